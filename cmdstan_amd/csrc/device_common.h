// Device helpers shared by the sampler and model kernels (gfx950, wave64).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define NUTS_WAVE 64

namespace nutsgpu {

// ------------------------------------------------------------ Philox4x32-10
// Salmon et al., SC'11.  Counter = (idx lo, idx hi, chain, purpose), key = seed.
struct U4 { uint32_t x, y, z, w; };

__device__ __forceinline__ U4 philox10(U4 c, uint32_t k0, uint32_t k1) {
#pragma unroll
  for (int r = 0; r < 10; ++r) {
    if (r > 0) { k0 += 0x9E3779B9u; k1 += 0xBB67AE85u; }
    const uint64_t p0 = (uint64_t)0xD2511F53u * c.x;
    const uint64_t p1 = (uint64_t)0xCD9E8D57u * c.z;
    U4 o;
    o.x = (uint32_t)(p1 >> 32) ^ c.y ^ k0;
    o.y = (uint32_t)p1;
    o.z = (uint32_t)(p0 >> 32) ^ c.w ^ k1;
    o.w = (uint32_t)p0;
    c = o;
  }
  return c;
}

enum : uint32_t { STREAM_UNIFORM = 0u, STREAM_NORMAL = 1u, STREAM_INIT = 2u };

__device__ __forceinline__ U4 stream_block(uint64_t seed, uint32_t chain, uint32_t purpose, uint64_t idx) {
  U4 c{(uint32_t)idx, (uint32_t)(idx >> 32), chain, purpose};
  return philox10(c, (uint32_t)seed, (uint32_t)(seed >> 32));
}

// (k + 0.5) * 2^-52 with k the top 52 of 64 random bits: exact, strictly in (0,1).
__device__ __forceinline__ double bits_to_unit(uint32_t a, uint32_t b) {
  const uint64_t k = ((uint64_t)a << 20) | (uint64_t)(b >> 12);
  return ((double)k + 0.5) * 2.220446049250313080847e-16;
}

__device__ __forceinline__ double stream_uniform(uint64_t seed, uint32_t chain, uint32_t purpose, uint64_t idx) {
  U4 r = stream_block(seed, chain, purpose, idx);
  return bits_to_unit(r.x, r.y);
}

// Box-Muller; element `which` (0: cos, 1: sin) of pair `idx`.  Out of line: the
// logarithm and the two angle reductions are 6 KB of instructions, and the
// state machine draws momenta in two places.
static __device__ __noinline__ double stream_normal(uint64_t seed, uint32_t chain, uint64_t idx, int which) {
  U4 r = stream_block(seed, chain, STREAM_NORMAL, idx);
  const double u1 = bits_to_unit(r.x, r.y);
  const double u2 = bits_to_unit(r.z, r.w);
  const double rad = sqrt(-2.0 * log(u1));
  const double ang = 6.283185307179586476925286766559 * u2;
  return which ? rad * sin(ang) : rad * cos(ang);
}

// ----------------------------------------------------------------- reductions
// One butterfly step on both halves of a double by a rotation inside rows of 16
// lanes: once lanes 8 apart hold the same value, rotating by 4 is the exchange
// of lanes 4 apart, and so on down.
template <int CTRL>
__device__ __forceinline__ double dpp_move(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xF, 0xF, false);
  return __hiloint2double(hi, lo);
}

__device__ __forceinline__ double uniform_value(double v) {
  return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(v)),
                          __builtin_amdgcn_readfirstlane(__double2loint(v)));
}

// Sums of N values over the wave, every lane gets them: the lane-xor butterfly
// (32, 16, 8, 4, 2, 1) with the additions of __shfl_xor's form -- the same bits
// -- on the vector unit's lane moves instead of six dependent trips through the
// LDS permute unit per value; the N chains interleave.
template <int N>
__device__ __forceinline__ void wave_sum_n(double (&v)[N]) {
#pragma unroll
  for (int k = 0; k < N; ++k) {  // upper half of a copy swapped for the lower: (lower, lower) + (upper, upper)
    const auto lo = __builtin_amdgcn_permlane32_swap(__double2loint(v[k]), __double2loint(v[k]), false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap(__double2hiint(v[k]), __double2hiint(v[k]), false, false);
    v[k] = __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
  }
#pragma unroll
  for (int k = 0; k < N; ++k) {  // the same with rows of 16
    const auto lo = __builtin_amdgcn_permlane16_swap(__double2loint(v[k]), __double2loint(v[k]), false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap(__double2hiint(v[k]), __double2hiint(v[k]), false, false);
    v[k] = __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
  }
#pragma unroll
  for (int k = 0; k < N; ++k) v[k] += dpp_move<0x128>(v[k]);  // row_ror:8
#pragma unroll
  for (int k = 0; k < N; ++k) v[k] += dpp_move<0x124>(v[k]);  // row_ror:4
#pragma unroll
  for (int k = 0; k < N; ++k) v[k] += dpp_move<0x122>(v[k]);  // row_ror:2
#pragma unroll
  for (int k = 0; k < N; ++k) v[k] = uniform_value(v[k] + dpp_move<0x121>(v[k]));  // row_ror:1
}

__device__ __forceinline__ double wave_sum(double v) {
  double a[1] = {v};
  wave_sum_n(a);
  return a[0];
}

// Positions of a batched gradient -> chains.  With the chains' request flags
// (`need`, at most 64 chains) every wave finds them by one ballot: position p is
// the p-th chain whose flag is set, so the launch needs no compaction kernel
// before it.  Otherwise the list idx (null: position = row) of *n_active (null:
// C) chains.
struct ActiveChains {
  int n;            // active positions
  int chain;        // flags: the chain of position `lane`
  bool flags;
  const int* idx;
  __device__ __forceinline__ ActiveChains(const int* need, const int* idx_, const int* n_active, int C)
      : chain(0), flags(need != nullptr), idx(idx_) {
    if (flags) {
      const int l = threadIdx.x & 63;
      const bool f = l < C && need[l] != 0;
      const unsigned long long m = __ballot(f);
      n = __popcll(m);
      const int r = __popcll(m & ((1ull << l) - 1));  // set flags below this lane
      chain = __builtin_amdgcn_ds_permute(4 * (f ? r : n + l - r), l);  // lane -> position, a permutation
    } else {
      n = n_active ? *n_active : C;
    }
  }
  // chain of a position, 0 past the last one; every lane of the wave takes part
  __device__ __forceinline__ int at(int pos) const {
    if (flags) {
      const int c = __shfl(chain, pos & 63, 64);
      return pos < n ? c : 0;
    }
    return pos < n ? (idx ? idx[pos] : pos) : 0;
  }
};

// and of 0/1 flags
__device__ __forceinline__ int wave_and(int v) { return __all(v != 0) ? 1 : 0; }

// ------------------------------------------------------------ scalar math
// 1/d for d in [1, 8]: the hardware reciprocal estimate refined by two Newton
// steps (no range reduction is needed in this range); within an ulp or two of
// the correctly rounded quotient, at about half the instructions of a division
__device__ __forceinline__ double recip_small(double d) {
  double x = __builtin_amdgcn_rcp(d);
  x = __builtin_fma(x, __builtin_fma(-d, x, 1.0), x);
  return __builtin_fma(x, __builtin_fma(-d, x, 1.0), x);
}

// Sum of log(1 + t) over many t in [0, 1] as the logarithm of their product: one
// fused multiply-add per term and one logarithm at the end.  u is the product
// minus one, (1 + u)(1 + t) - 1 = u (1 + t) + t, so a t far below the rounding
// of 1 counts in full; fold() after at most 900 terms brings 1 + u back into
// [1, 2) (u stays as it is while it is below 1).  Every operand is positive and
// rounds by 2^-53 of itself, so after n terms u, and with it log1p(u), is off by
// at most n 2^-52 of itself: like adding up n logarithms, measured no worse
// than 5e-15 (sum 5e-15) for 3000 terms up to |eta| = 10 and 2e-14 (sum 1e-14)
// at 50.  The product of the rounded 1 + t itself loses what of t lies below
// 2^-53: 1e-13 of the sum at |eta| = 10, all of it above 37.
struct LogProduct {
  double u = 0.0;
  int e = 0;
  __device__ __forceinline__ void times(double t, double one_plus_t) { u = __builtin_fma(u, one_plus_t, t); }
  __device__ __forceinline__ void fold() {
    const int x = __builtin_amdgcn_frexp_exp(1.0 + u) - 1;
    e += x;
    u = __builtin_amdgcn_ldexp(u, -x) + (__builtin_amdgcn_ldexp(1.0, -x) - 1.0);
  }
  // log1p(u) for u in [0, 1): log of the rounded d = 1 + u, plus what d leaves out
  // of u (over d, but that is within half a rounding of the result).  log1p's own
  // code is longer: glm_mfma_f64 at N = 10000, D = 25, 4 points 5.63 us with it, 5.47.
  __device__ __forceinline__ double log_value() {
    fold();
    const double d = 1.0 + u;
    return (log(d) + (u - (d - 1.0))) + (double)e * 0.69314718055994531;
  }
};

__device__ __forceinline__ double log1p_exp(double a) {
  return a > 0.0 ? a + log1p(exp(-a)) : log1p(exp(a));
}

// stan::math::log_sum_exp(double, double)
__device__ __forceinline__ double log_sum_exp2(double a, double b) {
  const double inf = __builtin_inf();
  if (a == -inf) return b;
  if (a == inf && b == inf) return inf;
  // one exponential and one logarithm in the code: the difference is not positive
  const double d = a > b ? b - a : a - b;
  return (a > b ? a : b) + log1p(exp(d));
}

__device__ __forceinline__ double inv_logit(double x) {
  if (x >= 0) return 1.0 / (1.0 + exp(-x));
  const double e = exp(x);
  return e / (1.0 + e);
}

}  // namespace nutsgpu
