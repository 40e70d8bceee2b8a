"""Measured workloads of the sampler: what a user of this framework runs, through
its public entry points, over the sizes it is used at.

Four kinds of call:

* ``sample``    ``Model.sample``: warmup and draws of every chain of a model or of a
                batch of models, host arrays out.
* ``gradient``  ``nuts_log_prob_grad_noalloc``: FP64 log densities and gradients of
                many points in device buffers (graph capture, serving loops).
* ``log_prob``  ``Model.log_prob_grad``: the ``log_prob`` method on host arrays, here
                with the FP32 and BF16 contraction of the logistic regression.
* ``flow``      ``Flow``: the learned reparameterisation's map, its pullback and its
                training gradient on host arrays.

Results that a call computes in FP32 (the reduced contractions, the FP32 leapfrog,
the flow) are handed on as FP32; everything else stays FP64.
"""
import ctypes
import math

import torch  # first: the library then shares torch's HIP runtime
import numpy as np

import cmdstan_amd as ca
from cmdstan_amd._lib import last_error, lib

FLOW_LAYERS, FLOW_HIDDEN = 8, 128


def listed():
    return [
        # the four-chain default run of a tiny model (bernoulli example: N = 10, 1000 + 1000): latency only
        dict(name="sample_bernoulli", kind="sample", family="bernoulli", N=10, chains=4, warmup=1000, draws=1000,
             metric="diag_e"),
        # sampling phase of a 100-dimensional correlated Gaussian, dense metric, four chains: the usual dense_e run
        dict(name="sample_gauss_dense", kind="sample", family="gauss", D=100, chains=4, warmup=0, draws=200,
             metric="dense_e"),
        # many non-centered hierarchical models of uneven size in one batch, a bounded part of each draw kept
        dict(name="sample_hier_batch", kind="sample", family="hier_normal_nc", models=64, Jmin=8, Jmax=2000,
             chains=32, warmup=0, draws=12, metric="diag_e", precision="fp64"),
        # sampling phase of a logistic regression as most users run it: four chains, a moderate table
        dict(name="sample_logistic_few", kind="sample", family="logistic_regression", N=10000, D=25, chains=4,
             warmup=0, draws=250, metric="diag_e"),
        # the sampling phase of the headline workload: 100000 x 100, 1024 chains
        dict(name="sample_logistic_many", kind="sample", family="logistic_regression", N=100000, D=100, chains=1024,
             warmup=0, draws=10, metric="diag_e"),
        # sampling phase of a centered hierarchical logistic regression, 400 groups x 10 covariates (D = 4020)
        dict(name="sample_hier_logistic", kind="sample", family="hier_logistic_cp", N=50000, G=400, K=10, chains=256,
             warmup=0, draws=10, metric="diag_e"),
        # the same family small enough for a dense metric (given, as from a metric file)
        dict(name="sample_dense_block", kind="sample", family="hier_logistic_cp", N=5000, G=50, K=10, chains=64,
             warmup=0, draws=10, metric="dense_e"),
        # one FP64 gradient of all chains at the headline shape
        dict(name="gradient_fp64", kind="gradient", family="logistic_regression", N=100000, D=100, points=1024),
        # FP64 gradients of a wide table (more than 128 coefficients), a modest number of points
        dict(name="gradient_fp64_wide", kind="gradient", family="logistic_regression", N=10000, D=500, points=64),
        # a wide table stored in BF16, 512 points
        dict(name="log_prob_bf16_wide", kind="log_prob", N=50000, D=1000, points=512, precision="bf16"),
        # the flow of the 4020-dimensional model at 256 rows: what a leaf of NUTS on the flow adds
        dict(name="flow_pullback", kind="flow", op="pullback", G=400, K=10, rows=256),
        # and the gradient of one training batch
        dict(name="flow_loss_grad", kind="flow", op="loss_grad", G=400, K=10, rows=256),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    """Another case of the listed kinds; sizes over the whole range, ragged ones included."""
    kind = rng.choice(["sample_small", "sample_gauss", "sample_hier", "sample_logistic", "sample_adapted",
                       "sample_hier_logistic", "gradient", "gradient_wide", "gradient_hier", "log_prob",
                       "log_prob_wide", "flow", "flow"])
    if kind == "sample_small":
        return dict(kind="sample", family="bernoulli", N=_log_int(rng, 5, 20000), chains=_log_int(rng, 1, 64),
                    warmup=_log_int(rng, 100, 1000), draws=_log_int(rng, 100, 1000), metric="diag_e")
    if kind == "sample_gauss":
        return dict(kind="sample", family="gauss", D=_log_int(rng, 2, 160), chains=_log_int(rng, 1, 64), warmup=0,
                    draws=rng.randint(40, 200), metric=rng.choice(["diag_e", "dense_e"]))
    if kind == "sample_hier":
        return dict(kind="sample", family="hier_normal_nc", models=_log_int(rng, 2, 64), Jmin=8,
                    Jmax=_log_int(rng, 40, 2000), chains=_log_int(rng, 4, 32), warmup=0, draws=rng.randint(4, 12),
                    metric="diag_e", precision=rng.choice(["fp64", "fp64", "fp32"]))
    if kind == "sample_logistic":
        return dict(kind="sample", family="logistic_regression", N=_log_int(rng, 500, 20000), D=_log_int(rng, 2, 64),
                    chains=_log_int(rng, 1, 16), warmup=0, draws=rng.randint(50, 250), metric="diag_e")
    if kind == "sample_adapted":
        return dict(kind="sample", family="logistic_regression", N=_log_int(rng, 10000, 100000),
                    D=_log_int(rng, 10, 100), chains=_log_int(rng, 64, 1024), warmup=0, draws=rng.randint(5, 10),
                    metric="diag_e")
    if kind == "sample_hier_logistic":
        K = rng.randint(2, 10)
        dense = rng.random() < 0.4
        G = _log_int(rng, 10, 50) if dense else _log_int(rng, 10, 400)
        return dict(kind="sample", family="hier_logistic_cp", N=G * rng.randint(20, 125), G=G, K=K,
                    chains=_log_int(rng, 4, 64 if dense else 256), warmup=0, draws=rng.randint(4, 10), metric="dense_e" if dense else "diag_e")
    if kind == "gradient":
        return dict(kind="gradient", family="logistic_regression", N=_log_int(rng, 1000, 100000),
                    D=_log_int(rng, 2, 128), points=_log_int(rng, 1, 1024))
    if kind == "gradient_wide":
        return dict(kind="gradient", family="logistic_regression", N=_log_int(rng, 1000, 10000),
                    D=_log_int(rng, 129, 500), points=_log_int(rng, 1, 64))
    if kind == "gradient_hier":
        G = _log_int(rng, 10, 400)
        return dict(kind="gradient", family="hier_logistic_cp", N=G * rng.randint(20, 125), G=G, K=rng.randint(1, 10),
                    points=_log_int(rng, 1, 256))
    if kind == "log_prob":
        return dict(kind="log_prob", N=_log_int(rng, 2000, 100000), D=_log_int(rng, 4, 128),
                    points=_log_int(rng, 16, 1024), precision=rng.choice(["fp32", "bf16"]))
    if kind == "log_prob_wide":
        return dict(kind="log_prob", N=_log_int(rng, 5000, 50000), D=_log_int(rng, 136, 1000),
                    points=_log_int(rng, 16, 512), precision=rng.choice(["bf16", "bf16", "fp32"]))
    return dict(kind="flow", op=rng.choice(["forward", "inverse", "pullback", "loss_grad"]), G=_log_int(rng, 20, 400),
                K=rng.randint(2, 10), rows=_log_int(rng, 16, 256))


# ------------------------------------------------------------------ data of a case
def _sigmoid(x):
    return 1.0 / (1.0 + np.exp(-x))


def _logistic_data(case, rng):
    N, D = case["N"], case["D"]
    X = rng.standard_normal((N, D), dtype=np.float32).astype(np.float64)
    beta = rng.normal(0, math.sqrt(1.0 / D), D)
    y = (rng.random(N) < _sigmoid(X @ beta)).astype(np.int64)
    return dict(N=N, D=D, X=X, y=y), beta


def _hier_logistic_data(case, rng):
    N, G, K = case["N"], case["G"], case["K"]
    X = rng.standard_normal((N, K), dtype=np.float32).astype(np.float64)
    grp = np.arange(N) * G // N
    mu = rng.normal(0, 1, K)
    tau = np.abs(rng.normal(0, 1, K))
    beta = mu + tau * rng.standard_normal((G, K))
    y = (rng.random(N) < _sigmoid((X * beta[grp]).sum(axis=1))).astype(np.int64)
    q = np.concatenate([mu, np.log(tau + 0.05), beta.ravel()])
    return dict(N=N, K=K, G=G, X=X, y=y, group=grp + 1), q


def _hier_normal_data(rng, J):
    sigma = rng.uniform(5, 20, J)
    mu, tau = rng.normal(0, 5), abs(rng.standard_cauchy()) * 5
    theta = mu + tau * rng.standard_normal(J)
    return dict(J=J, y=rng.normal(theta, sigma), sigma=sigma)


def _gauss_data(rng, D):
    A = rng.standard_normal((D, D))
    return dict(D=D, mu=rng.standard_normal(D), P=A @ A.T / D + 0.5 * np.eye(D))


def _gradient_data(case, seed):
    """Data and the points of a gradient call: chains spread around the posterior."""
    rng = np.random.default_rng(seed)
    if case.get("family") == "hier_logistic_cp":
        data, centre = _hier_logistic_data(case, rng)
        spread = 0.1
    else:
        data, centre = _logistic_data(case, rng)
        spread = 3.0 * math.sqrt(5.0 / case["N"])
    q = centre + spread * rng.standard_normal((case["points"], centre.size))
    return data, q


def _flow_masks(D, n_glob, group):
    """Coupling masks: globals + even groups | odd, globals + odd | even, all groups | globals."""
    loc = np.arange(n_glob, D)
    even, odd = loc[((loc - n_glob) // group) % 2 == 0], loc[((loc - n_glob) // group) % 2 == 1]
    glob = np.arange(n_glob)
    per = [(np.r_[glob, even], odd), (np.r_[glob, odd], even), (loc, glob)]
    return [per[l % 3] for l in range(FLOW_LAYERS)]


def _flow_data(case, seed):
    rng = np.random.default_rng(seed)
    K, n = case["K"], case["rows"]
    D, H = 2 * K + case["G"] * K, FLOW_HIDDEN
    parts = []
    for a, b in _flow_masks(D, 2 * K, K):
        for fan_in, fan_out in ((len(a), H), (H, H)):
            lim = math.sqrt(6.0 / (fan_in + fan_out))
            parts += [rng.uniform(-lim, lim, fan_in * fan_out), np.zeros(fan_out)]
        parts += [rng.normal(0, 0.02, H * 2 * len(b)), rng.normal(0, 0.02, 2 * len(b))]
    params = np.concatenate(parts).astype(np.float32)
    loc, scale = rng.normal(0, 1, D), np.exp(rng.normal(-1, 0.5, D))
    rows, gx = rng.standard_normal((n, D)), rng.standard_normal((n, D))
    if case["op"] in ("inverse", "loss_grad"):
        rows = loc + scale * rows
    return D, params, loc, scale, rows, gx


# ------------------------------------------------------------------ prepare / run
def _prepare_sample(case, seed):
    """The model and what a run of the sampling phase is started with: the state warmup leaves behind
    (chains spread around the posterior, step size, metric).  Warmup itself runs the same kernels, but its
    step-size feedback turns a last-bit difference into different trajectories; the bernoulli case has it."""
    rng = np.random.default_rng(seed)
    fam, dense = case["family"], case["metric"] == "dense_e"
    args = dict(num_chains=case["chains"], num_warmup=case["warmup"], num_samples=case["draws"],
                metric=case["metric"], seed=seed % 100003 + 1, adapt_engaged=case["warmup"] > 0)
    spread = None
    if fam == "bernoulli":
        data = dict(N=case["N"], y=(rng.random(case["N"]) < 0.2).astype(np.int64))
    elif fam == "gauss":
        data = _gauss_data(rng, case["D"])
        cov = np.linalg.inv(data["P"])
        centre, spread, eps = data["mu"], np.sqrt(np.diag(cov)), 0.9 * case["D"] ** -0.25
        metric = cov if dense else spread ** 2
        eps *= 1.0 if dense else 0.4
    elif fam == "hier_normal_nc":
        # uneven dimensions take no arrays: unit metric from small random positions
        sizes = np.random.default_rng(case["models"])  # the sizes belong to the case, not to the seed
        data = [_hier_normal_data(rng, int(J))
                for J in sizes.integers(case["Jmin"], case["Jmax"] + 1, case["models"])]
        args.update(max_saved_params=10, precision=case["precision"], init=0.5, stepsize=0.04)
    elif fam == "hier_logistic_cp":
        # scales from the information of a group's rows
        data, centre = _hier_logistic_data(case, rng)
        K, G = case["K"], case["G"]
        tau = np.exp(centre[K:2 * K])
        var = np.concatenate([tau ** 2 / G, np.full(K, 0.6 / G),
                              np.tile(1.0 / (0.15 * case["N"] / G + 1.0 / tau ** 2), G)])
        spread, eps, metric = 0.5 * np.sqrt(var), 0.15, np.diag(var) if dense else var
    else:
        data, centre = _logistic_data(case, rng)
        spread = np.full(case["D"], math.sqrt(5.0 / case["N"]))
        eps, metric = 0.6, spread ** 2
    if spread is not None:
        args.update(stepsize=eps, inv_metric=metric,
                    init=centre + spread * rng.standard_normal((case["chains"], spread.size)))
    return dict(kind="sample", model=ca.Model(fam, data), args=args)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "sample":
        return _prepare_sample(case, seed)
    if kind == "gradient":
        data, q = _gradient_data(case, seed)
        model = ca.Model(case["family"], data)
        dq = torch.from_numpy(q).cuda()
        return dict(kind=kind, model=model, q=dq, n=case["points"], lp=torch.empty(case["points"], dtype=dq.dtype,
                                                                                 device=dq.device),
                    grad=torch.empty_like(dq))
    if kind == "log_prob":
        data, q = _gradient_data(case, seed)
        return dict(kind=kind, model=ca.Model("logistic_regression", data), q=q, precision=case["precision"])
    D, params, loc, scale, rows, gx = _flow_data(case, seed)
    flow = ca.sampler.Flow(D, n_layers=FLOW_LAYERS, hidden=FLOW_HIDDEN, n_glob=2 * case["K"], group_size=case["K"],
                           max_rows=case["rows"])
    flow.set_params(params)
    flow.set_standardization(loc, scale)
    return dict(kind=kind, op=case["op"], flow=flow, rows=rows, gx=gx)


def run(state):
    kind = state["kind"]
    if kind == "sample":
        fit = state["model"].sample(**state["args"])
        vectors = np.float32 if state["args"].get("precision") == "fp32" else np.float64
        return dict(draws=np.concatenate([d.ravel() for d in fit.draws]).astype(vectors, copy=False),
                    stepsize=fit.stepsize, n_leapfrog=fit.n_leapfrog, status=fit.status,
                    inv_metric=np.concatenate([m.ravel() for m in fit.inv_metric]).astype(vectors, copy=False))
    if kind == "gradient":
        stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        ptr = [ctypes.c_void_p(state[k].data_ptr()) for k in ("q", "lp", "grad")]
        if lib().nuts_log_prob_grad_noalloc(state["model"].h, 0, ptr[0], state["n"], 1, ptr[1], ptr[2], stream) != 0:
            raise RuntimeError(last_error())
        return dict(lp=state["lp"], grad=state["grad"])
    if kind == "log_prob":
        lp, grad = state["model"].log_prob_grad(state["q"], precision=state["precision"])
        return dict(lp=lp.astype(np.float32), grad=grad.astype(np.float32))
    flow, op, rows = state["flow"], state["op"], state["rows"]
    if op == "pullback":
        return dict(gz=flow.pullback_grad(rows, state["gx"]).astype(np.float32))
    if op == "loss_grad":
        loss, grad = flow.loss_grad(rows)
        return dict(loss=np.float32(loss), grad=grad)
    out, logdet = flow.forward(rows) if op == "forward" else flow.inverse(rows)
    return dict(rows=out.astype(np.float32), logdet=logdet.astype(np.float32))


# ------------------------------------------------------------------ work of one pass
def _gradient_work(family, case, points, dim):
    """(bytes, flops) of one batched gradient: data once, a position and a gradient row per point."""
    rows = 16.0 * points * dim
    if family == "logistic_regression":
        return 8.0 * case["N"] * (dim + 1) + rows, 4.0 * case["N"] * dim * points
    if family == "hier_logistic_cp":
        return 8.0 * case["N"] * (case["K"] + 1) + rows, 4.0 * case["N"] * case["K"] * points
    if family == "gauss":
        return 8.0 * dim * dim + rows, 2.0 * dim * dim * points
    return 2 * rows, 12.0 * dim * points


def work(case):
    kind = case["kind"]
    if kind == "gradient":
        D = case.get("D") or (2 + case["G"]) * case["K"]
        b, f = _gradient_work(case["family"], case, case["points"], D)
        return dict(bytes=b, flops=f)
    if kind == "log_prob":
        size = 4 if case["precision"] == "fp32" else 2
        N, D, n = case["N"], case["D"], case["points"]
        return dict(bytes=float(N) * D * size + 8.0 * N + 16.0 * n * D, flops=4.0 * N * D * n)
    if kind == "flow":
        K, n, H = case["K"], case["rows"], FLOW_HIDDEN
        D = 2 * K + case["G"] * K
        mlp = sum(len(a) * H + H * H + 2 * H * len(b) for a, b in _flow_masks(D, 2 * K, K))
        passes = {"forward": 1, "inverse": 1, "pullback": 2, "loss_grad": 3}[case["op"]]
        extra = 8.0 * n * D if case["op"] == "pullback" else 0.0
        out = 4.0 * mlp if case["op"] == "loss_grad" else 8.0 * n * D
        return dict(bytes=4.0 * mlp + 8.0 * n * D + extra + out, flops=2.0 * passes * mlp * n)
    # one gradient per leapfrog step, and per step the chain's position, momentum, gradient, metric and one kept
    # state read and written once; steps per transition as these step sizes give them (trees of depth 2 to 6)
    steps = {"bernoulli": 2.7, "gauss": 15.0, "hier_normal_nc": 95.0, "hier_logistic_cp": 31.0,
             "logistic_regression": 7.0}[case["family"]]
    fam, transitions = case["family"], case["warmup"] + case["draws"]
    chains = case["chains"] * case.get("models", 1)
    if fam == "bernoulli":
        dim = 1
    elif fam == "hier_normal_nc":
        dim = 2 + (case["Jmin"] + case["Jmax"]) // 2
    elif fam == "hier_logistic_cp":
        dim = (2 + case["G"]) * case["K"]
    else:
        dim = case["D"]
    b, f = _gradient_work(fam, case, chains, dim)
    vectors = 8.0 * 11 * dim * chains
    if case["metric"] == "dense_e":
        vectors += 8.0 * dim * dim * chains
    return dict(bytes=steps * transitions * (b + vectors), flops=steps * transitions * f)


# ------------------------------------------------------------------ the values in 64 bits
def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _log_density(case, data, q):
    """Log density (up to a constant, Jacobian included) of each row of q."""
    dev = q.device
    X = torch.as_tensor(data["X"], device=dev)
    y = torch.as_tensor(data["y"], device=dev, dtype=torch.float64)

    def likelihood(eta, y):
        ls = torch.nn.functional.logsigmoid
        return (y * ls(eta) + (1 - y) * ls(-eta)).sum(dim=1)

    if case.get("family", "logistic_regression") == "logistic_regression":
        if case.get("precision") == "bf16":  # the stored table
            X = X.to(torch.bfloat16).double()
        elif case.get("precision") == "fp32":
            X = X.float().double()
        return likelihood(q @ X.T, y) - 0.5 * (q * q).sum(dim=1) / 2.5 ** 2
    K, G = case["K"], case["G"]
    mu, v, beta = q[:, :K], q[:, K:2 * K], q[:, 2 * K:].reshape(-1, G, K)
    tau = torch.exp(v)
    z = (beta - mu[:, None, :]) / tau[:, None, :]
    lp = (-0.5 * z * z - v[:, None, :]).sum(dim=(1, 2))
    lp = lp + (-0.5 * mu * mu / 25.0 - 0.5 * tau * tau + v).sum(dim=1)
    grp = torch.as_tensor(data["group"], device=dev) - 1
    eta = sum(X[:, k] * beta[:, grp, k] for k in range(K))
    return lp + likelihood(eta, y)


def _flow_mlp(p, off, a, b, u):
    """(s, t) of one coupling layer whose parameters start at p[off]."""
    H, out = FLOW_HIDDEN, u[:, a]
    for layer, (fan_in, fan_out) in enumerate(((len(a), H), (H, H), (H, 2 * len(b)))):
        W = p[off:off + fan_in * fan_out].reshape(fan_in, fan_out)
        out = out @ W + p[off + fan_in * fan_out:off + fan_in * fan_out + fan_out]
        off += fan_in * fan_out + fan_out
        if layer < 2:
            out = torch.tanh(out)
    return 3.0 * torch.tanh(out[:, :len(b)] / 3.0), out[:, len(b):]


def _exact_flow(case, seed):
    D, params, loc, scale, rows, gx = _flow_data(case, seed)
    dev = _device()
    t = lambda x: torch.as_tensor(x, device=dev, dtype=torch.float64)  # noqa: E731
    p, loc, scale, rows, gx = t(params), t(loc), t(scale), t(rows), t(gx)
    masks, offs, at = _flow_masks(D, 2 * case["K"], case["K"]), [], 0
    H = FLOW_HIDDEN
    for a, b in masks:
        offs.append(at)
        at += len(a) * H + H + H * H + H + H * 2 * len(b) + 2 * len(b)
    op = case["op"]
    need_p = op == "loss_grad"
    p.requires_grad_(need_p)
    rows.requires_grad_(op == "pullback")
    cols = [(torch.as_tensor(a, device=dev), torch.as_tensor(b, device=dev)) for a, b in masks]

    def couple(u, b, ub):
        return u.index_copy(1, b, ub)

    if op in ("forward", "pullback"):
        u, ld = rows, 0.0
        for (a, b), o in zip(cols, offs):
            s, sh = _flow_mlp(p, o, a, b, u)
            u, ld = couple(u, b, u[:, b] * torch.exp(s) + sh), ld + s.sum(dim=1)
        x, ld = loc + scale * u, ld + torch.log(scale).sum()
        if op == "forward":
            return dict(rows=x.cpu().numpy(), logdet=ld.cpu().numpy())
        ((gx * x).sum() - ld.sum()).backward()
        return dict(gz=rows.grad.cpu().numpy())
    u, ld = (rows - loc) / scale, 0.0
    for (a, b), o in reversed(list(zip(cols, offs))):
        s, sh = _flow_mlp(p, o, a, b, u)
        u, ld = couple(u, b, (u[:, b] - sh) * torch.exp(-s)), ld - s.sum(dim=1)
    ld = ld - torch.log(scale).sum()
    if op == "inverse":
        return dict(rows=u.cpu().numpy(), logdet=ld.cpu().numpy())
    loss = (0.5 * (u * u).sum(dim=1) - ld).mean()
    loss.backward()
    return dict(loss=float(loss.detach()), grad=p.grad.cpu().numpy())


def exact(case, seed):
    if case["kind"] == "sample":
        return None  # a chain of random transitions: no closed form
    if case["kind"] == "flow":
        return _exact_flow(case, seed)
    data, q = _gradient_data(case, seed)
    lps, grads = [], []
    step = max(1, int(2e8 // case["N"]))  # points per slice: a few GB of intermediates
    for k in range(0, q.shape[0], step):
        part = torch.tensor(q[k:k + step], device=_device(), requires_grad=True)
        lp = _log_density(case, data, part)
        grads.append(torch.autograd.grad(lp.sum(), part)[0].cpu().numpy())
        lps.append(lp.detach().cpu().numpy())
    return dict(lp=np.concatenate(lps), grad=np.concatenate(grads))
