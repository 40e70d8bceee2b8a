"""The device workspace pool, with a host allocator in the device's place: what stays idle is bounded
per handle and over the process, goes with its handle and is given back when memory runs out."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_pool(tmp_path):
    exe = str(tmp_path / "dev_pool_check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-pthread", "-Wall", "-o", exe,
                    os.path.join(HERE, "dev_pool_check.cpp")], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout + r.stderr
