"""Tuned launches forced to every candidate of their class, beyond the products of test_gpu_tuner and the
whole-line shape of test_gpu_elementwise: f32, c64 and symmetric c128 products, and transposing
element-wise launches whose lines or tiles are cut, with and without streaming hints.

A first process tunes and records its choices in a cache file (the tuner's own format); fresh processes
run the same calls with every recorded choice forced to each index its class has. Small-integer
operands make every product exact, and element-wise results are compared bit for bit.
"""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

_GEMM = r"""
import sys
import numpy as np
sys.path.insert(0, sys.argv[1]); sys.path.insert(0, sys.argv[1] + "/tests")
import rstsr_amd as rt
from test_gpu_gemm_tile import embed, ints, product
dev = rt.DeviceHIP(0)
rng = np.random.default_rng(41)
bad = []
for dt in (np.float32, np.complex64, np.complex128):
    for m, n, k in [(300, 261, 97), (128, 129, 33), (70, 515, 200)]:
        a, b = ints(rng, (m, k), dt), ints(rng, (k, n), dt)
        want = product(a, b).astype(dt)
        for fa, fb in ("cc", "cf", "fc", "ff"):
            if not np.array_equal((embed(dev, a, fa) % embed(dev, b, fb)).to_numpy(), want):
                bad.append((np.dtype(dt).char, m, n, k, fa, fb))
    for k, n in [(97, 300), (130, 129)]:
        x = ints(rng, (k, n), dt)
        for f in "cf":
            t = embed(dev, x, f)
            if not np.array_equal((t.transpose() % t).to_numpy(), product(x.T, x).astype(dt)):
                bad.append((np.dtype(dt).char, "sym", k, n, f))
dev.synchronize()
print("BAD", bad) if bad else print("ALL_OK", flush=True)
"""

_EW = r"""
import sys
import numpy as np
sys.path.insert(0, sys.argv[1])
import rstsr_amd as rt
dev = rt.DeviceHIP(0)
rng = np.random.default_rng(42)
bad = []
# whole tiles, whole lines with ragged tiles, cut lines; the last of each moves more than 288 MB
shapes = {np.float32: [(4096, 2304), (4000, 2080), (3001, 2803), (8000, 3104), (5003, 5001)],
          np.float64: [(2048, 2304), (2000, 2080), (3001, 2003), (5008, 2608), (5003, 2501)],
          np.complex128: [(2048, 1152), (2008, 1000), (2003, 1001), (4001, 1603), (60000, 20)]}
for dt, shs in shapes.items():
    for m, n in shs:
        x = rng.integers(-50, 51, size=(n, m)).astype(dt)
        y = rng.integers(-50, 51, size=(m, n)).astype(dt)
        r = rng.integers(1, 9, size=(n, 1)).astype(dt)
        t, u, v = (rt.asarray(z, device=dev) for z in (x, y, r))
        t, v = t.transpose(), v.transpose()
        for name, got, want in (("copy", t.to_contig(), x.T), ("plus", u + t, y + x.T), ("times", t * u, x.T * y),
                                ("row", t * v, x.T * r.T), ("both", t - t, x.T - x.T)):
            if not np.array_equal(got.to_numpy(), want):
                bad.append((np.dtype(dt).char, m, n, name))
dev.synchronize()
print("BAD", bad) if bad else print("ALL_OK", flush=True)
"""


def _force_all(tmp_path, script, prefix, ncand):
    cache = tmp_path / "tune.txt"
    env = dict(os.environ, RSTSR_HIP_TUNE_CACHE=str(cache))
    env.pop("RSTSR_HIP_NO_TUNE", None)

    def child():
        r = subprocess.run([sys.executable, "-c", script, ROOT], env=env, capture_output=True, text=True, timeout=100)
        assert r.returncode == 0, r.stderr[-2000:]
        assert "ALL_OK" in r.stdout, r.stdout[-2000:]

    child()
    keys = sorted({ln.split()[0] for ln in cache.read_text().splitlines() if ln.startswith(prefix)})
    for c in range(4):
        cache.write_text("".join(f"{k} {min(c, ncand(k) - 1)}\n" for k in keys))
        child()
        assert len(cache.read_text().splitlines()) == len(keys)  # nothing was tuned anew
    return keys


def test_products(tmp_path):
    keys = _force_all(tmp_path, _GEMM, "gemm:", lambda k: 2 if k.startswith("gemm:c:") else 3)
    for tag in ("s", "c", "z2"):
        forms = {int(k.rsplit(":f", 1)[1]) for k in keys if k.startswith(f"gemm:{tag}:")}
        assert len(forms) >= 4 and any(f & 8 for f in forms), (tag, forms)


def test_elementwise(tmp_path):
    # candidates: two orders for lines cut in launches of up to 8-byte outputs, otherwise four
    keys = _force_all(tmp_path, _EW, "ew|", lambda k: 2 if k.startswith("ew|c|") and k.split("|")[3] != "16" else 4)
    assert any(k.startswith("ew|c|") for k in keys) and any(not k.startswith("ew|c|") for k in keys)
