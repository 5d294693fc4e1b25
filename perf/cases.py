"""The work this backend is measured on: calls a user's program makes through the public entry points.

Every case is a dict of plain values. ``kind`` names the path, the other keys its sizes, data type
and options:

    plain       the small plain configuration: broadcast add, an axis sum, an axis argmax and a matmul
    broadcast   elementwise product of a permuted, stepped 3-d view with a broadcast vector
    contig      contiguous copy of a permuted, stepped 3-d view
    reduce      sum, max and argmax of a permuted, stepped 3-d view, over axis 0 and over axes (1, 2)
    softmax     row softmax of a matrix: max_axes, subtract, exp, sum_axes, divide
    matvec      matrix times vector (or vector times matrix)
    matmul      plain matmul, optionally with transposed operands
    trsm        triangular solve with many right-hand sides through the BLAS driver
    grouped     many uneven matmuls in one grouped call
    ri          (ia|jb) = sum_P B[P,i,a] B[P,j,b], batched over i
    split       f64 matmul by the split-precision path, entries over a wide exponent range
    chain       complex128 step: broadcast add, product, split-precision matmul, axis sum

Sizes are those of the repository's five benchmark configurations where one exists, and generic
(odd and ragged ones among them) otherwise.
"""
import ctypes
import math

import numpy as np
import torch

import rstsr_amd as rt
from rstsr_amd import abi

_TORCH = {"f32": torch.float32, "f64": torch.float64, "i32": torch.int32, "c64": torch.complex64,
          "c128": torch.complex128}
_NUMPY = {"f32": np.float32, "f64": np.float64, "i32": np.int32, "c64": np.complex64, "c128": np.complex128}
_SIZE = {"f32": 4, "f64": 8, "i32": 4, "c64": 8, "c128": 16}
# argmax indices are u64; their bytes are handed on as i64, which torch can index and compare
_TYPESTR = {np.dtype(np.float32): "<f4", np.dtype(np.float64): "<f8", np.dtype(np.int32): "<i4",
            np.dtype(np.complex64): "<c8", np.dtype(np.complex128): "<c16", np.dtype(np.uint64): "<i8"}

# BLAS driver flags (cblas values): row major, left, lower / upper, no transpose, non-unit diagonal
_ROW_MAJOR, _LEFT, _NO_TRANS, _NON_UNIT = 101, 141, 111, 131
_UPLO = {"lower": 122, "upper": 121}


# ---------------------------------------------------------------- tensors both sides share


class _Storage:
    """A tensor's device storage, as the array interface torch reads without a copy."""

    def __init__(self, t):
        shape, stride, offset = t.layout
        it = np.dtype(t.dtype).itemsize
        self.tensor = t  # keeps the storage alive as long as torch's view of it
        self.__cuda_array_interface__ = {
            "shape": tuple(shape), "strides": tuple(s * it for s in stride), "typestr": _TYPESTR[np.dtype(t.dtype)],
            "data": (t.as_ptr() + offset * it, False), "version": 2}


def _torch(t):
    """torch's view of a tensor of this package: no copy, no synchronisation."""
    return torch.as_tensor(_Storage(t), device="cuda")


def _tensor(x):
    """A c-contiguous tensor of this package holding the torch tensor `x`."""
    t = rt.empty(x.shape, _NUMPY[{v: k for k, v in _TORCH.items()}[x.dtype]])
    _torch(t).copy_(x)
    return t


def _gen(seed, salt=0):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 64 + salt)
    return g


def _normal(shape, dtype, g, scale=1.0):
    """N(0, scale); complex: both parts. Integers: uniform over [-2^20, 2^20]."""
    if dtype == "i32":
        return torch.randint(-(1 << 20), (1 << 20) + 1, tuple(shape), generator=g, device="cuda", dtype=torch.int32)
    if dtype in ("c64", "c128"):
        real = torch.float32 if dtype == "c64" else torch.float64
        x = torch.randn(tuple(shape) + (2,), generator=g, device="cuda", dtype=real)
        return torch.view_as_complex(x.mul_(scale))
    return torch.randn(tuple(shape), generator=g, device="cuda", dtype=_TORCH[dtype]).mul_(scale)


def _uniform(shape, dtype, g, lo, hi):
    if dtype == "i32":
        return _normal(shape, dtype, g)
    if dtype in ("c64", "c128"):
        real = torch.float32 if dtype == "c64" else torch.float64
        x = torch.rand(tuple(shape) + (2,), generator=g, device="cuda", dtype=real)
        return torch.view_as_complex(x.mul_(hi - lo).add_(lo))
    return torch.rand(tuple(shape), generator=g, device="cuda", dtype=_TORCH[dtype]).mul_(hi - lo).add_(lo)


def _perm(case):
    return [int(c) for c in case["perm"]]


def _view_shape(case):
    """Shape of the permuted view with its last axis stepped."""
    s = [case["n%d" % p] for p in _perm(case)]
    s[2] = -(-s[2] // case["step"])
    return s


def _group_sizes(case, seed_free=20261202 + 3):
    """m, n, k of a grouped call: uniform multiples of `mult` in [lo, hi]; fixed for a case."""
    r = np.random.default_rng(seed_free)
    lo, hi, mult = case["lo"], case["hi"], case["mult"]
    return [tuple(int(v) * mult for v in r.integers(lo // mult, hi // mult + 1, size=3)) for _ in range(case["count"])]


def _inputs(case, seed):
    """The torch tensors a case starts from, from the seed alone."""
    g, k = _gen(seed), case["kind"]
    if k == "plain":
        n0, n1, n2, q = case["n0"], case["n1"], case["n2"], case["q"]
        return {"a": _uniform((n0, n1, n2), "f64", g, -1, 1), "b": _uniform((n2,), "f64", g, -1, 1),
                "p": _normal((q, q), "f64", g), "q": _normal((q, q), "f64", g)}
    if k in ("broadcast", "contig", "reduce"):
        x = {"x": _normal([case["n0"], case["n1"], case["n2"]], case["dtype"], g)}
        if k == "broadcast":
            x["b"] = _uniform([1, case["n1"], 1], case["dtype"], g, 0.5, 2.0)
        return x
    if k == "softmax":
        return {"x": _normal((case["rows"], case["cols"]), case["dtype"], g, 3.0)}
    if k == "matvec":
        a = _normal((case["m"], case["n"]), case["dtype"], g)
        return {"a": a, "v": _normal((case["m"] if case["left"] else case["n"],), case["dtype"], g)}
    if k == "matmul":
        m, n, kk = case["m"], case["n"], case["k"]
        return {"a": _normal((kk, m) if case["ta"] else (m, kk), case["dtype"], g),
                "b": _normal((n, kk) if case["tb"] else (kk, n), case["dtype"], g)}
    if k == "trsm":
        s = case["n"]
        a = _normal((s, s), case["dtype"], g, 0.5 / math.sqrt(s))
        a.diagonal().copy_(_uniform((s,), case["dtype"], g, 1.0, 2.0))
        return {"a": a, "b": _normal((s, case["rhs"]), case["dtype"], g)}
    if k == "grouped":
        return {"p": [(_normal((m, kk), case["dtype"], g), _normal((kk, n), case["dtype"], g))
                      for m, n, kk in _group_sizes(case)]}
    if k == "ri":
        return {"b": _normal((case["naux"], case["nocc"], case["nvir"]), "f64", g, 0.1)}
    if k == "split":
        def wide(shape):
            x = _normal(shape, "f64", g)
            return x.mul_(torch.exp2(torch.randint(-8, 9, tuple(shape), generator=g, device="cuda").double()))
        return {"a": wide((case["m"], case["k"])), "b": wide((case["k"], case["n"]))}
    if k == "chain":
        n = case["n"]
        return {"v": _normal((n,), "c128", g), "z1": _normal((n, n), "c128", g), "z2": _normal((n, n), "c128", g)}
    raise ValueError(k)


# ---------------------------------------------------------------- the cases


def listed():
    return [
        # a small user script, call by call: every launch is short, so latency and launch count weigh most
        {"name": "plain small f64", "kind": "plain", "n0": 64, "n1": 128, "n2": 256, "q": 512},
        # bandwidth-bound broadcast arithmetic on a permuted, stepped view (tensor contractions' prologues)
        {"name": "broadcast mul f64", "kind": "broadcast", "dtype": "f64", "n0": 256, "n1": 512, "n2": 1024,
         "perm": "201", "step": 2},
        # layout change of a medium tensor with odd extents: no row is a multiple of a tile or a 16-byte word
        {"name": "contig ragged f32", "kind": "contig", "dtype": "f32", "n0": 255, "n1": 509, "n2": 333, "perm": "210",
         "step": 1},
        # reductions of a large strided view over its leading axis and over the two trailing ones
        {"name": "reduce f64", "kind": "reduce", "dtype": "f64", "n0": 256, "n1": 512, "n2": 1024, "perm": "201",
         "step": 2},
        # per-row statistics and normalisation of many short odd rows
        {"name": "softmax short rows f32", "kind": "softmax", "dtype": "f32", "rows": 50021, "cols": 233},
        # matrix-vector product of an iterative solver (eigenvectors, linear systems)
        {"name": "matvec f64", "kind": "matvec", "dtype": "f64", "m": 8000, "n": 8000, "left": False},
        # single-precision matmul, ragged, one operand transposed
        {"name": "matmul ragged f32", "kind": "matmul", "dtype": "f32", "m": 2000, "n": 1511, "k": 3001, "ta": False,
         "tb": True},
        # triangular solve after a Cholesky or LU factorisation
        {"name": "trsm lower f64", "kind": "trsm", "dtype": "f64", "n": 2000, "rhs": 1600, "uplo": "lower"},
        # 512 uneven contractions in one grouped call
        {"name": "grouped 512 f64", "kind": "grouped", "dtype": "f64", "count": 512, "lo": 32, "hi": 1024, "mult": 8},
        # RI-style four-index integrals: the largest product and the largest output
        {"name": "ri (ia|jb) f64", "kind": "ri", "naux": 1600, "nocc": 60, "nvir": 400},
        # dense square product by the split-precision path
        {"name": "split 8192 f64", "kind": "split", "m": 8192, "n": 8192, "k": 8192},
        # complex propagation step
        {"name": "chain 4096 c128", "kind": "chain", "n": 4096},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    k = rng.choice(["plain", "broadcast", "contig", "reduce", "softmax", "matvec", "matmul", "trsm", "grouped", "ri",
                    "split", "chain"])
    if k == "plain":
        return {"kind": k, "n0": _log(rng, 4, 128), "n1": _log(rng, 8, 256), "n2": _log(rng, 16, 512),
                "q": _log(rng, 32, 768)}
    if k in ("broadcast", "contig", "reduce"):
        types = ["f64", "f32", "i32"] if k == "reduce" else ["f64", "f32", "i32", "c128"]
        return {"kind": k, "dtype": rng.choice(types), "n0": _log(rng, 16, 512), "n1": _log(rng, 16, 768),
                "n2": _log(rng, 16, 1024), "perm": rng.choice(["201", "210", "120", "102", "021"]),
                "step": rng.choice([1, 2])}
    if k == "softmax":
        cols = _log(rng, 16, 8192)
        return {"kind": k, "dtype": rng.choice(["f32", "f64"]), "rows": max(16, _log(rng, 1 << 16, 1 << 24) // cols),
                "cols": cols}
    if k == "matvec":
        return {"kind": k, "dtype": rng.choice(["f64", "f64", "f32", "c128"]), "m": _log(rng, 64, 12000),
                "n": _log(rng, 64, 12000), "left": rng.random() < 0.3}
    if k == "matmul":
        m, n, kk = (_log(rng, 48, 4096) for _ in range(3))
        while m * n * kk > 10 ** 10:  # no larger than the listed one
            m, n, kk = m * 3 // 4, n * 3 // 4, kk * 3 // 4
        return {"kind": k, "dtype": rng.choice(["f64", "f64", "f32", "f32", "c128", "c64"]), "m": m, "n": n, "k": kk,
                "ta": rng.random() < 0.3, "tb": rng.random() < 0.3}
    if k == "trsm":
        return {"kind": k, "dtype": rng.choice(["f64", "f64", "f32", "c128"]), "n": _log(rng, 96, 4096),
                "rhs": _log(rng, 16, 4096), "uplo": rng.choice(["lower", "upper"])}
    if k == "grouped":
        lo = rng.choice([16, 32, 64])
        return {"kind": k, "dtype": rng.choice(["f64", "f64", "c128"]), "count": _log(rng, 16, 512), "lo": lo,
                "hi": _log(rng, 4 * lo, 1024) // 8 * 8, "mult": rng.choice([1, 8])}
    if k == "ri":
        return {"kind": k, "naux": _log(rng, 200, 1600), "nocc": _log(rng, 6, 60), "nvir": _log(rng, 40, 400)}
    if k == "split":
        return {"kind": k, "m": _log(rng, 1024, 8192), "n": _log(rng, 1024, 8192), "k": _log(rng, 512, 8192)}
    return {"kind": k, "n": _log(rng, 768, 4096)}


def prepare(case, seed):
    """The tensors (and the problem list or the solve's arguments) a program holds before the call."""
    x, k = _inputs(case, seed), case["kind"]
    s = {"case": case}
    if k in ("broadcast", "contig", "reduce"):
        cut = (slice(None), slice(None), slice(None, None, case["step"]))
        s["x"] = _tensor(x["x"]).transpose(_perm(case))[cut]
        if k == "broadcast":
            s["b"] = _tensor(x["b"]).transpose(_perm(case))[cut]
    elif k == "matmul":
        a, b = _tensor(x["a"]), _tensor(x["b"])
        s["a"], s["b"] = a.transpose() if case["ta"] else a, b.transpose() if case["tb"] else b
    elif k == "trsm":
        s["a"], s["b"] = _tensor(x["a"]), _tensor(x["b"])
        s["y"] = rt.empty((case["n"], case["rhs"]), _NUMPY[case["dtype"]])
        s["one"] = np.array(1, dtype=_NUMPY[case["dtype"]])
    elif k == "grouped":
        # the products lie one after the other in one tensor, so that they can be handed on together
        c = rt.empty((sum(a.shape[0] * b.shape[1] for a, b in x["p"]),), _NUMPY[case["dtype"]])
        s["p"], at = [], 0
        for a, b in x["p"]:
            m, n = a.shape[0], b.shape[1]
            s["p"].append((_tensor(a), _tensor(b), c[at:at + m * n].reshape([m, n])))
            at += m * n
        s["c"] = _torch(c)
    elif k == "ri":
        b = _tensor(x["b"])
        n = case["nocc"] * case["nvir"]
        s["l"] = b.transpose([1, 2, 0])           # [i, a, P]
        s["r"] = b.reshape([case["naux"], n])     # [P, (j b)]
    else:
        for name, t in x.items():
            s[name] = _tensor(t)
    torch.cuda.synchronize()  # the tensors' own stream starts after torch's has filled them
    return s


def run(s):
    case = s["case"]
    k = case["kind"]
    if k == "plain":
        t = s["a"] + s["b"]
        return {"add": _torch(t), "sum": _torch(t.sum_axes(1)), "argmax": _torch(t.argmax_axes(2)),
                "matmul": _torch(s["p"] % s["q"])}
    if k == "broadcast":
        return _torch(s["x"] * s["b"])
    if k == "contig":
        return _torch(s["x"].to_contig())
    if k == "reduce":
        x = s["x"]
        return {"%s %s" % (n, ax): _torch(f(ax)) for n, f in
                (("sum", x.sum_axes), ("max", x.max_axes), ("argmax", x.argmax_axes)) for ax in (0, (1, 2))}
    if k == "softmax":
        x = s["x"]
        e = (x - x.max_axes(1).reshape([case["rows"], 1])).exp()
        return _torch(e / e.sum_axes(1).reshape([case["rows"], 1]))
    if k == "matvec":
        return _torch(s["v"] % s["a"] if case["left"] else s["a"] % s["v"])
    if k == "matmul":
        return _torch(s["a"] % s["b"])
    if k == "trsm":
        a, y = s["a"], s["y"]
        y.assign(s["b"])
        abi.check(abi.lib().rstsr_hip_driver_trsm(
            ctypes.c_void_p(y.device._ctx_ptr()), rt._code(y.dtype), rt.GEMM_PLAIN, _ROW_MAJOR, _LEFT,
            _UPLO[case["uplo"]], _NO_TRANS, _NON_UNIT, case["n"], case["rhs"], s["one"].ctypes.data, a.as_ptr(),
            case["n"], y.as_ptr(), case["rhs"]))
        return _torch(y)
    if k == "grouped":
        rt.gemm_grouped(s["p"])
        return s["c"]
    if k == "ri":
        return _torch(s["l"] % s["r"])
    if k == "split":
        return _torch(rt.matmul(s["a"], s["b"], mode="ozaki"))
    z = (s["z1"] + s["v"]) * s["z2"]
    y = rt.matmul(z, s["z2"], mode="ozaki")
    return {"y": _torch(y), "sum": _torch(y.sum_axes(1))}


def work(case):
    """Bytes (each input read once, each output written once) and operations of one pass. A complex
    product counts four real ones, a triangular solve and a symmetric product their half."""
    k = case["kind"]
    e = _SIZE[case.get("dtype", "f64")]
    cx = 4 if case.get("dtype") in ("c64", "c128") else 1
    if k == "plain":
        n = case["n0"] * case["n1"] * case["n2"]
        q = case["q"]
        return {"bytes": 8 * (2 * n + n // case["n1"] + n // case["n2"] + 3 * q * q), "flops": 2 * n + 2 * q ** 3}
    if k in ("broadcast", "contig", "reduce"):
        v = _view_shape(case)
        n = v[0] * v[1] * v[2]
        if k == "reduce":
            return {"bytes": e * n + (2 * e + 8) * (n // v[0] + v[0]), "flops": 6 * n}
        return {"bytes": 2 * e * n, "flops": n if k == "broadcast" else 0}
    if k == "softmax":
        n = case["rows"] * case["cols"]
        return {"bytes": 2 * e * n, "flops": 5 * n}
    if k == "matvec":
        m, n = case["m"], case["n"]
        return {"bytes": e * (m * n + m + n), "flops": 2 * cx * m * n}
    if k == "matmul":
        m, n, kk = case["m"], case["n"], case["k"]
        return {"bytes": e * (m * kk + kk * n + m * n), "flops": 2 * cx * m * n * kk}
    if k == "trsm":
        s, r = case["n"], case["rhs"]
        return {"bytes": e * (s * s // 2 + 2 * s * r), "flops": cx * s * s * r}
    if k == "grouped":
        g = _group_sizes(case)
        return {"bytes": e * sum(m * kk + kk * n + m * n for m, n, kk in g),
                "flops": 2 * cx * sum(m * n * kk for m, n, kk in g)}
    if k == "ri":
        n = case["nocc"] * case["nvir"]
        return {"bytes": 8 * (case["naux"] * n + n * n), "flops": n * (n + 1) * case["naux"]}
    if k == "split":
        m, n, kk = case["m"], case["n"], case["k"]
        return {"bytes": 8 * (m * kk + kk * n + m * n), "flops": 2 * m * n * kk}
    n = case["n"]
    return {"bytes": 16 * (3 * n * n + 2 * n), "flops": 8 * n ** 3 + 10 * n * n}


def exact(case, seed):
    """What run() returns, by plain torch in 64 bits (indices and integers: no value of this kind)."""
    x, k = _inputs(case, seed), case["kind"]

    def wide(t):
        return t.to(torch.complex128 if t.is_complex() else torch.float64)

    if k == "plain":
        t = x["a"] + x["b"]
        return {"add": t, "sum": t.sum(1), "argmax": None, "matmul": x["p"] @ x["q"]}
    if k in ("broadcast", "contig", "reduce"):
        if case["dtype"] == "i32":
            return None
        v = x["x"].permute(_perm(case))[:, :, :: case["step"]]
        if k == "broadcast":
            return wide(v) * wide(x["b"]).permute(_perm(case))[:, :, :: case["step"]]
        if k == "contig":
            return wide(v).contiguous()
        out = {}
        for ax in (0, (1, 2)):
            out["sum %s" % (ax,)] = wide(v).sum(ax)
            out["max %s" % (ax,)] = wide(v).amax(ax)
            out["argmax %s" % (ax,)] = None
        return out
    if k == "softmax":
        return torch.softmax(wide(x["x"]), 1)
    if k == "matvec":
        return wide(x["v"]) @ wide(x["a"]) if case["left"] else wide(x["a"]) @ wide(x["v"])
    if k == "matmul":
        a, b = wide(x["a"]), wide(x["b"])
        return (a.T if case["ta"] else a) @ (b.T if case["tb"] else b)
    if k == "trsm":
        return torch.linalg.solve_triangular(wide(x["a"]), wide(x["b"]), upper=case["uplo"] == "upper")
    if k == "grouped":
        return torch.cat([(wide(a) @ wide(b)).reshape(-1) for a, b in x["p"]])
    if k == "ri":
        b = x["b"].reshape(case["naux"], -1)
        n = case["nvir"]
        return torch.stack([b[:, i * n:(i + 1) * n].T.contiguous() @ b for i in range(case["nocc"])])
    if k == "split":
        return x["a"] @ x["b"]
    y = ((x["z1"] + x["v"]) * x["z2"]) @ x["z2"]
    return {"y": y, "sum": y.sum(1)}

