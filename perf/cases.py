"""Workloads of the library as its users run them, for timing and for comparing outputs.

Operands are tracked objects that already live in HBM (what an application linked against or
preloaded with the library has after its first calls), and a pass calls the Fortran-ABI entry
points as a C or Fortran program does: scalars by reference, arrays by host address.  The batch
slot and the split-precision product, which have entry points of their own, take device addresses.

Matrices are column-major.  Here one is a tensor of shape (columns, leading dimension), so
storage order and the rows past m in each column (random, never to be touched) come with it.
"""
import ctypes
import math

import numpy as np
import torch

import libgpublas_amd as gb

F64, F32 = "float64", "float32"
SLICE_INT8 = 2


# --------------------------------------------------------------------------- cases
def listed():
    return [
        # the smallest products an application hands over (one block of a blocked factorisation,
        # a small element matrix): launches and latency
        {"name": "dgemm_small", "op": "gemm", "prec": "d", "ta": "N", "tb": "N",
         "m": 100, "n": 100, "k": 100, "pad": 0, "beta": 0.5},
        # the library's first benchmark configuration: an ordinary mid-size product
        {"name": "dgemm_1024", "op": "gemm", "prec": "d", "ta": "N", "tb": "N",
         "m": 1024, "n": 1024, "k": 1024, "pad": 0, "beta": 0.5},
        # the sizes that applications really have: no multiple of anything, odd leading
        # dimensions, a transposed factor
        {"name": "dgemm_odd", "op": "gemm", "prec": "d", "ta": "T", "tb": "N",
         "m": 2047, "n": 1531, "k": 1789, "pad": 0, "beta": 0.5},
        # the largest product of the Level-3 sweep
        {"name": "dgemm_8192", "op": "gemm", "prec": "d", "ta": "N", "tb": "T",
         "m": 8192, "n": 8192, "k": 8192, "pad": 0, "beta": 0.5},
        # single precision, the smaller corner of the Level-3 sweep
        {"name": "sgemm_4096", "op": "gemm", "prec": "s", "ta": "N", "tb": "N",
         "m": 4096, "n": 4096, "k": 4096, "pad": 0, "beta": 0.5},
        # rank-k update of one triangle (normal equations, Cholesky), the sweep's size
        {"name": "dsyrk_8192x2048", "op": "syrk", "prec": "d", "uplo": "L", "ta": "N",
         "n": 8192, "k": 2048, "pad": 0, "beta": 0.5},
        # solve with many right-hand sides, the sweep's size
        {"name": "dtrsm_8192x4096", "op": "trsm", "prec": "d", "side": "L", "uplo": "L",
         "ta": "N", "diag": "N", "m": 8192, "n": 4096, "pad": 0},
        # the same in single precision on an odd size, from the right with a transpose, as the
        # panel solve of a blocked Cholesky
        {"name": "strsm_odd", "op": "trsm", "prec": "s", "side": "R", "uplo": "L", "ta": "T",
         "diag": "N", "m": 3001, "n": 1502, "pad": 1},
        # the opt-in split-precision product at FP64 accuracy
        {"name": "split_4096", "op": "split", "m": 4096, "n": 4096, "k": 4096, "slices": 7},
        # the memory-bound chain of an iterative solver, the library's headline workload
        {"name": "chain_8192", "op": "chain", "n": 8192},
        # the other Level-2 calls (transposed product, rank-1 update, triangular solve) on an
        # odd size
        {"name": "level2_odd", "op": "level2", "n": 5001, "pad": 2},
        # many small uneven calls collected into one grouped launch (the serving loop's batch)
        {"name": "batch_32", "op": "batch", "gemms": 20, "gemvs": 8, "trsms": 4, "top": 512,
         "mix": 1},
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ranges; sizes log-uniform, mostly odd ones among them."""
    kind = rng.choice(["gemm", "gemm", "gemm", "syrk", "trsm", "trsm", "split", "chain", "level2",
                       "batch"])
    pad = rng.choice([0, 0, 1, 2, 7])
    if kind == "gemm":
        return {"op": "gemm", "prec": rng.choice("ds"), "ta": rng.choice("NT"),
                "tb": rng.choice("NT"), "m": _logint(rng, 32, 5000), "n": _logint(rng, 32, 5000),
                "k": _logint(rng, 32, 5000), "pad": pad, "beta": rng.choice([0.0, 0.5, 1.0])}
    if kind == "syrk":
        return {"op": "syrk", "prec": rng.choice("ds"), "uplo": rng.choice("LU"),
                "ta": rng.choice("NT"), "n": _logint(rng, 64, 6000), "k": _logint(rng, 64, 4000),
                "pad": pad, "beta": rng.choice([0.0, 0.5, 1.0])}
    if kind == "trsm":
        return {"op": "trsm", "prec": rng.choice("ds"), "side": rng.choice("LR"),
                "uplo": rng.choice("LU"), "ta": rng.choice("NT"), "diag": "N",
                "m": _logint(rng, 64, 5000), "n": _logint(rng, 64, 5000), "pad": pad}
    if kind == "split":
        return {"op": "split", "m": _logint(rng, 512, 4096), "n": _logint(rng, 512, 4096),
                "k": _logint(rng, 512, 4096), "slices": rng.choice([7, 8])}
    if kind == "chain":
        return {"op": "chain", "n": _logint(rng, 256, 12000)}
    if kind == "level2":
        return {"op": "level2", "n": _logint(rng, 256, 9000), "pad": pad}
    return {"op": "batch", "gemms": rng.randint(4, 20), "gemvs": rng.randint(2, 12),
            "trsms": rng.randint(1, 8), "top": _logint(rng, 128, 1024),
            "mix": rng.randint(2, 1 << 20)}


# --------------------------------------------------------------------------- inputs
class _Device:
    """A tracked array's device copy, as torch reads it."""

    def __init__(self, addr, shape, dtype):
        self.__cuda_array_interface__ = {"shape": shape, "typestr": np.dtype(dtype).str,
                                         "data": (addr, False), "version": 2}


def _tracked(t):
    """The tensor's values in a tracked (HBM-resident) array of the same storage order."""
    dtype = str(t.dtype).replace("torch.", "")
    a = gb.tracked_empty(tuple(t.shape), np.dtype(dtype), order="C")
    torch.as_tensor(_Device(gb.device_ptr(a), tuple(t.shape), dtype), device="cuda").copy_(t)
    return a


class _Inputs:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(int(seed))

    def uniform(self, shape, dtype=F64):
        t = torch.rand(shape, generator=self.g, device="cuda", dtype=getattr(torch, dtype))
        return t.mul_(2).sub_(1)

    def triangle(self, n, ld, dtype=F64):
        """A matrix whose triangles are factors as a Cholesky or LU factorisation of a matrix of
        unit-size entries leaves them: off-diagonal entries in [-1, 1], diagonal about sqrt(n)."""
        t = self.uniform((n, ld), dtype)
        d = torch.rand(n, generator=self.g, device="cuda", dtype=t.dtype)
        t[:, :n].diagonal().copy_((1 + d) * math.sqrt(n))
        return t


def _dtype(case):
    return F32 if case.get("prec") == "s" else F64


def _matrices(case, seed):
    """The operands of one case, as tensors in the library's storage order."""
    r, op, dt = _Inputs(seed), case["op"], _dtype(case)
    pad = case.get("pad", 0)
    if op in ("gemm", "split"):
        m, n, k = case["m"], case["n"], case["k"]
        an = case.get("ta", "N") == "N"
        bn = case.get("tb", "N") == "N"
        a = r.uniform((k if an else m, (m if an else k) + pad), dt)
        b = r.uniform((n if bn else k, (k if bn else n) + pad), dt)
        return a, b, r.uniform((n, m + pad), dt)
    if op == "syrk":
        n, k = case["n"], case["k"]
        a = r.uniform((k, n + pad) if case["ta"] == "N" else (n, k + pad), dt)
        return a, r.uniform((n, n + pad), dt)
    if op == "trsm":
        m, n = case["m"], case["n"]
        na = m if case["side"] == "L" else n
        ldb = m + pad + (m + pad) % 2  # even: two floats move as one 8-byte word below
        return r.triangle(na, na + pad, dt), r.uniform((n, ldb), dt)
    if op == "chain":
        n = case["n"]
        return r.uniform((n, n)), r.uniform((n,)), r.uniform((n,)), r.uniform((n,))
    if op == "level2":
        n = case["n"]
        return (r.triangle(n, n + pad), r.uniform((n, n + pad)),
                *(r.uniform((n,)) for _ in range(5)))
    return None


def _batch_calls(case):
    """The calls of one batch: 60 % GEMM of both precisions, GEMV and left lower TRSM, sizes
    log-uniform, as the serving trace has them."""
    import random
    rng = random.Random(case["mix"])
    top, calls = case["top"], []
    for i in range(case["gemms"]):
        calls.append(("gemm", "ds"[i % 2], rng.choice("NT"), rng.choice("NT"),
                      *(_logint(rng, 32, top) for _ in range(3))))
    for _ in range(case["gemvs"]):
        calls.append(("gemv", rng.choice("NT"), _logint(rng, 256, 4 * top),
                      _logint(rng, 256, 4 * top)))
    for _ in range(case["trsms"]):
        calls.append(("trsm", _logint(rng, 64, top), 256))
    return calls


def _batch_operands(case, seed):
    r, got = _Inputs(seed), []
    for c in _batch_calls(case):
        if c[0] == "gemm":
            _, prec, ta, tb, m, n, k = c
            dt = F32 if prec == "s" else F64
            got.append((r.uniform((k, m) if ta == "N" else (m, k), dt),
                        r.uniform((n, k) if tb == "N" else (k, n), dt), r.uniform((n, m), dt)))
        elif c[0] == "gemv":
            _, tr, m, n = c
            got.append((r.uniform((n, m)), r.uniform((n if tr == "N" else m,)),
                        r.uniform((m if tr == "N" else n,))))
        else:
            # diagonal 1024 + u with alpha 1024: repeated solves stay of unit size
            m, nrhs = c[1], c[2]
            a = r.uniform((m, m))
            a.diagonal().add_(1025)
            got.append((a, r.uniform((nrhs, m))))
    return got


# --------------------------------------------------------------------------- passes
def _ch(c):
    return ctypes.byref(ctypes.c_char(c.encode()))


def _int(v):
    return ctypes.byref(ctypes.c_int(v))


def _real(v, dt=F64):
    return ctypes.byref(ctypes.c_float(v) if dt == F32 else ctypes.c_double(v))


def _at(a):
    return ctypes.c_void_p(a.ctypes.data)


def prepare(case, seed):
    """Tracked operands in HBM and the argument lists of the calls, as a program keeps them."""
    lib, op, dt = gb.library(), case["op"], _dtype(case)
    gb.set_cutoff(0)  # every call goes to the device
    one, mone = _int(1), _real(1.0, dt)
    if op == "batch":
        return _prepare_batch(case, seed)
    tensors = _matrices(case, seed)
    if op == "split":
        m, n, k = case["m"], case["n"], case["k"]
        a, b, c = tensors
        f = lib.gpublas_dev_dgemm_split_fmt
        p = ctypes.c_void_p
        args = (None, case["slices"], SLICE_INT8, ctypes.c_char(b"N"), ctypes.c_char(b"N"), m, n, k,
                ctypes.c_double(1.0), p(a.data_ptr()), m, p(b.data_ptr()), k,
                ctypes.c_double(0.0), p(c.data_ptr()), m)
        torch.cuda.synchronize()
        return {"calls": [(f, args)], "out": [c], "keep": tensors}
    arrays = [_tracked(t) for t in tensors]
    torch.cuda.synchronize()
    ld = [_int(a.shape[-1]) for a in arrays]
    x = case["op"]
    if x == "gemm":
        f = lib.dgemm_ if dt == F64 else lib.sgemm_
        a, b, c = arrays
        calls = [(f, (_ch(case["ta"]), _ch(case["tb"]), _int(case["m"]), _int(case["n"]),
                      _int(case["k"]), mone, _at(a), ld[0], _at(b), ld[1],
                      _real(case["beta"], dt), _at(c), ld[2]))]
        out = [c]
    elif x == "syrk":
        f = lib.dsyrk_ if dt == F64 else lib.ssyrk_
        a, c = arrays
        calls = [(f, (_ch(case["uplo"]), _ch(case["ta"]), _int(case["n"]), _int(case["k"]), mone,
                      _at(a), ld[0], _real(case["beta"], dt), _at(c), ld[1]))]
        out = [c]
    elif x == "trsm":
        # the right-hand sides are copied first, so that every pass solves the same system; the
        # library copies 8-byte words, two floats each in single precision
        f = lib.dtrsm_ if dt == F64 else lib.strsm_
        a, b0 = arrays
        b = _tracked(tensors[1])
        torch.cuda.synchronize()
        words = b.nbytes // 8
        calls = [(lib.dcopy_, (_int(words), _at(b0), one, _at(b), one)),
                 (f, (_ch(case["side"]), _ch(case["uplo"]), _ch(case["ta"]), _ch(case["diag"]),
                      _int(case["m"]), _int(case["n"]), mone, _at(a), ld[0], _at(b), ld[1]))]
        arrays.append(b)
        out = [b]
    elif x == "chain":
        a, v, y, z = arrays
        n = _int(case["n"])
        calls = [(lib.dgemv_, (_ch("N"), n, n, mone, _at(a), n, _at(v), one, _real(0.0), _at(y),
                               one)),
                 (lib.daxpy_, (n, _real(0.3), _at(y), one, _at(z), one)),
                 (lib.ddot_, (n, _at(y), one, _at(z), one)),
                 (lib.dnrm2_, (n, _at(z), one)),
                 (lib.idamax_, (n, _at(z), one))]
        out = [y, z]
    else:
        t, a, v, y, u, w, s = arrays
        n = _int(case["n"])
        calls = [(lib.dgemv_, (_ch("T"), n, n, mone, _at(a), ld[1], _at(v), one, _real(0.0),
                               _at(y), one)),
                 (lib.dger_, (n, n, _real(1e-3), _at(u), one, _at(w), one, _at(a), ld[1])),
                 (lib.dcopy_, (n, _at(y), one, _at(s), one)),
                 (lib.dtrsv_, (_ch("L"), _ch("N"), _ch("N"), n, _at(t), ld[0], _at(s), one))]
        out = [y, a, s]
    return {"calls": calls, "out": out, "keep": arrays}


def _prepare_batch(case, seed):
    operands = _batch_operands(case, seed)
    b = gb.Batch(use_graph=True)
    adds, out = [], []
    for c, t in zip(_batch_calls(case), operands):
        at = [x.data_ptr() for x in t]
        ld = [x.shape[-1] for x in t]
        if c[0] == "gemm":
            f = b.dgemm if c[1] == "d" else b.sgemm
            adds.append((f, (c[2], c[3], *c[4:], 1.0, at[0], ld[0], at[1], ld[1], 0.0, at[2],
                             ld[2])))
        elif c[0] == "gemv":
            adds.append((b.dgemv, (*c[1:], 1.0, at[0], ld[0], at[1], 1, 0.0, at[2], 1)))
        else:
            adds.append((b.dtrsm, ("L", "L", "N", "N", c[1], c[2], 1024.0, at[0], ld[0], at[1],
                                   ld[1])))
        out.append(t[-1])
    torch.cuda.synchronize()
    return {"batch": _Slot(b), "adds": adds, "out": out, "keep": operands}


class _Slot:
    """A batch slot that is given back with the state that holds it."""

    def __init__(self, batch):
        self.batch = batch

    def __del__(self):
        self.batch.close()


def run(state):
    if "batch" in state:
        for f, args in state["adds"]:
            if f(*args) != 0:
                raise RuntimeError("the batch slot did not take a call")
        state["batch"].batch.run()
        return list(state["out"])
    got = []
    for f, args in state["calls"]:
        r = f(*args)
        if f.__name__ in ("ddot_", "dnrm2_", "idamax_"):
            got.append(r)
        elif f.__name__.startswith("gpublas_") and r != 0:
            raise RuntimeError("%s: error %d" % (f.__name__, r))
    return list(state["out"]) + got


# --------------------------------------------------------------------------- work, tolerance
def _gemm_work(m, n, k, es, beta):
    return {"bytes": es * (m * k + k * n + m * n * (1 if beta == 0 else 2)),
            "flops": 2 * m * n * k}


def work(case):
    op, es = case["op"], 4 if case.get("prec") == "s" else 8
    if op in ("gemm", "split"):
        return _gemm_work(case["m"], case["n"], case["k"], es, case.get("beta", 0.0))
    n = case.get("n", 0)
    if op == "syrk":
        tri = n * (n + 1) // 2
        return {"bytes": es * (n * case["k"] + tri * (1 if case["beta"] == 0 else 2)),
                "flops": 2 * tri * case["k"]}
    if op == "trsm":
        m = case["m"]
        na = m if case["side"] == "L" else n
        return {"bytes": es * (na * (na + 1) // 2 + 2 * m * n), "flops": na * m * n}
    if op == "chain":  # dgemv, then z read and written once, y and z read by the reductions
        return {"bytes": 8 * (n * n + 9 * n), "flops": 2 * n * n + 6 * n}
    if op == "level2":
        return {"bytes": 8 * (3 * n * n + n * (n + 1) // 2 + 8 * n), "flops": 5 * n * n}
    total = {"bytes": 0, "flops": 0}
    for c in _batch_calls(case):
        if c[0] == "gemm":
            w = _gemm_work(*c[4:], 4 if c[1] == "s" else 8, 0.0)
        elif c[0] == "gemv":
            w = {"bytes": 8 * (c[2] * c[3] + c[2] + c[3]), "flops": 2 * c[2] * c[3]}
        else:
            w = {"bytes": 8 * (c[1] * c[1] // 2 + 2 * c[1] * c[2]), "flops": c[1] * c[1] * c[2]}
        total = {k: total[k] + w[k] for k in total}
    return total


def tolerance(case):
    """Sums of products of up to 8192 terms, in the precision of the operands; about four times
    the distance from the results in 64 bits that was measured (FP32 up to 1.1e-6, FP64 1.1e-15,
    seven 7-bit slices 1.1e-14)."""
    if case.get("prec") == "s" or case["op"] == "batch":
        return {"rel": 5e-6}
    return {"rel": 5e-14 if case["op"] == "split" else 5e-15}


# --------------------------------------------------------------------------- in 64 bits
def _solve(t, b, side, uplo, ta):
    """op(T)^-1 B or B op(T)^-1 with the `uplo` triangle of t; plain matrices in and out."""
    t = torch.tril(t) if uplo == "L" else torch.triu(t)
    t = t if ta == "N" else t.T
    return torch.linalg.solve_triangular(t, b, upper=(uplo == "U") == (ta == "N"),
                                         left=side == "L")


def exact(case, seed):
    op = case["op"]
    if op == "batch":
        got = []
        for c, t in zip(_batch_calls(case), _batch_operands(case, seed)):
            t = [x.double() for x in t]
            if c[0] == "gemm":
                a, b = t[0].T if c[2] == "N" else t[0], t[1].T if c[3] == "N" else t[1]
                got.append((a @ b).T.contiguous())
            elif c[0] == "gemv":
                got.append((t[0].T if c[1] == "N" else t[0]) @ t[1])
            else:
                got.append(1024.0 * _solve(t[0].T, t[1].T, "L", "L", "N").T.contiguous())
        return got
    t = [x.double() for x in _matrices(case, seed)]
    if op in ("gemm", "split"):
        a, b, c = t
        m, n, k = case["m"], case["n"], case["k"]
        a = a[:, :m].T if case.get("ta", "N") == "N" else a[:, :k]
        b = b[:, :k].T if case.get("tb", "N") == "N" else b[:, :n]
        c[:, :m] = (a @ b).T + case.get("beta", 0.0) * c[:, :m]
        return [c]
    n = case["n"]
    if op == "syrk":
        a, c = t
        a = a[:, :n].T if case["ta"] == "N" else a[:, :case["k"]]
        full = c[:, :n].T
        new = a @ a.T + case["beta"] * full
        low = torch.ones_like(new, dtype=torch.bool).tril()
        full = torch.where(low if case["uplo"] == "L" else low.T, new, full)
        c[:, :n] = full.T
        return [c]
    if op == "trsm":
        a, b = t
        m = case["m"]
        na = m if case["side"] == "L" else n
        b[:, :m] = _solve(a[:, :na].T, b[:, :m].T, case["side"], case["uplo"], case["ta"]).T
        return [b]
    if op == "chain":
        a, v, _, z = t
        y = a.T @ v
        z = z + 0.3 * y
        return [y, z, float(y @ z), float(torch.linalg.vector_norm(z)),
                int(z.abs().argmax()) + 1]
    lt, a, v, _, u, w, _ = t
    y = a[:, :n] @ v
    a[:, :n] += 1e-3 * torch.outer(w, u)
    s = _solve(lt[:, :n].T, y[:, None], "L", "L", "N")[:, 0]
    return [y, a, s]
