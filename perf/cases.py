"""The solve paths of this library at the sizes its users run, as measurable cases.

A case is a plain dict; `prepare` makes what a program holds before the call
(matrices in HBM, factors, the handle), `run` is one pass through the public
interface, `work` the bytes and flops the pass cannot do without and `exact`
the result from plain torch / numpy in 64 bits.

Kinds:
    gesv     PDGESV on a matrix in HBM (Handle.dgesv): factors, IPIV and X
    getrf    PDGETRF alone on a rectangular matrix (Handle.dgetrf)
    getrs    PDGETRS, plain or transposed, with factors in hand
    gesvx    the expert driver PDGESVX (equilibrate, factor, condition, refine)
    batched  many small uneven systems in one call (Handle.gesv_batched)
    mixed    the mixed-precision solve with a named precision and refinement
    auto     the same with the learned selector's choice
    host     the drop-in PDGESV on host arrays (staging included)

Matrices are what the library's tests and benchmark use: standard normal or
uniform entries for the FP64 paths, A = U diag(sigma) V^T with sigma geometric
from 1 to 1/kappa for the mixed solve, uniform entries plus a diagonal for the
batch (`_batch_inputs`).  A program that solves keeps its A, so `run`
copies it into the array the solver overwrites, as such a program does.
"""
import math
from pathlib import Path

import numpy as np
import torch

import scalapack_amd
from scalapack_amd import api
from scalapack_amd.device import Handle

MODEL = Path(scalapack_amd.__file__).parent / "data" / "selector_model.npz"


def listed():
    return [
        # a small dense system, the size of LU.dat's test matrices: launches
        # and latency are all there is
        {"name": "gesv_150", "kind": "gesv", "n": 150, "nrhs": 1, "lda": 150, "nb": 64},
        # configuration 1: N = 1024, NRHS = 1, NB = 64
        {"name": "gesv_1024", "kind": "gesv", "n": 1024, "nrhs": 1, "lda": 1024, "nb": 64},
        # an order that fits nothing: odd N, LDA = N (column starts unaligned)
        {"name": "gesv_3001", "kind": "gesv", "n": 3001, "nrhs": 7, "lda": 3001, "nb": 128},
        # configuration 2: N = 16384, NRHS = 16, NB = 256
        {"name": "gesv_16384", "kind": "gesv", "n": 16384, "nrhs": 16, "lda": 16384, "nb": 256},
        # a tall block column with an odd row count, as a block algorithm above
        # the library factors it
        {"name": "getrf_tall", "kind": "getrf", "m": 30011, "n": 600, "lda": 30016, "nb": 256},
        # many right-hand sides against one factorization
        {"name": "getrs_many", "kind": "getrs", "n": 5000, "nrhs": 400, "trans": "N"},
        # the transposed solve with a handful of right-hand sides
        {"name": "getrs_trans", "kind": "getrs", "n": 8192, "nrhs": 16, "trans": "T"},
        # the expert driver at a middling odd order
        {"name": "gesvx_2003", "kind": "gesvx", "n": 2003, "nrhs": 3, "fact": "E", "trans": "N"},
        # configuration 4's distribution: N log-uniform in [32, 512], NRHS 1..8
        {"name": "batched_fp64", "kind": "batched", "batch": 2000, "nlo": 32, "nhi": 512,
         "prec": "fp64"},
        # a larger batch of smaller FP32 systems
        {"name": "batched_fp32", "kind": "batched", "batch": 4000, "nlo": 8, "nhi": 160,
         "prec": "fp32"},
        # the headline: N = 32768 to FP64 backward error, the selector's choice
        {"name": "auto_32768", "kind": "auto", "n": 32768, "nrhs": 1, "kappa": 1e2},
        # a Fortran program's call: host arrays through the drop-in
        {"name": "host_1500", "kind": "host", "n": 1500, "nrhs": 2, "nb": 64},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gesv", "gesv", "gesv", "getrf", "getrs", "getrs", "gesvx", "batched",
                       "mixed", "host"])
    nb = rng.choice([64, 128, 256, 512])
    if kind == "gesv":
        n = _log_int(rng, 100, 14000)
        lda = rng.choice([n, (n + 63) // 64 * 64])
        return {"kind": kind, "n": n, "nrhs": rng.randint(1, 16), "lda": lda, "nb": nb}
    if kind == "getrf":
        m, n = _log_int(rng, 200, 30000), _log_int(rng, 100, 2000)
        if rng.random() < 0.25:
            m, n = n, m // 4 + 100
        return {"kind": kind, "m": m, "n": n, "lda": rng.choice([m, (m + 63) // 64 * 64]),
                "nb": nb}
    if kind == "getrs":
        return {"kind": kind, "n": _log_int(rng, 200, 8000), "nrhs": _log_int(rng, 1, 600),
                "trans": rng.choice(["N", "N", "T"])}
    if kind == "gesvx":
        return {"kind": kind, "n": _log_int(rng, 200, 4000), "nrhs": rng.randint(1, 6),
                "fact": rng.choice(["E", "N"]), "trans": rng.choice(["N", "T"])}
    if kind == "batched":
        nlo = _log_int(rng, 4, 48)
        return {"kind": kind, "batch": _log_int(rng, 300, 3000), "nlo": nlo,
                "nhi": rng.choice([64, 130, 256, 512]), "prec": rng.choice(["fp64", "fp32"])}
    if kind == "mixed":
        return {"kind": kind, "n": _log_int(rng, 2000, 14000), "nrhs": rng.randint(1, 3),
                "kappa": rng.choice([1e1, 1e2, 1e3]),
                "prec": rng.choice(["fp32", "bf16x3", "bf16x6"]),
                "refine": rng.choice(["ir", "gmres"])}
    return {"kind": "host", "n": _log_int(rng, 100, 2500), "nrhs": rng.randint(1, 4), "nb": nb}


# --------------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(rows, cols, g):
    """`cols` columns of `rows` standard normal doubles: row k is column k."""
    return torch.randn(cols, rows, dtype=torch.float64, device="cuda", generator=g)


def _padded(t, ld):
    """The columns of `t` with leading dimension `ld` (zeros below)."""
    if ld == t.shape[1]:
        return t
    out = torch.zeros(t.shape[0], ld, dtype=t.dtype, device=t.device)
    out[:, : t.shape[1]] = t
    return out


def _hartley(t):
    """The orthonormal discrete Hartley transform of every row of `t`, in place."""
    n = t.shape[1]
    step = max(1, (1 << 27) // n)
    for i in range(0, t.shape[0], step):
        f = torch.fft.fft(t[i:i + step])
        t[i:i + step] = (f.real - f.imag) / math.sqrt(n)
    return t


def _signs(n, g):
    return torch.randint(0, 2, (n,), device="cuda", generator=g).double() * 2 - 1


def _spectral(n, kappa, g):
    """U diag(sigma) V^T, sigma geometric 1 .. 1/kappa, U and V products of two
    randomly signed Hartley transforms (dense, random-looking, exact kappa)."""
    a = torch.diag(torch.logspace(0.0, -math.log10(kappa), n, dtype=torch.float64, device="cuda"))
    for _ in range(2):
        for _ in range(2):
            a = _hartley(a.mul_(_signs(n, g)))
        a = a.t().contiguous()
    return a


def _batch_sizes(case):
    """Sizes of the batch: log-uniform, fixed by the case (a program that
    solves the same population again has them unchanged)."""
    rng = np.random.default_rng([case["batch"], case["nlo"], case["nhi"]])
    n = np.exp(rng.uniform(math.log(case["nlo"]), math.log(case["nhi"]), case["batch"]))
    return np.rint(n).astype(np.int32), rng.integers(1, 9, case["batch"]).astype(np.int32)


def _inputs(case, seed):
    """The problem alone: (A, B, x) with A's rows the columns of the matrix;
    x the solution B was made from, or None."""
    g = _gen(seed)
    kind = case["kind"]
    if kind in ("mixed", "auto"):
        a = _spectral(case["n"], case["kappa"], g)
        x = _normal(case["n"], case["nrhs"], g)
        return a, x @ a, x
    if kind == "getrf":
        return _normal(case["m"], case["n"], g), None, None
    if kind == "gesvx" and case["fact"] == "E":
        # rows and columns of very different size, what equilibration is for
        a = _normal(case["n"], case["n"], g)
        a *= 10.0 ** torch.empty(case["n"], dtype=torch.float64, device="cuda").uniform_(
            -3, 3, generator=g)
        return a, _normal(case["n"], case["nrhs"], g), None
    return _normal(case["n"], case["n"], g), _normal(case["n"], case["nrhs"], g), None


def _batch_inputs(case, seed):
    """Flat values of all A and of all B, and the systems' offsets in them.
    Uniform entries; FP64: n I added to every other system, a row-permuted
    multiple of I to the rest, which leaves them pivoting everywhere but keeps
    the worst of thousands from being singular in all but name; FP32: the
    permuted multiple of I larger and in every system, so that the FP32
    solutions have digits to compare."""
    g = _gen(seed)
    n, nrhs = _batch_sizes(case)
    offa = np.concatenate([[0], np.cumsum(n.astype(np.int64) ** 2)])
    offb = np.concatenate([[0], np.cumsum(n.astype(np.int64) * nrhs)])
    offp = np.concatenate([[0], np.cumsum(n.astype(np.int64))])
    a = torch.rand(int(offa[-1]), dtype=torch.float64, device="cuda", generator=g) * 2 - 1
    b = torch.randn(int(offb[-1]), dtype=torch.float64, device="cuda", generator=g)
    # flat positions of the added entries: one per column
    rng = np.random.default_rng(seed)
    where, add = [], []
    for s, ns in enumerate(n.tolist()):
        cols = np.arange(ns, dtype=np.int64)
        if case["prec"] == "fp32":
            where.append(offa[s] + cols * ns + rng.permutation(ns))
            add.append(np.full(ns, 2.0 * math.sqrt(ns)))
        elif s % 2 == 0:
            where.append(offa[s] + cols * (ns + 1))
            add.append(np.full(ns, float(ns)))
        else:
            where.append(offa[s] + cols * ns + rng.permutation(ns))
            add.append(np.full(ns, 0.6 * math.sqrt(ns)))
    a[torch.from_numpy(np.concatenate(where)).cuda()] += torch.from_numpy(
        np.concatenate(add)).cuda()
    if case["prec"] == "fp32":
        a, b = a.float(), b.float()
    return a, b, n, nrhs, offa, offb, offp


# -------------------------------------------------------------------- prepare
def prepare(case, seed):
    kind = case["kind"]
    if kind == "batched":
        return _prepare_batched(case, seed)
    if kind == "host":
        return _prepare_host(case, seed)
    a, b, _ = _inputs(case, seed)
    st = {"case": case}
    if kind == "gesv":
        st.update(h=Handle(nb=case["nb"]), a0=_padded(a, case["lda"]), b0=b)
        st.update(a=torch.empty_like(st["a0"]), b=torch.empty_like(b), ipiv=_ints(case["n"]))
    elif kind == "getrf":
        st.update(h=Handle(nb=case["nb"]), a0=_padded(a, case["lda"]))
        st.update(a=torch.empty_like(st["a0"]), ipiv=_ints(min(case["m"], case["n"])))
    elif kind == "getrs":
        n = case["n"]
        st.update(h=Handle(), a=a, ipiv=_ints(n), b0=b, b=torch.empty_like(b))
        st["h"].dgetrf(n, n, a, n, st["ipiv"])
    elif kind == "gesvx":
        n = case["n"]
        st.update(h=Handle(), a0=a, b0=b, a=torch.empty_like(a), af=torch.empty_like(a),
                  b=torch.empty_like(b), x=torch.empty_like(b), ipiv=_ints(n),
                  r=torch.zeros(n, dtype=torch.float64, device="cuda"),
                  c=torch.zeros(n, dtype=torch.float64, device="cuda"))
    else:  # mixed, auto: A is not modified
        st.update(h=Handle(nb=512), a=a, b=b, x=torch.empty_like(b), ipiv=_ints(case["n"]))
        if kind == "auto":
            with np.load(MODEL) as z:
                st["h"].selector_set_model(z["params"])
    return st


def _ints(n):
    return torch.zeros(n, dtype=torch.int32, device="cuda")


def _prepare_batched(case, seed):
    a, b, n, nrhs, offa, offb, offp = _batch_inputs(case, seed)
    st = {"case": case, "h": Handle(), "a0": a, "b0": b, "a": torch.empty_like(a),
          "b": torch.empty_like(b), "n": n, "nrhs": nrhs, "ipiv": _ints(int(offp[-1])),
          "info": _ints(case["batch"])}

    def addresses(t, off):
        return torch.from_numpy(t.data_ptr() + off[:-1] * t.element_size()).cuda()

    st.update(pa=addresses(st["a"], offa), pb=addresses(st["b"], offb),
              pp=addresses(st["ipiv"], offp))
    return st


def _host_arrays(case, seed):
    rng = np.random.default_rng(seed)
    n = case["n"]
    return (np.asfortranarray(rng.uniform(-1, 1, (n, n))),
            np.asfortranarray(rng.standard_normal((n, case["nrhs"]))))


def _prepare_host(case, seed):
    a, b = _host_arrays(case, seed)
    n, nb = case["n"], case["nb"]
    ctx = api.blacs_gridinit(1, 1)
    desca, _ = api.descinit(n, n, nb, nb, 0, 0, ctx, n)
    descb, _ = api.descinit(n, case["nrhs"], nb, nb, 0, 0, ctx, n)
    return {"case": case, "a0": a, "b0": b, "a": np.empty_like(a), "b": np.empty_like(b),
            "desca": desca, "descb": descb, "ipiv": np.zeros(n + nb, np.int32)}


# ------------------------------------------------------------------------ run
def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "gesv":
        n = case["n"]
        st["a"].copy_(st["a0"])
        st["b"].copy_(st["b0"])
        info = st["h"].dgesv(n, case["nrhs"], st["a"], case["lda"], st["ipiv"], st["b"], n)
        return {"lu": st["a"], "ipiv": st["ipiv"], "x": st["b"], "info": info}
    if kind == "getrf":
        st["a"].copy_(st["a0"])
        info = st["h"].dgetrf(case["m"], case["n"], st["a"], case["lda"], st["ipiv"])
        return {"lu": st["a"], "ipiv": st["ipiv"], "info": info}
    if kind == "getrs":
        n = case["n"]
        st["b"].copy_(st["b0"])
        st["h"].dgetrs_trans(case["trans"], n, case["nrhs"], st["a"], n, st["ipiv"], st["b"], n)
        return {"x": st["b"]}
    if kind == "gesvx":
        n = case["n"]
        st["a"].copy_(st["a0"])
        st["b"].copy_(st["b0"])
        info, equed, rcond, _ferr, _berr = st["h"].dgesvx(
            case["fact"], case["trans"], n, case["nrhs"], st["a"], n, st["af"], n, st["ipiv"],
            st["r"], st["c"], st["b"], n, st["x"], n)
        # FERR and BERR are the sizes of rounding errors: no digits to compare
        return {"x": st["x"], "a": st["a"], "af": st["af"], "ipiv": st["ipiv"], "rcond": rcond,
                "info": info, "equed": ord(equed)}
    if kind == "batched":
        st["a"].copy_(st["a0"])
        st["b"].copy_(st["b0"])
        st["h"].gesv_batched(case["prec"], st["n"], st["nrhs"], st["pa"], st["n"], st["pp"],
                             st["pb"], st["n"], st["info"])
        return {"lu": st["a"], "ipiv": st["ipiv"], "x": st["b"], "info": st["info"]}
    if kind == "host":
        n = case["n"]
        st["a"][...] = st["a0"]
        st["b"][...] = st["b0"]
        info = api.pdgesv(n, case["nrhs"], st["a"], 1, 1, st["desca"], st["ipiv"], st["b"], 1, 1,
                          st["descb"])
        return {"lu": st["a"], "ipiv": st["ipiv"][:n], "x": st["b"], "info": info}
    n = case["n"]
    if kind == "auto":
        _choice, _it, info = st["h"].dxgesv_auto(n, case["nrhs"], st["a"], n, st["ipiv"], st["b"],
                                                 n, st["x"], n)
    else:
        _it, info = st["h"].dxgesv(n, case["nrhs"], st["a"], n, st["ipiv"], st["b"], n, st["x"],
                                   n, prec=case["prec"], refine=case["refine"])
    return {"x": st["x"], "info": info}


# ----------------------------------------------------------------------- work
def _lu_flops(m, n):
    k = min(m, n)
    return 2.0 * k * (m * n - (m + n) * k / 2.0 + k * k / 3.0)


def work(case):
    kind = case["kind"]
    if kind == "batched":
        n, nrhs = (v.astype(np.float64) for v in _batch_sizes(case))
        size = 8 if case["prec"] == "fp64" else 4
        return {"bytes": float(2 * size * (n * n + n * nrhs).sum()),
                "flops": float((2 * n ** 3 / 3 + 2 * n * n * nrhs).sum())}
    if kind == "getrf":
        m, n = case["m"], case["n"]
        return {"bytes": 16.0 * m * n, "flops": _lu_flops(m, n)}
    n, nrhs = case["n"], case["nrhs"]
    solve = 2.0 * n * n * nrhs
    if kind == "getrs":
        return {"bytes": 8.0 * n * n + 16.0 * n * nrhs, "flops": solve}
    flops = _lu_flops(n, n) + solve
    if kind == "gesvx":
        # A read, A and AF written; PDGERFS's residual and weights, one solve
        return {"bytes": 24.0 * n * n + 24.0 * n * nrhs, "flops": flops + 3 * solve}
    if kind in ("mixed", "auto"):  # A is only read
        return {"bytes": 8.0 * n * n + 16.0 * n * nrhs, "flops": flops}
    return {"bytes": 16.0 * n * n + 16.0 * n * nrhs, "flops": flops}


# ---------------------------------------------------------------------- exact
def _lu64(a):
    """LU with partial pivoting of a CPU float64 matrix: (packed factors, pivots)."""
    return torch.linalg.lu_factor(a)


def exact(case, seed):
    kind = case["kind"]
    if kind == "batched":
        return _exact_batched(case, seed)
    if kind == "host":
        a, b = (torch.from_numpy(v) for v in _host_arrays(case, seed))
        lu, piv = _lu64(a)
        return {"lu": lu.numpy(), "ipiv": None, "x": torch.linalg.lu_solve(lu, piv, b).numpy(),
                "info": None}
    a, b, x = _inputs(case, seed)
    if x is not None:
        return {"x": x, "info": None}
    if kind == "getrf":
        lu, _ = _lu64(a.t().cpu())
        return {"lu": _padded(lu.t().contiguous(), case["lda"]), "ipiv": None, "info": None}
    at = a.t().cpu()
    bt = b.t().cpu()
    if kind == "gesvx":
        out = dict.fromkeys(("a", "af", "ipiv", "rcond", "info", "equed"))
        m = at if case["trans"] == "N" else at.t()
        out["x"] = torch.linalg.solve(m, bt).t().contiguous()
        return out
    if kind == "getrs":
        m = at if case["trans"] == "N" else at.t()
        return {"x": torch.linalg.solve(m, bt).t().contiguous()}
    lu, piv = _lu64(at)
    x = torch.linalg.lu_solve(lu, piv, bt).t().contiguous()
    return {"lu": _padded(lu.t().contiguous(), case["lda"]), "ipiv": None, "x": x, "info": None}


def _exact_batched(case, seed):
    a, b, n, nrhs, offa, offb, _ = _batch_inputs(case, seed)
    a, b = a.double().cpu(), b.double().cpu()
    lus, xs = [], []
    for s, (ns, rs) in enumerate(zip(n.tolist(), nrhs.tolist())):
        lu, piv = _lu64(a[offa[s]:offa[s + 1]].view(ns, ns).t())
        x = torch.linalg.lu_solve(lu, piv, b[offb[s]:offb[s + 1]].view(rs, ns).t())
        lus.append(lu.t().reshape(-1))
        xs.append(x.t().reshape(-1))
    return {"lu": torch.cat(lus), "ipiv": None, "x": torch.cat(xs), "info": None}
