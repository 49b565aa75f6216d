"""The work a user of eigen_amd has it do, as cases to time.

A case is a dict of plain values; ``listed()`` names the fixed ones, ``draw``
gives more of the same ranges.  ``prepare`` makes the inputs (and the plan, for
the batched paths that have one) on the GPU, ``run`` is one pass through the
public entry points, ``work`` the bytes and operations it cannot do without,
``exact`` the same outputs from torch in 64 bits.
"""
import math

import torch

import eigen_amd as ea
from eigen_amd import batched, mixed

F64 = torch.float64
# the sizes of a flight controller's small filters and fits
SMALL = "6,9,12,15,18,24"


def listed():
    return [
        # C = A B of a handful of state vectors: one launch, nothing to hide it behind
        {"name": "gemm_96", "kind": "gemm", "m": 96, "n": 80, "k": 64, "ta": "N", "tb": "N",
         "beta": 0.0},
        # an ordinary product of odd sizes with a transposed operand (A^T B)
        {"name": "gemm_ragged", "kind": "gemm", "m": 1000, "n": 777, "k": 1301, "ta": "T",
         "tb": "N", "beta": 0.0},
        # the benchmark's largest product
        {"name": "gemm_8192", "kind": "gemm", "m": 8192, "n": 8192, "k": 8192, "ta": "N",
         "tb": "N", "beta": 0.0},
        # T X = B with a block of right-hand sides (triangularView().solve)
        {"name": "trsm_2000x500", "kind": "trsm", "m": 2000, "n": 500, "side": "L", "uplo": "L",
         "trans": "N"},
        # PartialPivLU factor and solve: one system of a dense model
        {"name": "lu_1024", "kind": "lu", "n": 1024, "nrhs": 1},
        # the same at the benchmark's size
        {"name": "lu_16384", "kind": "lu", "n": 16384, "nrhs": 1},
        # the benchmark's headline: mixed-precision LU refined to FP64 accuracy
        {"name": "mixed_16384", "kind": "mixed", "n": 16384, "nrhs": 1, "precision": "fp16x3"},
        # LLT factor and solve of a large SPD system with 16 right-hand sides
        {"name": "llt_8192", "kind": "llt", "n": 8192, "nrhs": 16, "uplo": "L"},
        # a million small SPD systems, one right-hand side each, in one launch
        {"name": "batched_llt", "kind": "batched_llt", "count": 1000000, "sizes": SMALL},
        # many general systems of uneven size, four right-hand sides each
        {"name": "batched_lu", "kind": "batched_lu", "count": 65536, "lo": 16, "hi": 256,
         "nrhs": 4},
        # symmetric small systems: LDLT compute and solve
        {"name": "batched_ldlt", "kind": "batched_ldlt", "count": 1000000, "sizes": SMALL},
        # a filter's measurement update and downdate of its Cholesky factors
        {"name": "batched_rank1", "kind": "batched_rank1", "count": 1000000, "sizes": SMALL},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gemm", "gemm", "trsm", "lu", "mixed", "llt", "batched_llt", "batched_lu",
                       "batched_ldlt", "batched_rank1"])
    if kind == "gemm":
        m, n, k = (_log(rng, 16, 8192) for _ in range(3))
        return {"kind": kind, "m": m, "n": n, "k": k, "ta": rng.choice("NT"),
                "tb": rng.choice("NT"), "beta": rng.choice([0.0, 0.0, 1.0])}
    if kind == "trsm":
        return {"kind": kind, "m": _log(rng, 32, 4096), "n": _log(rng, 2, 2048),
                "side": rng.choice("LLR"), "uplo": rng.choice("LU"), "trans": rng.choice("NT")}
    if kind == "lu":
        return {"kind": kind, "n": _log(rng, 24, 12000), "nrhs": rng.choice([1, 1, 3, 16, 100])}
    if kind == "mixed":
        return {"kind": kind, "n": _log(rng, 300, 16384), "nrhs": rng.choice([1, 1, 2]),
                "precision": rng.choice(["fp16x3", "fp16x3", "fp32"])}
    if kind == "llt":
        return {"kind": kind, "n": _log(rng, 24, 8192), "nrhs": rng.choice([1, 5, 16, 64]),
                "uplo": rng.choice("LLU")}
    if kind == "batched_lu":
        lo = _log(rng, 4, 128)
        return {"kind": kind, "count": _log(rng, 200, 30000), "lo": lo,
                "hi": rng.randint(lo + 1, 256), "nrhs": rng.randint(1, 8)}
    top = {"batched_llt": 32, "batched_ldlt": 64, "batched_rank1": 96}[kind]
    sizes = sorted(rng.sample(range(2, top + 1), rng.randint(1, 6)))
    count = min(_log(rng, 500, 1000000), int(2.4e8 / (sum(s * s for s in sizes) / len(sizes))))
    return {"kind": kind, "count": count, "sizes": ",".join(str(s) for s in sizes)}


# ------------------------------------------------------------------- inputs --
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _randn(g, rows, cols):
    """N(0,1), column-major."""
    return torch.randn(cols, rows, dtype=F64, device="cuda", generator=g).t()


def _sizes(c):
    """The systems' sizes: the layout belongs to the case, values to the seed."""
    g = _gen(c["count"])
    if "sizes" in c:
        sz = torch.tensor([int(s) for s in c["sizes"].split(",")], device="cuda")
        return sz[torch.randint(0, sz.numel(), (c["count"],), generator=g, device="cuda")]
    return torch.randint(c["lo"], c["hi"] + 1, (c["count"],), generator=g, device="cuda")


def _offsets(lengths):
    return (torch.cumsum(lengths, 0) - lengths).contiguous()


def _groups(n, offA, chunk=1 << 25):
    """(size, system indices, flat positions of their entries), a bounded part at a time."""
    for s in torch.unique(n).tolist():
        idx = torch.nonzero(n == s).flatten()
        for ii in idx.split(max(1, chunk // (s * s))):
            yield s, ii, offA[ii][:, None] + torch.arange(s * s, device="cuda")[None, :]


def _packed_spd(c, g, dtype):
    """Packed SPD systems B B^T + n I, B N(0,1)."""
    n = _sizes(c)
    offA, offb = _offsets(n * n), _offsets(n)
    A = torch.empty(int((n * n).sum()), dtype=dtype, device="cuda")
    for s, ii, flat in _groups(n, offA):
        B = torch.randn(ii.numel(), s, s, generator=g, device="cuda", dtype=dtype)
        S = torch.bmm(B, B.transpose(1, 2).contiguous())
        S += s * torch.eye(s, device="cuda", dtype=dtype)
        A[flat.flatten()] = S.reshape(-1)
    b = torch.randn(int(n.sum()), generator=g, device="cuda", dtype=dtype)
    return n, offA, A, offb, b


def _packed_factors(c, g):
    """Packed lower Cholesky factors of such systems (Bartlett's form: N(0,1)
    below the diagonal, chi-like on it) and a vector for each."""
    n = _sizes(c)
    offL, offv = _offsets(n * n), _offsets(n)
    L = torch.empty(int((n * n).sum()), dtype=F64, device="cuda")
    for s, ii, flat in _groups(n, offL):
        M = torch.randn(ii.numel(), s, s, generator=g, device="cuda", dtype=F64)
        d = torch.sqrt(2.0 * s - torch.arange(s, device="cuda") +
                       M.diagonal(dim1=1, dim2=2).abs())
        M = torch.tril(M, -1) + torch.diag_embed(d)
        L[flat.flatten()] = M.transpose(1, 2).reshape(-1)
    v = torch.randn(int(n.sum()), generator=g, device="cuda", dtype=F64)
    return n, offL, L, offv, v


def _packed_newton(c, g):
    """Packed general systems as an implicit integrator has them (I - h J,
    scaled: N(0,1) couplings beside a term of 2 sqrt(n) per unknown), with the
    equations, hence the rows, in an order of their own."""
    n = _sizes(c)
    offA, offB = _offsets(n * n), _offsets(n * c["nrhs"])
    A = torch.randn(int((n * n).sum()), generator=g, device="cuda", dtype=F64)
    B = torch.randn(int((n * c["nrhs"]).sum()), generator=g, device="cuda", dtype=F64)
    N = int(n.sum())
    offn = _offsets(n)
    system = torch.repeat_interleave(torch.arange(n.numel(), device="cuda"), n)
    col = torch.arange(N, device="cuda") - offn[system]
    # a random order of each system's rows: sort random keys within the system
    key = system.to(F64) + torch.rand(N, generator=g, device="cuda", dtype=F64)
    row = torch.argsort(key) - offn[system]
    nn = n[system]
    A[offA[system] + col * nn + row] += 2.0 * torch.sqrt(nn.to(F64))
    return n, offA, A, offB, B


def prepare(case, seed):
    c, g = case, _gen(seed)
    kind = c["kind"]
    s = {"case": dict(c)}
    if kind == "gemm":
        s["A"] = _randn(g, c["m"], c["k"]) if c["ta"] == "N" else _randn(g, c["k"], c["m"])
        s["B"] = _randn(g, c["k"], c["n"]) if c["tb"] == "N" else _randn(g, c["n"], c["k"])
        if c["beta"]:
            s["C"] = _randn(g, c["m"], c["n"])
    elif kind == "trsm":
        na = c["m"] if c["side"] == "L" else c["n"]
        T = _randn(g, na, na) * (0.5 / math.sqrt(na))
        T.diagonal().add_(1.5)  # the other triangle holds values too: it is not read
        s["T"], s["B"] = T, _randn(g, c["m"], c["n"])
    elif kind in ("lu", "mixed"):
        s["A"], s["b"] = _randn(g, c["n"], c["n"]), _randn(g, c["n"], c["nrhs"])
    elif kind == "llt":
        G = _randn(g, c["n"], c["n"])
        S = (G @ G.t()) / c["n"]
        S.diagonal().add_(1.0)
        s["A"], s["b"] = ea.colmajor(S), _randn(g, c["n"], c["nrhs"])
    elif kind == "batched_lu":
        n, s["offA"], s["A"], s["offB"], s["B"] = _packed_newton(c, g)
        s["n"] = n.to(torch.int32)
        s["X"] = torch.empty_like(s["B"])
        s["info"] = torch.empty_like(s["n"])
        s["plan"] = batched.BatchedLuPlan(s["n"], c["nrhs"])
    elif kind == "batched_rank1":
        n, s["offL"], s["L"], s["offv"], s["v"] = _packed_factors(c, g)
        s["n"] = n.to(torch.int32)
        s["up"] = torch.ones(c["count"], dtype=F64, device="cuda")
        s["down"] = torch.full((c["count"],), -0.5, dtype=F64, device="cuda")
    else:
        dtype = torch.float32 if kind == "batched_llt" else F64
        n, s["offA"], s["A"], s["offb"], s["b0"] = _packed_spd(c, g, dtype)
        s["n"] = n.to(torch.int32)
        s["b"] = torch.empty_like(s["b0"])
        if kind == "batched_llt":
            s["info"] = torch.empty_like(s["n"])
            s["plan"] = batched.BatchedPlan(s["n"], 32)
        else:
            s["F"] = torch.empty_like(s["A"])
            s["max_n"] = int(n.max())
    return s


# --------------------------------------------------------------------- pass --
def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "gemm":
        if c["beta"]:
            C = s["C"].clone(memory_format=torch.preserve_format)
            return ea.gemm(s["A"], s["B"], C, beta=c["beta"], transa=c["ta"], transb=c["tb"])
        return ea.gemm(s["A"], s["B"], transa=c["ta"], transb=c["tb"])
    if kind == "trsm":
        X = s["B"].clone(memory_format=torch.preserve_format)
        return ea.triangular_solve(s["T"], X, side=c["side"], uplo=c["uplo"], trans=c["trans"])
    if kind == "lu":
        lu = ea.PartialPivLU(s["A"])
        return {"x": lu.solve(s["b"]), "lu": lu.matrixLU(), "t": lu.transpositionsP()}
    if kind == "mixed":
        return mixed.gesv_ir(s["A"], s["b"], precision=c["precision"])[0]
    if kind == "llt":
        f = ea.LLT(s["A"], uplo=c["uplo"])
        return {"x": f.solve(s["b"]), "f": f.matrixLLT(), "info": f.info()}
    if kind == "batched_llt":
        s["b"].copy_(s["b0"])  # solved in place
        s["plan"].solve_llt(s["offA"], s["A"], s["offb"], s["b"], s["info"])
        return {"x": s["b"], "info": s["info"]}
    if kind == "batched_lu":
        s["plan"].solve(s["offA"], s["n"], s["A"], s["offB"], s["B"], s["X"], s["info"])
        return {"x": s["X"], "info": s["info"]}
    if kind == "batched_ldlt":
        s["F"].copy_(s["A"])  # factored and solved in place
        s["b"].copy_(s["b0"])
        T, offT, sign, info = batched.ldlt_batched(s["offA"], s["n"], s["F"], s["offb"],
                                                   max_n=s["max_n"])
        batched.ldlt_solve_batched(s["offA"], s["n"], s["F"], offT, T, s["offb"], s["b"],
                                   max_n=s["max_n"])
        return {"x": s["b"], "f": s["F"], "t": T, "sign": sign, "info": info}
    i1 = batched.llt_rank_update_batched(s["offL"], s["n"], s["L"], s["offv"], s["v"], s["up"])
    i2 = batched.llt_rank_update_batched(s["offL"], s["n"], s["L"], s["offv"], s["v"], s["down"])
    return {"l": s["L"], "info": [i1, i2]}


def work(case):
    c = case
    kind = c["kind"]
    if kind == "gemm":
        m, n, k = c["m"], c["n"], c["k"]
        return {"bytes": 8.0 * (m * k + k * n + (2 if c["beta"] else 1) * m * n),
                "flops": 2.0 * m * n * k}
    if kind == "trsm":
        m, n = c["m"], c["n"]
        na = m if c["side"] == "L" else n
        return {"bytes": 8.0 * (na * (na + 1) / 2 + 2.0 * m * n), "flops": 1.0 * na * m * n}
    if kind in ("lu", "mixed", "llt"):
        n, r = c["n"], c["nrhs"]
        flops = (1.0 / 3.0 if kind == "llt" else 2.0 / 3.0) * n ** 3 + 2.0 * r * n * n
        mats = {"lu": 2.0, "mixed": 1.0, "llt": 1.0}[kind]  # A read (and the factor written)
        return {"bytes": 8.0 * (mats * n * n + 2.0 * n * r), "flops": flops}
    if "sizes" in c:
        ns = [int(x) for x in c["sizes"].split(",")]
    else:
        ns = list(range(c["lo"], c["hi"] + 1))
    per = c["count"] / len(ns)

    def total(f):
        return per * sum(f(n) for n in ns)

    if kind == "batched_lu":
        r = c["nrhs"]
        return {"bytes": total(lambda n: 8.0 * (n * n + 2 * n * r)),
                "flops": total(lambda n: 2.0 / 3.0 * n ** 3 + 2.0 * r * n * n)}
    if kind == "batched_llt":  # the lower triangle and b in, x out
        return {"bytes": total(lambda n: 4.0 * (n * (n + 1) / 2 + 2 * n)),
                "flops": total(lambda n: n ** 3 / 3.0 + 2.0 * n * n)}
    if kind == "batched_ldlt":  # the triangle in and out, b in, x out
        return {"bytes": total(lambda n: 8.0 * (n * (n + 1) + 2 * n) + 4.0 * n),
                "flops": total(lambda n: n ** 3 / 3.0 + 2.0 * n * n)}
    return {"bytes": 2 * total(lambda n: 8.0 * (n * (n + 1) + n)),  # two updates
            "flops": 2 * total(lambda n: 3.0 * n * n)}


# ---------------------------------------------------------- in 64 bits, torch --
def _solve_groups(s, n, off, offx, rhs, nrhs):
    x = torch.empty_like(rhs, dtype=F64)
    for k, ii, flat in _groups(n, off):
        M = s["A"][flat.flatten()].to(F64).reshape(-1, k, k).transpose(1, 2)
        at = (offx[ii][:, None] + torch.arange(k * nrhs, device="cuda")[None, :]).flatten()
        y = rhs[at].to(F64).reshape(-1, nrhs, k).transpose(1, 2)
        z = torch.linalg.solve(M.cpu(), y.cpu()).cuda()
        x[at] = z.transpose(1, 2).reshape(-1)
    return x


def exact(case, seed):
    c = case
    kind = c["kind"]
    s = prepare(case, seed)
    if kind == "gemm":
        A = s["A"] if c["ta"] == "N" else s["A"].t()
        B = s["B"] if c["tb"] == "N" else s["B"].t()
        return A @ B + (c["beta"] * s["C"] if c["beta"] else 0.0)
    if kind == "trsm":
        T = torch.tril(s["T"]) if c["uplo"] == "L" else torch.triu(s["T"])
        T, upper = (T, c["uplo"] == "U") if c["trans"] == "N" else (T.t(), c["uplo"] == "L")
        return torch.linalg.solve_triangular(T, s["B"], upper=upper, left=c["side"] == "L")
    if kind in ("lu", "mixed"):
        lu, piv = torch.linalg.lu_factor(s["A"].cpu())  # LAPACK's pivots: first largest
        x = torch.linalg.lu_solve(lu, piv, s["b"].cpu())
        return {"x": x, "lu": lu, "t": None} if kind == "lu" else x
    if kind == "llt":
        L = torch.linalg.cholesky(s["A"])
        f = torch.tril(L) + torch.triu(s["A"], 1)
        if c["uplo"] == "U":
            f = torch.triu(L.t()) + torch.tril(s["A"], -1)
        return {"x": torch.cholesky_solve(s["b"], L), "f": f, "info": None}
    n = s["n"].to(torch.int64)
    if kind == "batched_lu":
        return {"x": _solve_groups(s, n, s["offA"], s["offB"], s["B"], c["nrhs"]), "info": None}
    if kind == "batched_llt":
        return {"x": _solve_groups(s, n, s["offA"], s["offb"], s["b0"], 1), "info": None}
    if kind == "batched_ldlt":
        return {"x": _solve_groups(s, n, s["offA"], s["offb"], s["b0"], 1), "f": None, "t": None,
                "sign": None, "info": None}
    out = torch.empty_like(s["L"])
    for k, ii, flat in _groups(n, s["offL"]):
        L = s["L"][flat.flatten()].reshape(-1, k, k).transpose(1, 2).contiguous()
        v = s["v"][(s["offv"][ii][:, None] + torch.arange(k, device="cuda")).flatten()]
        v = v.reshape(-1, k, 1)
        S = L @ L.transpose(1, 2).contiguous() + 0.5 * v * v.reshape(-1, 1, k)
        M = torch.tril(torch.linalg.cholesky(S.cpu()).cuda()) + torch.triu(L, 1)
        out[flat.flatten()] = M.transpose(1, 2).reshape(-1)
    return {"l": out, "info": [None, None]}
