"""Performance cases: the level-3 work a program gives this library.

Operands are column-major, as the BLAS has them: a column-major M x N matrix
with leading dimension M is a contiguous (N, M) torch tensor.  Device cases
hold their operands in HBM and run on the library's own stream; the host
cases pass pageable numpy arrays through the BLAS ABI.
"""
import ctypes as C
import math

import numpy as np
import torch

import blasx_amd as bx

KINDS = {"s": (np.float32, torch.float32), "d": (np.float64, torch.float64),
         "z": (np.complex128, torch.complex128)}
ESIZE = {"s": 4, "d": 8, "z": 16}
LARGEST = 2.0 * 8192 ** 3


def listed():
    return [
        # a single small call, where latency counts: one block of a blocked
        # algorithm
        dict(name="dgemm_256", kind="gemm", type="d", ta="N", tb="N", M=256, N=256, K=256, pad=0,
             alpha=1.0, beta=0.0),
        # an ordinary call whose sizes and leading dimensions are odd
        dict(name="dgemm_1001_odd_tn", kind="gemm", type="d", ta="T", tb="N", M=1001, N=999,
             K=1003, pad=0, alpha=1.5, beta=0.0),
        # a block of vectors against a large matrix (the benchmark's skinny
        # workload): block Krylov, subspace iteration
        dict(name="dgemm_4096x64x4096", kind="gemm", type="d", ta="N", tb="N", M=4096, N=64,
             K=4096, pad=0, alpha=1.0, beta=0.0),
        # the trailing update of a blocked factorisation: C -= A B^T with a
        # narrow K, operands inside larger arrays
        dict(name="dgemm_update_3200_k256_nt", kind="gemm", type="d", ta="N", tb="T", M=3200,
             N=3200, K=256, pad=896, alpha=-1.0, beta=1.0),
        # the large product, the benchmark's kind, at a size that runs in ms
        dict(name="dgemm_8192", kind="gemm", type="d", ta="N", tb="N", M=8192, N=8192, K=8192,
             pad=0, alpha=1.0, beta=0.0),
        # single precision, ragged in every dimension
        dict(name="sgemm_2001x3003x1502_nt", kind="gemm", type="s", ta="N", tb="T", M=2001,
             N=3003, K=1502, pad=0, alpha=1.0, beta=0.0),
        # complex, conjugate-transposed left operand (overlap matrices)
        dict(name="zgemm_1500x1000x1200_cn", kind="gemm", type="z", ta="C", tb="N", M=1500,
             N=1000, K=1200, pad=0, alpha=1.0, beta=0.0),
        # many independent products in one call: the serving mix's element
        # types and transposes, small to ordinary sizes
        dict(name="grouped_mix_32", kind="grouped", count=32, low=64, high=1024, mix=7),
        # a triangular solve with many right-hand sides
        dict(name="dtrsm_2048x1024", kind="trsm", M=2048, N=1024, uplo="L", trans="N"),
        # a Gram matrix: rank-k update of one triangle
        dict(name="dsyrk_3000x1000", kind="syrk", N=3000, K=1000, uplo="L", trans="N"),
        # FP64 accuracy from the INT8 matrix cores, default accuracy
        dict(name="dgemm_crt_4096", kind="crt", M=4096, N=4096, K=4096, ta="N", tb="N"),
        # the drop-in BLAS call on a program's own (pageable) arrays
        dict(name="cblas_dgemm_host_2048", kind="host", M=2048, N=2048, K=2048, ta="N", tb="N"),
    ]


def _lu(rng, low, high):
    """Log-uniform; half of them odd, a quarter a multiple of 64."""
    v = int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))
    r = rng.random()
    if r < 0.25:
        v = (v + 32) // 64 * 64
    elif r < 0.75:
        v |= 1
    return max(low, min(high, v))


def draw(rng):
    while True:
        kind = rng.choice(["gemm"] * 7 + ["grouped", "trsm", "syrk", "crt", "host"])
        if kind == "gemm":
            # the serving mix's shapes: M, N, K log-uniform in [64, 8192]
            t = rng.choice("dddddssszz")
            ops = "NTC" if t == "z" else "NT"
            c = dict(kind=kind, type=t, ta=rng.choice(ops), tb=rng.choice(ops),
                     M=_lu(rng, 64, 8192), N=_lu(rng, 64, 8192), K=_lu(rng, 64, 8192),
                     pad=rng.choice([0, 0, 0, 5, 64]), alpha=1.0, beta=0.0)
            if rng.random() < 0.25:
                c["alpha"], c["beta"] = -1.0, 1.0
        elif kind == "grouped":
            c = dict(kind=kind, count=rng.randint(4, 64), low=64, high=rng.choice([256, 512, 1024]),
                     mix=rng.randrange(1 << 20))
        elif kind == "trsm":
            # an even number of right-hand sides (the copy moves 16 bytes at a time)
            c = dict(kind=kind, M=_lu(rng, 1024, 4096), N=_lu(rng, 64, 4096) & ~1,
                     uplo=rng.choice("LU"), trans=rng.choice("NT"))
        elif kind == "syrk":
            c = dict(kind=kind, N=_lu(rng, 1024, 6144), K=_lu(rng, 64, 4096),
                     uplo=rng.choice("LU"), trans=rng.choice("NT"))
        elif kind == "crt":
            c = dict(kind=kind, M=_lu(rng, 1024, 6144), N=_lu(rng, 1024, 6144),
                     K=_lu(rng, 1024, 6144), ta=rng.choice("NT"), tb=rng.choice("NT"))
        else:
            c = dict(kind=kind, M=_lu(rng, 1024, 3072), N=_lu(rng, 1024, 3072),
                     K=_lu(rng, 1024, 3072), ta=rng.choice("NT"), tb=rng.choice("NT"))
        if work(c)["flops"] <= LARGEST:
            return c


# ------------------------------------------------------------------ inputs
def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _uniform(g, cols, ld, t):
    """A column-major ld x cols matrix, uniform in [-1, 1) (both parts)."""
    if t == "z":
        return torch.view_as_complex(
            torch.rand((cols, ld, 2), generator=g, dtype=torch.float64, device="cuda") * 2 - 1)
    return torch.rand((cols, ld), generator=g, dtype=KINDS[t][1], device="cuda") * 2 - 1


def _stored(op, rows, cols):
    return (rows, cols) if op == "N" else (cols, rows)


def _gemm_operands(c, g, t):
    ra, ca = _stored(c["ta"], c["M"], c["K"])
    rb, cb = _stored(c["tb"], c["K"], c["N"])
    p = c.get("pad", 0)
    return (_uniform(g, ca, ra + p, t), _uniform(g, cb, rb + p, t),
            _uniform(g, c["N"], c["M"] + p, t))


def _mix(c):
    """The grouped case's problems: the serving mix's element types (60% FP64,
    30% FP32, 10% complex128) and random transposes."""
    r = np.random.default_rng(c["mix"])
    out = []
    for _ in range(c["count"]):
        t = "dsz"[int(r.choice(3, p=[0.6, 0.3, 0.1]))]
        M, N, K = (int(v) for v in np.exp(r.uniform(math.log(c["low"]), math.log(c["high"]), 3)))
        ops = "NTC" if t == "z" else "NT"
        out.append(dict(type=t, ta=ops[r.integers(len(ops))], tb=ops[r.integers(len(ops))], M=M,
                        N=N, K=K))
    return out


def _dynrange(g, cols, rows):
    """(u - 1/2) exp(phi x), phi = 0.5: the split-precision benchmark's inputs."""
    u = torch.rand((cols, rows), generator=g, dtype=torch.float64, device="cuda") - 0.5
    x = torch.randn((cols, rows), generator=g, dtype=torch.float64, device="cuda")
    return u * torch.exp(0.5 * x)


def _triangle(c, g):
    """A well-conditioned triangular factor (both triangles stored)."""
    n = c["M"]
    t = _uniform(g, n, n, "d") / math.sqrt(n)
    t += torch.diag(torch.rand(n, generator=g, dtype=torch.float64, device="cuda") + 1.0)
    return t


def prepare(case, seed):
    k = case["kind"]
    L = bx.lib()
    if k == "host":
        r = np.random.default_rng(seed)
        ra, ca = _stored(case["ta"], case["M"], case["K"])
        rb, cb = _stored(case["tb"], case["K"], case["N"])
        A = np.asfortranarray(r.uniform(-1, 1, (ca, ra)).T)
        B = np.asfortranarray(r.uniform(-1, 1, (cb, rb)).T)
        return dict(c=case, A=A, B=B, C=np.zeros((case["M"], case["N"]), order="F"))
    g = _generator(seed)
    s = dict(c=case)
    if k == "gemm":
        s["A"], s["B"], s["C"] = _gemm_operands(case, g, case["type"])
    elif k == "grouped":
        s["mats"], descs = [], []
        for p in _mix(case):
            A, B, Cm = _gemm_operands(p, g, p["type"])
            s["mats"].append((A, B, Cm))
            descs.append(bx.make_desc(KINDS[p["type"]][0], p["ta"], p["tb"], p["M"], p["N"],
                                      p["K"], 1.0, A.data_ptr(), A.shape[1], B.data_ptr(),
                                      B.shape[1], 0.0, Cm.data_ptr(), Cm.shape[1]))
        s["descs"] = descs
    elif k == "trsm":
        s["T"] = _triangle(case, g)
        s["B"] = _uniform(g, case["N"], case["M"], "d")
        s["X"] = torch.empty_like(s["B"])
        v, i, d = C.c_void_p, C.c_int, C.c_double
        L.cblas_dtrsm.argtypes = [i, i, i, i, i, i, i, d, v, i, v, i]
    elif k == "syrk":
        rows, cols = _stored(case["trans"], case["N"], case["K"])
        s["A"] = _uniform(g, cols, rows, "d")
        s["C"] = torch.zeros((case["N"], case["N"]), dtype=torch.float64, device="cuda")
        v, i, d = C.c_void_p, C.c_int, C.c_double
        L.cblas_dsyrk.argtypes = [i, i, i, i, i, d, v, i, d, v, i]
    else:
        ra, ca = _stored(case["ta"], case["M"], case["K"])
        rb, cb = _stored(case["tb"], case["K"], case["N"])
        s["A"], s["B"] = _dynrange(g, ca, ra), _dynrange(g, cb, rb)
        s["C"] = torch.zeros((case["N"], case["M"]), dtype=torch.float64, device="cuda")
    return s


# ------------------------------------------------------------------ one pass
def run(s):
    c = s["c"]
    k = c["kind"]
    if k == "gemm":
        A, B, Cm = s["A"], s["B"], s["C"]
        bx.device_gemm(c["ta"], c["tb"], c["M"], c["N"], c["K"], c["alpha"], A.data_ptr(),
                       A.shape[1], B.data_ptr(), B.shape[1], c["beta"], Cm.data_ptr(),
                       Cm.shape[1], KINDS[c["type"]][0])
        return Cm
    if k == "grouped":
        bx.gemm_grouped_device(s["descs"])
        return [m[2] for m in s["mats"]]
    if k == "trsm":
        # the program keeps its right-hand sides: X = B, then solve in place
        L, X, B, T = bx.lib(), s["X"], s["B"], s["T"]
        L.blasx_device_copy(X.data_ptr(), B.data_ptr(), B.numel() * 8, None)
        L.cblas_dtrsm(bx.COL_MAJOR, 141, 122 if c["uplo"] == "L" else 121, bx.TRANS[c["trans"]],
                      131, c["M"], c["N"], 1.0, T.data_ptr(), c["M"], X.data_ptr(), c["M"])
        return X
    if k == "syrk":
        A, Cm = s["A"], s["C"]
        bx.lib().cblas_dsyrk(bx.COL_MAJOR, 122 if c["uplo"] == "L" else 121,
                             bx.TRANS[c["trans"]], c["N"], c["K"], 1.0, A.data_ptr(), A.shape[1],
                             0.0, Cm.data_ptr(), c["N"])
        return Cm
    if k == "crt":
        A, B, Cm = s["A"], s["B"], s["C"]
        bx.dgemm_crt_device(c["ta"], c["tb"], c["M"], c["N"], c["K"], 1.0, A.data_ptr(),
                            A.shape[1], B.data_ptr(), B.shape[1], 0.0, Cm.data_ptr(), c["M"])
        return Cm
    bx.gemm(c["ta"], c["tb"], 1.0, s["A"], s["B"], 0.0, s["C"])
    return s["C"]


# ------------------------------------------------------------------ the same in 64 bits
def _op(x, op):
    """op of a stored column-major matrix given as its (cols, rows) tensor,
    in 64 bits, as an ordinary (rows of op) x (columns of op) tensor."""
    if x.dtype == torch.float32:
        x = x.double()
    m = x.T if op == "N" else x
    return m.conj() if op == "C" else m


def _exact_gemm(c, A, B, Cm, alpha, beta):
    ra, ca = _stored(c["ta"], c["M"], c["K"])
    rb, cb = _stored(c["tb"], c["K"], c["N"])
    P = alpha * (_op(A[:, :ra], c["ta"]) @ _op(B[:, :rb], c["tb"]))
    out = Cm.double() if Cm.dtype == torch.float32 else Cm.clone()
    out[:, :c["M"]] = P.T + (beta * out[:, :c["M"]] if beta else 0)
    return out


def exact(case, seed):
    k = case["kind"]
    s = prepare(case, seed)
    if k == "gemm":
        return _exact_gemm(case, s["A"], s["B"], s["C"], case["alpha"], case["beta"])
    if k == "grouped":
        return [_exact_gemm(p, *m, 1.0, 0.0) for p, m in zip(_mix(case), s["mats"])]
    if k == "trsm":
        T = s["T"].T.cpu()
        T = torch.tril(T) if case["uplo"] == "L" else torch.triu(T)
        upper = (case["uplo"] == "U") == (case["trans"] == "N")
        T = T if case["trans"] == "N" else T.T
        return torch.linalg.solve_triangular(T.contiguous(), s["B"].T.cpu().contiguous(),
                                             upper=upper).T.contiguous()
    if k == "syrk":
        A = _op(s["A"], case["trans"])
        P = A @ A.T
        # the tensor holds the column-major C transposed
        return torch.triu(P) if case["uplo"] == "L" else torch.tril(P)
    if k == "crt":
        return (_op(s["A"], case["ta"]) @ _op(s["B"], case["tb"])).T.contiguous()
    A = s["A"] if case["ta"] == "N" else s["A"].T
    B = s["B"] if case["tb"] == "N" else s["B"].T
    return np.asfortranarray(A @ B)


# ------------------------------------------------------------------ sizes and tolerances
def _gemm_work(t, M, N, K, beta):
    e = ESIZE[t]
    return (e * (M * K + K * N + M * N * (2 if beta else 1)),
            (8.0 if t == "z" else 2.0) * M * N * K)


def work(case):
    k = case["kind"]
    if k == "gemm":
        b, f = _gemm_work(case["type"], case["M"], case["N"], case["K"], case["beta"])
    elif k == "grouped":
        b = f = 0
        for p in _mix(case):
            pb, pf = _gemm_work(p["type"], p["M"], p["N"], p["K"], 0)
            b, f = b + pb, f + pf
    elif k == "trsm":
        # the stored triangle, B read and X written; M^2 N multiply-adds / 2
        M, N = case["M"], case["N"]
        b, f = 8 * (M * (M + 1) // 2 + 2 * M * N), float(M) * M * N
    elif k == "syrk":
        N, K = case["N"], case["K"]
        b, f = 8 * (N * K + N * (N + 1) // 2), float(N) * (N + 1) * K
    else:
        b, f = _gemm_work("d", case["M"], case["N"], case["K"], 0)
    return {"bytes": b, "flops": f}


def tolerance(case):
    """A sum of K products with random signs rounds like a random walk: its
    relative error grows as u sqrt(K).  Measured against 64-bit (FP32) or
    reordered (FP64) sums: 0.3 u sqrt(K) for products, rank updates and solves
    alike; stated at four times that."""
    k = case["kind"]
    if k == "gemm":
        u, n = (2.0 ** -24 if case["type"] == "s" else 2.0 ** -53), case["K"]
    elif k == "grouped":
        # FP32 problems among FP64 ones: one figure for all of them
        u, n = 2.0 ** -24, case["high"]
    elif k == "trsm":
        u, n = 2.0 ** -53, case["M"]
    else:
        u, n = 2.0 ** -53, case["K"]
    return {"rel": 1.25 * u * (1.0 + math.sqrt(n))}
