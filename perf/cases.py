"""What users of this BLAS have it do, as cases that can be timed and checked.

The library's work on MI355X is dense linear algebra on device memory: matrix products in FP16, FP32 and FP64 of any
shape, layout and alignment, products of a few activation rows with resident weights (decode), triangular solves and
rank-k updates, and the level-1/2 steps of an iterative solver. Each case below is one such use; `draw` spreads its sizes
over the range the use has, with odd and unaligned sizes among them. Everything runs through the C ABI
(include/gen9blas.h, include/gen9blas_hip.h) or the Python module over it, on device operands in no-wait mode, the way
a program that keeps its data on the GPU calls it.

    listed()  draw(rng)  prepare(case, seed)  run(state)  work(case)  tolerance(case)  exact(case, seed)
"""
import ctypes
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "gen9-gpu-blas_amd"))
import gen9blas  # noqa: E402

# C ABI type codes and the torch types of their elements
CODE = {"H": 0, "S": 1, "HS": 2, "D": 3}
TORCH = {"H": torch.float16, "HS": torch.float16, "S": torch.float32, "D": torch.float64}
SIZE = {"H": 2, "HS": 2, "S": 4, "D": 8}


def listed():
    return [
        # a large square FP16 product, the library's headline configuration
        {"name": "hgemm_4096", "op": "gemm", "type": "H", "tA": 0, "tB": 0, "M": 4096, "N": 4096, "K": 4096, "beta": 0.0},
        # a prompt of 1000 tokens through the first feed-forward weights of a transformer, packed once and resident
        {"name": "hgemm_prompt", "op": "packed", "type": "HS", "M": 1000, "N": 11008, "K": 4096, "layers": 1},
        # 48 sequences decoded together: each layer's weights are read once for 48 activation rows
        {"name": "decode_batch", "op": "packed", "type": "HS", "M": 48, "N": 4096, "K": 4096, "layers": 16},
        # one sequence decoded: a pass over the packed weights of 16 layers (512 MiB, beyond the last-level cache)
        {"name": "decode_token", "op": "packed", "type": "H", "M": 1, "N": 4096, "K": 4096, "layers": 16},
        # x·W with the weights as a framework lays them out (K×N rows), a few activation rows, several layers
        {"name": "skinny_rows", "op": "skinny", "type": "H", "tB": 0, "M": 4, "N": 4096, "K": 4096, "layers": 8},
        # a large FP32 product with a ragged row count, weights stored N×K, added to a scaled C
        {"name": "sgemm_odd", "op": "gemm", "type": "S", "tA": 0, "tB": 1, "M": 3000, "N": 11008, "K": 4096, "beta": 0.5},
        # an ordinary FP32 product of a numerical program, in round decimal numbers
        {"name": "sgemm_1000", "op": "gemm", "type": "S", "tA": 0, "tB": 0, "M": 1000, "N": 1000, "K": 1000, "beta": 0.0},
        # an FP64 product AᵀB (projections, normal equations)
        {"name": "dgemm_ragged", "op": "gemm", "type": "D", "tA": 1, "tB": 0, "M": 1500, "N": 1300, "K": 1700, "beta": 0.0},
        # many medium FP32 products in one call (blocks of a factorisation, elements of a mesh, attention heads)
        {"name": "sgemm_batch", "op": "batched", "type": "S", "count": 64, "M": 250, "N": 250, "K": 250},
        # forward substitution on many right-hand sides after an FP64 factorisation
        {"name": "dtrsm", "op": "trsm", "type": "D", "uplo": "L", "trans": False, "M": 2000, "N": 500},
        # a Gram matrix XᵀX of many FP32 samples with 1000 features (regression, covariance)
        {"name": "ssyrk_gram", "op": "syrk", "type": "S", "N": 1000, "K": 20000},
        # one gradient step of a least-squares solver: two GEMVs with a matrix of odd row length, and level 1
        {"name": "lsq_step", "op": "lsq", "type": "S", "M": 6000, "N": 1501},
    ]


# ---------------------------------------------------------------------------------------------------------------
# More cases of the same ranges
# ---------------------------------------------------------------------------------------------------------------
def _dim(rng, lo, hi):
    """A size spread over the logarithm of [lo, hi]: whole tiles, multiples of 8, and any number, a third each."""
    n = round(math.exp(rng.uniform(math.log(lo), math.log(hi))))
    step = rng.choice((64, 8, 1))
    n = max(step, round(n / step) * step)
    return n if n <= hi else hi // step * step


def _weight_shape(rng, lo=1024, hi=11008):
    """Weight shapes of linear layers: widths in multiples of 64, sometimes (an output head) any N."""
    n, k = (round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / 64) * 64 for _ in range(2))
    return (n - rng.randrange(64) if rng.random() < 0.25 else n), k


# most flops of a drawn product, so that it costs no more than the largest listed case
MOST_FLOPS = {"H": 2.7e11, "HS": 2.7e11, "S": 2.2e11, "D": 8e10}


def draw(rng):
    op = rng.choice(("gemm", "gemm", "gemm", "prompt", "decode_batch", "decode_token", "skinny", "batched", "trsm", "syrk",
                     "lsq"))
    if op == "gemm":
        t = rng.choice(("H", "HS", "S", "D"))
        while True:
            M, N, K = (_dim(rng, 128, 8192) for _ in range(3))
            if 2.0 * M * N * K <= MOST_FLOPS[t]:
                break
        return {"op": "gemm", "type": t, "tA": rng.randrange(2), "tB": rng.randrange(2), "M": M, "N": N, "K": K,
                "beta": rng.choice((0.0, 0.0, 0.5, 0.9))}
    if op == "prompt":
        N, K = _weight_shape(rng)
        return {"op": "packed", "type": rng.choice(("H", "HS")), "M": round(math.exp(rng.uniform(math.log(129), math.log(2500)))),
                "N": N, "K": K, "layers": 1}
    if op in ("decode_batch", "decode_token"):
        N, K = _weight_shape(rng)
        M = rng.randint(17, 128) if op == "decode_batch" else rng.randint(1, 16)
        return {"op": "packed", "type": rng.choice(("H", "HS")), "M": M, "N": N, "K": K,
                "layers": min(16, max(2, (512 << 20) // (2 * N * K)))}
    if op == "skinny":
        t, (N, K) = rng.choice(("H", "H", "S")), _weight_shape(rng)
        return {"op": "skinny", "type": t, "tB": rng.randrange(2), "M": rng.randint(1, 16), "N": N, "K": K,
                "layers": min(8, max(2, (512 << 20) // (SIZE[t] * N * K)))}
    if op == "batched":
        t = rng.choice(("S", "S", "H", "D"))
        M, N, K = (_dim(rng, 32, 512) for _ in range(3))
        most = MOST_FLOPS[t] / 8 / (2.0 * M * N * K)
        return {"op": "batched", "type": t, "count": max(1, min(rng.randint(8, 256), int(most))), "M": M, "N": N, "K": K}
    if op == "trsm":
        return {"op": "trsm", "type": rng.choice(("S", "D")), "uplo": rng.choice("LU"), "trans": rng.random() < 0.5,
                "M": _dim(rng, 128, 4096), "N": _dim(rng, 16, 2048)}
    if op == "syrk":
        t = rng.choice(("S", "D"))
        N = _dim(rng, 128, 2048)
        K = _dim(rng, 2000, 40000)
        return {"op": "syrk", "type": t, "N": N, "K": min(K, int(MOST_FLOPS[t] / (float(N) * N)))}
    M = _dim(rng, 1000, 40000)
    return {"op": "lsq", "type": rng.choice(("S", "D")), "M": M, "N": min(_dim(rng, 200, 8192), (1 << 27) // M)}


# ---------------------------------------------------------------------------------------------------------------
# Inputs: from the seed alone
# ---------------------------------------------------------------------------------------------------------------
def _inputs(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    t = TORCH[case["type"]]

    def normal(*shape, scale=1.0):
        x = torch.randn(shape, generator=g, device="cuda", dtype=torch.float64 if t == torch.float64 else torch.float32)
        return x.mul_(scale).to(t)

    op = case["op"]
    if op == "gemm":
        M, N, K = case["M"], case["N"], case["K"]
        scale = 1 / math.sqrt(K)
        A = normal(K, M) if case["tA"] else normal(M, K)
        B = normal(N, K, scale=scale) if case["tB"] else normal(K, N, scale=scale)
        return {"A": A, "B": B, "C": normal(M, N) if case["beta"] else torch.zeros((M, N), dtype=t, device="cuda")}
    if op in ("packed", "skinny"):
        M, N, K, L = case["M"], case["N"], case["K"], case["layers"]
        tB = case.get("tB", 1)
        return {"x": normal(L, M, K), "W": [normal(*((N, K) if tB else (K, N)), scale=1 / math.sqrt(K)) for _ in range(L)]}
    if op == "batched":
        c, M, N, K = case["count"], case["M"], case["N"], case["K"]
        return {"A": normal(c, M, K), "B": normal(c, K, N, scale=1 / math.sqrt(K))}
    if op == "trsm":
        # a well-conditioned triangular factor: N(0, 1/n) off the diagonal, 1 to 2 on it
        M, N = case["M"], case["N"]
        T = normal(M, M, scale=1 / math.sqrt(M))
        T = torch.tril(T, -1) if case["uplo"] == "L" else torch.triu(T, 1)
        T += torch.diag(1 + torch.rand(M, generator=g, device="cuda", dtype=torch.float32).to(t))
        return {"A": T, "B": normal(M, N)}
    if op == "syrk":
        return {"X": normal(case["K"], case["N"])}
    M, N = case["M"], case["N"]
    return {"A": normal(M, N, scale=1 / math.sqrt(N)), "x": normal(N), "b": normal(M)}


class _Packed:
    """Weights packed once by gen9blas_pack_b and kept on the device until the object goes."""

    def __init__(self, code, W):
        N, K = W.shape
        gen9blas._init()
        self.handle = gen9blas._lib.gen9blas_pack_b(code, 1, K, N, W.data_ptr(), K)
        if not self.handle:
            raise RuntimeError(gen9blas._lib.gen9blas_error().decode())

    def __del__(self):
        if getattr(self, "handle", None):
            gen9blas._lib.gen9blas_packed_b_free(self.handle)


def _checked(rc):
    if rc:
        raise RuntimeError(gen9blas._lib.gen9blas_error().decode())


# ---------------------------------------------------------------------------------------------------------------
# A pass
# ---------------------------------------------------------------------------------------------------------------
def prepare(case, seed):
    """What a program holds before the call: operands on the GPU, packed weights, result buffers."""
    gen9blas._init()
    gen9blas.set_nowait(True)   # device operands: calls queue on the library's stream and return
    op, code = case["op"], CODE[case["type"]]
    d = _inputs(case, seed)
    state = {"op": op}
    if op == "gemm":
        A, B, C = d["A"], d["B"], d["C"]
        state.update(A=A.t() if case["tA"] else A, B=B.t() if case["tB"] else B, C=C, beta=case["beta"],
                     accurate=case["type"] == "HS")
    elif op in ("packed", "skinny"):
        M, N, K, L = case["M"], case["N"], case["K"], case["layers"]
        x = d["x"]
        y = torch.empty((L, M, N), dtype=x.dtype, device="cuda")
        state.update(x=x, y=y)
        one, zero = ctypes.c_double(1.0), ctypes.c_double(0.0)
        if op == "packed":
            state["packs"] = [_Packed(code, W) for W in d["W"]]
            state["fn"] = gen9blas._lib.gen9blas_gemm_pb
            state["calls"] = [(0, M, one, x[i].data_ptr(), K, w.handle, zero, y[i].data_ptr(), N)
                              for i, w in enumerate(state["packs"])]
        else:
            state["W"] = d["W"]
            state["fn"] = gen9blas._lib.gen9blas_gemm
            state["calls"] = [(code, 0, case["tB"], M, N, K, one, x[i].data_ptr(), K, w.data_ptr(), K if case["tB"] else N,
                               zero, y[i].data_ptr(), N) for i, w in enumerate(d["W"])]
    elif op == "batched":
        c, M, N = case["count"], case["M"], case["N"]
        state.update(d, C=torch.empty((c, M, N), dtype=d["A"].dtype, device="cuda"))
    elif op == "trsm":
        state.update(d, uplo=case["uplo"], trans=case["trans"])
    elif op == "syrk":
        N = case["N"]
        state.update(d, C=torch.zeros((N, N), dtype=d["X"].dtype, device="cuda"))
    else:
        # the solver's buffers and its calls, as a C program has them: r = A·x − b, g = Aᵀ·r, x1 = x − 0.1·g, |g|
        A, x, b = d["A"], d["x"], d["b"]
        M, N = A.shape
        r, grad, x1 = torch.empty_like(b), torch.empty_like(x), torch.empty_like(x)
        norm = ctypes.c_double()
        state.update(d, r=r, g=grad, x1=x1, norm=norm)
        a, xp, bp, rp, gp, x1p = (t.data_ptr() for t in (A, x, b, r, grad, x1))
        num = ctypes.c_double
        lib = gen9blas._lib
        state["calls"] = [
            (lib.gen9blas_copy, (code, M, bp, 1, rp, 1)),
            (lib.gen9blas_gemv, (code, 0, M, N, num(1.0), a, N, xp, 1, num(-1.0), rp, 1)),
            (lib.gen9blas_gemv, (code, 1, M, N, num(1.0), a, N, rp, 1, num(0.0), gp, 1)),
            (lib.gen9blas_copy, (code, N, xp, 1, x1p, 1)),
            (lib.gen9blas_axpy, (code, N, num(-0.1), gp, 1, x1p, 1)),
            (lib.gen9blas_nrm2, (code, N, gp, 1, ctypes.byref(norm))),
        ]
    return state


def run(state):
    op = state["op"]
    if op == "gemm":
        # with beta, C is the program's accumulator: each pass scales it and adds the product
        return gen9blas.gemm(state["A"], state["B"], 1.0, state["beta"], state["C"], state["accurate"])
    if op in ("packed", "skinny"):
        fn = state["fn"]
        for args in state["calls"]:
            _checked(fn(*args))
        return state["y"]
    if op == "batched":
        return gen9blas.gemm_batched(state["A"], state["B"], C=state["C"])
    if op == "trsm":
        return gen9blas.trsm(state["A"], state["B"], uplo=state["uplo"], transA=state["trans"])
    if op == "syrk":
        return gen9blas.syrk(state["X"], trans=True, C=state["C"])   # the lower triangle of XᵀX
    for fn, args in state["calls"]:
        _checked(fn(*args))
    return {"r": state["r"], "g": state["g"], "x": state["x1"], "norm": state["norm"].value}


# ---------------------------------------------------------------------------------------------------------------
# What a pass cannot do without, and how close two correct implementations come
# ---------------------------------------------------------------------------------------------------------------
def work(case):
    op, es = case["op"], SIZE[case["type"]]
    if op == "gemm":
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": es * (M * K + K * N + M * N * (2 if case["beta"] else 1)), "flops": 2.0 * M * N * K}
    if op in ("packed", "skinny"):
        M, N, K, L = case["M"], case["N"], case["K"], case["layers"]
        return {"bytes": L * es * (M * K + K * N + M * N), "flops": L * 2.0 * M * N * K}
    if op == "batched":
        c, M, N, K = case["count"], case["M"], case["N"], case["K"]
        return {"bytes": c * es * (M * K + K * N + M * N), "flops": c * 2.0 * M * N * K}
    if op == "trsm":
        M, N = case["M"], case["N"]
        return {"bytes": es * (M * (M + 1) // 2 + 2 * M * N), "flops": 1.0 * M * M * N}
    if op == "syrk":
        N, K = case["N"], case["K"]
        return {"bytes": es * (N * K + N * (N + 1) // 2), "flops": 1.0 * N * (N + 1) * K}
    # A is needed twice: the second product needs all of the first one's result
    M, N = case["M"], case["N"]
    return {"bytes": es * (2 * M * N + 3 * M + 5 * N), "flops": 4.0 * M * N}


def tolerance(case):
    """FP16 results are rounded once (2^-11 of the value): two correct sums differ by an ulp in some places. FP32 and
    FP64: sums of up to 40000 products in another order; a solve adds the growth of its substitution."""
    t = case["type"]
    if t in ("H", "HS"):
        return {"rel": 1e-3, "max": 1e-2}
    if t == "S":
        return {"rel": 1e-5, "max": 2e-4} if case["op"] == "trsm" else {"rel": 4e-6, "max": 1e-4}
    return {"rel": 4e-14, "max": 2e-12} if case["op"] == "trsm" else {"rel": 1e-14, "max": 5e-13}


def exact(case, seed):
    """The same results in 64 bits, from torch."""
    d, op = _inputs(case, seed), case["op"]

    def mm(a, b):
        return torch.mm(a.double(), b.double())

    if op == "gemm":
        r = mm(d["A"].t() if case["tA"] else d["A"], d["B"].t() if case["tB"] else d["B"])
        return r + case["beta"] * d["C"].double() if case["beta"] else r
    if op in ("packed", "skinny"):
        tB = case.get("tB", 1)
        return torch.stack([mm(d["x"][i], w.t() if tB else w) for i, w in enumerate(d["W"])])
    if op == "batched":
        return torch.stack([mm(a, b) for a, b in zip(d["A"], d["B"])])
    if op == "trsm":
        A = d["A"].double()
        upper = (case["uplo"] == "U") != case["trans"]
        return torch.linalg.solve_triangular(A.t().contiguous() if case["trans"] else A, d["B"].double(), upper=upper)
    if op == "syrk":
        return torch.tril(mm(d["X"].t(), d["X"]))
    A, x, b = (d[k].double() for k in ("A", "x", "b"))
    r = A @ x - b
    g = A.t() @ r
    return {"r": r, "g": g, "x": x - 0.1 * g, "norm": float(g.norm())}
