"""Matrix products of ragged and unaligned shapes on the GPU, bit-exact on small integers.

Operands are views into NaN-filled device buffers, at an element offset and with a row stride of their own, so that a
value read from outside an operand that reaches a result shows as NaN; C lies in a buffer of a sentinel value that must
survive around it. The integers are small enough that every product and sum is exact in each type.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DT = {"H": "float16", "S": "float32", "D": "float64"}


def _view(torch, rng, dt, shape, pad, off, count=1, fill=float("nan")):
    """(count, rows, cols) small integers in a `fill` buffer: row stride cols + pad, first element at `off`."""
    rows, cols = shape
    ld = cols + pad
    span = rows * ld + 4   # even, as a batch stride of the direct-copy FP16 kernel must be
    buf = torch.full((off + count * span + 64,), fill, dtype=getattr(torch, dt), device="cuda")
    v = torch.as_strided(buf, (count, rows, cols), (span, ld, 1), off)
    v.copy_(torch.from_numpy(rng.integers(-2, 3, (count, rows, cols)).astype(np.float64)).cuda())
    return buf, v, ld, span


def check(g9, torch, kind, M, N, K, ta, tb, pad=0, off=0, beta=0.0, count=1, seed=0):
    """One gemm / gemm_batched call against the same product in float64."""
    rng, dt = np.random.default_rng(seed), DT[kind]
    _, a, lda, sa = _view(torch, rng, dt, (K, M) if ta else (M, K), pad, off, count)
    _, b, ldb, sb = _view(torch, rng, dt, (N, K) if tb else (K, N), pad, off, count)
    cb, c, ldc, sc = _view(torch, rng, dt, (M, N), pad, off, count, fill=77.0)
    opa, opb = (x.double().transpose(1, 2) if t else x.double() for x, t in ((a, ta), (b, tb)))
    want = torch.stack([torch.mm(x.contiguous(), y.contiguous()) for x, y in zip(opa, opb)]) * 2.0
    if beta:
        want += beta * c.double()
    else:
        c.fill_(float("nan"))   # beta = 0: C is not read
    keep = cb.clone()
    torch.as_strided(keep, c.shape, c.stride(), off).copy_(want)
    code = {"H": 0, "S": 1, "D": 3}[kind]
    g9._call("gemm_batched", code, ta, tb, M, N, K, 2.0, a.data_ptr(), lda, sa, b.data_ptr(), ldb, sb, beta, c.data_ptr(),
             ldc, sc, count)
    torch.cuda.synchronize()
    bad = (cb != keep).nonzero()
    assert bad.numel() == 0, f"{kind} {M}x{N}x{K} tA={ta} tB={tb} pad={pad} off={off} beta={beta} count={count}: " \
                             f"{bad.shape[0]} wrong elements, first at {bad[0].item() - off}, row stride {ldc}"


# tile edges (one past, one short, a remainder of one element) and k remainders around the k-step of each type (64
# FP16, 32 FP32, 16 FP64; twice that for tiles with two k groups)
RAGGED = [(129, 127, 65), (65, 255, 31), (257, 130, 129), (320, 192, 97), (200, 1000, 17), (19, 24, 200), (513, 512, 33),
          (1000, 1001, 111)]


@pytest.mark.parametrize("kind", ["H", "S", "D"])
@pytest.mark.parametrize("M,N,K", RAGGED)
def test_gemm_ragged_steps(g9, torch_dev, kind, M, N, K):
    """Tiles that cross the matrix's edges load full k-steps unchecked and their last k-step with checks."""
    for ta, tb in [(0, 0), (1, 0), (0, 1), (1, 1)]:
        for pad, off, beta in [(0, 0, 0.0), (1, 1, -1.0), (2, 2, 0.0), (8, 0, 0.5)]:
            check(g9, torch_dev, kind, M, N, K, ta, tb, pad, off, beta, seed=M + N + K)


@pytest.mark.parametrize("kind", ["H", "S", "D"])
def test_gemm_ragged_batch_and_tiny_strides(g9, torch_dev, kind):
    """Batches of unaligned matrices, and operands whose rows are shorter than one 16-byte load (N or M of 1-3)."""
    for ta, tb in [(0, 0), (1, 0), (0, 1), (1, 1)]:
        check(g9, torch_dev, kind, 70, 90, 75, ta, tb, 1, 1, 0.0, count=5, seed=5)
        for M, N in [(200, 1), (2, 300), (3, 5)]:
            check(g9, torch_dev, kind, M, N, 150, ta, tb, 0, 0, 0.0, count=3, seed=M + N)


# few tiles and a long k: K split into slices whose sums a second kernel adds (K = 3841: with 12 or 16 slices of FP16, 24
# of FP32, the last slice is one k; K = 4160: whole k-steps, the last slice one of them with 8 slices of 9)
@pytest.mark.parametrize("kind", ["H", "S", "D"])
@pytest.mark.parametrize("M,N,K", [(64, 64, 3841), (100, 60, 3841), (48, 300, 4160), (130, 129, 3009), (20, 700, 2050)])
def test_gemm_slices_of_k(g9, torch_dev, kind, M, N, K):
    for ta, tb in [(0, 0), (1, 0), (0, 1), (1, 1)]:
        for pad, off, beta in [(0, 0, 0.0), (1, 1, -1.0), (2, 2, 0.5)]:
            check(g9, torch_dev, kind, M, N, K, ta, tb, pad, off, beta, seed=M + K)


@pytest.mark.parametrize("kind", ["H", "S", "D"])
@pytest.mark.parametrize("N,K", [(70, 3841), (129, 2000), (64, 65), (333, 700), (1, 50), (3, 130)])
def test_syrk_ragged_and_long(g9, torch_dev, kind, N, K):
    """The triangle of X·Xᵀ and Xᵀ·X on unaligned views: edge tiles, slices of K, the other triangle left alone."""
    torch, dt = torch_dev, DT[kind]
    code = {"H": 0, "S": 1, "D": 3}[kind]
    for trans in (0, 1):
        for uplo in (0, 1):
            for pad, off, beta in [(0, 0, 0.0), (1, 1, -1.0)]:
                rng = np.random.default_rng(N + K + trans)
                _, x, ldx, _ = _view(torch, rng, dt, (K, N) if trans else (N, K), pad, off)
                cb, c, ldc, _ = _view(torch, rng, dt, (N, N), pad, off, fill=77.0)
                xd = x[0].double()
                full = (torch.mm(xd.t().contiguous(), xd) if trans else torch.mm(xd, xd.t().contiguous())) * 2.0 + beta * c[0].double()
                mask = torch.ones(N, N, dtype=torch.bool, device="cuda")
                mask = torch.triu(mask) if uplo else torch.tril(mask)
                keep = cb.clone()
                torch.as_strided(keep, (N, N), (ldc, 1), off)[mask] = full[mask].to(keep.dtype)
                if not beta:
                    c[0][mask] = float("nan")
                g9._call("syrk", code, uplo, trans, N, K, 2.0, x.data_ptr(), ldx, beta, c.data_ptr(), ldc)
                torch.cuda.synchronize()
                assert torch.equal(cb, keep), f"{kind} N={N} K={K} trans={trans} uplo={uplo} pad={pad} beta={beta}"


@pytest.mark.parametrize("M,N,K,count", [(1, 1, 1, 1), (31, 33, 15, 1), (32, 32, 64, 1), (33, 65, 1536, 1), (33, 65, 1537, 1),
                                         (500, 513, 200, 1), (520, 520, 70, 1), (65, 31, 129, 20)])
def test_dgemm_few_tiles(g9, torch_dev, M, N, K, count):
    """FP64 products of few tiles (32x32, four k groups of 16 k): edges of tiles, groups without a k-step, both sides of the
    lines in tiles and K that choose them."""
    for ta, tb in [(0, 0), (1, 0), (0, 1), (1, 1)]:
        for pad, off, beta in [(0, 0, 0.0), (1, 1, -1.0)]:
            check(g9, torch_dev, "D", M, N, K, ta, tb, pad, off, beta, count=count, seed=M + K)


@pytest.mark.parametrize("kind", ["H", "S", "D"])
@pytest.mark.parametrize("M,N", [(33, 1), (130, 2), (600, 1), (257, 3), (600, 7), (1025, 2)])
def test_trmm_narrow(g9, torch_dev, kind, M, N):
    """Triangular products with rows of B shorter than one 16-byte load (checked loads of B beside unchecked ones of A)."""
    torch, dt = torch_dev, DT[kind]
    for uplo in (0, 1):
        rng = np.random.default_rng(M + N)
        a, x = rng.integers(-1, 2, (M, M)).astype(np.float64), rng.integers(-2, 3, (M, N)).astype(np.float64)
        A = torch.from_numpy(a).to("cuda", getattr(torch, dt))
        bb, b, ldb, _ = _view(torch, rng, dt, (M, N), 0, 1)
        b[0].copy_(torch.from_numpy(x))
        g9._call("trmm", {"H": 0, "S": 1, "D": 3}[kind], 0, uplo, 0, 0, M, N, 1.0, A.data_ptr(), M, b.data_ptr(), ldb)
        torch.cuda.synchronize()
        want = (np.triu(a) if uplo else np.tril(a)) @ x
        assert np.array_equal(b[0].double().cpu().numpy(), want), f"{kind} {M}x{N} uplo={uplo}"
        assert torch.isnan(bb[:1]).all() and torch.isnan(bb[1 + M * N:]).all()


ORDER_CHILD = r"""
import sys, numpy as np, torch
sys.path.insert(0, sys.argv[1])
import gen9blas as g
gen = torch.Generator(device="cuda").manual_seed(1)
rnd = lambda *s, dt: torch.randn(s, generator=gen, device="cuda", dtype=torch.float64).to(dt)
for dt in (torch.float32, torch.float64):
    for K in (64, 96, 700, 704, 2048):
        for ta in (0, 1):
            for tb in (0, 1):
                a, b = rnd(1200, K, dt=dt), rnd(K, 900, dt=dt)
                A = a.t().contiguous().t() if ta else a
                B = b.t().contiguous().t() if tb else b
                C = g.gemm(A, B)
                for M, N in ((1100, 900), (128, 128), (64, 200), (1200, 70), (257, 129)):
                    assert torch.equal(g.gemm(A[:M], B[:, :N]), C[:M, :N]), ("gemm", dt, K, ta, tb, M, N)
        X = rnd(300, K, dt=dt)
        S = g.syrk(X)
        for N in (64, 100, 256):
            assert torch.equal(torch.tril(g.syrk(X[:N])), torch.tril(S[:N, :N])), ("syrk", dt, K, N)
    for n in (320, 700):
        T = rnd(n, n, dt=dt) / n ** 0.5 + 2 * torch.eye(n, dtype=dt, device="cuda")
        B = rnd(n, 4096, dt=dt)
        for uplo in "LU":
            for name in ("trmm", "trsm"):
                want = getattr(g, name)(T, B, uplo=uplo)
                for N in (16, 64, 500, 1500):
                    got = getattr(g, name)(T, B[:, :N].contiguous(), uplo=uplo)
                    assert torch.equal(got, want[:, :N]), (name, dt, n, uplo, N)
print("ok")
"""


def test_forced_split_fixes_the_order(tmp_path):
    """With GEN9BLAS_SPLITK set, an element of an FP32 or FP64 product is the same whatever the other sizes of the call: the
    k groups, slices and tiles that the number of tiles would choose are off, and whole tiles sum in the edge tiles' order."""
    import os
    import subprocess
    import sys
    script = tmp_path / "order.py"
    script.write_text(ORDER_CHILD)
    pkg = os.path.join(os.path.dirname(os.path.dirname(os.path.realpath(__file__))), "gen9-gpu-blas_amd")
    r = subprocess.run([sys.executable, str(script), pkg], env=dict(os.environ, GEN9BLAS_SPLITK="0"), capture_output=True,
                       text=True, timeout=110)
    assert r.returncode == 0 and r.stdout.strip().endswith("ok"), r.stderr[-2000:]


@pytest.mark.parametrize("N,K", [(2050, 128), (2050, 129), (2049, 40), (1984, 33)])
def test_ssyrk_short_k(g9, torch_dev, N, K):
    """FP32 rank-K updates on both sides of the lines in K and in tiles between the kernels."""
    test_syrk_ragged_and_long(g9, torch_dev, "S", N, K)


@pytest.mark.parametrize("M,N,K", [(300, 333, 127), (300, 333, 128), (300, 336, 127), (129, 1001, 33)])
def test_sgemm_short_k(g9, torch_dev, M, N, K):
    """FP32 NT products with a short K, rows of C of whole 64-byte sectors or not."""
    for pad, off, beta in [(0, 0, 0.5), (1, 1, 0.0), (2, 2, -1.0)]:
        check(g9, torch_dev, "S", M, N, K, 0, 1, pad, off, beta, seed=N + K)
        check(g9, torch_dev, "S", M, N, K, 0, 1, pad, off, beta, count=3, seed=N + K)
