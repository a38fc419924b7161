"""Matrix products whose operands have row strides of millions of elements (a window on very long rows), bit-exact on small
integers.

The kernels address a tile with 32-bit offsets where its rows span less than 4 GiB and with 64-bit offsets beyond that:
31, 63 or 127 rows (fewer in a smaller matrix) of a k-contiguous operand, 7·16 bytes' worth of k rows (112 strides of one
byte) of an mn-contiguous one. The strides below lie on both sides of each line. Everything around an operand is NaN.
"""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DT = {"H": "float16", "S": "float32", "D": "float64"}
CODE = {"H": 0, "S": 1, "D": 3}
MN_LAST = (2 ** 32 - 256) // 112   # the largest stride of an mn-contiguous operand that takes 32-bit offsets


@pytest.fixture(scope="module")
def space(torch_dev):
    buf = torch_dev.empty(12_600_000_000, dtype=torch_dev.uint8, device="cuda")
    yield buf
    del buf
    torch_dev.cuda.empty_cache()


def _place(torch, space, dt, x, ld):
    """x at row stride ld in `space`, which is NaN elsewhere."""
    d = getattr(torch, dt)
    t = torch.from_numpy(x).to("cuda", d)
    space[:(x.shape[0] * ld + 64) * t.element_size()].fill_(255)
    v = torch.as_strided(space.view(d), x.shape, (ld, 1))
    v.copy_(t)
    return v


def _ints(rng, *shape):
    return rng.integers(-2, 3, shape).astype(np.float64)


# (type, tA, tB, M, N, K, operand with the long stride, its stride)
GEMM = [("D", 0, 1, 40, 40, 70, "A", (1 << 20) - 1), ("D", 0, 1, 40, 40, 1700, "A", (1 << 20) + 1),
        ("D", 0, 1, 40, 40, 70, "A", 17318416), ("D", 0, 1, 40, 40, 70, "A", 17318417),
        ("D", 0, 0, 40, 40, 1700, "A", 17500000),   # few tiles, long k: slices of K
        ("D", 1, 0, 40, 70, 40, "A", MN_LAST), ("D", 1, 1, 40, 70, 40, "A", MN_LAST + 1),
        ("D", 0, 0, 300, 35, 40, "B", MN_LAST), ("D", 0, 0, 300, 35, 40, "B", MN_LAST + 1),
        ("D", 1, 1, 33, 40, 70, "B", 17318417),
        ("S", 0, 1, 70, 40, 70, "A", (1 << 22)), ("S", 0, 1, 70, 40, 70, "A", 17043520),
        ("S", 0, 0, 70, 40, 70, "A", 17043521), ("S", 0, 1, 70, 40, 1700, "A", 17100000),
        ("S", 1, 0, 50, 40, 70, "A", MN_LAST), ("S", 1, 1, 50, 40, 70, "A", MN_LAST + 1), ("S", 0, 0, 50, 40, 70, "B", MN_LAST + 1),
        ("H", 0, 1, 70, 40, 130, "A", 31122950), ("H", 0, 0, 70, 40, 130, "A", 31122951), ("H", 0, 1, 70, 40, 1700, "A", 31200000),
        ("H", 1, 0, 50, 40, 130, "A", MN_LAST), ("H", 0, 0, 50, 40, 130, "B", MN_LAST + 1)]


@pytest.mark.parametrize("kind,ta,tb,M,N,K,which,ld", GEMM)
def test_gemm_long_strides(g9, torch_dev, space, kind, ta, tb, M, N, K, which, ld):
    torch, rng, dt = torch_dev, np.random.default_rng(K + M), DT[kind]
    a, b, c0 = _ints(rng, *((K, M) if ta else (M, K))), _ints(rng, *((N, K) if tb else (K, N))), _ints(rng, M, N)
    want = 2.0 * ((a.T if ta else a) @ (b.T if tb else b)) - c0
    dev = {n: torch.from_numpy(x).to("cuda", getattr(torch, dt)) for n, x in (("A", a), ("B", b), ("C", c0))}
    lds = {n: dev[n].shape[1] for n in "ABC"}
    dev[which], lds[which] = _place(torch, space, dt, {"A": a, "B": b}[which], ld), ld
    g9._call("gemm", CODE[kind], ta, tb, M, N, K, 2.0, dev["A"].data_ptr(), lds["A"], dev["B"].data_ptr(), lds["B"], -1.0,
             dev["C"].data_ptr(), N)
    assert np.array_equal(dev["C"].double().cpu().numpy(), want)


@pytest.mark.parametrize("kind,trans,N,K,ld", [("D", 0, 40, 1700, (1 << 20) + 1), ("D", 0, 40, 1700, 13800000), ("D", 0, 40, 70, 13800000),
                                               ("D", 1, 40, 40, MN_LAST + 1), ("S", 0, 70, 300, 17100000),
                                               ("S", 1, 40, 70, MN_LAST + 1), ("H", 0, 70, 130, 31200000)])
def test_syrk_long_strides(g9, torch_dev, space, kind, trans, N, K, ld):
    torch, rng, dt = torch_dev, np.random.default_rng(N + K), DT[kind]
    x, c0 = _ints(rng, *((K, N) if trans else (N, K))), _ints(rng, N, N)
    X, c = _place(torch, space, dt, x, ld), torch.from_numpy(c0).to("cuda", getattr(torch, dt))
    for uplo in (0, 1):
        full = (x.T @ x if trans else x @ x.T) + c0
        want = np.where(np.triu(np.ones((N, N))) if uplo else np.tril(np.ones((N, N))), full, c0)
        g9._call("syrk", CODE[kind], uplo, trans, N, K, 1.0, X.data_ptr(), ld, 1.0, c.data_ptr(), N)
        assert np.array_equal(c.double().cpu().numpy(), want), uplo
        c.copy_(torch.from_numpy(c0))


@pytest.mark.parametrize("kind,M,N,side", [("D", 40, 36, 0), ("S", 70, 40, 0), ("H", 130, 40, 0)])
def test_trmm_long_strides(g9, torch_dev, space, kind, M, N, side):
    torch, rng, dt = torch_dev, np.random.default_rng(M), DT[kind]
    a, b = _ints(rng, M, M), _ints(rng, M, N)
    ld = MN_LAST + 1
    for uplo in (0, 1):
        B = _place(torch, space, dt, b, ld)
        A = torch.from_numpy(a).to("cuda", getattr(torch, dt))
        g9._call("trmm", CODE[kind], side, uplo, 0, 0, M, N, 1.0, A.data_ptr(), M, B.data_ptr(), ld)
        torch.cuda.synchronize()
        want = (np.triu(a) if uplo else np.tril(a)) @ b
        assert np.array_equal(B.double().cpu().numpy(), want), uplo


@pytest.mark.parametrize("routine", ["gemm", "syrk"])
def test_long_strides_keep_the_split(g9, torch_dev, space, routine):
    """FP64 products of few rows on long rows are split over K whatever the row stride: a stride past 2^20 elements takes at
    most twice as long as one below it (one workgroup per tile, as without slices of K, took 16 and 100 times as long)."""
    torch, n, K = torch_dev, 100, 200_000
    space[:3_000_000_000].view(torch.float64).fill_(1.0)
    c = torch.empty((n, n), dtype=torch.float64, device="cuda")
    p, q = space.data_ptr(), space.data_ptr() + 1_000_000_000

    def best(ld):
        if routine == "gemm":
            args = ("gemm", 3, 0, 1, n, n, K, 1.0, p, ld, q, ld, 0.0, c.data_ptr(), n)
        else:
            args = ("syrk", 3, 0, 0, n, K, 1.0, p, ld, 0.0, c.data_ptr(), n)
        times = []
        for _ in range(4):
            t = time.perf_counter()
            g9._call(*args)
            times.append(time.perf_counter() - t)
        assert float(c[n - 1, 0]) == K
        return min(times[1:])

    below, above = best((1 << 20) - 8), best((1 << 20) + 8)
    assert above <= 2 * below, f"{routine}: {above * 1e6:.0f} us with a row stride above 2^20, {below * 1e6:.0f} below"
