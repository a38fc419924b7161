"""The split-K work space when device memory is short: hipMalloc fails from a size on (a stand-in loaded before the library
in a child process, so that no memory is really used up).

Products that would split K then run in fewer slices or unsplit, with the same exact results on small integers; no call
fails or leaves an error text, the smaller work buffer that other routines use stays, and a failed reservation is not
tried again by every product.
"""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

STAND_IN = r"""
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stddef.h>
size_t fail_from = (size_t)-1, refused, given;
int hipMalloc(void **p, size_t n) {
    static int (*real)(void **, size_t);
    if (!real) {
        void *h = dlopen("libamdhip64.so.7", RTLD_LAZY | RTLD_NOLOAD);
        real = h ? (int (*)(void **, size_t))dlsym(h, "hipMalloc") : 0;
        if (!real) return 999;
    }
    if (n >= fail_from) {
        refused++;
        return 2;   /* hipErrorOutOfMemory */
    }
    given++;
    return real(p, n);
}
"""

CHILD = r"""
import ctypes, sys
stand_in = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
import numpy as np, torch
sys.path.insert(0, sys.argv[2])
import gen9blas as g
var = lambda n: ctypes.c_size_t.in_dll(stand_in, n)
gen = torch.Generator(device="cuda").manual_seed(2)
ints = lambda *s, dt: torch.randint(-2, 3, s, generator=gen, device="cuda").to(dt)
calls = []
for dt, M, N, K in ((torch.float16, 64, 64, 8192), (torch.float16, 48, 300, 4160), (torch.float32, 130, 130, 5000)):
    a, b = ints(M, K, dt=dt), ints(K, N, dt=dt)
    calls.append((lambda a=a, b=b, c=torch.empty(M, N, dtype=dt, device="cuda"): g.gemm(a, b, 1.0, 0.0, c), torch.mm(a.double(), b.double())))
for dt, N, K in ((torch.float64, 64, 4096), (torch.float64, 300, 7001), (torch.float32, 333, 3000)):
    x = ints(N, K, dt=dt)
    calls.append((lambda x=x, c=torch.zeros(N, N, dtype=dt, device="cuda"): g.syrk(x, C=c), torch.tril(torch.mm(x.double(), x.double().t().contiguous()))))
v = ints(100000, dt=torch.float32)
vv = float((v.double() ** 2).sum())
def check(times):
    for _ in range(times):
        for f, want in calls:
            assert torch.equal(f().double(), want)
            assert g._lib.gen9blas_last_status() == 0 and b"hipMalloc" not in g._lib.gen9blas_error()
    assert g.dot(v, v) == vv
assert g.dot(v, v) == vv                       # the small work buffer
assert var("given").value > 0, "the stand-in is not in the library's way"
var("fail_from").value = 1
check(10)                                      # 60 products, 51 of them ask
first = var("refused").value
assert 0 < first <= 12, first
var("fail_from").value = 16 << 20              # 8 MiB can be had
check(60)
had = var("given").value
assert var("refused").value - first <= 12, var("refused").value
var("fail_from").value = (1 << 64) - 1
check(60)
assert var("given").value == had + 1           # the whole work space, once
check(2)
assert var("given").value == had + 1
print("ok")
"""


def test_short_of_memory(tmp_path):
    src, lib, child = tmp_path / "short.c", tmp_path / "short.so", tmp_path / "child.py"
    src.write_text(STAND_IN)
    child.write_text(CHILD)
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-o", str(lib), str(src), "-ldl"], check=True, timeout=60)
    pkg = os.path.join(os.path.dirname(os.path.dirname(os.path.realpath(__file__))), "gen9-gpu-blas_amd")
    env = {k: v for k, v in os.environ.items() if not k.startswith("GEN9BLAS_")}
    r = subprocess.run([sys.executable, str(child), str(lib), pkg], env=env, capture_output=True, text=True, timeout=110)
    assert r.returncode == 0 and r.stdout.strip().endswith("ok"), r.stderr[-2000:]
