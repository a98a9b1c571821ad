"""GPU: memory that derived tables do not get.  A search whose extra tables
cannot be allocated runs the kernels that need none.  The allocator's refusal
is forced from the host, in a child process whose hipMalloc goes through a
small shim."""
import math
import subprocess
import sys

import pytest

from .conftest import ROOT

pytestmark = pytest.mark.gpu

SHIM = r"""
#include <cstddef>
typedef int (*malloc_fn)(void **, size_t);
static malloc_fn real;
static size_t refused[8];
static int count, hits;
extern "C" void shim_real(void *f) { real = (malloc_fn)f; }
extern "C" void shim_refuse(size_t bytes) { refused[count++] = bytes; }
extern "C" int shim_hits() { return hits; }
extern "C" int hipMalloc(void **p, size_t bytes)
{
    for (int i = 0; i < count; ++i)
        if (bytes == refused[i]) {
            ++hits;
            return 2;   // hipErrorOutOfMemory
        }
    return real(p, bytes);
}
"""

CHILD = r"""
import ctypes as C, sys
sys.path.insert(0, sys.argv[1])
shim = C.CDLL(sys.argv[2], mode=C.RTLD_GLOBAL)
hip = C.CDLL("libamdhip64.so.7")
shim.shim_real(C.cast(hip.hipMalloc, C.c_void_p))
shim.shim_refuse.argtypes = [C.c_size_t]
import numpy as np
import fiuncho_amd as fa
order, snps, cases, ctrls, step, missing, batch = [int(x) for x in sys.argv[3:10]]
g = np.random.default_rng(3).integers(0, 3, size=(snps, cases + ctrls)).astype(np.int8)
if missing:
    g[np.random.default_rng(4).random(g.shape) < 0.01] = -1
d = fa.Dataset.from_genotypes(g, (np.arange(cases + ctrls) >= cases).astype(np.uint8))
dist = fa.Distribution(snps, order - 1, step, 0)
want = fa.GpuSearch(algorithm=fa.ALGO_DIRECT).run_arrays(d, order, dist, 50)
for b in sys.argv[10:]:
    shim.shim_refuse(int(b))
for _ in range(2):
    if batch:
        got = fa.search_batch([(d, order, dist, 50)])[0][0]
    else:
        got = fa.GpuSearch().run_arrays(d, order, dist, 50)
    assert got[0].tolist() == want[0].tolist() and np.array_equal(got[1], want[1])
assert shim.shim_hits() > 0, "nothing was refused"
print("same list without the tables")
"""


def quads(samples):
    return (samples + 511) // 512 * 4    # rows are padded to 512 samples


@pytest.mark.parametrize("batch", [0, 1])
@pytest.mark.parametrize("order,snps,cases,ctrls,step,missing,what", [
    (4, 98, 512, 512, 1, 0, "table"),     # counts of three SNPs
    (4, 98, 512, 512, 1, 0, "image"),     # the two-row image they are counted from
    (3, 160, 5120, 5120, 3, 0, "table"),
    (3, 150, 2560, 2560, 1, 1, "image"),  # the three-row image
    (2, 700, 512, 512, 1, 0, "table"),    # the sampling pass of a whole scan
])
def test_refused_tables_fall_back(tmp_path, order, snps, cases, ctrls, step, missing, what, batch):
    src, lib, child = tmp_path / "shim.cpp", tmp_path / "shim.so", tmp_path / "child.py"
    src.write_text(SHIM)
    child.write_text(CHILD)
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-o", str(lib), str(src)], check=True, timeout=60)
    n_pad = (snps + 63) // 64 * 64
    q = quads(cases) + quads(ctrls)
    m = order - 1
    size = {"table": (math.comb(snps, m) << m) * 4, "image": (12 if missing else 8) * q * n_pad * 16}[what]
    print(f"case: order {order} {snps}x{cases}+{ctrls} {what} of {size} bytes refused, batch {batch}", flush=True)
    p = subprocess.run([sys.executable, str(child), ROOT, str(lib)] +
                       [str(x) for x in (order, snps, cases, ctrls, step, missing, batch, size)],
                       capture_output=True, text=True, timeout=100, cwd=ROOT)
    assert p.returncode == 0, p.stdout + p.stderr[-2000:]
    assert "same list without the tables" in p.stdout
