"""GPU: batched scans around a head -- order 4, shares, datasets with uncalled
genotypes -- in ranges that split and overflow, and the sampled threshold's
share of a small candidate buffer.  Bar: the popcount kernels' list of each
search alone, bit for bit."""
import numpy as np
import pytest

import fiuncho_amd as fa

from .test_gpu_tuples import genotypes

pytestmark = pytest.mark.gpu

DIRECT, MARGINAL = fa.ALGO_DIRECT, fa.ALGO_MARGINAL


def dataset(snps, cases, ctrls, seed, missing):
    g = genotypes(snps, cases + ctrls, seed, missing)
    return fa.Dataset.from_genotypes(g, (np.arange(cases + ctrls) >= cases).astype(np.uint8))


@pytest.mark.parametrize("step_ms,cap", [(0.0, 0), (0.05, 8192)])
def test_batch_of_scans_around_a_head(step_ms, cap):
    shapes = [   # order, snps, cases, ctrls, (step, offset), missing, outputs
        (4, 98, 2100, 1900, (1, 0), 0, 100),
        (4, 70, 3000, 3300, (2, 1), 0, 4096),
        (3, 220, 4000, 4100, (3, 1), 0, 1000),
        (3, 210, 2600, 2500, (2, 105), 0, 50),
        (2, 1200, 5200, 5000, (3, 2), 0, 4096),
        (2, 800, 4000, 4500, (1, 0), 0.01, 300),
        (3, 160, 2500, 2600, (1, 0), 0.02, 100),
        (3, 200, 4000, 4000, (4, 9), 0.01, 4096),
        (2, 300, 700, 600, (1, 0), 0, 50),          # beside them, one of the persistent kernel
    ]
    scans, want = [], []
    for i, (order, snps, cases, ctrls, (step, offset), missing, outputs) in enumerate(shapes):
        print(f"case: batch of order {order} {snps}x{cases}+{ctrls} share ({step},{offset}) missing {missing}", flush=True)
        d = dataset(snps, cases, ctrls, 300 + i, missing)
        dist = fa.Distribution(snps, order - 1, step, offset)
        scans.append((d, order, dist, outputs))
        want.append(fa.GpuSearch(algorithm=DIRECT if missing else MARGINAL).run_arrays(d, order, dist, outputs))
    cfg = fa.batch_config(step_ms=step_ms, candidate_cap=cap)
    for _ in range(2):
        got, stats = fa.search_batch(scans, cfg)
        for s, g, w in zip(shapes, got, want):
            assert g[0].tolist() == w[0].tolist() and np.array_equal(g[1], w[1]), s
    assert stats.steps > (8 if step_ms else 0)
    for s in scans:
        s[0].close()


@pytest.mark.parametrize("order,snps,cases,ctrls,outputs", [(2, 2000, 1000, 900, 4096), (3, 300, 700, 900, 2000),
                                                             (4, 98, 500, 600, 4000)])
def test_sampled_threshold_fits_a_small_buffer(order, snps, cases, ctrls, outputs):
    # the buffer of 8,192 candidates takes the first slice, which is the whole
    # scan after a sampled threshold
    print(f"case: batch of order {order} {snps}x{cases}+{ctrls} top-{outputs}, 8,192 candidates", flush=True)
    d = dataset(snps, cases, ctrls, 400 + order, 0)
    dist = fa.Distribution(snps, order - 1)
    want = fa.GpuSearch(algorithm=MARGINAL).run_arrays(d, order, dist, outputs)
    (got,), stats = fa.search_batch([(d, order, dist, outputs)], fa.batch_config(candidate_cap=8192))
    assert got[0].tolist() == want[0].tolist() and np.array_equal(got[1], want[1])
    assert stats.redo_ranges == 0
    d.close()
