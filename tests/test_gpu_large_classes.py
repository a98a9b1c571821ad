"""GPU: order 3 on the matrix cores with 2^24 samples or more in both classes
together, each class below.  Each class's counts are exact in FP32, their sums
are not.  Bar: the popcount kernel's list, bit for bit."""
import numpy as np
import pytest

import fiuncho_amd as fa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("snps,cases,ctrls", [(6, 8389000, 8390000), (40, 15000000, 2000000)])
def test_order3_above_2_24_samples(snps, cases, ctrls):
    print(f"case: order 3 {snps}x{cases}+{ctrls}", flush=True)
    d = fa.Dataset.synth(fa.synth_spec(snps, cases, ctrls, seed=91, planted=(0, 2, snps - 1)))
    dist = fa.Distribution(snps, 2)
    want = fa.GpuSearch(algorithm=fa.ALGO_MARGINAL).run_arrays(d, 3, dist, 30)
    for conf in ({}, {"algorithm": fa.ALGO_MFMA, "variant": 3}, {"algorithm": fa.ALGO_MFMA, "sample_threshold": False}):
        s = fa.GpuSearch(**conf)
        got = s.run_arrays(d, 3, dist, 30)
        assert s.last_stats.algorithm == fa.ALGO_MFMA
        assert got[0].tolist() == want[0].tolist() and np.array_equal(got[1], want[1]), conf
    (batched,), _ = fa.search_batch([(d, 3, dist, 30)])
    assert batched[0].tolist() == want[0].tolist() and np.array_equal(batched[1], want[1])
    share = fa.Distribution(snps, 2, 2, 1)
    want = fa.GpuSearch(algorithm=fa.ALGO_MARGINAL).run_arrays(d, 3, share, 30)
    got = fa.GpuSearch(algorithm=fa.ALGO_MFMA).run_arrays(d, 3, share, 30)
    assert got[0].tolist() == want[0].tolist() and np.array_equal(got[1], want[1])
    d.close()
