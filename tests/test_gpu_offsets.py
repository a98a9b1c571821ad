"""GPU: distributions of step 1 that start past the first prefix, on the
matrix-core tiles of orders 2 and 3.  Bar: the popcount kernel's list, bit for
bit."""
import numpy as np
import pytest

import fiuncho_amd as fa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order,snps,offset,outputs", [
    (2, 300, 1, 200), (2, 300, 64, 200), (2, 300, 191, 200), (2, 300, 298, 5), (2, 300, 299, 5), (2, 300, 1000, 5),
    (3, 90, 1, 200), (3, 90, 88, 200), (3, 90, 2000, 200), (3, 90, 4003, 5),
])
def test_scans_from_an_offset(order, snps, offset, outputs):
    print(f"case: order {order} {snps} SNPs from prefix {offset}", flush=True)
    d = fa.Dataset.synth(fa.synth_spec(snps, 700, 900, seed=77))
    dist = fa.Distribution(snps, order - 1, 1, offset)
    want = fa.GpuSearch(algorithm=fa.ALGO_DIRECT).run_arrays(d, order, dist, outputs)
    batched, _ = fa.search_batch([(d, order, dist, outputs)])
    for got in [batched[0]] + [fa.GpuSearch(**c).run_arrays(d, order, dist, outputs)
                               for c in ({}, {"algorithm": fa.ALGO_MFMA, "sample_threshold": False})]:
        assert got[0].tolist() == want[0].tolist() and np.array_equal(got[1], want[1])
    d.close()
