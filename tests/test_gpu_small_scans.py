"""GPU: order-2 scans in the 64 x 64 tile at the edges of its bands, of 16-bit
counts and of the waiting merges, and batched ranges in launches of their own.
Bar: the popcount kernel's list (combinations, order and float MI bit for
bit), for batches the single search's."""
import numpy as np
import pytest

import fiuncho_amd as fa

from .test_gpu_tuples import genotypes

pytestmark = pytest.mark.gpu


def dataset(snps, cases, ctrls, seed):
    g = genotypes(snps, cases + ctrls, seed, 0)
    return fa.Dataset.from_genotypes(g, (np.arange(cases + ctrls) >= cases).astype(np.uint8))


@pytest.mark.parametrize("snps,cases,ctrls,step,offset,outputs", [
    (2, 200, 100, 1, 0, 5),             # one pair
    (64, 300, 129, 1, 0, 2016),         # every pair of one tile
    (512, 700, 900, 1, 0, 100),         # one whole band of 8 tile rows
    (513, 640, 384, 1, 0, 100),         # a second band of one tile
    (1090, 1500, 1, 1, 0, 4096),        # a third band; a class of one sample; the longest list
    (130, 65535, 300, 1, 0, 300),       # the largest 16-bit counts
    (130, 65536, 300, 1, 0, 300),       # counts above: scored one by one
    (300, 900, 700, 7, 5, 50),          # a share too small for the scan around a head
])
def test_order2_tiles(snps, cases, ctrls, step, offset, outputs):
    print(f"case: order 2 {snps}x{cases}+{ctrls} share ({step},{offset})", flush=True)
    d = dataset(snps, cases, ctrls, 7 * snps)
    dist = fa.Distribution(snps, 1, step, offset)
    want = fa.GpuSearch(algorithm=fa.ALGO_MARGINAL).run_arrays(d, 2, dist, outputs)
    for conf in ({}, {"algorithm": fa.ALGO_MFMA, "variant": 2, "sample_threshold": False},
                 {"algorithm": fa.ALGO_MFMA, "variant": 2, "chunk_combos": 262144},
                 {"algorithm": fa.ALGO_MFMA, "variant": 2, "sample_threshold": False, "candidate_cap": 64}):
        got = fa.GpuSearch(**conf).run_arrays(d, 2, dist, outputs)
        assert got[0].tolist() == want[0].tolist() and np.array_equal(got[1], want[1]), conf
    d.close()


@pytest.mark.parametrize("shapes", [
    ((4000, 2, 2100, 2200, 50), (500, 3, 1300, 1350, 20), (150, 3, 400, 500, 20)),    # two above the size, one below
    ((8300, 2, 5000, 4100, 100), (800, 3, 600, 700, 100)),                            # the wide tiles
    ((1500, 2, 66000, 500, 20), (200, 3, 65600, 300, 20)),                            # classes above 16-bit counts
])
def test_batched_ranges_in_their_own_launches(shapes):
    scans = []
    for snps, order, cases, ctrls, outputs in shapes:
        print(f"case: batch of order {order} {snps}x{cases}+{ctrls}", flush=True)
        scans.append((dataset(snps, cases, ctrls, snps + order), order, fa.Distribution(snps, order - 1), outputs))
    batched, _ = fa.search_batch(scans)
    for (d, order, dist, outputs), got in zip(scans, batched):
        want = fa.GpuSearch().run_arrays(d, order, dist, outputs)
        assert got[0].tolist() == want[0].tolist() and np.array_equal(got[1], want[1])
        d.close()
