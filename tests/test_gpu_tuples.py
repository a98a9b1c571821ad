"""GPU: the matrix-core scans around a head of order - 2 SNPs, which AUTO takes
for order 4, for round-robin shares and for datasets with uncalled genotypes
above a size.  Bar: the same list (combinations, order and float MI bit for
bit) as the popcount kernels, which count by AND + popcount, and as the
oracle's FP64 ranking where it is quick."""
import numpy as np
import pytest

import fiuncho_amd as fa
import oracle as O

pytestmark = pytest.mark.gpu

DIRECT, MARGINAL = fa.ALGO_DIRECT, fa.ALGO_MARGINAL


def genotypes(snps, samples, seed, missing):
    r = np.random.default_rng(seed)
    maf = r.uniform(0.05, 0.5, size=(snps, 1))
    g = (r.random((snps, samples)) < maf).astype(np.int8) + (r.random((snps, samples)) < maf).astype(np.int8)
    if missing:
        g[r.random(g.shape) < missing] = -1
    return g


@pytest.mark.parametrize("order,snps,cases,ctrls,step,offset,missing,outputs,other", [
    (4, 60, 3000, 2100, 1, 0, 0, 200, MARGINAL),      # ragged last quads, partial column tiles
    (4, 49, 128, 10300, 1, 0, 0, 300, DIRECT),        # one quad of cases; a short b block
    (4, 98, 640, 384, 1, 0, 0, 100, MARGINAL),        # whole quads; 64-column tiles with one column over
    (4, 81, 4000, 3300, 5, 4, 0, 100, MARGINAL),      # a share
    (3, 200, 5000, 4400, 3, 2, 0, 100, MARGINAL),     # shares of order 3: progressions shorter and
    (3, 131, 20000, 33, 2, 1, 0, 300, MARGINAL),      # longer than a block of 64, one tiny class
    (3, 400, 9100, 9000, 90, 395, 0, 50, MARGINAL),     # a step above a block, an offset above the step
    (2, 1000, 7000, 6001, 3, 1, 0, 100, MARGINAL),    # share of order 2
    (2, 700, 9000, 1000, 1, 0, 0.01, 100, DIRECT),    # uncalled genotypes: every cell counted
    (2, 701, 9000, 11000, 2, 1, 0.02, 100, DIRECT),
    (3, 150, 2500, 2000, 1, 0, 0.02, 100, DIRECT),
    (3, 193, 2500, 4000, 3, 1, 0.02, 100, DIRECT),
])
def test_tuple_scans(order, snps, cases, ctrls, step, offset, missing, outputs, other):
    print(f"case: order {order} {snps}x{cases}+{ctrls} share ({step},{offset}) missing {missing}", flush=True)
    g = genotypes(snps, cases + ctrls, 1000 * order + snps, missing)
    is_ctrl = np.random.default_rng(snps).permutation(np.arange(cases + ctrls) >= cases).astype(np.uint8)
    d = fa.Dataset.from_genotypes(g, is_ctrl)
    dist = fa.Distribution(snps, order - 1, step, offset)
    want = fa.GpuSearch(algorithm=other).run_arrays(d, order, dist, outputs)
    for conf in ({}, {"sample_threshold": False, "chunk_combos": 30000, "candidate_cap": 512}):
        got = fa.GpuSearch(**conf).run_arrays(d, order, dist, outputs)
        assert got[0].tolist() == want[0].tolist(), conf
        assert np.array_equal(got[1], want[1]), conf
    if order < 4:
        od = O.pack(g, is_ctrl)
        oc, om, _ = O.search(od, order, outputs, step=step, offset=offset, threads=1, mi_mode=2)
        assert got[0].tolist() == oc.tolist() and np.array_equal(got[1], om)
    d.close()


@pytest.mark.parametrize("snps,cases,ctrls,outputs,variants", [
    (70, 66000, 100, 200, (3, 4)),      # a class above 16-bit counts: scored from LDS, block by block
    (66, 900, 65600, 4000, (4,)),
    (130, 500, 520, 4096, (3, 4, 5, 6)),   # no threshold at first: every triple is marked, full lists
    (67, 65000, 300, 50, (4, 6)),       # the largest 16-bit counts
])
def test_order3_epilogues(snps, cases, ctrls, outputs, variants):
    print(f"case: order 3 epilogues {snps}x{cases}+{ctrls}", flush=True)
    g = genotypes(snps, cases + ctrls, 50 + snps, 0)
    is_ctrl = (np.arange(cases + ctrls) >= cases).astype(np.uint8)
    d = fa.Dataset.from_genotypes(g, is_ctrl)
    dist = fa.Distribution(snps, 2)
    want = fa.GpuSearch(algorithm=MARGINAL).run_arrays(d, 3, dist, outputs)
    for v in variants:
        for sample in (True, False):
            s = fa.GpuSearch(algorithm=fa.ALGO_MFMA, variant=v, sample_threshold=sample)
            got = s.run_arrays(d, 3, dist, outputs)
            assert got[0].tolist() == want[0].tolist() and np.array_equal(got[1], want[1]), (v, sample)
    (batched, _) = fa.search_batch([(d, 3, dist, outputs)])
    assert batched[0][0].tolist() == want[0].tolist() and np.array_equal(batched[0][1], want[1])
    d.close()
