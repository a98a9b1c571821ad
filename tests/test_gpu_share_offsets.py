"""GPU: shares whose offset is at or above the step.  The share starts inside
the first head, so prefixes of the same residue before it -- (0, b) with b
above the head -- are not part of it.  A combination planted in one of them
is the strongest of the whole scan and must not be returned.  Bar: the
oracle's FP64 ranking, the popcount kernels' list bit for bit, and the rank
of every returned prefix."""
import numpy as np
import pytest

import fiuncho_amd as fa
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order,snps,cases,ctrls,step,offset,planted,missing", [
    (3, 160, 5500, 5200, 3, 7, (0, 5, 130), 0),       # the share starts at (0, 8)
    (3, 200, 8000, 8000, 8, 20, (0, 13, 180), 0),     # (0, 5) and (0, 13) before (0, 21)
    (3, 170, 5000, 5600, 2, 101, (0, 100, 165), 0),   # in a later column tile than the block's first
    (3, 160, 5500, 5200, 3, 7, (0, 5, 130), 0.01),    # every cell counted
    (3, 170, 5000, 5600, 2, 101, (0, 100, 165), 0.01),
    (2, 700, 9000, 9000, 2, 101, (99, 640), 0),       # free tiles
    (2, 700, 9000, 9000, 2, 101, (99, 640), 0.01),
    (4, 60, 5000, 4500, 2, 9, (0, 1, 9, 50), 0),
])
def test_share_starts_at_its_offset(order, snps, cases, ctrls, step, offset, planted, missing):
    print(f"case: order {order} {snps}x{cases}+{ctrls} share ({step},{offset}) missing {missing}", flush=True)
    spec = fa.synth_spec(snps, cases, ctrls, seed=31 + order, planted=planted, penetrance=(0.05, 0.95))
    _, g, _, _ = fa.synth_generate(spec, words=False, geno=True)
    if missing:
        g[np.random.default_rng(7).random(g.shape) < missing] = -1
    is_ctrl = (np.arange(cases + ctrls) >= cases).astype(np.uint8)
    d = fa.Dataset.from_genotypes(g, is_ctrl)
    dist = fa.Distribution(snps, order - 1, step, offset)
    outputs = 100
    rank = {tuple(p): r for r, p in enumerate(O.dist_prefixes(snps, order - 1, 1, 0).tolist())}
    # the planted combination is of the share's residue and comes before it
    assert rank[planted[:-1]] < offset and (rank[planted[:-1]] - offset) % step == 0
    whole, _ = fa.GpuSearch().run_arrays(d, order, fa.Distribution(snps, order - 1), 1)
    assert whole[0].tolist() == list(planted)
    want = fa.GpuSearch(algorithm=fa.ALGO_DIRECT).run_arrays(d, order, dist, outputs)
    if order < 4:
        oc, om, _ = O.search(O.pack(g, is_ctrl), order, outputs, step=step, offset=offset, threads=1, mi_mode=2)
        assert want[0].tolist() == oc.tolist() and np.array_equal(want[1], om)
    batched, _ = fa.search_batch([(d, order, dist, outputs)])
    for got in (fa.GpuSearch().run_arrays(d, order, dist, outputs),
                fa.GpuSearch(sample_threshold=False, chunk_combos=30000).run_arrays(d, order, dist, outputs),
                batched[0]):
        for c in got[0].tolist():
            r = rank[tuple(c[:-1])]
            assert r >= offset and (r - offset) % step == 0, c
        assert got[0].tolist() == want[0].tolist() and np.array_equal(got[1], want[1])
    d.close()
