"""GPU: which kernels a search takes.  A tuning entry and the options that
name a kernel are honoured also where AUTO has a scan around a head, and such
a scan is left alone where it would be the slower one.  Kernels that count
differently also cut their scans differently, so the launches of an explicit
algorithm, or the units of a batch, tell which one ran."""
import math

import numpy as np
import pytest

import fiuncho_amd as fa
from fiuncho_amd import tune

from .test_zz_no_alloc import run_static

from .test_zz_no_alloc import run_static

pytestmark = pytest.mark.gpu

AUTO, DIRECT, MARGINAL, MFMA = fa.ALGO_AUTO, fa.ALGO_DIRECT, fa.ALGO_MARGINAL, fa.ALGO_MFMA


@pytest.fixture(autouse=True)
def empty_table():
    tune.clear()
    yield
    tune.clear()


def run(d, order, dist, outputs, **conf):
    s = fa.GpuSearch(**conf)
    r = s.run_arrays(d, order, dist, outputs)
    return r, s.last_stats


def same(a, b):
    return a[0].tolist() == b[0].tolist() and np.array_equal(a[1], b[1])


@pytest.mark.parametrize("algorithm", [DIRECT, MARGINAL])
def test_order4_tuning_entry_is_honoured(algorithm):
    print(f"case: order-4 entry {algorithm}", flush=True)
    d = fa.Dataset.synth(fa.synth_spec(98, 300, 324, seed=61))
    dist = fa.Distribution(98, 3)
    chunk = 3000
    want, explicit = run(d, 4, dist, 50, algorithm=algorithm, chunk_combos=chunk)
    auto, plain = run(d, 4, dist, 50, chunk_combos=chunk)
    assert plain.launches != explicit.launches    # AUTO's scan around a head is another one
    tune.set_table([tune.Entry(4, 0, 1000, 0, 100000, algorithm)])
    got, stats = run(d, 4, dist, 50, chunk_combos=chunk)
    assert stats.algorithm == algorithm and stats.launches == explicit.launches
    batched, bs = fa.search_batch([(d, 4, dist, 50)])
    assert bs.units >= math.comb(98, 3)           # prefixes; a scan around a head has C(98, 2) heads
    for r in (auto, got, batched[0]):
        assert same(r, want)
    d.close()


def test_batch_tuner_adds_no_entry_slower_than_the_default():
    print("case: batch tuner, order 4 above the size of the scan around a head", flush=True)
    table = tune.autotune_batch([tune.BatchClass(4, 0, 1000, 0, 100000, 140, 4000, count=2)], units=(0, 4), repeats=2)
    assert not [e for e in table if e.order == 4]
    table = tune.autotune([tune.ShapeClass(4, 0, 1000, 0, 100000, 120, 2000)], outputs=20, repeats=1)
    assert not [e for e in table if e.order == 4]


@pytest.mark.parametrize("order,snps,conf", [
    (2, 1100, {"mfma_int8": True}),
    (2, 1100, {"variant": 2}),
    (3, 220, {"variant": 2}),
])
def test_options_that_name_a_kernel_keep_it_on_shares(order, snps, conf):
    print(f"case: order {order} share with {conf}", flush=True)
    d = fa.Dataset.synth(fa.synth_spec(snps, 9000, 8000, seed=62))
    dist = fa.Distribution(snps, order - 1, 3, 1)
    chunk = 262144 if order == 2 else 5000
    want, explicit = run(d, order, dist, 50, algorithm=MFMA if order == 2 else MARGINAL, chunk_combos=chunk, **conf)
    auto, plain = run(d, order, dist, 50, chunk_combos=chunk)
    assert plain.launches != explicit.launches
    got, stats = run(d, order, dist, 50, chunk_combos=chunk, **conf)
    assert stats.launches == explicit.launches and stats.variant == explicit.variant
    assert same(got, want) and same(auto, want)
    d.close()


@pytest.mark.parametrize("snps,cases,ctrls", [(200, 4700, 4700), (193, 65535, 300)])
def test_static_search_of_a_share_has_the_pair_table_of_an_earlier_search(snps, cases, ctrls):
    print(f"case: static share {snps}x{cases}+{ctrls}", flush=True)
    d = fa.Dataset.synth(fa.synth_spec(snps, cases, ctrls, seed=63))
    dist = fa.Distribution(snps, 2, 3, 1)
    want = fa.GpuSearch().run_arrays(d, 3, dist, 40)
    got = run_static(d, 3, dist, 40)
    assert got[2].algorithm == MARGINAL and same(got, want)
    # that table, made of the share's count tables, serves the other kernels
    whole = fa.Distribution(snps, 2)
    direct = fa.GpuSearch(algorithm=DIRECT).run_arrays(d, 3, whole, 300)
    for algorithm in (MARGINAL, MFMA):
        assert same(fa.GpuSearch(algorithm=algorithm).run_arrays(d, 3, whole, 300), direct)
    d.close()


@pytest.mark.parametrize("order,snps,samples,step,missing,head", [
    (3, 5000, 4000, 1024, 0, False),     # 2 b's per head: 11.8 ms around a head, 4.2 by popcount
    (3, 5000, 4000, 16, 0, True),        # 156
    (3, 3000, 2000, 1000, 0.01, False),  # with uncalled genotypes
    (3, 1000, 8000, 4, 0.01, True),
    (4, 500, 8000, 5000, 0, False),
    (4, 100, 16000, 8, 0, True),
])
def test_sparse_shares_stay_with_the_popcount_scan(order, snps, samples, step, missing, head):
    print(f"case: order {order} {snps}x{samples} share of {step}", flush=True)
    spec = fa.synth_spec(snps, samples // 2, samples // 2, seed=64)
    if missing:
        _, g, _, _ = fa.synth_generate(spec, words=False, geno=True)
        g[np.random.default_rng(8).random(g.shape) < missing] = -1
        d = fa.Dataset.from_genotypes(g, (np.arange(samples) >= samples // 2).astype(np.uint8))
    else:
        d = fa.Dataset.synth(spec)
    dist = fa.Distribution(snps, order - 1, step, step // 2)
    # launches of whole heads or of whole prefixes: about 1,000, in counts that differ
    heads = math.comb(snps, order - 2)
    per_launch = max(1, heads // 1000)
    chunk = int((per_launch + 0.9) * max(1.0, math.comb(snps, order) / step / heads))
    want, explicit = run(d, order, dist, 50, algorithm=DIRECT if missing else MARGINAL, chunk_combos=chunk)
    got, stats = run(d, order, dist, 50, chunk_combos=chunk)
    assert (stats.launches != explicit.launches) == head
    assert same(got, want)
    d.close()


def test_unsampled_share_stays_with_the_popcount_scan():
    # 8.3 ms by popcount, 10.3 around a head, whose exact MI it floods
    print("case: order 3 800x6000 share of 8, no sample", flush=True)
    d = fa.Dataset.synth(fa.synth_spec(800, 3000, 3000, seed=66))
    dist = fa.Distribution(800, 2, 8, 3)
    conf = {"chunk_combos": 25000, "sample_threshold": False}   # 1.9 heads
    want, explicit = run(d, 3, dist, 50, algorithm=MARGINAL, **conf)
    got, stats = run(d, 3, dist, 50, **conf)
    auto, sampled = run(d, 3, dist, 50, chunk_combos=25000)
    assert stats.launches == explicit.launches != sampled.launches
    assert same(got, want) and same(auto, want)
    d.close()
