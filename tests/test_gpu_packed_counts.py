"""GPU: scans whose counts travel as 16-bit pairs, on tables at the edge of
what fits: rows that hold more bits than their class has samples, samples
with two genotypes of a SNP, SNPs uncalled throughout a class, and samples
that every SNP misses.  Bar: the popcount kernels' list, bit for bit, which
count with AND + popcount."""
import numpy as np
import pytest

import fiuncho_amd as fa

from .test_gpu_tuples import genotypes

pytestmark = pytest.mark.gpu

DIRECT, MARGINAL = fa.ALGO_DIRECT, fa.ALGO_MARGINAL


def same(a, b):
    return a[0].tolist() == b[0].tolist() and np.array_equal(a[1], b[1])


def check(d, order, dist, outputs, other):
    want = fa.GpuSearch(algorithm=other).run_arrays(d, order, dist, outputs)
    batched, _ = fa.search_batch([(d, order, dist, outputs)])
    for got in (fa.GpuSearch().run_arrays(d, order, dist, outputs),
                fa.GpuSearch(sample_threshold=False).run_arrays(d, order, dist, outputs), batched[0]):
        assert same(got, want)
    return want


def wide_rows(snps, bits, called, seed, overlap):
    """Words of `snps` SNPs, nearly all of genotype 0: `bits` cases, and of the
    controls' 9,216 bits only the first `called` set; `overlap`: every sample
    has two genotypes."""
    r = np.random.default_rng(seed)
    cw, tw = bits // 64, 144
    words = np.zeros((snps, 3 * (cw + tw)), np.uint64)
    for s in range(snps):
        at = 0
        for size, n in ((bits, bits), (9216, called)):
            z = r.random(size) < 0.005
            one = z & (r.random(size) < 0.5)
            rows = [~z, one, z & ~one]
            if overlap:
                rows[1] = rows[1] | rows[0]
            for row in rows:
                row[n:] = False
                words[s, at:at + size // 64] = np.packbits(row).view(np.uint64)
                at += size // 64
    return words.reshape(-1), cw, tw


@pytest.mark.parametrize("order,snps,step,overlap", [
    (2, 500, 1, False), (2, 500, 3, False), (3, 80, 1, False), (3, 80, 2, False), (4, 49, 1, False),
    (2, 500, 1, True), (2, 500, 2, True), (3, 80, 1, True), (3, 90, 2, True),
])
def test_rows_with_more_bits_than_16_bit_counts(order, snps, step, overlap):
    print(f"case: order {order} {snps} SNPs, rows above 16-bit counts, step {step} overlap {overlap}", flush=True)
    # above 2^16: one row, or a SNP's rows together; few enough controls that
    # the MI of these tables stays positive
    bits, called = (33280, 200) if overlap else (66560, 2000)
    words, cw, tw = wide_rows(snps, bits, called, 5 * order + step, overlap)
    d = fa.Dataset.from_words(words, snps, cw, tw, 33280 if overlap else 60000, 9000)
    want = check(d, order, fa.Distribution(snps, order - 1, step, 0), 60, DIRECT)
    assert len(want[1]) == 60 and (want[1] > 0).all()
    d.close()


@pytest.mark.parametrize("order,snps,cases,ctrls", [(2, 700, 5000, 4300), (3, 140, 2600, 2500)])
def test_snps_uncalled_in_one_class(order, snps, cases, ctrls):
    print(f"case: order {order} {snps}x{cases}+{ctrls}, SNPs uncalled in a class", flush=True)
    g = genotypes(snps, cases + ctrls, 70 + order, 0.01)
    g[3, :cases] = -1              # no case called
    g[snps - 2, cases:] = -1       # no control called
    g[snps // 2, :] = -1           # nobody
    d = fa.Dataset.from_genotypes(g, (np.arange(cases + ctrls) >= cases).astype(np.uint8))
    check(d, order, fa.Distribution(snps, order - 1), 200, DIRECT)
    check(d, order, fa.Distribution(snps, order - 1, 2, 1), 200, DIRECT)
    d.close()


@pytest.mark.parametrize("order,snps,cases,ctrls,step", [
    (2, 900, 6000, 5700, 2), (3, 200, 5000, 4700, 3), (4, 64, 2100, 2300, 1), (4, 64, 2100, 2300, 3),
    (2, 300, 700, 500, 1), (3, 130, 700, 500, 1),
])
def test_samples_that_every_snp_misses(order, snps, cases, ctrls, step):
    print(f"case: order {order} {snps}x{cases}+{ctrls} step {step}, samples without a call", flush=True)
    g = genotypes(snps, cases + ctrls, 80 + order, 0)
    g[:, np.random.default_rng(9).random(cases + ctrls) < 0.03] = -1
    d = fa.Dataset.from_genotypes(g, (np.arange(cases + ctrls) >= cases).astype(np.uint8))
    check(d, order, fa.Distribution(snps, order - 1, step, step - 1), 200, MARGINAL)
    d.close()
