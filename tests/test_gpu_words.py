"""GPU: the host-layout words read back from a dataset, also while a stream of
the process records a graph."""
import numpy as np
import pytest
import torch

import fiuncho_amd as fa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("snps,cases,ctrls", [(1, 1, 1), (70, 500, 700), (900, 40000, 33000)])
def test_words_round_trip(snps, cases, ctrls):
    print(f"case: words of {snps}x{cases}+{ctrls}", flush=True)
    words, _, cw, tw = fa.synth_generate(fa.synth_spec(snps, cases, ctrls, seed=95), words=True)
    d = fa.Dataset.from_words(words, snps, cw, tw, cases, ctrls)
    assert np.array_equal(d.words(), words)
    d.close()


def test_words_while_a_graph_is_recorded():
    print("case: words during capture", flush=True)
    words, _, cw, tw = fa.synth_generate(fa.synth_spec(300, 900, 800, seed=96), words=True)
    d = fa.Dataset.from_words(words, 300, cw, tw, 900, 800)
    x = torch.arange(1000, device="cuda", dtype=torch.float32)
    y = x * 2 + 1
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        y = x * 2 + 1
        got = d.words()
    assert np.array_equal(got, words)
    for i in range(3):
        x.fill_(float(i))
        g.replay()
        torch.cuda.synchronize()
        assert np.array_equal(d.words(), words)
        assert (y == 2 * i + 1).all()
    d.close()
