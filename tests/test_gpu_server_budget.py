"""GPU: the scan server's memory budget.  The padding of the order-3 pair
table, 256 KB, is not what decides whether a request can be served: a budget
that holds its tables, staging, binomials and pairs does."""
import numpy as np
import pytest

import fiuncho_amd as fa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("budget", [330 << 10, 450 << 10, 4 << 20])   # 302 KB without the padding, 564 KB with it
def test_order3_request_within_a_small_budget(budget):
    print(f"case: server budget {budget}", flush=True)
    snps, cases, ctrls = 90, 700, 650
    words, _, cw, tw = fa.synth_generate(fa.synth_spec(snps, cases, ctrls, seed=64), words=True)
    d = fa.Dataset.from_words(words, snps, cw, tw, cases, ctrls)
    want = fa.GpuSearch().run_arrays(d, 3, fa.Distribution(snps, 2), 20)
    srv = fa.Server(fa.batch_config(memory_budget=budget))
    ids = [srv.submit(order=3, outputs=20, words=words, snps=snps, cases_words=cw, ctrls_words=tw, cases=cases,
                      ctrls=ctrls) for _ in range(2)]
    for rid in ids:
        got = srv.wait(rid, timeout_ms=30000.0)
        assert got[0].tolist() == want[0].tolist() and np.array_equal(got[1], want[1])
    srv.close()
    d.close()


def test_request_above_the_budget_is_refused():
    words, _, cw, tw = fa.synth_generate(fa.synth_spec(90, 700, 650, seed=64), words=True)
    srv = fa.Server(fa.batch_config(memory_budget=250 << 10))
    with pytest.raises(fa.FiuError):
        srv.submit(order=3, outputs=20, words=words, snps=90, cases_words=cw, ctrls_words=tw, cases=700, ctrls=650)
    srv.close()
