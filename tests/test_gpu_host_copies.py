"""The engine's copies of a batch between host and device memory: sources going up as parts of
the staging buffer packed by several threads, transfers coming down by halves of it. A batch of
many parts (each part of the buffer used more than once, a row of results across both halves)
equals the same pairs loaded one k1 at a time, and the oracle; a block of one pair and source type
that is larger than a part equals the oracle.
"""
import numpy as np
import pytest

from song_amd import lib as L
from tests.conftest import oracle_pairs, product_pairs, run_oracle

MANY = dict(has_T=1, has_E=1, m_list=[0, 1, 2], l_max_los_t=4, l_max_los_p=4, k_size=9,
            k_min=2e-3, k_max=0.03, k3_size=60, tau_size=400, l_size=40, l_max=400, dk_fine=3e-5,
            xx_max=600.0)


@pytest.mark.gpu
def test_many_parts(oracle):
    s = L.Scenario(L.Config(**MANY))
    s.prepare()
    eng = L.Engine(0)
    eng.set_shape(L.FORM_FP64, 1, 2, 0, 0)  # one kernel for every batch
    eng.load(s)
    eng.run()
    eng.store(s)
    whole = s.gather()
    pairs = [(i, j) for i in range(MANY["k_size"]) for j in range(i + 1)]
    n_types = 2 * (5 + 4 + 3)  # source types of a pair, at least T and E by (L, m)
    assert whole.nbytes > 40 << 20 and len(pairs) * 400 * 60 * 8 * n_types > 128 << 20
    ref = oracle_pairs(s, oracle, [pairs[0], pairs[-1]])
    got = product_pairs(s, whole, pairs)
    for p in ref:
        assert np.array_equal(got[p], ref[p]), p
    for i in range(MANY["k_size"]):
        eng.load(s, i, i + 1)
        eng.run()
        eng.store(s)
    assert np.array_equal(s.gather(), whole)


@pytest.mark.gpu
def test_block_larger_than_a_part(oracle):
    cfg = L.Config(has_T=1, has_E=0, m_list=[0], l_max_los_t=0, k_size=2, k_min=0.004, k_max=0.008,
                   k3_size=250, tau_size=2300, l_size=4, l_max=60, dk_fine=1e-3, xx_max=200.0)
    ref = run_oracle(L.Scenario(cfg), oracle)
    s = L.Scenario(cfg)
    s.prepare()
    eng = L.Engine(0)
    eng.load(s)
    eng.run()
    eng.store(s)
    assert np.array_equal(s.gather(), ref)
