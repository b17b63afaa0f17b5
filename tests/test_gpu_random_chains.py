"""kd_dropout and kd_bernoulli over counts that are drawn in chains (more than 300 blocks of 312): around
the chains of 64 blocks and the rounds of 64 chains, from positions inside a block, against the C
oracle's sequential draws bit for bit, the state after them included."""
import numpy as np
import pytest

import kd
import support
from test_oracle_random import draws, dropout_input, same, seeded

pytestmark = pytest.mark.gpu

P = support.ptr
CHAIN, ROUND = 64 * 312, 4096 * 312


@pytest.mark.parametrize("count,skip", [(300 * 312, 312), (299 * 312, 0), (300 * 312 + 1, 12), (5 * CHAIN - 1, 100), (5 * CHAIN + 1, 312),
                                        (ROUND, 312), (ROUND + 1, 312), (ROUND - 311, 311), (2 * ROUND + 313, 7),
                                        (3 * ROUND + 40 * CHAIN + 17, 5000)])
def test_draws_in_chains(kdb, oracle, count, skip):
    x = dropout_input(count, np.float32, 5)
    want, want_mask = np.zeros_like(x), np.zeros_like(x)
    want_state = seeded(oracle, 11)
    draws(oracle, want_state, skip)
    state = want_state.copy()
    assert oracle.oracle_dropout(kd.F32, P(want), P(want_mask), P(x), count, 0.9, P(want_state)) == 0
    dx, dout, dmask = kdb.to_device(x), kdb.empty(x.shape, x.dtype), kdb.empty(x.shape, x.dtype)
    kdb.check(kdb.lib.kd_dropout(kd.F32, dout.ptr, dmask.ptr, dx.ptr, count, 0.9, P(state)), "kd_dropout")
    np.testing.assert_array_equal(state, want_state)
    np.testing.assert_array_equal(dmask.numpy(), want_mask)
    assert same(dout.numpy(), want)


@pytest.mark.parametrize("dtype,npt", [(kd.F64, np.float64), (kd.I64, np.int64), (kd.BOOL, np.bool_)])
def test_masks_in_chains(kdb, oracle, dtype, npt):
    count = 9 * CHAIN + 5
    want = np.zeros(count, npt)
    want_state = seeded(oracle, 3)
    draws(oracle, want_state, 41)
    state = want_state.copy()
    assert oracle.oracle_bernoulli(dtype, P(want), count, 0.25, P(want_state)) == 0
    out = kdb.empty((count,), npt)
    kdb.check(kdb.lib.kd_bernoulli(dtype, out.ptr, count, 0.25, P(state)), "kd_bernoulli")
    np.testing.assert_array_equal(out.numpy(), want)
    np.testing.assert_array_equal(state, want_state)
