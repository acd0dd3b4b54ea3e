"""Signing contexts with fewer attempt slots than items: rounds over a part of
the items at a time, the persistent kernel beyond 32 items per slot, and one
slot for so many items that its workgroup runs tens of thousands of rounds."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def _check(mode, n, nslots):
    from cudilithium_amd.api import SignContext
    m = np.random.default_rng(n).integers(0, 256, (n, 40), dtype=np.uint8)
    _, sk = oracle.keypair_counter_batch(mode, n, rand_index=n)
    exp, att = oracle.sign_batch(mode, m, sk)
    ctx = SignContext(mode, n, nslots)
    assert np.array_equal(ctx.sign([r.tobytes() for r in m], sk), exp)
    assert np.array_equal(ctx.attempt_counts(n), att)
    return int(att.sum())


@pytest.mark.parametrize("mode", [2, 3, 5])
@pytest.mark.parametrize("n,nslots", [(333, 333), (333, 64), (333, 11), (333, 10), (333, 7), (40, 1), (17, 1), (1, 1)])
def test_few_slots_match_oracle(mode, n, nslots):
    _check(mode, n, nslots)


def test_no_limit_on_the_rounds_that_a_long_queue_takes():
    # 20,000 rounds without a signature are an error; with signatures they are not
    assert _check(2, 6000, 1) > 20000


@pytest.mark.parametrize("mode", [2, 3, 5])
@pytest.mark.parametrize("n", [1536, 1537])
def test_challenge_forms_change_at_3072_attempts(mode, n):
    # two attempts for each item in the first round: 3,072 with a wave each, 3,074 with a row
    _check(mode, n, 2 * n)
