"""Signing at the batch sizes where its launches change: one item, a few, the
edges of a list chunk (512 entries), the line between the forms of the message
hash and the one between one and two chains of rounds; signatures and attempt counts equal the oracle's, through
the device entry point and through the drop-in call with few temp rows."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def _batch(mode, n, seed):
    rng = np.random.default_rng(seed)
    _, sk = oracle.keypair_counter_batch(mode, n, rand_index=seed)
    lens = rng.integers(0, 300, n)
    lens[n // 2] = 4096  # one chain much longer than the others
    return [rng.integers(0, 256, int(k), dtype=np.uint8).tobytes() for k in lens], sk


@pytest.mark.parametrize("mode", [2, 3, 5])
@pytest.mark.parametrize("n", [1, 17, 511, 513, 2049, 4096, 4097])
def test_signatures_and_attempts_match_oracle(mode, n):
    from cudilithium_amd.api import SignContext
    msgs, sk = _batch(mode, n, 1000 * mode + n)
    exp, att = oracle.sign_batch(mode, msgs, sk)
    ctx = SignContext(mode, n)
    for _ in range(2):  # the lists and control words start over on each call
        assert np.array_equal(ctx.sign(msgs, sk), exp)
        assert np.array_equal(ctx.attempt_counts(n), att)
        assert ctx.executed_attempts() >= int(att.sum())


@pytest.mark.parametrize("n", [8192, 8193, 12287, 12288, 12801])
def test_large_batches_match_oracle(n):
    from cudilithium_amd.api import SignContext
    msgs, sk = _batch(2, n, n)
    exp, att = oracle.sign_batch(2, msgs, sk)
    ctx = SignContext(2, n)
    assert np.array_equal(ctx.sign(msgs, sk), exp)
    assert np.array_equal(ctx.attempt_counts(n), att)


@pytest.mark.parametrize("n,threshold", [(1, 1), (3, 1), (600, 1), (600, 7), (600, 600), (513, 2048)])
def test_dropin_pools_hold_the_rounds(n, threshold):
    from cudilithium_amd.api import Dilithium
    mode = 3
    m = np.random.default_rng(n).integers(0, 256, (n, 33), dtype=np.uint8)
    _, sk = oracle.keypair_counter_batch(mode, n, rand_index=n)
    assert np.array_equal(Dilithium(mode).sign(m, sk, exec_threshold=threshold), oracle.sign_batch(mode, m, sk)[0])
