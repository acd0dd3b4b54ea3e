"""The persistent kernel: alone under every tiling (the phase profile runs it,
whatever the batch), and taking over the items that the planned rounds left,
from the middle of their nonces and of the list."""
import math

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [2, 3, 5])
@pytest.mark.parametrize("spb,claim", [(1, 0), (8, 0), (8, 3), (16, 0), (16, 5), (32, 0), (32, 16), (32, 1)])
def test_every_tiling_signs_a_queue(mode, spb, claim):
    from cudilithium_amd.api import SignContext
    n, nslots = 150, 96  # several refills of each workgroup
    m = np.random.default_rng(spb + claim).integers(0, 256, (n, 70), dtype=np.uint8)
    msgs = [r.tobytes() for r in m]
    _, sk = oracle.keypair_counter_batch(mode, n, rand_index=spb)
    exp, att = oracle.sign_batch(mode, msgs, sk)
    for blocks in (0, 2):
        ctx = SignContext(mode, n, nslots)
        ctx.set_tiling(spb, 0, blocks)
        ctx.set_claim(claim)
        ctx.profile_phases(True)
        assert np.array_equal(ctx.sign(msgs, sk), exp)
        assert np.array_equal(ctx.attempt_counts(n), att)
        assert all(v > 0 for v in ctx.phase_cycles().values())


# messages (8 bytes, little-endian) that take 53 / 53 / 52 attempts under the
# first of the counter keys from 9 on
HARD = {2: (839135, 53), 3: (37878, 53), 5: (61193, 52)}


def _left_after_the_rounds(mode, attempts, nslots):
    """Items (with their next nonce) that the rounds planned for a batch leave."""
    target = min(nslots, 16384)
    fail = 1 - 1 / {2: 4.25, 3: 5.1, 5: 3.85}[mode]

    def plan(u):
        m = min(max(target // u if u else 0, 2), 32, nslots)
        return min(nslots // m, u), m
    expected, left = float(len(attempts)), [(i, 0) for i in range(len(attempts))]
    for _ in range(48):
        if expected <= 0.05:
            break
        count, m = plan(len(left))
        left = [(i, nonce + m) for i, nonce in left[:count] if attempts[i] > nonce + m] + left[count:]
        count, m = plan(math.ceil(expected))
        expected = max(0.0, expected - count) + min(expected, count) * fail ** m
    return left


@pytest.mark.parametrize("mode", [2, 3, 5])
@pytest.mark.parametrize("n,nslots", [(1, 1), (40, 64), (600, 1500), (600, None)])
def test_items_left_by_the_rounds_are_finished(mode, n, nslots):
    from cudilithium_amd.api import SignContext
    hard, attempts = HARD[mode]
    _, sk = oracle.keypair_counter_batch(mode, n, rand_index=9)
    # every item the hard one, but for each tenth an ordinary one
    msgs = [(hard if i % 10 or n == 1 else i).to_bytes(8, "little") for i in range(n)]
    sk = np.repeat(sk[:1], n, 0)
    exp, att = oracle.sign_batch(mode, msgs, sk)
    assert att[n - 1] == attempts
    ctx = SignContext(mode, n, nslots)
    left = _left_after_the_rounds(mode, att, ctx.slots)
    assert left and any(nonce > 0 for _, nonce in left)
    for _ in range(2):
        assert np.array_equal(ctx.sign(msgs, sk), exp)
        assert np.array_equal(ctx.attempt_counts(n), att)
        assert ctx.status() == 0
