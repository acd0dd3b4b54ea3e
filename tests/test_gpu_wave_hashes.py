"""Hashes and ExpandA with one sponge per wavefront: message lengths around the ends of
words and SHAKE256 blocks (the sponge also holds 32 bytes of tr), at unaligned
offsets, and the batch sizes at which signing and verification change between
one wave and fewer lanes per hash; bytes and verdicts equal the oracle's."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

# len + 32 over: empty, a word's ends, one block less a byte ... two blocks
LENGTHS = [0, 1, 3, 4, 5, 7, 8, 9, 95, 96, 97, 102, 103, 104, 105, 111, 112, 113, 238, 239, 240, 241, 375, 376, 1111]


def _msgs(rng, lens):
    return [rng.integers(0, 256, int(k), dtype=np.uint8).tobytes() for k in lens]


def _verdicts(mode, rng, sig, msgs, pk):
    sig = sig.copy()
    flip = np.arange(1, len(sig), 3)
    sig[flip, rng.integers(0, sig.shape[1], len(flip))] ^= 1
    return sig, oracle.verify_batch(mode, sig, msgs, pk)


@pytest.mark.parametrize("mode", [2, 3, 5])
def test_message_lengths_match_oracle(mode):
    from cudilithium_amd import api
    rng = np.random.default_rng(mode)
    msgs = _msgs(rng, LENGTHS)
    n = len(msgs)
    pk, sk = oracle.keypair_counter_batch(mode, n, rand_index=77)
    exp, att = oracle.sign_batch(mode, msgs, sk)
    ctx = api.SignContext(mode, n)
    assert np.array_equal(ctx.sign(msgs, sk), exp)
    assert np.array_equal(ctx.attempt_counts(n), att)
    rp = rng.integers(0, 256, (n, 64), dtype=np.uint8)
    rnd = ctx.sign_randomized(msgs, rp, sk)
    assert (oracle.verify_batch(mode, rnd, msgs, pk) == 0).all()
    sig, ret = _verdicts(mode, rng, exp, msgs, pk)
    assert np.array_equal(api.verify_device(mode, sig, msgs, pk), ret)
    ks = api.KeyStore(mode, n)
    ks.load(0, pk, sk)
    idx = np.arange(n, dtype=np.uint32)
    assert np.array_equal(ctx.sign_resident(ks, idx, msgs), exp)
    assert np.array_equal(ks.verify(idx, sig, msgs), ret)


@pytest.mark.parametrize("n", [1, 1024, 1025, 2048, 2049, 3072, 3073])
def test_batch_size_edges_match_oracle(n):
    from cudilithium_amd import api
    mode = 2
    rng = np.random.default_rng(n)
    msgs = _msgs(rng, rng.integers(0, 150, n))
    pk, sk = oracle.keypair_counter_batch(mode, n, rand_index=n)
    exp, _ = oracle.sign_batch(mode, msgs, sk)
    ctx = api.SignContext(mode, n)
    assert np.array_equal(ctx.sign(msgs, sk), exp)
    sig, ret = _verdicts(mode, rng, exp, msgs, pk)
    assert np.array_equal(api.verify_device(mode, sig, msgs, pk), ret)
    ks = api.KeyStore(mode, n)
    ks.load(0, pk, sk)
    idx = np.arange(n, dtype=np.uint32)[::-1].copy()
    assert np.array_equal(ctx.sign_resident(ks, idx, msgs[::-1]), exp[::-1])
    assert np.array_equal(ks.verify(idx, sig[::-1].copy(), msgs[::-1]), ret[::-1])


# slow seeds of tests/test_gpu_expand_fold.py have entries of A with many
# rejected candidates; n K L around the limit of 8,192 entries
@pytest.mark.parametrize("mode,n", [(2, 5), (2, 512), (2, 513), (3, 273), (3, 274), (5, 146), (5, 147)])
def test_entry_per_wave_matches_oracle(mode, n):
    from cudilithium_amd import api
    rng = np.random.default_rng(n)
    msgs = _msgs(rng, rng.integers(0, 150, n))
    pk, sk = oracle.keypair_counter_batch(mode, n, rand_index=15351 - n // 2)
    exp, att = oracle.sign_batch(mode, msgs, sk)
    ctx = api.SignContext(mode, n)
    assert np.array_equal(ctx.sign(msgs, sk), exp)
    assert np.array_equal(ctx.attempt_counts(n), att)
    sig, ret = _verdicts(mode, rng, exp, msgs, pk)
    sig[0] = 0xFF  # z out of range and hint bytes that break the rules
    ret[0] = -1
    assert np.array_equal(api.verify_device(mode, sig, msgs, pk), ret)


@pytest.mark.parametrize("mode,n", [(5, 1), (2, 3072), (3, 3073), (2, 8192), (2, 8193)])
def test_keys_match_oracle(mode, n):
    from cudilithium_amd import api
    pk, sk = api.keypair_device(mode, n=n, rand_index=n)
    epk, esk = oracle.keypair_counter_batch(mode, n, rand_index=n)
    assert np.array_equal(pk, epk) and np.array_equal(sk, esk)
