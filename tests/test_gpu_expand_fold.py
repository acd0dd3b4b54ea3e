"""ExpandA folded into matrix-vector products (keygen and verification) for
keys whose rejection sampling falls behind the window of live coefficients,
and at batch sizes that leave a wave's last places empty.

The seeds give, in at least one entry of A, five rejected candidates within
the first 168 or 224 (a window allows for four); found by counting candidates
>= q of SHAKE128(rho || l || k)."""
import hashlib

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

SLOW = [11448, 15351, 32739, 10322, 53407]


def _seeds(n):
    """n seeds, the slow ones spread over the batch."""
    ids = np.arange(n) + 1
    where = np.arange(0, n, 3)[:len(SLOW)]
    ids[where] = SLOW[:len(where)]
    return np.array([list(int(i).to_bytes(32, "little")) for i in ids], dtype=np.uint8)


def test_the_seeds_are_slow():
    for seed, k, l, cand in ((11448, 0, 2, 224), (15351, 4, 0, 168), (32739, 0, 3, 168), (10322, 1, 6, 224),
                             (53407, 1, 2, 168)):
        rho = hashlib.shake_256(seed.to_bytes(32, "little")).digest(32)
        b = np.frombuffer(hashlib.shake_128(rho + bytes([l, k])).digest(168 * 4), np.uint8).reshape(-1, 3).astype(int)
        t = b[:, 0] | b[:, 1] << 8 | (b[:, 2] & 127) << 16
        assert (t[:cand] >= 8380417).sum() == 5


@pytest.mark.parametrize("mode", [2, 3, 5])
@pytest.mark.parametrize("n", [1, 2, 3, 5, 14, 67])
def test_keys_and_verdicts_match_oracle(mode, n):
    from cudilithium_amd import api
    seeds = _seeds(n)
    pk, sk = api.keypair_device(mode, seeds=seeds)
    epk, esk = oracle.keypair_batch(mode, seeds)
    assert np.array_equal(pk, epk) and np.array_equal(sk, esk)
    m = np.random.default_rng(n).integers(0, 256, (n, 45), dtype=np.uint8)
    sig, _ = oracle.sign_batch(mode, m, esk)
    d = api.Dilithium(mode)
    assert (d.verify(sig, m, epk) == 0).all()
    sig[::2, 40] ^= 1  # z of every other item
    got = d.verify(sig, m, epk)
    assert np.array_equal(got, oracle.verify_batch(mode, sig, m, epk))
    assert np.array_equal(got, np.where(np.arange(n) % 2 == 0, -1, 0))
