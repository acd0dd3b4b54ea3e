"""Tilings that calls read: resident verification under every item count per
workgroup, at batch sizes of each of its hash forms, and the tuner that times
that call."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.fixture
def tiling():
    from cudilithium_amd import api, autotune
    yield lambda mode, v: api.L().dil_set_kernel_tiling(autotune.TILE_KINDS["verify"], mode, -1, v)
    autotune.apply_cache(api.L())


@pytest.mark.parametrize("mode,values", [(2, (2, 4, 8, 16)), (3, (2, 4, 8)), (5, (2, 4, 8))])
def test_resident_verification_under_every_tiling(tiling, mode, values):
    from cudilithium_amd import api
    rng = np.random.default_rng(mode)
    nkeys, n = 37, 4099
    pk, sk = oracle.keypair_counter_batch(mode, nkeys, rand_index=mode)
    idx = rng.integers(0, nkeys, n).astype(np.uint32)
    m = rng.integers(0, 256, (n, 50), dtype=np.uint8)
    msgs = [r.tobytes() for r in m]
    sig, _ = oracle.sign_batch(mode, msgs, sk[idx])
    flip = np.arange(0, n, 7)
    sig[flip, rng.integers(0, sig.shape[1], len(flip))] ^= 16
    ret = oracle.verify_batch(mode, sig, msgs, pk[idx])
    store = api.KeyStore(mode, nkeys)
    store.load(0, pk)
    for v in values:
        assert tiling(mode, v) == 0
        for k in (1, 17, 3072, 3079, n):  # waves, rows, lane pairs; last workgroups of 1 .. v items
            for flags in (None, api.HASH_LONG_MESSAGES):
                assert np.array_equal(store.verify(idx[:k], sig[:k], msgs[:k], flags), ret[:k]), (v, k, flags)
    assert tiling(mode, 32) != 0 and (mode == 2 or tiling(mode, 16) != 0)


def test_verify_tuner_times_the_call_that_reads_the_tiling(tiling, monkeypatch):
    from cudilithium_amd import api, autotune
    L = api.L()
    calls = []
    timed = L.dil_verify_device_resident

    def resident(*args):
        calls.append(L.dil_get_kernel_tiling(autotune.TILE_KINDS["verify"], 2, 50))
        return timed(*args)
    monkeypatch.setattr(L, "dil_verify_device_resident", resident)
    autotune.tune_kernel("verify", 2, 50, reps=1, values=(2, 8), log=lambda s: None)
    assert set(calls) == {2, 8}
