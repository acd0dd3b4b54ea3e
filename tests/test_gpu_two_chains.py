"""Batches that run as two chains of rounds on two streams: every mode, an odd
count, resident keys, caller's randomness, and calls from several host threads
on streams of their own, each of which forks a second stream."""
import threading

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu
N_ITEMS = 12289


def _batch(mode):
    rng = np.random.default_rng(mode)
    m = rng.integers(0, 256, (N_ITEMS, 40), dtype=np.uint8)
    _, sk = oracle.keypair_counter_batch(mode, 64, rand_index=mode)
    idx = rng.integers(0, 64, N_ITEMS).astype(np.uint32)
    return rng, m, [r.tobytes() for r in m], sk, idx


@pytest.mark.parametrize("mode", [2, 3, 5])
def test_two_chains_match_oracle(mode):
    from cudilithium_amd import api
    rng, m, msgs, sk, idx = _batch(mode)
    exp, att = oracle.sign_batch(mode, msgs, sk[idx])
    ctx = api.SignContext(mode, N_ITEMS)
    assert np.array_equal(ctx.sign(msgs, sk[idx]), exp)
    assert np.array_equal(ctx.attempt_counts(N_ITEMS), att)
    rnd = rng.integers(0, 256, (N_ITEMS, 64), dtype=np.uint8)
    assert np.array_equal(ctx.sign_randomized(msgs, rnd, sk[idx]), oracle.sign_rnd_batch(mode, m, sk[idx], rnd)[0])
    pk, _ = oracle.keypair_counter_batch(mode, 64, rand_index=mode)
    store = api.KeyStore(mode, 64)
    store.load(0, pk, sk)
    res = api.SignContext(mode, N_ITEMS, resident_only=True)
    assert np.array_equal(res.sign_resident(store, idx, msgs), exp)


def test_two_chains_from_several_threads():
    from cudilithium_amd import api
    from cudilithium_amd.device import DeviceBuffer, Stream
    mode = 2
    _, _, msgs, sk, idx = _batch(mode)
    exp, _ = oracle.sign_batch(mode, msgs, sk[idx])
    d_sk, dm = DeviceBuffer.from_array(np.ascontiguousarray(sk[idx])), api.DeviceMessages(msgs)
    out, errors = [None] * 4, []

    def caller(t):
        try:
            ctx, st = api.SignContext(mode, N_ITEMS), Stream()
            d_sig = DeviceBuffer(exp.nbytes)
            for _ in range(3):
                ctx.sign_device(d_sig, d_sk, dm, stream=st.handle)
            st.synchronize()
            out[t] = d_sig.download(exp.shape, np.uint8)
        except Exception as e:  # noqa: BLE001
            errors.append(e)
    threads = [threading.Thread(target=caller, args=(t,)) for t in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors
    for got in out:
        assert np.array_equal(got, exp)
