"""The calls this engine is measured on: batched keygen, signing,
verification and NTT through the public entry points, from one signature to
card-filling batches, with inputs resident in HBM, resident keys, captured
graphs and host buffers.

A case is a dict of plain values:

    name     (listed cases only)
    op       "sign" | "verify" | "keygen" | "ntt"
    mode     2, 3 or 5 (0 for ntt)
    n        items (polynomials for ntt)
    path     "device"    inputs in device memory, one call
             "graph"     the same call captured once, replayed per pass
             "resident"  keys held expanded in a KeyStore (the serving form)
             "pinned"    the drop-in call on pinned host buffers
             "pageable"  the drop-in call on ordinary numpy arrays
             "pipeline" | "forward" | "inverse" for ntt
    mlo, mhi message lengths: log-uniform in [mlo, mhi] bytes, or all mlo
             when equal (the drop-in calls take one length for the batch)
    long     True: the long-message hashing option of the resident calls
"""
from __future__ import annotations

import math

import numpy as np
import torch

from cudilithium_amd import api, ntt, workmodel

Q = 8380417
# signatures take this many attempts on average (the specification's
# rejection probabilities)
ATTEMPTS = {2: 4.25, 3: 5.1, 5: 3.85}
PK_BYTES = {2: 1312, 3: 1952, 5: 2592}
SK_BYTES = {2: 2528, 3: 4000, 5: 4864}
SIG_BYTES = {2: 2420, 3: 3293, 5: 4595}
EXEC_THRESHOLD = 2048  # the reference callers' default


def _case(name, op, mode, n, path, mlo=0, mhi=0, long=False):
    c = {"op": op, "mode": mode, "n": n, "path": path, "mlo": mlo, "mhi": mhi, "long": long}
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # a signing service's full batch: keys and messages of all lengths
        # from a line of text to a page, already in HBM (the benchmark's
        # default workload)
        _case("sign3_16384", "sign", 3, 16384, "device", 32, 4096),
        # the highest security level at an ordinary, odd batch size, replayed
        # as a graph by a loop that signs batch after batch
        _case("sign5_3001_graph", "sign", 5, 3001, "graph", 32, 4096),
        # one caller's slice of the reference's stream mode
        _case("sign2_1000", "sign", 2, 1000, "device", 32, 32),
        # a serving lane under light load: a handful of requests under
        # resident keys, where latency counts
        _case("sign3_17_resident", "sign", 3, 17, "resident", 32, 4096),
        # the reference's published benchmark conditions: 10,000 items,
        # 32-byte messages, pinned host buffers, copies included
        _case("sign2_10000_pinned", "sign", 2, 10000, "pinned", 32, 32),
        # a chain or log auditor's bulk check, one key per item
        _case("verify5_65536_graph", "verify", 5, 65536, "graph", 1024, 1024),
        # a serving lane with a backlog: known signers, messages of all lengths
        _case("verify3_2500_resident", "verify", 3, 2500, "resident", 32, 4096),
        # the few signatures of one request, checked on their own: launches
        # and latency
        _case("verify2_16", "verify", 2, 16, "device", 64, 64),
        # the reference's published conditions again
        _case("verify2_10000_pinned", "verify", 2, 10000, "pinned", 32, 32),
        # provisioning: a batch of keys from caller-drawn seeds
        _case("keygen3_16384", "keygen", 3, 16384, "device"),
        # the reference's published conditions again (counter seeds)
        _case("keygen2_10000_pinned", "keygen", 2, 10000, "pinned"),
        # the standalone transform as a library call: INTT(NTT(a) o b)
        _case("ntt_65536", "ntt", 0, 65536, "pipeline"),
    ]


def _log_int(rng, lo, hi):
    """An integer in [lo, hi], spread over its logarithm."""
    return min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))


def draw(rng):
    op = rng.choice(["sign", "sign", "verify", "verify", "keygen", "ntt"])
    if op == "ntt":
        return _case(None, "ntt", 0, _log_int(rng, 1, 65536), rng.choice(["pipeline", "forward", "inverse"]))
    mode = rng.choice([2, 3, 5])
    if op == "keygen":
        path = rng.choice(["device", "graph", "pinned", "pageable"])
        return _case(None, op, mode, _log_int(rng, 1, 16384 if path in ("pinned", "pageable") else 32768), path)
    path = rng.choice(["device", "graph", "resident", "pinned", "pageable"])
    least = 1 if op == "sign" else 16  # a verdict alone says little about its inputs
    mlo, mhi = rng.choice([(32, 32), (64, 64), (1024, 1024), (32, 4096), (1, 512)])
    if path in ("pinned", "pageable"):
        # 0: the drop-in calls accept an empty message
        mlo = mhi = rng.choice([0, 32, 59, 64, 1024])
        return _case(None, op, mode, _log_int(rng, least, 16384), path, mlo, mhi)
    if path == "resident" and rng.random() < 0.25:
        # messages too long for one lane to hash without holding up the batch
        return _case(None, op, mode, _log_int(rng, least, 256), path, 4096, 65536, True)
    return _case(None, op, mode, _log_int(rng, least, 16384 if op == "sign" else 32768), path, mlo, mhi)


# ------------------------------------------------------------------ inputs

def _stream():
    """The stream a torch program is on, as the entry points take it."""
    return torch.cuda.current_stream().cuda_stream or None


class _Buf:
    """A torch tensor handed to the entry points, which take device buffers
    by their address."""

    def __init__(self, t):
        self.t, self.ptr, self.nbytes = t, t.data_ptr(), t.numel() * t.element_size()


def _zeros(shape, dtype=torch.uint8):
    return _Buf(torch.zeros(shape, dtype=dtype, device="cuda"))


class _Messages:
    """n messages in device memory: flat bytes, 8-aligned offsets, lengths."""

    def __init__(self, lens, gen):
        offs = np.zeros(len(lens), np.int64)
        offs[1:] = np.cumsum((lens[:-1] + 7) // 8 * 8)
        total = int(offs[-1] + (lens[-1] + 7) // 8 * 8)
        self.n, self.host_lens = len(lens), lens
        self.data = _Buf(_random_bytes((max(8, total),), gen))
        self.offs = _Buf(torch.from_numpy(offs).cuda())
        self.lens = _Buf(torch.from_numpy(lens.astype(np.int32)).cuda())


def _random_bytes(shape, gen):
    return torch.randint(0, 256, shape, dtype=torch.uint8, device="cuda", generator=gen)


def _lengths(case, rs):
    lo, hi, n = case["mlo"], case["mhi"], case["n"]
    if lo == hi:
        return np.full(n, lo, np.int64)
    return np.floor(lo * (hi / lo) ** rs.random(n)).astype(np.int64)


def _check(r):
    if r:
        raise RuntimeError(f"status {r}")


def _keygen_device(mode, seeds, n):
    """Keys of `seeds` (n x 32, on the device), left on the device."""
    pk, sk = _zeros((n, PK_BYTES[mode])), _zeros((n, SK_BYTES[mode]))
    wrow = (api.L().dil_keypair_work_row_bytes(mode) + 255) // 256 * 256
    work = _zeros((n, wrow))
    _check(api.L().dil_keypair_device(mode, pk.ptr, PK_BYTES[mode], sk.ptr, SK_BYTES[mode], seeds.ptr, 32, 0, n,
                                      work.ptr, wrow, _stream()))
    torch.cuda.synchronize()
    return pk, sk


def _pinned(a):
    """The array in pinned host memory; the tensor behind it lives as long as
    the array does."""
    return torch.from_numpy(a).pin_memory().numpy()


def _flip(sig, rs):
    """One flipped bit in a tenth of the signatures (they must be rejected), or
    in half of a few."""
    n, nbytes = sig.shape
    rows = np.flatnonzero(rs.random(n) < (0.1 if n >= 256 else 0.5))
    bits = rs.integers(0, 8 * nbytes, len(rows))
    mask = torch.from_numpy((1 << (bits % 8)).astype(np.uint8)).cuda()
    r, c = torch.from_numpy(rows).cuda(), torch.from_numpy(bits // 8).cuda()
    sig[r, c] = sig[r, c] ^ mask


class _State:
    pass


def prepare(case, seed):
    op, mode, n, path = case["op"], case["mode"], case["n"], case["path"]
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    rs = np.random.default_rng(seed)
    st = _State()
    st.case = case
    api.L()
    if op == "ntt":
        # coefficients uniform in [-q, q), as the transforms' callers hold them
        st.a = _Buf(torch.randint(-Q, Q, (n, 256), dtype=torch.int32, device="cuda", generator=gen))
        if path == "pipeline":
            st.b = _Buf(torch.randint(-Q, Q, (n, 256), dtype=torch.int32, device="cuda", generator=gen))
            st.c = _zeros((n, 256), torch.int32)
        else:
            st.c = _zeros((n, 256), torch.int32)  # the in-place calls work on a copy
        torch.cuda.synchronize()
        return st
    seeds = _Buf(_random_bytes((n, 32), gen))
    if op == "keygen":
        return _prepare_keygen(st, mode, n, path, seeds, rs)
    lens = _lengths(case, rs)
    host = path in ("pinned", "pageable")
    if path == "resident":
        nkeys = max(1, min(n, 1024))  # signers with resident keys; several requests of a batch share one
        st.store = api.KeyStore(mode, nkeys)
        st.store.keygen(0, seeds.t[:nkeys].cpu().numpy())
        st.idx = _Buf(torch.from_numpy(rs.integers(0, nkeys, n).astype(np.int32)).cuda())
    else:
        st.pk, st.sk = _keygen_device(mode, seeds, n)
    st.msgs = _Messages(lens, gen)
    st.sig = _zeros((n, SIG_BYTES[mode]))
    st.ctx = api.SignContext(mode, n, resident_only=path == "resident")
    if case["long"]:
        st.ctx.set_message_hashing(api.HASH_LONG_MESSAGES)
    if op == "verify":
        _sign(st)
        torch.cuda.synchronize()
        _flip(st.sig.t, rs)
        st.ctx = None
        if not host:
            st.wrow = api.L().dil_verify_work_row_bytes(mode)
            st.work, st.ret = _zeros((n, st.wrow)), _zeros((n,), torch.int32)
    if host:
        _prepare_dropin(st, op, mode, n, path, int(lens[0]))
    elif path == "graph":
        if op == "sign":
            st.graph = st.ctx.graph(st.sig, st.sk, st.msgs)
        else:
            st.graph = api.verify_graph(mode, st.ret, st.sig, st.pk, st.msgs, st.work, st.wrow)
    torch.cuda.synchronize()
    return st


def _prepare_keygen(st, mode, n, path, seeds, rs):
    if path in ("pinned", "pageable"):
        st.rand_index = int(rs.integers(0, 1 << 40))
        st.pool = api.reference_pool(mode, api.POOL_KEYPAIR, n)
        outs = np.zeros((n, PK_BYTES[mode]), np.uint8), np.zeros((n, SK_BYTES[mode]), np.uint8)
        st.h_pk, st.h_sk = [_pinned(o) for o in outs] if path == "pinned" else outs
    else:
        st.seeds = seeds
        st.pk, st.sk = _zeros((n, PK_BYTES[mode])), _zeros((n, SK_BYTES[mode]))
        st.wrow = (api.L().dil_keypair_work_row_bytes(mode) + 255) // 256 * 256
        st.work = _zeros((n, st.wrow))
        if path == "graph":
            st.graph = api.keypair_graph(mode, st.pk, st.sk, n, st.work, st.wrow, st.seeds)
    torch.cuda.synchronize()
    return st


def _prepare_dropin(st, op, mode, n, path, mlen):
    """Host arrays, pools and tables as the reference's callers allocate them."""
    msg = np.zeros((n, 0), np.uint8)
    if mlen:
        pitch = (mlen + 7) // 8 * 8
        msg = st.msgs.data.t.cpu().numpy()[:n * pitch].reshape(n, pitch)[:, :mlen]
    arrays = {"msg": np.ascontiguousarray(msg)}
    st.mlen = mlen
    if op == "sign":
        arrays["sk"] = st.sk.t.cpu().numpy()
        arrays["sig"] = np.zeros((n, SIG_BYTES[mode]), np.uint8)
        st.pool = api.reference_pool(mode, api.POOL_SIGN, n, mlen)
        st.temp = api.reference_pool(mode, api.POOL_SIGN_TEMP, EXEC_THRESHOLD)
        st.lut = api.TaskLut(n, EXEC_THRESHOLD)
    else:
        arrays["pk"] = st.pk.t.cpu().numpy()
        arrays["sig"] = st.sig.t.cpu().numpy()
        arrays["ret"] = np.zeros(n, np.int32)
        st.pool = api.reference_pool(mode, api.POOL_VERIFY, n, mlen)
    st.ctx = st.sig = st.pk = st.sk = st.msgs = None
    if path == "pinned":
        arrays = {k: _pinned(v) for k, v in arrays.items()}
    st.h = arrays


# -------------------------------------------------------------------- pass

def _sign(st):
    if st.case["path"] == "resident":
        st.ctx.sign_resident_device(st.store, st.idx, st.sig, st.msgs, stream=_stream())
    else:
        st.ctx.sign_device(st.sig, st.sk, st.msgs, stream=_stream())


def run(st):
    c = st.case
    op, mode, n, path = c["op"], c["mode"], c["n"], c["path"]
    s = _stream()
    if op == "ntt":
        if path == "pipeline":
            ntt.pipeline_device(st.c, st.a, st.b, n, stream=s)
        else:
            st.c.t.copy_(st.a.t)
            (ntt.forward_device if path == "forward" else ntt.inverse_device)(st.c, n, stream=s)
        return st.c.t
    if path == "graph":
        st.graph.launch(s)
    elif op == "keygen":
        if path == "device":
            _check(api.L().dil_keypair_device(mode, st.pk.ptr, PK_BYTES[mode], st.sk.ptr, SK_BYTES[mode],
                                              st.seeds.ptr, 32, 0, n, st.work.ptr, st.wrow, s))
        else:
            api.crypto_sign_keypair(mode, st.h_pk, st.h_sk, st.pool, st.pool.pitch, n, s, st.rand_index)
            return st.h_pk, st.h_sk
    elif op == "sign":
        if path in ("pinned", "pageable"):
            api.crypto_sign_signature(mode, st.h["sig"], SIG_BYTES[mode], st.h["msg"], st.mlen, st.mlen, st.h["sk"],
                                      st.pool, st.pool.pitch, st.temp, st.temp.pitch, st.lut, EXEC_THRESHOLD, n, s)
            return st.h["sig"]
        _sign(st)
    elif path in ("pinned", "pageable"):
        api.crypto_sign_verify(mode, st.h["ret"], st.h["sig"], SIG_BYTES[mode], SIG_BYTES[mode], st.h["msg"], st.mlen,
                               st.mlen, st.h["pk"], st.pool, st.pool.pitch, n, s)
        return st.h["ret"]
    elif path == "resident":
        m = st.msgs
        _check(api.L().dil_verify_device_resident_ex(st.store.handle, st.idx.ptr, st.ret.ptr, st.sig.ptr,
                                                     SIG_BYTES[mode], m.data.ptr, m.offs.ptr, m.lens.ptr, n,
                                                     st.work.ptr, st.wrow,
                                                     api.HASH_LONG_MESSAGES if c["long"] else 0, s))
    else:
        m = st.msgs
        _check(api.L().dil_verify_device(mode, st.ret.ptr, st.sig.ptr, SIG_BYTES[mode], st.pk.ptr, PK_BYTES[mode],
                                         m.data.ptr, m.offs.ptr, m.lens.ptr, n, st.work.ptr, st.wrow, s))
    if op == "sign":
        return st.sig.t
    if op == "verify":
        return st.ret.t
    return st.pk.t, st.sk.t


# -------------------------------------------------------------------- work

def work(case):
    """Bytes in and out once, and 32-bit integer operations of the algorithm
    (workmodel's constants; signing at its mean number of attempts)."""
    op, mode, n, path = case["op"], case["mode"], case["n"], case["path"]
    if op == "ntt":
        if path == "pipeline":
            return {"bytes": 3 * 1024 * n, "flops": workmodel.NTT_PIPELINE_OPS * n}
        return {"bytes": 2 * 1024 * n,
                "flops": (workmodel.FWD_NTT_OPS if path == "forward" else workmodel.INV_NTT_OPS) * n}
    if op == "keygen":
        return {"bytes": n * (32 + PK_BYTES[mode] + SK_BYTES[mode]), "flops": n * workmodel.keygen_ops(mode)}
    lo, hi = case["mlo"], case["mhi"]
    mlen = int(lo if lo == hi else (hi - lo) / math.log(hi / lo))  # mean of the log-uniform law
    k, l = workmodel.PARAMS[mode][:2]
    if op == "sign":
        ops = ATTEMPTS[mode] * workmodel.sign_attempt_ops(mode) + workmodel.sign_fixed_ops(mode, mlen)
        per = SIG_BYTES[mode] + mlen
        if path == "resident":  # A, s1^, s2^, t0^ are held with the key and are read
            ops -= (5 * k * l) * workmodel.OPS_KECCAK + (l + 2 * k) * workmodel.FWD_NTT_OPS
            per += 4
            return {"bytes": int(n * per + min(n, 1024) * 1024 * (k * l + l + 2 * k)), "flops": int(n * ops)}
        return {"bytes": int(n * (per + SK_BYTES[mode])), "flops": int(n * ops)}
    ops, per = workmodel.verify_ops(mode, mlen), SIG_BYTES[mode] + mlen + 4
    if path == "resident":
        ops -= (5 * k * l + PK_BYTES[mode] // 136 + 1) * workmodel.OPS_KECCAK + k * workmodel.FWD_NTT_OPS
        return {"bytes": int(n * (per + 4) + min(n, 1024) * 1024 * (k * l + k)), "flops": int(n * ops)}
    return {"bytes": int(n * (per + PK_BYTES[mode])), "flops": int(n * ops)}
