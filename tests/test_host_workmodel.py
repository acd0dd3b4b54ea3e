"""Work counts behind the benchmark's roofline fractions: a fraction of the
card's issue rate counts the least instructions of the work, not the
operations that three-input instructions join."""
import pytest

from cudilithium_amd import workmodel as w


@pytest.mark.parametrize("mode,perms", [(2, 20 + 7 + 1), (3, 25 + 7 + 1), (5, 35 + 9 + 1)])
def test_least_instructions_of_an_attempt(mode, perms):
    k, l = w.PARAMS[mode][:2]
    transforms = l * w.FWD_NTT_OPS + k * w.INV_NTT_OPS + k * l * w.POINTWISE_OPS
    assert w.sign_attempt_instr(mode) == 4320 * perms + transforms < w.sign_attempt_ops(mode)
    assert w.sign_fixed_instr(mode, 32) == 4320 * (1 + 1 + 5 * k * l) < w.sign_fixed_ops(mode, 32)


@pytest.mark.parametrize("mode", [2, 3, 5])
def test_verification_is_split_by_launch(mode):
    k, l, w1, pk = w.PARAMS[mode]
    for keccak in (w.OPS_KECCAK, w.INSTR_KECCAK):
        ops = w.verify_kernel_ops(mode, 1024, keccak)
        assert ops["vf_prep"] == keccak  # the challenge
        assert ops["vf_final"] == keccak * ((64 + k * w1) // 136 + 1)
        hashes = pk // 136 + 1 + (32 + 1024) // 136 + 1 + 5 * k * l  # tr, mu and A: all in vf_main
        assert ops["vf_main"] - hashes * keccak == w.verify_ops(mode, 1024, 0)
