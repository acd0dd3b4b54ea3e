"""The host side of signing calls, without a GPU: tests/cxx/host_calls.cpp
stands in for the HIP runtime and checks what the library enqueues and
allocates through its public entry points."""
import os
import subprocess

import pytest

EXE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cxx", "bin", "host_calls")


def _run(what):
    if not os.path.exists(EXE):
        pytest.fail(f"{EXE} not built; run __graft_entry__.build()")
    r = subprocess.run([EXE, what], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr


def test_second_chain_is_joined_after_any_error():
    _run("join")


def test_contexts_allocate_the_slots_asked_for():
    _run("slots")


def test_fixed_stage_ends_on_both_streams():
    _run("timing")
