"""A rule of the kernel sources that no run can show (LDS operations of one
wave happen to execute in order): the table of twiddle factors is filled by all
lanes and read by all lanes, so a fence or barrier stands between."""
import pathlib
import re

import pytest

CSRC = pathlib.Path(__file__).resolve().parents[1] / "cudilithium_amd" / "csrc"


def _loads():
    for path in sorted(CSRC.glob("*.h*")):
        text = path.read_text()
        for m in re.finditer(r"^ +zeta_lds_load\(([\w.]+)\);", text, re.M):
            yield pytest.param(text[m.end():], m.group(1), id=f"{path.name}:{text.count(chr(10), 0, m.start()) + 1}")


@pytest.mark.parametrize("after,table", _loads())
def test_fence_between_filling_and_reading_the_twiddles(after, table):
    use = re.search(rf"\b{re.escape(table)}\b", after)
    assert use and re.search(r"wave_lds_sync\(\);|__syncthreads\(\);", after[:use.start()])
