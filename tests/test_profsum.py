"""The kernel names that profiles are summarised by, and the records bench.py
reads, follow the sources."""
import json
import re
from pathlib import Path

import pytest

from neutrongt_amd.profsum import TIMER_NAMES

ROOT = Path(__file__).resolve().parents[1]
CSRC = [f.read_text() for f in sorted((ROOT / "neutrongt_amd" / "csrc").glob("*.hip"))]
TIMERS = {t for text in CSRC for t in re.findall(r'KernelTimer\s+\w+\(\s*"(\w+)"', text)}


@pytest.mark.parametrize("kernel", sorted(TIMER_NAMES))
def test_every_profiled_kernel_exists_with_its_timer(kernel):
    assert any(re.search(r"__global__[^;{]*\bvoid\s+%s\(" % kernel, text) for text in CSRC), kernel
    assert TIMER_NAMES[kernel] in TIMERS


def test_every_timed_attention_kernel_can_be_recorded():
    named = set(TIMER_NAMES.values())
    want = {t for t in TIMERS if re.fullmatch(r"(dense|sparse)_(prep|fwd|bwd_kv|bwd_q)", t)}
    assert want and want <= named
    fx = [k for text in CSRC for k in re.findall(r"void (k_fx_\w+)\(const", text)]
    assert fx and set(fx) <= set(TIMER_NAMES)


def test_traffic_records_name_launched_timers():
    """A record of a kernel that is gone would be printed as another's traffic."""
    for key in json.loads((ROOT / "profiles" / "traffic.json").read_text()):
        assert key.split(":")[1] in TIMERS, key
