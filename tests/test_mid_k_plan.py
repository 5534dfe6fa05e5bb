"""fs_mid_k_plan, the mid-k kernel's layout (host only)."""
import os
import sys

import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
from ferro_amd import _lib, workloads as W  # noqa: E402


@pytest.mark.parametrize("B,V,k,want", [
    (256, 262144, 2048, (16, 16)),      # more workgroups than fit at once: the largest segments
    (40, 262144, 50, (16, 16)),         # 1280 workgroups of 8192 logits would need a second round
    (24, 100003, 200, (4, 25)), (1, 4096, 65, (4, 1)), (17, 262144, 100, (8, 32)),
    (16, 262144, 100, (8, 32)),         # 64 segments of 4096 logits: more than may wait for each other (below)
    (1, 32 * 65 - 1, 65, None),         # fewer than two lane maxima per candidate
    (256, 262145, 100, None),           # 17 lists of 16384 logits
    (1, 262144, 2049, None),
])
def test_layouts(B, V, k, want):
    assert _lib.mid_k_plan(256, W.make_params(B, temperature=0.8, top_k=k, frequency_penalty=0.1), V) == want


def test_which_rows_fit():
    p = W.make_params(8, temperature=0.8, top_k=70)
    assert _lib.mid_k_plan(256, p, 65536) == (4, 16)
    p["top_k"][3] = 3000                # between the largest k and every token
    assert _lib.mid_k_plan(256, p, 65536) is None
    p["temperature"][3] = 0.0           # greedy: top_k does not matter
    assert _lib.mid_k_plan(256, p, 65536) == (4, 16)
    p["temperature"][3] = 0.8
    p["top_k"][3] = 0                   # every token a candidate: without min-p
    assert _lib.mid_k_plan(256, p, 65536) == (4, 16)
    p["min_p"][3] = 0.05
    assert _lib.mid_k_plan(256, p, 65536) is None


def test_waiting_segments_leave_room():
    """A row's segments wait for each other. Each of four hardware queues can hold one row that is not dispatched whole:
    what waits of those must not fill an XCD (32 CUs of four workgroups)."""
    for V in (4096, 65536, 65537, 131073, 140000, 178740, 200000, 262144):
        for B in (1, 2, 7, 16, 40, 300):
            for k in (1, 65, 0):
                plan = _lib.mid_k_plan(256, W.make_params(B, temperature=0.8, top_k=k, frequency_penalty=0.1), V)
                if plan is not None:
                    assert 4 * (plan[1] - 1) < 4 * 32, (B, V, k, plan)
