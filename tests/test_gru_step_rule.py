"""Which kernel a GRU step takes, over hidden sizes, batches and alignments."""

from __future__ import annotations

import pytest


@pytest.mark.parametrize("H,B,want", [(16, 1, "fused"), (512, 400, "fused"), (8192, 1, "fused"), (8208, 1, None),
                                      (1, 1, "ragged"), (250, 128, "ragged"), (250, 161, None),  # 640 workgroups
                                      (515, 72, "ragged"), (515, 80, None),     # 585 and 650 workgroups
                                      (777, 40, "ragged"), (777, 41, None),     # 36 and 43 MB of W_hh read
                                      (1001, 24, "ragged"), (1001, 25, None),   # 36 and 48 MB
                                      (1300, 8, "ragged"), (1300, 9, None),     # one row of workgroups, two
                                      (5001, 8, "ragged"), (5127, 8, None), (8193, 1, None)])
def test_step_kernel(H, B, want):
    from ttrl_amd.engine.recurrent import _step_kernel

    assert _step_kernel(H, B, True, False) == want
    # a cell that keeps its two launches keeps them off the fused layout alone
    assert _step_kernel(H, B, True, True) == ("fused" if want == "fused" else None)


def test_unaligned_operands_are_ragged():
    from ttrl_amd.engine.recurrent import _step_kernel

    assert _step_kernel(512, 16, False, False) == "ragged"
    assert _step_kernel(512, 16, False, True) is None
