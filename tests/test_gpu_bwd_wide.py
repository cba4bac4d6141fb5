"""The gradient kernel for layers whose recurrent weights take the registers and the LDS of the CUs of a batch group."""

from __future__ import annotations

import numpy
import pytest
import torch

from returnn_amd import lib

from _gpu_util import announce, env
from test_gpu_bwd import _rel_to_max, _run

pytestmark = pytest.mark.gpu


# the narrowest and the widest layer, a width of the padded problem, a last group of fewer rows, a second launch with one group, one frame, more
# frames than the rings have slots, frames that are not visited
@pytest.mark.parametrize(
    "T,B,n,start,step", [(6, 64, 2048, 0, 1), (9, 33, 1088, 1, -1), (1, 48, 1280, 0, 1), (7, 70, 1152, 0, 2), (3, 40, 1080, 0, -1), (11, 64, 1984, 2, 1)]
)
def test_gradient_of_wide_layers(T, B, n, start, step):
    announce("wide gradient", T, B, n, start, step)
    with env(RTN_LSTM2_BWD_WIDE=2):  # (also where the groups of one tile per workgroup take no more launches)
        got, want, _ = _run(T, B, n, "bf16", start, step, seed=T + n)
        plan = lib.bwd_plan_text()
    assert "name=k_lstm2_bwd_wide" in plan, plan
    for name, a, b in zip(("DX", "DW", "Dy0", "Dc0"), got, want):
        assert numpy.isfinite(a).all(), name
        assert _rel_to_max(a, b) <= 2e-2, (name, _rel_to_max(a, b))  # (the bound of the other bf16 gradient tests)


def test_wrong_xcd_count_exchanges_at_device_scope():
    announce("wide gradient with a wrong XCD count")
    with env(RTN_LSTM2_XCDS=4, RTN_LSTM2_BWD_WIDE=2):
        got, want, _ = _run(6, 40, 1152, "bf16", 0, 1, seed=3)
        plan = lib.bwd_plan_text()
    assert "name=k_lstm2_bwd_wide" in plan, plan
    for name, a, b in zip(("DX", "DW", "Dy0", "Dc0"), got, want):
        assert _rel_to_max(a, b) <= 2e-2, (name, _rel_to_max(a, b))


def test_repeated_calls_agree():
    announce("wide gradient, repeated")
    first, _, _ = _run(12, 64, 2048, "bf16", 0, 1, seed=5)
    for _ in range(3):
        again, _, _ = _run(12, 64, 2048, "bf16", 0, 1, seed=5)
        for name, a, b in zip(("DX", "Dy0", "Dc0"), first, again):
            assert numpy.array_equal(a, b), name
    torch.cuda.synchronize()
