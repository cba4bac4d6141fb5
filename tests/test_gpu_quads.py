"""Float32 layers whose recurrent product goes in quads of rows, against per-step launches, bit for bit."""

from __future__ import annotations

import numpy
import pytest
import torch

from returnn_amd import lib, torch_native_op

from _gpu_util import announce, random_problem, run_raw, to_dev

pytestmark = pytest.mark.gpu

# (T, B, n, quads): one, two and three quads per group with full and cut last quads, every number of macro steps per wavefront,
# 16 and 32 cells per workgroup, widths that cut the last workgroup or a chunk of 16 bytes, the batch in two launches
CASES = [
    (6, 1, 512, 1), (9, 30, 500, 1), (6, 90, 512, 3), (7, 64, 512, 1), (5, 125, 505, 2), (4, 190, 448, 3),
    (8, 5, 256, 1), (6, 70, 200, 2), (6, 130, 256, 3), (7, 62, 270, 1), (4, 199, 301, 2), (6, 88, 128, 1), (6, 81, 99, 1),
]  # fmt: skip


@pytest.mark.parametrize("start,step", [(0, 1), (1, -1)])
@pytest.mark.parametrize("T,B,n,quads", CASES)
def test_quads_equal_per_step_launches(T, B, n, quads, start, step):
    announce("quads of rows", T, B, n, start, step)
    p = random_problem(7800 + n + B, T, B, n)
    p = (*p[:4], (numpy.random.default_rng(n).uniform(size=(T, B)) < 0.8).astype(numpy.float32))
    rc, status, want = run_raw(*p, start, step, dtype="f32", mode="stepwise")
    assert rc == 0 and status == 0
    rc, status, got = run_raw(*p, start, step, dtype="f32")
    plan = lib.describe_plan(T, B, n, lib.DTYPE_F32, lib.MODE_AUTO)
    assert " row_quads=%d" % quads in plan, plan
    assert rc == 0 and status == 0
    for name, a, b in zip("YCHd", got, want):
        assert numpy.isfinite(a).all(), name
        assert numpy.array_equal(a, b), "%s differs from per-step launches (%s)" % (name, plan)


def test_two_directions_in_one_launch():
    announce("quads of rows, two calls")
    calls = []
    for k in range(2):
        X, W, y0, c0, i = random_problem(7900 + k, 7, 18, 500)
        calls.append((*(to_dev(a, "f32") for a in (X, W, y0, c0, i)), 0, 1 if k else -1))
    outs = torch_native_op.native_lstm2_multi(calls)
    for c, o in zip(calls, outs):
        for a, b in zip(o, torch_native_op.native_lstm2_multi([c], mode="stepwise")[0]):
            assert torch.equal(a, b)
