"""The kernel for layers whose recurrent weights fit one compute unit, against per-step launches, bit for bit (widths below 32,
whose per-step launches are element-wise kernels with another order of additions, against the oracle)."""

from __future__ import annotations

import numpy
import pytest
import torch

from oracle import lstm2_oracle as oracle
from returnn_amd import lib, torch_native_op

from _gpu_util import announce, random_problem, run_raw, to_dev

pytestmark = pytest.mark.gpu

# every build, full and cut widths, batches of one, of less than a workgroup's rows, of a remainder; fewer frames than are
# fetched ahead
CASES = [
    (9, 1, 32, "f32"), (3, 4, 64, "f32"), (1, 5, 40, "f32"), (12, 17, 63, "f32"), (7, 3, 33, "f32"), (6, 66, 64, "f32"),
    (9, 1, 32, "bf16"), (2, 4, 64, "bf16"), (6, 6, 33, "bf16"), (13, 9, 96, "bf16"), (4, 18, 127, "bf16"), (8, 5, 128, "bf16"), (5, 7, 90, "bf16"),
]  # fmt: skip


@pytest.mark.parametrize("start,step", [(0, 1), (0, -1), (1, 2)])
@pytest.mark.parametrize("T,B,n,dtype", CASES)
def test_small_layers_equal_per_step_launches(T, B, n, dtype, start, step):
    if start >= T:
        start = 0
    announce("solo kernel", T, B, n, dtype, start, step)
    p = random_problem(7500 + n + B, T, B, n)
    p = (*p[:4], (numpy.random.default_rng(n).uniform(size=(T, B)) < 0.8).astype(numpy.float32))
    rc, status, want = run_raw(*p, start, step, dtype=dtype, mode="stepwise")
    assert rc == 0 and status == 0
    rc, status, got = run_raw(*p, start, step, dtype=dtype)
    plan = lib.describe_plan(T, B, n, lib.DTYPE_BF16 if dtype == "bf16" else lib.DTYPE_F32, lib.MODE_AUTO)
    assert "kernel=mfma_regw_solo" in plan, plan
    assert rc == 0 and status == 0
    for name, a, b in zip("YCHd", got, want):
        assert numpy.isfinite(a).all(), name
        assert numpy.array_equal(a, b), "%s differs from per-step launches (%s)" % (name, plan)


@pytest.mark.parametrize("n", [1, 3, 7, 20, 31])
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_tiny_layers_against_the_oracle(n, dtype):
    announce("solo kernel, tiny", n, dtype)
    p = random_problem(7600 + n, 6, 5, n)
    want = oracle.native_lstm2_fwd(*p, 0, -1)
    rc, status, got = run_raw(*p, 0, -1, dtype=dtype)
    assert rc == 0 and status == 0
    for name, a, b in zip("YCHd", got, want):
        assert numpy.abs(a - b).max() <= (2e-2 if dtype == "bf16" else 2e-6), name


def test_several_calls_and_final_outputs():
    announce("solo kernel, five calls")
    T, B, n = 7, 5, 96
    calls = []
    for k in range(5):
        X, W, y0, c0, i = random_problem(7700 + k, T, B, n)
        calls.append((*(to_dev(a, "bf16") for a in (X, W, y0)), to_dev(c0, "f32"), to_dev(i, "f32"), 0, 1 if k % 2 else -1))
    outs = torch_native_op.native_lstm2_multi(calls)
    for c, o in zip(calls, outs):
        single = torch_native_op.native_lstm2_multi([c], mode="stepwise")[0]
        for a, b in zip(o, single):
            assert torch.equal(a, b)


# one row per workgroup: every build, widths with copied cells (whole quads of them, a wavefront of them, cut quads); and the number of
# rows up to which a workgroup has one, which depends on the build's wavefronts, from both sides
@pytest.mark.parametrize("T,B,n,dtype,groups", [
    (5, 3, 32, "f32", 3), (4, 2, 65, "f32", 2), (6, 5, 96, "f32", 5), (3, 130, 97, "f32", 130), (9, 129, 128, "f32", 129), (5, 2, 34, "bf16", 2), (5, 3, 68, "bf16", 3), (3, 2, 1, "f32", 2),
    (2, 1024, 32, "f32", 1024), (2, 512, 64, "f32", 512), (2, 513, 64, "f32", 129), (2, 256, 128, "f32", 256), (2, 512, 40, "bf16", 512), (2, 520, 40, "bf16", 130),
    (2, 256, 96, "bf16", 256), (2, 257, 96, "bf16", 65),
])  # fmt: skip
def test_a_row_per_workgroup(T, B, n, dtype, groups):
    announce("solo kernel, rows", T, B, n, dtype)
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the limits are those of 256 CUs")
    plan = lib.describe_plan(T, B, n, lib.DTYPE_BF16 if dtype == "bf16" else lib.DTYPE_F32, lib.MODE_AUTO)
    assert "kernel=mfma_regw_solo" in plan and " groups=%i " % groups in plan, plan
    p = random_problem(7800 + n + B, T, B, n)
    p = (*p[:4], (numpy.random.default_rng(n).uniform(size=(T, B)) < 0.8).astype(numpy.float32))
    for step in (1, -1):
        rc, status, got = run_raw(*p, 0, step, dtype=dtype)
        assert rc == 0 and status == 0
        if n < 32:
            want, bars = oracle.native_lstm2_fwd(*p, 0, step), 2e-6
        else:
            rc, status, want = run_raw(*p, 0, step, dtype=dtype, mode="stepwise")
            assert rc == 0 and status == 0
            bars = 0.0
        for name, a, b in zip("YCHd", got, want):
            assert numpy.isfinite(a).all(), name
            assert numpy.abs(a - b).max() <= bars, (name, plan)


@pytest.mark.parametrize("n,dtype", [(70, "f32"), (34, "bf16"), (128, "bf16")])
def test_values_that_are_not_finite_stay_in_their_row(n, dtype):
    announce("solo kernel, not finite", n, dtype)
    T, B = 6, 3
    X, W, y0, c0, i = random_problem(7900 + n, T, B, n)
    i[:] = 1.0
    rc, status, clean = run_raw(X, W, y0, c0, i, 0, 1, dtype=dtype)
    assert rc == 0 and status == 0
    for value in (numpy.inf, numpy.nan):
        X[2, 1, n - 1] = value
        rc, status, got = run_raw(X, W, y0, c0, i, 0, 1, dtype=dtype)
        assert rc == 0 and status == 0
        for name, a, b in zip("YCH", got, clean):
            assert numpy.array_equal(a[:, [0, 2]], b[:, [0, 2]]) and numpy.array_equal(a[:2], b[:2]), name
        rc, status, want = run_raw(X, W, y0, c0, i, 0, 1, dtype=dtype, mode="stepwise")
        for name, a, b in zip("YCHd", got, want):
            assert numpy.array_equal(a, b, equal_nan=True), name
