"""The kernel for layers whose recurrent weights take the registers and the LDS of the whole device, against per-step
launches, bit for bit."""

from __future__ import annotations

import numpy
import pytest
import torch

from returnn_amd import lib

from _gpu_util import announce, env, get_op, random_problem, run_raw, to_dev
from test_gpu_pitch import POISON, _fwd_multi, _pair_problem

pytestmark = pytest.mark.gpu

# the narrowest and the widest layer of every build, few rows, full and partly filled turns, an odd width
CASES = [
    (7, 16, 4096, "bf16", 0, 1), (6, 1, 4096, "bf16", 0, -1), (5, 37, 3104, "bf16", 1, 1), (6, 32, 3072, "bf16", 0, 1), (5, 17, 2080, "bf16", 0, -2),
    (6, 50, 2399, "bf16", 0, 1), (6, 3, 1056, "f32", 0, 1), (5, 33, 2048, "f32", 0, -1), (5, 16, 2816, "f32", 0, 1), (4, 19, 2080, "f32", 1, 1),
]  # fmt: skip


@pytest.mark.parametrize("T,B,n,dtype,start,step", CASES)
def test_wide_layers_equal_per_step_launches(T, B, n, dtype, start, step):
    announce("wide kernel", T, B, n, dtype, start, step)
    p = random_problem(7000 + n + B, T, B, n)
    i = (numpy.random.default_rng(n).uniform(size=(T, B)) < 0.8).astype(numpy.float32)
    p = (*p[:4], i)
    rc, status, want = run_raw(*p, start, step, dtype=dtype, mode="stepwise")
    assert rc == 0 and status == 0
    rc, status, got = run_raw(*p, start, step, dtype=dtype)
    plan = lib.describe_plan(T, B, n, lib.DTYPE_BF16 if dtype == "bf16" else lib.DTYPE_F32, lib.MODE_AUTO)
    assert "kernel=mfma_regw_wide" in plan, plan
    assert rc == 0 and status == 0
    for name, a, b in zip("YCHd", got, want):
        assert numpy.isfinite(a).all(), name
        assert numpy.array_equal(a, b), "%s differs from per-step launches (%s)" % (name, plan)


def test_wrong_xcd_count_exchanges_at_device_scope():
    announce("wide kernel with a wrong XCD count")
    p = random_problem(71, 6, 5, 2304)
    rc, status, want = run_raw(*p, 0, 1, dtype="bf16", mode="stepwise")
    assert rc == 0 and status == 0
    with env(RTN_LSTM2_XCDS=4):
        rc, status, got = run_raw(*p, 0, 1, dtype="bf16")
    assert rc == 0 and status == 0
    for name, a, b in zip("YCHd", got, want):
        assert numpy.array_equal(a, b), name


def test_bounded_wait_expires_cleanly():
    announce("wide kernel, bounded wait")
    p = random_problem(72, 9, 4, 2304)
    with env(RTN_LSTM2_TIMEOUT_TICKS=0):
        rc, status, got = run_raw(*p, 0, 1, dtype="bf16")
    assert rc == 0 and status in (lib.RTN_OK, lib.RTN_ERR_ABORTED)
    if status == lib.RTN_ERR_ABORTED:
        assert numpy.isnan(got[3]).any() and numpy.isnan(got[0][-1]).any()
    rc, status, got = run_raw(*p, 0, 1, dtype="bf16")
    rc2, status2, want = run_raw(*p, 0, 1, dtype="bf16", mode="stepwise")
    assert (rc, status, rc2, status2) == (0, 0, 0, 0)
    for name, a, b in zip("YCHd", got, want):
        assert numpy.array_equal(a, b), name


@pytest.mark.parametrize("T,B,n,dtype", [(1, 65, 4096, "bf16"), (2, 80, 2080, "bf16"), (3, 300, 1280, "f32"), (2, 49, 2816, "f32")])
def test_few_frames_of_many_rows_run_as_one_launch_per_step(T, B, n, dtype):
    """Turns that load all of W for 16 or 32 rows are only taken where there are frames enough to make up for it; asked for,
    they give the same bits.  A workspace that is enough for a longer call is enough for a shorter one on another plan."""
    announce("wide layers, few frames", T, B, n, dtype)
    p = random_problem(7100 + n, T, B, n)
    dt = lib.DTYPE_BF16 if dtype == "bf16" else lib.DTYPE_F32
    plan = lib.describe_plan(T, B, n, dt, lib.MODE_AUTO)
    assert "mode=graph" in plan and "kernel=mfma_lds" in plan, plan
    assert "kernel=mfma_regw_wide" in lib.describe_plan(200, 16, n, dt, lib.MODE_AUTO)
    assert lib.workspace_bytes(T, B, n, dt, lib.MODE_AUTO) <= lib.workspace_bytes(200, B, n, dt, lib.MODE_AUTO)
    rc, status, got = run_raw(*p, 0, 1, dtype=dtype)
    assert rc == 0 and status == 0
    with env(RTN_LSTM2_KERNEL=3):
        plan = lib.describe_plan(T, B, n, dt, lib.MODE_AUTO)
        rc, status, want = run_raw(*p, 0, 1, dtype=dtype)
    assert "kernel=mfma_regw_wide" in plan and rc == 0 and status == 0
    for name, a, b in zip("YCHd", got, want):
        assert numpy.array_equal(a, b), name
    # ... and recorded into a graph, as launches per step
    op = get_op()
    args = [to_dev(a, dtype) for a in p[:3]] + [to_dev(a, "f32") for a in p[3:]]
    before = lib.capture_report()
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.graph(graph, stream=side):
        recorded = op(*args, 0, 1)
    assert lib.capture_report() == before
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        for name, a, b in zip("YCHd", recorded, want):
            assert numpy.array_equal(a.float().cpu().numpy(), b), name


# every build whose streams go in pieces of rows: a last workgroup of fewer tiles, a last turn of fewer rows, pieces of 8 and 16 bytes
@pytest.mark.parametrize("T,B,n,dtype,gap_x,gap_y", [(4, 17, 4096, "bf16", 0, 0), (5, 9, 2080, "bf16", 8, 8), (4, 33, 2576, "bf16", 0, 16), (4, 1, 1040, "f32", 4, 0), (5, 35, 2032, "f32", 0, 4)])
def test_rows_with_a_pitch(T, B, n, dtype, gap_x, gap_y):
    announce("wide kernel, pitched", T, B, n, dtype, gap_x, gap_y)
    problems = _pair_problem(7200 + n, T, B, n)
    with env(RTN_LSTM2_KERNEL=3):
        assert "kernel=mfma_regw_wide" in lib.describe_plan(T, B, n, lib.DTYPE_BF16 if dtype == "bf16" else lib.DTYPE_F32, lib.MODE_AUTO)
        got, _, Yj = _fwd_multi(problems, (1, -1), dtype, "auto", gap_x=gap_x, gap_y=gap_y, pitched=True)
    want, _, _ = _fwd_multi(problems, (1, -1), dtype, "stepwise", gap_x=0, gap_y=0, pitched=False)
    for k in range(2):
        for name, a, b in zip("YCHd", got[k], want[k]):
            assert bool(torch.isfinite(a).all()) and torch.equal(a, b), (k, name)
    if gap_y:
        assert bool((torch.cat([Yj[:, :, n : n + gap_y], Yj[:, :, 2 * n + gap_y :]], dim=-1) == POISON).all())
