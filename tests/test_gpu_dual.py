"""Large batches, whose rows two persistent launches would take in turn, in one launch of interleaved groups: against per-step
launches, bit for bit."""

from __future__ import annotations

import re

import numpy
import pytest
import torch

from returnn_amd import lib

from _gpu_util import announce, env, get_op, random_problem, run_raw, to_dev

pytestmark = pytest.mark.gpu

# two and three turns, full and cut groups, a last group without rows, cut widths, one to a few steps
CASES = [(6, 256, 1024, 0, 1), (1, 255, 1024, 0, 1), (2, 130, 1024, 0, -1), (9, 300, 1000, 1, -1), (5, 230, 608, 0, 2), (7, 170, 776, 0, 1)]


@pytest.mark.parametrize("T,B,n,start,step", CASES)
def test_interleaved_turns_equal_per_step_launches(T, B, n, start, step):
    announce("dual kernel", T, B, n, start, step)
    p = random_problem(8000 + n + B, T, B, n)
    p = (*p[:4], (numpy.random.default_rng(n).uniform(size=(T, B)) < 0.8).astype(numpy.float32))
    rc, status, want = run_raw(*p, start, step, dtype="bf16", mode="stepwise")
    assert rc == 0 and status == 0
    plan = lib.describe_plan(T, B, n, lib.DTYPE_BF16, lib.MODE_AUTO)
    assert " interleaved=2" in plan and "launches=1 " not in plan, plan
    for xcds in (None, 4):  # (4: the groups are found on two XCDs each and exchange at device scope)
        with env(RTN_LSTM2_XCDS=xcds):
            rc, status, got = run_raw(*p, start, step, dtype="bf16")
        assert rc == 0 and status == 0
        for name, a, b in zip("YCHd", got, want):
            assert numpy.isfinite(a).all(), name
            assert numpy.array_equal(a, b), "%s differs from per-step launches (%s)" % (name, plan)


def test_turns_one_by_one_where_two_do_not_fit():
    """The plan's two turns in one launch need another kernel than the turns: where the device does not hold that one, the call
    runs as two launches, with the same results (counted as recorded under stream capture)."""
    announce("dual kernel that does not fit")
    X, W, y0, c0, i = random_problem(8100, 5, 200, 1024)
    args = [to_dev(a, "bf16") for a in (X, W, y0)] + [to_dev(a, "f32") for a in (c0, i)]
    op = get_op()
    launches = []
    for per_cu in (None, 0):
        with env(RTN_LSTM2_DUAL_PER_CU=per_cu):
            want = op(*args, 0, 1)
            torch.cuda.synchronize()
            before = sum(int(v) for v in re.findall(r"\d+(?= as)", lib.capture_report()))
            graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.graph(graph, stream=side):
                got = op(*args, 0, 1)
            launches.append(sum(int(v) for v in re.findall(r"\d+(?= as)", lib.capture_report())) - before)
        for _ in range(3):
            graph.replay()
            torch.cuda.synchronize()
            for name, a, b in zip("YCHd", got, want):
                assert torch.equal(a, b), name
    assert launches == [1, 2], launches


# layers that no XCD holds: groups over all XCDs with four tiles of cells, alone, two turns in one launch, an odd number of turns, a last group of
# few rows, rows that do not fill a group, a width that cuts a chunk (turns one by one), one to a few steps
SPREAD = [(5, 20, 1300, 0, 1, 1), (4, 32, 2048, 0, -1, 1), (6, 64, 2048, 0, 1, 2), (1, 33, 2048, 0, 1, 2), (2, 90, 1280, 0, -1, 2), (7, 128, 1096, 1, 2, 3), (5, 50, 1604, 0, -1, 2),
          (9, 55, 1056, 0, 1, 2)]  # fmt: skip


@pytest.mark.parametrize("T,B,n,start,step,launches", SPREAD)
def test_groups_over_all_xcds_equal_per_step_launches(T, B, n, start, step, launches):
    announce("four tiles and dual kernel over all XCDs", T, B, n, start, step)
    p = random_problem(8200 + n + B, T, B, n)
    p = (*p[:4], (numpy.random.default_rng(n).uniform(size=(T, B)) < 0.8).astype(numpy.float32))
    plan = lib.describe_plan(T, B, n, lib.DTYPE_BF16, lib.MODE_AUTO)
    assert "kernel=mfma_regw mt=4 nt=1" in plan and " launches=%i " % launches in plan and (launches == 1 or " interleaved=2" in plan), plan
    rc, status, want = run_raw(*p, start, step, dtype="bf16", mode="stepwise")
    assert rc == 0 and status == 0
    for no_dual in (None, 1):
        with env(RTN_LSTM2_NO_DUAL=no_dual):
            rc, status, got = run_raw(*p, start, step, dtype="bf16")
        assert rc == 0 and status == 0
        for name, a, b in zip("YCHd", got, want):
            assert numpy.isfinite(a).all(), name
            assert numpy.array_equal(a, b), "%s differs from per-step launches (%s)" % (name, plan)


def test_interleaved_turns_over_all_xcds_drain_after_an_expired_wait():
    """A wait bound of zero ticks, as an environment sets it: the launch ends, what it handed out is marked if a wait expired, and the next call is sound."""
    announce("dual kernel over all XCDs, bounded wait")
    T, B, n = 12, 64, 1280
    p = random_problem(8300, T, B, n)
    with env(RTN_LSTM2_TIMEOUT_TICKS=0):
        rc, status, got = run_raw(*p, 0, 1, dtype="bf16")
    assert rc == 0 and status in (lib.RTN_OK, lib.RTN_ERR_ABORTED)
    if status == lib.RTN_ERR_ABORTED:
        assert numpy.isnan(got[3]).any() and numpy.isnan(got[0][-1]).any()
    rc, status, got = run_raw(*p, 0, 1, dtype="bf16")
    rc2, status2, want = run_raw(*p, 0, 1, dtype="bf16", mode="stepwise")
    assert rc == rc2 == 0 and status == status2 == 0
    for name, a, b in zip("YCHd", got, want):
        assert numpy.array_equal(a, b), name
