"""Large batches, whose rows two persistent launches would take in turn, in one launch of interleaved groups: against per-step
launches, bit for bit."""

from __future__ import annotations

import numpy
import pytest

from returnn_amd import lib

from _gpu_util import announce, env, random_problem, run_raw

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
