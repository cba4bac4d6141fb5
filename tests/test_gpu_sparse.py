"""
Groups of up to 8 rows of a bfloat16 layer, whose product goes in sparse matrix instructions: against per-step launches (dense
matrix instructions, pinned against the oracle by the parity tests), bit for bit.
"""

from __future__ import annotations

import numpy
import pytest

from returnn_amd import lib
from _gpu_util import announce, random_problem, run_multi_raw, run_raw
from test_gpu_bwd import _rel_to_max, _run

pytestmark = pytest.mark.gpu

# T: the streams move in turns of four frames; n: 2, 4 and 8 tiles of cells per workgroup, shares of W with and without a second half
# and pairs that not every wavefront has, widths that cut a chunk of 16 bytes; rows: one, a full group, a last group with fewer
CASES = [
    (1, 1, 1024, 0, 1), (2, 8, 1024, 0, -1), (3, 64, 1024, 0, 1), (4, 5, 992, 0, 1), (5, 32, 1000, 0, -1), (6, 17, 768, 1, 1), (7, 3, 800, 0, 1),
    (8, 7, 512, 0, 1), (9, 60, 512, 0, -1), (10, 2, 416, 0, 1), (11, 12, 300, 1, -1), (12, 1, 256, 0, 1), (13, 90, 256, 0, 1),
    (14, 8, 288, 0, 1), (23, 4, 160, 2, 3), (22, 6, 171, 0, 1),
]  # fmt: skip


@pytest.mark.parametrize("T,B,n,start,step", CASES)
def test_sparse_products_equal_per_step_launches(T, B, n, start, step):
    announce("sparse products", T, B, n, start, step)
    p = random_problem(5300 + n + B, T, B, n)
    p = (*p[:4], (numpy.random.default_rng(n).uniform(size=(T, B)) < 0.8).astype(numpy.float32))
    plan = lib.describe_plan(T, B, n, lib.DTYPE_BF16, lib.MODE_AUTO)
    assert " product=sparse" in plan, plan
    rc, status, want = run_raw(*p, start, step, dtype="bf16", mode="stepwise")
    assert rc == 0 and status == 0
    rc, status, got = run_raw(*p, start, step, dtype="bf16")
    assert rc == 0 and status == 0, "status %i" % status
    for name, a, b in zip("YCHd", got, want):
        assert numpy.array_equal(a, b), "%s differs from per-step launches (%s)" % (name, plan)


def test_large_infinite_and_nan_states_stay_in_their_row():
    """An initial output far from a hidden state's range, an infinity and a NaN (their bits are not the "not yet written" ones): as with per-step launches."""
    T, B, n = 6, 8, 1024
    announce("sparse products, unusual states", T, B, n)
    p = list(random_problem(97, T, B, n, ragged=False))
    p[2][1, 5], p[2][3, 700], p[2][6, 31] = 3e38, numpy.inf, numpy.nan
    plan, got, words = run_multi_raw([(*p, 0, 1), (*p, 0, -1)], dtype="bf16")
    assert " product=sparse" in plan and all(w[:2] == (0, 0) for w in words), (plan, words)
    for outs, step in zip(got, (1, -1)):
        rc, status, want = run_raw(*p, 0, step, dtype="bf16", mode="stepwise")
        assert rc == 0 and status == 0
        for name, a, b in zip("YCHd", outs, want):
            assert numpy.array_equal(a, b, equal_nan=True), name
        assert numpy.isfinite(outs[0][:, [0, 2, 4, 5, 7]]).all()


# (the frames' inputs come four at a time where a wavefront's share of W is small; the first frame stands in front of the loop)
@pytest.mark.parametrize("dtype,B,n", [("bf16", 9, 256), ("bf16", 17, 512), ("bf16", 6, 96), ("f32", 7, 128)])
@pytest.mark.parametrize("T", [1, 2, 3, 4, 5, 6, 7, 9, 10])
def test_gradients_of_any_number_of_frames(T, dtype, B, n):
    announce("gradient, inputs in turns", T, B, n, dtype)
    for start, step in [(0, 1), (0, -2)]:
        got, want, _ = _run(T, B, n, dtype, start, step, seed=T + n)
        assert "name=k_lstm2_bwd_local " in lib.bwd_plan_text()
        for name, a, b in zip(("DX", "DW", "Dy0", "Dc0"), got, want):
            assert _rel_to_max(a, b) <= (2e-2 if dtype == "bf16" else 2e-5), (name, _rel_to_max(a, b))
