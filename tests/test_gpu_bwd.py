"""
GPU parity of the NativeLstm2 gradient op (C ABI ``rtn_native_lstm2_bwd``) against the CPU oracle of the reference's
gradient code, on the forward results of the HIP path itself.

Tolerances.  The tolerances asked of the op are those of the forward outputs only; gradients are sums over up to T*B terms
whose summation order differs between MFMA tiles and a sequential loop, so they are judged relative to the largest
magnitude of each array: float32 within 2e-5 of it (the float32 oracle itself is that far from the float64 oracle),
bfloat16 (bf16 activations, gates and DX; float32 accumulation) within 2e-2 of it.
"""

from __future__ import annotations

import numpy
import pytest
import torch

from oracle import lstm2_oracle as oracle
from returnn_amd import lib, synthetic, torch_native_op
from _gpu_util import announce, get_op, random_problem, to_dev

pytestmark = pytest.mark.gpu


def _rel_to_max(got, want):
    scale = max(float(numpy.abs(want).max()), 1e-30)
    return float(numpy.abs(got - want).max()) / scale


def _run(T, B, n, dtype, start, step, seed=0, scale_x=0.5):
    X, W, y0, c0, i = random_problem(seed, T, B, n, scale_x=scale_x)
    rng = numpy.random.default_rng(seed + 1000)
    DY = rng.normal(0, 1.0, (T, B, n)).astype(numpy.float32)
    Dd = rng.normal(0, 1.0, (B, n)).astype(numpy.float32)
    op = get_op()
    Xd, Wd, y0d, DYd = (to_dev(a, dtype) for a in (X, W, y0, DY))
    c0d, id_, Ddd = (to_dev(a, "f32") for a in (c0, i, Dd))
    Y, C, H, d = op(Xd, Wd, y0d, c0d, id_, start, step)
    got = torch_native_op.native_lstm2_grad(Wd, y0d, c0d, id_, start, step, Y, C, H, DYd, Ddd)
    torch.cuda.synchronize()
    got = [g.float().cpu().numpy() for g in got]
    # the checker gets what the GPU's gradient op got: the GPU's own forward results and the same (rounded) inputs
    f = lambda t: t.float().cpu().numpy().astype(numpy.float64)  # noqa: E731
    want = oracle.native_lstm2_bwd(f(Xd), f(Wd), f(y0d), c0, i, start, step, f(Y), f(C), f(H), f(DYd), Dd, dtype=numpy.float64)
    return got, want, (X, W, y0, c0, i, DY, Dd)


@pytest.mark.parametrize("start,step", [(0, 1), (0, -1), (1, 2), (2, -3)])
@pytest.mark.parametrize("T,B,n", [(7, 3, 16), (12, 20, 64), (9, 40, 128), (6, 5, 20), (5, 2, 3), (5, 9, 48), (4, 12, 400), (3, 9, 1024), (4, 20, 720)])
def test_bwd_f32(T, B, n, start, step):
    announce("bwd f32", T, B, n, start, step)
    got, want, _ = _run(T, B, n, "f32", start, step, seed=T + n)
    for name, a, b in zip(("DX", "DW", "Dy0", "Dc0"), got, want):
        assert a.shape == b.shape
        assert _rel_to_max(a, b) <= 2e-5, (name, _rel_to_max(a, b))


@pytest.mark.parametrize("step", [1, -1])
@pytest.mark.parametrize("T,B,n", [(10, 16, 64), (16, 32, 256), (6, 5, 24), (6, 20, 768), (5, 33, 800), (5, 7, 48), (4, 24, 1280)])
def test_bwd_bf16(T, B, n, step):
    announce("bwd bf16", T, B, n, step)
    got, want, _ = _run(T, B, n, "bf16", 0, step, seed=T + n)
    for name, a, b in zip(("DX", "DW", "Dy0", "Dc0"), got, want):
        assert _rel_to_max(a, b) <= 2e-2, (name, _rel_to_max(a, b))


# (rows per group, tiles per workgroup, wavefronts per workgroup): decompositions of the persistent gradient kernel that the
# plan picks for other shapes than the ones above -- one (row, k) pair per thread with 2 and 4 tiles, whole and half ring
# frames, 8 wavefronts -- forced here on a small problem with ragged sequence lengths and a last group of fewer rows.
@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("rows,tiles,waves", [(8, 2, 4), (8, 4, 4), (4, 2, 4), (3, 4, 4), (16, 2, 4), (12, 1, 4), (8, 1, 8), (8, 2, 8), (8, 4, 8)])
def test_bwd_forced_decompositions(rows, tiles, waves, dtype):
    from _gpu_util import env

    T, B, n = 9, 21, 256
    announce("bwd forced decomposition", rows, tiles, waves, dtype)
    with env(RTN_LSTM2_BWD_KERNEL=2, RTN_LSTM2_BWD_ROWS=rows, RTN_LSTM2_BWD_MT=tiles, RTN_LSTM2_BWD_WAVES=waves):
        got, want, _ = _run(T, B, n, dtype, 1, 2 if tiles == 2 else -1, seed=rows + 10 * tiles + waves)
        plan = lib.bwd_plan_text()
    if "bwd_regw" not in plan:
        pytest.skip("no persistent kernel for this decomposition: " + plan)
    assert "rows_per_group=%i" % rows in plan and "tiles=%i" % tiles in plan and "waves=%i" % waves in plan, plan
    bar = 2e-2 if dtype == "bf16" else 2e-5
    for name, a, b in zip(("DX", "DW", "Dy0", "Dc0"), got, want):
        assert numpy.isfinite(a).all(), name
        assert _rel_to_max(a, b) <= bar, (name, _rel_to_max(a, b), plan)


def test_bwd_ring_that_does_not_fit_its_section_is_refused():
    """Groups of one row, which only the environment asks for, have frames of eight: the ring would reach into the section behind its own."""
    from _gpu_util import env

    announce("bwd ring beyond its section")
    with env(RTN_LSTM2_BWD_KERNEL=2, RTN_LSTM2_BWD_ROWS=1):
        with pytest.raises(RuntimeError, match="exchange ring"):
            _run(200, 21, 64, "f32", 0, 1)


def test_bwd_ring_is_held_against_its_own_section_alone():
    """The same at a width whose workspace has the rings of another kernel behind the exchange ring."""
    from _gpu_util import env

    announce("bwd ring beyond its section, wide layer")
    with env(RTN_LSTM2_BWD_KERNEL=2, RTN_LSTM2_BWD_ROWS=1):
        with pytest.raises(RuntimeError, match="exchange ring"):
            _run(4, 24, 1280, "bf16", 0, 1)


# float32 groups of up to 8 rows on one XCD each: one and two quads of rows with 1, 2 and 4 tiles, cut quads and groups, every
# number of macro steps per wavefront, odd widths
@pytest.mark.parametrize("B,n,tiles,quads", [(1, 512, 1, 1), (30, 500, 1, 1), (61, 512, 2, 1), (37, 512, 1, 2), (128, 512, 2, 2), (97, 301, 2, 2), (60, 256, 1, 1), (205, 224, 2, 2),
                                             (300, 256, 4, 2), (17, 128, 1, 1), (9, 64, 1, 1), (6, 33, 1, 1)])
def test_bwd_quads_of_rows(B, n, tiles, quads):
    announce("bwd quads of rows", B, n, tiles, quads)
    for start, step in [(0, 1), (1, -2)]:
        got, want, _ = _run(6, B, n, "f32", start, step, seed=B + n)
        plan = lib.bwd_plan_text()
        assert "bwd_regw_xcd" in plan and "tiles=%i " % tiles in plan and "row_quads=%i" % quads in plan and "name=k_lstm2_bwd_local " in plan, plan
        for name, a, b in zip(("DX", "DW", "Dy0", "Dc0"), got, want):
            assert numpy.isfinite(a).all(), name
            assert _rel_to_max(a, b) <= 2e-5, (name, _rel_to_max(a, b), plan)


# The kernel for groups of up to 8 rows on one XCD each: one, two and four tiles, shares of one, of an odd and of a full number of
# macro steps per wavefront, cut groups, and runs of one and two frames (the first is in front of the kernel's loop).
@pytest.mark.parametrize("dtype,B,n", [("bf16", 3, 16), ("bf16", 9, 80), ("bf16", 21, 208), ("bf16", 17, 512), ("bf16", 30, 1024), ("bf16", 130, 256), ("bf16", 250, 256),
                                       ("f32", 2, 16), ("f32", 5, 144), ("f32", 13, 512), ("f32", 61, 512), ("f32", 250, 256)])
def test_bwd_groups_of_one_xcd(dtype, B, n):
    """Against the oracle and against the plan that spreads a group over the XCDs (another kernel: equal to rounding, 1e-5 of the
    largest magnitude in float32, one bfloat16 step of it in bfloat16).  Rows are independent: errors that are not finite stay in
    their row, and every other row keeps its bits."""
    from _gpu_util import env

    announce("bwd groups of one xcd", dtype, B, n)
    bar, step_bar = (2e-2, 2.0**-7) if dtype == "bf16" else (2e-5, 1e-5)
    for T, start, step in [(1, 0, 1), (2, 0, -1), (7, 1, 2)]:
        got, want, _ = _run(T, B, n, dtype, start, step, seed=T + B + n)
        plan = lib.bwd_plan_text()
        assert "bwd_regw_xcd" in plan and "name=k_lstm2_bwd_local " in plan, plan
        with env(RTN_LSTM2_BWD_LOCAL=0):
            spread, _, _ = _run(T, B, n, dtype, start, step, seed=T + B + n)
            assert "bwd_regw_xcd" not in lib.bwd_plan_text() and "name=k_lstm2_bwd_regw " in lib.bwd_plan_text(), lib.bwd_plan_text()
        for name, a, b, c in zip(("DX", "DW", "Dy0", "Dc0"), got, want, spread):
            assert _rel_to_max(a, b) <= bar, (T, name, _rel_to_max(a, b), plan)
            assert _rel_to_max(a, c) <= step_bar, (T, name, _rel_to_max(a, c), plan)
    X, W, y0, c0, i = random_problem(n, 5, B, n)
    i[:] = 1.0
    Xd, Wd, y0d = (to_dev(a, dtype) for a in (X, W, y0))
    c0d, id_ = to_dev(c0, "f32"), to_dev(i, "f32")
    Y, C, H, _ = get_op()(Xd, Wd, y0d, c0d, id_, 0, 1)
    DY, Dd = torch.ones_like(Y), torch.ones_like(c0d)
    clean = torch_native_op.native_lstm2_grad(Wd, y0d, c0d, id_, 0, 1, Y, C, H, DY, Dd)
    row = B // 2
    for value in (float("inf"), float("nan")):
        DY[3, row, n // 2] = value
        hit = torch_native_op.native_lstm2_grad(Wd, y0d, c0d, id_, 0, 1, Y, C, H, DY, Dd)
        others = [b for b in range(B) if b != row]
        assert torch.equal(hit[0][:, others], clean[0][:, others]) and torch.equal(hit[2][others], clean[2][others]) and torch.equal(hit[3][others], clean[3][others])
        assert not torch.isfinite(hit[0][:4, row].float()).all(-1).any()
        assert torch.equal(hit[0][4, row], clean[0][4, row])


# Groups of up to 8 rows on one XCD each: their own kernel, the general one where fewer of the launch's groups fit the device with that, groups
# over all XCDs, launches per frame; and what the weight gradient came from.
@pytest.mark.parametrize("dtype,B,n,kernel,plan,weights", [
    ("bf16", 30, 512, 0, "bwd_regw_xcd k_lstm2_bwd_local", "rocblas,k_weight_last"), ("bf16", 200, 512, 0, "bwd_regw_xcd k_lstm2_bwd_regw", "rocblas"),
    ("bf16", 5, 2048, 0, "bwd_regw k_lstm2_bwd_regw", "rocblas,k_weight_last"), ("f32", 9, 64, 0, "bwd_regw_xcd k_lstm2_bwd_local", "k_weight_grad"),
    ("f32", 9, 64, 1, "bwd_step k_bwd_step", "k_weight_grad"), ("bf16", 4, 24, 0, "bwd_generic k_bwd_pointwise", "k_weight_grad"), ("f32", 70, 30, 0, "bwd_generic k_bwd_pointwise", "rocblas")])  # fmt: skip
def test_bwd_plan_names_its_kernels(dtype, B, n, kernel, plan, weights):
    from _gpu_util import env

    announce("bwd plan names", dtype, B, n, kernel)
    with env(RTN_LSTM2_BWD_KERNEL=kernel):
        got, want, _ = _run(3, B, n, dtype, 0, 1, seed=n)
        fields = dict(word.split("=", 1) for word in lib.bwd_plan_text().split())
    assert (fields["kernel"] + " " + fields["name"], fields["weight_gradient"]) == (plan, weights), lib.bwd_plan_text()
    for name, a, b in zip(("DX", "DW", "Dy0", "Dc0"), got, want):
        assert _rel_to_max(a, b) <= (2e-2 if dtype == "bf16" else 2e-5), name


def test_bwd_read_delay_only_moves_time():
    """The delay between a frame's stores and the read of its ring slot (and whether it adapts) decides how often a read is
    repeated, never what is read: every setting gives the same bits, on a plan with one pair per thread and on one without."""
    from _gpu_util import env

    announce("bwd read delay")
    for tiles in (2, 1):
        results = []
        for delay, inc in [(None, None), (0, 0), (64, 0), (3, 2)]:
            with env(RTN_LSTM2_BWD_KERNEL=2, RTN_LSTM2_BWD_ROWS=8, RTN_LSTM2_BWD_MT=tiles, RTN_LSTM2_BWD_POLL_DELAY=delay, RTN_LSTM2_BWD_DELAY_INC=inc):
                got, _, _ = _run(12, 19, 256, "bf16", 0, -1, seed=5)
                assert "bwd_regw" in lib.bwd_plan_text() and "tiles=%i" % tiles in lib.bwd_plan_text(), lib.bwd_plan_text()
            results.append(got)
        for other in results[1:]:
            for name, a, b in zip(("DX", "DW", "Dy0", "Dc0"), other, results[0]):
                assert numpy.array_equal(a, b), (tiles, name)


def test_bwd_groups_found_on_several_xcds_fall_back_to_device_scope():
    """With half the true XCD count the groups of an XCD-local gradient plan land on two XCDs each: the kernel's check
    finds that out and exchanges the ring at device scope (and adapts its read delay): the same bits, no abort."""
    from _gpu_util import env

    announce("bwd xcd-local with a wrong XCD count")
    T, B, n = 10, 32, 512
    want, _, _ = _run(T, B, n, "bf16", 0, 1, seed=3)
    plan = lib.bwd_plan_text()
    assert "bwd_regw_xcd" in plan, plan
    with env(RTN_LSTM2_XCDS=4):
        got, _, _ = _run(T, B, n, "bf16", 0, 1, seed=3)
        assert "bwd_regw_xcd" in lib.bwd_plan_text(), lib.bwd_plan_text()
    for name, a, b in zip(("DX", "DW", "Dy0", "Dc0"), got, want):
        assert numpy.isfinite(a).all(), name
        assert numpy.array_equal(a, b), name


def test_bwd_cfg2_reduced_f32():
    announce("bwd cfg2 reduced")
    p = synthetic.make_config("cfg2", T=60)
    rng = numpy.random.default_rng(2)
    DY = rng.normal(0, 1.0, (p.T, p.B, p.n)).astype(numpy.float32)
    Dd = rng.normal(0, 1.0, (p.B, p.n)).astype(numpy.float32)
    op = get_op()
    args = [to_dev(a, "f32") for a in (p.X, p.W, p.y0, p.c0, p.i)]
    Y, C, H, d = op(*args, 0, 1)
    got = torch_native_op.native_lstm2_grad(args[1], args[2], args[3], args[4], 0, 1, Y, C, H, to_dev(DY, "f32"), to_dev(Dd, "f32"))
    f = lambda t: t.float().cpu().numpy()  # noqa: E731
    want = oracle.native_lstm2_bwd(p.X, p.W, p.y0, p.c0, p.i, 0, 1, f(Y), f(C), f(H), DY, Dd, dtype=numpy.float64)
    for name, a, b in zip(("DX", "DW", "Dy0", "Dc0"), got, want):
        assert _rel_to_max(f(a), b) <= 2e-5, (name, _rel_to_max(f(a), b))


def test_bwd_autograd_function_matches_torch_lstm():
    """End to end through autograd: loss on Y and d, gradients equal those of torch.nn.LSTM on the CPU (float64)."""
    announce("bwd autograd")
    from test_oracle_bwd import torch_lstm_grads

    get_op()
    T, B, n = 9, 6, 32
    rng = numpy.random.default_rng(4)
    X = rng.normal(0, 0.7, (T, B, 4 * n)).astype(numpy.float32)
    W = (rng.normal(0, 1.0, (n, 4 * n)) / numpy.sqrt(n)).astype(numpy.float32)
    y0 = rng.normal(0, 0.4, (B, n)).astype(numpy.float32)
    c0 = rng.normal(0, 0.4, (B, n)).astype(numpy.float32)
    lens = numpy.array([9, 4, 1, 7, 9, 2])
    mask = (numpy.arange(T)[:, None] < lens[None, :]).astype(numpy.float32)
    GY = rng.normal(0, 1.0, (T, B, n)).astype(numpy.float32)
    Gd = rng.normal(0, 1.0, (B, n)).astype(numpy.float32)
    for reverse in (False, True):
        want = torch_lstm_grads(*(a.astype(numpy.float64) for a in (X, W, y0, c0)), lens, reverse, GY.astype(numpy.float64), Gd.astype(numpy.float64))
        leaves = [to_dev(a, "f32").requires_grad_(True) for a in (X, W, y0, c0)]
        Y, C, H, d = torch_native_op.NativeLstm2Function.apply(*leaves, to_dev(mask, "f32"), 0, -1 if reverse else 1)
        assert not C.requires_grad and not H.requires_grad
        loss = (Y * to_dev(GY, "f32")).sum() + (d * to_dev(Gd, "f32")).sum()
        loss.backward()
        for name, leaf, b in zip(("X", "W", "y0", "c0"), leaves, want):
            assert _rel_to_max(leaf.grad.cpu().numpy().astype(numpy.float64), b) <= 2e-5, (name, reverse)


def test_bwd_edge_cases_and_errors():
    announce("bwd edge cases")
    get_op()
    cabi = lib.load()
    B, n = 3, 16
    z = lambda *s: torch.zeros(s, device="cuda:0")  # noqa: E731
    Dd = torch.ones((B, n), device="cuda:0")
    DX, DW, Dy0, Dc0 = torch_native_op.native_lstm2_grad(z(n, 4 * n), z(B, n), z(B, n), z(0, B), 0, 1, z(0, B, n), z(0, B, n),
                                                         z(0, B, 4 * n), z(0, B, n), Dd)  # fmt: skip
    assert DX.shape == (0, B, 4 * n) and float(DW.abs().max()) == 0 and float(Dy0.abs().max()) == 0 and bool((Dc0 == 1).all())
    with pytest.raises(RuntimeError, match="start"):
        torch_native_op.native_lstm2_grad(z(n, 4 * n), z(B, n), z(B, n), z(4, B), 9, 1, z(4, B, n), z(4, B, n), z(4, B, 4 * n), z(4, B, n), Dd)
    with pytest.raises(RuntimeError, match="shape"):
        torch_native_op.native_lstm2_grad(z(n, 4 * n), z(B, n), z(B, n), z(4, B), 0, 1, z(4, B, n), z(4, B, n), z(4, B, n), z(4, B, n), Dd)
    with pytest.raises(RuntimeError, match="HIP"):
        torch_native_op.native_lstm2_grad(*(t.cpu() for t in (z(n, 4 * n), z(B, n), z(B, n), z(4, B))), 0, 1,
                                          *(t.cpu() for t in (z(4, B, n), z(4, B, n), z(4, B, 4 * n), z(4, B, n), Dd)))  # fmt: skip
    assert cabi.rtn_native_lstm2_bwd_workspace_bytes(10, B, n, 0) > 0
    assert cabi.rtn_native_lstm2_bwd_workspace_bytes(-1, B, n, 0) == 0


@pytest.mark.parametrize("T,B,n,dtype", [(14, 32, 256, "bf16"), (9, 20, 64, "f32"), (20, 32, 1024, "bf16"), (6, 5, 20, "f32"), (7, 70, 128, "bf16"), (6, 9, 100, "f32"), (5, 12, 200, "bf16")])
def test_bwd_multi_equals_single_calls(T, B, n, dtype):
    """
    The two directions of a layer through ``rtn_native_lstm2_bwd_multi``: against the oracle to the same bar as a single
    call, and against two single calls.  The joint launch may use another decomposition (k tiles per workgroup), which
    changes the order in which the MFMA partial sums are added: equal to float32 rounding, i.e. within 1e-5 of the
    largest magnitude in float32 and within one bfloat16 step (2^-7) of it in bfloat16.
    """
    announce("bwd multi", T, B, n, dtype)
    X, W, y0, c0, i = random_problem(50 + T + n, T, B, n)
    Wb = numpy.ascontiguousarray(W[::-1])  # another matrix for the other direction
    rng = numpy.random.default_rng(77)
    DY = [rng.normal(0, 1.0, (T, B, n)).astype(numpy.float32) for _ in range(2)]
    Dd = [rng.normal(0, 1.0, (B, n)).astype(numpy.float32) for _ in range(2)]
    op = get_op()
    Xd, y0d = to_dev(X, dtype), to_dev(y0, dtype)
    Wd = [to_dev(W, dtype), to_dev(Wb, dtype)]
    DYd = [to_dev(a, dtype) for a in DY]
    c0d, id_ = to_dev(c0, "f32"), to_dev(i, "f32")
    Ddd = [to_dev(a, "f32") for a in Dd]
    steps = (1, -1)
    fw = [op(Xd, Wd[k], y0d, c0d, id_, 0, steps[k]) for k in range(2)]
    calls = [(Wd[k], y0d, c0d, id_, 0, steps[k], fw[k][0], fw[k][1], fw[k][2], DYd[k], Ddd[k]) for k in range(2)]
    multi = torch_native_op.native_lstm2_grad_multi(calls)
    single = [torch_native_op.native_lstm2_grad(*c) for c in calls]
    torch.cuda.synchronize()
    f = lambda t: t.float().cpu().numpy().astype(numpy.float64)  # noqa: E731
    tol = 2e-5 if dtype == "f32" else 2e-2
    for k in range(2):
        Y, C, H, _ = fw[k]
        want = oracle.native_lstm2_bwd(f(Xd), f(Wd[k]), f(y0d), c0, i, 0, steps[k], f(Y), f(C), f(H), f(DYd[k]), Dd[k], dtype=numpy.float64)
        for name, a, s, b in zip(("DX", "DW", "Dy0", "Dc0"), multi[k], single[k], want):
            assert _rel_to_max(f(a), b) <= tol, (k, name, _rel_to_max(f(a), b))
            assert _rel_to_max(f(a), f(s)) <= (1e-5 if dtype == "f32" else 2.0**-7), (k, name, _rel_to_max(f(a), f(s)))


def test_bwd_multi_errors_and_empty():
    announce("bwd multi errors")
    get_op()
    cabi = lib.load()
    stream = torch.cuda.current_stream().cuda_stream
    assert cabi.rtn_native_lstm2_bwd_multi(None, 0, 4, 2, 32, lib.DTYPE_F32, None, 0, stream) == 0  # nothing to do
    assert cabi.rtn_native_lstm2_bwd_multi(None, 2, 4, 2, 32, lib.DTYPE_F32, None, 0, stream) == lib.RTN_ERR_ARG
    assert cabi.rtn_native_lstm2_bwd_multi_workspace_bytes(2, 4, 2, 32, lib.DTYPE_F32) == 2 * cabi.rtn_native_lstm2_bwd_workspace_bytes(4, 2, 32, lib.DTYPE_F32)
    with pytest.raises(RuntimeError, match="one shape"):
        z = lambda *s: torch.zeros(*s, device="cuda:0")  # noqa: E731
        a = (z(8, 32), z(2, 8), z(2, 8), z(3, 2), 0, 1, z(3, 2, 8), z(3, 2, 8), z(3, 2, 32), z(3, 2, 8), z(2, 8))
        b = (z(8, 32), z(2, 8), z(2, 8), z(4, 2), 0, 1, z(4, 2, 8), z(4, 2, 8), z(4, 2, 32), z(4, 2, 8), z(2, 8))
        torch_native_op.native_lstm2_grad_multi([a, b])


@pytest.mark.parametrize("T,B,n,dtype", [(40, 16, 256, "bf16"), (12, 9, 1024, "f32"), (10, 40, 128, "f32")])
def test_bwd_bounded_wait_expires_cleanly(T, B, n, dtype):
    """A wait bound of zero ticks forced from the host: the persistent gradient kernel (the ordinary variant, the one
    with half of W in LDS, and a batch in several groups) must still drain; the status call then reports success
    (nobody had to wait) or the abort, and the next ordinary call on the same workspace is unaffected."""
    from _gpu_util import env

    announce("bwd bounded wait", T, B, n, dtype)
    X, W, y0, c0, i = random_problem(77 + n, T, B, n)
    rng = numpy.random.default_rng(78)
    DY = rng.normal(0, 1.0, (T, B, n)).astype(numpy.float32)
    Dd = rng.normal(0, 1.0, (B, n)).astype(numpy.float32)
    op = get_op()
    Xd, Wd, y0d, DYd = (to_dev(a, dtype) for a in (X, W, y0, DY))
    c0d, id_, Ddd = (to_dev(a, "f32") for a in (c0, i, Dd))
    Y, C, H, d = op(Xd, Wd, y0d, c0d, id_, 0, 1)
    cabi = lib.load()
    dt = lib.DTYPE_BF16 if dtype == "bf16" else lib.DTYPE_F32
    act = torch.bfloat16 if dtype == "bf16" else torch.float32
    DX = torch.empty((T, B, 4 * n), dtype=act, device="cuda:0")
    DW = torch.empty((n, 4 * n), dtype=torch.float32, device="cuda:0")
    Dy0 = torch.empty((B, n), dtype=act, device="cuda:0")
    Dc0 = torch.empty((B, n), dtype=torch.float32, device="cuda:0")
    ws = torch.empty((max(int(cabi.rtn_native_lstm2_bwd_workspace_bytes(T, B, n, dt)), 256),), dtype=torch.uint8, device="cuda:0")
    stream = torch.cuda.current_stream().cuda_stream

    def call():
        return cabi.rtn_native_lstm2_bwd(
            Wd.data_ptr(), y0d.data_ptr(), c0d.data_ptr(), id_.data_ptr(), 0, 1, Y.data_ptr(), C.data_ptr(), H.data_ptr(),
            DYd.data_ptr(), Ddd.data_ptr(), DX.data_ptr(), DW.data_ptr(), Dy0.data_ptr(), Dc0.data_ptr(), T, B, n, dt,
            ws.data_ptr(), ws.numel(), stream,
        )  # fmt: skip

    with env(RTN_LSTM2_TIMEOUT_TICKS=0, RTN_LSTM2_BWD_KERNEL=2):
        assert call() == 0
    status = cabi.rtn_native_lstm2_fwd_status(ws.data_ptr(), stream)
    assert status in (lib.RTN_OK, lib.RTN_ERR_ABORTED)
    if status == lib.RTN_ERR_ABORTED:
        # visible without the status query too: NaN where every caller looks
        assert bool(torch.isnan(Dc0).any()) and bool(torch.isnan(Dy0.float()).any()), "no NaN marks after an expired wait"
    assert call() == 0
    assert cabi.rtn_native_lstm2_fwd_status(ws.data_ptr(), stream) == lib.RTN_OK
    torch.cuda.synchronize()
    f = lambda t: t.float().cpu().numpy().astype(numpy.float64)  # noqa: E731
    want = oracle.native_lstm2_bwd(f(Xd), f(Wd), f(y0d), c0, i, 0, 1, f(Y), f(C), f(H), f(DYd), Dd, dtype=numpy.float64)
    for name, a, b in zip(("DX", "DW", "Dy0", "Dc0"), (DX, DW, Dy0, Dc0), want):
        assert _rel_to_max(f(a), b) <= (2e-5 if dtype == "f32" else 2e-2), name


@pytest.mark.parametrize("T,B,n,dtype", [(10, 8, 128, "bf16"), (8, 5, 100, "f32"), (6, 3, 20, "f32")])
def test_forward_and_gradient_recorded_into_a_callers_graph(T, B, n, dtype):
    """A training step under stream capture: forward op and gradient op (persistent kernel and weight gradient, or one
    launch per frame) are recorded into the caller's graph after one eager run (which creates the library's rocBLAS handle).
    The graph is replayed three times with new inputs and eager work in between; every replay must agree with the
    eager gradient op (another decomposition: equal up to rounding) and with the oracle."""
    announce("captured training step", T, B, n, dtype)
    op = get_op()
    rng = numpy.random.default_rng(5)
    problems = [random_problem(1200 + k, T, B, n) for k in range(3)]
    grads_in = [(rng.normal(0, 1.0, (T, B, n)).astype(numpy.float32), rng.normal(0, 1.0, (B, n)).astype(numpy.float32)) for _ in range(3)]
    X, W, y0, c0, i = problems[0]
    Xd, Wd, y0d, DYd = (to_dev(a, dtype) for a in (X, W, y0, grads_in[0][0]))
    c0d, id_, Ddd = (to_dev(a, "f32") for a in (c0, i, grads_in[0][1]))

    def step():
        Y, C, H, d = op(Xd, Wd, y0d, c0d, id_, 0, 1)
        return (Y, C, H, d), torch_native_op.native_lstm2_grad(Wd, y0d, c0d, id_, 0, 1, Y, C, H, DYd, Ddd)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()  # eager warm-up on the capture stream
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        fwd_out, grad_out = step()
    f = lambda t: t.float().cpu().numpy().astype(numpy.float64)  # noqa: E731
    tol = 2e-5 if dtype == "f32" else 2e-2
    for k in range(3):
        Xk, Wk, y0k, c0k, ik = problems[k]
        for dst, src, dt in ((Xd, Xk, dtype), (Wd, Wk, dtype), (y0d, y0k, dtype), (DYd, grads_in[k][0], dtype), (c0d, c0k, "f32"),
                             (id_, ik, "f32"), (Ddd, grads_in[k][1], "f32")):  # fmt: skip
            dst.copy_(to_dev(src, dt))
        graph.replay()
        torch.cuda.synchronize()
        got_f = [t.clone() for t in fwd_out]
        got_g = [t.clone() for t in grad_out]
        eager_f, eager_g = step()
        torch.cuda.synchronize()
        for name, a, b in zip("YCHd", got_f, eager_f):
            assert torch.equal(a, b), (k, name)
        for name, a, b in zip(("DX", "DW", "Dy0", "Dc0"), got_g, eager_g):
            assert _rel_to_max(f(a), f(b)) <= tol, (k, name, "against the eager op")
        want = oracle.native_lstm2_bwd(f(Xd), f(Wd), f(y0d), c0k, ik, 0, 1, f(got_f[0]), f(got_f[1]), f(got_f[2]), f(DYd), grads_in[k][1], dtype=numpy.float64)
        for name, a, b in zip(("DX", "DW", "Dy0", "Dc0"), got_g, want):
            assert _rel_to_max(f(a), b) <= tol, (k, name, "against the oracle")


def test_gradient_from_two_host_threads_on_their_own_streams():
    """Two host threads, each with a stream of its own, run forward and gradient at the same time (the weight-gradient
    GEMMs go through a rocBLAS handle per thread, so neither can have its stream changed by the other).  Every result must
    equal what the main thread computes alone."""
    import threading

    announce("bwd from two threads")
    op = get_op()
    shapes = [(14, 6, 128, "bf16"), (11, 5, 160, "f32")]
    inputs, want = [], []
    for k, (T, B, n, dtype) in enumerate(shapes):
        X, W, y0, c0, i = random_problem(640 + k, T, B, n)
        rng = numpy.random.default_rng(650 + k)
        DY = rng.normal(0, 1.0, (T, B, n)).astype(numpy.float32)
        Dd = rng.normal(0, 1.0, (B, n)).astype(numpy.float32)
        Xd, Wd, y0d, DYd = (to_dev(a, dtype) for a in (X, W, y0, DY))
        c0d, id_, Ddd = (to_dev(a, "f32") for a in (c0, i, Dd))
        inputs.append((Xd, Wd, y0d, c0d, id_, DYd, Ddd))
        Y, C, H, _ = op(Xd, Wd, y0d, c0d, id_, 0, 1)
        want.append(torch_native_op.native_lstm2_grad(Wd, y0d, c0d, id_, 0, 1, Y, C, H, DYd, Ddd))
    torch.cuda.synchronize()
    results, errors = {}, []

    def work(k):
        try:
            Xd, Wd, y0d, c0d, id_, DYd, Ddd = inputs[k]
            stream = torch.cuda.Stream()
            with torch.cuda.stream(stream):
                for r in range(6):
                    Y, C, H, _ = op(Xd, Wd, y0d, c0d, id_, 0, 1)
                    results[(k, r)] = torch_native_op.native_lstm2_grad(Wd, y0d, c0d, id_, 0, 1, Y, C, H, DYd, Ddd)
            stream.synchronize()
        except Exception as exc:  # noqa: BLE001
            errors.append((k, exc))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(len(shapes))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not errors, errors
    for (k, r), grads in sorted(results.items()):
        for name, a, b in zip(("DX", "DW", "Dy0", "Dc0"), grads, want[k]):
            if name == "DW":  # rocBLAS may sum in another order from run to run
                assert _rel_to_max(a.double().cpu().numpy(), b.double().cpu().numpy()) <= 1e-5, (k, r, name)
            else:
                assert torch.equal(a, b), "thread %i, round %i: %s differs from the single-threaded result" % (k, r, name)


@pytest.mark.parametrize("dtype,bar", [("f32", 2e-5), ("bf16", 2e-2)])
@pytest.mark.parametrize("B,n", [(5, 72), (3, 30)])
def test_autograd_functions_of_two_directions(B, n, dtype, bar):
    """The differentiable calls of both directions, on separate gates and on one projection, against two of one direction."""
    T = 6
    announce("autograd of two directions", B, n, dtype)
    get_op()
    single, pair, bidir = torch_native_op.NativeLstm2Function, torch_native_op.NativeLstm2PairFunction, torch_native_op.NativeLstm2BidirFunction
    leaves, weights = [], []
    for k in range(2):
        X, W, y0, c0, i = random_problem(6100 + k, T, B, n)
        leaves.append([to_dev(a, dtype) for a in (X, W, y0)] + [to_dev(c0, "f32")])
        mask = to_dev(i, "f32")
        rng = numpy.random.default_rng(6200 + k)
        weights.append((to_dev(rng.normal(0, 1, (T, B, n)), dtype), to_dev(rng.normal(0, 1, (B, n)), "f32")))

    def gradients(run):
        args = [[t.clone().requires_grad_() for t in direction] for direction in leaves]
        Y, d = run(*args)
        torch.autograd.backward(list(Y) + list(d), [w for w, _ in weights] + [w for _, w in weights])
        return [t.detach() for t in (*Y, *d)] + [t.grad for direction in args for t in direction]

    def run_single(f, b):
        outs = [single.apply(*f, mask, 0, 1), single.apply(*b, mask, 0, -1)]
        return [o[0] for o in outs], [o[3] for o in outs]

    def run_pair(f, b):
        Yf, _, _, df, Yb, _, _, db = pair.apply(*f, *b, mask)
        return [Yf, Yb], [df, db]

    def run_bidir(f, b):
        Y, df, db = bidir.apply(torch.cat((f[0], b[0]), -1), *f[1:], *b[1:], mask)
        return [Y[..., :n], Y[..., n:]], [df, db]

    want = gradients(run_single)
    for run in (run_pair, run_bidir):
        for k, (a, b) in enumerate(zip(gradients(run), want)):
            assert a.shape == b.shape and a.dtype == b.dtype
            if k < 4:
                assert torch.equal(a, b), (run.__name__, k)
            assert _rel_to_max(a.float().cpu().numpy(), b.float().cpu().numpy()) <= bar, (run.__name__, k)


# one part and many, full and partly filled, rows that leave wavefronts without any; widths of one lane, of cut blocks, of pieces
# of 8 and of 16 bytes
@pytest.mark.parametrize("rows,width", [(1, 4), (3, 12), (63, 260), (64, 8), (65, 516), (129, 1000), (1000, 4000), (8200, 300), (20000, 2048)])
@pytest.mark.parametrize("dtype,out_dtype", [("f32", "f32"), ("bf16", "bf16"), ("bf16", "f32"), ("f32", "bf16")])
def test_column_sums(rows, width, dtype, out_dtype):
    announce("column sums", rows, width, dtype, out_dtype)
    get_op()
    cabi = lib.load()
    code = {"f32": lib.DTYPE_F32, "bf16": lib.DTYPE_BF16}
    x = torch.randn((rows, width), generator=torch.Generator().manual_seed(rows + width)).to(torch.bfloat16 if dtype == "bf16" else torch.float32)
    xd = x.to("cuda:0")
    out = torch.full((width + 64,), 7.0, dtype=torch.bfloat16 if out_dtype == "bf16" else torch.float32, device="cuda:0")
    size = int(cabi.rtn_column_sums_workspace_bytes(rows, width))
    ws = torch.full((size + 256,), 0x5A, dtype=torch.uint8, device="cuda:0")
    lib.check(cabi.rtn_column_sums(xd.data_ptr(), rows, width, code[dtype], out.data_ptr(), code[out_dtype], ws.data_ptr(), size, torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    assert bool((ws[size:] == 0x5A).all()) and bool((out[width:] == 7.0).all())
    want = x.double().sum(0)
    # (at most 128 parts of max(64, rows / 128) rows, rounded up to 16: chains of a sixteenth of either, and 4 more additions in each launch)
    part = -(-max(64, -(-rows // 128)) // 16) * 16
    chain = part // 16 + 1 + -(-rows // part) // 16 + 1 + 8
    bound = chain * 2.0**-24 * x.double().abs().sum(0) + (2.0**-8 * want.abs() if out_dtype == "bf16" else 0)
    assert bool(((out[:width].double().cpu() - want).abs() <= bound).all())
    if size:
        assert cabi.rtn_column_sums(xd.data_ptr(), rows, width, 0, out.data_ptr(), 0, ws.data_ptr(), size - 1, None) == lib.RTN_ERR_WORKSPACE
    assert cabi.rtn_column_sums(xd.data_ptr(), rows, width + 1, 0, out.data_ptr(), 0, ws.data_ptr(), size, None) == lib.RTN_ERR_SHAPE


# widths whose rows are not aligned to 16 bytes run on padded copies: pieces of 2, 4 and 8 bytes, rows beyond a multiple of four, one and two
# calls (more arrays than one launch of the copies takes), a pitch that decides the piece
@pytest.mark.parametrize("dtype,B,n", [("bf16", 5, 33), ("bf16", 3, 34), ("bf16", 7, 60), ("bf16", 2, 101), ("f32", 5, 33), ("f32", 3, 34), ("f32", 1, 65)])
def test_bwd_padded_copies(dtype, B, n):
    announce("bwd padded copies", dtype, B, n)
    bar = 2e-2 if dtype == "bf16" else 2e-5
    for T, step in [(1, 1), (6, -1)]:
        got, want, (X, W, y0, c0, i, DY, Dd) = _run(T, B, n, dtype, 0, step, seed=T + n)
        for name, a, b in zip(("DX", "DW", "Dy0", "Dc0"), got, want):
            assert a.shape == b.shape and _rel_to_max(a, b) <= bar, (T, name, _rel_to_max(a, b))
        Xd, Wd, y0d, DYd = (to_dev(a, dtype) for a in (X, W, y0, DY))
        c0d, id_, Ddd = (to_dev(a, "f32") for a in (c0, i, Dd))
        Y, C, H, _ = get_op()(Xd, Wd, y0d, c0d, id_, 0, step)
        wide = torch.full((T, B, n + 19), float("nan"), dtype=DYd.dtype, device="cuda:0")  # (rows further apart, and not aligned like the width)
        wide[..., 16 : 16 + n] = DYd
        calls = [(Wd, y0d, c0d, id_, 0, step, Y, C, H, dy, Ddd) for dy in (DYd, wide[..., 16 : 16 + n])]
        for grads in torch_native_op.native_lstm2_grad_multi(calls):
            for name, a, b in zip(("DX", "DW", "Dy0", "Dc0"), grads, got):
                assert _rel_to_max(a.float().cpu().numpy(), b) <= (1e-5 if dtype == "f32" else 2.0**-7), (T, name)


# the weight gradient of small layers in slices of the rows: one slice and many, rows that leave a slice cut or empty, widths that cut a tile,
# rows further apart than they are wide (two calls side by side), no frame but the first
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("T,B,n,count", [(1, 3, 32, 1), (2, 1, 64, 2), (9, 15, 4, 1), (40, 33, 100, 2), (130, 9, 68, 1), (65, 64, 256, 1), (30, 7, 192, 2), (300, 40, 36, 1), (64, 131, 384, 1)])
def test_bwd_weight_gradient_of_small_layers(T, B, n, count, dtype):
    """Against float64 products of what the op itself returned (dx0 is DX of the first visited frame where no frame is masked): the order of
    additions is all that differs, so within a few float32 roundings of the sum of magnitudes (64 of them, for up to 12 000 terms in slices)."""
    announce("bwd weight gradient", T, B, n, count, dtype)
    X, W, y0, c0, i = random_problem(n + T, T, B, n)
    i[:] = 1.0  # (no padding: dx0 is DX of the first frame)
    rng = numpy.random.default_rng(T)
    Xd, Wd, y0d = (to_dev(a, dtype) for a in (X, W, y0))
    c0d, id_ = to_dev(c0, "f32"), to_dev(i, "f32")
    op = get_op()
    wide = to_dev(rng.normal(0, 1, (T, B, 2 * n)), dtype)
    calls = []
    for k in range(count):
        Y, C, H, _ = op(Xd, Wd, y0d, c0d, id_, 0, 1 - 2 * k)
        calls.append((Wd, y0d, c0d, id_, 0, 1 - 2 * k, Y, C, H, wide[..., k * n : (k + 1) * n], to_dev(rng.normal(0, 1, (B, n)), "f32")))
    f = lambda t: t.float().cpu().numpy().astype(numpy.float64)  # noqa: E731
    results = torch_native_op.native_lstm2_grad_multi(calls)
    assert ("weight_gradient=k_weight_grad" in lib.bwd_plan_text()) == (n <= 256 or dtype == "f32"), lib.bwd_plan_text()
    for call, (DX, DW, _, _) in zip(calls, results):
        Y, DX = f(call[6]), f(DX)
        if call[5] < 0:
            Y, DX = Y[::-1], DX[::-1]
        before = numpy.concatenate([f(y0d)[None], Y[:-1]]).reshape(T * B, n)
        DX = DX.reshape(T * B, 4 * n)
        bound = 64 * 2.0**-24 * (numpy.abs(before).T @ numpy.abs(DX)) + 1e-30
        assert (numpy.abs(f(DW) - before.T @ DX) <= bound).all()


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_bwd_without_frames_or_cells_writes_its_outputs_only(dtype):
    """Gradients of no frames (Dy0 of three rows of five cells: an odd number of elements) and of no cells (LstmLowMem's DX): zeros, up to the last element."""
    announce("bwd zeros", dtype)
    get_op()
    cabi = lib.load()
    act, code = (torch.bfloat16, lib.DTYPE_BF16) if dtype == "bf16" else (torch.float32, lib.DTYPE_F32)
    stream = torch.cuda.current_stream().cuda_stream
    B, n = 3, 5
    z = lambda *s: torch.zeros(s, device="cuda")  # noqa: E731
    out = torch.full((32,), 7.0, dtype=act, device="cuda")
    any_, Dd, DW, Dc0 = z(64), torch.ones((B, n), device="cuda"), z(n, 4 * n), z(B, n)
    lib.check(cabi.rtn_native_lstm2_bwd(*[any_.data_ptr()] * 4, 0, 1, *[any_.data_ptr()] * 4, Dd.data_ptr(), any_.data_ptr(), DW.data_ptr(), out.data_ptr(), Dc0.data_ptr(),
                                        0, B, n, code, None, 0, stream))  # fmt: skip
    assert bool((out[: B * n] == 0).all()) and bool((out[B * n :] == 7.0).all()) and torch.equal(Dc0, Dd)
    out.fill_(7.0)
    args = [any_.data_ptr()] * 15
    args[10] = out.data_ptr()
    lib.check(cabi.rtn_lstm_low_mem_bwd(*args[:6], 0, 1, *args[6:], 3, 1, 5, 0, code, None, 0, stream))
    assert bool((out[:15] == 0).all()) and bool((out[15:] == 7.0).all())


@pytest.mark.parametrize("T,B,n", [(260, 32, 324), (260, 33, 268), (3, 2, 324)])
def test_bwd_smallest_accepted_workspace(T, B, n):
    """Widths padded on the fly whose slices of the weight gradient take more bytes than the padded width's: on the least workspace that the
    entry accepts nothing is written behind it, and the weight gradient is that of float64 products (bound as above)."""
    announce("bwd least workspace", T, B, n)
    X, W, y0, c0, i = random_problem(n, T, B, n)
    i[:] = 1.0
    args = [to_dev(a, "f32") for a in (X, W, y0, c0, i)]
    Y, C, H, _ = get_op()(*args, 0, 1)
    rng = numpy.random.default_rng(9)
    DY, Dd = to_dev(rng.normal(0, 1, (T, B, n)), "f32"), to_dev(rng.normal(0, 1, (B, n)), "f32")
    DX, DW, Dy0, Dc0 = (torch.empty(shape, device="cuda") for shape in ((T, B, 4 * n), (n, 4 * n), (B, n), (B, n)))
    cabi = lib.load()

    def call(ws, size):
        return cabi.rtn_native_lstm2_bwd(*[a.data_ptr() for a in args[1:]], 0, 1, Y.data_ptr(), C.data_ptr(), H.data_ptr(), DY.data_ptr(), Dd.data_ptr(), DX.data_ptr(),
                                         DW.data_ptr(), Dy0.data_ptr(), Dc0.data_ptr(), T, B, n, lib.DTYPE_F32, ws, size, torch.cuda.current_stream().cuda_stream)  # fmt: skip

    assert call(None, 0) == lib.RTN_ERR_WORKSPACE
    need = int(lib.last_error().split("workspace of ")[1].split()[0])
    ws = torch.full((need + 2**21,), 0x5A, dtype=torch.uint8, device="cuda")
    lib.check(call(ws.data_ptr(), need))
    torch.cuda.synchronize()
    assert bool((ws[need:] == 0x5A).all())
    f = lambda t: t.cpu().numpy().astype(numpy.float64)  # noqa: E731
    before, dx = numpy.concatenate([f(args[2])[None], f(Y)[:-1]]).reshape(T * B, n), f(DX).reshape(T * B, 4 * n)
    bound = 64 * 2.0**-24 * (numpy.abs(before).T @ numpy.abs(dx)) + 1e-30
    assert (numpy.abs(f(DW) - before.T @ dx) <= bound).all()


# a^T b in slices of the rows: widths that cut a tile, odd ones and rows that are farther apart (by element), one row, a slice's edge, and
# more rows than a round of every slice takes
@pytest.mark.parametrize("rows,m,n", [(1, 4, 1), (127, 64, 64), (129, 68, 77), (700, 180, 45), (9001, 256, 40), (20000, 128, 3)])
@pytest.mark.parametrize("dtype,out_dtype", [("f32", "f32"), ("bf16", "bf16"), ("bf16", "f32")])
@pytest.mark.parametrize("pad", [0, 3])
def test_transposed_product(rows, m, n, dtype, out_dtype, pad):
    announce("transposed product", rows, m, n, dtype, out_dtype, pad)
    code = {"f32": 0, "bf16": 1}
    rng = numpy.random.default_rng(6)
    a = to_dev(rng.normal(0, 1, (rows, m + 4 * pad)), dtype)
    b = to_dev(rng.normal(0, 1, (rows, n + pad)), dtype)
    out = torch.full((m, n), float("nan"), device="cuda", dtype=torch.float32 if out_dtype == "f32" else torch.bfloat16)
    cabi = lib.load()
    size = int(cabi.rtn_transposed_product_workspace_bytes(rows, m, n, code[dtype]))
    assert size > 0
    ws = torch.empty(size, dtype=torch.uint8, device="cuda")

    def call(size=size, lda=m + 4 * pad):
        return cabi.rtn_transposed_product(a.data_ptr(), lda, b.data_ptr(), n + pad, rows, m, n, code[dtype], out.data_ptr(), code[out_dtype], ws.data_ptr(), size, torch.cuda.current_stream().cuda_stream)

    assert call(size - 1) == lib.RTN_ERR_WORKSPACE and call(lda=m + 2) == lib.RTN_ERR_SHAPE
    lib.check(call())
    wide = a[:, :m].cpu().double(), b[:, :n].cpu().double()
    want, size_of_terms = wide[0].t() @ wide[1], wide[0].abs().t() @ wide[1].abs()
    # float32 sums of `rows` terms in any order, then the rounding of the result
    bound = size_of_terms * (rows + 8) * 2.0**-24 + want.abs() * (2.0**-8 if out_dtype == "bf16" else 2.0**-23) + 1e-30
    assert bool(((out.cpu().double() - want).abs() <= bound).all())
    assert int(cabi.rtn_transposed_product_workspace_bytes(rows, m + 2, n, code[dtype])) == 0  # (not whole quads)
    assert int(cabi.rtn_transposed_product_workspace_bytes(rows, 4096, 4096, code[dtype])) == 0  # (the library's)


# The weight gradient in the op's type: own kernel (n = 64), last share in a pass of its own (few rows; tiles of the output cut, no long product
# with one frame), library and conversion (many rows, also every second frame), padded copies (n = 45); one of the two calls only: a launch each.
@pytest.mark.parametrize("T,B,n,step", [(7, 5, 64, 1), (6, 5, 420, 1), (1, 3, 512, 1), (9, 64, 1024, -1), (5, 260, 512, 1), (7, 4, 512, 2), (5, 3, 45, 1)])
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("wanted", [(True, True), (False, True)])
def test_bwd_weight_gradient_in_the_ops_type(T, B, n, step, dtype, wanted):
    announce("bwd weight gradient type", T, B, n, step, dtype, wanted)
    cabi = lib.load()
    act, code = (torch.bfloat16, lib.DTYPE_BF16) if dtype == "bf16" else (torch.float32, lib.DTYPE_F32)
    op = get_op()
    arr, keep = (lib.Lstm2BwdCall * 2)(), []
    for k in range(2):
        X, W, y0, c0, i = random_problem(700 + k, T, B, n)
        args = [to_dev(X, dtype), to_dev(W, dtype), to_dev(y0, dtype), to_dev(c0, "f32"), to_dev(i, "f32")]
        s = step if k == 0 else -step
        Y, C, H, _ = op(*args, 0, s)
        rng = numpy.random.default_rng(60 + k)
        DY, Dd = to_dev(rng.normal(0, 1, (T, B, n)), dtype), to_dev(rng.normal(0, 1, (B, n)), "f32")
        DX = torch.empty((T, B, 4 * n), dtype=act, device="cuda")
        DW = torch.full((n, 4 * n), float("nan"), device="cuda")
        DW_act = torch.full((n, 4 * n), float("nan"), device="cuda", dtype=act) if wanted[k] else None
        Dy0, Dc0 = torch.empty((B, n), dtype=act, device="cuda"), torch.empty((B, n), device="cuda")
        arr[k] = lib.Lstm2BwdCall(*[a.data_ptr() for a in args[1:]], 0, s, Y.data_ptr(), C.data_ptr(), H.data_ptr(), DY.data_ptr(), Dd.data_ptr(), DX.data_ptr(),
                                  DW.data_ptr(), Dy0.data_ptr(), Dc0.data_ptr(), 0, 0, 0, DW_act.data_ptr() if wanted[k] else None)  # fmt: skip
        g = lambda t: t.float().cpu().numpy().astype(numpy.float64)  # noqa: E731
        want = oracle.native_lstm2_bwd(g(args[0]), g(args[1]), g(args[2]), c0, i, 0, s, g(Y), g(C), g(H), g(DY), g(Dd), dtype=numpy.float64)[1]
        keep.append((args, Y, C, H, DY, Dd, DX, DW, DW_act, Dy0, Dc0, want))
    ws = torch.empty(int(cabi.rtn_native_lstm2_bwd_multi_workspace_bytes(2, T, B, n, code)), dtype=torch.uint8, device="cuda")
    lib.check(cabi.rtn_native_lstm2_bwd_multi(arr, 2, T, B, n, code, ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream))
    way = "k_weight_grad" if n <= 64 else "rocblas,k_weight_last" if B <= 64 else "rocblas"
    assert lib.bwd_plan_text().endswith(" weight_gradient=" + way), lib.bwd_plan_text()
    for k in range(2):
        got, want = keep[k][8] if wanted[k] else keep[k][7], keep[k][11]
        scale = float(numpy.abs(want).max())
        # (the bounds of the gradient tests above; the result itself rounds to 2^-9 of its size)
        assert float(numpy.abs(got.float().cpu().numpy() - want).max()) <= scale * (2e-2 if dtype == "bf16" else 2e-5)
        if wanted[k] and dtype == "f32":
            assert got.dtype == torch.float32
    if wanted[0]:
        arr[0].DW_act += 4
        assert cabi.rtn_native_lstm2_bwd_multi(arr, 2, T, B, n, code, ws.data_ptr(), ws.numel(), None) == lib.RTN_ERR_ARG


# No error on the final cell state, without an array for it: persistent kernels (one XCD, all), one launch per frame, padded copies, no frame at all
@pytest.mark.parametrize("T,B,n,kernel", [(6, 5, 64, 0), (5, 20, 1280, 0), (4, 3, 32, 1), (4, 3, 45, 0), (0, 3, 32, 0)])
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_bwd_without_error_on_the_final_state(T, B, n, kernel, dtype):
    from _gpu_util import env

    announce("bwd without Dd", T, B, n, kernel, dtype)
    cabi = lib.load()
    act, code = (torch.bfloat16, lib.DTYPE_BF16) if dtype == "bf16" else (torch.float32, lib.DTYPE_F32)
    X, W, y0, c0, i = random_problem(810, T, B, n)
    args = [to_dev(X, dtype), to_dev(W, dtype), to_dev(y0, dtype), to_dev(c0, "f32"), to_dev(i, "f32")]
    Y, C, H, _ = get_op()(*args, 0, 1)
    DY = to_dev(numpy.random.default_rng(61).normal(0, 1, (T, B, n)), dtype)
    zeros = torch.zeros((B, n), device="cuda")
    ws = torch.empty(int(cabi.rtn_native_lstm2_bwd_multi_workspace_bytes(1, T, B, n, code)), dtype=torch.uint8, device="cuda")
    results = []
    for absent in (False, True):
        outs = [torch.full(s, float("nan"), device="cuda", dtype=d) for s, d in (((T, B, 4 * n), act), ((n, 4 * n), torch.float32), ((B, n), act), ((B, n), torch.float32))]
        call = (lib.Lstm2BwdCall * 1)(lib.Lstm2BwdCall(*[a.data_ptr() for a in args[1:]], 0, 1, Y.data_ptr(), C.data_ptr(), H.data_ptr(), DY.data_ptr(),
                                                       None if absent else zeros.data_ptr(), *[o.data_ptr() for o in outs], 0, 0, 0, None, int(absent)))  # fmt: skip
        with env(RTN_LSTM2_BWD_KERNEL=kernel):
            lib.check(cabi.rtn_native_lstm2_bwd_multi(call, 1, T, B, n, code, ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream))
            name = "k_bwd_step" if kernel == 1 or (n, dtype) == (1280, "f32") else "k_lstm2_bwd_regw" if n == 1280 else "k_lstm2_bwd_local"
            assert T == 0 or "name=%s " % name in lib.bwd_plan_text(), lib.bwd_plan_text()
        results.append(outs)
        call[0].Dd, call[0].Dd_is_zero = None, 0
        assert cabi.rtn_native_lstm2_bwd_multi(call, 1, T, B, n, code, ws.data_ptr(), ws.numel(), None) == lib.RTN_ERR_ARG
    for k, (a, b) in enumerate(zip(*results)):
        assert torch.isfinite(a.float()).all()
        # (the products' partial sums may be added in another order)
        assert torch.equal(a, b) if k != 1 else float((a - b).abs().max()) <= 2.0**-20 * max(1.0, float(a.abs().max())) * (T * B) ** 0.5, k
