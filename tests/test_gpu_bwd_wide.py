"""The gradient kernel for layers whose recurrent weights take the registers and the LDS of the CUs of a batch group."""

from __future__ import annotations

import numpy
import pytest
import torch

from returnn_amd import lib, torch_native_op

import test_gpu_bwd
import test_gpu_siblings as siblings
from _gpu_util import announce, env, get_op, random_problem, to_dev
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


def test_recorded_gradients_agree_with_eager_ones():
    """Two problems of five groups each, in several launches: every replay arms the rings anew."""
    announce("wide gradient, recorded")
    T, B, n = 9, 70, 1280
    get_op()
    X, W, y0, c0, i = random_problem(31, T, B, n)
    Xd, Wd, y0d, c0d, id_ = to_dev(X, "bf16"), to_dev(W, "bf16"), to_dev(y0, "bf16"), to_dev(c0, "f32"), to_dev(i, "f32")
    DY, Dd = Xd[:, :, :n].contiguous(), c0d.clone()

    def step():
        fw = torch_native_op.native_lstm2_multi([(Xd, Wd, y0d, c0d, id_, 0, 1), (Xd, Wd, y0d, c0d, id_, 0, -1)])
        return torch_native_op.native_lstm2_grad_multi([(Wd, y0d, c0d, id_, 0, (1, -1)[k], *fw[k][:3], DY, Dd) for k in range(2)])

    with env(RTN_LSTM2_BWD_WIDE=2):
        want = step()
        assert "problems=2" in lib.bwd_plan_text() and "name=k_lstm2_bwd_wide" in lib.bwd_plan_text(), lib.bwd_plan_text()
        torch.cuda.synchronize()
        graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.graph(graph, stream=side):
            got = step()
        for _ in range(3):
            graph.replay()
            again = step()  # the program's own work in between
            torch.cuda.synchronize()
            for k in range(2):
                for name, a, b, c in zip(("DX", "DW", "Dy0", "Dc0"), got[k], want[k], again[k]):
                    if name == "DW":  # (rocBLAS may sum in another order)
                        assert float((a - b).abs().max()) <= 1e-5 * float(b.abs().max()), (k, name)
                    else:
                        assert torch.equal(a, b) and torch.equal(c, b), (k, name)


def _gradients(problems, dtype="bf16"):
    """:param problems: of (T, B, n); -> the gradients of all of them, as one call"""
    calls = []
    for k, (T, B, n) in enumerate(problems):
        X, W, y0, c0, i = random_problem(41 + k, T, B, n)
        rng = numpy.random.default_rng(42 + k)
        Xd, Wd, y0d, c0d, id_ = to_dev(X, dtype), to_dev(W, dtype), to_dev(y0, dtype), to_dev(c0, "f32"), to_dev(i, "f32")
        Y, C, H, _ = get_op()(Xd, Wd, y0d, c0d, id_, 0, (1, -1)[k % 2])
        DY, Dd = to_dev(rng.normal(0, 1, (T, B, n)), dtype), to_dev(rng.normal(0, 1, (B, n)), "f32")
        calls.append((Wd, y0d, c0d, id_, 0, (1, -1)[k % 2], Y, C, H, DY, Dd))
    got = torch_native_op.native_lstm2_grad_multi(calls)
    return got, lib.bwd_plan_text(), calls


# both sides of the rule: as many launches as with one tile per workgroup, 2 for 3, 1 for 2; problems that share a launch
@pytest.mark.parametrize(
    "count,B,n,wide",
    [(1, 64, 2048, True), (1, 32, 2048, False), (2, 32, 2048, True), (2, 16, 2048, False), (1, 64, 1280, True), (1, 40, 1280, False), (1, 80, 1088, False), (1, 96, 1408, True)],
)
def test_rule_takes_it_where_it_spares_launches(count, B, n, wide):
    """Without an override; the general kernel splits the contraction in another way: equal to one bfloat16 step of the largest magnitude."""
    announce("wide gradient, rule", count, B, n)
    problems = [(3, B, n)] * count
    got, plan, _ = _gradients(problems)
    assert ("name=k_lstm2_bwd_wide" in plan) == wide and ("name=k_lstm2_bwd_regw" in plan) != wide, plan
    if wide:
        with env(RTN_LSTM2_BWD_WIDE=0):
            want, plan, _ = _gradients(problems)
        assert "name=k_lstm2_bwd_regw" in plan, plan
        for a, b in zip(got, want):
            for name, x, y in zip(("DX", "DW", "Dy0", "Dc0"), a, b):
                assert bool(torch.isfinite(x).all()) and float((x.float() - y.float()).abs().max()) <= 2.0**-7 * float(y.float().abs().max()), name


# (a launch takes two problems; calls with more run one by one)
@pytest.mark.parametrize("count,last", [(2, 2), (3, 1)])
def test_problems_with_groups_of_their_own(count, last):
    announce("wide gradient, problems", count)
    problems = [(5, 16, 1152)] * count
    with env(RTN_LSTM2_BWD_WIDE=2):
        got, plan, calls = _gradients(problems)
        assert "problems=%i" % last in plan and "name=k_lstm2_bwd_wide" in plan, plan
        alone = [torch_native_op.native_lstm2_grad(*c) for c in calls]
        assert "name=k_lstm2_bwd_wide" in lib.bwd_plan_text()
    for a, b in zip(got, alone):
        for name, x, y in zip(("DX", "Dy0", "Dc0"), (a[0], a[2], a[3]), (b[0], b[2], b[3])):
            assert torch.equal(x, y), name


def test_no_error_on_the_final_state_is_an_error_of_zero():
    announce("wide gradient without Dd")
    T, B, n = 4, 40, 1152
    with env(RTN_LSTM2_BWD_WIDE=2):
        _, _, calls = _gradients([(T, B, n)])
        W, y0, c0, i, _, _, Y, C, H, DY, Dd = calls[0]
        want = torch_native_op.native_lstm2_grad(*calls[0][:-1], torch.zeros_like(Dd))
        got = [torch.full_like(t, float("nan")) for t in want]
        c = lib.Lstm2BwdCall(*(t.data_ptr() for t in (W, y0, c0, i)), 0, 1, *(t.data_ptr() for t in (Y, C, H, DY)), None, *(t.data_ptr() for t in got), 0, 0, 0, None, 1)
        ws = torch.empty(int(lib.load().rtn_native_lstm2_bwd_multi_workspace_bytes(1, T, B, n, lib.DTYPE_BF16)), dtype=torch.uint8, device="cuda")
        lib.check(lib.load().rtn_native_lstm2_bwd_multi((lib.Lstm2BwdCall * 1)(c), 1, T, B, n, lib.DTYPE_BF16, ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
        assert "name=k_lstm2_bwd_wide" in lib.bwd_plan_text()
    for name, x, y in zip(("DX", "Dy0", "Dc0"), (got[0], got[2], got[3]), (want[0], want[2], want[3])):
        assert torch.equal(x, y), name


def test_other_ops_on_the_same_kernel():
    """LstmGenericBase (cell states in H, nothing carried over a masked frame) and LstmLowMem (errors of the output before the mask)."""
    with env(RTN_LSTM2_BWD_WIDE=2):
        siblings.test_generic_base_gradient(5, 40, 1152, "bf16")
        assert "name=k_lstm2_bwd_wide" in lib.bwd_plan_text(), lib.bwd_plan_text()
        announce("wide gradient, low_mem")
        got, want = siblings._low_mem_grad_case(60, 5, 40, 64, 1152, 0, 1, "bf16")
        assert "name=k_lstm2_bwd_wide" in lib.bwd_plan_text(), lib.bwd_plan_text()
    for a, b in zip(got, want):
        assert numpy.isfinite(a).all() and _rel_to_max(a, b) <= 3e-2, _rel_to_max(a, b)  # (the bound of that op's other tests)


def test_bounded_wait_expires_cleanly():
    with env(RTN_LSTM2_BWD_WIDE=2):
        test_gpu_bwd.test_bwd_bounded_wait_expires_cleanly(6, 40, 1152, "bf16")
        assert "name=k_lstm2_bwd_wide" in lib.bwd_plan_text(), lib.bwd_plan_text()
