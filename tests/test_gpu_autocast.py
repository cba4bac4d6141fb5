"""
The layers under ``torch.autocast``: their projection is a matrix product like torch's own (operands and result in the
region's type, errors back in the operands' types), and the recurrence runs in the type that result has for the op.
"""

from __future__ import annotations

import pytest
import torch

from returnn_amd.lstm import LSTM, BlstmEncoder, LstmState
from returnn_amd.torch_native_op import NativeLstm2Function

from _gpu_util import announce

pytestmark = pytest.mark.gpu

T, B, N_IN, N = 7, 5, 24, 64
TYPES = [torch.bfloat16, torch.float16]


def _layer(seed, bias=True, dtype=torch.float32):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    m = LSTM(N_IN, N, with_bias=bias, device="cuda", dtype=dtype)
    m.reset_parameters(gen)
    if bias:
        with torch.no_grad():
            m.bias.uniform_(-0.5, 0.5, generator=gen)
    return m, gen


def _run_type(amp):
    return torch.bfloat16 if amp == torch.bfloat16 else torch.float32


def _reference(m, x, state, mask, direction, amp):
    """Torch's own projection in the region, the op with its gradient on what it gives."""
    with torch.autocast("cuda", dtype=amp):
        x2 = x.reshape(-1, N_IN)
        P = torch.mm(x2, m.ff.t()) if m.bias is None else torch.addmm(m.bias, x2, m.ff.t())
    Y, _, _, d = NativeLstm2Function.apply(P.view(x.shape[0], B, 4 * N), m.rec, state.h, state.c, mask, 0, direction)
    return Y, d


@pytest.mark.parametrize("amp", TYPES, ids=str)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=str)
@pytest.mark.parametrize("bias", [True, False])
@pytest.mark.parametrize("backward_inside", [True, False])
def test_training_step(amp, dtype, bias, backward_inside):
    announce("autocast training step", amp, dtype, bias, backward_inside)
    m, gen = _layer(11, bias, dtype)
    x = torch.randn((T, B, N_IN), device="cuda", generator=gen).to(dtype).requires_grad_()
    state = LstmState(
        h=torch.randn((B, N), device="cuda", generator=gen).mul(0.3).to(dtype).requires_grad_(),
        c=torch.randn((B, N), device="cuda", generator=gen).requires_grad_(),
    )
    lens = torch.tensor([7, 1, 4, 6, 7], device="cuda")
    mask = (torch.arange(T, device="cuda")[:, None] < lens[None, :]).float()
    leaves = [x, state.h, state.c, *m.parameters()]

    def gradients(Y, d):
        dY, dd = (torch.linspace(-1, 1, t.numel(), device="cuda").view(t.shape).to(t.dtype) for t in (Y, d))
        return torch.autograd.grad([Y, d], leaves, [dY, dd])

    want = _reference(m, x, state, mask, -1, amp)
    want_grads = gradients(*want)
    with torch.autocast("cuda", dtype=amp):
        y, st = m(x, state=state, seq_lens=lens, direction=-1)
        if backward_inside:
            grads = gradients(y, st.c)
    if not backward_inside:
        grads = gradients(y, st.c)
    assert y.dtype == _run_type(amp) and st.h.dtype == y.dtype and st.c.dtype == torch.float32
    for got, ref in zip((y, st.c), want):
        assert torch.equal(got, ref)
    for leaf, got, ref in zip(leaves, grads, want_grads):
        assert got.dtype == leaf.dtype and torch.isfinite(got).all()
        # (the same products, of the same values: at most another split of a sum over T * B = 35 rows or 4n = 256 columns,
        # each product of which a float32 sum rounds by 2^-24 of what it has gathered so far, before the last rounding to the
        # operands' type, half a unit of which is 2^-9 in bfloat16)
        assert float((got.double() - ref.double()).norm()) <= 2**-8 * float(ref.double().norm())


def test_training_with_the_default_state_of_an_encoder():
    announce("autocast encoder")
    gen = torch.Generator(device="cuda").manual_seed(13)
    m = BlstmEncoder(N_IN, N, 2, device="cuda")
    m.reset_parameters(gen)
    x = torch.randn((T, B, N_IN), device="cuda", generator=gen)
    lens = torch.tensor([3, 7, 7, 2, 5], device="cuda")
    dy = torch.randn((T, B, 2 * N), device="cuda", generator=gen)

    def step(source, amp):
        source = source.clone().requires_grad_()
        m.zero_grad(set_to_none=True)
        with torch.autocast("cuda", dtype=torch.bfloat16, enabled=amp):
            y = m(source, seq_lens=lens)
        y.backward(dy.to(y.dtype))
        return [y.detach(), source.grad] + [p.grad for p in m.parameters()]

    got = step(x, True)
    want = step(x.bfloat16(), False)  # parameters cast to the run's type, outside any region
    assert got[0].dtype == torch.bfloat16 and all(g.dtype == torch.float32 for g in got[1:])
    for a, b in zip(got, want):
        # (the same operations but for the recurrent weights' gradients, which are rounded to bfloat16 on the way without the
        # region: half a unit, 2^-9)
        assert float((a.double() - b.double()).norm()) <= 2**-8 * float(b.double().norm())


@pytest.mark.parametrize("amp", TYPES, ids=str)
def test_parameters_stay_usable_in_the_region(amp):
    """The region keeps the casts of leaf parameters for its later operations: those must not lose the way back to them."""
    announce("autocast, parameters used again", amp)
    m, gen = _layer(17)
    x = torch.randn((T, B, N_IN), device="cuda", generator=gen)
    with torch.autocast("cuda", dtype=amp):
        m(x, state=m.default_initial_state(batch_dims=(B,)))
        z = torch.addmm(m.bias, x.reshape(-1, N_IN), m.ff.t())
    z.backward(torch.ones_like(z))
    assert m.bias.grad is not None and torch.equal(m.bias.grad, torch.full_like(m.bias, T * B))


@pytest.mark.parametrize("amp", TYPES, ids=str)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=str)
def test_one_step_is_a_sequence_of_one_frame(amp, dtype):
    announce("autocast, one step", amp, dtype)
    m, gen = _layer(19, dtype=dtype)
    x = torch.randn((B, N_IN), device="cuda", generator=gen).to(dtype)
    state = LstmState(h=torch.randn((B, N), device="cuda", generator=gen).mul(0.3).to(dtype), c=torch.randn((B, N), device="cuda", generator=gen))
    with torch.no_grad(), torch.autocast("cuda", dtype=amp):
        y, st = m(x, state=state)
        want, want_st = m(x[None], state=state)
    assert y.dtype == want.dtype == _run_type(amp) and st.h.dtype == y.dtype and st.c.dtype == torch.float32
    assert torch.equal(y, st.h)
    # (the one-step kernel keeps the projection in float32, the sequence rounds it to the region's type: half a unit of values
    # below 4, 2^-7 in bfloat16, which the gates pass on with a slope of at most 1 for each of cell-in, input and forget --
    # the cells here stay below 4 -- and the output's own rounding)
    tol = 2**-5 if amp == torch.bfloat16 else 2**-8
    for got, ref in ((y, want[0]), (st.c, want_st.c)):
        assert float((got.double() - ref.double()).abs().max()) <= tol
