"""One step of a layer, projection included (``rtn_lstm_step``), against the same step in float64 on the CPU."""

from __future__ import annotations

import pytest
import torch

from _gpu_util import announce
import returnn_amd.lstm as lstm_mod

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize(
    "B,n_in,n,bias",
    [(1, 1, 1, True), (1, 40, 32, False), (3, 33, 7, True), (16, 512, 64, True), (17, 31, 100, True), (33, 80, 1000, False), (64, 65, 72, True),
     (65, 16, 33, True), (130, 200, 136, True), (12, 512, 1024, True)],
)  # fmt: skip
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_step_against_float64(B, n_in, n, bias, dtype):
    announce("lstm_step", B, n_in, n, bias, dtype)
    from returnn_amd.lstm import LSTM, LstmState

    act = torch.bfloat16 if dtype == "bf16" else torch.float32
    gen = torch.Generator().manual_seed(B + 7 * n_in + 31 * n)
    m = LSTM(n_in, n, with_bias=bias)
    m.reset_parameters(gen)
    if bias:
        with torch.no_grad():
            m.bias.uniform_(-0.5, 0.5, generator=gen)
    m = m.to(act).requires_grad_(False)
    x, h = (torch.randn((B, k), generator=gen).mul(0.5).to(act) for k in (n_in, n))
    c = torch.randn((B, n), generator=gen)
    gates = x.double() @ m.ff.double().t() + h.double() @ m.rec.double()
    if bias:
        gates = gates + m.bias.double()
    g, i, f, o = gates.chunk(4, dim=1)
    want_c = torch.sigmoid(f) * c.double() + torch.sigmoid(i) * torch.tanh(g)
    want_y = torch.sigmoid(o) * torch.tanh(want_c)
    y, st = m.to("cuda:0")(x.cuda(), state=LstmState(h=h.cuda(), c=c.cuda()))
    torch.cuda.synchronize()
    assert y.dtype == act and st.h.dtype == act and st.c.dtype == torch.float32
    assert torch.equal(y, st.h) and y.data_ptr() != st.h.data_ptr()
    tol = 1e-2 if dtype == "bf16" else 2e-6
    for got, want in ((y, want_y), (st.c, want_c)):
        assert float((got.cpu().double() - want).abs().max()) <= tol


@pytest.mark.parametrize("B,n_in,n,dtype", [(385, 2048, 2048, "bf16"), (65, 2048, 4096, "f32"), (641, 512, 1024, "f32"), (4096, 1024, 1000, "bf16")])
def test_many_rows_run_as_a_sequence_of_one_frame(B, n_in, n, dtype):
    """Where the one-step kernel would read the weights too often, the projection is a GEMM and the recurrent kernels follow:
    the bits of a sequence of one frame.  (The one-step kernel adds in another order: one share of the batch has other bits.)"""
    announce("lstm_step, many rows", B, n_in, n, dtype)
    from returnn_amd.lstm import LSTM, LstmState

    act = torch.bfloat16 if dtype == "bf16" else torch.float32
    gen = torch.Generator(device="cuda").manual_seed(B)
    m = LSTM(n_in, n, device="cuda", dtype=act).requires_grad_(False)
    m.reset_parameters(gen)
    x, h = (torch.randn((B, k), device="cuda", generator=gen).to(act) for k in (n_in, n))
    st = LstmState(h=h, c=torch.randn((B, n), device="cuda", generator=gen))
    y, new = m(x, state=st)
    want, want_new = m(x[None], state=st)
    assert torch.equal(y, want[0]) and torch.equal(new.h, want_new.h) and torch.equal(new.c, want_new.c)
    assert new.h.data_ptr() != y.data_ptr()
    few, _ = m(x[:64], state=LstmState(h=h[:64], c=st.c[:64]))
    # (bfloat16: the sequence rounds the projection, values below 4 by up to 2^-7, which the four gates pass on with slopes of
    # at most 1 + 1/4 + |c| / 4 + 1/4 < 2.75, and each output is rounded by 2^-9; float32: two orders of sums of up to 6144
    # products, whose rounding errors of 2^-25 of sums below 4 add up like a random walk: 80 * 2^-23 < 1e-5)
    assert not torch.equal(few, y[:64]) and float((few.float() - y[:64].float()).abs().max()) <= (2**-5 if dtype == "bf16" else 1e-5)


@pytest.mark.parametrize("source,params", [("f32", "f32"), ("bf16", "bf16"), ("bf16", "f32"), ("f32", "bf16")])
def test_module_step_takes_the_same_way_as_the_function(source, params):
    """The module's step without views of its parameters against :func:`lstm` with prepared ones, in every combination of types, plain and
    under autocast; what it must hand on -- a gradient wanted, shapes that do not fit, CPU tensors -- does what it did."""
    dtypes = {"f32": torch.float32, "bf16": torch.bfloat16}
    B, k, n = 5, 24, 40
    gen = torch.Generator(device="cuda").manual_seed(3)
    module = lstm_mod.LSTM(k, n, device="cuda", dtype=dtypes[params])
    module.reset_parameters(gen)
    x = torch.randn((B, k), device="cuda", generator=gen).to(dtypes[source])
    h = torch.randn((B, n), device="cuda", generator=gen).to(dtypes[source])
    c = torch.randn((B, n), device="cuda", generator=gen)
    state = lstm_mod.LstmState(h=h, c=c)
    for region in (False, True):
        with torch.autocast("cuda", dtype=torch.bfloat16, enabled=region):
            with torch.no_grad():
                y, new = module(x, state=state)
                want, (want_h, want_c) = lstm_mod.lstm(x, state_h=h, state_c=c, weights=module.weights(dtypes[source]))
                back, _ = module(x, state=state, direction=-1)
            assert torch.equal(y, want) and torch.equal(new.h, want_h) and torch.equal(new.c, want_c) and torch.equal(back, y)
            assert y.dtype == want.dtype and new.h.dtype == want_h.dtype and new.c.dtype == torch.float32
    y, _ = module(x, state=state)
    assert y.requires_grad
    y.float().sum().backward()
    assert module.ff.grad is not None and bool(torch.isfinite(module.rec.grad.float()).all())
    with torch.no_grad():
        with pytest.raises(ValueError, match="state_h"):
            module(x, state=lstm_mod.LstmState(h=h[:, :-1], c=c))
        with pytest.raises(ValueError, match="in_dim"):
            module(x[:, :-1], state=state)
        with pytest.raises(ValueError, match="direction"):
            module(x, state=state, direction=2)
        with pytest.raises(RuntimeError, match="HIP"):
            module(x.cpu(), state=state)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_step_of_a_module_with_weights_of_its_own(dtype):
    """What a subclass's ``weights`` returns is what a step computes with: the bits of the same step of a plain layer with those parameters."""
    class Halved(lstm_mod.LSTM):
        def weights(self, act):
            w = super().weights(act)
            return w._replace(rec=0.5 * w.rec)

    announce("lstm_step, own weights", dtype)
    B, k, n = 5, 24, 40
    gen = torch.Generator(device="cuda").manual_seed(4)
    halved, plain = (cls(k, n, device="cuda", dtype=dtype).requires_grad_(False) for cls in (Halved, lstm_mod.LSTM))
    halved.reset_parameters(gen)
    plain.load_state_dict(halved.state_dict())
    plain.rec.mul_(0.5)
    x, h = (torch.randn((B, j), device="cuda", generator=gen).to(dtype) for j in (k, n))
    state = lstm_mod.LstmState(h=h, c=torch.randn((B, n), device="cuda", generator=gen))
    (y, new), (want, want_new) = halved(x, state=state), plain(x, state=state)
    assert torch.equal(y, want) and torch.equal(new.h, want_new.h) and torch.equal(new.c, want_new.c)
