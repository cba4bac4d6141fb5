"""The gates' non-linearities in float32 against 64 bits: with recurrent weights of zero, H of a frame is the non-linearity of X."""

from __future__ import annotations

import pytest
import torch

from _gpu_util import announce, get_op

pytestmark = pytest.mark.gpu

INF, NAN = float("inf"), float("nan")
# around where one formula takes over from another, and what must not come out of a range reduction as something else
EDGES = [0.0, -0.0, 0.75, -0.75, 0.7499999, -0.7500001, 1e-30, -1e-40, 16.6, -16.7, -86.9, -87.1, 88.8, 99.9, 101.0, -104.0, 3.4e38, -3.4e38, INF, -INF, NAN]


# one row per workgroup, groups on one XCD, a width that leaves no room for staging
@pytest.mark.parametrize("n", [64, 512, 2304])
@pytest.mark.parametrize("limit", [0.0, 0.2, 1.0, 4.0, 30.0, 80.0])
def test_float32_gates(n, limit):
    announce("float32 gates", n, limit)
    T, B = 3, 4
    if limit:
        X = (torch.rand(T, B, 4 * n, generator=torch.Generator().manual_seed(n), dtype=torch.float32) * 2 - 1) * limit
    else:
        X = torch.tensor(EDGES, dtype=torch.float32).repeat(T * B * 4 * n // len(EDGES) + 1)[: T * B * 4 * n].view(T, B, 4 * n)
    zero = torch.zeros(B, n, device="cuda")
    H = get_op()(X.cuda(), torch.zeros(n, 4 * n, device="cuda"), zero, zero.clone(), torch.ones(T, B, device="cuda"), 0, 1)[2].double().cpu()
    x = X.double()
    want = torch.cat([torch.tanh(x[..., :n]), torch.sigmoid(x[..., n:])], dim=-1)
    # (what left the first frame's y as NaN or infinity goes through the weights of zero into every gate of the row)
    frames = slice(0, 1) if not limit else slice(None)
    got, want = H[frames], want[frames]
    assert torch.equal(got.isnan(), want.isnan())
    # 4 ulp: e^x from the hardware and its correction 1.5 ulp, which are up to 3 of a result in the upper half of a binade, and 0.5 for each of
    # the two roundings behind it; below the normal numbers zero
    ulp = torch.exp2(torch.floor(torch.log2(want.abs().clamp(min=2.0**-126))) - 23)
    error = (got - want).abs().nan_to_num(0.0)
    allowed = torch.where(want.abs() < 2.0**-125, torch.full_like(ulp, 2.0**-125), 4 * ulp).nan_to_num(1.0)
    assert bool((error <= allowed).all()), float((error / allowed).max())


@pytest.mark.parametrize("n", [64, 512, 2304])
def test_small_results_of_sigmoid(n):
    """Down to where e^-x is no float32 any more a sigmoid is not cut off."""
    announce("float32 gates, small results", n)
    T, B = 2, 4
    X = -80.0 - 8.7228 * torch.rand(T, B, 4 * n, generator=torch.Generator().manual_seed(n), dtype=torch.float32)
    X[0, 0, n : n + 4] = torch.tensor([-87.0, -87.33655, -87.4, -88.722])
    zero = torch.zeros(B, n, device="cuda")
    H = get_op()(X.cuda(), torch.zeros(n, 4 * n, device="cuda"), zero, zero.clone(), torch.ones(T, B, device="cuda"), 0, 1)[2].cpu()
    got, want = H[..., n:].double(), torch.sigmoid(X[..., n:].double())
    # 4 ulp as above; below the normal numbers an ulp is the smallest number, and a result is rounded to it twice
    ulp = torch.exp2(torch.floor(torch.log2(want.clamp(min=2.0**-126))) - 23)
    assert bool(((got - want).abs() <= 4 * ulp).all()), float(((got - want).abs() / ulp).max())


@pytest.mark.parametrize("n", [64, 512, 2304])
def test_tanh_keeps_the_sign_of_zero(n):
    """A cell state of -0, to which a gate adds what rounds to -0, comes out as -0."""
    announce("float32 gates, signed zero", n)
    T, B = 3, 2
    X = torch.zeros(T, B, 4 * n, dtype=torch.float32)
    X[..., :n] = -1e-45  # times a sigmoid below a half: rounds to -0
    X[..., n : 2 * n] = -5.0
    X[:, 1, :n] = 1e-45
    W, y0, c0 = torch.zeros(n, 4 * n, device="cuda"), torch.zeros(B, n), torch.zeros(B, n)
    y0[0] = c0[0] = -0.0
    Y, C, _, d = get_op()(X.cuda(), W, y0.cuda(), c0.cuda(), torch.ones(T, B, device="cuda"), 0, 1)
    assert not Y.any() and not C.any()
    assert bool(torch.signbit(C[:, 0]).all()) and bool(torch.signbit(Y[:, 0]).all()) and bool(torch.signbit(d[0]).all())
    assert not torch.signbit(C[:, 1]).any() and not torch.signbit(Y[:, 1]).any()
