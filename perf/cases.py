"""
The calls by which the speed of this package is judged: what its users do with it, through its public entry points.

Five kinds of calls:

``op``       the forward op as a torch operator on gates projected before (``make_op(NativeLstm2)``), one direction
``pair``     the two directions of a bidirectional layer as one call (``native_lstm2_multi``)
``step``     one step of a recurrent decoder: the :class:`LSTM` module on ``[B, in]``, as in a search loop
``layer``    the :class:`LSTM` module on whole sequences: inference, or a training step
``encoder``  the :class:`BlstmEncoder`: inference, or a training step

Sequences are right-padded with lengths uniform in [T/2, T] where ``ragged`` (the longest fills the batch), as batches of
speech or text are; the lengths lie on the GPU.
"""

import math

import torch

from returnn_amd import native_op
from returnn_amd.lstm import LSTM, BlstmEncoder, LstmState
from returnn_amd.torch_native_op import make_op, native_lstm2_multi

_DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16}


def listed():
    return [
        # a small layer on short sequences: launches and the way to them are all there is
        {"name": "op_small", "kind": "op", "T": 32, "B": 4, "n": 64, "dtype": "f32", "ragged": False, "step": 1},
        # one step of a decoder in beam search (beam 12), called once per output label
        {"name": "decode_step", "kind": "step", "B": 12, "in_dim": 512, "n": 1024, "dtype": "bf16"},
        # float32 forward of a middle-sized layer, ragged batch
        {"name": "op_f32", "kind": "op", "T": 500, "B": 64, "n": 512, "dtype": "f32", "ragged": True, "step": 1},
        # the recurrences of a bidirectional layer of a speech encoder (the repository's headline workload)
        {"name": "pair_bf16", "kind": "pair", "T": 1000, "B": 32, "n": 1024, "dtype": "bf16", "ragged": True},
        # one long utterance, recognised by itself
        {"name": "op_single_sequence", "kind": "op", "T": 4000, "B": 1, "n": 1024, "dtype": "bf16", "ragged": False, "step": 1},
        # a layer whose recurrent weights do not fit on the chip
        {"name": "op_wide", "kind": "op", "T": 200, "B": 16, "n": 4096, "dtype": "bf16", "ragged": False, "step": 1},
        # scoring many sequences at once
        {"name": "op_large_batch", "kind": "op", "T": 200, "B": 256, "n": 1024, "dtype": "bf16", "ragged": True, "step": -1},
        # a layer whose width is no power of two, and an odd batch of ragged sequences
        {"name": "layer_odd_width", "kind": "layer", "T": 333, "B": 11, "in_dim": 200, "n": 1000, "dtype": "bf16", "ragged": True,
         "train": False, "step": -1},
        # training of a language model's layer: wide, truncated sequences
        {"name": "layer_train", "kind": "layer", "T": 64, "B": 64, "in_dim": 1024, "n": 2048, "dtype": "bf16", "ragged": True,
         "train": True, "step": 1},
        # the reference's own training benchmark: five bidirectional layers of 500, chunks of 50 frames, 40 of them
        {"name": "encoder_train_chunks", "kind": "encoder", "T": 50, "B": 40, "in_dim": 80, "n": 500, "layers": 5, "dtype": "f32",
         "ragged": False, "train": True},
        # a speech encoder of six bidirectional layers: recognition
        {"name": "encoder_forward", "kind": "encoder", "T": 1000, "B": 32, "in_dim": 80, "n": 1024, "layers": 6, "dtype": "bf16",
         "ragged": True, "train": False},
        # the same encoder in training
        {"name": "encoder_train", "kind": "encoder", "T": 1000, "B": 32, "in_dim": 80, "n": 1024, "layers": 6, "dtype": "bf16",
         "ragged": True, "train": True},
    ]  # fmt: skip


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    """Layer widths: multiples of 64 or of 32 as most configurations have them, and any others."""
    n = _log_int(rng, lo, hi)
    unit = rng.choice((64, 32, 1, 1))
    return max(unit, n // unit * unit)


def draw(rng):
    kind = rng.choice(("op", "op", "pair", "step", "layer", "layer", "encoder", "encoder"))
    while True:
        case = {"kind": kind, "n": _width(rng, 32, 4096 if kind == "op" else 2048), "B": _log_int(rng, 1, 256), "dtype": rng.choice(("f32", "bf16"))}
        if kind == "step":
            case["in_dim"] = _width(rng, 32, 2048)
            return case
        case["T"] = _log_int(rng, 8, 2000)
        case["ragged"] = rng.random() < 0.7
        if kind in ("op", "layer"):
            case["step"] = rng.choice((1, -1))
        if kind in ("layer", "encoder"):
            case["in_dim"] = _width(rng, 40, 2048)
            case["train"] = rng.random() < 0.5
        if kind == "encoder":
            case["layers"] = rng.randint(1, 6)
        # no more than the largest listed case: in arithmetic (float32's rate is a fraction of bf16's), memory and time steps
        w = work(case)
        rows = case["T"] * case["B"] * case.get("layers", 1) * (2 if kind in ("pair", "encoder") else 1)
        steps = case["T"] * case.get("layers", 1) * (3 if case.get("train") else 1) * max(1.0, case["n"] / 1024)
        if w["flops"] * (8 if case["dtype"] == "f32" else 1) < 6e12 and rows * case["n"] < 2e8 and steps < 6000:
            return case


def _uniform(shape, limit, dtype, gen):
    return torch.empty(shape, device="cuda").uniform_(-limit, limit, generator=gen).to(dtype)


def _normal(shape, std, dtype, gen):
    return (torch.randn(shape, device="cuda", generator=gen) * std).to(dtype)


def _lengths(case, gen):
    T, B = case["T"], case["B"]
    if not case["ragged"]:
        return torch.full((B,), T, dtype=torch.int64, device="cuda")
    lens = torch.randint(max(1, T // 2), T + 1, (B,), device="cuda", generator=gen)
    lens[0] = T
    return lens


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    act = _DTYPES[case["dtype"]]
    kind, B, n = case["kind"], case["B"], case["n"]
    state = {"case": case}
    if kind in ("op", "pair"):
        T = case["T"]
        lens = _lengths(case, gen)
        mask = (torch.arange(T, device="cuda")[:, None] < lens[None, :]).to(torch.float32)
        calls = []
        for step in (case["step"],) if kind == "op" else (1, -1):
            X = _normal((T, B, 4 * n), 0.1, act, gen)
            W = _uniform((n, 4 * n), 1.0 / math.sqrt(n), act, gen)
            y0, c0 = _normal((B, n), 0.01, act, gen), _normal((B, n), 0.01, torch.float32, gen)
            calls.append((X, W, y0, c0, mask, 0, step))
        state["calls"] = calls
        state["op"] = make_op(native_op.NativeLstm2)
        return state
    train = case.get("train", False)
    if kind == "encoder":
        m = BlstmEncoder(case["in_dim"], n, case["layers"], device="cuda", dtype=act)
    else:
        m = LSTM(case["in_dim"], n, device="cuda", dtype=act)
    m.reset_parameters(gen)
    m.requires_grad_(train)
    state["module"] = m
    if kind == "step":
        # in the middle of a sequence: the state of the step before
        state["x"] = _normal((B, case["in_dim"]), 1.0, act, gen)
        state["state"] = LstmState(h=_normal((B, n), 0.3, act, gen), c=_normal((B, n), 0.5, torch.float32, gen))
        return state
    T = case["T"]
    state["x"] = _normal((T, B, case["in_dim"]), 1.0, act, gen).requires_grad_(train)
    state["lens"] = _lengths(case, gen) if case["ragged"] else None
    if train:
        state["dy"] = _normal((T, B, (2 if kind == "encoder" else 1) * n), 1.0 / math.sqrt(T * B), act, gen)
    if kind == "layer":
        state["state"] = m.default_initial_state(batch_dims=(B,))
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "op":
        return state["op"](*state["calls"][0])
    if kind == "pair":
        return native_lstm2_multi(state["calls"])
    m, x = state["module"], state["x"]
    if kind == "step":
        with torch.no_grad():
            y, st = m(x, state=state["state"])
        return y, st.h, st.c
    if not case["train"]:
        with torch.no_grad():
            if kind == "layer":
                y, st = m(x, state=state["state"], seq_lens=state["lens"], direction=case["step"])
                return y, st.h, st.c
            return m(x, seq_lens=state["lens"])
    # a training step up to the optimizer: gradients of all parameters and of the input, given the error of the output
    x.grad = None
    m.zero_grad(set_to_none=True)
    if kind == "layer":
        y, _ = m(x, state=state["state"], seq_lens=state["lens"], direction=case["step"])
    else:
        y = m(x, seq_lens=state["lens"])
    y.backward(state["dy"])
    return [y, x.grad] + [p.grad for p in m.parameters()]


def work(case):
    kind, B, n = case["kind"], case["B"], case["n"]
    T = case.get("T", 1)
    e = 4 if case["dtype"] == "f32" else 2
    # frames that belong to a sequence (padding needs no arithmetic, but is read and written)
    frames = T * B * (0.75 if case.get("ragged") else 1.0)
    if kind in ("op", "pair"):
        # per frame and sequence X and H (4n), Y (n) and, in float32, C and the mask; W and the states once
        one = T * B * (e * 9 * n + 4 * n + 4) + e * 4 * n * n + B * n * (e + 12)
        count = 1 if kind == "op" else 2
        return {"bytes": count * one, "flops": count * 8.0 * frames * n * n}
    directions = 2 if kind == "encoder" else 1
    weights = flops = 0.0
    for layer in range(case.get("layers", 1)):
        in_dim = case["in_dim"] if layer == 0 else directions * n
        weights += directions * 4 * n * (in_dim + n + 1)
        flops += directions * 8.0 * frames * n * (in_dim + n)
    activations = T * B * (case["in_dim"] + directions * n)
    if kind == "step":
        return {"bytes": e * (weights + B * (case["in_dim"] + 3 * n)) + 8.0 * B * n, "flops": flops}
    if case["train"]:  # the error of the output is read, those of input and weights are written
        return {"bytes": 2.0 * e * (weights + activations), "flops": 3 * flops}
    return {"bytes": e * (weights + activations), "flops": flops}


def tolerance(case):
    train = case.get("train", False)
    if case["dtype"] == "f32":
        return {"rel": 2e-5 if train else 1e-5}
    # stacked layers round their activations, and the errors of them, to bf16 in between
    return {"rel": 2e-2 if train or case.get("layers", 1) > 1 else 1e-2}
