"""The work that performance is measured on: what programs have this package do, through its public entry points.

Seven kinds of pass, each with the sizes, types and options it is used with:

  step           one decoded token of a cell: ``cell.step(x, state)``, the state fed back from token to token
  layer_step     one decoded token of an sLSTM layer: ``layer.step(x, ...)``, both states fed back
  decoder        one decoded token of a layer replayed from graphs: ``GraphedLayerDecoder.step(x)``
  forward        a sequence (prefill, evaluation) through a cell: ``cell(wx, state, reset_mask=...)``
  layer_forward  the same through a layer, its states kept for the tokens after it
  train          forward and backward through a cell: outputs, state and the gradients of input, R and bias
  layer_train    forward and backward through a layer: outputs and the gradients of input and every parameter

``docs`` is the mean length of the documents packed into a row (0: rows are not packed, no mask is passed);
``carried`` says whether the call continues from a state.
"""
import math

import torch

from xlstm_amd.cell import sLSTMCell, sLSTMCellConfig
from xlstm_amd.decode import GraphedLayerDecoder
from xlstm_amd.layer import sLSTMLayer, sLSTMLayerConfig

_DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}


def _case(kind, dtype, B, T, NH, dh, docs=0, carried=False, name=None):
    case = {"kind": kind, "dtype": dtype, "B": B, "T": T, "NH": NH, "dh": dh, "docs": docs, "carried": carried}
    return dict(case, name=name) if name else case


def listed():
    return [
        # one stream of tokens from a small cell: nothing but the latency of a call
        _case("step", "bf16", 1, 1, 4, 128, carried=True, name="step_single_stream"),
        # a serving batch of decode steps (the decode configuration of the benchmark)
        _case("step", "bf16", 256, 1, 8, 256, carried=True, name="step_batch"),
        # a layer decoded eagerly, token by token, for a handful of streams
        _case("layer_step", "bf16", 16, 1, 4, 256, carried=True, name="layer_step"),
        # a serving batch through a layer, replayed from graphs
        _case("decoder", "bf16", 256, 1, 8, 256, carried=True, name="decoder_batch"),
        # a short float32 sequence (the smallest configuration of the benchmark)
        _case("forward", "fp32", 4, 256, 4, 128, name="forward_fp32_short"),
        # packed documents (the headline configuration of the benchmark)
        _case("forward", "bf16", 16, 2048, 4, 256, docs=512, name="forward_packed"),
        # the largest heads: R does not fit a compute unit (the stress configuration of the benchmark)
        _case("forward", "bf16", 64, 4096, 4, 1024, name="forward_large_heads"),
        # a ragged prefill chunk of a layer that continues from its states, odd batch and length
        _case("layer_forward", "bf16", 7, 333, 4, 192, carried=True, name="layer_prefill_ragged"),
        # training at the headline shape
        _case("train", "bf16", 16, 2048, 4, 256, docs=512, name="train_packed"),
        # float32 training, odd sizes, a state carried over from the chunk before (truncated backpropagation)
        _case("train", "fp32", 6, 250, 4, 96, carried=True, name="train_fp32_chunk"),
        # training of the largest heads
        _case("train", "bf16", 16, 512, 4, 1024, name="train_large_heads"),
        # training of a whole layer with float32 parameters on packed documents
        _case("layer_train", "fp32", 8, 512, 4, 128, docs=192, name="layer_train_fp32"),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "step", "layer_step", "decoder", "forward", "forward", "forward", "layer_forward",
                       "train", "train", "train", "layer_train"])
    layer = kind in ("layer_step", "decoder", "layer_forward", "layer_train")
    if kind == "layer_train":
        dtype = "fp32"
    elif kind in ("decoder", "layer_step"):
        dtype = "bf16"  # a layer is served in bfloat16
    else:
        dtype = rng.choice(["bf16", "bf16", "fp32"])
    NH = rng.choice([1, 2, 3, 4, 4, 6, 8, 8, 12, 16])
    most = 1024 if dtype == "bf16" else 512
    if layer and dtype == "bf16":  # the head dims that a layer's own kernels take
        dh = rng.choice([64, 64, 128, 128, 192, 256, 256, 320, 384, 512, 768, 1024])
    elif rng.random() < 0.6:  # the usual head dims
        dh = rng.choice([d for d in (16, 32, 64, 64, 96, 128, 128, 192, 256, 256, 384, 512, 768, 1024) if d <= most])
    else:
        dh = max(2, _log_uniform(rng, 16, most) // 8) * 8
    while NH * dh > 4096:
        NH = (NH + 1) // 2
    B = _log_uniform(rng, 1, 256)
    if kind in ("step", "layer_step", "decoder"):
        return _case(kind, dtype, B, 1, NH, dh, carried=True)
    trains = kind in ("train", "layer_train")
    T = _log_uniform(rng, 8, 2048 if not trains else (1024 if dtype == "bf16" else 512))
    if trains and dh > (512 if dtype == "bf16" else 256):
        T = min(T, 384)
    # no more elements than the headline shape holds (float32: half of it)
    room = (16 * 2048 * 1024) // (2 if dtype == "fp32" else 1)
    while B * T * NH * dh > room:
        if B > 16:
            B = (B + 1) // 2
        else:
            T = (T + 1) // 2
    docs = rng.choice([0, max(4, T // 2), max(4, T // 8)])
    return _case(kind, dtype, B, T, NH, dh, docs=docs, carried=kind != "layer_train" and rng.random() < 0.5)


def _randn(case, *shape):
    return torch.randn(*shape, device="cuda", dtype=_DTYPES[case["dtype"]])


def _carried_state(case):
    """A state as the cell leaves it: y of a sigmoid times a mean of tanh values, a positive normaliser."""
    s = torch.randn(4, case["B"], case["NH"] * case["dh"], device="cuda")
    s[0].tanh_()
    s[2].abs_().add_(1.0)
    return s


def _documents(case):
    """Document starts of packed rows (lengths geometric), or None."""
    if not case["docs"]:
        return None
    mask = torch.rand(case["B"], case["T"], device="cuda") < 1.0 / case["docs"]
    if not case["carried"]:
        mask[:, 0] = True
    return mask


def prepare(case, seed):
    torch.manual_seed(seed)
    B, T, NH, dh, kind = case["B"], case["T"], case["NH"], case["dh"], case["kind"]
    D, dtype = NH * dh, _DTYPES[case["dtype"]]
    st = {"kind": kind}
    if kind in ("step", "forward", "train"):
        with torch.device("cuda"):
            cell = sLSTMCell(sLSTMCellConfig(hidden_size=D, num_heads=NH, backend="hip", recurrent_weight_init="standard"))
        st["cell"] = cell
        st["x"] = _randn(case, B, T, 4 * D)
        st["state"] = _carried_state(case) if case["carried"] else None
        st["mask"] = _documents(case)
        if kind == "step":
            cell.keep_state_fp32 = True  # the state of a decode loop stays in float32
        if kind == "train":
            st["x"].requires_grad_(True)
            # as the group norm behind a cell hands it back: [B, S, NH, DH] in memory
            st["d_out"] = _randn(case, B, T, NH, dh).transpose(1, 2)
        else:
            cell.eval()
        return st
    with torch.device("cuda"):
        layer = sLSTMLayer(sLSTMLayerConfig(embedding_dim=D, num_heads=NH, conv1d_kernel_size=4, backend="hip",
                                            recurrent_weight_init="standard"))
    layer = layer.to(dtype)
    st["layer"] = layer
    st["x"] = _randn(case, B, T, D)
    st["mask"] = _documents(case)
    if kind == "layer_train":
        st["x"].requires_grad_(True)
        st["params"] = list(layer.parameters())
        st["d_out"] = _randn(case, B, T, D)
        return st
    layer.eval()
    if kind == "decoder":
        dec = GraphedLayerDecoder(layer, B, dtype=dtype)
        dec.load_state(_randn(case, B, 3, D), _carried_state(case))
        st["decoder"] = dec
        return st
    layer.slstm_cell.keep_state_fp32 = True
    st["states"] = {}
    if case["carried"]:
        st["states"] = {"conv_state": _randn(case, B, 3, D), "slstm_state": _carried_state(case)}
        if kind == "layer_step":
            st["states"]["conv_state"] = (_randn(case, B, 4, D),)
    return st


def run(st):
    kind = st["kind"]
    if kind == "step":
        with torch.no_grad():
            h, st["state"] = st["cell"].step(st["x"], st["state"])
        return h, st["state"]
    if kind == "layer_step":
        with torch.no_grad():
            out, st["states"] = st["layer"].step(st["x"], **st["states"])
        return out, st["states"]
    if kind == "decoder":
        out = st["decoder"].step(st["x"])
        return out, st["decoder"].state()
    if kind == "forward":
        with torch.no_grad():
            return st["cell"](st["x"], st["state"], reset_mask=st["mask"])
    if kind == "layer_forward":
        with torch.no_grad():
            return st["layer"](st["x"], return_last_state=True, reset_mask=st["mask"], **st["states"])
    if kind == "train":
        cell = st["cell"]
        out, state = cell(st["x"], st["state"], reset_mask=st["mask"])
        grads = torch.autograd.grad(out, (st["x"], *cell.parameters()), st["d_out"])
        return out, state, grads
    out = st["layer"](st["x"], reset_mask=st["mask"])
    grads = torch.autograd.grad(out, (st["x"], *st["params"]), st["d_out"])
    return out, grads


def work(case):
    B, T, NH, dh, kind = case["B"], case["T"], case["NH"], case["dh"], case["kind"]
    D = NH * dh
    e = 2 if case["dtype"] == "bf16" else 4
    rows = B * T
    state = 16 * B * D
    contraction = 8 * rows * D * dh  # R.y of the four gates, and likewise the four projections of a layer
    weights = 4 * D * dh
    mask = rows if case["docs"] else 0
    if kind in ("step", "forward"):
        read = 4 * rows * D * e + (state if case["carried"] else 0) + weights * (e if kind == "step" else 4) + 16 * D + mask
        written = rows * D * e + (state if kind == "step" else 4 * B * D * e)
        return {"bytes": read + written, "flops": contraction}
    if kind == "train":
        read = 4 * rows * D * e + rows * D * e + (state if case["carried"] else 0) + weights * 4 + 16 * D + mask
        written = rows * D * e + 4 * B * D * e + 4 * rows * D * e + weights * 4 + 16 * D
        return {"bytes": read + written, "flops": 3 * contraction}
    parameters = (2 * weights + 4 * D + 6 * D) * e  # R, projections, bias, convolution, norm
    if kind == "layer_train":
        return {"bytes": 4 * rows * D * e + mask + 2 * parameters, "flops": 6 * contraction}
    states = (2 if case["carried"] else 1) * (state + 3 * B * D * e)
    return {"bytes": 2 * rows * D * e + states + parameters + mask, "flops": 2 * contraction}


def tolerance(case):
    # float32: sums of float32 products through a recurrence of up to thousands of steps.  bfloat16: hidden states and
    # gate deltas are rounded to 8 bits every step, outputs once more.
    return {"rel": 2e-5, "max": 2e-3} if case["dtype"] == "fp32" else {"rel": 1e-2, "max": 0.3}
