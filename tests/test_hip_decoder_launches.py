"""A decoder's steps launched directly against its graphs, mixed token by token: the same states and outputs whichever runs."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("B,NH,dh", [(3, 2, 64), (70, 4, 256), (33, 2, 1024)])
def test_direct_steps_and_replays_may_be_mixed(monkeypatch, B, NH, dh):
    from xlstm_amd.decode import GraphedLayerDecoder
    from xlstm_amd.layer import sLSTMLayer, sLSTMLayerConfig

    print("case decoder launches", B, NH, dh, flush=True)
    D = NH * dh
    torch.manual_seed(B)
    layer = sLSTMLayer(sLSTMLayerConfig(embedding_dim=D, num_heads=NH, backend="hip", recurrent_weight_init="standard")).to(DEV).bfloat16().eval()
    x = torch.randn(9, B, 1, D, device=DEV).bfloat16()
    ring, state = torch.randn(B, 3, D, device=DEV).bfloat16(), torch.rand(4, B, D, device=DEV) + 0.5
    decoders = [GraphedLayerDecoder(layer, B) for _ in range(2)]
    for dec in decoders:
        dec.load_state(ring, state)
    first = None
    if dh <= 512:  # (float32: PyTorch's convolution, products and norm around the cell, up to the cell's largest head)
        plain = sLSTMLayer(layer.config).to(DEV).eval()
        plain.load_state_dict(layer.state_dict())
        with torch.no_grad():
            first = plain.step(x[0].float(), conv_state=ring.float(), slstm_state=state.clone())[0]
    launch, launched = GraphedLayerDecoder._launch, []
    monkeypatch.setattr(GraphedLayerDecoder, "_launch", lambda self, t: launched.append(launch(self, t)) or launched[-1])
    replayed = decoders[0]
    for t in range(9):
        forms = {3: x[t].float(), 4: x[t].transpose(0, 1).contiguous().transpose(0, 1), 5: torch.randn(B, 2, D, device=DEV).bfloat16()[:, :1]}
        token = forms.get(t, x[t])
        if t == 6:
            token = decoders[1].out.clone()
        monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)  # (no direct launch)
        want = replayed.step(token).clone()
        monkeypatch.undo()
        monkeypatch.setattr(GraphedLayerDecoder, "_launch", lambda self, t: launched.append(launch(self, t)) or launched[-1])
        got = decoders[1].step(decoders[1].out if t == 6 else token)  # (t 6: the output fed back is read before it is written)
        if t == 0 and first is not None:  # (the layer's bfloat16 kernels: 2e-2)
            assert float((got.float() - first).norm() / first.norm()) < 2e-2
        assert torch.equal(got, want), t
        assert torch.equal(decoders[1].state()["slstm_state"], replayed.state()["slstm_state"]), t
        assert torch.equal(decoders[1].state()["conv_state"][0], replayed.state()["conv_state"][0]), t
        if t == 4:
            replayed = decoders[0]
            decoders[0].load_state(decoders[1].state()["conv_state"], decoders[1].state()["slstm_state"])
    assert launched and launched[-1] and launched.count(True) == 9
    assert not got.requires_grad
    handle = layer.dropout.register_forward_hook(lambda *_: None)  # (what the direct path leaves to the graphs)
    got, want = decoders[1].step(x[0]), decoders[0].step(x[0])
    handle.remove()
    assert not launched[-1] and torch.equal(got, want)


@pytest.mark.parametrize("B,NH,dh", [(3, 2, 64), (600, 2, 128), (70, 4, 256), (33, 2, 1024)])
def test_the_token_is_in_the_decoders_buffer(B, NH, dh):
    """``step(x)`` leaves the token in ``dec.x``: whoever holds that buffer reads it there, and ``step()`` behind it takes it
    once more."""
    from xlstm_amd.decode import GraphedLayerDecoder
    from xlstm_amd.layer import sLSTMLayer, sLSTMLayerConfig

    print("case decoder token", B, NH, dh, flush=True)
    D = NH * dh
    torch.manual_seed(B)
    layer = sLSTMLayer(sLSTMLayerConfig(embedding_dim=D, num_heads=NH, backend="hip", recurrent_weight_init="standard")).to(DEV).bfloat16().eval()
    x = torch.randn(3, B, 1, D, device=DEV).bfloat16()
    dec, twice = GraphedLayerDecoder(layer, B), GraphedLayerDecoder(layer, B)
    held = dec.x
    for token in (x[0], x[1], x[2].float()):
        got = dec.step(token).clone()
        assert torch.equal(held, token.bfloat16()) and dec.x is held
        assert torch.equal(got, twice.step(token))
        got = dec.step().clone()
        assert torch.equal(got, twice.step(token))
        assert torch.equal(held, token.bfloat16())
    held[:2].copy_(x[0][:2])  # (its producer writes a part of it)
    mixed = held.clone()
    assert torch.equal(dec.step(), twice.step(mixed))
    assert torch.equal(dec.step(x[1][:1]), twice.step(x[1][:1].expand(B, 1, D)))  # (one token for all rows)
    assert torch.equal(held, x[1][:1].expand(B, 1, D))
