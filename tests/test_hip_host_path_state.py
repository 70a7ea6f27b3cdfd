"""What the native host path keeps between the calls of a cell: a workspace that a recorded graph writes, nothing of the
parameters."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _cell(NH, dh, dtype=torch.float32):
    from xlstm_amd.cell import sLSTMCell, sLSTMCellConfig

    torch.manual_seed(dh)
    cell = sLSTMCell(sLSTMCellConfig(hidden_size=NH * dh, num_heads=NH, backend="hip", recurrent_weight_init="standard"))
    return cell.to(DEV, dtype).eval()


@pytest.mark.parametrize("dh", [64, 256])
def test_bias_is_read_on_every_call(dh):
    """A bfloat16 bias written through ``.data`` keeps its version."""
    print("case bias", dh, flush=True)
    cell = _cell(2, dh, torch.bfloat16)
    x = torch.randn(3, 5, 8 * dh, device=DEV, dtype=torch.bfloat16)
    with torch.no_grad():
        cell(x)
        cell._bias_.data.add_(0.5)
        out, state = cell(x)
        other = _cell(2, dh, torch.bfloat16)
        other.load_state_dict(cell.state_dict())
        want, want_state = other(x)
    assert torch.equal(out, want) and torch.equal(state, want_state)


@pytest.mark.parametrize("warm", [False, True])
def test_workspace_of_a_graph_outlives_many_streams(warm):
    """A cell's call under capture (its first call, or behind one on the same stream), then calls on more streams than the
    cell keeps workspaces for: replays still write memory of their own."""
    print("case graph and streams", warm, flush=True)
    cell = _cell(2, 256, torch.bfloat16)
    x = torch.randn(3, 6, 8 * 256, device=DEV, dtype=torch.bfloat16)
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with torch.no_grad():
        want, want_state = _cell(2, 256, torch.bfloat16)(x)  # (loads the kernels: a cell of its own)
        torch.cuda.synchronize()
        if warm:
            with torch.cuda.stream(side):
                cell(x)
            side.synchronize()
        with torch.cuda.graph(graph, stream=side):
            out, state = cell(x)
            recorded = cell._workspace(3, x.device)
        torch.cuda.synchronize()
        ptr, size = recorded.data_ptr(), recorded.numel()
        del recorded
        for s in [torch.cuda.Stream() for _ in range(24)]:
            with torch.cuda.stream(s):
                o, _ = cell(x)
            s.synchronize()
            assert torch.equal(o, want)
        with torch.cuda.stream(side):
            held = [torch.full((size,), 0xA5, dtype=torch.uint8, device=DEV) for _ in range(8)]
        torch.cuda.synchronize()
        for _ in range(3):
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, want) and torch.equal(state, want_state)
            out.zero_()
        for t in held:
            assert t.data_ptr() != ptr and bool((t == 0xA5).all())
    cell.check_status()
