"""What the native host path keeps between the calls of a cell (the plans that recorded graphs read, nothing of the parameters),
what it gives graphs of their own, whom it calls, what it waits for and how it fails."""
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


def test_modules_put_in_the_place_of_a_layers_are_called():
    """A dropout without a rate, a wrapped cell: the layer runs them as modules."""
    from xlstm_amd.layer import sLSTMLayer, sLSTMLayerConfig

    print("case replaced modules", flush=True)
    torch.manual_seed(0)
    layer = sLSTMLayer(sLSTMLayerConfig(embedding_dim=128, num_heads=2, conv1d_kernel_size=4, backend="hip",
                                        recurrent_weight_init="standard")).to(DEV, torch.bfloat16).eval()
    x = torch.randn(2, 6, 128, device=DEV, dtype=torch.bfloat16)

    class Doubled(torch.nn.Module):
        def forward(self, y):
            return y * 2

    class Wrapped(torch.nn.Module):
        def __init__(self, cell):
            super().__init__()
            self.inner, self.calls = cell, 0

        def forward(self, *args, **kw):
            self.calls += 1
            return self.inner(*args, **kw)

    with torch.no_grad():
        want = layer(x)
        layer.dropout = torch.nn.Identity()
        assert torch.equal(layer(x), want)
        layer.group_norm.weight.data.fill_(0.25)
        layer.group_norm.eps, eps = 10.0, layer.group_norm.eps  # (the norm then sees the scale of its input)
        plain = layer(x)
        layer.dropout = Doubled()
        assert not torch.equal(layer(x), plain)
        layer.dropout, layer.group_norm.eps = torch.nn.Dropout(0.0), eps
        plain = layer(x)
        layer.slstm_cell = Wrapped(layer.slstm_cell)
        assert torch.equal(layer(x), plain) and layer.slstm_cell.calls == 1


def test_graphs_of_a_cell_have_workspaces_of_their_own():
    """Two graphs recorded on one stream, replayed on two streams at a time, beside eager calls on the stream of the capture
    (a head is spread over 9 compute units: three calls at a time fit an XCD)."""
    print("case workspaces of graphs", flush=True)
    cell = _cell(2, 136, torch.bfloat16)
    xs = [torch.randn(3, 40, 8 * 136, device=DEV, dtype=torch.bfloat16) for _ in range(3)]
    side, streams = torch.cuda.Stream(), [torch.cuda.Stream() for _ in range(2)]
    with torch.no_grad():
        want = [_cell(2, 136, torch.bfloat16)(x) for x in xs]
        torch.cuda.synchronize()
        with torch.cuda.stream(side):
            cell(xs[2])
        used = {cell._native().last_workspace().data_ptr()}
        torch.cuda.synchronize()
        graphs, outs, held = [], [], []
        for x in xs[:2]:
            graphs.append(torch.cuda.CUDAGraph())
            with torch.cuda.graph(graphs[-1], stream=side):
                outs.append(cell(x))
            held.append(cell._native().last_workspace())
            used.add(held[-1].data_ptr())
        assert len(used) == 3
        del held
        for _ in range(10):
            torch.cuda.synchronize()
            for g, s in zip(graphs, streams):
                with torch.cuda.stream(s):
                    g.replay()
            with torch.cuda.stream(side):
                got = cell(xs[2])
            torch.cuda.synchronize()
            for a, b in zip([*outs, got], want):
                assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])
            for o in outs:
                o[0].zero_()
    cell.check_status()


def test_plan_of_a_graph_outlives_other_batch_sizes():
    """A decoder's graphs, then eager steps of another batch size and of changed parameters on the same layer, with every block
    that is free given back to the driver: replays still read the R and the bias that they were recorded with."""
    from xlstm_amd.decode import GraphedLayerDecoder
    from xlstm_amd.layer import sLSTMLayer, sLSTMLayerConfig

    print("case graph and plans", flush=True)
    torch.manual_seed(0)
    layer = sLSTMLayer(sLSTMLayerConfig(embedding_dim=1024, num_heads=2, conv1d_kernel_size=4, backend="hip",
                                        recurrent_weight_init="standard")).to(DEV, torch.bfloat16).eval()
    xs = [torch.randn(4, 1, 1024, device=DEV, dtype=torch.bfloat16) for _ in range(4)]
    dec = GraphedLayerDecoder(layer, 4)
    want = [dec.step(x).clone() for x in xs]
    dec.reset()
    with torch.no_grad():
        for B in (6, 7):
            layer.step(torch.randn(B, 1, 1024, device=DEV, dtype=torch.bfloat16), slstm_state=torch.zeros(4, B, 1024, device=DEV))
        layer.slstm_cell._recurrent_kernel_.mul_(1.0)
        layer.step(xs[0], slstm_state=torch.zeros(4, 4, 1024, device=DEV))
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    for x, w in zip(xs, want):
        assert torch.equal(dec.step(x), w)


@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_first_step_of_a_cell_under_capture(dtype, masked):
    """A decode step whose first call is recorded (nothing of it has run when it returns), then eager steps in front of any
    replay, other parameters, replays."""
    print("case first step under capture", dtype, masked, flush=True)
    x = torch.randn(3, 1, 8 * 256, device=DEV, dtype=dtype)
    state = torch.rand(4, 3, 512, device=DEV) + 0.5
    mask = torch.tensor([[True], [False], [False]], device=DEV) if masked else None
    cells = [_cell(2, 256) for _ in range(2)]
    for cell in cells:
        cell.keep_state_fp32 = True
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with torch.no_grad():
        want = cells[1].step(x, state, mask)  # (loads the kernels: a cell of its own)
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=side):
            out = cells[0].step(x, state, mask)
        got = cells[0].step(x, state, mask)
        assert all(torch.equal(a, b) for a, b in zip(got, want))
        for _ in range(3):
            graph.replay()
            torch.cuda.synchronize()
            assert all(torch.equal(a, b) for a, b in zip(out, want))
            out[0].zero_()
            got = cells[0].step(x, state, mask)
            assert all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("module,method,where", [
    (module, method, where) for module, method in (("slstm_cell", "forward"), ("slstm_cell", "step"), ("dropout", "forward"))
    for where in ("instance", "class", "compiled") if (method, where) != ("step", "compiled")])
def test_methods_put_in_the_place_of_a_modules_are_called(monkeypatch, module, method, where):
    """A layer calls a ``forward`` or ``step`` that was replaced on its cell or dropout, or on their class, and a module that
    was compiled in place - behind calls that went through the native host path."""
    from xlstm_amd.layer import sLSTMLayer, sLSTMLayerConfig

    print("case replaced method", where, module, method, flush=True)
    torch.manual_seed(0)
    layer = sLSTMLayer(sLSTMLayerConfig(embedding_dim=128, num_heads=2, conv1d_kernel_size=4, backend="hip",
                                        recurrent_weight_init="standard")).to(DEV, torch.bfloat16).eval()
    layer.slstm_cell.keep_state_fp32 = True
    x = torch.randn(2, 6, 128, device=DEV, dtype=torch.bfloat16)
    calls = []

    def run():
        with torch.no_grad():
            out, states = layer(x[:, :4], return_last_state=True)
            outs = [out]
            for t in (4, 5):
                out, states = layer.step(x[:, t:t + 1].contiguous(), **states)
                outs.append(out)
        return torch.cat(outs, 1)

    want = run()
    target = getattr(layer, module)
    if where == "compiled":  # what Module.compile leaves on the module
        plain = target._call_impl
        target._compiled_call_impl = lambda *a, **kw: (calls.append(1), plain(*a, **kw))[1]
    elif where == "instance":
        plain = getattr(target, method)
        setattr(target, method, lambda *a, **kw: (calls.append(1), plain(*a, **kw))[1])
    else:
        plain = getattr(type(target), method)
        monkeypatch.setattr(type(target), method, lambda self, *a, **kw: (calls.append(1), plain(self, *a, **kw))[1])
    # (the dropout runs behind the sequence and behind every step, the cell's forward and step once per call of that kind)
    assert torch.equal(run(), want) and len(calls) == {"forward": 3 if module == "dropout" else 1, "step": 2}[method]


@pytest.mark.parametrize("trains", [False, True])
def test_out_of_memory_is_reported_as_such(trains):
    """Programs catch ``torch.OutOfMemoryError`` to go on with a smaller batch."""
    print("case out of memory", trains, flush=True)
    cell = _cell(2, 64)
    x = torch.randn(8, 4096, 512, device=DEV, requires_grad=trains)
    total = torch.cuda.get_device_properties(0).total_memory
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    large = torch.empty(2 << 30, dtype=torch.uint8, device=DEV)
    del large
    kept = torch.empty(2 << 20, dtype=torch.uint8, device=DEV)  # (a block with a tensor in it stays, whatever else of it is free)
    torch.cuda.empty_cache()
    free = torch.cuda.memory_reserved() - torch.cuda.memory_allocated()
    assert free > kept.numel()
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (1 << 20)) / total)
    try:
        with torch.set_grad_enabled(trains), pytest.raises(torch.OutOfMemoryError):
            held = [cell(x) for _ in range(64 + free // (16 << 20))]  # (16 MiB of outputs each)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    with torch.set_grad_enabled(trains):
        assert bool(torch.isfinite(cell(x)[0]).all())
    cell.check_status()


@pytest.mark.parametrize("trains", [False, True])
def test_check_status_waits_for_the_cells_own_calls(trains):
    """All of them, and not what other streams of the device run."""
    import time

    print("case check_status", trains, flush=True)
    cell = _cell(2, 64)
    x = torch.randn(2, 16384, 512, device=DEV, requires_grad=trains)  # (some 8 ms in one direction)
    a = torch.randn(8192, 8192, device=DEV, dtype=torch.bfloat16)
    others, own = torch.cuda.Event(), torch.cuda.Event()

    def busy_elsewhere():  # some 0.3 s on a stream whose hardware queue is not the current stream's
        for side in [torch.cuda.Stream() for _ in range(8)]:
            torch.cuda.synchronize()
            with torch.cuda.stream(side):
                for _ in range(400):
                    a @ a
                others.record()
            a[0].clone()
            own.record()
            own.synchronize()
            if not others.query():
                return
        pytest.skip("every stream shares the current one's hardware queue")

    with torch.set_grad_enabled(trains):
        torch.autograd.grad(cell(x)[0].sum(), x) if trains else cell(x)  # (loads the kernels)
        busy_elsewhere()
        begin = time.perf_counter()
        out, _ = cell(x)
        if trains:
            torch.autograd.grad(out, x, torch.ones_like(out))
        cell.check_status()
        waited, pending = time.perf_counter() - begin, not others.query()
        own.record()
        own.synchronize()
        rest = time.perf_counter() - begin - waited
    assert pending and waited > 4e-3 and rest < 0.5 * waited, (pending, waited, rest)
