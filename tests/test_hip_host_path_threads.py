"""The native host path among other threads: the GIL is given up while it allocates and launches, and threads that share a
cell - one stream or several, one batch size or several - get their own results."""
import ctypes
import shutil
import subprocess
import threading

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

_PROBE = r"""
extern int PyGILState_Check(void);
static int held, calls;
int probe(void) { ++calls; held += PyGILState_Check(); return -5; }  /* (XS_ERR_UNSUPPORTED: nothing is launched) */
int probe_calls(void) { return calls; }
int probe_held(void) { return held; }
"""


def _layer(NH=2, dh=64):
    from xlstm_amd.layer import sLSTMLayer, sLSTMLayerConfig

    torch.manual_seed(dh)
    layer = sLSTMLayer(sLSTMLayerConfig(embedding_dim=NH * dh, num_heads=NH, conv1d_kernel_size=4, backend="hip",
                                        recurrent_weight_init="standard")).to(DEV, torch.bfloat16).eval()
    layer.slstm_cell.keep_state_fp32 = True
    return layer


@pytest.mark.skipif(shutil.which("gcc") is None, reason="needs a C compiler")
@pytest.mark.parametrize("entry", ["xs_slstm_step", "xs_slstm_forward_watched", "xs_slstm_train_forward", "xs_causal_conv_silu",
                                   "xs_headwise_gates", "xs_headwise_group_norm"])
def test_launches_run_without_the_gil(tmp_path, entry):
    from torch.nn.modules import module as torch_module

    from xlstm_amd import _lib
    from xlstm_amd.functional import EngineError

    print("case gil", entry, flush=True)
    source, lib = tmp_path / "probe.c", tmp_path / "libprobe.so"
    source.write_text(_PROBE)
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-o", str(lib), str(source)], check=True)
    probe = ctypes.PyDLL(str(lib))
    engine, host = _lib.load(), _lib.host()
    addresses = {name: ctypes.cast(getattr(engine, name), ctypes.c_void_p).value for name in _lib.EXPORTS}
    hooks = (EngineError, torch_module._global_forward_hooks, torch_module._global_forward_pre_hooks)
    layer = _layer()
    cell = layer.slstm_cell
    x = torch.randn(2, 4, 128, device=DEV, dtype=torch.bfloat16)
    wx = torch.randn(2, 4, 512, device=DEV, dtype=torch.bfloat16)
    tokens = [x[:, t:t + 1].contiguous() for t in range(3)]
    calls = {"xs_slstm_step": [lambda s: cell.step(wx[:, :1].contiguous(), s["slstm_state"]), lambda s: layer.step(tokens[2], **s)],
             "xs_slstm_forward_watched": [lambda s: cell(wx), lambda s: layer(x)],
             "xs_slstm_train_forward": [lambda s: cell(wx)]}.get(entry, [lambda s: layer(x), lambda s: layer.step(tokens[2], **s)])
    with torch.no_grad():
        _, states = layer.step(tokens[0], slstm_state=torch.zeros(4, 2, 128, device=DEV))  # (makes the plan)
        _, states = layer.step(tokens[1], **states)
    host.bind({**addresses, entry: ctypes.cast(probe.probe, ctypes.c_void_p).value}, *hooks)
    try:
        for call in calls:
            before = probe.probe_calls()
            with torch.set_grad_enabled(entry == "xs_slstm_train_forward"), pytest.raises(EngineError, match="error -5"):
                call(states)
            assert probe.probe_calls() == before + 1
    finally:
        host.bind(addresses, *hooks)
    assert probe.probe_held() == 0


@pytest.mark.parametrize("streams", [False, True])
def test_threads_share_a_cell(streams):
    """Sequence calls, training calls and decode steps of two batch sizes from four threads on one cell: on one stream (one
    workspace: the launches of a call stay together) and on a stream each."""
    print("case threads", streams, flush=True)
    from xlstm_amd.cell import sLSTMCell, sLSTMCellConfig

    torch.manual_seed(0)
    NH, dh, T = 2, 136, 24  # (a head is spread over 9 compute units: the calls of all threads fit an XCD at a time)
    cell = sLSTMCell(sLSTMCellConfig(hidden_size=NH * dh, num_heads=NH, backend="hip", recurrent_weight_init="standard")).to(DEV)
    cell.keep_state_fp32 = True
    xs = [torch.randn(B, T, 4 * NH * dh, device=DEV).bfloat16() for B in (3, 5, 8, 8)]

    def sequence(x):
        with torch.no_grad():
            return cell(x)

    def training(x):
        x = x.detach().requires_grad_(True)
        out, state = cell(x)
        return out, state, *torch.autograd.grad(out, x, torch.ones_like(out))

    def decode(x):
        with torch.no_grad():
            state, outs = torch.zeros(4, x.shape[0], NH * dh, device=DEV), []
            for t in range(6):
                out, state = cell.step(x[:, t:t + 1].contiguous(), state)
                outs.append(out)
        return (*outs, state)

    work = [(sequence, xs[2]), (training, xs[3]), (decode, xs[0]), (decode, xs[1])]
    want = [f(x) for f, x in work]
    torch.cuda.synchronize()
    failures = []

    def run(i):
        f, x = work[i]
        stream = torch.cuda.Stream() if streams else torch.cuda.default_stream()
        try:
            with torch.cuda.stream(stream):
                for _ in range(20):
                    got = f(x)
                    stream.synchronize()
                    if not all(torch.equal(a, b) for a, b in zip(got, want[i])):
                        failures.append((f.__name__, i))
        except Exception as e:  # noqa: BLE001  (reported by the main thread)
            failures.append((f.__name__, i, repr(e)))

    threads = [threading.Thread(target=run, args=(i,)) for i in range(len(work))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failures, failures[:5]
    cell.check_status()


@pytest.mark.parametrize("of_layer", [False, True])
def test_a_plan_replaced_while_a_step_is_looked_at(of_layer):
    """Python code that runs in the middle of a step (here an attribute of the cell's config that steps the cell with another
    batch size, as another thread may at that point): the step takes the plan of its own batch size."""
    print("case plan replaced", of_layer, flush=True)
    layer = _layer()
    cell = layer.slstm_cell
    steps = {True: lambda x, s: layer.step(x, slstm_state=s), False: cell.step}[of_layer]
    xs = [torch.randn(B, 1, 128 if of_layer else 512, device=DEV, dtype=torch.bfloat16) for B in (3, 7)]
    states = [torch.rand(4, x.shape[0], 128, device=DEV) + 0.5 for x in xs]

    class Config:
        def __init__(self, config):
            self.config, self.armed = config, False

        def __getattr__(self, name):
            if name == "output_shape" and self.armed:
                self.armed = False
                steps(xs[1], states[1])
            return getattr(self.config, name)

    with torch.no_grad():
        want = steps(xs[0], states[0])[0]
        cell.config = Config(cell.config)
        assert torch.equal(steps(xs[0], states[0])[0], want)
        cell.config.armed = True
        assert torch.equal(steps(xs[0], states[0])[0], want) and not cell.config.armed
