"""CPU tests of the host-side mirror of the reference cell interface (no kernels run)."""
import dataclasses

import pytest
import torch

from xlstm_amd.cell import ParameterProxy, sLSTMCell, sLSTMCell_hip, sLSTMCellConfig


def _cell(**kw):
    cfg = sLSTMCellConfig(hidden_size=kw.pop("hidden_size", 64), num_heads=kw.pop("num_heads", 4), **kw)
    return sLSTMCell(cfg, skip_backend_init=True)


def test_backend_switch():
    assert isinstance(_cell(), sLSTMCell_hip)
    with pytest.raises(RuntimeError, match="unknown backend"):
        sLSTMCell(sLSTMCellConfig(hidden_size=64, backend="nope"))


def test_config_defaults_match_reference_fields():
    # field names and defaults of xlstm/blocks/slstm/cell.py:61-119 (backend default aside)
    cfg = sLSTMCellConfig(hidden_size=128)
    d = dataclasses.asdict(cfg)
    for k, v in dict(num_heads=4, num_states=4, function="slstm", bias_init="powerlaw_blockdependent",
                     recurrent_weight_init="zeros", num_gates=4, input_shape="BSGNH", output_shape="BNSH",
                     dtype="bfloat16", dtype_b="float32", enable_automatic_mixed_precision=True).items():
        assert d[k] == v, k
    assert cfg.dtype_r == "bfloat16" and cfg.dtype_s == "bfloat16" and cfg.dtype_a == "float32"
    assert cfg.head_dim == 32 and cfg.input_dim == 512


def test_hidden_size_must_divide():
    with pytest.raises(ValueError, match="must be divisible"):
        _cell(hidden_size=66, num_heads=4)


def test_layout_round_trips():
    # the doctests of cell.py:623-626,646-649 for the hip layouts
    cell = _cell(hidden_size=64, num_heads=2, recurrent_weight_init="standard", bias_init="standard")
    rk, b = cell._recurrent_kernel, cell._bias
    assert torch.equal(cell._recurrent_kernel_ext2int(cell._recurrent_kernel_int2ext(rk)), rk)
    assert torch.equal(cell._bias_ext2int(cell._bias_int2ext(b)), b)
    assert tuple(cell.recurrent_kernel.shape) == (2, 32, 4, 32)
    assert tuple(cell.bias.shape) == (2, 4, 32)


def test_internal_layout_is_k_contiguous_vanilla_layout():
    cell = _cell(hidden_size=32, num_heads=2, recurrent_weight_init="standard")
    ext = cell.recurrent_kernel[:]
    NH, dh = 2, 16
    for h, d, g, a in [(0, 3, 1, 5), (1, 15, 3, 0), (1, 0, 0, 15)]:
        assert cell._recurrent_kernel_[h, g * dh + a, d] == ext[h, d, g, a]
    bext = cell.bias[:]
    for h, g, a in [(0, 1, 3), (1, 3, 15)]:
        assert cell._bias_[h * 4 * dh + g * dh + a] == bext[h, g, a]


def test_inits_closed_forms():
    cell = _cell(hidden_size=64, num_heads=4)  # defaults: zeros R, power-law forget bias
    assert torch.count_nonzero(cell.recurrent_kernel[:]) == 0
    b = cell.bias[:]
    dh = 16
    want = -(-5.0 + 12.0 * (torch.arange(dh) / (dh - 1)) ** 0.3)
    for h in range(4):
        assert torch.allclose(b[h, 1], want)
        assert torch.count_nonzero(b[h, [0, 2, 3]]) == 0
    cell = _cell(hidden_size=64, num_heads=4, bias_init="small_init", recurrent_weight_init="standard")
    b = cell.bias[:]
    assert torch.allclose(b[2, 1], torch.linspace(3.0, 6.0, dh))
    r = cell.recurrent_kernel[:]
    assert r.abs().max() <= 1 / 8 and r.std() > 0.05  # U(+-1/sqrt(64))
    blockdep = sLSTMCell(sLSTMCellConfig(hidden_size=64, _block_idx=3, _num_blocks=7), skip_backend_init=True)
    want = -(-5.0 + 12.0 * (torch.arange(dh) / (dh - 1)) ** (0.3 + 1.3 * 0.5))
    assert torch.allclose(blockdep.bias[0, 1], want)


def test_proxy_setitem_writes_internal_layout():
    cell = _cell(hidden_size=32, num_heads=2)
    cell.recurrent_kernel[1, 2, 3, 4] = 7.0
    assert cell._recurrent_kernel_[1, 3 * 16 + 4, 2] == 7.0
    assert isinstance(cell.recurrent_kernel, ParameterProxy)


def test_permute_output_shapes():
    # shapes documented at cell.py:355-362
    for shape, want in (("SBH", (5, 3, 16)), ("BSH", (3, 5, 16)), ("BNSH", (3, 2, 5, 8)), ("SBNH", (5, 3, 2, 8))):
        cell = _cell(hidden_size=16, num_heads=2, output_shape=shape)
        assert tuple(cell._permute_output(torch.zeros(5, 3, 16)).shape) == want


def test_bad_input_size_and_cpu_tensor_fail_loudly():
    cell = _cell(hidden_size=64, num_heads=4)
    with pytest.raises(AssertionError, match="Input size mismatch"):
        cell(torch.zeros(1, 1, 255))
    with pytest.raises(ValueError, match="no CPU path"):
        with torch.no_grad():
            cell(torch.zeros(1, 1, 256))
    with pytest.raises(AssertionError, match="state must be"):
        with torch.no_grad():
            cell(torch.zeros(1, 1, 256), torch.zeros(4, 2, 64))


def test_state_dict_names_match_reference():
    assert set(_cell().state_dict().keys()) == {"_recurrent_kernel_", "_bias_"}


def test_reference_checkpoint_layouts_convert_to_hip():
    """Internal tensors as the reference's vanilla and cuda cells store them (fixture written from
    those classes) land in the hip cell with the same EXTERNAL view."""
    import os

    import numpy as np
    import torch

    from xlstm_amd.cell import reference_cell_params_to_hip, reference_state_dict_to_hip, sLSTMCell, sLSTMCellConfig

    z = np.load(os.path.join(os.path.dirname(__file__), "golden", "ckpt_layouts.npz"))
    NH = int(z["num_heads"])
    r_ext, b_ext = torch.from_numpy(z["r_ext"]), torch.from_numpy(z["b_ext"])
    for backend in ("vanilla", "cuda"):
        cell = sLSTMCell(sLSTMCellConfig(hidden_size=r_ext.shape[0] * r_ext.shape[1], num_heads=NH, backend="hip",
                                         dtype="float32"), skip_backend_init=True)
        sd = {"slstm_cell._recurrent_kernel_": torch.from_numpy(z[f"r_{backend}"]),
              "slstm_cell._bias_": torch.from_numpy(z[f"b_{backend}"]), "other.weight": torch.ones(2)}
        conv = reference_state_dict_to_hip(sd, backend, NH)
        assert conv["other.weight"] is sd["other.weight"]
        cell.load_state_dict({"_recurrent_kernel_": conv["slstm_cell._recurrent_kernel_"],
                              "_bias_": conv["slstm_cell._bias_"]})
        assert torch.equal(cell.recurrent_kernel[:], r_ext), backend
        assert torch.equal(cell.bias[:], b_ext), backend
    # the two source layouts really differ from each other (the fixture is not vacuous)
    assert z["r_vanilla"].shape != z["r_cuda"].shape and not np.array_equal(z["b_vanilla"], z["b_cuda"])
    import pytest
    with pytest.raises(ValueError):
        reference_cell_params_to_hip(torch.from_numpy(z["r_cuda"]), torch.from_numpy(z["b_cuda"]), "vanilla", NH)
    with pytest.raises(ValueError):
        reference_cell_params_to_hip(torch.from_numpy(z["r_cuda"]), torch.from_numpy(z["b_cuda"]), "triton", NH)


def test_cell_can_be_copied_and_pickled():
    """copy.deepcopy / pickle of a cell (torch does it for EMA copies, DDP, checkpoints of whole modules): the
    parameter proxies follow the copy, the per-cell runtime objects (workspaces, events, decode plan) do not."""
    import copy
    import pickle

    import torch

    from xlstm_amd.cell import sLSTMCell, sLSTMCellConfig

    c = sLSTMCell(sLSTMCellConfig(hidden_size=64, num_heads=4, backend="hip", recurrent_weight_init="standard"),
                  skip_backend_init=True)
    for other in (copy.deepcopy(c), pickle.loads(pickle.dumps(c))):
        assert other._rt is not c._rt and other.recurrent_kernel.module is other
        assert torch.equal(other.recurrent_kernel[:], c.recurrent_kernel[:]) and torch.equal(other.bias[:], c.bias[:])
        other.bias[0, 1] = torch.zeros(16)
        assert not torch.equal(other.bias[:], c.bias[:])


def test_the_choice_of_the_training_path_is_by_the_call_alone(monkeypatch):
    """Sizes, types and the cell's own setting; not what has become of a function of the package."""
    from xlstm_amd import cell as cell_module

    cell = _cell(hidden_size=512, num_heads=2)
    short, long = torch.zeros(1, 8, 2048), torch.zeros(1, 400, 2048)
    for watch in (False, True):
        if watch:
            plain = cell_module.F_hip.slstm_backward
            monkeypatch.setattr(cell_module.F_hip, "slstm_backward", lambda *a, **kw: plain(*a, **kw))
        assert cell._trains_natively(short) and cell._trains_natively(long) and cell._trains_natively(short.bfloat16())
        assert not cell._trains_natively(long.bfloat16())  # (row tiles of 4 rows x 64 units, forward and backward)
    cell.keep_backward_coefficients = False
    assert not cell._trains_natively(short)


def test_a_cell_in_a_cycle_is_collected():
    """A hook on a parameter whose closure refers to the module: a cycle through the native host path's reference to the
    cell's parameters, which the collector has to see."""
    import gc
    import weakref

    from xlstm_amd import _lib

    cell = _cell(hidden_size=16, num_heads=2)
    native = cell._native()
    assert gc.is_tracked(native) and cell._parameters in gc.get_referents(native)
    cell._bias_.register_hook(lambda grad, cell=cell: grad)
    gone = weakref.ref(cell)
    del cell, native
    gc.collect()
    assert gone() is None
    # a path without parameters (as the collector leaves one to finalizers): nothing runs, nothing crashes
    path = _lib.host().CellPath({}, 2, 8)
    x = torch.zeros(1, 3, 64)
    assert path.step(x[:, :1], x, None, None, None, None, None, False) is None and path.poll(False) is False


_COUNTER = r"""
#include <dlfcn.h>
static int thrown;
void __cxa_throw(void *object, void *type, void (*destructor)(void *)) {
  ++thrown;
  ((void (*)(void *, void *, void (*)(void *)))dlsym(dlopen("libstdc++.so.6", RTLD_NOW), "__cxa_throw"))(object, type, destructor);
}
int count_thrown(void) { int n = thrown; thrown = 0; return n; }
"""

_CALLS = r"""
import ctypes, sys
counter = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)  # (in front of every library that throws)
import torch
from xlstm_amd import _lib
from xlstm_amd.cell import sLSTMCell, sLSTMCellConfig
from xlstm_amd.layer import sLSTMLayer, sLSTMLayerConfig

host = _lib.host()

def layer_calls(dtype=torch.bfloat16, dh=64, T=3, hook=False, **kw):
    layer = sLSTMLayer(sLSTMLayerConfig(embedding_dim=2 * dh, num_heads=2, backend="hip", **kw)).to(dtype)
    if hook:
        layer.slstm_cell.register_forward_hook(lambda *a: None)
    x = torch.zeros(2, T, 2 * dh, dtype=dtype)
    with torch.no_grad():
        native = layer.slstm_cell._native()
        assert host.layer_forward(layer, native, x, None, None, True, None) is None
        assert host.layer_step(layer, native, x[:, :1], None, torch.zeros(4, 2, 2 * dh), None, None, None, None, None) is None

def cell_calls(x, state=None, mask=None, **kw):
    cell = sLSTMCell(sLSTMCellConfig(hidden_size=32, num_heads=2, backend="hip", **kw))
    native = cell._native()
    for grad in (False, True):
        with torch.set_grad_enabled(grad):
            assert native.forward(x, state, mask, cell.config, False) is None
            assert native.train(x, state, mask, cell.config, False, 1 << 40) is None
            assert native.step(x, state, mask, None, None, None, cell.config, False) is None

try:  # (an error of the library's own throws: the counter counts)
    torch.empty(1).reshape(2)
except RuntimeError:
    pass
assert counter.count_thrown() > 0
layer_calls(), layer_calls(torch.float32), layer_calls(dh=48), layer_calls(T=1), layer_calls(conv1d_kernel_size=0), layer_calls(dropout=0.5)
layer_calls(conv1d_kernel_size=6), layer_calls(group_norm_weight=False), layer_calls(output_shape="SBH"), layer_calls(hook=True)
x = torch.zeros(3, 4, 128)
state = torch.zeros(4, 3, 32)
cell_calls(x), cell_calls(x.half()), cell_calls(x.bfloat16(), state.bfloat16()), cell_calls(x[:, :1], state), cell_calls(x, state, torch.zeros(3, 4))
cell_calls(x.double(), input_shape="SBGNH"), cell_calls(x[0]), cell_calls(x[:, :1], state, input_shape="SBGNH"), cell_calls(x[:, :0])
cell_calls(x, output_shape="nope"), cell_calls(x, state, 3), cell_calls(x, "state")
print("thrown", counter.count_thrown())
"""


def test_calls_of_the_general_path_cost_no_exception(tmp_path):
    """Half precision, other head dims, no convolution, dropout, one-token calls, other layouts: the native host path says
    that it does not cover them by a return value."""
    import os
    import shutil
    import subprocess
    import sys

    from tests.conftest import ROOT

    if shutil.which("gcc") is None:
        pytest.skip("needs a C compiler")
    source, counter = tmp_path / "counter.c", tmp_path / "libcounter.so"
    source.write_text(_COUNTER)
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-w", "-o", str(counter), str(source), "-ldl"], check=True)
    res = subprocess.run([sys.executable, "-c", _CALLS, str(counter)], cwd=ROOT, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True,
                         timeout=300, env=dict(os.environ, PYTHONPATH=ROOT))
    assert res.returncode == 0 and "thrown 0" in res.stdout, res.stdout
