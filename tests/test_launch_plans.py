"""How the engine cuts a sequence call into launches, without a GPU: the host side of the library over a stand-in for the HIP
runtime that reports a device of 256 compute units and counts launches.  Every call that is taken must find a kernel for
every slice of its heads; a call that is refused must be refused in front of its first launch."""
import os
import shutil
import subprocess
import sys

import pytest

from tests.conftest import ROOT

_RUNTIME = r"""
typedef struct { unsigned x, y, z; } dim3_;
static int launches;
int hipGetDevice(int *d) { *d = 0; return 0; }
int hipDeviceGetAttribute(int *v, int attr, int dev) { *v = 256; return 0; }
int hipFuncSetAttribute(const void *f, int attr, int v) { return 0; }
int hipGetLastError(void) { return 0; }
int __hipPushCallConfiguration(dim3_ g, dim3_ b, unsigned long lds, void *s) { return 0; }
int __hipPopCallConfiguration(dim3_ *g, dim3_ *b, unsigned long *lds, void **s) {
  g->x = g->y = g->z = b->x = b->y = b->z = 1; *lds = 0; *s = 0;
  return 0;
}
int hipLaunchKernel(const void *f, dim3_ g, dim3_ b, void **args, unsigned long lds, void *s) { ++launches; return 0; }
int count_launches(void) { int n = launches; launches = 0; return n; }
"""

_SWEEP = r"""
import ctypes, sys
runtime = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)  # (in front of the engine: its calls resolve to the stand-in)
from xlstm_amd import _lib
lib = _lib.load()

def call(bf16, NH, dh, B, T=3, coef=None):
    a = _lib.SlstmArgs()
    H = NH * dh
    a.B, a.T, a.NH, a.dh = B, T, NH, dh
    a.wx_dtype, a.r_dtype = (_lib.XS_BF16 if bf16 else _lib.XS_F32), _lib.XS_F32
    a.wx_stride_b, a.wx_stride_t = 4 * H * T, 4 * H
    a.wx, a.r, a.bias, a.h_out, a.s_out, a.workspace = (i << 40 for i in range(1, 7))  # (device addresses: never read here)
    a.workspace_bytes = lib.xs_slstm_workspace_bytes(B, T, NH, dh)
    if coef:
        return lib.xs_slstm_train_forward(ctypes.byref(a), 7 << 40, None)
    return lib.xs_slstm_forward(ctypes.byref(a))

bad, calls, several = [], 0, 0
for bf16 in (True, False):
    dims = [8, 16, 24, 40, 48, 64, 72, 96, 104, 128, 136, 192, 256, 264, 384, 512] + ([640, 768, 1024] if bf16 else [])
    for dh in dims:
        for NH in [*range(1, 41), 48, 56, 64, 72, 96, 128, 129]:
            for B in (1, 3, 4, 5, 8, 9, 16, 17, 31, 32, 33, 40, 48, 49, 64, 65, 80, 96, 97, 128, 129, 200, 256):
                for coef in (False, True):
                    rc = call(bf16, NH, dh, B, coef=coef)
                    n = runtime.count_launches()
                    calls += 1
                    several += n > 2
                    if rc != 0 or n == 0:
                        bad.append((bf16, NH, dh, B, coef, rc, n, _lib.last_error()))
print(calls, several, len(bad), bad[:5])
# a call that no kernel takes: refused, and nothing has been launched
assert call(False, 40, 520, 33) == _lib.XS_ERR_UNSUPPORTED and runtime.count_launches() == 0
assert call(True, 4, 1032, 3) == _lib.XS_ERR_UNSUPPORTED and runtime.count_launches() == 0
assert several > 1000
sys.exit(1 if bad else 0)
"""


@pytest.mark.skipif(shutil.which("gcc") is None, reason="needs a C compiler")
def test_every_slice_of_heads_finds_a_kernel(tmp_path):
    source, stand_in = tmp_path / "runtime.c", tmp_path / "libruntime.so"
    source.write_text(_RUNTIME)
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-w", "-o", str(stand_in), str(source)], check=True)
    res = subprocess.run([sys.executable, "-c", _SWEEP, str(stand_in)], cwd=ROOT, stdout=subprocess.PIPE, stderr=subprocess.STDOUT,
                         text=True, timeout=300, env=dict(os.environ, PYTHONPATH=ROOT))
    assert res.returncode == 0, res.stdout
