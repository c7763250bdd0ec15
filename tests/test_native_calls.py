"""The host side of a layer in native code, on the CPU: what a map keeps of a call survives copies of the map, and what the
extension hands to the library.  The extension runs in a process of its own beside a library of stubs, on tensors over host memory that
say they are on a GPU (they are only ever described, never read)."""
import copy
import ctypes
import os
import shutil
import subprocess
import sys

import pytest
import torch

from pcengine_amd import _lib, backend, build

KV = 8


def plain_map():
    """A 2x2x2 stride-2 map of four pairs, as the builds leave it."""
    i32 = lambda n: torch.arange(n, dtype=torch.int32)
    km = backend.KernelMap(ks=(2, 2, 2), stride=(2, 2, 2), pad=(0, 0, 0), subm=False, n_in=4, n_out=3, kv=KV, M=4, qsum=128, imap=i32(4),
                           omap=i32(4), knnz=i32(KV), kpos=i32(KV + 1), qkpos=i32(KV + 1), out_coords=torch.zeros((3, 4), dtype=torch.int32),
                           icsr=i32(5), icode=i32(4), ocsr=i32(4), ocode=i32(4), islot=i32(4), oslot=i32(4))
    km.kpos_host = (_lib.c_int32 * (KV + 1))(*range(100, 100 + KV + 1))
    km.qkpos_host = (_lib.c_int32 * (KV + 1))(*range(200, 200 + KV + 1))
    return km


@pytest.mark.parametrize("how", [copy.deepcopy, copy.copy])
def test_copies_of_a_map_read_their_own_host_arrays(how):
    km = plain_map()
    assert backend._lay_out(km, backend.DATAFLOW_FDS, torch.Size((KV, 32, 48)), torch.float32, False, True)
    other = how(km)
    addresses = {ctypes.addressof(a) for a in (km.kpos_host, km.qkpos_host, other.kpos_host, other.qkpos_host)}
    for _, view, _, _, _ in other.__dict__.get("_calls", {}).values():
        assert not any(isinstance(v, int) and v in addresses for v in view)
        host = [v for v in view if isinstance(v, ctypes.Array)]
        assert len(host) == 2 and host[0] is other.kpos_host and host[1] is other.qkpos_host


STUB = r"""
#include <dlfcn.h>
#include <stdint.h>
int calls, held_lock, kpos_last, qkpos_last;
static int call(void) {
  int (*check)(void) = (int (*)(void))dlsym(RTLD_DEFAULT, "PyGILState_Check");
  ++calls;
  if (check && check()) ++held_lock;
  return 0;
}
int pce_conv_fwd_oso() { return call(); }
int pce_conv_fwd_osb() { return call(); }
int pce_conv_fwd_os() { return call(); }
int pce_conv_fwd_os_parts() { return call(); }
int pce_conv_fwd_dense() { return call(); }
int64_t pce_bn_workspace_bytes() { return 256; }
int pce_bn_forward() { return call(); }
int pce_bn_backward() { return call(); }
int pce_conv_wgrad() { return call(); }
int pce_conv_fwd_fds(const void *in, const void *w, const void *wp, void *out, int32_t dtype, int64_t n_in, int64_t n_out, int32_t c_in,
                     int32_t c_out, int32_t kv, int32_t mid, const int32_t *imap, const int32_t *omap, const int32_t *oslot,
                     const int32_t *kpos, const int32_t *qkpos, const int32_t *kpos_host, const int32_t *qkpos_host) {
  kpos_last = kpos_host[kv];
  qkpos_last = qkpos_host[kv];
  return call();
}
"""

CHILD = r"""
import copy, ctypes, gc, importlib.util, os, sys
import torch
from pcengine_amd import _lib, backend
from tests.test_native_calls import KV, plain_map
torch.cuda._lazy_init = lambda: None
backend._stream = lambda device: 0


class Managed(ctypes.Structure):     # DLManagedTensor of dlpack.h
    _fields_ = [("data", ctypes.c_void_p), ("device_type", ctypes.c_int), ("device_id", ctypes.c_int), ("ndim", ctypes.c_int),
                ("code", ctypes.c_uint8), ("bits", ctypes.c_uint8), ("lanes", ctypes.c_uint16), ("shape", ctypes.POINTER(ctypes.c_int64)),
                ("strides", ctypes.POINTER(ctypes.c_int64)), ("byte_offset", ctypes.c_uint64), ("ctx", ctypes.c_void_p),
                ("deleter", ctypes.c_void_p)]


capsule = ctypes.pythonapi.PyCapsule_New
capsule.restype, capsule.argtypes = ctypes.py_object, [ctypes.c_void_p, ctypes.c_char_p, ctypes.c_void_p]
alive = []


def on_gpu(t):
    code, bits = {torch.float16: (2, 16), torch.float32: (2, 32), torch.int32: (0, 32), torch.uint8: (1, 8)}[t.dtype]
    dims = (ctypes.c_int64 * t.dim())(*t.shape), (ctypes.c_int64 * t.dim())(*t.stride())
    m = Managed(t.data_ptr(), 10, 0, t.dim(), code, bits, 1, dims[0], dims[1], 0, None, None)
    alive.append((m, dims, t))
    return torch._C._from_dlpack(capsule(ctypes.addressof(m), b"dltensor", None))


where = sys.argv[1]
stub = ctypes.CDLL(os.path.join(where, "libpcengine_amd.so"))
spec = importlib.util.spec_from_file_location("_host", os.path.join(where, "_host.so"))
host = importlib.util.module_from_spec(spec)
spec.loader.exec_module(host)
_lib.host = lambda: host
for name in _lib._NATIVE:
    setattr(_lib, name, getattr(host, name))
seen = lambda name: ctypes.c_int.in_dll(stub, name).value
lib = torch.library.Library("aten", "IMPL")        # memory of outputs
lib.impl("empty.memory_format", lambda size, **kw: on_gpu(torch.zeros(size, dtype=kw["dtype"], device="cpu")), "CUDA")

f32 = lambda *shape: on_gpu(torch.zeros(shape))
km = plain_map()
for name in ("imap", "omap", "kpos", "qkpos", "icsr", "icode", "ocsr", "ocode", "islot", "oslot"):
    setattr(km, name, on_gpu(getattr(km, name)))
run = lambda m: backend.conv_forward(f32(4, 32), f32(KV, 32, 48), m, backend.DATAFLOW_FDS, buffer=f32(4 * 48), out=f32(3, 48))

# a copy of the map, once the map it was made from is gone
run(km)
assert (seen("kpos_last"), seen("qkpos_last")) == (100 + KV, 200 + KV), "the layer did not run natively"
other = copy.deepcopy(km, {id(t): t for t in km.__dict__.values() if torch.is_tensor(t)})
other.kpos_host[KV], other.qkpos_host[KV] = 7, 8
run(other)
assert (seen("kpos_last"), seen("qkpos_last")) == (7, 8), (seen("kpos_last"), seen("qkpos_last"))

# other Python threads may run while the library is called
held, calls = seen("held_lock"), seen("calls")
x = f32(4, 48)
assert torch.is_tensor(backend.dense_forward(x, f32(48, 40)))
y = backend.bn_forward(x, None, None, None, None, True, 0.1, 1e-5)
assert len(backend.bn_backward(x, x, None, y[1], y[2], True)) == 3
assert backend.conv_wgrad(f32(4, 32), f32(3, 48), km).shape == (KV, 32, 48)
assert seen("calls") == calls + 4, "a call did not run natively"
assert seen("held_lock") == 0, f"{seen('held_lock')} of {seen('calls')} calls held the interpreter's lock"
"""


def test_calls_of_the_extension(tmp_path):
    if not os.path.exists(build.HOST_PATH):
        build.build(force=True)
    shutil.copy(build.HOST_PATH, tmp_path / "_host.so")
    (tmp_path / "stub.c").write_text(STUB)
    subprocess.run(["gcc", "-D_GNU_SOURCE", "-shared", "-fPIC", "-w", "-o", str(tmp_path / "libpcengine_amd.so"), str(tmp_path / "stub.c"), "-ldl"], check=True)
    child = subprocess.run([sys.executable, "-c", CHILD, str(tmp_path)], cwd=build.ROOT, capture_output=True, text=True, timeout=300)
    assert child.returncode == 0, child.stderr[-3000:]


def test_an_extension_of_another_torch_is_refused(tmp_path, monkeypatch):
    if not os.path.exists(build.HOST_PATH):
        build.build(force=True)
    with open(build.HOST_PATH, "rb") as f:
        built = f.read()
    version = torch.__version__.encode()
    other = tmp_path / "_host.so"
    other.write_bytes(built.replace(b"for torch " + version, b"for torch " + b"9" * len(version)))
    for module in (_lib, build):
        monkeypatch.setattr(module, "HOST_PATH", str(other))
    monkeypatch.setattr(_lib, "_host", None)
    assert not build.up_to_date()
    with pytest.raises(_lib.PCEError, match="another torch"):
        _lib.host()
