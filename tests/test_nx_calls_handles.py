"""The handles of the host path in C (raven_amd/host_c/nx_calls.c) as Python objects, and the module as a file."""

import copy
import gc
import subprocess
import sys
import sysconfig
import weakref
from pathlib import Path

from raven_amd import build
from raven_amd import dtype as dt
from raven_amd.nx_backend import Tensor
from raven_amd.view import View

ROOT = Path(__file__).resolve().parent.parent


class Thing:
    ptr = None


def in_a_process(script):
    r = subprocess.run([sys.executable, "-c", script], cwd=ROOT, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return r.stdout.split()


def test_a_tensor_kept_by_its_context_goes_with_it():
    context = Thing()
    context.kept = Tensor(Thing(), View.create((2,)), dt.float32, context)
    ref = weakref.ref(context)
    del context
    gc.collect()
    assert ref() is None


def test_a_handle_can_be_copied():
    t = Tensor(Thing(), View.create((2, 3)), dt.float32, Thing())
    u = copy.copy(t)
    assert u is not t
    assert all(getattr(u, name) is getattr(t, name) for name in ("buffer", "view", "shape", "dtype", "context"))


def test_storage_kept_by_its_context_goes_back():
    """With stand-ins for the library, whose entry points the module holds for the whole process."""
    assert in_a_process("""
import ctypes as C, gc
from raven_amd._nxcalls import Calls, DeviceBuffer, Tensor, bind
from raven_amd import _ffi, dtype as dt
from raven_amd.nx_backend import View
def alloc(ctx, n, p):
    C.cast(p, C.POINTER(C.c_void_p))[0] = 4096
    return 0
def free(ctx, p):
    print("freed", ctx, p)
    return 0
alloc = C.CFUNCTYPE(C.c_int, C.c_void_p, C.c_size_t, C.c_void_p)(alloc)
free = C.CFUNCTYPE(C.c_int, C.c_void_p, C.c_void_p)(free)
bind({name: C.cast({"nxh_free": free}.get(name, alloc), C.c_void_p).value for name in _ffi.SIGNATURES})
class Context(Calls):
    pass
c = Context()
c._h = 77
c.kept = Tensor(DeviceBuffer(c, 64), View.create((16,)), dt.float32, c)
del c
gc.collect()
""") == ["freed", "77", "4096"]


def test_the_module_is_this_pythons_and_its_absence_is_named():
    assert build.CALLS_LIB.name.endswith(sysconfig.get_config_var("EXT_SUFFIX")) and build.CALLS_LIB.exists()
    assert "cpython" in sys.modules["raven_amd._nxcalls"].__file__
    out = in_a_process("""
import sys
sys.modules["raven_amd._nxcalls"] = None
try:
    import raven_amd.nx_backend
except ImportError as e:
    print("built" in str(e), "g.build()" in str(e))
""")
    assert out == ["True", "True"]
