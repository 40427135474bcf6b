"""csrc/native_calls.cpp without a GPU: built against a stand-in of the library's entry points.

The stand-ins count their calls; CPU tensors take the place of GPU ones and wrapping the result can be made
to fail.  What is checked is the promise that None means "nothing has been launched", on which the Python
layer makes the call again by itself.
"""

import ctypes
import importlib.machinery
import importlib.util
import os
import subprocess

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "nano-vllm-practice_amd")

HARNESS = r"""
#include <Python.h>
#include <ATen/Functions.h>
#include <c10/hip/HIPStream.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <torch/csrc/autograd/python_variable.h>
#include <stdexcept>
extern "C" { int fail_wrap = 0; }
static PyObject* stub_wrap(const at::Tensor& t) {
    if (fail_wrap == 1) throw std::runtime_error("no wrapper");
    if (fail_wrap == 2) return PyErr_NoMemory();
    return THPVariable_Wrap(t);
}
namespace c10::hip {
struct StubStream { void* stream() const { return nullptr; } };
inline StubStream stub_stream(int) { return {}; }
}
#define THPVariable_Wrap stub_wrap
#define is_cuda is_cpu
#define getCurrentHIPStreamMasqueradingAsCUDA stub_stream
#include "native_calls.cpp"
"""


@pytest.fixture(scope="module")
def native(tmp_path_factory):
    """(module, counts, rc, fail_wrap): the harness bound to stand-ins that count and return rc[0]."""
    spec = importlib.util.spec_from_file_location("femto_build", os.path.join(PKG, "build.py"))
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    d = tmp_path_factory.mktemp("native")
    src, lib = d / "harness.cpp", d / "femto_native.so"
    src.write_text(HARNESS)
    cmd = [str(src) if a.endswith("native_calls.cpp") else "-O0" if a == "-O2" else a
           for a in build.native_command(str(lib))]
    subprocess.run(cmd + [f"-I{PKG}/csrc"], check=True, capture_output=True, text=True)
    loader = importlib.machinery.ExtensionFileLoader("femto_native", str(lib))
    module = importlib.util.module_from_spec(importlib.util.spec_from_loader("femto_native", loader))
    loader.exec_module(module)
    counts, rc, keep = {}, [0], {}

    def entry(name, restype, result):
        def call():
            counts[name] = counts.get(name, 0) + 1
            return result()

        keep[name] = ctypes.CFUNCTYPE(restype)(call)  # cdecl: the callee ignores the arguments it does not read

    message = ctypes.create_string_buffer(b"stand-in refused")
    entry("femto_attn_last_error", ctypes.c_void_p, lambda: ctypes.addressof(message))
    for name in ("femto_paged_attention_gemv", "femto_paged_attention_gemm", "femto_qk_norm_rope_cache_write",
                 "femto_flash_attention"):
        entry(name, ctypes.c_int, lambda: rc[0])
    for name in ("femto_paged_attention_gemv_workspace_size", "femto_paged_attention_gemm_workspace_size"):
        entry(name, ctypes.c_size_t, lambda: 0)
    module.bind({n: ctypes.cast(f, ctypes.c_void_p).value for n, f in keep.items()})
    module.keep = keep, message
    return module, counts, rc, ctypes.c_int.in_dll(ctypes.CDLL(str(lib)), "fail_wrap")


def _calls(module):
    """entry point -> (library function, call)"""
    i32 = lambda *s: torch.zeros(s, dtype=torch.int32)
    b16 = lambda *s: torch.zeros(s, dtype=torch.bfloat16)
    pool, rope = b16(4, 2, 16, 128), torch.zeros(64, 128)
    return {
        "gemv": ("femto_paged_attention_gemv",
                 lambda q=b16(4, 3, 128): module.gemv(q, pool, pool, i32(3, 2), i32(3), 20, True, None, {})),
        "gemm": ("femto_paged_attention_gemm",
                 lambda q=b16(4, 5, 128): module.gemm(q, pool, pool, i32(2), 5, i32(1, 2), i32(1), i32(5), True, {})),
        "prologue": ("femto_qk_norm_rope_cache_write",
                     lambda q=b16(3, 4, 128): module.prologue(q, b16(3, 2, 128), b16(3, 2, 128), b16(128), b16(128), 1e-6,
                                                              rope, rope, i32(3), pool, pool, i32(3, 2), None, 1, None)),
        "flash": ("femto_flash_attention",
                  lambda q=b16(1, 4, 5, 128): module.flash(q, b16(1, 2, 9, 128), b16(1, 2, 9, 128))),
    }


ENTRIES = ["gemv", "gemm", "prologue", "flash"]


@pytest.mark.parametrize("name", ENTRIES)
def test_call_returns_the_output(native, name):
    module, counts, _, _ = native
    fn, call = _calls(module)[name]
    before = counts.get(fn, 0)
    out = call()
    assert isinstance(out, torch.Tensor) and out.dtype == torch.bfloat16 and counts[fn] == before + 1


@pytest.mark.parametrize("name", ENTRIES)
@pytest.mark.parametrize("how", [1, 2], ids=["throws", "python_error"])
def test_none_means_nothing_was_launched(native, name, how):
    """No Python object for the result: declined before the library is called, with no error left set."""
    module, counts, _, fail_wrap = native
    fn, call = _calls(module)[name]
    before = counts.get(fn, 0)
    fail_wrap.value = how
    try:
        assert call() is None
    finally:
        fail_wrap.value = 0
    assert counts.get(fn, 0) == before


@pytest.mark.parametrize("name", ENTRIES)
def test_library_errors_raise(native, name):
    module, counts, rc, _ = native
    fn, call = _calls(module)[name]
    before, rc[0] = counts.get(fn, 0), 1
    try:
        with pytest.raises(RuntimeError, match="stand-in refused"):
            call()
    finally:
        rc[0] = 0
    assert counts[fn] == before + 1


@pytest.mark.parametrize("name", ENTRIES)
def test_declined_forms(native, name):
    """Wrong types, ranks and subclasses are left to the Python path."""
    module, counts, _, _ = native
    fn, call = _calls(module)[name]
    before = counts.get(fn, 0)

    class Sub(torch.Tensor):
        pass

    q = torch.zeros((1, 4, 5, 128) if name == "flash" else (3, 4, 128) if name == "prologue" else
                    (4, 3 if name == "gemv" else 5, 128), dtype=torch.bfloat16)
    for bad in (q.double(), q[0], q.as_subclass(Sub), None, [1.0], q.half()):
        assert call(bad) is None
    assert counts.get(fn, 0) == before
