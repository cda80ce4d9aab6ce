"""The staging of state copies (fvgpu_stage.h) over a stand-in for the HIP
runtime that lives in host memory: what a copy does with errors that were
pending before it and with calls that fail under it.  And on the GPU: the
entry points that copy through it right after launching kernels report a
launch error."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "myfvcomcode_amd", "csrc")

# The calls that fvgpu_stage.h makes: copies are done at once, errors are
# kept per thread as the runtime keeps them, and any call can be told to fail.
HIP = r"""
#pragma once
#include <cstdlib>
#include <cstring>
#include <string>
enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2, hipErrorLaunchFailure = 719 };
enum hipMemoryType { hipMemoryTypeUnregistered = 0, hipMemoryTypeHost = 1 };
enum hipMemcpyKind { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2 };
typedef void* hipStream_t;
typedef void* hipEvent_t;
struct hipPointerAttribute_t { hipMemoryType type; };
constexpr unsigned hipHostMallocDefault = 0, hipEventDisableTiming = 2;
inline thread_local hipError_t last = hipSuccess;
inline std::string failing;   // the call that is told to fail
inline bool attributes_answer = true;   // whether an ordinary pointer is answered or refused
inline int live = 0;          // events and pinned buffers that exist
inline hipError_t ret(const char* f, hipError_t e = hipSuccess) {
  if (failing == f) e = hipErrorOutOfMemory;
  if (e != hipSuccess) last = e;
  return e;
}
inline hipError_t hipGetLastError() { const hipError_t e = last; last = hipSuccess; return e; }
inline hipError_t hipPeekAtLastError() { return last; }
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void*) {
  a->type = hipMemoryTypeUnregistered;
  return ret("hipPointerGetAttributes", attributes_answer ? hipSuccess : hipErrorInvalidValue);
}
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  const hipError_t e = ret("hipHostMalloc");
  if (e == hipSuccess) { *p = std::malloc(n); __atomic_add_fetch(&live, 1, __ATOMIC_SEQ_CST); }
  return e;
}
inline hipError_t hipHostFree(void* p) { std::free(p); __atomic_sub_fetch(&live, 1, __ATOMIC_SEQ_CST); return hipSuccess; }
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  if (!d || !s) return ret("hipMemcpyAsync", hipErrorInvalidValue);
  const hipError_t e = ret("hipMemcpyAsync");
  if (e == hipSuccess) std::memcpy(d, s, n);
  return e;
}
inline hipError_t hipStreamSynchronize(hipStream_t) { return ret("hipStreamSynchronize"); }
inline hipError_t hipGetDevice(int* d) { *d = 0; return ret("hipGetDevice"); }
inline hipError_t hipSetDevice(int) { return ret("hipSetDevice"); }
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  const hipError_t r = ret("hipEventCreateWithFlags");
  if (r == hipSuccess) { *e = std::malloc(1); __atomic_add_fetch(&live, 1, __ATOMIC_SEQ_CST); }
  return r;
}
inline hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return ret("hipEventRecord"); }
inline hipError_t hipEventSynchronize(hipEvent_t) { return ret("hipEventSynchronize"); }
inline hipError_t hipEventDestroy(hipEvent_t e) { std::free(e); __atomic_sub_fetch(&live, 1, __ATOMIC_SEQ_CST); return hipSuccess; }
"""

MAIN = r"""
#include "fvgpu_stage.h"
#include <cstdio>
#include <new>
#include <vector>
thread_local int news = -1;   // allocations of this thread that succeed before one fails; -1: all
void* operator new(size_t n) {
  if (news >= 0 && news-- == 0) throw std::bad_alloc();
  if (void* p = std::malloc(n ? n : 1)) return p;
  throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }
#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)
static const size_t sizes[] = {8, HostStage::SMALL, HostStage::SMALL + 1, 40u << 20};
static std::vector<char> bytes(size_t n) {
  std::vector<char> v(n);
  for (size_t i = 0; i < n; ++i) v[i] = (char)(i * 2654435761u >> 13);
  return v;
}
int main() {
BODY
  return 0;
}
"""


def _run(tmp_path, body):
    (tmp_path / "hip").mkdir(exist_ok=True)
    (tmp_path / "hip" / "hip_runtime.h").write_text(HIP)
    src = tmp_path / "main.cpp"
    src.write_text(MAIN.replace("BODY", body))
    exe = str(tmp_path / "main")
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I" + str(tmp_path), "-I" + CSRC, str(src), "-o", exe],
                   check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)


def test_copies_and_pending_errors(tmp_path):
    """What goes up comes down, and an error that was pending before a copy is
    still pending after it, whether the runtime answers for ordinary pointers
    or refuses them, and whether or not pinned memory can be had."""
    _run(tmp_path, r"""
  for (bool answer : {true, false})
    for (const char* f : {"", "hipHostMalloc"})
      for (hipError_t before : {hipSuccess, hipErrorLaunchFailure})
        for (size_t n : sizes) {
          attributes_answer = answer;
          failing = f;
          HostStage st;
          std::vector<char> a = bytes(n), dev(n), b(n);
          last = before;
          CHECK(st.to_device(dev.data(), a.data(), n, nullptr, 0) == hipSuccess);
          CHECK((last != hipSuccess) == (before != hipSuccess));
          CHECK(st.to_host(b.data(), dev.data(), n, nullptr, 0) == hipSuccess);
          CHECK((last != hipSuccess) == (before != hipSuccess));
          CHECK(a == dev && a == b);
          st.release();
          CHECK(live == 0);
        }
""")


def test_null_host_memory_is_refused(tmp_path):
    _run(tmp_path, r"""
  for (size_t n : sizes) {
    HostStage st;
    std::vector<char> dev(n);
    CHECK(st.to_device(dev.data(), nullptr, n, nullptr, 0) == hipErrorInvalidValue);
    CHECK(st.to_host(nullptr, dev.data(), n, nullptr, 0) == hipErrorInvalidValue);
    CHECK(st.to_host(nullptr, dev.data(), 0, nullptr, 0) == hipSuccess);
    st.release();
  }
""")


def test_no_memory_for_the_helpers(tmp_path):
    """A copy whose helper threads cannot be had is done by the caller; no
    exception leaves it, whichever allocation fails."""
    _run(tmp_path, r"""
  for (size_t n : sizes)
    for (int k = 0; k < 6; ++k) {
      HostStage st;
      std::vector<char> a = bytes(n), dev(n), b(n);
      news = k;
      const hipError_t up = st.to_device(dev.data(), a.data(), n, nullptr, 0);
      news = k;
      const hipError_t down = st.to_host(b.data(), dev.data(), n, nullptr, 0);
      news = -1;
      CHECK(up == hipSuccess && down == hipSuccess);
      CHECK(a == dev && a == b);
      st.release();
      CHECK(live == 0);
    }
""")


@pytest.mark.gpu
def test_null_arguments_are_errors(built):
    """Null host memory at the entry points that copy: an error, whatever the
    size, and the handle goes on."""
    import numpy as np
    import myfvcomcode_amd as F
    L = F.gpu_lib()
    m = F.Model.build(1, nx=181, ny=121, kb=12, n_seamounts=1)   # T1 above the size that is copied by chunks
    m.set_river(5, 1.0)
    dev = F.DeviceModel(m)
    dev.run(1)
    print("case: null host memory", flush=True)
    for n in ("el", "t1"):
        k = len(dev.get(n))
        assert L.fvgpu_get_state(dev._h, n.encode(), None, k) != 0
        assert L.fvgpu_put_state(dev._h, n.encode(), None, k) != 0
    assert L.fvgpu_set_forcing(dev._h, b"wind", None, 2 * (m.n + 1)) != 0
    assert L.fvgpu_set_forcing(dev._h, b"tdis", None, 1) != 0
    off = np.zeros(2, np.int64)
    assert L.fvgpu_ensemble_update(dev._h, b"el", 2, off.ctypes.data, off.ctypes.data, 2, 2, None) != 0
    assert L.fvgpu_ensemble_update(dev._h, b"el", 2, None, None, 2, 2, off.ctypes.data) != 0
    t = F.Trainer(np.ones((64, 8), np.float32), np.ones((64, 2), np.float32), bmax=64)
    assert L.fvmlp_set_params(t._h, None) != 0
    t.set_params(np.zeros(L.fvmlp_nparams(), np.float32))
    assert L.fvmlp_get_params(t._h, None) != 0
    assert L.fvmlp_grad(t._h, None, 64, None, None) != 0
    assert L.fvmlp_infer(t._h, 0, 64, 1, None) != 0
    assert np.isfinite(t.grad(batch=64)[1]).all()
    dev.run(1)
    assert dev.diagnostics().iint == 2


@pytest.mark.gpu
@pytest.mark.parametrize("call", ["external_step", "diagnostics"])
def test_launch_error_is_reported(built, call):
    """An error that is pending when the kernels have been enqueued (here that
    of an API call with an invalid device) is the call's result, not lost in
    the copy that follows."""
    import myfvcomcode_amd as F
    L = F.gpu_lib()
    m = F.Model.build(0, nx=21, ny=11, kb=4)
    dev = F.DeviceModel(m)
    dev.run(1)
    dev.synchronize()
    iint = dev.diagnostics().iint
    print("case: %s with an error pending" % call, flush=True)
    assert L.hipSetDevice(9999) != 0
    with pytest.raises(RuntimeError):
        getattr(dev, call)()
    assert dev.diagnostics().iint == iint
    dev.run(1)
    assert dev.diagnostics().iint == iint + 1
