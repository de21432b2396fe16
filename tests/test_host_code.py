"""Host-side C++ of the library, in small programs built and run without a GPU."""
import os
import re
import subprocess

import pytest

from exahype_amd import build, capi

ROCM = os.path.dirname(os.path.dirname(os.path.realpath(build.hipcc())))


def _run(tmp_path, source, *link):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(source)
    res = subprocess.run(["g++", "-std=c++20", "-O1", "-w", "-D__HIP_PLATFORM_AMD__", f"-I{ROCM}/include",
                          f"-I{build.ROOT}/include", f"-I{build.ROOT}/include/exahype_amd/device",
                          f"-I{build.HERE}/csrc", "-o", str(exe), str(src), *link], capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-3000:]
    return subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)


@pytest.fixture(scope="module")
def library():
    capi.lib()
    return [build.LIB, f"-Wl,-rpath,{build.HERE}", f"-L{ROCM}/lib", "-lamdhip64", f"-Wl,-rpath,{ROCM}/lib"]


def test_linear_surface_integral_is_not_the_nonlinear_one(tmp_path, library):
    """The update pass holds the nonlinear surface integral only and refuses a
    linear solver (before any launch)."""
    res = _run(tmp_path, r"""
#include "aderdg.hpp"
#include <cstdio>
int main() {
  int bad = 0;
  for (int mode : {exa::kUpdSurface | exa::kUpdUpdate, exa::kUpdSurface | exa::kUpdWriteLduh}) {
    exa::SolverDesc sd{};
    sd.pde = exa::kPdeElastic;
    sd.order = 4;
    sd.nvar = 9;
    sd.npar = 3;
    sd.terms = exa::kNCP;
    sd.precision = exa::kFP64;
    sd.linear = 1;
    exa::UpdateArgs a{};
    bad += exa::launch_update(sd, mode, a, 1, nullptr) != hipErrorNotSupported;
  }
  return bad;
}
""", *library)
    assert res.returncode == 0, res.stderr


def test_limiter_counters_are_allocated_whole():
    """Every owner of the limiter kernels' counters allocates and clears all of
    them, whichever its calls read today."""
    owners = 0
    for name in sorted(os.listdir(os.path.join(build.HERE, "csrc"))):
        text = open(os.path.join(build.HERE, "csrc", name)).read()
        for stmt in re.findall(r"[^;{}]*flags[^;{}]*;", text):
            if re.search(r"\b(hipMalloc|A\(|alloc\(|hipMemset)", stmt) and not re.search(r"CreateWithFlags", stmt):
                assert "kLimFlagBytes" in stmt, (name, stmt.strip())
                owners += 1
    assert owners >= 3


# the runtime's calls as host functions that count: device memory is host memory
FAKE_HIP = r"""
#include "capi_util.hpp"
#include <cstdio>
#include <cstdlib>
#include <numeric>
#include <vector>
static int ups, downs, sets;
extern "C" {
hipError_t hipMalloc(void** p, size_t n) { *p = std::malloc(n); std::memset(*p, 0x5a, n); return hipSuccess; }
hipError_t hipFree(void* p) { std::free(p); return hipSuccess; }
hipError_t hipMemset(void* p, int v, size_t n) { ++sets; std::memset(p, v, n); return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipMemcpy(void* to, const void* from, size_t n, hipMemcpyKind k) {
  ++(k == hipMemcpyHostToDevice ? ups : downs);
  std::memcpy(to, from, n);
  return hipSuccess;
}
}
#define CHECK(c) if (!(c)) { std::printf("line %d: %s\n", __LINE__, #c); return 1; }
"""


@pytest.mark.parametrize("scratch,inputs,packed", [(0, 4096, True), (1 << 19, 900 << 10, True), (1 << 21, 64, True),
                                                   (0, 1 << 20, False), (64, 2 << 20, False)])
def test_buffers_of_a_call(tmp_path, scratch, inputs, packed):
    """One copy each way up to 1 MiB of inputs and outputs, whatever the scratch;
    array by array above.  Inputs, outputs, both, cleared and empty parts."""
    res = _run(tmp_path, FAKE_HIP + r"""
int main() {
  const size_t n = %d / 8, m = 256;
  std::vector<double> in(n), io(m, 2.0), out(m), zero(m, -1.0);
  std::iota(in.begin(), in.end(), 1.0);
  CallBuffers b;
  const int i_in = b.in(in.data(), n * 8), i_out = b.out(out.data(), m * 8), i_none = b.in(nullptr, 0);
  const int i_io = b.inout(io.data(), io.data(), m * 8), i_zero = b.out(zero.data(), m * 8, true);
  const int i_scratch = b.scratch(%d), i_z2 = b.zeroed(m * 8);
  CHECK(b.up() == hipSuccess);
  CHECK(i_none != i_in && i_scratch != i_z2);
  for (size_t k = 0; k < m; ++k) {  // the call's kernel
    CHECK(b.d(i_zero)[k] == 0.0 && b.d(i_z2)[k] == 0.0);
    b.d(i_out)[k] = b.d(i_in)[k %% n] + b.d(i_io)[k];
    b.d(i_io)[k] *= 3.0;
  }
  std::memset(b.d(i_scratch), 0, %d);
  CHECK(b.down() == hipSuccess);
  for (size_t k = 0; k < m; ++k) CHECK(out[k] == in[k %% n] + 2.0 && io[k] == 6.0 && zero[k] == 0.0);
  std::printf("up %%d down %%d set %%d\n", ups, downs, sets);
  return 0;
}
""" % (inputs, scratch, scratch))
    assert res.returncode == 0, res.stdout
    assert res.stdout.split() == (["up", "1", "down", "1", "set", "0"] if packed else
                                  ["up", "2", "down", "3", "set", "3"])


def test_buffers_of_a_call_too_many_parts(tmp_path):
    """More parts than a call can have are refused, not written past the table."""
    res = _run(tmp_path, FAKE_HIP + r"""
int main() {
  struct { CallBuffers b; } x;
  double v[64] = {};
  for (int k = 0; k < 64; ++k) CHECK(x.b.in(v + k, 8) < 16);
  CHECK(x.b.up() == hipErrorInvalidValue);
  return 0;
}
""")
    assert res.returncode == 0, res.stdout + res.stderr


def test_riemann_call_on_a_small_stack(tmp_path, library):
    """The single-face Riemann call runs on a thread with 96 KiB of stack (its
    status is that of the device, absent or not)."""
    res = _run(tmp_path, r"""
#include "exahype_amd.h"
#include <cstdio>
#include <pthread.h>
static exa_solver s;
static double FL[320], FR[320], QL[384], QR[384];
static void* call(void* status) {
  *static_cast<int*>(status) = exa_riemann_solver_nonlinear(&s, FL, FR, QL, QR, 0.1, 1);
  return nullptr;
}
int main() {
  s.pde = EXA_PDE_EULER;
  s.order = 3;
  s.num_variables = 5;
  s.terms = EXA_TERM_FLUX;
  s.cfl = 0.9;
  for (int k = 0; k < 80; k += 5) QL[k] = QR[k] = 1.0, QL[k + 4] = QR[k + 4] = 2.5;
  int here = -1, there = -2;
  call(&here);  // the runtime starts on this thread
  pthread_attr_t a;
  pthread_t t;
  pthread_attr_init(&a);
  if (pthread_attr_setstacksize(&a, 96 << 10) != 0 || pthread_create(&t, &a, call, &there) != 0) return 2;
  pthread_join(t, nullptr);
  std::printf("%d %d\n", here, there);
  return here == there && here != EXA_E_INVALID && here != EXA_E_UNSUPPORTED ? 0 : 1;
}
""", "-lpthread", *library)
    assert res.returncode == 0, (res.returncode, res.stdout, res.stderr)
