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
