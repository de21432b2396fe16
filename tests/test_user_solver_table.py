"""The user-solver route on the host side: the table EXA_USER_SOLVER exports
from the example shared object (a host function; no GPU call).  The hook
flags must see the PDE's __device__ hooks from host code, and the launch
functions must all be present."""
import ctypes
import os
import subprocess

import pytest

from exahype_amd import build, capi


@pytest.mark.parametrize("order", [3, 5])
def test_example_table(order):
    fn = getattr(capi.user_example(), f"exa_user_euler_order{order}")
    fn.restype = ctypes.POINTER(capi.UserSolverTable)
    t = fn().contents
    assert t.abi_version == 1
    assert (t.order, t.num_variables, t.num_parameters, t.terms) == (order, 5, 0, capi.TERM_FLUX)
    assert t.cfl == 0.9
    assert t.has_boundary_values == 1
    assert t.has_adjust == 1
    assert all((t.predictor, t.corrector, t.stable_dt, t.adjust))


@pytest.mark.parametrize("name,order,npar", [("order1_many", 1, 10), ("order2", 2, 3), ("order4", 4, 3)])
def test_flux_free_example_table(name, order, npar):
    fn = getattr(capi.user_example(), f"exa_user_elastic_{name}")
    fn.restype = ctypes.POINTER(capi.UserSolverTable)
    t = fn().contents
    assert (t.order, t.num_variables, t.num_parameters, t.terms) == (order, 9, npar, capi.TERM_NCP)
    assert t.has_boundary_values == 0 and t.has_adjust == 0
    assert all((t.predictor, t.corrector, t.stable_dt, t.adjust))


# (order + 1, variables, parameters, terms, type) a user solver may have, at the
# corners of the predictor's choices of what it keeps where
LAYOUTS = [(2, 1, 3, "ncp", "double"), (3, 1, 3, "ncp", "float"), (2, 9, 10, "ncp", "double"),
           (4, 5, 60, "ncp", "double"), (7, 3, 24, "ncp", "float"), (4, 1, 3, "ncp", "double"),
           (6, 5, 60, "flux", "double"), (6, 5, 60, "flux+ncp", "double"), (6, 5, 0, "flux", "double"),
           (4, 5, 0, "flux+ncp", "double"), (7, 5, 0, "flux", "float")]


def test_predictor_layouts_of_user_solvers(tmp_path):
    """Sizes that need no device workspace and whose epilogue fits the arrays of
    the layout (compile-time constants, checked by the host compiler).  Each was
    accepted before the gradients were taken from the iterate in place and
    before the double form of order 5 ran its time slices in a rolled loop."""
    checks = []
    for b, v, p, terms, t in LAYOUTS:
        ncp, flux = ("true" if k in terms else "false" for k in ("ncp", "flux"))
        layout = f"exa::PredictorLayout<{b}, {v}, {v + p}, {ncp}, {t}, 144, {flux}>"
        checks.append(f"static_assert({layout}::ws_bytes == 0);\n"
                      f"static_assert(!{layout}::IN_PLACE || ({layout}::NQL == {b} && {b * v} >= {v + p}));\n")
    src = tmp_path / "layouts.hip"
    src.write_text('#include "exahype_amd/device/predictor.hpp"\n' + "".join(checks))
    include = os.path.join(build.ROOT, "include")
    res = subprocess.run([build.hipcc(), "--offload-arch=gfx950", "--offload-host-only", "-std=c++20", "-w",
                          "-fsyntax-only", "-I" + include, "-I" + os.path.join(include, "exahype_amd", "device"),
                          str(src)], capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-3000:]
