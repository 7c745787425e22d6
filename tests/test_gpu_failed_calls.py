"""Calls that fail for want of memory leave a simulation that steps on
correctly.  Each case runs in a child process whose HIP allocations pass
through a small library that refuses them on request (hipMalloc beyond a
size), as the runtime does when memory is short:

* a mesh upload that cannot allocate falls back to static geometry with the
  masks and walls in place: the steps after it equal the FP32 oracle's with
  those, bit for bit, whether the geometry before it was a moving sphere alone
  or one set over a static obstacle."""
import ctypes
import os
import subprocess
import sys

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SHIM = r"""
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stddef.h>
static size_t largest = (size_t)-1;
void refuse(size_t bytes_above) { largest = bytes_above; }
static void* real(const char* name) {
    return dlsym(dlopen("libamdhip64.so.7", RTLD_NOW | RTLD_NOLOAD), name);
}
int hipMalloc(void** p, size_t n) {
    if (n > largest) { *p = NULL; return 2; }      /* hipErrorOutOfMemory */
    return ((int (*)(void**, size_t))real("hipMalloc"))(p, n);
}
"""


def failed_mesh(bh, bfref, cases, refuse, over_static):
    p = cases.translating_sphere_params()
    n = p.nx * p.ny * p.nz
    with bh.BirdFlowSimulation(cases.solver_config(p)) as sim:
        if over_static:
            mask = np.zeros((p.nz, p.ny, p.nx), np.uint8)
            mask[3:6, 3:6, 3:6] = 1
            sim.set_geometry(mask.ravel(), np.tile(np.float32([0.02, 0.0, 0.0, 0.3]), (n, 1)))
            sim.init_equilibrium()
            sim.advance(1)
        sim.set_translating_sphere(cases.SPHERE_CENTER_RADIUS, cases.SPHERE_GEOMETRY_VELOCITY,
                                   cases.SPHERE_WALL_VELOCITY)
        if not over_static:
            sim.init_equilibrium()
            sim.advance(6)
        points = np.tile(np.float32([[5, 5, 5], [9, 5, 5], [5, 9, 5]]), (2, 1, 1))
        refuse(0)
        try:
            sim.upload_mesh(points, np.float32([0.0, 1.0]), np.uint32([[0, 1, 2]]), np.uint8([1]), 0.5)
            raise AssertionError("the upload was not refused")
        except bh.BirdFlowError as err:
            print("upload refused:", err, flush=True)
        finally:
            refuse(2 ** 64 - 1)
        mask, wall = sim.read_geometry()
        assert mask.any()
        f = sim.read_populations()
        sim.advance(3)
        got, loads = sim.read_populations(), sim.load_history(3)
    for s in range(3):
        f, ref, _, _ = bfref.step(p, f, mask, mask, wall)
        assert np.abs(loads[s, :6] - ref[:6]).max() <= 1e-12 * np.abs(ref[:6]).max(), s
    assert np.array_equal(got, f)


CHILDREN = {"mesh after a sphere": (failed_mesh, False), "mesh after a sphere over an obstacle": (failed_mesh, True)}


@pytest.mark.gpu
@pytest.mark.parametrize("case", list(CHILDREN))
def test_steps_after_a_refused_call(case, tmp_path):
    print("case:", case, flush=True)
    source, library = tmp_path / "refuse.c", tmp_path / "refuse.so"
    source.write_text(SHIM)
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(library), str(source), "-ldl"], check=True)
    run = subprocess.run([sys.executable, os.path.abspath(__file__), str(library), case], timeout=100,
                         capture_output=True, text=True)
    print(run.stdout[-2000:], run.stderr[-2000:], flush=True)
    assert run.returncode == 0 and "refused" in run.stdout


if __name__ == "__main__":
    shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)    # before the HIP library: its names win
    shim.refuse.argtypes = [ctypes.c_size_t]
    for sub in ("oracle", "numi-gpu-physics_amd", "tests"):
        sys.path.insert(0, os.path.join(os.path.dirname(HERE), sub))
    import bfref
    import birdflow_hip as bh
    import cases
    child, argument = CHILDREN[sys.argv[2]]
    child(bh, bfref, cases, shim.refuse, argument)
