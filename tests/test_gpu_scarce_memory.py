"""A small system without windows where the rows of lower ids find no memory: the
list and the forces are there all the same, over the half list.  A child process
whose hipMalloc (a shim ahead of the runtime's) refuses that one size."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

SHIM = r"""
#include <stddef.h>
typedef int (*malloc_fn)(void**, size_t);
static malloc_fn real;
static size_t refused_size;
static int refusals;
void shim_set(malloc_fn f, size_t size) { real = f; refused_size = size; }
int shim_refusals(void) { return refusals; }
int hipMalloc(void** p, size_t size)
{
    if (refused_size && size == refused_size) { refusals++; return 2; }
    return real(p, size);
}
"""

CHILD = r"""
import ctypes, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)   # ahead of the runtime
sys.path[:0] = sys.argv[2:5]
import numpy as np
import torch
runtime = [line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line][0]
real = ctypes.cast(ctypes.CDLL(runtime).hipMalloc, ctypes.c_void_p)
shim.shim_set.argtypes = [ctypes.c_void_p, ctypes.c_size_t]
shim.shim_set(real, 0)
from sponge_amd.lib import Nonbonded
from test_gpu_full_rows import _edges, _water


def forces(nb):
    nb.nl_update(forced=True)
    nb.clear_fixed_forces()
    nb.lj_direct(frc=False)
    f = nb.fixed_forces()
    assert nb.status() == 0
    return f


for name, s in (("orthorhombic", _water(700, 28.0, 8.0)),
                ("triclinic", _edges(3000, (40.0, 44.0, 48.0), (85.0, 87.0, 84.0)))):
    n = s["n"]
    nb = Nonbonded(s, cutoff=8.0, max_atom_in_grid_numbers=300)
    assert not nb.window_info()["windowed"]
    want = forces(nb)
    nb.close()
    before = shim.shim_refusals()
    shim.shim_set(real, 2 * n * n)
    nb = Nonbonded(s, cutoff=8.0, max_atom_in_grid_numbers=300)
    assert shim.shim_refusals() == before + 1
    assert np.array_equal(forces(nb), want)
    nb.close()
    if name == "orthorhombic":
        nb = Nonbonded(s, cutoff=8.0)
        assert nb.window_info()["windowed"] and nb.set_window_shape(0, 0, 0)
        assert shim.shim_refusals() == before + 2
        assert np.array_equal(forces(nb), want)
        nb.close()
    shim.shim_set(real, 0)
    print("ok", name, flush=True)
"""


def test_half_list_alone_without_memory_for_the_lower_ids(tmp_path):
    from conftest import ROOT
    (tmp_path / "shim.c").write_text(SHIM)
    shim = str(tmp_path / "shim.so")
    subprocess.run(["cc", "-shared", "-fPIC", "-O1", "-o", shim, str(tmp_path / "shim.c")],
                   check=True)
    (tmp_path / "child.py").write_text(CHILD)
    paths = [os.path.join(ROOT, "sponge2.0_amd", "python"), os.path.join(ROOT, "oracle"),
             os.path.join(ROOT, "tests")]
    r = subprocess.run([sys.executable, "-u", str(tmp_path / "child.py"), shim] + paths,
                       capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.split() == ["ok", "orthorhombic", "ok", "triclinic"]
