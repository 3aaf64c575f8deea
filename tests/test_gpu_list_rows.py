"""The windowed list builder where it can go wrong: cells of more than a
wavefront of atoms, stencils of more than one chunk of candidates, cells whose
atoms are in different periodic images, axes that are an exact number of list
cells and axes that are not.  The public list holds the pairs of the oracle's
cell-list build with the reference's float distance test and exclusion rule."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _stretched(box):
    """Low-density particles over a box of three different edges."""
    from sponge_amd.native_io import box_to_cell
    from test_gpu_pair_units import _gas
    s = _gas(4000, 50.0)
    scale = np.asarray(box, np.float32) / s["box"]
    s["crd"] = (s["crd"] * scale).astype(np.float32)
    s["box"] = np.asarray(box, np.float32)
    s["cell"], s["rcell"] = box_to_cell(s["box"])
    return s


def _dense(n):
    from test_gpu_pair_units import _gas
    return _gas(n, 32.0)


def _water():
    from sponge_amd import systems
    return systems.tip3p_box(1500, 35.6, seed=6, cutoff=8.0)


CASES = {
    # 72 atoms per cell, 4,500 candidates; windows near the whole LDS
    "dense": dict(make=lambda: _dense(9000), cutoff=10.0, max_nb=2600, shape=(1, 1, 1)),
    # the smallest window is larger than the preferred share of the LDS
    "large_windows": dict(make=lambda: _dense(6400), cutoff=10.0, max_nb=2000),
    "exact_edges": dict(make=lambda: _stretched((30.0, 60.0, 36.0)), cutoff=10.0, max_nb=1200),
    "wide_cells": dict(make=lambda: _stretched((35.9, 47.9, 41.9)), cutoff=10.0, max_nb=1200),
    "water": dict(make=_water, cutoff=8.0, max_nb=600),
}


@pytest.mark.parametrize("images", [False, True])
@pytest.mark.parametrize("name", sorted(CASES))
def test_windowed_list_matches_oracle(name, images):
    import oracle
    from sponge_amd.lib import Nonbonded
    c = CASES[name]
    s = c["make"]()
    if images:
        rng = np.random.default_rng(8)
        shift = (rng.integers(-2, 3, s["crd"].shape) * s["box"]).astype(np.float32)
        shift[rng.random(s["n"]) < 0.6] = 0.0
        s["crd"] = (s["crd"] + shift).astype(np.float32)
    nb = Nonbonded(s, cutoff=c["cutoff"], skin=2.0, max_neighbor_numbers=c["max_nb"],
                   max_atom_in_grid_numbers=256)
    if "shape" in c:
        assert nb.set_window_shape(*c["shape"])
    assert nb.window_info()["windowed"]
    nb.nl_update(forced=True)
    gc, gr = nb.nl_rows()
    assert nb.status() == 0
    oc, orows, _ = oracle.nl_build(s["crd"], s["cell"], s["rcell"], nb.cutoff, 2.0,
                                   (s["excl_start"], s["excl_numbers"], s["excl_list"]),
                                   max_nb=nb.max_nb)
    np.testing.assert_array_equal(gc, oc)
    for i in range(s["n"]):
        assert np.array_equal(np.sort(gr[i, :gc[i]]), np.sort(orows[i, :oc[i]])), i
    ic, _ = nb.internal_rows()
    assert ic.sum() == gc.sum()
    nb.close()
