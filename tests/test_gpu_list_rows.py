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


def _clustered(box):
    """One of seven particles around a corner of the reference's grids, which
    are 6 A wide, well inside a cell that shares its axis evenly."""
    s = _stretched(box)
    rng = np.random.default_rng(2)
    near = rng.random(s["n"]) < 0.15
    s["crd"][near] = 6.0 + rng.normal(0, 0.6, (int(near.sum()), 3))
    return s


def _tilted():
    from test_gpu_full_rows import _edges
    return _edges(6000, (40.0, 44.0, 48.0), (85.0, 87.0, 84.0))


def _most_in_a_grid(s, cutoff, even=False):
    """Atoms of the fullest grid of the reference (grids of (cutoff + skin) / 2,
    the last of an axis with the remainder; neighbor_list.cpp:206-275), or of
    cells that share each axis evenly."""
    f = np.float32
    c = np.asarray(s["cell"], f)
    gl = (f(cutoff) + f(2.0)) * f(0.5)
    edge = c[[0, 2, 5]]
    per = np.floor(edge / gl).astype(np.int64)
    r = np.array(s["crd"], f)
    k3 = np.floor(r[:, 2] / c[5])
    r[:, 2] -= k3 * c[5]
    r[:, 1] -= k3 * c[4]
    k2 = np.floor(r[:, 1] / c[2])
    r[:, 1] -= k2 * c[2]
    r[:, 0] -= k3 * c[3] + k2 * c[1]
    r[:, 0] -= np.floor(r[:, 0] / c[0]) * c[0]
    width = edge / per.astype(f) if even else np.full(3, gl)
    g = np.clip((r / width).astype(np.int64), 0, per - 1)
    return int(np.bincount((g[:, 0] * per[1] + g[:, 1]) * per[2] + g[:, 2]).max())


OVERFLOW = {
    "exact_edges": dict(make=lambda: _stretched((30.0, 60.0, 36.0)), cutoff=10.0),
    # the reference's corner grid holds several times the atoms of an even cell
    "wide_cells": dict(make=lambda: _stretched((35.9, 47.9, 41.9)), cutoff=10.0),
    # an even cell holds several times the atoms of the reference's fullest grid
    "clustered": dict(make=lambda: _clustered((35.9, 47.9, 41.9)), cutoff=10.0, max_nb=2600),
    "triclinic": dict(make=_tilted, cutoff=8.0, plain=True),
}


@pytest.mark.parametrize("plain", [False, True])
@pytest.mark.parametrize("name", sorted(OVERFLOW))
def test_grid_overflow_report(name, plain):
    """The overflow flag counts the reference's grids, whatever the cells that
    the list is built over: raised from the first atom above the limit."""
    from sponge_amd.lib import FLAG_CELL_OVERFLOW, Nonbonded
    c = OVERFLOW[name]
    s = c["make"]()
    most = _most_in_a_grid(s, c["cutoff"])
    if name == "wide_cells":
        assert 2 * _most_in_a_grid(s, c["cutoff"], even=True) < most
    if name == "clustered":
        assert _most_in_a_grid(s, c["cutoff"], even=True) > 3 * most
    for limit in (most - 1, most):
        nb = Nonbonded(s, cutoff=c["cutoff"], skin=2.0, max_neighbor_numbers=c.get("max_nb", 1200),
                       max_atom_in_grid_numbers=limit)
        if plain and nb.window_info()["windowed"]:
            assert nb.set_window_shape(0, 0, 0)
        elif not c.get("plain") and limit <= 256 and not plain:
            assert nb.window_info()["windowed"]
        for _ in range(2):
            nb.nl_update(forced=True)
            assert nb.status(clear=True) == (FLAG_CELL_OVERFLOW if limit < most else 0)
        nb.close()
