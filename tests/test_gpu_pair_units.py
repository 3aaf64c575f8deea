"""The force-only windowed pair kernel where its units can go wrong: short
rows and lists shorter than a unit, more units than lanes, pairs that come into
range between rebuilds, atoms in other periodic images, types without LJ, LJ
tables exchanged under a built list, windows beyond the LDS map.  All compared
bit for bit with the float twin over the list that the library built."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _gas(n=3000, box=64.0, seed=3, zero=()):
    """Charged LJ particles of three types at low density; types in `zero` have no LJ."""
    from sponge_amd.native_io import box_to_cell
    rng = np.random.default_rng(seed)
    per = int(np.ceil(n ** (1 / 3)))
    g = (np.arange(per) + 0.5) * (box / per)
    crd = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3)[:n]
    crd = (crd + rng.uniform(-1.0, 1.0, crd.shape)) % box
    eps = np.array([0.0 if t in zero else 0.1 + 0.05 * t for t in range(3)])
    i, j = np.tril_indices(3)
    e4 = 4.0 * np.sqrt(eps[i] * eps[j])
    cell, rcell = box_to_cell(np.full(3, box, np.float32))
    return dict(n=n, crd=crd.astype(np.float32),
                charge=rng.normal(0, 5.0, n).astype(np.float32), lj_ntypes=3,
                lj_a=(12.0 * e4 * 3.0 ** 12).astype(np.float32),
                lj_b=(6.0 * e4 * 3.0 ** 6).astype(np.float32),
                lj_type=rng.integers(0, 3, n).astype(np.int32), box=np.full(3, box, np.float32),
                angle=np.full(3, 90.0, np.float32), cell=cell, rcell=rcell,
                excl_start=np.zeros(n, np.int32), excl_numbers=np.zeros(n, np.int32),
                excl_list=np.zeros(0, np.int32), cutoff=8.0)


def _water(n_waters=3000, box=44.8, cutoff=8.0, seed=5):
    from sponge_amd import systems
    return systems.tip3p_box(n_waters, box, seed=seed, cutoff=cutoff)


def _check(nb, s, crd, **tables):
    import oracle
    import torch
    counts, rows = nb.nl_rows()
    nb.crd.copy_(torch.as_tensor(crd))
    t = dict(s, **tables)
    want, _, _, _ = oracle.pair_twin(crd, t["charge"], t["lj_type"], t["lj_a"], t["lj_b"],
                                     t["cell"], t["rcell"], nb.cutoff, nb.beta, counts, rows,
                                     virial=False)
    for mode in (0, 1):  # window sums through the stage and by atomic adds
        nb.set_direct_j(mode)
        nb.clear_fixed_forces()
        nb.lj_direct(frc=False)
        assert np.array_equal(nb.fixed_forces(), want)
    assert nb.status() == 0


CASES = {
    # rows of a few entries in a list whose rows are shorter than a unit
    "short_rows": dict(make=lambda: _gas(1500, 64.0), shape=(1, 1, 1), max_nb=60),
    "empty_rows": dict(make=lambda: _gas(150, 64.0), shape=(2, 2, 2), max_nb=60),
    "no_lj_type": dict(make=lambda: _gas(zero=(1,)), shape=(1, 2, 1), max_nb=400),
    "no_lj_at_all": dict(make=lambda: _gas(zero=(0, 1, 2)), shape=(2, 1, 2), max_nb=400),
    "water_small_blocks": dict(make=_water, shape=(1, 1, 1), max_nb=1200),
    # most units per wavefront: above the 64 that the lanes hold
    "water_large_blocks": dict(make=lambda: _water(6000, 56.5, cutoff=9.0), shape=(2, 2, 6),
                               max_nb=1200),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_units_match_twin(name):
    from sponge_amd.lib import Nonbonded
    c = CASES[name]
    s = c["make"]()
    nb = Nonbonded(s, skin=2.0, max_neighbor_numbers=c["max_nb"], max_atom_in_grid_numbers=256)
    assert nb.set_window_shape(*c["shape"])
    nb.nl_update(forced=True)
    _check(nb, s, s["crd"])
    rng = np.random.default_rng(9)
    # between rebuilds: pairs of the skin come into range
    moved = (s["crd"] + rng.normal(0, 0.35, s["crd"].shape)).astype(np.float32)
    _check(nb, s, moved)
    # other periodic images of some atoms
    shift = (rng.integers(-2, 3, s["crd"].shape) * s["box"]).astype(np.float32)
    shift[rng.random(s["n"]) < 0.7] = 0.0
    _check(nb, s, (moved + shift).astype(np.float32))
    # a window beyond the LDS map adds to the global accumulators
    nb.set_window_capacity(64)
    _check(nb, s, moved)
    nb.close()


def test_new_lj_tables_under_a_built_list():
    """A type without LJ is told from the tables of the moment, not those of the rebuild."""
    from sponge_amd import lib
    s = _gas(zero=(1,))
    nb = lib.Nonbonded(s, skin=2.0, max_neighbor_numbers=400)
    nb.nl_update(forced=True)
    _check(nb, s, s["crd"])
    new = _gas()
    a, b, t = new["lj_a"], new["lj_b"], s["lj_type"]
    lib.check(nb.L.snb_lj_initial(nb.ctx, 3, a.ctypes.data, b.ctypes.data, t.ctypes.data,
                                  nb.cutoff), "snb_lj_initial")
    _check(nb, s, s["crd"], lj_a=a, lj_b=b)
    nb.close()


def test_row_stream_modes_accepted_and_refused():
    """snb_lj_set_row_stream takes the modes that it documents and no other."""
    from sponge_amd.lib import Nonbonded
    nb = Nonbonded(_gas(150, 64.0), skin=2.0, max_neighbor_numbers=60)
    for mode in (-1, 0, 1):
        nb.set_row_stream(mode)
    for mode in (-2, 2):
        with pytest.raises(RuntimeError):
            nb.set_row_stream(mode)
    nb.close()
