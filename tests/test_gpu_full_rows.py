"""The row kernel over a small system's list in both directions: rows shorter
and longer than a wavefront's share, exclusions, other periodic images, a
triclinic cell, rows cut at their capacity, the largest such system and the
first one beyond it.  Bit for bit against the float twin over the half list.
Triclinic cells of more than six list cells an axis, whose neighbour-cell table
is not symmetric, in a test of their own."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _water(n_waters, box, cutoff, angle=None):
    from sponge_amd import systems
    from sponge_amd.native_io import box_to_cell
    s = systems.tip3p_box(n_waters, box, seed=7, cutoff=cutoff)
    if angle is not None:
        s["angle"] = np.array(angle, np.float32)
        f = s["crd"] / s["box"]
        s["cell"], s["rcell"] = c, _ = box_to_cell(s["box"], s["angle"])
        s["crd"] = np.stack([f[:, 0] * c[0] + f[:, 1] * c[1] + f[:, 2] * c[3],
                             f[:, 1] * c[2] + f[:, 2] * c[4], f[:, 2] * c[5]],
                            axis=1).astype(np.float32)
    return s


CASES = {
    "two_atoms": dict(n=2, box=24.0, cutoff=8.0),
    "short_rows": dict(n=90, box=24.0, cutoff=6.0),
    "water": dict(waters=700, box=28.0, cutoff=8.0),
    "long_rows": dict(waters=700, box=28.0, cutoff=12.0),
    "triclinic": dict(waters=700, box=30.0, cutoff=7.0, angle=(80.0, 75.0, 70.0)),
    "cut_rows": dict(waters=400, box=24.0, cutoff=8.0, max_nb=40),
    "largest": dict(n=8192, box=64.0, cutoff=8.0),
    "beyond": dict(n=8193, box=64.0, cutoff=8.0),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_full_rows_match_twin(name):
    import oracle
    import torch
    from sponge_amd.lib import Nonbonded
    from test_gpu_pair_units import _gas
    c = CASES[name]
    if "n" in c:
        s = _gas(c["n"], c["box"])
    else:
        s = _water(c["waters"], c["box"], c["cutoff"], c.get("angle"))
    nb = Nonbonded(s, cutoff=c["cutoff"], skin=2.0, max_neighbor_numbers=c.get("max_nb", 1200),
                   max_atom_in_grid_numbers=256)
    if nb.window_info()["windowed"]:
        assert nb.set_window_shape(0, 0, 0)
    nb.nl_update(forced=True)
    counts, rows = nb.nl_rows()
    cut = name == "cut_rows"
    assert nb.status(clear=True) == (1 if cut else 0)
    rng = np.random.default_rng(4)
    moved = (s["crd"] + rng.normal(0, 0.3, s["crd"].shape)).astype(np.float32)
    shift = (rng.integers(-1, 2, s["crd"].shape) * s["box"]).astype(np.float32)
    if "angle" in c:
        shift[:] = 0.0
    for crd in (s["crd"], moved, (moved + shift).astype(np.float32)):
        nb.crd.copy_(torch.as_tensor(crd))
        want, _, _, _ = oracle.pair_twin(crd, s["charge"], s["lj_type"], s["lj_a"], s["lj_b"],
                                         s["cell"], s["rcell"], nb.cutoff, nb.beta, counts, rows,
                                         virial=False)
        for mode in (-1, 0):
            nb.set_row_lds(mode)
            nb.clear_fixed_forces()
            nb.lj_direct(frc=False)
            assert np.array_equal(nb.fixed_forces(), want), mode
    assert np.abs(want).max() > 0 or c.get("n") == 2
    nb.close()


def _edges(n, edges, angle):
    """Low-density particles in a triclinic cell of three edges."""
    from sponge_amd.native_io import box_to_cell
    from test_gpu_pair_units import _gas
    s = _gas(n, 44.0)
    f = s["crd"] / s["box"]
    s["box"], s["angle"] = np.array(edges, np.float32), np.array(angle, np.float32)
    s["cell"], s["rcell"] = c, _ = box_to_cell(s["box"], s["angle"])
    s["crd"] = np.stack([f[:, 0] * c[0] + f[:, 1] * c[1] + f[:, 2] * c[3],
                         f[:, 1] * c[2] + f[:, 2] * c[4], f[:, 2] * c[5]],
                        axis=1).astype(np.float32)
    return s


TRICLINIC = {
    "positive_tilts": lambda: _water(2400, 43.0, 8.0, (80.0, 75.0, 70.0)),
    "mixed_tilts": lambda: _water(2400, 46.0, 8.0, (100.0, 95.0, 105.0)),
    "truncated_octahedron": lambda: _water(2200, 45.0, 8.0, (109.47, 109.47, 109.47)),
    "three_edges": lambda: _edges(6000, (40.0, 44.0, 48.0), (85.0, 87.0, 84.0)),
}


@pytest.mark.parametrize("name", sorted(TRICLINIC))
def test_full_rows_of_one_sided_cell_pairs(name):
    """The reference's table of neighbour cells may hold cell j for cell i and
    not i for j; the lower id's cell decides whether a pair is in the half
    list, and both of its atoms get its force or neither does."""
    import oracle
    import torch
    from sponge_amd.lib import Nonbonded
    s = TRICLINIC[name]()
    nb = Nonbonded(s, cutoff=8.0, skin=2.0)
    assert not nb.window_info()["windowed"]
    nb.nl_update(forced=True)
    counts, rows = nb.nl_rows()
    assert nb.status() == 0
    # the half list is the reference's: pairs within the list radius by the table
    # of the lower id's cell; some of those pairs the other cell's table lacks
    rule = oracle.nl_cell_rule(s["crd"], s["cell"], nb.cutoff, 2.0)
    oc, orows, _ = oracle.nl_build(s["crd"], s["cell"], s["rcell"], nb.cutoff, 2.0,
                                   (s["excl_start"], s["excl_numbers"], s["excl_list"]),
                                   max_nb=nb.max_nb)
    from_below = from_above = 0
    for i in range(s["n"]):
        j = np.sort(orows[i, :oc[i]])
        me = np.full(len(j), i)
        below, above = rule(me, j), rule(j, me)
        from_below += np.count_nonzero(below & ~above)
        from_above += np.count_nonzero(above & ~below)
        assert np.array_equal(np.sort(rows[i, :counts[i]]), j[below]), i
    print("case", name, "one-sided pairs", from_below, from_above, flush=True)
    assert from_below > 0 and from_above > 0
    rng = np.random.default_rng(4)
    moved = (s["crd"] + rng.normal(0, 0.3, s["crd"].shape)).astype(np.float32)
    for crd in (s["crd"], moved):
        nb.crd.copy_(torch.as_tensor(crd))
        want, _, _, _ = oracle.pair_twin(crd, s["charge"], s["lj_type"], s["lj_a"], s["lj_b"],
                                         s["cell"], s["rcell"], nb.cutoff, nb.beta, counts, rows,
                                         virial=False)
        for mode, energy in ((-1, False), (0, False), (-1, True)):
            nb.set_row_lds(mode)
            nb.clear_fixed_forces()
            nb.lj_direct(need_energy=energy, frc=False)
            got = nb.fixed_forces()
            assert np.all(got.sum(axis=1) == 0), (mode, energy)
            assert np.array_equal(got, want), (mode, energy)
    nb.close()
