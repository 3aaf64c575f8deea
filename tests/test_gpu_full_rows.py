"""The row kernel over a small system's list in both directions: rows shorter
and longer than a wavefront's share, exclusions, other periodic images, a
triclinic cell, rows cut at their capacity, the largest such system and the
first one beyond it.  Bit for bit against the float twin over the half list."""
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
