"""The reciprocal pipeline's own stream after the choice of it has changed: a
call that comes before the next list update starts after the work queued on the
context's stream, not at an event recorded before the change.  The reciprocal
forces are those of a fresh context at the coordinates written last."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

WINDOWED, PLAIN = 150, 300  # max_atom_in_grid_numbers: above 256 the path without windows


def _system():
    from sponge_amd import systems
    return systems.tip3p_box(2000, 39.2, seed=13, cutoff=8.0)


def _initial(nb, max_in_grid):
    from sponge_amd import lib
    lib.check(nb.L.snb_nl_initial(nb.ctx, nb.cutoff, 2.0, nb.cell, nb.rcell, nb.max_nb,
                                  max_in_grid, 0, 0.5), "snb_nl_initial")


def _reinitialise(nb):
    # a windowed list's update, then a path of one stream, then windows again
    nb.nl_update(forced=True)
    _initial(nb, PLAIN)
    assert not nb.window_info()["windowed"]
    nb.nl_update(forced=True)
    nb.reciprocal(step=0, frc=False)
    _initial(nb, WINDOWED)


def _reinitialise_pending(nb):
    # the pipeline still queued on its own stream when the path changes
    nb.nl_update(forced=True)
    nb.reciprocal(step=0, frc=False)
    _initial(nb, PLAIN)


def _window_shape(nb):
    nb.nl_update(forced=True)
    shape = nb.window_info()
    assert nb.set_window_shape(0, 0, 0)
    nb.nl_update(forced=True)
    assert nb.set_window_shape(shape["a"], shape["b"], shape["s"])


def _overlap(nb):
    nb.nl_update(forced=True)
    nb.set_pme_overlap(False)
    nb.reciprocal(step=0, frc=False)
    nb.set_pme_overlap(True)


def _row_kernel(nb):
    _initial(nb, PLAIN)
    nb.set_row_lds(1)
    nb.nl_update(forced=True)
    nb.set_row_lds(-1)
    nb.reciprocal(step=0, frc=False)
    nb.set_row_lds(1)


CHANGES = {"reinitialise": _reinitialise, "reinitialise_pending": _reinitialise_pending,
           "window_shape": _window_shape, "overlap": _overlap, "row_kernel": _row_kernel}


@pytest.mark.parametrize("name", sorted(CHANGES))
def test_pipeline_starts_after_queued_coordinates(name):
    import torch
    from sponge_amd.lib import Nonbonded
    s = _system()
    rng = np.random.default_rng(3)
    moved = (s["crd"] + rng.normal(0, 0.3, s["crd"].shape)).astype(np.float32)
    fresh = Nonbonded(dict(s, crd=moved), max_atom_in_grid_numbers=WINDOWED)
    fresh.reciprocal(step=0, frc=False)
    want = fresh.fixed_forces()
    fresh.close()
    nb = Nonbonded(s, max_atom_in_grid_numbers=WINDOWED)
    assert nb.window_info()["windowed"]
    print("case", name, flush=True)
    CHANGES[name](nb)
    nb.clear_fixed_forces()
    new = torch.as_tensor(moved).to(nb.dev)
    a = torch.rand(8192, 8192, device=nb.dev)
    torch.cuda.synchronize()
    for _ in range(4):  # milliseconds of work ahead of the coordinates
        a = (a @ a) * 1e-4
    nb.crd.copy_(new)
    nb.reciprocal(step=0, frc=False)
    assert np.array_equal(nb.fixed_forces(), want)
    nb.close()
