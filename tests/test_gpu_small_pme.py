"""The reciprocal pipeline of small systems (atoms binned by one workgroup,
forward planes in one kernel) against the kernels that all sizes have in
common, which recorded step batches use: the same steps, bit for bit, around
the most atoms, the most bricks and planes of both kinds that the small path takes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = {
    "few_atoms": dict(waters=216, box=18.7, grid=(20, 24, 28)),
    "most_atoms": dict(waters=5461, box=54.7, grid=(56, 56, 56)),
    "more_atoms": dict(waters=5462, box=54.7, grid=(56, 56, 56)),
    "most_bricks": dict(waters=216, box=18.7, grid=(128, 128, 128)),
    "more_bricks": dict(waters=216, box=18.7, grid=(128, 140, 128)),
    "odd_planes": dict(waters=216, box=18.7, grid=(9, 49, 45)),
    "large_plane": dict(waters=216, box=18.7, grid=(16, 60, 60)),
    "larger_plane": dict(waters=216, box=18.7, grid=(16, 80, 64)),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_small_pipeline_matches_general(name):
    import torch
    from sponge_amd import systems
    from sponge_amd.lib import Nonbonded, StepBatch
    c = CASES[name]
    s = systems.tip3p_box(c["waters"], c["box"], seed=4, cutoff=7.0)
    got = []
    for batched in (False, True):
        st = torch.cuda.Stream()
        nb = Nonbonded(s, cutoff=7.0, refresh_interval=2, grid=c["grid"], stream=st)
        nb.set_pme_overlap(False)
        nb.set_export(False)
        with torch.cuda.stream(st):
            nb.md_initial(s, temperature=300.0, tau=0.1, seed=3, dt=0.001)
            for k in range(2):
                nb.md_step(step=k, forced_nl=(k == 0))
            if not batched:
                for k in range(2, 4):
                    nb.md_step(step=k)
        st.synchronize()
        if batched:
            b = StepBatch()
            b.record(nb, 2, 2)
            b.plan()
            b.launch(st)
            st.synchronize()
            b.close()
        assert nb.status() == 0
        got.append((nb.crd.cpu().numpy(), nb.vel.cpu().numpy()))
        nb.close()
    np.testing.assert_array_equal(got[0][0], got[1][0])
    np.testing.assert_array_equal(got[0][1], got[1][1])
    assert np.isfinite(got[0][1]).all()
