"""set_state / get_state: the reference's r(3,P,N) (src/universe_mod.f90:38-67)
laid out on the device and back, exactly, at the edges of the tiles of 256
atom-beads that the layout kernel works in; in mixed bead mode a classical
atom's bead 0 is reported in every bead."""
import numpy as np
import pytest

from md_tian2_amd import geometry, mdt

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nbeads", [(1, 1, 1), (1, 2, 3), (16, 1, 5), (64, 10, 1)])
@pytest.mark.parametrize("mixed", [0, 1])
def test_state_round_trip(gpu_ctx, nbeads, mixed):
    rng = np.random.default_rng(3)
    systems = []
    for p, (n, layers) in zip(nbeads, ((1, 1), (3, 4), (8, 4))):  # 2, 37 and 257 atoms
        s = geometry.h_on_slab("Au", n=n, nlayers=layers, nfixed=1 if layers > 1 else 0, rng=rng, nbeads=p)
        s.r = rng.normal(0, 10.0, s.r.shape)
        s.v = rng.normal(0, 1.0, s.v.shape)
        systems.append(s)
    b = mdt.Batch(gpu_ctx, systems, dt=0.1, tsurf=300.0, tproj=300.0)
    if mixed:
        b.set_bead_mode(1)
    for s, o in zip(systems, b.get_state()):
        r, v = s.r.copy(), s.v.copy()
        if mixed:
            r[1:] = r[1:, :1]
            v[1:] = v[1:, :1]
        assert np.array_equal(o["r"], r)
        assert np.array_equal(o["v"], v)
    b.close()
