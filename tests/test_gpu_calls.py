"""compute_emt through the one-launch call path: odd and even atom counts, one
and several beads, the shape changing from call to call and staying, each call
against the oracle at the 1e-9 eV and eV/A of the EMT parity tests; a type
outside 1..4 is refused and leaves the next call unharmed, and so does what
an earlier call of the shape was flagged with."""
import numpy as np
import pytest

import oracle
from md_tian2_amd import geometry, mdt, nene, pesfile

pytestmark = pytest.mark.gpu


def test_calls_of_changing_shapes(gpu_ctx, pes_hau):
    rng = np.random.default_rng(17)
    shapes = [(1, 1, 1), (3, 4, 1), (3, 4, 1), (2, 2, 3), (3, 4, 5), (7, 4, 1), (3, 4, 5), (1, 1, 64)]
    for n, layers, p in shapes:  # 2, 37, 37, 9, 37, 197, 37 and 2 atoms
        s = geometry.h_on_slab("Au", n=n, nlayers=layers, nfixed=0, rng=rng, nbeads=p, z0=1.7)
        s.r += rng.normal(0, 0.05, s.r.shape)
        cols, pesm = pesfile.emt_tables(pes_hau, s.type_names)
        gpu_ctx.set_emt(cols, pesm)
        e, f, d = gpu_ctx.compute_emt(s)
        er, fr, dr = oracle.emt_energy_forces(s, cols, pesm)
        assert np.abs(e - er).max() <= 1e-9 * max(1.0, np.abs(er).max())
        assert np.abs(f - fr).max() <= 1e-9
        assert np.allclose(d, dr, rtol=1e-12, atol=1e-15)
        bad = s.copy()
        bad.idx[-1] = 4  # 0-based: type 5
        with pytest.raises(mdt.MdtError):
            gpu_ctx.compute_emt(bad)
        assert np.array_equal(gpu_ctx.compute_emt(s)[1], f)


def test_an_earlier_calls_status_is_gone(gpu_ctx, pes_hau):
    import os

    rng = np.random.default_rng(18)
    good = geometry.h_on_slab("Au", n=3, nlayers=4, rng=rng, z0=1.7)
    cols, pesm = pesfile.emt_tables(pes_hau, good.type_names)
    gpu_ctx.set_emt(cols, pesm)
    gpu_ctx.set_nn(nene.load(os.path.join(os.path.dirname(mdt.LIB_PATH), "nn", "hau_radial")), good.type_names)
    er, fr, _ = oracle.emt_energy_forces(good, cols, pesm)

    def check():
        e, f, _ = gpu_ctx.compute_emt(good)
        assert abs(e[0] - er[0]) <= 1e-9 * max(1.0, abs(er[0])) and np.abs(f - fr).max() <= 1e-9

    check()
    # a successful network call outside the training range
    out = good.copy()
    out.r[:, 0] *= 0.9
    out.simbox = out.simbox * 0.9
    assert gpu_ctx.compute_nene(out)[2]
    check()
    # a call that fails: two atoms on one point
    bad = good.copy()
    bad.r[5] = bad.r[6]
    with pytest.raises(mdt.MdtError):
        gpu_ctx.compute_emt(bad)
    check()
