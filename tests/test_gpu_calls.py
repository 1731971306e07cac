"""compute_emt through the one-launch call path: odd and even atom counts, one
and several beads, the shape changing from call to call and staying, each call
against the oracle at the 1e-9 eV and eV/A of the EMT parity tests; a type
outside 1..4 is refused and leaves the next call unharmed."""
import numpy as np
import pytest

import oracle
from md_tian2_amd import geometry, mdt, pesfile

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
