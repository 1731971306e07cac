"""The propagators' chunks (runs of atoms with all their beads, at most 256
atom-beads to a workgroup) against the oracle where they can go wrong: one
atom left over, a chunk of a few atoms, bead numbers that do not divide 256,
one-bead slabs of more than 256 atoms, the COM velocity summed over chunks.
Bars as in the propagators' own tests: 1e-8 over ten steps of RPMD.
"""
import numpy as np
import pytest

import oracle
from md_tian2_amd import geometry, mdt, pesfile

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,layers,P,proj,latt", [
    (3, 4, 7, geometry.PROP_PILE, geometry.PROP_LANGEVIN),    # 36 atoms to a chunk: one left over
    (3, 4, 10, geometry.PROP_VERLET, geometry.PROP_ANDERSEN),  # COM removal without PILE, transforms of every atom
    (3, 4, 64, geometry.PROP_PILE, geometry.PROP_LANGEVIN),   # 4 atoms to a chunk
    (3, 4, 6, geometry.PROP_PILE, geometry.PROP_PILE),        # every atom thermostatted and transformed
    (8, 4, 2, geometry.PROP_VERLET, geometry.PROP_LANGEVIN),  # 257 atoms: three chunks, no COM removal
    (8, 4, 1, geometry.PROP_PILE, geometry.PROP_LANGEVIN),    # 257 one-bead atoms: one left over
    (3, 4, 1, geometry.PROP_VERLET, geometry.PROP_ANDERSEN),  # one chunk
])
def test_chunk_edges_against_the_oracle(gpu_ctx, pes_hpt, n, layers, P, proj, latt):
    g = np.random.default_rng(100 * n + P)
    systems = [geometry.h_on_slab("Pt", n=n, nlayers=layers, nbeads=P, rng=g, z0=2.2, proj_algo=proj, latt_algo=latt,
                                  tsurf=100.0) for _ in range(2)]
    for s in systems:
        s.r += g.normal(0, 0.02, s.r.shape) * ~s.fixed
    cols, pesm = pesfile.emt_tables(pes_hpt, systems[0].type_names)
    gpu_ctx.set_emt(cols, pesm)
    # even bead numbers where every atom is transformed: the reference's normal modes are not orthonormal for odd ones
    nsteps = 4 if P > 16 or n > 4 else 10
    b = mdt.Batch(gpu_ctx, systems, dt=0.1, tsurf=100.0, tproj=120.0, pile_tau=50.0, andersen_time=1.0, seed=77)
    b.compute_forces()
    b.step(nsteps)
    out = b.get_state()
    b.close()
    for t, (s, o) in enumerate(zip(systems, out)):
        st = oracle.OracleState(s, cols, pesm, step=0.1, tsurf=100.0, tproj=120.0, pile_tau=50.0, andersen_time=1.0)
        st.calc_force()
        st.run(77, t, 1, nsteps)
        assert np.abs(o["r"] - st.r).max() <= 1e-8
        assert np.abs(o["v"] - st.v).max() <= 1e-8 * max(1.0, np.abs(st.v).max())
        assert np.abs(o["epot"] - st.epot).max() <= 1e-8 * max(1.0, np.abs(st.epot).max())
