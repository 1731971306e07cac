"""A captured chunk of steps follows a later mdt_batch_set_propagation: the host
chooses the propagator kernel and whether the COM velocity is removed (Andersen
or PILE atoms, src/md_algo.f90:37-71), and a graph captured before the change
holds the old choice.  Replayed and directly launched steps run the same kernels,
so the states are bitwise equal."""
import numpy as np
import pytest

from md_tian2_amd import geometry, mdt, pesfile

pytestmark = pytest.mark.gpu

V, L, A, P = geometry.PROP_VERLET, geometry.PROP_LANGEVIN, geometry.PROP_ANDERSEN, geometry.PROP_PILE


def _set_algo(b, algo):
    n = len(b.systems)
    i32 = np.ascontiguousarray(algo, dtype=np.int32)
    isp = np.ascontiguousarray(b.systems[0].is_proj, dtype=np.int32)
    t = np.full(n, 100.0)
    mdt._check(mdt.lib().mdt_batch_set_propagation(b.h, len(algo), mdt._ip(i32), mdt._ip(isp), 0.1, mdt._dp(t), mdt._dp(t),
                                                   50.0, 1.0))


# ring polymers (COM removal off and on), one-bead slabs (the lane-per-atom
# propagator and the chunked one)
@pytest.mark.parametrize("beads", [4, 1])
@pytest.mark.parametrize("first,then", [((P, P), (V, L)), ((V, L), (P, P)), ((V, A), (V, V)), ((V, V), (V, A))])
@pytest.mark.parametrize("split", [0, 1])
def test_replay_after_new_propagators(gpu_ctx, pes_hau, beads, first, then, split):
    g = np.random.default_rng(40 + beads)
    systems = [geometry.h_on_slab("Au", n=3, nlayers=4, nbeads=beads, rng=g, z0=2.2, tsurf=100.0) for _ in range(2)]
    for s in systems:
        s.r += g.normal(0, 0.02, s.r.shape) * ~s.fixed
    cols, pesm = pesfile.emt_tables(pes_hau, systems[0].type_names)
    gpu_ctx.set_emt(cols, pesm)
    out = []
    for chunk in (0, 5):
        b = mdt.Batch(gpu_ctx, systems, dt=0.1, tsurf=100.0, tproj=100.0, pile_tau=50.0, andersen_time=1.0, seed=5)
        b.set_split(split)
        b.set_graph(chunk)
        _set_algo(b, first)
        b.compute_forces()
        b.step(10)
        _set_algo(b, then)
        b.step(10)
        out.append(b.get_state())
        b.close()
    for a, c in zip(*out):
        for k in ("r", "v", "f", "epot"):
            assert np.array_equal(a[k], c[k]), k
