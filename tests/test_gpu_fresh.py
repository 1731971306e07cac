"""New positions before every force call: from the second such call on, k_replica's
rows serve one launch (read from LDS as scanned where few workgroups run, cut
but not kept where many do), all types in them; calls that go on from their positions
build rows to keep.  Every form sums the same rounded terms: forces and
energies of fresh positions have the same bits in all of them, and equal the
oracle's to the 1e-9 of the rows' other tests."""
import numpy as np
import pytest

import oracle
from md_tian2_amd import geometry, mdt, pesfile

pytestmark = pytest.mark.gpu


def _systems(n, layers, ntraj, beads, g):
    out = []
    for k in range(ntraj):
        s = geometry.h_on_slab("Au", n=n, nlayers=layers, nfixed=2, nbeads=beads, rng=g, z0=1.6 + 0.01 * (k % 400), tsurf=300.0)
        s.r[1:] += g.normal(0, 0.05, s.r[1:].shape) * ~s.fixed[1:]
        out.append(s)
    return out


# one wavefront's lanes and more, an even cell of 10 A (half-cell ties), folded layers,
# lanes that loop over the atoms, batches on both sides of the few-workgroup bound
@pytest.mark.parametrize("n,layers,ntraj,beads", [(3, 4, 3, 1), (4, 4, 3, 1), (4, 4, 600, 1), (6, 4, 520, 1), (5, 7, 2, 1),
                                                  (8, 8, 2, 1), (12, 6, 1, 1), (3, 4, 5, 4)])
@pytest.mark.parametrize("precision", [0, 1])
def test_fresh_positions(gpu_ctx, pes_hau, n, layers, ntraj, beads, precision):
    g = np.random.default_rng(1000 * n + ntraj)
    systems = _systems(n, layers, ntraj, beads, g)
    cols, pesm = pesfile.emt_tables(pes_hau, systems[0].type_names)
    gpu_ctx.set_emt(cols, pesm)

    def batch(keep):
        b = mdt.Batch(gpu_ctx, systems, dt=0.2, tsurf=300.0, tproj=300.0, seed=3)
        b.set_precision(precision)
        b.set_keep(keep)
        return b

    forms = [batch(-1), batch(0), batch(1)]
    for call in range(4):
        rs = [s.r + g.normal(0, 0.02, s.r.shape) * ~s.fixed for s in systems]
        got = []
        for k, b in enumerate(forms):
            b.set_state(rs)
            b.compute_forces()
            if k == 2 and beads == 1:  # goes on from its positions: its rows are kept ones
                # (with beads every call takes the ring-polymer step)
                b.compute_forces()
            got.append(b.get_state())
        for o in got[1:]:
            for a, c in zip(got[0], o):
                for key in ("f", "epot"):
                    assert np.array_equal(a[key], c[key]), (call, key)
        if beads == 1:
            s = systems[-1].copy()
            s.r = rs[-1]
            e, f, _ = oracle.emt_energy_forces(s, cols, pesm)
            tol = 1e-9 if precision == 0 else 1e-5
            assert np.abs(got[0][-1]["epot"] - e).max() <= tol * max(1.0, np.abs(e).max())
            assert np.abs(got[0][-1]["f"] - f).max() <= tol * max(1.0, np.abs(f).max())
    for b in forms:
        b.close()


@pytest.mark.parametrize("ntraj", [3, 1030])
@pytest.mark.parametrize("chunk", [0, 1, 4])
def test_steps_between_fresh_positions(gpu_ctx, pes_hau, ntraj, chunk):
    """Single steps and runs of steps after each new state, launched directly and from
    graphs, as halves and whole: the states equal those with rows rebuilt at every
    launch to rounding (1e-9, as the kept lists' tests)."""
    g = np.random.default_rng(ntraj + chunk)
    systems = _systems(3, 4, ntraj, 1, g)
    cols, pesm = pesfile.emt_tables(pes_hau, systems[0].type_names)
    gpu_ctx.set_emt(cols, pesm)
    forms = []
    for keep in (-1, 0):
        b = mdt.Batch(gpu_ctx, systems, dt=0.2, tsurf=300.0, tproj=300.0, seed=3)
        b.set_keep(keep)
        b.set_graph(chunk)
        forms.append(b)
    v = [s.v for s in systems]
    for nsteps in (1, 1, 1, 5, 1, 1, 8):
        rs = [s.r + g.normal(0, 0.02, s.r.shape) * ~s.fixed for s in systems]
        got = []
        for b in forms:
            b.set_state(rs, v)
            b.compute_forces()
            b.set_state(rs, v)
            b.step(nsteps)
            got.append(b.get_state())
        for a, c in zip(*got):
            assert np.abs(a["r"] - c["r"]).max() <= 1e-9
            assert np.abs(a["f"] - c["f"]).max() <= 1e-9 * max(1.0, np.abs(c["f"]).max())
    for b in forms:
        b.close()
