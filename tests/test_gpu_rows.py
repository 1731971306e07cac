"""k_replica's rows, pieces and flat lists at the sizes where they can go wrong.

Rows hold the pairs of the majority EMT type and are cut into pieces sorted by
length; the at most 4 atoms of the other type have lists of their own (flat
lists); batches of up to 512 workgroups keep the scanned rows in LDS.  Every
case is compared with the oracle's compute_emt restatement (pairs under the
minimum image, src/pes_emt_mod.f90:1204-1206).

Tolerance 1e-9 of the largest force (at least 1 eV/A): a pair's force is
rounded to 2^-43 eV/A (1.1e-13; at most 128 pairs an atom: 2e-12), its
terms are good to some 1e-13 relative (1 / sqrt to 4e-15, exponents up to 26 / A
times a distance of 6 A), and the sums cancel by no more than the number of
pairs."""
import numpy as np
import pytest

import oracle
from md_tian2_amd import geometry, mdt, pesfile

pytestmark = pytest.mark.gpu


def _check(ctx, pes, systems, steps=0, tol=1e-9, sample=3):
    cols, pesm = pesfile.emt_tables(pes, systems[0].type_names)
    ctx.set_emt(cols, pesm)
    b = mdt.Batch(ctx, systems, dt=0.2, tsurf=300.0, tproj=300.0, seed=3)
    b.compute_forces()
    if steps:
        b.step(steps)
    assert not b.status().any()
    out = b.get_state()
    for q in np.linspace(0, len(systems) - 1, min(sample, len(systems))).astype(int):
        s = systems[q].copy()
        s.r = out[q]["r"].copy()
        e, f, _ = oracle.emt_energy_forces(s, cols, pesm)
        assert np.abs(out[q]["epot"] - e).max() <= tol * max(1.0, np.abs(e).max())
        assert np.abs(out[q]["f"] - f).max() <= tol * max(1.0, np.abs(f).max()), (q, np.abs(out[q]["f"] - f).max())
    b.close()


# one wavefront's worth of atoms and one more, a single atom of the metal, even
# cells (half-cell ties: entries without a fixed image), launches on both sides of
# the few-workgroup bound, with the rows of the first launch and kept ones
@pytest.mark.parametrize("n,layers,ntraj", [(1, 1, 2), (3, 7, 512), (4, 4, 513), (4, 4, 3), (3, 4, 600), (6, 4, 5)])
@pytest.mark.parametrize("steps", [0, 25])
def test_rows_and_batch_sizes(gpu_ctx, pes_hau, n, layers, ntraj, steps):
    rng = np.random.default_rng(100 * n + layers)
    systems = []
    for k in range(ntraj):
        s = geometry.h_on_slab("Au", n=n, nlayers=layers, nfixed=min(2, layers - 1), rng=rng, z0=1.6 + 0.01 * (k % 400), einc=2.0)
        s.r[1:] += rng.normal(0, 0.04, s.r[1:].shape) * ~s.fixed[1:]
        systems.append(s)
    _check(gpu_ctx, pes_hau, systems, steps=steps)


# projectile-type atoms: 4 (flat lists, also of each other) and 5 (rows of both types)
@pytest.mark.parametrize("nh", [0, 2, 4, 5])
@pytest.mark.parametrize("steps", [0, 20])
def test_flat_atoms(gpu_ctx, pes_hau, nh, steps):
    rng = np.random.default_rng(7 + nh)
    systems = []
    for _ in range(3):
        s = geometry.h_on_slab("Au", n=5, nlayers=4, rng=rng, z0=1.5)
        top = np.flatnonzero(s.idx == 1)[:nh - 1] if nh else []
        for j in top:  # a top-layer atom becomes a projectile-type one above its site
            s.idx[j] = 0
            s.mass[j] = s.mass[0]
            s.r[j, 0, 2] += 1.2
            s.v[j] = 0.0
        if nh == 0:
            s.idx[0] = 1
            s.r[0, 0, 2] = 2.6
        systems.append(s)
    _check(gpu_ctx, pes_hau, systems, steps=steps)


def test_flat_list_overflow(gpu_ctx, pes_hau):
    """An H inside a compressed lattice has more near partners than its list
    holds: both passes test every atom instead."""
    rng = np.random.default_rng(5)
    s = geometry.h_on_slab("Au", n=8, nlayers=8, a=2.9, rng=rng, z0=0.0)
    s.r[0, 0, :] = s.r[1 + 64 * 3 + 27, 0, :] + [0.8, 0.5, 0.9]
    cols, pesm = pesfile.emt_tables(pes_hau, s.type_names)
    gpu_ctx.set_emt(cols, pesm)
    b = mdt.Batch(gpu_ctx, [s], dt=0.1)
    b.tune(tpa=1, nbcap=160)
    b.compute_forces()
    o = b.get_state()[0]
    e, f, _ = oracle.emt_energy_forces(s, cols, pesm)
    d = s.r[1:, 0] - s.r[0, 0]
    fr = d @ np.linalg.inv(s.simbox).T
    d = (fr - np.rint(fr)) @ s.simbox.T
    assert (np.linalg.norm(d, axis=1) < 6.0).sum() > 128
    assert np.abs(o["epot"] - e).max() <= 1e-9 * np.abs(e).max()
    assert np.abs(o["f"] - f).max() <= 1e-9 * max(1.0, np.abs(f).max())


def test_large_terms(gpu_ctx, pes_hau):
    """Overlapping atoms: pair forces beyond the 255 eV/A that the fast
    conversion takes, in rows (Au-Au) and in a flat list (H-Au)."""
    s = geometry.h_on_slab("Au", n=5, nlayers=4, rng=np.random.default_rng(2), z0=1.5)
    s.r[2, 0, :] = s.r[1, 0, :] + [0.15, 0.1, 0.2]
    s.r[0, 0, :] = s.r[12, 0, :] + [0.05, 0.02, 0.08]
    cols, pesm = pesfile.emt_tables(pes_hau, s.type_names)
    gpu_ctx.set_emt(cols, pesm)
    b = mdt.Batch(gpu_ctx, [s], dt=0.1)
    b.compute_forces()
    o = b.get_state()[0]
    e, f, _ = oracle.emt_energy_forces(s, cols, pesm)
    assert np.abs(o["epot"] - e).max() <= 1e-9 * max(1.0, np.abs(e).max())
    assert np.abs(o["f"] - f).max() <= 1e-9 * max(1.0, np.abs(f).max())


@pytest.mark.parametrize("precision", [0, 1])
def test_far_image_of_a_kept_pair(gpu_ctx, pes_hau, precision):
    """In a strongly skewed cell the image that a kept pair rounds to may be 60 A
    away while another one, which it could round to, is near: the pair is listed and
    counts nothing.  Two atoms half a cell apart along two axes, a and b
    nearly parallel: both fractional differences just below 1/2 give (a + b) / 2, one
    of them above 1/2 would give (a - b) / 2, 3.2 A long."""
    s = geometry.h_on_slab("Au", n=1, nlayers=4, nfixed=1, z0=1.7)  # H and 4 Au
    s.simbox = np.array([[60.0, 60.0, 0.0], [0.0, 6.4, 0.0], [0.0, 0.0, 40.0]])
    frac = np.array([[0.1, 0.32, 0.55], [0.1, 0.1, 0.5], [0.5999, 0.5998, 0.5], [0.1, 0.1, 0.58], [0.6001, 0.5998, 0.58]])
    s.r[:, 0] = frac @ s.simbox.T
    cols, pesm = pesfile.emt_tables(pes_hau, s.type_names)
    gpu_ctx.set_emt(cols, pesm)
    e, f, _ = oracle.emt_energy_forces(s, cols, pesm)
    assert np.abs(f).max() > 1e-3
    b = mdt.Batch(gpu_ctx, [s], dt=0.1)
    b.set_precision(precision)
    b.set_keep(1)
    for _ in range(2):  # the build and a launch on the kept rows
        b.compute_forces()
    o = b.get_state()[0]
    b.close()
    tol = 1e-9 if precision == 0 else 1e-5  # the FP32 pair terms' bar
    assert np.abs(o["epot"] - e).max() <= tol * max(1.0, np.abs(e).max())
    assert np.abs(o["f"] - f).max() <= tol * max(1.0, np.abs(f).max())


def test_flat_sums_do_not_depend_on_the_order(gpu_ctx, pes_hau):
    """An H pushed by 60 atoms at once, each by less than the fast conversion's
    limit, together by more than FP64 holds in steps of the grid: its force has the
    same bits in whatever order the atoms are numbered."""
    g = np.random.default_rng(3)
    s = geometry.h_on_slab("Au", n=6, nlayers=4, rng=g, z0=2.7)
    s.r[1:61, 0] = s.r[0, 0] + [0.5, 0.0, 0.0] + g.normal(0, 0.08, (60, 3))
    cols, pesm = pesfile.emt_tables(pes_hau, s.type_names)
    gpu_ctx.set_emt(cols, pesm)
    _, f, _ = oracle.emt_energy_forces(s, cols, pesm)
    assert np.abs(f[0, 0]).max() > 4096.0
    systems = []
    for k in range(8):
        q = s.copy()
        q.r[1:] = s.r[1:][g.permutation(s.natoms - 1)] if k else s.r[1:]
        systems.append(q)
    b = mdt.Batch(gpu_ctx, systems, dt=0.1)
    b.tune(tpa=1, nbcap=144)
    b.compute_forces()
    out = b.get_state()
    b.close()
    assert np.abs(out[0]["f"][0] - f[0]).max() <= 1e-9 * np.abs(f).max()
    for o in out[1:]:
        assert np.array_equal(o["f"][0], out[0]["f"][0])


@pytest.mark.parametrize("lost", [0, 20])
@pytest.mark.parametrize("keep", [0, 1])
def test_an_atom_without_a_position(gpu_ctx, pes_hau, lost, keep):
    """An atom at NaN (an H or an Au of a trajectory that blew up) has no partners;
    the batch goes on and the other atoms' forces are those without it."""
    s = geometry.h_on_slab("Au", n=5, nlayers=4, rng=np.random.default_rng(8), z0=1.6)
    cols, pesm = pesfile.emt_tables(pes_hau, s.type_names)
    gpu_ctx.set_emt(cols, pesm)
    rest = np.delete(np.arange(s.natoms), lost)
    w = geometry.System(s.type_names, s.idx[rest], s.mass[rest], s.fixed[rest], s.algo, s.simbox, s.r[rest], s.v[rest])
    _, f, _ = oracle.emt_energy_forces(w, cols, pesm)
    q = s.copy()
    q.r[lost] = np.nan
    b = mdt.Batch(gpu_ctx, [s, q], dt=0.1)
    b.set_keep(keep)
    for _ in range(2):
        b.compute_forces()
    assert not b.status().any()
    o = b.get_state()
    b.close()
    assert np.abs(o[1]["f"][rest] - f).max() <= 1e-9 * max(1.0, np.abs(f).max())
    assert not o[1]["f"][lost].any()
    _, f, _ = oracle.emt_energy_forces(s, cols, pesm)
    assert np.abs(o[0]["f"] - f).max() <= 1e-9 * max(1.0, np.abs(f).max())
