"""The angular network kernels' wavefront per centre, where it can go wrong:
centres with 0, 1, 2 and 3 neighbours, lists around and above 64 entries, the
image search and the minimum image, angular functions of one and of several
neighbour-pair classes, and every number of wavefronts per workgroup.
Against the NENE oracle with the bars of the network's other tests (2e-4
eV/atom, 5e-3 eV/A); against each other bitwise.
"""
import numpy as np
import pytest

import nene_oracle as no
from md_tian2_amd import geometry, mdt, nene

pytestmark = pytest.mark.gpu

TYPES = [("H", True), ("Au", False)]


def _universe(pos, cell):
    """Atom 0 is H, the others Au."""
    N = len(pos)
    return geometry.System(TYPES, np.array([0] + [1] * (N - 1), np.int32),
                           np.array([geometry.MASS_AMU["H"]] + [geometry.MASS_AMU["Au"]] * (N - 1)) * geometry.AMU2MASS,
                           np.zeros((N, 1, 3), bool), np.array([geometry.PROP_VERLET, geometry.PROP_VERLET], np.int32),
                           np.asarray(cell, float), np.asarray(pos, float).reshape(N, 1, 3).copy(), np.zeros((N, 1, 3)))


def _cluster(n):
    pos = [[0, 0, 0], [1.7, 0, 0], [-0.4, 2.1, 0.3], [0.5, -0.9, 2.6]][:n]
    return _universe(np.array(pos, float) + 30.0, np.eye(3) * 60.0)


def _bulk(ncell, g):
    """H in an octahedral site of fcc Au: 78 and more neighbours within 6.5 A."""
    b = geometry.bulk_fcc("Au", ncell=ncell)
    pos = np.concatenate([[[2.04, 0.0, 0.0]], b.r[:, 0]])
    return _universe(pos + g.normal(0, 0.05, pos.shape), b.simbox)


def _slab(g, n):
    s = geometry.h_on_slab("Au", n=n, nlayers=4, rng=g, z0=1.6)
    return _universe(s.r[:, 0] + g.normal(0, 0.05, s.r[:, 0].shape), s.simbox)


def _model(frames, g, classes):
    """hau_design with random weights, scaled on the frames; classes: angular
    functions on H-Au pairs beside the Au-Au ones (not factored)."""
    m = nene.hau_design()
    if classes:
        H, AU = 1, 79
        m.sf[AU] += [nene.SymFunc(3, H, AU, eta, 0.0, lam, z, m.rcmax()) for eta in (0.01, 0.05) for z in (1.0, 2.0) for lam in (-1.0, 1.0)]
        m.sort()
    for z in m.elements:
        m.gmin[z], m.gmax[z], m.gavg[z] = np.zeros(m.nsf(z)), np.ones(m.nsf(z)), np.zeros(m.nsf(z))
    nene.init_weights(m, g)
    om, Gs = no.Model(m), {1: [], 79: []}
    for s in frames:
        G = om.descriptors(om.elem_index([1] + [79] * (s.natoms - 1)), s.r[:, 0] / nene.BOHR2ANG, s.simbox.T / nene.BOHR2ANG)
        Gs[1].append(G[:1])
        Gs[79].append(G[1:])
    nene.set_scaling(m, {z: np.concatenate(v) for z, v in Gs.items()}, margin=0.5)
    return m


@pytest.mark.parametrize("classes", [False, True])
def test_centres_against_the_oracle(gpu_ctx, classes):
    g = np.random.default_rng(31)
    frames = [_cluster(1), _cluster(2), _cluster(3), _cluster(4), _bulk(3, g), _bulk(4, g), _slab(g, 3), _slab(g, 6)]
    frames = frames[1:]  # a lone atom has no descriptors to scale by; it is checked below
    m = _model(frames, g, classes)
    om = no.Model(m)
    gpu_ctx.set_nn(m, TYPES)
    for s in [_cluster(1)] + frames:
        e, f, _ = gpu_ctx.compute_nene(s)
        E, _, F, _ = om.energy_forces(om.elem_index([1] + [79] * (s.natoms - 1)), s.r[:, 0] / nene.BOHR2ANG,
                                      s.simbox.T / nene.BOHR2ANG)
        assert abs(e[0] - E * nene.HA2EV) / s.natoms <= 2e-4, s.natoms
        assert np.abs(f[:, 0] - F * nene.HABOHR2EVANG).max() <= 5e-3, s.natoms


def test_workgroup_sizes_agree_bitwise(gpu_ctx):
    """Up to 256 replicas run 16 wavefronts each, more 8."""
    g = np.random.default_rng(32)
    frames = [_slab(g, 3) for _ in range(5)]
    gpu_ctx.set_nn(_model(frames, g, False), TYPES)
    got = []
    for n in (5, 257):
        b = mdt.Batch(gpu_ctx, [frames[k % 5] for k in range(n)], dt=0.1)
        b.set_pes(1)
        b.compute_forces()
        got.append(b.get_state())
        b.close()
    for out in got[1:]:
        for k, o in enumerate(out):
            assert np.array_equal(o["f"], got[0][k % 5]["f"]) and np.array_equal(o["epot"], got[0][k % 5]["epot"])


def test_forces_keep_single_precision(gpu_ctx):
    """The shipped angular network on thermal slabs, against 64 bits: forces to 1e-5 and
    energies to 2e-6 eV/atom.  A pair's terms round some 12 times (2^-24 each) and its
    exponent, up to 30, once (2^-24 30 = 2e-6); sums over many pairs average, and the
    network, whose operands keep 24 bits, adds a few 2^-24 a layer, so the
    2-norm stays some 3e-6 and below 1e-5.  Operands of 16 bits (two bf16 parts: 2^-17
    = 8e-6 each, over three layers and the way back) or the hardware's sine and
    cosine (2^-18 absolute) give 2e-5."""
    import os

    g = np.random.default_rng(33)
    m = nene.load(os.path.join(os.path.dirname(mdt.LIB_PATH), "nn", "hau"))
    om = no.Model(m)
    gpu_ctx.set_nn(m, TYPES)
    diff = norm = 0.0
    for n in (3, 5, 6):
        for z in (1.6, 3.0):
            s = geometry.h_on_slab("Au", n=n, nlayers=4, rng=g, z0=z)
            u = _universe(s.r[:, 0] + g.normal(0, 0.05, s.r[:, 0].shape), s.simbox)
            e, f, _ = gpu_ctx.compute_nene(u)
            E, _, F, _ = om.energy_forces(om.elem_index([1] + [79] * (u.natoms - 1)), u.r[:, 0] / nene.BOHR2ANG,
                                          u.simbox.T / nene.BOHR2ANG)
            F = F * nene.HABOHR2EVANG
            diff += ((f[:, 0] - F) ** 2).sum()
            norm += (F ** 2).sum()
            assert abs(e[0] - E * nene.HA2EV) / u.natoms <= 2e-6
    print("network forces: relative error %.2e" % np.sqrt(diff / norm))
    assert np.sqrt(diff / norm) <= 1e-5
