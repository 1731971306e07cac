"""Host code of the C interface on two devices, without a GPU: libmdt_gpu.so runs on
a HIP runtime that keeps device memory in host memory and executes no kernel
(tests/native/fake_hip.cpp).  Whichever device the calling thread has current, a
call allocates, copies and launches on its context's.  A skin switched off and
on again leaves the launch shape that tuning chose."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SETUP = """
import ctypes, os, sys
sys.path.insert(0, %r)
import numpy as np
from md_tian2_amd import geometry, mdt, nene, pesfile
hip = ctypes.CDLL(None)
def other(dev):  # what else the thread does with the other device
    hip.hipSetDevice(dev)
pes = pesfile.load_pes(os.path.join(%r, "md_tian2_amd", "pes", "EMT-HAu.pes"))
rng = np.random.default_rng(1)
systems = [geometry.h_on_slab("Au", n=3, nlayers=4, nbeads=p, rng=rng, z0=2.0) for p in (1, 4)]
cols, pesm = pesfile.emt_tables(pes, systems[0].type_names)
""" % (ROOT, ROOT)

TWO = SETUP + """
ctx = [mdt.Context(d) for d in (0, 1)]
for c in ctx:
    c.set_emt(cols, pesm)
b = [mdt.Batch(ctx[d], [systems[k] for k in (0, 1)], dt=0.1, tsurf=300.0, tproj=300.0) for d in (0, 1)]
for d in (0, 1):
    for call in (lambda x: x.set_state([s.r for s in systems], [s.v for s in systems]),
                 lambda x: x.get_state(),
                 lambda x: x.compute_forces(),
                 lambda x: x.step(3),
                 lambda x: x.status(clear=True),
                 lambda x: x.set_observe(proj_ul=6.05, adsorption=(2.5, 3.5)),
                 lambda x: x.step(2),
                 lambda x: x.observables(),
                 lambda x: x.tune(0),
                 lambda x: x.set_bead_mode(1) or x.set_bead_mode(0),
                 lambda x: x.ctx.compute_emt(systems[1]),
                 lambda x: x.get_state()):
        other(1 - d)
        call(b[d])
what = ctypes.create_string_buffer(200)
n = hip.fake_hip_violations(what, 200)
print(n, what.value.decode())
sys.exit(1 if n or not hip.fake_hip_launches() else 0)
"""


@pytest.fixture(scope="module")
def fake_hip(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("hip") / "fake_hip.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-o", so,
                    os.path.join(ROOT, "tests", "native", "fake_hip.cpp")], check=True)
    return so


def run(so, script, **env):
    pre = ":".join(x for x in (os.environ.get("LD_PRELOAD", ""), so) if x)
    return subprocess.run([sys.executable, "-c", script], env={**os.environ, "LD_PRELOAD": pre, **env}, timeout=100,
                          capture_output=True, text=True)


def test_every_call_uses_its_contexts_device(fake_hip):
    out = run(fake_hip, TWO, FAKE_HIP_DEVICES="2")
    assert out.returncode == 0, out.stdout + out.stderr


SKIN = SETUP + """
s = geometry.h_on_slab("Au", n=6, nlayers=4, rng=rng)
c = mdt.Context(0)
c.set_emt(cols, pesm)
b = mdt.Batch(c, [s] * 600, dt=0.1)
tune_at, shapes = float(os.environ["TUNE_AT"]), []
b.set_list_skin(tune_at)
b.tune(0)
shapes.append(b.class_shapes())
for skin in (0.0, 0.3):
    b.set_list_skin(skin)
    shapes.append(b.class_shapes())
print([(x[0]["tpa"], x[0]["keep"], x[0]["block"]) for x in shapes])
"""


# the second candidate is one lane per atom on half the lanes: 145 atoms, 128 lanes
@pytest.mark.parametrize("tune_at,want", [("0.3", [(1, 1, 128), (1, 0, 128), (1, 1, 128)]),
                                          ("0.0", [(1, 0, 128), (1, 0, 128), (1, 1, 128)])])
def test_skin_off_and_on_keeps_the_tuned_shape(fake_hip, tune_at, want):
    out = run(fake_hip, SKIN, TUNE_AT=tune_at, FAKE_HIP_BEST="2")
    assert out.returncode == 0, out.stderr
    assert out.stdout.strip() == str(want)


FULL = SETUP + """
s = geometry.h_on_slab("Au", n=3, nlayers=4, rng=rng)
c = mdt.Context(0)
c.set_emt(cols, pesm)
b = mdt.Batch(c, [s] * 20000, dt=0.1)
b.compute_forces()
n0 = hip.fake_hip_launches()
b.compute_forces()
n1 = hip.fake_hip_launches()
b.step(2)
b.get_state()
print(b.class_shapes()[0]["keep"], n1 - n0)
"""


# 20000 trajectories of 37 atoms: 125 MB of state, 540 MB of lists
@pytest.mark.parametrize("mb,want", [(800, "1 1"), (360, "0 3")])
def test_a_batch_whose_lists_do_not_fit_still_runs(fake_hip, mb, want):
    """Without room for a list slot per replica the lists are rebuilt in fewer slots, a
    slice of the batch at a time."""
    out = run(fake_hip, FULL, FAKE_HIP_BYTES=str(mb << 20))
    assert out.returncode == 0, out.stderr
    assert out.stdout.strip() == want
