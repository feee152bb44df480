"""3D per-cell kernels on both sides of the size from which their memory variables go past the caches (by the
arrays that a step touches: codes, one set of maps, a set per axis): equal to the marching kernels bit for bit."""

import dataclasses

import numpy as np
import pytest

from fullwave25_amd import engine
from tests.helpers import raw_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("model,shape", [("codes", (150, 150, 180)), ("codes", (144, 150, 190)), ("maps", (150, 152, 121)),
                                         ("maps", (145, 150, 128)), ("axes", (120, 112, 110)), ("axes", (119, 112, 128)),
                                         ("spacing", (150, 152, 121)), ("spacing", (145, 150, 128))])
def test_per_cell_kernels_equal_the_marching_ones(monkeypatch, model, shape):
    rng = np.random.default_rng(31)
    nt = 4
    relax = {"v": {"kappa": 1.05, "d": (9e3, 4e5), "alpha": (3e6, 9e7)}, "p": {"kappa": 1.02, "d": (3e4, 5e5), "alpha": (1.5e7, 1.1e8)}}
    c = np.where(np.arange(shape[0])[:, None, None] < shape[0] // 2, 1500.0, 1560.0) * np.ones(shape)
    pts = np.stack([rng.integers(8, n - 8, 80) for n in shape], 1)
    inp = raw_inputs(shape, c=1500.0 if model == "axes" else c, nt=nt, relax=relax, icc=pts[:20], outc=pts[10:], isotropic=model != "axes",
                     icmat=rng.standard_normal((20, nt)).astype(np.float32))
    if model == "axes":
        inp.maps["bpmlz2"] = inp.maps["bpmlz2"] * np.float32(0.75)
    if model == "spacing":
        inp = dataclasses.replace(inp, dz=inp.dx * 1.2)
    p0 = np.zeros(shape, np.float32)
    core = tuple(slice(8, n - 8) for n in shape)
    p0[core] = rng.standard_normal(shape).astype(np.float32)[core]
    got = []
    for kernels in ("percell", "pipe:512:16"):
        print(f"{model} {shape}: {kernels}", flush=True)
        monkeypatch.setenv("FULLWAVE_HIP_KERNELS", kernels)
        with engine.HipSimulation(inp) as sim:
            sim.set_relaxation_codes(model != "maps")
            sim.set_field("p", p0)
            sim.run(nt)
            got.append([sim.sensors()] + [sim.field(f) for f in ("p", "vx", "vy", "vz")])
    assert np.abs(got[0][1]).max() > 0
    for a, b in zip(*got):
        np.testing.assert_array_equal(a, b)
