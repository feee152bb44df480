"""Handles that change after they have run: an adjoint bound to one with captured steps, codes taken away,
maps uploaded again. The next run equals a fresh handle's bit for bit."""

import ctypes

import numpy as np
import pytest

from fullwave25_amd import engine
from tests.helpers import raw_inputs

pytestmark = pytest.mark.gpu


def inputs(shape, nt=24, **more):
    rng = np.random.default_rng(sum(shape))
    c = np.full(shape, 1500.0)
    c[shape[0] // 2:] = 1560.0
    pts = np.stack([rng.integers(8, n - 8, 60) for n in shape], 1)
    sig = rng.standard_normal((20, nt)).astype(np.float32)
    return raw_inputs(shape, c=c, rho=950 + 100 * rng.random(shape), nt=nt, icc=pts[:20], icmat=sig, outc=pts[10:50],
                      icczero=pts[50:], modt=2, **more)


def fresh(inp):
    with engine.HipSimulation(inp) as sim:
        sim.run(inp.nt)
        return sim.sensors(), sim.field("p")


@pytest.mark.parametrize("kernels", ["stream:64:5", "tile:32", "percell", "brick:32:1"])
def test_adjoint_on_a_handle_with_captured_steps(monkeypatch, kernels):
    """fw_adj_create replaces a handle's kernels and its point table after steps were captured."""
    inp = inputs((24, 26, 44) if kernels.startswith("brick") else (60, 300))
    monkeypatch.delenv("FULLWAVE_HIP_KERNELS", raising=False)
    want = fresh(inp)
    monkeypatch.setenv("FULLWAVE_HIP_KERNELS", kernels)
    with engine.HipSimulation(inp) as sim:
        sim.set_graph_steps(4)
        sim.run(inp.nt)
        np.testing.assert_array_equal(sim.sensors(), want[0])
        adj = ctypes.c_void_p()
        engine._check(sim.lib, sim.lib.fw_adj_create(sim._h, 8, ctypes.byref(adj)))
        try:
            for _ in range(2):
                sim.reset()
                sim.run(inp.nt)
                np.testing.assert_array_equal(sim.sensors(), want[0])
                np.testing.assert_array_equal(sim.field("p"), want[1])
        finally:
            sim.lib.fw_adj_destroy(adj)


@pytest.mark.parametrize("graph_steps", [0, 4])
@pytest.mark.parametrize("isotropic", [True, False])
def test_bricks_whose_codes_go_and_come_back(monkeypatch, isotropic, graph_steps):
    """Brick kernels need relaxation codes: codes switched off and on, one axis map that differs and the
    old one again, between runs of one handle."""
    monkeypatch.delenv("FULLWAVE_HIP_KERNELS", raising=False)
    relax = {"v": {"kappa": 1.05, "d": (9e3, 4e5), "alpha": (3e6, 9e7)}, "p": {"kappa": 1.02, "d": (3e4, 5e5), "alpha": (1.5e7, 1.1e8)}}
    inp = inputs((24, 26, 44), isotropic=isotropic, relax=relax)
    want = fresh(inp)
    name = "bpmlx2" if isotropic else "bpmlz2"
    own = inp.maps[name] * np.linspace(0.2, 1.0, inp.maps[name].size, dtype=np.float32).reshape(inp.shape)
    changed = inputs((24, 26, 44), isotropic=isotropic, relax=relax)
    changed.maps[name] = own
    other = fresh(changed)
    assert (other[1] != want[1]).any()
    brick = {"variant": "brick", "width": 32, "chunk": 1}
    with engine.HipSimulation(inp) as sim:
        sim.set_kernel_config({"velocity": brick, "pressure": brick})
        sim.set_graph_steps(graph_steps)

        def again(ref):
            for _ in range(2):
                sim.reset()
                sim.run(inp.nt)
                np.testing.assert_array_equal(sim.sensors(), ref[0])
                np.testing.assert_array_equal(sim.field("p"), ref[1])

        again(want)
        sim.set_relaxation_codes(False)
        again(want)
        sim.set_relaxation_codes(True)
        again(want)
        sim.upload(name, own)
        again(other)
        sim.upload(name, inp.maps[name])
        again(want)


def test_adjoint_outlives_its_simulation():
    """Closing the simulation first leaves an adjoint that refuses to run and closes like any other."""
    from fullwave25_amd.adjoint import HipAdjoint

    inp = inputs((24, 26, 44))
    adj = HipAdjoint(inp, checkpoint_every=8)
    adj.forward()
    weights = np.ones((inp.n_records, inp.ncoordsout), np.float32)
    assert np.abs(adj.backward(weights)[0]).max() > 0
    adj.sim.close()
    with pytest.raises(engine.EngineError, match="destroyed"):
        adj.forward()
    with pytest.raises(engine.EngineError, match="destroyed"):
        adj.backward(weights)
    adj.close()
