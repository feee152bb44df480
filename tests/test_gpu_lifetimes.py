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
