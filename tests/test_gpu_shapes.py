"""Every forward kernel family and shape computes the same sums in the same order
(``tap``, ``memory_step``, ``corrected``, ``velocity_step``, ``pressure_step`` in fw_internal.h), so
traces and fields agree bit for bit, at the grid sizes where a tile can go wrong: one row or one
column quad more or less than whole tiles, the smallest grid, unequal spacings, one sound speed
(the wavefront-wide coefficient path) and a medium that changes from cell to cell."""

import dataclasses

import numpy as np
import pytest

from fullwave25_amd import engine
from tests.helpers import raw_inputs

pytestmark = pytest.mark.gpu
SHAPES = ["stream:64:5", "stream:256:16", "tile:8", "tile:16", "tile:32"]


def medium(shape, kind, nt=24, **more):
    """A loaded grid (initial pressure everywhere) of one medium, of patches, or of cells."""
    rng = np.random.default_rng(sum(shape))
    relax = {"v": {"kappa": 1.05, "d": (9e3, 4e5), "alpha": (3e6, 9e7)}, "p": {"kappa": 1.02, "d": (3e4, 5e5), "alpha": (1.5e7, 1.1e8)}}
    c, rho = 1540.0, 1000.0
    if kind != "one":
        c = np.full(shape, 1500.0)
        c[shape[0] // 3:] = 1560.0
        c[:, shape[1] // 2:] += 20.0
        rho = 950 + 100 * rng.random(shape)
    if kind == "cells":
        c = rng.choice([1500.0, 1523.0, 1580.0], size=shape)
    nd = len(shape)
    src = [[n // 2 for n in shape], [8] * nd]
    out = [[n - 9 for n in shape], [n // 2 + 3 for n in shape], [9] * nd]
    sig = rng.standard_normal((2, nt)).astype(np.float32)
    return raw_inputs(shape, c=c, rho=rho, nt=nt, relax=relax, icc=src, icmat=sig, outc=out, **more)


def run(inp, shape, monkeypatch, codes=True):
    monkeypatch.setenv("FULLWAVE_HIP_KERNELS", shape)
    p0 = np.random.default_rng(1).standard_normal(inp.shape).astype(np.float32)
    ghost = tuple(slice(8, n - 8) for n in inp.shape)
    start = np.zeros(inp.shape, np.float32)
    start[ghost] = p0[ghost]
    with engine.HipSimulation(inp) as sim:
        sim.set_relaxation_codes(codes)
        sim.set_field("p", start)
        sim.run(inp.nt)
        fields = ["p", "vx", "vy"] + (["vz"] if inp.ndim == 3 else [])
        return [sim.sensors()] + [sim.field(f) for f in fields]


@pytest.mark.parametrize("kind", ["one", "patches", "cells"])
@pytest.mark.parametrize("shape", [(17, 20), (32, 144), (33, 148), (47, 128), (49, 276), (81, 132)])
def test_2d_families_agree_bit_for_bit(monkeypatch, shape, kind):
    inp = medium(shape, kind)
    if kind == "patches":
        inp = dataclasses.replace(inp, dy=inp.dx * 1.25)
    want = run(inp, "percell", monkeypatch)
    assert np.abs(want[1]).max() > 0
    for s in SHAPES:
        print(f"{shape} {kind}: {s}", flush=True)
        for codes in (True, False):
            for got, ref in zip(run(inp, s, monkeypatch, codes), want):
                np.testing.assert_array_equal(got, ref)


@pytest.mark.parametrize("kind", ["one", "patches", "cells"])
@pytest.mark.parametrize("shape", [(17, 19, 21), (21, 26, 96), (18, 33, 131)])
def test_3d_families_agree_bit_for_bit(monkeypatch, shape, kind):
    inp = medium(shape, kind, nt=10)
    if kind == "patches":
        inp = dataclasses.replace(inp, dz=inp.dx * 1.2)
    want = run(inp, "percell", monkeypatch)
    assert np.abs(want[1]).max() > 0
    for s in ("percell", "stream:512:5", "pipe:512:4", "pipelite:512:7", "pipelite:1024:3"):
        print(f"{shape} {kind}: {s}", flush=True)
        for codes in (True, False):
            for got, ref in zip(run(inp, s, monkeypatch, codes), want):
                np.testing.assert_array_equal(got, ref)


@pytest.mark.parametrize("model", ["isotropic", "exponential"])
@pytest.mark.parametrize("kind", ["one", "patches", "cells"])
@pytest.mark.parametrize("shape", [(17, 17, 17), (20, 24, 40), (21, 25, 41), (18, 33, 109), (19, 32, 131)])
def test_3d_bricks_equal_the_per_cell_kernels(monkeypatch, shape, kind, model):
    """Brick kernels at the edges of bricks (4 x 8 x 32 cells): one cell, whole bricks, one more; shared,
    per-cell and mixed coefficients; both orders of the bricks; sources, pressure release and sensors on
    corners, ghost border and brick edges fused into the pressure launch and on their own; two shots; the
    adjoint's taped run. Bit for bit."""
    from fullwave25_amd.adjoint import HipAdjoint

    rng = np.random.default_rng(11)
    corners = np.stack(np.meshgrid(*[[0, n - 1] for n in shape], indexing="ij"), -1).reshape(-1, 3)
    inside = np.stack([rng.integers(0, n, 30) for n in shape], 1)
    edge = inside.copy()
    edge[:, -1] = np.minimum(rng.choice([8, 31, 32, 33], 30), shape[-1] - 1)
    src, out, air = (np.concatenate([corners, inside[i::3], edge[i::3]]) for i in range(3))
    nt = 9
    more = {}
    if model == "exponential":
        more = {"a_exp": 0.98 + 0.02 * rng.random(shape)}
    c = {"one": 1540.0, "patches": np.where(np.arange(shape[0])[:, None, None] < shape[0] // 2, 1500.0, 1560.0) * np.ones(shape),
         "cells": rng.choice([1500.0, 1523.0, 1580.0], size=shape)}[kind]
    inp = raw_inputs(shape, c=c, rho=950 + 100 * rng.random(shape), nt=nt, icc=src, modt=2, outc=np.concatenate([out, src[4:], air[:6]]),
                     icmat=rng.standard_normal((len(src), nt)).astype(np.float32), icczero=air, **more)
    want = run(inp, "percell", monkeypatch)
    assert np.abs(want[1]).max() > 0
    for order in (0, 1):
        for fused in ("1", "0"):
            monkeypatch.setenv("FULLWAVE_HIP_FUSED_BOUNDARY", fused)
            print(f"{shape} {kind} {model}: order {order} fused {fused}", flush=True)
            for got, ref in zip(run(inp, f"brick:32:{order}", monkeypatch), want):
                np.testing.assert_array_equal(got, ref)
    monkeypatch.delenv("FULLWAVE_HIP_FUSED_BOUNDARY")
    shots = np.stack([inp.icmat, 0.5 * inp.icmat[::-1]])
    traces = {}
    for k in ("percell", "brick:32:1"):
        monkeypatch.setenv("FULLWAVE_HIP_KERNELS", k)
        with engine.HipSimulation(inp, shots=shots) as sim:
            sim.run(nt)
            traces[k] = sim.sensors()
    np.testing.assert_array_equal(traces["brick:32:1"], traces["percell"])
    monkeypatch.delenv("FULLWAVE_HIP_KERNELS")
    weights = rng.standard_normal((inp.n_records, inp.ncoordsout)).astype(np.float32)
    grads = []
    for variant, width in (("percell", 0), ("brick", 32)):
        one = {"variant": variant, "width": width, "chunk": 0}
        with HipAdjoint(inp, checkpoint_every=4, kernel_config={"velocity": one, "pressure": one}) as adj:
            assert adj.sim.kernel_config()["velocity"]["variant"] == variant
            adj.forward()
            grads.append(adj.backward(weights))
    for a, b in zip(*grads):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("model", ["isotropic", "exponential"])
@pytest.mark.parametrize("kind", ["one", "patches", "cells"])
@pytest.mark.parametrize("shape", [(19, 21, 22), (20, 24, 40), (21, 25, 41), (30, 33, 109)])
def test_3d_reverse_bricks_meet_the_per_cell_gathers(monkeypatch, shape, kind, model):
    """The reverse step on bricks: gradients as the per-cell kernels' (the same terms summed in another
    order: sums of 60 terms with unit roundoff 6e-8, 3.6e-6 a gather, over 9 steps of two gathers: 6.5e-5
    of the largest value), the same bit for bit for any checkpoint spacing (the fused start of a step and
    the start on its own), with records on source and release points and brick edges."""
    from fullwave25_amd.adjoint import HipAdjoint

    rng = np.random.default_rng(12)
    nt = 9
    pts = np.stack([rng.integers(8, n - 8, 60) for n in shape], 1)
    pts[:12, -1] = np.minimum(rng.choice([8, 31, 32, 33], 12), shape[-1] - 9)
    src, air = pts[:16], pts[16:24]
    out = np.concatenate([pts[24:], src[:6], air[:4], pts[30:36]])
    c = {"one": 1540.0, "patches": np.where(np.arange(shape[0])[:, None, None] < shape[0] // 2, 1500.0, 1560.0) * np.ones(shape),
         "cells": rng.choice([1500.0, 1523.0, 1580.0], size=shape)}[kind]
    more = {"a_exp": 0.98 + 0.02 * rng.random(shape)} if model == "exponential" else {}
    inp = raw_inputs(shape, c=c, rho=950 + 100 * rng.random(shape), nt=nt, icc=src, outc=out, icczero=air,
                     icmat=rng.standard_normal((len(src), nt - 3)).astype(np.float32), **more)
    weights = rng.standard_normal((inp.n_records, inp.ncoordsout)).astype(np.float32)
    got = {}
    for mode, every in (("percell", nt), ("bricks", nt), ("bricks", 4), ("bricks", 1)):
        monkeypatch.setenv("FULLWAVE_HIP_ADJ_GATHERS", mode)
        print(f"{shape} {kind} {model}: {mode} every {every}", flush=True)
        with HipAdjoint(inp, checkpoint_every=every) as adj:
            adj.forward()
            got[mode, every] = adj.backward(weights)
    for k in range(2):
        ref, new = got["percell", nt][k], got["bricks", nt][k]
        assert np.abs(ref).max() > 0
        assert np.abs(new - ref).max() <= 6.5e-5 * np.abs(ref).max()
        for every in (4, 1):
            np.testing.assert_array_equal(got["bricks", every][k], new)


@pytest.mark.parametrize("model", ["isotropic", "per_axis", "exponential"])
@pytest.mark.parametrize("kind", ["one", "patches", "cells"])
@pytest.mark.parametrize("shape", [(21, 26), (24, 80), (25, 81), (40, 150), (67, 211)])
def test_2d_reverse_tiles_equal_the_per_cell_gathers(monkeypatch, shape, kind, model):
    """The reverse step on tiles of 8 x 64 cells, at the edges of tiles (part of one, whole tiles, one more),
    with tiles of one coefficient set, of several, and of both kinds side by side (patches), equal to the
    per-cell kernels bit for bit, for any checkpoint spacing."""
    from fullwave25_amd.adjoint import HipAdjoint

    rng = np.random.default_rng(14)
    nt = 9
    pts = np.stack([rng.integers(8, n - 8, 60) for n in shape], 1)
    pts[:12, -1] = np.minimum(rng.choice([8, 71, 72, 73], 12), shape[-1] - 9)
    src, air = pts[:16], pts[16:24]
    out = np.concatenate([pts[24:], src[:6], air[:4], pts[30:36]])
    c = {"one": 1540.0, "patches": np.where(np.arange(shape[0])[:, None] < shape[0] // 2, 1500.0, 1560.0) * np.ones(shape),
         "cells": rng.choice([1500.0, 1523.0, 1580.0], size=shape)}[kind]
    more = {"a_exp": 0.98 + 0.02 * rng.random(shape)} if model == "exponential" else {"isotropic": model == "isotropic"}
    inp = raw_inputs(shape, c=c, rho=950 + 100 * rng.random(shape), nt=nt, icc=src, outc=out, icczero=air,
                     icmat=rng.standard_normal((len(src), nt - 3)).astype(np.float32), **more)
    if kind == "patches":
        inp = dataclasses.replace(inp, dy=inp.dx * 1.25)
    weights = rng.standard_normal((inp.n_records, inp.ncoordsout)).astype(np.float32)
    got = []
    for mode, every in (("percell", nt), ("tiles", nt), ("tiles", 4)):
        monkeypatch.setenv("FULLWAVE_HIP_ADJ_GATHERS", mode)
        print(f"{shape} {kind} {model}: {mode} every {every}", flush=True)
        with HipAdjoint(inp, checkpoint_every=every) as adj:
            adj.forward()
            got.append(adj.backward(weights))
    assert np.abs(got[0][0]).max() > 0
    for new in got[1:]:
        for g, ref in zip(new, got[0]):
            np.testing.assert_array_equal(g, ref)


@pytest.mark.parametrize("model", ["isotropic", "per_axis", "exponential"])
@pytest.mark.parametrize("shape", [(17, 17), (21, 65), (40, 200), (17, 18, 19), (19, 21, 67)])
def test_per_cell_boundary_work_matches_boundary_launch(monkeypatch, shape, model):
    """The per-cell pressure kernels do the step's sources, pressure release and sensors for the points
    of their tiles: points in the ghost border, at the grid's corners and on tile edges, repeated and on
    each other, equal to the boundary pass launched on its own, bit for bit."""
    rng = np.random.default_rng(3)
    nd = len(shape)
    corners = np.stack(np.meshgrid(*[[0, n - 1] for n in shape], indexing="ij"), -1).reshape(-1, nd)
    inside = np.stack([rng.integers(0, n, 40) for n in shape], 1)
    edge = inside.copy()
    edge[:, -1] = np.minimum(rng.choice([8, 63, 64, 65], 40), shape[-1] - 1)
    src, out, air = (np.concatenate([corners, inside[i::3], edge[i::3]]) for i in range(3))
    out = np.concatenate([out, src[4:], air[:6], out[:3]])
    sig = rng.standard_normal((len(src), 9)).astype(np.float32)
    kw = {"isotropic": model != "per_axis"}
    if model == "exponential":
        kw = {"a_exp": 0.98 + 0.02 * rng.random(shape)}
    inp = raw_inputs(shape, c=rng.choice([1500.0, 1523.0], size=shape), rho=950 + 100 * rng.random(shape), nt=17, icc=src,
                     icmat=sig, outc=out, icczero=air, modt=2, **kw)
    got = {}
    for fused in ("1", "0"):
        monkeypatch.setenv("FULLWAVE_HIP_FUSED_BOUNDARY", fused)
        got[fused] = run(inp, "percell", monkeypatch)
    assert np.abs(got["1"][0]).max() > 0
    for a, b in zip(got["1"], got["0"]):
        np.testing.assert_array_equal(a, b)


def test_checkpointed_run_on_other_kernels_keeps_its_points(monkeypatch):
    """An adjoint replaces marching kernels by the tiled ones: the untaped steps of a checkpointed
    forward run then record the same traces as a plain run, bit for bit."""
    from fullwave25_amd.adjoint import HipAdjoint

    monkeypatch.delenv("FULLWAVE_HIP_KERNELS", raising=False)
    rng = np.random.default_rng(9)
    shape = (60, 300)
    pts = np.stack([rng.integers(8, n - 8, 200) for n in shape], 1)
    sig = rng.standard_normal((50, 30)).astype(np.float32)
    inp = raw_inputs(shape, c=rng.choice([1500.0, 1523.0], size=shape), nt=30, icc=pts[:50], icmat=sig, outc=pts[40:190],
                     icczero=pts[190:])
    pin = {k: {"variant": "stream", "width": 64, "chunk": 5} for k in ("velocity", "pressure")}
    with engine.HipSimulation(inp) as sim:
        sim.run(inp.nt)
        want = sim.sensors()
    with HipAdjoint(inp, checkpoint_every=7, kernel_config=pin) as adj:
        got = adj.forward()
    assert np.abs(want).max() > 0
    np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("kernels", ["percell", "tile:8", "stream:128:8", "pipe:512:4"])
@pytest.mark.parametrize("shape", [(33, 148), (17, 21), (18, 26, 43)])
def test_per_axis_maps_that_are_the_same_run_as_isotropic(monkeypatch, shape, kernels):
    """Per-axis inputs with one set of maps on every axis equal the isotropic run bit for bit; one
    voxel of one axis map that differs (also uploaded after a run) takes the per-axis path again and
    meets the FP64 oracle at the engine's tolerance (relative L2 1e-4)."""
    import oracle

    if kernels.startswith("pipe") != (len(shape) == 3) and kernels != "percell":
        pytest.skip("family of the other dimension")
    if kernels.startswith("tile") and shape[1] % 4:
        pytest.skip("unaligned rows")
    iso, axes = medium(shape, "cells", nt=16), medium(shape, "cells", nt=16, isotropic=False)
    want = run(iso, kernels, monkeypatch)
    for got, ref in zip(run(axes, kernels, monkeypatch), want):
        np.testing.assert_array_equal(got, ref)
    last = "y" if len(shape) == 2 else "z"
    m = axes.maps[f"bpml{last}2"].copy()
    m[(*(n // 2 for n in shape[:-1]), shape[-1] // 2 + 1)] *= 0.25  # beside the source
    other = dataclasses.replace(axes, maps={**axes.maps, f"bpml{last}2": m})
    got = run(other, kernels, monkeypatch)
    with engine.HipSimulation(axes) as sim:  # the map arrives after a run
        sim.run(1)
        sim.upload(f"bpml{last}2", m)
        sim.reset()
        start = np.zeros(shape, np.float32)
        core = tuple(slice(8, n - 8) for n in shape)
        start[core] = np.random.default_rng(1).standard_normal(shape).astype(np.float32)[core]
        sim.set_field("p", start)
        sim.run(other.nt)
        np.testing.assert_array_equal(sim.field("p"), got[1])
    o = oracle.OracleSimulation(other, 64)
    o.set_field("p", start)
    o.run(other.nt)
    err = np.linalg.norm(got[1] - o.field("p")) / np.linalg.norm(o.field("p"))
    assert err <= 1e-4, err
    assert (got[1] != want[1]).any()
