"""The reverse step of 2D grids with many sound speeds on tall tiles (16 x 64 cells, each with a table of
its own sets): from 32 sets and 1280 tiles of 8 x 64, where half of those or more hold several. Equal to the
per-cell kernels bit for bit, at the edges of tall tiles and of the rule."""

import numpy as np
import pytest

from tests.helpers import raw_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["cells", "layers", "few"])
@pytest.mark.parametrize("shape,sets", [((656, 1040), 32), ((649, 1041), 33), ((665, 1047), 256), ((641, 1039), 40), ((656, 1024), 250)])
def test_2d_reverse_tall_tiles_equal_the_per_cell_gathers(monkeypatch, shape, sets, kind):
    from fullwave25_amd.adjoint import HipAdjoint

    rng = np.random.default_rng(21)
    nt = 5
    speed = rng.integers(0, sets, shape)
    if kind == "layers":
        speed = np.broadcast_to((np.arange(shape[0]) * sets // shape[0])[:, None], shape).copy()
    if kind == "few":  # several sets in a corner, one elsewhere
        speed[:, shape[1] // 3:] = 7
    speed.flat[:sets] = np.arange(sets)  # every set occurs: in the ghost border, beside updated cells of others
    pts = np.stack([rng.integers(8, n - 8, 200) for n in shape], 1)
    inp = raw_inputs(shape, c=1450.0 + speed, rho=950 + 100 * rng.random(shape), nt=nt, icc=pts[:40], outc=pts[30:],
                     icmat=rng.standard_normal((40, nt)).astype(np.float32), icczero=pts[40:50])
    assert inp.dmap.shape[-1] == sets
    weights = rng.standard_normal((inp.n_records, inp.ncoordsout)).astype(np.float32)
    got = []
    for mode, every in (("percell", nt), ("tiles", nt), ("tiles", 2)):
        monkeypatch.setenv("FULLWAVE_HIP_ADJ_GATHERS", mode)
        print(f"{shape} {sets} {kind}: {mode} every {every}", flush=True)
        with HipAdjoint(inp, checkpoint_every=every) as adj:
            adj.forward()
            got.append(adj.backward(weights))
    assert np.abs(got[0][0]).max() > 0
    for new in got[1:]:
        for g, ref in zip(new, got[0]):
            np.testing.assert_array_equal(g, ref)
