"""Sums of unsplit walks: one step with the walks chosen by the library equals
the same step with the per-lane walk forced, bit for bit, for clumps at and
around the number of neighbours whose terms the staged walk holds (30 in one
z-layer of cells, 32 in two), and for dense ones walked as a union whose
lists overflow (64 and beyond)."""
import numpy as np
import pytest

import sph_scenes

pytestmark = pytest.mark.gpu
F32 = np.float32
H = 0.1


def _clumps(sizes, straddle, seed=3):
    rng = np.random.default_rng(seed)
    pos, edge = [], H * (1.0 + 2.0 ** -10)  # of a cell
    for k, m in enumerate(sizes):
        p = rng.uniform(-0.2 * H, 0.2 * H, size=(m, 3))
        # cell centres (counted from the wall at -2, one padding cell beside
        # it), clear of the axes; straddling: the clump's middle on the
        # upper face of the cell
        c = -2.0 + edge * np.array([6.5 + 7 * (k % 3), 8.5 + 5 * (k // 3), 9.5 + 3 * k])
        c[2] += 0.5 * edge * straddle
        pos.append(p + c)
    pos = np.concatenate(pos).astype(F32)
    vel = rng.normal(0.0, 0.1, size=pos.shape).astype(F32)
    return sph_scenes.Scene("clumps", pos, vel, float(F32(0.02 * (H / 0.15) ** 3)), 1000.0, 1.0, 1.04, H, -9.8, 0.2,
                            1e-3, (-2.0, -2.0, -2.0), (2.0, 2.0, 2.0))


@pytest.mark.parametrize("straddle", [0, 1])
@pytest.mark.parametrize("sizes", [(2, 3, 5, 9), (29, 30, 31), (31, 32, 33), (34, 35, 36), (64, 65, 66),
                                   (150, 200), (390, 409)])
def test_unsplit_sums_equal_the_lane_walks(sph, sizes, straddle):
    sc = _clumps(sizes, straddle)
    out = []
    for lane_walk in (False, True):
        with sph.Context(sc.n, sph.settings(*sc.settings_args()), sph.box(sc.box_lo, sc.box_hi), sc.dt,
                         lane_walk=lane_walk) as ctx:
            ctx.upload(sc.pos, sc.vel)
            assert not ctx.walk_dump()["split"].any(), "premise: no task is split"
            ctx.step(2)
            out.append(ctx.download())
    for key in ("pos", "vel", "rho", "pressure", "ids"):
        assert out[0][key].tobytes() == out[1][key].tobytes(), key
