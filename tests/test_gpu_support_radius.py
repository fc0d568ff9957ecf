"""The neighbour test is the settings' h2, whatever their h: a caller's
settings with h2 below or above h * h keep it in every walk of the density and
force passes (neighbour lists, whole and split union walks, per lane), as the
reference's loops do (src/sph.cpp:40-66, 92-118: dist2 < settings.h2, then
h - r of either sign).  One clump in a single grid cell and a single reference
cell, so that every pair is a candidate; counts exactly, densities and forces
within the parity bar of the 64-bit oracle (the 32-bit one's own sums of 5000
terms are up to 1.3 bars from it)."""
import numpy as np
import pytest

import parity_util as pu

pytestmark = pytest.mark.gpu
F32 = np.float32
H = 0.1
EDGE = H * (1.0 + 2.0 ** -10)  # of a grid cell; the first one starts one edge below the wall at -2
ARGS = (0.02 * (H / 0.15) ** 3, 1000.0, 1.0, 1.04, H, -9.8, 0.2)


def _clump(n, seed):
    """n points in a box of 0.7 h inside one grid cell and one reference cell."""
    rng = np.random.default_rng(seed)
    corner = []
    for first in (6, 9, 12):
        lo = next(x for x in (-2.0 + EDGE * (k + 0.02 * j) for k in range(first + 20, first + 30) for j in range(15))
                  if 0.02 < (x / H) % 1.0 < 0.28)
        corner.append(lo)
    at = rng.uniform(0.0, 0.7 * H, (n, 3))
    at[:2] = [[0.05 * H] * 3, [0.65 * H] * 3]  # 1.04 h apart
    pos = (np.array(corner) + at).astype(F32)
    cell = np.floor((pos.astype(np.float64) + 2.0 + EDGE) / EDGE)
    assert (cell == cell[0]).all() and (np.trunc(pos / F32(H)) == np.trunc(pos[0] / F32(H))).all()
    return pos, rng.normal(0.0, 0.1, (n, 3)).astype(F32)


# 30 with lists, 700 whole union walks, 5000 split ones
@pytest.mark.parametrize("n", [30, 700, 5000])
@pytest.mark.parametrize("lane_walk", [False, True])
@pytest.mark.parametrize("factor", [0.6, 1.0, 1.2])
def test_h2_is_the_neighbour_test(sph, orc64, n, lane_walk, factor):
    pos, vel = _clump(n, n)
    s, s_o = sph.settings(*ARGS), orc64.settings(*ARGS)
    s.h2 = float(F32(factor) * F32(s.h2))
    s_o.h2 = s.h2
    lo, hi = (-2.0,) * 3, (2.0,) * 3
    with sph.Context(n, s, sph.box(lo, hi), 1e-3, keep_force=True, lane_walk=lane_walk) as ctx:
        ctx.upload(pos, vel)
        count = ctx.walk_dump()["count"]
        ctx.step(1)
        p, _ = ctx.download_particles(transforms=False)
        ids = ctx.download()["ids"]
    got = np.zeros_like(p)
    got[ids] = p
    p_o = orc64.particles(pos, vel, ids=np.arange(n))
    table = orc64.prepare(p_o, s_o)
    off, idx = orc64.neighbors(p_o, table, s_o)
    orc64.density(p_o, table, s_o)
    orc64.forces(p_o, table, s_o)
    orc64.free_table(table)
    order = p_o["acceleration"][:, 0].astype(np.int64)
    ref, rows = np.zeros_like(p_o), [None] * n
    ref[order] = p_o
    for k in range(n):
        rows[order[k]] = order[idx[off[k]:off[k + 1]]]
    beyond = [np.linalg.norm(pos[r].astype(np.float64) - pos[i], axis=1).max(initial=0.0) > H
              for i, r in enumerate(rows)]
    assert np.array_equal(count, [len(r) for r in rows])
    assert any(beyond) == (factor > 1.0), "premise: pairs farther than h only with the larger h2"
    pu.assert_rho_p(got["density"], got["pressure"], ref["density"], ref["pressure"], s_o)
    # sum of the terms' magnitudes, as parity_util.force_scale, with |h - r|
    scale = np.zeros(n)
    for i, r in enumerate(rows):
        d = np.linalg.norm(pos[r].astype(np.float64) - pos[i], axis=1)
        hr = np.abs(H - d)
        press = ref["pressure"][i].astype(np.float64) + ref["pressure"][r]
        dv = np.linalg.norm(vel[r].astype(np.float64) - vel[i], axis=1)
        m = float(s_o.mass)
        scale[i] = np.sum(m * np.abs(press) / (2.0 * ref["density"][r]) * abs(float(s_o.spikyGrad)) * hr * hr +
                          float(s_o.viscosity) * m * dv / ref["density"][r] * float(s_o.spikyLap) * hr)
    pu.assert_force(got["force"], ref["force"].astype(np.float64), scale, f"n={n} factor={factor}")
