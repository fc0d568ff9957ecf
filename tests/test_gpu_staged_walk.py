"""The staged walk of short stencils (k_plan_list): one step with the walks
chosen by the library against the same step with the per-lane walk forced,
bit for bit, and against the oracle (neighbour counts and lists exactly,
densities within the parity bar), at the edges of what it accepts: waves of
one to many x-rows, partial waves, rows that end at the grid's border, rows
and lists at and over their limits, colliding buckets, h above 1."""
import numpy as np
import pytest

import parity_util as pu
import sph_scenes
from test_gpu_production_walks import OracleState, _check_dump

pytestmark = pytest.mark.gpu
F32 = np.float32


def _scene(pos, h=0.1, box=2.0):
    pos = np.ascontiguousarray(pos, dtype=F32)
    vel = np.random.default_rng(5).normal(0.0, 0.1, size=pos.shape).astype(F32)
    return sph_scenes.Scene("staged", pos, vel, float(F32(0.02 * (h / 0.15) ** 3)), 1000.0, 1.0, 1.04, h, -9.8, 0.2,
                            1e-3, (-box, -box, -box), (box, box, box))


def _uniform(n, ext, seed=1, h=0.1, box=2.0):
    return _scene(np.random.default_rng(seed).uniform(-ext, ext, size=(n, 3)), h, box)


def _case(name):
    rng = np.random.default_rng(17)
    if name.startswith("n="):  # partial and whole waves, dense enough for neighbours
        n = int(name[2:])
        return _uniform(n, 0.05 * n ** (1.0 / 3.0))
    if name == "column":  # a column of cells along z: a wave spans many x-rows (more than the staged seven)
        return _scene(np.stack([rng.uniform(0, 0.1, 600), rng.uniform(0, 0.1, 600), rng.uniform(-1.9, 1.9, 600)], 1))
    if name == "seven rows":  # about nine particles per cell of a column: waves of six to eight x-rows
        return _scene(np.stack([rng.uniform(0, 0.1, 350), rng.uniform(0, 0.1, 350), rng.uniform(-1.9, 1.9, 350)], 1))
    if name == "line":  # along x: one x-row, far more cells than lanes
        return _scene(np.stack([rng.uniform(-1.9, 1.9, 1000), rng.uniform(0, 0.02, 1000),
                                rng.uniform(0, 0.02, 1000)], 1))
    if name == "border":  # particles at and beyond the walls: cells at the ends of every axis
        p = rng.uniform(-0.35, 0.35, size=(2000, 3))
        p[:600] = np.sign(p[:600]) * rng.uniform(0.25, 0.349, size=(600, 3))
        return _scene(p, box=0.3)
    if name == "row limit":  # rows of 96 candidates and more beside shorter ones
        p = rng.uniform(-0.5, 0.5, size=(1500, 3))
        p[:300] = rng.uniform(0.0, 1.0, size=(300, 3)) * [0.3, 0.1, 0.1]
        p[300:390] = [0.9, 0.9, 0.9] + rng.uniform(0.0, 1.0, size=(90, 3)) * [0.3, 0.1, 0.1]
        return _scene(p)
    if name == "list limit":  # clumps of 60 to 70 within h: lists of 63, 64 and 65 entries
        p = [rng.uniform(-0.02, 0.02, size=(m, 3)) + c for m, c in
             zip((63, 64, 65, 66, 67), rng.permutation(8)[:5, None] * [0.4, 0.3, -0.35] - [1.2, 1.0, -1.1])]
        return _scene(np.concatenate(p))
    if name == "collisions":  # the axis columns, where buckets double
        return _scene(rng.uniform(-0.12, 0.12, size=(400, 3)))
    if name == "h above 1":
        return _uniform(500, 4.0, h=1.5, box=10.0)
    raise ValueError(name)


CASES = ["n=1", "n=2", "n=63", "n=64", "n=65", "n=129", "n=3375", "column", "seven rows", "line", "border", "row limit",
         "list limit", "collisions", "h above 1"]


@pytest.mark.parametrize("name", CASES)
def test_staged_walk_equals_lane_walk_and_oracle(sph, orc32, name):
    sc = _case(name)
    out = []
    for lane_walk in (False, True):
        with sph.Context(sc.n, sph.settings(*sc.settings_args()), sph.box(sc.box_lo, sc.box_hi), sc.dt,
                         lane_walk=lane_walk) as ctx:
            ctx.upload(sc.pos, sc.vel)
            dump = ctx.walk_dump(lists=True)
            assert not dump["split"].any(), "premise: no task is split"
            ost = OracleState(orc32, sc, sc.pos, sc.vel)
            try:
                _check_dump(dump, ost.rows(np.arange(sc.n)), np.arange(sc.n), f"{name}, lane_walk={lane_walk}")
            finally:
                ost.close()
            ctx.step(1)
            out.append(ctx.download())
    for key in ("pos", "vel", "rho", "pressure", "ids"):
        assert out[0][key].tobytes() == out[1][key].tobytes(), f"{name}: {key} differs between the walks"
    s_o = orc32.settings(*sc.settings_args())
    ref, _, _, _, _ = pu.oracle_step(orc32, sc.pos, sc.vel, s_o, sc.dt, orc32.box(sc.box_lo, sc.box_hi))
    got = {k: np.zeros_like(out[0][k]) for k in ("rho", "pressure")}
    for k in got:
        got[k][out[0]["ids"]] = out[0][k]
    pu.assert_rho_p(got["rho"], got["pressure"], ref["density"], ref["pressure"], s_o, name)
