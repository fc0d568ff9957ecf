"""The union walk of dense waves (candidates staged in LDS, no test per
candidate): one step against the oracle (neighbour counts exactly, density,
pressure and force within the parity bar) where it can go wrong: waves whose
lanes lie in separate clumps (segments), split and whole walks, chunks that
end inside a row, h above 1 (no clamp to [0, 1]); and values that are not
finite, which must reach only the particles they reach on the per-lane
walk."""
import numpy as np
import pytest

import parity_util as pu
import sph_scenes
from test_gpu_production_walks import OracleState, _check_dump, _check_forces

pytestmark = pytest.mark.gpu
F32 = np.float32


def _clumps(sizes, centres, h=0.1, sigma=0.4, seed=3, box=2.0):
    rng = np.random.default_rng(seed)
    pos = np.concatenate([rng.normal(0.0, sigma * h, size=(m, 3)) + c for m, c in zip(sizes, centres)]).astype(F32)
    vel = rng.normal(0.0, 0.1, size=pos.shape).astype(F32)
    return sph_scenes.Scene("clumps", pos, vel, float(F32(0.02 * (h / 0.15) ** 3)), 1000.0, 1.0, 1.04, h, -9.8, 0.2,
                            1e-3, (-box, -box, -box), (box, box, box))


# centres keep clear of the axis planes, whose buckets collide (such waves walk per lane)
SCENES = {
    "one clump, whole walks": lambda: _clumps([700], [[0.75, 0.95, -0.85]]),
    "one clump, split walks": lambda: _clumps([5000], [[0.75, 0.95, -0.85]]),
    "clumps in one x-row": lambda: _clumps([900, 911, 923], [[-1.3, 0.95, 0.85], [0.55, 0.95, 0.85], [1.4, 0.95, 0.85]],
                                           sigma=0.2),
    "clumps in separate rows": lambda: _clumps([450 + 17 * k for k in range(8)],
                                               [[0.5 + 0.1 * (k % 2), 0.45 + 0.15 * k, 0.55 + 0.12 * k] for k in range(8)],
                                               sigma=0.15),
    "h above 1": lambda: _clumps([3000], [[7.5, 9.5, -8.5]], h=1.5, box=20.0),
}


@pytest.mark.parametrize("name", SCENES)
@pytest.mark.parametrize("scale", [1.0, 0.5])
def test_union_walk_matches_the_oracle(sph, orc32, name, scale):
    sc = SCENES[name]()
    with sph.Context(sc.n, sph.settings(*sc.settings_args()), sph.box(sc.box_lo, sc.box_hi), sc.dt,
                     cell_scale=scale) as ctx:
        ctx.upload(sc.pos, sc.vel)
        dump = ctx.walk_dump(lists=True)
        ctx.step(1)
        d = ctx.download()
    assert dump["union"].mean() > 0.5, "premise: most waves walk a union"
    ids = np.arange(sc.n)
    ost = OracleState(orc32, sc, sc.pos, sc.vel)
    try:
        _check_dump(dump, ost.rows(ids), ids, name)
        if scale == 1.0:
            _check_forces(sph, orc32, sc, sc.pos, sc.vel, ids, ost, name)
        rho, prs = ost.rho_p_by_id() if ost.have_density else (None, None)
    finally:
        ost.close()
    if rho is not None:
        got = {k: np.zeros_like(d[k]) for k in ("rho", "pressure")}
        for k in got:
            got[k][d["ids"]] = d[k]
        pu.assert_rho_p(got["rho"], got["pressure"], rho, prs, ost.s, name)


@pytest.mark.parametrize("what", ["nan position", "inf position", "nan velocity", "inf velocity", "huge velocity"])
def test_values_that_are_not_finite_stay_where_they_belong(sph, what):
    """Particle 5 (in the clump) and one in its neighbourhood but out of
    reach carry the value: the union walk gives the per-lane walk's result,
    particle for particle, with the same ones not finite."""
    sc = _clumps([1500], [[0.75, 0.95, -0.85]])
    sc.pos = np.concatenate([sc.pos, [[0.75 + 0.19, 0.95 + 0.19, -0.85]]]).astype(F32)
    sc.vel = np.concatenate([sc.vel, np.zeros((1, 3), F32)])
    value = {"nan": np.nan, "inf": np.inf, "huge": 1e30}[what.split()[0]]
    for i in (5, sc.n - 1):
        (sc.pos if "position" in what else sc.vel)[i, 1] = value
    got = []
    for lane_walk in (False, True):
        with sph.Context(sc.n, sph.settings(*sc.settings_args()), sph.box(sc.box_lo, sc.box_hi), sc.dt,
                         lane_walk=lane_walk, keep_force=True) as ctx:
            ctx.upload(sc.pos, sc.vel)
            ctx.step(1)
            p, _ = ctx.download_particles(transforms=False)
            ids = ctx.download()["ids"]
        out = np.zeros_like(p)
        out[ids] = p
        got.append(out)
    u, l = got
    for key in ("position", "velocity", "force", "density"):
        a, b = u[key].astype(np.float64), l[key].astype(np.float64)
        assert np.array_equal(np.isnan(a), np.isnan(b)), f"{what}: {key} is NaN elsewhere"
        assert np.array_equal(np.isinf(a), np.isinf(b)), f"{what}: {key} is inf elsewhere"
        # both walks add the same terms in parts of their own: 2^-23 per
        # addition, of sums whose terms are at most the largest of them all
        ok = np.isfinite(a)
        tol = 1500 * 2.0 ** -23 * np.abs(b[ok]).max() if key == "force" else 1e-5 * np.abs(b[ok]) + 1e-5
        if what != "huge velocity" or key == "density":
            assert np.all(np.abs(a[ok] - b[ok]) <= tol), f"{what}: {key}"
