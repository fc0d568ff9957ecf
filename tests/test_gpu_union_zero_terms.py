"""Union walks meet candidates that are no neighbours, and places without a
candidate, without a test each: what these add must be nothing at all, also
where lengths come near the distance such places are put at, or the force's
constants overflow float on their own.  Compared with the per-lane walk, which
tests every candidate."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
F32 = np.float32


def _both(sph, s, box, pos, vel, steps=1):
    out = []
    for lane_walk in (False, True):
        with sph.Context(len(pos), s, box, 1e-3, lane_walk=lane_walk, keep_force=True) as ctx:
            ctx.upload(pos, vel)
            dump = ctx.walk_dump(lists=True)
            ctx.step(steps)
            p, _ = ctx.download_particles(transforms=False)
            ids = ctx.download()["ids"]
        by_id = np.zeros_like(p)
        by_id[ids] = p
        out.append((dump, by_id))
    return out


@pytest.mark.parametrize("n", [700, 5000])
def test_constants_that_overflow(sph, n):
    """A clump, and in its cell one particle out of everyone's reach: the
    force constant times the pressure overflows, for that one times zero."""
    h = 0.1
    s = sph.settings(mass=0.02, h=h)
    s.spikyGrad = -3.0e38
    edge = h * (1.0 + 2.0 ** -10)
    low = -2.0 + edge * np.array([24.0, 27.0, 31.0])  # of a cell, clear of the axes
    rng = np.random.default_rng(n)
    pos = low + edge * rng.uniform(0.02, 0.2, (n, 3))
    pos[n // 2] = low + 0.97 * edge
    pos = pos.astype(F32)
    assert np.linalg.norm(np.delete(pos, n // 2, 0).astype(float) - pos[n // 2], axis=1).min() > h
    vel = rng.normal(0.0, 0.1, (n, 3)).astype(F32)
    (dump, got), (_, ref) = _both(sph, s, sph.box((-2.0,) * 3, (2.0,) * 3), pos, vel)
    assert dump["union"].all() and not dump["listed"].any(), "premise: union walks, force included"
    assert dump["count"][n // 2] == 0 and not ref["force"][n // 2].any()
    for key in ("force", "position", "velocity", "density"):
        assert np.array_equal(got[key][n // 2], ref[key][n // 2]), key


@pytest.mark.parametrize("h", [1e15, 2e17, 1e18])
def test_lengths_like_the_far_places(sph, h):
    """Some of the particles lie where the walks put places without a
    candidate, or within h of there."""
    rng = np.random.default_rng(4)
    s = sph.settings(mass=0.02, h=h)
    far = np.full((3, 3), [[1.0e18], [2.0 ** 60], [1.02e18]])
    pos = np.concatenate([rng.uniform(-2.5, 2.5, (2000, 3)) * h + far[1], far,
                          rng.uniform(-0.3, 0.3, (500, 3)) * h, rng.uniform(-1.0, 1.0, (500, 3)) * [h, h, 40 * h]])
    pos = pos.astype(F32)
    vel = rng.normal(0.0, 0.1, pos.shape).astype(F32)
    (got, p), (ref, q) = _both(sph, s, sph.box((-4e18,) * 3, (4e18,) * 3), pos, vel)
    for key in ("count", "listed", "list_count", "list"):
        same = got["listed"] & ref["listed"] if key.startswith("list") else slice(None)
        assert np.array_equal(got[key][same], ref[key][same]), key
    for key in ("density", "position"):
        # NaN (a square of h^6 overflows) in the same places, the same otherwise
        a, b = p[key].astype(np.float64), q[key].astype(np.float64)
        assert np.array_equal(np.isnan(a), np.isnan(b)), key
        assert np.array_equal(a[~np.isnan(a)], b[~np.isnan(a)]), key
