"""A scene on cells of h / 2 gives the same bytes alone and beside scenes on
cells of h (where another kernel plans its walks): clumps whose cut stencils
hold up to, and their whole ones more than, the 409 candidates that leave a
walk whole, denser and sparser ones, slow lanes."""
import numpy as np
import pytest

import sph_amd as A

pytestmark = pytest.mark.gpu
H = 0.1
S = A.settings(mass=0.002, h=H)
BOX = A.box((-2.0, -2.0, -2.0), (2.0, 2.0, 2.0))


def _clumps(m, width, seed):
    rng = np.random.default_rng(seed)
    centres = rng.uniform(-1.2, 1.2, (6, 3))
    pos = np.concatenate([c + rng.uniform(-0.5, 0.5, (m, 3)) * width * H for c in centres] +
                         [rng.uniform(-1.5, 1.5, (1500, 3))])
    return pos.astype(np.float32), rng.normal(0.0, 0.05, pos.shape).astype(np.float32)


@pytest.mark.parametrize("m,width", [(60, 1.0), (300, 1.5), (420, 1.5), (500, 2.0), (700, 2.5), (1500, 3.0), (800, 0.4)])
def test_fine_scene_alone_and_beside_a_coarse_one(m, width):
    pos, vel = _clumps(m, width, m)
    other = _clumps(200, 1.5, 7)
    got = []
    with A.Context(len(pos), S, BOX, 1e-4, cell_scale=0.5) as c:
        c.upload(pos, vel)
        c.step(2)
        got.append(c.download())
    with A.Batch([A.scene_desc(len(other[0]), S, BOX, 1e-4), A.scene_desc(len(pos), S, BOX, 1e-4, cell_scale=0.5)]) as b:
        b.upload(0, *other)
        b.upload(1, pos, vel)
        b.step(2)
        got.append(b.download(1))
    for key in ("ids", "rho", "pressure", "pos", "vel"):
        assert got[0][key].tobytes() == got[1][key].tobytes(), key
