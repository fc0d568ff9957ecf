"""Replacing one scene of a batch leaves its grid, keys and automatic cell
size to the next call that needs them: each such call sees what it would see
after a first upload, the other scenes' particles keep what the last step left
them, and what no grid can hold is refused by the upload."""
import numpy as np
import pytest

import sph_amd as A

pytestmark = pytest.mark.gpu
F32 = np.float32
S = A.settings(mass=0.02, h=0.1)
BOX = A.box((-2.0, -2.0, -2.0), (2.0, 2.0, 2.0))
SIDE = 52  # a lattice of 52^3 particles chooses cells of h / 2
N = SIDE ** 3


def _lattice(seed=3):
    g = np.stack(np.meshgrid(*[np.arange(SIDE)] * 3, indexing="ij"), -1).reshape(-1, 3)
    return (g * 0.05 - 1.5 + np.random.default_rng(seed).uniform(-0.005, 0.005, g.shape)).astype(F32)


def _cloud(n, seed):
    rng = np.random.default_rng(seed)
    return rng.uniform(-0.5, 0.5, (n, 3)).astype(F32), rng.normal(0.0, 0.5, (n, 3)).astype(F32)


def _batch():
    return A.Batch([A.scene_desc(N, S, BOX, 1e-3, auto_grid=True), A.scene_desc(3000, S, BOX, 1e-3)])


def _replaced():
    """A batch that has run, its scene 0 replaced since by the lattice."""
    b = _batch()
    b.upload(0, _lattice(8))
    b.upload(1, *_cloud(3000, 5))
    b.step(2)
    b.upload(0, _lattice())
    return b


def test_walk_dump_of_a_replaced_scene():
    with _replaced() as b:
        got = b.walk_dump(0, lists=True)
    with _batch() as b:  # the same company: which kernel walks depends on it
        b.upload(0, _lattice())
        b.upload(1, *_cloud(3000, 5))
        ref = b.walk_dump(0, lists=True)
    for key, value in ref.items():  # the lists' order is that of the cells
        assert np.array_equal(got[key], value), key


def test_autotune_of_a_replaced_scene():
    with _replaced() as b:
        b.autotune(2)
        assert b.grid_info(0)[0] == 0.5


def test_other_scenes_keep_their_hashes():
    with _replaced() as b:
        b.step(1)
        before = b.download_particles(1)[0]
        assert len(np.unique(before["hash"])) > 1
        b.upload(0, _lattice())
        for query in (lambda: b.grid_info(0), lambda: b.walk_dump(0), lambda: b.grid_info(1)):
            query()
            assert b.download_particles(1)[0].tobytes() == before.tobytes()
            assert not b.download_particles(0)[0]["hash"].any()  # no step yet
        b.upload(0, _lattice(9))
        assert b.grid_info(0)[0] == 0.5
        assert b.download_particles(1)[0].tobytes() == before.tobytes()
        assert not b.download_particles(0)[0]["hash"].any()
        b.upload(1, *_cloud(3000, 6))
        assert not b.download_particles(1)[0]["hash"].any()
        b.step(1)
        fresh = b.download_particles(1)[0]
    with A.Context(3000, S, BOX, 1e-3) as c:
        c.upload(*_cloud(3000, 6))
        c.step(1)
        assert c.download_particles()[0].tobytes() == fresh.tobytes()


def test_upload_refuses_what_no_grid_holds():
    """Two scenes of 17 million particles may have 64 cells a particle: both
    spread out, 2^31.006 cells."""
    n = 17_000_000
    h = 0.01
    s = A.settings(mass=1e-9, h=h)
    edge = h * (1.0 + 2.0 ** -10)
    # 1030 x 1023 x 1023 cells, one of them beside each wall: 63.4 a particle
    size = np.array([1027.5, 1020.5, 1020.5]) * edge
    box = A.box((0.0, 0.0, 0.0), (0.0, 0.0, 0.0))
    pos = np.random.default_rng(1).random((n, 3), dtype=F32)
    with A.Batch([A.scene_desc(n, s, box, 1e-3)] * 2) as b:
        b.upload(0, pos)
        b.upload(1, pos)
        pos *= size.astype(F32)
        pos[0], pos[1] = 0.0, size
        b.upload(0, pos)
        with pytest.raises(A.SphError) as err:
            b.upload(1, pos)
        assert err.value.code == A.SPH_E_LIMIT
        with pytest.raises(A.SphError) as err:
            b.step(1)
        assert err.value.code == A.SPH_E_LIMIT
