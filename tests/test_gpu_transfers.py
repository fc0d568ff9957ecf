"""Uploads and downloads at the edges of their paths (through an object's
own pinned memory, directly, or in pieces by several threads), and the step's
graph when scenes are replaced: what is uploaded comes back byte for byte, and
a replaced scene steps as a fresh one, bit for bit."""
import numpy as np
import pytest

import sph_amd as A

pytestmark = pytest.mark.gpu
F32 = np.float32
S = A.settings(mass=0.02, h=0.1)
BOX = A.box((-2.0, -2.0, -2.0), (2.0, 2.0, 2.0))


def _state(n, seed, ext=1.5):
    rng = np.random.default_rng(seed)
    return rng.uniform(-ext, ext, (n, 3)).astype(F32), rng.normal(0.0, 0.1, (n, 3)).astype(F32)


# 36 bytes a particle come down, 24 go up, through pieces of 2 MiB:
# 58,254 and 87,381 particles are the last small download and upload
@pytest.mark.parametrize("n", [1, 63, 257, 58254, 58255, 87381, 87382, 466033, 500001])
def test_round_trip(n):
    pos, vel = _state(n, n)
    pos[n // 2] = [np.nan, -np.inf, -0.0]
    with A.Context(n, S, BOX, 1e-3) as c:
        for v in (vel, None):
            c.upload(pos, v)
            got = c.download()
            assert got["pos"].tobytes() == pos.tobytes()
            assert got["vel"].tobytes() == (np.zeros_like(pos) if v is None else v).tobytes()
            assert np.array_equal(got["ids"], np.arange(n))
            assert not got["rho"].any() and not got["pressure"].any()


def _same(x, y):
    return all(x[k].tobytes() == y[k].tobytes() for k in ("pos", "vel", "rho", "pressure", "ids"))


@pytest.mark.parametrize("graph", [True, False])
def test_replaced_scenes(graph):
    sizes = (100, 1000, 4097)
    first = [_state(n, n, 0.4) for n in sizes]
    # other extents (another grid), and a coordinate the bounds leave out
    second = [_state(n, n + 7, ext) for n, ext in zip(sizes, (1.9, 0.1, 0.7))]
    second[1][0][5, 1] = np.inf
    with A.Batch([A.scene_desc(n, S, BOX, 1e-3) for n in sizes]) as b:
        b.set_graph(graph)
        for k, (p, v) in enumerate(first):
            b.upload(k, p, v)
        b.step(3)
        for _ in range(2):  # the second time into an unchanged layout
            for k in (1, 0):
                b.upload(k, *second[k])
            b.step(4)
            got = [b.download(k) for k in range(3)]
        for k, (state, steps) in enumerate(((second[0], 4), (second[1], 4), (first[2], 11))):
            with A.Context(sizes[k], S, BOX, 1e-3) as c:
                c.upload(*state)
                c.step(steps)
                assert _same(got[k], c.download()), k


# 60 bytes a particle go up (and 64 beside them), 124 come down
@pytest.mark.parametrize("n", [1, 300, 16912, 16913, 34951, 34952, 140000])
def test_frame_sizes(n):
    pos, vel = _state(n, n)
    p = A.make_particles(pos, vel)
    before = p.tobytes()
    out, xf = A.update_particles(p, S, 1e-3, BOX)
    alone, none = A.update_particles(p, S, 1e-3, BOX, transforms=False)
    assert p.tobytes() == before and none is None
    assert out.tobytes() == alone.tobytes()
    assert np.array_equal(xf[:, 12:15], out["position"])
    if n <= A.NOALLOC_MAX_PARTICLES:
        ref, rxf = A.update_particles_noalloc(p, S, 1e-3, BOX)
        assert out.tobytes() == ref.tobytes() and xf.tobytes() == rxf.tobytes()


def test_threads_share_the_staging_memory():
    """Downloads above 2 MiB from several threads at once, each its own scene."""
    import threading

    sizes, bad = (120000, 90001, 200003), []

    def work(n):
        try:
            with A.Context(n, S, BOX, 1e-3) as c:
                for k in range(4):
                    pos, vel = _state(n, 10 * n + k)
                    c.upload(pos, vel)
                    got = c.download()
                    if got["pos"].tobytes() != pos.tobytes() or got["vel"].tobytes() != vel.tobytes():
                        bad.append((n, k))
        except Exception as e:  # noqa: BLE001
            bad.append((n, repr(e)))

    threads = [threading.Thread(target=work, args=(n,)) for n in sizes]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


def test_grid_info_after_a_scene_is_replaced():
    """The automatic grid's choice for a replaced scene shows at once, as
    after the first upload, and is the one it steps on."""
    n = 140608  # 52^3, a uniform lattice: chooses cells of h / 2
    g = np.stack(np.meshgrid(*[np.arange(52)] * 3, indexing="ij"), -1).reshape(-1, 3)
    pos = (g * 0.05 - 1.5 + np.random.default_rng(3).uniform(-0.005, 0.005, g.shape)).astype(F32)
    small, _ = _state(500, 5, 0.3)
    with A.Batch([A.scene_desc(n, S, BOX, 1e-3, auto_grid=True), A.scene_desc(500, S, BOX, 1e-3)]) as b:
        b.upload(0, pos)
        b.upload(1, small)
        first = b.grid_info(0)
        b.step(2)
        b.upload(0, pos)
        assert b.grid_info(0)[0] == first[0] == 0.5
        b.step(2)
        again = b.download(0)
    with A.Context(n, S, BOX, 1e-3, auto_grid=True) as c:
        c.upload(pos)
        c.step(2)
        assert _same(again, c.download())
