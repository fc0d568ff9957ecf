"""Which kernel walks what: the cases of the staged walks' and the union walk's
tests take the walks they are there for.  On cells of h the rule for staging a
wave task is followed from the positions (its x-rows of cells, candidates and
row lengths); on finer cells its sure ends are."""
import numpy as np
import pytest

import test_gpu_fine_walk
import test_gpu_staged_walk
import test_gpu_union_walk

pytestmark = pytest.mark.gpu


def _dump(sph, sc, cell_scale):
    with sph.Context(sc.n, sph.settings(*sc.settings_args()), sph.box(sc.box_lo, sc.box_hi), sc.dt,
                     cell_scale=cell_scale) as ctx:
        ctx.upload(sc.pos, sc.vel)
        return ctx.walk_dump()


class Waves:
    """The wave tasks of a scene: its particles in cell order, 64 to a wave."""

    def __init__(self, sc, cell_scale):
        edge = float(np.float32(sc.h)) * (1.0 + 2.0 ** -10) * cell_scale
        p = sc.pos.astype(np.float64)
        low = np.minimum(np.array(sc.box_lo), p.min(0))
        extent = np.maximum(np.array(sc.box_hi), p.max(0)) - low
        while True:  # cells widen until there are at most 64 a particle
            dims = np.floor(extent / edge).astype(int) + 3
            if dims.prod() <= max(64 * sc.n, 65536):
                break
            edge *= 1.25
        self.cell = np.clip(np.floor((p - (low - edge)) / edge).astype(int), 0, dims - 1)
        self.reach = int(np.ceil(1.0 / cell_scale))
        count = np.zeros(dims, int)
        np.add.at(count, tuple(self.cell.T), 1)
        R = self.reach
        self.count = np.pad(count, ((1 + R, R), (R, R), (R, R)))  # along x: one more in front, for differences
        self.below = np.cumsum(self.count, 0)
        order = np.lexsort((np.arange(sc.n), self.cell[:, 0], self.cell[:, 1], self.cell[:, 2]))
        self.tasks = [order[k:k + 64] for k in range(0, sc.n, 64)]

    def rows(self, x0, x1, y, z):
        """Candidates in each row of the stencil of cells x0 .. x1 of row (y, z)."""
        W = 2 * self.reach + 1
        at = self.below[:, y:y + W, z:z + W]
        return (at[x1 + 1 + W - 1] - at[x0]).ravel()

    def segments(self, task):
        """(first, last cell, y, z) of each x-row of the task's cells."""
        out = []
        for x, y, z in self.cell[task]:
            if out and out[-1][2:] == [y, z]:
                out[-1][1] = x
            else:
                out.append([x, x, y, z])
        return out

    def own(self, i):
        x, y, z = self.cell[i]
        return self.rows(x, x, y, z)


def _coarse_rule(w, task):
    """True / False: staged or not on cells of h; None: depends on the cut."""
    seg = w.segments(task)
    own = [w.own(i) for i in task]
    if len(seg) > 7 or max(r.sum() for r in own) > 409 or \
            sum((-(-w.rows(*s) // 4) * 4).sum() for s in seg) > 1296:
        return False
    return True if max(r.max() for r in own) + 3 <= 96 else None


def _fine_rule(w, task):
    own = [w.own(i) for i in task]
    if max(r.max() for r in own) <= 30 and max(r.sum() for r in own) <= 409:
        return True
    # the lane's own cell, at least, stays in its row
    cells = w.count[tuple((w.cell[task] + [1 + w.reach, w.reach, w.reach]).T)]
    return False if cells.max() > 30 else None


def _check(w, rule, staged):
    seen = set()
    for task in w.tasks:
        assert len(set(staged[task])) == 1
        want = rule(w, task)
        seen.add(want)
        assert want is None or staged[task[0]] == want, (w.segments(task), want)
    return seen


@pytest.mark.parametrize("name", test_gpu_staged_walk.CASES)
def test_staged_on_cells_of_h(sph, name):
    sc = test_gpu_staged_walk._case(name)
    w = Waves(sc, 1.0)
    seen = _check(w, _coarse_rule, _dump(sph, sc, 1.0)["staged"])
    if name in ("n=64", "n=129", "n=3375", "seven rows", "line", "row limit"):
        assert False in seen
    assert True in seen or name in ("n=63", "n=64", "collisions")


@pytest.mark.parametrize("name", ["lattice", "row of 31", "sparse"] + test_gpu_staged_walk.CASES)
def test_staged_on_cells_of_half_h(sph, name):
    sc = test_gpu_fine_walk._fine_case(name)
    dump = _dump(sph, sc, 0.5)
    if name == "h above 1":  # left to the density pass
        assert not dump["staged"].any()
        return
    seen = _check(Waves(sc, 0.5), _fine_rule, dump["staged"])
    assert True in seen or name in ("line", "list limit", "collisions")
    if name in ("row of 31", "line", "row limit", "list limit", "collisions"):
        assert False in seen


@pytest.mark.parametrize("name", test_gpu_union_walk.SCENES)
@pytest.mark.parametrize("scale", [1.0, 0.5])
def test_union_walks_are_not_staged_ones(sph, name, scale):
    dump = _dump(sph, test_gpu_union_walk.SCENES[name](), scale)
    union = dump["box"] & ~dump["staged"]
    assert union.mean() > 0.5
    if "whole" in name:
        assert (union & ~dump["split"] & ~dump["listed"]).any()
    if "split" in name:
        assert (union & dump["split"]).any()


@pytest.mark.parametrize("size", [470, 1500])
@pytest.mark.parametrize("scale", [1.0, 0.5])
def test_segment_walks_match_the_oracle(sph, orc32, monkeypatch, size, scale):
    """Clumps of a cell, some of whose waves hold the end of one and the start
    of the next, cells apart: each walked for its own lanes (470: whole waves,
    1500: split)."""
    # cells of 0.1 beside the wall at -2, middles clear of the axes
    centres = [-2.0 + 0.1 * (1.0 + 2.0 ** -10) * (np.array([26.0 + 3 * k, 25.0 + 5 * (k % 3), 24.0 + 4 * k]) + 0.3)
               for k in range(4)]
    sc = test_gpu_union_walk._clumps([size + 9 * k for k in range(4)], centres, sigma=0.06)
    dump = _dump(sph, sc, scale)
    segments = dump["box"] & dump["segments"] & ~dump["staged"]
    assert (segments & (dump["split"] == (size > 1000))).any(), "premise: waves of two clumps"
    monkeypatch.setitem(test_gpu_union_walk.SCENES, "cells apart", lambda: sc)
    test_gpu_union_walk.test_union_walk_matches_the_oracle(sph, orc32, "cells apart", scale)


@pytest.mark.parametrize("value", [np.nan, np.inf, 1e30, 1e17])
def test_values_in_segment_walks_stay_where_they_belong(sph, value):
    """Clumps whose lists overflow, unsplit on either walk: the force of waves
    that hold two of them, one with a velocity that is not finite or huge, is
    the per-lane walk's bit for bit."""
    centres = [-2.0 + 0.1 * (1.0 + 2.0 ** -10) * (np.array([26.0 + 3 * k, 25.0 + 5 * (k % 3), 24.0 + 4 * k]) + 0.3)
               for k in range(4)]
    sc = test_gpu_union_walk._clumps([200 + 9 * k for k in range(4)], centres, sigma=0.06)
    sc.vel[205, 1] = value  # in the second clump
    dump = _dump(sph, sc, 1.0)
    assert (dump["box"] & dump["segments"] & ~dump["split"] & ~dump["listed"]).any(), "premise: waves of two clumps"
    got = []
    for lane_walk in (False, True):
        with sph.Context(sc.n, sph.settings(*sc.settings_args()), sph.box(sc.box_lo, sc.box_hi), sc.dt,
                         lane_walk=lane_walk, keep_force=True) as ctx:
            ctx.upload(sc.pos, sc.vel)
            assert not ctx.walk_dump()["split"].any()
            ctx.step(1)
            got.append(ctx.download_particles(transforms=False)[0])
    for key in ("position", "velocity", "force", "density", "pressure"):
        assert np.array_equal(got[0][key], got[1][key], equal_nan=True), key
    assert not np.isfinite(got[0]["force"]).all() or np.isfinite(value)
    assert np.isfinite(got[0]["force"]).any()


@pytest.mark.parametrize("cell_scale", [1.7, 2.0, 2.6])
@pytest.mark.parametrize("spacing", [0.5, 0.64, 0.9])
def test_union_walks_that_record_lists(sph, orc32, spacing, cell_scale):
    """Whole union walks of the density pass with lists of a few to some thirty
    neighbours (cells larger than h, too many candidates to be staged): lists,
    counts and densities are the oracle's, sums the per-lane walk's bit for bit
    where that one is not split either."""
    h = 0.1
    g = np.stack(np.meshgrid(*[np.arange(12)] * 3, indexing="ij"), -1).reshape(-1, 3) * spacing * h
    pos = g + np.random.default_rng(7).uniform(-0.1, 0.1, g.shape) * spacing * h + [0.83, 0.71, -1.94]
    sc = test_gpu_staged_walk._scene(pos)
    dump = _dump(sph, sc, cell_scale)
    whole = dump["box"] & ~dump["staged"] & ~dump["split"] & dump["listed"]
    if 409 < 27 * (cell_scale / spacing) ** 3 < 800:  # too long to be staged, short enough to be left whole
        assert whole.any(), "premise: whole union walks with lists"
    out = []
    for lane_walk in (False, True):
        with sph.Context(sc.n, sph.settings(*sc.settings_args()), sph.box(sc.box_lo, sc.box_hi), sc.dt,
                         cell_scale=cell_scale, lane_walk=lane_walk) as ctx:
            ctx.upload(sc.pos, sc.vel)
            d = ctx.walk_dump(lists=True)
            ids = np.arange(sc.n)
            ost = test_gpu_union_walk.OracleState(orc32, sc, sc.pos, sc.vel)
            try:
                test_gpu_union_walk._check_dump(d, ost.rows(ids), ids, f"lane_walk={lane_walk}")
                ost.forces(ids[:1])  # computes the densities
                rho, prs = ost.rho_p_by_id()
            finally:
                ost.close()
            ctx.step(1)
            got = ctx.download()
            by_id = {k: np.zeros_like(got[k]) for k in ("rho", "pressure")}
            for k in by_id:
                by_id[k][got["ids"]] = got[k]
            test_gpu_union_walk.pu.assert_rho_p(by_id["rho"], by_id["pressure"], rho, prs, ost.s)
            out.append((d, got))
    assert np.array_equal(out[0][1]["ids"], out[1][1]["ids"])
    ids = out[0][1]["ids"]
    same = ~(out[0][0]["split"] | out[1][0]["split"])[ids]
    for key in ("rho", "pressure"):
        assert out[0][1][key][same].tobytes() == out[1][1][key][same].tobytes(), key


@pytest.mark.parametrize("n", [1, 65, 130, 300, 511, 1300, 5000, 9001])
@pytest.mark.parametrize("clumps", [0, 1, 5])
def test_every_task_and_part_is_taken_once(sph, orc32, n, clumps):
    """From one block to hundreds, unsplit tasks alone, with a few parts beside
    them, and many: counts exactly and densities within the parity bar."""
    rng = np.random.default_rng(n)
    pos = rng.uniform(-0.06, 0.06, (n, 3)) * n ** (1.0 / 3.0) + 1.1
    m = n // 2 if clumps else 0  # half of the particles in clumps
    pos[:m] = (rng.uniform(0.6, 1.6, (clumps or 1, 3))[np.arange(m) % (clumps or 1)] + rng.normal(0.0, 0.02, (m, 3)))
    sc = test_gpu_staged_walk._scene(pos, box=4.0)
    with sph.Context(sc.n, sph.settings(*sc.settings_args()), sph.box(sc.box_lo, sc.box_hi), sc.dt) as ctx:
        ctx.upload(sc.pos, sc.vel)
        count = ctx.walk_dump()["count"]
        ctx.step(1)
        got = ctx.download()
    ost = test_gpu_union_walk.OracleState(orc32, sc, sc.pos, sc.vel)
    try:
        assert np.array_equal(count, [len(r) for r in ost.rows(np.arange(n))])
        ost.forces(np.arange(1))  # computes the densities
        rho, prs = ost.rho_p_by_id()
    finally:
        ost.close()
    by_id = {k: np.zeros_like(got[k]) for k in ("rho", "pressure")}
    for k in by_id:
        by_id[k][got["ids"]] = got[k]
    test_gpu_union_walk.pu.assert_rho_p(by_id["rho"], by_id["pressure"], rho, prs, ost.s)
