"""The staged walk on cells finer than h (k_plan_fine): one step with the
walks chosen by the library against the same step with the per-lane walk
forced, bit for bit, and neighbour counts and lists against the oracle, at the
edges of what it accepts: partial waves, more x-rows than it stages, a row of
31 and 32 candidates, lists of 63 to 65 entries, the grid's border."""
import numpy as np
import pytest

from test_gpu_production_walks import OracleState, _check_dump
from test_gpu_staged_walk import CASES, _case, _scene, _uniform

pytestmark = pytest.mark.gpu


def _fine_case(name):
    rng = np.random.default_rng(23)
    if name == "lattice":  # spacing h / 2, whole waves and rows
        g = np.stack(np.meshgrid(*[np.arange(24)] * 3, indexing="ij"), -1).reshape(-1, 3) * 0.05 - 0.6
        return _scene(g + rng.uniform(-0.005, 0.005, size=g.shape))
    if name == "row of 31":  # clumps about a cell wide, 28 to 33 in a row of cells
        p = [rng.uniform(-0.02, 0.02, size=(m, 3)) * [1.0, 0.5, 0.5] + [0.3 * k + 0.775, 0.925, 0.4 * k - 0.975]
             for k, m in enumerate((28, 30, 31, 32, 33))]
        return _scene(np.concatenate(p + [rng.uniform(-1.5, -0.3, size=(700, 3))]))
    if name == "sparse":  # up to sixty x-rows of cells in a wave
        return _uniform(900, 1.9)
    return _case(name)


@pytest.mark.parametrize("cell_scale", [0.5, 0.7])
@pytest.mark.parametrize("name", ["lattice", "row of 31", "sparse"] + CASES)
def test_fine_walk_equals_lane_walk_and_oracle(sph, orc32, name, cell_scale):
    sc = _fine_case(name)
    out, whole = [], np.ones(sc.n, dtype=bool)
    for lane_walk in (False, True):
        with sph.Context(sc.n, sph.settings(*sc.settings_args()), sph.box(sc.box_lo, sc.box_hi), sc.dt,
                         cell_scale=cell_scale, lane_walk=lane_walk) as ctx:
            ctx.upload(sc.pos, sc.vel)
            dump = ctx.walk_dump(lists=True)
            whole &= ~dump["split"]
            ost = OracleState(orc32, sc, sc.pos, sc.vel)
            try:
                _check_dump(dump, ost.rows(np.arange(sc.n)), np.arange(sc.n), f"{name}, lane_walk={lane_walk}")
            finally:
                ost.close()
            ctx.step(1)
            out.append(ctx.download())
    # A split task's sums differ by rounding, and with them what its
    # neighbours feel: then the densities of the others are compared.
    ids = out[0]["ids"]
    assert np.array_equal(ids, out[1]["ids"])
    assert whole.any()
    for key in ("pos", "vel", "rho", "pressure") if whole.all() else ("rho", "pressure"):
        assert out[0][key][whole[ids]].tobytes() == out[1][key][whole[ids]].tobytes(), \
            f"{name}: {key} differs between the walks"
