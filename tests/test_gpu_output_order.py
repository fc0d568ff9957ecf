"""Order of a drop-in frame's output: by 16-bit bucket, ties by input index,
for buckets at and around the size that is sorted instead of counted in (64),
the sizes at which the sort's layout changes, and its largest."""
import numpy as np
import pytest

import sph_amd as A

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("noalloc", [False, True])
@pytest.mark.parametrize("sizes", [(1,), (2, 63), (64, 65), (66, 127, 128, 129), (1023, 1024, 1025), (4097,),
                                   (8193, 300), (16384, 64)])
def test_output_order(sizes, noalloc):
    h = 0.5
    rng = np.random.default_rng(sum(sizes))
    # each clump in a cell of h of its own, and a few particles elsewhere
    pos = [rng.uniform(0.1 * h, 0.9 * h, (m, 3)) + h * np.array([2 * k + 1, 3, 2]) for k, m in enumerate(sizes)]
    pos = np.concatenate(pos + [rng.uniform(-7.5, -1.0, (200, 3)) * [1, -1, 1]]).astype(np.float32)
    pos = pos[rng.permutation(len(pos))]
    p = A.make_particles(pos, np.zeros_like(pos))
    p["acceleration"][:, 0] = np.arange(len(p))  # carried through
    s, box = A.settings(mass=1e-6, h=h), A.box_reference_cpu()
    step = A.update_particles_noalloc if noalloc else A.update_particles
    out, xf = step(p, s, 1e-6, box)
    index = out["acceleration"][:, 0].astype(np.int64)
    assert np.array_equal(np.sort(index), np.arange(len(p)))
    assert max(np.bincount(out["hash"])) >= max(sizes)
    assert np.array_equal(np.lexsort((index, out["hash"])), np.arange(len(p)))
    assert np.array_equal(xf[:, 12:15], out["position"])
