"""The gradient maximum over the blocked brick layout: row remainders in every
axis, one voxel of core, several overlaps, both voxel types, the maximum placed
in a corner, at the ends of rows and in the last row."""
import numpy as np
import pytest

from tuvok_amd import HIPRaycaster

pytestmark = pytest.mark.gpu


def closed_form(vol):
    top = np.iinfo(vol.dtype).max
    p = np.pad(vol.astype(np.float64), 1)
    d = [(p[1:-1, 1:-1, :-2] - p[1:-1, 1:-1, 2:]), (p[1:-1, :-2, 1:-1] - p[1:-1, 2:, 1:-1]),
         (p[:-2, 1:-1, 1:-1] - p[2:, 1:-1, 1:-1])]
    g = [x / (2.0 * top) for x in d]
    return np.float32(np.sqrt(g[0] * g[0] + g[1] * g[1] + g[2] * g[2]).max())


@pytest.mark.parametrize("dtype", [np.uint8, np.uint16])
@pytest.mark.parametrize("dims,brick,ov", [((1, 1, 1), 3, 1), ((3, 1, 2), 4, 1), ((16, 16, 16), 18, 1),
                                           ((33, 20, 17), 18, 1), ((47, 9, 13), 20, 2), ((130, 5, 66), 66, 1),
                                           ((255, 3, 1), 258, 1)])
def test_max_gradient_rows(dims, brick, ov, dtype):
    top = np.iinfo(dtype).max
    rng = np.random.default_rng(3)
    base = rng.integers(0, top // 8, dims[::-1]).astype(dtype)
    spots = {(0, 0, 0), tuple(n - 1 for n in dims), (dims[0] // 2, 0, dims[2] - 1), (min(7, dims[0] - 1), dims[1] // 2, 0),
             (min(8, dims[0] - 1), dims[1] - 1, dims[2] // 2)}
    for x, y, z in spots:
        vol = base.copy()
        vol[z, y, x] = top
        with HIPRaycaster(0) as r:
            r.LoadVolume(vol, (brick,) * 3, ov, max_lods=1)
            assert np.float32(r.MaxGradientMagnitude()) == closed_form(vol)
