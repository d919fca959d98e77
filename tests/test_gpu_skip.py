"""The march that goes by stretches that cannot contribute (datasets with a cell
grid) against the march that samples every step: a budgeted pool has no grid, so
its frames, sample counts and hits must equal the resident pool's bit for bit."""
import ctypes as C
import threading

import numpy as np
import pytest

from tuvok_amd import RM_1DTRANS, RM_2DTRANS, RM_ISOSURFACE, HIPRaycaster, RenderBatch, _abi, rotation_y

pytestmark = pytest.mark.gpu


def sparse_volume(dims, dtype, seed):
    """Islands, thin sheets and single voxels in an empty volume, some at its faces."""
    rng = np.random.default_rng(seed)
    top = np.iinfo(dtype).max
    v = np.zeros(dims[::-1], dtype)
    for _ in range(6):
        c = [int(rng.integers(0, n)) for n in dims]
        r = [int(rng.integers(1, 9)) for _ in range(3)]
        s = tuple(slice(max(0, c[a] - r[a]), c[a] + r[a]) for a in (2, 1, 0))
        v[s] = rng.integers(top // 3, top, v[s].shape)
    v[:, dims[1] // 2, :] = top // 2
    for _ in range(20):
        v[tuple(int(rng.integers(0, n)) for n in dims[::-1])] = top
    return v


def table(kind):
    t = np.zeros((256, 4), np.uint8)
    t[:, :3] = np.arange(256)[:, None]
    t[:, 3] = {"ramp": np.maximum(np.arange(256) - 60, 0) // 2, "gaps": np.where(np.arange(256) % 64 > 50, 30, 0),
               "all": 20, "last": np.where(np.arange(256) == 255, 200, 0), "none": 0,
               "low": np.where(np.arange(256) < 3, 2, 0)}[kind]
    return t


def frames(r, rots):
    r.SetCountSamples(True)
    f = r.PaintViews(rots)
    n = r.last_stats.samples
    r.SetCountSamples(False)
    assert np.array_equal(f, r.PaintViews(rots))
    return f, n


@pytest.mark.parametrize("dtype", [np.uint8, np.uint16])
@pytest.mark.parametrize("dims,brick,ov,edge", [((70, 53, 61), 18, 1, False), ((64, 64, 192), 66, 1, False),
                                                ((45, 90, 33), 34, 2, True), ((40, 40, 40), 12, 0, False),
                                                ((300, 3, 50), 130, 1, True)])
def test_skipped_stretches(dims, brick, ov, edge, dtype):
    vol = sparse_volume(dims, dtype, 7)
    rots = [rotation_y(a) for a in (0.0, 0.7, 2.1)]
    with HIPRaycaster(0) as r, HIPRaycaster(0) as q:
        for x in (r, q):
            x.LoadVolume(vol, (brick,) * 3, ov, clamp_to_edge=edge, max_lods=1)
            x.SetClampToEdge(edge)
            x.SetViewParameters(45.0, 0.01, 1000.0)
            x.SetViewPosition((0.1, 0.2, 1.7))
            x.Resize(97, 83)
        q.SetPoolBudget(q.GetDatasetDesc().pool_bytes - 1)
        for mode, tf, lit, srm, ert in ((RM_1DTRANS, "ramp", False, 1.0, 0.0), (RM_1DTRANS, "ramp", True, 2.0, 2.0 ** -11),
                                        (RM_1DTRANS, "gaps", True, 1.0, 0.0), (RM_1DTRANS, "gaps", False, 0.7, 2.0 ** -11),
                                        (RM_1DTRANS, "all", False, 1.0, 0.0), (RM_1DTRANS, "last", True, 1.0, 0.0),
                                        (RM_1DTRANS, "low", False, 1.0, 0.0), (RM_1DTRANS, "none", True, 1.0, 0.0),
                                        (RM_ISOSURFACE, None, True, 1.0, 0.0), (RM_ISOSURFACE, None, True, 3.0, 2.0 ** -11)):
            for x in (r, q):
                if tf:
                    x.Set1DTrans(table(tf))
                x.SetRendermode(mode)
                x.SetUseLighting(lit)
                x.SetSampleRateModifier(srm)
                x.SetEarlyRayTermination(ert)
                x.SetIsoValue(np.iinfo(dtype).max * 0.4)
            (a, na), (b, nb) = frames(r, rots), frames(q, rots)
            assert np.array_equal(a, b), (mode, tf, lit, srm)
            if mode == RM_1DTRANS or ert == 0.0:   # the hit skip of a frame rendered in parts sees only its part
                assert na == nb
            assert tf in ("last", "none") or a[..., 3].max() > 0   # only the very top value: samples may miss it


def test_brick_uploaded_again_reaches_every_context():
    """A brick of a shared dataset changes: the other context's next frame and a
    batch see it, although both rendered (and skipped) with the old grid before."""
    dims, brick = (32, 32, 32), 34
    empty = np.zeros((34, 34, 34), np.uint8)
    full = np.zeros((34, 34, 34), np.uint8)
    full[10:20, 10:20, 10:20] = 255
    with HIPRaycaster(0) as a, HIPRaycaster(0) as b:
        a.SetBricks(np.uint8, dims, (brick,) * 3, 1, [(0, 0, (0.0, 255.0))], lod_count=1)
        a.UploadBrick(0, 0, empty)
        b.ShareDataset(a)
        for x in (a, b):
            x.Set1DTrans(table("ramp"))
            x.SetRendermode(RM_1DTRANS)
            x.SetUseLighting(False)
            x.SetViewParameters(45.0, 0.01, 1000.0)
            x.SetViewPosition((0.0, 0.0, 1.8))
            x.Resize(64, 64)
            assert x.Paint()[..., 3].max() == 0
        batch = RenderBatch(0)
        batch.Add(b, None, 64, 64)
        batch.Render()
        assert batch.Frame(0)[..., 3].max() == 0
        a.UploadBrick(0, 0, full)
        fb = b.Paint()
        assert fb[..., 3].max() > 0.5
        assert np.array_equal(fb, a.Paint())
        batch.Render()
        assert np.array_equal(batch.Frame(0), fb)
        batch.close()


@pytest.mark.parametrize("dtype", [np.uint8, np.uint16])
@pytest.mark.parametrize("again", [1, 3, 27])
def test_cell_grid_after_uploads(dtype, again):
    """Bricks uploaded again after the grid was made (one, a few, most): the grid
    equals that of the same bricks handed over at first, and the frame too."""
    dims, core = (40, 44, 36), 14
    grid = [-(-d // core) for d in dims]
    rng = np.random.default_rng(11)
    keys, first, second = [], [], []
    for z in range(grid[2]):
        for y in range(grid[1]):
            for x in range(grid[0]):
                n = [(core if p + 1 < g or d % core == 0 else d % core) + 2 for p, g, d in zip((x, y, z), grid, dims)]
                keys.append((0, len(keys), (0.0, float(np.iinfo(dtype).max))))
                first.append(rng.integers(0, 3, n[::-1]).astype(dtype))
                second.append(rng.integers(0, np.iinfo(dtype).max, n[::-1]).astype(dtype))
    pick = rng.permutation(len(keys))[:min(again, len(keys))]
    out = []
    for late in (True, False):
        with HIPRaycaster(0) as r:
            r.SetBricks(dtype, dims, (core + 2,) * 3, 1, keys, lod_count=1)
            for i, b in enumerate(first):
                r.UploadBrick(0, i, b if late or i not in pick else second[i])
            r.Set1DTrans(table("ramp"))
            r.SetRendermode(RM_1DTRANS)
            r.SetUseLighting(False)
            r.SetViewParameters(45.0, 0.01, 1000.0)
            r.SetViewPosition((0.0, 0.0, 1.8))
            r.Resize(80, 60)
            if late:
                r.Paint()
                for i in pick:
                    r.UploadBrick(0, int(i), second[i])
            out.append((r.Paint(), r.CellGrid()))
    assert np.array_equal(out[0][1], out[1][1])
    assert np.array_equal(out[0][0], out[1][0])


@pytest.mark.parametrize("learned", [False, True])
def test_uploads_beside_another_contexts_frames(learned):
    """One thread uploads the bricks of a shared dataset again (the same voxels) and
    renders, so that the grid is made anew each time; frames and batches of another
    context on another thread stay what they were."""
    core = 14
    vol = sparse_volume((2 * core, core, core), np.uint8, 3)
    with HIPRaycaster(0) as ref:
        ref.LoadVolume(vol, (core + 2,) * 3, 1, max_lods=1)
        bricks = [ref.GetBrick(i) for i in range(2)]
    with HIPRaycaster(0) as a, HIPRaycaster(0) as b:
        a.SetBricks(np.uint8, (2 * core, core, core), (core + 2,) * 3, 1, [(0, i, (0.0, 255.0)) for i in range(2)],
                    lod_count=1)
        for i in range(2):
            a.UploadBrick(0, i, bricks[i])
        b.ShareDataset(a)
        for x in (a, b):
            x.Set1DTrans(table("ramp"))
            x.SetRendermode(RM_1DTRANS)
            x.SetUseLighting(False)
            x.SetViewParameters(45.0, 0.01, 1000.0)
            x.SetViewPosition((0.0, 0.0, 1.8))
            x.Resize(64, 48)
        if learned:
            b.SetStepProposal(None, fixed_log2=0)
        want = b.Paint()
        assert want[..., 3].max() > 0
        batch = RenderBatch(0)
        batch.Add(b, None, 64, 48)
        batch.Render()
        want_batch = batch.Frame(0)
        bad, rounds = [], [0, 0]

        def upload():
            try:
                for k in range(60):
                    a.UploadBrick(0, k % 2, bricks[k % 2])
                    a.Paint()
                    rounds[0] += 1
            except Exception as e:
                bad.append(e)

        def render():
            try:
                for k in range(60):
                    if not np.array_equal(b.Paint(), want):
                        bad.append(k)
                    batch.Render()
                    if not np.array_equal(batch.Frame(0), want_batch):
                        bad.append(("batch", k))
                    rounds[1] += 1
            except Exception as e:
                bad.append(e)

        ts = [threading.Thread(target=f) for f in (upload, render)]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
        batch.close()
        assert not bad and rounds == [60, 60]


def test_2d_frames_make_no_grid():
    """A fixed-step 2D frame of bricks handed over one by one neither reads nor makes
    the cell grid (its ranges of 4^3 voxels are 8 MiB here); a 1D frame makes it."""
    def free():
        a, b = C.c_size_t(), C.c_size_t()
        assert _abi.load().hipMemGetInfo(C.byref(a), C.byref(b)) == 0   # of the library's own HIP runtime
        return a.value

    core, g = 126, 4
    tf2 = np.full((16, 16, 4), 3, np.uint8)
    with HIPRaycaster(0) as r:
        r.LoadVolume(np.full((20, 20, 20), 9, np.uint8), (18,) * 3, 1, max_lods=1)
        r.Set2DTrans(tf2)
        r.Set1DTrans(table("ramp"))
        r.SetRendermode(RM_2DTRANS)
        r.SetUseLighting(False)
        r.SetViewParameters(45.0, 0.01, 1000.0)
        r.SetViewPosition((0.0, 0.0, 1.8))
        r.Resize(64, 64)
        r.Paint()   # the frame's own buffers
        r.SetBricks(np.uint8, (core * g,) * 3, (core + 2,) * 3, 1, [(0, i, (0.0, 255.0)) for i in range(g ** 3)],
                    lod_count=1)
        brick = np.full((core + 2,) * 3, 7, np.uint8)
        for i in range(g ** 3):
            r.UploadBrick(0, i, brick)
        before = free()
        assert r.Paint()[..., 3].max() > 0
        r.UploadBrick(0, 5, brick)
        r.Paint()
        assert before - free() <= 4 << 20
