"""Bricking in memory that earlier datasets used: loads of several sizes in turn,
from two threads with a renderer each, give the bricks that a first load gives."""
import ctypes as C
import threading

import numpy as np
import pytest

from tuvok_amd import HIPRaycaster, TvkError, _abi, release_memory

pytestmark = pytest.mark.gpu


def test_blocks_of_earlier_datasets():
    rng = np.random.default_rng(5)
    vols = [rng.integers(1, 65535, d).astype(np.uint16) for d in ((40, 33, 50), (64, 64, 64), (9, 70, 31), (66, 64, 62))]
    want = []
    for v in vols:
        with HIPRaycaster(0) as r:
            r.LoadVolume(v, (18, 18, 18), 1)
            want.append((r.GetPool(), r.MaxGradientMagnitude()))
    bad, done = [], [0, 0]

    def work(start):
        try:
            with HIPRaycaster(0) as r:
                for k in range(8):
                    i = (start + k) % len(vols)
                    r.LoadVolume(vols[i], (18, 18, 18), 1, keep_linear=True)
                    if k % 2:
                        r.Rebrick((34, 34, 34), 1)
                        r.Rebrick((18, 18, 18), 1)
                    if not np.array_equal(r.GetPool(), want[i][0]) or r.MaxGradientMagnitude() != want[i][1]:
                        bad.append((start, k))
                    done[start] += 1
        except Exception as e:
            bad.append((start, e))

    ts = [threading.Thread(target=work, args=(s,)) for s in (0, 1)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad and done == [8, 8]


def test_released_memory_is_the_device_s_again():
    """What a replaced dataset leaves is kept, and given back when asked for."""
    def free():
        a, b = C.c_size_t(), C.c_size_t()
        assert _abi.load().hipMemGetInfo(C.byref(a), C.byref(b)) == 0
        return a.value

    with HIPRaycaster(0) as r:
        release_memory()
        r.LoadVolume(np.zeros((8, 8, 8), np.uint8), (18,) * 3, 1, max_lods=1)
        before = free()
        r.LoadVolume(np.zeros((400, 400, 400), np.uint8), (66,) * 3, 1, max_lods=1)
        pool = r.GetDatasetDesc().pool_bytes
        r.LoadVolume(np.zeros((8, 8, 8), np.uint8), (18,) * 3, 1, max_lods=1)
        assert before - free() >= pool   # kept
        release_memory()
        assert before - free() <= 8 << 20
        with pytest.raises(TvkError):
            release_memory(-1)
        assert r.GetBrick(0).max() == 0   # the dataset in use stays
