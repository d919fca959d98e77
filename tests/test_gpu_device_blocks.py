"""Bricking in memory that earlier datasets used: loads of several sizes in turn,
from two threads with a renderer each, give the bricks that a first load gives."""
import threading

import numpy as np
import pytest

from tuvok_amd import HIPRaycaster

pytestmark = pytest.mark.gpu


def test_blocks_of_earlier_datasets():
    rng = np.random.default_rng(5)
    vols = [rng.integers(1, 65535, d).astype(np.uint16) for d in ((40, 33, 50), (64, 64, 64), (9, 70, 31), (66, 64, 62))]
    want = []
    for v in vols:
        with HIPRaycaster(0) as r:
            r.LoadVolume(v, (18, 18, 18), 1)
            want.append((r.GetPool(), r.MaxGradientMagnitude()))
    bad = []

    def work(start):
        with HIPRaycaster(0) as r:
            for k in range(8):
                i = (start + k) % len(vols)
                r.LoadVolume(vols[i], (18, 18, 18), 1, keep_linear=True)
                if k % 2:
                    r.Rebrick((34, 34, 34), 1)
                    r.Rebrick((18, 18, 18), 1)
                if not np.array_equal(r.GetPool(), want[i][0]) or r.MaxGradientMagnitude() != want[i][1]:
                    bad.append((start, k))

    ts = [threading.Thread(target=work, args=(s,)) for s in (0, 1)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
