"""Pinned memory of downloads: taken while one runs, from blocks that the
contexts share, and not with every scene that is made."""
import threading

import numpy as np
import pytest

from lustrine_amd import scenes

pytestmark = pytest.mark.gpu


def _mapped_mb():
    """Memory that the process maps from the device's driver, the device's and pinned."""
    mapped = 0
    with open("/proc/self/maps") as f:
        for line in f:
            if "/dev/dri/" in line and line.split()[1].startswith("rw"):
                a, b = line.split()[0].split("-")
                mapped += int(b, 16) - int(a, 16)
    return mapped / 2 ** 20


def _init(gpu_mod, g, x0, side):
    g.pbf_init(gpu_mod.pbf_params(scenes.small(1, 1, 1, box=(side,) * 3)), x0, None)


def test_scenes_reserve_no_pinned_memory(gpu_mod):
    # a download of 28 n bytes uses 2 MB of pinned memory below 8 MB and 16 MB
    # from there on; the scenes' own arrays are alike on both sides
    kept, grown = [], []
    try:
        for n in (299500, 299700):
            x0 = (np.random.default_rng(n).random((n, 3), np.float32) * np.float32(120) + np.float32(2)).astype(np.float32)
            each = []
            for _ in range(9):
                before = _mapped_mb()
                kept.append(gpu_mod.Gpu(0))
                _init(gpu_mod, kept[-1], x0, 128)
                each.append(_mapped_mb() - before)
                if len(each) == 1:  # what a first download brings with it
                    kept[-1].pbf_download()
            grown.append(float(np.median(each)))
            for g in kept[-9:]:
                assert np.array_equal(g.pbf_download()[0], x0)
        print(f"a scene each: {grown[0]:.1f} and {grown[1]:.1f} MB")
        assert grown[1] - grown[0] < 14 / 2
    finally:
        for g in kept:
            g.close()


@pytest.mark.parametrize("sizes", [(300, 300000, 5000, 800000, 70000, 300001)])
def test_contexts_download_at_the_same_time(gpu_mod, sizes):
    # more contexts than idle blocks are kept, of several sizes, each on its own thread
    bad = []

    def work(k, n):
        rng = np.random.default_rng(k)
        with gpu_mod.Gpu(0) as g:
            for rep in range(3):
                x0 = (rng.random((n, 3), np.float32) * np.float32(120) + np.float32(2)).astype(np.float32)
                _init(gpu_mod, g, x0, 128)
                for _ in range(3):
                    x, v, ids = g.pbf_download(order=rep % 2)
                    if not (np.array_equal(x, x0) and not v.any() and np.array_equal(ids, np.arange(n))):
                        bad.append((k, n, rep))

    th = [threading.Thread(target=work, args=q) for q in enumerate(sizes)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad
