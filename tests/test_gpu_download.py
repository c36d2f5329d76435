"""Downloads through pinned memory: every array equals what the device holds,
at sizes around the chunks and the switch to several threads, for each subset
of the arrays, into memory that the runtime knows and into ordinary memory."""
import ctypes as C

import numpy as np
import pytest

from lustrine_amd import scenes

pytestmark = pytest.mark.gpu

F, I = C.POINTER(C.c_float), C.POINTER(C.c_int)


def _f(a):
    return None if a is None else a.ctypes.data_as(F)


def _i(a):
    return None if a is None else a.ctypes.data_as(I)


# 28 bytes a particle: one chunk, one byte row either side of a 1 MB chunk,
# the last size on one thread and the first on four (8 MB), many chunks
SIZES = [1, 2, 37449, 37450, 299593, 299594, 700001]


@pytest.mark.parametrize("n", SIZES)
def test_pbf_download(gpu_mod, n):
    rng = np.random.default_rng(n)
    side = 128.0
    cfg = scenes.small(1, 1, 1, box=(int(side),) * 3)
    x0 = (rng.random((n, 3), np.float32) * np.float32(side - 4) + np.float32(2)).astype(np.float32)
    v0 = rng.standard_normal((n, 3)).astype(np.float32)
    with gpu_mod.Gpu(0) as g:
        g.pbf_init(gpu_mod.pbf_params(cfg), x0, v0)
        for order in (0, 1):
            x, v, ids = g.pbf_download(order=order)
            assert np.array_equal(ids, np.arange(n))  # no step yet: input order
            assert np.array_equal(x, x0) and np.array_equal(v, v0)
        for sub in range(1, 8):
            a = [np.full((n, 3), 7, np.float32), np.full((n, 3), 7, np.float32), np.full(n, 7, np.int32)]
            p = [q if sub >> k & 1 else None for k, q in enumerate(a)]
            assert g._lib.lus_pbf_download(g._h, 0, _f(p[0]), _f(p[1]), _i(p[2])) == 0
            for k, want in enumerate((x0, v0, np.arange(n, dtype=np.int32))):
                assert np.array_equal(a[k], want if sub >> k & 1 else np.full_like(want, 7))


def test_permuted_rows_match_input_order(gpu_mod):
    cfg = scenes.small(41, 37, 43, box=(64, 64, 64))
    x0 = cfg.positions()
    with gpu_mod.Gpu(0) as g:
        g.pbf_init(gpu_mod.pbf_params(cfg), x0, None)
        g.pbf_step(np.float32(cfg.dt), 2)
        sx, sv, sid = g.pbf_download(order=0)
        ox, ov, oid = g.pbf_download(order=1)
    assert np.array_equal(np.sort(sid), np.arange(len(x0))) and np.array_equal(oid, np.arange(len(x0)))
    assert np.array_equal(ox[sid], sx) and np.array_equal(ov[sid], sv)


@pytest.mark.parametrize("n", [1, 100000])
def test_sand_download_subsets_and_pinned_memory(gpu_mod, n):
    rng = np.random.default_rng(n)
    x0 = (rng.random((n, 3), np.float32) * np.float32(60) + np.float32(2)).astype(np.float32)
    v0 = rng.standard_normal((n, 3)).astype(np.float32)
    att = rng.integers(0, 4, n).astype(np.int32)
    with gpu_mod.Gpu(0) as g:
        g.sand_init(gpu_mod.sand_params(64, 64, 64), x0, v0, att, None, None)
        want = (x0, x0, v0, att)
        for sub in range(1, 16):
            a = [np.full((n, 3), 7, np.float32) for _ in range(3)] + [np.full(n, 7, np.int32)]
            p = [q if sub >> k & 1 else None for k, q in enumerate(a)]
            assert g._lib.lus_sand_download(g._h, _f(p[0]), _f(p[1]), _f(p[2]), _i(p[3]), None) == 0
            for k in range(4):
                assert np.array_equal(a[k], want[k] if sub >> k & 1 else np.full_like(want[k], 7))
        hip = C.CDLL("libamdhip64.so.7")  # the runtime that the library has loaded
        mem = C.c_void_p()
        assert hip.hipHostMalloc(C.byref(mem), C.c_size_t(12 * n), C.c_uint(0)) == 0
        pinned = np.ctypeslib.as_array(C.cast(mem, F), (n, 3))
        pinned[:] = 7
        star = np.zeros((n, 3), np.float32)
        assert g._lib.lus_sand_download(g._h, C.cast(mem, F), _f(star), None, None, None) == 0
        assert np.array_equal(pinned, x0) and np.array_equal(star, x0)
        del pinned
        assert hip.hipHostFree(mem) == 0
