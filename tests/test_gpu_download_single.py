"""Downloads of ids, flags, the permutation or lambdas alone take no memory on
the device: nothing has to be packed."""
import ctypes as C

import numpy as np
import pytest
import torch

from lustrine_amd import scenes

pytestmark = pytest.mark.gpu

N = 1000003
F, I = C.POINTER(C.c_float), C.POINTER(C.c_int)


def _free_mb():
    return torch.cuda.mem_get_info()[0] / 2 ** 20


def _points(seed):
    rng = np.random.default_rng(seed)
    return (rng.random((N, 3), np.float32) * np.float32(120) + np.float32(2)).astype(np.float32)


def _ints():
    return np.full(N, -7, np.int32)


def test_ids_alone(gpu_mod):
    with gpu_mod.Gpu(0) as g:
        cfg = scenes.small(1, 1, 1, box=(128, 128, 128))
        g.pbf_init(gpu_mod.pbf_params(cfg, exact=False, iterations=1), _points(1), None)
        g.pbf_step(np.float32(cfg.dt), 1)
        got, before = [], _free_mb()
        for order in (0, 1):
            ids = _ints()
            assert g._lib.lus_pbf_download(g._h, order, None, None, ids.ctypes.data_as(I)) == 0
            got.append(ids)
        assert before - _free_mb() < 8.0
        assert np.array_equal(got[0], g.pbf_download(order=0)[2])
        assert np.array_equal(got[1], np.arange(N))


def test_flags_and_permutation_alone(gpu_mod):
    att = np.random.default_rng(3).integers(0, 2, N).astype(np.int32)
    with gpu_mod.Gpu(0) as g:
        g.sand_init(gpu_mod.sand_params(128, 128, 128), _points(2), None, att, None, None)
        g.sand_step(np.float32(0.016))
        a, p, a2, p2 = _ints(), _ints(), _ints(), _ints()
        before = _free_mb()
        assert g._lib.lus_sand_download(g._h, None, None, None, a.ctypes.data_as(I), None) == 0
        assert g._lib.lus_sand_download(g._h, None, None, None, None, p.ctypes.data_as(I)) == 0
        assert g._lib.lus_sand_download(g._h, None, None, None, a2.ctypes.data_as(I), p2.ctypes.data_as(I)) == 0
        assert g._lib.lus_sand_download(g._h, None, None, None, None, None) == 0
        assert before - _free_mb() < 8.0
        want = g.sand_download()
    for x, y in ((a, want[3]), (p, want[4]), (a2, want[3]), (p2, want[4])):
        assert np.array_equal(x, y)


def test_lambdas_alone(gpu_mod, oracle):
    n, total = 1000, 400000
    p = np.zeros((total, 3), np.float32)
    p[:n] = scenes.lattice(10, 10, 10, origin=(6.0, 6.0, 6.0))
    lam = np.random.default_rng(4).random(total).astype(np.float32)
    with gpu_mod.Gpu(0) as g:
        g.fluid_init(gpu_mod.fluid_params(oracle.init_constants(24, 24, 24, 0.5, 1.0, 4.0)), p, p, np.zeros_like(p),
                     (0, n), (total - 1, total - 1), lambdas=lam)
        got, before = np.zeros(total, np.float32), _free_mb()
        assert g._lib.lus_fluid_download(g._h, None, None, None, got.ctypes.data_as(F)) == 0
        assert before - _free_mb() < 8.0
        assert np.array_equal(got, lam) and np.array_equal(g.fluid_download()[0], p)
