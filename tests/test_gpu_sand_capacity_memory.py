"""The memory of a fixed list capacity: a smaller one gives it back, and the
last step's lists stay readable through every change."""
import numpy as np
import pytest
import torch

from test_gpu_sand_lists import DT, _clump_and_layer, _params

pytestmark = pytest.mark.gpu


def _free_mb():
    return torch.cuda.mem_get_info()[0] / 2 ** 20


@pytest.mark.parametrize("long_lists", [True, False])
def test_a_smaller_capacity_gives_memory_back(gpu_mod, long_lists):
    pos, sol = _clump_and_layer(True)
    if not long_lists:
        pos = pos[:11 * 3 * 9]  # the layer alone: no list past its fixed place
    sp, index = _params(gpu_mod, len(pos), sol)
    with gpu_mod.Gpu(0) as g:
        g.sand_init(sp, pos, None, None, sol, index)
        g.sand_set_list_capacity(100000)  # before the first step
        g.sand_step(DT)
        want = g.sand_neighbors()
        assert (np.diff(want[0]).max() > 128) == long_lists
        need = int(want[0][-1])
        small = _free_mb()
        for entries in (100_000_000, need, 100_000_000, 1000):  # 450 MB and less than 1
            g.sand_set_list_capacity(entries)
            got = g.sand_neighbors()
            assert all(np.array_equal(a, b) for a, b in zip(got, want))
            used = small - _free_mb()
            assert (used > 400.0) if entries > 10 * need else (used < 50.0)
        g.sand_set_list_capacity(4 * need)
        for _ in range(3):
            g.sand_step(DT)
        state = g.sand_download()
    with gpu_mod.Gpu(0) as g:
        g.sand_init(sp, pos, None, None, sol, index)
        for _ in range(4):
            g.sand_step(DT)
        assert all(np.array_equal(a, b) for a, b in zip(state, g.sand_download()))
