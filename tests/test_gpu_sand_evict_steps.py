"""Sand steps after an eviction (src/Lustrine.cpp:806-836) in every form of the
step: waiting, enqueued with a fixed capacity, replayed.  The captured steps
hold the particle count, and the lists' solid entries start at it."""
import numpy as np
import pytest

from lustrine_amd import scenes

pytestmark = pytest.mark.gpu

BOX = (20, 20, 20)
DT = np.float32(0.016)
FORMS = {"waiting": (0, False), "capacity": (200000, False), "graph": (200000, True)}


def _scene(gpu_mod, form, substeps=4):
    pos = scenes.jittered_lattice(12, 12, 12, origin=(2.0, 3.0, 2.0), amplitude=0.25, seed=7)
    sol = scenes.lattice(BOX[0], 2, BOX[2], origin=(0.0, 0.0, 0.0))
    total = BOX[0] * BOX[1] * BOX[2]
    sp = gpu_mod.sand_params(*BOX, kernel_radius_scale=3.1, substeps=substeps)
    sp.ptr_solid_start = total - len(sol)
    g = gpu_mod.Gpu(0)
    g.sand_init(sp, pos, None, None, sol, np.arange(total - 1, total - 1 - len(sol), -1, dtype=np.int32))
    capacity, graph = FORMS[form]
    if capacity:
        g.sand_set_list_capacity(capacity)
    if graph:
        g.sand_set_graph(True)
    return g


def _evicted(gpu_mod, form, steps):
    with _scene(gpu_mod, form) as g:
        for _ in range(4):
            g.sand_step(DT)
        cells = np.random.default_rng(5).choice(13 ** 3, 300, replace=False)
        n = g.n_sand
        assert g.sand_sink_evict(cells) < n
        for _ in range(steps):
            g.sand_step(DT)
        state = g.sand_download()
        return state, g.sand_neighbors()


@pytest.mark.parametrize("steps", [1, 2, 5])
@pytest.mark.parametrize("form", ["capacity", "graph"])
def test_steps_after_eviction(gpu_mod, form, steps):
    want, want_lists = _evicted(gpu_mod, "waiting", steps)
    got, lists = _evicted(gpu_mod, form, steps)
    for a, b in zip(got, want):  # the state first: lists of another count name other solids
        assert np.array_equal(a, b)
    for a, b in zip(lists, want_lists):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("substeps", [0, 4])
@pytest.mark.parametrize("form", list(FORMS))
def test_steps_of_an_emptied_scene(gpu_mod, form, substeps):
    # nothing left to step: no pass reads a slot, and every result is empty
    with _scene(gpu_mod, form, substeps) as g:
        g.sand_step(DT)
        assert g.sand_sink_evict(np.arange(13 ** 3)) == 0
        for _ in range(3):
            g.sand_step(DT)
        assert all(len(a) == 0 for a in g.sand_download())
        off, idx = g.sand_neighbors()
        assert off.tolist() == [0] and len(idx) == 0
        assert g.sand_query_cells([0, 0, 0], BOX, False) == 0
