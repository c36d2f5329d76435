"""simulate_sand's neighbour lists: fixed places, and the pool for lists past
them.  Bit for bit against the oracle (permutation, lists in the reference's
order, positions, velocities) where lists lie on both sides of a fixed place's
end in one wave, over solids and without, with slots past the symmetric
limit; a capacity of exactly the lists' length steps without waiting, one less
is reported."""
import numpy as np
import pytest

from lustrine_amd import scenes

pytestmark = pytest.mark.gpu

BOX = (20, 20, 20)
DT = np.float32(0.016)


def _clump_and_layer(solids):
    # lists of about 220 entries (the clump) beside lists of 5 to 20
    clump = scenes.jittered_lattice(5, 6, 7, cell=0.3, origin=(8.0, 8.0, 8.0), amplitude=0.02, seed=3)
    layer = scenes.jittered_lattice(11, 3, 9, origin=(2.0, 3.0, 2.0), amplitude=0.2, seed=4)
    pos = np.concatenate([layer, clump]).astype(np.float32)
    return pos, scenes.lattice(20, 2, 20, origin=(0.0, 0.0, 0.0)) if solids else None


def _params(gpu_mod, n, sol, limit=None):
    ns = 0 if sol is None else len(sol)
    total = max(n + ns, BOX[0] * BOX[1] * BOX[2])
    sp = gpu_mod.sand_params(*BOX, kernel_radius_scale=3.1)
    sp.ptr_solid_start = total - ns if limit is None else limit
    return sp, (np.arange(total - 1, total - 1 - ns, -1, dtype=np.int32) if ns else None)


def _run(gpu_mod, pos, sol, capacity=0, graph=False, steps=2, limit=None, variant=0):
    sp, index = _params(gpu_mod, len(pos), sol, limit)
    out = []
    with gpu_mod.Gpu(0) as g:
        g.sand_init(sp, pos, None, None, sol, index)
        g.sand_set_variant(variant)
        if capacity:
            g.sand_set_list_capacity(capacity)
        if graph:
            g.sand_set_graph(True)
        for _ in range(steps):
            g.sand_step(DT, False, False, None)
            out.append(g.sand_download() + g.sand_neighbors())
    return out


def _same(a, b):
    return all(np.array_equal(p, q) for s, t in zip(a, b) for p, q in zip(s, t))


@pytest.mark.parametrize("solids", [False, True])
def test_long_and_short_lists_match_reference(gpu_mod, oracle, solids):
    pos, sol = _clump_and_layer(solids)
    n = len(pos)
    st = oracle.SandStream(oracle.init_constants(*BOX, 0.5, 1.0, 3.1), pos, sol)
    got = _run(gpu_mod, pos, sol)
    for k in range(2):
        st.step(DT)
        off, idx = st.neighbors()
        length = np.diff(off)
        assert k or (length.max() > 128 and length.min() < 32)
        assert np.array_equal(got[k][5], off) and np.array_equal(got[k][6], idx)
        assert np.array_equal(got[k][4], st.perm())
        for a, b in zip(got[k][:3], (st.p[:n], st.ps[:n], st.v[:n])):
            assert np.array_equal(a, b)


@pytest.mark.parametrize("solids", [False, True])
def test_capacity_of_exactly_the_length(gpu_mod, solids):
    pos, sol = _clump_and_layer(solids)
    want = _run(gpu_mod, pos, sol)
    need = max(int(s[5][-1]) for s in want)
    for graph in (False, True):
        assert _same(_run(gpu_mod, pos, sol, capacity=need, graph=graph), want)
    with pytest.raises(gpu_mod.LusError, match="capacity"):
        _run(gpu_mod, pos, sol, capacity=need - 1)


@pytest.mark.parametrize("variant", [0, 2])
def test_slots_past_the_symmetric_limit(gpu_mod, variant):
    # slot i's pushed entries (j < i, and i's second one) exist only below the limit
    pos, _ = _clump_and_layer(False)
    n = len(pos)
    full = _run(gpu_mod, pos, None, steps=1, variant=variant)[0]
    limit = n // 2 + 3
    off, idx = full[5], full[6]
    cut = _run(gpu_mod, pos, None, steps=1, variant=variant, limit=limit)[0]
    for i in range(n):
        row = idx[off[i]:off[i + 1]]
        if i >= limit:
            row = np.unique(row[row >= i])
        assert np.array_equal(cut[6][cut[5][i]:cut[5][i + 1]], row), i


def test_no_substeps_keeps_the_prediction(gpu_mod):
    pos, sol = _clump_and_layer(True)
    sp, index = _params(gpu_mod, len(pos), sol)
    sp.substeps = 0
    with gpu_mod.Gpu(0) as g:
        g.sand_init(sp, pos, None, None, sol, index)
        g.sand_step(DT, False, False, None)
        x, xs, v, _, perm = g.sand_download()
    # v = dt g, x = x0 + dt v, v = (x - x0) / dt, in binary32
    x0 = pos[perm]
    want = x0 + (np.array([sp.gravity[a] for a in range(3)], np.float32) * DT) * DT
    assert np.array_equal(x, want) and np.array_equal(xs, x)
    assert np.array_equal(v, (want - x0) / DT)


def _heap(n, seed, spacing=0.9):
    side = int(np.ceil(n ** (1.0 / 3.0))) + 1
    lat = scenes.jittered_lattice(side, side, side, cell=spacing, origin=(3.0, 3.0, 3.0), amplitude=0.25, seed=seed)
    return lat[:n].astype(np.float32)


@pytest.mark.parametrize("solids", [False, True])
@pytest.mark.parametrize("spacing", [0.9, 0.6])
def test_small_and_large_scene_forms_agree(gpu_mod, solids, spacing):
    # the same heap alone (four waves per 64 slots, four lanes per particle)
    # and beside a far layer that takes the scene past the small form's size
    from lustrine_amd.gpu import sand_params

    box = (200, 60, 200)
    sol = scenes.lattice(40, 2, 40, origin=(0.0, 0.0, 0.0)) if solids else None
    heap = _heap(5003, 3, spacing)
    far = scenes.lattice(180, 2, 200, origin=(60.0, 20.0, 1.0))[:61000]
    far = far[far[:, 0] < box[0] - 2]
    far2 = scenes.lattice(130, 2, 190, origin=(62.0, 30.0, 2.0))
    big = np.concatenate([heap, far, far2]).astype(np.float32)
    assert len(heap) <= 65536 < len(big)
    out = []
    for pos in (heap, big):
        ns = 0 if sol is None else len(sol)
        total = max(len(pos) + ns, box[0] * box[1] * box[2])
        sp = sand_params(*box, kernel_radius_scale=3.1)
        sp.ptr_solid_start = total - ns
        index = np.arange(total - 1, total - 1 - ns, -1, dtype=np.int32) if ns else None
        with gpu_mod.Gpu(0) as g:
            g.sand_init(sp, pos, None, None, sol, index)
            g.sand_step(DT, False, False, None)
            x, _, v, _, perm = g.sand_download()
            off, idx = g.sand_neighbors()
        back = np.argsort(perm)  # slot of input particle i
        lists = []
        for i in range(len(heap)):
            row = idx[off[back[i]]:off[back[i] + 1]]
            # solids by their offset from the top of the reference's slots
            lists.append(np.where(row < len(pos), perm[np.minimum(row, len(pos) - 1)], row - total))
        out.append((x[back[:len(heap)]], v[back[:len(heap)]], lists))
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
    for a, b in zip(out[0][2], out[1][2]):
        assert np.array_equal(a, b)


def test_lists_stay_readable_when_a_capacity_is_set(gpu_mod):
    # the last step's long lists lie in the pool; a small capacity set after it
    # leaves them as they are
    pos, sol = _clump_and_layer(True)
    sp, index = _params(gpu_mod, len(pos), sol)
    with gpu_mod.Gpu(0) as g:
        g.sand_init(sp, pos, None, None, sol, index)
        g.sand_step(DT, False, False, None)
        off, idx = g.sand_neighbors()
        for entries in (100, 10 * int(off[-1]), 0):
            g.sand_set_list_capacity(entries)
            a, b = g.sand_neighbors()
            assert np.array_equal(a, off) and np.array_equal(b, idx)
