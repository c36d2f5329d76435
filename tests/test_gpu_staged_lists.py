"""The list forms of a step -- wave-staged build (lus_pbf_set_build(1)) and
block-staged lists (2) -- against the gathered one (0): the same neighbour sets in the same order, so the same bits in every pass that
walks them -- the plain solver, the learned step's features and the training
rows -- at sizes around a wave and a block, for columns of cells shorter and
longer than a block, dense cells (rows past what is staged) and lists past
their capacity."""
import numpy as np
import pytest

from lustrine_amd import learned, scenes

pytestmark = pytest.mark.gpu

# lattice, box, jitter: ragged, tall columns, wide layers, a dense clump
SCENES = [((1, 1, 1), (8, 8, 8), 0.0), ((3, 5, 7), (12, 12, 12), 0.1), ((9, 6, 11), (24, 16, 24), 0.3),
          ((5, 4, 130), (16, 12, 260), 0.1), ((70, 2, 33), (144, 12, 72), 0.3), ((40, 20, 41), (84, 44, 84), 0.02)]


def scene(lat, box, jitter, seed, squeeze=1.0):
    cfg = scenes.PbfConfig(name="t", lattice=lat, box=box, jitter=jitter, seed=seed)
    pos = cfg.positions()
    if squeeze != 1.0:
        pos = (pos * np.float32(squeeze) + np.float32(1.0)).astype(np.float32)
    vel = np.random.default_rng(seed).normal(0.0, 1.0, pos.shape).astype(np.float32)
    return cfg, pos, vel


def plain(gpu_mod, cfg, pos, vel, staged, exact, steps=3, lanes=1):
    with gpu_mod.Gpu(0) as g:
        g.pbf_set_build(staged)
        g.pbf_set_lanes(lanes)
        g.pbf_init(gpu_mod.pbf_params(cfg, exact=exact), pos, vel)
        g.pbf_set_mode(False, check=True)
        g.pbf_step(np.float32(cfg.dt), steps)
        out = g.pbf_download(order=0)
        return out + (g.pbf_retest_count(), g.pbf_last_max_constraint(), g.pbf_learned_stats(True)[2:])


def same(a, b):
    for x, y in zip(a, b):
        if isinstance(x, tuple):
            same(x, y)
        else:
            assert np.array_equal(x, y, equal_nan=True)


@pytest.mark.parametrize("exact", [True, False])
@pytest.mark.parametrize("k", range(len(SCENES)))
def test_plain_steps(gpu_mod, k, exact):
    cfg, pos, vel = scene(*SCENES[k], seed=k)
    want = plain(gpu_mod, cfg, pos, vel, 0, exact)
    for staged in (1, 2):
        same(plain(gpu_mod, cfg, pos, vel, staged, exact), want)


@pytest.mark.parametrize("exact", [True, False])
@pytest.mark.parametrize("squeeze", [0.8, 0.6, 0.45])
def test_dense_scenes(gpu_mod, squeeze, exact):
    # 2 to 11 times the rest density: full cells, long rows, lists past 128 entries
    cfg, pos, vel = scene((24, 16, 24), (48, 32, 48), 0.05, 7, squeeze)
    want = plain(gpu_mod, cfg, pos, vel, 0, exact, steps=2)
    for staged in (1, 2):
        same(plain(gpu_mod, cfg, pos, vel, staged, exact, steps=2), want)


@pytest.mark.parametrize("k", [2, 5])
def test_learned_steps(gpu_mod, k):
    cfg, pos, vel = scene(*SCENES[k], seed=k)
    net = learned.load()[0]
    out = []
    for staged in (0, 1, 2):
        with gpu_mod.Gpu(0) as g:
            g.pbf_set_build(staged)
            g.pbf_init(gpu_mod.pbf_params(cfg, iterations=6, exact=False), pos, vel)
            g.pbf_set_network(net)
            g.pbf_set_mode(True, 2, 0.05)  # some steps rerun
            g.pbf_step(np.float32(cfg.dt), 4)
            out.append(g.pbf_download(order=0) + tuple(np.asarray(q) for q in g.pbf_learned_stats(True)))
    same(out[0], out[1])
    same(out[0], out[2])


@pytest.mark.parametrize("exact", [True, False])
def test_recorded_rows(gpu_mod, exact):
    cfg, pos, vel = scene(*SCENES[2], seed=3)
    out = []
    for staged in (0, 1, 2):
        with gpu_mod.Gpu(0) as g:
            g.pbf_set_build(staged)
            g.pbf_init(gpu_mod.pbf_params(cfg, exact=exact), pos, vel)
            t = g.trainer(4 * cfg.n)
            for _ in range(3):
                t.record_step(np.float32(cfg.dt), 3)
            out.append(t.download())
            t.close()
    same(out[0], out[1])
    same(out[0], out[2])


def test_batch(gpu_mod):
    # scenes of different sizes in one grid: blocks that span scenes
    cfgs = [scenes.dam_break_of_size(n, n) for n in (40, 700, 2500, 90)]
    pos = np.concatenate([c.positions() for c in cfgs])
    out = []
    for staged in (0, 1, 2):
        with gpu_mod.Gpu(0) as g:
            g.pbf_set_build(staged)
            g.pbf_set_lanes(1)
            g.pbf_batch_init(gpu_mod.pbf_params(cfgs[0], exact=False), [c.n for c in cfgs], [c.box for c in cfgs], pos)
            g.pbf_step(np.float32(cfgs[0].dt), 3)
            out.append(g.pbf_download(order=1))
    same(out[0], out[1])
    same(out[0], out[2])


@pytest.mark.parametrize("exact", [True, False])
@pytest.mark.parametrize("lat", [(64, 32, 64), (64, 33, 64)])
def test_either_side_of_the_layered_build(gpu_mod, lat, exact):
    # 131072 particles: a wave per stencil layer; 135168: a lane per particle
    cfg, pos, vel = scene(lat, (140, 72, 140), 0.2, 5)
    same(plain(gpu_mod, cfg, pos, vel, 1, exact, steps=1), plain(gpu_mod, cfg, pos, vel, 0, exact, steps=1))
