"""Graph replays between steps of another form: what the library notes of the
last step (list form, block maxima) and the cell keys at hand have to be the
replayed steps'.  Each sequence against the same one without graphs."""
import numpy as np
import pytest

from lustrine_amd import scenes
from oracle import mlp as M

pytestmark = pytest.mark.gpu


def _dense(n, side, seed):
    """n particles squeezed into a cube that the box holds them in: lists past 128 entries."""
    rng = np.random.default_rng(seed)
    pos = rng.uniform(1.0, side - 1.0, (n, 3)).astype(np.float32)
    return scenes.small(1, 1, 1, box=(side,) * 3), pos


@pytest.mark.parametrize("lanes,build", [(0, 2), (4, 2), (1, 2), (0, 1)])
def test_recorded_steps_between_replays(gpu_mod, lanes, build):
    # plain steps with four lanes keep flat lists, recorded ones (one lane)
    # block-staged lists: the retest count reads one table or the other
    cfg, pos = _dense(4000, 10, 3)
    dt = np.float32(cfg.dt)
    out = []
    for graph in (False, True):
        with gpu_mod.Gpu(0) as g:
            g.pbf_set_build(build)
            g.pbf_set_lanes(lanes)
            g.pbf_init(gpu_mod.pbf_params(cfg, exact=False), pos)
            g.pbf_set_graph(graph)
            t = g.trainer(4 * len(pos))
            g.pbf_step(dt, 3)  # one ordinary step, then a captured pair
            for _ in range(2):
                t.record_step(dt, 1)
            g.pbf_step(dt, 2)  # replayed
            got = [g.pbf_retest_count(), g.pbf_last_max_constraint(), *g.pbf_download(order=0)]
            if len(out) and got[0] == out[0][0]:  # (its passes walk the table that the count was read from)
                assert all(u > 0.0 for u in g.pbf_time_kernels(reps=2).values())
            out.append(got)
    assert out[0][0] > 0
    for a, b in zip(*out):
        assert np.array_equal(a, b)


def _moving(seed):
    """Particles fast enough to be predicted in other cells with other step lengths."""
    cfg = scenes.small(12, 10, 12, box=(24, 20, 24), seed=seed)
    pos = cfg.positions()
    vel = np.random.default_rng(seed).uniform(-60.0, 60.0, pos.shape).astype(np.float32)
    return cfg, pos, vel


@pytest.mark.parametrize("exact", [True, False])
def test_steps_of_another_length_between_replays(gpu_mod, exact):
    # the captured steps sort by keys that the step before them wrote for their dt
    cfg, pos, vel = _moving(8)
    dt = np.float32(cfg.dt)
    out = []
    for graph in (False, True):
        with gpu_mod.Gpu(0) as g:
            g.pbf_init(gpu_mod.pbf_params(cfg, exact=exact), pos, vel)
            g.pbf_set_graph(graph)
            g.pbf_step(dt, 3)
            for _ in range(2):
                g.pbf_step(np.float32(0.125) * dt, 1)
            for _ in range(3):
                g.pbf_step(dt, 2)
            out.append(g.pbf_download(order=0))
    for a, b in zip(*out):
        assert np.array_equal(a, b)


def test_recorded_steps_between_learned_replays(gpu_mod):
    # learned steps write no keys: their captured key kernel counts into a
    # cleared histogram, which a recorded step leaves filled
    cfg, pos, vel = _moving(9)
    dt = np.float32(cfg.dt)
    out = []
    for graph in (False, True):
        with gpu_mod.Gpu(0) as g:
            g.pbf_init(gpu_mod.pbf_params(cfg, exact=True), pos, vel)
            g.pbf_set_network(np.concatenate([np.zeros(32), np.ones(32), np.zeros(M.N_PARAMS), [1.0]]))
            g.pbf_set_mode(learned=True, learned_iterations=2, bound=0.2)
            g.pbf_set_graph(graph)
            t = g.trainer(2 * len(pos))
            g.pbf_step(dt, 2)
            for _ in range(2):
                t.record_step(dt, 1)
            for _ in range(3):
                g.pbf_step(dt, 2)
            out.append((*g.pbf_download(order=0), *g.pbf_learned_stats(True)))
    for a, b in zip(*out):
        assert np.array_equal(a, b)
