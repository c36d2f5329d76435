"""Graph replays between steps of another form: what the library notes of the
last step (list form, block maxima) and the cell keys at hand have to be the
replayed steps'.  Each sequence against the same one without graphs."""
import numpy as np
import pytest

from lustrine_amd import scenes

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
