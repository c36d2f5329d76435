"""simulate_fluid's data-flow sweep at the edges of its two forms.  Up to 65,536
particles a wave holds one of them and a block four, above that four and
sixteen; either takes a list 64 entries at a time.  So: counts around a block
of the first form, lists of 63 to 129 entries, counts either side of the switch
and on and past a whole block of the second form, with lists past one and two
chunks there too.  Bar as in test_gpu_fluid_sweep.py."""
import numpy as np
import pytest

from test_gpu_fluid_sweep import REL, cloud, step_both

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5])
def test_counts_around_a_block(gpu_mod, oracle, n):
    p = np.zeros((24 ** 3, 3), np.float32)
    p[:n] = cloud(n, 1.0, n)
    step_both(gpu_mod, oracle, p, (0, n), (len(p) - 1, len(p) - 1))


@pytest.mark.parametrize("n", [63, 64, 65, 127, 128, 129])
def test_lists_around_a_chunk(gpu_mod, oracle, n):
    # every particle within h = 2 of every other (and in its own list): n entries each
    p = np.zeros((24 ** 3, 3), np.float32)
    p[:n] = cloud(n, 0.9, n)
    assert step_both(gpu_mod, oracle, p, (0, n), (len(p) - 1, len(p) - 1)) == n


@pytest.mark.parametrize("n,cluster", [(65536, 65), (65537, 64), (65552, 65), (65553, 129)])
def test_counts_around_the_switch(gpu_mod, oracle, n, cluster):
    m = n - cluster
    p = np.zeros((48 ** 3, 3), np.float32)
    p[:m] = cloud(m, 40.0, 1) * np.float32(0.9)
    p[m:n] = cloud(cluster, 0.9, 2) + np.float32(40.0)  # away from the block: lists of `cluster` entries
    none = (len(p) - 1, len(p) - 1)
    s = oracle.init_constants(48, 48, 48, 0.5, 1.0, 4.0)
    po, pso, vo, lo = p.copy(), p.copy(), np.zeros_like(p), np.zeros(len(p), np.float32)
    oracle.simulate_fluid(s, po, pso, vo, lo, (0, n), none, 1.0 / 60.0)
    with gpu_mod.Gpu(0) as g:
        g.fluid_init(gpu_mod.fluid_params(s), p, p, np.zeros_like(p), (0, n), none)
        g.fluid_step(1.0 / 60.0)
        gp, gps, gv, gl = g.fluid_download()
    assert np.array_equal(gl[:n], lo[:n])
    assert np.array_equal(gps[:n], gp[:n])
    assert np.abs(gp.astype(np.float64) - po).max() <= REL * np.abs(po).max()
