"""The data-flow form of simulate_fluid's sequential sweep: particle counts up
to 4,099 and past the switch to four particles per wave (65,536), lists within
and past the 64 entries taken at a time (several chunks), moving slots that do
not start at 0 with solids before and after them, and exponents other
than 4.  Same bar as test_gpu_fluid.py: positions within 1e-5 relative of the
FP32 oracle (the one call that differs, the power in s_coor, is off by one ulp
for about 7 in 10,000 arguments), lambdas of the step bit for bit.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

REL = 1e-5


def cloud(n, side, seed):
    """n points of a jittered lattice squeezed into a cube of the given side."""
    m = int(np.ceil(n ** (1.0 / 3.0)))
    g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    r = np.random.default_rng(seed)
    p = (g + 0.5 + r.uniform(-0.2, 0.2, g.shape)) * (side / m) + 6.0
    return p[r.permutation(n)].astype(np.float32)  # waits run through the whole array


def step_both(gpu_mod, oracle, p, sand, solid, exponent=4.0):
    s = oracle.init_constants(24, 24, 24, 0.5, 1.0, 4.0)
    s.s_corr_n = exponent
    total = p.shape[0]
    po, pso, vo, lo = p.copy(), p.copy(), np.zeros_like(p), np.zeros(total, np.float32)
    oracle.simulate_fluid(s, po, pso, vo, lo, sand, solid, 1.0 / 60.0)
    with gpu_mod.Gpu(0) as g:
        g.fluid_init(gpu_mod.fluid_params(s), p, p, np.zeros_like(p), sand, solid)
        g.fluid_step(1.0 / 60.0)
        gp, gps, gv, gl = g.fluid_download()
        levels, entries = g.fluid_stats()
    a, b = sand
    assert np.array_equal(gl[a:b], lo[a:b])
    err = np.abs(gp.astype(np.float64) - po).max() / np.abs(po).max()
    print(f"n {b - a}: {entries} entries, longest chain {levels}, x rel {err:.2e}")
    assert err <= REL
    assert np.array_equal(gps[a:b], gp[a:b])           # positions_star = positions after the sweep
    assert np.array_equal(np.delete(gp, np.s_[a:b], 0), np.delete(p, np.s_[a:b], 0))
    assert 1 <= levels <= b - a
    return entries / (b - a)


@pytest.mark.parametrize("n", [7, 8, 9, 31, 32, 33, 255, 257, 4099])
def test_sweep_counts(gpu_mod, oracle, n):
    p = np.zeros((24 ** 3, 3), np.float32)
    p[:n] = cloud(n, float(np.ceil(n ** (1.0 / 3.0))), n)
    step_both(gpu_mod, oracle, p, (0, n), (len(p) - 1, len(p) - 1))


@pytest.mark.parametrize("n,side", [(48, 1.2), (49, 1.2), (97, 1.5), (300, 2.0)])
def test_sweep_long_lists(gpu_mod, oracle, n, side):
    # nearly every particle within h of every other: lists of up to n entries
    p = np.zeros((24 ** 3, 3), np.float32)
    p[:n] = cloud(n, side, n)
    assert step_both(gpu_mod, oracle, p, (0, n), (len(p) - 1, len(p) - 1)) > 0.5 * n


@pytest.mark.parametrize("exponent", [4.0, 3.0, 2.5])
def test_sweep_slots_and_exponents(gpu_mod, oracle, exponent):
    # solids in the slots below the moving ones (never waited for), unused slots above
    n, ns = 700, 200
    p = np.zeros((24 ** 3, 3), np.float32)
    p[:ns] = cloud(ns, 6.0, 5)
    p[:ns, 1] = np.float32(5.5)
    p[ns:ns + n] = cloud(n, 8.0, 6)
    step_both(gpu_mod, oracle, p, (ns, ns + n), (0, ns), exponent)


def test_sweep_large_scene(gpu_mod, oracle):
    # past 65,536 particles the sweep holds four particles per wave; a dense
    # cluster gives lists past one chunk there too
    n = 70003
    p = np.zeros((48 ** 3, 3), np.float32)
    p[:n - 150] = cloud(n - 150, 40.0, 1)
    p[n - 150:n] = cloud(150, 1.6, 2)
    s = oracle.init_constants(48, 48, 48, 0.5, 1.0, 4.0)
    po, pso, vo, lo = p.copy(), p.copy(), np.zeros_like(p), np.zeros(len(p), np.float32)
    oracle.simulate_fluid(s, po, pso, vo, lo, (0, n), (len(p) - 1, len(p) - 1), 1.0 / 60.0)
    with gpu_mod.Gpu(0) as g:
        g.fluid_init(gpu_mod.fluid_params(s), p, p, np.zeros_like(p), (0, n), (len(p) - 1, len(p) - 1))
        g.fluid_step(1.0 / 60.0)
        gp, gps, gv, gl = g.fluid_download()
    assert np.array_equal(gl[:n], lo[:n])
    assert np.abs(gp.astype(np.float64) - po).max() <= REL * np.abs(po).max()
