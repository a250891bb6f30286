"""P2G and G2P of small scenes run a bucket in more waves than the general
launch. At the edges of a wave, a bucket and of both rules (capacities of up to
1,024 and 2,048 buckets) a substep in each launch shape is the same up to float
summation order.

Tolerance: a node sums at most 27 * 16 particle terms in an order that
differs, so its mass and momentum are off by at most 432 * 2^-24 = 2.6e-5 of
the terms' sizes and its velocity by twice that of the largest term, taken as
4 (|v| <= 1, and the affine and stress parts of a term below 3): 2.1e-4 in v,
dt of it in x, 4 / dx * 1.5 of it in C and dt of that in F."""
import dataclasses

import numpy as np
import pytest

from zpc_amd import scenes as S

pytestmark = pytest.mark.gpu


def _scene(n):
    rng = np.random.default_rng(n)
    base = S.tiny_scene(dx=1.0 / 64)
    side = (n / 8) ** (1 / 3) + 0.5  # cells: 8 particles each
    x = ((4.3 + side * rng.random((n, 3))) / 64).astype(np.float32)
    v, C, F, m, _ = S._state(x, base.material)
    v = rng.uniform(-0.5, 0.5, v.shape).astype(np.float32)
    return dataclasses.replace(base, x=x, v=v, C=C, F=F, m=m, table_size=S._table_size_for(x, 1.0 / 64))


def _same(sc, a, b):
    dv = 2.1e-4
    dC = 6.0 * 64 * dv
    for name, tol in (("x", sc.dt * dv + 1e-7), ("v", dv), ("C", dC), ("F", sc.dt * dC + 1e-6)):
        assert np.max(np.abs(a[name] - b[name])) <= tol, name


@pytest.mark.parametrize("reorder", [False, True])
@pytest.mark.parametrize("capacity", [1024, 1025, 2048, 2049])
@pytest.mark.parametrize("n", [600, 64000])
def test_launch_at_the_capacity_lines(n, capacity, reorder):
    from zpc_amd import rocm

    sc = _scene(n)
    got = []
    for tiles in ((0, 0), (576, 128)):
        sim = rocm.Simulator(sc, reorder=reorder, grid_capacity=capacity)
        sim.pol.set_launch_tiles(*tiles)
        sim.substep()
        sim.sync()
        got.append(sim.parts.host())
    _same(sc, *got)


@pytest.mark.parametrize("reorder", [False, True])
@pytest.mark.parametrize("n", [1, 64, 577, 4096, 76800, 76801, 262144, 262145])
def test_wide_launch_matches_general(n, reorder):
    from zpc_amd import rocm

    sc = _scene(n)
    got = []
    for tiles in ((0, 0), (256, 128)):
        sim = rocm.Simulator(sc, reorder=reorder)
        sim.pol.set_launch_tiles(*tiles)
        sim.substep()
        sim.sync()
        got.append(sim.parts.host())
    _same(sc, *got)
