"""P2G and the substep at negative coordinates, where the rounding of X - 0.5
can leave the local position l just below 0.5: floor(l - 0.5) is -1 there and
the B-spline's argument l + 1, in every transfer as in the oracle. Particles
sit on such positions in one, two and three axes, between ordinary ones.

Tolerances: m and m v are sums of a few float32 products, 1e-5 of the largest;
the force holds a float32 SVD's error of some 5e-7 on strains of 0.02, 1e-4;
state after the substep 1e-4. A weight off by one node changes them by O(1)."""
import dataclasses

import numpy as np
import pytest

from oracle import oracle as O
from zpc_amd import scenes as S

from test_gpu_parity import _oracle_particles, _rocm, rel_err

pytestmark = pytest.mark.gpu


def _below(dx, cell):
    """The position nearest -(cell + 0.5) dx whose float32 l is below 0.5."""
    f = np.float32
    x = f(-(cell + 0.5)) * f(dx)
    for _ in range(200):
        X = f(x / f(dx))
        if f(X - np.floor(f(X - f(0.5)))) < f(0.5):
            return x
        x = np.nextafter(x, f(-np.inf), dtype=np.float32)
    return None


@pytest.mark.parametrize("dx", [1.0 / 64, 1.0 / 48])
def test_weights_at_negative_positions(dx):
    f = np.float32
    edge = [x for x in (_below(f(dx), c) for c in (63, 127, 255)) if x is not None]
    assert edge
    rng = np.random.default_rng(9)
    pos = []
    for e in edge:
        for axes in range(8):
            p = e + rng.uniform(-3, 3, 3) * dx
            for d in range(3):
                if axes >> d & 1:
                    p[d] = e
            pos += [p, e + rng.uniform(-3, 3, 3) * dx]
    x = np.asarray(pos, np.float32)
    base = S.tiny_scene(dx=dx)
    v, C, F, m, _ = S._state(x, base.material)
    v = rng.uniform(-0.5, 0.5, v.shape).astype(np.float32)
    F = (F + 0.02 * rng.standard_normal(F.shape)).astype(np.float32)
    sc = dataclasses.replace(base, x=x, v=v, C=C, F=F, m=m, colliders=[], table_size=S._table_size_for(x, dx))
    X = (x / f(dx)).astype(np.float32)
    assert ((X - np.floor(X - f(0.5))) < 0.5).any(1).sum() >= 4 * len(edge)

    rocm = _rocm()
    prm = O.make_params(sc)
    ctx = O.Context()
    ctx.activate(sc.table_size, sc.x, sc.dx)
    ctx.enlarge()
    ctx.bucket_sort(sc.x, sc.dx)
    ctx.p2g(prm, _oracle_particles(sc))
    want, _, _ = ctx.grids()
    sim = rocm.Simulator(sc)
    sim.clear_table()
    sim.activate()
    sim.enlarge()
    sim.bucket_sort()
    sim.clear_grid()
    sim.p2g()
    sim.sync()
    got = sim.grid.data[:sim.nblocks()].cpu().numpy()
    assert got.shape == want.shape
    for ch, name, tol in ((slice(0, 1), "m", 1e-5), (slice(1, 4), "mv", 1e-5), (slice(4, 7), "rhs", 1e-4)):
        assert rel_err(got[:, ch], want[:, ch]) < tol, name

    sim = rocm.Simulator(sc)
    sim.substep()
    sim.sync()
    ps = _oracle_particles(sc)
    O.Context().run(prm, ps, 1)
    out = sim.parts.host()
    for name in ("x", "v", "C", "F"):
        assert rel_err(out[name], getattr(ps, name)) < 1e-4, name
