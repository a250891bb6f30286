"""Bucket sort at the edges of its segment lists: particles of two blocks
interleaved so that each bucket's list has a given number of segments (one
wave, the LDS sort's powers of two and its limit of 2,048, the radix sort
beyond), as short and as long runs, through the stand-alone operator and
through a substep. Integer results: exact against a stable argsort."""
import dataclasses

import numpy as np
import pytest

from zpc_amd import scenes as S

pytestmark = pytest.mark.gpu


def _scene(segments, run, tail):
    """`segments` runs of `run` particles alternating between two blocks, then
    `tail` particles of a third, all inside their blocks."""
    dx = 1.0 / 64
    n = segments * run
    block = np.repeat(np.arange(segments) % 2, run)
    block = np.concatenate([block, np.full(tail, 2)])
    rng = np.random.default_rng(segments * 31 + run)
    lo = np.array([[20, 20, 20], [24, 20, 20], [20, 28, 20]])  # node of each block's first cell
    pos = (lo[block] + 2.0 + 3.0 * rng.random((n + tail, 3))) * dx
    base = S.tiny_scene(dx=dx)
    x = pos.astype(np.float32)
    v, C, F, m, _ = S._state(x, base.material)
    return dataclasses.replace(base, x=x, v=v, C=C, F=F, m=m, table_size=1024), block


@pytest.mark.parametrize("driver", ["operator", "substep"])
@pytest.mark.parametrize("segments,run", [(2, 1), (2, 640), (126, 3), (128, 1), (130, 1), (130, 70), (512, 1),
                                          (514, 1), (1026, 8), (2046, 1), (2050, 1), (2050, 8), (4094, 1), (4096, 1),
                                          (4096, 8), (4098, 1), (4098, 8), (8190, 1), (8192, 1), (8194, 1),
                                          (8194, 5), (20002, 1)])
def test_segment_lists_exact(driver, segments, run):
    from zpc_amd import rocm

    sc, block = _scene(segments, run, tail=3)
    c = np.floor(sc.x * np.float32(64) + np.float32(0.5)).astype(np.int64) - 2
    key = np.floor_divide(c, 4)
    _, first, inv = np.unique(key, axis=0, return_index=True, return_inverse=True)
    rank = np.empty(len(first), np.int64)
    rank[np.argsort(first)] = np.arange(len(first))
    bucket = rank[inv.reshape(-1)]
    want = np.argsort(bucket, kind="stable")
    counts = np.bincount(bucket)
    sim = rocm.Simulator(sc)
    if driver == "substep":
        sim.substep()
    else:
        sim.clear_table()
        sim.activate()
        sim.enlarge()
        sim.bucket_sort()
    sim.sync()
    gc, go, gi = sim.buckets.host(sim.nblocks(), sc.n)
    k = len(counts)
    assert np.array_equal(gc[:k], counts) and not gc[k:].any()
    assert np.array_equal(go[:k], np.cumsum(counts) - counts) and np.all(go[k:] == sc.n)
    assert np.array_equal(gi, want)


@pytest.mark.parametrize("driver", ["operator", "substep", "graph"])
@pytest.mark.parametrize("segments,run", [(2, 1), (6, 640), (130, 70), (300, 256), (9, 1024), (700, 3001)])
def test_counters_runs_and_new_keys(driver, segments, run):
    """The diagnostic counters: particle runs of the last bucket sort, whatever
    tiles the sort cuts them into (both tile sizes), and the new keys of the
    last insertion (the enlargement's)."""
    from zpc_amd import rocm

    sc, block = _scene(segments, run, tail=3)
    sim = rocm.Simulator(sc, reorder=driver == "graph")
    if driver == "operator":
        sim.clear_table()
        sim.activate()
        sim.sync()
        assert sim.pol.counters()[0] == 3
        sim.enlarge()
        sim.bucket_sort()
    elif driver == "substep":
        sim.substep()
    else:  # particles in bucket order from the second substep on: a run per block
        sim.substeps(4, graph=True)
    sim.sync()
    got = sim.pol.counters()
    assert got[0] == sim.nblocks() - 3
    assert got[2] == (3 if driver == "graph" else segments + 1)
    assert sim.pol.counters()[2] == got[2]
