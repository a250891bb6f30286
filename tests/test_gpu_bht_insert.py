"""Insertion at the edges of its steps: words of 64 keys, tiles of 1,024, the
line of 2^20 keys, runs of equal keys across them, mostly distinct keys, and more
distinct keys than twice the table's slots
(the deduplication starts again with a larger hash); sampling on positions that
share blocks and on positions that do not. Whole numbers: exact against the
sequential insertion; samples are the same operations in the same order, equal
to 1e-6."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("run", [1, 7, 64])
@pytest.mark.parametrize("T,n", [(4096, 1), (4096, 63), (4096, 64), (4096, 65), (4096, 1023), (4096, 1025),
                                 (4096, 4097), (64, 1500), (64, 40000), (32768, (1 << 20) - 1),
                                 (32768, 1 << 20), (32768, (1 << 20) + 65)])
def test_insert_edges(T, n, run):
    import torch
    from zpc_amd import rocm

    rng = np.random.default_rng(n + run)
    span = 40 if T == 64 else 12
    keys = np.repeat(rng.integers(-span, span, size=((n + run - 1) // run, 3)), run, axis=0)[:n].astype(np.int32)
    h = O.HostBht(T)
    ref = h.insert(keys)
    t = rocm.DeviceBht(T)
    got = t.insert(torch.as_tensor(keys).cuda()).cpu().numpy()
    if int(h.success[0]):
        t.pol.sync()
        cnt = int(t.cnt.item())
        assert cnt == int(h.cnt[0])
        assert np.array_equal(t.keys.cpu().numpy().reshape(-1), h.keys)
        assert np.array_equal(t.active.cpu().numpy().reshape(-1)[:3 * cnt], h.active[:3 * cnt])
        assert np.array_equal(got, ref)
        return
    # a full table: a key's first occurrence takes its number or the failure
    # token, a repeat -1 (where the sequential insertion fails once more)
    with pytest.raises(rocm.ZsmpmError) as e:
        t.pol.sync()
    assert e.value.code == -7
    first = np.zeros(n, bool)
    first[np.unique(keys, axis=0, return_index=True)[1]] = True
    rank = np.cumsum(first) - 1
    assert np.array_equal(got[~first], np.full(int((~first).sum()), -1))
    assert np.all((got[first] == rank[first]) | (got[first] == O.BHT_FAILURE))
    assert np.all(got[first & (rank >= T - 20)] == O.BHT_FAILURE)


@pytest.mark.parametrize("n", [1000, 32768, (1 << 20) + 77])
def test_insert_distinct_into_a_used_table(n):
    """Nearly all keys are first occurrences, and half of them are in the table."""
    import torch
    from zpc_amd import rocm

    rng = np.random.default_rng(n)
    keys = rng.integers(-4000, 4000, size=(n, 3)).astype(np.int32)
    h = O.HostBht(1 << 22)
    t = rocm.DeviceBht(1 << 22)
    for part in (keys[::2], keys):
        part = np.ascontiguousarray(part)
        ref = h.insert(part)
        got = t.insert(torch.as_tensor(part).cuda()).cpu().numpy()
        assert int(h.success[0])
        assert np.array_equal(got, ref)
    t.pol.sync()
    assert np.array_equal(t.keys.cpu().numpy().reshape(-1), h.keys)


def test_insert_far_over_the_table_on_used_scratch():
    """More distinct keys than the table's hash takes, and more than the waves
    in flight hold: tiles that begin after the hash was found full are skipped,
    and what the scratch holds there from another insertion must not be read."""
    import torch
    from zpc_amd import rocm

    pol = rocm.Policy()
    g = torch.Generator().manual_seed(5)
    keys = torch.randint(-400000, 400000, (5000011, 3), generator=g, dtype=torch.int32)  # all distinct
    # another layout of the same scratch, filled with slots, indices and packed keys
    big = rocm.DeviceBht(1 << 20, pol)
    big.insert((keys % 64).contiguous().cuda())
    pol.sync()
    assert big.size() == 64 ** 3
    T = 64
    t = rocm.DeviceBht(T, pol)
    got = t.insert(keys.cuda()).cpu().numpy()
    with pytest.raises(rocm.ZsmpmError) as e:
        pol.sync()
    assert e.value.code == -7
    rank = np.arange(keys.shape[0])
    assert np.all((got == rank) | (got == O.BHT_FAILURE))
    assert np.all(got[T - 20:] == O.BHT_FAILURE)
    kept = got[got != O.BHT_FAILURE]
    assert np.array_equal(t.active.cpu().numpy()[kept], keys.numpy()[kept])


@pytest.mark.parametrize("order", ["sorted", "shuffled"])
@pytest.mark.parametrize("n", [1, 65, 30001])
def test_sample_orders(n, order):
    import torch
    from zpc_amd import rocm

    rng = np.random.default_rng(n)
    x = rng.uniform(-0.4, 0.4, size=(n, 3)).astype(np.float32)
    if order == "sorted":
        x = x[np.lexsort((x[:, 2], np.floor(x[:, 1] * 50), np.floor(x[:, 0] * 50)))]
    M = np.diag([0.02, 0.02, 0.02, 1.0])
    g = rocm.DeviceSparseGrid(4000, 2, M, background=-3.0)
    g.activate(torch.as_tensor(x).cuda())
    g.pol.sync()
    g.data.copy_(torch.as_tensor(rng.standard_normal(tuple(g.data.shape)).astype(np.float32)))
    got = g.sample(0, torch.as_tensor(x).cuda(), 2).cpu().numpy().reshape(n, 2)
    one = np.stack([g.sample(c, torch.as_tensor(np.repeat(x[i:i + 1], 3, 0)).cuda()).cpu().numpy()[:1]
                    for i in range(min(n, 40)) for c in (0, 1)]).reshape(-1, 2)
    assert np.allclose(got[:len(one)], one, rtol=0, atol=1e-6)
    # against the cell values gathered on the host
    nb = int(g.table.cnt.item())
    act = g.table.active.cpu().numpy().reshape(-1, 3)[:nb]
    index = {tuple(k): b for b, k in enumerate(act)}
    data = g.data.cpu().numpy().reshape(-1, 2, 512)
    X = x.astype(np.float64) / 0.02
    pick = rng.permutation(n)[:300]
    for i in pick:
        c = np.floor(X[i]).astype(int)
        f = X[i] - c
        want = np.zeros(2)
        for o in range(8):
            d = np.array([o >> 2, (o >> 1) & 1, o & 1])
            a = c + d
            b = index.get(tuple(a & ~7))
            k = ((a[0] & 7) * 8 + (a[1] & 7)) * 8 + (a[2] & 7)
            val = np.full(2, -3.0) if b is None else data[b, :, k]
            want += np.prod(np.where(d == 1, f, 1 - f)) * val
        # X in float32 is off by 20 * 2^-23 cells, times slopes of at most 8
        assert np.all(np.abs(got[i] - want) <= 1e-4), i
