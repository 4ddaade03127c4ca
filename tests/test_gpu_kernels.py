"""The operator kernels at the sizes where their tiling can go wrong: edges of
tiles, remainders, empty and full selections, misaligned buffers."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from oracle import oracle as O  # noqa: E402


@pytest.fixture(scope="module")
def ops():
    import torch
    assert torch.cuda.is_available()
    from sycldb_amd import ops as M
    return M


def dev(a, off=0):
    """The array on the device, `off` elements past an aligned start."""
    import torch
    t = torch.zeros(len(a) + off, dtype=torch.from_numpy(a[:0]).dtype, device="cuda")
    t[off:] = torch.from_numpy(a)
    return t[off:]


def flags_of(rng, n, density):
    """Flags of any nonzero byte value, a share `density` of them set."""
    return np.where(rng.random(n) < density, rng.integers(1, 256, n), 0).astype(np.uint8)


# a wave's tile is 4,096 rows, a block's four of them; off: flags not 16-byte aligned
@pytest.mark.parametrize("n", [1, 15, 16, 17, 1023, 1024, 1025, 4095, 4096, 4097, 16384, 16385, 70_001])
@pytest.mark.parametrize("density,off", [(0.0, 0), (0.03, 0), (0.6, 3), (1.0, 0), (1.0, 16)])
def test_compact_count_sum_tile_edges(ops, n, density, off):
    import torch
    rng = np.random.default_rng(n)
    fl = flags_of(rng, n, density)
    col = rng.integers(-2**31, 2**31, n).astype(np.int32)
    f, c = dev(fl, off), dev(col, off % 4)
    ids = torch.full((n + 1,), -1, dtype=torch.int32, device="cuda")
    count = torch.zeros(1, dtype=torch.int32, device="cuda")
    ops.compact(f, ids, count, n=n)
    want = np.flatnonzero(fl)
    assert int(count.item()) == len(want) == ops.count_true_flags(f, n)
    got = ids.cpu().numpy()
    assert (got[:len(want)] == want).all() and (got[len(want):] == -1).all()
    acc = torch.zeros(1, dtype=torch.int64, device="cuda")
    ops.sum_flagged(c, f, acc, n=n)
    assert int(acc.item()) == int(col[want].astype(np.int64).sum())


def test_compact_scan_takes_several_steps(ops):
    """More tiles than one step of the scan takes (16,384), with a remainder."""
    import torch
    n = (1 << 26) + 4096 * 5 + 7
    g = torch.Generator("cuda").manual_seed(3)
    f = (torch.rand(n, generator=g, device="cuda") < 0.2).to(torch.uint8)
    ids = torch.full((n,), -1, dtype=torch.int32, device="cuda")
    count = torch.zeros(1, dtype=torch.int32, device="cuda")
    ops.compact(f, ids, count)
    want = f.nonzero().squeeze(1).int()
    k = int(count.item())
    assert k == len(want) and bool((ids[:k] == want).all()) and bool((ids[k:] == -1).all())


# a wave lists up to 512 rows of its 2,048-row tile at once: sparse, just
# around that, and dense tiles; 1 to 5 keys; keys in and out of their ranges
@pytest.mark.parametrize("density", [0.0, 0.01, 0.24, 0.26, 1.0])
@pytest.mark.parametrize("n,nkeys,off", [(1, 1, 0), (2047, 2, 0), (2049, 3, 0), (32768, 4, 0), (33_001, 5, 0), (40_003, 2, 1)])
def test_groupby_lds_tiles(ops, density, n, nkeys, off):
    import torch
    rng = np.random.default_rng(n + nkeys)
    spans = [(-2, 3), (1992, 1998), (0, 4), (7, 9), (10, 12)][:nkeys]
    mins, maxs = [a for a, _ in spans], [b for _, b in spans]
    prod = int(np.prod([b - a + 1 for a, b in spans]))
    stray = 1 if nkeys <= 2 else 0
    keys = [rng.integers(a - stray, b + 1 + stray, n).astype(np.int32) for a, b in spans]
    agg = rng.integers(-2**31, 2**31, n).astype(np.int32)
    fl = flags_of(rng, n, density)
    sums, seen = (torch.zeros(prod, dtype=d, device="cuda") for d in (torch.int64, torch.int32))
    outk = [torch.full((prod,), -7, dtype=torch.int32, device="cuda") for _ in spans]
    ops.groupby_dense([dev(k, off) for k in keys], mins, maxs, dev(agg, off), dev(fl, off), outk, sums, seen, prod, n=n)
    w_sums, w_seen = np.zeros(prod, np.uint64), np.zeros(prod, np.uint32)
    w_keys = [np.full(prod, -7, np.int32) for _ in spans]
    O.groupby_dense(keys, mins, maxs, agg, fl, w_keys, w_sums, w_seen, prod)
    assert (sums.cpu().numpy().view(np.uint64) == w_sums).all()
    assert (seen.cpu().numpy().view(np.uint32) == w_seen).all()
    if not stray:  # out-of-range rows leave which of a slot's rows stores its keys open
        for a, b in zip(outk, w_keys):
            assert (a.cpu().numpy()[w_seen != 0] == b[w_seen != 0]).all()


def test_groupby_lds_largest_range(ops):
    """The largest slot count held in LDS, and one more (global atomics)."""
    import torch
    rng = np.random.default_rng(11)
    n = 50_000
    for prod in (8065, 8066):
        key = rng.integers(0, prod, n).astype(np.int32)
        agg = rng.integers(-1000, 1000, n).astype(np.int32)
        fl = flags_of(rng, n, 0.3)
        sums, seen = (torch.zeros(prod, dtype=d, device="cuda") for d in (torch.int64, torch.int32))
        out = torch.zeros(prod, dtype=torch.int32, device="cuda")
        ops.groupby_dense([dev(key)], [0], [prod - 1], dev(agg), dev(fl), [out], sums, seen, prod)
        want = np.bincount(key[fl != 0], weights=agg[fl != 0], minlength=prod).astype(np.int64)
        assert (sums.cpu().numpy() == want).all()
        assert ((seen.cpu().numpy() != 0) == (np.bincount(key[fl != 0], minlength=prod) > 0)).all()


# Probes over at least 4M rows and 16 rows per table slot: the 16-bit table in
# LDS up to 65,536 slots; the presence bitmap in LDS, whole up to 2^20 slots,
# folded above; few matches (listed) and many (gathered where they lie), few
# and many flagged rows; values too wide for 16 bits; in place; a ragged end.
@pytest.mark.parametrize("length,match,flagged,wide", [
    (1, 1.0, 1.0, False), (61_130, 0.04, 0.01, False), (65_536, 1.0, 0.5, False), (65_536, 0.5, 1.0, True),
    (65_537, 0.03, 1.0, False), (65_537, 0.9, 0.3, True), (300_000, 0.2, 0.02, False), (280_001, 0.0, 1.0, False)])
def test_probe_full_lds_tables(ops, length, match, flagged, wide):
    import torch
    rng = np.random.default_rng(length)
    n, mn = 4_500_003, -1000
    mx = mn + length - 1
    pairs = np.zeros(2 * length, np.int32)
    pairs[0::2] = np.where(rng.random(length) < match, 1, rng.integers(0, 2, length) * 2)  # 2 is no match
    pairs[1::2] = rng.integers(-5, 65_529 if not wide else 2**31, length)
    probe = rng.integers(mn - length // 8 - 1, mx + length // 8 + 2, n).astype(np.int32)
    probe[:3] = [-2**31, 2**31 - 1, mx]
    fl = flags_of(rng, n, flagged)
    tf, vo = dev(fl), torch.full((n,), -77, dtype=torch.int32, device="cuda")
    ops.full_join(dev(probe), vo, tf, n, dev(pairs), mn, mx)
    want, want_v = np.zeros(n, np.uint8), np.full(n, -77, np.int32)
    O.probe_full(probe, want_v, fl, want, pairs, mn, mx)
    assert (tf.cpu().numpy() == want).all() and (vo.cpu().numpy() == want_v).all()


@pytest.mark.parametrize("n", [4 << 20, (4 << 20) + 1, (4 << 20) + 2047])
@pytest.mark.parametrize("length", [1000, 70_000])
def test_probe_full_lds_ends(ops, n, length):
    """Rows in whole tiles of 2,048 only, and one and 2,047 past them."""
    import torch
    rng = np.random.default_rng(n)
    pairs = np.zeros(2 * length, np.int32)
    pairs[0::2] = rng.random(length) < 0.5
    pairs[1::2] = rng.integers(0, 1000, length)
    probe = rng.integers(-5, length + 5, n).astype(np.int32)
    fl = flags_of(rng, n, 0.5)
    tf, vo = dev(fl), torch.full((n,), -77, dtype=torch.int32, device="cuda")
    ops.full_join(dev(probe), vo, tf, n, dev(pairs), 0, length - 1)
    want, want_v = np.zeros(n, np.uint8), np.full(n, -77, np.int32)
    O.probe_full(probe, want_v, fl, want, pairs, 0, length - 1)
    assert (tf.cpu().numpy() == want).all() and (vo.cpu().numpy() == want_v).all()


@pytest.mark.parametrize("length,match", [(1_400_000, 0.04), (1_400_000, 0.7), (2_097_152, 0.01), (2_097_153, 0.01)])
def test_probe_full_folded_filter(ops, length, match):
    """Tables of more slots than the filter has bits, up to its largest fold
    and one slot past it (no filter)."""
    import torch
    g = torch.Generator("cuda").manual_seed(length)
    n, mn = 16 * length + 5, 7
    pairs = torch.zeros(2 * length, dtype=torch.int32, device="cuda")
    pairs[0::2] = (torch.rand(length, generator=g, device="cuda") < match).int()
    pairs[1::2] = torch.randint(100, 1100, (length,), generator=g, device="cuda", dtype=torch.int32)
    probe = torch.randint(mn - 50, mn + length + 50, (n,), generator=g, device="cuda", dtype=torch.int32)
    fl = (torch.rand(n, generator=g, device="cuda") < 0.9).to(torch.uint8)
    out, vo = torch.full((n,), 9, dtype=torch.uint8, device="cuda"), torch.full((n,), -7, dtype=torch.int32, device="cuda")
    ops.probe_full(probe, vo, fl, out, pairs, mn, mn + length - 1)
    s = probe - mn
    inside = (s >= 0) & (s < length)
    s = torch.where(inside, s, 0).long()
    hit = (fl != 0) & inside & (pairs[0::2][s] == 1)
    assert bool((out == hit).all()) and bool((vo == torch.where(hit, pairs[1::2][s], -7)).all())


# Semi probes over at least 4M rows and 128 rows per table slot read a bitmap
# in LDS: one slot, around the 16 slots a thread packs, a table that is not
# 16-byte aligned (no bitmap), the largest table and one slot more; in place.
@pytest.mark.parametrize("length,off,flagged", [
    (1, 0, 1.0), (15, 0, 0.5), (17, 0, 1.0), (61_130, 0, 0.02), (61_130, 1, 1.0), (300_000, 0, 0.9),
    (655_360, 0, 0.9), (655_361, 0, 0.9)])
def test_probe_semi_lds_tables(ops, length, off, flagged):
    import torch
    g = torch.Generator("cuda").manual_seed(length)
    n, mn = max(128 * length, 4 << 20) + 3, -1000
    ht = torch.zeros(length + off, dtype=torch.uint8, device="cuda")
    ht[off:] = torch.randint(0, 3, (length,), generator=g, device="cuda", dtype=torch.uint8) * 127
    ht = ht[off:]
    probe = torch.randint(mn - length // 8 - 1, mn + length + length // 8 + 1, (n,), generator=g, device="cuda",
                          dtype=torch.int32)
    probe[:3] = torch.tensor([-2**31, 2**31 - 1, mn + length - 1], dtype=torch.int32, device="cuda")
    fl = (torch.rand(n, generator=g, device="cuda") < flagged).to(torch.uint8) * 3
    s = probe - mn  # the two extreme keys wrap to far outside
    inside = (s >= 0) & (s < length)
    want = (fl != 0) & inside & (ht[torch.where(inside, s, 0)] != 0)
    ops.filter_join(probe, fl, n, ht, mn, mn + length - 1)
    assert bool((fl == want).all())

