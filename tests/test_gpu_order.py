"""cumm_hip_order_pairs (order_inst.hip): masks, order, tables by position and launch hints of finished pair
tables, against the host builders - sizes around the chunks and tiles, one and two tables, one to
four mask words, kernel volumes from 1 to 125."""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")      # (before the library: one HIP runtime in the process)

import helpers as H
from cumm_amd import _capi, pairs
from cumm_amd import tensorview as tv

pytestmark = pytest.mark.gpu


def _table(rng, kv, n, density):
    t = np.where(rng.random((kv, n)) < density, rng.integers(0, max(n, 1), size=(kv, n)), -1).astype(np.int32)
    t[kv // 2, : n // 2] = np.arange(n // 2)
    return t


UNWRITTEN = -7


def _order(tables, ksize, reverse, entry="cumm_hip_order_pairs"):
    lib, kv = _capi.lib(), tables[0].shape[0]
    words = (kv + 31) // 32
    sides, keep, outs = (_capi.OrderSide * 2)(), [], []
    for s, t in zip(sides, tables):
        n = t.shape[1]
        d = H.dev(t, "i32")
        o = {"mask": tv.empty([n, words], tv.uint32, 0), "order": tv.empty([n], tv.int32, 0), "pos": H.dev(np.full((kv, n), UNWRITTEN, np.int32), "i32"),
             "rev": H.dev(np.full((kv, n), UNWRITTEN, np.int32), "i32")}
        s.indices, s.n, s.sorted_mask, s.argsort = d.byte_pointer(), n, o["mask"].byte_pointer(), o["order"].byte_pointer()
        s.by_position = o["pos"].byte_pointer()
        s.by_position_reversed = o["rev"].byte_pointer() if reverse else None
        keep.append(d)
        outs.append(o)
    need = int(getattr(lib, entry + "_workspace")(sides, len(tables), kv))
    ws = H.dev(np.full(need, 0xA5, np.uint8), "u8")
    _capi.check(getattr(lib, entry)(sides, len(tables), (ctypes.c_int32 * 3)(*ksize), ws.byte_pointer(), ws.nbytes, 0))
    _capi.check(lib.cumm_hip_device_synchronize())
    return [{k: H.host(v) for k, v in o.items()} for o in outs], outs


@pytest.mark.parametrize("ksize", [(3, 3, 3), (1, 1, 1), (2, 2, 2), (4, 4, 2), (3, 3, 5), (5, 5, 5)])
@pytest.mark.parametrize("n,n2", [(1, 0), (63, 64), (256, 257), (4096, 4097), (9000, 130), (270000, 1000)])
def test_masks_order_and_tables(ksize, n, n2):
    kv = int(np.prod(ksize))
    if n > 100000 and kv > 40:
        n = 40000      # (the same branches with a smaller table)
    print("case order", ksize, n, n2, flush=True)
    rng = np.random.default_rng(n + kv)
    tables = [_table(rng, kv, n, 0.05 if kv > 8 else 0.4)] + ([_table(rng, kv, n2, 0.3)] if n2 else [])
    got, dev = _order(tables, ksize, reverse=n2 == 0 or n == 256)
    for t, g, d in zip(tables, got, dev):
        m = pairs.masks_from_pairs(t)
        order = g["order"]
        assert np.array_equal(np.sort(order), np.arange(t.shape[1]))
        np.testing.assert_array_equal(g["mask"], m[order])
        np.testing.assert_array_equal(g["pos"], pairs.pairs_by_position(t, order))
        if n2 == 0 or n == 256:
            np.testing.assert_array_equal(g["rev"], g["pos"][::-1])
        if m.shape[1] == 1:
            s = g["mask"][:, 0]
            count = np.array([bin(int(v)).count("1") for v in s])
            assert np.all(np.diff(count) >= 0)
            light = count[1:] <= 5
            same = np.diff(count) == 0
            assert np.all(np.diff(s.astype(np.int64))[light & same] >= 0)      # exact up to five offsets
            # stable: equal words of up to five offsets in row order
            eq = (np.diff(s.astype(np.int64)) == 0) & light
            assert np.all(np.diff(order)[eq] > 0)
            bits = (1 << kv) - 1 if kv < 32 else 0xFFFFFFFF
            if t is tables[-1] or t.shape[1] != tables[-1].shape[1]:
                hints = pairs.hints_device(d["mask"].view([t.shape[1]]), bits)
                if hints != (-1, -1):      # (the two arrays' slots may coincide: then the second one's stand)
                    assert hints == (pairs.light_prefix(s, bits, 3), pairs.heavy_from(s, bits))
    again, _ = _order(tables, ksize, reverse=False)
    for g, a in zip(got, again):
        np.testing.assert_array_equal(g["order"], a["order"])


def test_a_tile_has_as_few_offsets_as_in_the_exact_order():
    """What the order is for: the offsets of all tiles of 64, on a cloud, against the 32-bit sort by count and
    value (one word) and against the order by count and hash (5 x 5 x 5)."""
    coords, grid = H.small_cloud(5, 6000)
    for ksize in ((3, 3, 3), (5, 5, 5)):
        host = pairs.subm_pairs(coords, grid, ksize)
        (g,), _ = _order([host.indices_fwd], ksize, reverse=False)
        m = pairs.masks_from_pairs(host.indices_fwd)
        other = pairs.sort_by_mask(m[:, 0], (1 << 27) - 1, by_offset_count=True)[1] if m.shape[1] == 1 else pairs.sort_by_mask_words(m)[1]

        def steps(order):
            s = m[order]
            pad = np.zeros(((len(s) + 63) // 64 * 64, s.shape[1]), np.uint32)
            pad[: len(s)] = s
            w = np.bitwise_or.reduce(pad.reshape(-1, 64, s.shape[1]), axis=1)
            return sum(bin(int(v)).count("1") for v in w.ravel())
        assert steps(g["order"]) <= steps(other) * 1.01 + 2


@pytest.mark.parametrize("n,n2", [(511, 513), (512 * 64, 512 * 64 + 1), (1, 512 * 128 + 1), (512 * 64 * 8, 70),
                                  (512 * 64 * 8 + 1, 3), (512 * 64 * 24, 1030), (512 * 64 * 24 + 1, 512 * 64 * 8),
                                  (512 * 64 * 48 - 1, 40), (512 * 64 * 48 + 513, 600000)])
def test_counts_of_many_blocks(n, n2):
    """The digits' counts per block of 512 positions, summed in runs of blocks: a block, a run, the runs of one
    trip of 8, 24 and 48 blocks, and more; exact and stable up to five offsets."""
    print("case order blocks", n, n2, flush=True)
    rng = np.random.default_rng(n)
    tables = [np.where(rng.random((8, m)) < 0.3, np.int32(3), np.int32(-1)) for m in (n, n2)]
    got, _ = _order(tables, (2, 2, 2), reverse=False)
    for t, g in zip(tables, got):
        m = pairs.masks_from_pairs(t)[:, 0].astype(np.int64)
        count = np.array([bin(v).count("1") for v in range(256)])[m]
        light = count <= 5
        want = np.lexsort((m, count))
        assert np.array_equal(g["order"][: int(light.sum())], want[: int(light.sum())])
        assert np.array_equal(np.sort(g["order"]), np.arange(len(m))) and np.array_equal(g["mask"][:, 0], m[g["order"]])


def test_most_positions():
    """A table of one offset just under 2^31 bytes: 2^20 blocks of counts, whose sums begin 2^31 bytes into the
    matrix."""
    print("case order most positions", flush=True)
    lib, n = _capi.lib(), (1 << 29) - 1
    index = torch.arange(n, dtype=torch.int32, device="cuda")
    on = (index * 40503 & 0x300) == 0
    table = torch.where(on, index, torch.tensor(-1, dtype=torch.int32, device="cuda"))
    mask, order, by_position = (torch.empty(n, dtype=torch.int32, device="cuda") for _ in range(3))
    sides = (_capi.OrderSide * 2)()
    sides[0].indices, sides[0].n, sides[0].sorted_mask = table.data_ptr(), n, mask.data_ptr()
    sides[0].argsort, sides[0].by_position, sides[0].by_position_reversed = order.data_ptr(), by_position.data_ptr(), None
    ws = torch.empty(int(lib.cumm_hip_order_pairs_workspace(sides, 1, 1)), dtype=torch.uint8, device="cuda")
    _capi.check(lib.cumm_hip_order_pairs(sides, 1, (ctypes.c_int32 * 3)(1, 1, 1), ws.data_ptr(), ws.numel(), 0))
    _capi.check(lib.cumm_hip_device_synchronize())
    without = n - int(on.sum())
    assert bool((mask[:without] == 0).all()) and bool((mask[without:] == 1).all())
    for begin, end, want in ((0, without, False), (without, n, True)):      # stable: ascending, each of its kind
        rows = order[begin:end]
        assert bool((rows[1:] > rows[:-1]).all()) and int(rows[0]) >= 0 and int(rows[-1]) < n
        assert bool((by_position[begin:end] == (rows if want else -1)).all())


@pytest.mark.parametrize("ksize,n,n2", [((3, 3, 3), 1, 0), ((3, 3, 3), 1023, 0), ((3, 3, 3), 1025, 64), ((4, 4, 2), 5000, 0), ((1, 1, 1), 700, 0),
                                        ((1, 1, 2), 1024, 2049), ((3, 3, 3), 512 * 128 + 1, 0), ((3, 3, 3), 512 * 128 * 4 + 513, 1000),
                                        ((2, 2, 2), 1 << 20, 3), ((2, 2, 2), 3, (1 << 20) + 1), ((2, 2, 2), 1 << 19, 0), ((5, 5, 5), 3000, 0)])
def test_one_pass(ksize, n, n2):
    """cumm_hip_order_pairs_coarse: a permutation that repeats, ascending by number of offsets (without the middle
    one where a reversed table is asked for), stable and exact up to two of them; tables and hints as always.
    Chunks of 1024 positions, runs of 8 and 32 blocks, the last table that takes one pass and the first of two."""
    print("case one pass", ksize, n, n2, flush=True)
    rng, kv, reverse = np.random.default_rng(n + n2), int(np.prod(ksize)), n2 == 0
    tables = [_table(rng, kv, m, 0.08 if kv > 8 else 0.3) for m in (n, n2) if m]
    got, dev = _order(tables, ksize, reverse, "cumm_hip_order_pairs_coarse")
    again, _ = _order(tables, ksize, reverse, "cumm_hip_order_pairs_coarse")
    for t, g, a, d in zip(tables, got, again, dev):
        m = pairs.masks_from_pairs(t)
        order = g["order"]
        assert np.array_equal(np.sort(order), np.arange(t.shape[1])) and np.array_equal(order, a["order"])
        np.testing.assert_array_equal(g["mask"], m[order])
        want = pairs.pairs_by_position(t, order)
        # (written where a run of 128 positions has the offset; elsewhere what was there)
        runs = np.logical_or.reduceat(want >= 0, np.arange(0, t.shape[1], 128), axis=1)
        written = np.repeat(runs, 128, axis=1)[:, :t.shape[1]]
        np.testing.assert_array_equal(g["pos"], np.where(written, want, UNWRITTEN))
        if reverse:
            np.testing.assert_array_equal(g["rev"], g["pos"][::-1])
        if m.shape[1] > 1:
            continue
        word = m[:, 0].astype(np.int64)
        if reverse:
            low = (1 << (kv // 2)) - 1
            word = (word & low) | (word >> (kv // 2 + 1) << (kv // 2))
        count = sum((word >> b) & 1 for b in range(kv))
        assert np.all(np.diff(count[order]) >= 0)
        exact = int((count <= 2).sum())
        np.testing.assert_array_equal(order[:exact], np.lexsort((word, count))[:exact])
        bits, s = (1 << kv) - 1 if kv < 32 else 0xFFFFFFFF, g["mask"][:, 0]
        hints = pairs.hints_device(d["mask"].view([t.shape[1]]), bits)
        if hints != (-1, -1) and (t is tables[-1] or t.shape[1] != tables[-1].shape[1]):
            assert hints[0] == pairs.light_prefix(s, bits, 3)
