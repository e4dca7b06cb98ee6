"""The backward's sort of short calls (tiles sorted in LDS, merged by rank)
against numpy's stable sort, bit for bit, and its chunk plan through the
distinct rows it counts.

Sizes sit at the edges of a tile (4096 entries), of one tile (whose plan is
part of the sort's launch) and of the calls sorted by tiles without a hint
(12 tiles) and with one; orders are table by table (as a lookup emits them),
tables backwards, arbitrary, all one key and all sentinels.
"""

import numpy as np
import pytest
import torch

from mdl_amd import _lib

pytestmark = pytest.mark.gpu

TILE = 4096


def _keys(rng, order, n, rows):
    base = np.concatenate([[0], np.cumsum(rows)])
    total = int(base[-1])
    if order == "sentinels":
        return np.full(n, total, dtype=np.uint32), total
    if order == "one key":
        return np.full(n, total // 2, dtype=np.uint32), total
    if order == "any":
        keys = rng.integers(0, total, size=n)
    else:
        table = np.sort(rng.integers(0, len(rows), size=n))
        if order == "backwards":
            table = table[::-1]
        keys = base[table] + (rng.random(n) ** 3 * np.asarray(rows)[table]).astype(np.int64)
    keys[rng.random(n) < 0.05] = total  # ids without a gradient
    return keys.astype(np.uint32), total


@pytest.mark.parametrize("rows", [[300], [5, 100000, 1, 4000], [20000] * 40, [3] * 700])
@pytest.mark.parametrize("order", ["by table", "backwards", "any", "one key", "sentinels"])
def test_tile_sort_matches_stable_sort(device, order, rows):
    rng = np.random.default_rng(len(rows) + len(order))
    T = len(rows)
    tables = np.zeros(T, dtype=_lib.TABLE_DTYPE)
    tables["row_base"] = np.concatenate([[0], np.cumsum(rows)[:-1]])
    tables["num_rows"] = rows
    tables["dim"] = rng.choice([16, 64, 100], size=T)
    tables["feature"] = -1
    tdev = torch.from_numpy(tables.view(np.uint8)).to(device)
    L = _lib.lib()
    stream = torch.cuda.current_stream(device).cuda_stream
    sizes = [1, 63, 65, TILE - 1, TILE, TILE + 1, 3 * TILE + 77, 12 * TILE, 12 * TILE + 1]
    for n in sizes:
        for present, hints in [(n, 1), (max(n - 100, 0), 1), (n // 3, 1), (n, 0)]:
            keys, total = _keys(rng, order, n, rows)
            for key_bits in (int(total).bit_length(), 32):  # odd and even pass counts among them
                print("CASE tile_sort", order, T, n, present, hints, key_bits, flush=True)
                k = torch.from_numpy(keys.view(np.int32).copy()).to(device)
                p = torch.arange(n, dtype=torch.int32, device=device) + 7
                count = torch.tensor([present], dtype=torch.int64, device=device)
                ws = torch.empty(int(L.mdl_backward_workspace_bytes(n, T, 128)), dtype=torch.uint8, device=device)
                urange = torch.full((2 * T,), -1, dtype=torch.int64, device=device)
                _lib.check(L.mdl_backward_count_hinted(
                    tdev.data_ptr(), T, 128, k.data_ptr(), p.data_ptr(), n, count.data_ptr(), key_bits, hints,
                    urange.data_ptr(), ws.data_ptr(), ws.numel(), stream), "mdl_backward_count_hinted")
                if ((key_bits + 7) // 8) % 2:
                    # an odd number of radix passes ends in the workspace's first two arrays
                    pad = (4 * n + 255) // 256 * 256
                    k, p = ws[: 4 * n].view(torch.int32), ws[pad: pad + 4 * n].view(torch.int32)
                got_k = k.cpu().numpy().view(np.uint32)[:present]
                got_p = p.cpu().numpy()[:present]
                want = np.argsort(keys[:present], kind="stable")
                assert np.array_equal(got_k, keys[:present][want])
                assert np.array_equal(got_p, want + 7)
                ur = urange.cpu().numpy().reshape(T, 2)
                uniq = np.unique(keys[:present])
                lo = tables["row_base"]
                distinct = np.searchsorted(uniq, lo + tables["num_rows"]) - np.searchsorted(uniq, lo)
                assert np.array_equal(ur[:, 1] - ur[:, 0], distinct)


@pytest.mark.parametrize("tiles, extra, counted", [
    (100, 0, True), (128, 0, True), (127, 77, True), (100, 5, False), (512, 0, False), (512, 1, False),
    (1024, 0, False), (1024, 1, False),
])
@pytest.mark.parametrize("order", ["by table", "any"])
def test_tile_sort_of_many_tiles(device, order, tiles, extra, counted):
    """Hinted calls up to the bound with a device count (the count at, below
    and far below the capacity), and without one up to 1024 tiles, where the
    radix passes take over: more tiles than a block has threads, and, in no
    order, every tile in a block's list of those that overlap."""

    n, rows = tiles * TILE + extra, [50000] * 63 + [7]
    rng = np.random.default_rng(tiles + extra)
    T = len(rows)
    tables = np.zeros(T, dtype=_lib.TABLE_DTYPE)
    tables["row_base"] = np.concatenate([[0], np.cumsum(rows)[:-1]])
    tables["num_rows"] = rows
    tables["dim"] = 64
    tables["feature"] = -1
    tdev = torch.from_numpy(tables.view(np.uint8)).to(device)
    keys, total = _keys(rng, order, n, rows)
    L = _lib.lib()
    ws = torch.empty(int(L.mdl_backward_workspace_bytes(n, T, 64)), dtype=torch.uint8, device=device)
    for present in ([n, n - TILE - 3, n // 40] if counted else [n]):
        print("CASE many tiles", order, n, present, flush=True)
        k = torch.from_numpy(keys.view(np.int32).copy()).to(device)
        p = torch.arange(n, dtype=torch.int32, device=device)
        count = torch.tensor([present], dtype=torch.int64, device=device)
        urange = torch.full((2 * T,), -1, dtype=torch.int64, device=device)
        _lib.check(L.mdl_backward_count_hinted(
            tdev.data_ptr(), T, 64, k.data_ptr(), p.data_ptr(), n, count.data_ptr() if counted else None, 32, 1,
            urange.data_ptr(), ws.data_ptr(), ws.numel(), torch.cuda.current_stream(device).cuda_stream),
            "mdl_backward_count_hinted")
        want = np.argsort(keys[:present], kind="stable")
        assert np.array_equal(p.cpu().numpy()[:present], want)
        assert np.array_equal(k.cpu().numpy().view(np.uint32)[:present], keys[:present][want])
        uniq = np.unique(keys[:present])
        lo = tables["row_base"]
        ur = urange.cpu().numpy().reshape(T, 2)
        assert np.array_equal(ur[:, 0], np.searchsorted(uniq, lo))
        assert np.array_equal(ur[:, 1], np.searchsorted(uniq, lo + tables["num_rows"]))


def test_sort_hints_follow_the_stretches():
    """One short stretch per table takes the tile sort; one long one, or
    stretches of too many tile pairs together, the radix sort."""

    def hints(counts):
        c = np.asarray(counts, dtype=np.int64)
        return int(_lib.lib().mdl_sort_hints(c.ctypes.data, len(c)))

    assert hints([4096 * 3] * 32) == 1
    assert hints([0, 1, 4096]) == 1
    assert hints([4096 * 9]) == 1
    assert hints([4096 * 9 + 1]) == 0
    assert hints([4096 * 9] * 200) == 0


def test_sort_hints_stop_where_the_radix_sort_is_faster():
    """Tables of several tiles each, many of them: every tile meets the others
    of its table, and the merge's blocks no longer run all at once."""

    def hints(counts):
        c = np.asarray(counts, dtype=np.int64)
        return int(_lib.lib().mdl_sort_hints(c.ctypes.data, len(c)))

    assert hints([TILE * 9] * 28) == 1
    assert hints([TILE * 9] * 56) == 0
    assert hints([TILE * 8] * 100) == 0
    assert hints([TILE * 4] * 200) == 1
    assert hints([TILE] * 1000) == 1


@pytest.mark.parametrize("tiles, counted, merges", [(128, True, True), (129, True, False), (129, False, True)])
def test_hint_of_another_batch_is_followed_up_to_a_bound(device, tiles, counted, merges):
    """A call with a device count was hinted from another batch, whose tables
    this one's ids may not spread over: past 128 tiles it takes the radix
    passes, whose time does not depend on that."""

    n, rows = tiles * TILE - 3, 1 << 20
    print("CASE hint bound", tiles, counted, flush=True)
    tables = np.zeros(64, dtype=_lib.TABLE_DTYPE)
    tables["row_base"] = np.arange(64) * rows
    tables["num_rows"] = rows
    tables["dim"] = 16
    tables["feature"] = -1
    keys = np.random.default_rng(tiles).integers(0, rows, size=n).astype(np.uint32)  # one table's
    tdev = torch.from_numpy(tables.view(np.uint8)).to(device)
    k = torch.from_numpy(keys.view(np.int32).copy()).to(device)
    p = torch.arange(n, dtype=torch.int32, device=device)
    count = torch.tensor([n], dtype=torch.int64, device=device)
    L = _lib.lib()
    ws = torch.empty(int(L.mdl_backward_workspace_bytes(n, 64, 16)), dtype=torch.uint8, device=device)
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        _lib.check(L.mdl_backward_sort_hinted(
            tdev.data_ptr(), 64, 16, k.data_ptr(), p.data_ptr(), n, count.data_ptr() if counted else None, 32, 1,
            ws.data_ptr(), ws.numel(), torch.cuda.current_stream(device).cuda_stream), "mdl_backward_sort_hinted")
        torch.cuda.synchronize()
    names = " ".join(e.key for e in prof.key_averages())
    assert ("rank_merge_kernel" in names) == merges
    assert ("radix_downsweep" in names) != merges
    want = np.argsort(keys, kind="stable")
    assert np.array_equal(p.cpu().numpy(), want)
    assert np.array_equal(k.cpu().numpy().view(np.uint32), keys[want])
