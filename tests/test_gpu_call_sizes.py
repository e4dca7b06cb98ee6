"""Kernels whose launch shape follows the call's size, at the sizes where the
shape changes: the offsets scan (one block, tiles), the list gather (passes of
256 rows, entries four at a time), the radix passes' widths, the chunk plan of
few and of many tables, the grouped update's units, and the bag pooling
backward's windows.  Whole numbers bit for bit; sums against float64 with the
bound of fp32 summation (unit roundoff times the terms, about 1e-6 here)."""

import numpy as np
import pytest
import torch

from mdl_amd import _lib, ops
from mdl_amd.features import bag_csr, bag_csr_tensor
from mdl_amd.optim import ShardedRowWiseAdagrad
from mdl_amd.pooling import pool_bags
from mdl_amd.sparse_step import SparseStep

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 8191, 8192, 8193, 16384, 16385, 2048 * 40 + 1])
def test_offsets_scan(device, n):
    print("CASE scan", n, flush=True)
    rng = np.random.default_rng(n)
    ln = rng.integers(0, 1 << 34, size=n)
    got = ops.lengths_to_offsets(torch.from_numpy(ln).to(device)).cpu().numpy()
    assert np.array_equal(got, np.concatenate([[0], np.cumsum(ln)]))


@pytest.mark.parametrize("n", [2, 3, 63, 2047, 2048, 2049, 2050, 4095, 8193 + 511, 24577])
def test_offsets_scan_of_one_block_and_of_tiles(device, n):
    """Lengths two a thread (2048 at most), eight a thread through LDS, and a
    second tile of one that ends inside a wave; the last offset alone when
    the lengths before it are zeros."""

    print("CASE scan places", n, flush=True)
    rng = np.random.default_rng(n)
    for ln in (rng.integers(-5, 1 << 40, size=n), np.eye(1, n, n - 1, dtype=np.int64)[0]):
        got = ops.lengths_to_offsets(torch.from_numpy(ln).to(device)).cpu().numpy()
        assert np.array_equal(got, np.concatenate([[0], np.cumsum(ln)]))


@pytest.mark.parametrize("dim, n", [(64, 9000), (256, 40000), (256, 150000), (256, 500000), (256, 600000)])
def test_distinct_rows_of_many_chunks(device, dim, n):
    """The distinct rows of several tables where their chunks' head counts are
    scanned two a thread, in one tile, in several and by launches of tiles."""

    print("CASE heads", dim, n, flush=True)
    rng = np.random.default_rng(n)
    rows = [1, 70000, 5, 400000]
    tables = np.zeros(len(rows), dtype=_lib.TABLE_DTYPE)
    tables["row_base"] = np.concatenate([[0], np.cumsum(rows)[:-1]])
    tables["num_rows"] = rows
    tables["dim"] = dim
    tables["feature"] = -1
    total = sum(rows)
    keys = rng.integers(0, total + total // 50, size=n)
    keys = np.minimum(keys, total).astype(np.uint32)
    L = _lib.lib()
    tdev = torch.from_numpy(tables.view(np.uint8)).to(device)
    k = torch.from_numpy(keys.view(np.int32).copy()).to(device)
    p = torch.arange(n, dtype=torch.int32, device=device)
    ws = torch.empty(int(L.mdl_backward_workspace_bytes(n, len(rows), dim)), dtype=torch.uint8, device=device)
    urange = torch.full((2 * len(rows),), -1, dtype=torch.int64, device=device)
    _lib.check(L.mdl_backward_count(
        tdev.data_ptr(), len(rows), dim, k.data_ptr(), p.data_ptr(), n, None, total.bit_length(), urange.data_ptr(),
        ws.data_ptr(), ws.numel(), torch.cuda.current_stream(device).cuda_stream), "mdl_backward_count")
    ur = urange.cpu().numpy().reshape(-1, 2)
    uniq = np.unique(keys)
    lo = tables["row_base"]
    below = np.searchsorted(uniq, lo)
    assert np.array_equal(ur[:, 0], below)
    assert np.array_equal(ur[:, 1], np.searchsorted(uniq, lo + tables["num_rows"]))


@pytest.mark.parametrize("rows", [1, 255, 256, 257, 2049])
@pytest.mark.parametrize("longest", [0, 3, 1200])
@pytest.mark.parametrize("truncation", ["head", "tail"])
def test_list_gather(device, rows, longest, truncation):
    print("CASE lists", rows, longest, truncation, flush=True)
    rng = np.random.default_rng(rows + longest)
    lists = [rng.integers(1, 1 << 40, size=rng.integers(0, longest + 1)).tolist() for _ in range(rows)]
    flat = np.array([x for r in lists for x in r], dtype=np.int64)
    offsets = np.concatenate([[0], np.cumsum([len(r) for r in lists])])
    for keep in (None, 2, 700):
        want, _, lengths = bag_csr(lists, max_length=keep, truncation=truncation)
        for exact in (True, False):
            got = bag_csr_tensor(torch.from_numpy(flat).to(device), torch.from_numpy(offsets).to(device),
                                 max_length=keep, truncation=truncation, exact=exact)
            values = got["values"].cpu().numpy()
            assert np.array_equal(values[: len(want)], want)
            assert not values[len(want):].any() and (not exact or len(values) == len(want))
            assert np.array_equal(got["lengths"].cpu().numpy(), lengths)


@pytest.mark.parametrize("bits", [1, 7, 8, 9, 14, 17, 25, 28, 31, 32])
def test_radix_pass_widths(device, bits):
    """mdl_sort_pairs sorts on the low ``bits`` bits, stably, whatever the
    widths its passes take."""

    L = _lib.lib()
    rng = np.random.default_rng(bits)
    for n in (1, 4097, 300001):
        print("CASE radix", bits, n, flush=True)
        keys = rng.integers(0, 1 << 32, size=n, dtype=np.uint32)
        low = keys & np.uint32((1 << bits) - 1)
        k = torch.from_numpy(keys.view(np.int32).copy()).to(device)
        p = torch.arange(n, dtype=torch.int32, device=device)
        ka, pa = torch.empty_like(k), torch.empty_like(p)
        ws = torch.empty(int(L.mdl_sort_workspace_bytes(n)), dtype=torch.uint8, device=device)
        alt = np.zeros(1, dtype=np.int32)
        _lib.check(L.mdl_sort_pairs(k.data_ptr(), p.data_ptr(), ka.data_ptr(), pa.data_ptr(), n, bits, ws.data_ptr(),
                                    ws.numel(), alt.ctypes.data, torch.cuda.current_stream(device).cuda_stream),
                   "mdl_sort_pairs")
        assert int(alt[0]) == ((bits + 7) // 8) % 2
        want = np.argsort(low, kind="stable")
        got_k, got_p = (ka, pa) if alt[0] else (k, p)
        assert np.array_equal(got_p.cpu().numpy(), want)
        assert np.array_equal(got_k.cpu().numpy().view(np.uint32), keys[want])


@pytest.mark.parametrize("tables", [1, 128, 129])
@pytest.mark.parametrize("batch", [8, 700])
def test_step_of_few_and_many_tables(device, tables, batch):
    """One step of single-valued features, a table each: the plan's one launch
    (128 tables at most) and two, in calls of one tile and of several."""

    print("CASE plan", tables, batch, flush=True)
    gen = torch.Generator(device=device).manual_seed(tables + batch)
    rows, dim = 60, 16
    w = torch.randn(tables, rows, dim, device=device, generator=gen)
    acc = torch.rand(tables, rows, device=device, generator=gen)
    ids = torch.randint(0, rows, (tables, batch), device=device, generator=gen)
    grad = torch.randn(batch, tables * dim, device=device, generator=gen)
    w64, acc64 = w.double(), acc.double()
    for t in range(tables):
        live = ids[t] != 0
        g = torch.zeros(rows, dim, dtype=torch.float64, device=device)
        g.index_add_(0, ids[t][live], grad[:, t * dim: (t + 1) * dim].double()[live])
        hit = torch.zeros(rows, dtype=torch.bool, device=device)
        hit[ids[t][live]] = True
        acc64[t] += g.square().mean(1)
        w64[t] -= torch.where(hit[:, None], 0.1 * g / (acc64[t].sqrt() + 1e-8)[:, None], 0.0)
    want = torch.cat([w[t][ids[t]] for t in range(tables)], 1)
    out = torch.empty_like(grad)
    plan = ops.GroupPlan()
    for t in range(tables):
        plan.add_feature(w[t], pooling="none", state=acc[t])
    cols = [slice(t * dim, (t + 1) * dim) for t in range(tables)]
    step = SparseStep(plan, ids.reshape(-1), None, [batch] * tables, [0] * tables, [out[:, c] for c in cols],
                      [grad[:, c] for c in cols])
    step.step(0.1, 1e-8)
    assert torch.equal(out, want)
    torch.testing.assert_close(acc.double(), acc64, rtol=1e-5, atol=1e-6)
    torch.testing.assert_close(w.double(), w64, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("dim", [8, 64, 260, 600])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_update_units(device, dim, dtype):
    """Row counts at the edges of an update unit (256 rows) and of a wave's
    share of it (32), several tables in one launch, an empty one among them."""

    print("CASE update", dim, dtype, flush=True)
    gen = torch.Generator(device=device).manual_seed(dim)
    counts = [1, 31, 32, 33, 0, 255, 256, 257, 1000]
    params, want = [], []
    opt_sums = []
    for n in counts:
        p = torch.nn.Parameter(torch.randn(1500, dim, device=device, generator=gen).to(dtype))
        rows = torch.randperm(1500, device=device, generator=gen)[:n].sort().values
        vals = torch.randn(n, dim, device=device, generator=gen).to(dtype)
        acc = torch.rand(1500, device=device, generator=gen)
        a64, w64 = acc.double(), p.detach().double()
        a64[rows] += vals.double().square().mean(1)
        w64[rows] -= 0.1 * vals.double() / (a64[rows].sqrt() + 1e-8)[:, None]
        p.grad = torch.sparse_coo_tensor(rows[None], vals, (1500, dim), is_coalesced=True)
        params.append(p)
        want.append((w64, a64))
        opt_sums.append(acc)
    opt = ShardedRowWiseAdagrad(params, lr=0.1, eps=1e-8)
    for p, acc in zip(params, opt_sums):
        opt.state[p]["sum"] = acc
    opt.step()
    # fp32: a few roundings; bf16: one rounding of the weight to 8 bits
    tol = {"rtol": 1e-5, "atol": 1e-5} if dtype == torch.float32 else {"rtol": 2.0 ** -8, "atol": 1e-3}
    for p, acc, (w64, a64) in zip(params, opt_sums, want):
        torch.testing.assert_close(acc.double(), a64, rtol=1e-5, atol=1e-6)
        torch.testing.assert_close(p.detach().double(), w64, **tol)


@pytest.mark.parametrize("lengths", [[511, 1, 0, 513], [1024], [0, 0, 3], [2000, 7, 300]])
@pytest.mark.parametrize("dim", [3, 24, 64, 600])
def test_pool_backward_windows(device, lengths, dim):
    """Bags around the backward's 512-position windows: each position's
    gradient is its bag's, divided like the reference, bit for bit."""

    print("CASE pool windows", lengths, dim, flush=True)
    gen = torch.Generator(device=device).manual_seed(dim)
    ln = torch.tensor(lengths, device=device)
    n = int(ln.sum())
    emb = torch.randn(n, dim, device=device, generator=gen).requires_grad_()
    ids = torch.randint(0, 4, (n,), device=device, generator=gen)
    (out,) = pool_bags([(emb, ids, ln, "exclude")])
    g = torch.randn(len(lengths), dim, device=device, generator=gen)
    out.backward(g)
    bag = torch.repeat_interleave(torch.arange(len(lengths), device=device), ln)
    live = (ids != 0).float()
    count = torch.zeros(len(lengths), device=device).index_add_(0, bag, live).clamp(min=1)
    want = (g.cpu() / count.cpu()[:, None])[bag.cpu()] * live.cpu()[:, None]
    assert torch.equal(emb.grad.cpu(), want)
