"""Parity of the HIP library against the CPU oracle on seeded inputs.  Every
test goes through libzen_hip.so's C ABI (directly or via the package's thin
wrappers).  Bar: bit-exact for indices, slots, order and bit-copied values;
merged sums bit-exact against the fp32 sequential oracle (same order of adds)
and within 1e-6 relative of the fp64 truth."""
import ctypes

import numpy as np
import pytest
import torch

from gpu_util import make_grad, to_dev, to_np

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def zen():
    import zen_repro_amd
    from zen_repro_amd import _lib

    _lib.lib()
    assert torch.cuda.is_available()
    return zen_repro_amd


# ------------------------------------------------------------------ sort


@pytest.mark.parametrize("count", [1, 63, 64, 65, 1000, 4095, 4096, 4097, 70001, 1 << 20])
@pytest.mark.parametrize("bits", [1, 8, 9, 17, 30, 32])
def test_sort_pairs_is_stable_sort(zen, count, bits):
    from zen_repro_amd import _lib

    rng = np.random.default_rng(count * 131 + bits)
    hi = (1 << bits) - 1
    # few distinct keys on purpose: stability must show
    keys = rng.integers(0, min(hi, 500) + 1, count, dtype=np.uint64).astype(np.uint32)
    if bits >= 9:
        keys = (keys * np.uint32(max(1, hi // 501))).astype(np.uint32)
    vals = np.arange(count, dtype=np.uint32)
    dk = to_dev(keys.view(np.int32))
    dv = to_dev(vals.view(np.int32))
    L = _lib.lib()
    ws = torch.empty(L.zen_sort_pairs_workspace(count), dtype=torch.uint8, device="cuda")
    st = torch.zeros(1, dtype=torch.int32, device="cuda")
    rc = L.zen_sort_pairs(_lib.ptr(dk), _lib.ptr(dv), count, None, bits, _lib.ptr(ws), ws.numel(),
                          _lib.ptr(st), _lib.stream_of(dk.device))
    assert rc == 0 and st.item() == 0
    order = np.argsort(keys, kind="stable")
    assert np.array_equal(to_np(dk).view(np.uint32), keys[order])
    assert np.array_equal(to_np(dv).view(np.uint32), vals[order])


def test_sort_pairs_device_count(zen):
    from zen_repro_amd import _lib

    cap, live = 50000, 12345
    rng = np.random.default_rng(9)
    keys = rng.integers(0, 1 << 20, cap, dtype=np.uint64).astype(np.uint32)
    vals = np.arange(cap, dtype=np.uint32)
    dk, dv = to_dev(keys.view(np.int32)), to_dev(vals.view(np.int32))
    cnt = torch.tensor([live], dtype=torch.int32, device="cuda")
    L = _lib.lib()
    ws = torch.empty(L.zen_sort_pairs_workspace(cap), dtype=torch.uint8, device="cuda")
    st = torch.zeros(1, dtype=torch.int32, device="cuda")
    assert L.zen_sort_pairs(_lib.ptr(dk), _lib.ptr(dv), cap, _lib.ptr(cnt), 20, _lib.ptr(ws), ws.numel(),
                            _lib.ptr(st), _lib.stream_of(dk.device)) == 0
    order = np.argsort(keys[:live], kind="stable")
    assert np.array_equal(to_np(dk).view(np.uint32)[:live], keys[:live][order])
    assert np.array_equal(to_np(dv).view(np.uint32)[:live], vals[:live][order])
    assert np.array_equal(to_np(dk).view(np.uint32)[live:], keys[live:])  # tail untouched


@pytest.mark.parametrize("count,sentinel,live,distinct", [
    (1 << 16, 1 << 20, None, None), (70001, 743440384, None, None), (1 << 20, (1 << 30) + 7, None, None),
    (3800000, 743440384, None, None), (1 << 20, 5000011, 300000, None), (1 << 18, 1 << 24, None, 700),
])
def test_bucket_sort_pairs_is_stable_sort(zen, count, sentinel, live, distinct):
    """Evenly spread keys below the sentinel, some at or above it; duplicates keep their arrival order."""
    from zen_repro_amd import _lib

    rng = np.random.default_rng(count + sentinel % 1000)
    keys = rng.integers(0, sentinel, count, dtype=np.uint64).astype(np.uint32)
    if distinct:  # many equal keys
        keys = (keys // np.uint32(sentinel // distinct) * np.uint32(sentinel // distinct)).astype(np.uint32)
    tail = rng.random(count) < 0.05
    keys[tail] = sentinel + (rng.integers(0, 2, int(tail.sum())).astype(np.uint32))
    vals = np.arange(count, dtype=np.uint32)
    dk, dv = to_dev(keys.view(np.int32)), to_dev(vals.view(np.int32))
    n = count if live is None else live
    cnt = None if live is None else torch.tensor([live], dtype=torch.int32, device="cuda")
    L = _lib.lib()
    assert L.zen_bucket_sort_fits(count, sentinel)
    ws = torch.empty(L.zen_sort_pairs_workspace(count), dtype=torch.uint8, device="cuda")
    st = torch.zeros(1, dtype=torch.int32, device="cuda")
    rc = L.zen_bucket_sort_pairs(_lib.ptr(dk), _lib.ptr(dv), count, _lib.ptr(cnt), sentinel, _lib.ptr(ws),
                                 ws.numel(), _lib.ptr(st), _lib.stream_of(dk.device))
    assert rc == 0 and st.item() == 0
    below = np.flatnonzero(keys[:n] < sentinel)
    order = below[np.argsort(keys[below], kind="stable")]
    got_k, got_v = to_np(dk).view(np.uint32), to_np(dv).view(np.uint32)
    assert np.array_equal(got_k[:len(order)], keys[order])
    assert np.array_equal(got_v[:len(order)], vals[order])
    rest = np.flatnonzero(keys[:n] >= sentinel)  # behind, as a set, each still with its own value
    assert np.array_equal(np.sort(got_v[len(order):n]), rest)
    assert np.array_equal(got_k[len(order):n], keys[got_v[len(order):n]])
    assert np.array_equal(got_k[n:], keys[n:])


def test_bucket_sort_pairs_crowded_range_asks_for_retry(zen):
    from zen_repro_amd import _lib

    count, sentinel = 1 << 17, 1 << 24
    keys = np.random.default_rng(5).integers(0, 20000, count, dtype=np.uint64).astype(np.uint32)  # one key range
    dk, dv = to_dev(keys.view(np.int32)), to_dev(np.arange(count, dtype=np.int32))
    L = _lib.lib()
    ws = torch.empty(L.zen_sort_pairs_workspace(count), dtype=torch.uint8, device="cuda")
    st = torch.zeros(1, dtype=torch.int32, device="cuda")
    assert L.zen_bucket_sort_pairs(_lib.ptr(dk), _lib.ptr(dv), count, None, sentinel, _lib.ptr(ws), ws.numel(),
                                   _lib.ptr(st), _lib.stream_of(dk.device)) == 0
    assert st.item() == _lib.STAT_RETRY
    assert not L.zen_bucket_sort_fits(1000, sentinel) and not L.zen_bucket_sort_fits(count, 1000)
    assert L.zen_bucket_sort_pairs(_lib.ptr(dk), _lib.ptr(dv), 1000, None, sentinel, _lib.ptr(ws), ws.numel(),
                                   _lib.ptr(st), _lib.stream_of(dk.device)) == _lib.EINVAL


# ------------------------------------------------------------------ hash


@pytest.mark.parametrize("n,P", [(1 << 20, 4), (1003, 4), (38597376 // 16, 16), (999983, 7), (64, 64)])
def test_hash_index(zen, oracle, n, P):
    idx = torch.full((n,), -7, dtype=torch.int32, device="cuda")
    zen.hash_index(idx, P)
    assert np.array_equal(to_np(idx), oracle.hash_index(n, P))


def test_hash_index_rejects(zen):
    with pytest.raises(ValueError):
        zen.hash_index(torch.zeros(3, dtype=torch.int32, device="cuda"), 4)
    with pytest.raises(AssertionError):
        zen.hash_index(torch.zeros(8, dtype=torch.int64, device="cuda"), 4)


@pytest.mark.parametrize("n,P", [(1 << 16, 8), (1003, 4), (300000, 16)])
def test_calculate_mapping(zen, oracle, n, P):
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(P), None, None)
    got = lba.calculate_mapping(n)
    want = oracle.mapping(n, P)
    assert len(got) == P
    for g, w in zip(got, want):
        assert g.dtype == torch.int64 and np.array_equal(to_np(g), w)


# ---------------------------------------------------------------- insert

INSERT_CASES = [
    (4096, 4, 0.01, 1), (4096, 4, 0.3, 1), (1 << 16, 16, 0.05, 1), (1 << 16, 8, 0.5, 1),
    (100000, 5, 0.2, 1), (1 << 18, 32, 0.01, 1), (60000, 6, 0.35, 2), (50000, 4, 0.25, 1.5),
    (1000000, 4, 0.4, 1),  # rehash 1: > 8192 serial entries per partition (sorted in global memory)
]


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("rehash", [1, 2, 3])
@pytest.mark.parametrize("n,P,density,scale", INSERT_CASES)
def test_sparse_balance_tables_byte_identical(zen, oracle, n, P, density, scale, rehash, dtype):
    g = make_grad(oracle, n, density, dtype, seed=n + P)
    g[0] = g[g != 0][0] if (g != 0).any() else 1  # index 0 nonzero: must never be stored
    m, sn = oracle.table_sizes(n, P, scale)
    mem_o, ser_o, off_o, st_o = oracle.sparse_balance(g, m, sn, P, rehash)
    d = to_dev(g)
    mem = torch.zeros(m, dtype=torch.int32, device="cuda")
    ser = torch.zeros(sn, dtype=torch.int32, device="cuda")
    assert zen.sparse_balance(d, mem, ser, P, rehash) is None  # like the reference's
    pending = zen.last_status()
    assert np.array_equal(to_np(pending.offsets), off_o)
    assert int(pending.status.item()) == st_o
    assert np.array_equal(to_np(mem), mem_o)
    if st_o == 0:
        assert np.array_equal(to_np(ser), ser_o)


@pytest.mark.parametrize("n,P,entries", [
    (1 << 18, 1, 2), (1 << 18, 1, 8193),  # one turn of the region's sort: the smallest, many
    (1 << 20, 1, 16384), (1 << 20, 1, 16385), (1 << 20, 1, 64512), (1 << 20, 1, 64513),  # one turn, two, as many as fit, one more
    (1 << 22, 2, 40000),    # piled up at the end of the tensor
    (60000, 1025, 600),     # more partitions than a workgroup collects for
])
def test_serial_regions_at_the_edges_of_their_sort(zen, oracle, n, P, entries):
    """One level only, and `entries` indices more than there are slots taken: pairs of indices that share a slot."""
    m, sn = oracle.table_sizes(n, P)
    t = np.arange(n, dtype=np.uint32)
    slot = (((np.uint32(573729859) * t + np.uint32(0xCC9E2D51)) * t + np.uint32(0x1B873593)) * t + np.uint32(10001861)) % np.uint32(m)
    order = np.argsort(slot, kind="stable")[1:]
    order = order[order != 0]
    twin = order[1:][slot[order[1:]] == slot[order[:-1]]]  # every one loses its slot to the one in front of it
    if n == 1 << 22:
        twin = np.sort(twin)[-entries:]
    chosen = np.random.default_rng(entries).permutation(twin)[:entries]
    assert len(chosen) >= min(entries, 2)
    g = np.zeros(n, np.float32)
    g[chosen] = 1.0
    place = np.empty(n, np.int64)
    place[order] = np.arange(len(order))
    g[order[place[chosen] - 1]] = 1.0
    mem_o, ser_o, off_o, st_o = oracle.sparse_balance(g, m, sn, P, 1)
    mem = torch.zeros(m, dtype=torch.int32, device="cuda")
    ser = torch.zeros(sn, dtype=torch.int32, device="cuda")
    zen.sparse_balance(to_dev(g), mem, ser, P, 1)
    assert int(zen.last_status().status.item()) == st_o and np.array_equal(to_np(zen.last_status().offsets), off_o)
    assert np.array_equal(to_np(mem), mem_o)
    if st_o == 0:
        assert np.array_equal(to_np(ser), ser_o)


def test_sparse_balance_overflow_is_flagged_not_oob(zen, oracle):
    n, P = 40000, 4
    g = np.ones(n, np.float32)
    m, sn = oracle.table_sizes(n, P)
    mem_o, _, off_o, st_o = oracle.sparse_balance(g, m, sn, P, 1)
    assert st_o == oracle.SERIAL_OVERFLOW
    mem = torch.zeros(m, dtype=torch.int32, device="cuda")
    ser = torch.zeros(sn + 64, dtype=torch.int32, device="cuda")  # guard zone behind the table
    assert zen.sparse_balance(to_dev(g), mem, ser[:sn], P, 1) is None  # like the reference's
    pending = zen.last_status()
    assert int(pending.status.item()) & 1
    with pytest.raises(RuntimeError):
        pending.check()
    assert np.array_equal(to_np(mem), mem_o)
    assert np.array_equal(to_np(pending.offsets), off_o)
    assert not to_np(ser)[sn:].any()


def test_sparse_balance_argument_errors(zen):
    g = torch.zeros(64, dtype=torch.bfloat16, device="cuda")
    mem = torch.zeros(64, dtype=torch.int32, device="cuda")
    ser = torch.zeros(4, dtype=torch.int32, device="cuda")
    with pytest.raises(AssertionError):
        zen.sparse_balance(g.cpu(), mem, ser, 4, 3)
    with pytest.raises(AssertionError):
        zen.sparse_balance(g.half(), mem, ser, 4, 3)
    with pytest.raises(AssertionError):
        zen.sparse_balance(g, mem.long(), ser, 4, 3)
    with pytest.raises(RuntimeError):
        zen.sparse_balance(g[::2], mem, ser, 4, 3)
    with pytest.raises(ValueError):
        zen.sparse_balance(g, mem[:62], ser, 4, 3)  # table not a multiple of P


def test_reference_style_compaction_over_tables(zen, oracle):
    # balance_sparse_tensor + get_sub_sparse_tensors, the reference's two-step route
    n, P = 100000, 5
    g = make_grad(oracle, n, 0.2, "bf16", seed=77)
    tp = zen.TensorPartition(P, 1, 3)
    d = to_dev(g)
    mem, ser = tp.balance_sparse_tensor(d)
    i1, v1, s1 = tp.get_sub_sparse_tensors(d, mem)
    i2, v2, s2 = tp.get_sub_sparse_tensors(d, ser)
    idx_o, val_o, splits_o, st = oracle.load_balance(g, P, 1, 3)
    assert st == 0 and s2.sum().item() > 0  # the serial region is in use at this density
    got_i = np.concatenate([np.concatenate([to_np(a), to_np(b)]) for a, b in zip(i1, i2)])
    got_v = np.concatenate([np.concatenate([to_np(a), to_np(b)]) for a, b in zip(v1, v2)])
    assert np.array_equal(got_i, idx_o) and np.array_equal(got_v, val_o)
    assert np.array_equal(to_np(s1 + s2), splits_o)


@pytest.mark.parametrize("m, parts, shift, density", [
    (1, 1, 0, 1.0), (7, 3, 1, 0.6), (1023, 1, 3, 0.2), (1025, 2, 2, 0.2), (4099, 4, 1, 0.0), (70001, 70000, 0, 0.5),
    (100003, 16, 3, 1.0), (9000, 9000, 0, 0.3), ((1 << 23) + 5, 3, 1, 0.05)])
@pytest.mark.parametrize("dtype", ["bf16", "f32"])
def test_table_lists(zen, oracle, m, parts, shift, density, dtype):
    # partition edges off every vector boundary, stretches of one partition and many, full and empty tables, entries
    # that count from the end, slots behind the last whole partition
    n = 50000
    rng = np.random.default_rng(m + parts)
    table = rng.integers(-n, n, m, dtype=np.int32)
    table[rng.random(m) >= density] = 0
    g = make_grad(oracle, n, 1.0, dtype, seed=m)
    room = torch.zeros(m + shift, dtype=torch.int32, device="cuda")
    room[shift:] = to_dev(table)
    d = to_dev(g)
    tp = zen.TensorPartition(parts, 1, 3)
    assert tp._plain_table(d, room[shift:])
    idx, val, splits = tp.get_sub_sparse_tensors(d, room[shift:])
    cut = table[:m // parts * parts].reshape(parts, -1)
    sizes = (cut != 0).sum(1)
    want = cut[cut != 0]
    assert len(idx) == len(val) == parts and np.array_equal(to_np(splits), sizes)
    assert [t.numel() for t in idx] == sizes.tolist() == [t.numel() for t in val]
    assert np.array_equal(to_np(torch.cat(idx)), want) and np.array_equal(to_np(torch.cat(val)), g[want])


@pytest.mark.parametrize("m, parts", [(1, 1), (5000, 1), (1 << 24, 1), ((1 << 23) + 4, 5), (16400, 1024), (16400, 1025)])
def test_table_lists_by_either_entry(zen, m, parts):
    # the walk that adds up the partitions' sizes itself (one to 64 groups of workgroups a partition, partitions of a
    # single one) and the one with a workgroup behind it for that; the gather that follows either
    from zen_repro_amd import _lib
    gen = torch.Generator(device="cuda").manual_seed(m + parts)
    n = 100000
    table = torch.randint(1, n, (m,), generator=gen, device="cuda", dtype=torch.int32)
    table *= torch.rand(m, generator=gen, device="cuda") < 0.05
    grad = torch.randn(n, generator=gen, device="cuda")
    cut = table[:m // parts * parts]
    want, sizes = cut[cut != 0], (cut.view(parts, -1) != 0).sum(1)
    idx, val, splits = zen.TensorPartition(parts, 1, 3).get_sub_sparse_tensors(grad, table)
    assert torch.equal(splits, sizes) and [t.numel() for t in idx] == sizes.tolist()
    assert torch.equal(torch.cat(idx), want) and torch.equal(torch.cat(val), grad[want.long()])
    L, dev = _lib.lib(), table.device
    ws = torch.empty(L.zen_table_lists_workspace(m, parts), dtype=torch.uint8, device=dev)
    splits, status = torch.full((parts,), -1, device=dev), torch.zeros(1, dtype=torch.int32, device=dev)
    assert L.zen_table_find(_lib.ptr(table), m, parts, n, _lib.ptr(splits), _lib.ptr(ws), ws.numel(), _lib.ptr(status),
                            _lib.stream_of(dev)) == 0
    total = int(sizes.sum())
    out_idx, out_val = torch.empty_like(want), torch.empty(total, device=dev)
    assert L.zen_table_gather(_lib.ptr(table), m, parts, _lib.ptr(grad), 0, n, _lib.ptr(out_idx), _lib.ptr(out_val), total,
                              _lib.ptr(ws), ws.numel(), _lib.stream_of(dev)) == 0
    assert torch.equal(splits, sizes) and torch.equal(out_idx, want) and torch.equal(out_val, grad[want.long()])
    words = _lib.host_words(parts + 1)
    rc = L.zen_table_find_sizes(_lib.ptr(table), m, parts, n, _lib.ptr(splits), None, _lib.ptr(ws), ws.numel(),
                                _lib.ptr(status), words.ptr, words.words, _lib.stream_of(dev))
    assert rc == -1  # the zeroed words are missing


def test_table_lists_what_torch_indexes(zen):
    # an entry past the tensor is an error; autograd, other types and strided tensors are indexed by torch
    g = torch.arange(100, dtype=torch.float32, device="cuda") + 1
    mem = torch.tensor([0, 3, 0, -1, 99, 0], dtype=torch.int32, device="cuda")
    tp = zen.TensorPartition(2, 1, 3)
    with pytest.raises(IndexError):
        tp.get_sub_sparse_tensors(g[:99], mem)
    wide = g.repeat_interleave(2)[::2]
    leaf = g.clone().requires_grad_()
    for t in (wide, g.half(), leaf):
        assert not tp._plain_table(t, mem)
        idx, val, splits = tp.get_sub_sparse_tensors(t, mem)
        assert torch.cat(idx).tolist() == [3, -1, 99] and torch.cat(val).tolist() == [4, 100, 100]
        assert splits.tolist() == [1, 2]
    torch.cat(val).sum().backward()
    assert leaf.grad[99].item() == 2 and leaf.grad[3].item() == 1


# ---------------------------------------------------------------- select


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("n", [5000, 1 << 16, 1 << 20, 3 * (1 << 20) + 17])
def test_topk_threshold(zen, oracle, n, dtype):
    g = make_grad(oracle, n, 1.0, dtype, seed=n)
    d = to_dev(g)
    for k in (1, 2, n // 200, n // 100, n // 3, n):
        thr = zen.topk_threshold(d, k)
        key, count = (int(x) & 0xFFFFFFFF for x in to_np(thr))
        assert key == oracle.kth_key(g, k), (n, dtype, k)
        keys = (g & 0x7FFF) if dtype == "bf16" else (g.view(np.uint32) & 0x7FFFFFFF)
        assert count == int((keys >= key).sum())


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("n,s", [(5000, 50), (1 << 20, 10486), (3 * (1 << 20) + 17, 1 << 20), (1 << 16, 1 << 18)])
def test_sample_threshold(zen, oracle, n, s, dtype):
    """The threshold over tensor[sample_index] (train.py:78-82) in one call: positions drawn with replacement
    (more positions than elements in the last case), against the k-th largest key of the gathered sample."""
    import importlib

    C = importlib.import_module("zen_repro_amd.compress")
    from zen_repro_amd import _lib

    g = make_grad(oracle, n, 1.0, dtype, seed=n + s)
    d = to_dev(g)
    rng = np.random.default_rng(s)
    at = rng.integers(0, n, s)
    at[0], at[-1] = 0, n - 1
    at_dev = torch.from_numpy(at).cuda()
    keys = (g & 0x7FFF) if dtype == "bf16" else (g.view(np.uint32) & 0x7FFFFFFF)
    for k in (1, max(1, s // 100), s // 2 + 1, s):
        thr, status = C.sample_threshold(d, at_dev, k)
        key, count = (int(x) & 0xFFFFFFFF for x in to_np(thr))
        assert int(status) == 0
        assert key == oracle.kth_key(g[at], k), (n, s, dtype, k)
        assert count == int((keys[at] >= key).sum())
    # an unaligned view of the tensor, and a position outside it: flagged, counted as a zero
    thr, status = C.sample_threshold(d[1:], at_dev[: s // 2].clamp(max=n - 2), max(1, s // 200))
    assert int(status) == 0
    assert int(to_np(thr)[0]) & 0xFFFFFFFF == oracle.kth_key(g[1:][np.minimum(at[: s // 2], n - 2)], max(1, s // 200))
    bad = at.copy()
    bad[s // 3] = n
    bad[s // 2] = -1
    thr, status = C.sample_threshold(d, torch.from_numpy(bad).cuda(), max(1, s // 100))
    assert int(status) == _lib.STAT_BAD_INDEX
    sample = g[np.clip(bad, 0, n - 1)].copy()
    sample[[s // 3, s // 2]] = 0
    assert int(to_np(thr)[0]) & 0xFFFFFFFF == oracle.kth_key(sample, max(1, s // 100))


def test_topk_threshold_heavy_ties_and_zeros(zen, oracle):
    n = 1 << 18
    g = np.zeros(n, np.float32)
    g[::7] = 0.5
    g[::11] = -0.5
    g[5::13] = 2.0
    d = to_dev(g)
    for k in (1, 1000, int((g != 0).sum()), n):
        thr = zen.topk_threshold(d, k)
        assert int(to_np(thr)[0]) == oracle.kth_key(g, k)


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
def test_compress_masked_copy(zen, oracle, dtype):
    import importlib

    C = importlib.import_module("zen_repro_amd.compress")

    n = (1 << 18) + 5
    g = make_grad(oracle, n, 1.0, dtype, seed=5)
    d = to_dev(g)
    k = n // 100
    thr = C.topk_threshold(d, k)
    want, kept = oracle.mask_dense(g, oracle.kth_key(g, k))
    assert np.array_equal(to_np(C.mask_below(d, thr)), want)
    # unaligned views take the scalar path
    got = C.mask_below(d[1:], C.topk_threshold(d[1:], k))
    want1, _ = oracle.mask_dense(g[1:], oracle.kth_key(g[1:], k))
    assert np.array_equal(to_np(got), want1)
    # the reference-shaped entry: caller-supplied sample positions
    rng = np.random.default_rng(1)
    sample = rng.integers(0, n, -(-n // 100))
    out = zen.compress(5, d, torch.from_numpy(sample).cuda())
    ks = len(sample) * 5 // 100
    want2, _ = oracle.mask_dense(g, oracle.kth_key(g[sample], ks))
    assert np.array_equal(to_np(out), want2)
    small = d[:4096]
    assert zen.compress(1, small) is small  # train.py:77-78
    # threshold over the samples of several ranks (train.py:56-73); the exchange is the caller's
    others = [make_grad(oracle, n, 1.0, dtype, seed=6 + r) for r in range(3)]
    everyone = np.concatenate([g[sample]] + [o[sample] for o in others])
    gather = lambda mine: torch.cat([mine] + [to_dev(o)[torch.from_numpy(sample).cuda()] for o in others])  # noqa: E731
    out = zen.compress_with_allgather(5, d, zen.LocalGroup(4), torch.from_numpy(sample).cuda(), gather)
    want3, _ = oracle.mask_dense(g, oracle.kth_key(everyone, len(everyone) * 5 // 100))
    assert np.array_equal(to_np(out), want3)
    assert np.array_equal(to_np(zen.compress_with_allgather(5, d, zen.LocalGroup(1), torch.from_numpy(sample).cuda())),
                          want2)
    with pytest.raises(RuntimeError):
        zen.compress_with_allgather(5, d, zen.LocalGroup(4))


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("n,density", [(1, 1.0), (100, 0.5), (8192, 0.0), (8193, 1.0), (1 << 20, 0.01),
                                       (5 * (1 << 20) + 3, 0.3), (40 * 1000 * 1000 + 3, 0.5),
                                       (70 * 1000 * 1000, 0.004)])
def test_encode_sparse_tensor(zen, oracle, n, density, dtype):
    g = make_grad(oracle, n, density, dtype, seed=n * 3 + 1)
    if n > 4:
        g[3] = 0x8000 if dtype == "bf16" else -0.0  # negative zero is a zero
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(4), None, None)
    idx, val = lba.encode_sparse_tensor(to_dev(g))
    idx_o, val_o = oracle.encode(g)
    assert idx.dtype == torch.int64
    assert np.array_equal(to_np(idx), idx_o) and np.array_equal(to_np(val), val_o)
    if n > 64:
        off = to_dev(g)[3:]
        i2, v2 = lba.encode_sparse_tensor(off)
        io, vo = oracle.encode(g[3:])
        assert np.array_equal(to_np(i2), io) and np.array_equal(to_np(v2), vo)


def test_select_capacity_flag(zen, oracle):
    from zen_repro_amd import _lib

    n = 100000
    g = make_grad(oracle, n, 0.5, "f32", seed=2)
    d = to_dev(g)
    L = _lib.lib()
    cap = 1000
    oi = torch.full((cap + 16,), -1, dtype=torch.int32, device="cuda")
    ov = torch.zeros(cap + 16, dtype=torch.float32, device="cuda")
    cnt = torch.zeros(1, dtype=torch.int64, device="cuda")
    st = torch.zeros(1, dtype=torch.int32, device="cuda")
    ws = torch.empty(L.zen_select_workspace(n, 0), dtype=torch.uint8, device="cuda")
    assert L.zen_select(_lib.ptr(d), 0, n, None, _lib.ptr(oi), 0, _lib.ptr(ov), cap, _lib.ptr(cnt),
                        _lib.ptr(ws), ws.numel(), _lib.ptr(st), _lib.stream_of(d.device)) == 0
    io, _ = oracle.encode(g)
    assert cnt.item() == len(io) and st.item() == _lib.STAT_CAPACITY
    assert np.array_equal(to_np(oi)[:cap], io[:cap].astype(np.int32))
    assert (to_np(oi)[cap:] == -1).all()


# ---------------------------------------------------------- load balance

LB_CASES = [
    (8192, 4, 0.01, 1, 3), (1 << 16, 16, 0.005, 1, 3), (1 << 16, 8, 0.3, 1, 3), (1 << 18, 32, 0.05, 1, 2),
    (100000, 5, 0.4, 1, 1), (1 << 20, 16, 0.01, 1, 3), (60000, 6, 0.2, 2, 3), (50000, 4, 0.25, 1.5, 3),
    (1 << 20, 64, 0.001, 1, 3),
]


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("n,P,density,scale,rehash", LB_CASES)
def test_load_balance_bit_exact(zen, oracle, n, P, density, scale, rehash, dtype, mode):
    """mode 0: sort-based owner resolution; mode 1: owner table like the reference."""
    g = make_grad(oracle, n, density, dtype, seed=n ^ P)
    g[0] = 0x3F80 if dtype == "bf16" else 1.0
    idx_o, val_o, splits_o, st_o = oracle.load_balance(g, P, scale, rehash)
    tp = zen.TensorPartition(P, scale, rehash)
    d = to_dev(g)
    for rep in range(2):  # the second call reuses the (re-zeroed) owner table
        if st_o:
            with pytest.raises(RuntimeError):
                tp.load_balance(d, mode=mode)
            continue
        indices, values, splits = tp.load_balance(d, mode=mode)
        assert np.array_equal(to_np(splits), splits_o)
        assert np.array_equal(np.concatenate([to_np(i) for i in indices]), idx_o)
        assert np.array_equal(np.concatenate([to_np(v) for v in values]), val_o)
        assert indices[0].dtype == torch.int32 and values[0].dtype == d.dtype
    m, _ = oracle.table_sizes(n, P, scale)
    assert not tp._table(d.device, m).any()  # left empty for the next call


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
def test_topk_then_load_balance(zen, oracle, dtype):
    n, P = 1 << 20, 16
    g = make_grad(oracle, n, 1.0, dtype, seed=123)
    k = n // 200
    key = oracle.kth_key(g, k)
    masked, kept = oracle.mask_dense(g, key)
    idx_o, val_o, splits_o, st_o = oracle.load_balance(masked, P, 1, 3)
    d = to_dev(g)
    thr = zen.topk_threshold(d, k)
    tp = zen.TensorPartition(P, 1, 3)
    indices, values, splits = tp.load_balance(d, thr=thr, capacity=2 * k + 1024)
    assert st_o == 0
    assert np.array_equal(to_np(splits), splits_o)
    assert np.array_equal(np.concatenate([to_np(i) for i in indices]), idx_o)
    assert np.array_equal(np.concatenate([to_np(v) for v in values]), val_o)
    part = oracle.hash_index(n, P)
    for p, i in enumerate(indices):
        assert (part[to_np(i)] == p).all()


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("dtype,shape", [("bf16", "flat"), ("f32", "flat"), ("bf16", "columns")])
def test_load_balance_fused_topk(zen, oracle, dtype, shape, mode):
    """k-largest selection inside the call: the one-pass sampled route (mode 0,
    tensors of 2^24 elements and more) and the exact full-histogram route must
    both equal oracle top-k followed by oracle load balance."""
    from zen_repro_amd import _lib

    n, P = (1 << 25) + 4096, 16
    rng = np.random.default_rng(11)
    x = (rng.standard_normal(n) * 1e-3).astype(np.float32)
    if shape == "columns":  # a few hot columns of a 4096-wide matrix: a stride-aligned sample would be fooled
        x.reshape(-1, 4096)[:, ::509] *= 50.0
    g = oracle.f32_to_bf16_bits(x) if dtype == "bf16" else x
    k = n // 200
    key = oracle.kth_key(g, k)
    masked, kept = oracle.mask_dense(g, key)
    idx_o, val_o, splits_o, st_o = oracle.load_balance(masked, P, 1, 3)
    assert st_o == 0
    tp = zen.TensorPartition(P, 1, 3)
    d = to_dev(g)
    thr_out = torch.zeros(2, dtype=torch.int32, device="cuda")
    oi, ov, splits, status = tp.load_balance_flat(d, capacity=int(1.3 * k) + 4096, k=k, mode=mode, thr_out=thr_out)
    assert status.item() == 0
    assert to_np(thr_out).tolist() == [key, kept]
    assert np.array_equal(to_np(splits), splits_o)
    total = int(splits_o.sum())
    assert np.array_equal(to_np(oi)[:total], idx_o)
    assert np.array_equal(to_np(ov)[:total], val_o)
    if mode == 0:  # the reference-shaped call picks the mode by itself
        indices, values, _ = tp.load_balance(d, capacity=int(1.3 * k) + 4096, k=k)
        assert np.array_equal(np.concatenate([to_np(i) for i in indices]), idx_o)


def test_load_balance_sampled_floor_too_high_asks_for_retry(zen, oracle):
    """k larger than the number of nonzeros the floor lets through cannot
    happen with a fair sample; force it with a tensor whose large values all
    hide from the 1-in-256 sample's expectation: nearly all zeros."""
    from zen_repro_amd import _lib

    n, P = 1 << 25, 8
    g = np.zeros(n, np.float32)
    rng = np.random.default_rng(5)
    hot = rng.choice(n, 3000, replace=False)
    g[hot] = rng.standard_normal(3000).astype(np.float32)
    k = 2000
    tp = zen.TensorPartition(P, 1, 3)
    d = to_dev(g)
    indices, values, splits = tp.load_balance(d, capacity=8192, k=k)  # retries in general mode if it must
    key = oracle.kth_key(g, k)
    masked, _ = oracle.mask_dense(g, key)
    idx_o, val_o, splits_o, _ = oracle.load_balance(masked, P, 1, 3)
    assert np.array_equal(to_np(splits), splits_o)
    assert np.array_equal(np.concatenate([to_np(i) for i in indices]), idx_o)


def test_load_balance_capacity_flag(zen, oracle):
    n, P = 1 << 16, 4
    g = make_grad(oracle, n, 0.5, "f32", seed=4)
    tp = zen.TensorPartition(P, 1, 3)
    with pytest.raises(RuntimeError, match="capacity"):
        tp.load_balance(to_dev(g), capacity=100)


# ----------------------------------------------------------------- merge


def make_payloads(oracle, rng, n, peers, per_peer, overlap, dtype):
    pool = rng.choice(n, max(1, int(per_peer * overlap)), replace=False)
    idx, val = [], []
    for _ in range(peers):
        shared = rng.choice(pool, int(per_peer * overlap), replace=False) if overlap > 0 else np.empty(0, np.int64)
        own = rng.integers(0, n, per_peer - len(shared))
        i = np.concatenate([shared, own]).astype(np.int32)
        rng.shuffle(i)
        v = (rng.standard_normal(len(i)) * 1e-3).astype(np.float32)
        idx.append(i)
        val.append(oracle.f32_to_bf16_bits(v) if dtype == "bf16" else v)
    return idx, val


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("n,peers,per_peer,overlap", [(1000, 4, 50, 0.2), (1 << 20, 16, 5000, 0.3),
                                                      (1 << 22, 64, 3000, 0.4), (4096, 8, 4096, 0.9),
                                                      (1 << 16, 1, 1, 0.0)])
def test_merge_sparse(zen, oracle, n, peers, per_peer, overlap, dtype):
    rng = np.random.default_rng(n + peers)
    idx, val = make_payloads(oracle, rng, n, peers, per_peer, overlap, dtype)
    ci, cv = np.concatenate(idx), np.concatenate(val)
    want_i, want_v = oracle.merge_sparse(ci, cv, n)
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(peers), None, None)
    gi, gv = lba.merge_sparse([to_dev(i) for i in idx], [to_dev(v) for v in val], n)
    assert gi.dtype == torch.int64 and gv.dtype == torch.float32
    assert np.array_equal(to_np(gi), want_i)
    # same adds in the same order: bit-exact against the sequential fp32 oracle
    assert np.array_equal(to_np(gv).view(np.uint32), want_v.view(np.uint32))
    # and within 1e-6 (relative to the summed magnitudes) of the fp64 truth
    truth = oracle.decode(ci, cv, n, "f64")[want_i]
    vf = oracle.bf16_bits_to_f32(cv) if dtype == "bf16" else cv
    scale = np.zeros(n)
    np.add.at(scale, ci, np.abs(vf.astype(np.float64)))
    assert (np.abs(to_np(gv) - truth) <= 1e-6 * scale[want_i] + 1e-30).all()


@pytest.mark.parametrize("mode", [0, 1])
def test_merge_modes_agree_with_oracle(zen, oracle, mode):
    rng = np.random.default_rng(77 + mode)
    n = 3000017
    idx, val = make_payloads(oracle, rng, n, 16, 20000, 0.3, "bf16")
    ci, cv = np.concatenate(idx), np.concatenate(val)
    want_i, want_v = oracle.merge_sparse(ci, cv, n)
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(16), None, None)
    gi, gv, cnt, st = lba.merge_sparse_flat(to_dev(ci), to_dev(cv), n, mode=mode)
    assert st.item() == 0 and cnt.item() == len(want_i)
    assert np.array_equal(to_np(gi)[:len(want_i)], want_i.astype(np.int32))
    assert np.array_equal(to_np(gv)[:len(want_i)].view(np.uint32), want_v.view(np.uint32))


def test_merge_piled_up_keys_fall_back_to_general_mode(zen, oracle):
    from zen_repro_amd import _lib

    n = 1 << 20
    rng = np.random.default_rng(3)
    idx = np.concatenate([np.full(100000, 12345), rng.integers(0, n, 50000)]).astype(np.int32)
    val = (rng.standard_normal(len(idx)) * 1e-3).astype(np.float32)
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(4), None, None)
    _, _, cnt, st = lba.merge_sparse_flat(to_dev(idx), to_dev(val), n, mode=_lib.MODE_FAST)
    assert st.item() == _lib.STAT_RETRY  # one key range holds more than a workgroup sorts in LDS
    gi, gv = lba.merge_sparse(to_dev(idx), to_dev(val), n)  # retries by itself
    wi, wv = oracle.merge_sparse(idx, val, n)
    assert np.array_equal(to_np(gi), wi) and np.array_equal(to_np(gv).view(np.uint32), wv.view(np.uint32))
    dense = lba.decode_sparse_tensors(to_dev(idx), to_dev(val), n)
    assert np.array_equal(to_np(dense), oracle.decode(idx, val, n, "f32acc"))


def test_merge_cancellation_nan_and_bad_index(zen, oracle):
    from zen_repro_amd import _lib

    n = 64
    idx = np.array([5, 9, 5, 63, 9, 0, 0, 17], np.int32)
    val = np.array([1.0, 2.0, -1.0, 4.0, np.nan, 3.0, -3.0, -0.0], np.float32)
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(2), None, None)
    gi, gv = lba.merge_sparse(to_dev(idx), to_dev(val), n)
    wi, wv = oracle.merge_sparse(idx, val, n)
    assert to_np(gi).tolist() == wi.tolist() == [9, 63]
    assert np.array_equal(to_np(gv).view(np.uint32) & 0x7FC00000, wv.view(np.uint32) & 0x7FC00000)
    bad = np.array([5, 64, -1, 7], np.int64)
    for mode in (0, 1):
        i2, v2, cnt, st = lba.merge_sparse_flat(to_dev(bad), to_dev(np.ones(4, np.float32)), n, idx64=True, mode=mode)
        assert cnt.item() == 2 and st.item() == _lib.STAT_BAD_INDEX
        assert to_np(i2)[:2].tolist() == [5, 7]


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
def test_decode_sparse_tensors_dense(zen, oracle, dtype):
    rng = np.random.default_rng(8)
    n, peers = 1 << 18, 8
    idx, val = make_payloads(oracle, rng, n, peers, 4000, 0.3, dtype)
    ci, cv = np.concatenate(idx), np.concatenate(val)
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(peers), None, None)
    dense = lba.decode_sparse_tensors([to_dev(i) for i in idx], [to_dev(v) for v in val], n)
    f32 = oracle.decode(ci, cv, n, "f32acc")
    want = oracle.f32_to_bf16_bits(f32) if dtype == "bf16" else f32
    got = to_np(dense)
    assert dense.dtype == (torch.bfloat16 if dtype == "bf16" else torch.float32)
    assert np.array_equal(got, want)
    # single-tensor form with int64 indices (comm.py:40-44)
    d2 = lba.decode_sparse_tensors(to_dev(ci.astype(np.int64)), to_dev(cv), n)
    assert np.array_equal(to_np(d2), want)
    if dtype == "bf16":
        # against the reference's own accumulation dtype: 1e-3 relative
        native = oracle.bf16_bits_to_f32(oracle.decode(ci, cv, n, "native"))
        scale = np.zeros(n)
        np.add.at(scale, ci, np.abs(oracle.bf16_bits_to_f32(cv).astype(np.float64)))
        assert (np.abs(oracle.bf16_bits_to_f32(got) - native) <= 2e-2 * scale + 1e-30).all()


def ascending_lists(oracle, rng, n, nlists, per_list, shared, dtype, idx_dtype):
    """nlists strictly ascending index lists over [0, n); a fraction `shared` of every list comes from one pool
    (lists meet on those indices), the rest lies in the list's own residue class (disjoint)."""
    pool = rng.choice(n // nlists, max(1, int(per_list * shared) * 2), replace=False) * nlists
    idx, val = [], []
    for l in range(nlists):
        common = rng.choice(pool, int(per_list * shared), replace=False) if shared > 0 else np.empty(0, np.int64)
        own = rng.choice(n // nlists, per_list - len(common), replace=False) * nlists + (l if l else 0)
        i = np.unique(np.concatenate([common, own])).astype(idx_dtype)
        v = (rng.standard_normal(len(i)) * 1e-3).astype(np.float32)
        v[::97] = -0.0  # +0 + -0 = +0: the dense element stays a plain zero
        idx.append(i)
        val.append(oracle.f32_to_bf16_bits(v) if dtype == "bf16" else v)
    return idx, val


@pytest.mark.parametrize("idx_dtype", [np.int64, np.int32])
@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("n,nlists,per_list,shared", [
    ((1 << 22) + 4099, 16, 20000, 0.0),   # the second exchange: disjoint shards; size not a multiple of the tile
    (1 << 22, 16, 20000, 0.4),            # method 1: every rank's own selection, lists meet on many indices
    (1 << 20, 1, 5000, 0.0),
    (3000, 5, 40, 0.5),                   # less than one tile
    (1 << 21, 64, 3000, 0.1),
])
def test_decode_ascending_lists_without_a_sort(zen, oracle, n, nlists, per_list, shared, dtype, idx_dtype):
    """zen_decode_dense_sorted through decode_sparse_tensors(ascending=True): bit-identical to the oracle's
    sequential fp32 scatter_add (and therefore to zen_decode_dense), straight through the C-ABI too."""
    from zen_repro_amd import _lib

    rng = np.random.default_rng(n % 977 + nlists)
    idx, val = ascending_lists(oracle, rng, n, nlists, per_list, shared, dtype, idx_dtype)
    ci, cv = np.concatenate(idx), np.concatenate(val)
    f32 = oracle.decode(ci.astype(np.int64), cv, n, "f32acc")
    want = oracle.f32_to_bf16_bits(f32) if dtype == "bf16" else f32
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(max(nlists, 2)), None, None)
    d_idx, d_val = [to_dev(i) for i in idx], [to_dev(v) for v in val]
    got = lba.decode_sparse_tensors(d_idx, d_val, n, ascending=True)
    assert np.array_equal(to_np(got).view(want.dtype), want)
    assert np.array_equal(to_np(lba.decode_sparse_tensors(d_idx, d_val, n)).view(want.dtype), want)
    # the entry point itself: it must have taken the lists as they are (status 0), into a buffer full of ones
    L = _lib.lib()
    flat_i, flat_v = to_dev(ci), to_dev(cv)
    dense = torch.full((n,), 1.0, dtype=flat_v.dtype, device="cuda")
    starts = (ctypes.c_int64 * (nlists + 1))(0, *np.cumsum([len(i) for i in idx]).tolist())
    ws = torch.empty(L.zen_decode_dense_sorted_workspace(n, nlists), dtype=torch.uint8, device="cuda")
    status = _lib.status_word("cuda")
    rc = L.zen_decode_dense_sorted(_lib.ptr(flat_i), int(idx_dtype == np.int64), _lib.ptr(flat_v), _lib.dtype_code(flat_v),
                                   starts, nlists, _lib.ptr(dense), n, _lib.ptr(ws), ws.numel(), _lib.ptr(status),
                                   _lib.stream_of("cuda"))
    assert rc == 0 and status.item() == 0
    assert np.array_equal(to_np(dense).view(want.dtype), want)


@pytest.mark.parametrize("n", [256 * 8192, 256 * 8192 + 1, 4096 * 8192, 4096 * 8192 + 1])
def test_decode_ascending_tells_the_host(zen, oracle, n):
    """Tiles that search for themselves, up to the last size that does, and tiles with a kernel in front: right lists bit
    for bit, a descent seen, and the call after it right again."""
    rng = np.random.default_rng(n)
    idx, val = ascending_lists(oracle, rng, n, 4, 20000, 0.1, "bf16", np.int64)
    want = oracle.f32_to_bf16_bits(oracle.decode(np.concatenate(idx), np.concatenate(val), n, "f32acc"))
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(4), None, None)
    d_idx, d_val = [to_dev(i) for i in idx], [to_dev(v) for v in val]
    swapped = [i.copy() for i in idx]
    swapped[3][[-2, -1]] = swapped[3][[-1, -2]]
    for _ in range(2):
        assert np.array_equal(to_np(lba._decode_ascending(d_idx, d_val, n)).view(want.dtype), want)
        assert lba._decode_ascending([to_dev(i) for i in swapped], d_val, n) is None


@pytest.mark.parametrize("n", [200000, 20000000, 100000000])
def test_decode_ascending_is_complete_for_every_stream(zen, n):
    """When the call has returned another stream may overwrite the lists and read the tensor, without a wait."""
    gen = torch.Generator(device="cuda").manual_seed(n)
    idx = [torch.nonzero(torch.rand(n, generator=gen, device="cuda") < 0.02).view(-1) for _ in range(3)]
    val = [torch.randn(i.numel(), generator=gen, device="cuda").bfloat16() for i in idx]
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(3), None, None)
    want = lba._decode_ascending(idx, val, n)
    side = torch.cuda.Stream()
    for _ in range(3):
        i, v = [t.clone() for t in idx], [t.clone() for t in val]
        torch.cuda.synchronize()
        got = lba._decode_ascending(i, v, n)
        with torch.cuda.stream(side):
            seen = got.clone()
            for t in i + v:
                t.zero_()
        torch.cuda.synchronize()
        assert torch.equal(seen, want) and torch.equal(got, want)


def test_decode_ascending_declines_what_is_not_ascending(zen, oracle):
    """A list with a descent, a repeated index inside one list or an index outside the dense tensor raise
    ZEN_STAT_RETRY; decode_sparse_tensors then answers through the general entry point (or raises, for the
    bad index, as the reference's scatter_add_ does)."""
    from zen_repro_amd import _lib

    n = 1 << 20
    rng = np.random.default_rng(3)
    idx, val = ascending_lists(oracle, rng, n, 4, 3000, 0.2, "f32", np.int64)
    L = _lib.lib()

    def status_of(lists):
        flat_i, flat_v = to_dev(np.concatenate(lists)), to_dev(np.concatenate(val))
        dense = torch.empty(n, dtype=torch.float32, device="cuda")
        starts = (ctypes.c_int64 * 5)(0, *np.cumsum([len(i) for i in lists]).tolist())
        ws = torch.empty(L.zen_decode_dense_sorted_workspace(n, 4), dtype=torch.uint8, device="cuda")
        status = _lib.status_word("cuda")
        rc = L.zen_decode_dense_sorted(_lib.ptr(flat_i), 1, _lib.ptr(flat_v), _lib.F32, starts, 4, _lib.ptr(dense), n,
                                       _lib.ptr(ws), ws.numel(), _lib.ptr(status), _lib.stream_of("cuda"))
        assert rc == 0
        return int(status.item())

    assert status_of(idx) == 0
    swapped = [i.copy() for i in idx]
    swapped[2][[100, 101]] = swapped[2][[101, 100]]          # one descent
    assert status_of(swapped) == _lib.STAT_RETRY
    twice = [i.copy() for i in idx]
    twice[1][500] = twice[1][499]                             # the same index twice in one list
    assert status_of(twice) == _lib.STAT_RETRY
    beyond = [i.copy() for i in idx]
    beyond[3][-1] = n + 5                                     # ascending, but outside the tensor
    assert status_of(beyond) == _lib.STAT_RETRY
    below = [i.copy() for i in idx]
    below[0][0] = -3
    assert status_of(below) == _lib.STAT_RETRY
    # through the wrapper the result is right all the same
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(4), None, None)
    for lists in (swapped, twice):
        got = lba.decode_sparse_tensors([to_dev(i) for i in lists], [to_dev(v) for v in val], n, ascending=True)
        assert np.array_equal(to_np(got), oracle.decode(np.concatenate(lists), np.concatenate(val), n, "f32acc"))
    with pytest.raises(RuntimeError):
        lba.decode_sparse_tensors([to_dev(i) for i in beyond], [to_dev(v) for v in val], n, ascending=True)
    # bad arguments are the host's business
    ws = torch.empty(1024, dtype=torch.uint8, device="cuda")
    status = _lib.status_word("cuda")
    bad = (ctypes.c_int64 * 3)(0, 10, 5)
    assert L.zen_decode_dense_sorted(_lib.ptr(ws), 1, _lib.ptr(ws), _lib.F32, bad, 2, _lib.ptr(ws), 100, _lib.ptr(ws),
                                     ws.numel(), _lib.ptr(status), None) == _lib.EINVAL
    ok = (ctypes.c_int64 * 2)(0, 10)
    assert L.zen_decode_dense_sorted(_lib.ptr(ws), 1, _lib.ptr(ws), _lib.F32, ok, 1, _lib.ptr(ws), 1 << 30,
                                     _lib.ptr(ws), ws.numel(), _lib.ptr(status), None) == _lib.EWORKSPACE


@pytest.mark.parametrize("form", ["strided indices", "strided values", "two index types", "two value types", "one buffer"])
def test_decode_ascending_lists_in_any_layout(zen, oracle, form):
    """Ascending lists that are no plain runs of one type are put into one buffer first and decoded all the same."""
    rng = np.random.default_rng(72)
    n = 40000
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(4), None, None)
    idx, val = ascending_lists(oracle, rng, n, 4, 3000, 0.2, "f32", np.int64)
    if form == "two value types":  # both types hold the values exactly
        val = [oracle.bf16_bits_to_f32(oracle.f32_to_bf16_bits(v)) for v in val]
    d_idx, d_val = [to_dev(i) for i in idx], [to_dev(v) for v in val]
    want = oracle.decode(np.concatenate(idx), np.concatenate(val), n, "f32acc")
    strided = lambda t: torch.stack([t, torch.full_like(t, 7)], dim=1)[:, 0]
    if form == "strided indices":
        d_idx[2] = strided(d_idx[2])
    elif form == "strided values":
        d_val = [strided(v) for v in d_val]
    elif form == "two index types":
        d_idx[1] = d_idx[1].int()
    elif form == "two value types":
        d_val[3] = d_val[3].bfloat16()
    else:
        d_val = torch.cat(d_val)
    got = lba.decode_sparse_tensors(d_idx, d_val, n, ascending=True)
    assert got.dtype == torch.float32 and np.array_equal(to_np(got).view(np.uint32), want.view(np.uint32))


def test_stack_tensors_views_are_not_copied(zen):
    buf = torch.arange(100, device="cuda", dtype=torch.int32)
    parts = [buf[0:10], buf[10:45], buf[45:100]]
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(3), None, None)
    assert lba.stack_tensors(parts).data_ptr() == buf.data_ptr()
    other = [buf[0:10], buf[20:30]]
    assert lba.stack_tensors(other).tolist() == list(range(10)) + list(range(20, 30))


def test_zero_pool_pieces_are_zero_apart_and_per_stream(zen):
    """Status words, counts and split sizes are cut from pooled zeroed blocks: every piece is zero, aligned,
    handed out once, and belongs to the stream that was current when its block was made."""
    from zen_repro_amd import _lib

    pool = _lib.ZeroPool()
    a = pool.take("cuda", 1, torch.int32)
    b = pool.take("cuda", 16, torch.int64)
    c = pool.take("cuda", 3, torch.int32)
    for t, n, dt in ((a, 1, torch.int32), (b, 16, torch.int64), (c, 3, torch.int32)):
        assert t.dtype == dt and t.numel() == n and t.data_ptr() % 16 == 0 and int(t.abs().sum()) == 0
    spans = sorted((t.data_ptr(), t.data_ptr() + t.numel() * t.element_size()) for t in (a, b, c))
    assert all(spans[i][1] <= spans[i + 1][0] for i in range(2))
    a.fill_(7)  # a holder may write: the neighbours stay zero
    assert int(b.abs().sum()) == 0 and int(c.abs().sum()) == 0
    base = a.data_ptr()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        d = pool.take("cuda", 1, torch.int32)
        assert int(d.item()) == 0
    assert not (base <= d.data_ptr() < base + pool.BLOCK)  # another stream, another block
    # a block that is used up is replaced, not reused
    seen = set()
    for _ in range(2 * pool.BLOCK // 16 + 3):
        t = pool.take("cuda", 1, torch.int32)
        assert t.data_ptr() not in seen
        seen.add(t.data_ptr())
    assert int(t.item()) == 0
    big = pool.take("cuda", pool.BLOCK, torch.uint8)  # too large for a block: a tensor of its own
    assert big.numel() == pool.BLOCK and int(big.sum()) == 0


def test_profile_every_nth_launch(zen, oracle):
    """zen_profile_every(n): of a tag's launches since recording began, the first and every n-th after it
    carry events."""
    from zen_repro_amd import _lib

    vals = to_dev(make_grad(oracle, 1 << 16, 0.05, "f32", seed=5))
    try:
        _lib.profile_enable(True, only="k_compress", every=3)
        for _ in range(7):
            zen.compress(10, vals)
        torch.cuda.synchronize()
        got = _lib.profile_read()
        assert set(got) == {"k_compress"} and got["k_compress"][1] == 3 and got["k_compress"][0] > 0
        _lib.profile_enable(True, every=1)
        for _ in range(2):
            zen.compress(10, vals)
        assert _lib.profile_read()["k_compress"][1] == 2
        with pytest.raises(ValueError):
            _lib.profile_enable(True, every=0)
    finally:
        _lib.profile_enable(False)
        _lib.check(_lib.lib().zen_profile_every(1), "profile_every")


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("idx64", [False, True])
@pytest.mark.parametrize("count", [0, 1, 2047, 2049, 300000])
def test_round_merged_sums(zen, oracle, dtype, idx64, count):
    """zen_round_compact: what comm.py:125-127 makes of the merged sums (a dense tensor of the gradient's type,
    then its nonzeros): every fp32 sum rounded once to the type, entries that round to zero dropped, order
    kept; only the first `count` entries (a device value) are looked at.  Sums that are tiny, negative zeros,
    NaN and infinities included."""
    cap = count + 100
    rng = np.random.default_rng(count + 7)
    sums = (rng.standard_normal(cap) * 1e-3).astype(np.float32)
    sums[rng.integers(0, cap, cap // 5)] = 0.0
    sums[rng.integers(0, cap, cap // 7)] = -0.0
    sums[rng.integers(0, cap, cap // 9)] = 1e-41 if dtype == "bf16" else 1e-45  # bf16: rounds to zero
    sums[rng.integers(0, cap, 3)] = np.nan
    sums[rng.integers(0, cap, 3)] = -np.inf
    idx = np.sort(rng.choice(1 << 30, cap, replace=False)).astype(np.int64 if idx64 else np.int32)
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(4), None, None)
    tdt = torch.bfloat16 if dtype == "bf16" else torch.float32
    cnt = torch.tensor([count], dtype=torch.int64, device="cuda")
    o_idx, o_val, kept, status = lba.round_merged_flat(to_dev(idx), to_dev(sums), cnt, tdt)
    assert int(status) == 0
    rounded = torch.from_numpy(sums[:count]).to(tdt)
    keep = (rounded != 0).numpy()  # NaN != 0 is true, -0.0 != 0 false: what torch.nonzero keeps
    u = int(kept)
    assert u == int(keep.sum())
    assert np.array_equal(to_np(o_idx)[:u], idx[:count][keep])
    bits = torch.int16 if dtype == "bf16" else torch.int32
    got, want = o_val[:u].cpu(), rounded[torch.from_numpy(keep)]
    nan = torch.isnan(want)
    assert torch.equal(torch.isnan(got), nan)  # a NaN stays a NaN (which of the NaN patterns is the converter's business)
    assert torch.equal(got[~nan].view(bits), want[~nan].view(bits))


@pytest.mark.parametrize("dtype", ["fp32", "bf16"])
@pytest.mark.parametrize("s", [1, 1023, 8192, 8193, 16384, 16385, 4096 * 15 + 1, 4096 * 256 + 77])
@pytest.mark.parametrize("kind", ["normal", "sparse", "constant"])
def test_sample_threshold_at_the_edges_of_its_kernels(zen, oracle, s, dtype, kind):
    """One workgroup (up to 8192 positions of bf16, 16384 of fp32), a few, all of them; a sample nearly all of which is zero and one whose
    elements are all equal, so that one histogram bin takes everything.  Keys and counts are whole numbers: exact."""
    import importlib

    C = importlib.import_module("zen_repro_amd.compress")
    n = 70001
    g = make_grad(oracle, n, 0.02 if kind == "sparse" else 1.0, dtype, seed=s)
    if kind == "constant":
        g[:] = g[5]
    at = np.random.default_rng(s).integers(0, n, s)
    keys = ((g & 0x7FFF) if dtype == "bf16" else (g.view(np.uint32) & 0x7FFFFFFF))[at]
    order = np.sort(keys)[::-1]
    for k in sorted({1, max(1, s // 100), max(1, s // 2), s}):
        thr, status = C.sample_threshold(to_dev(g), torch.from_numpy(at).cuda(), k)
        key, count = (int(x) & 0xFFFFFFFF for x in to_np(thr))
        assert int(status) == 0 and key == int(order[k - 1]) and count == int((keys >= key).sum()), (k, kind)


@pytest.mark.parametrize("dtype", ["fp32", "bf16"])
@pytest.mark.parametrize("n", [1, 511, 65536, 65537, 300001, 8192 * 2048 + 5])
@pytest.mark.parametrize("density", [0.01, 0.125, 0.6])
def test_ordered_compaction_at_the_edges_of_its_kernels(zen, oracle, n, dtype, density):
    """One workgroup (up to 65536 elements) and a stretch per wave; fewer entries than an eighth of a stretch, about
    that many (stretches on either side of it) and more; an aligned and an unaligned tensor; too little room."""
    from zen_repro_amd.comm import _select_raw
    from zen_repro_amd import _lib

    g = make_grad(oracle, n + 1, density, dtype, seed=n)
    keys = (g & 0x7FFF) if dtype == "bf16" else (g.view(np.uint32) & 0x7FFFFFFF)
    d = to_dev(g)
    for shift in (0, 1):
        want = np.flatnonzero(keys[shift:])
        idx, val, count, bits = _select_raw(d[shift:], None, True)
        assert bits == 0 and count == want.size
        assert np.array_equal(to_np(idx), want) and np.array_equal(to_np(val), to_np(to_dev(g[shift:][want])))
        room = want.size // 2
        idx, val, count, bits = _select_raw(d[shift:], None, False, capacity=room)
        assert count == want.size and bits == (_lib.STAT_CAPACITY if want.size > room else 0)
        assert np.array_equal(to_np(idx), want[:room])


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("n,P,density,scale,rehash", [
    (4097, 4, 0.1, 1, 3), (32768, 256, 0.05, 1, 3), (32771, 4, 0.3, 1, 3), (32768, 2, 0.15, 1, 1),  # one workgroup, and just beyond
    (32768, 257, 0.02, 1, 3), (20000, 8, 0.2, 2, 3),                      # more partitions, more slots than it takes
    (262143, 16, 0.1, 1, 3), (1 << 18, 1000, 0.02, 1, 3),                 # ragged stretches, many partitions in one
    (1048575, 2, 0.15, 1, 2), (3000001, 16, 0.1, 1, 3), (1 << 22, 64, 0.01, 1, 3),  # long serial tails; the largest
])
def test_load_balance_through_the_owner_table(zen, oracle, n, P, density, scale, rehash, dtype):
    """Nonzeros, a threshold and a top-k selection, twice on the same table; whole numbers and copies: exact."""
    g = make_grad(oracle, n, density, dtype, seed=n ^ P)
    g[0] = 0x3F80 if dtype == "bf16" else 1.0
    tp = zen.TensorPartition(P, scale, rehash)
    d = to_dev(g)
    k = max(1, int(n * density) // 2)  # fewer than there are nonzeros: the wide buckets (top-k from 2^20 slots on) decline others
    key = oracle.kth_key(g, k)
    masked, _ = oracle.mask_dense(g, key)
    whole = oracle.load_balance(g, P, scale, rehash)
    part = oracle.load_balance(masked, P, scale, rehash)
    thr = zen.topk_threshold(d, k)
    for (idx_o, val_o, splits_o, st_o), kw in ((whole, {}), (part, {"thr": thr}), (part, {"k": k})):
        if st_o:
            continue  # a serial region overflowed
        for capacity in (len(idx_o), len(idx_o) + 77):
            oi, ov, splits, status = tp.load_balance_flat(d, capacity=max(1, capacity), **kw)
            assert status.item() == 0
            assert np.array_equal(to_np(splits), splits_o)
            assert np.array_equal(to_np(oi)[:len(idx_o)], idx_o) and np.array_equal(to_np(ov)[:len(idx_o)], val_o)
    m, _ = oracle.table_sizes(n, P, scale)
    assert not tp._table(d.device, m).any()


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("n,P,density,rehash", [
    (1 << 21, 16, 0.15, 3),          # thousands of level-2/3 moves
    (1 << 21, 16, 0.15, 2),          # two levels: serial entries in every partition
    ((1 << 21) + 1237, 16, 0.03, 3),  # a length that is no multiple of anything, and a table that is none of 4096
    ((1 << 20) + 2, 3, 0.05, 1),     # one level: whoever loses its slot ends in the serial list
    (1 << 21, 4, 0.2, 1),            # more of those than a partition carries: declined
])
def test_nonzeros_on_the_wide_buckets_while_a_sample_waits(zen, oracle, n, P, density, rehash, dtype):
    """A sample waits in the table of its call, which then is no owner table, and tables of 2^20 to 2^22 slots are too
    small for the bucket slabs: selections of any density on the wide buckets, from tensors that begin on 16 bytes and
    between, and from one without nonzeros.  The call the sample was taken for finds it untouched."""
    from zen_repro_amd import _lib

    g = make_grad(oracle, n, density, dtype, seed=n + rehash)
    g[-1] = 0x3F80 if dtype == "bf16" else 1.0
    idx_o, val_o, splits_o, st_o = oracle.load_balance(g, P, 1, rehash)
    x = (np.random.default_rng(n).standard_normal(n) * 1e-3).astype(np.float32)
    x[0] = 0
    if dtype == "bf16":
        x = (x.view(np.uint32) >> 16).astype(np.uint16)
    k, capacity = 4000, len(idx_o) + 1024
    masked, kept = oracle.mask_dense(x, int(oracle.kth_key(x, k)))
    tp = zen.TensorPartition(P, 1, rehash)
    m, _ = tp.table_sizes(n)
    sampled = to_dev(x)
    tp.prepare(sampled, k, 2 * k)
    assert tp._ahead_state(sampled.device, 0)["pending"]
    code = _lib.BF16 if dtype == "bf16" else _lib.F32
    assert _lib.lib().zen_load_balance_path(n, m, code, capacity, P, 0, _lib.MODE_FAST) == 3
    buf = to_dev(np.concatenate([g[:3], g]))
    for d in (to_dev(g), buf[3:]):
        oi, ov, splits, status = tp.load_balance_flat(d, capacity=capacity)
        if (density, rehash) == (0.2, 1):
            assert status.item() & _lib.STAT_RETRY
            return
        assert st_o == 0 and status.item() == 0 and np.array_equal(to_np(splits), splits_o)
        assert np.array_equal(to_np(oi)[:len(idx_o)], idx_o) and np.array_equal(to_np(ov)[:len(idx_o)], val_o)
    _, _, splits, status = tp.load_balance_flat(torch.zeros_like(buf[3:]), capacity=capacity)
    assert status.item() == 0 and not splits.any()
    assert tp._ahead_state(sampled.device, 0)["pending"]
    idx_o, val_o, splits_o, _ = oracle.load_balance(masked, P, 1, rehash)
    oi, ov, splits, status = tp.load_balance_flat(sampled, capacity=2 * k, k=k)
    assert not tp._ahead_state(sampled.device, 0)["pending"]
    assert status.item() == 0 and np.array_equal(to_np(splits), splits_o)
    assert np.array_equal(to_np(oi)[:kept], idx_o) and np.array_equal(to_np(ov)[:kept], val_o)
    assert not tp._table(sampled.device, m).any()


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("n,P,density,rehash", [
    (9219, 4, 0.1, 3), (32768, 4, 0.6, 3),            # one workgroup: a list of selected indices, several of them
    (49152, 3, 0.1, 3), (49151, 3, 0.1, 2),           # partitions that end with a stretch, and in front of its end
    (1 << 18, 1000, 0.02, 3), (3000001, 16, 0.1, 1),  # dozens of partitions to a stretch; long serial tails
])
def test_owner_table_tells_the_host(zen, oracle, n, P, density, rehash, dtype):
    """The calls that wait for the sizes, which the last kernel itself stores."""
    g = make_grad(oracle, n, density, dtype, seed=n + 3 * P)
    idx_o, val_o, splits_o, st_o = oracle.load_balance(g, P, 1, rehash)
    assert st_o == 0
    tp = zen.TensorPartition(P, 1, rehash)
    d = to_dev(g)
    for rep in range(2):
        indices, values, splits = tp.load_balance(d)
        assert [len(i) for i in indices] == list(splits_o) and np.array_equal(to_np(splits), splits_o)
        assert np.array_equal(to_np(torch.cat(indices)), idx_o) and np.array_equal(to_np(torch.cat(values)), val_o)
    with pytest.raises(RuntimeError, match="capacity"):
        tp.load_balance(d, capacity=len(idx_o) - 1)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("r", [1, 1023, 1025, 4096, 6144, 6145])
@pytest.mark.parametrize("n", [1, 1000, 262144, 262145, 2147483647])
def test_merge_in_one_workgroup(zen, oracle, n, r, dtype):
    """One workgroup up to 6144 entries, just beyond it the wide buckets or the sort; every entry on one index, few and many
    of them; dense results of up to a megabyte, and longer ones."""
    gen = torch.Generator().manual_seed(r + n % 1000)
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(4), None, None)
    for spread in (1, min(n, 700), n):
        idx = torch.randint(0, spread, (r,), generator=gen, dtype=torch.int64) * (n // spread) + (n - 1) % (n // spread)
        val = (torch.randn(r, generator=gen) * 1e-3).to(dtype)
        val[r // 2] = -0.0
        which, place = np.unique(idx.numpy(), return_inverse=True)  # (the oracle's dense tensor: as long as needed)
        w_idx, w_val = oracle.merge_sparse(place, to_np(val), len(which))
        w_idx = which[w_idx]
        d_idx, d_val = idx.cuda(), val.cuda()
        m_idx, m_val = lba.merge_sparse(d_idx, d_val, n)
        assert np.array_equal(to_np(m_idx), w_idx) and np.array_equal(to_np(m_val).view(np.uint32), w_val.view(np.uint32))
        rounded = torch.from_numpy(w_val).to(dtype)
        kept = rounded != 0
        m_idx, m_val = lba.merge_rounded(d_idx.int(), d_val, n, dtype)
        assert np.array_equal(to_np(m_idx), w_idx[kept.numpy()]) and torch.equal(m_val.cpu(), rounded[kept])
        if n <= 262145:
            want = torch.zeros(n, dtype=dtype)
            want[torch.from_numpy(w_idx.astype(np.int64))] = rounded
            assert torch.equal(lba.decode_sparse_tensors(d_idx, d_val, n).cpu(), want)
            with pytest.raises(RuntimeError, match="range"):
                lba.decode_sparse_tensors(torch.where(d_idx == d_idx[0], n, d_idx), d_val, n)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("r", [64, 65, 1025, 2048, 4097, 6143, 6144])
@pytest.mark.parametrize("kind", ["narrow", "run", "eight of each", "half narrow", "half on one"])
def test_merge_in_one_workgroup_of_indices_that_pile_up(zen, oracle, kind, r, dtype):
    """Lists whose indices lie in few of the ranges they are sorted by, some outside the tensor among them: sums, order and
    flags as ever, and a time that does not go with the square of the length (it was fifty times that of a spread list;
    the sum of many values of one index is a chain of its own)."""
    from zen_repro_amd import _lib

    n = 1 << 30
    gen = torch.Generator().manual_seed(r)
    idx = {"narrow": lambda: torch.randint(0, 1 << 18, (r,), generator=gen),
           "run": lambda: torch.randperm(r, generator=gen),
           "eight of each": lambda: torch.randint(0, max(1, r // 8), (r,), generator=gen),
           "half narrow": lambda: torch.where(torch.arange(r) % 2 == 0, torch.randint(0, n // 4, (r,), generator=gen),
                                              torch.randint(0, 1 << 18, (r,), generator=gen)),
           "half on one": lambda: torch.where(torch.arange(r) % 2 == 0, torch.randint(0, n // 4, (r,), generator=gen), 7)}[kind]()
    idx = idx + n // 2
    spread = torch.randint(0, n, (r,), generator=gen).cuda()
    val = (torch.randn(r, generator=gen) * 1e-3).to(dtype)
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(4), None, None)
    d_val = val.cuda()
    for bad in (0, 3):
        idx[torch.randperm(r, generator=gen)[:bad]] = torch.tensor([-1, n, 1 << 40])[:bad]
        good = ((idx >= 0) & (idx < n)).numpy()
        which, place = np.unique(idx.numpy()[good], return_inverse=True)
        w_idx, w_val = oracle.merge_sparse(place, to_np(val)[good], len(which))
        m_idx, m_val, count, status = lba.merge_sparse_flat(idx.cuda(), d_val, n)
        assert status.item() == (_lib.STAT_BAD_INDEX if bad else 0) and count.item() == len(w_idx)
        assert np.array_equal(to_np(m_idx)[:len(w_idx)], which[w_idx])
        assert np.array_equal(to_np(m_val)[:len(w_idx)].view(np.uint32), w_val.view(np.uint32))
    d_idx = idx.cuda()

    def quickest(i):
        times = []
        for _ in range(20):
            begin, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            begin.record()
            lba.merge_sparse_flat(i, d_val, n)
            end.record()
            end.synchronize()
            times.append(begin.elapsed_time(end))
        return min(times)

    assert kind == "half on one" or quickest(d_idx) < 10 * quickest(spread)


@pytest.mark.parametrize("words", [1, 1023, 1024, (1 << 16) - 1, 1 << 16, (1 << 19) + 1])
def test_read_back_of_any_length(zen, words):
    """Both types, a word and a list of `words` of them, up to and past what goes through the pinned buffer."""
    from zen_repro_amd import _lib

    wide = torch.arange(words, dtype=torch.int64, device="cuda") * (1 << 33) - 5
    narrow = torch.tensor([-7], dtype=torch.int32, device="cuda")
    assert list(_lib.read_back(wide, narrow)) == wide.tolist() + [-7]
    assert list(_lib.read_back(narrow, wide.int(), narrow)) == [-7] + wide.int().tolist() + [-7]


def test_read_back_leaves_the_core_to_others_in_a_long_wait(zen):
    """Behind tens of milliseconds of work the waiting thread sleeps nearly all the time, and what comes back is what
    the stream's work left."""
    import time

    from zen_repro_amd import _lib

    x = torch.ones(8192, 8192, device="cuda")
    word = torch.zeros(1, dtype=torch.int64, device="cuda")
    _lib.read_back(word)
    y = x @ x
    torch.cuda.synchronize()
    for _ in range(6):
        y = x @ x
    word += 5
    wall, core = time.perf_counter(), time.thread_time()
    assert list(_lib.read_back(word)) == [5]
    wall, core = time.perf_counter() - wall, time.thread_time() - core
    assert core < max(0.5 * wall, 0.004)  # a millisecond is watched through


def test_table_lists_of_very_many_partitions(zen, oracle):
    """get_sub_sparse_tensors with 2^19 partitions of eight slots."""
    P = 1 << 19
    rng = np.random.default_rng(81)
    g_np = rng.standard_normal(8 * P).astype(np.float32)
    memory = np.where(rng.random(8 * P) < 0.2, rng.integers(1, 8 * P, 8 * P), 0).astype(np.int32)
    tp = zen.TensorPartition(P, 1, 3)
    indices, values, splits = tp.get_sub_sparse_tensors(to_dev(g_np), to_dev(memory))
    assert np.array_equal(to_np(splits), (memory.reshape(P, 8) != 0).sum(axis=1))
    assert len(indices) == P and np.array_equal(to_np(torch.cat(indices)), memory[memory != 0])
    assert np.array_equal(to_np(torch.cat(values)), g_np[memory[memory != 0]])


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("r,n", [(1, 5000), (1023, 5000), (4096, 5000), (4096, 1 << 30), (4097, 20000), (30000, 40000), (9000, 16385)])
@pytest.mark.parametrize("copies", [1, 16, 0])
def test_merge_of_short_lists(zen, oracle, r, n, copies, dtype):
    """One workgroup (up to 4096 entries) and narrow wide buckets; indices that differ, that come about sixteen times
    and (0) that are all the same.  Sums in order of arrival: bit for bit, in fp32 and rounded once."""
    rng = np.random.default_rng(r + n + copies)
    distinct = 1 if copies == 0 else max(1, min(n - 1, r // copies))
    pool = rng.choice(n - 1, distinct, replace=False) + 1 if n < 1 << 20 else rng.integers(1, n, distinct)
    idx = rng.permutation(np.resize(pool, r)).astype(np.int32)
    val = make_grad(oracle, r, 1.0, dtype, seed=r)
    mi, mv = oracle.merge_sparse(idx, val, n)
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(4), None, None)
    di, dv = torch.from_numpy(idx).cuda(), to_dev(val)
    gi, gv = lba.merge_sparse(di, dv, n)
    assert np.array_equal(to_np(gi), mi) and np.array_equal(to_np(gv).view(np.uint32), mv.view(np.uint32))
    ri, rv = lba.merge_rounded(di, dv, n, dv.dtype)
    want = torch.from_numpy(mv).to(dv.dtype)
    keep = want != 0
    assert torch.equal(ri.cpu(), torch.from_numpy(mi)[keep]) and torch.equal(rv.cpu(), want[keep])
    if n <= 1 << 20:
        dense = torch.zeros(n, dtype=dv.dtype)
        dense[torch.from_numpy(mi).long()] = want
        assert torch.equal(lba.decode_sparse_tensors(di, dv, n).cpu(), dense)


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("n,P,flags", [
    (3000, 5, 0),               # one workgroup
    (300000, 7, 0),             # the owner table
    (6000000, 3, 0),            # wide buckets
    (6000000, 3, "slabs"),      # bucket slabs: the sizes come before the entries are in their places
    (300000, 600, "general"),
])
def test_sizes_the_host_is_told_by_the_calls_own_kernels(zen, oracle, n, P, flags, dtype):
    from zen_repro_amd import _lib

    mode = {0: None, "slabs": _lib.MODE_FAST | _lib.MODE_SLABS, "general": _lib.MODE_GENERAL}[flags]
    g = make_grad(oracle, n, 0.05, dtype, seed=n + P)
    idx_o, val_o, splits_o, st_o = oracle.load_balance(g, P, 1, 3)
    assert st_o == 0
    tp = zen.TensorPartition(P, 1, 3)
    d = to_dev(g)
    for rep in range(3):  # the same words are asked again
        indices, values, splits = tp.load_balance(d, mode=mode)
        assert [t.numel() for t in indices] == [t.numel() for t in values] == splits_o.tolist()
        assert np.array_equal(to_np(splits), splits_o)
        assert np.array_equal(to_np(torch.cat(indices)), idx_o) and np.array_equal(to_np(torch.cat(values)), val_o)
        zeros = tp.load_balance(torch.zeros_like(d), mode=mode)
        assert [t.numel() for t in zeros[0]] == [0] * P and not zeros[2].any()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("r,n", [(0, 1000), (1, 1000), (3000, 20000), (20000, 40000), (200000, 1 << 23)])
def test_count_the_host_is_told_by_the_merge(zen, r, n, dtype):
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(4), None, None)
    gen = torch.Generator(device="cuda").manual_seed(r + n)
    idx = torch.randint(0, n, (r,), generator=gen, device="cuda", dtype=torch.int32)
    val = torch.randint(1, 4, (r,), generator=gen, device="cuda").to(dtype)  # sums are exact
    want = torch.zeros(n, device="cuda").scatter_add_(0, idx.long(), val.float())
    at = torch.nonzero(want).view(-1)
    for flags in (0, zen._lib.MODE_SLABS):
        lba.fast_flags = flags
        got_idx, got_val = lba.merge_rounded(idx, val, n, dtype)
        assert torch.equal(got_idx, at) and torch.equal(got_val, want[at].to(dtype))


@pytest.mark.parametrize("s", [1, 1024, 1025, 5120, 5121, 16384, 16385, 65536, 65537, 270000])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_sample_threshold_of_every_size(zen, s, dtype):
    """One workgroup, several with the search in the second launch, with a third: the k-th largest and how many reach
    it, for distinct magnitudes, few different ones, magnitudes that share their upper half, and mostly zeros."""
    from zen_repro_amd import _lib

    L, dev = _lib.lib(), torch.device("cuda", torch.cuda.current_device())
    gen = torch.Generator(device="cuda").manual_seed(s)
    n = 300007
    noise = torch.randn(n, generator=gen, device="cuda")
    near = (torch.randint(0x3f800000, 0x3f800900, (n,), generator=gen, device="cuda", dtype=torch.int32)).view(torch.float32)
    at = torch.randint(0, n, (s,), generator=gen, device="cuda")
    for values in (noise, (noise * 3).round(), near, noise * (noise > 2.5)):
        t = values.to(dtype)
        code = _lib.dtype_code(t)
        keys = t[at].float().abs().view(torch.int32)
        ordered = torch.sort(keys, descending=True)[0]
        ws = torch.empty(L.zen_sample_threshold_workspace(s, code), dtype=torch.uint8, device=dev)
        for k in {1, s, max(1, s // 20), max(1, s // 2)}:
            thr = torch.full((2,), -1, dtype=torch.int32, device=dev)
            status = torch.zeros(1, dtype=torch.int32, device=dev)
            assert L.zen_sample_threshold(_lib.ptr(t), code, n, _lib.ptr(at), s, k, _lib.ptr(thr), _lib.ptr(ws), ws.numel(),
                                          _lib.ptr(status), _lib.stream_of(dev)) == 0
            want = ordered[k - 1].item()
            assert thr.tolist() == [want >> 16 if dtype == torch.bfloat16 else want, (keys >= want).sum().item()]
            assert status.item() == 0


@pytest.mark.parametrize("s", [128 * 1024, 128 * 1024 + 1, 255 * 1024 + 5, 256 * 4096 * 2, 256 * 4096 * 2 + 1, 256 * 4096 * 3 - 5,
                               256 * 4096 * 5 + 9, 256 * 65535 + 1])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_sample_threshold_in_rounds(zen, s, dtype):
    """As many workgroups as the search sums up in one batch and one more; one to sixteen rounds of 4096 places a workgroup, whole
    and cut off; more workgroups than compute units.  Places outside the tensor count as zero, in every round.  Exact."""
    import importlib

    from zen_repro_amd import _lib

    C = importlib.import_module("zen_repro_amd.compress")
    gen = torch.Generator(device="cuda").manual_seed(s)
    n = 300007
    t = torch.randn(n, generator=gen, device="cuda").to(dtype)
    at = torch.randint(0, n, (s,), generator=gen, device="cuda")
    for outside in (False, True):
        if outside:
            at[torch.randint(0, s, (1000,), generator=gen, device="cuda")] = n
            at[s - 1] = -1
        keys = torch.where((at >= 0) & (at < n), t[at.clamp(0, n - 1)], torch.zeros((), dtype=dtype, device="cuda"))
        keys = keys.float().abs().view(torch.int32)
        ordered = torch.sort(keys, descending=True)[0]
        for k in (1, s // 20, s):
            thr, status = C.sample_threshold(t, at, k)
            want = ordered[k - 1].item()
            assert thr.tolist() == [want >> 16 if dtype == torch.bfloat16 else want, (keys >= want).sum().item()]
            assert int(status) == (_lib.STAT_BAD_INDEX if outside else 0)


@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("n", [65537, 65536 + 2048, 65536 + 2049, 200001, 20000000])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_selection_of_every_density(zen, n, shift, dtype):
    """What a wave keeps of its findings is full at 512: rows with none, with a few, with all of their elements, and
    stretches with one kind of row behind the other; stretches cut off in a row, views from an odd element on."""
    from zen_repro_amd import comm

    gen = torch.Generator(device="cuda").manual_seed(n)
    room = torch.randn(n + shift, generator=gen, device="cuda").to(dtype)
    at = torch.arange(n + shift, device="cuda")
    lots = torch.rand(n + shift, generator=gen, device="cuda")
    for keep in (lots < 0.0, lots < 0.002, lots < 0.1, lots < 0.124, lots < 0.5, lots < 2.0, at // 512 % 3 == 0,
                 (at // 256 % 5 == 0) | (lots < 0.05), at >= n + shift - 1):
        t = torch.where(keep, room, torch.zeros_like(room))[shift:]
        want = torch.nonzero(t).view(-1)
        idx, val, count, bits = comm._select_raw(t, None, True)
        assert count == want.numel() and bits == 0 and torch.equal(idx, want) and torch.equal(val, t[want])


@pytest.mark.parametrize("n", [1, 65536, 65537, 1000003])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_count_the_host_is_told_by_the_selection(zen, n, dtype):
    """In one workgroup and in stretches, with room for all and for some; the workspace is used again at once, by the
    same stream and by another one."""
    from zen_repro_amd import comm

    gen = torch.Generator(device="cuda").manual_seed(n)
    a, b = ((torch.randn(n, generator=gen, device="cuda") *
             (torch.rand(n, generator=gen, device="cuda") < 0.3)).to(dtype) for _ in range(2))
    want = [torch.nonzero(t).view(-1) for t in (a, b)]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    for capacity in (n, max(1, want[0].numel() // 2)):
        out = [comm._select_raw(a, None, True, capacity), comm._select_raw(b, None, True, n)]
        with torch.cuda.stream(side):
            out.append(comm._select_raw(a, None, True, capacity))
        torch.cuda.synchronize()
        for (idx, val, count, bits), at, t, room in zip(out, (want[0], want[1], want[0]), (a, b, a), (capacity, n, capacity)):
            assert count == at.numel() and bits == (zen._lib.STAT_CAPACITY if count > room else 0)
            assert torch.equal(idx, at[:room]) and torch.equal(val, t[at[:room]])
