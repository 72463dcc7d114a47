"""Parity of the bucket-slab fast paths (large inputs) against the CPU oracle:
load balance with many collisions (levels 2 and 3, serial entries, declined
calls that fall back to the general mode), merge with heavy duplication, bad
indices and 64-bit indices, and calls in flight on two streams with their own
slots.  Every test first checks through zen_*_path that the sizes really take
the slab path.  Bar: bit-exact, as in test_gpu_parity.py."""
import numpy as np
import pytest
import torch

from gpu_util import make_grad, to_dev, to_np

pytestmark = pytest.mark.gpu

SLAB = 2
WIDE = 3
FLAGS = 0  # OR-ed into the fast mode of every merge and its path query in this module (set per run, below)
BALANCE_FLAGS = 0  # the same for the load balances


@pytest.fixture(scope="module", autouse=True, params=["wide", "slabs"])
def fast_path(request):
    """Every test of this module runs twice: on the wide buckets (MODE_WIDE takes load balances there wherever they
    fit) and with MODE_SLABS, which keeps the calls on the bucket slabs."""
    global FLAGS, BALANCE_FLAGS
    import zen_repro_amd
    from zen_repro_amd import _lib

    FLAGS = _lib.MODE_SLABS if request.param == "slabs" else 0
    BALANCE_FLAGS = FLAGS or _lib.MODE_WIDE
    zen_repro_amd.TensorPartition.fast_flags = BALANCE_FLAGS
    zen_repro_amd.LoadBalanceAllreduce.fast_flags = FLAGS
    yield request.param
    FLAGS = BALANCE_FLAGS = 0
    zen_repro_amd.TensorPartition.fast_flags = 0
    zen_repro_amd.LoadBalanceAllreduce.fast_flags = 0


def on_fast_path(code):
    """Whether a zen_*_path answer is the path this run is about."""
    return code == (SLAB if FLAGS else WIDE)


def balance_mode(k):
    """The mode of a load_balance_flat call of this run on whose slot no sample waits."""
    from zen_repro_amd import _lib

    return _lib.MODE_FAST | BALANCE_FLAGS | (0 if k else _lib.MODE_NO_SAMPLES)


@pytest.fixture(scope="module")
def zen():
    import zen_repro_amd
    from zen_repro_amd import _lib

    _lib.lib()
    assert torch.cuda.is_available()
    return zen_repro_amd


def lb_path(zen, n, P, dtype, capacity, k=0, mode=0, scale=1):
    from zen_repro_amd import _lib

    m = int(n * scale // P * P)
    return _lib.lib().zen_load_balance_path(n, m, 1 if dtype == "bf16" else 0, capacity, P, k, mode | balance_mode(k))


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("n,P,density,rehash", [
    ((1 << 23), 16, 0.15, 3),        # 15 % of the slots taken: thousands of level-2/3 moves per partition
    ((1 << 23), 16, 0.15, 2),        # two levels: serial entries in every partition
    ((1 << 23) + 4096, 8, 0.05, 3),  # table size not a power of two
    ((1 << 24), 64, 0.01, 3),
    (6000000, 3, 0.02, 3),           # partitions not a power of two, odd bucket widths
])
def test_slab_load_balance_bit_exact(zen, oracle, n, P, density, rehash, dtype):
    from zen_repro_amd import _lib

    n = n // P * P
    g = make_grad(oracle, n, density, dtype, seed=n ^ (P * 131) ^ rehash)
    g[0] = 0x3F80 if dtype == "bf16" else 1.0  # index 0 holds a value and is never transmitted
    idx_o, val_o, splits_o, st_o = oracle.load_balance(g, P, 1, rehash)
    assert st_o == 0
    capacity = int(len(idx_o) * 1.1) + 1024
    assert on_fast_path(lb_path(zen, n, P, dtype, capacity))
    tp = zen.TensorPartition(P, 1, rehash)
    d = to_dev(g)
    for rep in range(2):  # the second call finds the borrowed table zero again
        oi, ov, splits, status = tp.load_balance_flat(d, capacity=capacity, mode=_lib.MODE_FAST)
        assert status.item() == 0
        assert np.array_equal(to_np(splits), splits_o)
        total = int(splits_o.sum())
        assert np.array_equal(to_np(oi)[:total], idx_o)
        assert np.array_equal(to_np(ov)[:total], val_o)
    m, _ = oracle.table_sizes(n, P, 1)
    assert not tp._table(d.device, m).any()


def slab_buckets(m, P, capacity):
    """Buckets of a partition (slab_geometry): 3584 entries each, or fuller ones where that saves a round of 512."""
    bpp = min(-(-capacity // (3584 * P)), 4096 // P)
    fewer = (-(-bpp * P // 512) - 1) * 512 // P
    return fewer if fewer and capacity // (fewer * P) <= 4608 else bpp


def slab_settles(m, P, capacity):
    """Whether the losers of level 1 are settled group by group (plan_slab)."""
    losers = 0.5 * capacity ** 2 / m * (1.4 if m % 4 == 0 and m & (m - 1) else 1)
    return losers > min(max((190 if P > 256 else 250) * slab_buckets(m, P, capacity) * P, 50000), 400000)


@pytest.mark.parametrize("P,log2,density,room,rehash,settled", [
    (16, 24, 0.25, 1.0, 3, True),
    (128, 24, 0.27, 1.02, 2, True),   # nearly as full as buckets may be
    (32, 24, 0.278, 1.0, 3, True),    # 943 of a part's 1024 cells taken, 1065 if losers with a smaller owner took one ...
    (32, 24, 0.2812, 1.0, 3, True),   # ... 966 and 1091
    (1, 26, 0.08, 1.35, 3, True),     # one partition of all groups
    (7, 24, 0.22, 1.05, 3, True),     # the last group of a partition has fewer buckets
    (300, 24, 0.22, 1.05, 3, True),   # more than 256 partitions: groups of one bucket ...
    (1000, 24, 0.24, 1.02, 2, True),
    (300, 25, 0.155, 1.05, 3, True),  # ... of two, the last of a partition of one
    (650, 25, 0.185, 1.0, 3, True),   # ... of three
    (16, 22, 0.127, 1.0, 3, False),   # fewer than 50 000 losers
    (16, 22, 0.135, 1.0, 3, True),
    (16, 24, 0.1, 1.0, 3, False),     # fewer than 250 to a bucket
    (16, 24, 0.105, 1.0, 3, True),
    (16, 24, 0.11, 2.0, 3, True),     # a capacity twice what is selected
    (257, 24, 0.13, 1.0, 3, False),   # fewer than 190 to a bucket
    (257, 24, 0.136, 1.0, 3, True),
])
@pytest.mark.parametrize("fast_path", ["slabs"], indirect=True)
def test_slab_load_balance_of_settled_losers(zen, oracle, P, log2, density, room, rehash, settled):
    from zen_repro_amd import _lib

    n = ((1 << log2) + 160) // P * P
    g = make_grad(oracle, n, density, "bf16", seed=P + rehash)
    idx_o, val_o, splits_o, st_o = oracle.load_balance(g, P, 1, rehash)
    capacity = int(len(idx_o) * room)
    assert st_o == 0 and lb_path(zen, n, P, "bf16", capacity) == SLAB
    assert slab_settles(n, P, capacity) == settled
    tp = zen.TensorPartition(P, 1, rehash)
    d = to_dev(g)
    for rep in range(2):  # the second call finds the counters and the map zero again
        oi, ov, splits, status = tp.load_balance_flat(d, capacity=capacity, mode=_lib.MODE_FAST)
        assert status.item() == 0
        assert np.array_equal(to_np(splits), splits_o)
        assert np.array_equal(to_np(oi)[:len(idx_o)], idx_o)
        assert np.array_equal(to_np(ov)[:len(idx_o)], val_o)
    m, _ = oracle.table_sizes(n, P, 1)
    assert not tp._table(d.device, m).any()


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("rehash", [2, 3])
@pytest.mark.parametrize("fast_path", ["slabs"], indirect=True)
def test_slab_load_balance_of_losers_in_one_place(zen, oracle, rehash, dtype):
    """More losers than a group's list takes (the rest go their way from their buckets' own lists, beside what the group has
    left over), and a bucket with more losers than its workgroup has threads."""
    from zen_repro_amd import _lib
    from zen_repro_amd.workloads import hash_slot

    n, P, capacity = (1 << 24) + 160, 16, 3500000
    npp, bpp, per_group = n // P, 62, 4  # 3584 entries to a bucket; groups of at least four buckets, 256 of them
    listed = int(1.25 * 0.7 * capacity * (capacity / n) / (P * 16)) + 512

    def bucket(slot):  # of the partition
        return slot % npp * ((bpp << 32) // npp) >> 32

    t = torch.arange(1, n, device="cuda")
    first = hash_slot(t, n)
    second = (hash_slot(t, 1 << 32) - 10001861 + 100703) % (1 << 32) % npp
    order = torch.argsort(first, stable=True)  # by slot, then index: whoever is not the first of its slot loses it
    twin = torch.zeros(n - 1, dtype=torch.bool, device="cuda")
    twin[order[1:]] = first[order[1:]] == first[order[:-1]]
    mate = torch.zeros(n - 1, dtype=torch.int64, device="cuda")  # ... to the index in front of it
    mate[order[1:]] = order[:-1]
    to_group = twin & (first // npp == 5) & (bucket(second) // per_group == 3)
    in_bucket = twin & (first // npp == 9) & (bucket(first) == 17)
    chosen = torch.cat([torch.nonzero(to_group).view(-1)[:listed + 400], torch.nonzero(in_bucket).view(-1)[:1300]])
    assert chosen.numel() == listed + 1700
    g = make_grad(oracle, n, 0.03, dtype, seed=rehash)
    at = torch.cat([chosen, mate[chosen]]).cpu().numpy() + 1
    g[at] = 0x3F80 if dtype == "bf16" else 1.0
    idx_o, val_o, splits_o, st_o = oracle.load_balance(g, P, 1, rehash)
    assert st_o == 0 and len(idx_o) < capacity and lb_path(zen, n, P, dtype, capacity) == SLAB
    assert slab_settles(n, P, capacity)
    tp = zen.TensorPartition(P, 1, rehash)
    d = to_dev(g)
    for rep in range(2):  # the second call finds the counters and the map zero again
        oi, ov, splits, status = tp.load_balance_flat(d, capacity=capacity, mode=_lib.MODE_FAST)
        assert status.item() == 0
        assert np.array_equal(to_np(splits), splits_o)
        assert np.array_equal(to_np(oi)[:len(idx_o)], idx_o)
        assert np.array_equal(to_np(ov)[:len(idx_o)], val_o)
    assert not tp._table(d.device, n).any()


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("P,density,room,losers,settled", [
    # losers that are settled group by group, and that each go their way
    (16, 0.2, 1.05, 451039, True),
    (3, 0.16, 1.1, 202997, True),
    (16, 0.1, 2.0, 119306, True),
    (16, 0.1, 1.1, 119306, True),
    (3, 0.125, 1.0, 125090, True),  # just past the line
    (3, 0.12, 1.0, 115574, False),  # just below it
])
@pytest.mark.parametrize("fast_path", ["slabs"], indirect=True)
def test_slab_load_balance_of_many_losers(zen, oracle, P, density, room, losers, settled, dtype):
    from zen_repro_amd import _lib
    from zen_repro_amd.workloads import hash_slot

    n = ((1 << 24) + 160) // P * P  # (no power of two, where the hash has fewer collisions)
    g = make_grad(oracle, n, density, dtype, seed=P)
    idx_o, val_o, splits_o, st_o = oracle.load_balance(g, P, 1, 3)
    capacity = int(len(idx_o) * room)
    assert st_o == 0 and lb_path(zen, n, P, dtype, capacity) == SLAB
    assert len(idx_o) - torch.unique(hash_slot(torch.from_numpy(idx_o.astype(np.int64)), n)).numel() == losers
    assert slab_settles(n, P, capacity) == settled
    tp = zen.TensorPartition(P, 1, 3)
    d = to_dev(g)
    for rep in range(2):  # the second call finds the counters zero again
        oi, ov, splits, status = tp.load_balance_flat(d, capacity=capacity, mode=_lib.MODE_FAST)
        assert status.item() == 0
        assert np.array_equal(to_np(splits), splits_o)
        assert np.array_equal(to_np(oi)[:len(idx_o)], idx_o)
        assert np.array_equal(to_np(ov)[:len(idx_o)], val_o)
    indices, values, splits = tp.load_balance(d, capacity=capacity)  # the host is told by the last of these launches
    assert np.array_equal(to_np(splits), splits_o)
    assert np.array_equal(to_np(torch.cat(indices)), idx_o)
    assert np.array_equal(to_np(torch.cat(values)), val_o)


@pytest.mark.parametrize("n,P,density,rehash,room", [
    ((6 << 20) - 3, 3, 0.05, 3, 1.1),   # the largest owner tables, a tenth selected and little
    ((10 << 20) - 6, 16, 0.001, 3, 1.1),
    ((6 << 20) + 2, 2, 0.1, 3, 1.1),    # just beyond them: the slabs
    ((10 << 20) + 16, 16, 0.001, 3, 1.1),
    ((6 << 20) + 5, 2, 0.3, 2, 1.1),    # too dense for the slabs' buckets
    (7000000, 3, 0.1, 2, 0.5),          # room for half: declined, and taken again with more
])
@pytest.mark.parametrize("dtype", ["bf16", "f32"])
def test_call_that_waits_gives_the_same_on_every_path(zen, oracle, n, P, density, rehash, room, dtype, monkeypatch):
    """load_balance waits for its sizes, which takes it off the wide buckets where the slabs fit (and nothing asks for
    them)."""
    monkeypatch.setattr(zen.TensorPartition, "fast_flags", FLAGS)
    g = make_grad(oracle, n, density, dtype, seed=n + P)
    idx_o, val_o, splits_o, st_o = oracle.load_balance(g, P, 1, rehash)
    assert st_o == 0
    tp = zen.TensorPartition(P, 1, rehash)
    indices, values, splits = tp.load_balance(to_dev(g), capacity=int(len(idx_o) * room) + 1024, grow=True)
    assert np.array_equal(to_np(splits), splits_o)
    assert [len(i) for i in indices] == list(splits_o)
    assert np.array_equal(to_np(torch.cat(indices)), idx_o) and np.array_equal(to_np(torch.cat(values)), val_o)
    assert not tp._table(torch.device("cuda"), oracle.table_sizes(n, P, 1)[0]).any()


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("P,per_part", [(4, 800), (4, 960), (4, 1000), (2, 1024), (16, 1024)])
@pytest.mark.parametrize("fast_path", ["wide"], indirect=True)  # (the slabs have neither)
def test_slab_load_balance_at_a_round_of_records(zen, oracle, P, per_part, dtype):
    """Wide buckets whose slabs' parts hold fewer records than the workgroup has threads, more, or some of each: it keeps
    them in registers in the first case and loads them round by round in the others.  Hundreds lose their slot."""
    n = 1 << 20
    k = per_part * 8 * 16
    x = (np.random.default_rng(P * per_part).standard_normal(n) * 1e-3).astype(np.float32)
    x[0] = 0
    g = x if dtype == "f32" else (x.view(np.uint32) >> 16).astype(np.uint16)
    masked, kept = oracle.mask_dense(g, int(oracle.kth_key(g, k)))
    idx_o, val_o, splits_o, st_o = oracle.load_balance(masked, P, 1, 3)
    capacity = kept + 1024
    assert st_o == 0 and lb_path(zen, n, P, dtype, capacity, k=k) == WIDE
    tp = zen.TensorPartition(P, 1, 3)
    oi, ov, splits, status = tp.load_balance_flat(to_dev(g), capacity=capacity, k=k)
    assert status.item() == 0 and np.array_equal(to_np(splits), splits_o)
    assert np.array_equal(to_np(oi)[:kept], idx_o) and np.array_equal(to_np(ov)[:kept], val_o)
    assert not tp._table(torch.device("cuda"), n).any()


@pytest.mark.parametrize("rehash", [1, 2, 3])
@pytest.mark.parametrize("P,k", [(4, 400), (4, 30000), (4, 45000), (4, 46300), (4, 48000), (1, 23000), (16, 92000), (3, 60000)])
@pytest.mark.parametrize("fast_path", ["wide"], indirect=True)  # (the slabs have neither)
def test_slab_load_balance_of_few_losers(zen, oracle, P, k, rehash):
    """Partitions with fewer and more entries that lose their first slot than their workgroups work out by themselves."""
    n = -(-(1 << 20) // P) * P
    x = (np.random.default_rng(P * k).standard_normal(n) * 1e-3).astype(np.float32)
    x[0] = 0
    masked, kept = oracle.mask_dense(x, int(oracle.kth_key(x, k)))
    idx_o, val_o, splits_o, st_o = oracle.load_balance(masked, P, 1, rehash)
    assert st_o == 0 and lb_path(zen, n, P, "f32", kept + 1024, k=k) == WIDE
    tp = zen.TensorPartition(P, 1, rehash)
    for _ in range(2):
        oi, ov, splits, status = tp.load_balance_flat(to_dev(x), capacity=kept + 1024, k=k)
        assert status.item() == 0 and np.array_equal(to_np(splits), splits_o)
        assert np.array_equal(to_np(oi)[:kept], idx_o) and np.array_equal(to_np(ov)[:kept], val_o)
    assert not tp._table(torch.device("cuda"), n).any()


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
def test_slab_load_balance_odd_length_unaligned_and_empty(zen, oracle, dtype):
    """A tensor whose length is no multiple of anything and whose first element is not 16-byte aligned (the
    streaming kernel's element-wise loads and its ragged last tile), and a tensor of zeros."""
    from zen_repro_amd import _lib

    n, P = (1 << 23) + 1237, 16
    g = make_grad(oracle, n, 0.03, dtype, seed=4242)
    g[-1] = 0x3F80 if dtype == "bf16" else 1.0  # the very last element is selected
    idx_o, val_o, splits_o, st_o = oracle.load_balance(g, P, 1, 3)
    assert st_o == 0
    capacity = len(idx_o) + 2048
    assert on_fast_path(lb_path(zen, n, P, dtype, capacity))
    buf = to_dev(np.concatenate([g[:3], g]))
    d = buf[3:]
    assert d.data_ptr() % 16 != 0
    tp = zen.TensorPartition(P, 1, 3)
    oi, ov, splits, status = tp.load_balance_flat(d, capacity=capacity)
    total = int(splits_o.sum())
    assert status.item() == 0 and np.array_equal(to_np(splits), splits_o)
    assert np.array_equal(to_np(oi)[:total], idx_o) and np.array_equal(to_np(ov)[:total], val_o)
    # the same tensor 16-byte aligned: whole vectors stream, the few elements behind the last one (the
    # selected last element among them) go through a stage of their own
    a = to_dev(g)
    assert a.data_ptr() % 16 == 0 and n % 8 != 0
    oi, ov, splits, status = tp.load_balance_flat(a, capacity=capacity)
    assert status.item() == 0 and np.array_equal(to_np(splits), splits_o)
    assert np.array_equal(to_np(oi)[:total], idx_o) and np.array_equal(to_np(ov)[:total], val_o)
    zeros = torch.zeros(n, dtype=d.dtype, device="cuda")
    oi, ov, splits, status = tp.load_balance_flat(zeros, capacity=capacity)
    assert status.item() == 0 and int(splits.sum()) == 0


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("P,scale,rehash", [
    (8, 21, 3),       # buckets of 131 075 slots: just past the narrowest width the bucket kernels come in
    (64, 100, 2),     # the second width
    (3000, 5000, 3),  # 333 333 slots: as many buckets as there may be, and wider than two workgroups to a unit allow
    (1, 33, 3),       # 366 667 as the records call for: more buckets, so that their bitmaps fit
    (1, 60, 2),       # 666 667, and too few records for more buckets: by comparisons, like the case before the last
    (4, 60, 1),       # the same with one level: whoever loses it goes to the serial lists
    (2500, 7400, 3),  # 592 000
    (2049, 10800, 2),  # 1 047 600: the widest there is
])
def test_slab_load_balance_at_every_bucket_width(zen, oracle, P, scale, rehash, dtype):
    from zen_repro_amd import _lib

    n = 200000 // P * P
    g = make_grad(oracle, n, 0.3, dtype, seed=P + scale)
    idx_o, val_o, splits_o, st_o = oracle.load_balance(g, P, scale, rehash)
    capacity = len(idx_o) + 1024
    if not FLAGS and lb_path(zen, n, P, dtype, capacity, scale=scale) != WIDE:
        pytest.skip("covered by the other run")
    assert st_o == 0 and on_fast_path(lb_path(zen, n, P, dtype, capacity, scale=scale))
    tp = zen.TensorPartition(P, scale, rehash)
    oi, ov, splits, status = tp.load_balance_flat(to_dev(g), capacity=capacity, mode=_lib.MODE_FAST)
    assert status.item() == 0
    assert np.array_equal(to_np(splits), splits_o)
    assert np.array_equal(to_np(oi)[:len(idx_o)], idx_o)
    assert np.array_equal(to_np(ov)[:len(idx_o)], val_o)


def test_slab_load_balance_declines_and_general_mode_takes_over(zen, oracle):
    """One rehash level at 15 % load sends every level-1 loser to the serial
    lists: far more than the slab path carries per partition.  It must say so
    (RETRY), and the reference-shaped call must come back with the right
    answer from the general mode."""
    from zen_repro_amd import _lib

    n, P = (1 << 23) + 16000, 16  # not a power of two: about 8000 level-1 losers per partition
    g = make_grad(oracle, n, 0.15, "bf16", seed=99)
    idx_o, val_o, splits_o, st_o = oracle.load_balance(g, P, 1, 1)
    assert st_o == 0
    capacity = int(len(idx_o) * 1.1) + 1024
    assert on_fast_path(lb_path(zen, n, P, "bf16", capacity))
    tp = zen.TensorPartition(P, 1, 1)
    d = to_dev(g)
    _, _, _, status = tp.load_balance_flat(d, capacity=capacity, mode=_lib.MODE_FAST)
    assert status.item() & _lib.STAT_RETRY
    tp._table(d.device, n).zero_()
    indices, values, splits = tp.load_balance(d, capacity=capacity)
    assert np.array_equal(to_np(splits), splits_o)
    assert np.array_equal(np.concatenate([to_np(i) for i in indices]), idx_o)
    assert np.array_equal(np.concatenate([to_np(v) for v in values]), val_o)


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("fast_path", ["wide"], indirect=True)  # (the slabs set nothing aside)
def test_wide_load_balance_declines_a_bucket_of_shared_slots(zen, oracle, dtype):
    """6300 records of one bucket share their slot with another: three times what a workgroup has room to set aside."""
    from zen_repro_amd import _lib
    from zen_repro_amd.workloads import hash_slot

    n, P, capacity = (1 << 20) + 64, 4, 130000
    t = torch.arange(1, n)
    t = t[hash_slot(t, n) < n // P // 32 - 200]
    slots = hash_slot(t, n)
    assert 6144 < torch.count_nonzero(torch.bincount(slots)[slots] > 1) < t.numel() < 8192
    g = np.zeros(n, dtype=np.uint16 if dtype == "bf16" else np.float32)
    g[t.numpy()] = 0x3F80 if dtype == "bf16" else 1.0
    idx_o, val_o, splits_o, st_o = oracle.load_balance(g, P, 1, 3)
    assert st_o == 0 and lb_path(zen, n, P, dtype, capacity) == WIDE
    tp = zen.TensorPartition(P, 1, 3)
    d = to_dev(g)
    for _ in range(2):
        _, _, _, status = tp.load_balance_flat(d, capacity=capacity, mode=_lib.MODE_FAST)
        assert status.item() & _lib.STAT_RETRY
        tp._table(d.device, n).zero_()
    indices, values, splits = tp.load_balance(d, capacity=capacity)
    assert np.array_equal(to_np(splits), splits_o)
    assert np.array_equal(to_np(torch.cat(indices)), idx_o) and np.array_equal(to_np(torch.cat(values)), val_o)


def test_slab_load_balance_too_many_candidates_declines(zen, oracle):
    """A capacity far below what is selected: the candidate list overflows, the
    call declines instead of writing out of bounds."""
    from zen_repro_amd import _lib

    n, P = 1 << 23, 8
    g = make_grad(oracle, n, 0.05, "f32", seed=5)
    capacity = 1 << 16  # about a sixth of the nonzeros
    assert on_fast_path(lb_path(zen, n, P, "f32", capacity))
    tp = zen.TensorPartition(P, 1, 3)
    _, _, _, status = tp.load_balance_flat(to_dev(g), capacity=capacity, mode=_lib.MODE_FAST)
    assert status.item() & (_lib.STAT_RETRY | _lib.STAT_CAPACITY)


def test_slab_load_balance_fused_topk_fp32(zen, oracle):
    """fp32 top-k inside the call on the slab path: the candidates' histogram resolves 15 key bits, the last
    16 come from a second histogram over the candidates of the threshold's bin.  The k-th value is shared
    by many elements (ties are kept), element 0 lies in the threshold's bin above the threshold (it counts
    towards k and is never transmitted), and the very last element holds the largest value."""
    n, P = (1 << 24) + 24, 16
    rng = np.random.default_rng(77)
    x = (rng.standard_normal(n) * 1e-3).astype(np.float32)
    k = n // 100
    key0 = int(oracle.kth_key(x, k))
    tie = np.array([key0], dtype=np.uint32).view(np.float32)[0]
    x[rng.integers(1, n - 1, 300)] = -tie                                    # 300 more elements at the k-th magnitude
    x[0] = np.array([key0 + 5], dtype=np.uint32).view(np.float32)[0]         # same bin of 65536 keys, above it
    x[-1] = 1.0
    key = int(oracle.kth_key(x, k))
    assert key >> 16 == key0 >> 16
    masked, kept = oracle.mask_dense(x, key)
    assert kept > k and masked[0] != 0
    idx_o, val_o, splits_o, st_o = oracle.load_balance(masked, P, 1, 3)
    assert st_o == 0 and 0 not in idx_o
    capacity = int(1.25 * k) + 4096
    assert on_fast_path(lb_path(zen, n, P, "f32", capacity, k=k))
    tp = zen.TensorPartition(P, 1, 3)
    d = to_dev(x)
    thr_out = torch.zeros(2, dtype=torch.int32, device="cuda")
    for rep in range(2):  # the second call finds its counters cleared again
        oi, ov, splits, status = tp.load_balance_flat(d, capacity=capacity, k=k, thr_out=thr_out)
        assert status.item() == 0
        assert to_np(thr_out).tolist() == [key, kept]
        assert np.array_equal(to_np(splits), splits_o)
        total = int(splits_o.sum())
        assert np.array_equal(to_np(oi)[:total], idx_o)
        assert np.array_equal(to_np(ov)[:total], val_o)


def test_fused_topk_fp32_wherever_the_kth_key_lies_in_its_bin(zen, oracle, fast_path):
    """The fp32 threshold's last 16 bits for a k-th key at the top, the bottom and the middle of the threshold's
    bin of 65536 keys, at even and odd keys and either side of multiples of 128 and 256 (the refinement's last
    workgroup finds the 256 keys that hold the rank, then the key among them)."""
    n, P = (1 << 20) if fast_path == "wide" else (1 << 24), 4
    rng = np.random.default_rng(5)
    x = (rng.standard_normal(n) * 0.2).astype(np.float32)
    base = 0x3F000000  # 0.5: the bin is [0.5, 0.50390625)
    keys = x.view(np.uint32) & 0x7FFFFFFF
    x[(keys >> 16) == (base >> 16)] = 0.3  # nobody else in that bin
    x[0] = 0.25
    lows = [65535, 65534, 65409, 65408, 65407, 65280, 65279, 32769, 32768, 32767, 257, 256, 255, 129, 128, 127, 1, 0]
    at = rng.choice(np.arange(1, n), 3 * len(lows), replace=False)
    sign = np.where(rng.random(len(at)) < 0.5, 0x80000000, 0).astype(np.uint32)
    x.view(np.uint32)[at] = (np.repeat(np.array(lows, np.uint32), 3) + np.uint32(base)) | sign  # three of each
    ordered = np.sort(x.view(np.uint32) & 0x7FFFFFFF)
    above = n - int(np.searchsorted(ordered, base + 65536, "left"))
    assert int(oracle.kth_key(x, above + 4)) == base + lows[1]
    capacity = int(1.5 * above) + 4096
    tp = zen.TensorPartition(P, 1, 3)
    d = to_dev(x)
    thr_out = torch.zeros(2, dtype=torch.int32, device="cuda")
    for j in range(1, 3 * len(lows) + 1):
        k = above + j
        key = base + lows[(j - 1) // 3]  # the k-th largest key: the ((j - 1) // 3)-th of the planted ones
        kept = n - int(np.searchsorted(ordered, key, "left"))
        assert on_fast_path(lb_path(zen, n, P, "f32", capacity, k=k))
        _, _, splits, status = tp.load_balance_flat(d, capacity=capacity, k=k, thr_out=thr_out)
        assert status.item() == 0, (j, status.item())
        assert to_np(thr_out).tolist() == [key, kept], j
        assert int(to_np(splits).sum()) == kept - int((x.view(np.uint32)[0] & 0x7FFFFFFF) >= key)  # index 0 is never handed on


def test_slab_load_balance_threshold_given(zen, oracle):
    """Selection by a threshold the caller computed (topk_threshold) instead of k."""
    from zen_repro_amd import _lib

    n, P = 1 << 24, 16
    rng = np.random.default_rng(8)
    g = oracle.f32_to_bf16_bits((rng.standard_normal(n) * 1e-3).astype(np.float32))
    k = n // 100
    key = oracle.kth_key(g, k)
    masked, kept = oracle.mask_dense(g, key)
    idx_o, val_o, splits_o, _ = oracle.load_balance(masked, P, 1, 3)
    d = to_dev(g)
    thr = zen.topk_threshold(d, k)
    capacity = kept + 4096
    assert on_fast_path(lb_path(zen, n, P, "bf16", capacity))
    tp = zen.TensorPartition(P, 1, 3)
    oi, ov, splits, status = tp.load_balance_flat(d, thr=thr, capacity=capacity)
    assert status.item() == 0 and np.array_equal(to_np(splits), splits_o)
    assert np.array_equal(to_np(oi)[:kept], idx_o) and np.array_equal(to_np(ov)[:kept], val_o)


def test_two_slots_in_flight_give_the_same_answer(zen, oracle):
    """Two encodes and two merges enqueued on four streams, each pair with its
    own slot (workspace and table): same bytes as one call alone."""
    n, P = 1 << 24, 16
    rng = np.random.default_rng(21)
    g = oracle.f32_to_bf16_bits((rng.standard_normal(n) * 1e-3).astype(np.float32))
    d = to_dev(g)
    k = n // 200
    capacity = int(1.3 * k) + 4096
    assert on_fast_path(lb_path(zen, n, P, "bf16", capacity, k=k))
    tp = zen.TensorPartition(P, 1, 3)
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(P), None, None)
    mi = to_dev(rng.integers(1, n, 400000).astype(np.int32))
    mv = to_dev((rng.standard_normal(400000) * 1e-3).astype(np.float32))
    ref = tp.load_balance_flat(d, capacity=capacity, k=k)
    ref_m = lba.merge_sparse_flat(mi, mv, n)
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(4)]
    outs = []
    for rep in range(3):
        for slot in range(2):
            with torch.cuda.stream(streams[slot]):
                outs.append(("e", tp.load_balance_flat(d, capacity=capacity, k=k, slot=slot)))
            with torch.cuda.stream(streams[2 + slot]):
                outs.append(("m", lba.merge_sparse_flat(mi, mv, n, slot=slot)))
    torch.cuda.synchronize()
    total = int(ref[2].sum())
    for kind, o in outs:
        if kind == "e":
            assert o[3].item() == 0 and torch.equal(o[2], ref[2])
            assert torch.equal(o[0][:total], ref[0][:total]) and torch.equal(o[1][:total], ref[1][:total])
        else:
            cnt = int(ref_m[2])
            assert o[3].item() == 0 and int(o[2]) == cnt
            assert torch.equal(o[0][:cnt], ref_m[0][:cnt]) and torch.equal(o[1][:cnt], ref_m[1][:cnt])


# ------------------------------------------------------------------ merge


def test_resident_launches_on_streams_that_take_turns(zen, oracle):
    """Calls on the default stream and on two others in every order, none waited for, each with a slot of its own."""
    n, P, k = 3 << 20, 8, 20000
    rng = np.random.default_rng(77)
    tp = zen.TensorPartition(P, 1, 3)
    streams = [torch.cuda.default_stream(), torch.cuda.Stream(), torch.cuda.Stream()]
    cases = []
    for slot in range(4):
        g = (rng.standard_normal(n) * 1e-3).astype(np.float32)
        masked, _ = oracle.mask_dense(g, oracle.kth_key(g, k))
        cases.append((to_dev(g), oracle.load_balance(masked, P, 1, 3)))
    torch.cuda.synchronize()
    got = []
    for call, which in enumerate([0, 0, 1, 1, 0, 2, 1, 0, 0, 2, 2, 0]):
        with torch.cuda.stream(streams[which]):
            got.append(tp.load_balance_flat(cases[call % 4][0], capacity=2 * k, k=k, slot=call))
    torch.cuda.synchronize()
    for call, (oi, ov, splits, status) in enumerate(got):
        idx_o, val_o, splits_o, _ = cases[call % 4][1]
        assert status.item() == 0 and np.array_equal(to_np(splits), splits_o)
        assert np.array_equal(to_np(oi)[:len(idx_o)], idx_o) and np.array_equal(to_np(ov)[:len(idx_o)], val_o)


def payloads(oracle, rng, n, peers, per_peer, overlap, dtype):
    pool = rng.choice(n, max(1, int(per_peer * overlap) * 2), replace=False)
    idx, val = [], []
    for _ in range(peers):
        shared = rng.choice(pool, int(per_peer * overlap), replace=False) if overlap > 0 else np.empty(0, np.int64)
        own = rng.integers(0, n, per_peer - len(shared))
        i = np.concatenate([shared, own])
        rng.shuffle(i)
        v = (rng.standard_normal(len(i)) * 1e-3).astype(np.float32)
        idx.append(i)
        val.append(oracle.f32_to_bf16_bits(v) if dtype == "bf16" else v)
    return np.concatenate(idx), np.concatenate(val)


@pytest.mark.parametrize("idx64", [False, True])
@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("n,peers,per_peer,overlap", [
    (1 << 24, 16, 20000, 0.3),
    (50000000, 64, 4000, 0.5),   # every shared index arrives 64 times
    (1 << 24, 16, 20000, 0.9),   # nine records in ten share their index with fifteen others: more than a
                                 # workgroup sets aside for ranking in a second round
    ((1 << 23) + 12345, 4, 30000, 0.0),
])
def test_slab_merge_bit_exact(zen, oracle, n, peers, per_peer, overlap, dtype, idx64):
    from zen_repro_amd import _lib

    rng = np.random.default_rng(n % 1000 + peers)
    ci, cv = payloads(oracle, rng, n, peers, per_peer, overlap, dtype)
    ci = ci.astype(np.int64 if idx64 else np.int32)
    assert on_fast_path(_lib.lib().zen_merge_path(len(ci), n, _lib.MODE_FAST | FLAGS))
    want_i, want_v = oracle.merge_sparse(ci, cv, n)
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(peers), None, None)
    gi, gv, cnt, st = lba.merge_sparse_flat(to_dev(ci), to_dev(cv), n, idx64=idx64, mode=_lib.MODE_FAST)
    assert st.item() == 0 and cnt.item() == len(want_i)
    assert np.array_equal(to_np(gi)[:len(want_i)], want_i.astype(np.int64 if idx64 else np.int32))
    # same adds in the same order as a sequential scatter_add_: bit-exact
    assert np.array_equal(to_np(gv)[:len(want_i)].view(np.uint32), want_v.view(np.uint32))
    # and the dense form of the same merge
    dense = lba.decode_sparse_tensors(to_dev(ci), to_dev(cv), n)
    f32 = oracle.decode(ci, cv, n, "f32acc")
    assert np.array_equal(to_np(dense), oracle.f32_to_bf16_bits(f32) if dtype == "bf16" else f32)


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("times", [2, 3, 4, 5, 6, 7, 8, 9, 11, 16, 17, 37])
def test_merge_of_groups_of_every_length(zen, oracle, times, dtype):
    """Every index comes `times` times, and one in three once: groups are ranked, and runs that began in front of a
    thread's records summed, four records at a time."""
    from zen_repro_amd import _lib

    n, r = (1 << 23) + 3, 200000
    rng = np.random.default_rng(times)
    ci = np.concatenate([np.tile(rng.integers(0, n, r * 2 // 3 // times), times), rng.integers(0, n, r // 3)])
    rng.shuffle(ci)
    cv = (rng.standard_normal(len(ci)) * 1e-3).astype(np.float32)
    if dtype == "bf16":
        cv = oracle.f32_to_bf16_bits(cv)
    assert on_fast_path(_lib.lib().zen_merge_path(len(ci), n, _lib.MODE_FAST | FLAGS))
    want_i, want_v = oracle.merge_sparse(ci, cv, n)
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(4), None, None)
    gi, gv, cnt, st = lba.merge_sparse_flat(to_dev(ci), to_dev(cv), n, mode=_lib.MODE_FAST)
    assert st.item() == 0 and cnt.item() == len(want_i)
    assert np.array_equal(to_np(gi)[:len(want_i)], want_i.astype(np.int32))
    assert np.array_equal(to_np(gv)[:len(want_i)].view(np.uint32), want_v.view(np.uint32))


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("piled", [3072, 3073, 4096, 4097, 5120, 5121, 6143, 6144])
def test_slab_merge_at_a_row_of_records(zen, oracle, piled, dtype):
    """The first of fourteen bucket slabs holds exactly `piled` records, a quarter of them on 64 indices, the others some
    2800: the merge is written out for every number of rows of 1024 records, up to the slab's room."""
    from zen_repro_amd import _lib

    n, r, width = 14 << 19, 43000, 1 << 19
    rng = np.random.default_rng(piled)
    ci = rng.integers(width + 64, n, r)
    first = rng.integers(0, width - 64, piled)
    few = rng.choice(piled, piled // 4, replace=False)
    first[few] = rng.choice(first, 64)[rng.integers(0, 64, len(few))]
    ci[rng.choice(r, piled, replace=False)] = first
    cv = (rng.standard_normal(r) * 1e-3).astype(np.float32)
    if dtype == "bf16":
        cv = oracle.f32_to_bf16_bits(cv)
    want_i, want_v = oracle.merge_sparse(ci, cv, n)
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(4), None, None)
    lba.fast_flags = _lib.MODE_SLABS
    assert _lib.lib().zen_merge_path(r, n, _lib.MODE_FAST | _lib.MODE_SLABS) == 2
    gi, gv, cnt, st = lba.merge_sparse_flat(to_dev(ci), to_dev(cv), n, mode=_lib.MODE_FAST)
    assert st.item() == 0 and cnt.item() == len(want_i)
    assert np.array_equal(to_np(gi)[:len(want_i)], want_i.astype(np.int32))
    assert np.array_equal(to_np(gv)[:len(want_i)].view(np.uint32), want_v.view(np.uint32))


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("piled", [5120, 5121, 9216, 9217, 13312, 13313, 16383, 16384])
def test_wide_merge_at_a_number_of_places(zen, oracle, piled, dtype):
    """The first of 128 wide buckets holds exactly `piled` records, a quarter of them on 64 indices: the sums are written out
    for 5, 9, 13 and 17 places a thread."""
    from zen_repro_amd import _lib

    n, r, width = 1 << 24, 128 * 8000, 1 << 17
    rng = np.random.default_rng(piled)
    ci = rng.integers(width + 64, n, r)
    first = rng.integers(0, width - 64, piled)
    few = rng.choice(piled, piled // 4, replace=False)
    first[few] = rng.choice(first, 64)[rng.integers(0, 64, len(few))]
    ci[rng.choice(r, piled, replace=False)] = first
    cv = (rng.standard_normal(r) * 1e-3).astype(np.float32)
    if dtype == "bf16":
        cv = oracle.f32_to_bf16_bits(cv)
    want_i, want_v = oracle.merge_sparse(ci, cv, n)
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(4), None, None)
    gi, gv, cnt, st = lba.merge_sparse_flat(to_dev(ci), to_dev(cv), n, mode=_lib.MODE_FAST)
    # (on the slabs alone a bucket of a third of them is too much)
    if not FLAGS:
        assert st.item() == 0 and cnt.item() == len(want_i)
        assert np.array_equal(to_np(gi)[:len(want_i)], want_i.astype(np.int32))
        assert np.array_equal(to_np(gv)[:len(want_i)].view(np.uint32), want_v.view(np.uint32))
    dense = lba.decode_sparse_tensors(to_dev(ci), to_dev(cv), n)
    f32 = oracle.decode(ci, cv, n, "f32acc")
    assert np.array_equal(to_np(dense), oracle.f32_to_bf16_bits(f32) if dtype == "bf16" else f32)


@pytest.mark.parametrize("r", [1 << 19, (1 << 19) + 1, 1900000, 128 * 15360 + 1])
def test_merge_that_waits_gives_the_same_on_half_and_all_of_the_chip(zen, oracle, r):
    """One list of r entries around the sizes where the number of wide buckets changes, against merge_sparse_flat."""
    n = 20000000
    gen = torch.Generator(device="cuda").manual_seed(r)
    idx = torch.randint(0, n, (r,), generator=gen, device="cuda")
    val = torch.randn(r, generator=gen, device="cuda").to(torch.bfloat16)
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(4), None, None)
    w_idx, w_val = oracle.merge_sparse(to_np(idx), to_np(val), n)
    dense = lba.decode_sparse_tensors(idx, val, n)
    f_idx, f_val, count, status = lba.merge_sparse_flat(idx, val, n)
    assert status.item() == 0 and count.item() == len(w_idx)
    assert np.array_equal(to_np(f_idx)[:len(w_idx)], w_idx)
    assert np.array_equal(to_np(f_val)[:len(w_idx)].view(np.uint32), w_val.view(np.uint32))
    rounded = torch.from_numpy(w_val).to(torch.bfloat16)
    kept = rounded != 0
    want = torch.zeros(n, dtype=torch.bfloat16)
    want[torch.from_numpy(w_idx.astype(np.int64))] = rounded
    assert torch.equal(dense.cpu(), want)
    m_idx, m_val = lba.merge_rounded(idx, val, n, torch.bfloat16)
    assert np.array_equal(to_np(m_idx), w_idx[kept.numpy()]) and torch.equal(m_val.cpu(), rounded[kept])


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("piled", [1000, 1024, 1025, 2047, 2049, 3072, 3200])
def test_merge_at_a_round_of_records(zen, oracle, piled, dtype):
    """The first of 128 wide buckets gets all its records from every eighth batch of 4096 entries, which is one part of its
    slab: up to one and two records a thread, more, and more than the workgroup takes."""
    from zen_repro_amd import _lib

    n, batches = 1 << 24, 336
    rng = np.random.default_rng(piled)
    ci = rng.integers(n // 128, n, batches * 4096)
    at = rng.choice(batches // 8 * 4096, piled, replace=False)
    ci[at // 4096 * 8 * 4096 + at % 4096] = rng.integers(0, n // 128, piled)
    cv = (rng.standard_normal(len(ci)) * 1e-3).astype(np.float32)
    if dtype == "bf16":
        cv = oracle.f32_to_bf16_bits(cv)
    want_i, want_v = oracle.merge_sparse(ci, cv, n)
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(4), None, None)
    gi, gv, cnt, st = lba.merge_sparse_flat(to_dev(ci), to_dev(cv), n, mode=_lib.MODE_FAST)
    if piled > 3072 and not FLAGS:
        assert st.item() == _lib.STAT_RETRY
    else:
        assert st.item() == 0 and cnt.item() == len(want_i)
        assert np.array_equal(to_np(gi)[:len(want_i)], want_i.astype(np.int32))
        assert np.array_equal(to_np(gv)[:len(want_i)].view(np.uint32), want_v.view(np.uint32))
    dense = lba.decode_sparse_tensors(to_dev(ci), to_dev(cv), n)
    f32 = oracle.decode(ci, cv, n, "f32acc")
    assert np.array_equal(to_np(dense), oracle.f32_to_bf16_bits(f32) if dtype == "bf16" else f32)


def test_slab_merge_bad_indices_cancellation_and_pile_up(zen, oracle):
    from zen_repro_amd import _lib

    n = 1 << 24
    rng = np.random.default_rng(17)
    idx = rng.integers(0, n, 200000).astype(np.int64)
    val = (rng.standard_normal(len(idx)) * 1e-3).astype(np.float32)
    idx[1000:1100] = idx[0:100]          # pairs that cancel exactly
    val[1000:1100] = -val[0:100]
    idx[5000] = -7                        # out of range on both sides
    idx[5001] = n
    assert on_fast_path(_lib.lib().zen_merge_path(len(idx), n, _lib.MODE_FAST | FLAGS))
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(4), None, None)
    gi, gv, cnt, st = lba.merge_sparse_flat(to_dev(idx), to_dev(val), n, idx64=True, mode=_lib.MODE_FAST)
    assert st.item() == _lib.STAT_BAD_INDEX
    good = (idx >= 0) & (idx < n)
    wi, wv = oracle.merge_sparse(idx[good], val[good], n)
    assert cnt.item() == len(wi)
    assert np.array_equal(to_np(gi)[:len(wi)], wi) and np.array_equal(to_np(gv)[:len(wi)].view(np.uint32), wv.view(np.uint32))
    # one index received 50000 times: the slab path declines, the general mode answers
    idx2 = np.concatenate([np.full(50000, 4242), rng.integers(0, n, 100000)]).astype(np.int32)
    val2 = (rng.standard_normal(len(idx2)) * 1e-3).astype(np.float32)
    _, _, _, st2 = lba.merge_sparse_flat(to_dev(idx2), to_dev(val2), n, mode=_lib.MODE_FAST)
    assert st2.item() & _lib.STAT_RETRY
    gi2, gv2 = lba.merge_sparse(to_dev(idx2), to_dev(val2), n)
    wi2, wv2 = oracle.merge_sparse(idx2, val2, n)
    assert np.array_equal(to_np(gi2), wi2) and np.array_equal(to_np(gv2).view(np.uint32), wv2.view(np.uint32))


# ------------------------------------------------ counters are left at zero

def test_table_and_merge_workspace_are_zero_again_after_every_call(zen, oracle):
    """The slab paths clear no counters up front: they rely on the table (encode) and the head of the merge
    workspace being zero, and put them back to zero themselves.  Calls of different sizes and selections in a
    row, on one table and one workspace, must each give the oracle's answer and leave both all zero."""
    from zen_repro_amd import _lib

    L = _lib.lib()
    P = 8
    n = 1 << 23
    tp = zen.TensorPartition(P, 1, 3)
    rng = np.random.default_rng(5)
    g = (rng.standard_normal(n) * 1e-3).astype(np.float32)
    cases = [("f32", 0.004, 0), ("bf16", 0.01, 0), ("f32", 1.0, n // 200), ("bf16", 1.0, n // 100), ("f32", 0.002, 0)]
    for dtype, density, k in cases:
        x = np.where(rng.random(n) < density, g, 0).astype(np.float32)
        x_np = oracle.f32_to_bf16_bits(x) if dtype == "bf16" else x
        grad = to_dev(x_np)
        if k:
            key = oracle.kth_key(x_np, k)
            masked, kept = oracle.mask_dense(x_np, key)
            cap = kept + 1024
        else:
            masked, cap = x_np, int(np.count_nonzero(x)) + 1024
        m, _ = tp.table_sizes(n)
        assert on_fast_path(L.zen_load_balance_path(n, m, _lib.dtype_code(grad), cap, P, k, balance_mode(k)))
        idx, val, splits, st = tp.load_balance_flat(grad, None, cap, k=k)
        idx_o, val_o, splits_o, st_o = oracle.load_balance(masked, P, 1, 3)
        assert int(st.item()) == 0 and st_o == 0
        total = int(splits.sum())
        assert np.array_equal(splits.cpu().numpy(), splits_o)
        assert np.array_equal(idx[:total].cpu().numpy(), idx_o)
        assert np.array_equal(to_np(val[:total]), val_o)
        assert int(tp._table(grad.device, m).count_nonzero()) == 0, (dtype, density, k)

    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(P), None, None)
    dense_n = 1 << 26
    for r in (400_000, 3_000_000, 70_000):
        idx = rng.integers(1, dense_n, r).astype(np.int32)
        idx[rng.integers(0, r, r // 3)] = idx[rng.integers(0, r, r // 3)]  # duplicates
        val = (rng.standard_normal(r) * 1e-3).astype(np.float32)
        assert on_fast_path(L.zen_merge_path(r, dense_n, _lib.MODE_FAST | FLAGS))
        m_idx, m_val, count, st = lba.merge_sparse_flat(to_dev(idx), to_dev(val), dense_n)
        assert int(st.item()) == 0
        mi_o, mv_o = oracle.merge_sparse(idx, val, dense_n)
        c = int(count.item())
        assert np.array_equal(m_idx[:c].cpu().numpy(), mi_o)
        assert np.array_equal(m_val[:c].cpu().numpy().view(np.uint32), mv_o.view(np.uint32))
        ws = _lib.scratch.get(m_idx.device, "merge/0", 256, zero=True)
        assert int(ws[:L.zen_merge_zero_bytes()].count_nonzero()) == 0, r


def test_load_balance_without_a_capacity_takes_the_slab_path(zen, oracle):
    """TensorPartition.load_balance(tensor) as the reference calls it (tensor_load_balance.py:43): the capacity
    it works out for itself keeps a bucket-sized, sparse tensor on the fast paths, and the result is the
    oracle's."""
    from zen_repro_amd import _lib

    L = _lib.lib()
    n, P = 1 << 26, 16  # a 128 MB bf16 bucket (run_all.sh:22)
    g_np = make_grad(oracle, n, 0.005, "bf16", seed=21)
    grad = to_dev(g_np)
    tp = zen.TensorPartition(P, 1, 3)
    cap = tp._honest_capacity(grad, None, 0)
    m, _ = tp.table_sizes(n)
    assert cap < n // 100
    assert on_fast_path(L.zen_load_balance_path(n, m, _lib.BF16, cap, P, 0, balance_mode(0)))
    assert L.zen_load_balance_workspace(n, m, _lib.BF16, cap, P) < 1 << 28
    indices, values, splits = tp.load_balance(grad)
    idx_o, val_o, splits_o, st_o = oracle.load_balance(g_np, P, 1, 3)
    assert st_o == 0
    assert np.array_equal(splits.cpu().numpy(), splits_o)
    assert np.array_equal(torch.cat(indices).cpu().numpy(), idx_o)
    assert np.array_equal(to_np(torch.cat(values)), val_o)
    # with a threshold: the count that came with it sizes the call
    thr = zen.topk_threshold(grad, 200_000)
    assert tp._honest_capacity(grad, thr, 0) == int(thr[1].item()) + 1024
    indices, values, splits = tp.load_balance(grad, thr=thr)
    masked, kept = oracle.mask_dense(g_np, int(thr[0].item()))
    idx_o, val_o, splits_o, st_o = oracle.load_balance(masked, P, 1, 3)
    assert int(splits.sum()) == kept and np.array_equal(torch.cat(indices).cpu().numpy(), idx_o)


def test_sample_taken_ahead_gives_the_same_result(zen, oracle):
    """TensorPartition.prepare takes a top-k call's sample on another stream before the call: same bytes out
    as without, over several calls in a row with the two sets of sampling memory in turn, also when a sample
    is taken for a call that never comes (it is dropped), and the table is all zero afterwards."""
    from zen_repro_amd import _lib

    n, P = 1 << 25, 16
    rng = np.random.default_rng(31)
    side = torch.cuda.Stream()
    tp = zen.TensorPartition(P, 1, 3)
    grads, wants = [], []
    for i in range(3):
        g_np = oracle.f32_to_bf16_bits((rng.standard_normal(n) * 1e-3).astype(np.float32))
        k = n // 200 + 1000 * i
        key = oracle.kth_key(g_np, k)
        masked, kept = oracle.mask_dense(g_np, key)
        grads.append((to_dev(g_np), k, int(k * 1.25) + 4096))
        wants.append(oracle.load_balance(masked, P, 1, 3))
    torch.cuda.synchronize()
    m, _ = tp.table_sizes(n)
    assert on_fast_path(_lib.lib().zen_load_balance_path(n, m, _lib.BF16, grads[0][2], P, grads[0][1], balance_mode(grads[0][1])))

    def check(out, want):
        idx, val, splits, st = out
        idx_o, val_o, splits_o, st_o = want
        assert int(st.item()) == 0 and st_o == 0
        total = int(splits.sum())
        assert np.array_equal(splits.cpu().numpy(), splits_o)
        assert np.array_equal(idx[:total].cpu().numpy(), idx_o) and np.array_equal(to_np(val[:total]), val_o)

    # call i's sample is taken while call i - 1 is still being enqueued / running
    with torch.cuda.stream(side):
        tp.prepare(*grads[0])
    outs = []
    for i in range(6):
        g, k, cap = grads[i % 3]
        outs.append(tp.load_balance_flat(g, None, cap, k=k))
        if i + 1 < 6:
            with torch.cuda.stream(side):
                tp.prepare(*grads[(i + 1) % 3])
    for i, out in enumerate(outs):
        check(out, wants[i % 3])
    # a sample whose call comes later: the calls in between (other buckets on the same slot) leave it alone and
    # sample for themselves, in the other set of sampling memory
    with torch.cuda.stream(side):
        tp.prepare(*grads[1])
    g, k, cap = grads[2]
    check(tp.load_balance_flat(g, None, cap, k=k), wants[2])
    check(tp.load_balance_flat(grads[0][0], None, grads[0][2], k=grads[0][1]), wants[0])
    state = tp._ahead_state(g.device, 0)
    assert len(state["pending"]) == 1
    check(tp.load_balance_flat(grads[1][0], None, grads[1][2], k=grads[1][1]), wants[1])
    assert not state["pending"]
    # both sets hold samples of calls still to come and a third bucket turns up: the older sample gives way
    with torch.cuda.stream(side):
        tp.prepare(*grads[1])
        tp.prepare(*grads[2])
    assert len(state["pending"]) == 2
    check(tp.load_balance_flat(grads[0][0], None, grads[0][2], k=grads[0][1]), wants[0])
    assert len(state["pending"]) == 1
    check(tp.load_balance_flat(grads[1][0], None, grads[1][2], k=grads[1][1]), wants[1])  # samples again
    check(tp.load_balance_flat(g, None, cap, k=k), wants[2])                                # picks its sample up
    assert not state["pending"]
    torch.cuda.synchronize()
    assert int(tp._table(g.device, m).count_nonzero()) == 0


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("n,P", [(1 << 20, 4), ((1 << 21) + 4096, 8), (1 << 22, 16)])
def test_calls_that_take_no_sample_leave_a_waiting_one_alone(zen, oracle, n, P, dtype):
    """Tables of 2^20 to 4 Mi slots hold the samples taken ahead and serve as owner tables for calls without a k: with
    such calls (nonzeros, a threshold, the general mode) between a sample and its call, all of them give the oracle's
    results, the sample is picked up (dropped in front of the general mode), and the table ends all zero."""
    from zen_repro_amd import _lib

    rng = np.random.default_rng(57)
    sparse = make_grad(oracle, n, 0.01, dtype, seed=58)
    full = make_grad(oracle, n, 1.0, dtype, seed=59)
    k = n // 200
    cap, room = k + k // 4 + 4096, n // 64 + 4096
    key = oracle.kth_key(full, k)
    top = oracle.load_balance(oracle.mask_dense(full, key)[0], P, 1, 3)
    nonzeros = oracle.load_balance(sparse, P, 1, 3)
    a, b = to_dev(sparse), to_dev(full)
    thr = zen.topk_threshold(b, k)
    side = torch.cuda.Stream()
    tp = zen.TensorPartition(P, 1, 3)
    torch.cuda.synchronize()

    def check(out, want):
        idx, val, splits, st = out
        assert int(st.item()) == 0 and want[3] == 0
        total = int(splits.sum())
        assert np.array_equal(splits.cpu().numpy(), want[2])
        assert np.array_equal(idx[:total].cpu().numpy(), want[0]) and np.array_equal(to_np(val[:total]), want[1])

    calls = [lambda: (tp.load_balance_flat(a, None, room), nonzeros),
             lambda: (tp.load_balance_flat(b, thr, room), top),
             lambda: (tp.load_balance_flat(a, None, room, mode=_lib.MODE_GENERAL), nonzeros)]
    for i in rng.permutation(np.repeat(np.arange(3), 2)):
        with torch.cuda.stream(side):  # beside the call before, whose table it writes to
            tp.prepare(b, k, cap)
        state = tp._ahead_state(b.device, 0) if FLAGS == 0 else None
        assert state is None or len(state["pending"]) == 1
        out, want = calls[i]()
        assert state is None or len(state["pending"]) == (i < 2)
        top_out = tp.load_balance_flat(b, None, cap, k=k)
        assert state is None or not state["pending"]
        after = calls[i]()  # no sample waits now
        check(out, want)
        check(top_out, top)
        check(*after)
    torch.cuda.synchronize()
    assert int(tp._table(b.device, tp.table_sizes(n)[0]).count_nonzero()) == 0


def test_a_table_made_on_another_stream_is_waited_for(zen, oracle):
    """The first prepare of a size makes the table on its own stream, behind whatever that one is busy with; calls of
    other buckets on the current stream, which have no sample to wait for, find it filled all the same."""
    n, P = 1 << 22, 16
    a_np = make_grad(oracle, n, 0.01, "bf16", seed=65)
    b_np = make_grad(oracle, n, 1.0, "bf16", seed=66)
    k = n // 200
    cap, room = k + k // 4 + 4096, n // 64 + 4096
    top = oracle.load_balance(oracle.mask_dense(b_np, oracle.kth_key(b_np, k))[0], P, 1, 3)
    nonzeros = oracle.load_balance(a_np, P, 1, 3)
    a, b, c = to_dev(a_np), to_dev(b_np), to_dev(b_np)
    busy = torch.ones(2048, 2048, device="cuda")
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    tp = zen.TensorPartition(P, 1, 3)
    with torch.cuda.stream(side):
        for _ in range(20):
            busy = busy @ busy * 1e-4
        tp.prepare(b, k, cap)
    outs = [(tp.load_balance_flat(a, None, room), nonzeros), (tp.load_balance_flat(c, None, cap, k=k), top),
            (tp.load_balance_flat(b, None, cap, k=k), top)]
    for (idx, val, splits, st), (idx_o, val_o, splits_o, st_o) in outs:
        assert int(st.item()) == 0 and st_o == 0
        total = int(splits.sum())
        assert np.array_equal(splits.cpu().numpy(), splits_o)
        assert np.array_equal(idx[:total].cpu().numpy(), idx_o) and np.array_equal(to_np(val[:total]), val_o)


def test_merge_on_a_stream_that_runs_ahead(zen, oracle):
    """With the merge on a stream of its own and the current stream busy with something long, the merge comes before
    everything that the current stream still has to do: its count, status and workspace have to be zero by then, on
    the first call, whose blocks and workspaces are new, and on later ones with larger workspaces and new blocks."""
    from zen_repro_amd import _lib

    n, P = 1 << 22, 16
    a_np = make_grad(oracle, n, 0.01, "bf16", seed=67)
    cap = n // 64 + 4096
    want_e = oracle.load_balance(a_np, P, 1, 3)
    rng = np.random.default_rng(68)
    a = to_dev(a_np)
    busy = torch.ones(2048, 2048, device="cuda")
    side = torch.cuda.Stream()
    tp = zen.TensorPartition(P, 1, 3)
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(P), None, None)
    for per_peer in (3000, 9000, 9000):
        ci, cv = payloads(oracle, rng, n, P, per_peer, 0.25, "bf16")
        ci = ci.astype(np.int32)
        di, dv = to_dev(ci), to_dev(cv)
        want_i, want_v = oracle.merge_sparse(ci, cv, n)
        torch.cuda.synchronize()
        _lib.zeros.fresh(a.device)
        with torch.cuda.stream(side):
            _lib.zeros.fresh(a.device)
        for _ in range(20):
            busy = busy @ busy * 1e-4
        (idx, val, splits, st), (m_idx, m_val, count, m_st) = lba.encode_merge_flat(tp, a, cap, 0, di, dv, n,
                                                                                   merge_stream=side)
        torch.cuda.current_stream().wait_stream(side)
        assert int(st.item()) == 0 and int(m_st.item()) == 0 and int(count) == len(want_i)
        assert np.array_equal(to_np(m_idx)[:len(want_i)], want_i.astype(np.int32))
        assert np.array_equal(to_np(m_val)[:len(want_i)].view(np.uint32), want_v.view(np.uint32))
        total = int(splits.sum())
        assert np.array_equal(to_np(splits), want_e[2]) and np.array_equal(to_np(idx)[:total], want_e[0])


def test_sizes_kept_by_shape_are_bounded(zen, monkeypatch):
    """Steps that receive another number of entries each time: what is kept by the shape of a step stays small."""
    n, P = 1 << 20, 4
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(P), None, None)
    monkeypatch.setattr(lba, "_MOST_SHAPES", 8)
    grad = torch.zeros(n, device="cuda")
    grad[5::100] = 1.0
    for r in range(1, 30):
        idx = torch.arange(1, r + 1, dtype=torch.int32, device="cuda")
        e, (_, _, count, status) = lba.encode_merge_flat(lba.tensor_partition, grad, n // 64, 0, idx, idx.float(), n)
        assert int(count) == r and not int(status) and int(e[2].sum()) == grad[5::100].numel()
        assert len(lba._step_sizes) <= 8


def test_step_replayed_from_a_captured_graph(zen, oracle):
    """An encode (fused top-k) and a merge captured into a HIP graph, the merge forked onto a second stream:
    every replay, with eager calls on the same workspaces and a synchronisation in between, leaves the bytes
    the eager call leaves (the calls record kernels only: nothing a replay would skip or do twice)."""
    from zen_repro_amd import _lib

    n, P = 1 << 25, 16
    rng = np.random.default_rng(41)
    g_np = oracle.f32_to_bf16_bits((rng.standard_normal(n) * 1e-3).astype(np.float32))
    k = n // 200
    cap = int(k * 1.25) + 4096
    key = oracle.kth_key(g_np, k)
    masked, _ = oracle.mask_dense(g_np, key)
    idx_o, val_o, splits_o, st_o = oracle.load_balance(masked, P, 1, 3)
    per_peer = k // P
    peers_i = [rng.choice(n - 1, per_peer, replace=False).astype(np.int32) + 1 for _ in range(P)]
    flat_i = np.concatenate(peers_i)
    flat_v = oracle.f32_to_bf16_bits((rng.standard_normal(flat_i.size) * 1e-3).astype(np.float32))
    want_i, want_v = oracle.merge_sparse(flat_i, flat_v, n)
    grad, fi, fv = to_dev(g_np), to_dev(flat_i), to_dev(flat_v)
    tp = zen.TensorPartition(P, 1, 3)
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(P), None, None)
    m, _ = tp.table_sizes(n)
    assert on_fast_path(_lib.lib().zen_load_balance_path(n, m, _lib.BF16, cap, P, k, balance_mode(k)))
    assert on_fast_path(_lib.lib().zen_merge_path(flat_i.size, n, _lib.MODE_FAST | FLAGS))

    def check(enc, mrg):
        idx, val, splits, st = enc
        m_idx, m_val, m_count, m_st = mrg
        assert int(st.item()) == 0 and int(m_st.item()) == 0
        total = int(splits.sum())
        assert np.array_equal(splits.cpu().numpy(), splits_o)
        assert np.array_equal(idx[:total].cpu().numpy(), idx_o) and np.array_equal(to_np(val[:total]), val_o)
        u = int(m_count.item())
        assert u == len(want_i) and np.array_equal(m_idx[:u].cpu().numpy(), want_i.astype(np.int32))
        assert np.array_equal(m_val[:u].cpu().numpy().view(np.uint32), want_v.view(np.uint32))

    def eager():
        return (tp.load_balance_flat(grad, None, cap, k=k),
                lba.merge_sparse_flat(fi, fv, n, capacity=flat_i.size))

    check(*eager())  # also makes the workspaces, outside the capture
    torch.cuda.synchronize()
    side, cap_stream = torch.cuda.Stream(), torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=cap_stream):
        cur = torch.cuda.current_stream()
        _lib.zeros.fresh(grad.device)
        side.wait_stream(cur)
        enc = tp.load_balance_flat(grad, None, cap, k=k)
        with torch.cuda.stream(side):
            _lib.zeros.fresh(grad.device)
            mrg = lba.merge_sparse_flat(fi, fv, n, capacity=flat_i.size)
        cur.wait_stream(side)
    _lib.zeros.fresh(grad.device)
    for s_ in (side, cap_stream):
        with torch.cuda.stream(s_):
            _lib.zeros.fresh(grad.device)
    for _ in range(3):
        enc[0].fill_(-1)
        mrg[0].fill_(-1)
        graph.replay()
        torch.cuda.synchronize()
        check(enc, mrg)
        check(*eager())  # the same tables and workspaces, between two replays
        torch.cuda.synchronize()
    assert int(tp._table(grad.device, m).count_nonzero()) == 0


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
def test_threshold_of_an_earlier_call_replaces_the_sample(zen, oracle, dtype):
    """load_balance_flat(..., k, near=thr_out of an earlier call): no sample kernel, same bytes out, on the
    same gradient and on gradients a few per cent larger and smaller; a key that is far off (the gradient
    halved or doubled) makes the call decline (STAT_RETRY) or still gives the exact answer, never a wrong one."""
    from zen_repro_amd import _lib

    n, P = 1 << 24, 16
    rng = np.random.default_rng(53)
    base = (rng.standard_normal(n) * 1e-3).astype(np.float32)
    k = n // 200
    cap = int(k * 1.25) + 4096
    tp = zen.TensorPartition(P, 1, 3)
    m, _ = tp.table_sizes(n)
    code = _lib.BF16 if dtype == "bf16" else _lib.F32
    assert on_fast_path(_lib.lib().zen_load_balance_path(n, m, code, cap, P, k, balance_mode(k)))

    def bits(x):
        return oracle.f32_to_bf16_bits(x) if dtype == "bf16" else x

    def want(g_np):
        key = oracle.kth_key(g_np, k)
        masked, _ = oracle.mask_dense(g_np, key)
        return key, oracle.load_balance(masked, P, 1, 3)

    g0 = bits(base)
    thr_out = torch.zeros(2, dtype=torch.int32, device="cuda")
    g0_dev = to_dev(g0)
    dev = g0_dev.device
    first = tp.load_balance_flat(g0_dev, None, cap, k=k, thr_out=thr_out)
    key0, w0 = want(g0)
    assert int(first[3].item()) == 0 and int(thr_out[0].item()) == key0
    near = thr_out.clone()
    exact = 0
    for scale in (1.0, 1.02, 0.98, 0.5, 2.0):
        g_np = bits((base * np.float32(scale)).astype(np.float32))
        key, (idx_o, val_o, splits_o, st_o) = want(g_np)
        thr_now = torch.zeros(2, dtype=torch.int32, device="cuda")
        idx, val, splits, st = tp.load_balance_flat(to_dev(g_np), None, cap, k=k, thr_out=thr_now, near=near)
        status = int(st.item())
        if status & (_lib.STAT_RETRY | _lib.STAT_INTERNAL):
            assert scale in (0.5, 2.0), f"declined at scale {scale}"
            tp._table(dev, m).zero_()  # a declined call leaves the table for its caller to clear
            continue
        assert status == 0 and st_o == 0
        total = int(splits.sum())
        assert int(thr_now[0].item()) == key
        assert np.array_equal(splits.cpu().numpy(), splits_o)
        assert np.array_equal(idx[:total].cpu().numpy(), idx_o) and np.array_equal(to_np(val[:total]), val_o)
        exact += 1
    assert exact >= 3
    torch.cuda.synchronize()
    assert int(tp._table(dev, m).count_nonzero()) == 0


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
def test_encode_and_merge_in_one_call(zen, oracle, dtype):
    """encode_merge_flat (zen_encode_merge) against the two calls it stands for, bit for bit: a top-k bucket and
    the entries received for it, twice in a row (the second call finds every counter where the first left it),
    then with a sample taken ahead, and with the merge on a stream of its own."""
    from zen_repro_amd import _lib

    n, P, k = 1 << 25, 16, (1 << 25) // 100
    g = make_grad(oracle, n, 1.0, dtype, seed=31)
    rng = np.random.default_rng(5)
    ci, cv = payloads(oracle, rng, n, P, 20000, 0.25, dtype)
    ci = ci.astype(np.int32)
    cap = int(k * 1.25) + 4096
    d, di, dv = to_dev(g), to_dev(ci), to_dev(cv)
    tp = zen.TensorPartition(P, 1, 3)
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(P), None, None)
    e0 = tp.load_balance_flat(d, None, cap, k=k, slot=1)
    m0 = lba.merge_sparse_flat(di, dv, n, slot=1)
    torch.cuda.synchronize()
    assert e0[3].item() == 0 and m0[3].item() == 0
    total, cnt = int(e0[2].sum()), int(m0[2])
    side = torch.cuda.Stream()

    def same(e, m):
        torch.cuda.synchronize()
        assert e[3].item() == 0 and m[3].item() == 0
        assert torch.equal(e[2], e0[2]) and int(m[2]) == cnt
        assert torch.equal(e[0][:total], e0[0][:total]) and torch.equal(to_dev(to_np(e[1][:total])), to_dev(to_np(e0[1][:total])))
        assert torch.equal(m[0][:cnt], m0[0][:cnt]) and torch.equal(m[1][:cnt].view(torch.int32), m0[1][:cnt].view(torch.int32))

    for rep in range(2):
        same(*lba.encode_merge_flat(tp, d, cap, k, di, dv, n))
    tp.prepare(d, k, cap)
    same(*lba.encode_merge_flat(tp, d, cap, k, di, dv, n))
    side.wait_stream(torch.cuda.current_stream())
    same(*lba.encode_merge_flat(tp, d, cap, k, di, dv, n, merge_stream=side))
    torch.cuda.current_stream().wait_stream(side)
    m, _ = oracle.table_sizes(n, P, 1)
    assert not tp._table(d.device, m).any()


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
def test_sample_taken_along_by_the_call_before(zen, oracle, dtype):
    """encode_merge_flat(..., next_tensor=): the pass over one bucket takes the next bucket's sample along.  Four
    different gradients in a row on one slot, the third of another size (with its own k, capacity and table),
    each call handed its successor; every result equals the oracle's (so the floor the call before left behind
    selected nothing wrong), and every call after the first picks its sample up (no sample kernel of its own is
    launched: counted)."""
    from zen_repro_amd import _lib

    n, P = 1 << 24, 16
    sizes = [n, n, n // 4 * 3, n]
    ks = [s // 200 for s in sizes]
    caps = [int(k * 1.25) + 4096 for k in ks]
    grads = [make_grad(oracle, s, 1.0, dtype, seed=41 + i) for i, s in enumerate(sizes)]
    rng = np.random.default_rng(9)
    ci, cv = payloads(oracle, rng, n, P, 9000, 0.25, dtype)
    ci = ci.astype(np.int32)
    ds = [to_dev(g) for g in grads]
    di, dv = to_dev(ci), to_dev(cv)
    tp = zen.TensorPartition(P, 1, 3)
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(P), None, None)
    for s_, k_, c_ in zip(sizes, ks, caps):
        m, _ = oracle.table_sizes(s_, P, 1)
        assert on_fast_path(_lib.lib().zen_load_balance_path(s_, m, _lib.dtype_code(ds[0]), c_, P, k_, balance_mode(k_)))
    want_m = oracle.merge_sparse(ci, cv, n)
    _lib.profile_enable(True)
    outs = []
    for i in range(4):
        more = i + 1 < 4
        outs.append(lba.encode_merge_flat(tp, ds[i], caps[i], ks[i], di, dv, n, next_tensor=ds[i + 1] if more else None,
                                          next_k=ks[i + 1] if more else None,
                                          next_capacity=caps[i + 1] if more else None))
    torch.cuda.synchronize()
    launched = _lib.profile_read()
    _lib.profile_enable(False)
    assert launched["k_sample_hist"][1] == 1 and launched["k_select_stage"][1] == 4  # only the first call sampled for itself
    state = tp._ahead_state(ds[0].device, 0)
    assert state is not None and not state["pending"]
    for i, (e, mg) in enumerate(outs):
        assert e[3].item() == 0 and mg[3].item() == 0
        key = oracle.kth_key(grads[i], ks[i])
        sel, _ = oracle.mask_dense(grads[i], key)
        idx_o, val_o, splits_o, st_o = oracle.load_balance(sel, P, 1, 3)
        total = int(splits_o.sum())
        assert st_o == 0 and np.array_equal(to_np(e[2]), splits_o)
        assert np.array_equal(to_np(e[0])[:total], idx_o) and np.array_equal(to_np(e[1])[:total], val_o)
        cnt = int(mg[2])
        assert cnt == len(want_m[0]) and np.array_equal(to_np(mg[0])[:cnt], want_m[0].astype(np.int32))
        assert np.array_equal(to_np(mg[1])[:cnt].view(np.uint32), want_m[1].view(np.uint32))
    for s_ in set(sizes):
        assert not tp._table(ds[0].device, oracle.table_sizes(s_, P, 1)[0]).any()
    # a successor whose sizes take no path that keeps a sample is refused by the library, and not offered by the wrapper
    small = ds[0][: 1 << 12]
    e, _ = lba.encode_merge_flat(tp, ds[0], caps[0], ks[0], di, dv, n, next_tensor=small, next_k=20, next_capacity=64)
    assert e[3].item() == 0 and not tp._ahead_state(ds[0].device, 0)["pending"]


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("n,P", [(1 << 20, 4), (1 << 22, 16)])
def test_calls_without_a_k_around_calls_that_sample(zen, oracle, n, P, dtype):
    """encode_merge_flat with k == 0 and a next tensor whose call has a k, and the other way round, on tables that
    serve as owner tables for the one and hold samples for the other: the oracle's results, every call in one go."""
    sparse = make_grad(oracle, n, 0.01, dtype, seed=61)
    full = make_grad(oracle, n, 1.0, dtype, seed=62)
    k = n // 200
    cap = n // 64 + 4096
    top = oracle.load_balance(oracle.mask_dense(full, oracle.kth_key(full, k))[0], P, 1, 3)
    nonzeros = oracle.load_balance(sparse, P, 1, 3)
    rng = np.random.default_rng(63)
    ci, cv = payloads(oracle, rng, n, P, 900, 0.25, dtype)
    ci = ci.astype(np.int32)
    want_m = oracle.merge_sparse(ci, cv, n)
    a, b, di, dv = to_dev(sparse), to_dev(full), to_dev(ci), to_dev(cv)
    tp = zen.TensorPartition(P, 1, 3)
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(P), None, None)
    steps = [(a, 0), (b, k), (a, 0), (a, 0), (b, k), (b, k), (a, 0), (b, k)]
    outs = []
    for (t, kk), nxt in zip(steps, steps[1:] + [(None, None)]):
        outs.append(lba.encode_merge_flat(tp, t, cap, kk, di, dv, n, next_tensor=nxt[0], next_k=nxt[1]))
    for (t, kk), (e, mg) in zip(steps, outs):
        idx_o, val_o, splits_o, st_o = top if kk else nonzeros
        total = int(splits_o.sum())
        assert st_o == 0 and e[3].item() == 0 and mg[3].item() == 0
        assert np.array_equal(to_np(e[2]), splits_o)
        assert np.array_equal(to_np(e[0])[:total], idx_o) and np.array_equal(to_np(e[1])[:total], val_o)
        cnt = int(mg[2])
        assert cnt == len(want_m[0]) and np.array_equal(to_np(mg[0])[:cnt], want_m[0].astype(np.int32))
        assert np.array_equal(to_np(mg[1])[:cnt].view(np.uint32), want_m[1].view(np.uint32))
    state = tp._ahead_state(a.device, 0)
    assert state is None or not state["pending"]
    assert not tp._table(a.device, tp.table_sizes(n)[0]).any()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_workgroups_that_take_the_next_sample_leave_their_first_tiles_to_the_others(zen, dtype):
    """Sizes at which a workgroup has no tile of its own, one, two (as many as it leaves out), three and more, odd
    lengths and unaligned tensors among them: the calls that take their successor's sample along return what calls
    without one return."""
    P = 16
    per = {torch.bfloat16: 2, torch.float32: 1}[dtype]
    tensors = []
    gen = torch.Generator(device="cuda").manual_seed(5)
    for i, n in enumerate([(1 << 22) + 13, 7500003, 14500001, 14500000, 22000007, 30000011, 5000000]):
        flat = torch.randn(n * per + i % 3, generator=gen, device="cuda").to(dtype)
        tensors.append(flat[i % 3:])
    idx = torch.arange(1, 5001, dtype=torch.int32, device="cuda")
    val = torch.ones(5000, dtype=dtype, device="cuda")
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(P), None, None)
    tp, plain = zen.TensorPartition(P, 1, 3), zen.TensorPartition(P, 1, 3)
    ks = [t.numel() // 200 for t in tensors]
    caps = [k + k // 4 + 4096 for k in ks]
    for i, t in enumerate(tensors):
        more = {}
        if i + 1 < len(tensors):
            more = {"next_tensor": tensors[i + 1], "next_k": ks[i + 1], "next_capacity": caps[i + 1]}
        e, _ = lba.encode_merge_flat(tp, t, caps[i], ks[i], idx, val, t.numel(), **more)
        want = plain.load_balance_flat(t, capacity=caps[i], k=ks[i])
        total = int(want[2].sum())
        assert e[3].item() == 0 == want[3].item() and total >= ks[i]
        for got, ref in ((e[0][:total], want[0][:total]), (e[1][:total], want[1][:total]), (e[2], want[2])):
            assert torch.equal(got, ref)


@pytest.mark.parametrize("dtype, sub", [(torch.bfloat16, 8192), (torch.float32, 4096)])
@pytest.mark.parametrize("more", [-4097, -1, 0, 1, 8191])
def test_every_element_is_looked_at_once(zen, dtype, sub, more):
    """Around the tensor length where the select kernel hands out more of its tiles by ticket (sixteen sub-tiles for
    each of three workgroups per compute unit), with and without the next call's sample taken along: the sent entries
    are the tensor's, each once."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    n, P = sub * 16 * 3 * cus + more, 4
    k = n // 200
    gen = torch.Generator(device="cuda").manual_seed(sub + more)
    grad = torch.randn(n, generator=gen, device="cuda").to(dtype)
    grad[-3:] = 9
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(P), None, None)
    recv = (torch.arange(1, 5000, device="cuda", dtype=torch.int32), torch.ones(4999, device="cuda", dtype=dtype))
    for nxt in (None, grad):
        thr = torch.zeros(2, dtype=torch.int32, device="cuda")
        (idx, val, splits, status), _ = lba.encode_merge_flat(lba.tensor_partition, grad, k + k // 4 + 4096, k, *recv, n,
                                                              thr_out=thr, next_tensor=nxt)
        key, reached = thr.tolist()
        least = torch.tensor([key << 16 if dtype == torch.bfloat16 else key], dtype=torch.int32).view(torch.float32).item()
        passed = grad.abs() >= least
        assert status.item() == 0 and reached >= k and reached == int(passed.sum())
        passed[0] = False  # index 0 is never sent
        want, total = torch.nonzero(passed).view(-1), int(splits.sum())
        order = torch.sort(idx[:total])
        assert torch.equal(order[0].long(), want) and torch.equal(val[:total][order[1]], grad[want])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("r", [8 * 4096, 8 * 4096 + 1, 8 * 4096 + 511, 8 * 4096 + 512, 8 * 4096 + 513, 9 * 4096 - 1])
def test_slab_merge_of_cut_off_batches(zen, r, dtype):
    """The last batch of a list has one entry, a little less than a row of a workgroup's threads, a row, a little more, all of
    its entries but one; the coarse slabs' parts have a few.  Whole numbers: exact."""
    from zen_repro_amd import _lib

    n = 1 << 23
    assert _lib.lib().zen_merge_path(r, n, _lib.MODE_FAST | _lib.MODE_SLABS) == SLAB
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(4), None, None)
    lba.fast_flags = _lib.MODE_SLABS
    gen = torch.Generator(device="cuda").manual_seed(r)
    idx = torch.randint(0, n, (r,), generator=gen, device="cuda", dtype=torch.int32)
    idx[-1], idx[-2] = 0, n - 1
    val = torch.randint(1, 4, (r,), generator=gen, device="cuda").to(dtype)
    want = torch.zeros(n, device="cuda").scatter_add_(0, idx.long(), val.float())
    at = torch.nonzero(want).view(-1)
    got_idx, got_val = lba.merge_rounded(idx, val, n, dtype)
    assert torch.equal(got_idx, at) and torch.equal(got_val, want[at].to(dtype))
