"""CPU-only checks: the C-ABI library loads and exports what include/zen_hip.h
declares, argument validation happens on the host, the host-side helpers and
the synthetic workloads behave, and the CPU baseline restatement agrees with
the oracle.  No kernel is launched here."""
import ctypes
import json
import os
import re
import subprocess
import sys

import numpy as np
import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def L():
    from zen_repro_amd import _lib

    if not os.path.exists(_lib.LIB_PATH):
        _lib.build()
    return _lib.lib()


def test_every_declared_symbol_is_exported(L):
    header = open(os.path.join(ROOT, "include", "zen_hip.h")).read()
    header = re.sub(r"/\*.*?\*/", "", header, flags=re.S)
    names = set(re.findall(r"\b(zen_[a-z0-9_]+)\s*\(", header))
    assert len(names) >= 20
    raw = ctypes.CDLL(os.path.join(ROOT, "zen_repro_amd", "csrc", "libzen_hip.so"))
    for n in sorted(names):
        assert hasattr(raw, n), f"{n} declared in zen_hip.h but not exported"
    from zen_repro_amd import _lib

    declared = int(re.search(r"#define\s+ZEN_ABI_VERSION\s+(\d+)", header).group(1))
    assert L.zen_abi_version() == declared == _lib.ABI_VERSION


def test_workspace_queries_are_host_only(L):
    assert L.zen_topk_threshold_workspace() >= 2048 * 4
    a, b = L.zen_sort_pairs_workspace(1000), L.zen_sort_pairs_workspace(1 << 20)
    assert 0 < a < b
    assert L.zen_merge_workspace(1 << 20, 1 << 30) >= 4 * 4 * (1 << 20)
    assert L.zen_load_balance_workspace(1 << 24, 1 << 24, 1, 1 << 18, 16) >= 6 * 4 * (1 << 18)
    assert L.zen_select_workspace(1 << 24, 1) >= (1 << 24) // 8192 * 8
    assert L.zen_mapping_workspace(1 << 20, 8) >= 16 * (1 << 20)
    assert L.zen_decode_dense_workspace(1000, 5000) > L.zen_merge_workspace(1000, 5000)


def test_path_selection_is_host_only(L):
    """Which implementation a call takes depends on sizes alone."""
    # c3: 743 M bf16 elements, top 0.5 %, 16 partitions -> bucket slabs; the same as fp32 too
    from zen_repro_amd import _lib

    slabs = _lib.MODE_SLABS  # without it the answer depends on the device: 3 (wide buckets) on a chip of 256 compute units
    assert L.zen_load_balance_path(743440384, 743440384, 1, 4650000, 16, 3717201, slabs) == 2
    assert L.zen_load_balance_path(743440384, 743440384, 0, 4650000, 16, 3717201, slabs) == 2
    assert L.zen_load_balance_path(743440384, 743440384, 0, 4650000, 16, 0, slabs) == 2
    assert L.zen_load_balance_path(743440384, 743440384, 1, 4650000, 16, 3717201, 0) in (2, 3)
    assert L.zen_load_balance_path(743440384, 743440384, 1, 4650000, 16, 3717201, 1) == 0   # general mode
    assert L.zen_load_balance_path(1 << 20, 1 << 20, 1, 1 << 14, 4, 0, 0) == 1             # small table
    assert L.zen_load_balance_path(1 << 24, 1 << 24, 1, 1 << 24, 16, 0, 0) == 1            # capacity = everything
    assert L.zen_merge_path(3717200, 743440384, slabs) == 2
    assert L.zen_merge_path(3717200, 743440384, 0) in (2, 3)
    assert L.zen_merge_path(3717200, 743440384, 1) == 0
    assert L.zen_merge_path(1000, 1 << 20, 0) == 0


@pytest.mark.parametrize("P", [1, 64, 511, 513, 600, 700, 1024, 1025, 1365, 1366, 2048, 2049, 2500, 3000, 4096])
def test_the_widest_tables_stay_on_the_slabs(L, P):
    """However badly the partitions fill the 4096 buckets there may be: the largest table has a slab geometry."""
    from zen_repro_amd import _lib

    m = (2 ** 31 - 1) // P * P
    for dtype in (0, 1):
        for k in (0, m // 1000):
            assert L.zen_load_balance_path(m, m, dtype, m // 900, P, k, _lib.MODE_SLABS) == 2


def test_bad_arguments_are_rejected_on_the_host(L):
    from zen_repro_amd import _lib

    one = ctypes.c_void_p(256)  # never dereferenced: validation comes first
    assert L.zen_hash_index(None, 16, 4, None) == _lib.EINVAL
    assert L.zen_hash_index(one, 3, 4, None) == _lib.EINVAL          # n < P
    assert L.zen_hash_index(one, 1 << 31, 4, None) == _lib.EINVAL    # n >= 2^31
    assert L.zen_hash_index(one, 16, 0, None) == _lib.EINVAL
    assert b"partitions" in L.zen_last_error()
    # table not a multiple of P, bad dtype, oversize
    assert L.zen_sparse_balance(one, 1, 64, one, 62, one, 4, one, 4, 3, one, None) == _lib.EINVAL
    assert L.zen_sparse_balance(one, 7, 64, one, 64, one, 4, one, 4, 3, one, None) == _lib.EINVAL
    assert L.zen_sparse_balance(one, 1, 1 << 31, one, 64, one, 4, one, 4, 3, one, None) == _lib.EINVAL
    assert L.zen_topk_threshold(one, 0, 100, 0, one, one, 1 << 20, None) == _lib.EINVAL    # k < 1
    assert L.zen_topk_threshold(one, 0, 100, 101, one, one, 1 << 20, None) == _lib.EINVAL  # k > n
    assert L.zen_topk_threshold(one, 0, 100, 5, one, one, 16, None) == _lib.EWORKSPACE
    assert L.zen_load_balance(one, 1, 1024, 1022, 4, 3, None, 0, None, one, one, 64, one, one, 0, one, 1 << 30, one, None) == _lib.EINVAL
    assert L.zen_load_balance(one, 1, 1024, 1024, 4, 3, one, 5, None, one, one, 64, one, one, 0, one, 1 << 30, one, None) == _lib.EINVAL  # thr and k
    assert L.zen_load_balance(one, 1, 1024, 1024, 4, 3, None, 0, None, one, one, 64, one, one, 0, one, 16, one, None) == _lib.EWORKSPACE
    assert L.zen_merge(one, 0, one, 0, 10, 0, one, 0, one, 10, one, 0, one, 1 << 20, one, None) == _lib.EINVAL  # dense_n
    assert L.zen_merge(one, 0, one, 0, 10, 100, one, 0, one, 10, one, 7, one, 1 << 20, one, None) == _lib.EINVAL  # mode
    assert L.zen_merge(one, 0, one, 0, 10, 100, one, 0, one, 10, one, 0, one, 16, one, None) == _lib.EWORKSPACE
    assert L.zen_sort_pairs(one, one, 100, None, 33, one, 1 << 20, one, None) == _lib.EINVAL
    # zen_encode_merge: a next call of its own size must take a path that keeps a sample in its table
    n = 1 << 24
    a = _lib.EncodeMergeArgs(
        256, 1, n, n, 16, 3, None, n // 200, None, 256, 256, n // 100, 256, 256, _lib.MODE_FAST | _lib.MODE_SLABS, 256,
        1 << 40, 256, 256, 0, 256, 1000, n, 256, 0, 256, 1000, 256, _lib.MODE_FAST, 256, 1 << 40, 256, None, None,
        256, 20, 4096, 4096, 64, 256)
    assert L.zen_encode_merge(ctypes.byref(a)) == _lib.EINVAL and b"next call" in L.zen_last_error()
    assert L.zen_encode_merge(None) == _lib.EINVAL
    with pytest.raises(ValueError):
        _lib.check(_lib.EINVAL, "x")
    with pytest.raises(RuntimeError):
        _lib.check(_lib.EHIP, "x")


def test_wrappers_assert_like_the_reference():
    import zen_repro_amd as zen

    g = torch.zeros(64, dtype=torch.bfloat16)
    mem = torch.zeros(64, dtype=torch.int32)
    with pytest.raises(AssertionError):  # extensions/cuda/functions.py:5: CPU tensors are refused
        zen.sparse_balance(g, mem, mem[:4], 4, 3)
    with pytest.raises(AssertionError):
        zen.hash_index(mem, 4)


def test_missing_library_fails_loudly(monkeypatch):
    from zen_repro_amd import _lib

    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "LIB_PATH", "/nonexistent/libzen_hip.so")
    with pytest.raises(RuntimeError, match="no fallback"):
        _lib.lib()


def test_missing_native_host_side_fails_loudly():
    """Whatever is called first says what is to be built, also where the library itself has not been asked for."""
    code = ("import sys; sys.modules['zen_repro_amd._host'] = None\n"
            "import torch, zen_repro_amd as zen\n"
            "from zen_repro_amd import _lib\n"
            "lba = zen.LoadBalanceAllreduce.__new__(zen.LoadBalanceAllreduce)\n"
            "for call in (lambda: lba.stack_tensors([torch.zeros(2), torch.zeros(3)]), _lib.lib, _lib.zeros.native):\n"
            "    try:\n"
            "        call()\n"
            "    except RuntimeError as e:\n"
            "        assert 'make -C zen_repro_amd/csrc' in str(e) and 'no fallback' in str(e)\n"
            "        print('told')\n")
    out = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True)
    assert out.stdout.split() == ["told"] * 3, out.stderr


def test_table_sizes_follow_the_reference(oracle):
    from zen_repro_amd.tensor_load_balance import TensorPartition

    tp = TensorPartition.__new__(TensorPartition)
    for n, P, scale in [(1 << 20, 4, 1), (1003, 4, 1), (5000, 4, 1.5), (743440384, 16, 1), (100, 64, 2)]:
        tp.partitions, tp.memory_scale = P, scale
        assert tp.table_sizes(n) == oracle.table_sizes(n, P, scale)
        m, s = tp.table_sizes(n)
        assert m % P == 0 and s % P == 0 and s == n // P // 10 * P


def test_consecutive_views_are_recognised():
    from zen_repro_amd.comm import _as_one_buffer

    buf = torch.arange(50, dtype=torch.int32)
    whole = _as_one_buffer([buf[:10], buf[10:30], buf[30:]])
    assert whole is not None and whole.data_ptr() == buf.data_ptr() and whole.numel() == 50
    assert _as_one_buffer([buf[:10], buf[11:30]]) is None
    assert _as_one_buffer([buf[:10], torch.arange(5, dtype=torch.int32)]) is None
    assert _as_one_buffer([buf[:10], buf[10:20].long()]) is None


def test_workload_hash_matches_oracle(oracle):
    from zen_repro_amd import workloads

    rng = np.random.default_rng(0)
    for m in (1 << 20, 743440384, 1003, (1 << 31) - 1):
        t = rng.integers(0, m, 3000)
        got = workloads.hash_slot(torch.from_numpy(t), m).numpy()
        want = np.array([oracle.hash32(int(x)) % m for x in t])
        assert np.array_equal(got, want)


def test_peer_payloads_have_the_stated_shape(oracle):
    from zen_repro_amd import workloads

    cfg, g = workloads.make("c1", device="cpu", seed=0)
    assert g.numel() == 1 << 20 and g.dtype == torch.float32 and cfg.k == 10485
    per = 2600
    idx_l, val_l, flat_idx, flat_val = workloads.peer_payloads(cfg, per, device="cpu")
    assert len(idx_l) == 4 and flat_idx.numel() == 4 * per and flat_idx.dtype == torch.int32
    part = oracle.hash_index(cfg.n, cfg.partitions)
    sets = [set(i.tolist()) for i in idx_l]
    for i, s in zip(idx_l, sets):
        assert len(s) == per and (part[i.numpy()] == 0).all()
        slots = workloads.hash_slot(i.long(), cfg.n)
        assert (slots[1:] >= slots[:-1]).all()  # slot order, as an encoder emits
    common = set.intersection(*sets)
    assert len(common) == int(per * cfg.overlap)  # the shared pool, and nothing else
    assert idx_l[1].data_ptr() == flat_idx.data_ptr() + per * 4


@pytest.mark.parametrize("name,shrink", [("c2", 64), ("c3", 256), ("c4", 1024), ("c5", 64)])
def test_workloads_small(name, shrink):
    from zen_repro_amd import workloads

    cfg, g = workloads.make(name, device="cpu", seed=0, shrink=shrink)
    assert g.numel() == cfg.n and cfg.n % cfg.partitions == 0 and g.dtype == cfg.dtype
    nz = int(torch.count_nonzero(g))
    if name == "c3":
        assert nz > 0.99 * cfg.n and cfg.k == int(cfg.n * 0.005)
    elif name == "c2":
        # two gradient buckets: the embedding (row-sparse, taken as it is) and the dense rest (top 1 % by the path)
        emb, rest = workloads.buckets(cfg)
        assert emb.offset == 0 and rest.offset == emb.n and emb.n + rest.n == cfg.n
        assert emb.k == 0 and rest.k == rest.n // 100
        assert emb.n % cfg.partitions == 0 and rest.n % cfg.partitions == 0
        assert 0 < int(torch.count_nonzero(g[:emb.n])) < 0.05 * emb.n
        assert int(torch.count_nonzero(g[emb.n:])) > 0.99 * rest.n
    else:
        assert 0 < nz < 0.05 * cfg.n
        assert workloads.buckets(cfg) == [cfg]
    if name == "c4":
        idx = torch.nonzero(g, as_tuple=True)[0]
        h, r = workloads.bucket_imbalance(idx, cfg.n, cfg.partitions)
        assert h < 1.2 < r  # the hash flattens what range partitioning piles up


def test_cpu_baseline_restatement_agrees_with_oracle(oracle):
    from oracle import torch_path
    from zen_repro_amd import workloads

    cfg, g = workloads.make("c3", device="cpu", seed=0, shrink=1024)
    per = cfg.k // cfg.partitions
    idx_l, val_l, flat_idx, flat_val = workloads.peer_payloads(cfg, per, device="cpu")
    times, (indices, values, splits, status, m_idx, m_val) = torch_path.timed_pass(g, cfg.k, cfg.partitions, idx_l, val_l)
    bits = g.view(torch.int16).numpy().view(np.uint16)
    key = oracle.kth_key(bits, cfg.k)
    masked, _ = oracle.mask_dense(bits, key)
    idx_o, val_o, splits_o, st = oracle.load_balance(masked, cfg.partitions)
    assert status == st == 0
    assert np.array_equal(torch.cat(indices).numpy(), idx_o)
    assert np.array_equal(torch.cat(values).view(torch.int16).numpy().view(np.uint16), val_o)
    assert np.array_equal(splits.numpy(), splits_o)
    # merge: torch's CPU kernel sums bf16 in fp32 and rounds once
    f32 = oracle.decode(flat_idx.numpy(), flat_val.view(torch.int16).numpy().view(np.uint16), cfg.n, "f32acc")
    mi, mv = oracle.encode(oracle.f32_to_bf16_bits(f32))
    assert np.array_equal(m_idx.numpy(), mi)
    assert np.array_equal(m_val.view(torch.int16).numpy().view(np.uint16), mv)
    assert set(times) == {"select", "partition", "merge"}


def test_ranges_are_off_by_default_and_cost_nothing():
    """The named ranges (the reference's nvtx names) are plain null contexts unless switched on."""
    import contextlib

    from zen_repro_amd import _lib

    was = _lib._ranges_on
    try:
        _lib.ranges_enable(False)
        assert isinstance(_lib.annotate("load_balance"), contextlib.nullcontext)
        with _lib.annotate("load_balance"), _lib.annotate("decode_sparse_tensors"):
            pass
        _lib.ranges_enable(True)
        assert not isinstance(_lib.annotate("load_balance"), contextlib.nullcontext)
    finally:
        _lib.ranges_enable(was)


def test_a_waiting_sample_keeps_the_owner_table_away(L):
    """A sample taken ahead waits in its call's table (2^20 slots or more): a call that selects by threshold or takes
    the nonzeros may use every word of such a table only where it is told that none waits there."""
    from zen_repro_amd import _lib
    from zen_repro_amd.tensor_load_balance import TensorPartition

    n, room = 1 << 22, 1 << 14
    assert L.zen_load_balance_path(n, n, _lib.BF16, room, 4, 0, _lib.MODE_FAST) in (2, 3)
    assert L.zen_load_balance_path(n, n, _lib.BF16, room, 4, 0, _lib.MODE_FAST | _lib.MODE_NO_SAMPLES) == 1
    assert L.zen_load_balance_path((1 << 20) - 4, (1 << 20) - 4, _lib.BF16, room, 4, 0, _lib.MODE_FAST) == 1  # holds none
    assert L.zen_load_balance_path(n, n, _lib.BF16, room, 4, 4096, _lib.MODE_FAST | _lib.MODE_NO_SAMPLES) in (2, 3)

    tp = TensorPartition.__new__(TensorPartition)
    tp.partitions, tp.memory_scale, tp._on_buckets = 4, 1, {}
    state, dropped = {"free": [None, None], "pending": []}, []
    tp._ahead_state = lambda dev, slot: state
    tp._discard = lambda entry, slot, dev: dropped.append(entry)
    flat = torch.zeros(n, dtype=torch.bfloat16)
    take = lambda mode: tp._take_ahead(flat, n, 0, room, None, 0, mode, None, None)
    assert take(_lib.MODE_FAST) == (_lib.MODE_NO_SAMPLES, 0)
    state["pending"].append("a sample")
    assert take(_lib.MODE_FAST) == (0, 0) and state["pending"] and not dropped
    # the general mode has no other way than through the whole table: what waits there is dropped first
    assert take(_lib.MODE_GENERAL) == (_lib.MODE_NO_SAMPLES, 0) and not state["pending"] and dropped == ["a sample"]


def test_only_a_call_that_samples_books_the_next_sample(L):
    """Whether a call takes its successor's sample along follows from the call's own path: a call through the owner
    table does not, whatever the successor's k is, and so there is nothing for the successor to pick up."""
    from zen_repro_amd import _lib
    from zen_repro_amd.tensor_load_balance import TensorPartition

    n, room = 1 << 22, 1 << 14
    tp = TensorPartition.__new__(TensorPartition)
    tp.partitions, tp.memory_scale, tp._samples_next = 4, 1, {}
    state = {"free": [None, None], "pending": []}
    tp._ahead_state = lambda dev, slot, create=False: state
    flat, nxt = torch.zeros(n, dtype=torch.bfloat16), torch.ones(n, dtype=torch.bfloat16)
    book = lambda k, mode: tp._next_sample(flat, k, nxt, 4096, room, room, 0, mode, 0)[0]
    for _ in range(2):  # the second time from the cache
        assert book(0, _lib.MODE_FAST | _lib.MODE_NO_SAMPLES) is None
        assert book(0, _lib.MODE_FAST).data_ptr() == nxt.data_ptr()
        assert book(4096, _lib.MODE_FAST).data_ptr() == nxt.data_ptr()


def test_read_back_of_more_words_than_the_pinned_buffer_holds():
    """Split sizes of hundreds of thousands of partitions come back as plain copies."""
    from zen_repro_amd import _lib

    splits, status = torch.arange(1 << 20, dtype=torch.int64), torch.full((1,), 8, dtype=torch.int32)
    assert _lib.read_back(splits, status) == list(range(1 << 20)) + [8]


@pytest.mark.parametrize("capturing", [False, True])
def test_a_hook_without_a_stream_keeps_its_calls_in_order(monkeypatch, capturing):
    """The calls of one hook share workspaces: one that finds another current stream than the last waits for that
    one's; calls that stay on a stream wait for nothing."""
    import zen_repro_amd as zen
    from zen_repro_amd.hook import SparseCommHook

    class Stream:
        def __init__(self):
            self.cuda_stream = id(self)
            self.waited = []

        def wait_stream(self, other):
            self.waited.append(other)

    a, b = Stream(), Stream()
    now = [a]
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: now[0])
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: capturing)

    class Bucket:
        def buffer(self):
            return torch.zeros(8)

    class Lba:
        process_group = zen.LocalGroup(1)

    ran_on = []
    hook = SparseCommHook(Lba(), 1, 2, zen.LocalGroup(1))
    hook._reduce = lambda tensors, exchange: ran_on.append((now[0], list(now[0].waited))) or tensors
    hook(None, Bucket())  # passes the first bucket through
    for stream in (a, a, b, b, a):
        now[0] = stream
        hook(None, Bucket())
    waits = [[], [], [a], [a], [b]] if not capturing else [[]] * 5
    assert ran_on == list(zip((a, a, b, b, a), waits))


@pytest.mark.parametrize("capturing", [False, True])
def test_a_kept_buffer_is_waited_for_and_held_by_every_stream(monkeypatch, capturing):
    """A stream's first use of a buffer made on another one waits for its making and is remembered by the
    allocator; uses on the maker's stream, and second uses, do neither."""
    from zen_repro_amd import _lib

    log = []

    class Stream:
        def __init__(self, handle):
            self.cuda_stream = handle

        def wait_stream(self, other):
            log.append(("wait", self.cuda_stream, other.cuda_stream))

    class Buffer:
        def numel(self):
            return 256

        def record_stream(self, stream):
            log.append(("hold", stream.cuda_stream))

    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: capturing)
    streams = {h: Stream(h) for h in (1, 2, 3)}
    buf = Buffer()
    now = [1]
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: streams[now[0]])
    monkeypatch.setattr(_lib, "current_handle", lambda index: now[0])
    scratch = _lib.Scratch()
    scratch._bufs()[0, "a"] = _lib.Kept(buf, streams[1])
    for now[0] in (1, 2, 1, 2):
        assert scratch.get(torch.device("cuda", 0), "a", 1) is buf
    assert scratch.get(torch.device("cuda", 0), "a", 1, stream=streams[3]) is buf
    assert log == ([] if capturing else [("wait", 2, 1), ("hold", 2), ("wait", 3, 1), ("hold", 3)])


def test_streams_wait_for_a_call_that_returned_before_its_kernels_were_through(monkeypatch):
    """Split sizes reach the host before the last kernel of a load balance is done with the workspace: the streams
    that have used it before wait for the call's stream at their next use, the call's own does not."""
    from zen_repro_amd import _lib

    log = []

    class Stream:
        def __init__(self, handle):
            self.cuda_stream = handle

        def wait_stream(self, other):
            log.append((self.cuda_stream, other.cuda_stream))

    class Buffer:
        def numel(self):
            return 256

        def record_stream(self, stream):
            pass

    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    streams = {h: Stream(h) for h in (1, 2, 3)}
    now = [1]
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: streams[now[0]])
    monkeypatch.setattr(_lib, "current_handle", lambda index: now[0])
    device = torch.device("cuda", 0)
    scratch = _lib.Scratch()
    scratch._bufs()[0, "a"] = _lib.Kept(Buffer(), streams[1])
    scratch.left_running(device, "a")  # stream 1, the only one so far
    now[0] = 2
    scratch.get(device, "a", 1)
    assert log == [(2, 1)]
    scratch.left_running(device, "a")
    for now[0] in (2, 1, 2, 1):
        scratch.get(device, "a", 1)
    scratch.get(device, "a", 1, stream=streams[3])
    assert log == [(2, 1), (1, 2), (3, 2)]


@pytest.mark.parametrize("call", ["load_balance", "encode_sparse_tensor", "decode_sparse_tensors", "merge_rounded"])
@pytest.mark.parametrize("code", [0, -2])
def test_calls_that_return_early_leave_their_buffers_marked(monkeypatch, call, code):
    """The four calls whose kernels tell the host sizes or a status return while the last of them may still use the
    call's workspace (and table).  Two streams that have both used one take turns: each waits for the other's call,
    one that failed on the device's side among them (what clears the buffer again comes behind it)."""
    import zen_repro_amd as zen
    from zen_repro_amd import _lib

    class Stream:
        def __init__(self, handle):
            self.cuda_stream = handle

    class Library:  # every size 256, nothing launched
        def __getattr__(self, name):
            if name == "zen_last_error":
                return lambda: b"the device"
            told = name.endswith(("_sizes", "_count", "_status"))
            return lambda *args: 0 if name == "zen_merge_zero_bytes" else code if told else 256

    class Words:
        ptr, words, view = 0, 64, [0] * 64

    waits, held, now = [], [], [1]
    streams = {h: Stream(h) for h in (1, 2)}

    def join(kept, stream, new=False):
        waits.append((stream.cuda_stream, kept.maker.cuda_stream))
        kept.seen.add(stream.cuda_stream)

    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: streams[now[0]])
    monkeypatch.setattr(_lib, "lib", Library)
    monkeypatch.setattr(_lib, "device_index", lambda device: 0)
    monkeypatch.setattr(_lib, "current_handle", lambda index: now[0])
    monkeypatch.setattr(_lib, "require_gpu", lambda t, name: None)
    monkeypatch.setattr(_lib, "host_words", lambda n: Words)
    monkeypatch.setattr(_lib, "scratch", _lib.Scratch())
    monkeypatch.setattr(_lib, "zeros", _lib.ZeroPool())
    monkeypatch.setattr(_lib.Kept, "join", join)
    monkeypatch.setattr(torch.Tensor, "record_stream", lambda t, s: held.append((t.data_ptr(), s.cuda_stream)))
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(4), None, None)
    dense, idx = torch.ones(64), torch.arange(8, dtype=torch.int32)
    run = {"load_balance": lambda: lba.tensor_partition.load_balance(dense, capacity=64),
           "encode_sparse_tensor": lambda: lba.encode_sparse_tensor(dense),
           "decode_sparse_tensors": lambda: lba.decode_sparse_tensors(idx, dense[:8], 64),
           "merge_rounded": lambda: lba.merge_rounded(idx, dense[:8], 64, torch.float32)}[call]
    for now[0] in (1, 1, 2, 2, 1, 2):
        if code:
            with pytest.raises(RuntimeError, match="the device"):
                run()
        else:
            run()
    buffers = 2 if call == "load_balance" else 1
    assert waits == [w for w in [(2, 1), (1, 2), (2, 1)] for _ in range(buffers)]
    # two of them may still read their input, which the allocator is told of; the others are through with theirs
    reads = call in ("load_balance", "encode_sparse_tensor")
    assert held == ([(dense.data_ptr(), s) for s in (1, 1, 2, 2, 1, 2)] if reads else [])


@pytest.fixture(scope="module")
def deviceless(tmp_path_factory, L):
    """(name, fail_at, arguments) -> (return code, what was launched and waited for): the library's calls on a HIP
    runtime without a device (fake_hip.py)."""
    from zen_repro_amd import _lib

    here = os.path.dirname(os.path.abspath(__file__))
    fake = str(tmp_path_factory.mktemp("fake") / "fake_hip.so")
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", os.path.join(here, "fake_hip.cpp"), "-o", fake], check=True)
    child = subprocess.Popen([sys.executable, os.path.join(here, "fake_hip.py"), fake, _lib.LIB_PATH],
                             stdin=subprocess.PIPE, stdout=subprocess.PIPE, text=True)

    def call(name, fail_at, args):
        child.stdin.write(json.dumps([name, fail_at, args]) + "\n")
        child.stdin.flush()
        return json.loads(child.stdout.readline())

    yield call
    child.stdin.close()
    child.wait(timeout=60)


PTR, ROOM, STREAM = 4096, 1 << 50, 77  # an address nothing looks at, a workspace of any size, a stream
WAITING_CALLS = {
    "zen_balance_tables": [PTR, 1, 4096, PTR, 4096, PTR, 400, PTR, 4, 3, PTR, "host", 64, STREAM],
    "zen_bitmap_encode_status": [PTR, 1000, PTR, 1, 100, None, PTR, 4000, PTR, PTR, "host", 64, STREAM],
    "zen_select_count": [PTR, 1, 1 << 20, None, PTR, 1, PTR, 1 << 20, PTR, PTR, ROOM, PTR, "host", 64, STREAM],
    "zen_table_find_sizes": [PTR, 4096, 4, 4096, PTR, PTR, PTR, ROOM, PTR, "host", 64, STREAM],
    "zen_load_balance_sizes, one workgroup": [PTR, 1, 9000, 9000, 4, 3, None, 0, None, PTR, PTR, 1000, PTR, PTR, 0x4100, PTR, ROOM,
                                              PTR, "host", 64, STREAM],
    "zen_load_balance_sizes, owner table": [PTR, 1, 1 << 21, 1 << 21, 4, 3, None, 0, None, PTR, PTR, 1000, PTR, PTR, 0x4100, PTR,
                                            ROOM, PTR, "host", 64, STREAM],
    "zen_load_balance_sizes, slabs": [PTR, 0, 1 << 24, 1 << 24, 4, 3, None, 1000, None, PTR, PTR, 2000, PTR, PTR, 0x100, PTR, ROOM,
                                      PTR, "host", 64, STREAM],
    "zen_load_balance_sizes, wide buckets": [PTR, 0, 1 << 24, 1 << 24, 4, 3, None, 1000, None, PTR, PTR, 2000, PTR, PTR, 0x8100, PTR,
                                             ROOM, PTR, "host", 64, STREAM],
    "zen_load_balance_sizes, general": [PTR, 0, 1 << 16, 1 << 16, 4, 3, None, 0, None, PTR, PTR, 2000, PTR, PTR, 1, PTR, ROOM, PTR,
                                        "host", 64, STREAM],
    "zen_merge_rounded_count, one workgroup": [PTR, 0, PTR, 1, 1000, 1 << 20, PTR, 0, PTR, 1000, PTR, 0x100, PTR, ROOM, PTR, "host",
                                               64, STREAM],
    "zen_merge_rounded_count, wide buckets": [PTR, 0, PTR, 1, 100000, 1 << 24, PTR, 0, PTR, 1000, PTR, 0x100, PTR, ROOM, PTR, "host",
                                              64, STREAM],
    "zen_merge_rounded_count, slabs": [PTR, 0, PTR, 1, 400000, 1 << 26, PTR, 0, PTR, 1000, PTR, 0x2100, PTR, ROOM, PTR, "host", 64,
                                       STREAM],
    "zen_merge_rounded_count, general": [PTR, 0, PTR, 1, 10000, 1 << 24, PTR, 0, PTR, 1000, PTR, 1, PTR, ROOM, PTR, "host", 64, STREAM],
    "zen_decode_dense_status": [PTR, 1, PTR, 0, 100000, PTR, 1 << 24, 0x100, PTR, ROOM, PTR, "host", 64, STREAM],
    "zen_decode_dense_lists_status": [[PTR, PTR], 1, [PTR, PTR], 1, [50, 60], 2, PTR, 1 << 20, PTR, ROOM, PTR, "host", 64, STREAM],
    "zen_decode_dense_lists_status, many tiles": [[PTR, PTR], 1, [PTR, PTR], 1, [50, 60], 2, PTR, 1 << 26, PTR, ROOM, PTR, "host", 64,
                                                  STREAM],
    "zen_bitmap_dense_lists_status": [PTR, 1 << 20, 2, [PTR, PTR], [1 << 16, 1 << 16], [PTR, PTR], 1, [50, 60], PTR, PTR, ROOM, PTR,
                                      "host", 64, STREAM],
    "zen_read_back": [PTR, 3, 1, None, 0, 0, None, 0, 0, "host", 64, STREAM],
}


@pytest.mark.parametrize("what", list(WAITING_CALLS))
def test_a_failed_call_leaves_no_answer_on_its_way(deviceless, what):
    """A call that waits draws the ticket of its answer from the host's words, where a call that fails leaves them as
    they were: the next one would take a late answer of this one for its own.  So whichever launch fails, the stream has
    been waited for when the call returns."""
    from zen_repro_amd import _lib

    name, args = what.split(",")[0], WAITING_CALLS[what]
    _, log = deviceless(name, 0, args)
    launches = [line for line in log if line.startswith("launch")]
    assert launches and all(line.endswith(f" {STREAM}") for line in launches)
    for fail_at in range(1, 40):
        rc, log = deviceless(name, fail_at, args)
        if "fail" not in log:  # fewer checks than that
            break
        assert rc == _lib.EHIP and log[-2:] == ["fail", f"wait {STREAM}"]
    assert fail_at > 1 and log == launches


@pytest.mark.parametrize("what,tiles", [
    ("zen_bitmap_dense_lists_status", "k_fd_tiles"),
    ("zen_decode_dense_lists_status", "k_decode_tiles"),
    ("zen_decode_dense_lists_status, many tiles", "k_decode_tiles"),
])
def test_a_decode_is_done_when_its_status_is_known(deviceless, what, tiles):
    """The host is told by a kernel behind the tiles: nobody reads the lists any more when the call returns, the tensor is
    there for every stream, and what a tile has to say about the bitmaps' dictionary is in the status."""
    rc, log = deviceless(what.split(",")[0], 0, WAITING_CALLS[what])
    assert rc == 0 and tiles in log[-2] and "k_read_back" in log[-1]


def test_other_threads_run_while_a_call_allocates():
    """The native side lets go of the interpreter while it makes a call's tensors (long zeros here), as
    torch's own functions do: another thread goes on meanwhile."""
    import threading
    import time

    from zen_repro_amd import _lib

    memory, began, ended, seen = torch.zeros(8, dtype=torch.int32), [], [], []
    done = threading.Event()

    def watch():
        while not done.is_set():
            seen.append(time.perf_counter())
            time.sleep(1e-4)

    parts = 1 << 25  # 0.8 GB of words
    other = threading.Thread(target=watch)
    other.start()
    began.append(time.perf_counter())
    _lib.host.table_find(lambda *a: ended.append(time.perf_counter()) or 0, _lib.host.Zeros(), memory, parts, 8, 16, 0, 0, 0)
    done.set()
    other.join()
    inside = [began[0]] + [t for t in seen if began[0] < t < ended[0]] + [ended[0]]
    assert max(b - a for a, b in zip(inside, inside[1:])) < 0.5 * (ended[0] - began[0])


def test_every_call_gets_zeroed_words_of_its_own():
    """Status words and split sizes are cut from blocks: none is handed out twice, also where a block ends, where a
    piece is longer than a block, and where a stream starts afresh."""
    from zen_repro_amd import _lib

    zeros = _lib.host.Zeros()
    flat, ws = torch.zeros(8, dtype=torch.bfloat16), torch.zeros(16, dtype=torch.uint8)
    held, words = [], []  # (pieces begin at 16 bytes, those of status words at 8)
    for call in range(3000):
        parts, stream = (9000, 5) if call == 1500 else (5, 5 + call % 2)
        rc, idx, val, splits, status = _lib.host.load_balance(
            lambda *a: len(a), zeros, flat, 1, 8, parts, 3, None, 0, None, 4, 0, 0, ws, stream, 0, 0)
        assert rc == 19 and idx.shape == val.shape == (4,) and splits.shape == (parts,) and status.shape == (1,)
        assert not splits.any() and not status.any()
        assert splits.data_ptr() % 16 == 0 and status.data_ptr() % 8 == 0
        held += [splits, status]
        words += [(t.data_ptr(), t.data_ptr() + t.numel() * t.element_size()) for t in (splits, status)]
        splits.fill_(-1)
        status.fill_(-1)
        if call == 2000:
            zeros.fresh(-1, 5)
    words.sort()
    assert all(a[1] <= b[0] and b[0] % 8 == 0 for a, b in zip(words, words[1:]))


def test_compaction_kernels_keep_their_rows_in_registers(tmp_path):
    """The rows a wave has in flight are the kernels' speed: none of their registers may end up in memory, for
    aligned tensors and for views that begin at an odd element."""
    import shutil
    import subprocess

    csrc = os.path.join(ROOT, "zen_repro_amd", "csrc")
    plan = subprocess.run(["make", "-C", csrc, "-n", "-B", "--no-print-directory", "zen_compact.o"],
                          capture_output=True, text=True, check=True).stdout
    command = plan.strip().splitlines()[-1].split()
    if not shutil.which(command[0]):
        pytest.skip("no compiler")
    out = str(tmp_path / "zen_compact.s")
    command = command[:command.index("-c")] + ["--cuda-device-only", "-S", "zen_compact.hip", "-o", out]
    subprocess.run(command, cwd=csrc, check=True, stderr=subprocess.DEVNULL)
    spills = re.findall(r"\.name:\s+(\S+).*?\.vgpr_spill_count:\s+(\d+)", open(out).read(), flags=re.S)
    walks = [int(n) for name, n in spills if "k_compact" in name]
    assert len(walks) >= 12 and not any(walks)
