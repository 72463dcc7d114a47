"""Parity of the bitmap index codec (comm.py:59-99) against the CPU oracle
(itself pinned by numpy.packbits), its edge cases, a full-size round trip, and
the whole sparse all-reduce (comm.py:101-150, methods 1-3) with four ranks
played by four host threads on the one GPU.  Bar: bit-exact bitmaps and
indices; summed values within 1e-6 of the summed magnitudes (fp32) or one
bf16 rounding of the fp32 sum."""
import threading

import numpy as np
import pytest
import torch

from gpu_util import to_dev, to_np

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def zen():
    import zen_repro_amd
    from zen_repro_amd import _lib

    _lib.lib()
    assert torch.cuda.is_available()
    return zen_repro_amd


def lba_with_mapping(zen, n, P, rank):
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(P, rank), None, None)
    lba.mapping[n] = lba.calculate_mapping(n)
    return lba


@pytest.mark.parametrize("n, P", [(1, 1), (95, 1), (96, 2), (97, 1), (193, 3), (12 * 96 + 1, 4), (9000, 2)])
def test_bitmap_rank_entries(zen, oracle, n, P):
    """Every index of [0, n) by itself, around the edges of the rank dictionary's entries; lists that ascend, that
    repeat an index, that descend, and of lengths around what a workgroup takes."""
    n = n // P * P
    rng = np.random.default_rng(n)
    for rank in range(P):
        lba = lba_with_mapping(zen, n, P, rank)
        members = oracle.mapping(n, P)[rank]
        if not len(members):
            continue
        fits = np.arange(members[-1] + 1)  # an index that is no member marks the next one
        lists = [fits, fits[::-1].copy(), np.sort(np.concatenate([fits, fits]))]
        lists += [np.sort(rng.choice(fits, size)) for size in (1, 63, 64, 65, 255, 1023, 1024, 1025)]
        lists += [fits[i:i + 1] for i in range(max(0, len(fits) - 200), len(fits), 7)]
        for idx in lists:
            assert np.array_equal(to_np(lba.encode_bitmap(to_dev(idx), n)), oracle.bitmap_encode(members, idx))
        with pytest.raises(IndexError):
            lba.encode_bitmap(to_dev(np.array([members[-1] + 1])), n)


@pytest.mark.parametrize("idx_dtype", [torch.int64, torch.int32])
@pytest.mark.parametrize("n,P,rank,frac", [
    (1 << 12, 8, 3, 0.05),
    (1 << 20, 4, 0, 0.01),
    (1 << 20, 4, 3, 0.5),          # every second member
    (6000000, 3, 1, 0.001),        # partitions not a power of two
    ((1 << 22) + 40, 8, 7, 1.0),   # all members; list length not a multiple of 8
])
def test_bitmap_matches_oracle(zen, oracle, n, P, rank, frac, idx_dtype):
    n = n // P * P
    lba = lba_with_mapping(zen, n, P, rank)
    mp = oracle.mapping(n, P)
    for p in range(P):  # the lists themselves are the oracle's
        assert np.array_equal(to_np(lba.mapping[n][p]), mp[p])
    members = mp[rank]
    rng = np.random.default_rng(n ^ P ^ rank)
    pick = np.sort(rng.choice(members, max(1, int(len(members) * frac)), replace=False))
    want = oracle.bitmap_encode(members, pick)
    got = lba.encode_bitmap(to_dev(pick).to(idx_dtype), n)
    assert got.dtype == torch.uint8 and got.numel() == (len(members) + 7) // 8
    assert np.array_equal(to_np(got), want)
    # order of the indices does not matter, nor do repeats
    shuffled = np.concatenate([rng.permutation(pick), pick[:7]])
    assert np.array_equal(to_np(lba.encode_bitmap(to_dev(shuffled).to(idx_dtype), n)), want)
    # the same through the C-ABI without the rank table (search from an interpolated position)
    from zen_repro_amd import _lib

    L = _lib.lib()
    d_idx = to_dev(shuffled).to(idx_dtype)
    d_map = lba.mapping[n][rank]
    words = torch.full((L.zen_bitmap_words(len(members)),), -1, dtype=torch.int32, device="cuda")
    status = _lib.status_word("cuda")
    rc = L.zen_bitmap_encode(_lib.ptr(d_map), len(members), _lib.ptr(d_idx), int(idx_dtype == torch.int64),
                             d_idx.numel(), None, None, 0, _lib.ptr(words), _lib.ptr(status), _lib.stream_of("cuda"))
    assert rc == 0 and status.item() == 0
    assert np.array_equal(to_np(words.view(torch.uint8))[:len(want)], want)
    assert int(words.view(torch.uint8)[len(want):].sum()) == 0  # the padding up to a whole word is zero
    # decode: one bitmap per rank, each against that rank's list
    lba0 = lba_with_mapping(zen, n, P, 0)
    bitmaps, wants = [], []
    for p in range(P):
        sel = np.sort(rng.choice(mp[p], max(1, len(mp[p]) // 50), replace=False))
        bm = oracle.bitmap_encode(mp[p], sel)
        # what allgather_padding hands back may be a view at any byte offset
        holder = torch.zeros(len(bm) + 3, dtype=torch.uint8, device="cuda")
        holder[1 + (p % 3):1 + (p % 3) + len(bm)] = to_dev(bm)
        bitmaps.append(holder[1 + (p % 3):1 + (p % 3) + len(bm)])
        wants.append(sel)
        assert np.array_equal(oracle.bitmap_decode(mp[p], bm), sel)
    outs = lba0.decode_bitmap(bitmaps, n)
    assert len(outs) == P
    for p in range(P):
        assert outs[p].dtype == torch.int64
        assert np.array_equal(to_np(outs[p]), wants[p])


def test_bitmap_edge_cases(zen, oracle):
    n, P, rank = 1 << 16, 4, 2
    lba = lba_with_mapping(zen, n, P, rank)
    members = oracle.mapping(n, P)[rank]
    nbytes = (len(members) + 7) // 8
    solo = zen.LoadBalanceAllreduce(zen.LocalGroup(P, 0), None, None)  # decodes against this one list
    solo.mapping[n] = [lba.mapping[n][rank]]
    # nothing selected
    empty = lba.encode_bitmap(torch.empty(0, dtype=torch.int64, device="cuda"), n)
    assert empty.numel() == nbytes and int(empty.sum()) == 0
    assert solo.decode_bitmap([empty], n)[0].numel() == 0
    # an index that is no member marks the next member (searchsorted, left side)
    gap = np.setdiff1d(np.arange(members[5] + 1, members[-1]), members)[:9]
    want = oracle.bitmap_encode(members, gap)
    assert np.array_equal(to_np(lba.encode_bitmap(to_dev(gap), n)), want)
    assert want.sum() > 0
    # first and last member, and the values around them
    ends = np.array([0, members[0], members[-1]], dtype=np.int64)
    assert np.array_equal(to_np(lba.encode_bitmap(to_dev(ends), n)), oracle.bitmap_encode(members, ends))
    # beyond the last member: the reference indexes one past the end of its mask
    with pytest.raises(IndexError):
        lba.encode_bitmap(to_dev(np.array([members[-1] + 1], dtype=np.int64)), n)
    # a device-side count limits what is read
    pick = members[::3].copy()
    count = torch.tensor([100], dtype=torch.int64, device="cuda")
    bm, status = lba.encode_bitmap_flat(to_dev(pick), n, count=count)
    assert status.item() == 0
    assert np.array_equal(to_np(bm), oracle.bitmap_encode(members, pick[:100]))
    # padding after the last byte is ignored, bits past the last member too; a short bitmap is refused
    full = oracle.bitmap_encode(members, members)
    padded = np.concatenate([full, np.full(5, 0xFF, dtype=np.uint8)])
    padded[nbytes - 1] = 0xFF
    assert np.array_equal(to_np(solo.decode_bitmap([to_dev(padded)], n)[0]), members)
    with pytest.raises(IndexError):
        solo.decode_bitmap([to_dev(full[:-1])], n)


def test_bitmap_full_size_round_trip(zen):
    """c3's index space (743 M, 16 partitions): the merged indices of rank 0's
    received payloads -> bitmap -> indices, and the bitmap against the
    reference's own recipe (searchsorted, mask, weights 1..128) in torch ops."""
    from zen_repro_amd import workloads

    cfg, grad = workloads.make("c3", device="cuda", seed=0, shrink=1)
    del grad
    n, P = cfg.n, cfg.partitions
    lba = lba_with_mapping(zen, n, P, 0)
    members = lba.mapping[n][0]
    assert sum(m.numel() for m in lba.mapping[n]) == n
    _, _, flat_idx, flat_val = workloads.peer_payloads(cfg, cfg.k // P, device="cuda", seed=1)
    m_idx, _ = lba.merge_sparse(flat_idx, flat_val, n)
    bitmap = lba.encode_bitmap(m_idx, n)
    pos = torch.searchsorted(members, m_idx)
    mask = torch.zeros(members.numel() + 7, dtype=torch.uint8, device="cuda")
    mask[pos] = 1
    weights = 2 ** torch.arange(8, dtype=torch.uint8, device="cuda")
    want = (mask[:(members.numel() + 7) // 8 * 8].view(-1, 8) * weights).sum(dim=1).to(torch.uint8)
    assert torch.equal(bitmap, want)
    back = lba.decode_bitmap([bitmap], n)[0]
    assert torch.equal(back, m_idx)


class ThreadExchange:
    """The reference backend's calls (DDPbackend.py:13-41, 71-81) between host
    threads that each play one rank on the same GPU."""

    def __init__(self, size):
        self.size = size
        self.barrier = threading.Barrier(size)
        self.slots = [None] * size

    def view(self, rank):
        return _RankView(self, rank)

    def exchange(self, rank, item):
        torch.cuda.current_stream().synchronize()
        self.slots[rank] = item
        self.barrier.wait()
        got = list(self.slots)
        self.barrier.wait()
        return got


class _RankView:
    def __init__(self, ex, rank):
        self.ex, self.rank = ex, rank

    def allgather(self, tensor, async_op=True):
        return [t.clone() for t in self.ex.exchange(self.rank, tensor)]

    def allgather_padding(self, tensor, async_op=True):
        return [t.clone() for t in self.ex.exchange(self.rank, tensor)]

    def alltoallv(self, tensors, gather_splits):
        everyone = self.ex.exchange(self.rank, tensors)
        got = [everyone[src][self.rank].clone() for src in range(self.ex.size)]
        for src in range(self.ex.size):
            assert got[src].numel() == int(gather_splits[src][self.rank])
        return got


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("method", [1, 2, 3])
def test_sparse_allreduce_between_four_ranks(zen, method, dtype):
    """Every rank ends with the sum of all ranks' sparse tensors."""
    P, n = 4, 1 << 20
    gen = torch.Generator(device="cuda").manual_seed(7 + method)
    tensors = []
    for r in range(P):
        g = torch.randn(n, device="cuda", generator=gen) * 1e-3
        keep = torch.rand(n, device="cuda", generator=gen) < 0.01
        shared = torch.rand(n, device="cuda", generator=gen) < 0.002  # positions several ranks hold
        if r == 0:
            common = shared
        tensors.append(torch.where(keep | common, g, torch.zeros_like(g)).to(dtype))
    ex = ThreadExchange(P)
    results, errors = [None] * P, []

    def run(rank):
        try:
            torch.cuda.set_device(0)
            lba = zen.LoadBalanceAllreduce(zen.LocalGroup(P, rank), None, None)
            lba.ddp = ex.view(rank)
            results[rank] = lba.zen_sparse_comm(tensors[rank], method)
            torch.cuda.current_stream().synchronize()
        except BaseException as e:  # noqa: BLE001 - reported below, and the others must not wait for ever
            errors.append((rank, repr(e)))
            ex.barrier.abort()

    threads = [threading.Thread(target=run, args=(r,)) for r in range(P)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(timeout=100)
    assert not errors, errors
    total = torch.stack([t.double() for t in tensors]).sum(dim=0)
    scale = torch.stack([t.double().abs() for t in tensors]).sum(dim=0)
    for r in range(P):
        out = results[r]
        assert out.dtype == dtype and out.numel() == n
        assert torch.equal(out != 0, total != 0)
        err = (out.double() - total).abs()
        tol = scale * (1e-6 if dtype == torch.float32 else 2.0 ** -7)
        assert bool((err <= tol).all())
        assert torch.equal(out, results[0])


# ---------------------------------------------- bitmaps + values -> dense in one pass


def _shards(oracle, n, P, frac, dtype, seed):
    """Per rank: (members of its partition that are present, their values), as the merge of the first
    exchange would leave them: ascending indices of partition p, nonzero values."""
    rng = np.random.default_rng(seed)
    mp = oracle.mapping(n, P)
    idx, val = [], []
    for p in range(P):
        take = max(1, int(len(mp[p]) * frac))
        pick = np.sort(rng.choice(mp[p], take, replace=False))
        v = (rng.standard_normal(take) * 1e-3).astype(np.float32)
        v[v == 0] = 1e-3
        idx.append(pick)
        val.append(oracle.f32_to_bf16_bits(v) if dtype == "bf16" else v)
    return mp, idx, val


def _dense_truth(oracle, n, idx, val):
    """oracle.decode of all lists (fp32 accumulation, rounded once to the values' type)."""
    flat_i, flat_v = np.concatenate(idx), np.concatenate(val)
    f32 = oracle.decode(flat_i, flat_v, n, "f32acc")
    return oracle.f32_to_bf16_bits(f32) if flat_v.dtype == np.uint16 else f32


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("n,P,frac", [
    (1 << 16, 4, 0.05),
    ((1 << 20) + 48, 16, 0.06),      # a last tile that is not full
    (3000000, 3, 0.3),               # partitions not a power of two, n % 8192 != 0
    (1 << 20, 64, 0.02),             # the most lists the kernel takes
    (1 << 19, 2, 0.9),               # nearly every member present
    (1003 * 7, 7, 0.5),              # below one tile per ... and n % P == 0 with odd sizes
])
def test_bitmaps_to_dense_in_one_pass_matches_oracle(zen, oracle, n, P, frac, dtype):
    n = n // P * P
    mp, idx, val = _shards(oracle, n, P, frac, dtype, seed=n + P)
    bitmaps = [oracle.bitmap_encode(mp[p], idx[p]) for p in range(P)]
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(P, 0), None, None)
    got = lba.decode_bitmaps_dense([to_dev(b) for b in bitmaps], [to_dev(v) for v in val], n)
    want = _dense_truth(oracle, n, idx, val)
    assert got.numel() == n and np.array_equal(to_np(got), want)
    # the two-step path of the reference (decode_bitmap, then decode_sparse_tensors) gives the same bytes
    lba.mapping[n] = lba.calculate_mapping(n)
    idx_lists = lba.decode_bitmap([to_dev(b) for b in bitmaps], n)
    for p in range(P):
        assert np.array_equal(to_np(idx_lists[p]), idx[p])
    two_step = lba.decode_sparse_tensors(idx_lists, [to_dev(v) for v in val], n, ascending=True)
    assert torch.equal(two_step.view(torch.int16 if dtype == "bf16" else torch.int32),
                       got.view(torch.int16 if dtype == "bf16" else torch.int32))
    # a second call on the cached dictionary, other data
    mp, idx, val = _shards(oracle, n, P, frac / 2, dtype, seed=n + P + 1)
    bitmaps = [oracle.bitmap_encode(mp[p], idx[p]) for p in range(P)]
    got = lba.decode_bitmaps_dense([to_dev(b) for b in bitmaps], [to_dev(v) for v in val], n)
    assert np.array_equal(to_np(got), _dense_truth(oracle, n, idx, val))


def _far_members(mapping):
    """(list, number in the list) of the members 256 or more elements behind the one in front of them in their tile."""
    return [(p, int(j) + 1) for p, m in enumerate(mapping)
            for j in np.flatnonzero((np.diff(m) > 255) & (np.diff(m // 7168) == 0))]


@pytest.mark.parametrize("several", [False, True])
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("n, P", [(52974, 16), (141040, 16), (101419, 14)])
def test_bitmaps_to_dense_across_far_members(zen, oracle, n, P, dtype, several):
    """-0, a NaN and ordinary values in front of, at and behind a distance that does not fit its byte; the same with every
    chunk marked as one with several such distances, whose places are hashed out."""
    mp = oracle.mapping(n, P)
    p, j = _far_members(mp)[0]
    rng = np.random.default_rng(n)
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(P, 0), None, None)
    for at in (j - 1, j, j + 1):
        for bits, quiet in ((0x80000000, 0), (0x7f810000, 0x7fc10000), (0xffc00000, 0xffc00000), (0x3f800000, 0x3f800000)):
            for share in (1.0, 0.3, 0.02):
                pick = [rng.random(len(m)) < share for m in mp]
                pick[p][[j - 1, j, j + 1]] = at == np.array([j - 1, j, j + 1])
                idx = [m[t] for m, t in zip(mp, pick)]
                val = [(rng.standard_normal(len(i)) + 9.0).astype(np.float32).view(np.uint32) & 0xffff0000 for i in idx]
                val[p][np.flatnonzero(idx[p] == mp[p][at])] = bits
                want = np.zeros(n, np.uint32)
                for i, v in zip(idx, val):
                    want[i] = v
                want[mp[p][at]] = quiet
                bitmaps = [to_dev(oracle.bitmap_encode(m, i)) for m, i in zip(mp, idx)]
                values = [torch.from_numpy(v.view(np.int32)).cuda().view(torch.float32) for v in val]
                if dtype == "bf16":
                    values = [torch.from_numpy((v >> 16).astype(np.uint16).view(np.int16)).cuda().view(torch.bfloat16) for v in val]
                    want >>= 16
                got = lba.decode_bitmaps_dense(bitmaps, values, n)
                if several:
                    words = lba._dense_dicts[n][(n + 7167) // 7168 * 7296 + 512 + 255 & -256:].view(torch.int32)
                    words[:(n + 7167) // 7168 * 32].bitwise_or_(0xc000)
                    got = lba.decode_bitmaps_dense(bitmaps, values, n)
                got = got.view(torch.int32 if dtype == "f32" else torch.int16).cpu().numpy()
                assert np.array_equal(got.view(np.uint32 if dtype == "f32" else np.uint16), want), (at - j, bits, share)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("n, P", [
    (7679, 1), (7168, 2), (7681, 3), (2 * 7168 + 1, 16), (8191, 16), (8193, 17), (3 * 7168 - 1, 15),  # edges of the tiles
    (1030, 2), (16 * 8 + 5, 16), (100, 16),                      # lists of a chunk of 512 and a few more; of a few members
    (52974, 16), (83381, 16), (141040, 16), (167428, 15),        # a list with two members 256 or more elements apart
])
def test_bitmaps_to_dense_at_the_edges_of_the_dictionary(zen, oracle, n, P, dtype):
    """Every member set (lists end with their values), every other one, few and none, exact."""
    mp = oracle.mapping(n, P)
    rng = np.random.default_rng(n)
    if n > 50000:
        assert _far_members(mp)
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(P, 0), None, None)
    for share in (1.0, 0.5, 0.03, 0.0):
        idx = [m[rng.random(len(m)) < share] if share < 1 else m for m in mp]
        val = [(rng.standard_normal(len(i)) * 1e-3 + 1.0).astype(np.float32) for i in idx]
        if dtype == "bf16":
            val = [oracle.f32_to_bf16_bits(v) for v in val]
        bitmaps = [oracle.bitmap_encode(m, i) for m, i in zip(mp, idx)]
        got = lba.decode_bitmaps_dense([to_dev(b) for b in bitmaps], [to_dev(v) for v in val], n)
        assert np.array_equal(to_np(got), _dense_truth(oracle, n, idx, val)), share


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_bitmaps_to_dense_with_a_dictionary_that_leaves_the_tile(zen, oracle, dtype):
    """Distances that add up to places beyond the tile are refused, and nothing but the tensor suffers."""
    n, P = 3 * 7168, 2
    mp, idx, val = _shards(oracle, n, P, 0.4, dtype, seed=5)
    bitmaps = [to_dev(oracle.bitmap_encode(mp[p], idx[p])) for p in range(P)]
    values = [to_dev(v) for v in val]
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(P, 0), None, None)
    want = _dense_truth(oracle, n, idx, val)
    assert np.array_equal(to_np(lba.decode_bitmaps_dense(bitmaps, values, n)), want)
    dictionary = lba._dense_dicts[n]
    kept = dictionary.clone()
    dictionary[:n].fill_(255)  # the distances lie in front
    with pytest.raises(IndexError):
        lba.decode_bitmaps_dense(bitmaps, values, n)
    dictionary.copy_(kept)
    assert np.array_equal(to_np(lba.decode_bitmaps_dense(bitmaps, values, n)), want)


@pytest.mark.parametrize("form", ["strided values", "two value types"])
def test_bitmaps_to_dense_with_values_in_any_layout(zen, oracle, form):
    """Value lists that are not contiguous, or of two types (the dense tensor then has the one that holds both)."""
    n, P = 1 << 16, 4
    mp, idx, val = _shards(oracle, n, P, 0.1, "f32", seed=8)
    if form == "two value types":  # both types hold the values exactly
        val = [oracle.bf16_bits_to_f32(oracle.f32_to_bf16_bits(v)) for v in val]
    bitmaps = [to_dev(oracle.bitmap_encode(mp[p], idx[p])) for p in range(P)]
    values = [to_dev(v) for v in val]
    if form == "strided values":
        values = [torch.stack([v, torch.full_like(v, 7)], dim=1)[:, 0] for v in values]
    else:
        values[1] = values[1].bfloat16()
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(P, 0), None, None)
    got = lba.decode_bitmaps_dense(bitmaps, values, n)
    assert got.dtype == torch.float32 and np.array_equal(to_np(got), _dense_truth(oracle, n, idx, val))


def test_bitmaps_to_dense_is_complete_for_every_stream(zen):
    """When the call has returned another stream may overwrite bitmaps and values and read the tensor, without a wait."""
    n, P = 1 << 26, 16
    gen = torch.Generator(device="cuda").manual_seed(4)
    room = n // P + 8192  # (a partition's members: about n / P)
    bitmaps = [torch.randint(0, 256, (room // 8,), generator=gen, device="cuda", dtype=torch.uint8) for _ in range(P)]
    values = [torch.randn(room, generator=gen, device="cuda").bfloat16() for _ in range(P)]
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(P, 0), None, None)
    want = lba.decode_bitmaps_dense(bitmaps, values, n)
    side = torch.cuda.Stream()
    for _ in range(3):
        b, v = [t.clone() for t in bitmaps], [t.clone() for t in values]
        torch.cuda.synchronize()
        got = lba.decode_bitmaps_dense(b, v, n)
        with torch.cuda.stream(side):
            seen = got.clone()
            for t in b + v:
                t.zero_()
        torch.cuda.synchronize()
        assert torch.equal(seen, want) and torch.equal(got, want)


@pytest.mark.parametrize("special", range(12))
@pytest.mark.parametrize("n, P", [(8192, 1), (24576 + 80, 1), (3 * 8192 + 17, 3), (1 << 17, 16),
                                  (3 * 8192 + 17, 17), (1 << 16, 64)])  # places of 16 bits
def test_bitmaps_to_dense_special_values(zen, oracle, n, P, special):
    """0.0f + v for one element that needs it (-0, NaNs of either sign, quiet or not) and for those that do not, alone
    among ordinary ones, in whole tiles and in the last one; every member set, so that the values end with the list."""
    n = n // P * P
    bits = [0x8000, 0x7f81, 0x7fbf, 0x7fc0, 0x7fff, 0xff81, 0xffbf, 0xffff, 0x7f80, 0xff80, 0x0001, 0x8001][special]
    mp = oracle.mapping(n, P)
    values = [np.full(len(m), 0x3f80, np.uint16) for m in mp]
    at = [len(m) * special // 12 for m in mp]
    want = np.full(n, 0x3f80, np.uint16)
    for p in range(P):
        values[p][at[p]] = bits
        quiet = bits | 0x40 if bits & 0x7fff > 0x7f80 else 0 if bits == 0x8000 else bits
        want[mp[p][at[p]]] = quiet
    bitmaps = [to_dev(oracle.bitmap_encode(m, m)) for m in mp]
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(P, 0), None, None)
    got = lba.decode_bitmaps_dense(bitmaps, [torch.from_numpy(v.view(np.int16)).cuda().view(torch.bfloat16) for v in values], n)
    assert np.array_equal(got.view(torch.int16).cpu().numpy().view(np.uint16), want)


@pytest.mark.parametrize("n, P, n2, P2", [(1 << 18, 8, 100003, 4), (1 << 18, 32, 100003, 24), (8192 * 17, 17, 100003, 64)])
def test_bitmaps_to_dense_edge_cases(zen, oracle, n, P, n2, P2):
    mp, idx, val = _shards(oracle, n, P, 0.1, "f32", seed=3)
    bitmaps = [oracle.bitmap_encode(mp[p], idx[p]) for p in range(P)]
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(P, 0), None, None)
    want = _dense_truth(oracle, n, idx, val)
    # padding behind a bitmap (allgather_padding pads to the longest, DDPbackend.py:26-41; garbage bits past the
    # list's length are ignored, comm.py:97) and lists that do not sit in one buffer
    padded = [np.concatenate([b, np.full(5 + p, 0xFF, np.uint8)]) for p, b in enumerate(bitmaps)]
    last_bits = [len(mp[p]) % 8 for p in range(P)]
    for p in range(P):  # garbage in the unused bits of the last byte too
        if last_bits[p]:
            padded[p][len(bitmaps[p]) - 1] |= np.uint8((0xFF << last_bits[p]) & 0xFF)
    got = lba.decode_bitmaps_dense([to_dev(b) for b in padded], [to_dev(v) for v in val], n)
    assert np.array_equal(to_np(got), want)
    # -0.0 among the values becomes +0.0, as 0 + (-0) does in scatter_add_; NaN stays
    val2 = [v.copy() for v in val]
    val2[0][0] = -0.0
    val2[1][0] = np.nan
    got = to_np(lba.decode_bitmaps_dense([to_dev(b) for b in bitmaps], [to_dev(v) for v in val2], n))
    assert got.view(np.uint32)[idx[0][0]] == 0 and np.isnan(got[idx[1][0]])
    # an empty list (no bit set, no values)
    empty = [b.copy() for b in bitmaps]
    empty[2][:] = 0
    vals3 = [v if p != 2 else v[:0] for p, v in enumerate(val)]
    got = to_np(lba.decode_bitmaps_dense([to_dev(b) for b in empty], [to_dev(v) for v in vals3], n))
    want3 = want.copy()
    want3[idx[2]] = 0
    assert np.array_equal(got, want3)
    # a bitmap shorter than its list, and fewer values than set bits: the reference raises an index error
    short = [b if p != 1 else b[:-2] for p, b in enumerate(bitmaps)]
    with pytest.raises(IndexError):
        lba.decode_bitmaps_dense([to_dev(b) for b in short], [to_dev(v) for v in val], n)
    fewer = [v if p != 3 else v[:-1] for p, v in enumerate(val)]
    with pytest.raises(IndexError):
        lba.decode_bitmaps_dense([to_dev(b) for b in bitmaps], [to_dev(v) for v in fewer], n)
    # n % P != 0: some indices belong to no list (hash_index gives P for them, functions_cuda_kernel.cu:172-175)
    part = oracle.hash_index(n2, P2)
    mp2 = oracle.mapping(n2, P2)
    rng = np.random.default_rng(8)
    idx2 = [np.sort(rng.choice(m, len(m) // 3, replace=False)) for m in mp2]
    val2 = [(rng.standard_normal(len(i)) * 1e-3).astype(np.float32) + 1.0 for i in idx2]
    bm2 = [oracle.bitmap_encode(mp2[p], idx2[p]) for p in range(P2)]
    lba2 = zen.LoadBalanceAllreduce(zen.LocalGroup(P2, 0), None, None)
    got = to_np(lba2.decode_bitmaps_dense([to_dev(b) for b in bm2], [to_dev(v) for v in val2], n2))
    assert np.array_equal(got, _dense_truth(oracle, n2, idx2, val2)) and (got[part == P2] == 0).all()


@pytest.mark.parametrize("P", [1, 16])
def test_bitmaps_to_dense_of_few_lists_beyond_the_bytes(zen, P):
    """More elements than dictionaries of bytes serve: places of 16 bits, and at one list fifteen chunks to a tile, of
    which the later ones begin behind what the earlier have set."""
    from zen_repro_amd.workloads import hash_slot

    n = (1024 * 256 * 7168 + 8192 + 40) // P * P
    gen = torch.Generator(device="cuda").manual_seed(P)
    step = 1 << 26
    counts = [0] * P
    where, bits, values = [[] for _ in range(P)], [[] for _ in range(P)], [[] for _ in range(P)]
    for lo in range(0, n, step):
        t = torch.arange(lo, min(n, lo + step), device="cuda")
        part = hash_slot(t, n) // (n // P)
        chosen = torch.rand(t.numel(), generator=gen, device="cuda") < 1e-6
        if lo == 0 or lo + step >= n:  # three tiles in front, and the last ones, two thirds set
            chosen |= (torch.rand(t.numel(), generator=gen, device="cuda") < 0.66) & ((t < 3 * 8192) | (t >= n - 2 * 8192 - 100))
        for p in range(P):
            mine = part == p
            rank = torch.cumsum(mine, 0) - 1 + counts[p]
            counts[p] += int(mine.sum())
            at = mine & chosen
            where[p].append(t[at])
            bits[p].append(rank[at])
        del t, part, chosen, mine, rank, at
    bitmaps = []
    for p in range(P):
        where[p], rank = torch.cat(where[p]), torch.cat(bits[p]).cpu().numpy()
        bitmap = np.zeros((counts[p] + 7) // 8, np.uint8)
        np.bitwise_or.at(bitmap, rank >> 3, (1 << (rank & 7)).astype(np.uint8))
        bitmaps.append(to_dev(bitmap))
        values[p] = (torch.rand(where[p].numel(), generator=gen, device="cuda") + 1).to(torch.bfloat16)
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(P, 0), None, None)
    got = lba.decode_bitmaps_dense(bitmaps, values, n)
    assert got.numel() == n
    for p in range(P):
        assert torch.equal(got[where[p]], values[p])
    assert sum(int(torch.count_nonzero(part)) for part in got.split(step)) == sum(v.numel() for v in values)


# ---------------------------------------------------------- the DDP hook


class _StubBucket:
    """What the hook asks of a dist.GradBucket: its flat buffer (train.py:168)."""

    def __init__(self, tensor):
        self._t = tensor

    def buffer(self):
        return self._t


def test_comm_hook_on_one_rank(zen, oracle):
    """custom_comm_hook (train.py:167-183) with a stub bucket: the first call passes the bucket through, later
    ones return a completed future holding the compressed bucket (one rank: no exchange, train.py:178); the
    compression is the reference's sampled threshold with the sample positions given."""
    n = 1 << 20
    gen = torch.Generator(device="cuda").manual_seed(11)
    grad = (torch.randn(n, device="cuda", generator=gen) * 1e-3).to(torch.bfloat16)
    sample = torch.randint(0, n, ((n + 99) // 100,), device="cuda", generator=gen)
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(1, 0), None, None)
    hook = zen.SparseCommHook(lba, top_k=5, method=3, tp_group=zen.LocalGroup(1, 0), sample_index=lambda numel: sample)
    first = hook(None, _StubBucket(grad))
    assert first.done() and first.value() is grad  # train.py:170-174
    fut = hook(None, _StubBucket(grad))
    assert isinstance(fut, torch.futures.Future) and fut.done()
    out = fut.value()
    hook.stream.synchronize()
    # the reference's rule on the CPU: threshold = smallest of the top 5 % of the sampled magnitudes
    g = grad.float().cpu()
    s = g.abs()[sample.cpu()]
    thr = torch.topk(s, s.numel() * 5 // 100, largest=True, sorted=False)[0].min()
    want = torch.where(g.abs() >= thr, g, torch.zeros(())).to(torch.bfloat16)
    assert out.dtype == grad.dtype and torch.equal(out.cpu().view(torch.int16), want.view(torch.int16))
    # buckets of at most 4096 elements pass through (train.py:58-59)
    small = grad[:4096].clone()
    assert hook(None, _StubBucket(small)).value() is small


@pytest.mark.parametrize("method,fused", [(3, True), (3, False), (2, True), (1, True)])
def test_comm_hook_between_four_ranks(zen, method, fused):
    """The hook end to end with four ranks played by host threads: every rank's future holds the sum of all
    ranks' compressed buckets (method 3: buckets exchanged, merged, sent round as bitmaps and decoded in one
    pass), whether the threshold is handed to the all-reduce (fused) or applied to a copy of the bucket first
    as in the reference."""
    P, n = 4, 1 << 20
    gen = torch.Generator(device="cuda").manual_seed(5)
    grads = [(torch.randn(n, device="cuda", generator=gen) * 1e-3) for _ in range(P)]
    samples = [torch.randint(0, n, ((n + 99) // 100,), device="cuda", generator=gen) for _ in range(P)]
    ex = ThreadExchange(P)
    results, compressed, errors = [None] * P, [None] * P, []

    def run(rank):
        try:
            torch.cuda.set_device(0)
            lba = zen.LoadBalanceAllreduce(zen.LocalGroup(P, rank), None, None)
            lba.ddp = ex.view(rank)
            hook = zen.SparseCommHook(lba, top_k=2, method=method, tp_group=zen.LocalGroup(1, 0),
                                      sample_index=lambda numel, r=rank: samples[r], fused=fused)
            hook(None, _StubBucket(grads[rank]))  # the first call is passed through
            compressed[rank] = zen.compress_with_allgather(2, grads[rank], zen.LocalGroup(1, 0), sample_index=samples[rank])
            results[rank] = hook(None, _StubBucket(grads[rank])).value()
            hook.stream.synchronize()
            torch.cuda.current_stream().synchronize()
        except BaseException as e:  # noqa: BLE001
            errors.append((rank, repr(e)))
            ex.barrier.abort()

    threads = [threading.Thread(target=run, args=(r,)) for r in range(P)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(timeout=100)
    assert not errors, errors
    total = torch.stack([c.double() for c in compressed]).sum(dim=0)
    scale = torch.stack([c.double().abs() for c in compressed]).sum(dim=0)
    for r in range(P):
        out = results[r]
        assert out.numel() == n and torch.equal(out != 0, total != 0)
        assert bool(((out.double() - total).abs() <= scale * 1e-6).all())
        assert torch.equal(out, results[0])


@pytest.mark.parametrize("fused,headroom", [(True, 1.5), (True, 0.05), (False, 1.5)])
def test_comm_hook_on_a_bucket_of_training_size(zen, fused, headroom):
    """The hook between two ranks on a bucket of 64 Mi bf16 elements, the size at which the load balance takes
    its fast paths (asserted), with the threshold handed to the all-reduce (fused), with far too little room
    for the selection (the call is declined, falls back, learns the size and starts again), and the reference's
    way (masked copy first): all three give every rank the same tensor, the sum of the ranks' compressed
    buckets."""
    from zen_repro_amd import _lib

    P, n, top_k = 2, 64 << 20, 1
    gen = torch.Generator(device="cuda").manual_seed(21)
    grads = [(torch.randn(n, device="cuda", generator=gen) * 1e-3).to(torch.bfloat16) for _ in range(P)]
    samples = [torch.randint(0, n, ((n + 99) // 100,), device="cuda", generator=gen) for _ in range(P)]
    L = _lib.lib()
    m = zen.TensorPartition(P, 1, 3).table_sizes(n)[0]
    room = int(n * top_k / 100 * 1.5) + 4096
    assert L.zen_load_balance_path(n, m, _lib.BF16, room, P, 0, _lib.MODE_FAST) >= 2
    ex = ThreadExchange(P)
    results, compressed, errors = [None] * P, [None] * P, []

    def run(rank):
        try:
            torch.cuda.set_device(0)
            lba = zen.LoadBalanceAllreduce(zen.LocalGroup(P, rank), None, None)
            lba.ddp = ex.view(rank)
            hook = zen.SparseCommHook(lba, top_k=top_k, method=3, tp_group=zen.LocalGroup(1, 0),
                                      sample_index=lambda numel, r=rank: samples[r], fused=fused, headroom=headroom)
            hook(None, _StubBucket(grads[rank]))  # the first call is passed through
            compressed[rank] = zen.compress_with_allgather(top_k, grads[rank], zen.LocalGroup(1, 0),
                                                           sample_index=samples[rank])
            results[rank] = hook(None, _StubBucket(grads[rank])).value()
            torch.cuda.current_stream().synchronize()  # the hook made this stream wait for its own
        except BaseException as e:  # noqa: BLE001
            errors.append((rank, repr(e)))
            ex.barrier.abort()

    threads = [threading.Thread(target=run, args=(r,)) for r in range(P)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(timeout=150)
    assert not errors, errors
    # two bf16 values per index at most: their fp32 sum rounded once to bf16
    want = (compressed[0].float() + compressed[1].float()).to(torch.bfloat16)
    want = torch.where(want == 0, torch.zeros((), dtype=torch.bfloat16, device="cuda"), want)  # no negative zeros
    for r in range(P):
        assert results[r].dtype == torch.bfloat16 and results[r].numel() == n
        assert torch.equal(results[r].view(torch.int16), want.view(torch.int16))


def test_comm_hook_needs_a_backend_for_more_than_one_rank(zen):
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(2, 0), None, None)
    hook = zen.SparseCommHook(lba, top_k=1, method=3, tp_group=zen.LocalGroup(1, 0))
    grad = torch.zeros(8192, device="cuda")
    hook(None, _StubBucket(grad))
    with pytest.raises(RuntimeError):
        hook(None, _StubBucket(grad))


class _OneRank:
    """The exchange of a rank that receives `idx` and whose peers send nothing else; `cut` values of the second exchange
    are lost.  `sent`: what the second exchange was given, in copies taken on a stream of its own behind the call's."""

    def __init__(self, parts, idx, val, cut):
        self.parts, self.idx, self.val, self.cut = parts, idx, val, cut
        self.sent, self.side = [], torch.cuda.Stream()

    def allgather(self, tensor):
        return [tensor]

    def alltoallv(self, tensors, gather_splits):
        return [self.idx if tensors[0].dtype == torch.int32 else self.val]

    def allgather_padding(self, tensor):
        self.side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(self.side):
            self.sent.append(tensor.clone())
        self.side.synchronize()
        if tensor.dtype != torch.uint8:
            tensor = tensor[:tensor.numel() - self.cut]
        return [tensor] + [tensor[:0] if tensor.dtype != torch.uint8 else torch.zeros(1 << 14, dtype=torch.uint8, device="cuda")
                           for _ in range(self.parts - 1)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_allreduce_names_the_bitmap_that_is_wrong(zen, oracle, dtype):
    """An index beyond the last member raises what encode_bitmap raises, values that are too few what decode_bitmaps_dense
    does, and neither is left behind for the next call."""
    P = 4
    n = next(n for n in range(20000, 40000, P) if oracle.mapping(n, P)[0][-1] < n - 1)
    members = oracle.mapping(n, P)[0]
    good = torch.from_numpy(members[::3].astype(np.int32)).cuda()
    grad = torch.zeros(n, dtype=dtype, device="cuda")
    grad[1:50] = 1.0
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(P), None, None)

    def call(idx, cut):
        lba.ddp = _OneRank(P, idx, torch.ones(idx.numel(), dtype=dtype, device="cuda"), cut)
        return lba.zen_sparse_comm(grad, 3)

    want = torch.zeros(n, dtype=dtype, device="cuda")
    want[good.long()] = 1.0
    for _ in range(2):
        assert torch.equal(call(good, 0), want)
        with pytest.raises(IndexError, match="beyond the last member"):
            call(torch.cat([good, torch.tensor([n - 1], dtype=torch.int32, device="cuda")]), 0)
        with pytest.raises(IndexError, match="more set bits than values"):
            call(good, 1)
    assert torch.equal(call(good, 0), want)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,scale", [(30001, 1), (30000, 2)])
def test_allreduce_sends_no_bitmap_before_it_is_known_to_be_right(zen, oracle, n, scale, dtype):
    """Where list and table disagree (a length the ranks do not divide, a table of another size) an index beyond the last
    member raises in front of the second exchange: its bitmap has fewer bits than there are values, which no peer would
    notice."""
    P = 4
    rank = next(r for r in range(P) if oracle.mapping(n, P)[r][-1] < n - 1)
    members = oracle.mapping(n, P)[rank]
    idx = torch.from_numpy(np.append(members[::3], n - 1).astype(np.int32)).cuda()
    grad = torch.zeros(n, dtype=dtype, device="cuda")
    grad[1:50] = 1.0
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(P, rank), None, None, memory_scale=scale)
    lba.ddp = _OneRank(P, idx, torch.ones(idx.numel(), dtype=dtype, device="cuda"), 0)
    with pytest.raises(IndexError, match="beyond the last member"):
        lba.zen_sparse_comm(grad, 3)
    assert not lba.ddp.sent


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n", [30000, 30001])
def test_allreduce_sends_its_bitmap_in_the_order_of_the_stream(zen, oracle, n, dtype):
    """The second exchange is given the bitmap in the order of the call's stream, whatever that has in front of the marking,
    which the host waits for or does not."""
    P = 4
    members = oracle.mapping(n, P)[0]
    idx = torch.from_numpy(members[::3].astype(np.int32)).cuda()
    grad = torch.zeros(n, dtype=dtype, device="cuda")
    grad[1:50] = 1.0
    lba = zen.LoadBalanceAllreduce(zen.LocalGroup(P), None, None)
    lba.ddp = _OneRank(P, idx, torch.ones(idx.numel(), dtype=dtype, device="cuda"), 0)
    calculate = lba.calculate_mapping

    def slow(numel):  # called between the merge, which waits, and the marking
        lists = calculate(numel)
        torch.cuda._sleep(20000000)
        return lists

    lba.calculate_mapping = slow
    want = torch.zeros(n, dtype=dtype, device="cuda")
    want[idx.long()] = 1.0
    assert torch.equal(lba.zen_sparse_comm(grad, 3), want)
    bitmap, values = lba.ddp.sent
    assert np.array_equal(to_np(bitmap), oracle.bitmap_encode(members, members[::3]))
    assert torch.equal(values, torch.ones_like(values)) and values.numel() == idx.numel()
