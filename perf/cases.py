"""Workloads of this package at the sizes its users bring: what is measured when a kernel or the host path around
it changes.

A training program reaches the package in one of five ways, and each is a kind of case here:

  hook     SparseCommHook on one gradient bucket: sampled threshold, load balance, exchange, merge, second exchange
           and decode (methods 1 to 3).  The other ranks are played by a loopback exchange that hands out what they
           would have sent; top_k is 1, 5 or 10 per cent and a bucket 128 or 512 MB, as in the reference's runs.
  step     LoadBalanceAllreduce.encode_merge_flat, the call without host synchronisation: one bucket is encoded while
           the entries received for another are merged.  One bucket, or the buckets of a whole backward pass.
  dropin   compress and TensorPartition.load_balance, the reference's two calls in front of the exchange.
  table    TensorPartition.balance_sparse_tensor and get_sub_sparse_tensors, the reference's pieces one by one
           (sparse_balance fills the caller's hash table).
  merge    decode_sparse_tensors and encode_sparse_tensor on received payloads, the reference's pieces of the merge.

Everything is drawn from a seeded generator on the GPU.  Indices, orders and sums are defined bit for bit (sums are
taken in the order of arrival), so every result is exact.
"""
import math

import torch

from zen_repro_amd import (LoadBalanceAllreduce, LocalGroup, SparseCommHook, TensorPartition, compress,
                           topk_threshold)
from zen_repro_amd.workloads import hash_slot

_DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16}
_CHUNK = 1 << 26
_LEAST = {1: 10000, 5: 5000, 10: 5000}  # by top_k: a smaller sample of 1 % has no top_k per cent (4096 pass through)


def listed():
    return [
        # the last, small bucket of a backward pass (biases and norms): latency only
        {"name": "hook_9k_m2", "kind": "hook", "n": 9219, "dtype": "bf16", "parts": 4, "top_k": 10, "method": 2},
        # a small model in fp32 on four ranks, all-gather of everybody's selection
        {"name": "hook_1m_fp32_m1", "kind": "hook", "n": 1 << 20, "dtype": "fp32", "parts": 4, "top_k": 1, "method": 1},
        # a 128 MB bucket on sixteen ranks, index lists in the second exchange
        {"name": "hook_62m_m2", "kind": "hook", "n": 61953360, "dtype": "bf16", "parts": 16, "top_k": 5, "method": 2},
        # the same with the densest selection and bitmaps in the second exchange
        {"name": "hook_62m_m3", "kind": "hook", "n": 61953360, "dtype": "bf16", "parts": 16, "top_k": 10, "method": 3},
        # the default 512 MB bucket, 1 %, bitmaps
        {"name": "hook_268m_m3", "kind": "hook", "n": 1 << 28, "dtype": "bf16", "parts": 16, "top_k": 1, "method": 3},
        # one small bucket, exact top 1 % of fp32
        {"name": "step_1m_fp32", "kind": "step", "n": 1 << 20, "dtype": "fp32", "parts": 4, "data": "normal",
         "density": 0.01, "overlap": 0.2, "buckets": 1},
        # an embedding and a decoder layer of an 8B model in twelve buckets of 128 MB, exact top 0.5 % of bf16
        {"name": "step_12x62m", "kind": "step", "n": 61953360, "dtype": "bf16", "parts": 16, "data": "normal",
         "density": 0.005, "overlap": 0.25, "buckets": 12},
        # the same gradient as one tensor
        {"name": "step_743m", "kind": "step", "n": 743440384, "dtype": "bf16", "parts": 16, "data": "normal",
         "density": 0.005, "overlap": 0.25, "buckets": 1},
        # a very large fp32 gradient whose nonzeros sit in hot ranges
        {"name": "step_1g_fp32", "kind": "step", "n": 1 << 30, "dtype": "fp32", "parts": 32, "data": "hot",
         "density": 0.01, "overlap": 0.0, "buckets": 1},
        # the reference's calls in front of the exchange, mid-size fp32 bucket of an odd length
        {"name": "dropin_13m_fp32", "kind": "dropin", "n": 12865793, "dtype": "fp32", "parts": 8, "top_k": 1},
        # the reference's hash table, filled in place
        {"name": "table_16m", "kind": "table", "n": 1 << 24, "dtype": "bf16", "parts": 8, "density": 0.05, "rehash": 3},
        # the reference's merge of sixteen payloads of a 128 MB bucket
        {"name": "merge_62m", "kind": "merge", "n": 61953360, "dtype": "bf16", "parts": 16, "density": 0.05,
         "overlap": 0.25},
    ]


def _between(rng, lo, hi):
    return int(math.exp(rng.uniform(math.log(lo), math.log(hi))))


def draw(rng):
    kind = rng.choice(["hook", "hook", "step", "step", "dropin", "table", "merge"])
    dtype = rng.choice(["bf16", "bf16", "fp32"])
    if kind == "hook":
        method = rng.choice([1, 2, 3])
        parts = rng.choice([2, 4, 8, 16])
        top_k = rng.choice([1, 5, 10])
        n = _between(rng, _LEAST[top_k], min(1 << 28, 6200000 * 100 // top_k))
        if method == 1:
            n = min(n, 50000000 * 100 // (top_k * parts))
        if method == 3:  # the bitmaps' member lists and the table agree on lengths the ranks divide
            n = max(1, n // parts) * parts
        return {"kind": kind, "n": n, "dtype": dtype, "parts": parts, "top_k": top_k, "method": method}
    if kind == "step":
        data = rng.choice(["normal", "normal", "hot", "rows"])
        buckets = rng.choice([1, 1, 3])
        size = {"bf16": 2, "fp32": 4}[dtype]
        return {"kind": kind, "n": _between(rng, 1 << 16, (1 << 32) // size // buckets // 2), "dtype": dtype,
                "parts": rng.choice([4, 16, 32, 64]), "data": data, "density": rng.choice([0.001, 0.005, 0.01]),
                "overlap": rng.choice([0.0, 0.25, 0.4]), "buckets": buckets}
    parts = rng.choice([2, 4, 8, 16])
    if kind == "dropin":
        top_k = rng.choice([1, 5, 10])
        return {"kind": kind, "n": _between(rng, _LEAST[top_k], 61953360), "dtype": dtype, "parts": parts,
                "top_k": top_k}
    n = _between(rng, 5000, 61953360)
    if kind == "table":
        return {"kind": kind, "n": min(n, 1 << 24), "dtype": dtype, "parts": parts,
                "density": rng.choice([0.01, 0.05, 0.1]), "rehash": rng.choice([1, 2, 3])}
    return {"kind": kind, "n": n, "dtype": dtype, "parts": parts, "density": rng.choice([0.01, 0.05]),
            "overlap": rng.choice([0.0, 0.25])}


# ------------------------------------------------------------------ inputs

def _fixed():
    """A generator that is the same for every seed: a kind of gradient has one set of magnitudes, the seed says where
    they sit and with which sign, so that every seed selects as many entries."""
    return torch.Generator(device="cuda").manual_seed(1)


def _normal(n, dtype, gen):
    out = torch.empty(n, dtype=dtype, device="cuda")
    for lo in range(0, n, _CHUNK):
        part = out[lo:lo + _CHUNK]
        part.copy_(torch.randn(part.numel(), generator=gen, device="cuda") * 1e-3)
    return out


def _placed(base, shift, gen):
    """`base` moved round by `shift` places behind an element 0 that is never sent, with new signs."""
    out = torch.zeros(base.numel() + 1, dtype=base.dtype, device="cuda")
    out[1:1 + shift] = base[base.numel() - shift:]
    out[1 + shift:] = base[:base.numel() - shift]
    for part in out.split(_CHUNK):
        part.mul_(torch.randint(0, 2, (part.numel(),), generator=gen, device="cuda", dtype=torch.int8) * 2 - 1)
    return out


def _shift(n, gen, block=1):
    return int(torch.randint(0, n // block, (1,), generator=gen, device="cuda")) * block


def _dense_gradient(n, dtype, gen):
    """(gradient, 1 % sample positions): normal values, and the sample the threshold is taken from."""
    fixed, shift = _fixed(), _shift(n - 1, gen)
    base = _normal(n - 1, dtype, fixed)
    at = torch.randint(0, n - 1, (math.ceil(0.01 * n),), generator=fixed, device="cuda")
    return _placed(base, shift, gen), (at + shift) % (n - 1) + 1


def _sparse(n, dtype, where, density, gen):
    """A gradient with `density` of its elements nonzero: `hot` in Zipf(1.3)-filled blocks of 4096 elements, `rows`
    in whole rows of 768, `even` anywhere."""
    fixed = _fixed()
    out = _normal(n - 1, dtype, fixed)
    block = {"hot": 4096, "rows": 768, "even": 1}[where]
    count = -(-n // block)
    if where == "hot":
        w = torch.arange(1, count + 1, dtype=torch.float64, device="cuda").pow(-1.3)
        want = (w / w.sum() * (density * n)).clamp_(max=block)
        room = block - want
        spill = density * n - want.sum()
        fill = (want + torch.where(torch.cumsum(room, 0) <= spill, room, torch.zeros_like(room))) / block
    elif where == "rows":
        fill = torch.zeros(count, device="cuda")
        fill[torch.randperm(count, generator=fixed, device="cuda")[:max(1, int(count * density))]] = 1.0
    step = max(1, _CHUNK // block)
    for b in range(0, count, step):
        part = out[b * block:min(n, (b + step) * block)]
        chance = density if where == "even" else fill[b:b + step].to(torch.float32).repeat_interleave(block)[:part.numel()]
        part.mul_(torch.rand(part.numel(), generator=fixed, device="cuda") < chance)
    return _placed(out, _shift(n - 1, gen, block), gen)


def _destination(n, parts):
    """The indices of destination 0's range, in the order of their level-1 slots."""
    m = n // parts * parts
    idx, slots = [], []
    for lo in range(0, n, _CHUNK):
        t = torch.arange(max(lo, 1), min(n, lo + _CHUNK), device="cuda")
        s = hash_slot(t, m)
        mine = s < m // parts
        idx.append(t[mine])
        slots.append(s[mine])
    idx, slots = torch.cat(idx), torch.cat(slots)
    order = torch.sort(slots, stable=True)[1]
    return idx[order].to(torch.int32)


def _payloads(members, count, density, overlap, gen):
    """What `count` ranks send to one destination: each a selection of its members in slot order, `overlap` of it
    shared by all.  The rest is different from rank to rank as long as there are members enough."""
    size = members.numel()
    shared, own = int(size * density * overlap), max(1, int(size * density * (1 - overlap)))
    if shared + count * own > size:
        pool = torch.rand(size, generator=gen, device="cuda") < density * overlap
        return [members[pool | (torch.rand(size, generator=gen, device="cuda") < density * (1 - overlap))]
                for _ in range(count)]
    at = torch.randperm(size, generator=gen, device="cuda")[:shared + count * own].to(torch.int32)
    pool = at[:shared]
    return [members[torch.sort(torch.cat([pool, part]))[0]] for part in at[shared:].split(own)]


def _values(idx, dtype, gen):
    """Values for `idx`, those of one index with one sign (a sum that cancels exactly is not sent on)."""
    size = torch.randn(idx.numel(), generator=gen, device="cuda").abs() * 1e-3 + 1e-6
    return torch.where((idx & 4) == 0, size, -size).to(dtype)


def _cut(flat, sizes):
    return list(torch.split(flat, sizes))


class _Bucket:
    def __init__(self, tensor):
        self.tensor = tensor

    def buffer(self):
        return self.tensor


class _Loopback:
    """The exchange calls of the reference's backend on one GPU: what the other ranks send is there already, this
    rank's share is put beside it.  An all-to-all goes from and into one flat buffer, an all-gather goes from a
    padded buffer into one tensor a rank."""

    def __init__(self, received, gathered, room):
        # received: the other ranks' buckets by type, each as (buffer, room in front, sizes); gathered: the other
        # ranks' lists of the second exchange by type; room: entries a rank may send there
        self.received, self.gathered = received, gathered
        self.padded = {t: torch.zeros(room, dtype=t, device="cuda") for t in gathered}
        self.sent = []

    def allgather(self, tensor):
        self.sent.append(tensor)
        return [tensor]

    def alltoallv(self, tensors, splits):
        self.sent.append(torch.cat(tensors))
        buffer, room, sizes = self.received[tensors[0].dtype]
        own = tensors[0].numel()
        buffer[room - own:room].copy_(tensors[0])
        return _cut(buffer[room - own:], [own] + sizes)

    def allgather_padding(self, tensor):
        padded = self.padded[tensor.dtype]
        padded[:tensor.numel()].copy_(tensor)
        self.sent.append(padded)
        return [tensor] + self.gathered[tensor.dtype]


def _second_exchange(case, mapping, gen):
    """The other ranks' lists of the second exchange (method 1: of the only one), by type."""
    n, parts, dtype = case["n"], case["parts"], _DTYPES[case["dtype"]]
    density = case["top_k"] / 100
    if case["method"] == 1:
        lists = []
        for _ in range(parts - 1):
            lists.append(torch.cat([torch.nonzero(torch.rand(min(_CHUNK, n - lo), generator=gen, device="cuda") < density)
                                    .view(-1) + lo for lo in range(0, n, _CHUNK)]))
    else:
        merged = _merged_share(density, 0.25, parts)
        marked = torch.cat([torch.rand(min(_CHUNK, n - lo), generator=gen, device="cuda") < merged
                            for lo in range(0, n, _CHUNK)])
        if case["method"] == 3:
            lists, weights = [], torch.tensor([1, 2, 4, 8, 16, 32, 64, 128], dtype=torch.uint8, device="cuda")
            bitmaps = []
            for members in mapping[1:]:
                bits = torch.zeros(-(-members.numel() // 8) * 8, dtype=torch.uint8, device="cuda")
                bits[:members.numel()] = marked[members]
                lists.append(members[marked[members]])
                bitmaps.append((bits.view(-1, 8) * weights).sum(1, dtype=torch.uint8))
            return {torch.uint8: bitmaps, dtype: [_values(x, dtype, gen) for x in lists]}
        m = n // parts * parts
        marked[0] = False
        t = torch.nonzero(marked).view(-1)
        part = torch.cat([(hash_slot(x, m) // (m // parts)).to(torch.uint8) for x in t.split(_CHUNK)])
        lists = [t[part == p] for p in range(1, parts)]
    return {torch.int64: lists, dtype: [_values(x, dtype, gen) for x in lists]}


def _prepare_hook(case, gen):
    n, parts, dtype = case["n"], case["parts"], _DTYPES[case["dtype"]]
    lba = LoadBalanceAllreduce(LocalGroup(parts), None, None)
    if case["method"] == 3:
        lba.mapping[n] = lba.calculate_mapping(n)  # kept for as long as the program runs, like the reference's
    received = {}
    if case["method"] != 1:
        lists = _payloads(_destination(n, parts), parts - 1, case["top_k"] / 100, 0.25, gen)
        sizes = [x.numel() for x in lists]
        room = n // parts  # nobody sends more than a whole index range
        front = torch.zeros(room, dtype=torch.int32, device="cuda")
        received[torch.int32] = (torch.cat([front] + lists), room, sizes)
        received[dtype] = (_values(received[torch.int32][0], dtype, gen), room, sizes)
    room = n // parts + 8 if case["method"] != 1 else min(n, int(n * case["top_k"] / 50) + 4096)
    lba.ddp = _Loopback(received, _second_exchange(case, lba.mapping.get(n), gen), room)
    grad, sample = _dense_gradient(n, dtype, gen)
    hook = SparseCommHook(lba, case["top_k"], case["method"], LocalGroup(1), sample_index=lambda numel: sample)
    bucket = _Bucket(grad)
    hook(None, bucket)  # the first bucket passes through uncompressed
    return {"kind": "hook", "hook": hook, "bucket": bucket, "ddp": lba.ddp}


def _prepare_step(case, gen):
    n, parts, dtype, density = case["n"], case["parts"], _DTYPES[case["dtype"]], case["density"]
    lba = LoadBalanceAllreduce(LocalGroup(parts), None, None)
    members = _destination(n, parts)
    buckets = []
    for _ in range(case["buckets"]):
        if case["data"] == "normal":
            k = max(1, int(n * density))
            grad = _dense_gradient(n, dtype, gen)[0]
            sent = int(topk_threshold(grad, k)[1])
            capacity = int(k * 1.25) + 4096
        else:
            k = 0
            grad = _sparse(n, dtype, case["data"], density, gen)
            sent = int(torch.count_nonzero(grad))
            capacity = int(sent * 1.25) + 4096
        lists = _payloads(members, parts, density, case["overlap"], gen)
        idx = torch.cat(lists)
        val = _values(idx, dtype, gen)
        merged = lba.merge_sparse(idx, val, n)[0].numel()
        buckets.append({"grad": grad, "k": k, "capacity": min(n, capacity), "idx": idx, "val": val, "sent": sent,
                        "merged": merged})
    return {"kind": "step", "lba": lba, "n": n, "buckets": buckets}


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind = case["kind"]
    if kind == "hook":
        return _prepare_hook(case, gen)
    if kind == "step":
        return _prepare_step(case, gen)
    n, parts, dtype = case["n"], case["parts"], _DTYPES[case["dtype"]]
    if kind == "dropin":
        grad, sample = _dense_gradient(n, dtype, gen)
        return {"kind": kind, "grad": grad, "partition": TensorPartition(parts, 1, 3), "sample": sample,
                "top_k": case["top_k"]}
    if kind == "table":
        return {"kind": kind, "grad": _sparse(n, dtype, "even", case["density"], gen),
                "partition": TensorPartition(parts, 1, case["rehash"])}
    lists = _payloads(_destination(n, parts), parts, case["density"], case["overlap"], gen)
    sizes = [x.numel() for x in lists]
    idx = torch.cat(lists)
    return {"kind": kind, "lba": LoadBalanceAllreduce(LocalGroup(parts), None, None), "n": n,
            "idx": _cut(idx, sizes), "val": _cut(_values(idx, dtype, gen), sizes)}


# --------------------------------------------------------------------- run

_merge_streams = {}  # a program has one stream for its merges


def _merge_stream():
    device = torch.cuda.current_device()
    if device not in _merge_streams:
        _merge_streams[device] = torch.cuda.Stream()
    return _merge_streams[device]


def _run_step(state):
    lba, buckets = state["lba"], state["buckets"]
    main, side = torch.cuda.current_stream(), _merge_stream()
    side.wait_stream(main)  # what was received is there
    out = []
    for i, b in enumerate(buckets):
        nxt = buckets[i + 1] if i + 1 < len(buckets) else None
        more = {"next_tensor": nxt["grad"], "next_k": nxt["k"], "next_capacity": nxt["capacity"]} if nxt else {}
        (idx, val, splits, status), (m_idx, m_val, count, m_status) = lba.encode_merge_flat(
            lba.tensor_partition, b["grad"], b["capacity"], b["k"], b["idx"], b["val"], state["n"], merge_stream=side,
            **more)
        out.append({"idx": idx[:b["sent"]], "val": val[:b["sent"]], "splits": splits, "status": status,
                    "m_idx": m_idx[:b["merged"]], "m_val": m_val[:b["merged"]], "count": count, "m_status": m_status})
    main.wait_stream(side)  # the caller goes on with both
    if len(out) > 4:  # a long pass: the buffers and sizes of every bucket
        return [{key: o[key] for key in ("idx", "val", "splits", "m_idx", "m_val")} for o in out]
    return out


def run(state):
    kind = state["kind"]
    if kind == "hook":
        state["ddp"].sent = []
        dense = state["hook"](None, state["bucket"]).value()
        return {"dense": dense, "sent": state["ddp"].sent}
    if kind == "step":
        return _run_step(state)
    partition = state["partition"] if kind != "merge" else None
    if kind == "dropin":
        masked = compress(state["top_k"], state["grad"], state["sample"])
        indices, values, splits = partition.load_balance(masked)
        return {"masked": masked, "indices": torch.cat(indices), "values": torch.cat(values), "splits": splits}
    if kind == "table":
        grad = state["grad"]
        memory, serial = partition.balance_sparse_tensor(grad)
        found = [partition.get_sub_sparse_tensors(grad, t) for t in (memory, serial)]
        indices, values = ([t for pair in zip(found[0][i], found[1][i]) for t in pair] for i in (0, 1))
        return {"memory": memory, "serial": serial, "indices": torch.cat(indices), "values": torch.cat(values),
                "splits": found[0][2] + found[1][2]}
    dense = state["lba"].decode_sparse_tensors(state["idx"], state["val"], state["n"])
    idx, val = state["lba"].encode_sparse_tensor(dense)
    return {"dense": dense, "idx": idx, "val": val}


# ------------------------------------------------------------ what it takes

def _merged_share(density, overlap, ranks):
    """The share of a destination's index range that `ranks` selections of `density` cover together."""
    return density * overlap + (1 - density * overlap) * (1 - (1 - density * (1 - overlap)) ** ranks)


def work(case):
    n, parts, s = case["n"], case["parts"], {"bf16": 2, "fp32": 4}[case["dtype"]]
    kind = case["kind"]
    density = case["density"] if "density" in case else case["top_k"] / 100
    entries = n * density
    if kind == "hook":
        total = n * s + (8 + s) * math.ceil(0.01 * n) + n * s  # the bucket, its sample, the result
        if case["method"] == 1:
            return {"bytes": total + entries * (8 + s) * (1 + parts)}
        merged = n * _merged_share(density, 0.25, parts)
        total += 2 * entries * (4 + s)  # the buckets that leave and the entries that arrive
        if case["method"] == 2:
            return {"bytes": total + merged * (8 + s) * (1 + 1 / parts)}
        return {"bytes": total + (merged * s + n / 8) * (1 + 1 / parts)}
    if kind == "step":
        merged = n / parts * _merged_share(density, case["overlap"], parts)
        one = n * s + 2 * entries * (4 + s) + merged * 8 + parts * 8
        return {"bytes": one * case["buckets"]}
    if kind == "dropin":
        return {"bytes": 2 * n * s + (8 + s) * math.ceil(0.01 * n) + entries * (4 + s)}
    if kind == "table":
        # the table and the overflow region come out, are read again for the lists, and the lists come out
        return {"bytes": n * s + 2 * (4 * n + 4 * (n // 10)) + entries * (4 + s)}
    merged = n / parts * _merged_share(density, case["overlap"], parts)
    return {"bytes": entries * (4 + s) + n * s + merged * (8 + s)}


def tolerance(case):
    return "exact"
