"""Loader of libzen_hip.so (the C-ABI of include/zen_hip.h) and the small
amount of torch plumbing every wrapper shares: dtype codes, stream handles,
cached workspaces and status words.  There is no fallback: if the library is
missing or a call fails, an exception is raised."""
import ctypes
import os
import sys
import threading

import torch  # first: makes the process use torch's HIP runtime for libzen_hip too


class _Unbuilt:
    """Stands for zen_host.cpp's module where that does not load: whoever comes to use it is told."""

    def __init__(self, why):
        self._why = why

    def __getattr__(self, name):
        raise RuntimeError("zen_repro_amd/_host.so does not load: build it with `make -C zen_repro_amd/csrc` "
                           f"(or __graft_entry__.build()); there is no fallback path ({self._why})")


try:
    from . import _host as host  # zen_host.cpp: what the calls do around the library's functions
except ImportError as e:  # not built, or for another torch
    host = _Unbuilt(str(e))

F32, BF16 = 0, 1
OK, EINVAL, EHIP, EWORKSPACE = 0, -1, -2, -3
STAT_SERIAL_OVERFLOW, STAT_CAPACITY, STAT_INTERNAL, STAT_BAD_INDEX, STAT_RETRY = 1, 2, 4, 8, 16
MODE_FAST, MODE_GENERAL = 0, 1
MODE_ZEROED = 0x100  # zen_merge: the head of the workspace is zero (and stays so); zen_load_balance: splits is zero
MODE_PREPARED, MODE_SECOND, MODE_DISCARD = 0x200, 0x400, 0x800  # zen_load_balance: the sample was taken ahead (zen_load_balance_prepare)
MODE_FLOOR = 0x1000  # zen_load_balance with k > 0: thr holds a key close to the threshold, no sample is taken
MODE_SLABS = 0x2000  # fast mode without the wide-bucket path (bucket slabs where they fit)
MODE_NO_SAMPLES = 0x4000  # zen_load_balance with k == 0: no sample taken ahead waits in the table
MODE_WIDE = 0x8000  # fast mode on the wide buckets wherever they fit (zen_load_balance)

_HERE = os.path.dirname(os.path.abspath(__file__))
# ZEN_HIP_LIB names another build of the library (a debug build, a build with other compile-time settings)
LIB_PATH = os.environ.get("ZEN_HIP_LIB") or os.path.join(_HERE, "csrc", "libzen_hip.so")

# ZEN_ABI_VERSION of include/zen_hip.h this loader's signatures and structs are written for
ABI_VERSION = 11
TABLE_SIZES_MOST = 1024  # ZEN_TABLE_SIZES_MOST

_lib = None


class EncodeMergeArgs(ctypes.Structure):
    """zen_encode_merge_args of include/zen_hip.h."""
    _vp, _i32, _i64, _sz = ctypes.c_void_p, ctypes.c_int, ctypes.c_int64, ctypes.c_size_t
    _fields_ = [
        ("input", _vp), ("dtype", _i32), ("n", _i64), ("m", _i64), ("partitions", _i32), ("rehash", _i32),
        ("thr", _vp), ("k", _i64), ("thr_out", _vp), ("out_idx", _vp), ("out_val", _vp), ("capacity", _i64),
        ("splits", _vp), ("table", _vp), ("mode", _i32), ("workspace", _vp), ("workspace_bytes", _sz),
        ("status", _vp),
        ("recv_idx", _vp), ("recv_idx64", _i32), ("recv_val", _vp), ("r", _i64), ("dense_n", _i64),
        ("merged_idx", _vp), ("merged_idx64", _i32), ("merged_val", _vp), ("merged_capacity", _i64),
        ("merged_count", _vp), ("merge_mode", _i32), ("merge_workspace", _vp), ("merge_workspace_bytes", _sz),
        ("merge_status", _vp),
        ("stream", _vp), ("merge_stream", _vp),
        ("next_input", _vp), ("next_k", _i64), ("next_n", _i64), ("next_m", _i64), ("next_capacity", _i64),
        ("next_table", _vp),
    ]


def build():
    """Compile libzen_hip.so for gfx950 with hipcc (cross-compiles without a GPU)."""
    import subprocess

    subprocess.check_call(["make", "-C", os.path.join(_HERE, "csrc"), "-B", "-j8", "all"],
                          stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    return LIB_PATH


def lib():
    global _lib
    if _lib is not None:
        return _lib
    if not os.path.exists(LIB_PATH):
        raise RuntimeError(
            f"{LIB_PATH} is missing: build it with `make -C zen_repro_amd/csrc` "
            "(or __graft_entry__.build()); there is no fallback path")
    if host.ABI_VERSION != ABI_VERSION:
        raise RuntimeError("zen_repro_amd/_host.so is of another version: build it with `make -C zen_repro_amd/csrc`")
    L = ctypes.CDLL(LIB_PATH)
    vp, i32, i64, sz = ctypes.c_void_p, ctypes.c_int, ctypes.c_int64, ctypes.c_size_t
    sig = {
        "zen_abi_version": (i32, []),
        "zen_last_error": (ctypes.c_char_p, []),
        "zen_hash_index": (i32, [vp, i64, i32, vp]),
        "zen_mapping_workspace": (sz, [i64, i32]),
        "zen_mapping": (i32, [i64, i32, vp, vp, vp, sz, vp, vp]),
        "zen_bitmap_words": (sz, [i64]),
        "zen_bitmap_rank_words": (sz, [i64]),
        "zen_bitmap_ranks": (i32, [vp, i64, i64, vp, vp]),
        "zen_bitmap_encode": (i32, [vp, i64, vp, i32, i64, vp, vp, i64, vp, vp, vp]),
        "zen_bitmap_encode_status": (i32, [vp, i64, vp, i32, i64, vp, vp, i64, vp, vp, vp, i64, vp]),
        "zen_bitmap_decode_workspace": (sz, [i64]),
        "zen_bitmap_decode": (i32, [vp, i64, vp, i64, vp, i64, vp, vp, sz, vp, vp]),
        "zen_sparse_balance": (i32, [vp, i32, i64, vp, i64, vp, i64, vp, i32, i32, vp, vp]),
        "zen_balance_tables": (i32, [vp, i32, i64, vp, i64, vp, i64, vp, i32, i32, vp, vp, i64, vp]),
        "zen_encode_merge_samples_next": (i32, [i64, i64, i32, i64, i32, i64, i32]),
        "zen_topk_threshold_workspace": (sz, []),
        "zen_topk_threshold": (i32, [vp, i32, i64, i64, vp, vp, sz, vp]),
        "zen_topk_threshold_static": (i32, [vp, i32, i64, i64, vp, vp]),
        "zen_round_compact_workspace": (sz, [i64]),
        "zen_round_compact": (i32, [vp, i32, vp, vp, i64, i32, vp, vp, vp, vp, sz, vp, vp]),
        "zen_sample_threshold_workspace": (sz, [i64, i32]),
        "zen_sample_threshold": (i32, [vp, i32, i64, vp, i64, i64, vp, vp, sz, vp, vp]),
        "zen_compress": (i32, [vp, i32, i64, vp, vp, vp]),
        "zen_select_workspace": (sz, [i64, i32]),
        "zen_select": (i32, [vp, i32, i64, vp, vp, i32, vp, i64, vp, vp, sz, vp, vp]),
        "zen_select_count": (i32, [vp, i32, i64, vp, vp, i32, vp, i64, vp, vp, sz, vp, vp, i64, vp]),
        "zen_load_balance_workspace": (sz, [i64, i64, i32, i64, i32]),
        "zen_load_balance": (i32, [vp, i32, i64, i64, i32, i32, vp, i64, vp, vp, vp, i64, vp, vp, i32, vp, sz, vp, vp]),
        "zen_load_balance_sizes": (i32, [vp, i32, i64, i64, i32, i32, vp, i64, vp, vp, vp, i64, vp, vp, i32, vp, sz, vp, vp, i64,
                                         vp]),
        "zen_load_balance_prepare": (i32, [vp, i32, i64, i64, i32, i64, i64, vp, i32, vp, sz, vp]),
        "zen_load_balance_path": (i32, [i64, i64, i32, i64, i32, i64, i32]),
        "zen_merge_workspace": (sz, [i64, i64]),
        "zen_merge_path": (i32, [i64, i64, i32]),
        "zen_merge_zero_bytes": (sz, []),
        "zen_merge": (i32, [vp, i32, vp, i32, i64, i64, vp, i32, vp, i64, vp, i32, vp, sz, vp, vp]),
        "zen_encode_merge": (i32, [ctypes.POINTER(EncodeMergeArgs)]),
        "zen_merge_rounded": (i32, [vp, i32, vp, i32, i64, i64, vp, i32, vp, i64, vp, i32, vp, sz, vp, vp]),
        "zen_merge_rounded_count": (i32, [vp, i32, vp, i32, i64, i64, vp, i32, vp, i64, vp, i32, vp, sz, vp, vp, i64, vp]),
        "zen_decode_dense_lists_status": (i32, [vp, i32, vp, i32, vp, i32, vp, i64, vp, sz, vp, vp, i64, vp]),
        "zen_decode_dense_lists": (i32, [vp, i32, vp, i32, vp, i32, vp, i64, vp, sz, vp, vp]),
        "zen_decode_dense_workspace": (sz, [i64, i64]),
        "zen_decode_dense": (i32, [vp, i32, vp, i32, i64, vp, i64, i32, vp, sz, vp, vp]),
        "zen_decode_dense_status": (i32, [vp, i32, vp, i32, i64, vp, i64, i32, vp, sz, vp, vp, i64, vp]),
        "zen_decode_dense_sorted_workspace": (sz, [i64, i32]),
        "zen_decode_dense_sorted": (i32, [vp, i32, vp, i32, ctypes.POINTER(ctypes.c_int64), i32, vp, i64, vp, sz, vp, vp]),
        "zen_bitmap_dense_dict_bytes": (sz, [i64, i32]),
        "zen_bitmap_dense_dict": (i32, [i64, i32, vp, ctypes.POINTER(ctypes.c_int64), vp]),
        "zen_bitmap_dense_workspace": (sz, [i64, i32]),
        "zen_bitmap_dense": (i32, [vp, i64, i32, vp, ctypes.POINTER(ctypes.c_int64), vp, i32,
                                   ctypes.POINTER(ctypes.c_int64), vp, vp, sz, vp, vp]),
        "zen_bitmap_dense_lists_status": (i32, [vp, i64, i32, vp, vp, vp, i32, vp, vp, vp, sz, vp, vp, i64, vp]),
        "zen_bitmap_dense_lists": (i32, [vp, i64, i32, vp, vp, vp, i32, vp, vp, vp, sz, vp, vp]),
        "zen_sort_pairs_workspace": (sz, [i64]),
        "zen_sort_pairs": (i32, [vp, vp, i64, vp, i32, vp, sz, vp, vp]),
        "zen_bucket_sort_fits": (i32, [i64, ctypes.c_uint32]),
        "zen_bucket_sort_pairs": (i32, [vp, vp, i64, vp, ctypes.c_uint32, vp, sz, vp, vp]),
        "zen_host_words_alloc": (i32, [i64, ctypes.POINTER(vp)]),
        "zen_host_words_free": (i32, [vp]),
        "zen_read_back": (i32, [vp, i32, i32, vp, i32, i32, vp, i32, i32, vp, i64, vp]),
        "zen_count": (i32, [vp, i32, i64, vp, vp, vp]),
        "zen_table_lists_workspace": (sz, [i64, i32]),
        "zen_table_find": (i32, [vp, i64, i32, i64, vp, vp, sz, vp, vp]),
        "zen_table_find_sizes": (i32, [vp, i64, i32, i64, vp, vp, vp, sz, vp, vp, i64, vp]),
        "zen_table_gather": (i32, [vp, i64, i32, vp, i32, i64, vp, vp, i64, vp, sz, vp]),
        "zen_stream_read": (i32, [vp, sz, vp, vp]),
        "zen_profile_enable": (i32, [i32]),
        "zen_profile_only": (i32, [i32]),
        "zen_profile_every": (i32, [i32]),
        "zen_profile_tags": (i32, []),
        "zen_profile_name": (ctypes.c_char_p, [i32]),
        "zen_profile_read": (i32, [i32, ctypes.POINTER(ctypes.c_double), ctypes.POINTER(ctypes.c_int64)]),
    }
    for name, (res, args) in sig.items():
        fn = getattr(L, name)
        fn.restype, fn.argtypes = res, args
    if L.zen_abi_version() != ABI_VERSION:
        raise RuntimeError("libzen_hip.so: unexpected ABI version")
    _lib = L
    return L


def check(code, what):
    if code == OK:
        return
    msg = lib().zen_last_error().decode(errors="replace")
    if code == EINVAL:
        raise ValueError(f"{what}: {msg}")
    raise RuntimeError(f"{what} failed ({code}): {msg}")


def dtype_code(t):
    if t.dtype == torch.float32:
        return F32
    if t.dtype == torch.bfloat16:
        return BF16
    raise AssertionError(f"gradient dtype must be bfloat16 or float32, got {t.dtype}")


def ptr(t):
    """What a void * argument takes: the address, or None."""
    return t.data_ptr() if t is not None else None


def device_index(device):
    """Index of a torch device (or of the current one if it names none)."""
    try:
        index = device.index
        if index.__class__ is int:
            return index
    except AttributeError:
        pass
    index = torch.device(device).index
    return index if index is not None else torch.cuda.current_device()


# The current stream of the device of that index as an integer handle (hipStream_t).  Asked on every call of the hot
# path: torch's own shortcut, where it has one, is several microseconds quicker than a Stream object.
current_handle = getattr(torch._C, "_cuda_getCurrentRawStream",
                         lambda index: torch.cuda.current_stream(index).cuda_stream)


def stream_handle(device):
    return current_handle(device_index(device))


def stream_of(device):
    return stream_handle(device)


def require_gpu(t, name):
    # extensions/cuda/functions.py:5-7 asserts; functions_cuda.cpp:11-13 raises RuntimeError
    if t.is_cuda and t.is_contiguous():
        return
    assert t.is_cuda, f"{name} must be a GPU tensor"
    raise RuntimeError(f"{name} must be contiguous")


def untransformed(*tensors):
    """Whether nothing watches or rewrites torch's operations on these: no forward-mode level, vmap or other
    transform, no torch mode, no subclass.  A kernel call in their place would go unnoticed."""
    return (torch.autograd.forward_ad._current_level < 0 and torch._C._functorch.peek_interpreter_stack() is None
            and not torch._C._len_torch_function_stack() and not torch._C._len_torch_dispatch_stack()
            and all(type(t) in _PLAIN for t in tensors))


_PLAIN = (torch.Tensor, torch.nn.Parameter)


class Kept:
    """A buffer that is kept from call to call, and the streams it is used on.  A stream other than the one it
    was made on waits for its making (its fill) at its first use there, and the memory is not handed out again
    before the work of every such stream is done.  Neither while a stream is being captured into a graph: what
    came before the capture has finished, and whoever replays the graph keeps the buffer."""

    __slots__ = ("buf", "maker", "seen")

    def __init__(self, buf, maker):
        self.buf = buf
        self.maker = maker
        self.seen = {maker.cuda_stream}

    def join(self, stream, new=False):
        """A stream that is not in `seen` comes to use the buffer (`new`: which has just been made, in the same
        capture if there is one)."""
        if new or not torch.cuda.is_current_stream_capturing():
            stream.wait_stream(self.maker)
            self.buf.record_stream(stream)
            self.seen.add(stream.cuda_stream)

    def left_running(self, device, *inputs):
        """A call that waits for its sizes has returned while its last kernels may still use the buffer on the
        current stream: every other stream waits for that at its next use, like for the making.  `inputs` (None:
        not given): tensors those kernels still read, whose memory is not handed out before they have, also if it
        belongs to another stream's pool and its owner drops it now."""
        if len(self.seen) > 1:  # else no stream but this one has used it
            self.maker = torch.cuda.current_stream(device)
            self.seen = {self.maker.cuda_stream}
        for t in inputs:
            if t is not None:
                t.record_stream(self.maker)


class Scratch:
    """Cache of raw byte buffers per device and host thread, grown on demand
    and reused.  A buffer is tied to the stream order of its users, like any
    torch tensor; two threads that enqueue calls side by side (their kernels
    interleave even on one stream) never share one, and a thread's buffers go
    when the thread does."""

    def __init__(self):
        self._local = threading.local()

    def _bufs(self):
        bufs = getattr(self._local, "bufs", None)
        if bufs is None:
            bufs = self._local.bufs = {}
        return bufs

    def get(self, device, name, nbytes, zero=False, stream=None):
        """The buffer `name` of at least `nbytes` bytes (zeroed when it is made if `zero`), for use on `stream`
        (None: the current one)."""
        index = device_index(device)
        key = (index, name)
        try:
            bufs = self._local.bufs
        except AttributeError:
            bufs = self._bufs()
        kept = bufs.get(key)
        if kept is None or kept.buf.numel() < nbytes:
            alloc = torch.zeros if zero else torch.empty
            buf = alloc(max(int(nbytes), 256), dtype=torch.uint8, device=device)
            kept = bufs[key] = Kept(buf, torch.cuda.current_stream(index))
            if stream is not None and stream.cuda_stream not in kept.seen:
                kept.join(stream, new=True)
        elif (stream.cuda_stream if stream is not None else current_handle(index)) not in kept.seen:
            kept.join(torch.cuda.current_stream(index) if stream is None else stream)
        return kept.buf

    def left_running(self, device, name, *inputs):
        """See Kept.left_running."""
        self._bufs()[device_index(device), name].left_running(device, *inputs)

    def drop(self):
        """Forget the calling thread's buffers."""
        self._bufs().clear()


scratch = Scratch()


class ZeroPool:
    """Small zeroed device buffers (status words, counters, split sizes).  A
    fill kernel for four bytes costs the device as much as one for a megabyte,
    and a call on the hot path needs two or three such buffers: they are cut
    from a block that one fill zeroed.  Every piece is handed out once (its
    holder may write to it).  A block belongs to the host thread and the stream
    that were current when it was made, so a piece is only ever used in the
    stream order of its block's fill."""

    BLOCK = 1 << 16
    ALIGN = 16
    WORDS = 4096  # of one type to a block of single words

    def __init__(self):
        self._local = threading.local()

    def native(self):
        """The same for this thread's calls through zen_host.cpp, whose blocks are their own."""
        try:
            return self._local.native
        except AttributeError:
            self._local.native = host.Zeros()
            return self._local.native

    _SIZES = {torch.int32: 4, torch.int64: 8, torch.uint8: 1, torch.float32: 4}

    def _blocks(self):
        blocks = getattr(self._local, "blocks", None)
        if blocks is None:
            blocks = self._local.blocks = {}
        return blocks

    def word(self, device, dtype):
        """take(device, 1, dtype) for int32 and int64, which calls need most."""
        blocks = self._blocks()
        key = (device_index(device), stream_handle(device), dtype)
        entry = blocks.get(key)
        if entry is None or entry[1] == self.WORDS:
            entry = blocks[key] = [torch.zeros(self.WORDS, dtype=dtype, device=device), 0]
        at = entry[1]
        entry[1] = at + 1
        return entry[0][at:at + 1]

    def take(self, device, count, dtype, stream=None):
        """`count` zeros of `dtype`.  `stream`: a stream beside the current one that uses them too, and may be far
        ahead of it: it waits for the fill of every block, once."""
        size = self._SIZES.get(dtype)
        if size is None:
            size = torch.empty((), dtype=dtype).element_size()
        nbytes = count * size
        if nbytes > self.BLOCK // 4:
            piece = torch.zeros(count, dtype=dtype, device=device)
            if stream is not None:
                stream.wait_stream(torch.cuda.current_stream(device))
            return piece
        blocks = self._blocks()
        key = (device_index(device), stream_handle(device))
        entry = blocks.get(key)
        if entry is None or entry[1] + nbytes > self.BLOCK:
            # the block, how much of it is handed out, views of it by element type (made when first asked for), and
            # the streams its fill lies before
            entry = blocks[key] = [torch.zeros(self.BLOCK, dtype=torch.uint8, device=device), 0, {}, {key[1]}]
        if stream is not None and stream.cuda_stream not in entry[3]:
            stream.wait_stream(torch.cuda.current_stream(device))
            entry[3].add(stream.cuda_stream)
        at = entry[1]
        entry[1] = (at + nbytes + self.ALIGN - 1) // self.ALIGN * self.ALIGN
        typed = entry[2].get(dtype)
        if typed is None:
            typed = entry[2][dtype] = entry[0].view(dtype)
        first = at // size  # `at` is a multiple of ALIGN, which every element size divides
        return typed[first:first + count]

    def fresh(self, device):
        """Forget the current stream's block: the next piece comes from a new one.  Call this at the start of
        every HIP graph capture: the block made inside the capture, fill included, then belongs to that graph
        alone (its replays put its own status words and counts back to zero and nobody else's)."""
        blocks = self._blocks()
        key = (device_index(device), stream_handle(device))
        for k in [k for k in blocks if k[:2] == key]:
            del blocks[k]
        self.native().fresh(*key)


zeros = ZeroPool()


def status_word(device):
    return zeros.word(device, torch.int32)


class _HostWords:
    """Pinned host words of one host thread (zen_read_back stores into them); they go when the thread does."""

    def __init__(self, words):
        self.words = words
        pinned = ctypes.c_void_p()
        check(lib().zen_host_words_alloc(words, ctypes.byref(pinned)), "host_words")
        self.ptr = pinned.value
        self.view = (ctypes.c_int64 * words).from_address(self.ptr)

    def __del__(self):
        if not sys.is_finalizing() and getattr(self, "ptr", None):
            _lib.zen_host_words_free(self.ptr)


_host = threading.local()
_NO_SEGMENT = [(None, 0, 0) * (3 - n) for n in range(4)]
# Longer lists (split sizes of very many partitions) come as plain copies: one workgroup stores the words, and a
# thread's pinned memory stays below a megabyte.
_READ_BACK_MOST = 1 << 16


def host_words(n):
    """This host thread's pinned words, with room for `n` (at most _READ_BACK_MOST) of an answer."""
    try:
        words = _host.words
    except AttributeError:
        words = None
    if words is None or words.words <= n:
        words = _host.words = _HostWords(max(1024, min(2 * n, _READ_BACK_MOST + 1)))
    return words


def read_back(*tensors):
    """The values of up to three small contiguous int32 / int64 device tensors (split sizes, counts, status
    words), one list after the other, once the current stream has got there.  The way a call on this path
    waits for the device: one kernel instead of a conversion, a concatenation and a copy."""
    args = []
    n = 0
    for t in tensors:
        count = t.numel()
        n += count
        args += (t.data_ptr(), count, 1 if t.dtype is torch.int64 else 0)
    if n > _READ_BACK_MOST:
        return [word for t in tensors for word in t.tolist()]
    args += _NO_SEGMENT[len(tensors)]
    words = host_words(n)
    rc = _lib.zen_read_back(*args, words.ptr, words.words, stream_handle(tensors[0].device))
    if rc:
        check(rc, "read_back")
    return words.view[1:n + 1]


def describe_status(bits):
    names = []
    if bits & STAT_SERIAL_OVERFLOW:
        names.append("serial region overflow")
    if bits & STAT_CAPACITY:
        names.append("output capacity exceeded")
    if bits & STAT_INTERNAL:
        names.append("internal wait expired")
    if bits & STAT_BAD_INDEX:
        names.append("index out of range")
    if bits & STAT_RETRY:
        names.append("fast path declined the input (retry in general mode)")
    return ", ".join(names) or "ok"


def profile_enable(on=True, only=None, every=1):
    """Start (or stop) timing the tagged launches; `only` names the one kernel
    tag to time, `every` = n times every n-th launch of a tag."""
    L = lib()
    tag = -1
    if only is not None:
        names = [L.zen_profile_name(t).decode() for t in range(L.zen_profile_tags())]
        tag = names.index(only)
    check(L.zen_profile_only(tag), "profile_only")
    check(L.zen_profile_every(int(every)), "profile_every")
    check(L.zen_profile_enable(1 if on else 0), "profile_enable")


def profile_read():
    """{kernel name: (total ms, launches)} for every tag that recorded a launch."""
    L = lib()
    out = {}
    for tag in range(L.zen_profile_tags()):
        ms, cnt = ctypes.c_double(0), ctypes.c_int64(0)
        check(L.zen_profile_read(tag, ctypes.byref(ms), ctypes.byref(cnt)), "profile_read")
        if cnt.value:
            out[L.zen_profile_name(tag).decode()] = (ms.value, cnt.value)
    return out


# ---------------------------------------------------------------- ranges
# Named ranges around the steps of the path, under the names the reference gives its nvtx ranges (comm.py:66-144,
# tensor_load_balance.py:25-44, train.py:65-69, 176), so that a rocprofv3 --marker-trace run of a training step
# reads like an Nsight trace of the reference.  Off unless ZEN_ROCTX=1 is set or ranges_enable(True) is called:
# the hot calls then pay nothing for them.
import contextlib

_ranges_on = os.environ.get("ZEN_ROCTX", "") not in ("", "0")
_no_range = contextlib.nullcontext()


def ranges_enable(on=True):
    global _ranges_on
    _ranges_on = bool(on)


def annotate(name):
    """Context manager: a roctx range called `name` (torch.cuda.nvtx is roctx on ROCm), or nothing when ranges are off."""
    if not _ranges_on:
        return _no_range
    return torch.cuda.nvtx.range(name)
