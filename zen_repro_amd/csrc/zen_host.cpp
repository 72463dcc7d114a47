// What the Python calls do around the library's functions, one crossing from the interpreter to a call: outputs and
// zeroed words are made, addresses taken, the function called, results cut.  A call of a small bucket is bound by the
// host, and each of these steps costs a microsecond or two in the interpreter (an all-reduce of a 9 k-element bucket had
// some 65 us of it).
//
// A library function arrives as the ctypes object that stands for it, so that whoever replaces the library replaces it
// here too; ctypes lets other threads run while the function does.
#include <torch/extension.h>

#include <algorithm>
#include <map>
#include <optional>
#include <tuple>
#include <utility>
#include <vector>

#include "zen_hip.h"

namespace py = pybind11;
using at::Tensor;

namespace {

int64_t address(const Tensor &t) { return reinterpret_cast<int64_t>(t.data_ptr()); }

Tensor room(const Tensor &like, int64_t count, at::ScalarType type) {
  return at::empty({count}, like.options().dtype(type).requires_grad(false));
}

// What `make` returns, a call's new tensors, while other threads may hold the interpreter: an allocator that has to go to
// the device, or free memory first, takes its time (torch's own bindings let go of it too).
template <typename Make>
auto made(Make make) {
  py::gil_scoped_release others;
  return make();
}
using Two = std::tuple<Tensor, Tensor>;  // (in braces: made in this order)
using Three = std::tuple<Tensor, Tensor, Tensor>;
using Four = std::tuple<Tensor, Tensor, Tensor, Tensor>;
using Five = std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor>;

// Zeroed words for status words, counters and split sizes, cut from blocks that one fill zeroed.  Every piece is handed
// out once, in the order of the stream its block was made on.  One object to a host thread.
class Zeros {
 public:
  static constexpr int64_t kWords = 8192;
  static constexpr int64_t kSplit = 2;  // pieces begin at multiples of so many words: of 16 bytes, status words of 8

  Tensor words(const Tensor &like, int64_t stream, int64_t count) { return take(blocks_, like, stream, count, at::kLong, 0, nullptr); }
  Tensor status(const Tensor &like, int64_t stream) { return take(narrow_, like, stream, 1, at::kInt, 0, nullptr); }
  // `other`: a stream beside that uses the words too; *wait: it has to wait for the block's fill.
  Tensor words_for(const Tensor &like, int64_t stream, int64_t count, int64_t other, bool *wait) {
    return take(blocks_, like, stream, count, at::kLong, other, wait);
  }
  void fresh(int64_t device, int64_t stream) {
    blocks_.erase({device, stream});
    narrow_.erase({device, stream});
  }

 private:
  struct Block {
    Tensor all;
    int64_t used = 0;
    std::vector<int64_t> seen;
  };
  using Blocks = std::map<std::pair<int64_t, int64_t>, Block>;
  Blocks blocks_, narrow_;

  static Tensor take(Blocks &blocks, const Tensor &like, int64_t stream, int64_t count, at::ScalarType type, int64_t other,
                     bool *wait) {
    const auto options = like.options().dtype(type).requires_grad(false);
    if (count > kWords / 4) {
      if (wait) *wait = true;
      return at::zeros({count}, options);
    }
    Block &b = blocks[{like.device().index(), stream}];
    const int64_t step = (count + kSplit - 1) / kSplit * kSplit;
    if (!b.all.defined() || b.used + step > kWords) b = Block{at::zeros({kWords}, options), 0, {stream}};
    if (wait) {
      *wait = std::find(b.seen.begin(), b.seen.end(), other) == b.seen.end();
      if (*wait) b.seen.push_back(other);
    }
    const Tensor piece = b.all.narrow(0, b.used, count);
    b.used += step;
    return piece;
  }
};

// The covering view of one-dimensional tensors that sit back to back in one storage; none if they do not.
py::object one_buffer(const std::vector<Tensor> &tensors) {
  if (tensors.empty()) return py::none();
  const Tensor &first = tensors[0];
  if (first.dim() != 1 || !first.is_contiguous()) return py::none();
  const char *at = static_cast<const char *>(first.data_ptr());
  const void *storage = first.storage().data();
  const int64_t size = first.element_size();
  int64_t total = 0;
  for (const Tensor &t : tensors) {
    if (t.scalar_type() != first.scalar_type() || t.dim() != 1 || t.data_ptr() != at || !t.is_contiguous() ||
        t.storage().data() != storage)
      return py::none();
    total += t.numel();
    at += t.numel() * size;
  }
  return py::cast(first.as_strided({total}, {1}));
}

// Contiguous, of one type and on one device: what a kernel takes by their addresses.
bool plain_runs(const std::vector<Tensor> &tensors) {
  for (const Tensor &t : tensors)
    if (t.scalar_type() != tensors[0].scalar_type() || t.device() != tensors[0].device() || !t.is_contiguous()) return false;
  return true;
}

struct Lists {
  std::vector<int64_t> at, count;
  explicit Lists(const std::vector<Tensor> &tensors) {
    for (const Tensor &t : tensors) {
      at.push_back(address(t));
      count.push_back(t.numel());
    }
  }
  int64_t addresses() const { return reinterpret_cast<int64_t>(at.data()); }
  int64_t counts() const { return reinterpret_cast<int64_t>(count.data()); }
};

// Indices and values to their partitions.
py::tuple cut(const Tensor &indices, const Tensor &values, const std::vector<int64_t> &sizes) {
  int64_t total = 0;
  for (int64_t s : sizes) total += s;
  return py::make_tuple(at::split_with_sizes(indices.narrow(0, 0, total), sizes),
                        at::split_with_sizes(values.narrow(0, 0, total), sizes));
}

py::tuple load_balance(const py::object &fn, Zeros &zeros, const Tensor &flat, int code, int64_t m, int64_t partitions,
                       int rehash, const py::object &thr, int64_t k, const py::object &thr_out, int64_t capacity,
                       int64_t table, int64_t mode, const Tensor &ws, int64_t stream, int64_t host, int64_t words) {
  const auto [idx, val, splits, status] = made([&] {
    return Four{room(flat, capacity, at::kInt), room(flat, capacity, flat.scalar_type()), zeros.words(flat, stream, partitions),
                zeros.status(flat, stream)};
  });
  const py::object rc =
      host ? fn(address(flat), code, flat.numel(), m, partitions, rehash, thr, k, thr_out, address(idx), address(val),
                capacity, address(splits), table, mode, address(ws), ws.numel(), address(status), host, words, stream)
           : fn(address(flat), code, flat.numel(), m, partitions, rehash, thr, k, thr_out, address(idx), address(val),
                capacity, address(splits), table, mode, address(ws), ws.numel(), address(status), stream);
  return py::make_tuple(rc, idx, val, splits, status);
}

py::tuple merge(const py::object &fn, Zeros &zeros, const Tensor &indices, const Tensor &values, int code, int64_t dense_size,
                int64_t capacity, bool idx64, bool rounded, int64_t mode, const Tensor &ws, int64_t stream, int64_t host,
                int64_t words) {
  const auto [idx, val, count, status] = made([&] {
    return Four{room(values, capacity, idx64 ? at::kLong : at::kInt), room(values, capacity, rounded ? values.scalar_type() : at::kFloat),
                zeros.words(values, stream, 1), zeros.status(values, stream)};
  });
  const int from64 = indices.scalar_type() == at::kLong;
  const py::object rc =
      host ? fn(address(indices), from64, address(values), code, indices.numel(), dense_size, address(idx), idx64 ? 1 : 0,
                address(val), capacity, address(count), mode, address(ws), ws.numel(), address(status), host, words, stream)
           : fn(address(indices), from64, address(values), code, indices.numel(), dense_size, address(idx), idx64 ? 1 : 0,
                address(val), capacity, address(count), mode, address(ws), ws.numel(), address(status), stream);
  return py::make_tuple(rc, idx, val, count, status);
}

py::tuple select_count(const py::object &fn, Zeros &zeros, const Tensor &flat, int code, const py::object &thr, bool idx64,
                 int64_t capacity, const Tensor &ws, int64_t stream, int64_t host, int64_t words) {
  const auto [idx, val, count, status] = made([&] {
    return Four{room(flat, capacity, idx64 ? at::kLong : at::kInt), room(flat, capacity, flat.scalar_type()),
                zeros.words(flat, stream, 1), zeros.status(flat, stream)};
  });
  const py::object rc = fn(address(flat), code, flat.numel(), thr, address(idx), idx64 ? 1 : 0, address(val), capacity,
                           address(count), address(ws), ws.numel(), address(status), host, words, stream);
  return py::make_tuple(rc, idx, val);
}

py::tuple sample_threshold(const py::object &fn, Zeros &zeros, const Tensor &flat, int code, const Tensor &index, int64_t k,
                           const Tensor &ws, int64_t stream) {
  const auto [thr, status] = made([&] { return Two{room(flat, 2, at::kInt), zeros.status(flat, stream)}; });
  const py::object rc = fn(address(flat), code, flat.numel(), address(index), index.numel(), k, address(thr), address(ws),
                           ws.numel(), address(status), stream);
  return py::make_tuple(rc, thr, status);
}

py::tuple decode(const py::object &fn, Zeros &zeros, const Tensor &indices, const Tensor &values, int code, const Tensor &dense,
                 int64_t mode, const Tensor &ws, int64_t stream, int64_t host, int64_t words) {
  const Tensor status = made([&] { return zeros.status(values, stream); });
  const py::object rc = fn(address(indices), indices.scalar_type() == at::kLong ? 1 : 0, address(values), code,
                           indices.numel(), address(dense), dense.numel(), mode, address(ws), ws.numel(), address(status),
                           host, words, stream);
  return py::make_tuple(rc, status);
}

// Whether the lists are plain runs of one type on one device, with a value list to each index list.
bool matching_runs(const std::vector<Tensor> &indices, const std::vector<Tensor> &values) {
  if (indices.size() != values.size() || !plain_runs(indices) || !plain_runs(values)) return false;
  for (size_t i = 0; i < indices.size(); ++i)
    if (indices[i].numel() != values[i].numel() || indices[i].device() != values[i].device()) return false;
  return true;
}

py::tuple decode_lists(const py::object &fn, Zeros &zeros, const std::vector<Tensor> &indices,
                       const std::vector<Tensor> &values, int code, int64_t dense_size, const Tensor &ws, int64_t stream,
                       int64_t host, int64_t words) {
  const auto [dense, status] =
      made([&] { return Two{room(values[0], dense_size, values[0].scalar_type()), zeros.status(values[0], stream)}; });
  const Lists i(indices), v(values);
  const py::object rc = fn(i.addresses(), indices[0].scalar_type() == at::kLong ? 1 : 0, v.addresses(), code, i.counts(),
                           indices.size(), address(dense), dense_size, address(ws), ws.numel(), address(status), host, words,
                           stream);
  return py::make_tuple(rc, dense);
}

// `told`: a status word that is answered for with this call's own, of work in front of it on the stream.
py::tuple bitmaps_dense(const py::object &fn, Zeros &zeros, const std::vector<Tensor> &bitmaps,
                        const std::vector<Tensor> &values, int code, const Tensor &dict, int64_t numel, const Tensor &ws,
                        int64_t stream, int64_t host, int64_t words, const std::optional<Tensor> &told) {
  const auto [dense, status] = made([&] {
    return Two{room(values[0], numel, values[0].scalar_type()), told ? *told : zeros.status(values[0], stream)};
  });
  const Lists b(bitmaps), v(values);
  const py::object rc = fn(address(dict), numel, bitmaps.size(), b.addresses(), b.counts(), v.addresses(), code, v.counts(),
                           address(dense), address(ws), ws.numel(), address(status), host, words, stream);
  return py::make_tuple(rc, dense);
}

py::tuple bitmap_encode(const py::object &fn, Zeros &zeros, const Tensor &mapping, const Tensor &indices, const Tensor &ranks,
                        int64_t numel, int64_t count, int64_t stream, int64_t host, int64_t words) {
  const auto [bitmap, status] =
      made([&] { return Two{room(indices, std::max<int64_t>(count, 1) * 4, at::kByte), zeros.status(indices, stream)}; });
  const int idx64 = indices.scalar_type() == at::kLong ? 1 : 0;
  const py::object rc =
      host ? fn(address(mapping), mapping.numel(), address(indices), idx64, indices.numel(), py::none(), address(ranks), numel,
                address(bitmap), address(status), host, words, stream)
           : fn(address(mapping), mapping.numel(), address(indices), idx64, indices.numel(), py::none(), address(ranks), numel,
                address(bitmap), address(status), stream);
  return py::make_tuple(rc, bitmap.narrow(0, 0, (mapping.numel() + 7) / 8), status);
}

py::tuple tables(const py::object &fn, Zeros &zeros, const Tensor &input, int code, int64_t m, int64_t serial_n,
                 int64_t partitions, int rehash, int64_t stream, int64_t host, int64_t words) {
  const auto [memory, serial, offsets, status] = made([&] {
    return Four{room(input, m, at::kInt), room(input, serial_n, at::kInt), room(input, partitions, at::kInt), zeros.status(input, stream)};
  });
  const py::object rc = fn(address(input), code, input.numel(), address(memory), m, address(serial), serial_n,
                           address(offsets), partitions, rehash, address(status), host, words, stream);
  return py::make_tuple(rc, memory, serial, offsets, status);
}

py::tuple table_find(const py::object &fn, Zeros &zeros, const Tensor &memory, int64_t partitions, int64_t n, int64_t ws_bytes,
                     int64_t stream, int64_t host, int64_t words) {
  // beside the split sizes, the words in which the walk adds them up; no workspace that is kept from call to call: the
  // thread may walk another table before these lists are used up
  const auto [all, status, ws] = made([&] {
    return Three{zeros.words(memory, stream, 3 * partitions + 66), zeros.status(memory, stream), room(memory, ws_bytes, at::kByte)};
  });
  const Tensor splits = all.narrow(0, 0, partitions);
  const py::object rc =
      host ? fn(address(memory), memory.numel(), partitions, n, address(splits), address(all) + 8 * partitions, address(ws),
                ws_bytes, address(status), host, words, stream)
           : fn(address(memory), memory.numel(), partitions, n, address(splits), address(ws), ws_bytes, address(status), stream);
  return py::make_tuple(rc, splits, status, ws);
}

py::tuple table_gather(const py::object &fn, const Tensor &memory, const Tensor &flat, int code,
                       const std::vector<int64_t> &sizes, const Tensor &ws, int64_t stream) {
  int64_t total = 0;
  for (int64_t s : sizes) total += s;
  const auto [idx, val] = made([&] { return Two{room(flat, total, at::kInt), room(flat, total, flat.scalar_type())}; });
  const py::object rc = fn(address(memory), memory.numel(), sizes.size(), address(flat), code, flat.numel(), address(idx),
                           address(val), total, address(ws), ws.numel(), stream);
  return py::make_tuple(rc, at::split_with_sizes(idx, sizes), at::split_with_sizes(val, sizes));
}

// The buffers of a step (zen_encode_merge) and everything in its arguments that follows from them; `wait`: the merge's
// stream has to wait for the zeroed words.
py::tuple step_buffers(int64_t args, Zeros &zeros, const Tensor &flat, const Tensor &indices, const Tensor &values,
                       int64_t capacity, int64_t partitions, int64_t stream, int64_t merge_stream, const Tensor &ws,
                       const Tensor &merge_ws) {
  zen_encode_merge_args *a = reinterpret_cast<zen_encode_merge_args *>(args);
  const int64_t r = indices.numel();
  bool wait = false;
  // small: split sizes, merged count, the two status words
  const auto [idx, val, m_idx, m_val, small] = made([&] {
    return Five{room(flat, capacity, at::kInt), room(flat, capacity, flat.scalar_type()), room(flat, r, at::kInt),
                room(flat, r, at::kFloat),
                merge_stream ? zeros.words_for(flat, stream, partitions + 2, merge_stream, &wait)
                             : zeros.words(flat, stream, partitions + 2)};
  });
  const Tensor splits = small.narrow(0, 0, partitions), count = small.narrow(0, partitions, 1);
  const Tensor both = small.narrow(0, partitions + 1, 1).view(at::kInt);
  const Tensor status = both.narrow(0, 0, 1), m_status = both.narrow(0, 1, 1);
  a->input = flat.data_ptr();
  a->out_idx = static_cast<int32_t *>(idx.data_ptr());
  a->out_val = val.data_ptr();
  a->splits = static_cast<int64_t *>(splits.data_ptr());
  a->workspace = ws.data_ptr();
  a->workspace_bytes = (size_t)ws.numel();
  a->status = static_cast<int32_t *>(status.data_ptr());
  a->recv_idx = indices.data_ptr();
  a->recv_idx64 = indices.scalar_type() == at::kLong;
  a->recv_val = values.data_ptr();
  a->merged_idx = m_idx.data_ptr();
  a->merged_val = static_cast<float *>(m_val.data_ptr());
  a->merged_count = static_cast<int64_t *>(count.data_ptr());
  a->merge_workspace = merge_ws.data_ptr();
  a->merge_workspace_bytes = (size_t)merge_ws.numel();
  a->merge_status = static_cast<int32_t *>(m_status.data_ptr());
  a->stream = reinterpret_cast<void *>(stream);
  a->merge_stream = reinterpret_cast<void *>(merge_stream);
  return py::make_tuple(py::make_tuple(idx, val, splits, status), py::make_tuple(m_idx, m_val, count, m_status), wait);
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  py::class_<Zeros>(m, "Zeros").def(py::init<>()).def("fresh", &Zeros::fresh);
  m.attr("ABI_VERSION") = ZEN_ABI_VERSION;
  m.def("one_buffer", &one_buffer);
  m.def("plain_runs", &plain_runs);
  m.def("cut", &cut);
  m.def("load_balance", &load_balance);
  m.def("merge", &merge);
  m.def("select_count", &select_count);
  m.def("sample_threshold", &sample_threshold);
  m.def("decode", &decode);
  m.def("matching_runs", &matching_runs);
  m.def("decode_lists", &decode_lists);
  m.def("bitmaps_dense", &bitmaps_dense);
  m.def("bitmap_encode", &bitmap_encode);
  m.def("tables", &tables);
  m.def("table_find", &table_find);
  m.def("table_gather", &table_gather);
  m.def("step_buffers", &step_buffers);
}
