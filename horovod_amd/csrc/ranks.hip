// ranks.hip -- the sum over ranks of a fused response whose tensors all sit in this device's
// memory: every rank's tensors are read where they are, scaled (and narrowed), summed in rank
// order, scaled back (and widened) and stored into the outputs in one pass.  gfx950 only.
//
// The sequence it replaces -- each rank packs into a fusion buffer of its own, the buffers are
// summed into the first, which is unpacked -- moves every byte three times (2 per packing rank,
// world + 1 for the sum, 2 for the unpack: 27 passes over the tensors for 8 ranks where 9 do).
// It is bound by memory in both forms: ResNet-50's gradients (102 MB) of 8 ranks took 222 us of
// kernels and take 160 us in this one, BERT-large's with fp16 on the wire 4.2 ms and 2.4 ms (8 read
// streams from HBM: 5.8-6.1 TB/s).  Results are the same to the bit: the same roundings in the
// same order (to the wire type after the prescale and after every rank).
//
// There is no table in device memory.  A launch carries the addresses of up to kMaxRows tensors
// (what fits in 4 KiB of kernel arguments: 44 tensors of 8 ranks), a response of more is several
// launches.  A table would have to be built and copied for every new set of addresses, and new
// outputs are what an out-of-place call brings each time: with a cache of tables, BERT-large's
// step spent 16 ms on rebuilding them whenever more sets rotated than it held.
#include <algorithm>
#include <cstring>
#include <vector>

#include "ranks.h"

namespace hvdhip {
namespace {

constexpr int kTogether = 8;        // ranks whose loads are in flight at once

template <typename T, int VEC>
__device__ __forceinline__ void add_to(Arr<T, VEC>& acc, const Arr<T, VEC>& x) {
#pragma unroll
  for (int j = 0; j < VEC; ++j) acc.v[j] = (T)(acc.v[j] + x.v[j]);
}
// Halves as packed adds (one rounding, which equals fp32 add and narrowing: see reduce.hip).
template <>
__device__ __forceinline__ void add_to<half_t, 8>(Arr<half_t, 8>& acc, const Arr<half_t, 8>& x) {
  typedef half_t h2 __attribute__((ext_vector_type(2)));
  h2 a[4], b[4];
  __builtin_memcpy(a, acc.v, 16);
  __builtin_memcpy(b, x.v, 16);
#pragma unroll
  for (int w = 0; w < 4; ++w) a[w] = a[w] + b[w];
  __builtin_memcpy(acc.v, a, 16);
}
// Bytes four to a word, without a carry into the neighbour (see reduce.hip).
__device__ __forceinline__ void add_bytes(uint8_t* acc, const uint8_t* x) {
  uint32_t a[4], b[4];
  __builtin_memcpy(a, acc, 16);
  __builtin_memcpy(b, x, 16);
#pragma unroll
  for (int w = 0; w < 4; ++w)
    a[w] = ((a[w] & 0x7f7f7f7fu) + (b[w] & 0x7f7f7f7fu)) ^ ((a[w] ^ b[w]) & 0x80808080u);
  __builtin_memcpy(acc, a, 16);
}
template <>
__device__ __forceinline__ void add_to<uint8_t, 16>(Arr<uint8_t, 16>& acc, const Arr<uint8_t, 16>& x) {
  add_bytes(acc.v, x.v);
}
template <>
__device__ __forceinline__ void add_to<int8_t, 16>(Arr<int8_t, 16>& acc, const Arr<int8_t, 16>& x) {
  add_bytes(reinterpret_cast<uint8_t*>(acc.v), reinterpret_cast<const uint8_t*>(x.v));
}

// One workgroup per chunk of kWG * kVec elements: 4 KiB of the wider side, one 16-byte access per lane
// and rank, the loads of the first K ranks (K = min(world, 8)) all in flight before the first add.  The arguments stay in the scalar cache, so a
// workgroup waits for one vector load (the search) and one batch of scalar loads (its row) before its
// data loads go out.  Two or four accesses per lane in a loop (8 and 16 KiB) are 3-10 % slower at 8 ranks
// (BERT-large 446 -> 489 us), loads without the non-temporal hint 8 %; runs of 64 KiB to 1 MiB per XCD
// measure within 2 % of each other.
template <typename S, typename W, typename D, int K, int ST>
__global__ __launch_bounds__(kWG) void ranks_sum_k(uint32_t shift, uint32_t ordered, uint32_t nrows, uint32_t world,
                                                   double pre, double post, uint32_t flags, Rows rows) {
  constexpr int VEC = kVec<S, D>;
  constexpr uint32_t kTile = kWG * VEC;
  constexpr bool kBytes = sizeof(S) == 1;  // byte elements are read through windows (vecmem.h)
  const uint32_t chunk = xcd_tile(blockIdx.x, XcdOrder{shift, ordered});
  const uint32_t row = row_of(rows, nrows, chunk);
  const uint64_t* q = rows.q + row * (world + 2);  // {output, elements, input of rank 0, 1 ...}
  const uint64_t start = (uint64_t)(chunk - rows.first[row]) * kTile;
  const uint64_t left = q[1] - start;
  const uint32_t m = left < kTile ? (uint32_t)left : kTile;
  gptr<D> out = as_global<D>(q[0]) + start;
  const Window win = store_window<ST>(out, m * (uint32_t)sizeof(D));
  const typename Factor<W>::type fin = (typename Factor<W>::type)pre, fout = (typename Factor<W>::type)post;
  const bool scale_in = flags & kScaleIn, scale_out = flags & kScaleOut;
  auto source = [&](uint32_t rank) { return as_global<const S>(q[2 + rank]) + start; };
  gptr<const S> src[K];  // all at once, ahead of the branch
#pragma unroll
  for (int k = 0; k < K; ++k) src[k] = source(k);
  const uint32_t v = threadIdx.x, nv = m / VEC;
  if (v < nv) {
    auto load = [&](gptr<const S> p) {
      if constexpr (kBytes) {
        return ldw<S, VEC>(load_window(p, m), v * 16u);
      } else {
        return ldv<S, VEC>(p + (size_t)v * VEC);
      }
    };
    auto wire = [&](const Arr<S, VEC>& x) { return to_wire<S, W, VEC>(x, fin, scale_in); };
    Arr<S, VEC> x[K];
#pragma unroll
    for (int k = 0; k < K; ++k) x[k] = load(src[k]);
    Arr<W, VEC> acc = wire(x[0]);
#pragma unroll
    for (int k = 1; k < K; ++k) add_to<W, VEC>(acc, wire(x[k]));
    if constexpr (K == kTogether) {
      for (uint32_t r = K; r < world; ++r) add_to<W, VEC>(acc, wire(load(source(r))));
    }
    stw<ST, D, VEC>(win, v * (uint32_t)(VEC * sizeof(D)), from_wire<W, D, VEC>(acc, fout, scale_out));
  }
  const uint32_t t = nv * VEC + threadIdx.x;  // fewer than VEC elements remain
  if (t < m) {
    auto wire = [&](uint32_t r) { return to_wire<S, W, 1>(Arr<S, 1>{source(r)[t]}, fin, scale_in); };
    Arr<W, 1> acc = wire(0);
    for (uint32_t r = 1; r < world; ++r) add_to<W, 1>(acc, wire(r));
    out[t] = from_wire<W, D, 1>(acc, fout, scale_out).v[0];
  }
  if constexpr (ST == kStoreWT) {  // into a fusion buffer: zeros up to the next 16-byte boundary
    const uint32_t pad = (uint32_t)(0u - (uint32_t)q[1] * (uint32_t)sizeof(D)) & 15u;
    if (left <= kTile && threadIdx.x < pad) as_global<uint8_t>(q[0])[q[1] * sizeof(D) + threadIdx.x] = 0;
  }
}

// ---- host side ---------------------------------------------------------------------------------

template <typename S, typename W, typename D, int K, int ST>
hipError_t launch_rows(const RanksCall& c, const Rows& rows, uint32_t nrows, uint32_t chunks, bool last) {
  constexpr uint32_t kTileBytes = kWG * kVec<S, D> * (uint32_t)(sizeof(S) > sizeof(D) ? sizeof(S) : sizeof(D));
  const XcdOrder order = xcd_order(chunks, kTileBytes);
  return launch_with(last ? c.completion : nullptr, ranks_sum_k<S, W, D, K, ST>, chunks, c.stream, order.shift,
                     order.ordered, nrows, c.world, c.pre, c.post, c.flags, rows);
}

template <typename S, typename W, typename D, int ST>
hipError_t launch_by_world(const RanksCall& c, const Rows& rows, uint32_t nrows, uint32_t chunks, bool last) {
  switch (c.world) {
  case 1: return launch_rows<S, W, D, 1, ST>(c, rows, nrows, chunks, last);
  case 2: return launch_rows<S, W, D, 2, ST>(c, rows, nrows, chunks, last);
  case 3: return launch_rows<S, W, D, 3, ST>(c, rows, nrows, chunks, last);
  case 4: return launch_rows<S, W, D, 4, ST>(c, rows, nrows, chunks, last);
  case 5: return launch_rows<S, W, D, 5, ST>(c, rows, nrows, chunks, last);
  case 6: return launch_rows<S, W, D, 6, ST>(c, rows, nrows, chunks, last);
  case 7: return launch_rows<S, W, D, 7, ST>(c, rows, nrows, chunks, last);
  default: return launch_rows<S, W, D, kTogether, ST>(c, rows, nrows, chunks, last);
  }
}

// Fills launches with as many rows as their arguments hold.  A tensor that would take a launch beyond
// kMaxWorkgroups chunks is cut there and goes on in the next one.
template <typename S, typename W, typename D>
int run(const RanksCall& c) {
  constexpr uint64_t kTile = (uint64_t)kWG * kVec<S, D>;
  const uint32_t max_rows = std::min(kMaxRows, kQwords / (c.world + 2));
  int entry = 0;
  uint64_t done = 0;  // elements of the current entry that earlier launches took
  auto skip_empty = [&] { while (entry < c.n && c.counts[entry] == 0) ++entry; };
  skip_empty();
  if (entry == c.n) {
    if (c.completion) HVDHIP_CHECK(hipEventRecord(c.completion, c.stream));
    return 0;
  }
  Rows rows;
  while (entry < c.n) {
    uint32_t nrows = 0;
    uint64_t chunks = 0;
    uint64_t* q = rows.q;
    while (entry < c.n && nrows < max_rows && chunks < kMaxWorkgroups) {
      const uint64_t left = (uint64_t)c.counts[entry] - done;
      const uint64_t take = std::min(left, (kMaxWorkgroups - chunks) * kTile);
      rows.first[nrows++] = (uint32_t)chunks;
      *q++ = (uint64_t)(uintptr_t)c.outputs[entry] + done * sizeof(D);
      *q++ = take;
      for (uint32_t r = 0; r < c.world; ++r)
        *q++ = (uint64_t)(uintptr_t)c.inputs[(size_t)r * (size_t)c.n + (size_t)entry] + done * sizeof(S);
      chunks += (take + kTile - 1) / kTile;
      done += take;
      if (take == left) {
        done = 0;
        ++entry;
        skip_empty();
      }
    }
    for (uint32_t i = nrows; i < kMaxRows; ++i) rows.first[i] = ~0u;
    const bool last = entry == c.n;
    const hipError_t status = c.flags & kPadOut
                                  ? launch_by_world<S, W, D, kStoreWT>(c, rows, nrows, (uint32_t)chunks, last)
                                  : launch_by_world<S, W, D, kStoreNT>(c, rows, nrows, (uint32_t)chunks, last);
    HVDHIP_CHECK_LAUNCH("ranks_sum_k", status);
  }
  return 0;
}

// Whether an input overlaps an output anywhere but exactly at its own entry's.  Within an entry every lane
// reads all its inputs before it stores, and no other lane touches those addresses.
bool overlaps(const RanksCall& c, uint64_t in_size, uint64_t out_size) {
  struct Range {
    uint64_t lo, hi;
    int entry;
  };
  std::vector<Range> outs;
  outs.reserve((size_t)c.n);
  for (int i = 0; i < c.n; ++i)
    if (c.counts[i]) {
      const uint64_t lo = (uint64_t)(uintptr_t)c.outputs[i];
      outs.push_back(Range{lo, lo + (uint64_t)c.counts[i] * out_size, i});
    }
  if (outs.empty()) return false;
  auto before = [](const Range& a, const Range& b) { return a.lo < b.lo; };
  if (!std::is_sorted(outs.begin(), outs.end(), before)) std::sort(outs.begin(), outs.end(), before);
  for (size_t i = 0; i + 1 < outs.size(); ++i)
    if (outs[i].hi > outs[i + 1].lo) return true;
  const uint64_t lowest = outs.front().lo, highest = outs.back().hi;
  for (uint32_t r = 0; r < c.world; ++r) {
    const void* const* in = c.inputs + (size_t)r * (size_t)c.n;
    for (int i = 0; i < c.n; ++i) {
      const uint64_t lo = (uint64_t)(uintptr_t)in[i], hi = lo + (uint64_t)c.counts[i] * in_size;
      if (c.counts[i] == 0 || hi <= lowest || lo >= highest) continue;
      if (lo == (uint64_t)(uintptr_t)c.outputs[i] && in_size == out_size) continue;
      auto it = std::upper_bound(outs.begin(), outs.end(), Range{lo, 0, 0}, before);
      if (it != outs.begin() && std::prev(it)->hi > lo) return true;
      if (it != outs.end() && it->lo < hi) return true;
    }
  }
  return false;
}

bool scalable_dtype(int dtype) {
  switch (dtype) {
  case HVDHIP_UINT8: case HVDHIP_INT8: case HVDHIP_INT32: case HVDHIP_INT64:
  case HVDHIP_FLOAT16: case HVDHIP_FLOAT32: case HVDHIP_FLOAT64: return true;
  default: return false;
  }
}

}  // namespace
}  // namespace hvdhip

using namespace hvdhip;

int hvdhip::check_ranks_call(RanksCall* c, int in_dtype, int wire_dtype, int out_dtype) {
  if (c->n < 0 || (c->n > 0 && (!c->outputs || !c->inputs || !c->counts)))
    return fail(HVDHIP_ERR_INVALID_ARGUMENT, "bad entry arrays");
  const int64_t is = dtype_size(in_dtype), os = dtype_size(out_dtype);
  if (is < 0 || os < 0) return fail(HVDHIP_ERR_UNSUPPORTED_DTYPE, "unknown dtype");
  const bool same = in_dtype == wire_dtype && wire_dtype == out_dtype;
  const bool halves = wire_dtype == HVDHIP_FLOAT16 && (in_dtype == HVDHIP_FLOAT32 || in_dtype == HVDHIP_FLOAT16) &&
                      (out_dtype == HVDHIP_FLOAT32 || out_dtype == HVDHIP_FLOAT16);
  if (!same && !halves)
    return fail(HVDHIP_ERR_UNSUPPORTED_DTYPE, "dtypes %d, %d, %d: only FLOAT32 converts, to and from FLOAT16 on the wire",
                in_dtype, wire_dtype, out_dtype);
  if (c->world > 1 && wire_dtype == HVDHIP_BOOL)
    return fail(HVDHIP_ERR_UNSUPPORTED_DTYPE, "dtype %d cannot be summed", wire_dtype);
  if ((c->pre != 1.0 || c->post != 1.0) && !scalable_dtype(wire_dtype))
    return fail(HVDHIP_ERR_UNSUPPORTED_DTYPE, "dtype %d cannot be scaled by a factor other than 1", wire_dtype);
  for (int i = 0; i < c->n; ++i) {
    if (c->counts[i] < 0) return fail(HVDHIP_ERR_INVALID_ARGUMENT, "entry %d has a negative size", i);
    if (c->counts[i] == 0) continue;
    if (!c->outputs[i] || (uintptr_t)c->outputs[i] % (uintptr_t)os)
      return fail(HVDHIP_ERR_INVALID_ARGUMENT, "the output of entry %d is NULL or not aligned to its element size", i);
    for (int r = 0; r < (int)c->world; ++r) {
      const uintptr_t p = (uintptr_t)c->inputs[(size_t)r * (size_t)c->n + (size_t)i];
      if (!p || p % (uintptr_t)is)
        return fail(HVDHIP_ERR_INVALID_ARGUMENT, "rank %d of entry %d is NULL or not aligned to its element size", r, i);
    }
  }
  if (overlaps(*c, (uint64_t)is, (uint64_t)os))
    return fail(HVDHIP_ERR_OVERLAP, "an output overlaps another output or another entry's input");
  if (c->pre != 1.0) c->flags |= kScaleIn;
  if (c->post != 1.0) c->flags |= kScaleOut;
  if (wire_dtype == HVDHIP_FLOAT16) {
    c->pre = fp16_scale_factor(c->pre);
    c->post = fp16_scale_factor(c->post);
  }
  return 0;
}

extern "C" int hvdhip_ranks_sum(void* const* outputs, const void* const* inputs, const int64_t* num_elements, int n,
                                int world, int in_dtype, int wire_dtype, int out_dtype, double prescale,
                                double postscale, unsigned flags, void* stream, void* event) {
  if (world < 1 || world > HVDHIP_RANKS_SUM_MAX_WORLD)
    return fail(HVDHIP_ERR_INVALID_ARGUMENT, "world = %d is outside 1..%d", world, HVDHIP_RANKS_SUM_MAX_WORLD);
  if (flags & ~HVDHIP_RANKS_SUM_PAD_OUTPUTS) return fail(HVDHIP_ERR_INVALID_ARGUMENT, "unknown flags 0x%x", flags);
  RanksCall c = {outputs, inputs, num_elements, n, (uint32_t)world, prescale, postscale, 0,
                 static_cast<hipStream_t>(stream), static_cast<hipEvent_t>(event)};
  int rc = check_ranks_call(&c, in_dtype, wire_dtype, out_dtype);
  if (rc) return rc;
  if (flags & HVDHIP_RANKS_SUM_PAD_OUTPUTS) c.flags |= kPadOut;
  switch (wire_dtype) {
  case HVDHIP_UINT8: case HVDHIP_BOOL: rc = run<uint8_t, uint8_t, uint8_t>(c); break;
  case HVDHIP_INT8: rc = run<int8_t, int8_t, int8_t>(c); break;
  case HVDHIP_UINT16: case HVDHIP_INT16: rc = run<uint16_t, uint16_t, uint16_t>(c); break;
  case HVDHIP_INT32: rc = run<int32_t, int32_t, int32_t>(c); break;
  case HVDHIP_INT64: rc = run<int64_t, int64_t, int64_t>(c); break;
  case HVDHIP_FLOAT32: rc = run<float, float, float>(c); break;
  case HVDHIP_FLOAT64: rc = run<double, double, double>(c); break;
  default:
    rc = in_dtype == HVDHIP_FLOAT32 ? (out_dtype == HVDHIP_FLOAT32 ? run<float, half_t, float>(c) : run<float, half_t, half_t>(c))
                                    : (out_dtype == HVDHIP_FLOAT32 ? run<half_t, half_t, float>(c) : run<half_t, half_t, half_t>(c));
  }
  return rc ? rc : ok();
}
