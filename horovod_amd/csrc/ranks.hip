// ranks.hip -- the sum over ranks of a fused response whose tensors all sit in this device's
// memory: every rank's tensors are read where they are, scaled (and narrowed), summed in rank
// order, scaled back (and widened) and stored into the outputs in one pass.  gfx950 only.
//
// The sequence it replaces -- each rank packs into a fusion buffer of its own, the buffers are
// summed into the first, which is unpacked -- moves every byte three times (2 per packing rank,
// world + 1 for the sum, 2 for the unpack: 27 passes over the tensors for 8 ranks where 9 do).
// It is bound by memory in both forms: ResNet-50's gradients (102 MB) of 8 ranks took 222 us of
// kernels and take 146 us in this one, BERT-large's with fp16 on the wire 4.2 ms and 1.95 ms (8 read
// streams from HBM: 6.1-6.5 TB/s).  Results are the same to the bit: the same roundings in the
// same order (to the wire type after the prescale and after every rank).
//
// There is no table in device memory.  A launch carries the addresses of up to 128 tensors
// (what fits in 4 KiB of kernel arguments: 84 tensors of 8 ranks), a response of more is several
// launches.  A table would have to be built and copied for every new set of addresses, and new
// outputs are what an out-of-place call brings each time: with a cache of tables, BERT-large's
// step spent 16 ms on rebuilding them whenever more sets rotated than it held.
#include <algorithm>
#include <cstring>
#include <new>
#include <vector>

#include "ranks.h"

namespace hvdhip {
namespace {

constexpr int kTogether = 8;        // ranks whose loads are in flight at once

// ranks_split_k: K ranks over this many wavefronts, two ranks each (the last may have one), and vectors of a rank that a
// lane loads.
template <int K>
constexpr int kSplitWaves = K <= 4 ? 2 : 4;
template <int K>
constexpr int kSplitVecs = K == 2 * kSplitWaves<K> ? 1 : 2;

template <typename T, int VEC>
__device__ __forceinline__ void add_to(Arr<T, VEC>& acc, const Arr<T, VEC>& x) {
#pragma unroll
  for (int j = 0; j < VEC; ++j) {
    if constexpr (std::is_integral<T>::value) {  // wraps, which signed addition is not defined to do
      typedef typename std::make_unsigned<T>::type U;
      acc.v[j] = (T)((U)acc.v[j] + (U)x.v[j]);
    } else {
      acc.v[j] = (T)(acc.v[j] + x.v[j]);
    }
  }
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

// acc plus what load() gives for the ranks from `rank` to `world`, in rank order, with the loads of eight ranks in flight
// at a time and of four, two and one at the end.  One at a time, each waiting for the sum before it, bounds small
// tensors by latency: 1 KiB of fp32 and 16 ranks 6.3 us and 5.7 in batches, 64 ranks 32 and 9.4, 256 ranks 146 and 35;
// 32 MiB of uint8 and 32 ranks 244 and 178.  32 MiB of fp32 are bound by memory either way (16 ranks 92 and 92.5, 64
// ranks 331 and 344; batches of four or two the same).
template <int B, typename W, int N, typename Load, typename Wire>
__device__ __forceinline__ void add_ranks(Arr<W, N>& acc, uint32_t rank, uint32_t world, Load&& load, Wire&& wire) {
  for (; rank + B <= world; rank += B) {
    decltype(load(rank)) x[B];
#pragma unroll
    for (uint32_t k = 0; k < B; ++k) x[k] = load(rank + k);
#pragma unroll
    for (uint32_t k = 0; k < B; ++k) add_to<W, N>(acc, wire(x[k]));
  }
  if constexpr (B > 1) add_ranks<B / 2, W, N>(acc, rank, world, load, wire);
}

// What a workgroup needs of its row: of K ranks {output, elements, rank 0, 1 ...; wide_words(K + 1) if they are wide}, or
// of `world` ranks, more than eight.
static_assert(sizeof(ShortRows) + 40 <= 4096, "kernel arguments");
template <typename S, typename D, int K>
struct ShortRow {
  const ShortRows& rows;
  const uint32_t* d;
  uint32_t row;
  __device__ __forceinline__ ShortRow(const ShortRows& r, uint32_t nrows, uint32_t chunk, uint32_t)
      : rows(r), row(row_of(r, nrows, chunk)) {
    d = r.d + row * (K + 2 + (r.wide ? wide_words(K + 1) : 0));
  }
  __device__ __forceinline__ uint64_t elements() const { return d[1]; }
  __device__ __forceinline__ gptr<D> output() const { return as_global<D>(rows.base[0]) + distance(rows, d, 0, K + 2, 0); }
  __device__ __forceinline__ gptr<const S> input(uint32_t r) const {
    return as_global<const S>(rows.base[1 + r]) + distance(rows, d, 2 + r, K + 2, 1 + r);
  }
};
template <typename S, typename D>
struct LongRow {
  const uint64_t* q;  // {output, elements, input of rank 0, 1 ...}
  uint32_t row;
  __device__ __forceinline__ LongRow(const Rows& r, uint32_t nrows, uint32_t chunk, uint32_t world)
      : row(row_of(r, nrows, chunk)) {
    q = r.q + row * (world + 2);
  }
  __device__ __forceinline__ uint64_t elements() const { return q[1]; }
  __device__ __forceinline__ gptr<D> output() const { return as_global<D>(q[0]); }
  __device__ __forceinline__ gptr<const S> input(uint32_t r) const { return as_global<const S>(q[2 + r]); }
};
template <int K>
using RowsOf = typename std::conditional<K == kTogether, Rows, ShortRows>::type;  // of ranks_sum_k
template <typename S, typename D, int K>
using RowOf = typename std::conditional<K == kTogether, LongRow<S, D>, ShortRow<S, D, K>>::type;

// For 1, 2 and more than 8 ranks.  One workgroup per chunk of kWG * kVec elements: 4 KiB of the wider side, one 16-byte
// access per lane and rank, the loads of the first K ranks (K = min(world, 8)) all in flight before the first add.  The
// arguments stay in the scalar cache, so a workgroup waits for one vector load (the search) and one batch of scalar
// loads (its row) before its data loads go out.  Two or four accesses per lane in a loop (8 and 16 KiB) are 3-10 %
// slower at 8 ranks (BERT-large 446 -> 489 us), loads without the non-temporal hint 8 %; runs of 64 KiB to 1 MiB per
// XCD measure within 2 % of each other.
template <typename S, typename W, typename D, int K, int ST>
__global__ __launch_bounds__(kWG) void ranks_sum_k(uint32_t shift, uint32_t ordered, uint32_t nrows, uint32_t world,
                                                   double pre, double post, uint32_t flags, RowsOf<K> rows) {
  constexpr int VEC = kVec<S, D>;
  constexpr uint32_t kTile = kWG * VEC;
  constexpr bool kBytes = sizeof(S) == 1;  // byte elements are read through windows (vecmem.h)
  const uint32_t chunk = xcd_tile(blockIdx.x, XcdOrder{shift, ordered});
  const RowOf<S, D, K> row(rows, nrows, chunk, world);
  const uint64_t start = (uint64_t)(chunk - rows.first[row.row]) * kTile;
  const uint64_t left = row.elements() - start;
  const uint32_t m = left < kTile ? (uint32_t)left : kTile;
  gptr<D> out = row.output() + start;
  const Window win = store_window<ST>(out, m * (uint32_t)sizeof(D));
  const typename Factor<W>::type fin = (typename Factor<W>::type)pre, fout = (typename Factor<W>::type)post;
  const bool scale_in = flags & kScaleIn, scale_out = flags & kScaleOut;
  auto source = [&](uint32_t rank) { return row.input(rank) + start; };
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
      add_ranks<kTogether, W, VEC>(acc, K, world, [&](uint32_t r) { return load(source(r)); }, wire);
    }
    stw<ST, D, VEC>(win, v * (uint32_t)(VEC * sizeof(D)), from_wire<W, D, VEC>(acc, fout, scale_out));
  }
  const uint32_t t = nv * VEC + threadIdx.x;  // fewer than VEC elements remain
  if (t < m) {
    auto load = [&](uint32_t r) { return Arr<S, 1>{source(r)[t]}; };
    auto wire = [&](const Arr<S, 1>& x) { return to_wire<S, W, 1>(x, fin, scale_in); };
    Arr<W, 1> acc = wire(load(0));
    add_ranks<K == kTogether ? kTogether : 1, W, 1>(acc, 1, world, load, wire);
    out[t] = from_wire<W, D, 1>(acc, fout, scale_out).v[0];
  }
  if constexpr (ST == kStoreWT) {  // into a fusion buffer: zeros up to the next 16-byte boundary
    const uint32_t pad = (uint32_t)(0u - (uint32_t)row.elements() * (uint32_t)sizeof(D)) & 15u;
    if (left <= kTile && threadIdx.x < pad) as_global<uint8_t>(win.base)[left * sizeof(D) + threadIdx.x] = 0;
  }
}

// The same for 3 to 8 ranks, split over the wavefronts of a workgroup: wavefront w loads the tile of ranks w and
// w + WV, all meet in LDS as wire values, and the first U wavefronts add them in rank order and store.  What bounds the
// sum of many streams is how much of them is in flight: 2,048 workgroups of the kernel above have 64 MiB of 8 ranks under
// way, more than latency times bandwidth by far and spread over as many DRAM pages, and stream at 6.0 TB/s; a plain
// sum of 8 x 128 MiB gains when it is held to fewer resident wavefronts (201 -> 185 us) and most with this tile of
// 1 KiB per rank and two loads per lane (181 us).  fp32, 8 ranks: BERT-large's layers of one response 158.5 -> 151
// us (6.5 TB/s), with fp16 on the wire 159.5 -> 150.5, fp16 80.5 -> 76.5, ResNet-50's gradients 158 -> 151.5; 4 ranks
// 85.8 -> 83.7, 5 ranks 106 -> 99, 6 ranks 123 -> 118, below 16 MiB per rank no difference.  With an odd number of
// ranks a wavefront has one load to wait for, so a lane takes two vectors of each (5 ranks, one vector: 112 us); more
// per workgroup in a loop that loads ahead is slower (4 tiles: 161 us, 8: 176).  Runs of 256 KiB per XCD gain 1-4 % at
// 3 to 6 ranks; with 8 they lose 2-5 % on the responses of ResNet-50, BERT-large and GPT-2 XL and on single tensors from
// 64 MiB a rank on (200 MiB 288 and 304 us), and gain up to 16 MiB (4 MiB 9.1 and 7.9).
template <typename S, typename W, typename D, int K, int ST>
__global__ __launch_bounds__(64 * kSplitWaves<K>) void ranks_split_k(uint32_t shift, uint32_t ordered, uint32_t nrows,
                                                                     double pre, double post, uint32_t flags,
                                                                     ShortRows rows) {
  constexpr int VEC = kVec<S, D>, WV = kSplitWaves<K>, U = kSplitVecs<K>;
  constexpr uint32_t kTile = 64 * U * VEC;
  constexpr bool kBytes = sizeof(S) == 1;
  static_assert(U <= WV, "a wavefront per 64 vectors of the sum");
  __shared__ Arr<W, VEC> lds[K][64 * U];
  const uint32_t chunk = xcd_tile(blockIdx.x, XcdOrder{shift, ordered});
  const ShortRow<S, D, K> row(rows, nrows, chunk, K);
  const uint64_t start = (uint64_t)(chunk - rows.first[row.row]) * kTile;
  const uint64_t left = row.elements() - start;
  const uint32_t m = left < kTile ? (uint32_t)left : kTile;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
  const typename Factor<W>::type fin = (typename Factor<W>::type)pre, fout = (typename Factor<W>::type)post;
  const bool scale_in = flags & kScaleIn, scale_out = flags & kScaleOut;
  auto source = [&](uint32_t rank) { return row.input(rank) + start; };
  const bool second = K == 2 * WV || wave + WV < K;
  const gptr<const S> src[2] = {source(wave), source(second ? wave + WV : wave)};
  const uint32_t nv = m / VEC;
  auto load = [&](gptr<const S> p, uint32_t v) {
    if constexpr (kBytes) {
      return ldw<S, VEC>(load_window(p, m), v * 16u);
    } else {
      return ldv<S, VEC>(p + (size_t)v * VEC);
    }
  };
  Arr<S, VEC> x[U][2];
#pragma unroll
  for (uint32_t u = 0; u < U; ++u) {
    const uint32_t v = u * 64 + lane;
    if (v < nv) {
      x[u][0] = load(src[0], v);
      if (second) x[u][1] = load(src[1], v);
    }
  }
#pragma unroll
  for (uint32_t u = 0; u < U; ++u) {
    const uint32_t v = u * 64 + lane;
    if (v < nv) {
      lds[wave][v] = to_wire<S, W, VEC>(x[u][0], fin, scale_in);
      if (second) lds[wave + WV][v] = to_wire<S, W, VEC>(x[u][1], fin, scale_in);
    }
  }
  __syncthreads();
  gptr<D> out = row.output() + start;
  const Window win = store_window<ST>(out, m * (uint32_t)sizeof(D));
  const uint32_t v = threadIdx.x;
  if (v < nv) {
    Arr<W, VEC> acc = lds[0][v];
#pragma unroll
    for (int k = 1; k < K; ++k) add_to<W, VEC>(acc, lds[k][v]);
    stw<ST, D, VEC>(win, v * (uint32_t)(VEC * sizeof(D)), from_wire<W, D, VEC>(acc, fout, scale_out));
  }
  const uint32_t t = nv * VEC + threadIdx.x;  // fewer than VEC elements remain
  if (t < m) {
    auto wire = [&](uint32_t r) { return to_wire<S, W, 1>(Arr<S, 1>{source(r)[t]}, fin, scale_in); };
    Arr<W, 1> acc = wire(0);
    for (uint32_t r = 1; r < K; ++r) add_to<W, 1>(acc, wire(r));
    out[t] = from_wire<W, D, 1>(acc, fout, scale_out).v[0];
  }
  if constexpr (ST == kStoreWT) {  // into a fusion buffer: zeros up to the next 16-byte boundary
    const uint32_t pad = (uint32_t)(0u - (uint32_t)row.elements() * (uint32_t)sizeof(D)) & 15u;
    if (left <= kTile && threadIdx.x < pad) as_global<uint8_t>(win.base)[left * sizeof(D) + threadIdx.x] = 0;
  }
}

// ---- host side ---------------------------------------------------------------------------------

// A launch of ranks_split_k for K from 3 to 8, of ranks_sum_k for K = 1, 2 and (K = 0) more than 8 ranks.
template <int K>
constexpr bool kSplit = K >= 3;

// The rows of one launch.  add() refuses one that it has no room for.
class LongTable {
 public:
  explicit LongTable(uint32_t world) : world_(world), max_(std::min(kMaxRows, kQwords / (world + 2))) {}
  uint32_t rows() const { return n_; }
  // Elements that a row can have, a multiple of `tile`.
  static uint64_t most(uint64_t) { return ~0ull; }
  template <typename Input>
  bool add(uint32_t first, uint64_t output, uint64_t elements, Input&& input) {
    if (n_ == max_) return false;
    uint64_t* q = table_.q + n_ * (world_ + 2);
    *q++ = output;
    *q++ = elements;
    for (uint32_t r = 0; r < world_; ++r) *q++ = input(r);
    table_.first[n_++] = first;
    return true;
  }
  const Rows& finished() {
    for (uint32_t i = n_; i < kMaxRows; ++i) table_.first[i] = ~0u;
    n_ = 0;
    return table_;
  }

 private:
  const uint32_t world_, max_;
  uint32_t n_ = 0;
  Rows table_;
};

// IS and OS: bytes of an element on either side, which every address is a multiple of.
template <int K, uint32_t IS, uint32_t OS>
class ShortTable {
 public:
  explicit ShortTable(uint32_t) {}
  uint32_t rows() const { return n_; }
  static uint64_t most(uint64_t tile) { return kShortReach / tile * tile; }
  template <typename Input>
  bool add(uint32_t first, uint64_t output, uint64_t elements, Input&& input) {
    constexpr uint32_t short_max = std::min(kMaxShortRows, kShortWords / (K + 2));
    constexpr uint32_t wide_max = std::min(kMaxShortRows, kShortWords / (K + 2 + wide_words(K + 1)));
    if (n_ == short_max || (wide_ && n_ == wide_max)) return false;
    uint64_t* at = at_[n_];
    at[0] = output;
    for (uint32_t r = 0; r < K; ++r) at[1 + r] = input(r);
    uint64_t lo[K + 1], hi[K + 1];
    bool wide = wide_;
    for (uint32_t r = 0; r <= K; ++r) {
      lo[r] = n_ ? std::min(lo_[r], at[r]) : at[r];
      hi[r] = n_ ? std::max(hi_[r], at[r]) : at[r];
      const uint64_t span = (hi[r] - lo[r]) / (r ? IS : OS);  // 0 for the first row of a launch
      if (span > kShortReach) wide = true;
      if (span > kWideReach || (wide && n_ >= wide_max)) return false;
    }
    wide_ = wide;
    std::copy(lo, lo + K + 1, lo_);
    std::copy(hi, hi + K + 1, hi_);
    elements_[n_] = (uint32_t)elements;
    table_.first[n_++] = first;
    return true;
  }
  const ShortRows& finished() {
    constexpr uint32_t high = K + 2;
    const uint32_t words = high + (wide_ ? wide_words(K + 1) : 0);
    for (uint32_t i = 0; i < n_; ++i) {
      uint32_t* d = table_.d + i * words;
      std::fill(d + high, d + words, 0u);
      d[1] = elements_[i];
      set_distance(d, 0, high, 0, (at_[i][0] - lo_[0]) / OS, wide_);
      for (uint32_t r = 0; r < K; ++r) set_distance(d, 2 + r, high, 1 + r, (at_[i][1 + r] - lo_[1 + r]) / IS, wide_);
    }
    std::copy(lo_, lo_ + K + 1, table_.base);
    table_.wide = wide_ ? 0xff : 0;
    for (uint32_t i = n_; i < kMaxShortRows; ++i) table_.first[i] = ~0u;
    n_ = 0;
    wide_ = false;
    return table_;
  }

 private:
  uint32_t n_ = 0;
  bool wide_ = false;
  uint32_t elements_[kMaxShortRows];
  uint64_t lo_[K + 1], hi_[K + 1], at_[kMaxShortRows][K + 1];
  ShortRows table_;
};

template <typename S, typename W, typename D, int K, int ST, typename Table>
hipError_t launch_rows(const RanksCall& c, Table& table, uint32_t chunks, bool last) {
  constexpr uint32_t kVecBytes = kVec<S, D> * (uint32_t)(sizeof(S) > sizeof(D) ? sizeof(S) : sizeof(D));
  hipEvent_t completion = last ? c.completion : nullptr;
  const uint32_t nrows = table.rows();
  if constexpr (kSplit<K>) {
    const XcdOrder order = K < 8 ? xcd_order(chunks, 64 * kSplitVecs<K> * kVecBytes) : XcdOrder{0, 0};
    return launch_shaped(completion, ranks_split_k<S, W, D, K, ST>, chunks, 64 * kSplitWaves<K>, c.stream, order.shift,
                         order.ordered, nrows, c.pre, c.post, c.flags, table.finished());
  } else {
    const XcdOrder order = xcd_order(chunks, kWG * kVecBytes);
    return launch_with(completion, ranks_sum_k<S, W, D, K ? K : kTogether, ST>, chunks, c.stream, order.shift,
                       order.ordered, nrows, c.world, c.pre, c.post, c.flags, table.finished());
  }
}

// Fills launches with as many rows as their arguments hold.  A tensor that would take a launch beyond
// kMaxWorkgroups chunks, or has more elements than a row can say, is cut there and goes on in the next one.
template <typename S, typename W, typename D, int K>
int run_ranks(const RanksCall& c) {
  constexpr uint64_t kTile = (uint64_t)(kSplit<K> ? 64 * kSplitVecs<K> : kWG) * kVec<S, D>;
  typedef typename std::conditional<K != 0, ShortTable<K ? K : 1, sizeof(S), sizeof(D)>, LongTable>::type Table;
  int entry = 0;
  uint64_t done = 0;  // elements of the current entry that earlier launches took
  // One rank's tensor that is its own output and changes neither type nor scale is left where it is.
  const bool may_stay = K == 1 && std::is_same<S, W>::value && std::is_same<W, D>::value && c.flags == 0;
  auto skip_idle = [&] {
    while (entry < c.n && (c.counts[entry] == 0 || (may_stay && c.inputs[entry] == c.outputs[entry]))) ++entry;
  };
  skip_idle();
  if (entry == c.n) {
    if (c.completion) HVDHIP_CHECK(hipEventRecord(c.completion, c.stream));
    return 0;
  }
  Table table(c.world);
  while (entry < c.n) {
    uint64_t chunks = 0;
    while (entry < c.n && chunks < kMaxWorkgroups) {
      const uint64_t left = (uint64_t)c.counts[entry] - done;
      const uint64_t take = std::min(std::min(left, Table::most(kTile)), (kMaxWorkgroups - chunks) * kTile);
      auto input = [&](uint32_t r) {
        return (uint64_t)(uintptr_t)c.inputs[(size_t)r * (size_t)c.n + (size_t)entry] + done * sizeof(S);
      };
      if (!table.add((uint32_t)chunks, (uint64_t)(uintptr_t)c.outputs[entry] + done * sizeof(D), take, input)) break;
      chunks += (take + kTile - 1) / kTile;
      done += take;
      if (take == left) {
        done = 0;
        ++entry;
        skip_idle();
      }
    }
    const bool last = entry == c.n;
    const hipError_t status = c.flags & kPadOut
                                  ? launch_rows<S, W, D, K, kStoreWT>(c, table, (uint32_t)chunks, last)
                                  : launch_rows<S, W, D, K, kStoreNT>(c, table, (uint32_t)chunks, last);
    HVDHIP_CHECK_LAUNCH("ranks_sum_k", status);
  }
  return 0;
}

template <typename S, typename W, typename D>
int run(const RanksCall& c) {
  switch (c.world) {
  case 1: return run_ranks<S, W, D, 1>(c);
  case 2: return run_ranks<S, W, D, 2>(c);
  case 3: return run_ranks<S, W, D, 3>(c);
  case 4: return run_ranks<S, W, D, 4>(c);
  case 5: return run_ranks<S, W, D, 5>(c);
  case 6: return run_ranks<S, W, D, 6>(c);
  case 7: return run_ranks<S, W, D, 7>(c);
  case 8: return run_ranks<S, W, D, 8>(c);
  default: return run_ranks<S, W, D, 0>(c);
  }
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
  try {
    if (overlaps(*c, (uint64_t)is, (uint64_t)os))
      return fail(HVDHIP_ERR_OVERLAP, "an output overlaps another output or another entry's input");
  } catch (const std::bad_alloc&) {  // must not leave through a C interface
    return fail(HVDHIP_ERR_OUT_OF_MEMORY, "no host memory to compare %d outputs", c->n);
  }
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
