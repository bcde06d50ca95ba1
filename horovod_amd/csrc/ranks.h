// ranks.h -- shared by the kernels that read every rank's tensors where they sit in this device's memory
// (not installed): the addresses in a launch's arguments, an element's way to the wire type and back,
// and the checks of a call.
#ifndef HVDHIP_RANKS_H
#define HVDHIP_RANKS_H

#include "internal.h"
#include "vecmem.h"

namespace hvdhip {

constexpr uint32_t kMaxRows = 64;   // one lane of a wavefront looks at each
constexpr uint32_t kQwords = 440;   // addresses and counts: with `first` and the scalars below 4 KiB

// first[i]: the first chunk of row i; beyond the last row a number no chunk reaches.
// q: a few words per row, the same number for every row of a launch (addresses and the element count).
struct Rows {
  uint32_t first[kMaxRows];
  uint64_t q[kQwords];
};

// The row that `chunk` of a launch belongs to; every wavefront finds it by itself: a lane per row compares
// the row's first chunk, and the count of lanes at or below is the row.
__device__ __forceinline__ uint32_t row_of(const Rows& rows, uint32_t nrows, uint32_t chunk) {
  if (nrows <= 1) return 0;
  return (uint32_t)__popcll(__ballot(rows.first[threadIdx.x & 63] <= chunk)) - 1;
}

// The same for up to eight ranks with addresses as distances, in elements, from the lowest one of each rank (and of the
// outputs): 32 bits each, and where some are further apart 8 more, four to a word behind the row's others.  A launch
// carries up to 128 tensors so, 84 of eight ranks (65 with the wide distances) where 64-bit addresses leave room for 44.
// Each launch more costs the stream 4 to 5 us between one's drain and the next one's start: sums of eight ranks,
// ResNet-50's 161 gradients 153 -> 146 us, 320 tensors of 8 million elements in all 77 -> 63, 200 of 2 million 47 -> 38.
// (Two allocations of the framework's are easily 32 GiB apart: its small segments and its large ones.)
constexpr uint32_t kMaxShortRows = 128;  // two per lane of a wavefront
constexpr uint32_t kShortWords = 848;
struct ShortRows {
  uint32_t first[kMaxShortRows];  // as in Rows
  uint64_t base[9];               // outputs, rank 0, 1 ...
  uint32_t wide;                  // 0xff if the rows have the words with bits 32 to 39, else 0
  uint32_t d[kShortWords + 3];    // a few words per row; the last three are there to be loaded, not used
};
constexpr uint64_t kShortReach = 0xffffffffull, kWideReach = 0xffffffffffull;  // largest distances
constexpr uint32_t wide_words(uint32_t distances) { return (distances + 3) / 4; }

// Distance k of a row: its low word is d[low], the words of high bits start at d[high].
__device__ __forceinline__ uint64_t distance(const ShortRows& rows, const uint32_t* d, uint32_t low, uint32_t high,
                                             uint32_t k) {
  return d[low] | (uint64_t)(d[high + k / 4] >> k % 4 * 8 & rows.wide) << 32;
}
// The host's side of it: the row's words of high bits are zero before the first call.
inline void set_distance(uint32_t* d, uint32_t low, uint32_t high, uint32_t k, uint64_t value, bool wide) {
  d[low] = (uint32_t)value;
  if (wide) d[high + k / 4] |= (uint32_t)(value >> 32) << k % 4 * 8;
}

__device__ __forceinline__ uint32_t row_of(const ShortRows& rows, uint32_t nrows, uint32_t chunk) {
  if (nrows <= 1) return 0;
  const uint32_t lane = threadIdx.x & 63, low = rows.first[lane], high = rows.first[64 + lane];
  return (uint32_t)__popcll(__ballot(low <= chunk)) + (uint32_t)__popcll(__ballot(high <= chunk)) - 1;
}

enum : uint32_t { kScaleIn = 1, kScaleOut = 2, kPadOut = 4 };

// The factor of a scaled type, prepared once per workgroup from the doubles of the launch.
template <typename T>
struct Factor {
  typedef double type;
};
template <>
struct Factor<float> {
  typedef float type;
};
template <>
struct Factor<half_t> {
  typedef float type;
};

// ScaleBufferCPUImpl's element (ops/collective_operations.h:91-127), as in xfer.hip.  Device code contracts by default,
// and what follows here is a sum: the product has to be rounded by itself first.  A byte's product goes through 32 bits:
// straight to a byte it is undefined outside of the byte's range, and the compiler leaves what lies above eight bits in
// the register.
template <typename T>
__device__ __forceinline__ T scaled(T x, typename Factor<T>::type s) {
#pragma clang fp contract(off)
  if constexpr (sizeof(T) == 1) return (T)(int32_t)(s * x);
  return (T)(s * x);
}
template <>
__device__ __forceinline__ half_t scaled<half_t>(half_t x, float s) {
  return (half_t)opaque(s * (float)x);
}

template <typename S, typename D, int N>
__device__ __forceinline__ Arr<D, N> converted(const Arr<S, N>& x) {
  if constexpr (std::is_same<S, D>::value) {
    return x;
  } else {
    Arr<D, N> y;
#pragma unroll
    for (int j = 0; j < N; ++j) y.v[j] = (D)x.v[j];
    return y;
  }
}

// N elements on their way in (tensor type S to wire type W) and out (W to D): converted before or
// after the wire, scaled on it (compress, then scale: horovod/torch/compression.py:49-55 before the
// fp16 ScaleBuffer; the converting unpack scales the half and widens).  16-bit integers are summed and
// copied but never scaled.
template <typename W, int N>
__device__ __forceinline__ void scale_all(Arr<W, N>& x, typename Factor<W>::type s) {
  if constexpr (sizeof(W) == 1 && N == 16) {
    asm volatile("");  // or the compiler scales in any case and picks one of the two
    x = scaled_bytes(x, s);
  } else if constexpr (!std::is_same<W, uint16_t>::value) {
#pragma unroll
    for (int j = 0; j < N; ++j) x.v[j] = scaled<W>(x.v[j], s);
  }
}
template <typename S, typename W, int N>
__device__ __forceinline__ Arr<W, N> to_wire(const Arr<S, N>& x, typename Factor<W>::type s, bool scale) {
  Arr<W, N> y = converted<S, W, N>(x);
  if (scale) scale_all(y, s);
  return y;
}
template <typename W, typename D, int N>
__device__ __forceinline__ Arr<D, N> from_wire(Arr<W, N> x, typename Factor<W>::type s, bool scale) {
  if (scale) scale_all(x, s);
  return converted<W, D, N>(x);
}

template <typename S, typename D>
constexpr int kVec = 16 / (int)(sizeof(S) > sizeof(D) ? sizeof(S) : sizeof(D));

struct RanksCall {
  void* const* outputs;
  const void* const* inputs;  // rank-major: inputs[rank * n + entry]
  const int64_t* counts;
  int n;
  uint32_t world;
  double pre, post;
  uint32_t flags;
  hipStream_t stream;
  hipEvent_t completion;
};

// Checks the arguments of a call and fills in its flags and factors (HVDHIP_ERR_OVERLAP: an output overlaps
// another output, or an input that is not exactly its own entry's).
int check_ranks_call(RanksCall* c, int in_dtype, int wire_dtype, int out_dtype);

}  // namespace hvdhip

#endif  // HVDHIP_RANKS_H
