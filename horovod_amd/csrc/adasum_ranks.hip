// adasum_ranks.hip -- Adasum over the ranks of a fused response whose tensors all sit in this device's memory: the
// pairwise tree of Adasum::FusedAllreduce (ops/adasum/adasum.h:194-340), distances 1, 2, 4 ..., each tensor a
// layer of its own.  gfx950 only.
//
// The sequence it replaces -- every rank packs into a buffer, then per pair a pass for the sums and one for the
// scaled add, then an unpack -- moves 2 R + 5 (R - 1) + 2 vectors for R ranks, 53 for eight.  Here a level's scaled
// add and the next level's sums are one pass, and the ends read and write the tensors themselves:
//
//   dots_k   reads the ranks pairwise, leaves each pair's sums                                (R)
//   level_k  reads four vectors of a level, combines them to two, stores those for the next
//            level and leaves the sums of the two                            (R + R/2, R/2 + R/4 ...)
//   last_k   reads the last two, combines them, stores the result into the outputs            (2 + 1)
//
// A response of rows that fit the registers of a workgroup goes through the tree in one launch (tree_held_k).
//
// 29 vectors for eight ranks, in 4 launches instead of 23, and a launch of coeffs_k between two passes where a tensor has
// more than 512 chunks.  Every pass is bound by memory: a BERT-large layer (16 tensors, 50 MB, four of them of 1,024
// chunks) of eight ranks takes 230 us in 7 launches: dots_k 62, level_k 86 and 44, last_k 23.5 us, 6.8 TB/s over the 1.46
// GB that the passes move, and 15 us of coeffs_k; the separate steps move 2.67 GB in 443 us.  What level_k stores goes
// through the Infinity Cache to its reader (non-temporal stores take the passes 24 us more).  Sums of all pairs at once
// would spare the levels their own (17 vectors), but a level's norm as a difference of the ranks' products has no digits
// left where ranks nearly cancel.
//
// All roundings are those of the separate steps: to the wire type after the prescale, after every level's scaled add
// and in the output.  The sums are taken in double in an order that depends on the tensor's size alone.
#include <algorithm>
#include <cfloat>
#include <cmath>

#include "adasum_math.h"
#include "ranks.h"

namespace hvdhip {
namespace {

constexpr uint32_t kRanksAtOnce = 8;      // ranks whose addresses one launch carries
constexpr uint32_t kChunkBytes = 16384;   // of the wire type per workgroup and vector
constexpr uint32_t kSumsPerLane = 4;      // partial sums that a lane fetches at a time
// Chunks of a row up to which its consumers add the partial sums themselves (12 KiB per pair, from L2, beside the
// 32 to 64 KiB of data that a workgroup reads); beyond, a launch of coeffs_k per level does, 4.6 us.
constexpr uint32_t kReaddMax = 512;

template <typename W>
constexpr uint32_t kChunk = kChunkBytes / (uint32_t)sizeof(W);

// What a launch works on besides its rows.  Vectors between levels lie in the workspace, `in_stride` and
// `out_stride` bytes apart; sums[(pair * chunks + chunk) * 3] is a pair's triple for a chunk of the launch's rows.
struct Level {
  uint32_t nrows;
  uint32_t chunks;
  uint32_t words;  // per row in ShortRows::d
  uint32_t high;   // where in it the words of high bits start
  uint32_t first;  // pair (dots_k) or group of four vectors (level_k) that blockIdx.y = 0 works on
  uint32_t flags;
  uint64_t in_stride, out_stride;
  double pre, post, guard;
  const double* in_sums;
  const double* coeffs;  // [(pair * kMaxShortRows + row) * 2], or NULL: from in_sums
  double* out_sums;
};

// A row: {distance from base[0], elements in two words, distances from base[1], base[2] ...; wide_words() of them if they
// are wide}.
constexpr uint32_t kRowHead = 3;
static_assert(sizeof(ShortRows) + sizeof(Level) <= 4096, "kernel arguments");

struct Place {
  const uint32_t* d;
  uint32_t high;  // where the row's words of high bits are
  uint32_t row, chunk;
  uint64_t elements, start;  // of the row; element within it
  uint32_t m;                // elements of this chunk
  // What base[k] is the lowest one of.
  template <typename T>
  __device__ __forceinline__ gptr<T> at(const ShortRows& rows, uint32_t k) const {
    return as_global<T>(rows.base[k]) + distance(rows, d, k == 0 ? 0 : kRowHead - 1 + k, high, k);
  }
};
__device__ __forceinline__ uint64_t row_elements(const uint32_t* d) { return d[1] | (uint64_t)d[2] << 32; }
template <typename W>
__device__ __forceinline__ Place place(const ShortRows& rows, const Level& l) {
  Place p;
  p.chunk = blockIdx.x;
  p.row = row_of(rows, l.nrows, p.chunk);
  p.d = rows.d + p.row * l.words;
  p.high = l.high;
  p.elements = row_elements(p.d);
  p.start = (uint64_t)(p.chunk - rows.first[p.row]) * kChunk<W>;
  const uint64_t left = p.elements - p.start;
  p.m = left < kChunk<W> ? (uint32_t)left : kChunk<W>;
  return p;
}

// f(std::integral_constant<int, U>, v): U vectors per lane at v, v + kWG ... while whole rounds are left, then one
// at a time.
template <int U, typename F>
__device__ __forceinline__ void over_vectors(uint32_t nv, F&& f) {
  uint32_t v = threadIdx.x;
  for (; v + (U - 1) * kWG < nv; v += U * kWG) f(std::integral_constant<int, U>(), v);
  if constexpr (U > 1) {
    for (; v < nv; v += kWG) f(std::integral_constant<int, 1>(), v);
  }
}

// Two fma chains per sum.
struct Sums {
  double d[2] = {0., 0.}, a[2] = {0., 0.}, b[2] = {0., 0.};
  template <typename W, int N>
  __device__ __forceinline__ void add(const Arr<W, N>& x, const Arr<W, N>& y) {
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const double p = (double)x.v[j], q = (double)y.v[j];
      d[j & 1] = fma(p, q, d[j & 1]);
      a[j & 1] = fma(p, p, a[j & 1]);
      b[j & 1] = fma(q, q, b[j & 1]);
    }
  }
  __device__ __forceinline__ void store(const Level& l, uint32_t pair, uint32_t chunk) const {
    const Triple r = wg_reduce(Triple{d[0] + d[1], a[0] + a[1], b[0] + b[1]});
    if (threadIdx.x == 0) {
      double* out = l.out_sums + 3 * ((uint64_t)pair * l.chunks + chunk);
      out[0] = r.d;
      out[1] = r.a;
      out[2] = r.b;
    }
  }
};

// A lane's part of a row's `chunks` triples: every LANES-th from `lane` on, of which there is at least one.
template <uint32_t LANES>
__device__ __forceinline__ Triple lane_sum(const double* s, uint32_t chunks, uint32_t lane) {
  Triple t = {0., 0., 0.};
  for (uint32_t i = lane; i < chunks; i += LANES * kSumsPerLane) {
    Triple r[kSumsPerLane];
#pragma unroll
    for (uint32_t u = 0; u < kSumsPerLane; ++u) {  // unconditional, so that all are in flight together
      const uint64_t at = 3 * (uint64_t)(i + LANES * u < chunks ? i + LANES * u : lane);
      r[u] = Triple{s[at], s[at + 1], s[at + 2]};
    }
#pragma unroll
    for (uint32_t u = 0; u < kSumsPerLane; ++u) {
      const bool in = i + LANES * u < chunks;
      t.d += in ? r[u].d : 0.;
      t.a += in ? r[u].a : 0.;
      t.b += in ? r[u].b : 0.;
    }
  }
  return t;
}

// The sum of at most kReaddMax triples by one wavefront, in lane 63.  Whether a row's consumers add it or coeffs_k does
// on account of a longer row beside it, the order is this one: a tensor's result does not depend on its company.
__device__ __forceinline__ Triple short_row_sum(const double* s, uint32_t chunks, uint32_t lane) {
  Triple t = lane_sum<64>(s, chunks, lane);
  t.d = wave_sum(t.d);
  t.a = wave_sum(t.a);
  t.b = wave_sum(t.b);
  return t;
}

// The coefficients of NP consecutive pairs of a row.  Without a table of them, wavefront w adds pair w's partial
// sums.
template <int NP>
__device__ __forceinline__ void row_coeffs(const Level& l, const Place& p, uint32_t first_chunk, uint32_t chunks,
                                           uint32_t pair, double (&c)[2 * NP]) {
  if (l.coeffs) {
    const double* t = l.coeffs + 2 * ((uint64_t)pair * kMaxShortRows + p.row);
#pragma unroll
    for (int k = 0; k < NP; ++k) {
      c[2 * k] = t[2 * kMaxShortRows * k];
      c[2 * k + 1] = t[2 * kMaxShortRows * k + 1];
    }
    return;
  }
  __shared__ double shared[2 * NP];
  const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  if (wave < NP) {
    const double* s = l.in_sums + 3 * ((uint64_t)(pair + wave) * l.chunks + first_chunk);
    const Triple t = short_row_sum(s, chunks, lane);
    if (lane == 63) layer_coeffs(t, l.guard, &shared[2 * wave], &shared[2 * wave + 1]);
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 2 * NP; ++k) c[k] = shared[k];
}

template <typename W, int N>
__device__ __forceinline__ Arr<W, N> combined(double ca, const Arr<W, N>& a, double cb, const Arr<W, N>& b) {
  Arr<W, N> y;
#pragma unroll
  for (int j = 0; j < N; ++j) y.v[j] = Axpby<W>::f(ca, a.v[j], cb, b.v[j]);
  return y;
}

// Bases: anything, rank 0, 1 ...  KEEP: whose tensors the loads leave in the Infinity Cache for the
// pass that reads them again (1 every pair's first rank's, 2 all).
template <typename S, typename W, int KEEP>
__global__ __launch_bounds__(kWG) void dots_k(Level l, ShortRows rows) {
  constexpr int VEC = kVec<S, W>;
  if (blockIdx.x >= l.chunks) return;
  const Place p = place<W>(rows, l);
  const gptr<const S> a = p.at<const S>(rows, 1 + 2 * blockIdx.y) + p.start;
  const gptr<const S> b = p.at<const S>(rows, 2 + 2 * blockIdx.y) + p.start;
  const typename Factor<W>::type fin = (typename Factor<W>::type)l.pre;
  const bool scale_in = l.flags & kScaleIn;
  Sums sums;
  over_vectors<4>(p.m / VEC, [&](auto u, uint32_t v) {
    constexpr int U = decltype(u)::value;
    Arr<S, VEC> x[U], y[U];
#pragma unroll
    for (int i = 0; i < U; ++i) {
      x[i] = ldv<S, VEC, false>(a + (size_t)(v + i * kWG) * VEC);
      y[i] = ldv<S, VEC, KEEP != 2>(b + (size_t)(v + i * kWG) * VEC);
    }
#pragma unroll
    for (int i = 0; i < U; ++i)
      sums.add(to_wire<S, W, VEC>(x[i], fin, scale_in), to_wire<S, W, VEC>(y[i], fin, scale_in));
  });
  const uint32_t t = p.m / VEC * VEC + threadIdx.x;
  if (t < p.m)
    sums.add(to_wire<S, W, 1>(Arr<S, 1>{a[t]}, fin, scale_in), to_wire<S, W, 1>(Arr<S, 1>{b[t]}, fin, scale_in));
  sums.store(l, l.first + blockIdx.y, p.chunk);
}

// LEAVES, bases: workspace, rank 0, 1 ...; else the workspace alone, and the vectors are in_stride
// apart in it, where the two results take the places of two of the four.
template <typename S, typename W, bool LEAVES>
__global__ __launch_bounds__(kWG) void level_k(Level l, ShortRows rows) {
  constexpr int VEC = kVec<S, W>;
  if (blockIdx.x >= l.chunks) return;
  const Place p = place<W>(rows, l);
  const uint32_t quad = l.first + blockIdx.y;
  const typename Factor<W>::type fin = (typename Factor<W>::type)l.pre;
  const bool scale_in = LEAVES && (l.flags & kScaleIn);
  const uint64_t work = reinterpret_cast<uint64_t>(p.at<W>(rows, 0));
  gptr<const S> in[4];
#pragma unroll
  for (uint32_t k = 0; k < 4; ++k)
    in[k] = (LEAVES ? p.at<const S>(rows, 1 + 4 * blockIdx.y + k)
                    : as_global<const S>(work + (uint64_t)(4 * quad + k) * l.in_stride)) + p.start;
  Window out[2];
  gptr<W> to[2];
#pragma unroll
  for (uint32_t k = 0; k < 2; ++k) {
    to[k] = as_global<W>(work + (uint64_t)(2 * quad + k) * l.out_stride) + p.start;
    out[k] = store_window<kStoreWT>(to[k], p.m * (uint32_t)sizeof(W));
  }
  double c[4];
  row_coeffs<2>(l, p, rows.first[p.row], (uint32_t)((p.elements + kChunk<W> - 1) / kChunk<W>), 2 * quad, c);
  Sums sums;
  over_vectors<2>(p.m / VEC, [&](auto u, uint32_t v) {
    constexpr int U = decltype(u)::value;
    Arr<S, VEC> x[U][4];
#pragma unroll
    for (int i = 0; i < U; ++i) {
#pragma unroll
      for (int k = 0; k < 4; ++k) x[i][k] = ldv<S, VEC>(in[k] + (size_t)(v + i * kWG) * VEC);
    }
#pragma unroll
    for (int i = 0; i < U; ++i) {
      Arr<W, VEC> y[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) y[k] = to_wire<S, W, VEC>(x[i][k], fin, scale_in);
      const Arr<W, VEC> r0 = combined<W, VEC>(c[0], y[0], c[1], y[1]), r1 = combined<W, VEC>(c[2], y[2], c[3], y[3]);
      stw<kStoreWT, W, VEC>(out[0], (v + i * kWG) * (uint32_t)(VEC * sizeof(W)), r0);
      stw<kStoreWT, W, VEC>(out[1], (v + i * kWG) * (uint32_t)(VEC * sizeof(W)), r1);
      sums.add(r0, r1);
    }
  });
  const uint32_t t = p.m / VEC * VEC + threadIdx.x;
  if (t < p.m) {
    Arr<W, 1> y[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) y[k] = to_wire<S, W, 1>(Arr<S, 1>{in[k][t]}, fin, scale_in);
    const Arr<W, 1> r0 = combined<W, 1>(c[0], y[0], c[1], y[1]), r1 = combined<W, 1>(c[2], y[2], c[3], y[3]);
    to[0][t] = r0.v[0];
    to[1][t] = r1.v[0];
    sums.add(r0, r1);
  }
  sums.store(l, quad, p.chunk);
}

// LEAVES (two ranks), bases: output, rank 0, rank 1; else output, workspace.
template <typename S, typename W, typename D, bool LEAVES>
__global__ __launch_bounds__(kWG) void last_k(Level l, ShortRows rows) {
  constexpr int VEC = kVec<S, D>;
  if (blockIdx.x >= l.chunks) return;
  const Place p = place<W>(rows, l);
  const typename Factor<W>::type fin = (typename Factor<W>::type)l.pre, fout = (typename Factor<W>::type)l.post;
  const bool scale_in = LEAVES && (l.flags & kScaleIn), scale_out = l.flags & kScaleOut;
  const gptr<const S> a = p.at<const S>(rows, 1) + p.start;
  const gptr<const S> b = LEAVES ? p.at<const S>(rows, 2) + p.start
                                 : as_global<const S>(reinterpret_cast<uint64_t>(a) + l.in_stride);
  const gptr<D> to = p.at<D>(rows, 0) + p.start;
  const Window out = store_window<kStoreNT>(to, p.m * (uint32_t)sizeof(D));
  double c[2];
  row_coeffs<1>(l, p, rows.first[p.row], (uint32_t)((p.elements + kChunk<W> - 1) / kChunk<W>), 0, c);
  over_vectors<4>(p.m / VEC, [&](auto u, uint32_t v) {
    constexpr int U = decltype(u)::value;
    Arr<S, VEC> x[U], y[U];
#pragma unroll
    for (int i = 0; i < U; ++i) {
      x[i] = ldv<S, VEC>(a + (size_t)(v + i * kWG) * VEC);
      y[i] = ldv<S, VEC>(b + (size_t)(v + i * kWG) * VEC);
    }
#pragma unroll
    for (int i = 0; i < U; ++i) {
      const Arr<W, VEC> r = combined<W, VEC>(c[0], to_wire<S, W, VEC>(x[i], fin, scale_in), c[1],
                                             to_wire<S, W, VEC>(y[i], fin, scale_in));
      stw<kStoreNT, D, VEC>(out, (v + i * kWG) * (uint32_t)(VEC * sizeof(D)), from_wire<W, D, VEC>(r, fout, scale_out));
    }
  });
  const uint32_t t = p.m / VEC * VEC + threadIdx.x;
  if (t < p.m) {
    const Arr<W, 1> r = combined<W, 1>(c[0], to_wire<S, W, 1>(Arr<S, 1>{a[t]}, fin, scale_in), c[1],
                                       to_wire<S, W, 1>(Arr<S, 1>{b[t]}, fin, scale_in));
    to[t] = from_wire<W, D, 1>(r, fout, scale_out).v[0];
  }
}

// One workgroup per row and pair of a level: the coefficients, where some row has more chunks than kReaddMax.
struct RowStarts {
  uint32_t first[kMaxShortRows + 1];
};
__global__ __launch_bounds__(kWG) void coeffs_k(const double* __restrict__ sums, double* __restrict__ coeffs,
                                                uint32_t chunks, double guard, RowStarts rows) {
  const uint32_t row = blockIdx.x, pair = blockIdx.y;
  const uint32_t first = rows.first[row], count = rows.first[row + 1] - first;
  const double* s = sums + 3 * ((uint64_t)pair * chunks + first);
  double* c = coeffs + 2 * ((uint64_t)pair * kMaxShortRows + row);
  if (count <= kReaddMax) {
    if (threadIdx.x >= 64) return;
    const Triple r = short_row_sum(s, count, threadIdx.x);
    if (threadIdx.x == 63) layer_coeffs(r, guard, &c[0], &c[1]);
  } else {
    const Triple r = wg_reduce(lane_sum<kWG>(s, count, threadIdx.x));
    if (threadIdx.x == 0) layer_coeffs(r, guard, &c[0], &c[1]);
  }
}

// ---- rows that fit a workgroup -----------------------------------------------------------------

// A chunk of every rank in the registers of 256 lanes.  The vectors are pinned where they are used: the compiler would
// keep widened halves from the sums to the scaled add, in four times the registers.
template <typename W, int WORLD>
struct HeldRanks {
  static constexpr int VEC = 16 / (int)sizeof(W), kVecs = (int)(kChunkBytes / 16 / kWG);
  typedef RawSel<16>::type R;
  uint32_t m, nv, lane;
  R x[WORLD][kVecs];
  W t[WORLD];  // the element behind the last whole vector

  static __device__ __forceinline__ Arr<W, VEC> pinned(R& r) {
    asm("" : "+v"(r));
    return __builtin_bit_cast(Arr<W, VEC>, r);
  }
  __device__ __forceinline__ bool has_tail() const { return nv * VEC + lane < m; }

  __device__ __forceinline__ void load(const ShortRows& rows, const Place& at, uint32_t lane_,
                                       typename Factor<W>::type fin, bool scale_in) {
    m = at.m;
    nv = m / VEC;
    lane = lane_;
#pragma unroll
    for (int r = 0; r < WORLD; ++r) {
      const gptr<const W> p = at.at<const W>(rows, 1 + r) + at.start;
#pragma unroll
      for (int u = 0; u < kVecs; ++u)
        if (lane + u * kWG < nv) x[r][u] = __builtin_bit_cast(R, ldv<W, VEC>(p + (size_t)(lane + u * kWG) * VEC));
      if (has_tail()) t[r] = p[nv * VEC + lane];
    }
    if (!scale_in) return;
#pragma unroll
    for (int r = 0; r < WORLD; ++r) {
#pragma unroll
      for (int u = 0; u < kVecs; ++u)
        if (lane + u * kWG < nv) x[r][u] = __builtin_bit_cast(R, to_wire<W, W, VEC>(pinned(x[r][u]), fin, true));
      if (has_tail()) t[r] = to_wire<W, W, 1>(Arr<W, 1>{t[r]}, fin, true).v[0];
    }
  }
};

// The levels of the tree from PAIRS pairs on, the vectors in the first 2 * PAIRS places; the result ends in the first.
template <int PAIRS, typename W, int WORLD, int G>
__device__ __forceinline__ void held_levels(HeldRanks<W, WORLD>& h, uint32_t group, double guard,
                                            double (*red)[WORLD / 2][3][kWG / 64]) {
  constexpr int VEC = HeldRanks<W, WORLD>::VEC, kVecs = HeldRanks<W, WORLD>::kVecs;
  const uint32_t l64 = threadIdx.x & 63;
#pragma unroll
  for (int p = 0; p < PAIRS; ++p) {
    Sums sums;
#pragma unroll
    for (int u = 0; u < kVecs; ++u)
      if (h.lane + u * kWG < h.nv) sums.add(h.pinned(h.x[2 * p][u]), h.pinned(h.x[2 * p + 1][u]));
    if (h.has_tail()) sums.add(Arr<W, 1>{h.t[2 * p]}, Arr<W, 1>{h.t[2 * p + 1]});
    const double d = wave_sum(sums.d[0] + sums.d[1]), a = wave_sum(sums.a[0] + sums.a[1]),
                 b = wave_sum(sums.b[0] + sums.b[1]);
    if (l64 == 63) {
      red[group][p][0][h.lane / 64] = d;
      red[group][p][1][h.lane / 64] = a;
      red[group][p][2][h.lane / 64] = b;
    }
  }
  __syncthreads();
  // Every wavefront adds the chunks' sums for itself, a lane per coefficient, with the bits of wg_reduce and
  // short_row_sum.
  const uint32_t k = l64 < 2 * PAIRS ? l64 : 0;
  double d = 0., n = 0., c, other;
#pragma unroll
  for (int g = 0; g < G; ++g) {
    double rd = 0., rn = 0.;
#pragma unroll
    for (int w = 0; w < kWG / 64; ++w) {
      rd += red[g][k / 2][0][w];
      rn += red[g][k / 2][1 + k % 2][w];
    }
    d += rd;
    n += rn;
  }
  layer_coeffs(Triple{d, n, n}, guard, &c, &other);
#pragma unroll
  for (int p = 0; p < PAIRS; ++p) {
    const double ca = lane_value(c, 2 * p), cb = lane_value(c, 2 * p + 1);
#pragma unroll
    for (int u = 0; u < kVecs; ++u)
      if (h.lane + u * kWG < h.nv)
        h.x[p][u] = __builtin_bit_cast(typename HeldRanks<W, WORLD>::R,
                                       combined<W, VEC>(ca, h.pinned(h.x[2 * p][u]), cb, h.pinned(h.x[2 * p + 1][u])));
    if (h.has_tail()) h.t[p] = combined<W, 1>(ca, Arr<W, 1>{h.t[2 * p]}, cb, Arr<W, 1>{h.t[2 * p + 1]}).v[0];
  }
  if constexpr (PAIRS > 1) held_levels<PAIRS / 2, W, WORLD, G>(h, group, guard, red + G);
}

// The whole tree of rows of at most G chunks, a workgroup each: G groups of 256 lanes have a chunk of every rank.
// Bases: output, rank 0, 1 ...  The operations and their order are those of the launches it stands for, four of
// them for eight ranks, each of which costs the stream 4 to 5 us however little it does.  Bound by the chain of one
// workgroup: a level's sums, two trips through LDS and a divide, 1 us, and what a compute unit takes to load the ranks.
// fp32, us: 8 ranks of 10 rows of 1,000 elements 15.7 -> 6.6, of 44 rows of one chunk 19.6 -> 9.7, of two 20.2 -> 13.4,
// 2 ranks of 44 rows of two chunks 7.8 -> 4.4.  The lines: 8 ranks of two chunks are 182 registers at 512 lanes, and one
// row of them takes as long in fp16 (16.7) as level by level; with a narrower type on the wire the levels' lanes have
// other elements than the ranks', and a row's bits would depend on whether a longer row is beside it.
template <typename W, int WORLD, int G>
__global__ __launch_bounds__(G * kWG) void tree_held_k(Level l, ShortRows rows) {
  constexpr int VEC = HeldRanks<W, WORLD>::VEC, kVecs = HeldRanks<W, WORLD>::kVecs;
  const typename Factor<W>::type fin = (typename Factor<W>::type)l.pre, fout = (typename Factor<W>::type)l.post;
  const uint32_t group = threadIdx.x / kWG;
  Place p;
  p.row = blockIdx.x;
  p.d = rows.d + p.row * l.words;
  p.high = l.high;
  p.elements = row_elements(p.d);
  p.start = group * kChunk<W>;
  const uint32_t left = p.start < p.elements ? (uint32_t)(p.elements - p.start) : 0;
  p.m = left < kChunk<W> ? left : kChunk<W>;
  HeldRanks<W, WORLD> h;
  h.load(rows, p, threadIdx.x % kWG, fin, l.flags & kScaleIn);
  __shared__ double red[(WORLD == 8 ? 3 : WORLD == 4 ? 2 : 1) * G][WORLD / 2][3][kWG / 64];
  held_levels<WORLD / 2, W, WORLD, G>(h, group, l.guard, red);
  const bool scale_out = l.flags & kScaleOut;
  const gptr<W> to = p.at<W>(rows, 0) + p.start;
  const Window out = store_window<kStoreNT>(to, h.m * (uint32_t)sizeof(W));
#pragma unroll
  for (int u = 0; u < kVecs; ++u)
    if (h.lane + u * kWG < h.nv)
      stw<kStoreNT, W, VEC>(out, (h.lane + u * kWG) * 16u, from_wire<W, W, VEC>(h.pinned(h.x[0][u]), fout, scale_out));
  if (h.has_tail()) to[h.nv * VEC + h.lane] = from_wire<W, W, 1>(Arr<W, 1>{h.t[0]}, fout, scale_out).v[0];
}

// ---- host side ---------------------------------------------------------------------------------

uint64_t up256(uint64_t bytes) { return (bytes + 255) / 256 * 256; }

// Consecutive entries that go through the tree together: as many as a launch's arguments hold.
struct Group {
  int begin, end;             // entries, empty ones among them
  uint32_t nrows, chunks, max_row_chunks;
  uint64_t vector_bytes;      // of the wire type, every row padded to 256 bytes
  // workspace: vectors of the first level, then the sums of the levels in turn, then coefficients
  uint64_t sums_at[2], coeffs_at, bytes;
};

int next_group(const int64_t* counts, int n, int begin, uint32_t world, uint32_t wire_size, Group* out) {
  const uint32_t max_rows = std::min(kMaxShortRows, kShortWords / (kRowHead + std::min(world, kRanksAtOnce)));
  const uint64_t chunk = kChunkBytes / wire_size;
  const uint64_t max_chunks = kMaxWorkgroups / std::max(1u, world / 2);
  Group g = {begin, begin, 0, 0, 0, 0, {0, 0}, 0, 0};
  for (; g.end < n && g.nrows < max_rows; ++g.end) {
    const uint64_t count = (uint64_t)counts[g.end], c = (count + chunk - 1) / chunk;
    if (c == 0) continue;
    if (g.nrows && g.chunks + c > max_chunks) break;
    if (c > max_chunks) return fail(HVDHIP_ERR_TOO_LARGE, "entry %d needs more than 2^23 workgroups", g.end);
    ++g.nrows;
    g.chunks += (uint32_t)c;
    g.max_row_chunks = std::max(g.max_row_chunks, (uint32_t)c);
    g.vector_bytes += up256(count * wire_size);
  }
  const uint64_t triples = 3 * sizeof(double) * (uint64_t)g.chunks;
  g.sums_at[0] = world >= 4 ? world / 2 * g.vector_bytes : 0;
  g.sums_at[1] = g.sums_at[0] + up256(world / 2 * triples);
  g.coeffs_at = g.sums_at[1] + up256(world / 4 * triples);
  g.bytes = g.coeffs_at + up256(g.max_row_chunks > kReaddMax ? world / 2 * (uint64_t)kMaxShortRows * 2 * sizeof(double) : 0);
  *out = g;
  return 0;
}

int workspace_bytes(const int64_t* counts, int n, uint32_t world, uint32_t wire_size, uint64_t* bytes) {
  *bytes = 0;
  for (int at = 0; at < n;) {
    Group g;
    const int rc = next_group(counts, n, at, world, wire_size, &g);
    if (rc) return rc;
    *bytes = std::max(*bytes, g.bytes);
    at = g.end;
  }
  return 0;
}

template <typename S, typename W, typename D>
class Tree {
 public:
  Tree(const RanksCall& c, unsigned char* ws) : c_(c), ws_(ws) {}

  int run() {
    int last = c_.n;  // the completion event goes out with the last launch, so it has to be known
    while (last > 0 && c_.counts[last - 1] == 0) --last;
    if (last == 0) {
      if (c_.completion) HVDHIP_CHECK(hipEventRecord(c_.completion, c_.stream));
      return 0;
    }
    for (int at = 0; at < last;) {
      Group whole;  // what the workspace was sized for
      int rc = next_group(c_.counts, last, at, c_.world, sizeof(W), &whole);
      if (rc) return rc;
      for (; at < whole.end; at = g_.end) {
        rc = next_group(c_.counts, within_reach(at, whole.end, &wide_), at, c_.world, sizeof(W), &g_);
        if (rc) return rc;
        rc = group(g_.end == last ? c_.completion : nullptr);
        if (rc) return rc;
      }
    }
    return 0;
  }

 private:
  int group(hipEvent_t completion) {
    l_ = Level{};
    l_.nrows = g_.nrows;
    l_.chunks = g_.chunks;
    l_.flags = c_.flags;
    l_.pre = c_.pre;
    l_.post = c_.post;
    l_.guard = std::sqrt(DBL_MIN);
    const uint32_t world = c_.world, at_once = std::min(world, kRanksAtOnce);
    double* sums[2] = {reinterpret_cast<double*>(ws_ + g_.sums_at[0]), reinterpret_cast<double*>(ws_ + g_.sums_at[1])};
    if constexpr (std::is_same<S, W>::value && std::is_same<W, D>::value) {
      if (g_.max_row_chunks <= 2 && world <= kRanksAtOnce) {
        fill(0, world, true);
        const bool one = g_.max_row_chunks == 1;
        const hipError_t status = world == 2   ? (one ? held<2, 1>(completion) : held<2, 2>(completion))
                                  : world == 4 ? (one ? held<4, 1>(completion) : held<4, 2>(completion))
                                               : (one ? held<8, 1>(completion) : held<8, 2>(completion));
        HVDHIP_CHECK_LAUNCH("tree_held_k", status);
        return 0;
      }
    }
    // the ranks' sums, pairwise
    l_.out_sums = sums[0];
    for (uint32_t r = 0; r < world; r += at_once) {
      fill(r, at_once, world == 2);
      l_.first = r / 2;
      const uint64_t bytes = (uint64_t)world * g_.vector_bytes * sizeof(S) / sizeof(W);
      const dim3 grid(columns(), at_once / 2);
      const hipError_t status = bytes <= kKeepBytes ? launch(dots_k<S, W, 2>, grid, c_.stream, l_, rows_)
                                                    : launch(dots_k<S, W, 1>, grid, c_.stream, l_, rows_);
      HVDHIP_CHECK_LAUNCH("dots_k", status);
    }
    int rc = level_done(sums, 0, world / 2);
    if (rc) return rc;
    if (world == 2) {
      HVDHIP_CHECK_LAUNCH("last_k", launch_with(completion, last_k<S, W, D, true>, dim3(columns()), c_.stream, l_, rows_));
      return 0;
    }
    l_.out_stride = g_.vector_bytes;
    for (uint32_t r = 0; r < world; r += at_once) {
      if (world > at_once) fill(r, at_once, false);
      l_.first = r / 4;
      HVDHIP_CHECK_LAUNCH("level_k", launch(level_k<S, W, true>, dim3(columns(), at_once / 4), c_.stream, l_, rows_));
    }
    int side = 1;
    rc = level_done(sums, side, world / 4);
    if (rc) return rc;
    l_.first = 0;
    for (uint32_t vectors = world / 2; vectors > 2; vectors /= 2) {
      fill(0, 0, false);
      l_.in_stride = l_.out_stride;
      l_.out_stride = 2 * l_.in_stride;
      HVDHIP_CHECK_LAUNCH("level_k", launch(level_k<W, W, false>, dim3(columns(), vectors / 4), c_.stream, l_, rows_));
      side ^= 1;
      rc = level_done(sums, side, vectors / 4);
      if (rc) return rc;
    }
    l_.in_stride = l_.out_stride;
    fill(0, 0, true);
    HVDHIP_CHECK_LAUNCH("last_k", launch_with(completion, last_k<W, W, D, false>, dim3(columns()), c_.stream, l_, rows_));
    return 0;
  }

  template <int WORLD, int G>
  hipError_t held(hipEvent_t completion) const {
    return launch_shaped(completion, tree_held_k<W, WORLD, G>, dim3(g_.nrows), G * kWG, c_.stream, l_, rows_);
  }

  // Workgroups along a launch's chunks: a multiple of the XCDs, so that a chunk is on the same one for every pair and in
  // every level and finds there what the level before left in its L2 (the ranks, where they fit).  Against as many as
  // there are chunks: 8 ranks of 1 million fp32 31.2 -> 28.7 us, 4 of 2 million 24.3 -> 22.5, 8 of 1 million fp64
  // 45.5 -> 42.7; 8 of 5 million and the BERT-large layer the same.
  uint32_t columns() const { return (g_.chunks + kXcds - 1) / kXcds * kXcds; }

  // The sums that were just left on one side are the next launch's input.
  int level_done(double* const* sums, int side, uint32_t pairs) {
    l_.in_sums = sums[side];
    l_.out_sums = sums[side ^ 1];
    if (g_.max_row_chunks <= kReaddMax) return 0;
    RowStarts starts;
    std::copy(rows_.first, rows_.first + g_.nrows, starts.first);
    starts.first[g_.nrows] = g_.chunks;
    double* coeffs = reinterpret_cast<double*>(ws_ + g_.coeffs_at);
    l_.coeffs = coeffs;
    HVDHIP_CHECK_LAUNCH("coeffs_k", launch(coeffs_k, dim3(g_.nrows, pairs), c_.stream, l_.in_sums, coeffs, l_.chunks,
                                           l_.guard, starts));
    return 0;
  }

  // The end of the entries from `begin` on, at most `end`, that a group of short or of wide distances reaches, whichever
  // is further; of the wide ones fewer fit a launch's arguments.
  int within_reach(int begin, int end, bool* wide) const {
    const int narrow = within(begin, end, kShortReach);
    *wide = false;
    if (narrow == end) return end;
    const uint32_t bases = 1 + std::min(c_.world, kRanksAtOnce);
    uint32_t room = std::min(kMaxShortRows, kShortWords / (kRowHead - 1 + bases + wide_words(bases)));
    int most = begin;
    for (; most < end; ++most)
      if (c_.counts[most] && room-- == 0) break;
    const int far = within(begin, most, kWideReach);
    *wide = far > narrow;
    return std::max(far, narrow);
  }
  int within(int begin, int end, uint64_t most) const {
    auto reach = [&](auto&& address, uint64_t unit) {  // of one base, and never short of the first entry with elements
      uint64_t lo = ~0ull, hi = 0;
      for (int e = begin; e < end; ++e) {
        if (c_.counts[e] == 0) continue;
        const uint64_t at = address(e);
        lo = std::min(lo, at);
        hi = std::max(hi, at);
        if ((hi - lo) / unit > most) end = e;
      }
    };
    reach([&](int e) { return (uint64_t)(uintptr_t)c_.outputs[e]; }, sizeof(D));
    for (uint32_t r = 0; r < c_.world; ++r)
      reach([&](int e) { return (uint64_t)(uintptr_t)c_.inputs[(size_t)r * (size_t)c_.n + (size_t)e]; }, sizeof(S));
    uint64_t next = 0;
    reach([&](int e) { const uint64_t at = next; next += up256((uint64_t)c_.counts[e] * sizeof(W)); return at; }, sizeof(W));
    return end;
  }

  // Rows from the bases workspace or output and the tensors of `ranks` ranks from `first` on, or without ranks
  // workspace alone and output and workspace.
  void fill(uint32_t first, uint32_t ranks, bool to_output) {
    const bool work_too = to_output && ranks == 0;
    const uint32_t bases = 1 + (work_too ? 1 : ranks);
    const uint64_t work = (uint64_t)(uintptr_t)ws_;
    uint64_t at[kMaxShortRows][1 + kRanksAtOnce];
    uint64_t* base = rows_.base;
    std::fill(base, base + bases, ~0ull);
    l_.high = kRowHead - 1 + bases;
    l_.words = l_.high + (wide_ ? wide_words(bases) : 0);
    rows_.wide = wide_ ? 0xff : 0;
    uint32_t row = 0, chunks = 0;
    uint64_t offset = 0;
    for (int e = g_.begin; e < g_.end; ++e) {
      const uint64_t count = (uint64_t)c_.counts[e];
      if (count == 0) continue;
      at[row][0] = to_output ? (uint64_t)(uintptr_t)c_.outputs[e] : work + offset;
      if (work_too) at[row][1] = work + offset;
      for (uint32_t r = 0; r < ranks; ++r)
        at[row][1 + r] = (uint64_t)(uintptr_t)c_.inputs[(size_t)(first + r) * (size_t)c_.n + (size_t)e];
      for (uint32_t k = 0; k < bases; ++k) base[k] = std::min(base[k], at[row][k]);
      uint32_t* d = rows_.d + row * l_.words;
      d[1] = (uint32_t)count;
      d[2] = (uint32_t)(count >> 32);
      rows_.first[row++] = chunks;
      chunks += (uint32_t)((count + kChunk<W> - 1) / kChunk<W>);
      offset += up256(count * sizeof(W));
    }
    for (uint32_t i = 0; i < row; ++i) {
      uint32_t* d = rows_.d + i * l_.words;
      std::fill(d + l_.high, d + l_.words, 0u);
      set_distance(d, 0, l_.high, 0, (at[i][0] - base[0]) / (to_output ? sizeof(D) : sizeof(W)), wide_);
      for (uint32_t k = 1; k < bases; ++k)
        set_distance(d, kRowHead - 1 + k, l_.high, k, (at[i][k] - base[k]) / (work_too ? sizeof(W) : sizeof(S)), wide_);
    }
    for (; row < kMaxShortRows; ++row) rows_.first[row] = ~0u;
  }

  // Largest total of the ranks' tensors that the first pass leaves in the Infinity Cache whole: keeping all, half or
  // none of 2 x 50 MB takes 40.6 / 40.6 / 44.2 us and of 8 x 12 MB 70.5 / 70.6 / 71.9, but of 8 x 50 MB, which
  // do not fit, 229.5 / 223.6 / 226.5.
  static constexpr uint64_t kKeepBytes = (uint64_t)160 << 20;

  const RanksCall& c_;
  unsigned char* ws_;
  Group g_;
  Level l_;
  bool wide_;  // the group's distances take more than 32 bits
  ShortRows rows_;
};

template <typename S, typename W, typename D>
int run(const RanksCall& c, void* workspace) {
  return Tree<S, W, D>(c, static_cast<unsigned char*>(workspace)).run();
}

int check_world_and_type(int world, int wire_dtype) {
  if (world < 2 || (world & (world - 1)) || world > HVDHIP_ADASUM_RANKS_MAX_WORLD)
    return fail(HVDHIP_ERR_INVALID_ARGUMENT, "world = %d is not a power of two from 2 to %d", world,
                HVDHIP_ADASUM_RANKS_MAX_WORLD);
  if (wire_dtype != HVDHIP_FLOAT16 && wire_dtype != HVDHIP_FLOAT32 && wire_dtype != HVDHIP_FLOAT64)
    return fail(HVDHIP_ERR_UNSUPPORTED_DTYPE, "Adasum supports FLOAT16, FLOAT32 and FLOAT64, not dtype %d", wire_dtype);
  return 0;
}

}  // namespace
}  // namespace hvdhip

using namespace hvdhip;

extern "C" int64_t hvdhip_adasum_ranks_workspace(const int64_t* num_elements, int n, int world, int wire_dtype) {
  int rc = check_world_and_type(world, wire_dtype);
  if (rc) return rc;
  if (n < 0 || (n > 0 && !num_elements)) return fail(HVDHIP_ERR_INVALID_ARGUMENT, "bad entry arrays");
  for (int i = 0; i < n; ++i)
    if (num_elements[i] < 0) return fail(HVDHIP_ERR_INVALID_ARGUMENT, "entry %d has a negative size", i);
  uint64_t bytes = 0;
  rc = workspace_bytes(num_elements, n, (uint32_t)world, (uint32_t)dtype_size(wire_dtype), &bytes);
  return rc ? rc : (int64_t)bytes;
}

extern "C" int hvdhip_adasum_ranks(void* const* outputs, const void* const* inputs, const int64_t* num_elements, int n,
                                   int world, int in_dtype, int wire_dtype, int out_dtype, double prescale,
                                   double postscale, void* workspace, int64_t workspace_bytes, void* stream,
                                   void* event) {
  int rc = check_world_and_type(world, wire_dtype);
  if (rc) return rc;
  RanksCall c = {outputs, inputs, num_elements, n, (uint32_t)world, prescale, postscale, 0,
                 static_cast<hipStream_t>(stream), static_cast<hipEvent_t>(event)};
  rc = check_ranks_call(&c, in_dtype, wire_dtype, out_dtype);
  if (rc) return rc;
  const int64_t need = hvdhip_adasum_ranks_workspace(num_elements, n, world, wire_dtype);
  if (need < 0) return (int)need;
  if (need > 0 && (!workspace || (uintptr_t)workspace % 256 || workspace_bytes < need))
    return fail(HVDHIP_ERR_INVALID_ARGUMENT, "the workspace is not %lld bytes on a 256-byte boundary", (long long)need);
  switch (wire_dtype) {
  case HVDHIP_FLOAT32: rc = run<float, float, float>(c, workspace); break;
  case HVDHIP_FLOAT64: rc = run<double, double, double>(c, workspace); break;
  default:
    rc = in_dtype == HVDHIP_FLOAT32 ? (out_dtype == HVDHIP_FLOAT32 ? run<float, half_t, float>(c, workspace)
                                                                   : run<float, half_t, half_t>(c, workspace))
                                    : (out_dtype == HVDHIP_FLOAT32 ? run<half_t, half_t, float>(c, workspace)
                                                                   : run<half_t, half_t, half_t>(c, workspace));
  }
  return rc ? rc : ok();
}
