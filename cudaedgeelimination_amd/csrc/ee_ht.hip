// Hamilton-Tutte reply enumerations on the resident CSR: the Hamilton
// replies (pairs of a center's neighbours that survive the target edge's
// 2-opt and cost tests) and the end replies (a path end's active edges but
// the path-internal one), in the reference's deterministic order.
//
// Reference: CountHtRepliesKernel / WriteHtRepliesKernel /
// CountEndRepliesKernel / WriteEndRepliesKernel and their host drivers
// (src/cuda/ht_replies.cu:406-520, 585-752); CPU semantics
// AppendHtHamiltonRepliesUnchecked / AppendHtEndRepliesUnchecked
// (src/cpu/hamilton_tutte.cpp:230-277) with EdgesSurviveTwoOpt (:79-87).
//
// One wavefront per center.  Its lanes first compute, once per neighbour,
// the center edge's exact distance and its 2-opt verdict into LDS (the
// reference recomputes both per pair); then each lane takes one neighbour
// pair (pairs numbered in the reference's first-major order), and a ballot
// plus a popcount prefix place the surviving pairs in order.
//
// Two forms of the output.  Where the centers' rows are short (PlanVerdicts),
// one pass writes each pair's verdict as a bit into host memory, and the host
// writes the replies from the bits into the caller's buffer: a reply is its
// center and two neighbours, 12 bytes that the host has, against one bit.
// Otherwise a count pass, an offset scan and a write pass leave the replies
// on the device, which then never holds more than the replies themselves.
#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstring>
#include <stdexcept>
#include <type_traits>
#include <vector>

#include "ee_exact.h"
#include "ee_jvhost.h"
#include "ee_runtime.h"

namespace ee {
namespace {

constexpr uint32_t kHtBlock = 256;
constexpr uint32_t kHtWaves = kHtBlock / 64;
constexpr uint32_t kHtLdsNeighbors = 64;  // per wave; larger rows recompute per pair

struct HtNeighbor {
  int64_t center_cost;
  int32_t node;
  int32_t survives;
};

// kNear: both coordinate extents of the snapshot are below 2^25, so the
// differences fit int32 and the FP64 root with one exact remainder applies
// (ExactDistanceNear); otherwise the 64-bit integer path.
template <bool kNear>
__device__ inline int64_t Dist(const longlong2* xy, int32_t a, int32_t b, int type) {
  const longlong2 p = xy[a], q = xy[b];
  if constexpr (kNear) {
    return ExactDistanceNear(static_cast<int32_t>(p.x - q.x), static_cast<int32_t>(p.y - q.y), type);
  } else {
    return ExactDistance(p.x, p.y, q.x, q.y, type);
  }
}

// EdgesSurviveTwoOpt for the edge (a, b) against the target (tu, tv): at
// least one 2-opt orientation is not a strict improvement.  Distances of a
// distance-safe snapshot are below 2^32, so the 64-bit sums are exact.
template <bool kNear>
__device__ inline bool Survives(const longlong2* xy, int32_t tu, int32_t tv, int64_t target_cost,
                                int32_t a, int32_t b, int64_t ab, int type) {
  const int32_t lo = min(a, b), hi = max(a, b);
  const int64_t original = target_cost + ab;
  const int64_t first = Dist<kNear>(xy, tu, hi, type) + Dist<kNear>(xy, tv, lo, type);
  const int64_t second = Dist<kNear>(xy, tu, lo, type) + Dist<kNear>(xy, tv, hi, type);
  return first >= original || second >= original;
}

// First index of row i of the pairs (i, j > i) of d items, first-major.
__device__ inline uint64_t PairRowStart(uint64_t i, uint64_t d) { return i * (2 * d - i - 1) / 2; }

// Centers per scan chunk: one workgroup sums each chunk's reply counts, and
// the scan pass gives each chunk to one workgroup.
constexpr uint32_t kScanThreads = 256;
constexpr uint32_t kScanPerThread = 4;
constexpr uint32_t kScanChunk = kScanThreads * kScanPerThread;

template <bool kWrite, bool kNear>
__global__ __launch_bounds__(kHtBlock) void HtHamiltonKernel(
    const longlong2* __restrict__ xy, const int32_t* __restrict__ row_offsets,
    const int32_t* __restrict__ neighbors, int type, int32_t tu, int32_t tv,
    const int32_t* __restrict__ centers, uint64_t center_count, uint64_t* __restrict__ counts,
    const uint64_t* __restrict__ offsets, int32_t* __restrict__ replies) {
  __shared__ HtNeighbor cache[kHtWaves][kHtLdsNeighbors];
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  const uint64_t item = static_cast<uint64_t>(blockIdx.x) * kHtWaves + wave;
  if (item >= center_count) return;  // whole wavefronts leave together
  const int32_t c = centers[item];
  const int32_t begin = row_offsets[c];
  const uint64_t d = static_cast<uint64_t>(row_offsets[c + 1] - begin);
  const int64_t target_cost = Dist<kNear>(xy, tu, tv, type);
  const int64_t center_target = Dist<kNear>(xy, tu, c, type) + Dist<kNear>(xy, tv, c, type);
  const bool cached = d <= kHtLdsNeighbors;
  HtNeighbor* mine = cache[wave];
  if (cached && lane < d) {
    const int32_t nb = neighbors[begin + lane];
    const int64_t cost = Dist<kNear>(xy, c, nb, type);
    mine[lane] = {cost, nb, Survives<kNear>(xy, tu, tv, target_cost, c, nb, cost, type) ? 1 : 0};
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  const uint64_t pairs = d < 2 ? 0 : d * (d - 1) / 2;
  uint64_t out = kWrite ? offsets[item] : 0;
  const uint64_t out_end = kWrite ? offsets[item + 1] : 0;
  uint64_t found = 0;
  for (uint64_t base = 0; base < pairs; base += 64) {
    const uint64_t p = base + lane;
    bool keep = false;
    if (p < pairs) {
      // row i of pair p: the root estimate, then exact corrections
      const double b = static_cast<double>(2 * d - 1);
      uint64_t i = static_cast<uint64_t>(fmax(0.0, floor((b - sqrt(b * b - 8.0 * static_cast<double>(p))) / 2)));
      if (i > d - 2) i = d - 2;
      while (i > 0 && PairRowStart(i, d) > p) --i;
      while (i + 1 <= d - 2 && PairRowStart(i + 1, d) <= p) ++i;
      const uint64_t j = p - PairRowStart(i, d) + i + 1;
      HtNeighbor f, s;
      if (cached) {
        f = mine[i];
        s = mine[j];
      } else {
        f.node = neighbors[begin + i];
        s.node = neighbors[begin + j];
        f.center_cost = Dist<kNear>(xy, c, f.node, type);
        s.center_cost = Dist<kNear>(xy, c, s.node, type);
        f.survives = Survives<kNear>(xy, tu, tv, target_cost, c, f.node, f.center_cost, type);
        s.survives = Survives<kNear>(xy, tu, tv, target_cost, c, s.node, s.center_cost, type);
      }
      const bool is_target = min(f.node, s.node) == tu && max(f.node, s.node) == tv;
      if (!is_target && f.survives && s.survives) {
        const int64_t original = target_cost + f.center_cost + s.center_cost;
        const int64_t replacement = Dist<kNear>(xy, f.node, s.node, type) + center_target;
        keep = original <= replacement;
      }
      if (kWrite && keep) {
        const uint64_t ballot_below = __ballot(keep) & ((uint64_t{1} << lane) - 1);
        const uint64_t at = out + __popcll(ballot_below);
        if (at < out_end) {  // the count pass found exactly out_end - offsets[item]
          int32_t* r = replies + 3 * at;
          r[0] = c;
          r[1] = f.node;
          r[2] = s.node;
        }
      }
    }
    const uint64_t ballot = __ballot(keep);
    found += __popcll(ballot);
    if (kWrite) out += __popcll(ballot);
  }
  if (!kWrite && lane == 0) counts[item] = found;
}

// Words of verdict bits of a row of d neighbours.
__host__ __device__ inline uint32_t VerdictWords(uint32_t d) { return d < 2 ? 0 : (d * (d - 1) / 2 + 63) / 64; }

// A neighbour of the center under test: what the pair test needs of it.  x
// and y are the low words on near snapshots (differences stay exact).
template <bool kNear> struct HtRow {
  int64_t cost;
  typename std::conditional<kNear, uint32_t, int64_t>::type x, y;
  int32_t node;
  int32_t survives;
};

template <bool kNear>
__device__ inline int64_t RowDist(const HtRow<kNear>& a, const HtRow<kNear>& b, int type) {
  if constexpr (kNear) {
    return ExactDistanceNear(static_cast<int32_t>(a.x - b.x), static_cast<int32_t>(a.y - b.y), type);
  } else {
    return ExactDistance(a.x, a.y, b.x, b.y, type);
  }
}

// Neighbours per center in a wavefront's first phase.
constexpr uint32_t kVerdictGroup = 16;

// Verdict bits of each center's pairs, in words of their own, and their
// counts.  With a stride every center has that many words (zero past its
// pairs); otherwise VerdictWords of its row, and first_words[w] is the first
// of wavefront w's.  A wavefront takes kCenters consecutive centers, so its
// reads of centers and writes of words and counts are whole stretches of
// host memory.  Of 4, the centers gather their neighbours on 16 lanes each
// (rows of up to 16, the usual case; otherwise they take the wavefront one by
// one), then each center's pairs take the 64 lanes, out of LDS.  Bound by
// those gathers and the pair arithmetic: 41 us for the 30,000-node graph's
// 1.56 million pairs.  One center per wavefront, reading its id and writing
// its words over PCIe by itself, took 64 us there; 8 and 16 centers 41 and 50
// us, and 7 and 19 us more where few centers leave the chip to single
// wavefronts.  Rows beyond the LDS cache recompute both neighbours per pair
// and end the launch, so wherever there is one a wavefront takes one center.
template <bool kNear, uint32_t kCenters>
__global__ __launch_bounds__(kHtBlock) void HtVerdictKernel(
    const longlong2* __restrict__ xy, const int32_t* __restrict__ row_offsets,
    const int32_t* __restrict__ neighbors, int32_t nodes, int type, int32_t tu, int32_t tv,
    const int32_t* __restrict__ centers, uint32_t center_count, uint32_t stride,
    const uint32_t* __restrict__ first_words, uint64_t* __restrict__ bits, uint32_t* __restrict__ counts) {
  __shared__ HtRow<kNear> rows[kHtWaves][kHtLdsNeighbors];
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  const uint32_t number = blockIdx.x * kHtWaves + wave;
  const uint32_t first = number * kCenters;
  if (first >= center_count) return;  // whole wavefronts leave together
  const uint32_t here = min(kCenters, center_count - first);
  HtRow<kNear>* const mine = rows[wave];
  const int64_t target_cost = Dist<kNear>(xy, tu, tv, type);
  // lane i < here: center i of the wavefront, its row (empty for an id out of
  // range: the host refuses the call) and its distance to the target's ends
  int32_t my_center = 0, my_begin = 0, my_degree = 0;
  int64_t my_target = 0;
  if (lane < here) {
    const int32_t c = centers[first + lane];
    if (static_cast<uint32_t>(c) < static_cast<uint32_t>(nodes)) {
      my_center = c;
      my_begin = row_offsets[c];
      my_degree = row_offsets[c + 1] - my_begin;
      my_target = Dist<kNear>(xy, tu, c, type) + Dist<kNear>(xy, tv, c, type);
    }
  }
  const auto neighbor = [&](int32_t c, int32_t begin, uint32_t i) {
    HtRow<kNear> r;
    r.node = neighbors[begin + static_cast<int32_t>(i)];
    const longlong2 p = xy[r.node];
    r.x = static_cast<decltype(r.x)>(p.x);
    r.y = static_cast<decltype(r.y)>(p.y);
    r.cost = Dist<kNear>(xy, c, r.node, type);
    r.survives = Survives<kNear>(xy, tu, tv, target_cost, c, r.node, r.cost, type) ? 1 : 0;
    return r;
  };
  const auto lds = [] {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  uint64_t word = 0;       // lane l: word l of the stretch being filled
  uint32_t at = 0;         // words of the wavefront so far
  uint32_t my_count = 0;   // lane i: surviving pairs of center i
  uint64_t* const out = bits + (stride != 0 ? static_cast<uint64_t>(first) * stride : first_words[number]);
  const uint32_t q = lane / kVerdictGroup;
  const int32_t q_degree = __shfl(my_degree, static_cast<int>(q));
  const bool together = __ballot(q_degree > static_cast<int32_t>(kVerdictGroup)) == 0;
  if (together) {
    const int32_t c = __shfl(my_center, static_cast<int>(q)), begin = __shfl(my_begin, static_cast<int>(q));
    const uint32_t i = lane % kVerdictGroup;
    if (static_cast<int32_t>(i) < q_degree) mine[lane] = neighbor(c, begin, i);
    lds();
  }
  for (uint32_t k = 0; k < here; ++k) {  // uniform
    const int32_t c = __builtin_amdgcn_readlane(my_center, static_cast<int>(k));
    const int32_t begin = __builtin_amdgcn_readlane(my_begin, static_cast<int>(k));
    const uint32_t d = static_cast<uint32_t>(__builtin_amdgcn_readlane(my_degree, static_cast<int>(k)));
    const int64_t center_target = __shfl(static_cast<long long>(my_target), static_cast<int>(k));
    const bool cached = d <= kHtLdsNeighbors;
    const HtRow<kNear>* row = mine + (together ? k * kVerdictGroup : 0);
    if (!together) {
      if (cached && lane < d) mine[lane] = neighbor(c, begin, lane);
      lds();
    }
    const uint32_t pairs = d < 2 ? 0 : d * (d - 1) / 2;
    uint32_t found = 0;
    const uint32_t words = stride != 0 ? stride : VerdictWords(d);
    for (uint32_t w = 0; w < words; ++w) {
      const uint32_t p = w * 64 + lane;
      bool keep = false;
      if (p < pairs) {
        // row i of pair p: the root estimate (its argument is exact in
        // float), then exact corrections
        const float b = static_cast<float>(2 * d - 1);
        uint32_t i = static_cast<uint32_t>(fmaxf(0.0f, (b - sqrtf(b * b - 8.0f * static_cast<float>(p))) * 0.5f));
        if (i > d - 2) i = d - 2;
        while (i > 0 && i * (2 * d - i - 1) / 2 > p) --i;
        while (i + 1 <= d - 2 && (i + 1) * (2 * d - i - 2) / 2 <= p) ++i;
        const uint32_t j = p - i * (2 * d - i - 1) / 2 + i + 1;
        const HtRow<kNear> f = cached ? row[i] : neighbor(c, begin, i);
        const HtRow<kNear> s = cached ? row[j] : neighbor(c, begin, j);
        const bool is_target = min(f.node, s.node) == tu && max(f.node, s.node) == tv;
        if (!is_target && f.survives && s.survives) {
          const int64_t original = target_cost + f.cost + s.cost;
          const int64_t replacement = RowDist<kNear>(f, s, type) + center_target;
          keep = original <= replacement;
        }
      }
      const uint64_t ballot = __ballot(keep);
      found += static_cast<uint32_t>(__popcll(ballot));
      if (lane == (at & 63u)) word = ballot;
      ++at;
      if ((at & 63u) == 0) out[at - 64 + lane] = word;  // uniform
    }
    if (lane == k) my_count = found;
    if (!together) lds();  // the row is read before the next one replaces it
  }
  if (lane < (at & 63u)) out[(at & ~63u) + lane] = word;
  if (lane < here) counts[first + lane] = my_count;
}

// chunk_sums[c] = counts of chunk c (kScanChunk centers), one workgroup per
// chunk: plain stores, no atomics shared by the chunk's centers.
__global__ __launch_bounds__(kScanThreads) void HtChunkSumKernel(const uint64_t* __restrict__ counts, uint64_t n,
                                                                  unsigned long long* __restrict__ chunk_sums) {
  __shared__ unsigned long long wave_sums[kScanThreads / 64];
  const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6;
  const uint64_t first = static_cast<uint64_t>(blockIdx.x) * kScanChunk + static_cast<uint64_t>(t) * kScanPerThread;
  unsigned long long own = 0;
#pragma unroll
  for (uint32_t e = 0; e < kScanPerThread; ++e) own += first + e < n ? counts[first + e] : 0;
  for (uint32_t d = 32; d >= 1; d >>= 1) own += __shfl_xor(own, d, 64);
  if (lane == 0) wave_sums[wave] = own;
  __syncthreads();
  if (t == 0) {
    unsigned long long total = 0;
    for (uint32_t w = 0; w < kScanThreads / 64; ++w) total += wave_sums[w];
    chunk_sums[blockIdx.x] = total;
  }
}

// offsets[0] = 0, offsets[i + 1] = counts[0] + ... + counts[i], one
// workgroup per chunk of kScanChunk counts: the workgroup first sums the
// totals of the chunks before its own (chunk_sums, from HtChunkSumKernel),
// then scans its chunk, each thread holding 4 consecutive counts
// (wavefront shuffles, then the 4 wavefront totals in LDS).
__global__ __launch_bounds__(kScanThreads) void HtScanKernel(const uint64_t* __restrict__ counts,
                                                              uint64_t n,
                                                              const unsigned long long* __restrict__ chunk_sums,
                                                              uint64_t* __restrict__ offsets) {
  __shared__ unsigned long long partial[kScanThreads / 64];
  __shared__ unsigned long long wave_sums[kScanThreads / 64];
  const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6;
  const uint64_t chunk = blockIdx.x;
  // prefix of the chunks before this one
  unsigned long long before = 0;
  for (uint64_t c = t; c < chunk; c += kScanThreads) before += chunk_sums[c];
  for (uint32_t d = 32; d >= 1; d >>= 1) before += __shfl_xor(before, d, 64);
  if (lane == 0) partial[wave] = before;
  const uint64_t first = chunk * kScanChunk + static_cast<uint64_t>(t) * kScanPerThread;
  unsigned long long v[kScanPerThread];
  unsigned long long own = 0;
#pragma unroll
  for (uint32_t e = 0; e < kScanPerThread; ++e) {
    v[e] = first + e < n ? counts[first + e] : 0;
    own += v[e];
  }
  unsigned long long inc = own;  // inclusive scan of the threads' sums in the wavefront
  for (uint32_t d = 1; d < 64; d <<= 1) {
    const unsigned long long o = __shfl_up(inc, d, 64);
    if (lane >= d) inc += o;
  }
  if (lane == 63) wave_sums[wave] = inc;
  __syncthreads();
  unsigned long long run = inc - own;
  for (uint32_t w = 0; w < kScanThreads / 64; ++w) {
    run += partial[w];
    if (w < wave) run += wave_sums[w];
  }
  if (chunk == 0 && t == 0) offsets[0] = 0;
#pragma unroll
  for (uint32_t e = 0; e < kScanPerThread; ++e) {
    run += v[e];
    if (first + e < n) offsets[first + e + 1] = run;
  }
}

// End replies: one thread per task writes the endpoint's active edges but
// the internal one, canonical (u < v), from its precomputed offset.
__global__ __launch_bounds__(kHtBlock) void HtEndKernel(const int32_t* __restrict__ row_offsets,
                                                         const int32_t* __restrict__ neighbors,
                                                         const int32_t* __restrict__ tasks,
                                                         uint64_t task_count,
                                                         const uint64_t* __restrict__ offsets,
                                                         int32_t* __restrict__ replies) {
  const uint64_t i = static_cast<uint64_t>(blockIdx.x) * kHtBlock + threadIdx.x;
  if (i >= task_count) return;
  const int32_t e = tasks[2 * i], internal = tasks[2 * i + 1];
  uint64_t out = offsets[i];
  const uint64_t end = offsets[i + 1];
  for (int32_t a = row_offsets[e]; a < row_offsets[e + 1] && out < end; ++a) {
    const int32_t nb = neighbors[a];
    if (nb == internal) continue;
    replies[2 * out] = min(e, nb);
    replies[2 * out + 1] = max(e, nb);
    ++out;
  }
}

bool RowHas(const ee_graph_view& g, int32_t a, int32_t b) {
  const int32_t* lo = g.neighbors + g.row_offsets[a];
  const int32_t* hi = g.neighbors + g.row_offsets[a + 1];
  return std::binary_search(lo, hi, b);
}

// ValidateGraphShape (src/cuda/ht_replies.cu:521-553): distance type and
// integer, distance-safe coordinates; n >= 4; CSR offsets in bounds and
// ascending; rows strictly ascending, in range, without self loops, every
// entry mirrored in its neighbour's row; and the CSR holding exactly the
// active edges.  Every kernel access depends on it.
void ValidateHtGraph(const ee_graph_view& g) {
  if (g.dimension < 4) throw std::invalid_argument("HT reply snapshot needs at least four nodes");
  if (!DistanceSafe(g.x, g.y, g.dimension)) {
    throw std::invalid_argument("HT reply snapshot needs distance-safe integer coordinates");
  }
  const int32_t n = g.dimension;
  if (g.row_offsets[0] != 0) throw std::invalid_argument("CSR row_offsets[0] must be 0");
  for (int32_t v = 0; v < n; ++v) {
    if (g.row_offsets[v + 1] < g.row_offsets[v]) {
      throw std::invalid_argument("CSR row_offsets must be non-decreasing");
    }
  }
  int64_t active = 0;
  for (int32_t e = 0; e < g.edge_count; ++e) active += g.edge_active[e] != 0;
  if (static_cast<int64_t>(g.row_offsets[n]) != 2 * active) {
    throw std::invalid_argument("HT reply CSR must hold exactly the active edges");
  }
  for (int32_t v = 0; v < n; ++v) {
    int32_t previous = -1;
    for (int32_t a = g.row_offsets[v]; a < g.row_offsets[v + 1]; ++a) {
      const int32_t nb = g.neighbors[a];
      if (nb <= previous || nb < 0 || nb >= n || nb == v) {
        throw std::invalid_argument("HT reply CSR row is not strictly ascending and in range");
      }
      previous = nb;
    }
  }
  for (int32_t v = 0; v < n; ++v) {
    for (int32_t a = g.row_offsets[v]; a < g.row_offsets[v + 1]; ++a) {
      if (!RowHas(g, g.neighbors[a], v)) throw std::invalid_argument("HT reply CSR is not symmetric");
    }
  }
}

// Whether the resident snapshot is this one (coordinates, CSR and active
// flags); it then passed the HT checks when it was uploaded.
bool HtGraphMatches(const HtCache& c, const ee_graph_view& g) {
  const size_t n = static_cast<size_t>(g.dimension), m = static_cast<size_t>(g.edge_count);
  if (!c.valid || c.dimension != g.dimension || c.distance_type != g.distance_type || c.active.size() != m ||
      c.row_offsets.size() != n + 1 || std::memcmp(c.row_offsets.data(), g.row_offsets, (n + 1) * 4) != 0) {
    return false;
  }
  const struct {
    const void *cached, *given;
    size_t bytes;
  } arrays[] = {{c.x.data(), g.x, n * 8},
                {c.y.data(), g.y, n * 8},
                {c.neighbors.data(), g.neighbors, c.neighbors.size() * 4},
                {c.active.data(), g.edge_active, m}};
  // in pieces of 64 KiB; large snapshots on four host threads
  constexpr size_t kPiece = size_t{64} << 10;
  size_t pieces = 0;
  for (const auto& a : arrays) pieces += (a.bytes + kPiece - 1) / kPiece;
  std::atomic<bool> equal{true};
  ParallelFor(pieces, [&](size_t i) {
    for (const auto& a : arrays) {
      const size_t count = (a.bytes + kPiece - 1) / kPiece;
      if (i < count) {
        const size_t at = i * kPiece;
        if (std::memcmp(static_cast<const char*>(a.cached) + at, static_cast<const char*>(a.given) + at,
                        std::min(kPiece, a.bytes - at)) != 0) {
          equal = false;
        }
        return;
      }
      i -= count;
    }
  }, pieces < 8 ? 1 : 4);
  return equal;
}

// Keeps a device copy of a checked snapshot.
void UploadHtGraph(Context& ctx, const ee_graph_view& g) {
  HtCache& c = ctx.ht;
  const size_t n = static_cast<size_t>(g.dimension), m = static_cast<size_t>(g.edge_count);
  const size_t a = static_cast<size_t>(g.row_offsets[g.dimension]);
  c.valid = false;
  c.last_kind = 0;  // verdict bits go with their snapshot
  c.d_xy.Allocate(n, ctx.device);
  c.d_row_offsets.Allocate(n + 1, ctx.device);
  c.d_neighbors.Allocate(std::max<size_t>(a, 1), ctx.device);
  UploadItems(ctx, {{kUploadSpread64, c.d_xy.get(), g.x, n, 0, 0, 0},
                    {kUploadSpread64, c.d_xy.get(), g.y, n, 0, 0, 1},
                    {kUploadWords, c.d_row_offsets.get(), g.row_offsets, n + 1},
                    {kUploadWords, c.d_neighbors.get(), g.neighbors, a}});
  c.x.assign(g.x, g.x + n);
  c.y.assign(g.y, g.y + n);
  c.row_offsets.assign(g.row_offsets, g.row_offsets + n + 1);
  c.neighbors.assign(g.neighbors, g.neighbors + a);
  c.active.assign(g.edge_active, g.edge_active + m);
  c.near = NearExtent(g.x, g.y, g.dimension);
  c.max_degree = 0;
  for (size_t v = 0; v < n; ++v) {
    c.max_degree = std::max(c.max_degree, static_cast<uint32_t>(g.row_offsets[v + 1] - g.row_offsets[v]));
  }
  c.dimension = g.dimension;
  c.distance_type = g.distance_type;
  c.valid = true;
}

template <typename T> bool Reserve(DeviceArray<T>& a, size_t count, int device) {
  if (a.count() >= std::max<size_t>(count, 1)) return true;
  a.Allocate(Grow(a.count(), std::max<size_t>(count, 1)), device);
  return false;
}

uint64_t HtResidentBytes(const HtCache& c) {
  uint64_t host = 0;
  for (const HtCache::Verdicts& v : c.verdicts) host += v.centers.count() * 4 + v.bits.count() * 8;
  return host + c.d_xy.bytes() + c.d_row_offsets.bytes() + c.d_neighbors.bytes() + c.d_items.bytes() +
         c.d_counts.bytes() + c.d_offsets.bytes() + c.d_chunk_sums.bytes() + c.d_replies.bytes();
}

// Replies of centers [b, e), whose verdict bits begin at `bits`, in order, to
// `out`.
void WriteReplies(const HtCache& c, const HtCache::Verdicts& v, const uint64_t* bits, size_t b, size_t e,
                  int32_t* out) {
  for (size_t item = b; item < e; ++item) {
    const int32_t center = v.centers.get()[item];
    const int32_t* row = c.neighbors.data() + c.row_offsets[static_cast<size_t>(center)];
    const uint32_t d = static_cast<uint32_t>(c.row_offsets[static_cast<size_t>(center) + 1] -
                                             c.row_offsets[static_cast<size_t>(center)]);
    const uint32_t pairs = d < 2 ? 0 : d * (d - 1) / 2;
    const uint32_t words = VerdictWords(d);
    bool all = true;  // the usual case: every pair survives
    for (uint32_t w = 0; w < words; ++w) {
      const uint32_t left = pairs - w * 64;
      all = all && bits[w] == (left >= 64 ? ~uint64_t{0} : (uint64_t{1} << left) - 1);
    }
    if (all) {
      for (uint32_t i = 0; i + 1 < d; ++i) {
        const int32_t first = row[i];
        for (uint32_t j = i + 1; j < d; ++j) {
          out[0] = center;
          out[1] = first;
          out[2] = row[j];
          out += 3;
        }
      }
    } else {
      uint32_t i = 0, begin = 0, end = d - 1;  // pairs [begin, end) are those of neighbour i
      for (uint32_t w = 0; w < words; ++w) {
        for (uint64_t left = bits[w]; left != 0; left &= left - 1) {
          const uint32_t p = w * 64 + static_cast<uint32_t>(__builtin_ctzll(left));
          while (p >= end) {
            ++i;
            begin = end;
            end += d - 1 - i;
          }
          out[0] = center;
          out[1] = row[i];
          out[2] = row[p - begin + i + 1];
          out += 3;
        }
      }
    }
    bits += v.stride != 0 ? v.stride : words;
  }
}

// Host threads: writing 19 MB of replies takes 12 about 0.15 ms.  Below
// kSerialReplies waking them costs more than it saves: 37,500 replies take 17
// us on one thread, 48,500 21 and 103,000 46; 20, 20 and 25 on 12.
constexpr unsigned kReplyThreads = 12;
constexpr uint64_t kSerialReplies = 50000;

// Replies [first, first + count) of the last verdicts.
void CopyVerdictReplies(const HtCache& c, uint64_t first, uint64_t count, int32_t* out) {
  const HtCache::Verdicts& v = c.verdicts[c.current];
  const auto group_of = [&](uint64_t reply) {
    return static_cast<size_t>(std::upper_bound(v.group_first.begin(), v.group_first.end(), reply) -
                               v.group_first.begin()) - 1;
  };
  const size_t g0 = group_of(first), g1 = group_of(first + count - 1) + 1;
  ParallelFor(g1 - g0, [&](size_t i) {
    const size_t g = g0 + i;
    const size_t b = g * v.group, e = std::min(v.count, b + v.group);
    const uint64_t* bits = v.bits.get() + (v.stride != 0 ? b * v.stride : v.first_words()[b / v.per_wave]);
    const uint64_t from = v.group_first[g], to = v.group_first[g + 1];
    if (from >= first && to <= first + count) {
      WriteReplies(c, v, bits, b, e, out + 3 * (from - first));
      return;
    }
    std::vector<int32_t> whole(3 * (to - from));  // a group the range cuts
    WriteReplies(c, v, bits, b, e, whole.data());
    const uint64_t lo = std::max(from, first), hi = std::min(to, first + count);
    std::copy(whole.begin() + 3 * (lo - from), whole.begin() + 3 * (hi - from), out + 3 * (lo - first));
  }, count < kSerialReplies ? 1 : kReplyThreads);
}

void CheckHamilton(const ee_graph_view& g, int32_t tu, int32_t tv, const int32_t* centers, size_t count) {
  if (tu < 0 || tv >= g.dimension || tu == tv || !RowHas(g, tu, tv)) {
    throw std::invalid_argument("HT Hamilton replies: the target is not an active edge");
  }
  bool bad = false;
  for (size_t i = 0; i < count; ++i) {
    const int32_t c = centers[i];
    bad |= static_cast<uint32_t>(c) >= static_cast<uint32_t>(g.dimension) || c == tu || c == tv;
  }
  if (bad) throw std::invalid_argument("HT Hamilton replies: invalid center");
}

// How a call's verdict bits lie in host memory, or that it does not take them.
struct VerdictPlan {
  bool take = false;
  uint32_t stride = 0;    // words of every center, or 0: as many as its row needs
  uint32_t per_wave = 4;  // centers of a wavefront
  size_t words = 0;
};

// The rule goes by the rows of the given centers on the resident snapshot, not
// by its longest row: a hub among short rows costs its own words only.
//  - kUniformDegree: up to here (4 words) all centers get the longest row's
//    words and the host need not look at the rows; 32 bytes a center are less
//    than its replies.
//  - kMeanWords: the form is faster as far as both were measured, from the
//    smallest calls (one launch and one wait for four and three): whole calls
//    on k-NN graphs, 300 to 30,000 centers with 3 to 52 words each, 154-5,260
//    us by three passes and 71-1,950 by bits; complete graphs of 40 to 90
//    nodes (12 to 62 words) 91-455 and 60-190.  Beyond, replies are hundreds
//    of MB, which PCIe carries about as fast as host threads write them.
//  - kBitsDegree: pair numbers stay exact in the kernel's float root.
//  - kBitsBytes and kBitsCenters bound what a context keeps page-locked.
constexpr uint32_t kUniformDegree = 23;
constexpr size_t kMeanWords = 64;
constexpr uint32_t kBitsDegree = 512;
constexpr size_t kBitsBytes = size_t{32} << 20;
constexpr size_t kBitsCenters = kBitsBytes / sizeof(uint64_t);

VerdictPlan PlanVerdicts(const HtCache& c, const int32_t* centers, size_t count) {
  VerdictPlan p;
  if (count == 0 || count > kBitsCenters) return p;
  uint32_t longest = c.max_degree;
  if (c.max_degree <= kUniformDegree) {
    p.stride = std::max<uint32_t>(1, VerdictWords(c.max_degree));
    p.words = count * p.stride;
  } else {
    longest = 0;
    for (size_t i = 0; i < count; ++i) {
      const size_t v = static_cast<uint32_t>(centers[i]);
      if (v >= static_cast<size_t>(c.dimension)) continue;  // refused later
      const uint32_t d = static_cast<uint32_t>(c.row_offsets[v + 1] - c.row_offsets[v]);
      longest = std::max(longest, d);
      if (longest > kBitsDegree) return p;
      p.words += VerdictWords(d);
    }
  }
  p.per_wave = longest <= kHtLdsNeighbors ? 4 : 1;
  p.take = p.words <= kMeanWords * count && p.words * sizeof(uint64_t) <= kBitsBytes;
  return p;
}

// Starts the verdict pass on the resident snapshot into the buffer that does
// not hold the last call's; returns whether the buffers had room.
bool LaunchVerdicts(Context& ctx, int type, int32_t tu, int32_t tv, const int32_t* centers, size_t count,
                    const VerdictPlan& plan) {
  HtCache& c = ctx.ht;
  HtCache::Verdicts& v = c.verdicts[c.current ^ 1];
  v.stride = plan.stride;
  v.per_wave = plan.per_wave;
  v.count = count;
  // groups of the host's work, whole wavefronts: 256 centers or some 1,024
  // words (half of that took 5 us more for 30,000 centers, whose groups then
  // share more of the replies' untouched pages), and as many as threads
  const size_t most = std::min<size_t>(256, 1024 * count / std::max<size_t>(plan.words, 1));
  v.group = (std::min(most, (count + kReplyThreads - 1) / kReplyThreads) + 3) / 4 * 4;
  const size_t waves = (count + plan.per_wave - 1) / plan.per_wave;
  const size_t ints = 2 * count + (plan.stride != 0 ? 0 : waves), words = std::max<size_t>(plan.words, 1);
  const bool room = v.centers.count() >= ints && v.bits.count() >= words;
  for (HtCache::Verdicts& b : c.verdicts) {
    if (&b != &v && c.last_kind == 1 && c.last_bits) continue;  // growing would drop the last call's replies
    // both, so that the next call of this size finds room as this one's does
    b.centers.Reserve(std::min(Grow(b.centers.count(), ints), 3 * kBitsCenters));
    b.bits.Reserve(std::min(Grow(b.bits.count(), words), kBitsBytes / sizeof(uint64_t)));
  }
  std::memcpy(v.centers.get(), centers, count * sizeof(int32_t));
  if (plan.stride == 0) {
    uint32_t* const first_words = reinterpret_cast<uint32_t*>(v.centers.get()) + 2 * count;
    uint32_t run = 0;
    for (size_t i = 0; i < count; ++i) {
      if (i % plan.per_wave == 0) first_words[i / plan.per_wave] = run;
      const size_t node = static_cast<uint32_t>(centers[i]);
      if (node >= static_cast<size_t>(c.dimension)) continue;
      run += VerdictWords(static_cast<uint32_t>(c.row_offsets[node + 1] - c.row_offsets[node]));
    }
  }
  const auto kernel = plan.per_wave == 1 ? (c.near ? HtVerdictKernel<true, 1> : HtVerdictKernel<false, 1>)
                                         : (c.near ? HtVerdictKernel<true, 4> : HtVerdictKernel<false, 4>);
  const uint32_t* const device = reinterpret_cast<const uint32_t*>(v.centers.device());
  hipLaunchKernelGGL(kernel, dim3(static_cast<uint32_t>((waves + kHtWaves - 1) / kHtWaves)), dim3(kHtBlock), 0,
                     ctx.stream, c.d_xy.get(), c.d_row_offsets.get(), c.d_neighbors.get(), c.dimension, type, tu, tv,
                     v.centers.device(), static_cast<uint32_t>(count), plan.stride, device + 2 * count,
                     v.bits.device(), reinterpret_cast<uint32_t*>(v.centers.device() + count));
  CheckHip(hipGetLastError(), "HtVerdictKernel launch");
  return room;
}

// Offsets and group totals from the finished verdict pass's counts.
uint64_t CountVerdicts(HtCache& c, uint64_t* offsets) {
  HtCache::Verdicts& v = c.verdicts[c.current ^ 1];
  const uint32_t* counts = reinterpret_cast<const uint32_t*>(v.centers.get() + v.count);
  const size_t groups = (v.count + v.group - 1) / v.group;
  v.group_first.assign(groups + 1, 0);
  uint64_t run = 0;
  for (size_t g = 0; g < groups; ++g) {
    for (size_t i = g * v.group, e = std::min(v.count, i + v.group); i < e; ++i) {
      run += counts[i];
      offsets[i + 1] = run;
    }
    v.group_first[g + 1] = run;
  }
  return run;
}

// As HamiltonReplies below, by the verdict bits of the pass launched at
// `launched`.
void VerdictReplies(Context& ctx, std::chrono::steady_clock::time_point launched, uint64_t* offsets,
                    ee_ht_neighbor_pair* replies, uint64_t capacity, uint64_t* total, ee_ht_usage* u) {
  HtCache& c = ctx.ht;
  ctx.Sync();
  u->kernel_ms = MsSince(launched);
  const auto t0 = std::chrono::steady_clock::now();
  *total = CountVerdicts(c, offsets);
  c.current ^= 1;
  c.last_kind = 1;
  c.last_bits = true;
  c.last_total = *total;
  const uint64_t copy = std::min(*total, capacity);
  if (copy > 0) CopyVerdictReplies(c, 0, copy, reinterpret_cast<int32_t*>(replies));
  u->d2h_ms = MsSince(t0);
  u->resident_bytes = HtResidentBytes(c);
}

void HamiltonReplies(Context& ctx, const ee_graph_view* graph, int32_t target_u, int32_t target_v,
                     const int32_t* centers, size_t count, uint64_t* offsets,
                     ee_ht_neighbor_pair* replies, uint64_t capacity, uint64_t* total,
                     ee_ht_usage* usage) {
  ee_ht_usage u{};
  ctx.Activate();
  CheckGraphView(graph);
  const ee_graph_view& g = *graph;
  if (offsets == nullptr || total == nullptr || (count > 0 && centers == nullptr) ||
      (capacity > 0 && replies == nullptr)) {
    throw std::invalid_argument("HT Hamilton replies: NULL argument");
  }
  auto t0 = std::chrono::steady_clock::now();
  const int32_t tu = std::min(target_u, target_v), tv = std::max(target_u, target_v);
  // Where the snapshot looks like the resident one, the verdict pass goes out
  // first and the comparison runs beside it (the kernel leaves centers out of
  // range alone; nothing reaches the caller before the checks).
  const bool likely = count > 0 && tu >= 0 && tu != tv && tv < g.dimension && ctx.ht.valid &&
                      ctx.ht.dimension == g.dimension && ctx.ht.distance_type == g.distance_type &&
                      ctx.ht.active.size() == static_cast<size_t>(g.edge_count) &&
                      std::memcmp(ctx.ht.x.data(), g.x, std::min<size_t>(ctx.ht.x.size(), 64) * 8) == 0;
  VerdictPlan plan;
  if (likely) plan = PlanVerdicts(ctx.ht, centers, count);
  bool started = plan.take;
  std::chrono::steady_clock::time_point launched;
  const auto launch = [&] {
    u.workspace_hit = LaunchVerdicts(ctx, g.distance_type, tu, tv, centers, count, plan) ? 1 : 0;
    u.h2d_ms = MsSince(t0);
    launched = std::chrono::steady_clock::now();
  };
  if (started) launch();
  try {
    u.graph_hit = HtGraphMatches(ctx.ht, g) ? 1 : 0;
    if (!u.graph_hit) ValidateHtGraph(g);
    CheckHamilton(g, tu, tv, centers, count);
  } catch (...) {
    if (started) static_cast<void>(hipStreamSynchronize(ctx.stream));
    throw;
  }
  if (!u.graph_hit) {
    if (started) ctx.Sync();
    started = false;
    UploadHtGraph(ctx, g);
  }
  offsets[0] = 0;
  *total = 0;
  HtCache& c = ctx.ht;
  c.last_kind = 0;
  c.last_total = 0;
  if (count == 0) {
    if (usage) *usage = u;
    return;
  }
  if (!started) plan = PlanVerdicts(c, centers, count);
  if (plan.take) {
    if (!started) launch();
    VerdictReplies(ctx, launched, offsets, replies, capacity, total, &u);
    if (usage) *usage = u;
    return;
  }
  const uint64_t chunks = (count + kScanChunk - 1) / kScanChunk;
  bool ws = Reserve(c.d_items, count, ctx.device);
  ws = Reserve(c.d_counts, count, ctx.device) && ws;
  ws = Reserve(c.d_offsets, count + 1, ctx.device) && ws;
  ws = Reserve(c.d_chunk_sums, chunks, ctx.device) && ws;
  c.d_items.Upload(centers, count, ctx.stream);
  ctx.Sync();
  u.h2d_ms = MsSince(t0);

  // count pass and offset scan, then the exact reply count (the reference
  // sizes its reply buffer the same way, ht_replies.cu:626-637)
  t0 = std::chrono::steady_clock::now();
  const uint64_t blocks = (count + kHtWaves - 1) / kHtWaves;
  const auto count_kernel = c.near ? HtHamiltonKernel<false, true> : HtHamiltonKernel<false, false>;
  const auto write_kernel = c.near ? HtHamiltonKernel<true, true> : HtHamiltonKernel<true, false>;
  hipLaunchKernelGGL(count_kernel, dim3(static_cast<uint32_t>(blocks)), dim3(kHtBlock), 0,
                     ctx.stream, c.d_xy.get(), c.d_row_offsets.get(), c.d_neighbors.get(),
                     static_cast<int>(g.distance_type), tu, tv, c.d_items.get(),
                     static_cast<uint64_t>(count), c.d_counts.get(), nullptr, nullptr);
  CheckHip(hipGetLastError(), "HtHamiltonKernel count launch");
  hipLaunchKernelGGL(HtChunkSumKernel, dim3(static_cast<uint32_t>(chunks)), dim3(kScanThreads), 0, ctx.stream,
                     c.d_counts.get(), static_cast<uint64_t>(count), c.d_chunk_sums.get());
  CheckHip(hipGetLastError(), "HtChunkSumKernel launch");
  hipLaunchKernelGGL(HtScanKernel, dim3(static_cast<uint32_t>(chunks)), dim3(kScanThreads), 0,
                     ctx.stream, c.d_counts.get(), static_cast<uint64_t>(count),
                     c.d_chunk_sums.get(), c.d_offsets.get());
  CheckHip(hipGetLastError(), "HtScanKernel launch");
  c.d_offsets.Download(offsets, count + 1, ctx.stream);
  ctx.Sync();
  *total = offsets[count];
  uint64_t bound = 0;  // every neighbour pair of every center
  for (size_t i = 0; i < count; ++i) {
    const uint64_t d = static_cast<uint64_t>(g.row_offsets[centers[i] + 1] - g.row_offsets[centers[i]]);
    bound += d < 2 ? 0 : d * (d - 1) / 2;
  }
  if (*total > bound) throw std::logic_error("HT Hamilton replies exceed the pair bound");
  if (*total > UINT64_MAX / 3) throw std::overflow_error("HT Hamilton reply count overflows");
  ws = Reserve(c.d_replies, 3 * *total, ctx.device) && ws;
  u.workspace_hit = ws ? 1 : 0;
  hipLaunchKernelGGL(write_kernel, dim3(static_cast<uint32_t>(blocks)), dim3(kHtBlock), 0,
                     ctx.stream, c.d_xy.get(), c.d_row_offsets.get(), c.d_neighbors.get(),
                     static_cast<int>(g.distance_type), tu, tv, c.d_items.get(),
                     static_cast<uint64_t>(count), nullptr, c.d_offsets.get(), c.d_replies.get());
  CheckHip(hipGetLastError(), "HtHamiltonKernel write launch");
  ctx.Sync();
  u.kernel_ms = MsSince(t0);
  c.last_kind = 1;
  c.last_bits = false;
  c.last_total = *total;

  t0 = std::chrono::steady_clock::now();
  const uint64_t copy = std::min(*total, capacity);
  if (copy > 0) DownloadToCaller(ctx, replies, c.d_replies.get(), copy * sizeof(ee_ht_neighbor_pair));
  u.d2h_ms = MsSince(t0);
  u.resident_bytes = HtResidentBytes(c);
  if (usage) *usage = u;
}

// Replies [first, first + count) of the context's last reply call.
void CopyReplies(Context& ctx, uint64_t first, uint64_t count, void* out) {
  HtCache& c = ctx.ht;
  if (c.last_kind == 0) throw std::logic_error("HT copy replies: no reply call has completed");
  if (first > c.last_total || count > c.last_total - first) {
    throw std::invalid_argument("HT copy replies: range beyond the last call's replies");
  }
  if (count == 0) return;
  if (out == nullptr) throw std::invalid_argument("HT copy replies: NULL buffer");
  if (c.last_kind == 1 && c.last_bits) {
    CopyVerdictReplies(c, first, count, static_cast<int32_t*>(out));
    return;
  }
  ctx.Activate();
  const size_t record = c.last_kind == 1 ? sizeof(ee_ht_neighbor_pair) : sizeof(ee_node_edge);
  DownloadToCaller(ctx, out, reinterpret_cast<const char*>(c.d_replies.get()) + first * record, count * record);
}

void EndReplies(Context& ctx, const ee_graph_view* graph, const ee_ht_end_task* tasks, size_t count,
                uint64_t* offsets, ee_node_edge* replies, uint64_t capacity, uint64_t* total,
                ee_ht_usage* usage) {
  ee_ht_usage u{};
  ctx.Activate();
  CheckGraphView(graph);
  const ee_graph_view& g = *graph;
  if (offsets == nullptr || total == nullptr || (count > 0 && tasks == nullptr) ||
      (capacity > 0 && replies == nullptr)) {
    throw std::invalid_argument("HT end replies: NULL argument");
  }
  auto t0 = std::chrono::steady_clock::now();
  u.graph_hit = HtGraphMatches(ctx.ht, g) ? 1 : 0;
  if (!u.graph_hit) ValidateHtGraph(g);
  offsets[0] = 0;
  for (size_t i = 0; i < count; ++i) {
    const int32_t e = tasks[i].endpoint, in = tasks[i].internal_neighbor;
    if (e < 0 || e >= g.dimension || in < 0 || in >= g.dimension || e == in || !RowHas(g, e, in)) {
      throw std::invalid_argument("HT end replies: a task must name an active path-internal edge");
    }
    // the internal edge is in the row exactly once, so the rest are replies
    offsets[i + 1] = offsets[i] + static_cast<uint64_t>(g.row_offsets[e + 1] - g.row_offsets[e] - 1);
  }
  *total = offsets[count];
  if (!u.graph_hit) UploadHtGraph(ctx, g);
  HtCache& c = ctx.ht;
  c.last_kind = 0;
  c.last_total = 0;
  if (count == 0) {
    if (usage) *usage = u;
    return;
  }
  bool ws = Reserve(c.d_items, 2 * count, ctx.device);
  ws = Reserve(c.d_offsets, count + 1, ctx.device) && ws;
  ws = Reserve(c.d_replies, 2 * *total, ctx.device) && ws;
  u.workspace_hit = ws ? 1 : 0;
  static_assert(sizeof(ee_ht_end_task) == 8, "task layout");
  c.d_items.Upload(reinterpret_cast<const int32_t*>(tasks), 2 * count, ctx.stream);
  c.d_offsets.Upload(offsets, count + 1, ctx.stream);
  ctx.Sync();
  u.h2d_ms = MsSince(t0);
  t0 = std::chrono::steady_clock::now();
  const uint64_t blocks = (count + kHtBlock - 1) / kHtBlock;
  hipLaunchKernelGGL(HtEndKernel, dim3(static_cast<uint32_t>(blocks)), dim3(kHtBlock), 0, ctx.stream,
                     c.d_row_offsets.get(), c.d_neighbors.get(), c.d_items.get(),
                     static_cast<uint64_t>(count), c.d_offsets.get(), c.d_replies.get());
  CheckHip(hipGetLastError(), "HtEndKernel launch");
  ctx.Sync();
  u.kernel_ms = MsSince(t0);
  c.last_kind = 2;
  c.last_total = *total;
  t0 = std::chrono::steady_clock::now();
  const uint64_t copy = std::min(*total, capacity);
  if (copy > 0) DownloadToCaller(ctx, replies, c.d_replies.get(), copy * sizeof(ee_node_edge));
  u.d2h_ms = MsSince(t0);
  u.resident_bytes = HtResidentBytes(c);
  if (usage) *usage = u;
}

template <typename F> ee_status Guarded(F&& body) {
  try {
    body();
    return EE_OK;
  } catch (...) {
    return StatusFromException();
  }
}

}  // namespace
}  // namespace ee

extern "C" {

ee_status ee_ht_hamilton_replies(ee_ctx* ctx, const ee_graph_view* graph, int32_t target_u,
                                 int32_t target_v, const int32_t* centers, size_t center_count,
                                 uint64_t* offsets, ee_ht_neighbor_pair* replies, uint64_t capacity,
                                 uint64_t* total, ee_ht_usage* usage) {
  return ee::Guarded([&] {
    if (ctx == nullptr) throw std::invalid_argument("NULL context");
    ee::HamiltonReplies(*reinterpret_cast<ee::Context*>(ctx), graph, target_u, target_v, centers,
                        center_count, offsets, replies, capacity, total, usage);
  });
}

ee_status ee_ht_end_replies(ee_ctx* ctx, const ee_graph_view* graph, const ee_ht_end_task* tasks,
                            size_t task_count, uint64_t* offsets, ee_node_edge* replies,
                            uint64_t capacity, uint64_t* total, ee_ht_usage* usage) {
  return ee::Guarded([&] {
    if (ctx == nullptr) throw std::invalid_argument("NULL context");
    ee::EndReplies(*reinterpret_cast<ee::Context*>(ctx), graph, tasks, task_count, offsets, replies,
                   capacity, total, usage);
  });
}

ee_status ee_ht_copy_replies(ee_ctx* ctx, uint64_t first, uint64_t count, void* replies) {
  return ee::Guarded([&] {
    if (ctx == nullptr) throw std::invalid_argument("NULL context");
    ee::CopyReplies(*reinterpret_cast<ee::Context*>(ctx), first, count, replies);
  });
}

ee_status ee_ht_clear_cache(ee_ctx* ctx) {
  return ee::Guarded([&] {
    if (ctx == nullptr) throw std::invalid_argument("NULL context");
    ee::Context& c = *reinterpret_cast<ee::Context*>(ctx);
    c.Activate();
    c.ht = ee::HtCache{};
  });
}

}  // extern "C"
