// Transfers between caller memory and the device through page-locked host
// memory which kernels read and write in place: the ring itself (DirectIo),
// the host's side of taking tiles out of it, the download of device-resident
// cells and words, and the upload of task rows.
#include <algorithm>
#include <array>
#include <cstring>
#include <stdexcept>
#include <vector>

#include "ee_internal.h"
#include "ee_jvhost.h"
#include "ee_runtime.h"

namespace ee {
namespace {

// A wavefront's tile of resident cells, and the wavefronts of a launch.
// PCIe bounds the kernel (PackCells), so it runs few wavefronts with many
// tiles each, and tiles arrive in order while later ones are on their way.
constexpr uint32_t kWave = 64;
constexpr uint32_t kPackTile = 512;
constexpr uint32_t kPackWaves = 128;

// Cells [0, count) in transfer form to lo (and hi, for cells that may need
// their high byte), tile by tile, `mark` to marks[i] after tile i.
template <bool kWide>
__global__ __launch_bounds__(kWave) void PackCells(const int64_t* __restrict__ cells, uint32_t count,
                                                   uint32_t* __restrict__ lo, uint8_t* __restrict__ hi,
                                                   uint64_t* __restrict__ marks, uint64_t mark) {
  const uint32_t tiles = (count + kPackTile - 1) / kPackTile;
  for (uint32_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
    const uint32_t end = min(count, (tile + 1) * kPackTile);
#pragma unroll 4
    for (uint32_t i = tile * kPackTile + threadIdx.x; i < end; i += kWave) {
      const int64_t v = cells[i];
      const bool bad = v == INT64_MAX;
      lo[i] = bad ? kPackedInvalid : static_cast<uint32_t>(v);
      if (kWide) hi[i] = bad ? kPackedInvalidHi : static_cast<uint8_t>(v >> 32);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "");
    if (threadIdx.x == 0) __hip_atomic_store(marks + tile, mark, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// Words [0, count) to host memory, tile by tile, as PackCells.
__global__ __launch_bounds__(kWave) void CopyWords(const uint32_t* __restrict__ words, uint32_t count,
                                                   uint32_t* __restrict__ out, uint64_t* __restrict__ marks,
                                                   uint64_t mark) {
  const uint32_t tiles = (count + kPackTile - 1) / kPackTile;
  for (uint32_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
    const uint32_t end = min(count, (tile + 1) * kPackTile);
#pragma unroll 4
    for (uint32_t i = tile * kPackTile + threadIdx.x; i < end; i += kWave) out[i] = words[i];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "");
    if (threadIdx.x == 0) __hip_atomic_store(marks + tile, mark, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// ValidateTasks' rule for one row (12 words) of a segment.
__device__ inline bool RowIsValid(const int32_t* row, uint32_t k, int32_t n) {
  bool ok = row[11] >= 0;  // the high word of deleted_cost
  uint64_t deleted[kMaxK];
  for (uint32_t e = 0; e < static_cast<uint32_t>(kMaxK); ++e) {
    if (e >= k) break;
    const int32_t a = row[2 * e], b = row[2 * e + 1];
    ok = ok && a >= 0 && b >= 0 && a < n && b < n && a != b;
    deleted[e] = (static_cast<uint64_t>(min(a, b)) << 32) | static_cast<uint32_t>(max(a, b));
    for (uint32_t f = 0; f < e; ++f) ok = ok && deleted[f] != deleted[e];
  }
  return ok;
}

// One workgroup per 256 rows: it reads them from host memory in whole words,
// stores them to the row pool, and checks a row per thread out of LDS.  PCIe
// bounds it (56 GB/s: 12.6 MB in 225 us); the host's check of as many rows
// took 1.2 ms.  marks[i] once group i is done, *refused = 1 on a bad row.
constexpr uint32_t kIngestRows = 256;
constexpr uint32_t kRowWords = sizeof(ee_kopt_task) / 4;

__global__ __launch_bounds__(kIngestRows) void IngestRows(const uint32_t* __restrict__ staged, uint64_t first,
                                                          uint32_t count, const KoptRowSegment* __restrict__ segments,
                                                          uint32_t segment_count, uint32_t* __restrict__ rows,
                                                          uint32_t* __restrict__ refused, uint64_t* __restrict__ marks,
                                                          uint64_t mark) {
  __shared__ int32_t words[kIngestRows * kRowWords];
  const uint32_t row0 = blockIdx.x * kIngestRows;
  const uint32_t here = min(kIngestRows, count - row0);
  const uint32_t* from = staged + static_cast<uint64_t>(row0) * kRowWords;
  uint32_t* to = rows + (first + row0) * kRowWords;
#pragma unroll 4
  for (uint32_t q = threadIdx.x; q < here * kRowWords; q += kIngestRows) {
    const uint32_t v = from[q];
    words[q] = static_cast<int32_t>(v);
    to[q] = v;
  }
  __syncthreads();
  if (threadIdx.x < here) {
    const uint64_t row = first + row0 + threadIdx.x;
    uint32_t lo = 0, hi = segment_count - 1;  // the last segment that begins at or before the row
    while (lo < hi) {
      const uint32_t mid = lo + (hi - lo + 1) / 2;
      if (segments[mid].row_begin <= row) {
        lo = mid;
      } else {
        hi = mid - 1;
      }
    }
    if (!RowIsValid(words + threadIdx.x * kRowWords, segments[lo].k, segments[lo].n)) {
      __hip_atomic_store(refused, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "");
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "");
    __hip_atomic_store(marks + blockIdx.x, mark, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

constexpr uint32_t kPartThreads = 256;
constexpr uint32_t kPartBytes = 8192;  // of a part in a slot, at most; 4096 and 2048 measured slower

// A part of an upload item in a slot: `count` elements from byte `at` of the
// slot (16-byte aligned) to `to`.
struct UploadPart {
  uint64_t to;
  uint32_t at, count, kind, limit, add, lane;
};
static_assert(sizeof(UploadPart) == 32, "parts are read as whole 32-byte records");

// The parts of a slot to their arrays, in the forms of UploadKind.  A value
// at or above its limit is stored as `add` alone and refuses the upload.
// PCIe bounds it: a block holds a whole part in registers before it stores,
// and many blocks keep the link busy (1.44 MB of a JV call, host copy
// included, 67 us; parts of 2 KiB 95 us).  marks[b] once block b is done.
// Against copy commands from caller memory, one per array: 64 graphs with
// 435,000 edge slots built and uploaded in 2.5 ms, 5.1 ms before.
__global__ __launch_bounds__(kPartThreads) void StoreParts(const UploadPart* __restrict__ parts, uint32_t count,
                                                  const char* __restrict__ slot, uint32_t* __restrict__ refused,
                                                  uint64_t* __restrict__ marks, uint64_t mark) {
  constexpr uint32_t kHeld = kPartBytes / 4 / kPartThreads;  // a thread's words of a part, all in flight at once
  const uint32_t t = threadIdx.x;
  bool bad = false;
  for (uint32_t i = blockIdx.x; i < count; i += gridDim.x) {  // uniform
    const UploadPart part = parts[i];
    const uint32_t* from = reinterpret_cast<const uint32_t*>(slot + part.at);
    int32_t* to = reinterpret_cast<int32_t*>(part.to);
    if (part.kind == kUploadSpread64) {
      const int64_t* from64 = reinterpret_cast<const int64_t*>(from);
      int64_t* to64 = reinterpret_cast<int64_t*>(part.to);
      int64_t v[kHeld / 2];
#pragma unroll
      for (uint32_t j = 0; j < kHeld / 2; ++j) {
        const uint32_t q = j * kPartThreads + t;
        v[j] = q < part.count ? from64[q] : 0;
      }
#pragma unroll
      for (uint32_t j = 0; j < kHeld / 2; ++j) {
        const uint32_t q = j * kPartThreads + t;
        if (q < part.count) to64[2 * q + part.lane] = v[j];
      }
      continue;
    }
    const uint32_t words = part.kind == kUploadFlags ? (part.count + 3) / 4 : part.count;
    uint32_t v[kHeld];
#pragma unroll
    for (uint32_t j = 0; j < kHeld; ++j) {
      const uint32_t q = j * kPartThreads + t;
      v[j] = q < words ? from[q] : 0;
    }
#pragma unroll
    for (uint32_t j = 0; j < kHeld; ++j) {
      const uint32_t q = j * kPartThreads + t;
      if (q >= words) break;
      if (part.kind == kUploadWords) {
        const bool out = v[j] >= part.limit && part.limit != 0;
        bad |= out;
        to[q] = static_cast<int32_t>((out ? 0u : v[j]) + part.add);
      } else if (part.kind == kUploadSpread32) {
        to[2 * q + part.lane] = static_cast<int32_t>(v[j] + part.add);
      } else {
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) {
          if (4 * q + u < part.count) to[4 * q + u] = ((v[j] >> (8 * u)) & 0xffu) != 0 ? 1 : 0;
        }
      }
    }
  }
  if (bad) {
    __hip_atomic_store(refused, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "");
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "");
    __hip_atomic_store(marks + blockIdx.x, mark, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// Passes items [0, count) through the ring in launches of at most
// `slot_items`, each with a slot of slot_bytes: start(i, slot) stages and
// launches number i, finish(i, slot) takes what it left.
template <typename Start, typename Finish>
void ThroughRing(Context& ctx, size_t launches, Start&& start, Finish&& finish) {
  const size_t slots = std::min<size_t>(launches, DirectIo::kSlots);
  try {
    for (size_t i = 0; i < slots; ++i) start(i, i);
    for (size_t i = 0; i < launches; ++i) {
      finish(i, i % slots);
      if (i + slots < launches) start(i + slots, i % slots);
    }
  } catch (...) {
    static_cast<void>(hipStreamSynchronize(ctx.stream));  // the ring is free again
    throw;
  }
}

constexpr size_t kSlotBytes = DirectIo::kSlotBytes;
static_assert(kSlotBytes / 4 / kPackTile <= DirectIo::kSlotTiles, "a slot's tiles have marks");

}  // namespace

void DirectIo::Create() {
  marks_.Allocate(kSlots * kSlotTiles);
  mem_.Allocate(kBytes);
}

void DirectIo::WaitTile(size_t slot, size_t tile, uint64_t mark, hipStream_t stream) const {
  const uint64_t* at = marks_.host() + slot * kSlotTiles + tile;
  const auto seen = [&] { return __atomic_load_n(at, __ATOMIC_ACQUIRE) == mark; };
  for (uint64_t polls = 1; !seen(); ++polls) {
    __builtin_ia32_pause();
    // a kernel that ended, or failed, without the mark: look now and then
    if (polls % (uint64_t{1} << 16) != 0) continue;
    const hipError_t status = hipStreamQuery(stream);
    if (status == hipErrorNotReady || seen()) continue;
    CheckHip(status, "kernel writing to host memory");
    throw std::runtime_error("a kernel ended without marking a tile");
  }
}

void DirectIo::TakeTiles(size_t slot, uint64_t mark, hipStream_t stream, size_t tiles, size_t group,
                         unsigned threads, const std::function<void(size_t, size_t)>& take) const {
  // the work queued before the launch is waited for here, not on the process's
  // host threads, which run one caller's job at a time
  if (tiles > 0) WaitTile(slot, 0, mark, stream);
  ParallelFor((tiles + group - 1) / group, [&](size_t g) {
    const size_t first = g * group, last = std::min(tiles, first + group);
    for (size_t t = first; t < last; ++t) WaitTile(slot, t, mark, stream);
    take(first, last);
  }, threads);
}

// On the host threads from kSerialCells up (below, waking them costs more
// than it saves; the expansion of a large result needs about twelve to keep
// pace with PCIe).
void DirectIo::TakeCells(size_t slot, uint64_t mark, hipStream_t stream, const uint32_t* lo, const uint8_t* hi,
                         size_t count, size_t tile_cells, int64_t* cells) const {
  constexpr size_t kGroupCells = 16384, kSerialCells = 65536;
  constexpr unsigned kThreads = 12;
  TakeTiles(slot, mark, stream, (count + tile_cells - 1) / tile_cells, std::max<size_t>(1, kGroupCells / tile_cells),
            count < kSerialCells ? 1 : kThreads, [&](size_t first, size_t last) {
    const size_t b = first * tile_cells, e = std::min(count, last * tile_cells);
    ExpandCells(lo + b, hi != nullptr ? hi + b : nullptr, e - b, cells + b);
  });
}

// Half the bytes of a copy of the int64 cells (five eighths with high bytes)
// and no copy command.  21.8 MB of near cells (10.9 MB, 195 us of PCIe) take
// 265 us, 26.8 MB in three downloads 365 us instead of 736.  Slots of 4 MiB
// would save 30 us of gaps between launches, for 1.5 ms more of page-locked
// memory when a context is made; launches alternating on two
// streams, with slots of 1 or 2 MiB, measured slower (290-360 us).
void DownloadCells(Context& ctx, const int64_t* d_cells, size_t count, bool wide, int64_t* cells) {
  if (count == 0) return;
  if (d_cells == nullptr || cells == nullptr) throw std::logic_error("download with a NULL buffer");
  const size_t cell_bytes = wide ? 5 : 4;
  const size_t slot_cells = kSlotBytes / cell_bytes / kPackTile * kPackTile;
  const size_t launches = (count + slot_cells - 1) / slot_cells;
  const size_t plane = launches == 1 ? (count + 255) / 256 * 256 : slot_cells;
  const size_t slot_bytes = plane * cell_bytes;
  DirectIo& io = ctx.io;
  uint64_t marks[DirectIo::kSlots] = {};
  const auto cells_of = [&](size_t i) { return std::min(slot_cells, count - i * slot_cells); };
  ThroughRing(ctx, launches, [&](size_t i, size_t slot) {
    char* at = io.device() + slot * slot_bytes;
    marks[slot] = io.NextMark();
    const uint32_t n = static_cast<uint32_t>(cells_of(i));
    hipLaunchKernelGGL((wide ? PackCells<true> : PackCells<false>),
                       dim3(std::min<uint32_t>(kPackWaves, (n + kPackTile - 1) / kPackTile)), dim3(kWave), 0, ctx.stream,
                       d_cells + i * slot_cells, n, reinterpret_cast<uint32_t*>(at),
                       reinterpret_cast<uint8_t*>(at + plane * 4), io.device_marks(slot), marks[slot]);
    CheckHip(hipGetLastError(), "PackCells launch");
  }, [&](size_t i, size_t slot) {
    const char* at = io.host() + slot * slot_bytes;
    io.TakeCells(slot, marks[slot], ctx.stream, reinterpret_cast<const uint32_t*>(at),
                 wide ? reinterpret_cast<const uint8_t*>(at + plane * 4) : nullptr, cells_of(i), kPackTile,
                 cells + i * slot_cells);
  });
}

void DownloadToCaller(Context& ctx, void* dst, const void* src, size_t bytes, const std::function<void()>& begun) {
  if (bytes == 0) return;
  if (dst == nullptr || src == nullptr) throw std::logic_error("download with a NULL buffer");
  if (bytes % 4 != 0) throw std::logic_error("download of partial words");
  constexpr size_t kSlotWords = kSlotBytes / 4;
  const size_t count = bytes / 4, launches = (count + kSlotWords - 1) / kSlotWords;
  const size_t slot_words = std::min(kSlotWords, count);
  DirectIo& io = ctx.io;
  uint64_t marks[DirectIo::kSlots] = {};
  const auto words_of = [&](size_t i) { return std::min(kSlotWords, count - i * kSlotWords); };
  ThroughRing(ctx, launches, [&](size_t i, size_t slot) {
    marks[slot] = io.NextMark();
    const uint32_t n = static_cast<uint32_t>(words_of(i));
    hipLaunchKernelGGL(CopyWords, dim3(std::min<uint32_t>(kPackWaves, (n + kPackTile - 1) / kPackTile)), dim3(kWave),
                       0, ctx.stream, static_cast<const uint32_t*>(src) + i * kSlotWords, n,
                       reinterpret_cast<uint32_t*>(io.device()) + slot * slot_words, io.device_marks(slot),
                       marks[slot]);
    CheckHip(hipGetLastError(), "CopyWords launch");
  }, [&](size_t i, size_t slot) {
    const size_t n = words_of(i);
    if (i == 0) {
      io.WaitTile(slot, 0, marks[slot], ctx.stream);
      begun();
    }
    const uint32_t* from = reinterpret_cast<const uint32_t*>(io.host()) + slot * slot_words;
    uint32_t* to = static_cast<uint32_t*>(dst) + i * kSlotWords;
    // 64 KiB at a time, on host threads from 512 KiB up
    io.TakeTiles(slot, marks[slot], ctx.stream, (n + kPackTile - 1) / kPackTile, 32, n < (size_t{1} << 17) ? 1 : 8,
                 [&](size_t first, size_t last) {
                   const size_t b = first * kPackTile, e = std::min(n, last * kPackTile);
                   std::memcpy(to + b, from + b, (e - b) * 4);
                 });
  });
}

bool UploadRows(Context& ctx, const ee_kopt_task* rows, size_t count, const KoptRowSegment* d_segments,
                size_t segments, ee_kopt_task* d_rows) {
  if (count == 0) return true;
  constexpr size_t kHeader = 256;  // the refusal flag
  constexpr size_t kSlotRows = (kSlotBytes - kHeader) / sizeof(ee_kopt_task) / kIngestRows * kIngestRows;
  static_assert(kSlotRows / kIngestRows <= DirectIo::kSlotTiles, "a slot's groups have marks");
  if (segments == 0 || segments > UINT32_MAX) throw std::logic_error("row segments");
  const size_t launches = (count + kSlotRows - 1) / kSlotRows;
  const size_t slot_bytes = kHeader + std::min(kSlotRows, (count + 63) / 64 * 64) * sizeof(ee_kopt_task);
  DirectIo& io = ctx.io;
  uint64_t marks[DirectIo::kSlots] = {};
  const auto rows_of = [&](size_t i) { return std::min(kSlotRows, count - i * kSlotRows); };
  bool refused = false;
  ThroughRing(ctx, launches, [&](size_t i, size_t slot) {
    const size_t n = rows_of(i);
    char* at = io.host() + slot * slot_bytes;
    *reinterpret_cast<uint32_t*>(at) = 0;
    // 64 KiB at a time, on host threads from 256 KiB up
    const char* from = reinterpret_cast<const char*>(rows + i * kSlotRows);
    const size_t bytes = n * sizeof(ee_kopt_task), piece = size_t{64} << 10;
    ParallelFor((bytes + piece - 1) / piece, [&](size_t p) {
      std::memcpy(at + kHeader + p * piece, from + p * piece, std::min(piece, bytes - p * piece));
    }, bytes < (size_t{256} << 10) ? 1 : 8);
    char* device = io.device() + slot * slot_bytes;
    marks[slot] = io.NextMark();
    hipLaunchKernelGGL(IngestRows, dim3(static_cast<uint32_t>((n + kIngestRows - 1) / kIngestRows)), dim3(kIngestRows), 0,
                       ctx.stream, reinterpret_cast<const uint32_t*>(device + kHeader), static_cast<uint64_t>(i * kSlotRows),
                       static_cast<uint32_t>(n), d_segments, static_cast<uint32_t>(segments),
                       reinterpret_cast<uint32_t*>(d_rows), reinterpret_cast<uint32_t*>(device), io.device_marks(slot),
                       marks[slot]);
    CheckHip(hipGetLastError(), "IngestRows launch");
  }, [&](size_t i, size_t slot) {
    const size_t groups = (rows_of(i) + kIngestRows - 1) / kIngestRows;
    for (size_t g = 0; g < groups; ++g) io.WaitTile(slot, g, marks[slot], ctx.stream);
    refused = refused || *reinterpret_cast<const uint32_t*>(io.host() + slot * slot_bytes) != 0;
  });
  return !refused;
}

bool UploadItems(Context& ctx, const std::vector<UploadItem>& items, const std::function<void()>& then) {
  constexpr size_t kHeader = 256, kMaxParts = 2048, kMaxBlocks = 1024;
  constexpr size_t kTable = kMaxParts * sizeof(UploadPart), kData = kHeader + kTable;
  // slots of 2 MiB, filled one after the other: 1.4 MB through four slots of
  // 512 KiB took 27 us more, the gaps between the launches
  constexpr size_t room = kSlotBytes - kData;
  struct Slot {
    std::vector<UploadPart> parts;
    std::vector<const char*> from;
    size_t used = 0;
  };
  std::vector<Slot> plan;
  for (const UploadItem& item : items) {
    const size_t element = item.kind == kUploadFlags ? 1 : item.kind == kUploadSpread64 ? 8 : 4;
    const size_t out = item.kind == kUploadFlags ? 4 : item.kind == kUploadWords ? 4 : item.kind == kUploadSpread32 ? 8 : 16;
    for (size_t first = 0; first < item.count;) {
      // flags grow fourfold: a part of them holds a quarter
      const size_t most = (item.kind == kUploadFlags ? kPartBytes / 4 : kPartBytes) / element;
      const size_t n = std::min(item.count - first, most), bytes = (n * element + 15) / 16 * 16;
      if (plan.empty() || plan.back().parts.size() == kMaxParts || room - plan.back().used < bytes) plan.emplace_back();
      Slot& s = plan.back();
      s.parts.push_back({reinterpret_cast<uint64_t>(item.to) + first * out, static_cast<uint32_t>(kData + s.used),
                         static_cast<uint32_t>(n), static_cast<uint32_t>(item.kind), item.limit, item.add, item.lane});
      s.from.push_back(static_cast<const char*>(item.from) + first * element);
      s.used += bytes;
      first += n;
    }
  }
  if (plan.empty()) {
    then();
    return true;
  }
  size_t longest = 0;
  for (const Slot& s : plan) longest = std::max(longest, s.used);
  const size_t slot_bytes = (kData + longest + 255) / 256 * 256;
  DirectIo& io = ctx.io;
  uint64_t marks[DirectIo::kSlots] = {};
  bool refused = false;
  const auto blocks_of = [&](size_t i) { return std::min(plan[i].parts.size(), kMaxBlocks); };
  ThroughRing(ctx, plan.size(), [&](size_t i, size_t slot) {
    const Slot& s = plan[i];
    char* at = io.host() + slot * slot_bytes;
    *reinterpret_cast<uint32_t*>(at) = 0;
    std::memcpy(at + kHeader, s.parts.data(), s.parts.size() * sizeof(UploadPart));
    // sixteen parts at a time, on host threads where there are many
    constexpr size_t kGroup = 16;
    const size_t groups = (s.parts.size() + kGroup - 1) / kGroup;
    ParallelFor(groups, [&](size_t g) {
      for (size_t p = g * kGroup, e = std::min(s.parts.size(), p + kGroup); p < e; ++p) {
        const size_t element = s.parts[p].kind == kUploadFlags ? 1 : s.parts[p].kind == kUploadSpread64 ? 8 : 4;
        std::memcpy(at + s.parts[p].at, s.from[p], s.parts[p].count * element);
      }
    }, groups < 6 ? 1 : 8);
    char* device = io.device() + slot * slot_bytes;
    marks[slot] = io.NextMark();
    hipLaunchKernelGGL(StoreParts, dim3(static_cast<uint32_t>(blocks_of(i))), dim3(kPartThreads), 0, ctx.stream,
                       reinterpret_cast<const UploadPart*>(device + kHeader), static_cast<uint32_t>(s.parts.size()),
                       device, reinterpret_cast<uint32_t*>(device), io.device_marks(slot), marks[slot]);
    CheckHip(hipGetLastError(), "StoreParts launch");
    if (i + 1 == plan.size()) then();
  }, [&](size_t i, size_t slot) {
    for (size_t b = 0; b < blocks_of(i); ++b) io.WaitTile(slot, b, marks[slot], ctx.stream);
    refused = refused || *reinterpret_cast<const uint32_t*>(io.host() + slot * slot_bytes) != 0;
  });
  return !refused;
}

}  // namespace ee
