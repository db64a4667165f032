// Results that reach the caller through page-locked host memory which kernels
// write in place: the ring itself (DirectIo), the host's side of taking
// cells out of it, and the download of device-resident cells.
#include <algorithm>
#include <stdexcept>

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

}  // namespace

void DirectIo::Reserve(size_t bytes) {
  const auto device_of = [](void* host) {
    void* d = nullptr;
    CheckHip(hipHostGetDevicePointer(&d, host, 0), "hipHostGetDevicePointer");
    return d;
  };
  if (marks_.count() == 0) {
    marks_.Reserve(kSlots * kSlotTiles);
    device_marks_ = static_cast<uint64_t*>(device_of(marks_.get()));
  }
  for (const size_t size : kSizes) {
    if (bytes <= size) {
      bytes = size;
      break;
    }
  }
  if (bytes <= mem_.count()) return;
  mem_.Reserve(bytes);
  device_ = static_cast<char*>(device_of(mem_.get()));
}

void DirectIo::WaitTile(size_t slot, size_t tile, uint64_t mark, hipStream_t stream) const {
  const uint64_t* at = marks_.get() + slot * kSlotTiles + tile;
  const auto seen = [&] { return __atomic_load_n(at, __ATOMIC_ACQUIRE) == mark; };
  for (uint64_t polls = 1; !seen(); ++polls) {
    // a kernel that ended, or failed, without the mark: look now and then
    if (polls % (uint64_t{1} << 20) != 0) continue;
    const hipError_t status = hipStreamQuery(stream);
    if (status == hipErrorNotReady || seen()) continue;
    CheckHip(status, "kernel writing to host memory");
    throw std::runtime_error("a kernel ended without marking a tile");
  }
}

void DirectIo::TakeTiles(size_t slot, uint64_t mark, hipStream_t stream, size_t tiles, size_t group,
                         unsigned threads, const std::function<void(size_t, size_t)>& take) const {
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
// memory in a context's first large download; launches alternating on two
// streams, with slots of 1 or 2 MiB, measured slower (290-360 us).
void DownloadCells(Context& ctx, const int64_t* d_cells, size_t count, bool wide, int64_t* cells) {
  if (count == 0) return;
  if (d_cells == nullptr || cells == nullptr) throw std::logic_error("download with a NULL buffer");
  // whole tiles, 2 MiB to a slot: the ring's second size
  constexpr size_t kSlotBytes = size_t{2} << 20;
  static_assert(kSlotBytes / 4 / kPackTile <= DirectIo::kSlotTiles, "a slot's tiles have marks");
  const size_t cell_bytes = wide ? 5 : 4;
  const size_t slot_cells = kSlotBytes / cell_bytes / kPackTile * kPackTile;
  const size_t launches = (count + slot_cells - 1) / slot_cells;
  const size_t slots = std::min<size_t>(launches, DirectIo::kSlots);
  const size_t plane = launches == 1 ? (count + 255) / 256 * 256 : slot_cells;
  const size_t slot_bytes = plane * cell_bytes;
  DirectIo& io = ctx.io;
  io.Reserve(slots * slot_bytes);
  uint64_t marks[DirectIo::kSlots] = {};
  const auto cells_of = [&](size_t i) { return std::min(slot_cells, count - i * slot_cells); };
  const auto launch = [&](size_t i) {
    const size_t slot = i % slots;
    char* at = io.device() + slot * slot_bytes;
    uint8_t* hi = reinterpret_cast<uint8_t*>(at + plane * 4);
    marks[slot] = io.NextMark();
    const uint32_t n = static_cast<uint32_t>(cells_of(i));
    const uint32_t grid = std::min<uint32_t>(kPackWaves, (n + kPackTile - 1) / kPackTile);
    hipLaunchKernelGGL((wide ? PackCells<true> : PackCells<false>), dim3(grid), dim3(kWave), 0, ctx.stream,
                       d_cells + i * slot_cells, n, reinterpret_cast<uint32_t*>(at), hi, io.device_marks(slot),
                       marks[slot]);
    CheckHip(hipGetLastError(), "PackCells launch");
  };
  try {
    for (size_t i = 0; i < slots; ++i) launch(i);
    for (size_t i = 0; i < launches; ++i) {
      const size_t slot = i % slots;
      const char* at = io.host() + slot * slot_bytes;
      io.TakeCells(slot, marks[slot], ctx.stream, reinterpret_cast<const uint32_t*>(at),
                   wide ? reinterpret_cast<const uint8_t*>(at + plane * 4) : nullptr, cells_of(i), kPackTile,
                   cells + i * slot_cells);
      if (i + slots < launches) launch(i + slots);
    }
  } catch (...) {
    static_cast<void>(hipStreamSynchronize(ctx.stream));  // the ring is free again
    throw;
  }
}

}  // namespace ee
