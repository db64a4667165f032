// Host-side runtime types: device arrays, per-context caches, the context.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <chrono>
#include <cstdint>
#include <cstring>
#include <functional>
#include <string>
#include <vector>

#include "ee_internal.h"
#include "ee_pool.h"

namespace ee {

void SetLastError(const std::string& message);
const char* LastError();
// Maps the in-flight exception onto a status code (call inside catch).
ee_status StatusFromException();
double MsSince(std::chrono::steady_clock::time_point t0);
size_t Grow(size_t current, size_t required);
bool DistanceSafe(const int64_t* x, const int64_t* y, int32_t n);
// The graph content hash in two parts (ee_graph_content_hash = edges part
// continued from the prefix part).
uint64_t ContentHashPrefix(int32_t n, uint8_t distance_type, const int64_t* x, const int64_t* y);
uint64_t ContentHashEdges(uint64_t prefix, int32_t m, const int32_t* edge_u, const int32_t* edge_v,
                          const int64_t* edge_weight, const uint8_t* edge_active);
bool NearExtent(const int64_t* x, const int64_t* y, int32_t n);
KoptInstance MakeKoptInstance(uint64_t coord_base, const int64_t* x, const int64_t* y, int32_t n,
                              uint8_t distance_type);
int CountDevices();

// `bytes` of device memory on the current device or of page-locked host
// memory.  Where there is none, the memory that contexts keep for their next
// sessions and fleets is freed first.
void* NewDeviceMemory(size_t bytes);
void* NewHostMemory(size_t bytes, unsigned flags = hipHostMallocDefault);
void FreeMemory(bool host, void* ptr);

// Page-locked host staging of at least `count` elements (hipHostMalloc);
// growing discards the contents.  The pages are written once when allocated:
// the first host access to fresh page-locked memory faults every page in
// (about 0.4 ms per MB, and no less on several threads, which wait for one
// another there), which would otherwise land on the first run that fills or
// reads the staging.
template <typename T> class Pinned {
 public:
  Pinned() = default;
  ~Pinned() { Reset(); }
  Pinned(const Pinned&) = delete;
  Pinned& operator=(const Pinned&) = delete;
  Pinned(Pinned&& o) noexcept { Take(&o); }
  Pinned& operator=(Pinned&& o) noexcept {
    if (this != &o) {
      Reset();
      Take(&o);
    }
    return *this;
  }
  // With a pool, a kept block (contents left over) or a fresh one that goes
  // there when released.
  void Reserve(size_t count, MemoryPool* pool = nullptr) {
    if (count <= count_) return;
    Reset();
    size_t bytes = std::max<size_t>(count, 1) * sizeof(T);
    void* p = pool != nullptr ? pool->Take(true, bytes, &bytes) : nullptr;
    if (p == nullptr) {
      p = NewHostMemory(bytes);
      std::memset(p, 0, bytes);
    }
    ptr_ = static_cast<T*>(p);
    count_ = count;
    bytes_ = bytes;
    pool_ = pool;
  }
  T* get() { return ptr_; }
  const T* get() const { return ptr_; }
  // The address kernels use.
  T* device() const {
    void* d = nullptr;
    CheckHip(hipHostGetDevicePointer(&d, ptr_, 0), "hipHostGetDevicePointer");
    return static_cast<T*>(d);
  }
  size_t count() const { return count_; }

 private:
  void Reset() {
    if (ptr_ != nullptr && (pool_ == nullptr || !pool_->Give(true, ptr_, bytes_))) {
      static_cast<void>(hipHostFree(ptr_));
    }
    ptr_ = nullptr;
    count_ = bytes_ = 0;
    pool_ = nullptr;
  }
  void Take(Pinned* o) noexcept {
    ptr_ = o->ptr_;
    count_ = o->count_;
    bytes_ = o->bytes_;
    pool_ = o->pool_;
    o->ptr_ = nullptr;
    o->count_ = o->bytes_ = 0;
    o->pool_ = nullptr;
  }
  T* ptr_ = nullptr;
  size_t count_ = 0, bytes_ = 0;
  MemoryPool* pool_ = nullptr;
};

// Coherent, device-mapped host memory, cleared: kernels read and write it over
// the bus, and the host sees their stores while they run, as they see its.
// What one side polls while the other writes lies here.
template <typename T> class CoherentHost {
 public:
  CoherentHost() = default;
  ~CoherentHost() {
    if (host_ != nullptr) static_cast<void>(hipHostFree(host_));
  }
  CoherentHost(const CoherentHost&) = delete;
  CoherentHost& operator=(const CoherentHost&) = delete;
  void Allocate(size_t count) {
    const size_t bytes = std::max<size_t>(count, 1) * sizeof(T);
    host_ = static_cast<T*>(NewHostMemory(bytes, hipHostMallocMapped | hipHostMallocCoherent));
    count_ = count;
    std::memset(static_cast<void*>(host_), 0, bytes);
    void* d = nullptr;
    CheckHip(hipHostGetDevicePointer(&d, host_, 0), "hipHostGetDevicePointer");
    device_ = static_cast<T*>(d);
  }
  T* host() { return host_; }
  const T* host() const { return host_; }
  T* device() { return device_; }
  size_t count() const { return count_; }

 private:
  T* host_ = nullptr;
  T* device_ = nullptr;
  size_t count_ = 0;
};

// Owning device allocation of `count` elements of T on one device.
template <typename T> class DeviceArray {
 public:
  DeviceArray() = default;
  DeviceArray(size_t count, int device) { Allocate(count, device); }
  ~DeviceArray() { Reset(); }
  DeviceArray(const DeviceArray&) = delete;
  DeviceArray& operator=(const DeviceArray&) = delete;
  DeviceArray(DeviceArray&& o) noexcept { Take(&o); }
  DeviceArray& operator=(DeviceArray&& o) noexcept {
    if (this != &o) {
      Reset();
      Take(&o);
    }
    return *this;
  }

  // With a pool, a kept block or a fresh one that goes there when released.
  void Allocate(size_t count, int device, MemoryPool* pool = nullptr) {
    Reset();
    if (count == 0) return;
    if (count > SIZE_MAX / sizeof(T)) throw std::overflow_error("device allocation size overflows");
    CheckHip(hipSetDevice(device), "hipSetDevice");
    size_t bytes = count * sizeof(T);
    void* p = pool != nullptr ? pool->Take(false, bytes, &bytes) : nullptr;
    if (p == nullptr) p = NewDeviceMemory(bytes);
    ptr_ = static_cast<T*>(p);
    count_ = count;
    held_ = bytes;
    device_ = device;
    pool_ = pool;
  }

  void Upload(const T* host, size_t count, hipStream_t stream) { UploadAt(0, host, count, stream); }
  void UploadAt(size_t offset, const T* host, size_t count, hipStream_t stream) {
    if (count == 0) return;
    if (offset > count_ || count > count_ - offset) throw std::logic_error("H2D beyond device buffer");
    CheckHip(hipMemcpyAsync(ptr_ + offset, host, count * sizeof(T), hipMemcpyHostToDevice, stream),
             "hipMemcpyAsync H2D");
  }
  void Download(T* host, size_t count, hipStream_t stream) const {
    DownloadAt(0, host, count, stream);
  }
  void DownloadAt(size_t offset, T* host, size_t count, hipStream_t stream) const {
    if (count == 0) return;
    if (offset > count_ || count > count_ - offset) throw std::logic_error("D2H beyond device buffer");
    CheckHip(hipMemcpyAsync(host, ptr_ + offset, count * sizeof(T), hipMemcpyDeviceToHost, stream),
             "hipMemcpyAsync D2H");
  }

  T* get() { return ptr_; }
  const T* get() const { return ptr_; }
  size_t count() const { return count_; }
  uint64_t bytes() const { return static_cast<uint64_t>(count_) * sizeof(T); }

 private:
  void Reset() noexcept {
    if (ptr_ != nullptr && (pool_ == nullptr || !pool_->Give(false, ptr_, held_))) {
      static_cast<void>(hipSetDevice(device_));
      static_cast<void>(hipFree(ptr_));
    }
    ptr_ = nullptr;
    count_ = held_ = 0;
    device_ = -1;
    pool_ = nullptr;
  }
  void Take(DeviceArray* o) noexcept {
    ptr_ = o->ptr_;
    count_ = o->count_;
    held_ = o->held_;
    device_ = o->device_;
    pool_ = o->pool_;
    o->ptr_ = nullptr;
    o->count_ = o->held_ = 0;
    o->device_ = -1;
    o->pool_ = nullptr;
  }

  T* ptr_ = nullptr;
  size_t count_ = 0, held_ = 0;  // elements, and bytes of the block
  int device_ = -1;
  MemoryPool* pool_ = nullptr;
};

struct JvCache {
  bool valid = false;
  int32_t dimension = 0;
  uint8_t distance_type = 0;
  bool near = false;  // NearExtent of the cached coordinates
  // exact static key (host copies)
  std::vector<int64_t> x, y, edge_weight;
  std::vector<int32_t> edge_u, edge_v;
  // static: 8m + 8m + 16n bytes
  DeviceArray<int2> d_uv;
  DeviceArray<int64_t> d_weight;
  DeviceArray<longlong2> d_xy;
  // dynamic: 4m + 4(n+1) + 4A + 4A + 4m bytes
  DeviceArray<int32_t> d_active;
  DeviceArray<int32_t> d_row_offsets;
  DeviceArray<int32_t> d_neighbors;
  DeviceArray<int32_t> d_edge_ids;
  DeviceArray<int32_t> d_witnesses;
};

struct KoptCache {
  struct TemplateEntry {
    bool valid = false;
    uint64_t hash = 0;
    std::vector<ee_endpoint_matching> table;
  };
  bool snapshot_valid = false;
  int32_t dimension = 0;
  uint8_t distance_type = 0;
  bool near = false;  // NearExtent of the snapshot
  std::vector<int64_t> x, y;
  DeviceArray<longlong2> d_xy;
  std::array<TemplateEntry, 3> templates;
  std::array<KoptPlan, 3> host_plans;
  DeviceArray<KoptPlan> d_plans;
  DeviceArray<ee_kopt_task> d_tasks;  // rows made without an evaluation
  // largest evaluation through the ring so far, grown as the buffers are
  size_t task_room = 0, cell_room = 0;
  bool Reserve(size_t tasks, size_t cells);
};

// Page-locked host memory that kernels read and write in place, in up to
// kSlots slots: while one is on the device the host fills or empties
// another.  One per context, used by its thread between synchronisations.
//
// A kernel marks each tile's output with the launch's mark, a number no
// earlier launch used, once the output is in host memory; the host polls the
// marks and takes the output while the kernel runs, so both lie in coherent
// memory.  The marks have an area of their own, so that a word there is never
// anything but a mark.
class DirectIo {
 public:
  static constexpr size_t kSlots = 2;
  static constexpr size_t kSlotTiles = 4096;
  // The ring is made with the context and keeps its size: fresh page-locked
  // memory costs about 0.4 ms per MB, which a first large call would pay (a
  // ring of 2 MiB that grew to 4 made that of 4,096 k = 5 rows 1.5 ms, it is
  // 0.5 ms now).  Half of it per slot; slots of 1 MiB in 2 took a third longer
  // on large results (batch cells 400 -> 520 us).
  static constexpr size_t kBytes = size_t{4} << 20, kSlotBytes = kBytes / kSlots;
  void Create();
  char* host() { return mem_.host(); }
  char* device() { return mem_.device(); }
  uint64_t* device_marks(size_t slot) { return marks_.device() + slot * kSlotTiles; }
  uint64_t bytes() const { return mem_.count() + marks_.count() * sizeof(uint64_t); }
  uint64_t NextMark() { return ++mark_; }
  // Returns once tile `tile` of the slot's launch, on `stream`, carries
  // `mark`; throws if the stream has ended without it.  Any host thread.
  void WaitTile(size_t slot, size_t tile, uint64_t mark, hipStream_t stream) const;
  // Waits for the tiles of a launch that writes `count` cells in transfer
  // form, tile_cells to a tile, and expands them to int64 as they arrive.
  void TakeCells(size_t slot, uint64_t mark, hipStream_t stream, const uint32_t* lo, const uint8_t* hi,
                 size_t count, size_t tile_cells, int64_t* cells) const;
  // Waits for tiles [0, tiles) in groups, in order, and calls take(first,
  // last) for each group as it arrives, on up to `threads` host threads.
  void TakeTiles(size_t slot, uint64_t mark, hipStream_t stream, size_t tiles, size_t group, unsigned threads,
                 const std::function<void(size_t, size_t)>& take) const;

 private:
  CoherentHost<char> mem_;
  CoherentHost<uint64_t> marks_;
  uint64_t mark_ = 0;
};

// Device copy of one tour context for the deletion-set producer, kept while
// the caller passes the same tour, edge costs and selectable positions.
struct KoptCursorCache {
  bool valid = false;
  int32_t nodes = 0;  // node count of the snapshots the tour was checked for
  std::vector<int32_t> tour;
  std::vector<int64_t> edge_costs;
  std::vector<uint64_t> selectable;
  DeviceArray<int32_t> d_tour;
  DeviceArray<int64_t> d_edge_costs;
  DeviceArray<uint64_t> d_selectable;
  DeviceArray<uint32_t> d_positions;
  DeviceArray<uint32_t> d_status;  // bit 0: some deleted cost overflowed int64
};

// Device copy of one snapshot's coordinates and active CSR for the HT reply
// enumerations, kept while the caller passes the same arrays, plus their
// growing workspaces.
struct HtCache {
  bool valid = false;
  int32_t dimension = 0;
  uint8_t distance_type = 0;
  std::vector<int64_t> x, y;
  std::vector<int32_t> row_offsets, neighbors;
  std::vector<uint8_t> active;  // the snapshot passed the HT checks with these flags
  bool near = false;            // NearExtent: the FP64 distance path applies
  uint32_t max_degree = 0;
  DeviceArray<longlong2> d_xy;
  DeviceArray<int32_t> d_row_offsets, d_neighbors;
  DeviceArray<int32_t> d_items;      // centers, or (endpoint, internal) task pairs
  DeviceArray<uint64_t> d_counts;    // per item
  DeviceArray<uint64_t> d_offsets;   // per item + 1
  DeviceArray<unsigned long long> d_chunk_sums;  // reply totals per scan chunk of centers
  DeviceArray<int32_t> d_replies;    // triples or pairs, exactly the last call's replies
  int last_kind = 0;                 // last completed call: 1 Hamilton, 2 end replies
  uint64_t last_total = 0;           // its reply count
  // Hamilton replies as verdict bits: per center `stride` words in host
  // memory, or with stride 0 as many as its row needs, bit p set where pair p
  // survives.  The call under way uses the other buffer, so that a refused
  // one leaves the last one's replies.
  struct Verdicts {
    // the centers, then their reply counts, then (stride 0) the first word of
    // each wavefront's centers
    Pinned<int32_t> centers;
    Pinned<uint64_t> bits;
    size_t count = 0, stride = 0, per_wave = 4;
    size_t group = 256;                 // centers of a group of the host's work
    std::vector<uint64_t> group_first;  // replies before each group of centers, and in all
    const uint32_t* first_words() const { return reinterpret_cast<const uint32_t*>(centers.get()) + 2 * count; }
  };
  Verdicts verdicts[2];
  int current = 0;
  bool last_bits = false;            // the last Hamilton replies are verdicts[current]
};

struct Context {
  MemoryPool pool{FreeMemory};  // released last
  explicit Context(int requested_device);
  ~Context();
  Context(const Context&) = delete;
  Context& operator=(const Context&) = delete;

  void Activate() const;
  void Sync() const;
  // A second stream, for snapshot hashes beside the context's work; kept.
  hipStream_t HashStream();

  int device = -1;
  int compute_units = 0;
  hipStream_t stream = nullptr;
  hipStream_t hash_stream = nullptr;
  hipEvent_t ev_begin = nullptr, ev_end = nullptr;
  uint32_t jv_grid = 0;  // 0: one wavefront per edge slot or pair of slots
  uint32_t jv_edges_per_wave = 2;  // 2: pairs of edge slots on 32-lane halves
  KoptTuning kopt_tuning;
  JvCache jv;
  KoptCache kopt;
  KoptCursorCache cursor;
  HtCache ht;
  DirectIo io;
};

// Copies `bytes` (whole 4-byte words) of device memory to caller memory and
// waits, after the work queued before it on the context's stream: a kernel
// writes the words into the context's ring and host threads copy them out
// as they arrive.  `begun` runs when the first have, with all of that work done.
void DownloadToCaller(Context& ctx, void* dst, const void* src, size_t bytes,
                      const std::function<void()>& begun = [] {});

// The rows from row_begin to the next entry's are checked as k-opt task rows
// of this k on n nodes.
struct KoptRowSegment {
  uint64_t row_begin;
  uint32_t k;
  int32_t n;
};

// Copies task rows [0, count) into device memory through the context's ring,
// checking them on the way as ValidateTasks does, against `segments` entries
// on the device (and one more, where the last ends).  Returns once all rows
// are in place; false if some row is refused.
bool UploadRows(Context& ctx, const ee_kopt_task* rows, size_t count, const KoptRowSegment* d_segments,
                size_t segments, ee_kopt_task* d_rows);

// Device-resident cost cells [0, count) into caller memory, after the work
// queued before on the context's stream, in transfer form through the
// context's ring.  wide: some instance's coordinates are not near.
void DownloadCells(Context& ctx, const int64_t* d_cells, size_t count, bool wide, int64_t* cells);

// An array on its way to the device: `count` elements of `from`, caller or
// host memory, to the device address `to`.
enum UploadKind : uint32_t {
  kUploadWords,     // 32-bit words plus `add`; with a limit, words below it
  kUploadFlags,     // bytes to 32-bit 0 or 1
  kUploadSpread32,  // 32-bit words plus `add` to component `lane` of pairs
  kUploadSpread64,  // 64-bit words to component `lane` of pairs
};
struct UploadItem {
  UploadKind kind;
  void* to;
  const void* from;
  size_t count;
  uint32_t limit = 0, add = 0, lane = 0;
};
// Copies the items to the device through the context's ring, in few launches
// and no copy command; `then` runs once the last part is queued, with the
// arrays in place for work it queues on the context's stream.  Returns once
// the arrays are in place; false if some word reached its limit (the device
// then holds `add` alone in its place).
bool UploadItems(Context& ctx, const std::vector<UploadItem>& items, const std::function<void()>& then = [] {});

// Elements [offset, offset + count) of a device array into caller memory, as
// DownloadToCaller.
template <typename T>
void DownloadRange(Context& ctx, const DeviceArray<T>& a, size_t offset, size_t count, T* host) {
  if (count == 0) return;
  if (offset > a.count() || count > a.count() - offset) throw std::logic_error("D2H beyond device buffer");
  DownloadToCaller(ctx, host, a.get() + offset, count * sizeof(T));
}

// The deletion-set producer of ee_cursor.hip: the number of sets of size k
// the reference cursor enumerates over `selectable_count` positions, the
// checks of a tour view, and the row-building launch (sets [first, first +
// count) into d_tasks and, when not NULL, their sorted positions into
// d_positions; bit 0 of *d_status is set where a deleted cost overflows).
uint64_t CursorSetCount(uint32_t selectable_count, uint32_t k);
void CheckCursorTour(const ee_tour_view* tour, int32_t n);
void LaunchCursorRows(const int32_t* d_tour, const int64_t* d_edge_costs, const uint64_t* d_selectable,
                      uint32_t tour_length, uint32_t selectable_count, uint32_t k, uint64_t first,
                      uint32_t count, ee_kopt_task* d_tasks, uint32_t* d_positions, uint32_t* d_status,
                      hipStream_t stream);

// Looks up (once per device, with that device current) the device address of
// the no-allocation scratch array of ee_kopt_eval_costs_noalloc.
void InitNoAllocScratch(int device);

std::vector<ee_endpoint_matching> CanonicalTemplates(uint32_t k, uint64_t* hash);
KoptPlan BuildPlan(uint32_t k, const ee_endpoint_matching* templates, uint32_t count);
void ValidateTasks(int32_t n, uint32_t k, const ee_kopt_task* tasks, size_t count);
// Null arrays, dimensions, distance type and integer coordinates of a view.
void CheckGraphView(const ee_graph_view* g);

// The task rows of one plain evaluation: the caller's (which must pass
// ValidateTasks), or, with `tasks` null, those of the deletion sets from rank
// `first` of a checked tour context on the device, delivered to out_tasks
// and out_positions where these are not null.
struct KoptRows {
  const ee_kopt_task* tasks = nullptr;
  KoptCursor cursor{};
  uint64_t first = 0;
  ee_kopt_task* out_tasks = nullptr;
  uint32_t* out_positions = nullptr;
};

// The plain synchronous k-opt evaluation (snapshot and template caches, rows
// and output through the context's ring).  Exactly one of `costs`
// (task_count x template_count cells) and `masks` (task_count x
// ceil(template_count / 32) improving-template words) is non-null, masks only
// with made rows.
void EvalKoptRows(Context& ctx, const int64_t* x, const int64_t* y, int32_t n, uint8_t type, uint32_t k,
                  const ee_endpoint_matching* templates, uint32_t template_count, uint64_t generator_hash,
                  size_t task_count, const KoptRows& rows, int64_t* costs, uint32_t* masks, ee_kopt_usage* usage);

}  // namespace ee
