// Host runtime of the gfx950 backend: device selection, per-context
// device-resident caches and the C entry points of the reference-shaped
// (synchronous, host buffers in and out) paths.  Host-only helpers (errors,
// validation, the template generator) are in ee_host.cpp.
//
// Cache semantics follow the reference so that callers observe the same hit
// flags and resident byte counts:
//   JV    (src/cuda/jv_cuda.cu:360-478): the static part (coordinates, edge
//         endpoints, edge weights) is keyed by an exact element-wise compare;
//         the dynamic part (active flags, CSR, witnesses) lives in buffers
//         that grow to max(required, 2 x current).  Resident bytes are
//         24m + 20n + 4 + 8A on an exact first fit.
//   k-opt (src/cuda/kopt_cost.cu:205-295): coordinates keyed by exact
//         compare of (dimension, distance type, x, y); templates keyed per k
//         by (generator hash, content).  Rows and cells pass through the
//         context's ring, so the workspace flag is that of the reference's
//         buffers, followed by their sizes alone, and the resident bytes are
//         the device copies and the ring.
#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstring>
#include <memory>
#include <new>
#include <string>
#include <vector>

#include "ee_exact.h"
#include "ee_internal.h"
#include "ee_jvhost.h"
#include "ee_runtime.h"

namespace ee {

void CheckHip(hipError_t status, const char* what) {
  if (status != hipSuccess) {
    throw std::runtime_error(std::string(what) + ": " + hipGetErrorString(status));
  }
}

namespace {

// `allocate` until it succeeds or has failed without the contexts' kept memory.
template <typename F> void* NewMemory(size_t bytes, const char* what, F&& allocate) {
  void* p = nullptr;
  hipError_t status = allocate(&p);
  if (status == hipErrorOutOfMemory) {
    MemoryPool::ReleaseAll();
    static_cast<void>(hipGetLastError());  // a later launch's check is not to find the failure
    status = allocate(&p);
  }
  if (status == hipSuccess) return p;
  static_cast<void>(hipGetLastError());
  throw std::runtime_error(std::string(what) + "(" + std::to_string(bytes) + " bytes): " + hipGetErrorString(status));
}

}  // namespace

void* NewDeviceMemory(size_t bytes) {
  return NewMemory(bytes, "hipMalloc", [&](void** p) { return hipMalloc(p, bytes); });
}

void* NewHostMemory(size_t bytes, unsigned flags) {
  return NewMemory(bytes, "hipHostMalloc", [&](void** p) { return hipHostMalloc(p, bytes, flags); });
}

void FreeMemory(bool host, void* ptr) { static_cast<void>(host ? hipHostFree(ptr) : hipFree(ptr)); }

KoptInstance MakeKoptInstance(uint64_t coord_base, const int64_t* x, const int64_t* y, int32_t n,
                              uint8_t distance_type) {
  KoptInstance inst{};
  inst.coord_base = coord_base;
  inst.n = static_cast<uint32_t>(n);
  inst.distance_type = distance_type;
  inst.near = NearExtent(x, y, n) ? 1 : 0;
  return inst;
}

// ------------------------------------------------------------------ device
int CountDevices() {
  int count = 0;
  if (hipGetDeviceCount(&count) != hipSuccess) return 0;
  return count;
}

int SelectDevice(int requested) {
  const int count = CountDevices();
  if (count <= 0) throw Unavailable("no visible HIP device");
  if (requested >= 0) {
    if (requested >= count) throw Unavailable("requested HIP device ordinal is not visible");
    CheckHip(hipSetDevice(requested), "hipSetDevice");
    return requested;
  }
  int best = -1;
  size_t best_free = 0;
  for (int d = 0; d < count; ++d) {
    if (hipSetDevice(d) != hipSuccess) continue;
    size_t free_bytes = 0, total_bytes = 0;
    if (hipMemGetInfo(&free_bytes, &total_bytes) == hipSuccess &&
        (best < 0 || free_bytes > best_free)) {
      best = d;
      best_free = free_bytes;
    }
  }
  if (best < 0) throw Unavailable("no HIP device could report its free memory");
  CheckHip(hipSetDevice(best), "hipSetDevice");
  return best;
}

Context::Context(int requested) {
  device = SelectDevice(requested);
  InitNoAllocScratch(device);
  CheckHip(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking), "hipStreamCreate");
  CheckHip(hipEventCreate(&ev_begin), "hipEventCreate");
  CheckHip(hipEventCreate(&ev_end), "hipEventCreate");
  io.Create();
  hipDeviceProp_t prop{};
  if (hipGetDeviceProperties(&prop, device) == hipSuccess) {
    compute_units = prop.multiProcessorCount;
  }
}

Context::~Context() {
  static_cast<void>(hipSetDevice(device));
  static_cast<void>(hipStreamSynchronize(stream));
  jv = JvCache{};
  kopt = KoptCache{};
  static_cast<void>(hipEventDestroy(ev_begin));
  static_cast<void>(hipEventDestroy(ev_end));
  if (hash_stream != nullptr) {
    static_cast<void>(hipStreamSynchronize(hash_stream));
    static_cast<void>(hipStreamDestroy(hash_stream));
  }
  static_cast<void>(hipStreamDestroy(stream));
}

hipStream_t Context::HashStream() {
  if (hash_stream == nullptr) {
    CheckHip(hipStreamCreateWithFlags(&hash_stream, hipStreamNonBlocking), "hipStreamCreate");
  }
  return hash_stream;
}

void Context::Activate() const { CheckHip(hipSetDevice(device), "hipSetDevice"); }

void Context::Sync() const { CheckHip(hipStreamSynchronize(stream), "hipStreamSynchronize"); }

// ---------------------------------------------------------------------- JV
namespace {

void ValidateStaticJv(const ee_graph_view& g) {
  const int32_t n = g.dimension, m = g.edge_count;
  for (int32_t e = 0; e < m; ++e) {
    if (g.edge_u[e] < 0 || g.edge_u[e] >= n || g.edge_v[e] < 0 || g.edge_v[e] >= n) {
      throw std::invalid_argument("JV edge endpoint out of range");
    }
    if (g.edge_weight[e] < 0 || g.edge_weight[e] > (int64_t{1} << 62)) {
      throw std::invalid_argument("JV edge weight outside [0, 2^62]");
    }
  }
  if (!DistanceSafe(g.x, g.y, n)) {
    throw std::runtime_error("HIP JV needs integer coordinates whose squared distances fit uint64");
  }
}

// Row offsets that start at 0 and do not decrease; returns the entry count.
size_t CheckRowOffsets(const ee_graph_view& g) {
  if (g.row_offsets[0] != 0) throw std::invalid_argument("CSR row_offsets[0] must be 0");
  bool ordered = true;
  for (int32_t v = 0; v < g.dimension; ++v) ordered &= g.row_offsets[v + 1] >= g.row_offsets[v];
  if (!ordered) throw std::invalid_argument("CSR row_offsets must be non-decreasing");
  return static_cast<size_t>(g.row_offsets[g.dimension]);
}

// The first CSR entry that the device refused.
[[noreturn]] void RefuseCsr(const ee_graph_view& g, size_t adjacency) {
  for (size_t i = 0; i < adjacency; ++i) {
    if (g.neighbors[i] < 0 || g.neighbors[i] >= g.dimension) {
      throw std::invalid_argument("CSR neighbour out of range");
    }
    if (g.csr_edge_ids[i] < 0 || g.csr_edge_ids[i] >= g.edge_count) {
      throw std::invalid_argument("CSR edge id out of range");
    }
  }
  throw std::logic_error("the device refused CSR entries that the host accepts");
}

// Whether the cached static part has this snapshot's sizes and first entries.
bool StaticLooksAlike(const JvCache& c, const ee_graph_view& g) {
  const size_t n = static_cast<size_t>(g.dimension), m = static_cast<size_t>(g.edge_count);
  return c.valid && c.dimension == g.dimension && c.distance_type == g.distance_type && c.x.size() == n &&
         c.edge_u.size() == m && std::memcmp(c.x.data(), g.x, std::min<size_t>(n, 64) * 8) == 0 &&
         std::memcmp(c.edge_weight.data(), g.edge_weight, std::min<size_t>(m, 64) * 8) == 0;
}

bool StaticMatches(const JvCache& c, const ee_graph_view& g) {
  if (!StaticLooksAlike(c, g)) return false;
  const size_t n = static_cast<size_t>(g.dimension), m = static_cast<size_t>(g.edge_count);
  const struct {
    const void *cached, *given;
    size_t bytes;
  } arrays[] = {{c.x.data(), g.x, n * 8},
                {c.y.data(), g.y, n * 8},
                {c.edge_u.data(), g.edge_u, m * 4},
                {c.edge_v.data(), g.edge_v, m * 4},
                {c.edge_weight.data(), g.edge_weight, m * 8}};
  std::atomic<bool> equal{true};
  // the arrays on host threads of their own where they are large
  ParallelFor(5, [&](size_t i) {
    if (std::memcmp(arrays[i].cached, arrays[i].given, arrays[i].bytes) != 0) equal = false;
  }, m < 16384 ? 1 : 5);
  return equal;
}

}  // namespace

uint64_t JvResidentBytes(const JvCache& c) {
  return c.d_uv.bytes() + c.d_weight.bytes() + c.d_xy.bytes() + c.d_active.bytes() +
         c.d_row_offsets.bytes() + c.d_neighbors.bytes() + c.d_edge_ids.bytes() +
         c.d_witnesses.bytes();
}

// PrepareStaticGraph (jv_cuda.cu:384-430).  Returns true on a cache hit.
bool PrepareJvStatic(Context& ctx, const ee_graph_view& g) {
  JvCache& c = ctx.jv;
  if (StaticMatches(c, g)) return true;
  ValidateStaticJv(g);
  const size_t n = static_cast<size_t>(g.dimension), m = static_cast<size_t>(g.edge_count);
  DeviceArray<int2> d_uv(m, ctx.device);
  DeviceArray<int64_t> d_weight(m, ctx.device);
  DeviceArray<longlong2> d_xy(n, ctx.device);
  UploadItems(ctx, {{kUploadSpread32, d_uv.get(), g.edge_u, m, 0, 0, 0},
                    {kUploadSpread32, d_uv.get(), g.edge_v, m, 0, 0, 1},
                    {kUploadWords, d_weight.get(), g.edge_weight, 2 * m},
                    {kUploadSpread64, d_xy.get(), g.x, n, 0, 0, 0},
                    {kUploadSpread64, d_xy.get(), g.y, n, 0, 0, 1}});
  c.d_uv = std::move(d_uv);
  c.d_weight = std::move(d_weight);
  c.d_xy = std::move(d_xy);
  c.x.assign(g.x, g.x + n);
  c.y.assign(g.y, g.y + n);
  c.edge_u.assign(g.edge_u, g.edge_u + m);
  c.edge_v.assign(g.edge_v, g.edge_v + m);
  c.edge_weight.assign(g.edge_weight, g.edge_weight + m);
  c.dimension = g.dimension;
  c.distance_type = g.distance_type;
  c.near = NearExtent(g.x, g.y, g.dimension);
  c.valid = true;
  return false;
}

// PrepareWorkspace (jv_cuda.cu:442-470).  Returns true on a cache hit.
bool PrepareJvWorkspace(Context& ctx, size_t n, size_t m, size_t adjacency) {
  JvCache& c = ctx.jv;
  const bool hit = c.d_active.count() >= m && c.d_row_offsets.count() >= n + 1 &&
                   c.d_neighbors.count() >= adjacency && c.d_edge_ids.count() >= adjacency &&
                   c.d_witnesses.count() >= m;
  if (c.d_active.count() < m) c.d_active.Allocate(Grow(c.d_active.count(), m), ctx.device);
  if (c.d_row_offsets.count() < n + 1) {
    c.d_row_offsets.Allocate(Grow(c.d_row_offsets.count(), n + 1), ctx.device);
  }
  if (c.d_neighbors.count() < adjacency) {
    c.d_neighbors.Allocate(Grow(c.d_neighbors.count(), adjacency), ctx.device);
  }
  if (c.d_edge_ids.count() < adjacency) {
    c.d_edge_ids.Allocate(Grow(c.d_edge_ids.count(), adjacency), ctx.device);
  }
  if (c.d_witnesses.count() < m) c.d_witnesses.Allocate(Grow(c.d_witnesses.count(), m), ctx.device);
  return hit;
}

void CheckGraphView(const ee_graph_view* g) {
  if (g == nullptr) throw std::invalid_argument("graph view is NULL");
  if (g->dimension <= 0 || g->edge_count < 0) throw std::invalid_argument("bad graph dimensions");
  if (g->distance_type != EE_EUC_2D && g->distance_type != EE_CEIL_2D) {
    throw std::invalid_argument("unsupported distance type");
  }
  if (g->integer_coordinates == 0) {
    throw std::runtime_error("HIP JV supports integer coordinates only");
  }
  if (g->x == nullptr || g->y == nullptr || g->row_offsets == nullptr ||
      (g->edge_count > 0 && (g->edge_u == nullptr || g->edge_v == nullptr ||
                             g->edge_weight == nullptr || g->edge_active == nullptr)) ||
      (g->row_offsets[g->dimension] > 0 && (g->neighbors == nullptr || g->csr_edge_ids == nullptr))) {
    throw std::invalid_argument("graph view has a NULL array");
  }
}

JvLaunch JvArgs(Context& ctx, int32_t m, int type) {
  JvCache& c = ctx.jv;
  JvLaunch a{};
  a.edge_count = m;
  a.distance_type = type;
  a.near = c.near ? 1 : 0;
  a.edge_uv = c.d_uv.get();
  a.edge_weight = c.d_weight.get();
  a.edge_active = c.d_active.get();
  a.row_offsets = c.d_row_offsets.get();
  a.neighbors = c.d_neighbors.get();
  a.csr_edge_ids = c.d_edge_ids.get();
  a.xy = c.d_xy.get();
  a.witnesses = c.d_witnesses.get();
  a.one_per_wave = ctx.jv_edges_per_wave == 1 ? 1 : 0;
  return a;
}

// FindJvCandidatesCuda (jv_cuda.cu:488-566) without the final compaction.
// The dynamic arrays pass through the context's ring to a kernel that checks
// and widens them, the JV kernel queued behind it; while both run the host
// compares the static part with the resident copy.  On a 15,000-node 10-NN
// graph (1.4 MB of dynamic arrays, 53 us of JV kernel) 260 -> 154 us.
void FindJvCandidates(Context& ctx, const ee_graph_view& g, int32_t* witnesses, ee_jv_usage* usage) {
  ee_jv_usage u{};
  ctx.Activate();
  const int32_t m = g.edge_count;
  if (m == 0) {
    if (usage) *usage = u;
    return;
  }
  JvCache& c = ctx.jv;
  const size_t adjacency = CheckRowOffsets(g);
  // a snapshot that only looks like the resident one gets a second pass, once
  // it has been made resident
  bool workspace_hit = true;
  for (bool likely = StaticLooksAlike(c, g);; likely = false) {
    bool static_hit = likely;
    if (!likely) {
      for (size_t i = 0; i < adjacency; ++i) {
        if (static_cast<uint32_t>(g.neighbors[i]) >= static_cast<uint32_t>(g.dimension) ||
            static_cast<uint32_t>(g.csr_edge_ids[i]) >= static_cast<uint32_t>(m)) {
          RefuseCsr(g, adjacency);
        }
      }
      static_hit = PrepareJvStatic(ctx, g);
    }
    workspace_hit =
        PrepareJvWorkspace(ctx, static_cast<size_t>(g.dimension), static_cast<size_t>(m), adjacency) && workspace_hit;
    auto t0 = std::chrono::steady_clock::now();
    const bool accepted = UploadItems(
        ctx,
        {{kUploadFlags, c.d_active.get(), g.edge_active, static_cast<size_t>(m)},
         {kUploadWords, c.d_row_offsets.get(), g.row_offsets, static_cast<size_t>(g.dimension) + 1},
         {kUploadWords, c.d_neighbors.get(), g.neighbors, adjacency, static_cast<uint32_t>(g.dimension)},
         {kUploadWords, c.d_edge_ids.get(), g.csr_edge_ids, adjacency, static_cast<uint32_t>(m)}},
        [&] { LaunchJv(JvArgs(ctx, m, g.distance_type), ctx.jv_grid, ctx.stream); });
    u.h2d_ms = MsSince(t0);
    t0 = std::chrono::steady_clock::now();
    if (!accepted) {
      ctx.Sync();
      RefuseCsr(g, adjacency);
    }
    if (likely && !StaticMatches(c, g)) {
      ctx.Sync();
      continue;
    }
    u.static_hit = static_hit ? 1 : 0;
    u.workspace_hit = workspace_hit ? 1 : 0;
    u.resident_bytes = JvResidentBytes(c);
    DownloadToCaller(ctx, witnesses, c.d_witnesses.get(), static_cast<size_t>(m) * sizeof(int32_t), [&] {
      u.kernel_ms = MsSince(t0);
      t0 = std::chrono::steady_clock::now();
    });
    u.d2h_ms = MsSince(t0);
    break;
  }
  if (usage) *usage = u;
}

// ------------------------------------------------------------------- k-opt
// Device memory of the caches and the page-locked ring the kernels work in.
uint64_t KoptResidentBytes(const Context& ctx) {
  const KoptCache& c = ctx.kopt;
  return c.d_xy.bytes() + c.d_plans.bytes() + c.d_tasks.bytes() + ctx.io.bytes();
}

// Whether an evaluation of this size found room, with the growth rule of the
// other caches (the rows and cells themselves pass through the bounded ring).
bool KoptCache::Reserve(size_t tasks, size_t cells) {
  const bool hit = task_room >= tasks && cell_room >= cells;
  task_room = Grow(task_room, tasks);
  cell_room = Grow(cell_room, cells);
  return hit;
}

namespace {

// Which caches held what an evaluation needs.
struct KoptHits {
  bool snapshot, templates;
};

bool SnapshotMatches(const KoptCache& c, const int64_t* x, const int64_t* y, int32_t n, uint8_t type) {
  const size_t nn = static_cast<size_t>(n);
  return c.snapshot_valid && c.dimension == n && c.distance_type == type && c.x.size() == nn &&
         std::memcmp(c.x.data(), x, nn * 8) == 0 && std::memcmp(c.y.data(), y, nn * 8) == 0;
}

bool TemplatesMatch(const KoptCache& c, uint32_t k, const ee_endpoint_matching* templates, uint32_t template_count,
                    uint64_t generator_hash) {
  const KoptCache::TemplateEntry& entry = c.templates[k - 3];
  return entry.valid && entry.hash == generator_hash && entry.table.size() == template_count &&
         std::memcmp(entry.table.data(), templates, template_count * sizeof(ee_endpoint_matching)) == 0;
}

void CheckKoptInputs(const int64_t* x, const int64_t* y, int32_t n, uint8_t type, uint32_t k,
                     const ee_endpoint_matching* templates, uint32_t template_count, size_t task_count) {
  if (k < 3 || k > 5 || templates == nullptr || template_count == 0) {
    throw std::invalid_argument("HIP k-opt reconnect table is invalid");
  }
  if (x == nullptr || y == nullptr || n <= 0 || (type != EE_EUC_2D && type != EE_CEIL_2D)) {
    throw std::invalid_argument("HIP k-opt coordinates are invalid");
  }
  if (task_count > SIZE_MAX / template_count) throw std::overflow_error("k-opt cell count overflows");
}

KoptHits PrepareKoptCaches(Context& ctx, const int64_t* x, const int64_t* y, int32_t n, uint8_t type, uint32_t k,
                           const ee_endpoint_matching* templates, uint32_t template_count,
                           uint64_t generator_hash) {
  KoptCache& c = ctx.kopt;
  KoptHits hits{};
  hits.snapshot = SnapshotMatches(c, x, y, n, type);
  if (!hits.snapshot) {
    if (!DistanceSafe(x, y, n)) {
      throw std::invalid_argument("k-opt cost needs distance-safe integer coordinates");
    }
    const size_t nn = static_cast<size_t>(n);
    DeviceArray<longlong2> d_xy(nn, ctx.device);
    UploadItems(ctx, {{kUploadSpread64, d_xy.get(), x, nn, 0, 0, 0}, {kUploadSpread64, d_xy.get(), y, nn, 0, 0, 1}});
    c.d_xy = std::move(d_xy);
    c.x.assign(x, x + nn);
    c.y.assign(y, y + nn);
    c.dimension = n;
    c.distance_type = type;
    c.near = NearExtent(x, y, n);
    c.snapshot_valid = true;
  }
  // one plan slot per k
  hits.templates = TemplatesMatch(c, k, templates, template_count, generator_hash);
  if (!hits.templates) {
    const KoptPlan plan = BuildPlan(k, templates, template_count);
    if (c.d_plans.count() < 3) c.d_plans.Allocate(3, ctx.device);
    c.host_plans[k - 3] = plan;
    c.d_plans.UploadAt(k - 3, &c.host_plans[k - 3], 1, ctx.stream);
    ctx.Sync();
    KoptCache::TemplateEntry& entry = c.templates[k - 3];
    entry.table.assign(templates, templates + template_count);
    entry.hash = generator_hash;
    entry.valid = true;
  }
  return hits;
}

// The rows of one evaluation, cut into launches that pass through the
// context's page-locked ring.  A launch's slot holds an overflow flag, its
// task rows (the caller's, or made ones on their way out) and positions, where
// the caller wants them, and
// its output: mask words, or cells in transfer form (low words, then high
// bytes on instances that are not near).
struct KoptChunks {
  // One launch where everything fits the ring, slots of half of it otherwise:
  // 16,384 k = 4 rows (2.4 MB) take 108 us in one launch and 138 in two.  A
  // tile is 0.3 MB at most.  kPads: the parts of a slot start on 256 bytes.
  static constexpr size_t kPads = 5 * 256;

  // The bytes of a row in each part of a slot; a part may be empty.
  KoptChunks(size_t rows, uint32_t tile_rows, size_t task_bytes, size_t position_bytes, size_t low_bytes,
             size_t high_bytes)
      : rows_(rows) {
    const size_t per_row = task_bytes + position_bytes + low_bytes + high_bytes;
    const size_t tiles = (rows + tile_rows - 1) / tile_rows, tile_bytes = tile_rows * per_row;
    const bool whole = tiles <= DirectIo::kSlotTiles && tiles * tile_bytes + kPads <= DirectIo::kBytes;
    const size_t room = whole ? DirectIo::kBytes : DirectIo::kSlotBytes;
    const size_t fit = std::min<size_t>((room - kPads) / tile_bytes, DirectIo::kSlotTiles);
    if (fit == 0) throw std::logic_error("a k-opt tile exceeds the ring");
    count = (rows + fit * tile_rows - 1) / (fit * tile_rows);
    // launches of equal size, whole tiles each
    const size_t even = (rows + count - 1) / count;
    chunk_rows = std::min(rows, (even + tile_rows - 1) / tile_rows * tile_rows);
    count = (rows + chunk_rows - 1) / chunk_rows;
    positions_off = rows_off + Align256(chunk_rows * task_bytes);
    lo_off = positions_off + Align256(chunk_rows * position_bytes);
    hi_off = lo_off + Align256(chunk_rows * low_bytes);
    slot_bytes = hi_off + Align256(chunk_rows * high_bytes);
    slots = std::min<size_t>(count, DirectIo::kSlots);
  }
  static size_t Align256(size_t v) { return (v + 255) & ~size_t{255}; }
  size_t First(size_t chunk) const { return chunk * chunk_rows; }
  size_t Rows(size_t chunk) const { return std::min(chunk_rows, rows_ - First(chunk)); }

  size_t count = 0, chunk_rows = 0, slots = 0;
  static constexpr size_t rows_off = 256;
  size_t positions_off = 0, lo_off = 0, hi_off = 0, slot_bytes = 0;

 private:
  size_t rows_;
};

// body(first, end) over [0, n), in four parts on host threads from
// `serial_below` up.
template <typename F> void InParts(size_t n, size_t serial_below, F&& body) {
  constexpr size_t kParts = 4;
  if (n < serial_below) {
    body(size_t{0}, n);
    return;
  }
  ParallelFor(kParts, [&](size_t p) { body(n * p / kParts, n * (p + 1) / kParts); }, static_cast<unsigned>(kParts));
}

// Whether the caches look up to date, from their sizes and a sample of the
// coordinates.
bool LooksResident(const KoptCache& c, const int64_t* x, const int64_t* y, int32_t n, uint8_t type, uint32_t k,
                   const ee_endpoint_matching* templates, uint32_t template_count, uint64_t generator_hash) {
  if (!c.snapshot_valid || c.dimension != n || c.distance_type != type ||
      !TemplatesMatch(c, k, templates, template_count, generator_hash)) {
    return false;
  }
  const size_t sample = std::min<size_t>(static_cast<size_t>(n), 64) * sizeof(int64_t);
  return std::memcmp(c.x.data(), x, sample) == 0 && std::memcmp(c.y.data(), y, sample) == 0;
}

// Tiles of the launches that write to host memory.  Where cells go out, PCIe
// bounds them, so few wavefronts take several small tiles each: they keep
// the link busy and their first tiles arrive early, so the host expands while
// the rest crosses.  A k = 5 block of 4,096 rows takes 120 us (rows 4, 192
// wavefronts), 126 with 256 and 158 with one tile per wavefront, whose tiles
// all end together; k = 3 and 4, with less output per row, measured best at
// 256.  Masks are small, so the wavefronts' own chain bounds them: one short
// tile each (4,096 k = 5 sets: 59 us with 8 rows, 61 with 16, 64 with 4).
KoptTuning DirectTuning(uint32_t k, bool masks) {
  constexpr uint32_t kCellRows[3] = {64, 16, 4}, kMaskRows[3] = {32, 8, 8};
  KoptTuning t;
  std::copy_n(masks ? kMaskRows : kCellRows, 3, t.rows_per_tile);
  t.block = 64;
  t.grid = masks ? 0 : k == 5 ? 192 : 256;
  return t;
}

// The kernel reads the task rows from page-locked host memory, or makes them
// itself, and writes its output (and made rows) back there, cells in transfer
// form, tile by tile.  So a call has no copy command and no wait for the
// stream, and half the bytes of int64 cells cross PCIe (56 GB/s here, which
// bounds a block: 61 us for 4,096 k = 5 rows).  Host threads take tiles into
// the caller's buffers as their marks arrive.  Against an upload, a launch
// and a download with a wait each: one k = 5 row 56 -> 19 us, 1,237 k = 4
// rows 63 -> 34 us, 4,096 k = 5 rows 293 -> 121 us, 1,501 wide k = 5 rows
// 163 -> 83 us, 4,096 made k = 5 rows with their masks 125 -> 60 us.
// `check` runs on the host while the first launches are on the device; false
// drops their output and returns false, with nothing delivered.
bool RunDirect(Context& ctx, int32_t n, uint8_t type, uint32_t k, uint32_t template_count, size_t task_count,
               const KoptRows& rows, int64_t* costs, uint32_t* masks, const std::function<bool()>& check,
               ee_kopt_usage* usage) {
  ee_kopt_usage u{};
  KoptCache& c = ctx.kopt;
  const bool made = rows.tasks == nullptr, wide = !c.near && masks == nullptr;
  const uint32_t mask_words = (template_count + 31) / 32;
  const KoptTuning tuning = DirectTuning(k, masks != nullptr);
  const uint32_t tile_rows = tuning.rows_per_tile[k - 3];
  const KoptChunks chunks(task_count, tile_rows, made && rows.out_tasks == nullptr ? 0 : sizeof(ee_kopt_task),
                          rows.out_positions == nullptr ? 0 : 4 * k, 4 * (masks ? mask_words : template_count),
                          wide ? template_count : 0);
  DirectIo& io = ctx.io;

  KoptInstance inst{};
  inst.n = static_cast<uint32_t>(n);
  inst.distance_type = type;
  inst.near = c.near ? 1 : 0;
  bool present[3] = {false, false, false};
  present[k - 3] = true;
  uint64_t marks[DirectIo::kSlots] = {};
  const auto slot_of = [&](size_t chunk) { return chunk % chunks.slots * chunks.slot_bytes; };
  const auto launch = [&](size_t chunk) {
    const size_t count = chunks.Rows(chunk), slot = chunk % chunks.slots, at = slot_of(chunk);
    char* const device = io.device() + at;
    KoptSegment segment{0, k, 0, count, 0, 0, tile_rows, 0};
    KoptLaunch a{};
    KoptAssignTiles(&segment, 1, &inst, c.host_plans.data(), tuning, nullptr, &a);
    if (a.inline_count == 0) throw std::logic_error("a one-segment k-opt launch needs its inline table");
    a.xy = c.d_xy.get();
    a.plans = c.d_plans.get();
    if (made) {
      *reinterpret_cast<uint32_t*>(io.host() + at) = 0;
      a.row_status = reinterpret_cast<uint32_t*>(device);
      a.cursor = rows.cursor;
      a.row_first = rows.first + chunks.First(chunk);
      if (rows.out_tasks != nullptr) a.made_tasks = reinterpret_cast<ee_kopt_task*>(device + chunks.rows_off);
      if (rows.out_positions != nullptr) {
        a.made_positions = reinterpret_cast<uint32_t*>(device + chunks.positions_off);
      }
    } else {
      const ee_kopt_task* from = rows.tasks + chunks.First(chunk);
      ee_kopt_task* staged = reinterpret_cast<ee_kopt_task*>(io.host() + at + chunks.rows_off);
      InParts(count, 8192, [&](size_t b, size_t e) { std::memcpy(staged + b, from + b, (e - b) * sizeof(*from)); });
      a.tasks = reinterpret_cast<const ee_kopt_task*>(device + chunks.rows_off);
      a.bound_nodes = static_cast<uint32_t>(n);
    }
    if (masks) {
      a.masks = reinterpret_cast<uint32_t*>(device + chunks.lo_off);
      a.mask_words = mask_words;
    } else {
      a.packed_lo = reinterpret_cast<uint32_t*>(device + chunks.lo_off);
      a.packed_hi = wide ? reinterpret_cast<uint8_t*>(device + chunks.hi_off) : nullptr;
    }
    a.marks = io.device_marks(slot);
    a.mark = marks[slot] = io.NextMark();
    const size_t shared = KoptPrepareLayout(&a, c.host_plans.data(), present, tuning, c.near);
    LaunchKopt(a, tuning, shared, ctx.stream);
  };
  // made rows, their positions and mask words of tiles [first, last)
  const auto take_rows = [&](size_t chunk, size_t first, size_t last) {
    const size_t b = first * tile_rows, count = std::min(chunks.Rows(chunk), last * tile_rows) - b;
    const size_t row = chunks.First(chunk) + b;
    const char* at = io.host() + slot_of(chunk);
    if (rows.out_tasks != nullptr) {
      std::memcpy(rows.out_tasks + row, at + chunks.rows_off + b * sizeof(ee_kopt_task), count * sizeof(ee_kopt_task));
    }
    if (rows.out_positions != nullptr) {
      std::memcpy(rows.out_positions + row * k, at + chunks.positions_off + b * 4 * k, count * 4 * k);
    }
    if (masks != nullptr) {
      std::memcpy(masks + row * mask_words, at + chunks.lo_off + b * 4 * mask_words, count * 4 * mask_words);
    }
  };
  bool overflow = false;
  try {
    auto t0 = std::chrono::steady_clock::now();
    for (size_t i = 0; i < chunks.slots; ++i) launch(i);
    u.h2d_ms = MsSince(t0);
    t0 = std::chrono::steady_clock::now();
    if (!check()) {
      ctx.Sync();
      return false;
    }
    for (size_t i = 0; i < chunks.count; ++i) {
      const size_t slot = i % chunks.slots, count = chunks.Rows(i);
      io.WaitTile(slot, 0, marks[slot], ctx.stream);
      if (i == 0) {
        u.kernel_ms = MsSince(t0);
        t0 = std::chrono::steady_clock::now();
      }
      const char* from = io.host() + slot_of(i);
      if (masks == nullptr) {
        io.TakeCells(slot, marks[slot], ctx.stream, reinterpret_cast<const uint32_t*>(from + chunks.lo_off),
                     wide ? reinterpret_cast<const uint8_t*>(from + chunks.hi_off) : nullptr,
                     count * template_count, tile_rows * template_count, costs + chunks.First(i) * template_count);
      }
      if (made) {
        const size_t tiles = (count + tile_rows - 1) / tile_rows;
        // 256 rows at a time on this thread: a block's rows and words are a few
        // hundred KB, and four threads took 20 us where one takes 13
        io.TakeTiles(slot, marks[slot], ctx.stream, tiles, std::max<size_t>(1, 256 / tile_rows), 1,
                     [&](size_t first, size_t last) { take_rows(i, first, last); });
        overflow = overflow || *reinterpret_cast<const uint32_t*>(from) != 0;
      }
      if (i + chunks.slots < chunks.count) launch(i + chunks.slots);
    }
    u.d2h_ms = MsSince(t0);
  } catch (...) {
    static_cast<void>(hipStreamSynchronize(ctx.stream));  // the ring is free again
    throw;
  }
  if (overflow) throw std::runtime_error("k-opt cursor: deleted cost sum overflows int64_t");
  u.snapshot_hit = u.template_hit = 1;
  const size_t out_cells = masks ? (task_count * mask_words + 1) / 2 : task_count * template_count;
  u.workspace_hit = c.Reserve(task_count, out_cells) ? 1 : 0;
  u.resident_bytes = KoptResidentBytes(ctx);
  if (usage) *usage = u;
  return true;
}

}  // namespace

void EvalKoptRows(Context& ctx, const int64_t* x, const int64_t* y, int32_t n, uint8_t type, uint32_t k,
                  const ee_endpoint_matching* templates, uint32_t template_count, uint64_t generator_hash,
                  size_t task_count, const KoptRows& rows, int64_t* costs, uint32_t* masks, ee_kopt_usage* usage) {
  ctx.Activate();
  if ((costs == nullptr) == (masks == nullptr)) {
    throw std::invalid_argument("HIP k-opt needs exactly one of costs and masks");
  }
  KoptCache& c = ctx.kopt;
  const auto validate = [&] {
    if (rows.tasks != nullptr) ValidateTasks(n, k, rows.tasks, task_count);
  };
  // Where the caches look up to date, the launch goes out first, and the
  // full comparison with them and the check of the rows run beside it: the
  // kernel clamps node ids to the cached snapshot, and nothing reaches the
  // caller before both passed.  Otherwise rows and caches come first.
  const bool inputs = k >= 3 && k <= 5 && templates != nullptr && template_count > 0 && x != nullptr &&
                      y != nullptr && n > 0 && task_count <= SIZE_MAX / template_count;
  if (inputs && LooksResident(c, x, y, n, type, k, templates, template_count, generator_hash)) {
    const auto check = [&] {
      if (!SnapshotMatches(c, x, y, n, type)) return false;
      if (rows.tasks == nullptr) return true;
      try {
        InParts(task_count, 1024, [&](size_t b, size_t e) { ValidateTasks(n, k, rows.tasks + b, e - b); });
      } catch (const std::invalid_argument&) {
        validate();  // the first refused row's message
        throw;
      }
      return true;
    };
    if (RunDirect(ctx, n, type, k, template_count, task_count, rows, costs, masks, check, usage)) return;
  }
  validate();
  CheckKoptInputs(x, y, n, type, k, templates, template_count, task_count);
  const KoptHits hits = PrepareKoptCaches(ctx, x, y, n, type, k, templates, template_count, generator_hash);
  RunDirect(ctx, n, type, k, template_count, task_count, rows, costs, masks, [] { return true; }, usage);
  if (usage) {
    usage->snapshot_hit = hits.snapshot ? 1 : 0;
    usage->template_hit = hits.templates ? 1 : 0;
  }
}

void EvalKoptCosts(Context& ctx, const int64_t* x, const int64_t* y, int32_t n, uint8_t type,
                   uint32_t k, const ee_endpoint_matching* templates, uint32_t template_count,
                   uint64_t generator_hash, const ee_kopt_task* tasks, size_t task_count,
                   int64_t* costs, ee_kopt_usage* usage) {
  ctx.Activate();
  if (task_count == 0) {
    if (usage) *usage = ee_kopt_usage{};
    return;
  }
  if (tasks == nullptr || costs == nullptr) throw std::invalid_argument("HIP k-opt NULL buffer");
  KoptRows rows;
  rows.tasks = tasks;
  EvalKoptRows(ctx, x, y, n, type, k, templates, template_count, generator_hash, task_count, rows, costs, nullptr,
               usage);
}

}  // namespace ee

// =================================================================== C ABI
using ee::StatusFromException;

extern "C" {

int ee_device_count(void) { return ee::CountDevices(); }

ee_status ee_backend_available(int device, char* reason, size_t reason_capacity) {
  std::string why;
  const int count = ee::CountDevices();
  if (count <= 0) {
    why = "no visible HIP device";
  } else if (device >= count) {
    why = "requested HIP device ordinal is not visible";
  }
  if (reason && reason_capacity > 0) {
    const size_t len = std::min(why.size(), reason_capacity - 1);
    std::memcpy(reason, why.data(), len);
    reason[len] = '\0';
  }
  if (!why.empty()) {
    ee::SetLastError(why);
    return EE_ERR_UNAVAILABLE;
  }
  return EE_OK;
}

ee_status ee_ctx_create(int device, ee_ctx** out) {
  try {
    if (out == nullptr) throw std::invalid_argument("ee_ctx_create: out is NULL");
    *out = nullptr;
    *out = reinterpret_cast<ee_ctx*>(new ee::Context(device));
    return EE_OK;
  } catch (...) {
    return StatusFromException();
  }
}

void ee_ctx_destroy(ee_ctx* ctx) { delete reinterpret_cast<ee::Context*>(ctx); }

int ee_ctx_device(const ee_ctx* ctx) {
  return ctx ? reinterpret_cast<const ee::Context*>(ctx)->device : -1;
}

ee_status ee_ctx_set_jv_edges_per_wave(ee_ctx* ctx, uint32_t edges) {
  try {
    if (ctx == nullptr) throw std::invalid_argument("context is NULL");
    if (edges != 1 && edges != 2) throw std::invalid_argument("JV edges per wavefront must be 1 or 2");
    reinterpret_cast<ee::Context*>(ctx)->jv_edges_per_wave = edges;
    return EE_OK;
  } catch (...) {
    return StatusFromException();
  }
}

ee_status ee_jv_find_candidates(ee_ctx* ctx, const ee_graph_view* graph, int32_t* witnesses,
                                ee_jv_usage* usage) {
  try {
    if (ctx == nullptr) throw std::invalid_argument("context is NULL");
    ee::CheckGraphView(graph);
    if (graph->edge_count > 0 && witnesses == nullptr) {
      throw std::invalid_argument("witness buffer is NULL");
    }
    ee::FindJvCandidates(*reinterpret_cast<ee::Context*>(ctx), *graph, witnesses, usage);
    return EE_OK;
  } catch (...) {
    return StatusFromException();
  }
}

ee_status ee_jv_clear_cache(ee_ctx* ctx) {
  try {
    if (ctx == nullptr) throw std::invalid_argument("context is NULL");
    auto* c = reinterpret_cast<ee::Context*>(ctx);
    c->Activate();
    c->Sync();
    c->jv = ee::JvCache{};
    return EE_OK;
  } catch (...) {
    return StatusFromException();
  }
}

ee_status ee_kopt_eval_costs(ee_ctx* ctx, const int64_t* x, const int64_t* y, int32_t dimension,
                             uint8_t distance_type, uint32_t k,
                             const ee_endpoint_matching* templates, uint32_t template_count,
                             uint64_t generator_hash, const ee_kopt_task* tasks,
                             size_t task_count, int64_t* costs, ee_kopt_usage* usage) {
  try {
    if (ctx == nullptr) throw std::invalid_argument("context is NULL");
    ee::EvalKoptCosts(*reinterpret_cast<ee::Context*>(ctx), x, y, dimension, distance_type, k,
                      templates, template_count, generator_hash, tasks, task_count, costs, usage);
    return EE_OK;
  } catch (...) {
    return StatusFromException();
  }
}

ee_status ee_kopt_clear_cache(ee_ctx* ctx) {
  try {
    if (ctx == nullptr) throw std::invalid_argument("context is NULL");
    auto* c = reinterpret_cast<ee::Context*>(ctx);
    c->Activate();
    c->Sync();
    c->kopt = ee::KoptCache{};
    return EE_OK;
  } catch (...) {
    return StatusFromException();
  }
}

}  // extern "C"
