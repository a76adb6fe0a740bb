// Host side of the TBE lookup: plan construction (tra_tbe_create) and launch
// (tra_tbe_forward), plus the small library-level entry points.
#include <algorithm>
#include <atomic>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <tuple>
#include <memory>
#include <mutex>
#include <string>

#include "tbe_lookup_impl.h"

namespace tra {

static thread_local char g_err[512] = "";

void set_error(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
}

int hip_fail(hipError_t e, const char* what) {
  set_error("%s: %s", what, hipGetErrorString(e));
  return TRA_ERR_HIP;
}

// Explicit specializations live in tbe_lookup_<dtype>.hip.
template <>
int launch_lookup<TRA_INT8>(const LookupArgs&, int, const LaunchParams&, hipStream_t);
template <>
int launch_lookup<TRA_INT4>(const LookupArgs&, int, const LaunchParams&, hipStream_t);
template <>
int launch_lookup<TRA_INT2>(const LookupArgs&, int, const LaunchParams&, hipStream_t);
template <>
int launch_lookup<TRA_INT8 + kSplitHeader>(const LookupArgs&, int, const LaunchParams&, hipStream_t);
template <>
int launch_lookup<TRA_INT4 + kSplitHeader>(const LookupArgs&, int, const LaunchParams&, hipStream_t);
template <>
int launch_lookup<TRA_INT2 + kSplitHeader>(const LookupArgs&, int, const LaunchParams&, hipStream_t);
template <>
int launch_lookup<TRA_FP16>(const LookupArgs&, int, const LaunchParams&, hipStream_t);
template <>
int launch_lookup<TRA_FP32>(const LookupArgs&, int, const LaunchParams&, hipStream_t);
// ... and in tbe_group_<id type>_<weight mode>.hip.
template <>
void launch_group<int32_t, kUnweighted>(const GroupArgs&, const GroupPositions*, const GroupLaunch&, bool, hipStream_t);
template <>
void launch_group<int32_t, kPerSample>(const GroupArgs&, const GroupPositions*, const GroupLaunch&, bool, hipStream_t);
template <>
void launch_group<int32_t, kByPosition>(const GroupArgs&, const GroupPositions*, const GroupLaunch&, bool, hipStream_t);
template <>
void launch_group<int64_t, kUnweighted>(const GroupArgs&, const GroupPositions*, const GroupLaunch&, bool, hipStream_t);
template <>
void launch_group<int64_t, kPerSample>(const GroupArgs&, const GroupPositions*, const GroupLaunch&, bool, hipStream_t);
template <>
void launch_group<int64_t, kByPosition>(const GroupArgs&, const GroupPositions*, const GroupLaunch&, bool, hipStream_t);

// Launch shape of the pooled kernels.  Defaults are chosen from the problem
// size when a plan first sees a (batch size, route) pair and are remembered in
// the plan.  The tuning overrides (environment TRA_BALANCED, TRA_WINDOW,
// TRA_UNROLL, TRA_LDS, TRA_XCD, TRA_COST_FLOOR, TRA_FUSED_SCAN, TRA_CB) are read
// once, when the library is loaded; tra_set_tuning changes them afterwards
// (experiments and tests).  A forward never reads the environment.
struct Tuning {
  int balanced;  // 1: tbe_pooled_cu_kernel, one block per CU-sized window of bags
  int window;    // bags per block (0: derive from the problem size)
  int unroll;    // window kernel
  int lds_bytes;
};

struct Overrides {
  int balanced = -1;    // -1: decide by size
  int window = -1;      // <= 0: derive
  int unroll = -1;
  int lds = -1;
  int xcd = -1;         // 0: no XCD remap of the window kernel's blocks
  int cost_floor = -1;
  int fused_scan = -1;  // -1: decide by size
  int cb = -1;          // smaller lane chunks (plan creation)
  int fork = -1;        // 0: the launches of a multi-class call stay on the caller's stream
};

static int env_int(const char* name, int fallback) {
  const char* v = getenv(name);
  return v && *v ? atoi(v) : fallback;
}

static Overrides overrides_from_env() {
  Overrides o;
  o.balanced = env_int("TRA_BALANCED", -1);
  o.window = env_int("TRA_WINDOW", -1);
  o.unroll = env_int("TRA_UNROLL", -1);
  o.lds = env_int("TRA_LDS", -1);
  o.xcd = env_int("TRA_XCD", -1);
  o.cost_floor = env_int("TRA_COST_FLOOR", -1);
  o.fused_scan = env_int("TRA_FUSED_SCAN", -1);
  o.cb = env_int("TRA_CB", -1);
  o.fork = env_int("TRA_FORK", -1);
  return o;
}

static Overrides g_ovr = overrides_from_env();
// Bumped by tra_set_tuning: launch geometry remembered under an older value is recomputed.
static std::atomic<int> g_ovr_gen{0};

constexpr int kFewBags = 8;  // per compute unit

// How the sixteen-lane kernel takes the columns of a row from `off` on: the first slice of them.
struct GroupShape {
  int ne;  // columns per lane
  int lanes_log2;
  int cols;
};

// A row is one slice where sixteen lanes can hold it (16 columns of an integer row each, 16 bytes of others), else
// where 32 or 64 can; only what 64 cannot hold is cut.  The walk over the ids and its trip count belong to a wave,
// so two or one bags in it are better for wide rows than four bags of each of several slices.  Graph replays of 8
// tables, ~20 ids a bag, us, slices of sixteen lanes / this: int8 100 columns, 6400 bags 13.3 / 11.9; int8 512, 512 bags
// 10.9 / 10.2, 6400 bags 28.4 / 24.0; int8 300, 512 bags 10.5 / 8.3; int4 512, 6400 bags of 45 45.2 / 38.7; fp16 512
// 55.6 / 50.3; fp32 256 53.3 / 48.8.  What is cut starts with a slice of half the most columns a lane can hold (int8 300:
// 64 lanes of 4 columns 7.5 and 45.3 us at 512 bags of 20 and 6400 of 45, 32 of 8 8.3 and 43.1, 16 of 16 10.5 and 39.5).
// few: the call has few bags (kFewBags).  int8 rows that need 16 columns of each of sixteen lanes go by 32 lanes then,
// for a shorter chain per bag (us, 16 / 32 lanes: 192 columns, 128 bags of 3 5.4 / 4.7, of 20 8.9 / 7.2, 2048 bags
// 5.9 / 5.4 and 10.2 / 9.0, but 3072 bags 6.0 / 6.3 and 10.4 / 10.6, 6400 bags of up to 45 16.5 / 18.5).
static GroupShape group_shape(int dtype, int dim, int off, bool few) {
  const int bits = bits_of(dtype), left = dim - off;
  const int most = dtype == TRA_FP32 ? 4 : dtype == TRA_FP16 ? 8 : 16;
  for (int log2 = few && dtype == TRA_INT8 && dim > 128 ? 5 : 4; log2 <= 6; ++log2) {
    // (more than sixteen lanes, or a part of the row: with a header, the kernel's split kinds, whole dwords a lane)
    const int least = header_bytes(dtype) != 0 && (log2 > 4 || off > 0) ? 32 / bits : 1;
    for (int ne = least; ne <= most; ne *= 2)
      if (left % ne == 0 && ne << log2 >= left) return {ne, log2, left};
  }
  int cols = most << 6;
  while (cols > left) cols /= 2;
  int ne = most / 2, log2 = 4;
  while (ne << 6 < cols) ne *= 2;
  while (ne << log2 < cols) ++log2;
  return {ne, log2, cols};
}

// balanced: what the call's size says (the overrides come first).
static Tuning choose_tuning(bool balanced) {
  Tuning t;
  t.balanced = balanced ? 1 : 0;
  t.window = 0;
  t.unroll = 4;
  t.lds_bytes = 0;  // (the window kernel's own 107 KB leave a compute unit one block; an override has 53 KB of room)
  if (g_ovr.balanced >= 0) t.balanced = g_ovr.balanced;
  if (g_ovr.window >= 0) t.window = g_ovr.window;
  if (g_ovr.unroll >= 0) t.unroll = g_ovr.unroll;
  if (g_ovr.lds >= 0) t.lds_bytes = g_ovr.lds;
  if (t.window > kMaxWindow) t.window = kMaxWindow;
  if (t.window < 0) t.window = 0;
  return t;
}

// ... and in tbe_multi_<id type>_<weight mode>.hip.
template <>
void launch_multi<int32_t, kUnweighted>(const MultiArgs&, int, int, bool, hipStream_t);
template <>
void launch_multi<int32_t, kPerSample>(const MultiArgs&, int, int, bool, hipStream_t);
template <>
void launch_multi<int32_t, kByPosition>(const MultiArgs&, int, int, bool, hipStream_t);
template <>
void launch_multi<int64_t, kUnweighted>(const MultiArgs&, int, int, bool, hipStream_t);
template <>
void launch_multi<int64_t, kPerSample>(const MultiArgs&, int, int, bool, hipStream_t);
template <>
void launch_multi<int64_t, kByPosition>(const MultiArgs&, int, int, bool, hipStream_t);

}  // namespace tra

// Scratch of tra_tbe_forward_lengths_static: the offsets array and the scan's
// tile sums of one call.  One copy per GPU, held until the process ends.
constexpr int64_t kStaticScratchBytes = 8 << 20;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

namespace tra {

// Device address of `scratch` on each GPU (the array's name is only a host-side
// handle).  Resolved when the first plan is created on a device, that device
// being current.
constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mutex;
static void* g_scratch_ptr[kMaxDevices] = {};

static int resolve_static_scratch(int device) {
  if (device < 0 || device >= kMaxDevices) {
    set_error("device index %d is beyond the %d devices the library tracks", device, kMaxDevices);
    return TRA_ERR_TOO_LARGE;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (g_scratch_ptr[device] != nullptr) return TRA_OK;
  void* p = nullptr;
  hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
  if (e != hipSuccess) return hip_fail(e, "hipGetSymbolAddress(scratch)");
  if (p == nullptr || (uintptr_t)p % 256 != 0) {
    set_error("static scratch resolved to %p (expected a 256-byte aligned device address)", p);
    return TRA_ERR_HIP;
  }
  g_scratch_ptr[device] = p;
  return TRA_OK;
}

}  // namespace tra

using namespace tra;

// Launch geometry of one launch class for one (batch size, route).
struct ClassGeometry {
  SubClass sub[kMaxSub];
  int n_sub = 0;
  int grid = 0;
  int xcd_blocks = 0;
  int xcd_count = 1;
};

// Launch geometry of all classes in one launch.
struct MultiGeometry {
  int n_sub = 0;
  int grid = 0;
  int xcd_blocks = 0;
  int xcd_count = 1;
  SubClass sub[kMaxMultiSub];
};

// What a plan remembers about a call shape it has seen: the route and, per
// launch class, the grid and windows.  Recomputed when the tuning overrides change.
struct Geometry {
  int32_t batch_size = -1;
  int64_t nobag_indices = -1;  // sequence lookups size their grid by the id count
  int balanced = 0;
  int nobag = 0;
  int gen = -1;
  Tuning tune{};
  std::vector<ClassGeometry> cls;
  int multi = 0;
  MultiGeometry all;     // balanced calls in one launch
  GroupLaunch group{};  // pooled calls that are not balanced: windows (the grid is per launch)
};

constexpr int kGeometrySlots = 8;

// A call of at least this many launch classes runs them on two streams (see forward_impl).  The
// fork and the join cost about 10 us of dependencies between queues, every pair of neighbouring
// launches gains a few: with launches of 25 - 30 us each, two classes lose 11 %, three and four
// are even (-1 %, +0.5 %), five gain 8 %, seven (of about 50 us) 9 %.
constexpr size_t kForkMinClasses = 5;

struct GroupSlices {
  std::vector<GroupSlice> host;
  GroupSlice* dev = nullptr;
};

struct tra_tbe {
  int device = 0;
  int num_cus = 256;  // compute units of the device (hipDeviceProp_t::multiProcessorCount)
  int num_xcd = 8;    // accelerator dies, each with its own L2 (hipDeviceAttributeNumberOfXccs)
  int num_features = 0;
  bool same_dim = true;  // every feature has the same dim (required for POOL_NONE)
  int dim0 = 0;
  int max_key_pos = 0;          // largest feature position among the input keys
  size_t max_class_feats = 0;   // features of the largest launch class
  std::vector<FeatureDesc> slices;  // host copy
  FeatureDesc* slices_dev = nullptr;
  int32_t* feats_dev = nullptr;  // all classes' slice lists, concatenated
  FeatureDesc* cdescs_dev = nullptr;  // the descriptors in that order: cdescs[i] = slices[feats[i]]
  unsigned long long* err_dev = nullptr;
  void* static_scratch = nullptr;  // this device's copy of the library's static scratch array
  std::atomic<int> bad_to_row0{0};  // 1: ids outside their table pool row 0 (tra_tbe_set_bounds_check_mode)
  // The second stream of a multi-class call (plans of kForkMinClasses launch classes or more; default
  // priority), the events that fork it from and join it to the caller's stream, and which of the
  // two streams every class is launched on, in launch order (largest class first).
  std::mutex fork_mutex;
  hipStream_t side = nullptr;
  hipEvent_t ev_fork = nullptr;
  hipEvent_t ev_join = nullptr;
  std::vector<int> launch_order;     // class indices
  std::vector<uint8_t> on_side;      // per class index: 1 = launched on `side`
  std::vector<LaunchClass> classes;
  std::vector<LookupArgs> base_args;  // per class: everything a call does not change
  // All slices for one launch of windows, where that can be (else empty): lane chunks of at most 16 accumulators,
  // sorted by kind and lanes per row; at most kMaxPos of them, and kMaxMultiSub sub-classes.
  std::vector<int32_t> multi_feats;
  std::vector<int32_t> multi_lprs;
  std::vector<int32_t> multi_kinds;
  bool multi_aligned_fp16 = true;  // every slice's first output column is 16-byte aligned
  bool multi_aligned_fp32 = true;
  FeatureDesc* multi_descs_dev = nullptr;
  LookupArgs multi_base;
  // Column slices for the sixteen-lane kernel, in feature order.
  GroupSlices group_slices[2];  // [1]: calls of few bags (kFewBags), where they differ
  std::mutex geo_mutex;
  std::shared_ptr<const Geometry> geo[kGeometrySlots];
  int geo_next = 0;
};

extern "C" {

int tra_version(void) { return 1; }

const char* tra_last_error(void) { return g_err; }

int tra_device_arch(char* buf, int buf_len) {
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess || n == 0) {
    set_error("no HIP device");
    return TRA_ERR_NO_DEVICE;
  }
  int dev = 0;
  TRA_HIP(hipGetDevice(&dev));
  hipDeviceProp_t prop;
  TRA_HIP(hipGetDeviceProperties(&prop, dev));
  if (buf && buf_len > 0) {
    strncpy(buf, prop.gcnArchName, (size_t)buf_len - 1);
    buf[buf_len - 1] = 0;
  }
  if (strncmp(prop.gcnArchName, "gfx950", 6) != 0) {
    set_error("device arch %s is not gfx950", prop.gcnArchName);
    return TRA_ERR_NO_DEVICE;
  }
  return TRA_OK;
}

int tra_set_tuning(const char* name, int32_t value) {
  if (!name) {
    set_error("tra_set_tuning: null name");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  struct { const char* n; int* v; } const knobs[] = {
      {"balanced", &g_ovr.balanced}, {"window", &g_ovr.window}, {"unroll", &g_ovr.unroll},
      {"lds", &g_ovr.lds}, {"xcd", &g_ovr.xcd}, {"cost_floor", &g_ovr.cost_floor},
      {"fused_scan", &g_ovr.fused_scan}, {"cb", &g_ovr.cb}, {"fork", &g_ovr.fork}};
  for (const auto& k : knobs)
    if (strcmp(name, k.n) == 0) {
      *k.v = value < 0 ? -1 : value;
      g_ovr_gen.fetch_add(1, std::memory_order_relaxed);
      return TRA_OK;
    }
  set_error("tra_set_tuning: unknown knob '%s'", name);
  return TRA_ERR_INVALID_ARGUMENT;
}

int tra_tbe_create(const tra_table_spec* tables, int32_t num_tables,
                   const int32_t* feature_table_map, const int32_t* feature_positions,
                   int32_t num_features, tra_tbe_t* out) {
  if (!out || num_tables < 0 || num_features < 0 || (num_tables > 0 && !tables) ||
      (num_features > 0 && !feature_table_map)) {
    set_error("tra_tbe_create: null or negative argument");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  *out = nullptr;
  for (int t = 0; t < num_tables; ++t) {
    const tra_table_spec& s = tables[t];
    const int bits = bits_of(s.dtype);
    if (bits == 0) {
      set_error("table %d: unsupported dtype %d", t, s.dtype);
      return TRA_ERR_INVALID_ARGUMENT;
    }
    if (s.rows < 1) {
      // Skipped ids are redirected to row 0, so every table needs one.
      set_error("table %d has no rows", t);
      return TRA_ERR_INVALID_ARGUMENT;
    }
    if (s.dim <= 0 || (int64_t)s.dim * bits % 32 != 0) {
      set_error("table %d: dim %d with %d-bit elements is not a whole number of dwords", t,
                s.dim, bits);
      return TRA_ERR_INVALID_ARGUMENT;
    }
    const int need = s.dim * bits / 8 + header_bytes(s.dtype);
    if (s.row_bytes < need || s.row_bytes % 4 != 0 || s.offset % 4 != 0 || s.offset < 0) {
      set_error("table %d: row_bytes %d (need >= %d) and offset must be multiples of 4", t,
                s.row_bytes, need);
      return TRA_ERR_INVALID_ARGUMENT;
    }
  }
  auto plan = new tra_tbe();
  plan->num_features = num_features;
  int col = 0;
  // (dtype, cb, rows cut into several slices) -> slice ids
  std::map<std::tuple<int, int, int>, std::vector<int>> by_class;
  std::vector<int> slice_lpr;
  for (int f = 0; f < num_features; ++f) {
    const int t = feature_table_map[f];
    if (t < 0 || t >= num_tables || (feature_positions && feature_positions[f] < 0)) {
      delete plan;
      set_error("feature %d maps to table %d of %d (or has a negative position)", f, t,
                num_tables);
      return TRA_ERR_INVALID_ARGUMENT;
    }
    const tra_table_spec& s = tables[t];
    if (f == 0) plan->dim0 = s.dim;
    if (s.dim != plan->dim0) plan->same_dim = false;
    const int bits = bits_of(s.dtype);
    const int payload = s.dim * bits / 8;
    // Bytes per lane.  Rows of up to 64 payload bytes take 8-byte chunks: with
    // 16-byte chunks a wave would gather from 16-64 different rows per load,
    // which measured 9 % slower on the mixed-width workload (and 3 % faster on
    // the all-64-byte one).
    int cb = payload % 16 == 0 && payload > 64 ? 16 : (payload % 8 == 0 ? 8 : 4);
    {
      const int force = g_ovr.cb;  // tuning: smaller lane chunks, or 16 bytes wherever they divide the row
      if ((force == 8 || force == 4) && force < cb && payload % force == 0) cb = force;
      if (force == 16 && payload % 16 == 0) cb = 16;
    }
    const int max_slice = cb * kWaveSize;  // bytes one wave-wide lane group covers
    // A row with a header whose lanes take 8 or 4 bytes normally gets its header with the
    // first lane's chunk; cut into several slices, only the first slice could, so all its
    // slices go to a launch class of their own that loads the header separately.
    const int split = payload > max_slice && header_bytes(s.dtype) != 0 && cb <= 8 ? 1 : 0;
    for (int off = 0; off < payload; off += max_slice) {
      const int bytes = std::min(max_slice, payload - off);
      FeatureDesc d;
      d.table_offset = s.offset;
      d.rows = s.rows;
      d.dim = s.dim;
      d.row_bytes = s.row_bytes;
      d.out_col = col + off * 8 / bits;
      d.dtype = s.dtype;
      d.feature = feature_positions ? feature_positions[f] : f;
      d.payload_off = off;
      by_class[{s.dtype, cb, split}].push_back((int)plan->slices.size());
      plan->slices.push_back(d);
      slice_lpr.push_back(bytes / cb);
    }
    // The sixteen-lane kernel's slices.
    for (const bool few : {false, true})
      for (int off = 0; off < s.dim;) {
        const GroupShape shape = group_shape(s.dtype, s.dim, off, few);
        GroupSlice w;
        w.table_offset = s.offset;
        w.rows = s.rows;
        w.rows32 = (uint32_t)std::min<int64_t>(s.rows, int64_t(1) << 31);
        w.row_bytes = s.row_bytes;
        w.cols = shape.cols;
        w.out_col = col + off;
        w.payload = header_bytes(s.dtype) + off * bits / 8;
        w.key = feature_positions ? feature_positions[f] : f;
        w.even = w.out_col % 2 == 0 ? 1 : 0;
        w.first_slice = off == 0 ? 1 : 0;
        w.lanes_log2 = (uint8_t)shape.lanes_log2;
        // (near: row offset and place in the row are added in 32 bits)
        const bool split = header_bytes(s.dtype) != 0 && (shape.cols < s.dim || shape.lanes_log2 > 4);
        w.kind = group_kind(s.dtype, shape.ne, split ? kSplit : s.rows * s.row_bytes > 0xffffffffll ? kFar : kNear);
        for (int part = 0; part < (1 << shape.lanes_log2) / 16; ++part) {
          w.part = (uint8_t)part;
          plan->group_slices[few].host.push_back(w);
        }
        off += shape.cols;
      }
    col += s.dim;
  }
  // Classes: slices sorted by lanes-per-row; at most kMaxSub distinct values each.
  std::vector<int32_t> all_feats;
  for (auto& kv : by_class) {
    std::vector<int>& ids = kv.second;
    std::stable_sort(ids.begin(), ids.end(),
                     [&](int x, int y) { return slice_lpr[x] < slice_lpr[y]; });
    LaunchClass cur;
    int distinct = 0, last_lpr = -1;
    auto flush = [&]() {
      if (!cur.feats.empty()) plan->classes.push_back(cur);
      cur = LaunchClass();
      distinct = 0;
      last_lpr = -1;
    };
    for (int id : ids) {
      if (slice_lpr[id] != last_lpr) {
        if (distinct == kMaxSub) flush();
        ++distinct;
        last_lpr = slice_lpr[id];
      }
      cur.dtype = std::get<0>(kv.first);
      cur.cb = std::get<1>(kv.first);
      cur.split = std::get<2>(kv.first) != 0;
      cur.feats.push_back(id);
      cur.lprs.push_back(slice_lpr[id]);
    }
    flush();
  }
  hipError_t e = hipGetDevice(&plan->device);
  if (e == hipSuccess) {
    // The window kernel sizes its grid by the CU count and keeps consecutive
    // windows on one die: both come from the device, so a partitioned GPU
    // (fewer CUs, fewer dies) gets a launch that fits it.
    int cus = 0, xcds = 0;
    e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, plan->device);
    if (e == hipSuccess && hipDeviceGetAttribute(&xcds, hipDeviceAttributeNumberOfXccs, plan->device) != hipSuccess) {
      (void)hipGetLastError();
      xcds = 1;
    }
    if (e == hipSuccess) {
      if (cus < 1) {
        delete plan;
        set_error("tra_tbe_create: device reports %d compute units", cus);
        return TRA_ERR_NO_DEVICE;
      }
      plan->num_cus = cus;
      // Blocks are dealt to the dies round-robin; the remap assumes every die
      // has the same number of CUs.  Anything else: no remap.
      plan->num_xcd = (xcds >= 1 && cus % xcds == 0) ? xcds : 1;
      // Only tra_tbe_forward_lengths_static needs the static scratch: where it cannot be
      // resolved the plan is still good for every other entry point, and that one reports it.
      if (resolve_static_scratch(plan->device) == TRA_OK) {
        plan->static_scratch = g_scratch_ptr[plan->device];
      } else {
        (void)hipGetLastError();
        plan->static_scratch = nullptr;
      }
    }
  }
  size_t total = 0;
  for (auto& c : plan->classes) total += c.feats.size();
  if (e == hipSuccess && !plan->slices.empty()) {
    e = hipMalloc((void**)&plan->slices_dev, plan->slices.size() * sizeof(FeatureDesc));
    if (e == hipSuccess)
      e = hipMemcpy(plan->slices_dev, plan->slices.data(),
                    plan->slices.size() * sizeof(FeatureDesc), hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMalloc((void**)&plan->feats_dev, total * sizeof(int32_t));
    if (e == hipSuccess) {
      size_t pos = 0;
      for (auto& c : plan->classes) {
        c.feats_dev = plan->feats_dev + pos;
        all_feats.insert(all_feats.end(), c.feats.begin(), c.feats.end());
        pos += c.feats.size();
      }
      e = hipMemcpy(plan->feats_dev, all_feats.data(), total * sizeof(int32_t),
                    hipMemcpyHostToDevice);
    }
    if (e == hipSuccess) e = hipMalloc((void**)&plan->cdescs_dev, total * sizeof(FeatureDesc));
    if (e == hipSuccess) {
      std::vector<FeatureDesc> ordered;
      for (int32_t id : all_feats) ordered.push_back(plan->slices[id]);
      e = hipMemcpy(plan->cdescs_dev, ordered.data(), total * sizeof(FeatureDesc), hipMemcpyHostToDevice);
    }
  }
  if (plan->classes.size() >= 2 && plan->slices.size() == (size_t)num_features && num_features <= kMaxPos) {
    std::vector<std::tuple<int, int, int>> order;  // kind, lanes per row, slice
    for (int f = 0; f < num_features; ++f) {
      const FeatureDesc& d = plan->slices[f];
      const int bits = bits_of(d.dtype), payload = d.dim * bits / 8;
      // (the chunk of the classes, or less where a lane would hold more than 16 accumulators)
      int cb = payload % 16 == 0 && payload > 64 ? 16 : payload % 8 == 0 ? 8 : 4;
      cb = std::min(cb, 2 * bits);
      order.emplace_back(multi_kind(d.dtype, cb), payload / cb, f);
    }
    std::stable_sort(order.begin(), order.end());
    int subs = 0, widest = 0;
    for (size_t i = 0; i < order.size(); ++i) {
      subs += i == 0 || std::get<0>(order[i]) != std::get<0>(order[i - 1]) || std::get<1>(order[i]) != std::get<1>(order[i - 1]);
      widest = std::max(widest, std::get<1>(order[i]));
    }
    if (subs <= kMaxMultiSub && widest <= kWaveSize)
      for (const auto& o : order) {
        const FeatureDesc& d = plan->slices[std::get<2>(o)];
        plan->multi_kinds.push_back(std::get<0>(o));
        plan->multi_lprs.push_back(std::get<1>(o));
        plan->multi_feats.push_back(std::get<2>(o));
        plan->multi_aligned_fp16 = plan->multi_aligned_fp16 && (int64_t)d.out_col * 2 % 16 == 0;
        plan->multi_aligned_fp32 = plan->multi_aligned_fp32 && (int64_t)d.out_col * 4 % 16 == 0;
      }
  }
  if (e == hipSuccess && !plan->multi_feats.empty()) {
    std::vector<FeatureDesc> ordered;
    for (int32_t id : plan->multi_feats) ordered.push_back(plan->slices[id]);
    e = hipMalloc((void**)&plan->multi_descs_dev, ordered.size() * sizeof(FeatureDesc));
    if (e == hipSuccess)
      e = hipMemcpy(plan->multi_descs_dev, ordered.data(), ordered.size() * sizeof(FeatureDesc), hipMemcpyHostToDevice);
  }
  // (other lanes per bag are another number of descriptors; beyond kMaxPos position weights would take more launches)
  const size_t few_slices = plan->group_slices[1].host.size();
  if (few_slices == plan->group_slices[0].host.size() || few_slices > kMaxPos) plan->group_slices[1].host.clear();
  if (e == hipSuccess && !plan->group_slices[0].host.empty()) {
    // (both sets in one buffer)
    GroupSlices& few = plan->group_slices[1];
    std::vector<GroupSlice> all = plan->group_slices[0].host;
    all.insert(all.end(), few.host.begin(), few.host.end());
    GroupSlice* dev = nullptr;
    e = hipMalloc((void**)&dev, all.size() * sizeof(GroupSlice));
    plan->group_slices[0].dev = dev;
    if (e == hipSuccess) e = hipMemcpy(dev, all.data(), all.size() * sizeof(GroupSlice), hipMemcpyHostToDevice);
    if (!few.host.empty()) few.dev = dev + plan->group_slices[0].host.size();
  }
  if (e == hipSuccess) e = hipMalloc((void**)&plan->err_dev, sizeof(unsigned long long));
  if (e == hipSuccess) e = hipMemset(plan->err_dev, 0, sizeof(unsigned long long));
  if (e != hipSuccess) {
    tra_tbe_destroy(plan);
    return hip_fail(e, "tra_tbe_create");
  }
  for (const FeatureDesc& d : plan->slices) plan->max_key_pos = std::max(plan->max_key_pos, (int)d.feature);
  for (LaunchClass& cls : plan->classes) {
    for (int id : cls.feats) {
      cls.cols_aligned_fp16 = cls.cols_aligned_fp16 && (int64_t)plan->slices[id].out_col * 2 % 16 == 0;
      cls.cols_aligned_fp32 = cls.cols_aligned_fp32 && (int64_t)plan->slices[id].out_col * 4 % 16 == 0;
    }
    plan->max_class_feats = std::max(plan->max_class_feats, cls.feats.size());
    cls.odd = 2 * std::count_if(cls.lprs.begin(), cls.lprs.end(), odd_lanes) > (int64_t)cls.lprs.size();
    LookupArgs a;
    memset(&a, 0, sizeof(a));
    a.descs = plan->slices_dev;
    a.feats = cls.feats_dev;
    a.cdescs = plan->cdescs_dev + (cls.feats_dev - plan->feats_dev);
    a.err_count = plan->err_dev;
    for (size_t i = 0; i < cls.feats.size() && i < (size_t)kMaxPos; ++i)
      a.feat_pos[i] = (int16_t)plan->slices[cls.feats[i]].feature;
    plan->base_args.push_back(a);
  }
  memset(&plan->multi_base, 0, sizeof(plan->multi_base));
  plan->multi_base.cdescs = plan->multi_descs_dev;
  plan->multi_base.err_count = plan->err_dev;
  for (size_t i = 0; i < plan->multi_feats.size(); ++i)
    plan->multi_base.feat_pos[i] = (int16_t)plan->slices[plan->multi_feats[i]].feature;
  // Launch order and streams.  The launches of a call write disjoint output columns, so they may
  // overlap.  A launch leaves compute units idle before its first rows arrive and while its last
  // blocks finish; with consecutive launches on alternating streams the next launch's blocks fill
  // them.  Measured on 7 classes (64 mixed tables, 7.9 M ids): 379 us on one stream, 345 us on two
  // with the largest class first (348 us in plan order, 347 us smallest first, 355 us with the
  // classes dealt to the two streams by balanced work, where neighbours often share a stream), 376
  // and 385 us on three and four streams.  A class's work is taken as 128-byte lines per row,
  // summed over its features.
  {
    const size_t nc = plan->classes.size();
    std::vector<double> cost(nc, 0.0);
    for (size_t ci = 0; ci < nc; ++ci)
      for (int32_t lpr : plan->classes[ci].lprs)
        cost[ci] += std::max(1.0, std::ceil((double)lpr * plan->classes[ci].cb / 128.0));
    plan->launch_order.resize(nc);
    for (size_t ci = 0; ci < nc; ++ci) plan->launch_order[ci] = (int)ci;
    plan->on_side.assign(nc, 0);
    // (tuning: `fork` = k > 1 at plan creation lowers or raises the class count from which a plan forks)
    const size_t fork_min = g_ovr.fork > 1 ? (size_t)g_ovr.fork : kForkMinClasses;
    if (nc >= fork_min) {
      std::stable_sort(plan->launch_order.begin(), plan->launch_order.end(),
                       [&](int x, int y) { return cost[x] > cost[y]; });
      for (size_t k = 0; k < nc; ++k) plan->on_side[plan->launch_order[k]] = (uint8_t)(k & 1);
      if (hipStreamCreateWithFlags(&plan->side, hipStreamNonBlocking) != hipSuccess ||
          hipEventCreateWithFlags(&plan->ev_fork, hipEventDisableTiming) != hipSuccess ||
          hipEventCreateWithFlags(&plan->ev_join, hipEventDisableTiming) != hipSuccess) {
        const int rc = hip_fail(hipGetLastError(), "creating the second stream of a multi-class plan");
        tra_tbe_destroy(plan);
        return rc;
      }
    }
  }
  *out = plan;
  return TRA_OK;
}

int tra_tbe_destroy(tra_tbe_t tbe) {
  if (!tbe) return TRA_OK;
  if (tbe->slices_dev) (void)hipFree(tbe->slices_dev);
  if (tbe->feats_dev) (void)hipFree(tbe->feats_dev);
  if (tbe->cdescs_dev) (void)hipFree(tbe->cdescs_dev);
  if (tbe->group_slices[0].dev) (void)hipFree(tbe->group_slices[0].dev);
  if (tbe->multi_descs_dev) (void)hipFree(tbe->multi_descs_dev);
  if (tbe->err_dev) (void)hipFree(tbe->err_dev);
  if (tbe->side) (void)hipStreamDestroy(tbe->side);
  if (tbe->ev_join) (void)hipEventDestroy(tbe->ev_join);
  if (tbe->ev_fork) (void)hipEventDestroy(tbe->ev_fork);
  delete tbe;
  return TRA_OK;
}

// Largest number of features one window of the from-lengths kernel may span.
constexpr int kMaxWindowFeatures = 32;
// Lengths up to which the blocks of the sixteen-lane kernel sum the ones in front of their bags themselves.
constexpr int64_t kSmallFusedMaxLengths = 16384;

// A window of up to kMaxWindow bags spans kMaxWindow / B + 2 features at most.
static bool windows_derive_starts(int32_t batch_size) { return batch_size > 0 && kMaxWindow / batch_size + 2 <= kMaxWindowFeatures; }

// Ranking bags by length pays once every CU gets a few dozen bags; below that the sixteen-lane kernel is
// faster, and with several launch classes it stays so for longer, being one launch for all of them.  Graph
// replays of the whole call, us (sixteen-lane / window), ids a bag 3 and 20:
//   one class (int8 dim 64): 8192 bags 5.3 / 5.3 and 9.0 / 9.1; 13 K bags of 2 ids 6.2 / 5.6; 33 K bags 13.8 / 6.9
//   and 22.8 / 11.7
//   two classes, one launch of windows: 8192 bags 6.9 / 8.8 and 14.3 / 17; 33 K bags 17 / 12.6 and 34 / 20
//   seven classes, one launch of windows: 8192 bags 6.7 / 7.3 and 14.1 / 15.4; 33 K bags 17 / 9 and 34 / 18
// Where a plan has no such launch (over 128 features, cut rows), the window kernel is a launch per class and
// pays with the ids, not with the bags:
//   150 features, two classes: 12 K bags of 20 ids 11.0 / 24.4, 33 K of 4 15.2 / 20.6, 33 K of 20 25.7 / 25.6 (rows in
//   memory 27.3 / 29.1), 60 K of 20 44.3 / 43.2; with a cut fp32 row 33 K of 4 25.9 / 28.9, of 20 72.9 / 70.3
//   136 features, seven classes: 60 K bags of 2.5 ids 24 / 59, 33 K of 20 40 / 93, rows in memory 43 / 105
// One class of int8, fp16 or fp32 rows, bags of several ids: beyond 32 bags per compute unit (two blocks of the
// sixteen-lane kernel) that kernel's further blocks wait for the first ones:
//   8192 / 9216 bags of 20 ids, us: int8 128 columns 12.6 / 14.5 (windows 11.0 / 11.5), 256 17.0 / 20.4 (16.3 / 16.9);
//   fp16 64 8.8 / 9.9 (8.2 / 8.3), 128 11.5 / 12.6 (11.4 / 11.9); fp32 64 11.1 / 12.1 (11.0 / 11.6)
//   9216 weighted bags of 64-bit ids, of 3 and 20 ids: int8 64 7.1 / 6.9 and 11.2 / 10.7, 128 8.0 / 8.4 and 15.1 / 14.1;
//   but int4 128 7.6 / 8.4 and 12.4 / 13.2, int2 64 7.5 / 9.8 and 12.1 / 16.8
// Where a window spans too many features to derive its bags' starts a scan goes in front of it, which up to 16,384
// lengths the sixteen-lane kernel does without: 10 - 12 K bags of 2 ids 6.3 / 9.6, of 20 11.9 / 14.7, of 80 26 / 26 (from
// offsets, where neither has a scan, 5.7 / 5.3, 11.5 / 10.1, 26 / 22).
static Tuning tuning_of(const tra_tbe* tbe, int32_t batch_size, int64_t num_indices) {
  const int64_t cus = tbe->num_cus, bags = (int64_t)tbe->num_features * batch_size;
  if (tbe->classes.size() <= 1) {
    if (!windows_derive_starts(batch_size))
      return choose_tuning(bags >= 40 * cus && (num_indices >= 640 * cus || bags > kSmallFusedMaxLengths));
    const bool bytes = !tbe->classes.empty() && bits_of(tbe->classes[0].dtype) >= 8;
    return choose_tuning(bags >= 40 * cus || (bytes && bags > 32 * cus && num_indices >= 8 * bags));
  }
  if (tbe->multi_feats.empty()) return choose_tuning(bags >= 40 * cus && num_indices >= 2500 * cus);
  return choose_tuning(bags >= 40 * cus && (num_indices >= 640 * cus || bags >= 80 * cus));
}

// Whether a pooled call goes to the per-CU window kernel: the size heuristic
// (or its override) and the limits of the kernel's packed window entries.
static bool use_window_kernel(const tra_tbe* tbe, const Tuning& tune, bool nobag,
                              int32_t batch_size) {
  return !nobag && tune.balanced && batch_size <= (1 << kBagBits) && tbe->max_key_pos <= 32767 &&
         (int64_t)tbe->max_class_feats < (int64_t(1) << (32 - kBagBits)) &&
         (int64_t)tbe->max_class_feats * batch_size < (int64_t(1) << 31);
}

// The sixteen-lane kernel's slices for a call.
static const GroupSlices& group_slices_of(const tra_tbe* tbe, int32_t batch_size) {
  const bool few = (int64_t)tbe->num_features * batch_size <= kFewBags * (int64_t)tbe->num_cus;
  return tbe->group_slices[few && tbe->group_slices[1].dev != nullptr];
}

// Whether launches on a stream are being captured into a graph (or the runtime cannot say).
static bool captured(hipStream_t s) {
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s, &status) == hipSuccess) return status != hipStreamCaptureStatusNone;
  (void)hipGetLastError();
  return true;
}

// Where a call's launches go.
struct CallStream {
  hipStream_t stream;
  bool one_stream;  // never on the plan's second stream
  bool described;   // a call that is only described, and taken as not captured
};

// Whether a call of several launch classes that takes the window kernel does so in one launch (whatever the class, a
// block is a window of bags; the launches' fixed costs, and a window of each class too small to fill its block, are
// paid once).  Two classes, graph replays, us, a launch per class / one launch: 33 K bags of 20 ids 30 / 20, 131 K bags
// of 20 85 / 66, 262 K bags of 30 hot ids 182 / 151, of cold ids 280 / 277.  So: always where there is no second stream.
// Seven classes, thousands of ids per compute unit, rows in the caches and in memory:
//   on two streams, from offsets (from lengths: 6 - 10 / 0 - 4 more)
//     3.8: 77 / 26, 99 / 46   7.7: 92 / 45, 121 / 96   11.5: 117 / 63, 159 / 139   15.4: 110 / 84, 180 / 192   31: 171 / 156, 307 / 361
//   captured or from the entry that must not allocate, on one stream
//     11.5: 138 / 63, 193 / 139   15.4: 126 / 84, 205 / 192   23: 163 / 120, 267 / 277   31: 201 / 156, 330 / 361
static bool use_one_launch(const tra_tbe* tbe, int32_t batch_size, int64_t num_indices, const CallStream& c) {
  if (tbe->multi_feats.empty() || (int64_t)tbe->multi_feats.size() * batch_size >= (int64_t(1) << 31)) return false;
  if (tbe->side == nullptr || num_indices < 12000 * (int64_t)tbe->num_cus) return true;
  return num_indices < 18000 * (int64_t)tbe->num_cus && (c.one_stream || (!c.described && captured(c.stream)));
}

// One launch for several classes derives its offsets itself up to as many lengths as one scan launch takes (its blocks
// then sum 260 KB on average, about 4 us; the scan of more is two launches of 5 us each and the gaps).
constexpr int64_t kOneLaunchMaxLengths = 131072;

// Can a pooled call with these sizes take the window kernel in its
// from-lengths form (which needs no offsets)?
static bool fused_scan_possible(const tra_tbe* tbe, int32_t batch_size, int32_t num_keys,
                                int64_t num_indices, int32_t pooling_mode, const void* lengths, const CallStream& c) {
  if (pooling_mode == TRA_POOL_NONE || batch_size <= 0 || tbe->num_features == 0) return false;
  if ((uintptr_t)lengths % 16 != 0) return false;
  const Tuning tune = tuning_of(tbe, batch_size, num_indices);
  if (!use_window_kernel(tbe, tune, false, batch_size)) return false;
  const int fused = g_ovr.fused_scan;
  if (fused >= 0) return fused != 0;
  if (!windows_derive_starts(batch_size)) return false;
  // Every block of every launch sums the lengths in front of its window
  // (about 1.3 us + 1 us per 40k lengths, measured); a separate scan costs
  // about 7 us once.  Take whichever is less.
  const int64_t n = (int64_t)num_keys * batch_size;
  if (use_one_launch(tbe, batch_size, num_indices, c)) return n <= kOneLaunchMaxLengths;
  return (int64_t)tbe->classes.size() * (13 + n / 4000) < 70;
}

// A pooled call too small for the window kernel whose lengths are few enough
// that every block of the sixteen-lane kernel can sum the ones in front of its
// bags itself: one launch instead of a scan and a lookup.
static bool small_fused_scan_possible(const tra_tbe* tbe, int32_t batch_size, int32_t num_keys,
                                      int64_t num_indices, int32_t pooling_mode, const void* lengths) {
  if (pooling_mode == TRA_POOL_NONE || batch_size <= 0 || tbe->num_features == 0) return false;
  if ((uintptr_t)lengths % 16 != 0 || g_ovr.fused_scan == 0) return false;
  const Tuning tune = tuning_of(tbe, batch_size, num_indices);
  if (use_window_kernel(tbe, tune, false, batch_size)) return false;
  return (int64_t)num_keys * batch_size <= kSmallFusedMaxLengths;
}

int tra_tbe_launch_info(tra_tbe_t tbe, int32_t batch_size, int64_t num_indices,
                        int32_t pooling_mode, int32_t lengths_num_keys, char* buf,
                        int32_t buf_len) {
  if (!tbe || !buf || buf_len <= 0) {
    set_error("tra_tbe_launch_info: null argument");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  const bool nobag = pooling_mode == TRA_POOL_NONE;
  const Tuning tune = tuning_of(tbe, batch_size, num_indices);
  const bool balanced = use_window_kernel(tbe, tune, nobag, batch_size);
  const CallStream c{nullptr, false, true};
  // lengths entry point: same decision as tra_tbe_forward_lengths (aligned lengths and no capture assumed)
  const bool fused = lengths_num_keys > 0 &&
                     (fused_scan_possible(tbe, batch_size, lengths_num_keys, num_indices, pooling_mode,
                                          (const void*)16, c) ||
                      small_fused_scan_possible(tbe, batch_size, lengths_num_keys, num_indices, pooling_mode,
                                                (const void*)16));
  static const char* const kDtypeName[] = {"fp32", "fp16", "int8", "int4", "int2"};
  std::string text;
  const bool multi = balanced && use_one_launch(tbe, batch_size, num_indices, c);
  if (!nobag && (multi || !balanced)) {
    char line[120];
    snprintf(line, sizeof(line), "%s slices=%d%s", multi ? "tbe_pooled_multi_kernel" : "tbe_pooled_kernel",
             (int)(multi ? tbe->multi_feats.size() : group_slices_of(tbe, batch_size).host.size()), fused ? " from_lengths" : "");
    text = line;
  }
  // In launch order; a plan with a second stream alternates between the two.
  const bool two_streams = tbe->side != nullptr && balanced && g_ovr.fork != 0;
  for (const int ci : tbe->launch_order) {
    if (!text.empty() && !nobag && (multi || !balanced)) break;
    const LaunchClass& cls = tbe->classes[ci];
    char line[200];
    snprintf(line, sizeof(line), "%s%s dtype=%s lane_bytes=%d slices=%d%s%s",
             text.empty() ? "" : "; ",
             nobag ? "tbe_nobag_kernel" : "tbe_pooled_cu_kernel",
             kDtypeName[cls.dtype], cls.cb, (int)cls.feats.size(),
             two_streams ? (tbe->on_side[ci] ? " on the plan's second stream" : " on the caller's stream") : "",
             fused ? " from_lengths" : "");
    text += line;
  }
  if (lengths_num_keys > 0 && !fused) text = "scan_small_kernel or tile_sums_kernel + scan_tiles_kernel; " + text;
  snprintf(buf, (size_t)buf_len, "%s", text.c_str());
  return TRA_OK;
}

// Position weights of a call: one fp32 vector per input key, concatenated on
// the device; key_start / key_len (host) say where key p's vector sits.
struct PositionWeights {
  const float* table;
  int64_t table_len;
  const int32_t* key_start;
  const int32_t* key_len;
  int32_t num_keys;
};

// Where the ids of a sequence lookup's keys lie, when not given by offsets: int64 totals[num_keys] on the device,
// or the keys' first ids on the host (num_keys + 1 of them).
struct SequenceBounds {
  const int64_t* totals_dev;
  const int64_t* starts;
  int32_t num_keys;
};

// Windows of the sixteen-lane kernel: one bag per lane group until every compute unit has four blocks, then more (33 K
// bags of 3 and 20 ids, us: one bag per group 16.7 / 25.0, two 13.9 / 22.8, three 13.8 / 24.1, eight 15.5 / 30.3; 8 K
// bags: one 5.3 / 9.0, two 5.7 / 10.2).
static GroupLaunch group_windows(const tra_tbe* tbe, int32_t batch_size) {
  GroupLaunch l{};
  constexpr int groups = kBlockThreads / 16;
  const int64_t bags = (int64_t)group_slices_of(tbe, batch_size).host.size() * batch_size;
  const int64_t at_once = 4 * (int64_t)tbe->num_cus * groups;
  const int64_t per_group = std::min<int64_t>((bags + at_once - 1) / at_once, 16);
  l.per_group = (int)std::min<int64_t>(per_group, (batch_size + groups - 1) / groups);
  l.tiles = (batch_size + l.per_group * groups - 1) / (l.per_group * groups);
  return l;
}

}  // extern "C"

// Windows (bags per block) of a launch's sub-classes.  Every block should get
// about the same amount of work, so a sub-class's window shrinks with its row
// width.  A row costs its payload bytes, but never less than 256: below that the
// per-row requests (id, header, one line) dominate and rows of any width
// take the same time.  Aim at one block per CU; more passes when a window
// would not fit the kernel's LDS arrays.  Returns the grid.
static int balance_windows(const Tuning& tune, int num_cus, int32_t batch_size, SubClass* sub, const int* row_cost,
                           int n_sub) {
  const int64_t cost_floor = g_ovr.cost_floor >= 0 ? g_ovr.cost_floor : 256;
  auto bag_cost = [&](int i) { return std::max<int64_t>(row_cost[i], cost_floor); };
  int64_t total = 0, min_cost = INT64_MAX;
  for (int i = 0; i < n_sub; ++i) {
    total += (int64_t)sub[i].count * batch_size * bag_cost(i);
    min_cost = std::min(min_cost, bag_cost(i));
  }
  int64_t blocks = num_cus;
  while ((total + blocks - 1) / blocks > (int64_t)kMaxWindow * min_cost) blocks += num_cus;
  int64_t work_per_block = (total + blocks - 1) / blocks;
  auto window_of = [&](int i) {
    return std::max<int64_t>(64, std::min<int64_t>((work_per_block + bag_cost(i) - 1) / bag_cost(i), kMaxWindow));
  };
  // Rounding each sub-class up to whole windows must not spill a few
  // blocks into an extra pass: grow the share until the grid fits.
  for (int iter = 0; iter < 64; ++iter) {
    int64_t grid = 0;
    for (int i = 0; i < n_sub; ++i) grid += ((int64_t)sub[i].count * batch_size + window_of(i) - 1) / window_of(i);
    if (grid <= blocks) break;
    work_per_block += std::max<int64_t>(1, work_per_block / 128);
  }
  int grid = 0;
  for (int i = 0; i < n_sub; ++i) {
    const int64_t window = tune.window > 0 ? std::max<int64_t>(64, std::min<int64_t>(tune.window, kMaxWindow)) : window_of(i);
    sub[i].tiles_per_feat = 0;
    sub[i].window = (int)window;
    sub[i].tile_start = grid;
    grid += (int)(((int64_t)sub[i].count * batch_size + window - 1) / window);
  }
  return grid;
}

// Sub-classes of slices in launch order: runs of equal `same`.
template <typename Same>
static int cut_sub_classes(const tra_tbe* tbe, const std::vector<int32_t>& feats, const std::vector<int32_t>& lprs,
                           Same&& same, SubClass* sub) {
  int n = 0;
  for (size_t i = 0; i < feats.size();) {
    size_t j = i;
    while (j < feats.size() && same(i, j)) ++j;
    SubClass& sc = sub[n++];
    sc = SubClass();
    sc.first = (int)i;
    sc.count = (int)(j - i);
    sc.lpr = lprs[i];
    sc.key0 = tbe->slices[feats[i]].feature;
    for (size_t k = i; k < j; ++k)
      if (tbe->slices[feats[k]].feature != sc.key0 + (int)(k - i)) sc.key0 = -1;
    i = j;
  }
  return n;
}

// The XCD remap needs a grid that is a whole number of blocks per die
// (surplus blocks exit at once).
template <typename G>
static void deal_to_dies(const tra_tbe* tbe, int grid, G& g) {
  const int nx = tbe->num_xcd;
  g.grid = (grid + nx - 1) / nx * nx;
  g.xcd_count = 1;
  g.xcd_blocks = 0;
  if (nx > 1 && g_ovr.xcd != 0) {
    g.xcd_blocks = g.grid / nx;
    g.xcd_count = nx;
  }
}

// Grid and windows of every launch class for one call shape.
static void compute_geometry(const tra_tbe* tbe, const Tuning& tune, bool balanced, bool multi, bool nobag,
                             int32_t batch_size, int64_t num_indices, Geometry& g) {
  const int num_cus = tbe->num_cus;
  g.batch_size = batch_size;
  g.nobag_indices = nobag ? num_indices : -1;
  g.balanced = balanced ? 1 : 0;
  g.nobag = nobag ? 1 : 0;
  g.multi = multi ? 1 : 0;
  g.tune = tune;
  if (!balanced && !nobag) {
    g.group = group_windows(tbe, batch_size);
    return;
  }
  if (multi) {
    MultiGeometry& mg = g.all;
    const auto same = [&](size_t x, size_t y) {
      return tbe->multi_kinds[x] == tbe->multi_kinds[y] && tbe->multi_lprs[x] == tbe->multi_lprs[y];
    };
    mg.n_sub = cut_sub_classes(tbe, tbe->multi_feats, tbe->multi_lprs, same, mg.sub);
    int row_cost[kMaxMultiSub];
    for (int i = 0; i < mg.n_sub; ++i) {
      const FeatureDesc& d = tbe->slices[tbe->multi_feats[mg.sub[i].first]];
      // A bag's share of a block: per row the requests (as above), and the issue slots of its lanes, about 25 and three
      // per column that a lane holds.  (Bytes alone, us: two classes int8 dims 32 - 256, 33 K bags of 20 hot ids 28
      // against 20; seven classes 29 against 20, 262 K bags of 30 248 against 152, of 30 cold ids 349 against 309.
      // Half and twice the slots: 22.5 and 20.2, 21.4 and 21.2, 168 and 153, 365 and 334.)
      row_cost[i] = 256 + mg.sub[i].lpr * 25 + 3 * d.dim;
    }
    deal_to_dies(tbe, balance_windows(tune, num_cus, batch_size, mg.sub, row_cost, mg.n_sub), mg);
    return;
  }
  g.cls.assign(tbe->classes.size(), ClassGeometry());
  for (size_t ci = 0; ci < tbe->classes.size(); ++ci) {
    const LaunchClass& cls = tbe->classes[ci];
    ClassGeometry& cg = g.cls[ci];
    cg.n_sub = cut_sub_classes(tbe, cls.feats, cls.lprs, [&](size_t x, size_t y) { return cls.lprs[x] == cls.lprs[y]; },
                               cg.sub);
    if (balanced) {
      int row_bytes[kMaxSub];
      for (int i = 0; i < cg.n_sub; ++i) row_bytes[i] = cg.sub[i].lpr * cls.cb;
      deal_to_dies(tbe, balance_windows(tune, num_cus, batch_size, cg.sub, row_bytes, cg.n_sub), cg);
      continue;
    }
    int grid = 0;
    for (int i = 0; i < cg.n_sub; ++i) {
      SubClass& sc = cg.sub[i];
      sc.tile_start = grid;
      // Ids per tile: one step of the kernel's loop (16 to 1024 ids, by the row width), at least
      // 128 ids; less where that leaves fewer than two tiles per compute unit, down to one id
      // per lane group.  2.1 M int8 rows of 128 columns: 128 ids a tile 187 us, 256 ids 195 us,
      // 512 ids 197 us, 64 ids 201 us (8-byte lane chunks: 64 and 128 ids 187 us, 256 ids 197 us).
      // One block per tile: all of the call's ids may belong to this sub-class, and every feature
      // may leave a partial tile; blocks stride over the tiles if there are more.  No XCD
      // remap: consecutive tiles on the same die measured 5 % slower.
      const int per_block = kWavesPerBlock * (kWaveSize / sc.lpr);
      const int64_t step = (int64_t)per_block * kSequenceUnroll;
      const int64_t busy = 2 * (int64_t)num_cus;
      const int64_t full = step >= 128 ? step : (128 + step - 1) / step * step;
      sc.window = (int)(num_indices >= full * busy ? full : num_indices >= step * busy ? step : per_block);
      sc.tiles_per_feat = (int)std::min<int64_t>(num_indices / sc.window + sc.count, 1 << 20);
      grid += sc.tiles_per_feat;
    }
    cg.grid = grid;
    cg.xcd_count = 1;
    cg.xcd_blocks = 0;
  }
}

extern "C" {

// The grid of a sequence lookup follows the number of ids, which differs from call to call in
// service.  Geometries are kept per id count rounded up to a step of an eighth of its power of
// two (the blocks of a feature stride over its ids, so any grid of about the right size will
// do): neighbouring batch sizes share an entry instead of each evicting one.
static int64_t quantized_id_count(int64_t n) {
  if (n <= 1024) return 1024;
  int lg = 0;
  while ((int64_t(1) << (lg + 1)) <= n) ++lg;
  const int64_t step = int64_t(1) << (lg - 3);
  return (n + step - 1) / step * step;
}

static int forward_impl(tra_tbe_t tbe, const void* weights, const void* indices,
                        const void* offsets, bool from_lengths, int32_t idx_is_i64,
                        const float* per_sample_weights, int32_t batch_size, int64_t num_indices,
                        int32_t pooling_mode, int32_t out_dtype, void* out, int64_t out_stride,
                        void* stream, const PositionWeights* pw = nullptr, bool one_stream = false,
                        const SequenceBounds* seq = nullptr) {
  if (!tbe) {
    set_error("tra_tbe_forward: null plan");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  if (pooling_mode != TRA_POOL_SUM && pooling_mode != TRA_POOL_MEAN &&
      pooling_mode != TRA_POOL_NONE) {
    set_error("tra_tbe_forward: bad pooling mode %d", pooling_mode);
    return TRA_ERR_INVALID_ARGUMENT;
  }
  if (out_dtype != TRA_FP32 && out_dtype != TRA_FP16) {
    set_error("tra_tbe_forward: output dtype %d is not fp32/fp16", out_dtype);
    return TRA_ERR_UNSUPPORTED;
  }
  if (batch_size < 0) {
    set_error("tra_tbe_forward: negative batch size");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  const bool nobag = pooling_mode == TRA_POOL_NONE;
  if (tbe->num_features == 0 || batch_size == 0 || (nobag && num_indices == 0)) return TRA_OK;
  if (num_indices < 0) {
    set_error("tra_tbe_forward: num_indices is required");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  if (!weights || (!offsets && !seq) || !out || (!indices && num_indices != 0)) {
    set_error("tra_tbe_forward: null buffer");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  {
    // Rows are read as dwords; ids, bag boundaries and weights as whole elements.
    const uintptr_t isz = idx_is_i64 ? 8 : 4;
    if ((uintptr_t)weights % 4 != 0 || (uintptr_t)indices % isz != 0 ||
        (uintptr_t)offsets % isz != 0 || (uintptr_t)per_sample_weights % 4 != 0 ||
        (uintptr_t)out % (out_dtype == TRA_FP16 ? 2 : 4) != 0 ||
        (pw != nullptr && (uintptr_t)pw->table % 4 != 0)) {
      set_error("tra_tbe_forward: a buffer is not aligned to its element size");
      return TRA_ERR_INVALID_ARGUMENT;
    }
  }
  if (nobag && !tbe->same_dim) {
    set_error("tra_tbe_forward: sequence lookup needs one embedding dim for all tables");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  {
    int cur = -1;
    if (hipGetDevice(&cur) != hipSuccess || cur != tbe->device) {
      set_error("tra_tbe_forward: plan was created on device %d, current device is %d", tbe->device,
                cur);
      return TRA_ERR_INVALID_ARGUMENT;
    }
  }
  const int esz = out_dtype == TRA_FP16 ? 2 : 4;
  hipStream_t s = (hipStream_t)stream;
  // Route and launch geometry: remembered per (batch size, route) in the plan.
  std::shared_ptr<const Geometry> geo;
  {
    std::lock_guard<std::mutex> lock(tbe->geo_mutex);
    const int gen = g_ovr_gen.load(std::memory_order_relaxed);
    const Tuning tune = tuning_of(tbe, batch_size, num_indices);
    const int balanced = use_window_kernel(tbe, tune, nobag, batch_size) ? 1 : 0;
    const CallStream where{(hipStream_t)stream, one_stream, false};
    const int multi = balanced && use_one_launch(tbe, batch_size, num_indices, where) ? 1 : 0;
    const int64_t geo_indices = nobag ? quantized_id_count(num_indices) : num_indices;
    for (const auto& g : tbe->geo)
      if (g && g->batch_size == batch_size && g->gen == gen && g->balanced == balanced &&
          g->multi == multi && g->nobag == (int)nobag && (!nobag || g->nobag_indices == geo_indices)) {
        geo = g;
        break;
      }
    if (!geo) {
      auto g = std::make_shared<Geometry>();
      compute_geometry(tbe, tune, balanced != 0, multi != 0, nobag, batch_size, geo_indices, *g);
      g->gen = gen;
      geo = g;
      tbe->geo[tbe->geo_next] = geo;  // a call still launching from the replaced entry keeps it alive
      tbe->geo_next = (tbe->geo_next + 1) % kGeometrySlots;
    }
  }
  const Geometry& geo_local = *geo;
  const bool balanced = geo_local.balanced != 0;
  // A call of several launch classes runs them on two streams: the caller's stream forks into the
  // plan's second stream before the first launch and joins it after the last.  One call at a time
  // per plan enqueues such a sequence (the events are the plan's).  Not while the caller's stream
  // is being captured, not for the sixteen-lane kernel, not from the entry point that must not
  // allocate (an event's first record may), and `fork` = 0 (tuning) switches it off.
  bool forked = false;
  std::unique_lock<std::mutex> fork_lock(tbe->fork_mutex, std::defer_lock);
  if (tbe->side != nullptr && balanced && !geo_local.multi && !one_stream && g_ovr.fork != 0 && !captured(s)) {
    fork_lock.lock();
    TRA_HIP(hipEventRecord(tbe->ev_fork, s));
    TRA_HIP(hipStreamWaitEvent(tbe->side, tbe->ev_fork, 0));
    forked = true;
  }
  hipStream_t const caller_stream = s;
  // (an error on the way still joins the side streams before it is returned)
  auto join = [&](int rc) -> int {
    if (forked && (hipEventRecord(tbe->ev_join, tbe->side) != hipSuccess ||
                   hipStreamWaitEvent(caller_stream, tbe->ev_join, 0) != hipSuccess)) {
      if (rc == TRA_OK) rc = hip_fail(hipGetLastError(), "joining the second stream of a lookup call");
    }
    return rc;
  };
  const bool positions = pw != nullptr && !nobag && num_indices > 0;
  // Where the position weights of a launch's n features lie; key_of(i): the i-th one's key position.
  auto fill_positions = [&](int32_t* off, int32_t* len, size_t n_features, auto&& key_of) -> int {
    if (tbe->max_class_feats > (size_t)kMaxPos) {
      set_error("position-weighted lookup: a launch class has %d features, at most %d are supported",
                (int)tbe->max_class_feats, kMaxPos);
      return TRA_ERR_TOO_LARGE;
    }
    for (size_t i = 0; i < n_features; ++i) {
      const int key = key_of(i);
      if (key < 0 || key >= pw->num_keys) {
        set_error("position-weighted lookup: feature at key position %d, but %d keys were described", key, pw->num_keys);
        return TRA_ERR_INVALID_ARGUMENT;
      }
      const int64_t st = pw->key_start[key], n = pw->key_len[key];
      if (n < 0 || st < 0 || (n > 0 && st + n > pw->table_len)) {
        set_error("position-weighted lookup: key %d has weights [%lld, %lld) outside the table of %lld", key,
                  (long long)st, (long long)(st + n), (long long)pw->table_len);
        return TRA_ERR_INVALID_ARGUMENT;
      }
      off[i] = (int32_t)st;
      len[i] = (int32_t)n;
    }
    return TRA_OK;
  };
  // Lanes past the end of their bag still issue (clamped) id loads, so the
  // kernels need one readable element even when there are no ids at all.
  const void* const readable_ids = num_indices > 0 ? indices : (const void*)tbe->err_dev;
  // (no ids: nothing to weigh, and the weights pointer may not be readable)
  const float* const psw = nobag || num_indices == 0 || positions ? nullptr : per_sample_weights;
  // What a call adds to the arguments of a window or sequence launch of n features.
  auto fill = [&](LookupArgs& a, size_t n_features, auto&& key_of) -> int {
    a.weights = (const uint8_t*)weights;
    a.indices = readable_ids;
    a.offsets = offsets;
    a.psw = psw;
    if (positions) {
      const int rc = fill_positions(a.pw_off, a.pw_len, n_features, key_of);
      if (rc != TRA_OK) return rc;
      a.posw = pw->table;
    }
    a.out = out;
    a.out_stride = out_stride;
    a.bad_to_row0 = tbe->bad_to_row0.load(std::memory_order_relaxed);
    a.num_indices = num_indices > 0 ? num_indices : 1;
    a.B = batch_size;
    a.mean = pooling_mode == TRA_POOL_MEAN;
    a.out_fp16 = out_dtype == TRA_FP16;
    return TRA_OK;
  };
  auto vec_store = [&](const LaunchClass& cls) -> bool {
    const int ne = cls.cb * 8 / bits_of(cls.dtype);
    if ((uintptr_t)out % 16 != 0 || (int64_t)ne * esz % 16 != 0) return false;
    if (nobag) return (int64_t)tbe->dim0 * esz % 16 == 0;
    return out_stride * esz % 16 == 0 && (esz == 2 ? cls.cols_aligned_fp16 : cls.cols_aligned_fp32);
  };
  if (!balanced && !nobag) {
    GroupArgs a;
    a.weights = (const uint8_t*)weights;
    a.indices = readable_ids;
    a.offsets = offsets;
    a.psw = psw;
    a.posw = positions ? pw->table : nullptr;
    a.out = out;
    a.out_stride = out_stride;
    a.err_count = tbe->err_dev;
    a.num_indices = num_indices > 0 ? num_indices : 1;
    a.B = batch_size;
    a.mean = pooling_mode == TRA_POOL_MEAN;
    a.out_fp16 = out_dtype == TRA_FP16;
    a.pairs = (uintptr_t)out % 4 == 0 && out_stride % 2 == 0;
    a.bad_to_row0 = tbe->bad_to_row0.load(std::memory_order_relaxed) != 0;
    // (position weights: the launch arguments hold the layout of kMaxPos slices)
    const GroupSlices& all = group_slices_of(tbe, batch_size);
    const size_t step = positions ? kMaxPos : all.host.size();
    for (size_t s0 = 0; s0 < all.host.size(); s0 += step) {
      const size_t n = std::min(step, all.host.size() - s0);
      const GroupSlice* slices = all.host.data() + s0;
      a.slices = all.dev + s0;
      GroupPositions p;
      if (positions) {
        const int rc = fill_positions(p.off, p.len, n, [&](size_t i) { return slices[i].key; });
        if (rc != TRA_OK) return rc;
      }
      GroupLaunch l = geo_local.group;
      l.grid = (int)n * l.tiles;
      l.key0 = slices[0].key;
      for (size_t i = 1; i < n; ++i)
        if (slices[i].key != l.key0 + (int)i) {
          l.key0 = -1;
          break;
        }
      const auto go = [&](auto ids) {
        using IdxT = decltype(ids);
        if (positions)
          launch_group<IdxT, kByPosition>(a, &p, l, from_lengths, s);
        else if (psw != nullptr)
          launch_group<IdxT, kPerSample>(a, nullptr, l, from_lengths, s);
        else
          launch_group<IdxT, kUnweighted>(a, nullptr, l, from_lengths, s);
      };
      if (idx_is_i64) go(int64_t()); else go(int32_t());
      const hipError_t e = hipGetLastError();
      if (e != hipSuccess) return hip_fail(e, "tbe lookup launch");
    }
    return TRA_OK;
  }
  if (geo_local.multi) {
    const MultiGeometry& mg = geo_local.all;
    MultiArgs m;
    LookupArgs& a = m.common;
    a = tbe->multi_base;
    const int rc = fill(a, tbe->multi_feats.size(), [&](size_t i) { return tbe->slices[tbe->multi_feats[i]].feature; });
    if (rc != TRA_OK) return rc;
    a.xcd_blocks = mg.xcd_blocks;
    a.xcd_count = mg.xcd_count;
    const bool aligned = (uintptr_t)out % 16 == 0 && out_stride * esz % 16 == 0 &&
                         (esz == 2 ? tbe->multi_aligned_fp16 : tbe->multi_aligned_fp32);
    for (int i = 0; i < kMaxMultiSub; ++i) {
      m.tile_start[i] = i < mg.n_sub ? mg.sub[i].tile_start : INT32_MAX;
      m.kind[i] = 0;
      if (i >= mg.n_sub) continue;
      m.sub[i] = mg.sub[i];
      const FeatureDesc& d = tbe->slices[tbe->multi_feats[mg.sub[i].first]];
      const bool vec = aligned && d.dim / mg.sub[i].lpr * esz % 16 == 0;
      m.kind[i] = tbe->multi_kinds[mg.sub[i].first] | (vec ? kMultiVec : 0);
    }
    const auto go = [&](auto ids) {
      using IdxT = decltype(ids);
      if (a.posw != nullptr)
        launch_multi<IdxT, kByPosition>(m, mg.grid, geo_local.tune.lds_bytes, from_lengths, s);
      else if (a.psw != nullptr)
        launch_multi<IdxT, kPerSample>(m, mg.grid, geo_local.tune.lds_bytes, from_lengths, s);
      else
        launch_multi<IdxT, kUnweighted>(m, mg.grid, geo_local.tune.lds_bytes, from_lengths, s);
    };
    if (idx_is_i64) go(int64_t()); else go(int32_t());
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? TRA_OK : hip_fail(e, "tbe lookup launch");
  }
  for (const int ci : tbe->launch_order) {
    s = forked && tbe->on_side[ci] ? tbe->side : caller_stream;
    const LaunchClass& cls = tbe->classes[ci];
    const ClassGeometry& cg = geo_local.cls[ci];
    LookupArgs a = tbe->base_args[ci];
    const int filled = fill(a, cls.feats.size(), [&](size_t i) { return tbe->slices[cls.feats[i]].feature; });
    if (filled != TRA_OK) return join(filled);
    a.bounds_kind = kBoundsOffsets;
    if (seq != nullptr) {
      a.num_keys = seq->num_keys;
      a.offsets = seq->totals_dev;
      a.bounds_kind = seq->totals_dev ? kBoundsTotals : kBoundsHost;
      for (size_t i = 0; !seq->totals_dev && i < cls.feats.size(); ++i) {
        const int key = tbe->slices[cls.feats[i]].feature;
        a.pw_off[i] = (int32_t)seq->starts[key];
        a.pw_len[i] = (int32_t)(seq->starts[key + 1] - seq->starts[key]);
      }
    }
    a.vec_store = vec_store(cls) ? 1 : 0;
    memcpy(a.sub, cg.sub, sizeof(a.sub));
    a.n_sub = cg.n_sub;
    a.xcd_blocks = cg.xcd_blocks;
    a.xcd_count = cg.xcd_count;
    LaunchParams lp;
    lp.lds_bytes = geo_local.tune.lds_bytes;
    lp.grid = cg.grid;
    lp.unroll = geo_local.tune.unroll;
    lp.idx64 = idx_is_i64 != 0;
    lp.weighted = a.psw != nullptr || a.posw != nullptr;
    lp.from_lengths = from_lengths;
    lp.odd = cls.odd;
    int rc;
    if (nobag) {
      rc = launch_sequence(a, cls.dtype, cls.cb, cls.split, lp.idx64, lp.grid, s);
      if (rc != TRA_OK) return join(rc);
      continue;
    }
    switch (cls.dtype) {
      case TRA_INT8:
        rc = cls.split ? launch_lookup<TRA_INT8 + kSplitHeader>(a, cls.cb, lp, s) : launch_lookup<TRA_INT8>(a, cls.cb, lp, s);
        break;
      case TRA_INT4:
        rc = cls.split ? launch_lookup<TRA_INT4 + kSplitHeader>(a, cls.cb, lp, s) : launch_lookup<TRA_INT4>(a, cls.cb, lp, s);
        break;
      case TRA_INT2:
        rc = cls.split ? launch_lookup<TRA_INT2 + kSplitHeader>(a, cls.cb, lp, s) : launch_lookup<TRA_INT2>(a, cls.cb, lp, s);
        break;
      case TRA_FP16: rc = launch_lookup<TRA_FP16>(a, cls.cb, lp, s); break;
      default: rc = launch_lookup<TRA_FP32>(a, cls.cb, lp, s); break;
    }
    if (rc != TRA_OK) return join(rc);
  }
  return join(TRA_OK);
}

int tra_tbe_forward(tra_tbe_t tbe, const void* weights, const void* indices,
                    const void* offsets, int32_t idx_is_i64, const float* per_sample_weights,
                    int32_t batch_size, int64_t num_indices, int32_t pooling_mode,
                    int32_t out_dtype, void* out, int64_t out_stride, void* stream) {
  return forward_impl(tbe, weights, indices, offsets, false, idx_is_i64, per_sample_weights,
                      batch_size, num_indices, pooling_mode, out_dtype, out, out_stride, stream);
}

int tra_tbe_takes_key_starts(tra_tbe_t tbe) {
  return tbe && tbe->max_class_feats <= (size_t)kMaxPos ? 1 : 0;
}

int tra_tbe_forward_sequence(tra_tbe_t tbe, const void* weights, const void* indices, const int64_t* key_totals,
                             const int64_t* key_starts, int32_t num_keys, int32_t idx_is_i64, int64_t num_indices,
                             int32_t out_dtype, void* out, void* stream) {
  if (!tbe) {
    set_error("tra_tbe_forward_sequence: null plan");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  if ((key_totals == nullptr) == (key_starts == nullptr) || num_keys < 1 || tbe->max_key_pos >= num_keys) {
    set_error("tra_tbe_forward_sequence: one of key_totals and key_starts, for every key a feature sits at");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  if (key_totals != nullptr && (num_keys > kMaxTotalKeys || (uintptr_t)key_totals % 8 != 0)) {
    set_error("tra_tbe_forward_sequence: %d keys on the device (at most %d, 8-byte aligned)", num_keys, kMaxTotalKeys);
    return TRA_ERR_UNSUPPORTED;
  }
  if (key_starts != nullptr) {
    if (!tra_tbe_takes_key_starts(tbe) || num_indices > 0x7fffffff) {
      set_error("tra_tbe_forward_sequence: a launch class of %d column slices (at most %d) or %lld ids",
                (int)tbe->max_class_feats, kMaxPos, (long long)num_indices);
      return TRA_ERR_UNSUPPORTED;
    }
    for (int k = 0; k < num_keys; ++k)
      if (key_starts[k] < 0 || key_starts[k + 1] < key_starts[k] || key_starts[k + 1] > num_indices) {
        set_error("tra_tbe_forward_sequence: key %d lies outside the %lld ids", k, (long long)num_indices);
        return TRA_ERR_INVALID_ARGUMENT;
      }
  }
  const SequenceBounds seq{key_totals, key_starts, num_keys};
  return forward_impl(tbe, weights, indices, nullptr, false, idx_is_i64, nullptr, 1, num_indices, TRA_POOL_NONE,
                      out_dtype, out, 0, stream, nullptr, false, &seq);
}

int64_t tra_tbe_forward_lengths_workspace_bytes(int32_t num_keys, int32_t batch_size,
                                                int32_t idx_is_i64) {
  if (num_keys < 0 || batch_size < 0) return 0;
  const int64_t n = (int64_t)num_keys * batch_size;
  const int64_t off_bytes = ((n + 1) * (idx_is_i64 ? 8 : 4) + 255) / 256 * 256;
  return off_bytes + tra_cumsum_workspace_bytes(n);
}

}  // extern "C"

static int forward_lengths_impl(tra_tbe_t tbe, const void* weights, const void* indices,
                                const void* lengths, int32_t idx_is_i64,
                                const float* per_sample_weights, int32_t batch_size,
                                int32_t num_keys, int64_t num_indices, int32_t pooling_mode,
                                int32_t out_dtype, void* out, int64_t out_stride, void* workspace,
                                void* stream, const PositionWeights* pw, bool one_stream = false) {
  if (!tbe) {
    set_error("tra_tbe_forward_lengths: null plan");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  if (num_keys < 0 || batch_size < 0 || num_indices < 0) {
    set_error("tra_tbe_forward_lengths: negative size");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  for (const FeatureDesc& d : tbe->slices)
    if (d.feature >= num_keys) {
      set_error("tra_tbe_forward_lengths: feature position %d but only %d keys", d.feature,
                num_keys);
      return TRA_ERR_INVALID_ARGUMENT;
    }
  if (!lengths && (int64_t)num_keys * batch_size > 0) {
    set_error("tra_tbe_forward_lengths: null lengths");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  const CallStream where{(hipStream_t)stream, one_stream, false};
  if (fused_scan_possible(tbe, batch_size, num_keys, num_indices, pooling_mode, lengths, where) ||
      small_fused_scan_possible(tbe, batch_size, num_keys, num_indices, pooling_mode, lengths))
    return forward_impl(tbe, weights, indices, lengths, true, idx_is_i64, per_sample_weights,
                        batch_size, num_indices, pooling_mode, out_dtype, out, out_stride, stream, pw, one_stream);
  // Offsets first, then the ordinary lookup.
  const int64_t n = (int64_t)num_keys * batch_size;
  if (!workspace) {
    set_error("tra_tbe_forward_lengths: workspace of %lld bytes required",
              (long long)tra_tbe_forward_lengths_workspace_bytes(num_keys, batch_size, idx_is_i64));
    return TRA_ERR_INVALID_ARGUMENT;
  }
  const int64_t off_bytes = ((n + 1) * (idx_is_i64 ? 8 : 4) + 255) / 256 * 256;
  void* scan_ws = tra_cumsum_workspace_bytes(n) ? (void*)((uint8_t*)workspace + off_bytes) : nullptr;
  const int rc = tra_cumsum(lengths, n, idx_is_i64, workspace, scan_ws, stream);
  if (rc != TRA_OK) return rc;
  return forward_impl(tbe, weights, indices, workspace, false, idx_is_i64, per_sample_weights, batch_size, num_indices,
                      pooling_mode, out_dtype, out, out_stride, stream, pw, one_stream);
}

extern "C" {

int tra_tbe_forward_lengths(tra_tbe_t tbe, const void* weights, const void* indices,
                            const void* lengths, int32_t idx_is_i64,
                            const float* per_sample_weights, int32_t batch_size, int32_t num_keys,
                            int64_t num_indices, int32_t pooling_mode, int32_t out_dtype, void* out,
                            int64_t out_stride, void* workspace, void* stream) {
  return forward_lengths_impl(tbe, weights, indices, lengths, idx_is_i64, per_sample_weights,
                              batch_size, num_keys, num_indices, pooling_mode, out_dtype, out,
                              out_stride, workspace, stream, nullptr);
}

int64_t tra_tbe_forward_lengths_static_max_bytes(void) { return kStaticScratchBytes; }

int tra_tbe_forward_lengths_static(tra_tbe_t tbe, const void* weights, const void* indices,
                                   const void* lengths, int32_t idx_is_i64,
                                   const float* per_sample_weights, int32_t batch_size,
                                   int32_t num_keys, int64_t num_indices, int32_t pooling_mode,
                                   int32_t out_dtype, void* out, int64_t out_stride, void* stream) {
  if (!tbe) {
    set_error("tra_tbe_forward_lengths_static: null plan");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  const int64_t need = tra_tbe_forward_lengths_workspace_bytes(num_keys, batch_size, idx_is_i64);
  if (need > kStaticScratchBytes) {
    set_error("tra_tbe_forward_lengths_static: %d keys x %d samples need %lld bytes of scratch, the static "
              "buffer holds %lld; use tra_tbe_forward_lengths with a workspace",
              num_keys, batch_size, (long long)need, (long long)kStaticScratchBytes);
    return TRA_ERR_TOO_LARGE;
  }
  if (!tbe->static_scratch) {
    set_error("tra_tbe_forward_lengths_static: the static scratch was not resolved for device %d", tbe->device);
    return TRA_ERR_HIP;
  }
  return forward_lengths_impl(tbe, weights, indices, lengths, idx_is_i64, per_sample_weights,
                              batch_size, num_keys, num_indices, pooling_mode, out_dtype, out,
                              out_stride, tbe->static_scratch, stream, nullptr, /*one_stream=*/true);
}

int tra_tbe_forward_position_weighted(tra_tbe_t tbe, const void* weights, const void* indices,
                                      const void* bags, int32_t bags_are_lengths,
                                      int32_t idx_is_i64, const float* position_weights,
                                      int64_t position_weights_len, const int32_t* key_start,
                                      const int32_t* key_len, int32_t num_keys, int32_t batch_size,
                                      int64_t num_indices, int32_t pooling_mode, int32_t out_dtype,
                                      void* out, int64_t out_stride, void* workspace,
                                      void* stream) {
  if (!position_weights || position_weights_len < 1 || !key_start || !key_len || num_keys < 0) {
    set_error("tra_tbe_forward_position_weighted: null or empty position weight description");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  if (pooling_mode == TRA_POOL_NONE) {
    set_error("tra_tbe_forward_position_weighted: position weights apply to pooled lookups only");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  const PositionWeights pw{position_weights, position_weights_len, key_start, key_len, num_keys};
  if (bags_are_lengths)
    return forward_lengths_impl(tbe, weights, indices, bags, idx_is_i64, nullptr, batch_size,
                                num_keys, num_indices, pooling_mode, out_dtype, out, out_stride,
                                workspace, stream, &pw);
  return forward_impl(tbe, weights, indices, bags, false, idx_is_i64, nullptr, batch_size,
                      num_indices, pooling_mode, out_dtype, out, out_stride, stream, &pw);
}

int tra_tbe_set_bounds_check_mode(tra_tbe_t tbe, int32_t mode) {
  if (!tbe) {
    set_error("tra_tbe_set_bounds_check_mode: null plan");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  if (mode < -1 || mode > 3) {
    set_error("tra_tbe_set_bounds_check_mode: mode %d is none of FATAL 0, WARNING 1, IGNORE 2, NONE 3, unset -1", mode);
    return TRA_ERR_INVALID_ARGUMENT;
  }
  tbe->bad_to_row0.store(mode == 1 || mode == 2 ? 1 : 0, std::memory_order_relaxed);
  return TRA_OK;
}

int tra_tbe_error_count(tra_tbe_t tbe, void* stream, int64_t* count) {
  if (!tbe || !count) {
    set_error("tra_tbe_error_count: null argument");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  unsigned long long v = 0;
  hipStream_t s = (hipStream_t)stream;
  TRA_HIP(hipMemcpyAsync(&v, tbe->err_dev, sizeof(v), hipMemcpyDeviceToHost, s));
  TRA_HIP(hipStreamSynchronize(s));
  if (v != 0) {
    TRA_HIP(hipMemsetAsync(tbe->err_dev, 0, sizeof(v), s));
    TRA_HIP(hipStreamSynchronize(s));
  }
  *count = (int64_t)v;
  return TRA_OK;
}

}  // extern "C"
