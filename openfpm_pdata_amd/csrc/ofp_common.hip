// ofp_common.hip -- error state, plane arguments, fills and exclusive scans.
//
// The scans are three-phase (block reduce -> scan of block sums in one block ->
// block scan + offset), two-phase where the blocks are few enough that each sums
// the earlier blocks' totals itself, and one block where one will do: no
// inter-block waiting, so no kernel can spin.
#include "ofp_internal.hpp"

#include <atomic>
#include <cstring>
#include <list>
#include <mutex>

namespace ofp {

static std::atomic<uint64_t> g_realloc_epoch{0};

uint64_t realloc_epoch() { return g_realloc_epoch.load(std::memory_order_acquire); }
void bump_realloc_epoch() { g_realloc_epoch.fetch_add(1, std::memory_order_acq_rel); }

static thread_local std::string g_last_error;

// ---------------------------------------------------------- device blocks
namespace {
struct Kept {
  void* p;
  size_t cap;
  int dev;
  uint64_t stamp;  // number of the release
};
constexpr int kMaxPoolDevices = 64;
struct Pool {
  std::mutex m;
  std::list<Kept> kept;  // oldest first
  size_t held[kMaxPoolDevices] = {};
  size_t limit[kMaxPoolDevices] = {};  // 0: not asked yet
  uint64_t releases = 0;
  uint64_t synced[kMaxPoolDevices] = {};  // releases the device is known to have finished before
  size_t handles = 0;
};
Pool& pool() {
  static Pool* p = new Pool();  // lives until the process ends
  return *p;
}
// Most bytes kept on a device (under the lock): 1/128 of its memory.  Another
// allocator of the program cannot reach kept blocks, so the bound is what the lists
// that programs make anew need (2e6 particles with 46 entries: 0.8 GB), 2.25 GB of
// 288; larger blocks go back at once.
size_t keep_limit(Pool& P, int dev) {
  if (P.limit[dev] == 0) {
    hipDeviceProp_t prop;
    P.limit[dev] = hipGetDeviceProperties(&prop, dev) == hipSuccess ? prop.totalGlobalMem / 128 + 1 : 1;
  }
  return P.limit[dev];
}
// Sizes in steps of an eighth of their power of two, so counts that vary a
// little from call to call meet the same blocks; blocks too large to be kept have
// the size asked for.
size_t block_size(size_t b, size_t limit) {
  if (b > limit) return b;
  size_t step = 256;
  while (step * 16 < b) step *= 2;
  return (b + step - 1) / step * step;
}
// Takes the kept blocks that `which` names out of the pool (under its lock).
template <class F>
std::list<Kept> take_out(Pool& P, F&& which) {
  std::list<Kept> out;
  for (auto it = P.kept.begin(); it != P.kept.end();) {
    const auto next = std::next(it);
    if (which(*it)) {
      P.held[it->dev] -= it->cap;
      out.splice(out.end(), P.kept, it);
    }
    it = next;
  }
  return out;
}
void give_back(const std::list<Kept>& blocks) {
  for (const Kept& k : blocks) (void)hipFree(k.p);
}
}  // namespace

// Test hook: the next `count` allocations of lo to hi bytes fail, as on a full device
// (the runtime is asked for more than any device has).
namespace {
std::atomic<size_t> g_fail_lo{0}, g_fail_hi{0};
std::atomic<int> g_fail_count{0};
bool test_fails(size_t bytes) {
  if (g_fail_count.load(std::memory_order_relaxed) <= 0 || bytes < g_fail_lo || bytes > g_fail_hi) return false;
  return g_fail_count.fetch_sub(1) > 0;
}
}  // namespace

// Waits for everything submitted to the current device.  By hipFree, which waits
// implicitly, on an allocation made for it (3 us on an idle device): a
// hipDeviceSynchronize would end any capture under way, this thread's or another's,
// that allows hipMalloc.
static bool device_wait() {
  void* p = nullptr;
  if (hipMalloc(&p, 256) == hipSuccess && hipFree(p) == hipSuccess) return true;
  (void)hipGetLastError();
  return false;
}

int block_alloc(void** p, size_t bytes, size_t* cap, int* dev) {
  *p = nullptr;
  *cap = 0;
  OFP_HIP(hipGetDevice(dev));
  size_t want = bytes;
  Pool& P = pool();
  const int d = *dev;
  if (d >= 0 && d < kMaxPoolDevices) {
    Kept best{nullptr, 0, 0, 0};
    uint64_t before = 0;
    {
      std::lock_guard<std::mutex> lock(P.m);
      want = block_size(bytes, keep_limit(P, d));
      if (test_fails(bytes)) bytes = want = size_t(1) << 60;
      auto found = P.kept.end();
      for (auto it = P.kept.begin(); it != P.kept.end(); ++it)
        if (it->dev == d && it->cap >= want && it->cap <= want + want / 4 &&
            (found == P.kept.end() || it->cap < found->cap))
          found = it;
      if (found != P.kept.end()) {
        best = *found;
        P.held[d] -= best.cap;
        P.kept.erase(found);
        if (best.stamp > P.synced[d]) before = P.releases;
      }
    }
    if (best.p) {
      if (before) {
        const bool waited = device_wait();
        std::lock_guard<std::mutex> lock(P.m);
        if (waited) {
          if (P.synced[d] < before) P.synced[d] = before;
        } else {  // kept for later
          P.kept.push_back(best);
          P.held[d] += best.cap;
          best.p = nullptr;
        }
      }
      if (best.p) {
        *p = best.p;
        *cap = best.cap;
        return OFP_OK;
      }
    }
  }
  hipError_t e = hipMalloc(p, want);
  if (e == hipErrorOutOfMemory) {
    (void)hipGetLastError();
    std::list<Kept> mine;
    {
      std::lock_guard<std::mutex> lock(P.m);
      mine = take_out(P, [d](const Kept& k) { return k.dev == d; });
    }
    give_back(mine);
    e = hipMalloc(p, want);
    if (e == hipErrorOutOfMemory && want > bytes) e = hipMalloc(p, want = bytes);
  }
  if (e != hipSuccess) {
    // the return code alone carries the error: a caller that goes on without the
    // block would find the runtime's at its next launch
    (void)hipGetLastError();
    *p = nullptr;
    return set_error(OFP_E_HIP, "hipMalloc(%zu): %s", want, hipGetErrorString(e));
  }
  *cap = want;
  return OFP_OK;
}

void block_free(void* p, size_t cap, int dev) {
  Pool& P = pool();
  std::list<Kept> out;
  bool keep = false;
  if (dev >= 0 && dev < kMaxPoolDevices) {
    std::lock_guard<std::mutex> lock(P.m);
    const size_t limit = keep_limit(P, dev);
    if (P.handles > 0 && cap <= limit) {
      keep = true;
      P.kept.push_back(Kept{p, cap, dev, ++P.releases});
      P.held[dev] += cap;
      size_t over = P.held[dev] > limit ? P.held[dev] - limit : 0;
      out = take_out(P, [dev, &over](const Kept& k) {
        if (k.dev != dev || over == 0) return false;
        over -= k.cap < over ? k.cap : over;
        return true;
      });
    }
  }
  if (!keep) (void)hipFree(p);
  give_back(out);
}

HandleLife::HandleLife() {
  Pool& P = pool();
  std::lock_guard<std::mutex> lock(P.m);
  ++P.handles;
}

HandleLife::~HandleLife() {
  Pool& P = pool();
  std::list<Kept> out;
  {
    std::lock_guard<std::mutex> lock(P.m);
    if (--P.handles == 0) out = take_out(P, [](const Kept&) { return true; });
  }
  give_back(out);
}

int set_error(int code, const char* fmt, ...) {
  char buf[1024];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof buf, fmt, ap);
  va_end(ap);
  g_last_error = buf;
  return code;
}

void clear_error() { g_last_error.clear(); }

int make_plane_args(const ofp_plane* in, const ofp_plane* out, int n, PlaneArgs* a) {
  OFP_CHECK(n >= 0 && n <= kMaxPlanes, OFP_E_LIMIT, "at most %d planes per call (got %d)",
            kMaxPlanes, n);
  OFP_CHECK(n == 0 || in != nullptr, OFP_E_ARG, "null plane list");
  std::memset(a, 0, sizeof(*a));
  a->n = n;
  for (int k = 0; k < n; ++k) {
    OFP_CHECK(in[k].elem_bytes == 4 || in[k].elem_bytes == 8, OFP_E_ARG,
              "plane %d: elem_bytes must be 4 or 8 (got %u)", k, in[k].elem_bytes);
    OFP_CHECK(in[k].ptr != nullptr, OFP_E_ARG, "plane %d: null pointer", k);
    a->src[k] = reinterpret_cast<uint64_t>(in[k].ptr);
    a->esz[k] = in[k].elem_bytes;
    if (out) {
      OFP_CHECK(out[k].ptr != nullptr && out[k].elem_bytes == in[k].elem_bytes, OFP_E_ARG,
                "plane %d: output pointer null or element size differs", k);
      a->dst[k] = reinterpret_cast<uint64_t>(out[k].ptr);
    } else {
      a->dst[k] = a->src[k];
    }
  }
  return OFP_OK;
}

// ------------------------------------------------------------------ fills
template <class U>
__global__ void k_fill(U* p, U v, size_t n) {
  size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
  size_t step = size_t(gridDim.x) * blockDim.x;
  for (; i < n; i += step) p[i] = v;
}

template <class U>
static int fill_impl(U* p, U v, size_t n, hipStream_t s) {
  if (n == 0) return OFP_OK;
  unsigned g = grid_for(n, 256);
  if (g > 8192) g = 8192;
  k_fill<U><<<g, 256, 0, s>>>(p, v, n);
  OFP_LAUNCHED();
  return OFP_OK;
}

int fill_u32(uint32_t* p, uint32_t v, size_t n, hipStream_t s) { return fill_impl(p, v, n, s); }
int fill_u64(uint64_t* p, uint64_t v, size_t n, hipStream_t s) { return fill_impl(p, v, n, s); }

// ------------------------------------------------------------------ scans
constexpr int kScanBlock = 256;
constexpr int kScanItems = 16;
constexpr size_t kScanTile = size_t(kScanBlock) * kScanItems;  // 4096 per block
// One launch up to kScanOne elements, two up to kScanTwo tiles, three beyond.  A
// launch costs about 2 us of kernel and as much again before the next one starts:
// 8,192 elements 11.4 us in three launches, 7 in one.
constexpr int kScanOneBlock = 1024;
constexpr size_t kScanOne = size_t(kScanOneBlock) * kScanItems;
constexpr size_t kScanTwo = 512;

size_t scan_tmp_bytes(size_t n) {
  size_t nb = (n + kScanTile - 1) / kScanTile;
  return (nb + 1) * sizeof(uint64_t) * 2 + 256;
}

// Block-wide exclusive scan of one value per thread; returns the block total in
// *total (all threads).
template <class V, int kBlock = kScanBlock>
__device__ __forceinline__ V block_excl_scan(V v, V* lds, V* total) {
  const int lane = threadIdx.x & (kWave - 1);
  const int w = threadIdx.x / kWave;
  constexpr int nw = kBlock / kWave;
  V inc = wave_incl_scan(v);
  if (lane == kWave - 1) lds[w] = inc;
  __syncthreads();
  if (w == 0) {
    V t = lane < nw ? lds[lane] : V(0);
    V ti = wave_incl_scan(t);
    if (lane < nw) lds[lane] = ti - t;
    if (lane == nw - 1) lds[nw] = ti;
  }
  __syncthreads();
  V r = lds[w] + inc - v;
  *total = lds[nw];
  __syncthreads();
  return r;
}

template <class In, class V>
__global__ __launch_bounds__(kScanBlock) void k_scan_reduce(const In* in, size_t n,
                                                            V* partial) {
  __shared__ V lds[kScanBlock / kWave + 1];
  size_t base = size_t(blockIdx.x) * kScanTile;
  V acc = 0;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    size_t i = base + size_t(k) * kScanBlock + threadIdx.x;
    if (i < n) acc += V(in[i]);
  }
  V tot;
  (void)block_excl_scan<V>(acc, lds, &tot);
  if (threadIdx.x == 0) partial[blockIdx.x] = tot;
}

// One block scans the nb partial sums in place (exclusive): each thread sums a
// contiguous segment of them, the block scans the segment sums, and each
// thread writes its segment's prefixes.  The segment loads are independent, so
// a thread has several in flight.
template <class V>
__global__ __launch_bounds__(kScanBlock) void k_scan_partials(V* partial, size_t nb) {
  __shared__ V lds[kScanBlock / kWave + 1];
  const size_t per = (nb + kScanBlock - 1) / kScanBlock;
  const size_t a = size_t(threadIdx.x) * per;
  const size_t b = a + per < nb ? a + per : nb;
  V sum = 0;
#pragma unroll 8
  for (size_t i = a; i < b; ++i) sum += partial[i];
  V tot;
  V run = block_excl_scan<V>(sum, lds, &tot);
#pragma unroll 8
  for (size_t i = a; i < b; ++i) {
    const V x = partial[i];
    partial[i] = run;
    run += x;
  }
  if (threadIdx.x == 0) partial[nb] = tot;
}

// One tile: each thread owns kScanItems consecutive elements, read and written as
// whole 16-byte vectors in full tiles (the arrays are at least 4-byte aligned,
// which gfx950's multi-dword loads and stores need).  Returns the tile's total.
template <class In, class V, int kBlock>
__device__ __forceinline__ V scan_tile(const In* in, V* out, size_t n, size_t base, V before, V* lds) {
  const bool full = base + kScanItems <= n;
  In x[kScanItems];
  if (full) {
    __builtin_memcpy(x, in + base, sizeof(x));
  } else {
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) x[k] = base + k < n ? in[base + k] : In(0);
  }
  V acc = 0;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) acc += V(x[k]);
  V tot;
  const V ex = block_excl_scan<V, kBlock>(acc, lds, &tot);
  V run = ex + before;
  V y[kScanItems];
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    y[k] = run;
    run += V(x[k]);
  }
  if (full) {
    __builtin_memcpy(out + base, y, sizeof(y));
  } else {
#pragma unroll
    for (int k = 0; k < kScanItems; ++k)
      if (base + k < n) out[base + k] = y[k];
  }
  return tot;
}

template <class In, class V>
__global__ __launch_bounds__(kScanBlock) void k_scan_apply(const In* in, V* out, size_t n,
                                                           const V* partial, size_t nb) {
  __shared__ V lds[kScanBlock / kWave + 1];
  const size_t base = size_t(blockIdx.x) * kScanTile + size_t(threadIdx.x) * kScanItems;
  (void)scan_tile<In, V, kScanBlock>(in, out, n, base, partial[blockIdx.x], lds);
  if (blockIdx.x == 0 && threadIdx.x == 0) out[n] = partial[nb];
}

// partial: the tiles' sums (not scanned), nb <= kScanTwo of them.
template <class In, class V>
__global__ __launch_bounds__(kScanBlock) void k_scan_apply_two(const In* in, V* out, size_t n, const V* partial) {
  static_assert(kScanTwo == 2 * kScanBlock, "two sums per thread");
  __shared__ V lds[kScanBlock / kWave + 1];
  const uint32_t b = blockIdx.x, t = threadIdx.x;
  V v = t < b ? partial[t] : V(0);
  if (t + kScanBlock < b) v += partial[t + kScanBlock];
  V before;
  (void)block_excl_scan<V>(v, lds, &before);
  const size_t base = size_t(b) * kScanTile + size_t(t) * kScanItems;
  const V tot = scan_tile<In, V, kScanBlock>(in, out, n, base, before, lds);
  if (b == gridDim.x - 1 && t == 0) out[n] = before + tot;
}

template <class In, class V>
__global__ __launch_bounds__(kScanOneBlock) void k_scan_one(const In* in, V* out, size_t n) {
  __shared__ V lds[kScanOneBlock / kWave + 1];
  const V tot = scan_tile<In, V, kScanOneBlock>(in, out, n, size_t(threadIdx.x) * kScanItems, V(0), lds);
  if (threadIdx.x == 0) out[n] = tot;
}

template <class In, class V>
static int scan_impl(const In* in, V* out, size_t n, void* tmp, hipStream_t s) {
  size_t nb = (n + kScanTile - 1) / kScanTile;
  V* partial = reinterpret_cast<V*>(tmp);
  if (n == 0) {
    return fill_impl<V>(out, V(0), 1, s);
  }
  if (n <= kScanOne) {
    k_scan_one<In, V><<<1, kScanOneBlock, 0, s>>>(in, out, n);
    OFP_LAUNCHED();
    return OFP_OK;
  }
  k_scan_reduce<In, V><<<unsigned(nb), kScanBlock, 0, s>>>(in, n, partial);
  OFP_LAUNCHED();
  if (nb <= kScanTwo) {
    k_scan_apply_two<In, V><<<unsigned(nb), kScanBlock, 0, s>>>(in, out, n, partial);
    OFP_LAUNCHED();
    return OFP_OK;
  }
  k_scan_partials<V><<<1, kScanBlock, 0, s>>>(partial, nb);
  OFP_LAUNCHED();
  k_scan_apply<In, V><<<unsigned(nb), kScanBlock, 0, s>>>(in, out, n, partial, nb);
  OFP_LAUNCHED();
  return OFP_OK;
}

int scan_excl_u32(const uint32_t* in, uint32_t* out, size_t n, void* tmp, hipStream_t s) {
  return scan_impl<uint32_t, uint32_t>(in, out, n, tmp, s);
}
int scan_excl_u64(const uint64_t* in, uint64_t* out, size_t n, void* tmp, hipStream_t s) {
  return scan_impl<uint64_t, uint64_t>(in, out, n, tmp, s);
}
int scan_excl_u32_to_u64(const uint32_t* in, uint64_t* out, size_t n, void* tmp,
                         hipStream_t s) {
  return scan_impl<uint32_t, uint64_t>(in, out, n, tmp, s);
}

}  // namespace ofp

extern "C" {

const char* ofp_last_error(void) { return ofp::g_last_error.c_str(); }

int ofp_abi_version(void) { return OFP_ABI_VERSION; }

int ofp_trim(size_t* bytes) {
  ofp::Pool& P = ofp::pool();
  std::list<ofp::Kept> out;
  {
    std::lock_guard<std::mutex> lock(P.m);
    out = ofp::take_out(P, [](const ofp::Kept&) { return true; });
  }
  size_t sum = 0;
  for (const ofp::Kept& k : out) sum += k.cap;
  ofp::give_back(out);
  if (bytes) *bytes = sum;
  return OFP_OK;
}

// Test hook (not in the public header), see test_fails.
int ofp_test_fail_alloc_(size_t lo, size_t hi, int count) {
  ofp::g_fail_lo = lo;
  ofp::g_fail_hi = hi;
  ofp::g_fail_count = count;
  return OFP_OK;
}

// Test hook (not in the public header): queue_grid.
int ofp_test_queue_grid_(unsigned blocks, unsigned waves_per_block, unsigned* grid, unsigned* queues) {
  *grid = ofp::queue_grid(blocks, waves_per_block);
  *queues = ofp::kQueues;
  return OFP_OK;
}

int ofp_device_info(int* device, int* n_cu, char* arch, size_t arch_len) {
  int dev = 0;
  OFP_HIP(hipGetDevice(&dev));
  hipDeviceProp_t prop;
  OFP_HIP(hipGetDeviceProperties(&prop, dev));
  if (device) *device = dev;
  if (n_cu) *n_cu = prop.multiProcessorCount;
  if (arch && arch_len) {
    std::strncpy(arch, prop.gcnArchName, arch_len - 1);
    arch[arch_len - 1] = 0;
  }
  return OFP_OK;
}

}  // extern "C"
