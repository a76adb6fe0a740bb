// Ids per key of a KeyedJaggedTensor, on the device and on the host.
//
// Slicing a jagged result per key needs the keys' id counts on the host.  A
// device-to-host copy with a wait costs a copy engine's round trip and, behind
// other work, the wait for all of it; here the kernel that adds the lengths up
// also stores each total in pinned host memory, where the host reads it as
// soon as it is there, while whatever was queued behind the kernel runs.
#include <sched.h>

#include <atomic>
#include <mutex>

#include "tra_common.h"

namespace tra {

constexpr int kTotalsThreads = 256;
constexpr int kMailSlots = 64;
constexpr int kMailKeys = 1024;

__device__ __forceinline__ void store_total(int64_t v, int k, int64_t* dev, int64_t* host) {
  if (dev) dev[k] = v;
  if (host) publish_total(v, host + k);
}

// One block per key.
template <typename T>
__global__ __launch_bounds__(kTotalsThreads) void key_totals_kernel(const T* __restrict__ lengths, int32_t B,
                                                                    int64_t* dev, int64_t* host) {
  constexpr int V = 16 / (int)sizeof(T);
  struct __align__(16) Vec { T v[V]; };
  __shared__ int64_t s_part[kTotalsThreads / kWaveSize];
  const T* mine = lengths + (int64_t)blockIdx.x * B;
  int64_t sum = 0;
  int done = 0;
  if ((uintptr_t)mine % 16 == 0) {
    const int n = B / V;
    for (int i0 = 0; i0 < n; i0 += 4 * kTotalsThreads) {  // four loads in flight
      Vec x[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) x[u] = reinterpret_cast<const Vec*>(mine)[min(i0 + u * kTotalsThreads + (int)threadIdx.x, n - 1)];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        int64_t part = 0;
#pragma unroll
        for (int j = 0; j < V; ++j) part += (int64_t)x[u].v[j];
        sum += i0 + u * kTotalsThreads + (int)threadIdx.x < n ? part : 0;
      }
    }
    done = n * V;
  }
  for (int i = done + threadIdx.x; i < B; i += kTotalsThreads) sum += (int64_t)mine[i];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off, 64);
  if ((threadIdx.x & (kWaveSize - 1)) == 0) s_part[threadIdx.x / kWaveSize] = sum;
  __syncthreads();
  if (threadIdx.x == 0) {
    int64_t t = 0;
#pragma unroll
    for (int w = 0; w < kTotalsThreads / kWaveSize; ++w) t += s_part[w];
    store_total(t, blockIdx.x, dev, host);
  }
}

template <typename T>
__global__ __launch_bounds__(kTotalsThreads) void key_totals_of_offsets_kernel(const T* __restrict__ offsets, int32_t K,
                                                                               int32_t B, int64_t* dev, int64_t* host) {
  const int k = blockIdx.x * kTotalsThreads + threadIdx.x;
  if (k < K) store_total((int64_t)offsets[(int64_t)(k + 1) * B] - (int64_t)offsets[(int64_t)k * B], k, dev, host);
}

// The host side: kMailSlots slots of kMailKeys totals in one pinned allocation, made on first use and kept until the
// process ends.  A slot belongs to one call from begin to wait.
struct MailSlot {
  hipStream_t stream = nullptr;
  int num_keys = 0;
};
static std::mutex g_mail_mutex;
static int64_t* g_mail = nullptr;      // host address (the same pages are mapped into every GPU)
static int64_t* g_mail_dev = nullptr;  // their address there
static uint64_t g_mail_used = 0;
static MailSlot g_mail_slot[kMailSlots];

static int take_slot(int32_t* ticket) {
  std::lock_guard<std::mutex> lock(g_mail_mutex);
  if (!g_mail) {
    void* p = nullptr;
    const hipError_t e = hipHostMalloc(&p, sizeof(int64_t) * kMailSlots * kMailKeys,
                                       hipHostMallocPortable | hipHostMallocMapped | hipHostMallocCoherent);
    if (e != hipSuccess) return hip_fail(e, "hipHostMalloc(key totals)");
    void* d = nullptr;
    const hipError_t mapped = hipHostGetDevicePointer(&d, p, 0);
    if (mapped != hipSuccess) {
      (void)hipHostFree(p);
      return hip_fail(mapped, "hipHostGetDevicePointer(totals)");
    }
    g_mail = static_cast<int64_t*>(p);
    g_mail_dev = static_cast<int64_t*>(d);
  }
  if (~g_mail_used == 0) {
    set_error("tra_key_totals_begin: %d calls are waiting for their totals already", kMailSlots);
    return TRA_ERR_TOO_LARGE;
  }
  const int s = __builtin_ctzll(~g_mail_used);
  g_mail_used |= 1ull << s;
  *ticket = s;
  return TRA_OK;
}

void mail_cancel(int32_t ticket) {
  std::lock_guard<std::mutex> lock(g_mail_mutex);
  g_mail_used &= ~(1ull << ticket);
}

int mail_open(hipStream_t s, int n, int32_t* ticket, int64_t** device) {
  *ticket = -1;
  if (n > kMailKeys) {
    set_error("%d totals (at most %d reach the host)", n, kMailKeys);
    return TRA_ERR_TOO_LARGE;
  }
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone) {
    (void)hipGetLastError();
    set_error("the stream is being captured: its kernels do not run now, and the host cannot wait for their totals");
    return TRA_ERR_UNSUPPORTED;
  }
  int32_t slot = 0;
  const int rc = take_slot(&slot);
  if (rc != TRA_OK) return rc;
  int64_t* host = g_mail + (int64_t)slot * kMailKeys;
  for (int k = 0; k < n; ++k) host[k] = kMailEmpty;
  std::atomic_thread_fence(std::memory_order_release);
  *device = g_mail_dev + (int64_t)slot * kMailKeys;
  g_mail_slot[slot].stream = s;
  g_mail_slot[slot].num_keys = n;
  *ticket = slot;
  return TRA_OK;
}

}  // namespace tra

using namespace tra;

extern "C" {

int tra_key_totals_begin(const void* bags, int32_t bags_are_offsets, int32_t num_keys, int32_t batch_size,
                         int32_t is_i64, int64_t* totals, int32_t* ticket, void* stream) {
  if (!bags || num_keys < 1 || batch_size < 1 || (!totals && !ticket)) {
    set_error("tra_key_totals_begin: bad argument");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  hipStream_t s = (hipStream_t)stream;
  int64_t* host_dev = nullptr;
  if (ticket) *ticket = -1;
  // An error left by an earlier call is reported before anything is queued: what hipGetLastError says after the
  // launch is then the launch's own, and the slot is given back only where no kernel will store into it.
  const hipError_t earlier = hipGetLastError();
  if (earlier != hipSuccess) return hip_fail(earlier, "tra_key_totals_begin: an earlier call");
  if (ticket) {
    const int rc = mail_open(s, num_keys, ticket, &host_dev);
    if (rc != TRA_OK) return rc;
  }
  if (bags_are_offsets) {
    const dim3 g((num_keys + kTotalsThreads - 1) / kTotalsThreads);
    if (is_i64)
      hipLaunchKernelGGL(key_totals_of_offsets_kernel<int64_t>, g, dim3(kTotalsThreads), 0, s, (const int64_t*)bags,
                         num_keys, batch_size, totals, host_dev);
    else
      hipLaunchKernelGGL(key_totals_of_offsets_kernel<int32_t>, g, dim3(kTotalsThreads), 0, s, (const int32_t*)bags,
                         num_keys, batch_size, totals, host_dev);
  } else if (is_i64) {
    hipLaunchKernelGGL(key_totals_kernel<int64_t>, dim3(num_keys), dim3(kTotalsThreads), 0, s, (const int64_t*)bags,
                       batch_size, totals, host_dev);
  } else {
    hipLaunchKernelGGL(key_totals_kernel<int32_t>, dim3(num_keys), dim3(kTotalsThreads), 0, s, (const int32_t*)bags,
                       batch_size, totals, host_dev);
  }
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    if (ticket) {
      mail_cancel(*ticket);
      *ticket = -1;
    }
    return hip_fail(e, "tra_key_totals_begin");
  }
  return TRA_OK;
}

int tra_key_totals_wait(int32_t ticket, int64_t* totals) {
  if (ticket < 0 || ticket >= kMailSlots || !totals) {
    set_error("tra_key_totals_wait: bad ticket");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  const MailSlot slot = g_mail_slot[ticket];
  const int64_t* host = g_mail + (int64_t)ticket * kMailKeys;
  // The kernel's stores arrive one by one; each key is read until it is there.  Every few thousand reads the stream
  // is asked whether it has anything left to run at all: the wait ends with an error instead of never if the kernel
  // was lost to an earlier fault.
  for (int k = 0; k < slot.num_keys; ++k) {
    int64_t v;
    for (int spins = 0; (v = __atomic_load_n(host + k, __ATOMIC_RELAXED)) == kMailEmpty; ++spins) {
      if ((spins & 0xfff) == 0xfff) {
        const hipError_t e = hipStreamQuery(slot.stream);
        if (e != hipErrorNotReady && __atomic_load_n(host + k, __ATOMIC_RELAXED) == kMailEmpty) {
          // (the slot stays taken: nothing says that the kernel will not write to it after all)
          if (e == hipSuccess) {
            set_error("tra_key_totals_wait: the stream is idle and key %d has no total", k);
            return TRA_ERR_HIP;
          }
          return hip_fail(e, "tra_key_totals_wait");
        }
        if (e == hipErrorNotReady) (void)hipGetLastError();
        sched_yield();
      }
    }
    totals[k] = v;
  }
  mail_cancel(ticket);
  return TRA_OK;
}

}  // extern "C"
