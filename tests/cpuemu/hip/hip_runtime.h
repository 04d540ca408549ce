// CPU emulation of the HIP subset the library uses, for bounds checking with
// AddressSanitizer.  Kernels run on the host: one std::thread per GPU thread
// of a block, blocks one after another; __shared__ becomes static storage
// (shared by the threads of the running block); __syncthreads is a barrier
// that exited threads drop out of.
#pragma once
#include <algorithm>
#include <atomic>
#include <barrier>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <memory>
#include <stdexcept>
#include <mutex>
#include <thread>
#include <tuple>
#include <vector>

#define __global__
#define __device__
#define __host__
#define __forceinline__ inline
#define __launch_bounds__(...)
#define __shared__ static
#define __align__(n) alignas(n)

struct float4 { float x, y, z, w; };
struct float2 { float x, y; };
inline float4 make_float4(float a, float b, float c, float d) { return float4{a, b, c, d}; }
inline float2 make_float2(float a, float b) { return float2{a, b}; }
struct int2 { int x, y; };
struct int4 { int x, y, z, w; };
inline int4 make_int4(int a, int b, int c, int d) { return int4{a, b, c, d}; }
struct uint4 { unsigned x, y, z, w; };

struct dim3 {
  unsigned x = 1, y = 1, z = 1;
  dim3(unsigned a = 1, unsigned b = 1, unsigned c = 1) : x(a), y(b), z(c) {}
};
struct uint3e { unsigned x = 0, y = 0, z = 0; };
inline thread_local uint3e threadIdx, blockIdx;
inline thread_local dim3 blockDim, gridDim;

namespace emu {
inline std::barrier<> *bar = nullptr;
inline std::mutex atom_mu;
inline std::vector<float> shfl_buf;
inline void sync() { bar->arrive_and_wait(); }
}  // namespace emu

inline void __syncthreads() { emu::sync(); }
inline float __shfl_down(float v, int off, int width = 64) {
  const unsigned t = threadIdx.x;
  emu::shfl_buf[t] = v;
  emu::sync();
  const unsigned src = t + off;
  float r = v;
  if ((t % width) + off < (unsigned)width && src < blockDim.x) r = emu::shfl_buf[src];
  emu::sync();
  return r;
}
inline float __shfl(float v, int lane, int width = 64) {
  const unsigned t = threadIdx.x;
  emu::shfl_buf[t] = v;
  emu::sync();
  const float r = emu::shfl_buf[t / width * width + lane];
  emu::sync();
  return r;
}
inline int __syncthreads_or(int x) {
  emu::shfl_buf[threadIdx.x] = x ? 1.0f : 0.0f;
  emu::sync();
  int any = 0;
  for (unsigned t = 0; t < blockDim.x; t++) any |= emu::shfl_buf[t] != 0.0f;
  emu::sync();
  return any;
}
inline float unsafeAtomicAdd(float *p, float v) {
  std::lock_guard<std::mutex> g(emu::atom_mu);
  const float old = *p;
  *p = old + v;
  return old;
}
inline float atomicAdd(float *p, float v) { return unsafeAtomicAdd(p, v); }
#define __builtin_amdgcn_sched_barrier(m) ((void)0)
// as v_rcp_f32: one ulp off for about one significand in nine, right for the
// all-ones one
inline float __builtin_amdgcn_rcpf(float x) {
  const float y = 1.0f / x;
  unsigned b, r;
  std::memcpy(&b, &x, 4);
  std::memcpy(&r, &y, 4);
  b &= 0x7fffffu;
  const unsigned h = (b * 2654435761u) >> 16;
  if (b != 0x7fffffu && b != 0 && h % 9 == 0) r += h % 2 ? 1 : -1;
  float out;
  std::memcpy(&out, &r, 4);
  return out;
}
inline float sqrtf_(float x) { return std::sqrt(x); }

typedef int hipError_t;
enum { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorNotSupported = 801 };
typedef void *hipStream_t;
typedef void *hipEvent_t;
typedef void *hipGraph_t;
typedef void *hipGraphExec_t;
enum hipMemcpyKind { hipMemcpyHostToDevice, hipMemcpyDeviceToHost, hipMemcpyDeviceToDevice, hipMemcpyHostToHost };
enum { hipStreamCaptureModeThreadLocal = 0, hipEventDisableTiming = 2 };

inline const char *hipGetErrorString(hipError_t e) { return e ? "emulated error" : "no error"; }
inline hipError_t hipGetLastError() { return hipSuccess; }
namespace emu {
inline std::atomic<long> mallocs_left{-1};  // allocations that still succeed; -1: all
}
// for tests: the n-th allocation from now on and all after it fail (n < 0: none)
extern "C" __attribute__((used)) inline void emu_allow_mallocs(long n) { emu::mallocs_left = n; }
template <class T> inline hipError_t hipMalloc(T **p, size_t n) {
  *p = nullptr;
  if (emu::mallocs_left == 0) return hipErrorOutOfMemory;
  if (emu::mallocs_left > 0) emu::mallocs_left--;
  *p = static_cast<T *>(std::malloc(n ? n : 1));
  std::memset(*p, 0x7f, n);  // poison: reads of never-written device memory show up as huge values
  return hipSuccess;
}
inline hipError_t hipFree(void *p) { std::free(p); return hipSuccess; }
inline hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { std::memcpy(d, s, n); return hipSuccess; }
inline hipError_t hipStreamCreate(hipStream_t *s) { *s = (void *)1; return hipSuccess; }
inline hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
namespace emu {
inline std::atomic<int> launches{0};  // under way, of all host threads
inline std::atomic<long> launched{0}, waited{0}, most_queued{0};  // in all; waited for; most that were not
struct Event { long at = 0; };
}
// for tests: the most launches that were queued without a wait since the last call
extern "C" __attribute__((used)) inline long emu_most_queued() { return emu::most_queued.exchange(0); }
// what other host threads have launched ends before this returns
inline hipError_t hipStreamSynchronize(hipStream_t) {
  while (emu::launches) std::this_thread::yield();
  emu::waited = emu::launched.load();
  return hipSuccess;
}
inline hipError_t hipEventCreate(hipEvent_t *e) { *e = new emu::Event(); return hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
inline hipError_t hipEventDestroy(hipEvent_t e) { delete static_cast<emu::Event *>(e); return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
  static_cast<emu::Event *>(e)->at = emu::launched;
  return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t e) {
  emu::waited = std::max(emu::waited.load(), static_cast<emu::Event *>(e)->at);
  return hipSuccess;
}
// a launch takes one millisecond
inline hipError_t hipEventElapsedTime(float *ms, hipEvent_t a, hipEvent_t b) {
  *ms = static_cast<float>(static_cast<emu::Event *>(b)->at - static_cast<emu::Event *>(a)->at);
  return hipSuccess;
}
namespace emu {
// stream capture: launches and async copies are recorded as closures and
// replayed by hipGraphLaunch
struct Graph { std::vector<std::function<void()>> ops; };
inline thread_local Graph *capturing = nullptr;
}  // namespace emu
inline hipError_t hipStreamBeginCapture(hipStream_t, int) { emu::capturing = new emu::Graph(); return hipSuccess; }
inline hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) { *g = emu::capturing; emu::capturing = nullptr; return hipSuccess; }
inline hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t g, void *, void *, size_t) {
  *e = new emu::Graph(*static_cast<emu::Graph *>(g));
  return hipSuccess;
}
inline hipError_t hipGraphDestroy(hipGraph_t g) { delete static_cast<emu::Graph *>(g); return hipSuccess; }
inline hipError_t hipGraphExecDestroy(hipGraphExec_t g) { delete static_cast<emu::Graph *>(g); return hipSuccess; }
inline hipError_t hipGraphLaunch(hipGraphExec_t g, hipStream_t) {
  for (auto &op : static_cast<emu::Graph *>(g)->ops) op();
  return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
  if (emu::capturing) emu::capturing->ops.push_back([d, s, n] { std::memcpy(d, s, n); });
  else std::memcpy(d, s, n);
  return hipSuccess;
}

namespace emu {
template <class... P, class... A>
void launch(void (*k)(P...), dim3 grid, dim3 block, size_t, hipStream_t, A &&...args) {
  const unsigned nb = grid.x * grid.y * grid.z, nt = block.x * block.y * block.z;
  if (nb == 0 || nt == 0 || nt > 1024) { std::fprintf(stderr, "EMU: bad launch %u x %u\n", nb, nt); std::abort(); }
  std::tuple<P...> params(static_cast<P>(args)...);
  if (capturing) {
    capturing->ops.push_back([k, grid, block, params] {
      std::apply([&](auto... a) { launch(k, grid, block, 0, nullptr, a...); }, params);
    });
    return;
  }
  static std::mutex one_at_a_time;  // streams of several host threads
  launches++;
  launched++;
  most_queued = std::max(most_queued.load(), launched - waited);
  std::lock_guard<std::mutex> lock(one_at_a_time);
  shfl_buf.assign(nt, 0.0f);
  // nt pool threads run the blocks one after another; each block gets a fresh
  // barrier for __syncthreads, which a thread leaves when its kernel returns
  std::barrier<> start(nt + 1), done(nt + 1);
  std::unique_ptr<std::barrier<>> br;
  unsigned cur = 0;
  bool stop = false;
  std::vector<std::thread> th;
  th.reserve(nt);
  for (unsigned t = 0; t < nt; t++)
    th.emplace_back([&, t] {
      threadIdx.x = t; threadIdx.y = 0; threadIdx.z = 0;
      blockDim = block; gridDim = grid;
      for (;;) {
        start.arrive_and_wait();
        if (stop) return;
        blockIdx.x = cur; blockIdx.y = 0; blockIdx.z = 0;
        std::apply(k, params);
        br->arrive_and_drop();
        done.arrive_and_wait();
      }
    });
  for (unsigned b = 0; b < nb; b++) {
    br = std::make_unique<std::barrier<>>(nt);
    bar = br.get();
    cur = b;
    start.arrive_and_wait();
    done.arrive_and_wait();
  }
  stop = true;
  start.arrive_and_wait();
  for (auto &x : th) x.join();
  launches--;
}
}  // namespace emu
#define hipLaunchKernelGGL(...) emu::launch(__VA_ARGS__)
#define HIP_SYMBOL(x) (&(x))
inline hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
inline hipError_t hipSetDevice(int) { return hipSuccess; }
inline hipError_t hipGetSymbolAddress(void **p, const void *sym) { *p = const_cast<void *>(sym); return hipSuccess; }
