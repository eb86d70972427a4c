// hip_cpu_wave.h -- test infrastructure: hip_cpu_shim.h with what the
// matrix-core kernels of mdff_amd/csrc/fit.hip need on top, so that the
// iterations that run on the GPU run on the host too: waves of 64 lanes whose
// cross-lane operations meet, shared arrays of a workgroup, and memory that ends
// at a page no access may touch, so that a read or write past the end of a device
// array or of a launch's LDS ends the process.  Only tests/test_fit_wave_cpu.py
// builds and loads it.
#pragma once
#include <cstdio>
#include <map>
#include <memory>
#include <mutex>
#include <sys/mman.h>
#include <unistd.h>

#define __HIPCC__ 1
#define __syncthreads shim_syncthreads
#define hipMalloc shim_malloc
#define hipFree shim_free
#include "hip_cpu_shim.h"
#undef __syncthreads
#undef hipMalloc
#undef hipFree
#undef hipLaunchKernelGGL
#undef __shared__
#define __shared__ static thread_local   // a workgroup's lanes are contexts of one thread

// memory that ends (to 16 bytes) at a guard page, filled with a pattern that is
// NaN as a double
struct GuardMem {
  char* base;
  size_t bytes;
};
inline GuardMem guard_map(size_t n) {
  const size_t page = (size_t)sysconf(_SC_PAGESIZE), body = (std::max<size_t>(n, 16) + 15 + page - 1) / page * page;
  char* p = (char*)mmap(nullptr, body + page, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0);
  if (p == (char*)MAP_FAILED || mprotect(p + body, page, PROT_NONE) != 0) abort();
  memset(p, 0xff, body);
  return {p, body};
}
inline char* guard_end(const GuardMem& g, size_t n) { return g.base + g.bytes - ((n + 15) & ~(size_t)15); }

inline std::mutex g_mem_lock;
inline std::map<void*, GuardMem> g_mem;
inline hipError_t hipMalloc(void** p, size_t n) {
  const GuardMem g = guard_map(n);
  *p = guard_end(g, n);
  std::lock_guard<std::mutex> l(g_mem_lock);
  g_mem[*p] = g;
  return 0;
}
inline hipError_t hipFree(void* p) {
  std::lock_guard<std::mutex> l(g_mem_lock);
  auto it = g_mem.find(p);
  if (it == g_mem.end()) abort();
  munmap(it->second.base, it->second.bytes + (size_t)sysconf(_SC_PAGESIZE));
  g_mem.erase(it);
  return 0;
}
#define hipHostMallocMapped 1
#define hipHostMallocCoherent 2
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return hipMalloc(p, n); }
inline hipError_t hipHostFree(void* p) { return hipFree(p); }
inline hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned) { *d = h; return 0; }
#define hipFuncAttributeMaxDynamicSharedMemorySize 1
inline hipError_t hipFuncSetAttribute(const void*, int, int) { return 0; }
inline void __threadfence_system() { std::atomic_thread_fence(std::memory_order_seq_cst); }
#define __builtin_amdgcn_sched_barrier(x)
struct double2 {
  double x, y;
};

// lanes wait for their wave (cross-lane operations) or their workgroup
enum { LANE_RUN, LANE_WAVE, LANE_BLOCK, LANE_DONE };
struct WaveGroup {
  std::vector<char> state;
  std::vector<double> xa, xb;    // operands of the waves' operations, two in turn
  std::vector<int> turn;         // per lane
};
inline thread_local WaveGroup* g_wave = nullptr;
inline void lane_wait(int why) {
  g_wave->state[g_grp->cur] = (char)why;
  swapcontext(&g_grp->ctx[g_grp->cur], &g_grp->sched);
}
inline void __syncthreads() { lane_wait(LANE_BLOCK); }
// both operands of every lane of the wave, in place at a and b
inline void wave_exchange(double va, double vb, const double*& a, const double*& b) {
  const int lane = g_grp->cur, turn = (g_wave->turn[lane] ^= 1);
  const size_t nl = g_wave->state.size();
  g_wave->xa[turn * nl + lane] = va;
  g_wave->xb[turn * nl + lane] = vb;
  lane_wait(LANE_WAVE);
  a = g_wave->xa.data() + turn * nl + (lane & ~63);
  b = g_wave->xb.data() + turn * nl + (lane & ~63);
}
inline double __shfl_xor(double v, int mask) {
  const double *a, *b;
  const int lane = g_grp->cur & 63;
  wave_exchange(v, 0.0, a, b);
  return a[lane ^ mask];
}
// D = A B + C of 16 x 4 and 4 x 16: A(row = l % 16, k = l / 16), B(k = l / 16,
// col = l % 16), D(row = 4 r + l / 16, col = l % 16)
typedef double emu_f64x4 __attribute__((vector_size(32)));
inline emu_f64x4 __builtin_amdgcn_mfma_f64_16x16x4f64(double va, double vb, emu_f64x4 c, int, int, int) {
  const double *a, *b;
  const int lane = g_grp->cur & 63, col = lane & 15, g = lane >> 4;
  wave_exchange(va, vb, a, b);
  for (int r = 0; r < 4; ++r)
    for (int k = 0; k < 4; ++k) c[r] = std::fma(a[16 * k + 4 * r + g], b[16 * k + col], c[r]);
  return c;
}

template <typename F>
struct WaveLane {
  static void entry(unsigned lo, unsigned hi) {
    (*reinterpret_cast<F*>(((uintptr_t)hi << 32) | (uintptr_t)lo))();
    g_wave->state[g_grp->cur] = LANE_DONE;
  }
};

// a launch as emu_launch_f, with lds bytes of LDS and its lanes in waves
template <typename F>
void wave_launch(const char* name, F fn, dim3 g, dim3 b, size_t lds_bytes) {
  gridDim = g;
  blockDim = b;
  std::atomic<unsigned> next{0};
  auto work = [&]() {
    constexpr size_t kStack = 64 * 1024;
    const unsigned nl = b.x;
    const std::unique_ptr<char[]> stacks(new char[nl * kStack]);
    const GuardMem lds = guard_map(lds_bytes);
    EmuGroup grp;
    WaveGroup wv;
    grp.ctx.resize(nl);
    grp.done.resize(nl);
    wv.state.resize(nl);
    wv.xa.resize(2 * nl);
    wv.xb.resize(2 * nl);
    wv.turn.resize(nl);
    g_grp = &grp;
    g_wave = &wv;
    g_shared = (double*)guard_end(lds, lds_bytes);
    const unsigned nblocks = g.x * g.y * g.z;
    for (unsigned bx; (bx = next.fetch_add(1)) < nblocks;) {
      blockIdx = dim3(bx % g.x, (bx / g.x) % g.y, bx / (g.x * g.y));
      memset(lds.base, 0xff, lds.bytes);
      const uintptr_t p = reinterpret_cast<uintptr_t>(&fn);
      for (unsigned t = 0; t < nl; ++t) {
        getcontext(&grp.ctx[t]);
        grp.ctx[t].uc_stack.ss_sp = stacks.get() + t * kStack;
        grp.ctx[t].uc_stack.ss_size = kStack;
        grp.ctx[t].uc_link = &grp.sched;
        makecontext(&grp.ctx[t], (void (*)())&WaveLane<F>::entry, 2, (unsigned)(p & 0xffffffffu), (unsigned)(p >> 32));
        wv.state[t] = LANE_RUN;
      }
      for (;;) {
        for (unsigned t = 0; t < nl; ++t) {
          if (wv.state[t] != LANE_RUN) continue;
          grp.cur = (int)t;
          threadIdx = dim3(t, 0, 0);
          swapcontext(&grp.sched, &grp.ctx[t]);
        }
        // waves whose live lanes have all met go on, else the workgroup if all have
        unsigned count[4] = {0, 0, 0, 0}, released = 0;
        for (unsigned w = 0; w < nl; w += 64) {
          unsigned c[4] = {0, 0, 0, 0};
          const unsigned e = std::min(nl, w + 64);
          for (unsigned t = w; t < e; ++t) ++c[(int)wv.state[t]];
          if (c[LANE_WAVE] > 0 && c[LANE_BLOCK] == 0) {
            if (c[LANE_DONE] > 0) { fprintf(stderr, "%s: a wave operation without all lanes\n", name); abort(); }
            for (unsigned t = w; t < e; ++t) wv.state[t] = LANE_RUN;
            released += e - w;
          }
          for (int k = 0; k < 4; ++k) count[k] += c[k];
        }
        if (count[LANE_DONE] == nl) break;
        if (released) continue;
        if (count[LANE_WAVE] > 0) { fprintf(stderr, "%s: lanes wait for each other\n", name); abort(); }
        for (unsigned t = 0; t < nl; ++t)
          if (wv.state[t] == LANE_BLOCK) wv.state[t] = LANE_RUN;
      }
    }
    munmap(lds.base, lds.bytes + (size_t)sysconf(_SC_PAGESIZE));
  };
  const unsigned nth = std::min(8u, g.x * g.y * g.z);
  std::vector<std::thread> th;
  for (unsigned i = 1; i < nth; ++i) th.emplace_back(work);
  work();
  for (auto& x : th) x.join();
}
#define hipLaunchKernelGGL(K, G, B, SHM, ST, ...) \
  wave_launch(#K, [&]() { K(__VA_ARGS__); }, dim3(G), dim3(B), (size_t)(SHM))
