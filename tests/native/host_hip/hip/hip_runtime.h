// A host stand-in for <hip/hip_runtime.h>: enough of HIP to compile a kernel
// source for the CPU and run it there, so that what a kernel does between its
// barriers can be tested in orders that a GPU takes rarely.
//
// Every thread of a workgroup is a fiber.  A wave's lanes meet at each cross-lane
// operation and at wave barriers; between those the lanes run one after another,
// so LDS traffic between lanes that no such point orders is not ordered here
// either.  A wave runs until all its lanes wait at a workgroup barrier, and only
// then the next wave, in the order host_hip_order() chose: a wave that leaves a
// barrier early is a whole phase ahead of the others.  Waves that meet at
// different barriers of the source end the process.  LDS is a static
// object, atomics are plain operations (one thread of the host runs it all),
// and a launch returns when the grid has run.
#pragma once

#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <ucontext.h>

#include <functional>
#include <vector>

#define __global__
#define __device__
#define __host__
#define __forceinline__ inline
#define __launch_bounds__(...)
#define amdgpu_waves_per_eu(...) unused
#define __shared__ static

struct dim3 {
  unsigned x, y, z;
  dim3(unsigned x = 1, unsigned y = 1, unsigned z = 1) : x(x), y(y), z(z) {}
};
struct alignas(16) uint4 { uint32_t x, y, z, w; };
struct alignas(16) int4 { int32_t x, y, z, w; };
struct alignas(16) float4 { float x, y, z, w; };
inline uint4 make_uint4(uint32_t x, uint32_t y, uint32_t z, uint32_t w) { return {x, y, z, w}; }

typedef void* hipStream_t;
typedef int hipError_t;
constexpr hipError_t hipSuccess = 0;
constexpr int hipDeviceAttributeMultiprocessorCount = 0;
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
inline hipError_t hipDeviceGetAttribute(int* v, int, int) { *v = 256; return hipSuccess; }

template <class T> inline T min(T a, T b) { return b < a ? b : a; }
template <class T> inline T max(T a, T b) { return a < b ? b : a; }
inline uint32_t __float_as_uint(float f) { return __builtin_bit_cast(uint32_t, f); }
inline float __uint_as_float(uint32_t u) { return __builtin_bit_cast(float, u); }
inline int __popc(uint32_t v) { return __builtin_popcount(v); }
inline int __clz(int v) { return v ? __builtin_clz(static_cast<unsigned>(v)) : 32; }
inline uint32_t atomicAdd(uint32_t* p, uint32_t v) { const uint32_t o = *p; *p = o + v; return o; }
inline uint32_t atomicOr(uint32_t* p, uint32_t v) { const uint32_t o = *p; *p = o | v; return o; }

static dim3 threadIdx(0, 0, 0), blockIdx(0, 0, 0);

namespace host_hip {

constexpr int kWave = 64;
constexpr size_t kStack = 128 << 10;
enum State { kRun, kAtWave, kAtBarrier, kDone };

struct Slot {          // a lane's operands of a cross-lane operation
  uint64_t op = 0;     // its number (0: none yet)
  int kind = 0;
  uint32_t v[24] = {};
};
struct Fiber {
  ucontext_t ctx;
  State state;
  int line;            // of the barrier it waits at
  uint64_t ops;        // cross-lane operations so far
  Slot slot[2];        // by parity: a lane is at most one operation ahead of another's reads
};

inline std::vector<Fiber> fibers;
inline std::vector<char> stacks;
inline std::function<void()> body;
inline ucontext_t scheduler;
inline int current, wave_desc, lane_desc;

[[noreturn]] inline void fail(const char* what, int a, int b) {
  fprintf(stderr, "host_hip: %s (%d, %d)\n", what, a, b);
  abort();
}
inline void entry() {
  body();
  fibers[current].state = kDone;
  swapcontext(&fibers[current].ctx, &scheduler);
}
inline void wait(State s) {
  fibers[current].state = s;
  swapcontext(&fibers[current].ctx, &scheduler);
}
inline void barrier(int line) {
  fibers[current].line = line;
  wait(kAtBarrier);
}

// Deposit this lane's n dwords and wait for the wave's other lanes.
inline void meet(int kind, const uint32_t* v, int n) {
  Fiber& f = fibers[current];
  Slot& s = f.slot[++f.ops & 1];
  s.op = f.ops;
  s.kind = kind;
  memcpy(s.v, v, 4 * n);
  wait(kAtWave);
}
// Lane l's operands of the operation this lane is in, or none if it ended before.
inline const Slot* lane_slot(int l) {
  const Fiber& me = fibers[current];
  const int i = current / kWave * kWave + l;
  if (i >= static_cast<int>(fibers.size())) return nullptr;
  const Slot& s = fibers[i].slot[me.ops & 1];
  if (s.op != me.ops) return nullptr;
  if (s.kind != me.slot[me.ops & 1].kind) fail("lanes of a wave in different operations", s.kind, l);
  return &s;
}
inline int lane() { return current % kWave; }
inline uint32_t lane_value(int l, int i) {
  const Slot* s = lane_slot(l);
  return s ? s->v[i] : 0u;
}

// Run wave w until every lane waits at a barrier or has ended.
inline void run_wave(int w) {
  const int lo = w * kWave, hi = min(lo + kWave, static_cast<int>(fibers.size()));
  for (;;) {
    for (int j = lo; j < hi; j++) {
      current = lane_desc ? lo + hi - 1 - j : j;
      if (fibers[current].state != kRun) continue;
      threadIdx = dim3(current, 0, 0);
      swapcontext(&scheduler, &fibers[current].ctx);
    }
    bool at_wave = false;
    for (int i = lo; i < hi; i++) at_wave |= fibers[i].state == kAtWave;
    if (!at_wave) return;
    for (int i = lo; i < hi; i++) {
      if (fibers[i].state == kAtBarrier) fail("a lane at a barrier, others in a cross-lane operation", fibers[i].line, i);
      if (fibers[i].state == kAtWave) fibers[i].state = kRun;
    }
  }
}

inline void launch(dim3 grid, dim3 block, std::function<void()> kernel) {
  body = kernel;
  const int n = static_cast<int>(block.x), waves = (n + kWave - 1) / kWave;
  fibers.resize(n);
  stacks.resize(n * kStack);
  for (unsigned z = 0; z < grid.z; z++)
    for (unsigned y = 0; y < grid.y; y++)
      for (unsigned x = 0; x < grid.x; x++) {
        blockIdx = dim3(x, y, z);
        for (int i = 0; i < n; i++) {
          Fiber& f = fibers[i];
          f.state = kRun;
          f.ops = 0;
          f.slot[0].op = f.slot[1].op = 0;
          getcontext(&f.ctx);
          f.ctx.uc_stack.ss_sp = &stacks[i * kStack];
          f.ctx.uc_stack.ss_size = kStack;
          f.ctx.uc_link = nullptr;
          makecontext(&f.ctx, entry, 0);
        }
        for (bool live = true; live;) {
          for (int w = 0; w < waves; w++) run_wave(wave_desc ? waves - 1 - w : w);
          live = false;
          int line = 0;
          for (Fiber& f : fibers)
            if (f.state == kAtBarrier) {
              if (live && f.line != line) fail("waves at different barriers", line, f.line);
              live = true;
              line = f.line;
              f.state = kRun;
            }
        }
      }
}

struct Pair {
  uint32_t v[2];
  uint32_t operator[](int i) const { return v[i]; }
};
inline float fp8(uint32_t b) {   // E4M3 (OCP)
  const int e = (b >> 3) & 15, m = b & 7;
  if ((b & 127) == 127) return NAN;
  const float f = e ? ldexpf(1.f + m / 8.f, e - 7) : ldexpf(m / 8.f, -6);
  return b & 128 ? -f : f;
}

}  // namespace host_hip

// Order of the waves of a workgroup and of the lanes of a wave: ascending, or descending.
extern "C" inline void host_hip_order(int wave_desc, int lane_desc) {
  host_hip::wave_desc = wave_desc;
  host_hip::lane_desc = lane_desc;
}
extern "C" __attribute__((used)) void (*const host_hip_order_ref)(int, int) = host_hip_order;

#define __syncthreads() host_hip::barrier(__LINE__)
#define hipLaunchKernelGGL(kernel, grid, block, lds, stream, ...) \
  host_hip::launch(grid, block, [&] { kernel(__VA_ARGS__); })

// The gfx950 builtins, which the build renames from __builtin_amdgcn_* to host_amdgcn_*.
inline uint64_t __ballot(bool p) {
  const uint32_t v = p;
  host_hip::meet(1, &v, 1);
  uint64_t m = 0;
  for (int l = 0; l < host_hip::kWave; l++) m |= static_cast<uint64_t>(host_hip::lane_value(l, 0)) << l;
  return m;
}
inline int host_amdgcn_readlane(int value, int from) {
  const uint32_t v = value;
  host_hip::meet(2, &v, 1);
  return static_cast<int>(host_hip::lane_value(from, 0));
}
inline int host_amdgcn_readfirstlane(int value) {
  const uint32_t v = value;
  host_hip::meet(3, &v, 1);
  for (int l = 0; l < host_hip::kWave; l++)
    if (const host_hip::Slot* s = host_hip::lane_slot(l)) return static_cast<int>(s->v[0]);
  return value;
}
inline int host_amdgcn_ds_bpermute(int addr, int value) {
  const uint32_t v = value;
  host_hip::meet(4, &v, 1);
  return static_cast<int>(host_hip::lane_value((addr >> 2) & 63, 0));
}
inline int host_amdgcn_update_dpp(int old, int value, int ctrl, int row_mask, int, bool) {
  const uint32_t v = value;
  host_hip::meet(5, &v, 1);
  const int l = host_hip::lane(), row = l / 16, i = l % 16;
  int from = -1;
  if (ctrl < 0x100) from = (l & ~3) + ((ctrl >> (2 * (l & 3))) & 3);                     // quad_perm
  else if (ctrl > 0x110 && ctrl < 0x120) from = i >= ctrl - 0x110 ? l - (ctrl - 0x110) : -1;   // row_shr
  else if (ctrl > 0x120 && ctrl < 0x130) from = 16 * row + ((i - (ctrl - 0x120)) & 15);        // row_ror
  else if (ctrl == 0x142) from = row > 0 ? 16 * row - 1 : -1;                                  // row_bcast15
  else if (ctrl == 0x143) from = row > 1 ? 31 : -1;                                            // row_bcast31
  else host_hip::fail("unknown DPP control", ctrl, l);
  return (row_mask >> row) & 1 && from >= 0 ? static_cast<int>(host_hip::lane_value(from, 0)) : old;
}
inline host_hip::Pair host_amdgcn_swap(int kind, int rows, uint32_t a, uint32_t b) {
  const uint32_t v[2] = {a, b};
  host_hip::meet(kind, v, 2);
  const int l = host_hip::lane();
  return l & rows ? host_hip::Pair{{host_hip::lane_value(l - rows, 1), b}}
                  : host_hip::Pair{{a, host_hip::lane_value(l + rows, 0)}};
}
inline host_hip::Pair host_amdgcn_permlane16_swap(uint32_t a, uint32_t b, bool, bool) { return host_amdgcn_swap(6, 16, a, b); }
inline host_hip::Pair host_amdgcn_permlane32_swap(uint32_t a, uint32_t b, bool, bool) { return host_amdgcn_swap(7, 32, a, b); }
inline float host_amdgcn_fmed3f(float x, float lo, float hi) { return x != x ? fminf(lo, hi) : fmaxf(lo, fminf(x, hi)); }
inline void host_amdgcn_fence(int, const char*) {}
inline void host_amdgcn_sched_barrier(int) {}
inline void host_amdgcn_wave_barrier() { host_hip::meet(8, nullptr, 0); }
// FP8 products of 16 rows x 16 columns over 128 dims: lane (g, c) holds 32 dims of row and column c.
template <class A, class C>
inline C host_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(const A& a, const A& b, C acc, int, int, int, int, int, int) {
  uint32_t v[16];
  for (int i = 0; i < 8; i++) { v[i] = a[i]; v[8 + i] = b[i]; }
  host_hip::meet(9, v, 16);
  const int g = host_hip::lane() / 16, c = host_hip::lane() % 16;
  for (int e = 0; e < 4; e++)
    for (int kg = 0; kg < 4; kg++)
      for (int i = 0; i < 32; i++)
        acc[e] += host_hip::fp8(host_hip::lane_value(16 * kg + 4 * g + e, i / 4) >> (8 * (i % 4)) & 255) *
                  host_hip::fp8(host_hip::lane_value(16 * kg + c, 8 + i / 4) >> (8 * (i % 4)) & 255);
  return acc;
}
