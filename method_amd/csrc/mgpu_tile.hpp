// What the tiled sweeps of the step (mgpu_kernels.hip) and of the ensemble
// (mgpu_batch.hip) share: the deal of face items to threads and global accesses
// at a 32-bit offset from a scalar base.
#pragma once

#include "mgpu_kernels.hpp"

namespace mgpu {

constexpr int kThreads = 256;  // per workgroup

// How the (variable, face) items of a tile phase go to the threads, NV
// variables of kFaces faces each, face f of variable v starting its stencil at
// LDS offset v VSTRIDE + off(f). Where the faces fill the threads once (or
// half of them, for an even NV), a thread keeps one face and takes it through
// its variables, pass by pass: its LDS addresses are one base plus constants,
// and the few faces left over make one or two passes more. Dealing the items
// out in one flat row took a division and a bounds check per item and half,
// and the sweeps were bound by VALU issue then (79-85 % of the cycles): with this
// and the 32-bit offsets below the fused y + z launch has 2,090 FP64 of 2,625
// VALU instructions instead of 3,069, the x sweep 948 of 1,108 instead of
// 1,292, and the KH 256^3 WENO5 step went from 5.82-5.88 to 5.44 ms, 128^3
// WENO3 from 639 to 590 us, 1024^2 WENO3 from 228 to 209 us.
// Tiles of fewer faces keep the flat row, which leaves fewer threads idle.
template <int NV, int FACES, int VSTRIDE, class Off>
struct FaceItems {
  static constexpr int NB = FACES >= kThreads ? kThreads : (FACES >= kThreads / 2 && NV % 2 == 0 ? kThreads / 2 : 0);
  static constexpr int H = NB ? kThreads / NB : 1;      // variables taken side by side
  static constexpr int kRegular = NB ? NV / H : 0;      // passes over them
  static constexpr int kRest = FACES - NB;              // faces left over per variable (all of them in the flat row)
  static constexpr int kRestItems = NV * kRest;
  static constexpr int kPasses = kRegular + (kRestItems + kThreads - 1) / kThreads;
  static_assert(H * kRegular == (NB ? NV : 0), "whole passes");
  unsigned tid, reg_lds, reg_item;
  __device__ __forceinline__ explicit FaceItems(unsigned t) : tid(t), reg_lds(0), reg_item(0) {
    if (NB) {
      const unsigned f = t % (NB ? NB : 1), h = t / (NB ? NB : 1);
      reg_lds = Off::at(f) + h * VSTRIDE;
      reg_item = f + h * FACES;
    }
  }
  // Whether the thread has an item in pass k (a constant after unrolling for
  // the regular passes), its stencil's LDS offset and its place v FACES + f.
  __device__ __forceinline__ bool has(int k) const { return k < kRegular || tid + (k - kRegular) * kThreads < kRestItems; }
  __device__ __forceinline__ unsigned lds(int k) const {
    if (k < kRegular) return reg_lds + k * H * VSTRIDE;
    const unsigned e = tid + (k - kRegular) * kThreads, v = e / kRest;
    return Off::at(NB + e - v * kRest) + v * VSTRIDE;
  }
  __device__ __forceinline__ unsigned item(int k) const {
    if (k < kRegular) return reg_item + k * H * FACES;
    const unsigned e = tid + (k - kRegular) * kThreads, v = e / kRest;
    return NB + e - v * kRest + v * FACES;
  }
};

// The end of a face pass: its results are formed here, and no LDS read of a
// later pass moves up past it. Without it the passes pile up their stencils in
// registers (196-226 VGPRs in the x sweep, 140 spilled in the fused y + z one).
__device__ __forceinline__ void pass_end(double &a) { asm volatile("" : "+v"(a) : : "memory"); }
__device__ __forceinline__ void pass_end(double &a, double &b) { asm volatile("" : "+v"(a), "+v"(b) : : "memory"); }

// A cell's place in a variable's plane as a 32-bit byte offset from the
// plane's base: base and offset then are a scalar pair and one register of the
// access itself, where a 64-bit index takes an addition or two per access. Grids
// of more than 2^29 cells are refused (kMaxCells).
// The empty asm keeps the base a scalar pair: left to itself the compiler adds
// the offset first and then steps that sum from plane to plane.
// (It hides the pointer's origin too, so the address space is stated.)
typedef __attribute__((address_space(1))) double gdouble;
typedef __attribute__((address_space(1))) char gchar;
__device__ __forceinline__ gdouble *at_offset(const double *plane, unsigned o) {
  gdouble *p = (gdouble *)plane;
  asm("" : "+s"(p));
  return (gdouble *)((gchar *)p + o);
}
__device__ __forceinline__ double ld(const double *p, unsigned o) { return *at_offset(p, o); }
__device__ __forceinline__ double ld_nt(const double *p, unsigned o) { return __builtin_nontemporal_load(at_offset(p, o)); }
__device__ __forceinline__ void st(double *p, unsigned o, double x) { *at_offset(p, o) = x; }
__device__ __forceinline__ void st_nt(double *p, unsigned o, double x) { __builtin_nontemporal_store(x, at_offset(p, o)); }

// Cells whose cons2prim failed in a stage, for the retry that ends it: their
// list, its length fail[kFailCount] and a flag per cell, which is up if it equals
// this stage's mark. A retry that is over raises the mark (fail[kFailMark] + 1,
// up to 255) instead of taking the flags down again: that was the last
// workgroup's work, and with every cell of 200^3 failed a cons2prim took 16.7 ms
// where it takes 4.2 now (4.6 with a launch of 64 workgroups for the flags). The
// mark has its own cache line: read from the line that the length's atomics keep
// moving, it cost as much again as the Newton solves. Zeroed memory is an empty
// list.
constexpr int kFailMarks = 255;

__device__ __forceinline__ void note_failed(int *fail, long long *list, unsigned char *flag, long long q) {
  list[atomicAdd(&fail[kFailCount], 1)] = q;
  flag[q] = (unsigned char)(fail[kFailMark] + 1);
}

// Empties the list, by one workgroup of kThreads; n: the number of flags, which
// go down only when the marks are used up, once in 255 lists (hipMalloc aligns
// them, so 16 at a time).
__device__ __forceinline__ void forget_failed(int *fail, unsigned char *flag, long long n) {
  const int mark = fail[kFailMark] + 1;
  if (mark == kFailMarks) {
    for (long long k = threadIdx.x; k < n / 16; k += kThreads) reinterpret_cast<uint4 *>(flag)[k] = uint4{0, 0, 0, 0};
    for (long long k = n / 16 * 16 + threadIdx.x; k < n; k += kThreads) flag[k] = 0;
  }
  __syncthreads();  // every thread has read the mark
  if (threadIdx.x == 0) {
    fail[kFailCount] = 0;
    fail[kFailDone] = 0;
    fail[kFailMark] = mark == kFailMarks ? 0 : mark;
  }
}

// The end of a retry of a non-empty list over the whole grid: the last workgroup
// to get here empties the list. No workgroup does so before all have read its
// length and the flags, since each counts itself after that.
__device__ __forceinline__ void end_retry(int *fail, unsigned char *flag, long long n) {
  __shared__ int s_last;
  __threadfence();
  __syncthreads();
  if (threadIdx.x == 0) s_last = atomicAdd(&fail[kFailDone], 1) == (int)gridDim.x - 1;
  __syncthreads();
  if (!s_last) return;
  __threadfence();
  forget_failed(fail, flag, n);
}

}  // namespace mgpu
