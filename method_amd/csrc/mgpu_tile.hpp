// What the tiled sweeps of the step (mgpu_kernels.hip) and of the ensemble
// (mgpu_batch.hip) share: the deal of face items to threads and global accesses
// at a 32-bit offset from a scalar base.
#pragma once

#include <hip/hip_runtime.h>

namespace mgpu {

constexpr int kThreads = 256;  // per workgroup

// How the (variable, face) items of a tile phase go to the threads, NV
// variables of kFaces faces each, face f of variable v starting its stencil at
// LDS offset v VSTRIDE + off(f). Where the faces fill the threads once (or
// half of them, for an even NV), a thread keeps one face and takes it through
// its variables, pass by pass: its LDS addresses are one base plus constants,
// and the few faces left over make one or two passes more. Dealing the items
// out in one flat row took a division and a bounds check per item and half,
// and the sweeps are bound by VALU issue (79-85 % of the cycles): with this
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

}  // namespace mgpu
