/*
 * slb_step2.h -- the two-step kernel (slb_step2.hip): what the batched one
 * (slb_batch.hip) shares, and its interface to the single-lattice path
 * (slb_dev.hip).
 */
#ifndef SLB_STEP2_H
#define SLB_STEP2_H

#include "slb_kern.h"

/* LDS slot of a population that leaves its column: c_x = -1 diagonals, c_x =
 * 0 axes, c_x = +1 diagonals */
__host__ __device__ constexpr int XSLOT(int l) {
  return l == 8 ? 0 : l == 10 ? 1 : l == 12 ? 2 : l == 14 ? 3
       : l == 3 ? 4 : l == 4 ? 5 : l == 5 ? 6 : l == 6 ? 7
       : l == 7 ? 8 : l == 9 ? 9 : l == 11 ? 10 : 11;
}

/* byte offset of a node's population 0 in the tiled layout, from the byte
 * offset n of the node in an array of one T per node: a shift and a
 * multiply-add (population l: l tiles further) */
template <typename T>
__device__ __forceinline__ uint32_t pop_byte(uint32_t n) {
  constexpr int SH = POP_SHIFT + (sizeof(T) == 4 ? 2 : 3);
  return n + (n >> SH) * (uint32_t)(14 * POP_TILE * sizeof(T));
}

__device__ __forceinline__ void lds_barrier() {
  /* orders LDS only: the next plane's global loads stay in flight */
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

/* jt x kt nodes of a plane per block, ci planes; their counts */
struct Step2Plan {
  int jt, kt, ci, njt, nkt, nch;
};

/* Most columns (tile and rim) of a block: a thread and 2 x 12 values of the
 * CU's 160 KB of LDS each (FP32 98 KB; FP64 148 KB, and 168 registers, of
 * which three waves per SIMD fit). */
template <typename T> struct Step2Cfg { enum { NTHR = sizeof(T) == 4 ? 1024 : 768 }; };

/* How a column's accesses are addressed: the first of these that
 * slbd_step2_mode_ok allows.
 * 0: planes of whole population tiles (plane % 1024 == 0) and buffers under
 *    4 GB: a column's in-plane byte offset is fixed and a plane adds a scalar;
 * 1: any plane, buffers under 4 GB (two more operations per load);
 * 2: as 0 with 64-bit plane offsets: the in-plane byte offset has 32 bits, so
 *    planes are under 4 GB (a lattice of few planes can exceed that while its
 *    population indices still have 31 bits);
 * 3: any plane, 31-bit population indices. */
extern "C" int slbd_step2_mode_ok(int mode, long plane, long N, int prec);
extern "C" int slbd_step2_mode(long plane, long N, int prec);   /* -1: none */

struct Step2Args {
  const void *src;
  void *dst;
  const uint16_t *flags;
  const void *bx, *by, *bz;
  bool nt;
  int bf, mode;
  Step2Plan plan;
};

extern "C" int slbd_step2_pays(int esi, int esj, int esk, int prec, const Step2Plan *p);
extern "C" int slbd_step2_plan(int esi, int esj, int esk, int prec, Step2Plan *best);
void slbd_step2_launch(const Step2Args *a, const PhysArgs &A, const Geom &G, int prec,
                       hipStream_t st);

#endif
