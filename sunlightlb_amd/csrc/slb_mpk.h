/*
 * slb_mpk.h -- what the moment-propagation kernels of slb_dev.hip (factors,
 * single steps) and slb_mp2.hip (two steps per pass) share: the layout of the
 * link factors and the compact records.
 */
#ifndef SLB_MPK_H
#define SLB_MPK_H

#include "slb_kern.h"

struct MPArgs {
  double rho0, alpha, pads;
  int axis;
};

/* The share of what arrives that a solid node keeps, from its MP flags word
 * (bit 15: it adsorbs, bit 16: a boundary node). */
template <typename T>
__device__ __forceinline__ T mp_kept(uint32_t f, const MPArgs &A) {
  return (f & (1u << 15)) ? T(1) : ((f & (1u << 16)) && A.pads > 0.0) ? T(A.pads) : T(0);
}

/* weights in tiles of 1024 nodes: runs of 1024 four-value vectors (weights
 * 0-3, 4-7, 8-11) and one of 1024 three-value vectors (12-14), so a wave's
 * load of one run is contiguous */
template <typename I>
__device__ __forceinline__ I wt_idx(int c, I x) {
  const I tile = (x >> POP_SHIFT) * I(15 * POP_TILE), n = x & I(POP_TILE - 1);
  return c < 3 ? tile + (I(c) * I(POP_TILE) + n) * I(4) : tile + I(12 * POP_TILE) + n * I(3);
}
template <typename T>
struct __attribute__((aligned(sizeof(T)))) Wt3 {
  T a, b, c;
};

/* Compact node records of a run on link factors: {P} or {P, m1, m2} without
 * the 1/rho slot, which only the factors use (12 bytes per node FP32 with
 * moments instead of 16). */
template <typename T, int NM> struct CRec;
template <typename T> struct __attribute__((aligned(sizeof(T)))) CRec<T, 3> { T p, m1, m2; };
template <typename T> struct __attribute__((aligned(sizeof(T)))) CRec<T, 1> { T p; };

/* jt x kt nodes of a plane per block, ci planes; their counts (ci 0: no plan) */
struct MP2Plan {
  int jt, kt, ci, njt, nkt, nch;
};

extern "C" int slbd_mp2_plan(int esi, int esj, int esk, int prec, int nmom, MP2Plan *best);
extern "C" int slbd_mp2_pays(int esj, int esk, int nmom, const MP2Plan *p);
/* two steps from records q to records qout on the factors wt */
void slbd_mp2_launch(const void *wt, const void *q, void *qout, const uint32_t *mpf, int prec,
                     int nmom, const Geom &G, const MPArgs &A, const MP2Plan &Q, hipStream_t st);

#endif
