/*
 * slb_step2.h -- interface of the two-step kernel (slb_step2.hip) to the
 * single-lattice path (slb_dev.hip).
 */
#ifndef SLB_STEP2_H
#define SLB_STEP2_H

#include "slb_kern.h"

/* jt x kt nodes of a plane per block, ci planes; their counts */
struct Step2Plan {
  int jt, kt, ci, njt, nkt, nch;
};

/* Most columns (tile and rim) of a block: a thread and 2 x 12 values of the
 * CU's 160 KB of LDS each (FP32 98 KB; FP64 148 KB, and 168 registers, of
 * which three waves per SIMD fit). */
template <typename T> struct Step2Cfg { enum { NTHR = sizeof(T) == 4 ? 1024 : 768 }; };

struct Step2Args {
  const void *src;
  void *dst;
  const uint16_t *flags;
  const void *bx, *by, *bz;
  bool nt;
  int bf;
  Step2Plan plan;
};

int slbd_step2_plan(int esi, int esj, int esk, int prec, Step2Plan *best);
void slbd_step2_launch(const Step2Args *a, const PhysArgs &A, const Geom &G, int prec,
                       hipStream_t st);

#endif
