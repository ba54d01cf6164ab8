/*
 * slb_batch.hip -- many independent small lattices ("problems") stepped
 * together: one kernel launch per time step covers every node of every
 * problem, the step loop is captured in a HIP graph and replayed, and the
 * launch shape (block size, nodes per thread, persistent grid size) is chosen
 * by a timing autotuner.
 *
 * Each problem is one periodic box with its own size, solid map, relaxation
 * time and object velocities (one right-hand side of a resistance problem).
 * Problems of the same box share the node tables (flags, objidx).  The step
 * is the single-lattice fused pull step (bbl + propagate + collide, see
 * slb_dev.hip) with the moving-wall velocity of a solid node computed from
 * its object row (src/lbobjs.c:565-589) instead of a stored field; the force
 * variant accumulates the momentum exchange of src/lbkernel.c:464-618
 * directly into per-object force and torque (the distribf sums of
 * src/lbmeasure.c:236-263) in FP64.
 *
 * Work decomposition: a tile is a contiguous run of blockDim*NPT nodes of one
 * problem; the tile table lists (problem, first node) for all tiles.  A
 * persistent grid of G blocks walks the tile table with stride G.
 */
#include <string.h>
#include "slb_dev.h"
#include "slb_kern.h"
#include "slb_step2.h"

struct BProb {
  int esi, esj, esk, plane;
  long N;
  long pop_off;   /* first population of this problem in the arena (tiled
                     layout pidx, whole tiles per problem) */
  int jt, kt, ci; /* two-step tiles of the box (k_bstep2) */
  long wall_off;  /* first row of the wall terms, -1: walls at rest */
  long node_off;  /* first node of this problem's box in the node tables */
  int tab_off;    /* first object row (9 doubles each) */
  int nobj;
  int acc_off;    /* first object accumulator (6 doubles each) */
  int moving, stokes, skip_solid;
  double omega, comega, rho0;
  double bf[3];
};

#define BATCH_LDS_OBJ 64

/* Wall rows: per object row, in the working precision and scaled by
 * rho0/12, w0 = v - omega x pos (the velocity of the lattice origin in the
 * object's rigid motion) and omega, so that the wall velocity at solid node s
 * is U = w0 + omega x s and only c.U = c.w0 + c.(omega x s) enters a link. */
#define WROW 8

/* w_l c_l.U of link l with its solid end at (si, sj, sk) on the object of wall
 * row wr; multiply-adds written out, so that every caller gets the same value */
template <int l, typename T>
__device__ __forceinline__ T wall_term(const T *__restrict__ wr, int si, int sj, int sk) {
#pragma clang fp contract(off)
  const T sx = T(si), sy = T(sj), sz = T(sk);
  T cv = T(0);
  if (CX(l)) cv += T(CX(l)) * __builtin_elementwise_fma(-wr[5], sy, __builtin_elementwise_fma(wr[4], sz, wr[0]));
  if (CY(l)) cv += T(CY(l)) * __builtin_elementwise_fma(-wr[3], sz, __builtin_elementwise_fma(wr[5], sx, wr[1]));
  if (CZ(l)) cv += T(CZ(l)) * __builtin_elementwise_fma(-wr[4], sx, __builtin_elementwise_fma(wr[3], sy, wr[2]));
  return T(WL(l)) * cv;
}

template <typename T, bool FORCE, int NPT>
__global__ void __launch_bounds__(512)
k_bstep(const T *__restrict__ src, T *__restrict__ dst,
        const uint16_t *__restrict__ flags, const int32_t *__restrict__ objidx,
        const double *__restrict__ tab, const T *__restrict__ wtab,
        const BProb *__restrict__ probs,
        const int2 *__restrict__ tiles, int ntiles, int xcd_chunk, double *__restrict__ acc) {
  __shared__ double sacc[FORCE ? BATCH_LDS_OBJ * 6 : 1];
  /* Work items v = blockIdx.x, + gridDim.x, ...  Workgroups are dispatched
   * round robin over the 8 XCDs (each with its own L2), so block b runs on
   * XCD b % 8.  With xcd_chunk > 0 (and gridDim.x a multiple of 8) item v is
   * tile (v % 8) * xcd_chunk + v / 8: each XCD walks one contiguous eighth of
   * the tile table in order, and the rows a tile pulls from (j and i
   * neighbours, a few tiles away in a small box) were fetched into the same
   * L2 moments before instead of by another XCD. */
  const int nv = xcd_chunk > 0 ? 8 * xcd_chunk : ntiles;
  for (int v = blockIdx.x; v < nv; v += gridDim.x) {
    const int tile = xcd_chunk > 0 ? (v & 7) * xcd_chunk + (v >> 3) : v;
    if (tile >= ntiles) continue;
    const int2 td = tiles[tile];
    const BProb P = probs[td.x];
    const bool lds = FORCE && P.nobj <= BATCH_LDS_OBJ;
    if (lds) {
      for (int q = threadIdx.x; q < P.nobj * 6; q += blockDim.x) sacc[q] = 0.0;
      __syncthreads();
    }
    const T *s = src + P.pop_off;
    T *d = dst + P.pop_off;
    const uint16_t *fl = flags + P.node_off;
    const int32_t *oid = objidx + P.node_off;
    PhysArgs A;
    A.omega = P.omega; A.comega = P.comega; A.rho0 = P.rho0;
    A.stokes = P.stokes; A.skip_solid = P.skip_solid;
    A.bfx = P.bf[0]; A.bfy = P.bf[1]; A.bfz = P.bf[2];
    const bool bfon = (P.bf[0] != 0.0 || P.bf[1] != 0.0 || P.bf[2] != 0.0);
#pragma unroll
    for (int q = 0; q < NPT; q++) {
      /* 15 pop_nodes(N) < 2^31 per problem (checked at commit): 32-bit
       * node and population indices */
      const int x = td.y + q * (int)blockDim.x + (int)threadIdx.x;
      if (x >= P.N) continue;
      const int i = x / P.plane;
      const int rem = x - i * P.plane;
      const int j = rem / P.esk, k = rem - j * P.esk;
      const AxisOff32 oi = axis_off32(i, P.esi, P.plane);
      const AxisOff32 oj = axis_off32(j, P.esj, P.esk);
      const AxisOff32 ok = axis_off32(k, P.esk, 1);
      const unsigned f = fl[x];
      const bool solid = (f & FLAG_SOLID) != 0;
      T v[15];
      /* the node's loads issue at raised wave priority (8.57 -> 8.47 ms per
       * step on the 512-box batch, FP64 15.83 -> 15.20 ms) */
      __builtin_amdgcn_s_setprio(3);
      v[0] = s[pidx32(0, x)];
      Links<1, 15>::run([&](auto LL) {
        constexpr int l = decltype(LL)::value;
        const bool bb = (f >> (l - 1)) & 1u;
        const int idx = bb ? pidx32(OPP(l), x) : pidx32(l, x + nb_off<l, -1>(oi, oj, ok));
        v[l] = s[idx];
      });
      __builtin_amdgcn_s_setprio(0);
      if ((P.moving || FORCE) && (f & FLAG_LINKS)) {
        double Fx = 0.0, Fy = 0.0, Fz = 0.0;
        Links<1, 15>::run([&](auto LL) {
          constexpr int l = decltype(LL)::value;
          if ((f >> (l - 1)) & 1u) {
            const int xs = x + nb_off<l, -1>(oi, oj, ok);
            T cu = T(0);
            if (P.moving) {
              /* wall velocity U = (rho0/12)(v + w x r) of the solid end of
               * the link (vspread, src/lbobjs.c:565-589, r = s - pos without
               * minimum image) = w0 + w x s with the scaled wall row; only
               * its component along c_l enters */
              int sn = x;
              int si = i, sj = j, sk = k;
              if (!solid) {
                sn = xs;
                si = i - CX(l); si += (si < 0) ? P.esi : 0; si -= (si >= P.esi) ? P.esi : 0;
                sj = j - CY(l); sj += (sj < 0) ? P.esj : 0; sj -= (sj >= P.esj) ? P.esj : 0;
                sk = k - CZ(l); sk += (sk < 0) ? P.esk : 0; sk -= (sk >= P.esk) ? P.esk : 0;
              }
              cu = wall_term<l, T>(wtab + ((long)P.tab_off + oid[sn]) * WROW, si, sj, sk);
            }
            if (FORCE && solid) {
              const double a = (double)v[l];
              const double b = (double)s[pidx32(l, xs)];
              const double g = -2.0 * (a - b + (double)cu);
              if (CX(l)) Fx += CX(l) * g;
              if (CY(l)) Fy += CY(l) * g;
              if (CZ(l)) Fz += CZ(l) * g;
            }
            if (P.moving) v[l] += cu;
          }
        });
        if (FORCE && solid && (Fx != 0.0 || Fy != 0.0 || Fz != 0.0)) {
          const int o = oid[x];
          const double *po = tab + ((long)P.tab_off + o) * SLBD_OBJ_STRIDE;
          const double rx = i - po[0], ry = j - po[1], rz = k - po[2];
          const double tq[6] = {Fx, Fy, Fz, ry * Fz - rz * Fy, rz * Fx - rx * Fz, rx * Fy - ry * Fx};
          double *dstp = lds ? sacc + 6 * o : acc + 6 * ((long)P.acc_off + o);
#pragma unroll
          for (int c = 0; c < 6; c++) atomicAdd(dstp + c, tq[c]);
        }
      }
      if (!(P.skip_solid && solid)) {
        T jbx = T(0), jby = T(0), jbz = T(0);
        if (bfon && !solid) { jbx = T(P.bf[0]); jby = T(P.bf[1]); jbz = T(P.bf[2]); }
        collide_node<T>(v, jbx, jby, jbz, A);
      }
#pragma unroll
      /* non-temporal: a batch step streams tens of GB (8.95 -> 8.59 ms at 512 boxes) */
      for (int l = 0; l < 15; l++) __builtin_nontemporal_store(v[l], &d[pidx32(l, x)]);
    }
    if (lds) {
      __syncthreads();
      for (int q = threadIdx.x; q < P.nobj * 6; q += blockDim.x)
        if (sacc[q] != 0.0) atomicAdd(acc + 6 * (long)P.acc_off + q, sacc[q]);
      __syncthreads();
    }
  }
}

/* ---------------------------------------------------------------------- */
/* Wall terms.  The wall velocity term of a bounced link, w_l c_l.U, is the  */
/* same at every step: each node with bounced links of a box gets a place    */
/* (k_bwall_place), and each moving problem a row of 16 values per place     */
/* (value l - 1: link l's term, 0 where it does not bounce), so that a step   */
/* adds one row instead of looking up the solid end's object for each link.  */

__global__ void __launch_bounds__(256)
k_bwall_place(const uint16_t *__restrict__ flags, long N, int *__restrict__ place,
              int *__restrict__ count) {
  const long x = (long)blockIdx.x * 256 + threadIdx.x;
  const bool has = x < N && (flags[x] & FLAG_LINKS) != 0;
  const unsigned long long m = __ballot(has);
  const int lane = threadIdx.x & 63;
  int base = 0;
  if (lane == 0 && m) base = atomicAdd(count, __popcll(m));
  base = __shfl(base, 0, 64);
  if (x < N) place[x] = has ? base + __popcll(m & ((1ULL << lane) - 1)) : -1;
}

/* P: the box's first problem; blockIdx.y: its right-hand side, nrow rows each */
template <typename T>
__global__ void __launch_bounds__(256)
k_bwall_fill(const uint16_t *__restrict__ flags, const int32_t *__restrict__ objidx,
             const int *__restrict__ place, const T *__restrict__ wtab, BProb P, int nrow,
             T *__restrict__ rows) {
  const long xl = (long)blockIdx.x * 256 + threadIdx.x;
  if (xl >= P.N) return;
  const int x = (int)xl;
  const unsigned f = flags[x];
  if (!(f & FLAG_LINKS)) return;
  const bool solid = (f & FLAG_SOLID) != 0;
  const int i = x / P.plane, rem = x - i * P.plane, j = rem / P.esk, k = rem - j * P.esk;
  const AxisOff32 oi = axis_off32(i, P.esi, P.plane);
  const AxisOff32 oj = axis_off32(j, P.esj, P.esk);
  const AxisOff32 ok = axis_off32(k, P.esk, 1);
  const long tab = P.tab_off + (long)blockIdx.y * P.nobj;
  T *row = rows + (P.wall_off + (long)blockIdx.y * nrow + place[x]) * 16;
  row[14] = row[15] = T(0);
  Links<1, 15>::run([&](auto LL) {
    constexpr int l = decltype(LL)::value;
    T cu = T(0);
    if ((f >> (l - 1)) & 1u) {
      int sn = x, si = i, sj = j, sk = k;
      if (!solid) {
        sn = x + nb_off<l, -1>(oi, oj, ok);
        si = i - CX(l); si += (si < 0) ? P.esi : 0; si -= (si >= P.esi) ? P.esi : 0;
        sj = j - CY(l); sj += (sj < 0) ? P.esj : 0; sj -= (sj >= P.esj) ? P.esj : 0;
        sk = k - CZ(l); sk += (sk < 0) ? P.esk : 0; sk -= (sk >= P.esk) ? P.esk : 0;
      }
      cu = wall_term<l, T>(wtab + (tab + objidx[sn]) * WROW, si, sj, sk);
    }
    row[l - 1] = cu;
  });
}

/* Two steps per pass: k_step2 (slb_step2.hip) on the tiles of all problems,
 * a tile table of (problem, j0, k0, i0), one block each.  What differs: the
 * collision's parameters are the problem's, and moving walls add their rows.  A row is
 * loaded with the populations of its plane, and again for the second step,
 * ahead of the next plane's loads.  Looked up link by link, as k_bstep does,
 * the terms would be a chain of loads that every wave of the block waits for.
 * Measured, k_bstep / this kernel: 512 boxes of U{32..64} x 6 right-hand sides
 * FP32 8.35/5.63 ms per step, FP64 15.25/10.3-11.6; 32 boxes 434/331 us, 6 boxes
 * of U{28..40} 39/25.5.  NT (non-temporal stores): rows of boxes start off the
 * 128-byte lines, which tiles share: FP32 without on 6 boxes 25.5 against 35.5
 * us, on 60 696 against 713; FP64 on 32 boxes 629 against 617 with. */
/* most threads of a block (FP32 123 registers, FP64 212; FP32 with at most 512:
 * 392, 768: 344, 1024: 331 us per step on 32 boxes x 6) */
template <typename T> struct B2Cfg { enum { NTHR = sizeof(T) == 4 ? 1024 : 512 }; };

template <typename T, bool NT>
__global__ void __launch_bounds__(B2Cfg<T>::NTHR)
k_bstep2(const T *__restrict__ src, T *__restrict__ dst, const uint16_t *__restrict__ flags,
         const int *__restrict__ place, const T *__restrict__ rows,
         const BProb *__restrict__ probs, const int4 *__restrict__ tiles) {
  typedef T V4 __attribute__((ext_vector_type(4)));
  constexpr int M1 = B2Cfg<T>::NTHR + 1;
  __shared__ T buf[2][12 * M1];
  const int4 td = tiles[blockIdx.x];
  const BProb P = probs[td.x];
  const int j0 = td.y, k0 = td.z, i0 = td.w;
  const int kn = min(P.kt, P.esk - k0), jn = min(P.jt, P.esj - j0), np = min(P.ci, P.esi - i0);
  const int S = P.kt + 2, main = (P.jt + 2) * P.kt;
  const int q = (int)threadIdx.x;
  const int row = q < main ? q / P.kt : (q - main) >> 1;
  const int col = q < main ? 1 + q - row * P.kt : ((q - main) & 1) ? kn + 1 : 0;
  const bool valid = row <= jn + 1 && col <= kn + 1;
  const bool out = valid && row >= 1 && row <= jn && col >= 1 && col <= kn;
  if (!__any(valid)) {     /* a wave past the tile only keeps the barriers */
    for (int st = 0; st < np + 2; st++) lds_barrier();
    return;
  }
  const int lidx = valid ? row * S + col : M1 - 1;
  const int j = (j0 + min(row, jn + 1) - 1 + P.esj) % P.esj;
  const int k = (k0 + min(col, kn + 1) - 1 + P.esk) % P.esk;
  const int t0 = j * P.esk + k;
  const T *s = src + P.pop_off;
  T *d = dst + P.pop_off;
  const uint16_t *fl = flags + P.node_off;
  const int *pl_of = place + P.node_off;
  const T *wr = rows + P.wall_off * 16;
  const bool moving = P.wall_off >= 0;
  PhysArgs A;
  A.omega = P.omega; A.comega = P.comega; A.rho0 = P.rho0;
  A.stokes = P.stokes; A.skip_solid = P.skip_solid;
  A.bfx = P.bf[0]; A.bfy = P.bf[1]; A.bfz = P.bf[2];
  uint32_t off[9];         /* in-plane byte of (j - cy, k - cz): index 3 (cy + 1) + cz + 1 */
  {
    const AxisOff32 oj = axis_off32(j, P.esj, P.esk), ok = axis_off32(k, P.esk, 1);
#pragma unroll
    for (int c = 0; c < 9; c++)
      off[c] = (uint32_t)(t0 + (c / 3 == 0 ? oj.p : c / 3 == 2 ? oj.m : 0) +
                          (c % 3 == 0 ? ok.p : c % 3 == 2 ? ok.m : 0)) * (uint32_t)sizeof(T);
  }
  auto uni = [](int i) { return __builtin_amdgcn_readfirstlane(i); };
  auto wrap = [&](int i) { return i < 0 ? i + P.esi : (i >= P.esi ? i - P.esi : i); };
  auto bit = [](unsigned f, int l) { return (int)(f << (32 - l)) >> 31; };
  auto pick = [&](unsigned f, int l, T x, T y) -> T {
    const int m = bit(f, l);
    if constexpr (sizeof(T) == 4) {
      return __int_as_float((__float_as_int(x) & m) | (__float_as_int(y) & ~m));
    } else {
      return __hiloint2double((__double2hiint(x) & m) | (__double2hiint(y) & ~m),
                              (__double2loint(x) & m) | (__double2loint(y) & ~m));
    }
  };
  /* byte offset of population 0 of the node at byte n of a plane array */
  auto tiled = [&](int pl, uint32_t o) -> uint32_t {
    return pop_byte<T>((uint32_t)(pl * P.plane) * (uint32_t)sizeof(T) + o);
  };
  auto load = [&](T (&v)[15], int pm, int pl, int pp, unsigned f) {
    const uint32_t o0 = tiled(pl, off[4]);
    Links<0, 15>::run([&](auto LL) {
      constexpr int l = decltype(LL)::value;
      constexpr int c = 3 * (CY(l) + 1) + CZ(l) + 1;
      const int bb = l > 0 ? bit(f, l) : 0;
      /* both offsets from the lower of the two populations' runs: never negative */
      constexpr int lo = l < OPP(l) ? l : OPP(l);
      const uint32_t pulled = (l ? tiled(CX(l) > 0 ? pm : CX(l) < 0 ? pp : pl, off[c]) : o0) +
                              (uint32_t)((l - lo) * POP_TILE * (long)sizeof(T));
      const uint32_t own = o0 + (uint32_t)((OPP(l) - lo) * POP_TILE * (long)sizeof(T));
      v[l] = *(const T *)((const char *)(s + lo * POP_TILE) + ((own & bb) | (pulled & ~bb)));
    });
  };
  auto node = [&](int pl) { return pl * P.plane + t0; };
  auto walls = [&](T (&r)[16], unsigned f, int at) {
    if (f & FLAG_LINKS) {
#pragma unroll
      for (int c = 0; c < 4; c++) {
        const V4 v = *(const V4 *)(wr + (long)at * 16 + 4 * c);
        r[4 * c] = v[0]; r[4 * c + 1] = v[1]; r[4 * c + 2] = v[2]; r[4 * c + 3] = v[3];
      }
    }
  };
  auto update = [&](T (&v)[15], const T (&r)[16], unsigned f) {
    const bool solid = (f & FLAG_SOLID) != 0;
    if (moving && (f & FLAG_LINKS)) {
#pragma unroll
      for (int l = 1; l < 15; l++) v[l] += r[l - 1];
    }
    if (!(A.skip_solid && solid)) {
      T jbx = T(0), jby = T(0), jbz = T(0);
      if (!solid) { jbx = T(A.bfx); jby = T(A.bfy); jbz = T(A.bfz); }
      collide_node<T>(v, jbx, jby, jbz, A);
    }
  };
  T va[15], vb[15], a[15], dg[4], o[5];
  T ra[16], rb[16];        /* wall rows of plane pl, and of plane pl - 1 again */
  int pm = uni(wrap(i0 - 2 + P.esi)), pl = uni(wrap(i0 - 1)), pp = uni(i0);
  unsigned f = fl[node(pl)], fn = fl[node(pp)], fp = 0;
  int w = 0, wn = 0, wp = 0;   /* places in the wall rows */
  if (moving) {
    w = (f & FLAG_LINKS) ? pl_of[node(pl)] : 0;
    wn = (fn & FLAG_LINKS) ? pl_of[node(pp)] : 0;
  }
#pragma unroll
  for (int c = 0; c < 16; c++) { ra[c] = T(0); rb[c] = T(0); }
  load(va, pm, pl, pp, f);
  if (moving) walls(ra, f, w);
#pragma unroll
  for (int l = 0; l < 15; l++) a[l] = T(0);
#pragma unroll
  for (int m = 0; m < 4; m++) dg[m] = T(0);
#pragma unroll
  for (int m = 0; m < 5; m++) o[m] = T(0);
  int p2 = uni(wrap(pp + 1));
  unsigned f2 = fl[node(p2)];  /* flags run one plane further ahead than the populations */
  auto plane = [&](T (&v)[15], T (&nv)[15], T *B, int st) {
    const int p3 = uni(wrap(p2 + 1));
    unsigned f3 = 0;
    int w2 = 0;
    update(v, ra, f);
    Links<3, 15>::run([&](auto LL) {
      constexpr int l = decltype(LL)::value;
      B[XSLOT(l) * M1 + lidx] = v[l];
    });
    if (moving && st >= 2) walls(rb, fp, wp);
    if (st < np + 1) {
      load(nv, pl, pp, p2, fn);
      f3 = fl[node(p3)];
      if (moving) {
        walls(ra, fn, wn);
        if (f2 & FLAG_LINKS) w2 = pl_of[node(p2)];
      }
    }
    lds_barrier();
    if (out) {
      auto pull = [&](auto LL) -> T {
        constexpr int l = decltype(LL)::value;
        return B[XSLOT(l) * M1 + lidx - CY(l) * S - CZ(l)];
      };
      if (st >= 2) {
        a[2] = pick(fp, 2, o[0], v[2]);
        a[8] = pick(fp, 8, o[4], pull(std::integral_constant<int, 8>{}));
        a[10] = pick(fp, 10, o[3], pull(std::integral_constant<int, 10>{}));
        a[12] = pick(fp, 12, o[2], pull(std::integral_constant<int, 12>{}));
        a[14] = pick(fp, 14, o[1], pull(std::integral_constant<int, 14>{}));
        update(a, rb, fp);
        const uint32_t o0 = tiled(pm, off[4]);
        Links<0, 15>::run([&](auto LL) {
          constexpr int l = decltype(LL)::value;
          T *p = (T *)((char *)(d + l * POP_TILE) + o0);
          if constexpr (NT) __builtin_nontemporal_store(a[l], p);
          else *p = a[l];
        });
      }
      a[0] = v[0];
      a[1] = pick(f, 1, v[2], o[0]);
      a[7] = pick(f, 7, v[14], dg[0]);
      a[9] = pick(f, 9, v[12], dg[1]);
      a[11] = pick(f, 11, v[10], dg[2]);
      a[13] = pick(f, 13, v[8], dg[3]);
      a[3] = pick(f, 3, v[4], pull(std::integral_constant<int, 3>{}));
      a[4] = pick(f, 4, v[3], pull(std::integral_constant<int, 4>{}));
      a[5] = pick(f, 5, v[6], pull(std::integral_constant<int, 5>{}));
      a[6] = pick(f, 6, v[5], pull(std::integral_constant<int, 6>{}));
      dg[0] = pull(std::integral_constant<int, 7>{});
      dg[1] = pull(std::integral_constant<int, 9>{});
      dg[2] = pull(std::integral_constant<int, 11>{});
      dg[3] = pull(std::integral_constant<int, 13>{});
      o[0] = v[1]; o[1] = v[7]; o[2] = v[9]; o[3] = v[11]; o[4] = v[13];
    }
    fp = f; f = fn; fn = f2; f2 = f3;
    wp = w; w = wn; wn = w2;
    pm = pl; pl = pp; pp = p2; p2 = p3;
  };
  for (int st = 0;;) {
    plane(va, vb, buf[0], st);
    if (++st == np + 2) break;
    plane(vb, va, buf[1], st);
    if (++st == np + 2) break;
  }
}

template <typename T>
__global__ void k_bscale(double *__restrict__ a, long n, double s) {
  const long x = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (x < n) a[x] *= s;
}

/* Pull flags for one box from its object index and mask (as k_flags). */
__global__ void __launch_bounds__(256)
k_bflags(const int32_t *__restrict__ objidx, const int32_t *__restrict__ mask,
         uint16_t *__restrict__ flags, int esi, int esj, int esk) {
  const int plane = esj * esk;
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= plane) return;
  const int i = blockIdx.y, j = t / esk, k = t - j * esk;
  const long x = (long)i * plane + t;
  const AxisOff oi = axis_off(i, esi, plane);
  const AxisOff oj = axis_off(j, esj, esk);
  const AxisOff ok = axis_off(k, esk, 1);
  const int mx = mask[x];
  unsigned f = (objidx[x] >= 0) ? FLAG_SOLID : 0u;
  Links<1, 15>::run([&](auto LL) {
    constexpr int l = decltype(LL)::value;
    const int ms = mask[x + nb_off<l, -1>(oi, oj, ok)];
    if (((ms >> (l - 1)) & 1) || ((mx >> (OPP(l) - 1)) & 1)) f |= 1u << (l - 1);
  });
  flags[x] = (uint16_t)f;
}

/* ---------------------------------------------------------------------- */

struct BBox {
  int esi, esj, esk, nobj, nrhs, moving, stokes, skip_solid;
  double tau, rho0, bf[3];
  int32_t *objidx, *mask;   /* host copies until commit */
  double *tab;              /* nrhs * nobj rows */
};

struct slbd_batch {
  int prec;
  int nbox, cap;
  BBox *box;
  int committed;
  /* device arenas */
  void *pops[2];
  int cur;
  uint16_t *flags;
  int32_t *objidx;
  double *tab, *acc;
  void *wtab;               /* wall rows in the working precision */
  BProb *probs;
  int2 *tiles;
  int nprob, ntiles, nacc;
  double *hacc;             /* host copy of acc, brought up to date by every measure */
  long nnodes_total, npop_total, nnode_tab;
  /* two steps per pass: places and rows of the wall terms, tile table */
  int pairs;
  int *place;
  void *wrows;
  int4 *tiles2;
  int ntiles2, thr2;        /* tiles, threads per block */
  size_t bytes, pair_bytes; /* device memory held; by what pairs need alone */
  BProb *hprobs;
  int *box_first_prob;
  /* launch configuration */
  int block, npt, grid;
  int tiled_block, tiled_npt;   /* tile table built for this shape */
  int xcd_order;                /* XCD-contiguous tile order (k_bstep) */
  hipStream_t stream;
  /* captured step loops, one per live buffer: a graph replays the pointers
   * it was captured with, so the loop captured from buffer 0 must not run
   * when buffer 1 is live (after an odd number of plain steps) */
  hipGraphExec_t gexec[2];
  int graph_valid[2];
  hipEvent_t ev0, ev1;
};

/* Drop the captured step loops (launch shape or tile table changed). */
static void invalidate_graphs(slbd_batch *B) {
  for (int c = 0; c < 2; c++)
    if (B->graph_valid[c]) {
      HIPCHECK(hipGraphExecDestroy(B->gexec[c]));
      B->graph_valid[c] = 0;
    }
}

static size_t bts(int prec) { return prec == 32 ? 4 : 8; }

extern "C" slbd_batch *slbd_batch_create(int prec) {
  if (slbd_device_count() < 1) {
    fprintf(stderr, "sunlightlb: no HIP device is visible; the GPU library cannot run\n");
    exit(EXIT_FAILURE);
  }
  slbd_batch *B = (slbd_batch *)calloc(1, sizeof(slbd_batch));
  B->prec = (prec == 32) ? 32 : 64;
  B->block = 256; B->npt = 1; B->grid = 0;
  /* XCD-contiguous tile order: measured slower on the 512-box batch (8.59 ->
   * 8.76 ms per step), off unless SLB_BATCH_XCD=1 */
  B->xcd_order = getenv("SLB_BATCH_XCD") ? atoi(getenv("SLB_BATCH_XCD")) : 0;
  HIPCHECK(hipStreamCreateWithFlags(&B->stream, hipStreamNonBlocking));
  HIPCHECK(hipEventCreate(&B->ev0));
  HIPCHECK(hipEventCreate(&B->ev1));
  return B;
}

extern "C" int slbd_batch_add_box(slbd_batch *B, int esi, int esj, int esk,
                                  const int32_t *objidx, const int32_t *mask, int nobj,
                                  int nrhs, const double *tabs, double tau, double rho0,
                                  int stokes, int skip_solid, int moving, const double *bf) {
  if (B->committed || nrhs < 1) return -1;
  if (15 * pop_nodes((long)esi * esj * esk) > 0x7fffffffL) {
    fprintf(stderr, "slb_batch_add: a %d x %d x %d box is too large for a batch (at most "
            "2^31 populations per box)\n", esi, esj, esk);
    return -1;
  }
  if (B->nbox == B->cap) {
    B->cap = B->cap ? 2 * B->cap : 64;
    B->box = (BBox *)realloc(B->box, sizeof(BBox) * B->cap);
  }
  BBox *b = &B->box[B->nbox];
  const long N = (long)esi * esj * esk;
  b->esi = esi; b->esj = esj; b->esk = esk; b->nobj = nobj; b->nrhs = nrhs;
  b->moving = moving; b->stokes = stokes; b->skip_solid = skip_solid;
  b->tau = tau; b->rho0 = rho0;
  for (int c = 0; c < 3; c++) b->bf[c] = bf ? bf[c] : 0.0;
  b->objidx = (int32_t *)malloc(sizeof(int32_t) * N);
  b->mask = (int32_t *)malloc(sizeof(int32_t) * N);
  memcpy(b->objidx, objidx, sizeof(int32_t) * N);
  memcpy(b->mask, mask, sizeof(int32_t) * N);
  const size_t tb = sizeof(double) * SLBD_OBJ_STRIDE * (size_t)(nobj > 0 ? nobj : 1) * nrhs;
  b->tab = (double *)malloc(tb);
  if (nobj > 0) memcpy(b->tab, tabs, sizeof(double) * SLBD_OBJ_STRIDE * nobj * nrhs);
  return B->nbox++;
}

/* Device memory of a batch.  A limit set from the host (tests; 0: none) stands
 * for a device with that much left. */
static size_t mem_limit, last_bytes;

/* Set the limit; the bytes that the batch committed last holds. */
extern "C" size_t slbd_batch_mem_limit(size_t bytes) {
  mem_limit = bytes;
  return last_bytes;
}

static bool try_alloc(slbd_batch *B, void **p, size_t bytes) {
  *p = NULL;
  if (mem_limit && B->bytes + bytes > mem_limit) return false;
  if (hipMalloc(p, bytes) != hipSuccess) {
    (void)hipGetLastError();
    *p = NULL;
    return false;
  }
  B->bytes += bytes;
  return true;
}

/* Single steps from here on: their memory goes back. */
static void drop_pairs(slbd_batch *B) {
  void *ps[] = {B->place, B->wrows, B->tiles2};
  for (size_t q = 0; q < sizeof ps / sizeof ps[0]; q++)
    if (ps[q]) HIPCHECK(hipFree(ps[q]));
  B->bytes -= B->pair_bytes;
  B->pair_bytes = 0;
  B->place = NULL; B->wrows = NULL; B->tiles2 = NULL;
  B->pairs = 0;
}

template <typename P>
static void must_alloc(slbd_batch *B, P **p, size_t bytes) {
  void *v;
  if (!try_alloc(B, &v, bytes)) {
    if (B->pairs) {          /* what single steps need comes before the pairs' tables */
      HIPCHECK(hipStreamSynchronize(B->stream));
      drop_pairs(B);
      invalidate_graphs(B);
    }
    if (!try_alloc(B, &v, bytes)) {
      fprintf(stderr, "sunlightlb: out of device memory (%zu bytes for a batch)\n", bytes);
      exit(EXIT_FAILURE);
    }
  }
  *p = (P *)v;
}

/* memory that only the pairs need */
template <typename P>
static bool pair_alloc(slbd_batch *B, P **p, size_t bytes) {
  void *v;
  if (!try_alloc(B, &v, bytes)) return false;
  B->pair_bytes += bytes;
  *p = (P *)v;
  return true;
}

static void build_tiles(slbd_batch *B) {
  const long per = (long)B->block * B->npt;
  long nt = 0;
  for (int p = 0; p < B->nprob; p++) nt += (B->hprobs[p].N + per - 1) / per;
  int2 *h = (int2 *)malloc(sizeof(int2) * (nt > 0 ? nt : 1));
  long t = 0;
  for (int p = 0; p < B->nprob; p++)
    for (long s = 0; s < B->hprobs[p].N; s += per) { h[t].x = p; h[t].y = (int)s; t++; }
  if (B->tiles) {
    HIPCHECK(hipFree(B->tiles));
    B->bytes -= sizeof(int2) * (B->ntiles > 0 ? B->ntiles : 1);
  }
  must_alloc(B, &B->tiles, sizeof(int2) * (nt > 0 ? nt : 1));
  HIPCHECK(hipMemcpy(B->tiles, h, sizeof(int2) * nt, hipMemcpyHostToDevice));
  free(h);
  B->ntiles = (int)nt;
  B->tiled_block = B->block;
  B->tiled_npt = B->npt;
  invalidate_graphs(B);
}

/* k_bstep2's times, us, [FP64][moving walls]: a launch; a block's start, a plane's
 * barrier and load latency, a plane's work per thread (fitted to 250 batches of 1
 * to 512 problems; standard error 11%).  One step of k_bstep: a launch and its
 * first loads, then 30 values per node at 5.65 TB/s (7%). */
static const double PLAN_US[2][2][4] = {{{2.8, 0.4, 0.91, 0.0024}, {2.5, 0.5, 1.20, 0.0026}},
                                        {{1.5, 1.2, 1.03, 0.0046}, {2.0, 1.5, 1.13, 0.0043}}};
static const double SINGLE_US[2] = {3.5, 5.9}; /* walls at rest, moving */
/* Time of one block of k_bstep2, us: its start, then a barrier, the loads' latency
 * and the work of pts threads per plane. */
static double block_us(int prec, int moving, int pts, int ci) {
  const double *t = PLAN_US[prec == 64][moving != 0];
  return t[1] + (ci + 2) * (t[2] + t[3] * pts);
}

/* Whether a batch takes two steps per pass, and the tiles of every box (box: esi, esj, esk, right-hand sides, moving; tile: jt, kt,
 * ci), and the time of two steps in this way and as two single ones (us).  Tried
 * are tiles of at most `cap` threads (of these the split of a plane that costs
 * least, as slbd_step2_plan: FP64 512 boxes x 6 10.6 ms per step, 10.9 by block_us)
 * and chunks of at most `len` planes; a CU holds one block at a time.  Large tiles and long chunks do the least work, but
 * few problems then leave most CUs idle: one box of 64^3, FP32, us per step: 20
 * blocks (13 x 64 x 16) 21.4, 256 (8 x 64 x 2) 6.3, single steps 7.6; one right-hand
 * side of 6 of 64^3 35.1/19.3 (single / this), 2 x 2 of 256 x 256 x 4 25.3/15.2 (62 in
 * chunks of a quarter).  Many problems of a few hundred nodes each fill no
 * block and keep single steps: 384 of 8^3 6.5/14.2, 1536 of 6^3 12.3/32.2. */
extern "C" int slbd_bstep2_plan(int nbox, const int *box, int prec, int *tile, double us[2]) {
  static const int caps[] = {1024, 704, 512, 320, 192, 96};
  static const int lens[] = {1 << 30, 64, 48, 32, 24, 16, 12, 8, 6, 4, 3, 2, 1};
  const int most = prec == 32 ? B2Cfg<float>::NTHR : B2Cfg<double>::NTHR, cus = 256;
  int *jk = (int *)malloc(sizeof(int) * 2 * (size_t)nbox);
  if (!jk) { fprintf(stderr, "sunlightlb: out of host memory\n"); exit(EXIT_FAILURE); }
  double best = 0.0, nodes = 0.0;
  int moving = 0;
  for (int b = 0; b < nbox; b++) {
    const int *q = box + 5 * b;
    nodes += (double)q[0] * q[1] * q[2] * q[3];
    moving |= q[4] != 0;
  }
  for (size_t c = 0; c < sizeof caps / sizeof caps[0]; c++) {
    if (caps[c] > most) continue;
    for (int b = 0; b < nbox; b++) {
      const int *q = box + 5 * b;
      double bc = 0.0;
      int jt = 0, kt = 0;
      for (int nk = 1; nk <= (q[2] + 31) / 32 || jt == 0; nk++) {
        const int k = (q[2] + nk - 1) / nk, nkt = (q[2] + k - 1) / k;
        for (int jq = 1; jq <= q[1] && (jq + 2) * (k + 2) <= caps[c]; jq++) {
          const int njt = (q[1] + jq - 1) / jq, j = (q[1] + njt - 1) / njt;
          const double cost = (1.0 + 16.0 / k) * njt * nkt *
                              ((double)(j + 2) * (k + 2) + (double)j * k + 1000.0);
          if (jt == 0 || cost < bc) { bc = cost; jt = j; kt = k; }
        }
      }
      jk[2 * b] = jt; jk[2 * b + 1] = kt;
    }
    for (size_t l = 0; l < sizeof lens / sizeof lens[0]; l++) {
      double sum = 0.0, longest = 0.0;
      long blocks = 0;
      for (int b = 0; b < nbox; b++) {
        const int *q = box + 5 * b, jt = jk[2 * b], kt = jk[2 * b + 1];
        const int nch = lens[l] < q[0] ? (q[0] + lens[l] - 1) / lens[l] : 1, ci = (q[0] + nch - 1) / nch;
        const long n = (long)((q[1] + jt - 1) / jt) * ((q[2] + kt - 1) / kt) * ((q[0] + ci - 1) / ci) * q[3];
        const double t = block_us(prec, q[4], (jt + 2) * (kt + 2), ci);
        blocks += n;
        sum += n * t;
        if (t > longest) longest = t;
      }
      const double t = blocks <= cus ? longest : sum / cus + 0.5 * longest;
      if (best > 0.0 && t >= best) continue;
      best = t;
      for (int b = 0; b < nbox; b++) {
        const int *q = box + 5 * b;
        const int nch = lens[l] < q[0] ? (q[0] + lens[l] - 1) / lens[l] : 1;
        tile[3 * b] = jk[2 * b]; tile[3 * b + 1] = jk[2 * b + 1];
        tile[3 * b + 2] = (q[0] + nch - 1) / nch;
      }
    }
  }
  free(jk);
  us[0] = PLAN_US[prec == 64][moving][0] + best;
  us[1] = 2.0 * (SINGLE_US[moving] + nodes * 30.0 * (prec / 8) / 5.65e6);
  /* with a margin for the estimate: of 338 batches, 2 at 4 to 80 us per step were
   * then slower by more than 4% (6, 8%); FP32 at rest without it 7, by up to 21% */
  return us[0] < (prec == 32 && !moving ? 0.85 : 0.95) * us[1];
}

/* Two steps per pass: tiles of every box in chunks along i, and the wall terms. */
static void plan_pairs(slbd_batch *B) {
  const char *e = getenv("SLB_BATCH_STEP2");
  B->pairs = !(e && atoi(e) == 0);
  for (int p = 0; p < B->nprob; p++)   /* 32-bit byte offsets in a problem */
    if (15 * pop_nodes(B->hprobs[p].N) * (long)bts(B->prec) >= (1L << 32)) B->pairs = 0;
  if (!B->pairs) return;
  int *box = (int *)malloc(sizeof(int) * 8 * (size_t)B->nbox), *tile = box + 5 * (size_t)B->nbox;
  if (!box) { fprintf(stderr, "sunlightlb: out of host memory\n"); exit(EXIT_FAILURE); }
  for (int b = 0; b < B->nbox; b++) {
    const BBox *x = &B->box[b];
    const int q[5] = {x->esi, x->esj, x->esk, x->nrhs, x->moving};
    memcpy(box + 5 * b, q, sizeof q);
  }
  double us[2];
  if (!slbd_bstep2_plan(B->nbox, box, B->prec, tile, us) && !e) B->pairs = 0;
  int pts = 0;
  long total = 0;
  for (int b = 0, p = 0; b < B->nbox; b++)
    for (int r = 0; r < B->box[b].nrhs; r++, p++) {
      BProb *q = &B->hprobs[p];
      q->jt = tile[3 * b]; q->kt = tile[3 * b + 1]; q->ci = tile[3 * b + 2];
      if ((q->jt + 2) * (q->kt + 2) > pts) pts = (q->jt + 2) * (q->kt + 2);
      total += (long)((q->esj + q->jt - 1) / q->jt) * ((q->esk + q->kt - 1) / q->kt) *
               ((q->esi + q->ci - 1) / q->ci);
    }
  free(box);
  if (!B->pairs) return;
  int4 *h = (int4 *)malloc(sizeof(int4) * (total > 0 ? total : 1));
  long n = 0;
  for (int p = 0; p < B->nprob; p++) {
    const BProb *q = &B->hprobs[p];
    for (int i0 = 0; i0 < q->esi; i0 += q->ci)
      for (int j0 = 0; j0 < q->esj; j0 += q->jt)
        for (int k0 = 0; k0 < q->esk; k0 += q->kt) h[n++] = make_int4(p, j0, k0, i0);
  }
  B->ntiles2 = (int)n;
  B->thr2 = (pts + 63) & ~63;
  if (!pair_alloc(B, &B->tiles2, sizeof(int4) * (n > 0 ? n : 1))) {
    drop_pairs(B);
    free(h);
    return;
  }
  HIPCHECK(hipMemcpy(B->tiles2, h, sizeof(int4) * n, hipMemcpyHostToDevice));
  free(h);
  /* places of the boxes' boundary nodes, then the moving problems' rows */
  int *cnt, *hc = (int *)calloc(B->nbox, sizeof(int));
  if (!pair_alloc(B, &B->place, sizeof(int) * B->nnode_tab) ||
      !pair_alloc(B, &cnt, sizeof(int) * B->nbox)) {
    drop_pairs(B);
    free(hc);
    return;
  }
  HIPCHECK(hipMemsetAsync(cnt, 0, sizeof(int) * B->nbox, B->stream));
  long nrow = 0;
  for (int b = 0; b < B->nbox; b++) {
    const BProb *q = &B->hprobs[B->box_first_prob[b]];
    if (!B->box[b].moving) continue;
    hipLaunchKernelGGL(k_bwall_place, dim3((unsigned)((q->N + 255) / 256)), dim3(256), 0, B->stream,
                       B->flags + q->node_off, q->N, B->place + q->node_off, cnt + b);
    LAUNCHCHECK();
  }
  HIPCHECK(hipMemcpyAsync(hc, cnt, sizeof(int) * B->nbox, hipMemcpyDeviceToHost, B->stream));
  HIPCHECK(hipStreamSynchronize(B->stream));
  HIPCHECK(hipFree(cnt));
  B->bytes -= sizeof(int) * B->nbox;
  B->pair_bytes -= sizeof(int) * B->nbox;
  for (int b = 0; b < B->nbox; b++)
    if (B->box[b].moving)
      for (int r = 0; r < B->box[b].nrhs; r++) {
        B->hprobs[B->box_first_prob[b] + r].wall_off = nrow;
        nrow += hc[b];
      }
  /* a batch that fills the memory without the rows runs single steps */
  if (!pair_alloc(B, &B->wrows, bts(B->prec) * 16 * (nrow > 0 ? nrow : 1))) {
    drop_pairs(B);
    free(hc);
    return;
  }
  for (int b = 0; b < B->nbox; b++) {
    const BProb *q = &B->hprobs[B->box_first_prob[b]];
    if (q->wall_off < 0 || hc[b] == 0) continue;
    BProb q1 = *q;
    for (int r = 0; r < B->box[b].nrhs; r += 32768) { /* a grid's y extent is 16 bits wide */
      const int nr = B->box[b].nrhs - r < 32768 ? B->box[b].nrhs - r : 32768;
      const dim3 g((unsigned)((q->N + 255) / 256), (unsigned)nr);
      q1.wall_off = q->wall_off + (long)r * hc[b];
      q1.tab_off = q->tab_off + r * q->nobj;
      if (B->prec == 32)
        hipLaunchKernelGGL(k_bwall_fill<float>, g, dim3(256), 0, B->stream, B->flags + q->node_off,
                           B->objidx + q->node_off, B->place + q->node_off, (const float *)B->wtab,
                           q1, hc[b], (float *)B->wrows);
      else
        hipLaunchKernelGGL(k_bwall_fill<double>, g, dim3(256), 0, B->stream, B->flags + q->node_off,
                           B->objidx + q->node_off, B->place + q->node_off, (const double *)B->wtab,
                           q1, hc[b], (double *)B->wrows);
      LAUNCHCHECK();
    }
  }
  free(hc);
  HIPCHECK(hipStreamSynchronize(B->stream));
}

extern "C" int slbd_batch_commit(slbd_batch *B) {
  if (B->committed || B->nbox == 0) return -1;
  int nprob = 0, nacc = 0;
  long nodes = 0, pops = 0, ntab = 0;
  for (int b = 0; b < B->nbox; b++) {
    const long N = (long)B->box[b].esi * B->box[b].esj * B->box[b].esk;
    nprob += B->box[b].nrhs;
    nodes += N;
    pops += 15 * pop_nodes(N) * B->box[b].nrhs;
    ntab += (long)B->box[b].nobj * B->box[b].nrhs;
    nacc += B->box[b].nobj * B->box[b].nrhs;
  }
  B->nprob = nprob;
  B->nacc = nacc;
  B->nnode_tab = nodes;
  B->npop_total = pops;
  B->hprobs = (BProb *)calloc(nprob, sizeof(BProb));
  B->box_first_prob = (int *)malloc(sizeof(int) * B->nbox);
  must_alloc(B, &B->pops[0], bts(B->prec) * pops);
  must_alloc(B, &B->pops[1], bts(B->prec) * pops);
  HIPCHECK(hipMemsetAsync(B->pops[0], 0, bts(B->prec) * pops, B->stream));
  HIPCHECK(hipMemsetAsync(B->pops[1], 0, bts(B->prec) * pops, B->stream));
  must_alloc(B, &B->flags, sizeof(uint16_t) * nodes);
  must_alloc(B, &B->objidx, sizeof(int32_t) * nodes);
  int32_t *dmask;
  must_alloc(B, &dmask, sizeof(int32_t) * nodes);
  must_alloc(B, &B->tab, sizeof(double) * SLBD_OBJ_STRIDE * (ntab > 0 ? ntab : 1));
  must_alloc(B, &B->wtab, bts(B->prec) * WROW * (ntab > 0 ? ntab : 1));
  double *hw = (double *)calloc((size_t)WROW * (ntab > 0 ? ntab : 1), sizeof(double));
  must_alloc(B, &B->acc, sizeof(double) * 6 * (nacc > 0 ? nacc : 1));
  HIPCHECK(hipMemsetAsync(B->acc, 0, sizeof(double) * 6 * (nacc > 0 ? nacc : 1), B->stream));
  B->hacc = (double *)calloc(6 * (size_t)(nacc > 0 ? nacc : 1), sizeof(double));
  if (!B->hacc) { fprintf(stderr, "sunlightlb: out of host memory\n"); exit(EXIT_FAILURE); }
  long node_off = 0, pop_off = 0;
  int tab_off = 0, p = 0;
  for (int b = 0; b < B->nbox; b++) {
    BBox *x = &B->box[b];
    const long N = (long)x->esi * x->esj * x->esk;
    HIPCHECK(hipMemcpy(B->objidx + node_off, x->objidx, sizeof(int32_t) * N, hipMemcpyHostToDevice));
    HIPCHECK(hipMemcpy(dmask + node_off, x->mask, sizeof(int32_t) * N, hipMemcpyHostToDevice));
    if (x->nobj > 0)
      HIPCHECK(hipMemcpy(B->tab + (long)tab_off * SLBD_OBJ_STRIDE, x->tab,
                         sizeof(double) * SLBD_OBJ_STRIDE * x->nobj * x->nrhs,
                         hipMemcpyHostToDevice));
    for (long o = 0; o < (long)x->nobj * x->nrhs; o++) {
      const double *po = x->tab + o * SLBD_OBJ_STRIDE;   /* pos, vel, ang */
      double *w = hw + (tab_off + o) * WROW;
      const double us = x->rho0 / 12.0;
      w[0] = us * (po[3] - (po[7] * po[2] - po[8] * po[1]));
      w[1] = us * (po[4] - (po[8] * po[0] - po[6] * po[2]));
      w[2] = us * (po[5] - (po[6] * po[1] - po[7] * po[0]));
      w[3] = us * po[6]; w[4] = us * po[7]; w[5] = us * po[8];
    }
    hipLaunchKernelGGL(k_bflags, dim3((x->esj * x->esk + 255) / 256, x->esi), dim3(256), 0,
                       B->stream, B->objidx + node_off, dmask + node_off, B->flags + node_off,
                       x->esi, x->esj, x->esk);
    LAUNCHCHECK();
    B->box_first_prob[b] = p;
    for (int r = 0; r < x->nrhs; r++, p++) {
      BProb *q = &B->hprobs[p];
      q->esi = x->esi; q->esj = x->esj; q->esk = x->esk; q->plane = x->esj * x->esk;
      q->N = N;
      q->pop_off = pop_off;
      q->node_off = node_off;
      q->tab_off = tab_off + r * x->nobj;
      q->nobj = x->nobj;
      q->acc_off = tab_off + r * x->nobj;
      q->moving = x->moving; q->stokes = x->stokes; q->skip_solid = x->skip_solid;
      q->omega = 1.0 / x->tau; q->comega = 1.0 - q->omega; q->rho0 = x->rho0;
      for (int c = 0; c < 3; c++) q->bf[c] = x->bf[c];
      q->wall_off = -1;
      pop_off += 15 * pop_nodes(N);
    }
    node_off += N;
    tab_off += x->nobj * x->nrhs;
    free(x->objidx); free(x->mask); free(x->tab);
    x->objidx = x->mask = NULL; x->tab = NULL;
  }
  if (B->prec == 32) {
    float *hf = (float *)malloc(sizeof(float) * WROW * (ntab > 0 ? ntab : 1));
    for (long q = 0; q < (long)WROW * (ntab > 0 ? ntab : 1); q++) hf[q] = (float)hw[q];
    HIPCHECK(hipMemcpy(B->wtab, hf, sizeof(float) * WROW * (ntab > 0 ? ntab : 1),
                       hipMemcpyHostToDevice));
    free(hf);
  } else {
    HIPCHECK(hipMemcpy(B->wtab, hw, sizeof(double) * WROW * (ntab > 0 ? ntab : 1),
                       hipMemcpyHostToDevice));
  }
  free(hw);
  HIPCHECK(hipStreamSynchronize(B->stream));
  HIPCHECK(hipFree(dmask));
  B->bytes -= sizeof(int32_t) * nodes;
  /* what single steps need first: the pairs take what is left, or do without */
  must_alloc(B, &B->probs, sizeof(BProb) * nprob);
  build_tiles(B);
  plan_pairs(B);
  HIPCHECK(hipMemcpy(B->probs, B->hprobs, sizeof(BProb) * nprob, hipMemcpyHostToDevice));
  long tot = 0;
  for (int q = 0; q < nprob; q++) tot += B->hprobs[q].N;
  B->nnodes_total = tot;
  last_bytes = B->bytes;
  B->committed = 1;
  return 0;
}

template <typename T, bool FORCE, int NPT>
static void blaunch_t(slbd_batch *B) {
  int grid = (B->grid > 0 && B->grid < B->ntiles) ? B->grid : B->ntiles;
  int chunk = 0;
  if (B->xcd_order && B->ntiles >= 64) {
    chunk = (B->ntiles + 7) / 8;
    grid = (grid + 7) & ~7;   /* every block stays on one XCD's range */
  }
  hipLaunchKernelGGL((k_bstep<T, FORCE, NPT>), dim3(grid), dim3(B->block), 0, B->stream,
                     (const T *)B->pops[B->cur], (T *)B->pops[B->cur ^ 1], B->flags, B->objidx,
                     B->tab, (const T *)B->wtab, B->probs, B->tiles, B->ntiles, chunk, B->acc);
  LAUNCHCHECK();
  B->cur ^= 1;
}

template <typename T>
static void blaunch(slbd_batch *B, bool force) {
  if (force) {
    if (B->npt == 2) blaunch_t<T, true, 2>(B); else if (B->npt == 4) blaunch_t<T, true, 4>(B);
    else blaunch_t<T, true, 1>(B);
  } else {
    if (B->npt == 2) blaunch_t<T, false, 2>(B); else if (B->npt == 4) blaunch_t<T, false, 4>(B);
    else blaunch_t<T, false, 1>(B);
  }
}

static void bstep(slbd_batch *B, bool force) {
  if (B->tiled_block != B->block || B->tiled_npt != B->npt) build_tiles(B);
  if (B->prec == 32) blaunch<float>(B, force); else blaunch<double>(B, force);
}

template <typename T, bool NT>
static void bstep2_t(slbd_batch *B) {
  hipLaunchKernelGGL((k_bstep2<T, NT>), dim3((unsigned)B->ntiles2), dim3((unsigned)B->thr2), 0,
                     B->stream, (const T *)B->pops[B->cur], (T *)B->pops[B->cur ^ 1], B->flags,
                     B->place, (const T *)B->wrows, B->probs, B->tiles2);
  LAUNCHCHECK();
  B->cur ^= 1;
}

static void bstep2(slbd_batch *B) {
  if (B->prec == 32) bstep2_t<float, false>(B);
  else if (16 * B->npop_total > 256000000L) bstep2_t<double, true>(B);
  else bstep2_t<double, false>(B);
}

/* nsteps plain steps; pairs: two per launch as far as they go */
static void bsteps(slbd_batch *B, int nsteps, bool pairs) {
  int s = 0;
  if (pairs)
    for (; s + 2 <= nsteps; s += 2) bstep2(B);
  for (; s < nsteps; s++) bstep(B, false);
}

extern "C" void slbd_batch_config(slbd_batch *B, int block, int npt, int grid) {
  if (block != 64 && block != 128 && block != 256 && block != 512) block = 256;
  if (npt != 1 && npt != 2 && npt != 4) npt = 1;
  if (block != B->block || npt != B->npt || grid != B->grid) invalidate_graphs(B);
  B->block = block; B->npt = npt; B->grid = grid;
}

#define BATCH_GRAPH_STEPS 32

/* Capture BATCH_GRAPH_STEPS steps (a multiple of 4: as single steps or in pairs
 * they end on the buffer they began on) starting from the live buffer B->cur. */
static void build_graph(slbd_batch *B) {
  if (B->tiled_block != B->block || B->tiled_npt != B->npt) build_tiles(B);
  const int cur0 = B->cur;
  if (B->graph_valid[cur0]) return;
  hipGraph_t g;
  HIPCHECK(hipStreamBeginCapture(B->stream, hipStreamCaptureModeThreadLocal));
  bsteps(B, BATCH_GRAPH_STEPS, B->pairs != 0);
  HIPCHECK(hipStreamEndCapture(B->stream, &g));
  HIPCHECK(hipGraphInstantiate(&B->gexec[cur0], g, NULL, NULL, 0));
  HIPCHECK(hipGraphDestroy(g));
  B->cur = cur0;   /* an even number of steps returns to the same buffer */
  B->graph_valid[cur0] = 1;
}

extern "C" void slbd_batch_run(slbd_batch *B, int nsteps, int use_graph) {
  if (!B->committed) return;
  int s = 0;
  if (use_graph && nsteps >= BATCH_GRAPH_STEPS) {
    /* the loop captured from the live buffer (a shape change since the
     * last capture rebuilds the tile table and drops both loops) */
    if (B->tiled_block != B->block || B->tiled_npt != B->npt) build_tiles(B);
    build_graph(B);
    for (; s + BATCH_GRAPH_STEPS <= nsteps; s += BATCH_GRAPH_STEPS)
      HIPCHECK(hipGraphLaunch(B->gexec[B->cur], B->stream));
  }
  /* use_graph 0: the autotuner times the single-step launch shapes */
  bsteps(B, nsteps - s, B->pairs != 0 && use_graph != 0);
}

extern "C" const char *slbd_batch_run_kernel(const slbd_batch *B) {
  return B->committed && B->pairs ? "k_bstep2" : "k_bstep";
}

extern "C" double slbd_batch_time(slbd_batch *B, int nsteps, int use_graph) {
  if (use_graph && B->committed && nsteps >= BATCH_GRAPH_STEPS) build_graph(B);
  HIPCHECK(hipStreamSynchronize(B->stream));
  HIPCHECK(hipEventRecord(B->ev0, B->stream));
  slbd_batch_run(B, nsteps, use_graph);
  HIPCHECK(hipEventRecord(B->ev1, B->stream));
  HIPCHECK(hipEventSynchronize(B->ev1));
  float ms = 0.0f;
  HIPCHECK(hipEventElapsedTime(&ms, B->ev0, B->ev1));
  return (double)ms;
}

/* measure(): force accumulators zeroed, two force-collecting steps, halved
 * (src/lbmeasure.c:30-49). */
extern "C" void slbd_batch_measure(slbd_batch *B) {
  if (!B->committed) return;
  const long n = 6L * (B->nacc > 0 ? B->nacc : 1);
  HIPCHECK(hipMemsetAsync(B->acc, 0, sizeof(double) * n, B->stream));
  bstep(B, true);
  bstep(B, true);
  hipLaunchKernelGGL(k_bscale<double>, dim3((n + 255) / 256), dim3(256), 0, B->stream, B->acc, n, 0.5);
  LAUNCHCHECK();
  /* every problem's sums in one copy: 192 problems' forces read one by one
   * from the device took 7 ms */
  HIPCHECK(hipMemcpyAsync(B->hacc, B->acc, sizeof(double) * n, hipMemcpyDeviceToHost, B->stream));
  HIPCHECK(hipStreamSynchronize(B->stream));
}

extern "C" int slbd_batch_forces(slbd_batch *B, int box, int rhs, double *frc, double *trq) {
  if (!B->committed || box < 0 || box >= B->nbox || rhs < 0 || rhs >= B->box[box].nrhs) return -1;
  const BProb *q = &B->hprobs[B->box_first_prob[box] + rhs];
  if (q->nobj == 0) return 0;
  const double *h = B->hacc + 6L * q->acc_off;
  for (int o = 0; o < q->nobj; o++)
    for (int c = 0; c < 3; c++) {
      frc[3 * o + c] = h[6 * o + c];
      trq[3 * o + c] = h[6 * o + 3 + c];
    }
  return q->nobj;
}

extern "C" int slbd_batch_get_pops(slbd_batch *B, int box, int rhs, double *aos) {
  if (!B->committed || box < 0 || box >= B->nbox || rhs < 0 || rhs >= B->box[box].nrhs) return -1;
  HIPCHECK(hipStreamSynchronize(B->stream));
  const BProb *q = &B->hprobs[B->box_first_prob[box] + rhs];
  const size_t ts = bts(B->prec);
  const long np = 15 * pop_nodes(q->N);
  char *tmp = (char *)malloc(np * ts);
  HIPCHECK(hipMemcpy(tmp, (char *)B->pops[B->cur] + q->pop_off * ts, np * ts,
                     hipMemcpyDeviceToHost));
  for (int l = 0; l < 15; l++)
    for (long n = 0; n < q->N; n++)
      aos[15 * n + l] = (B->prec == 32) ? (double)((float *)tmp)[pidx(l, n)]
                                        : ((double *)tmp)[pidx(l, n)];
  free(tmp);
  return 0;
}

extern "C" long slbd_batch_nodes(const slbd_batch *B) { return B->nnodes_total; }
extern "C" int slbd_batch_nprob(const slbd_batch *B) { return B->nprob; }
extern "C" int slbd_batch_nbox(const slbd_batch *B) { return B->nbox; }
extern "C" int slbd_batch_box_dims(const slbd_batch *B, int box, int *dims) {
  if (box < 0 || box >= B->nbox) return -1;
  dims[0] = B->box[box].esi; dims[1] = B->box[box].esj; dims[2] = B->box[box].esk;
  return B->box[box].nrhs;
}
extern "C" void slbd_batch_get_config(const slbd_batch *B, int *cfg) {
  /* tile count of the configured shape (the table itself is rebuilt lazily
   * at the next run, so B->ntiles may still describe an earlier shape) */
  const long per = (long)B->block * B->npt;
  long nt = 0;
  for (int p = 0; p < B->nprob; p++) nt += (B->hprobs[p].N + per - 1) / per;
  cfg[0] = B->block; cfg[1] = B->npt; cfg[2] = B->grid; cfg[3] = (int)nt;
}
extern "C" int slbd_batch_cu_count(void) {
  hipDeviceProp_t prop;
  HIPCHECK(hipGetDeviceProperties(&prop, 0));
  return prop.multiProcessorCount;
}

extern "C" void slbd_batch_destroy(slbd_batch *B) {
  if (!B) return;
  HIPCHECK(hipStreamSynchronize(B->stream));
  invalidate_graphs(B);
  void *ps[] = {B->pops[0], B->pops[1], B->flags, B->objidx, B->tab, B->wtab, B->acc, B->probs,
                B->tiles, B->place, B->wrows, B->tiles2};
  for (size_t q = 0; q < sizeof ps / sizeof ps[0]; q++)
    if (ps[q]) HIPCHECK(hipFree(ps[q]));
  for (int b = 0; b < B->nbox; b++) { free(B->box[b].objidx); free(B->box[b].mask); free(B->box[b].tab); }
  free(B->box); free(B->hprobs); free(B->box_first_prob); free(B->hacc);
  HIPCHECK(hipEventDestroy(B->ev0));
  HIPCHECK(hipEventDestroy(B->ev1));
  HIPCHECK(hipStreamDestroy(B->stream));
  free(B);
}

/* Every problem back to rest (populations and force sums zero). */
extern "C" void slbd_batch_reset(slbd_batch *B) {
  if (!B->committed) return;
  HIPCHECK(hipMemsetAsync(B->pops[0], 0, bts(B->prec) * B->npop_total, B->stream));
  HIPCHECK(hipMemsetAsync(B->pops[1], 0, bts(B->prec) * B->npop_total, B->stream));
  HIPCHECK(hipMemsetAsync(B->acc, 0, sizeof(double) * 6 * (B->nacc > 0 ? B->nacc : 1), B->stream));
  memset(B->hacc, 0, sizeof(double) * 6 * (size_t)(B->nacc > 0 ? B->nacc : 1));
  HIPCHECK(hipStreamSynchronize(B->stream));
  B->cur = 0;
}
