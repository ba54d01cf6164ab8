/*
 * slb_mp2.hip -- two moment-propagation steps per pass over the link factors.
 *
 * A step on precomputed factors (k_mpstep_w, slb_dev.hip) reads 15 factors
 * per node for 3 values read and written: the factors are its traffic.
 * k_mpstep2 advances a tile of JT x KT (j, k) columns by two steps while it
 * marches along i, so that a node's factors are read once for both:
 *
 *   - the records of planes p - 1 .. p + 1 of the tile and a rim of two nodes
 *     lie in LDS (a ring of four planes, the next one in flight);
 *   - per plane p the block computes step t+1 of the tile and a rim of one
 *     node from them, into a second ring of four planes;
 *   - from planes p - 2 .. p of that ring it computes step t+2 of plane p - 1,
 *     with the factors it kept from the plane before.
 *
 * Bound by LDS reads and HBM together at 128^3 (30 records of 12
 * bytes per node and pair).
 * Measured, us per step, k_mpstep_w / this kernel: FP32 with moments 128^3
 * 26.5/19.7, 200^3 160/80.6, 256^3 322/153; FP64 128^3 78.7/44.2, one moment
 * 45.6/27.1.
 *
 * A thread owns one (j, k) column; one barrier per plane.  The factors of the
 * next plane are loaded a plane ahead; three register sets take turns by
 * name.  Sums run over the links in k_mpstep_w's order: bit-identical.
 */
#include "slb_dev.h"
#include "slb_kern.h"
#include "slb_mpk.h"

template <typename T> struct MP2Cfg { enum { NTHR = sizeof(T) == 4 ? 1024 : 640 }; };
#define MP2_LDS 163840

/* AX: axis of the displacement moments (NMOM 3) */
template <typename T, int NMOM, int AX, typename I>
__global__ void __launch_bounds__(MP2Cfg<T>::NTHR)
k_mpstep2(const T *__restrict__ wt, const CRec<T, NMOM> *__restrict__ Q,
          CRec<T, NMOM> *__restrict__ qout, const uint32_t *__restrict__ mpf, Geom G, MPArgs A,
          MP2Plan L) {
  typedef CRec<T, NMOM> R;
  typedef T V4 __attribute__((ext_vector_type(4)));
  extern __shared__ __attribute__((aligned(16))) unsigned char mp2_raw[];
  const int S1 = L.kt + 2, S2 = L.kt + 4;
  const int M1 = (L.jt + 2) * S1, M2 = (L.jt + 4) * S2;
  /* rings of four planes; the last place of each takes idle threads' writes */
  R *qs = (R *)mp2_raw;                /* [4][M2 + 1] */
  R *ts = qs + 4 * (M2 + 1);           /* [4][M1 + 1] */
  const int nb = gridDim.x;
  const int b = (nb & 7) == 0 ? (int)(blockIdx.x & 7) * (nb >> 3) + (int)(blockIdx.x >> 3)
                              : (int)blockIdx.x;
  const int kt = b % L.nkt, jt = (b / L.nkt) % L.njt, ch = b / (L.nkt * L.njt);
  const int k0 = kt * L.kt, j0 = jt * L.jt, i0 = ch * L.ci;
  const int kn = min(L.kt, G.esk - k0), jn = min(L.jt, G.esj - j0), np = min(L.ci, G.esi - i0);
  if (kn <= 0 || jn <= 0 || np <= 0) return;     /* the whole block */
  auto uni = [](int i) { return __builtin_amdgcn_readfirstlane(i); };
  auto wrapi = [&](int i) { return ((i % G.esi) + G.esi) % G.esi; };
  auto node = [&](int row, int col) {            /* rows and columns from the tile's corner */
    const int j = (((j0 + row) % G.esj) + G.esj) % G.esj;
    const int k = (((k0 + col) % G.esk) + G.esk) % G.esk;
    return j * G.esk + k;
  };
  /* the thread's column of step t+1: inner columns row by row, then the rim's */
  const int q = (int)threadIdx.x, main = (L.jt + 2) * L.kt;
  const int row = q < main ? q / L.kt : (q - main) >> 1;
  const int col = q < main ? 1 + q - row * L.kt : ((q - main) & 1) ? kn + 1 : 0;
  const bool valid = row <= jn + 1 && col <= kn + 1;
  const bool out = valid && row >= 1 && row <= jn && col >= 1 && col <= kn;
  const int t0 = node(min(row, jn + 1) - 1, min(col, kn + 1) - 1);
  const int l1 = valid ? row * S1 + col : M1;
  const int l2 = valid ? (row + 1) * S2 + col + 1 : S2 + 1;
  /* its two columns of the records in LDS */
  auto place = [&](int m) { return min(q + m * (int)blockDim.x, M2); };
  auto column = [&](int e) {
    const int r = e / S2, c = e - r * S2;
    return node(min(r, jn + 3) - 2, min(c, kn + 3) - 2);
  };
  const int ea = place(0), eb = place(1), ta = column(ea), tb = column(eb);
  /* (field by field: a record copied whole stays in scratch memory, and its
   * spill waits for every load in flight) */
  auto copy = [](R &d, const R &s) {
    d.p = s.p;
    if constexpr (NMOM > 1) { d.m1 = s.m1; d.m2 = s.m2; }
  };
  auto fetch = [&](R &ra, R &rb, int pl) {
    copy(ra, Q[(I)pl * (I)G.plane + (I)ta]);
    copy(rb, Q[(I)pl * (I)G.plane + (I)tb]);
  };
  auto put = [&](const R &ra, const R &rb, int slot) {
    copy(qs[slot * (M2 + 1) + ea], ra);
    copy(qs[slot * (M2 + 1) + eb], rb);
  };
  auto factors = [&](T (&w)[15], int pl) {
    const I x = (I)pl * (I)G.plane + (I)t0;
#pragma unroll
    for (int c = 0; c < 3; c++) {
      const V4 v = *(const V4 *)(wt + wt_idx<I>(c, x));
      w[4 * c] = v[0]; w[4 * c + 1] = v[1]; w[4 * c + 2] = v[2]; w[4 * c + 3] = v[3];
    }
    const Wt3<T> v = *(const Wt3<T> *)(wt + wt_idx<I>(3, x));
    w[12] = v.a; w[13] = v.b; w[14] = v.c;
  };
  /* k_mpstep_w's update of one node: sm, sc, sp the planes of its sources at
   * i - 1, i, i + 1, at its own place, rows S apart */
  auto update = [&](const T (&w)[15], uint32_t f, const R *sm, const R *sc, const R *sp,
                    int S) -> R {
    const R qx = *sc;
    T n0 = T(0), n1 = T(0), n2 = T(0);
    if ((f & 1u) || (f >> 17)) {
      const T pr = w[0];
      n0 += pr * qx.p;
      if constexpr (NMOM > 1) { n1 += pr * qx.m1; n2 += pr * qx.m2; }
    }
    Links<1, 15>::run([&](auto LL) {
      constexpr int l = decltype(LL)::value;
      const R *s = CX(l) > 0 ? sm : CX(l) < 0 ? sp : sc;
      const R qy = s[-CY(l) * S - CZ(l)];
      const T P = qy.p, pr = w[l];
      n0 += pr * P;
      if constexpr (NMOM > 1) {
        constexpr int dd = (AX == 0) ? CX(l) : (AX == 1) ? CY(l) : CZ(l);
        const T q1 = qy.m1;
        n1 += pr * (q1 + T(dd) * P);
        n2 += pr * (qy.m2 + T(2 * dd) * q1 + T(dd * dd) * P);
      }
    });
    R o;
    o.p = T(0);
    if constexpr (NMOM > 1) { o.m1 = T(0); o.m2 = T(0); }
    if (f & 1u) {
      o.p = n0;
      if constexpr (NMOM > 1) { o.m1 = n1; o.m2 = n2; }
    } else if (const T frac = mp_kept<T>(f, A); frac != T(0)) {
      o.p = qx.p + frac * n0;
      if constexpr (NMOM > 1) { o.m1 = qx.m1 + frac * n1; o.m2 = qx.m2 + frac * n2; }
    }
    return o;
  };
  R ra, rb;
#pragma unroll
  for (int u = 0; u < 3; u++) {                   /* planes i0 - 2, i0 - 1, i0 */
    fetch(ra, rb, uni(wrapi(i0 - 2 + u)));
    put(ra, rb, u);
  }
  int pm = uni(wrapi(i0 - 2)), pl = uni(wrapi(i0 - 1)), pp = uni(wrapi(i0));
  int p3 = uni(wrapi(i0 + 1));                    /* the plane in flight */
  fetch(ra, rb, p3);
  T wa[15], wb[15], wc[15];
  factors(wa, pl);
#pragma unroll
  for (int l = 0; l < 15; l++) { wb[l] = T(0); wc[l] = T(0); }
  uint32_t f = mpf[(long)pl * G.plane + t0], fp = 0;
  __syncthreads();
  auto plane = [&](const T (&w)[15], T (&wn)[15], const T (&wp)[15], int s) {
    put(ra, rb, (s + 3) & 3);
    uint32_t fn = 0;
    const int p4 = uni(p3 + 1 < G.esi ? p3 + 1 : 0);
    if (s < np + 1) {
      fetch(ra, rb, p4);
      factors(wn, pp);
      fn = mpf[(long)pp * G.plane + t0];
    }
    ts[(s & 3) * (M1 + 1) + l1] =
        update(w, f, qs + (s & 3) * (M2 + 1) + l2, qs + ((s + 1) & 3) * (M2 + 1) + l2,
               qs + ((s + 2) & 3) * (M2 + 1) + l2, S2);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    if (out && s >= 2) {
      const R *tr = ts + l1;
      const R o = update(wp, fp, tr + ((s + 2) & 3) * (M1 + 1), tr + ((s + 3) & 3) * (M1 + 1),
                         tr + (s & 3) * (M1 + 1), S1);
      qout[(long)pm * G.plane + t0] = o;
    }
    fp = f; f = fn;
    pm = pl; pl = pp; pp = uni(pp + 1 < G.esi ? pp + 1 : 0); p3 = p4;
  };
  /* planes i0 - 1 .. i0 + np: the first two only start the march */
  for (int s = 0;;) {
    plane(wa, wb, wc, s);
    if (++s == np + 2) break;
    plane(wb, wc, wa, s);
    if (++s == np + 2) break;
    plane(wc, wa, wb, s);
    if (++s == np + 2) break;
  }
}

/* Tiles: as slbd_step2_plan, the split of least cost over rounds of blocks,
 * with the same weights for short and unaligned rows (128^3 FP32: 13 x 64 19.6
 * us per step, 5 x 128 23.6, 26 x 26 27.2). */
extern "C" int slbd_mp2_plan(int esi, int esj, int esk, int prec, int nmom, MP2Plan *best) {
  const int cap = prec == 32 ? MP2Cfg<float>::NTHR : MP2Cfg<double>::NTHR;
  const long rec = (long)(prec / 8) * (nmom > 1 ? 3 : 1);
  const int cus = 256;
  double bc = 0.0;
  best->ci = 0;
  for (int nk = 1; nk <= (esk + 15) / 16; nk++) {
    const int kt = (esk + nk - 1) / nk, nkt = (esk + kt - 1) / kt;
    const double row = (1.0 + 16.0 / kt) * (nkt > 1 && kt % 32 ? 1.2 : 1.0);
    for (int jq = 1; jq <= esj; jq++) {
      const long m1 = (long)(jq + 2) * (kt + 2), m2 = (long)(jq + 4) * (kt + 4);
      if (m1 > cap || m2 > 2 * ((m1 + 63) & ~63L) || 4 * (m1 + m2 + 2) * rec > MP2_LDS) {
        if (m1 > cap) break;
        continue;
      }
      const int njt = (esj + jq - 1) / jq, jt = (esj + njt - 1) / njt;
      if (jt != jq) continue;
      for (int r = 1; r <= 3; r++) {
        const long tiles = (long)njt * nkt, fit = r * (long)cus / tiles;
        const int nch = fit < 1 ? 1 : fit > esi ? esi : (int)fit;
        const int ci = (esi + nch - 1) / nch, nc = (esi + ci - 1) / ci;
        const double cost = row * (double)((tiles * nc + cus - 1) / cus) * (ci + 2) *
                            ((double)m1 + (double)jt * kt + 1000.0);
        if (best->ci == 0 || cost < bc) {
          bc = cost;
          best->jt = jt; best->kt = kt; best->ci = ci;
          best->njt = njt; best->nkt = nkt; best->nch = nc;
        }
      }
    }
  }
  return best->ci > 0;
}

/* Whether two steps per pass are the faster way on the tiles of plan p, given
 * factors beyond the L2s.  `work`: nodes of step t+1 per node of the result,
 * the rim and the planes before and after a chunk included.  Not
 *   - with a work of more than 3.3 (one moment 3.5): single / two steps per
 *     pass, us per step with moments, FP32 1 x 1024 x 1024 14/23, 1 x 2923 x 899
 *     40/62, 1024 x 1024 x 1 14/17.5, FP64 1 x 2907 x 2023 196/270; one moment FP32
 *     1 x 1024 x 1024 12/16, but 1024 x 1024 x 1 (3.4) 11.8/10.8 and 1236 x 1 x 2635
 *     (3.2, moments) 38/23;
 *   - with moments and more than 2.3 in several rounds of blocks: FP32
 *     2 x 1024 x 1024 28.6/33.0 (one moment 23.2/23.2);
 *   - on planes of up to 128 nodes, a long march of a barrier and a load latency
 *     each (0.7-1.7 us per plane): 12000 x 10 x 10 FP32 17.4/33.5, one moment
 *     13.9/17.8, FP64 34/43, 24/26; but FP64 2236 x 2 x 70 14.8/12.2.
 * Elsewhere 0.47-0.95 of the time, a few FP32 shapes of 40-90 MB of factors
 * 1.0-1.07 (190 shapes). */
extern "C" int slbd_mp2_pays(int esj, int esk, int nmom, const MP2Plan *p) {
  const double work = (p->jt + 2.0) * (p->kt + 2.0) * (p->ci + 2.0) / ((double)p->jt * p->kt * p->ci);
  const long blocks = (long)p->njt * p->nkt * p->nch;
  if (work > (nmom > 1 ? 3.3 : 3.5)) return 0;
  if (nmom > 1 && work > 2.3 && blocks > 256) return 0;
  return (long)esj * esk > 128;
}

template <typename T, int NMOM, int AX>
static void launch_mp2(const void *wt, const void *q, void *qout, const uint32_t *mpf,
                       const Geom &G, const MPArgs &A, const MP2Plan &Q,
                       hipStream_t st) {
  typedef CRec<T, NMOM> R;
  const long m1 = (long)(Q.jt + 2) * (Q.kt + 2), m2 = (long)(Q.jt + 4) * (Q.kt + 4);
  const long thr = (m1 + 63) & ~63L;
  const size_t lds = 4 * (size_t)(m1 + m2 + 2) * sizeof(R);
  if (thr > MP2Cfg<T>::NTHR || m2 > 2 * thr || lds > MP2_LDS) {
    fprintf(stderr, "sunlightlb: a two-step tracer tile of %d x %d nodes does not fit a block\n",
            Q.jt, Q.kt);
    exit(EXIT_FAILURE);
  }
  const dim3 g((unsigned)(Q.njt * Q.nkt * Q.nch));
  hipLaunchKernelGGL((k_mpstep2<T, NMOM, AX, int>), g, dim3((unsigned)thr), lds, st, (const T *)wt,
                     (const R *)q, (R *)qout, mpf, G, A, Q);
  LAUNCHCHECK();
}

template <typename T>
static void launch_mp2_t(const void *wt, const void *q, void *qout, const uint32_t *mpf,
                         int nmom, const Geom &G, const MPArgs &A,
                         const MP2Plan &Q, hipStream_t st) {
  if (nmom == 1) launch_mp2<T, 1, 0>(wt, q, qout, mpf, G, A, Q, st);
  else if (A.axis == 0) launch_mp2<T, 3, 0>(wt, q, qout, mpf, G, A, Q, st);
  else if (A.axis == 1) launch_mp2<T, 3, 1>(wt, q, qout, mpf, G, A, Q, st);
  else launch_mp2<T, 3, 2>(wt, q, qout, mpf, G, A, Q, st);
}

void slbd_mp2_launch(const void *wt, const void *q, void *qout, const uint32_t *mpf,
                     int prec, int nmom, const Geom &G, const MPArgs &A,
                     const MP2Plan &Q, hipStream_t st) {
  if (prec == 32) launch_mp2_t<float>(wt, q, qout, mpf, nmom, G, A, Q, st);
  else launch_mp2_t<double>(wt, q, qout, mpf, nmom, G, A, Q, st);
}
