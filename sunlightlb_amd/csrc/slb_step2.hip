/*
 * slb_step2.hip -- two fused lattice-Boltzmann steps per pass over HBM.
 *
 * One step of k_step (slb_dev.hip) reads and writes every population once
 * and is bound by that traffic.  k_step2 advances a tile of JT x KT (j, k)
 * columns by two steps while it marches along i, so that two steps cost one
 * read and one write:
 *
 *   - per plane p the block computes step t+1 of the tile and a rim of one
 *     node around it ((JT + 2) x (KT + 2) columns, the pulls of k_step from
 *     the source buffer), and hands the 12 populations that leave their
 *     column to the neighbouring threads through LDS;
 *   - with plane p's populations there, step t+2 of plane p - 1 is complete:
 *     a population with c_x = -1 arrives from plane p now, one with c_x = 0
 *     was taken from the LDS one plane ago, one with c_x = +1 two planes ago
 *     (both wait in registers); the tile's nodes collide again and are
 *     written.
 *
 * Bound by HBM and its latency at 256^3: FP32 2.36 GB for two steps (1.17x
 * one read and one write), 80% of the copy rate, the VALU busy 40% of the
 * time; FP64 4.82 GB, 98%, 29%.  Measured, us per step, one
 * step at a time / this kernel: FP32 256^3 356.6/224.0 (252 on the slowest
 * card), 512^3 2957/1852,
 * 160^3 94.4/58.8, 96^3 20.7/12.6, 64^3 6.97/6.05; FP64 256^3 735/401,
 * 128^3 92.9/54.7, 32^3 5.69/3.87.
 *
 * A thread owns one (j, k) column over the whole march, so the index
 * arithmetic is done once.  The loads of plane p + 1 are issued between
 * plane p's first step and its barrier, and complete under its second step
 * (issued before the first step: 254 against 233 us per step at 256^3; after
 * the barrier: 252).  The two register sets alternate by name over an
 * unrolled pair of planes: copying one to the other makes each plane wait
 * for its loads and stores (239 us).  The LDS is double buffered: one barrier
 * per plane.  Every node runs the arithmetic of k_step (bounce-back,
 * collide_node): bit-identical results.  Walls are at rest: with the wall
 * terms of moving objects looked up link by link, their FP64 velocity loads and
 * the registers these take, the pair was slower than two steps (FP64 128^3 116
 * against 102 us per step, FP32 256^3 1323 against 388); rows of precomputed
 * terms, as k_bstep2 has them, were not tried here.
 */
#include "slb_dev.h"
#include "slb_kern.h"
#include "slb_step2.h"

/* MODE: slbd_step2_mode.  NT: non-temporal stores. */
template <typename T, int BF, int MODE, bool NT>
__global__ void __launch_bounds__(Step2Cfg<T>::NTHR)
k_step2(const T *__restrict__ src, T *__restrict__ dst, const uint16_t *__restrict__ flags,
        const T *__restrict__ bx, const T *__restrict__ by, const T *__restrict__ bz, Geom G,
        PhysArgs A, Step2Plan Q) {
  constexpr int M1 = Step2Cfg<T>::NTHR + 1;   /* the last slot takes the writes of idle threads */
  __shared__ T buf[2][12 * M1];
  /* blocks of one XCD (b % 8) take neighbouring tiles of one chunk: their
   * rims and k edges then hit the same L2 */
  const int nb = gridDim.x;
  const int b = (nb & 7) == 0 ? (int)(blockIdx.x & 7) * (nb >> 3) + (int)(blockIdx.x >> 3)
                              : (int)blockIdx.x;
  const int kt = b % Q.nkt, jt = (b / Q.nkt) % Q.njt, ch = b / (Q.nkt * Q.njt);
  const int k0 = kt * Q.kt, j0 = jt * Q.jt, i0 = ch * Q.ci;
  const int kn = min(Q.kt, G.esk - k0), jn = min(Q.jt, G.esj - j0), np = min(Q.ci, G.esi - i0);
  if (kn <= 0 || jn <= 0 || np <= 0) return;     /* the whole block */
  const int S = Q.kt + 2, main = (Q.jt + 2) * Q.kt;

  /* the KT inner columns row by row (aligned rows for the waves), then the
   * two rim columns */
  const int q = (int)threadIdx.x;
  const int row = q < main ? q / Q.kt : (q - main) >> 1;
  const int col = q < main ? 1 + q - row * Q.kt : ((q - main) & 1) ? kn + 1 : 0;
  const bool valid = row <= jn + 1 && col <= kn + 1;
  const bool out = valid && row >= 1 && row <= jn && col >= 1 && col <= kn;
  const int lidx = valid ? row * S + col : M1 - 1;
  /* periodic; threads past the tile repeat a node in range */
  const int j = (j0 + min(row, jn + 1) - 1 + G.esj) % G.esj;
  const int k = (k0 + min(col, kn + 1) - 1 + G.esk) % G.esk;
  const int t0 = j * G.esk + k;
  uint32_t off[9];         /* in-plane offset of (j - cy, k - cz): index 3 (cy + 1) + cz + 1 */
  {
    const AxisOff32 oj = axis_off32(j, G.esj, G.esk), ok = axis_off32(k, G.esk, 1);
#pragma unroll
    for (int c = 0; c < 9; c++) {
      const int t = t0 + (c / 3 == 0 ? oj.p : c / 3 == 2 ? oj.m : 0) +
                    (c % 3 == 0 ? ok.p : c % 3 == 2 ? ok.m : 0);
      off[c] = MODE == 3 ? (uint32_t)t
               : MODE == 1 ? (uint32_t)t * (uint32_t)sizeof(T)
                           : (uint32_t)pidx32(0, t) * (uint32_t)sizeof(T);
    }
  }
  auto uni = [](int i) { return __builtin_amdgcn_readfirstlane(i); };
  auto wrap = [&](int i) { return i < 0 ? i + G.esi : (i >= G.esi ? i - G.esi : i); };
  /* bit l of a flags word as a mask; x where it is set, else y */
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

  /* the 15 populations that stream into the column's node of plane pl (pm
   * and pp its neighbours): bounced links take the node's own opposite */
  auto load = [&](T (&v)[15], int pm, int pl, int pp, unsigned f) {
    const uint32_t o0 = MODE == 1 ? pop_byte<T>((uint32_t)pl * (uint32_t)G.plane * (uint32_t)sizeof(T) + off[4]) : 0;
    Links<0, 15>::run([&](auto LL) {
      constexpr int l = decltype(LL)::value;
      constexpr int c = 3 * (CY(l) + 1) + CZ(l) + 1;
      const int ps = CX(l) > 0 ? pm : CX(l) < 0 ? pp : pl;
      const int bb = l > 0 ? bit(f, l) : 0;
      if constexpr (MODE == 0) {
        const uint32_t pitch = 15u * (uint32_t)G.plane;
        const uint32_t pulled =
            ((uint32_t)ps * pitch + (uint32_t)(l * POP_TILE)) * (uint32_t)sizeof(T) + off[c];
        const uint32_t own =
            ((uint32_t)pl * pitch + (uint32_t)(OPP(l) * POP_TILE)) * (uint32_t)sizeof(T) + off[4];
        v[l] = *(const T *)((const char *)src + ((own & bb) | (pulled & ~bb)));
      } else if constexpr (MODE == 1) {
        /* both offsets from the lower of the two populations' runs: never negative */
        constexpr int lo = l < OPP(l) ? l : OPP(l);
        const uint32_t pulled =
            pop_byte<T>((uint32_t)ps * (uint32_t)G.plane * (uint32_t)sizeof(T) + off[c]) +
            (uint32_t)((l - lo) * POP_TILE * (long)sizeof(T));
        const uint32_t own = o0 + (uint32_t)((OPP(l) - lo) * POP_TILE * (long)sizeof(T));
        v[l] = *(const T *)((const char *)(src + lo * POP_TILE) + ((own & bb) | (pulled & ~bb)));
      } else if constexpr (MODE == 3) {
        const int o = bb ? pidx32(OPP(l), pl * G.plane + (int)off[4])
                         : pidx32(l, ps * G.plane + (int)off[c]);
        v[l] = src[o];
      } else {
        const long pitch = 15L * G.plane;
        const char *pulled = (const char *)(src + ((long)ps * pitch + l * POP_TILE)) + off[c];
        const char *own = (const char *)(src + ((long)pl * pitch + OPP(l) * POP_TILE)) + off[4];
        v[l] = *(const T *)(bb ? own : pulled);
      }
    });
  };
  /* collision of the column's node of plane pl */
  auto update = [&](T (&v)[15], int pl, unsigned f) {
    const bool solid = (f & FLAG_SOLID) != 0;
    if (!(A.skip_solid && solid)) {
      T jbx = T(0), jby = T(0), jbz = T(0);
      if (!solid) {
        jbx = T(A.bfx); jby = T(A.bfy); jbz = T(A.bfz);
        if (BF == 2) {
          const long x = (long)pl * G.plane + t0;
          jbx += bx[x]; jby += by[x]; jbz += bz[x];
        }
      }
      collide_node<T>(v, jbx, jby, jbz, A);
    }
  };
  auto flag = [&](int pl) -> unsigned { return flags[(long)pl * G.plane + t0]; };

  T va[15], vb[15];        /* a plane's arriving populations, then its step t+1; the next plane's */
  T a[15];                 /* step t+2 of plane pl - 1: what has arrived so far */
  T d[4], o[5];            /* c_x = +1 diagonals of plane pl - 1 for plane pl; own c_x = +1 */
  int pm = uni(wrap(i0 - 2 + G.esi)), pl = uni(wrap(i0 - 1)), pp = uni(i0);
  unsigned f = flag(pl), fn = flag(pp), fp = 0;
  load(va, pm, pl, pp, f);
#pragma unroll
  for (int l = 0; l < 15; l++) a[l] = T(0);
#pragma unroll
  for (int m = 0; m < 4; m++) d[m] = T(0);
#pragma unroll
  for (int m = 0; m < 5; m++) o[m] = T(0);

  /* one plane: v holds plane pl, nv receives plane pl + 1 */
  auto plane = [&](T (&v)[15], T (&nv)[15], T *B, int s) {
    const int p2 = uni(wrap(pp + 1));
    unsigned fn2 = 0;
    update(v, pl, f);
    Links<3, 15>::run([&](auto LL) {
      constexpr int l = decltype(LL)::value;
      B[XSLOT(l) * M1 + lidx] = v[l];
    });
    if (s < np + 1) {
      load(nv, pl, pp, p2, fn);
      fn2 = flag(p2);
    }
    lds_barrier();
    if (out) {
      auto pull = [&](auto LL) -> T {
        constexpr int l = decltype(LL)::value;
        return B[XSLOT(l) * M1 + lidx - CY(l) * S - CZ(l)];
      };
      if (s >= 2) {
        /* complete plane pl - 1: the c_x = -1 links arrive from plane pl */
        a[2] = pick(fp, 2, o[0], v[2]);
        a[8] = pick(fp, 8, o[4], pull(std::integral_constant<int, 8>{}));
        a[10] = pick(fp, 10, o[3], pull(std::integral_constant<int, 10>{}));
        a[12] = pick(fp, 12, o[2], pull(std::integral_constant<int, 12>{}));
        a[14] = pick(fp, 14, o[1], pull(std::integral_constant<int, 14>{}));
        update(a, pm, fp);
        const uint32_t o0 = MODE == 1 ? pop_byte<T>((uint32_t)pm * (uint32_t)G.plane * (uint32_t)sizeof(T) + off[4]) : 0;
        Links<0, 15>::run([&](auto LL) {
          constexpr int l = decltype(LL)::value;
          T *p;
          if constexpr (MODE == 0)
            p = (T *)((char *)dst + (((uint32_t)pm * (15u * (uint32_t)G.plane) +
                                      (uint32_t)(l * POP_TILE)) * (uint32_t)sizeof(T) + off[4]));
          else if constexpr (MODE == 1)
            p = (T *)((char *)(dst + l * POP_TILE) + o0);
          else if constexpr (MODE == 3)
            p = dst + pidx32(l, pm * G.plane + t0);
          else
            p = (T *)((char *)(dst + ((long)pm * (15L * G.plane) + l * POP_TILE)) + off[4]);
          if constexpr (NT) __builtin_nontemporal_store(a[l], p);
          else *p = a[l];
        });
      }
      /* plane pl: everything but its c_x = -1 links has arrived */
      a[0] = v[0];
      a[1] = pick(f, 1, v[2], o[0]);
      a[7] = pick(f, 7, v[14], d[0]);
      a[9] = pick(f, 9, v[12], d[1]);
      a[11] = pick(f, 11, v[10], d[2]);
      a[13] = pick(f, 13, v[8], d[3]);
      a[3] = pick(f, 3, v[4], pull(std::integral_constant<int, 3>{}));
      a[4] = pick(f, 4, v[3], pull(std::integral_constant<int, 4>{}));
      a[5] = pick(f, 5, v[6], pull(std::integral_constant<int, 5>{}));
      a[6] = pick(f, 6, v[5], pull(std::integral_constant<int, 6>{}));
      d[0] = pull(std::integral_constant<int, 7>{});
      d[1] = pull(std::integral_constant<int, 9>{});
      d[2] = pull(std::integral_constant<int, 11>{});
      d[3] = pull(std::integral_constant<int, 13>{});
      o[0] = v[1]; o[1] = v[7]; o[2] = v[9]; o[3] = v[11]; o[4] = v[13];
    }
    fp = f; f = fn; fn = fn2;
    pm = pl; pl = pp; pp = p2;
  };
  /* planes i0 - 1 .. i0 + np: the first two only start the march */
  for (int s = 0;;) {
    plane(va, vb, buf[0], s);
    if (++s == np + 2) break;
    plane(vb, va, buf[1], s);
    if (++s == np + 2) break;
  }
}

/* Tiles of a lattice: the split of least cost, the plane passes over all
 * rounds of blocks (one block per CU) times a pass's work: both steps'
 * nodes and a constant for the barrier and the load latency (1000 nodes, from
 * tiles of 13 x 64 and 8 x 64 nodes at 256^3).  Short rows cost more (FP32
 * 256^3: 4 x 128 tiles 224 us per step, 13 x 64 232, 26 x 32 270), and so do
 * rows that start off a 128-byte line (FP64 256^3: 84 x 9 509, 64 x 8 401), which
 * those of a lattice with such rows do whatever the tile's width (FP32 20 x 109 x
 * 665: 28 x 32 tiles 34.6, 7 x 84 17.6). */
extern "C" int slbd_step2_plan(int esi, int esj, int esk, int prec, Step2Plan *best) {
  const int cap = prec == 32 ? Step2Cfg<float>::NTHR : Step2Cfg<double>::NTHR;
  const int cus = 256, wide = prec == 32 ? 160 : 100;
  double bc = 0.0;
  best->ci = 0;
  for (int nk = (esk + wide - 1) / wide; nk <= (esk + 31) / 32; nk++) {
    const int kt = (esk + nk - 1) / nk, nkt = (esk + kt - 1) / kt;
    const int jmax = cap / (kt + 2) - 2;
    const bool line = (long)kt * (prec / 8) % 128 == 0 && (long)esk * (prec / 8) % 128 == 0;
    const double row = (1.0 + 16.0 / kt) * (nkt > 1 && !line ? 1.2 : 1.0);
    for (int jq = 1; jq <= jmax && jq <= esj; jq++) {
      const int njt = (esj + jq - 1) / jq, jt = (esj + njt - 1) / njt;
      for (int r = 1; r <= 3; r++) {     /* as many chunks as r rounds hold */
        const long tiles = (long)njt * nkt, fit = r * (long)cus / tiles;
        const int nch = fit < 1 ? 1 : fit > esi ? esi : (int)fit;
        const int ci = (esi + nch - 1) / nch, nc = (esi + ci - 1) / ci;
        const double cost = row * (double)((tiles * nc + cus - 1) / cus) * (ci + 2) *
                            ((double)(jt + 2) * (kt + 2) + (double)jt * kt + 1000.0);
        if (best->ci == 0 || cost < bc) {
          bc = cost;
          best->jt = jt; best->kt = kt; best->ci = ci;
          best->njt = (esj + jt - 1) / jt; best->nkt = nkt; best->nch = nc;
        }
      }
    }
  }
  return best->ci > 0;
}

extern "C" int slbd_step2_mode_ok(int mode, long plane, long N, int prec) {
  const long ts = prec == 32 ? 4 : 8, four = 1L << 32, np = 15 * pop_nodes(N);
  const bool whole = plane % POP_TILE == 0;
  switch (mode) {
    case 0: return whole && np * ts < four;
    case 1: return np * ts < four;
    case 2: return whole && 15 * plane * ts < four;
    case 3: return np <= 0x7fffffffL;
    default: return 0;
  }
}

extern "C" int slbd_step2_mode(long plane, long N, int prec) {
  for (int m = 0; m < 4; m++)
    if (slbd_step2_mode_ok(m, plane, N, prec)) return m;
  return -1;
}

/* Whether two steps per pass are the faster way on the tiles of plan p.  A
 * block computes step t+1 on a rim around its tile and on the planes before
 * and after its chunk: `work` nodes per node of the result.  Not
 *   - in several rounds of blocks with a work of more than 3.2, as a single
 *     plane of a large lattice has (three planes marched for one): single / two
 *     steps per pass, us per FP32 step, 1 x 1024 x 1024 19/23, 1 x 2923 x 899
 *     54/65, 1 x 1 x 65536 3.9/5.1 (FP64 36/41, 1 x 759 x 2191 77/91, 4.8/8.6);
 *     but 2 x 1024 x 1024 (2.4) 36/32 (FP64 97/60), 1236 x 1 x 2635 in one round
 *     (3.1) 89/67, 1 x 256 x 256 4.6/3.5;
 *   - on long chunks of planes of up to 160 nodes (FP64 80), a march of a barrier
 *     and a load latency each for next to nothing (1.0-1.4 us per plane): 65536 x 1 x 1
 *     42/140, 4096 x 1 x 1 5.8/10.8, 1671 x 12 x 2 5.2/6.1, 5000 x 8 x 8 9.2/14.9 (FP64
 *     13/17), 12000 x 10 x 10 27.7/31.5; but FP64 12000 x 10 x 10 55/43, and in
 *     chunks of 4 planes 1000 x 10 x 10 6.3/5.3;
 *   - on a few long rows, which are split over k into tiles of mostly rim:
 *     3 x 8 x 2034 3.8/4.7, 7 x 7 x 1294 5.0/5.2.
 * Elsewhere it is faster or, within the spread of two runs of such calls,
 * equal (380 shapes with one to three short axes, 64 to 16 million nodes, both
 * precisions: 0.5-0.9 of the time, a few of 20-100 thousand nodes 1.0-1.1). */
extern "C" int slbd_step2_pays(int esi, int esj, int esk, int prec, const Step2Plan *p) {
  const double work = (p->jt + 2.0) * (p->kt + 2.0) * (p->ci + 2.0) / ((double)p->jt * p->kt * p->ci);
  const long blocks = (long)p->njt * p->nkt * p->nch, plane = (long)esj * esk;
  if (blocks > 256 && work > 3.2) return 0;
  if (plane * (prec / 8) <= 640 && p->ci > 6) return 0;
  if (esk > 1000 && work > 5.0 && esi * plane > 8192) return 0;
  return 1;
}

template <typename T, int MODE, bool NT>
static void launch2(const Step2Args *a, const PhysArgs &A, const Geom &G, hipStream_t st) {
  const int pts = (a->plan.jt + 2) * (a->plan.kt + 2);
  /* a block's threads and LDS hold the tile and its rim */
  if (pts > Step2Cfg<T>::NTHR) {
    fprintf(stderr, "sunlightlb: a two-step tile of %d x %d nodes does not fit a block\n",
            a->plan.jt, a->plan.kt);
    exit(EXIT_FAILURE);
  }
  const dim3 g((unsigned)(a->plan.njt * a->plan.nkt * a->plan.nch)), n((unsigned)((pts + 63) & ~63));
  if (a->bf == 2)
    hipLaunchKernelGGL((k_step2<T, 2, MODE, NT>), g, n, 0, st, (const T *)a->src, (T *)a->dst,
                       a->flags, (const T *)a->bx, (const T *)a->by, (const T *)a->bz, G, A,
                       a->plan);
  else
    hipLaunchKernelGGL((k_step2<T, 1, MODE, NT>), g, n, 0, st, (const T *)a->src, (T *)a->dst,
                       a->flags, (const T *)a->bx, (const T *)a->by, (const T *)a->bz, G, A,
                       a->plan);
  LAUNCHCHECK();
}

template <typename T>
static void launch2_t(const Step2Args *a, const PhysArgs &A, const Geom &G, hipStream_t st) {
  if (!slbd_step2_mode_ok(a->mode, G.plane, G.N, (int)sizeof(T) * 8)) {
    fprintf(stderr, "sunlightlb: a two-step pass cannot address this lattice in mode %d\n", a->mode);
    exit(EXIT_FAILURE);
  }
  if (a->mode == 0) {
    if (a->nt) launch2<T, 0, true>(a, A, G, st); else launch2<T, 0, false>(a, A, G, st);
  } else if (a->mode == 1) {
    if (a->nt) launch2<T, 1, true>(a, A, G, st); else launch2<T, 1, false>(a, A, G, st);
  } else if (a->mode == 2) {
    if (a->nt) launch2<T, 2, true>(a, A, G, st); else launch2<T, 2, false>(a, A, G, st);
  } else {
    if (a->nt) launch2<T, 3, true>(a, A, G, st); else launch2<T, 3, false>(a, A, G, st);
  }
}

void slbd_step2_launch(const Step2Args *a, const PhysArgs &A, const Geom &G, int prec,
                       hipStream_t st) {
  if (prec == 32) launch2_t<float>(a, A, G, st);
  else launch2_t<double>(a, A, G, st);
}
