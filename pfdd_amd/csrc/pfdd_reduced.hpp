// pfdd_reduced.hpp -- the GL step in a reduced basis of the eigenstrains.
//
// The interaction matrix depends on the slip systems only through the
// symmetric parts of their eigenstrains: B_ab(k) = e_a : L(k) : e_b / mu with
// one fourth-order kernel L(k) = C - C.f G f.C for all pairs (Bmatrix,
// G.c:386-402).  The symmetric parts of S eigenstrains span R <= min(S, 6)
// dimensions (5 for the 12 FCC systems, whose strains are traceless; 2 for
// the three systems of one slip plane).  With a basis h_t of that span,
// e_a = sum_t al_at h_t,
//   sum_b B_ab xi_b^ = sum_t al_at [ sum_u K_tu(k) c_u^ ],
//   c_u = sum_b al_bu xi_b,   K_tu = h_t : L : h_u / mu,
// and the sums over a and b commute with the Fourier transform.  So a step
// transforms R component fields instead of S slip fields: the row kernel
// forms them from xi in real space right after the update, and expands the R
// transformed results to the S driving forces right before it.
//
// What bounds the step is memory traffic: per point 32 S + 32 R bytes in the
// row kernel and 3 x 32 R in the two N2 passes and the column kernel (FP64),
// against 160 S to 224 S with the transforms on the slip fields.  Measured per
// GL step, slip fields -> components: 128^3 x 12 FP64 682 -> 358 us, lean 346
// -> 218, 96^3 x 3 lean 121 -> 70, 256x256x192 x 3 FP64 1467 -> 836, 32^3 x 3
// FP64 33 -> 18; 256x256x128 x 12 mixed with stored B 3240 -> 1103 (15 stored
// values a k-point instead of 78).
//
// Layout: W[instance][N1][N2][N3][R], the components of a point together.
#pragma once
#include "pfdd_reduced.h"

namespace pfdd {

// ---------------------------------------------------------------- wave sums
template <int CTRL> __device__ __forceinline__ double dpp_mov(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, true);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
// Sums of four values over each row of 16 lanes at once: lane l with
// l % 4 = j returns the row's sum of v[j].  Each of the first two exchanges
// halves the values a lane carries, so four sums take 33 vector instructions
// instead of 4 x 12, and none of them goes through LDS.
__device__ __forceinline__ double row_sum4(const double (&v)[4]) {
  const bool b0 = threadIdx.x & 1, b1 = threadIdx.x & 2;
  const double k0 = (b0 ? v[1] : v[0]) + dpp_mov<0xB1>(b0 ? v[0] : v[1]);  // quad_perm 1,0,3,2
  const double k1 = (b0 ? v[3] : v[2]) + dpp_mov<0xB1>(b0 ? v[2] : v[3]);
  double k = (b1 ? k1 : k0) + dpp_mov<0x4E>(b1 ? k0 : k1);                 // quad_perm 2,3,0,1
  k += dpp_mov<0x124>(k);                                                  // row_ror 4
  k += dpp_mov<0x128>(k);                                                  // row_ror 8
  return k;
}

// ---------------------------------------------------------------- row kernel
// Two forms of the kernel, by the fields and components:
//  k_row_red    S <= 4 with R <= 3, and S <= 8 with R = 4: the update is
//               unrolled over the fields and all master points of a thread
//               are loaded before the transform, which hides their latency
//  k_row_red_n  any S: the fields pass through in chunks, the next chunk's
//               points loaded while one is updated (with 12 fields the first
//               form needs 146 registers and more in the mixed modes, and
//               measured 206 against 157 us at 128^3 x 12 mixed)
// Shape of a block.  The transform occupies R / 8 lanes per point (radix 8),
// so with one point per thread few lanes of a small R work in it: from N = 96
// on, R <= 3 takes PPT = 2 points per thread (4 in FP32 with R <= 2); shorter
// rows keep one, for more blocks on small grids (32^3 x 3: 7 against 9 us).
// Rows shorter than 32 fill a block of about 128 points with 128 / N of them,
// and the transform may then need more lanes than there are points.  N1 N2 rows
// need not be a multiple of ROWS: the last block may be short of rows.
template <typename T, int N, int R, int PPT_> struct RowRed {
  static constexpr int PPT = PPT_, ROWS = red_rows(N, PPT), PTS = ROWS * N, TPP = make_plan(N, RED_RL).tpp;
  static constexpr int LANES = ROWS * R * TPP, NEED = PTS / PPT > LANES ? PTS / PPT : LANES;
  static constexpr int NT = (NEED + 63) / 64 * 64;
  static constexpr int SH = 3, LD = padded_pitch<N, SH>(), NPEN = ROWS * R;
};
// The master advanced by a uniform offset (so that a thread's address is a
// scalar base and a 32-bit lane offset).
__device__ __forceinline__ Master<double> advance(Master<double> m, long o) { return {m.p + o}; }
__device__ __forceinline__ MasterF32C advance(MasterF32C m, long o) { return {m.r + o, m.im + o}; }
__device__ __forceinline__ MasterF32L advance(MasterF32L m, long o) { return {m.r + o}; }

// A pencil of the interleaved array as one thread sees it: element i at p[i * stride].
template <typename T> struct StridedPencil {
  cx<T>* p;
  long stride;
  static constexpr bool in_lds = false;
  __device__ __forceinline__ cx<T> load(int, int i) const { return p[i * stride]; }
  __device__ __forceinline__ void store(int, int i, cx<T> v) const { p[i * stride] = v; }
};

// The update's sine.  Cody-Waite reduction by pi/2 in three parts (the first
// with 33 bits, so that its products with |k| < 2^20 are exact), the remainder
// carried as r + t; sin r = r + r^3 S(r^2) and cos r = 1 - r^2/2 + r^4 C(r^2)
// on |r| <= pi/4 with S and C interpolated at Chebyshev nodes (6 terms each,
// relative errors 1.3e-17 and 5e-19).  Against 80-bit sinl over 5e6 arguments
// in each of |x| < 6.3 and |x| < 1000: at most 0.92 ulp, rms 0.295 (correct
// rounding gives 0.289).  31 vector instructions where the library's sine
// takes about 60.  Both hold for |x| < SIN_MAX; the row kernel sends larger
// arguments to big_sin (a function of its own: inlined, the library's long
// reduction takes 28 registers from the kernel).
constexpr double SIN_MAX = 4096.0;
static __device__ __attribute__((noinline, cold)) double big_sin(double x) { return sin(x); }
// The constants are kept in scalar registers (sgpr_const): left to itself the
// compiler, in the unrolled update, moves each into a vector register pair at
// every use, a third of the update's instructions.
__device__ __forceinline__ double sgpr_const(double v) {
  asm("" : "+s"(v));
  return v;
}
struct GlSin {
  const double inv = sgpr_const(0.6366197723675814), p1 = sgpr_const(-1.5707963267341256),
               p2 = sgpr_const(-6.077100506506192e-11), p3 = sgpr_const(-3.5215598651832e-27),
               s6 = sgpr_const(1.591805913698281e-10), s5 = sgpr_const(-2.5051130870968297e-08),
               s4 = sgpr_const(2.755731609787775e-06), s3 = sgpr_const(-0.0001984126983674956),
               s2 = sgpr_const(0.008333333333330943), s1 = sgpr_const(-0.16666666666666666),
               c6 = sgpr_const(-1.1382588535352522e-11), c5 = sgpr_const(2.0876145659059344e-09),
               c4 = sgpr_const(-2.755731726880539e-07), c3 = sgpr_const(2.4801587298760048e-05),
               c2 = sgpr_const(-0.0013888888888887393), c1 = sgpr_const(0.041666666666666664);
  __device__ __forceinline__ double operator()(double x) const {
    const double k = rint(x * inv);
    const double r1 = fma(k, p1, x), r = fma(k, p2, r1);
    const double t = fma(k, p3, fma(k, p2, r1 - r));
    const double z = r * r;
    double s = fma(z, s6, s5);
    s = fma(s, z, s4);
    s = fma(s, z, s3);
    s = fma(s, z, s2);
    s = fma(s, z, s1);
    s = r + fma(r * z, s, t);
    double c = fma(z, c6, c5);
    c = fma(c, z, c4);
    c = fma(c, z, c3);
    c = fma(c, z, c2);
    c = fma(c, z, c1);
    const double w = fma(-0.5, z, 1.0);
    c = w + fma(z * z, c, fma(-r, t, fma(-0.5, z, 1.0 - w)));
    const int q = (int)k;
    const double o = (q & 1) ? c : s;
    return (q & 2) ? -o : o;
  }
};
// The lean master's sine (xi carries 24 bits): reduction by pi, then 5 terms
// on |r| <= pi/2, absolute error 7e-11 where an FP32 sine of the reduced
// argument has 6e-8.
struct GlSinLean {
  const double inv = sgpr_const(0.3183098861837907), p1 = sgpr_const(-3.141592653589793),
               p2 = sgpr_const(-1.2246467991473532e-16), s5 = sgpr_const(-2.4079713707378346e-08),
               s4 = sgpr_const(2.753644296396837e-06), s3 = sgpr_const(-0.00019841086288980702),
               s2 = sgpr_const(0.008333332767631813), s1 = sgpr_const(-0.16666666663874308);
  __device__ __forceinline__ double operator()(double x) const {
    const double k = rint(x * inv);
    const double r = fma(k, p2, fma(k, p1, x));
    const double z = r * r;
    double s = fma(z, s5, s4);
    s = fma(s, z, s3);
    s = fma(s, z, s2);
    s = fma(s, z, s1);
    s = fma(r * z, s, r);
    return ((int)k & 1) ? -s : s;
  }
};

// One block: ROWS rows along N3 of all R components.  Inverse N3 transform
// (G.c:4638), then point by point: the S driving forces from the R components,
// plasticevolv (G.c:3470-3501) on the S fields, the new components from them,
// the fields' sums of Re xi / P; forward N3 transform (first pass of
// G.c:4599).  The first pass reads W into registers and the last writes it
// back.  A thread's master points are all loaded before the transform, which
// hides their latency.  Bound by HBM at R = 2 and 3 (256x256x192 x 3: FP64
// 322 us, 6.25 TB/s; mixed 214 us, 6.1 TB/s), with one point per thread and the
// points loaded a chunk ahead 395 and 377 us.  S <= SM.  grid = (row blocks,
// instances).
template <typename T, int N, int R, typename M, bool OPT>
__global__ void __launch_bounds__((RowRed<T, N, R, red_ppt(sizeof(T) == 8, N, R)>::NT), N == 512 ? 1 : 4)
k_row_red(cx<T>* __restrict__ W, M xi, const RedArgs a, const RedOpt<T> o, const cx<T>* __restrict__ tw,
          double* __restrict__ partials, const int* __restrict__ step_ctr) {
  using K = RowRed<T, N, R, red_ppt(sizeof(T) == 8, N, R)>;
  constexpr int NT = K::NT, LD = K::LD, TPP = K::TPP, SH = K::SH, ROWS = K::ROWS, PPT = K::PPT, SM = red_unrolled(R);
  static_assert(K::LANES <= NT && SM % 4 == 0 && NT >= MAXS, "block shape");
  __shared__ cx<T> sm[K::NPEN * LD];
  __shared__ cx<T> twl[N];
  __shared__ double tq[MAXS], rowsum[NT / 16][MAXS];
  const int t = threadIdx.x, S = a.S, inst = blockIdx.y;
  const long blk = blockIdx.x, P = a.P, pt0 = blk * (ROWS * N);
  // FFT lanes: component fastest, then the lane within the pencil, then the row
  const int fc = t % R, fq = (t / R) % TPP, fr = t / (R * TPP);
  const int nr = P / N - blk * ROWS < ROWS ? (int)(P / N - blk * ROWS) : ROWS;  // rows of this block
  const int pen = fr < nr ? fr * R + fc : 1 << 30;
  const StridedPencil<T> g{W + ((long)inst * P + pt0 + (long)fr * N) * R + fc, R};
  const LdsPencils<T, SH> l{sm, LD};
  TwStage<T, N, NT> ts;
  ts.load(tw);
  const long x0 = (long)inst * S * P + pt0;  // the block's first point of field 0
  typename M::Raw raw[PPT][SM];
#pragma unroll
  for (int f = 0; f < SM; f++)
    if (f < S) {
      const M m = advance(xi, x0 + (long)f * P);
#pragma unroll
      for (int p = 0; p < PPT; p++)  // (a lane without a point loads the block's first)
        raw[p][f] = m.raw(t + p * NT < nr * N ? t + p * NT : 0);
    }
  // the options' arrays, loaded with the master: the per-point shear (over
  // dslip) or the uniform one, and the frozen flags as bits
  double pq[OPT ? PPT : 1][OPT ? SM : 1];
  unsigned frozen[OPT ? PPT : 1];
  if constexpr (OPT) {
#pragma unroll
    for (int p = 0; p < PPT; p++) {
      const int e0 = t + p * NT < nr * N ? t + p * NT : 0;
      frozen[p] = 0;
#pragma unroll
      for (int f = 0; f < SM; f++) {
        if (f >= S) continue;
        if (o.taupp) pq[p][f] = o.taupp[((long)inst * P + pt0 + e0) * S + f];
        if (o.mask) frozen[p] |= (o.mask[x0 + (long)f * P + e0] ? 1u : 0u) << f;
      }
    }
  }
  if (t < S) {
    const double2 tr = a.tau[inst * S + t];
    tq[t] = (tr.x + tr.y * (double)step_ctr[1]) / a.dslip[t];
  }
  const bool project = OPT && o.project;
  if (!project) {
    fft_pencils<T, N, 1, RED_RL>(g, l, l, pen, 1 << 30, K::NPEN, fq, (T)1, twl, [&] { ts.store(twl); });
  } else {
    ts.store(twl);
    __syncthreads();
  }
  const std::conditional_t<lean_master<M>(), GlSinLean, GlSin> glsin;
  double gsum[SM];
#pragma unroll
  for (int f = 0; f < SM; f++) gsum[f] = 0.0;
#pragma unroll
  for (int p = 0; p < PPT; p++) {
    const int e0 = t + p * NT;  // the point within the block
    if (e0 >= nr * N) continue;
    cx<T>* cell = sm + (e0 / N) * (R * LD) + lds_pos<SH>(e0 % N);
    double2 r[R], s[R];
#pragma unroll
    for (int c = 0; c < R; c++) {
      const cx<T> v = cell[c * LD];
      r[c] = make_double2((double)v.x, (double)v.y);
      s[c] = make_double2(0.0, 0.0);
    }
#pragma unroll
    for (int f = 0; f < SM; f++) {
      if (f >= S) continue;
      double2 x = M::widen(raw[p][f]);
      if (!project) {
        double dr = 0.0, di = 0.0;
#pragma unroll
        for (int c = 0; c < R; c++) {
          dr += a.al[f][c] * r[c].x;
          di += a.al[f][c] * r[c].y;
        }
        double q = tq[f];
        bool live = true;
        if constexpr (OPT) {
          const long e = x0 + (long)f * P + e0;
          if (o.extra) {
            const cx<T> v = o.extra[e];
            dr += (double)v.x;
            di += (double)v.y;
          }
          if (o.taupp) q = (pq[p][f] + a.tau[inst * S + f].y * (double)step_ctr[1]) / a.dslip[f];
          live = !((frozen[p] >> f) & 1);
        }
        if (live) {
          const double arg = a.two_pi * x.x;
          double sn = glsin(arg);
          if (__builtin_expect(fabs(arg) > SIN_MAX, 0)) sn = big_sin(arg);
          x.x -= a.cd2[f] * (a.uq2 * dr * a.inv_n + a.asf_pi[f] * sn - q);  // G.c:3485-3489
          x.y -= a.uq2 * a.cd2[f] * (di * a.inv_n);
          advance(xi, x0 + (long)f * P).store(e0, x);
        }
      }
#pragma unroll
      for (int c = 0; c < R; c++) {
        s[c].x += a.al[f][c] * x.x;
        s[c].y += a.al[f][c] * x.y;
      }
      gsum[f] += x.x;
    }
#pragma unroll
    for (int c = 0; c < R; c++) cell[c * LD] = {(T)s[c].x, (T)s[c].y};
  }
#pragma unroll
  for (int f = 0; f < SM; f += 4) {
    if (f >= S) continue;
    const double v[4] = {gsum[f], gsum[f + 1], gsum[f + 2], gsum[f + 3]};
    const double rs = row_sum4(v);
    if ((t & 15) < 4) rowsum[t >> 4][f + (t & 15)] = rs;
  }
  __syncthreads();
  if (t < S && !project) {
    double v = 0.0;
    for (int w = 0; w < NT / 16; w++) v += rowsum[w][t];
    partials[((long)inst * S + t) * a.nblk + blk] = v * a.inv_n;
  }
  fft_pencils<T, N, 1, RED_RL>(l, l, g, pen, 1 << 30, K::NPEN, fq, (T)-1, twl);
}

// plasticevolv (G.c:3485-3489) with the shear already divided by dslip.
template <bool F32SIN>
__device__ __forceinline__ void gl_point_q(double2& x, double dre, double dim, double cd2, double asf_pi, double tq,
                                           const RedArgs& a) {
  const double arg = a.two_pi * x.x;
  double sn;
  if constexpr (F32SIN) {
    constexpr double TWO_PI_HI = 6.283185307179586, TWO_PI_LO = 2.4492935982947064e-16;
    const double k = rint(arg * (1.0 / TWO_PI_HI));
    sn = (double)sinf((float)fma(-k, TWO_PI_LO, fma(-k, TWO_PI_HI, arg)));
  } else {
    sn = sin(arg);
  }
  x.x -= cd2 * (a.uq2 * dre * a.inv_n + asf_pi * sn - tq);
  x.y -= a.uq2 * cd2 * (dim * a.inv_n);
}

// The form for any S.  Chunk length and register bound by measurement, at
// 128^3 x 12 and 256x256x128 x 12 (us): FP64 chunks of 4 without a bound 183
// and 786 (chunks of 2 with four waves a SIMD 177 and 820); the compensated
// mode chunks of 2 and four waves 155 and 559 (chunks of 4: 155 and 572); lean
// chunks of 4 and five waves 106 (115 without the bound).  FP64 runs at HBM
// speed (6.3 TB/s); the mixed modes are bound by vector issue (69% of the
// cycles).  Its sine is the library's: with GlSin it measured slower in FP64
// and lean (187 and 115 us), where the constants crowd out points in flight.
template <typename M> constexpr int row_n_chunk() { return __is_same(M, MasterF32C) ? 2 : 4; }
template <typename M> constexpr int row_n_waves() { return __is_same(M, MasterF32C) ? 4 : lean_master<M>() ? 5 : 1; }
template <typename T, int N, int R, typename M, bool OPT>
__global__ void __launch_bounds__((RowRed<T, N, R, 1>::NT), (row_n_waves<M>()))
k_row_red_n(cx<T>* __restrict__ W, M xi, const RedArgs a, const RedOpt<T> o, const cx<T>* __restrict__ tw,
          double* __restrict__ partials, const int* __restrict__ step_ctr) {
  using K = RowRed<T, N, R, 1>;
  constexpr int NT = K::NT, LD = K::LD, TPP = K::TPP, SH = K::SH, ROWS = K::ROWS, CH = row_n_chunk<M>();
  static_assert(K::LANES <= NT && NT >= MAXS, "block shape");
  __shared__ cx<T> sm[K::NPEN * LD];
  __shared__ cx<T> twl[N];
  __shared__ double tq[MAXS], rowsum[NT / 16][MAXS];
  const int t = threadIdx.x, S = a.S, inst = blockIdx.y;
  const long blk = blockIdx.x, P = a.P, pt0 = blk * (ROWS * N);  // one point per thread
  // FFT lanes: component fastest, then the lane within the pencil, then the row
  const int fc = t % R, fq = (t / R) % TPP, fr = t / (R * TPP);
  const int nr = P / N - blk * ROWS < ROWS ? (int)(P / N - blk * ROWS) : ROWS;  // rows of this block
  const int pen = fr < nr ? fr * R + fc : 1 << 30;
  const StridedPencil<T> g{W + ((long)inst * P + pt0 + (long)fr * N) * R + fc, R};
  const LdsPencils<T, SH> l{sm, LD};
  TwStage<T, N, NT> ts;
  ts.load(tw);
  const long xo = (long)inst * S * P + pt0 + (t < nr * N ? t : 0);  // this thread's point of field 0 (or the block's first)
  const bool has = t < nr * N;  // this thread has a point
  typename M::Raw cur[CH], nxt[CH];
#pragma unroll
  for (int j = 0; j < CH; j++)
    if (j < S) cur[j] = xi.raw(xo + (long)j * P);
  if (t < S) {
    const double2 tr = a.tau[inst * S + t];
    tq[t] = (tr.x + tr.y * (double)step_ctr[1]) / a.dslip[t];
  }
  const bool project = OPT && o.project;
  if (!project) {
    fft_pencils<T, N, 1, RED_RL>(g, l, l, pen, 1 << 30, K::NPEN, fq, (T)1, twl, [&] { ts.store(twl); });
  } else {
    ts.store(twl);
    __syncthreads();
  }
  cx<T>* cell = sm + (has ? (t / N) * (R * LD) + lds_pos<SH>(t % N) : 0);
  cx<T> r[R];
  double2 s[R];
#pragma unroll
  for (int c = 0; c < R; c++) {
    r[c] = cell[c * LD];
    s[c] = make_double2(0.0, 0.0);
  }
#pragma unroll 1
  for (int a0 = 0; a0 < S; a0 += CH) {
#pragma unroll
    for (int j = 0; j < CH; j++)
      if (a0 + CH + j < S) nxt[j] = xi.raw(xo + (long)(a0 + CH + j) * P);
    double gm[CH];
#pragma unroll
    for (int j = 0; j < CH; j++) {
      gm[j] = 0.0;
      if (a0 + j >= S || !has) continue;
      const int f = a0 + j;
      double2 x = M::widen(cur[j]);
      if (!project) {
        double dr = 0.0, di = 0.0;
#pragma unroll
        for (int c = 0; c < R; c++) {
          dr += a.al[f][c] * (double)r[c].x;
          di += a.al[f][c] * (double)r[c].y;
        }
        const long e = xo + (long)f * P;
        double q = tq[f];
        bool live = true;
        if constexpr (OPT) {
          if (o.extra) {
            const cx<T> v = o.extra[e];
            dr += (double)v.x;
            di += (double)v.y;
          }
          if (o.taupp)
            q = (o.taupp[((long)inst * P + pt0 + t) * S + f] + a.tau[inst * S + f].y * (double)step_ctr[1]) / a.dslip[f];
          if (o.mask) live = o.mask[e] == 0;
        }
        if (live) {
          gl_point_q<lean_master<M>()>(x, dr, di, a.cd2[f], a.asf_pi[f], q, a);
          xi.store(e, x);
        }
      }
#pragma unroll
      for (int c = 0; c < R; c++) {
        s[c].x += a.al[f][c] * x.x;
        s[c].y += a.al[f][c] * x.y;
      }
      gm[j] = x.x;
    }
    double v4[4] = {gm[0], gm[1], 0.0, 0.0};
    if constexpr (CH == 4) v4[2] = gm[2], v4[3] = gm[3];
    const double rs = row_sum4(v4);
    if ((t & 15) < CH) rowsum[t >> 4][a0 + (t & 15)] = rs;
#pragma unroll
    for (int j = 0; j < CH; j++) cur[j] = nxt[j];
  }
  if (has) {
#pragma unroll
    for (int c = 0; c < R; c++) cell[c * LD] = {(T)s[c].x, (T)s[c].y};
  }
  __syncthreads();
  if (t < S && !project) {
    double v = 0.0;
    for (int w = 0; w < NT / 16; w++) v += rowsum[w][t];
    partials[((long)inst * S + t) * a.nblk + blk] = v * a.inv_n;
  }
  fft_pencils<T, N, 1, RED_RL>(l, l, g, pen, 1 << 30, K::NPEN, fq, (T)-1, twl);
}

// ---------------------------------------------------------------- column kernel
// Columns per block TC: row segments (R TC complex) of 128 to 192 bytes where
// 48 KB of LDS allow it; about 256 k-points where N < 32.  At 512, whose rows
// lie megabytes apart, 72 KB: two blocks a CU with segments of 128 bytes beat
// four with 64 (512x128x512 x 3 FP64 669 against 821 us, mixed 445 against 462;
// at 384 they do not: 384x96x384 x 3 355 against 323).
// Radix limit: two passes (16) are faster in FP32 and, in FP64, at 48 and 96;
// FP64's radix-16 pass at 128, 192 and 256 leaves half the lanes idle and
// measured slower (128^3 x 3: 51 against 42 us, 256x256x192 x 3: 279 against 220).
template <typename T, int N, int R> struct ColRed {
  static constexpr int RL = sizeof(T) == 8 && N >= 128 ? 8 : RED_RL;
  static constexpr int TPP = make_plan(N, RL).tpp, LD = pitch<N>();
  static constexpr size_t CSZ = sizeof(cx<T>), LIMIT = (N >= 512 ? 72 : 48) * 1024;
  static constexpr int tc() {
    int t = 1;
    if (N < 32) {
      while (N * t * 2 <= 256 && t * 2 * R * TPP <= 512) t *= 2;
      return t;
    }
    while (t * 2 * R * CSZ <= 192 && (size_t)t * 2 * R * LD * CSZ <= LIMIT && t * 2 * R * TPP <= 1024) t *= 2;
    return t;
  }
  static constexpr int TC = tc(), NPEN = R * TC;
  static constexpr size_t LDS = ((size_t)NPEN * LD + N) * CSZ;  // tile and twiddles
  static constexpr int LANES = (NPEN * TPP + 63) / 64 * 64;
  static constexpr int PTS = N * TC < 512 ? N * TC : 512;
  static constexpr int NT = LANES > PTS ? LANES : (PTS + 63) / 64 * 64;
  static constexpr int KPT = (N * TC + NT - 1) / NT;  // k-points per thread
  // The wave vectors are loaded with the tile in FP64 (256x256x192 x 3: 209
  // against 223 us); in FP32 that measured slower (128^3 x 12: 45 against 42),
  // and so it did in FP64 at 192 (192^3 x 3: 150 against 127).
  static constexpr bool KEARLY = sizeof(T) == 8 && N % 3 != 0;
};

// The two stages of the per-field sums ride along as extra blocks of the
// launches that follow the row kernel anyway (as launches of their own they
// take 5 us each, of the 16 to 25 us that a step of a 32^3 grid takes): when
// the row kernel wrote many block sums per field, blocks of the forward N2
// pass fold them to FOLD per field, and one block of the column kernel turns
// those into the history row.  A field is added by one wave in a fixed order,
// which is k_finish_sums' order for up to FOLD_ABOVE sums.
__device__ __forceinline__ double wave_range_sum(const double* __restrict__ v, int b0, int b1) {
  double acc = 0.0;
  for (int b = b0 + ((int)threadIdx.x & 63); b < b1; b += 64) acc += v[b];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
  return acc;
}
template <int NT> __device__ __forceinline__ void fold_block(const FoldJob& j, int blk) {
  constexpr int NW = NT / 64;
  const int w = threadIdx.x >> 6, k = blk * NW + w;
  if (w >= NW || k >= j.F * FOLD) return;
  const int f = k / FOLD, part = k % FOLD;
  const int per = (j.nblk + FOLD - 1) / FOLD, b0 = part * per;
  const double s = wave_range_sum(j.in + (long)f * j.nblk, b0, b0 + per < j.nblk ? b0 + per : j.nblk);
  if ((threadIdx.x & 63) == 0) j.out[(long)f * FOLD + part] = s;
}
// The sums of fields f0 .. f0 + 3 (clamped to the last), their loads and
// exchanges in flight together: one field at a time, the 12 fields of a
// 32^3 grid took one wave 12 us, longer than the rest of the column kernel.
__device__ __forceinline__ void wave_sums4(const FinishJob& j, int f0, double (&s)[4]) {
  const double* v[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    v[i] = j.in + (long)(f0 + i < j.F ? f0 + i : j.F - 1) * j.nblk;
    s[i] = 0.0;
  }
  for (int b = (int)threadIdx.x & 63; b < j.nblk; b += 64)
#pragma unroll
    for (int i = 0; i < 4; i++) s[i] += v[i][b];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1)
#pragma unroll
    for (int i = 0; i < 4; i++) s[i] += __shfl_xor(s[i], o, 64);
}
// (The history row lies in host memory: it is written, never read back.)
constexpr int FINISH_LDS = 64;  // fields whose sums the block holds in LDS
__device__ __forceinline__ void finish_block(const FinishJob& j) {
  const int NT = blockDim.x, NW = NT / 64;
  __shared__ double fsum[FINISH_LDS];
  const int ninst = j.F / j.S, w = threadIdx.x >> 6;
  const bool lane0 = (threadIdx.x & 63) == 0;
  double* dst = j.out + (long)j.step_ctr[0] * ninst * (j.S + 1);
  double s[4];
  if (j.F <= FINISH_LDS) {
    for (int f0 = 4 * w; f0 < j.F; f0 += 4 * NW) {
      wave_sums4(j, f0, s);
#pragma unroll
      for (int i = 0; i < 4; i++)
        if (lane0 && f0 + i < j.F) dst[(f0 + i) / j.S * (j.S + 1) + (f0 + i) % j.S] = fsum[f0 + i] = s[i];
    }
    __syncthreads();
    for (int b = threadIdx.x; b < ninst; b += NT) {
      double tot = 0.0;
      for (int a = 0; a < j.S; a++) tot += fsum[b * j.S + a];
      dst[b * (j.S + 1) + j.S] = tot;
    }
  } else {  // an instance per wave
    for (int b = w; b < ninst; b += NW) {
      double tot = 0.0;
      for (int a0 = 0; a0 < j.S; a0 += 4) {
        wave_sums4(j, b * j.S + a0, s);
#pragma unroll
        for (int i = 0; i < 4; i++) {
          if (a0 + i >= j.S) continue;
          if (lane0) dst[b * (j.S + 1) + a0 + i] = s[i];
          tot += s[i];
        }
      }
      if (lane0) dst[b * (j.S + 1) + j.S] = tot;
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    j.step_ctr[0] = j.step_ctr[0] + 1;  // history row (read by every thread before the barrier above)
    j.step_ctr[1] = j.step_ctr[1] + 1;  // GL steps since the tau ramp was set
  }
}

// green6 with a reciprocal per distinct denominator (5 divisions instead of 25
// for a cubic material; the same to rounding).
__device__ __forceinline__ bool green6_rcp(const double f[3], const ElasticConsts* __restrict__ ec, double g[6]) {
  const double a = f[0] * f[0], b = f[1] * f[1], c = f[2] * f[2], fk2 = a + b + c;
  if (!(fk2 > 0.0)) return false;
  const double inv = 1 / fk2;
  double m0, m1, m2, w;  // 1 / m_i and (mu + lambda) / kk / |f|^2 of Bmatrix
  if (ec->iso) {
    m0 = m1 = m2 = ec->inv_mu;
    w = ec->g_iso * ec->mu * ec->mu * inv;
  } else {
    const double mu = ec->mu, mup = ec->mup * inv, ml = ec->mu + ec->ll;
    m0 = 1 / (mu + mup * a);
    m1 = 1 / (mu + mup * b);
    m2 = 1 / (mu + mup * c);
    w = ml / (1.0 + ml * inv * (m0 * a + m1 * b + m2 * c)) * inv;
  }
  const double p0 = f[0] * m0, p1 = f[1] * m1, p2 = f[2] * m2;
  g[0] = inv * (m0 - p0 * p0 * w);
  g[1] = inv * (-p0 * p1 * w);
  g[2] = inv * (-p0 * p2 * w);
  g[3] = inv * (m1 - p1 * p1 * w);
  g[4] = inv * (-p1 * p2 * w);
  g[5] = inv * (m2 - p2 * p2 * w);
  return true;
}

// Stored mode: K(k) as its upper triangle in the working precision, the
// R (R + 1) / 2 values of a k-point together (so that a column tile reads them
// in stretches, as it reads W), built once in FP64.  One thread per k-point.
constexpr int red_tri(int a, int b, int R) { return a * R - a * (a - 1) / 2 + (b - a); }  // a <= b
template <typename T, int R>
__global__ void __launch_bounds__(256)
k_build_K(T* __restrict__ Kst, const ElasticConsts* __restrict__ ec, long P) {
  const long pt = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (pt >= P) return;
  double f[3], g[6], u[R][3];
  kvec(pt, ec, f);
  const bool nz = green6(f, ec, g);
#pragma unroll
  for (int b = 0; b < R; b++) sig_f(ec, b, f, u[b]);
#pragma unroll
  for (int a = 0; a < R; a++) {
    double gu[3];
    gmul(g, u[a], gu);
#pragma unroll
    for (int b = a; b < R; b++)
      Kst[pt * (R * (R + 1) / 2) + red_tri(a, b, R)] =
          nz ? (T)((ec->SE[a][b] - (gu[0] * u[b][0] + gu[1] * u[b][1] + gu[2] * u[b][2])) * ec->inv_mu) : (T)0;
  }
}
template <typename T, int R>
__device__ __forceinline__ void contract_stored_lds(cx<T>* io, int stride, const T* __restrict__ k) {
  T kv[R * (R + 1) / 2];
#pragma unroll
  for (int i = 0; i < R * (R + 1) / 2; i++) kv[i] = k[i];
  cx<T> v[R];
#pragma unroll
  for (int b = 0; b < R; b++) v[b] = io[b * stride];
#pragma unroll
  for (int a = 0; a < R; a++) {
    cx<T> o = {(T)0, (T)0};
#pragma unroll
    for (int b = 0; b < R; b++) {
      const T w = kv[a <= b ? red_tri(a, b, R) : red_tri(b, a, R)];
      o.x += w * v[b].x;
      o.y += w * v[b].y;
    }
    io[a * stride] = o;
  }
}

// One block: TC neighbouring (i2, i3) columns of all R components.  Forward
// N1 transform (last pass of G.c:4599), the contraction K(k) at every k of
// the columns (G.c:4609-4629 in the basis h_t; ec holds the basis strains in
// the place of the eigenstrains), inverse N1 transform (first pass of
// G.c:4638).  grid = instances x column tiles, and one block for the sums.
template <typename T, int N, int R, bool STORED>
__global__ void __launch_bounds__((ColRed<T, N, R>::NT))
k_col_red(cx<T>* __restrict__ W, const ElasticConsts* __restrict__ ec, const T* __restrict__ Kst, long P, int blocks,
          const cx<T>* __restrict__ tw, const FinishJob fin) {
  using K = ColRed<T, N, R>;
  constexpr int NT = K::NT, LD = K::LD, TPP = K::TPP, TC = K::TC, NPEN = K::NPEN;
  extern __shared__ unsigned char lds_raw[];  // K::LDS
  cx<T>* sm = reinterpret_cast<cx<T>*>(lds_raw);
  cx<T>* twl = sm + NPEN * LD;
  if ((int)blockIdx.x >= blocks) {
    finish_block(fin);
    return;
  }
  const int t = threadIdx.x;
  const long cols = P / N, tiles = (cols + TC - 1) / TC;
  const long bt = xcd_tile(blockIdx.x, blocks), inst = bt / tiles, m0 = (bt - inst * tiles) * TC;
  const int fp = t % NPEN, fq = t / NPEN;
  const int nc = cols - m0 < TC ? (int)(cols - m0) : TC;  // columns of this block
  const int pen = fq < TPP && fp < nc * R ? fp : 1 << 30;
  const StridedPencil<T> g{W + (inst * P + m0) * R + fp, cols * R};
  const LdsPencils<T> l{sm, LD};
  TwStage<T, N, NT> ts;
  ts.load(tw);
  double f[K::KPT][3];  // wave vectors of this thread's k-points
  if constexpr (!STORED && K::KEARLY) {
#pragma unroll
    for (int k = 0; k < K::KPT; k++) {
      const int e = t + k * NT, c = e / N;
      kvec(c < nc ? (long)(e % N) * cols + m0 + c : 0, ec, f[k]);
    }
  }
  fft_pencils<T, N, 1, K::RL>(g, l, l, pen, 1 << 30, NPEN, fq, (T)-1, twl, [&] { ts.store(twl); });
#pragma unroll
  for (int k = 0; k < K::KPT; k++) {
    const int e = t + k * NT, c = e / N, n = e % N;
    if (c >= nc) continue;
    cx<T>* io = sm + c * (R * LD) + n;
    if constexpr (STORED) {
      contract_stored_lds<T, R>(io, LD, Kst + ((long)n * cols + m0 + c) * (R * (R + 1) / 2));
    } else {
      double gr[6];
      if constexpr (!K::KEARLY) kvec((long)n * cols + m0 + c, ec, f[k]);
      const bool nz = green6_rcp(f[k], ec, gr);
      contract_stress_form_lds<T, R>(io, LD, ec, f[k], gr, nz);
    }
  }
  __syncthreads();
  fft_pencils<T, N, 1, K::RL>(l, l, g, pen, 1 << 30, NPEN, fq, (T)1, twl);
}

// ---------------------------------------------------------------- N2 pass
// Transform along N2 of the [outer][N][inner] components (inner = N3 R), as
// k_fft_cols; the last tile of a row may be narrower than the others.
// grid = fold blocks, then outer x tiles.
template <typename T, int N>
__global__ void __launch_bounds__((cols_threads<T, N, RED_RL>()))
k_pass2_red(cx<T>* __restrict__ data, int inner, int blocks, T sign, const cx<T>* __restrict__ tw, const FoldJob fold,
            int nfold) {
  constexpr int TILE = tile_cols<T, N, RED_RL>(), LD = pitch<N>(), NT = cols_threads<T, N, RED_RL>();
  extern __shared__ unsigned char lds_raw[];  // cols_lds_bytes<T, N, RED_RL>()
  cx<T>* sm = reinterpret_cast<cx<T>*>(lds_raw);
  __shared__ cx<T> twl[N];
  if ((int)blockIdx.x < nfold) {
    fold_block<NT>(fold, blockIdx.x);
    return;
  }
  TwStage<T, N, NT> ts;
  ts.load(tw);
  const int tiles = (inner + TILE - 1) / TILE;
  const long bt = xcd_tile((int)blockIdx.x - nfold, blocks);
  const long o = bt / tiles;
  const int i0 = (int)(bt - o * tiles) * TILE, np = inner - i0 < TILE ? inner - i0 : TILE;
  const ColPencils<T> g{data + o * N * inner + i0, inner};
  const LdsPencils<T> l{sm, LD};
  fft_pencils<T, N, 1, RED_RL>(g, l, g, (int)threadIdx.x % TILE, 1 << 30, np, (int)threadIdx.x / TILE, sign, twl,
                       [&] { ts.store(twl); });
}

// ---------------------------------------------------------------- plane kernel
// One block: the N1 x N2 plane of one i3, all R components, in LDS: forward N2
// and N1, K(k), inverse N1 and N2 -- the two N2 passes and the column kernel in
// one launch and one trip through memory, with their arithmetic.  On small
// grids a launch costs 4 to 5 us whatever it does (32x2x32 x 2: 14.2 against
// 11.1 us a step, 256x2x256 x 3: 29.7 against 21.2); on many planes the two
// trips count (64 instances of 32^3 x 3: 184 against 119).  Threads:
// plane_threads(), one pencil share each.  grid = instances x N3, and one
// block for the sums.
template <typename T> struct PlaneN2 {  // N2 pencils of the plane in LDS: pencil p = n1 R + c
  cx<T>* sm;
  int R, ld;
  static constexpr bool in_lds = true;
  __device__ __forceinline__ cx<T>* at(int p, int i) const { return sm + (i * R + p % R) * ld + p / R; }
  __device__ __forceinline__ cx<T> load(int p, int i) const { return *at(p, i); }
  __device__ __forceinline__ void store(int p, int i, cx<T> v) const { *at(p, i) = v; }
};
template <typename T, int N1, int N2>
__global__ void __launch_bounds__(plane_max_threads(sizeof(T) == 8))
k_plane_red(cx<T>* __restrict__ W, const ElasticConsts* __restrict__ ec, const T* __restrict__ Kst, int n3, int R,
            int blocks, const cx<T>* __restrict__ tw1, const cx<T>* __restrict__ tw2, const FinishJob fin) {
  constexpr int LD = pitch<N1>(), RL1 = plane_rl(sizeof(T) == 8, N1), P = N1 * N2;
  constexpr int TPP1 = make_plan(N1, RL1).tpp, TPP2 = make_plan(N2, RED_RL).tpp;
  extern __shared__ unsigned char lds_raw[];  // plane_lds()
  cx<T>* sm = reinterpret_cast<cx<T>*>(lds_raw);
  cx<T>*twl1 = sm + N2 * R * LD, *twl2 = twl1 + N1;
  if ((int)blockIdx.x >= blocks) {
    finish_block(fin);
    return;
  }
  const int t = threadIdx.x;
  const int b = (int)xcd_tile(blockIdx.x, blocks), inst = b / n3, i3 = b - inst * n3;
  cx<T>* base = W + ((long)inst * P * n3 + i3) * R;
  const cx<T> w1 = tw1[t < N1 ? t : N1 - 1], w2 = tw2[t < N2 ? t : N2 - 1];
  const int np2 = N1 * R, p2 = t % np2, q2 = t / np2;
  const int np1 = N2 * R, p1 = t % np1, q1 = t / np1;
  const int pen2 = q2 < TPP2 ? p2 : 1 << 30, pen1 = q1 < TPP1 ? p1 : 1 << 30;
  const StridedPencil<T> g{base + (long)(p2 / R) * N2 * n3 * R + p2 % R, (long)n3 * R};
  const PlaneN2<T> l2{sm, R, LD};
  const LdsPencils<T> l1{sm, LD};
  fft_pencils<T, N2, 1, RED_RL>(g, l2, l2, pen2, 1 << 30, np2, q2, (T)-1, twl2, [&] {
    if (t < N1) twl1[t] = w1;
    if (t < N2) twl2[t] = w2;
  });
  fft_pencils<T, N1, 1, RL1>(l1, l1, l1, pen1, 1 << 30, np1, q1, (T)-1, twl1);
  for (int e = t; e < P; e += blockDim.x) {
    const int i1 = e % N1, i2 = e / N1;
    const long k = ((long)i1 * N2 + i2) * n3 + i3;
    cx<T>* io = sm + i2 * R * LD + i1;
    double f[3], gr[6];
    bool nz = false;
    if (!Kst) {
      kvec(k, ec, f);
      nz = green6_rcp(f, ec, gr);
    }
    switch (R) {
#define PFDD_R(RR)                                                                       \
  case RR:                                                                               \
    if (Kst) contract_stored_lds<T, RR>(io, LD, Kst + k * (RR * (RR + 1) / 2));          \
    else contract_stress_form_lds<T, RR>(io, LD, ec, f, gr, nz);                         \
    break;
      PFDD_R(1) PFDD_R(2) PFDD_R(3) PFDD_R(4) PFDD_R(5) PFDD_R(6)
#undef PFDD_R
    }
  }
  __syncthreads();
  fft_pencils<T, N1, 1, RL1>(l1, l1, l1, pen1, 1 << 30, np1, q1, (T)1, twl1);
  fft_pencils<T, N2, 1, RED_RL>(l2, l2, g, pen2, 1 << 30, np2, q2, (T)1, twl2);
}

}  // namespace pfdd
