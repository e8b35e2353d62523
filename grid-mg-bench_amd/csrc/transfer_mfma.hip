// Block transfers (project and promote) of several right-hand sides as matrix
// products on the FP32 / FP64 matrix cores.
//
// Per block and chirality k, with U the (block sites x Ef/2) x nb panel:
//   project:  c[i][r] = sum_q conj(U[q][i]) f[q][r]
//   promote:  f[q][r] = sum_i U[q][i] c[r][i]
// A complex product is four real 16x16x4 products on operands that stay
// interleaved in memory: a lane loads whole complex entries and hands the real
// and the imaginary parts to separate instructions, so nothing is staged or
// shuffled on the way in.  Lane layout of the 16x16x4 forms: A[m = l%16][k = l/16],
// B[k = l/16][n = l%16]; D[m][n = l%16] in register v holds m = 4 (l/16) + v in
// FP32 and m = 4 v + l/16 in FP64.
//
// What bounds them is HBM: the basis, V x Ef x nb entries, is read once per 16
// right-hand sides (the vector-unit kernels read it once per four), and the
// fine field is read or written once.  At 32^4, 4^4 blocks, nb 16, 12 rhs, FP32
// that is 2.8 GB a direction (3.24 and 2.84 measured): project 0.50 ms (1.45 ms in the
// vector form), promote 0.59 ms (1.27 ms).
//
// Both kernels are instantiated for the width of the basis.  VEC: nb allows
// vector loads of it; FAST: Ef = 12 and a fine field at a 16-byte address.
#include "aggregation.hpp"

#include <algorithm>

namespace mgc {

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef double f64x4 __attribute__((ext_vector_type(4)));

template <typename R> struct Mfma;
template <> struct Mfma<float> {
  typedef f32x4 acc_t;
  __device__ static __forceinline__ acc_t go(float a, float b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  __device__ static __forceinline__ int row(int lane_group, int v) { return 4 * lane_group + v; }
};
template <> struct Mfma<double> {
  typedef f64x4 acc_t;
  __device__ static __forceinline__ acc_t go(double a, double b, acc_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  __device__ static __forceinline__ int row(int lane_group, int v) { return 4 * v + lane_group; }
};

constexpr int TRC = 16;  // right-hand sides per workgroup: the columns of one tile

// N consecutive complex entries; pairs of FP32 entries in one 16-byte load
// where the caller knows p to be 16-byte aligned (PAIRED, even N)
template <typename R, int N, bool PAIRED>
__device__ __forceinline__ void load_run(const cplx<R>* p, cplx<R>* o) {
  if constexpr (sizeof(R) == 4 && PAIRED && N % 2 == 0) {
#pragma unroll
    for (int q = 0; q < N / 2; ++q) {
      const float4 t = reinterpret_cast<const float4*>(p)[q];
      o[2 * q] = {t.x, t.y};
      o[2 * q + 1] = {t.z, t.w};
    }
  } else {
#pragma unroll
    for (int q = 0; q < N; ++q) o[q] = p[q];
  }
}

// ---------------------------------------------------------------------------
// project.  One workgroup per (coarse site, 16 rhs, range of block sites).  A
// wavefront takes four sites at a time, one per lane group (the K index of the
// product), and EU elements of each: lane (g, j) loads the basis entries
// MT j .. MT j + MT - 1 of its site's rows and the elements of rhs j.  The
// products of CH elements (2 * 4 * CH of them) start from zero and are then added to
// the running sums; the wavefronts' sums meet in LDS.  The rounding error grows with
// the square root of the additions in a row, 8 CH and the running sums' after them;
// the vector form, with two stages over a block's rows, makes 2 sqrt(rows) at best.
// CH = 2 keeps below that from eight Dirac sites a block up (agg_transfer asks for
// them).  Where a workgroup has 64 sites or more, FP32 affords all six elements of a
// chirality in one chain, with fewer registers and additions; ranges shorter than
// that of a split panel take one element in FP64 (nb to 32, where registers allow).
// Error in FP32, nb 32: at 2^4 blocks 8.8e-8 (vector form 1.02e-7, six in a chain
// 1.31e-7), at 4^4 1.46e-7 (2.7e-7).  Two in a chain throughout, three elements a
// step in FP32: up to 1.18 times the time (32^4, 4^4 blocks, nb 16, 12 rhs).
// Sites past the range or outside the mask enter as zeros on both sides.
// ---------------------------------------------------------------------------
template <typename R, int MT, bool VEC, bool FAST, int CH>
__global__ __launch_bounds__(512) void k_project_mfma(
    const cplx<R>* __restrict__ U, const cplx<R>* __restrict__ f, cplx<R>* __restrict__ c,
    const int* __restrict__ blk_fine, int nb, int Vb, int Ef_, int nrhs, Lat4 blk, int kind,
    int point, int sites_per, cplx<R>* __restrict__ part) {
  typedef typename Mfma<R>::acc_t acc_t;
  // elements per step: as many loads in flight as the registers allow
  constexpr bool wide = sizeof(R) == 8;
  constexpr int EU = !FAST ? (wide ? 2 : 4) : !wide && (CH == 6 || MT == 1) ? 6 : 3;
  const int Ef = FAST ? 12 : Ef_;
  const int half = Ef / 2;
  extern __shared__ unsigned char smem_raw[];
  acc_t* s_acc = reinterpret_cast<acc_t*>(smem_raw);  // [waves / 2][MT][2][64]
  const int xc = blockIdx.x;
  const int r0 = blockIdx.y * TRC;
  const int nr = min(TRC, nrhs - r0);
  const int w = threadIdx.x >> 6, nw = blockDim.x >> 6;
  const int l = threadIdx.x & 63, g = l >> 4, j = l & 15;
  const int rj = min(j, nr - 1);  // columns past nr repeat the last one and are not stored
  // basis entries of this lane (those past nb repeat the last ones and are not stored)
  int im[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m)
    im[m] = VEC ? min(j, nb / MT - 1) * MT + m : min(j * MT + m, nb - 1);
  const cplx<R>* Ub = U + (size_t)xc * Vb * Ef * nb;
  const int* bf = blk_fine + (size_t)xc * Vb;
  const int sbeg = blockIdx.z * sites_per, send = min(Vb, sbeg + sites_per);
  acc_t tot[2][MT][2];
#pragma unroll
  for (int k = 0; k < 2; ++k)
#pragma unroll
    for (int m = 0; m < MT; ++m) tot[k][m][0] = tot[k][m][1] = acc_t{0, 0, 0, 0};
  for (int s0 = sbeg + 4 * w; s0 < send; s0 += 4 * nw) {
    const int s = s0 + g, sc = min(s, send - 1);
    const bool ok = s < send && (kind == 0 || site_in_mask(blk, s, kind, point));
    const cplx<R>* fp = f + ((size_t)bf[sc] * nrhs + r0 + rj) * Ef;
    const cplx<R>* up = Ub + (size_t)sc * Ef * nb;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
#pragma unroll 1
      for (int eb = 0; eb < half; eb += EU) {
        cplx<R> u[EU][MT], x[EU];
#pragma unroll
        for (int e = 0; e < EU; ++e) {
          const int ee = half * k + (FAST ? eb + e : min(eb + e, half - 1));
          if constexpr (VEC) {
            load_run<R, MT, true>(up + (size_t)ee * nb + im[0], u[e]);
          } else {
#pragma unroll
            for (int m = 0; m < MT; ++m) u[e][m] = up[(size_t)ee * nb + im[m]];
          }
          if constexpr (!FAST) x[e] = fp[ee];
        }
        if constexpr (FAST) load_run<R, EU, true>(fp + half * k + eb, x);
        // conj(u) x: re = u.re x.re + u.im x.im, im = u.re x.im - u.im x.re
#pragma unroll
        for (int e0 = 0; e0 < EU; e0 += CH) {
          acc_t acc[MT][2];
#pragma unroll
          for (int m = 0; m < MT; ++m) acc[m][0] = acc[m][1] = acc_t{0, 0, 0, 0};
#pragma unroll
          for (int e = e0; e < (e0 + CH < EU ? e0 + CH : EU); ++e) {
            const bool in = ok && (FAST || eb + e < half);
            if (!in) {
              x[e] = {R(0), R(0)};
#pragma unroll
              for (int m = 0; m < MT; ++m) u[e][m] = {R(0), R(0)};
            }
            const R nx = -x[e].re;
#pragma unroll
            for (int m = 0; m < MT; ++m) {
              acc[m][0] = Mfma<R>::go(u[e][m].re, x[e].re, acc[m][0]);
              acc[m][1] = Mfma<R>::go(u[e][m].re, x[e].im, acc[m][1]);
              acc[m][0] = Mfma<R>::go(u[e][m].im, x[e].im, acc[m][0]);
              acc[m][1] = Mfma<R>::go(u[e][m].im, nx, acc[m][1]);
            }
          }
#pragma unroll
          for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int t = 0; t < 2; ++t) tot[k][m][t] += acc[m][t];
        }
      }
    }
  }
  // the wavefronts' sums, one chirality at a time, in a fixed tree
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    for (int h = nw / 2; h >= 1; h /= 2) {
      __syncthreads();
      if (w >= h && w < 2 * h)
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
          for (int t = 0; t < 2; ++t)
            s_acc[(((w - h) * MT + m) * 2 + t) * 64 + l] = tot[k][m][t];
      __syncthreads();
      if (w < h)
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
          for (int t = 0; t < 2; ++t) tot[k][m][t] += s_acc[((w * MT + m) * 2 + t) * 64 + l];
    }
    if (w == 0 && j < nr) {
      cplx<R>* o = gridDim.z == 1
                       ? c + ((size_t)xc * nrhs + r0 + j) * 2 * nb + k * nb
                       : part + ((((size_t)xc * gridDim.y + blockIdx.y) * gridDim.z + blockIdx.z) *
                                     min(TRC, nrhs) + j) * 2 * nb + k * nb;
#pragma unroll
      for (int v = 0; v < 4; ++v)
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          const int i = Mfma<R>::row(g, v) * MT + m;
          if (i < nb) o[i] = {tot[k][m][0][v], tot[k][m][1][v]};
        }
    }
  }
}

// ---------------------------------------------------------------------------
// promote.  One workgroup per (coarse site, 16 rhs, range of 16-site groups).
// The columns of the product are 16 block sites (one per lane), the rows the
// right-hand sides and K the basis index in pairs: of each row lane group g
// holds the pairs g, 4 + g, ... (KP = ceil(nb / 8) of them, so that a load
// covers 64 bytes or more of a row); entries past nb, in the last pair only, enter
// as zeros on both sides.  The four wavefronts take EW elements each of a tile
// of EC = 4 EW elements (Ef = 12: the whole site, wavefronts 0 and 1 the first
// chirality; otherwise eight elements of one chirality at a time), and the tile
// leaves through LDS, so that a site's record is written in whole lines: stored
// from the product's registers, each lane's 16 bytes are a write request of
// their own (75 million of them at the size above, 1.68 ms against 0.6 ms).
// An element's 2 nb real products go to promote_chains chains at a time, new ones
// every promote_steps steps: the rounding error grows with the square root of a
// chain's length, and no chain is longer than those of the vector form, whose lanes
// for a row are two (FP64, four from nb 30 up) or one (FP32, two from nb 31, four
// from nb 60).
// Against one chain throughout that costs nothing to 10% of the time (FP64, nb
// 48, 12 rhs, 18^4: 290 -> 306 us) and takes the error at nb 48 from 3.3e-16 to
// 1.8e-16, in FP32 from 1.8e-7 to 1.3e-7.
// ---------------------------------------------------------------------------
constexpr int promote_ew(bool fast) { return fast ? 3 : 2; }
constexpr int promote_chains(int kp, size_t real) { return kp * real >= 16 || real == 8 ? 2 : 1; }
constexpr int promote_steps(int kp, size_t real) {
  return real == 4 ? 8 : kp <= 3 ? 2 * kp : 4;
}
// LDS entries of one site: nr x EC elements and 16 bytes against bank conflicts
template <typename R>
__host__ __device__ constexpr int promote_pitch(int nr, int ec) {
  return nr * ec + (int)(16 / sizeof(cplx<R>));
}

template <typename R, int KP, bool VEC, bool FAST>
__global__ __launch_bounds__(256) void k_promote_mfma(const cplx<R>* __restrict__ U,
                                                      const cplx<R>* __restrict__ c,
                                                      cplx<R>* __restrict__ f,
                                                      const int* __restrict__ blk_fine, int nb,
                                                      int Vb, int Ef_, int nrhs, int groups_per) {
  typedef typename Mfma<R>::acc_t acc_t;
  constexpr int EW = promote_ew(FAST), EC = 4 * EW;
  constexpr int KR = 2 * KP;  // basis entries per lane and row
  // a tile's basis entries are loaded together, and those of the next tile ahead
  // of this one's products, where the registers leave four wavefronts a SIMD
  constexpr bool AHEAD = KP * sizeof(R) <= 8, WHOLE = KP * sizeof(R) <= 24;
  const int Ef = FAST ? 12 : Ef_;
  const int half = Ef / 2;
  extern __shared__ unsigned char smem_raw[];
  cplx<R>* s_f = reinterpret_cast<cplx<R>*>(smem_raw);  // [16][pitch]
  const int xc = blockIdx.x;
  const int r0 = blockIdx.y * TRC;
  const int nr = min(TRC, nrhs - r0);
  const int pitch = promote_pitch<R>(nr, EC);
  const int w = threadIdx.x >> 6;
  const int l = threadIdx.x & 63, g = l >> 4, j = l & 15;
  const int rj = min(j, nr - 1);  // rows past nr repeat the last one and are not stored
  const cplx<R>* Ub = U + (size_t)xc * Vb * Ef * nb;
  const int* bf = blk_fine + (size_t)xc * Vb;
  // entry of step t, and whether it is past nb
  auto entry = [&](int t) { return 8 * (t / 2) + 2 * g + t % 2; };
  auto past = [&](int t) { return t / 2 == KP - 1 && entry(t) >= nb; };
  const int gbeg = blockIdx.z * groups_per, gend = min((Vb + 15) / 16, gbeg + groups_per);
  // the lane's entries of row e of its site in group sg
  auto fetch = [&](int sg, int e, cplx<R>(&u)[KR]) __attribute__((always_inline)) {
    const cplx<R>* up = Ub + ((size_t)min(sg * 16 + j, Vb - 1) * Ef + e) * nb;
    constexpr int ST = VEC ? 2 : 1;
#pragma unroll
    for (int t = 0; t < KR; t += ST) {
      load_run<R, ST, true>(up + (past(t) ? nb - ST : entry(t)), &u[t]);
      if (past(t))
#pragma unroll
        for (int v = 0; v < ST; ++v) u[t + v] = {R(0), R(0)};
    }
  };
  cplx<R> a[KR];
  R nai[KR];
  auto load_c = [&](int k) __attribute__((always_inline)) {
    const cplx<R>* cp = c + ((size_t)xc * nrhs + r0 + rj) * 2 * nb + k * nb;
#pragma unroll
    for (int t = 0; t < KR; ++t) {
      a[t] = cp[past(t) ? nb - 1 : entry(t)];
      if (past(t)) a[t] = {R(0), R(0)};
      nai[t] = -a[t].im;
    }
  };
  // products of one row and their way to LDS as element e of the tile
  auto product = [&](const cplx<R>(&u)[KR], int e) __attribute__((always_inline)) {
    // NC chains at a time, new ones every TG steps
    constexpr int NC = promote_chains(KP, sizeof(R)), TG = promote_steps(KP, sizeof(R));
    acc_t re, im;
#pragma unroll
    for (int t0 = 0; t0 < KR; t0 += TG) {
      acc_t sr[NC], si[NC];
#pragma unroll
      for (int q = 0; q < NC; ++q) sr[q] = si[q] = acc_t{0, 0, 0, 0};
#pragma unroll
      for (int t = t0; t < (t0 + TG < KR ? t0 + TG : KR); ++t) {
        acc_t &r = sr[t % NC], &i = si[t % NC];
        r = Mfma<R>::go(a[t].re, u[t].re, r);
        i = Mfma<R>::go(a[t].re, u[t].im, i);
        r = Mfma<R>::go(nai[t], u[t].im, r);
        i = Mfma<R>::go(a[t].im, u[t].re, i);
      }
      if (NC == 2) {
        sr[0] += sr[NC - 1];
        si[0] += si[NC - 1];
      }
      re = t0 ? re + sr[0] : sr[0];
      im = t0 ? im + si[0] : si[0];
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int r = Mfma<R>::row(g, v);
      if (r < nr) s_f[j * pitch + r * EC + e] = {re[v], im[v]};
    }
  };
  if constexpr (FAST) {
    load_c(w >> 1);
    cplx<R> nxt[AHEAD ? EW : 1][KR];
    if constexpr (AHEAD)
      if (gbeg < gend)
#pragma unroll
        for (int q = 0; q < EW; ++q) fetch(gbeg, w * EW + q, nxt[q]);
    for (int sg = gbeg; sg < gend; ++sg) {
      cplx<R> u[WHOLE ? EW : 1][KR];
      if constexpr (AHEAD) {
#pragma unroll
        for (int q = 0; q < EW; ++q)
#pragma unroll
          for (int t = 0; t < KR; ++t) u[q][t] = nxt[q][t];
        if (sg + 1 < gend)
#pragma unroll
          for (int q = 0; q < EW; ++q) fetch(sg + 1, w * EW + q, nxt[q]);
#pragma unroll
        for (int q = 0; q < EW; ++q) product(u[q], w * EW + q);
      } else if constexpr (WHOLE) {
#pragma unroll
        for (int q = 0; q < EW; ++q) fetch(sg, w * EW + q, u[q]);
#pragma unroll
        for (int q = 0; q < EW; ++q) product(u[q], w * EW + q);
      } else {
#pragma unroll 1
        for (int q = 0; q < EW; ++q) {
          fetch(sg, w * EW + q, u[0]);
          product(u[0], w * EW + q);
        }
      }
      __syncthreads();
      // whole records in units of 16 bytes
      constexpr int CU = 16 / (int)sizeof(cplx<R>);
      const int units = nr * EC / CU, ns = min(16, Vb - sg * 16);
      for (int t = threadIdx.x; t < ns * units; t += 256) {
        const int s = t / units, o = (t - s * units) * CU;
        *reinterpret_cast<float4*>(f + ((size_t)bf[sg * 16 + s] * nrhs + r0) * 12 + o) =
            *reinterpret_cast<const float4*>(s_f + s * pitch + o);
      }
      __syncthreads();
    }
  } else {
    for (int k = 0; k < 2; ++k) {
      load_c(k);
      for (int sg = gbeg; sg < gend; ++sg)
        for (int eb = 0; eb < half; eb += EC) {
          for (int q = 0; q < EW; ++q)
            if (eb + w * EW + q < half) {  // uniform over the wavefront
              cplx<R> u[KR];
              fetch(sg, half * k + eb + w * EW + q, u);
              product(u, w * EW + q);
            }
          __syncthreads();
          const int ne = min(EC, half - eb), units = nr * ne, ns = min(16, Vb - sg * 16);
          for (int t = threadIdx.x; t < ns * units; t += 256) {
            const int s = t / units, o = t - s * units, r = o / ne, e = o - r * ne;
            f[((size_t)bf[sg * 16 + s] * nrhs + r0 + r) * Ef + half * k + eb + e] =
                s_f[s * pitch + r * EC + e];
          }
          __syncthreads();
        }
    }
  }
}

template <typename R, int MT, bool VEC, bool FAST>
void project_launch(const mgc_aggregation* a, const cplx<R>* U, const cplx<R>* in, cplx<R>* out,
                    cplx<R>* part, int nrhs, int S, int kind, int point, hipStream_t s) {
  const int nchunk = (nrhs + TRC - 1) / TRC;
  const int sites_per = ((a->Vb + S - 1) / S + 3) / 4 * 4;
  const dim3 grid(a->Vc, nchunk, (a->Vb + sites_per - 1) / sites_per);
  // eight wavefronts per workgroup where four would leave the chip half empty,
  // fewer where the sites would leave some of them idle
  int waves = (size_t)grid.x * grid.y * grid.z < 2048 ? 8 : 4;
  while (waves > 1 && 4 * (waves - 1) >= sites_per) waves /= 2;
  const size_t sh = (size_t)waves / 2 * MT * 2 * 64 * sizeof(typename Mfma<R>::acc_t);
  auto k = k_project_mfma<R, MT, VEC, FAST, 2>;
  if constexpr (FAST && sizeof(R) == 4) {
    if (sites_per >= 64) k = k_project_mfma<R, MT, VEC, FAST, 6>;
  } else if constexpr (FAST && MT <= 2) {
    if (sites_per < 64 && grid.z > 1) k = k_project_mfma<R, MT, VEC, FAST, 1>;
  }
  k<<<grid, 64 * waves, sh, s>>>(U, in, out, a->blk_fine, a->nb, a->Vb, a->Ef, nrhs, a->blk, kind,
                                 point, sites_per, part);
  MGC_LAUNCH_CHECK();
  if (grid.z > 1) project_reduce<R>(part, out, a->Vc, nchunk, (int)grid.z, nrhs, a->nb, TRC, s);
}

template <typename R, int KP, bool VEC, bool FAST>
void promote_launch(const mgc_aggregation* a, const cplx<R>* U, const cplx<R>* in, cplx<R>* out,
                    int nrhs, hipStream_t s) {
  const int nchunk = (nrhs + TRC - 1) / TRC;
  // split a block's 16-site groups over workgroups until about 2048 of them
  // fill the chip
  const int groups = (a->Vb + 15) / 16;
  int S = (int)std::max<size_t>(1, 2048 / ((size_t)a->Vc * nchunk));
  S = std::min(S, groups);
  const int groups_per = (groups + S - 1) / S;
  const dim3 grid(a->Vc, nchunk, (groups + groups_per - 1) / groups_per);
  const size_t sh =
      (size_t)16 * promote_pitch<R>(std::min(nrhs, TRC), 4 * promote_ew(FAST)) * sizeof(cplx<R>);
  k_promote_mfma<R, KP, VEC, FAST><<<grid, 256, sh, s>>>(U, in, out, a->blk_fine, a->nb, a->Vb,
                                                         a->Ef, nrhs, groups_per);
  MGC_LAUNCH_CHECK();
}

// f(N, VEC, FAST as integral constants), N = n in 1 .. MAX
template <int MAX, typename F>
void with_shape(int n, bool vec, bool fast, F&& f) {
  if constexpr (MAX > 1)
    if (n < MAX) return with_shape<MAX - 1>(n, vec, fast, f);
  const std::integral_constant<int, MAX> N;
  if (vec && fast) f(N, std::true_type{}, std::true_type{});
  else if (vec) f(N, std::true_type{}, std::false_type{});
  else if (fast) f(N, std::false_type{}, std::true_type{});
  else f(N, std::false_type{}, std::false_type{});
}

bool aligned_fine(const mgc_aggregation* a, const void* fine) {
  return a->Ef == 12 && (uintptr_t)fine % 16 == 0;
}

}  // namespace

template <typename R>
void project_mfma(const mgc_aggregation* a, const cplx<R>* U, const cplx<R>* in, cplx<R>* out,
                  cplx<R>* part, int nrhs, int S, int kind, int point, hipStream_t s) {
  // VEC: each lane's MT entries are one run (and 16-byte aligned in FP32 when MT is even)
  const int mt = (a->nb + 15) / 16;
  with_shape<4>(mt, a->nb % mt == 0, aligned_fine(a, in), [&](auto MT, auto VEC, auto FAST) {
    if constexpr (MT() > 1 || VEC())  // one entry a lane is always a run
      project_launch<R, MT(), VEC(), FAST()>(a, U, in, out, part, nrhs, S, kind, point, s);
  });
}

template <typename R>
void promote_mfma(const mgc_aggregation* a, const cplx<R>* U, const cplx<R>* in, cplx<R>* out,
                  int nrhs, hipStream_t s) {
  // VEC: pairs of entries neither straddle nb nor (in FP32) a 16-byte boundary
  with_shape<8>((a->nb + 7) / 8, a->nb % 2 == 0, aligned_fine(a, out),
                [&](auto KP, auto VEC, auto FAST) {
                  promote_launch<R, KP(), VEC(), FAST()>(a, U, in, out, nrhs, s);
                });
}

template void project_mfma<float>(const mgc_aggregation*, const cplx<float>*, const cplx<float>*,
                                  cplx<float>*, cplx<float>*, int, int, int, int, hipStream_t);
template void project_mfma<double>(const mgc_aggregation*, const cplx<double>*,
                                   const cplx<double>*, cplx<double>*, cplx<double>*, int, int,
                                   int, int, hipStream_t);
template void promote_mfma<float>(const mgc_aggregation*, const cplx<float>*, const cplx<float>*,
                                  cplx<float>*, int, hipStream_t);
template void promote_mfma<double>(const mgc_aggregation*, const cplx<double>*,
                                   const cplx<double>*, cplx<double>*, int, hipStream_t);

}  // namespace mgc
