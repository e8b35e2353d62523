// Galerkin coarse-operator construction (CoarsenOperator) and the
// gamma5-hermiticity link reconstruction, FP64.
//
// Reference semantics:
//   include/CoarsenedMatrixBaseline.h:575-705   CoarsenOperator, inner/outer-mask form
//   include/CoarsenedMatrixUpstreamImprovedDirsave.h:835-932  backward links + self only,
//   include/CoarsenedMatrixUpstreamImprovedDirsave.h:999-1032 ConstructRemainingLinks
//   include/CoarsenedMatrixKernelsRework.h:141-167 shiftLinks (the converse direction)
//   include/CoarsenedMatrixRework.h:640-668     InvertSelfStencilPoint (done by set_links)
//
// With the chirally doubled basis v_{l*nb+c} = P_l u_c the links are
//   A_p(xc)[k*nb+c][l*nb+c'] = sum_{x in B(xc), outer_p} sum_{e in k} conj(u_c(x,e)) W_p^l(x,e,c')
//   W_p^l(x) = H_p(x) P_l u_{c'}(x + d_p),  H_p = -1/2 (1 - disp g_mu) (U_mu(x) | U_mu(x-mu)^dag)
// and the self link uses the block-restricted operator D_BB (diagonal term plus
// every hop that stays inside the block), which is the sum of the reference's
// Mdiag and inner-mask projections.
//
// One workgroup per (coarse site, point).  Per stage of SB fine sites the
// workgroup builds W for both chiralities in LDS (items (l, c', colour)), stages
// the block-panel rows of u, and every thread accumulates a TC x TC register
// tile of one chirality block (k, l) of the N x N link in FP64.
#include <algorithm>
#include <string>
#include <type_traits>

#include "aggregation.hpp"
#include "coarse_op.hpp"
#include "fine_op.hpp"

namespace mgc {

constexpr int CO_SB = 4;  // fine sites per stage

// Workgroup b -> (coarse site, point).  The points of one coarse site are
// consecutive in the dispatch sequence of one XCD (b % 8 is the XCD), so the
// workgroups that read one block panel run together on one L2; with a coarse
// volume that is not a multiple of 8 they are simply consecutive.
__device__ __forceinline__ void coarsen_work(int b, int np, int Vc, int& xc, int& pi) {
  if (Vc % 8 == 0) {
    const int i = b >> 3;
    xc = (i / np) * 8 + (b & 7);
    pi = i % np;
  } else {
    xc = b / np;
    pi = b % np;
  }
}

// Geometry of one (coarse site, point) work item of the construction.
struct CoGeom {
  const cplx<double>* basis;  // [xc][xb][e 12][nb] panels
  const cplx<double>* gauge;  // [mu][site][3][3]
  const cplx<double>* diag;   // [site][2][6][6]
  Lat4 fine, coarse, blk;
  int Vf, Vb;
  int xc, p, mu, disp, nsite;
  int cc[4], bs[4], fs[4], cs[4];

  __device__ CoGeom(const cplx<double>* b, const cplx<double>* g, const cplx<double>* d, Lat4 f,
                    Lat4 c, Lat4 bl, int vf, int vb, int x, int pt)
      : basis(b), gauge(g), diag(d), fine(f), coarse(c), blk(bl), Vf(vf), Vb(vb), xc(x), p(pt) {
    coarse.coords(xc, cc);
    bs[0] = 1; bs[1] = blk.L[0]; bs[2] = bs[1] * blk.L[1]; bs[3] = bs[2] * blk.L[2];
    fs[0] = 1; fs[1] = fine.L[0]; fs[2] = fs[1] * fine.L[1]; fs[3] = fs[2] * fine.L[2];
    cs[0] = 1; cs[1] = coarse.L[0]; cs[2] = cs[1] * coarse.L[1]; cs[3] = cs[2] * coarse.L[2];
    mu = p & 3;
    disp = p < 4 ? 1 : -1;
    // sites of this point: outer face of the block for p < 8, the whole block for p = 8
    // (blk.L[mu] by a select: a runtime index would put the geometry in scratch memory)
    const int Lmu = mu == 0 ? blk.L[0] : mu == 1 ? blk.L[1] : mu == 2 ? blk.L[2] : blk.L[3];
    nsite = (p == 8) ? Vb : Vb / Lmu;
  }
  // face site f: the coordinates other than mu run lexicographically over the
  // face, coordinate mu is the block's last (+mu) or first (-mu) layer
  __device__ int face_site(int f) const {
    if (p == 8) return f;
    int r = f, idx = 0, stride = 1;
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      int cd;
      if (d == mu) {
        cd = disp > 0 ? blk.L[d] - 1 : 0;
      } else {
        cd = r % blk.L[d];
        r /= blk.L[d];
      }
      idx += cd * stride;
      stride *= blk.L[d];
    }
    return idx;
  }
};

// One W item: W^lw(xb)[e, cp] for all 12 spin-colour elements, where
// W^l = H_p P_l u_cp for a hop (p < 8) and D_BB P_l u_cp (inner hops plus the
// diagonal) for p = 8.  The chirality lw is a runtime value, so that lanes
// of both chiralities run one instruction stream: ws[sl*3 + ci] holds spin
// 2 lw + sl (chirality lw), wo[k*3 + ci] spin 2 (1 - lw) + k, and the
// spin-dependent constants are chosen by selects between compile-time values
// (an index computed from lw would put the accumulators in scratch memory).
// The hops are taken HB at a time: the loads of the batch (link, and the
// neighbour's chirality-lw basis values) are issued before any is used.
// One hop per batch (HB = 1) measured fastest: with two the loads take ~230
// registers and one wavefront per SIMD; links staged in LDS for the
// wavefront's site cost a barrier per stage and ran slower.
template <int NB, int HB>
__device__ __forceinline__ void coarsen_w_lane(const CoGeom& g, const GammaTab& G, int xb, int lw,
                                               int cp, cplx<double> ws[6], cplx<double> wo[6]) {
  constexpr int ROW = 12 * NB;
  const int p = g.p;
#pragma unroll
  for (int e = 0; e < 6; ++e) {
    ws[e] = {0.0, 0.0};
    wo[e] = {0.0, 0.0};
  }
  // block and fine coordinates of this site
  int bc[4], x = 0;
  {
    int r = xb;
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      bc[d] = r % g.blk.L[d];
      r /= g.blk.L[d];
      x += (g.cc[d] * g.blk.L[d] + bc[d]) * g.fs[d];
    }
  }
  const int e0 = 6 * lw;  // first element of chirality lw
#pragma unroll
  for (int q0 = 0; q0 < 8; q0 += HB) {
    if (p != 8 && (p < q0 || p >= q0 + HB)) continue;  // uniform: a hop point uses one hop
    cplx<double> L[HB][9], B[HB][6];  // link U (row-major), basis (sl, colour)
    bool use[HB];
#pragma unroll
    for (int h = 0; h < HB; ++h) {
      const int q = q0 + h;
      const int qm = q & 3;
      const int disp = q < 4 ? 1 : -1;
      const bool inner = (unsigned)(bc[qm] + disp) < (unsigned)g.blk.L[qm];
      // self: inner hops only, by the reference's coordinate mask
      // (x_mu mod b != b-1 for +mu, != 0 for -mu)
      use[h] = p == 8 ? inner : q == p;
      if (!use[h]) continue;
      // fine neighbour y = x + disp*mu (periodic) and its panel row
      const int fq = g.cc[qm] * g.blk.L[qm] + bc[qm] + disp;
      const int y = x + disp * g.fs[qm] -
                    (fq < 0 ? -g.fine.L[qm] * g.fs[qm]
                            : fq >= g.fine.L[qm] ? g.fine.L[qm] * g.fs[qm] : 0);
      int ry;
      if (inner) {
        ry = g.xc * g.Vb + xb + disp * g.bs[qm];
      } else {
        const int cq = g.cc[qm] + disp;
        const int xn = g.xc + disp * g.cs[qm] -
                       (cq < 0 ? -g.coarse.L[qm] * g.cs[qm]
                               : cq >= g.coarse.L[qm] ? g.coarse.L[qm] * g.cs[qm] : 0);
        ry = xn * g.Vb + xb - disp * (g.blk.L[qm] - 1) * g.bs[qm];
      }
      const cplx<double>* U = g.gauge + ((size_t)qm * g.Vf + (q < 4 ? x : y)) * 9;
#pragma unroll
      for (int k = 0; k < 9; ++k) L[h][k] = U[k];
      const cplx<double>* uy = g.basis + (size_t)ry * ROW + (size_t)e0 * NB + cp;
#pragma unroll
      for (int k = 0; k < 6; ++k) B[h][k] = uy[k * NB];  // element e0 + k = 3 sl + j
    }
#pragma unroll
    for (int h = 0; h < HB; ++h) {
      if (!use[h]) continue;
      const int q = q0 + h;
      const int qm = q & 3;
      const double sg = q < 4 ? 1.0 : -1.0;
#pragma unroll
      for (int sl = 0; sl < 2; ++sl) {
        // gamma image of spin 2 lw + sl: spin s2 of the other chirality,
        // local index k = s2 - 2 (1 - lw), phase of s2
        const int s2a = G.col[qm][sl], s2b = G.col[qm][2 + sl];  // lw = 0, lw = 1
        const int ka = s2a - 2, kb = s2b;
        const cplx<double> pa = {(double)G.re[qm][s2a], (double)G.im[qm][s2a]};
        const cplx<double> pb = {(double)G.re[qm][s2b], (double)G.im[qm][s2b]};
        const cplx<double> ph = lw ? pb : pa;
        const int kimg = lw ? kb : ka;
#pragma unroll
        for (int ci = 0; ci < 3; ++ci) {
          cplx<double> chi = {0.0, 0.0};
#pragma unroll
          for (int j = 0; j < 3; ++j) {
            // row ci of U (q < 4) or of U^dag (q >= 4)
            const cplx<double> l = q < 4 ? L[h][ci * 3 + j]
                                         : cplx<double>{L[h][j * 3 + ci].re, -L[h][j * 3 + ci].im};
            cmac(chi, l, B[h][sl * 3 + j]);
          }
          // same-chirality part: -1/2 chi
          ws[sl * 3 + ci].re -= 0.5 * chi.re;
          ws[sl * 3 + ci].im -= 0.5 * chi.im;
          // gamma image: + sg/2 * phase(s2) * chi at spin s2
          const cplx<double> t = cmul(ph, chi);
          const cplx<double> v = {0.5 * sg * t.re, 0.5 * sg * t.im};
          if (ka == kb) {  // the same local spin for both chiralities (compile time)
            wo[ka * 3 + ci].re += v.re;
            wo[ka * 3 + ci].im += v.im;
          } else {
            const double f0 = kimg == 0 ? 1.0 : 0.0;
            wo[ci].re += f0 * v.re;
            wo[ci].im += f0 * v.im;
            wo[3 + ci].re += (1.0 - f0) * v.re;
            wo[3 + ci].im += (1.0 - f0) * v.im;
          }
        }
      }
    }
  }
  if (p == 8) {  // diagonal (mass + clover) term, block-diagonal in chirality
    const cplx<double>* D = g.diag + ((size_t)x * 2 + lw) * 36;
    const cplx<double>* ux = g.basis + ((size_t)g.xc * g.Vb + xb) * ROW + (size_t)e0 * NB + cp;
    cplx<double> v[6];
#pragma unroll
    for (int b = 0; b < 6; ++b) v[b] = ux[b * NB];
#pragma unroll
    for (int r = 0; r < 6; ++r) {
      cplx<double> a = {0.0, 0.0};
#pragma unroll
      for (int b = 0; b < 6; ++b) cmac(a, D[r * 6 + b], v[b]);
      ws[r].re += a.re;
      ws[r].im += a.im;
    }
  }
}

// FP64 vector form: one workgroup per (coarse site, point).  Per stage of
// CO_SB fine sites the workgroup builds W for both chiralities in LDS (items
// (l, c', colour)), stages the block-panel rows of u, and every thread
// accumulates a TC x TC register tile of one chirality block (k, l) of the
// N x N link.
template <int NB, int TC>
__global__ __launch_bounds__(4 * (NB / TC) * (NB / TC)) void k_coarsen(
    const cplx<double>* __restrict__ basis, const cplx<double>* __restrict__ gauge,
    const cplx<double>* __restrict__ diag, Lat4 fine, Lat4 coarse, Lat4 blk, int Vf, int Vb,
    const int* __restrict__ plist, int np, int Vc, cplx<double>* __restrict__ links) {
  constexpr int NT1 = NB / TC;
  constexpr int THREADS = 4 * NT1 * NT1;
  constexpr int ROW = 12 * NB;  // complex per panel row group (one fine site)
  __shared__ cplx<double> sU[CO_SB][12][NB];
  __shared__ cplx<double> sW[CO_SB][2][12][NB];
  const GammaTab G = gamma_table();

  int xc, pi;
  coarsen_work((int)blockIdx.x, np, Vc, xc, pi);
  const CoGeom g(basis, gauge, diag, fine, coarse, blk, Vf, Vb, xc, plist[pi]);
  const int tid = threadIdx.x;
  const int kl = tid / (NT1 * NT1);
  const int k = kl >> 1, l = kl & 1;
  const int rem = tid % (NT1 * NT1);
  const int cb = rem / NT1, pb = rem % NT1;

  cplx<double> acc[TC][TC];
#pragma unroll
  for (int i = 0; i < TC; ++i)
#pragma unroll
    for (int j = 0; j < TC; ++j) acc[i][j] = {0.0, 0.0};

  for (int s0 = 0; s0 < g.nsite; s0 += CO_SB) {
    // ---- stage u rows of the SB sites
    for (int idx = tid; idx < CO_SB * ROW; idx += THREADS) {
      const int s = idx / ROW, r = idx - s * ROW;
      // past the face end: load block site 0 (in bounds) and stage zero
      const bool ok = s0 + s < g.nsite;
      const int xb = ok ? g.face_site(s0 + s) : 0;
      const cplx<double> v = basis[((size_t)xc * Vb + xb) * ROW + r];
      (&sU[s][0][0])[r] = ok ? v : cplx<double>{0.0, 0.0};
    }
    // ---- W items (s, l', c'), all 12 elements each
    for (int it = tid; it < CO_SB * 2 * NB; it += THREADS) {
      const int s = it / (2 * NB);
      const int r = it - s * 2 * NB;
      const int lw = r / NB, cp = r - lw * NB;
      cplx<double> ws[6], wo[6];
      if (s0 + s < g.nsite) {
        coarsen_w_lane<NB, 1>(g, G, g.face_site(s0 + s), lw, cp, ws, wo);
      } else {
#pragma unroll
        for (int e = 0; e < 6; ++e) ws[e] = wo[e] = {0.0, 0.0};
      }
#pragma unroll
      for (int e = 0; e < 6; ++e) {
        sW[s][lw][6 * lw + e][cp] = ws[e];
        sW[s][lw][6 - 6 * lw + e][cp] = wo[e];
      }
    }
    __syncthreads();
    // ---- accumulate the (k, l) block: acc[c][c'] += sum_{e in k} conj(u(e,c)) W^l(e,c')
#pragma unroll
    for (int s = 0; s < CO_SB; ++s)
#pragma unroll
      for (int e6 = 0; e6 < 6; ++e6) {
        const int e = 6 * k + e6;
        cplx<double> a[TC], b[TC];
#pragma unroll
        for (int i = 0; i < TC; ++i) a[i] = sU[s][e][cb * TC + i];
#pragma unroll
        for (int j = 0; j < TC; ++j) b[j] = sW[s][l][e][pb * TC + j];
#pragma unroll
        for (int i = 0; i < TC; ++i)
#pragma unroll
          for (int j = 0; j < TC; ++j) cmac_conj(acc[i][j], a[i], b[j]);
      }
    __syncthreads();
  }
  // ---- write A_p(xc) rows k*NB + c, columns l*NB + c'
  constexpr int N = 2 * NB;
  cplx<double>* Ap = links + ((size_t)g.p * Vc + xc) * N * N;
#pragma unroll
  for (int i = 0; i < TC; ++i)
#pragma unroll
    for (int j = 0; j < TC; ++j)
      Ap[(size_t)(k * NB + cb * TC + i) * N + l * NB + pb * TC + j] = acc[i][j];
}

// FP64 MFMA form (v_mfma_f64_16x16x4_f64), one workgroup of four wavefronts
// per (coarse site, point), wavefront w owning the chirality block
// (k, l) = (w / 2, w % 2) of the N x N link.  Each block is the complex
// product C = sum_{s, e in k} conj(u(s,e))^T W^l(s,e), run as one real GEMM
// with the complex index folded into K (the scheme of the multi-rhs stencil):
//   A'[c][2m+t]   = (Re u, -Im u)(m, c)           for t = 0, 1 (m = (s, e))
//   B'[2m+t][2c'+v] = v = 0: (Re w, -Im w),  v = 1: (Im w, Re w)
// so that C'[c][2c'+v] = (Re, Im) C[c][c'].  Rows and columns past NB are zero
// padding of the 16 x 16 tiles and are never stored.  The staged u and W are
// kept as separate real and imaginary planes in LDS, so every lane's operand
// is one 8-byte read.
// MFMA 16x16x4 f64 lane layout: A[i = l%16][k = l/16], B[k = l/16][j = l%16],
// D[i = 4r + l/16][j = l%16] for result r < 4 (rows interleaved, unlike the
// FP32 16x16x4 form's 4(l/16) + r).
//
// What bounds it: the products (412 GFLOP at 32^4, 4^4 blocks, nb 32: 5.7 ms at
// the FP64 matrix rate) and the gathers of W: the self point reads 43 GB from beyond
// L2, over six times the panel, at 4.7 TB/s, the faces 12 GB (55 GB in all; 51 in one
// kernel with two workgroups a CU).  The workgroups of a CU overlap the two, so a stage is sized for three of them (38 KB of LDS: two sites at nb >
// 16, four below; up to 168 registers a lane).  For the registers a W item is
// one spin of one chirality (two lanes per column), the link, the same for a
// whole wavefront, is read into scalar registers, and the faces and the self
// point are kernels of their own.  Faces 4.7 ms (62% of the matrix rate), self
// 9.3 ms; one kernel at two workgroups a CU and a lane per column: 18.2 ms.
// All of a stage's loads in flight one stage ahead, at two workgroups: 16.5 ms.
constexpr int co_sites(int nb) { return nb > 16 ? 2 : 4; }  // fine sites per stage
typedef double doublex4 __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(4))) double* scalar_f64_ptr;

// the value of the neighbouring lane l ^ 1
__device__ __forceinline__ double swap_pair(double x) {
  union { double d; int i[2]; } a, b;
  a.d = x;
#pragma unroll
  for (int k = 0; k < 2; ++k)  // quad permutation (1, 0, 3, 2)
    b.i[k] = __builtin_amdgcn_mov_dpp(a.i[k], 0xB1, 0xF, 0xF, true);
  return b.d;
}

// One hop of one W item: lane (cp, sl) of chirality lw adds its spin's part of
// H_q P_lw u_cp to ws (spin 2 lw + sl) and the gamma image to wo (the spin of
// the other chirality that g_mu maps it to).  U: the link, B: the lane's three
// colours of the neighbour; bit mu of neg: the image spin's phase is negative.
template <int Q>
__device__ __forceinline__ void coarsen_hop(unsigned neg, scalar_f64_ptr U,
                                            const cplx<double> B[3], cplx<double> ws[3],
                                            cplx<double> wo[3]) {
  constexpr int mu = Q & 3;
  // half the phase of the image spin, +-1 (y, t) or +-i (x, z): bit mu of neg
  const double f =
      __hiloint2double((int)(0x3fe00000u ^ (((neg >> mu) ^ (Q < 4 ? 0u : 1u)) << 31)), 0);
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    cplx<double> chi = {0.0, 0.0};
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      // row i of U (forward) or of U^dag (backward)
      const int k = Q < 4 ? i * 3 + j : j * 3 + i;
      const cplx<double> l = {U[2 * k], Q < 4 ? U[2 * k + 1] : -U[2 * k + 1]};
      cmac(chi, l, B[j]);
    }
    ws[i].re -= 0.5 * chi.re;
    ws[i].im -= 0.5 * chi.im;
    if (mu % 2) {
      wo[i].re += f * chi.re;
      wo[i].im += f * chi.im;
    } else {
      wo[i].re -= f * chi.im;
      wo[i].im += f * chi.re;
    }
  }
}

template <int NB, bool SELF>
__global__ __launch_bounds__(256, 3) void k_coarsen_mfma(
    const cplx<double>* __restrict__ basis, const cplx<double>* __restrict__ gauge,
    const cplx<double>* __restrict__ diag, Lat4 fine, Lat4 coarse, Lat4 blk, int Vf, int Vb,
    const int* __restrict__ plist, int np, int Vc, cplx<double>* __restrict__ links) {
  constexpr int SB = co_sites(NB);
  constexpr int MT = (NB + 15) / 16;   // m-tiles (rows c)
  constexpr int NTL = (NB + 7) / 8;    // n-tiles (columns 2c'+v)
  constexpr int NBP = NB + 1;          // LDS row pitch (doubles) against bank conflicts
  constexpr int ROW = 12 * NB;
  constexpr int LPS = 256 / SB;        // lanes that build one site
  constexpr int NU = (ROW + LPS - 1) / LPS;  // staged u entries per lane
  constexpr int PL = SB * 12 * NBP;    // one plane of u; a plane of W is two
  static_assert(NB <= 32, "lanes of a W item");
  __shared__ double smem[6 * PL];
  double* const sUr = smem;            // u[site][e][c], with -Im u in sUi
  double* const sUi = smem + PL;
  double* const sWr = smem + 2 * PL;   // W[site][l][e][c']
  double* const sWi = smem + 4 * PL;

  int xc, pi;
  coarsen_work((int)blockIdx.x, np, Vc, xc, pi);
  // the same for all lanes, though divisions computed them in vector registers
  xc = __builtin_amdgcn_readfirstlane(xc);
  pi = __builtin_amdgcn_readfirstlane(pi);
  CoGeom g(basis, gauge, diag, fine, coarse, blk, Vf, Vb, xc, SELF ? 8 : plist[pi]);
#pragma unroll
  for (int d = 0; d < 4; ++d) g.cc[d] = __builtin_amdgcn_readfirstlane(g.cc[d]);
  g.nsite = __builtin_amdgcn_readfirstlane(g.nsite);
  const int p = SELF ? 8 : g.p;
  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63;
  const int kb = w >> 1, lb = w & 1;  // chirality block of this wavefront
  const int lk = l >> 4;              // k index of this lane within a k-step
  const int t = lk & 1;               // real (0) or imaginary (1) slot of K
  // A operand: row c = mt*16 + l%16, from the plane of t
  const double* aplane = t ? sUi : sUr;
  // B operand: column n = nt*16 + l%16, c' = n/2, v = n%2: plane Re for
  // t == v, else Im, negated for (t, v) = (1, 0)
  const int v = l & 1;
  const double* bplane = (t ^ v) ? sWi : sWr;
  const double bsign = (t == 1 && v == 0) ? -1.0 : 1.0;

  // W item of this lane: site ss of the stage (uniform over the wavefront),
  // chirality lw, spin 2 lw + sl, column cp
  const int ss = SB == 2 ? w >> 1 : w;
  const int lw = SB == 2 ? w & 1 : l >> 5;
  const int sl = l & 1;
  const int cp_raw = (SB == 2 ? l : l & 31) >> 1;
  const bool col = cp_raw < NB;
  const int cp = col ? cp_raw : NB - 1;
  const int e0 = 6 * lw + 3 * sl;  // first of this lane's elements
  const int li = SB == 2 ? tid & 127 : l;  // lane among those of the site

  unsigned neg = 0;  // bit mu: sign of the phase of this lane's image spin under g_mu
  {
    const GammaTab G = gamma_table();
#pragma unroll
    for (int mu = 0; mu < 4; ++mu)
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int s2 = G.col[mu][s];
        if (2 * lw + sl == s && G.re[mu][s2] + G.im[mu][s2] < 0) neg |= 1u << mu;
      }
  }

  doublex4 acc[MT][NTL];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NTL; ++nt) acc[mt][nt] = {0.0, 0.0, 0.0, 0.0};

  // block coordinates of this wavefront's site, advanced over the point's
  // sites (lexicographic over the block, or over the face without coordinate
  // mu, which stays at the block's last (+mu) or first (-mu) layer)
  int bc[4];
#pragma unroll
  for (int d = 0; d < 4; ++d) bc[d] = !SELF && d == g.mu && g.disp > 0 ? g.blk.L[d] - 1 : 0;
  auto advance = [&](int n) __attribute__((always_inline)) {
    for (int i = 0; i < n; ++i) {
      int carry = 1;
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        const bool fixed = !SELF && d == g.mu;
        const int c = bc[d] + (fixed ? 0 : carry);
        const bool wrap = !fixed && c == g.blk.L[d];
        carry = fixed ? carry : wrap ? 1 : 0;
        bc[d] = wrap ? 0 : c;
      }
    }
  };
  advance(ss);

  for (int s0 = 0; s0 < g.nsite; s0 += SB) {
    cplx<double> ur[NU], ws[3], wo[3];
#pragma unroll
    for (int e = 0; e < 3; ++e) ws[e] = wo[e] = {0.0, 0.0};
    // (opaque here, or the eight phases would be kept in registers over the loop)
    asm volatile("" : "+v"(neg));
    const bool ok = s0 + ss < g.nsite;  // uniform over the wavefront
    if (ok) {
      int xb = 0, x = 0;
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        xb += bc[d] * g.bs[d];
        x += (g.cc[d] * g.blk.L[d] + bc[d]) * g.fs[d];
      }
      xb = __builtin_amdgcn_readfirstlane(xb);
      x = __builtin_amdgcn_readfirstlane(x);
      const cplx<double>* ub = basis + ((size_t)xc * Vb + xb) * ROW;
#pragma unroll
      for (int q = 0; q < NU; ++q) ur[q] = ub[min(li + q * LPS, ROW - 1)];
      auto hop = [&](auto qc) __attribute__((always_inline)) {
        constexpr int q = decltype(qc)::value, qm = q & 3, disp = q < 4 ? 1 : -1;
        const bool inner = (unsigned)(bc[qm] + disp) < (unsigned)g.blk.L[qm];
        // self: inner hops, by the reference's coordinate mask (x_mu mod b !=
        // b-1 for +mu, != 0 for -mu)
        if (!(SELF ? inner : q == p)) return;  // uniform over the wavefront
        // fine neighbour y = x + disp*mu (periodic) and its panel row
        const int fq = g.cc[qm] * g.blk.L[qm] + bc[qm] + disp;
        const int y = x + disp * g.fs[qm] -
                      (fq < 0 ? -g.fine.L[qm] * g.fs[qm]
                              : fq >= g.fine.L[qm] ? g.fine.L[qm] * g.fs[qm] : 0);
        int ry;
        if (inner) {
          ry = xc * Vb + xb + disp * g.bs[qm];
        } else {
          const int cq = g.cc[qm] + disp;
          const int xn = xc + disp * g.cs[qm] -
                         (cq < 0 ? -g.coarse.L[qm] * g.cs[qm]
                                 : cq >= g.coarse.L[qm] ? g.coarse.L[qm] * g.cs[qm] : 0);
          ry = xn * Vb + xb - disp * (g.blk.L[qm] - 1) * g.bs[qm];
        }
        const int lsite = __builtin_amdgcn_readfirstlane(q < 4 ? x : y);
        const scalar_f64_ptr U =
            (scalar_f64_ptr)(uintptr_t)(gauge + ((size_t)qm * Vf + lsite) * 9);
        const cplx<double>* uy = basis + (size_t)__builtin_amdgcn_readfirstlane(ry) * ROW +
                                 (size_t)e0 * NB + cp;
        cplx<double> B[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) B[k] = uy[k * NB];
        coarsen_hop<q>(neg, U, B, ws, wo);
      };
      // g_x and g_y exchange the spins of a chirality: their images belong to
      // the other lane of the pair
      hop(std::integral_constant<int, 0>{});
      hop(std::integral_constant<int, 1>{});
      hop(std::integral_constant<int, 4>{});
      hop(std::integral_constant<int, 5>{});
#pragma unroll
      for (int e = 0; e < 3; ++e) wo[e] = {swap_pair(wo[e].re), swap_pair(wo[e].im)};
      hop(std::integral_constant<int, 2>{});
      hop(std::integral_constant<int, 3>{});
      hop(std::integral_constant<int, 6>{});
      hop(std::integral_constant<int, 7>{});
      if constexpr (SELF) {  // diagonal (mass + clover) term, block-diagonal in chirality
        const cplx<double>* D = diag + ((size_t)x * 2 + lw) * 36 + 18 * sl;
        const cplx<double>* ux = ub + (size_t)(6 * lw) * NB + cp;
#pragma unroll
        for (int b = 0; b < 6; ++b) {
          const cplx<double> vb = ux[b * NB];
#pragma unroll
          for (int r = 0; r < 3; ++r) cmac(ws[r], D[r * 6 + b], vb);
        }
      }
    } else {
#pragma unroll
      for (int q = 0; q < NU; ++q) ur[q] = {0.0, 0.0};
    }
    advance(SB);
    __syncthreads();  // the previous stage's products have been read
#pragma unroll
    for (int q = 0; q < NU; ++q) {
      const int r = li + q * LPS, e = r / NB, c = r - e * NB;
      if (ROW % LPS == 0 || r < ROW) {
        sUr[(ss * 12 + e) * NBP + c] = ur[q].re;
        sUi[(ss * 12 + e) * NBP + c] = -ur[q].im;
      }
    }
    if (col) {
      const int base = (ss * 2 + lw) * 12 * NBP + cp;
#pragma unroll
      for (int e = 0; e < 3; ++e) {
        sWr[base + (e0 + e) * NBP] = ws[e].re;
        sWi[base + (e0 + e) * NBP] = ws[e].im;
        const int eo = 6 - 6 * lw + 3 * sl + e;
        sWr[base + eo * NBP] = wo[e].re;
        sWi[base + eo * NBP] = wo[e].im;
      }
    }
    __syncthreads();
    // ---- the block's GEMM: per site three k-steps of two elements each
#pragma unroll 1
    for (int s = 0; s < SB; ++s)
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        const int e = 6 * kb + 2 * q + (lk >> 1);  // element of this lane's K slot
        double a[MT], b[NTL];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          const int c = mt * 16 + (l & 15);
          a[mt] = (NB % 16 == 0 || c < NB) ? aplane[(s * 12 + e) * NBP + c] : 0.0;
        }
#pragma unroll
        for (int nt = 0; nt < NTL; ++nt) {
          const int cq = (nt * 16 + (l & 15)) >> 1;
          b[nt] = (NB % 8 == 0 || cq < NB)
                      ? bsign * bplane[((s * 2 + lb) * 12 + e) * NBP + cq]
                      : 0.0;
        }
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int nt = 0; nt < NTL; ++nt)
            acc[mt][nt] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[mt], b[nt], acc[mt][nt], 0, 0, 0);
      }
  }
  // ---- write A_p(xc) rows k*NB + c, columns l*NB + c' (component v)
  constexpr int N = 2 * NB;
  double* Ap = reinterpret_cast<double*>(links + ((size_t)p * Vc + xc) * N * N);
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NTL; ++nt) {
      const int cq = (nt * 16 + (l & 15)) >> 1;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int c = mt * 16 + 4 * r + lk;
        if ((NB % 16 == 0 || c < NB) && (NB % 8 == 0 || cq < NB))
          Ap[((size_t)(kb * NB + c) * N + lb * NB + cq) * 2 + v] = acc[mt][nt][r];
      }
    }
}

// A_want(x) = sigma o adj(A_have(x + disp_want * mu)), FLAT layout, in place:
// a workgroup at a time per 32 x 32 tile of a link, transposed through LDS so that
// both sides run along rows.  Bound by HBM (8^4, N = 64: 2.1 GB).
constexpr int RT = 32;
__global__ __launch_bounds__(256) void k_reconstruct(cplx<double>* __restrict__ links, Lat4 lat,
                                                     int N, int nt, size_t tiles, int disp_have,
                                                     const int* __restrict__ nbr) {
  __shared__ cplx<double> sA[RT][RT + 1];
  const int V = lat.volume(), nb = N / 2;
  const int i = threadIdx.x % RT, j0 = threadIdx.x / RT;
  for (size_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
    const size_t m = tile / (nt * nt);  // link (mu, x)
    const int rem = (int)(tile - m * (nt * nt)), tr = rem / nt, tc = rem - tr * nt;
    const int mu = (int)(m / V), x = (int)(m - (size_t)mu * V);
    const int ph = disp_have > 0 ? mu : mu + 4;  // point we have
    const int pw = disp_have > 0 ? mu + 4 : mu;  // point we want
    // neighbour in direction disp_want = -disp_have: the want-point's own neighbour
    const int y = nbr[(size_t)x * 8 + pw];
    const cplx<double>* have = links + ((size_t)ph * V + y) * N * N;
    cplx<double>* want = links + ((size_t)pw * V + x) * N * N;
    for (int j = j0; j < RT; j += 256 / RT) {  // element (c, r) of the link we have
      const int c = tc * RT + j, r = tr * RT + i;
      if (c < N && r < N) sA[j][i] = have[(size_t)c * N + r];
    }
    __syncthreads();
    for (int j = j0; j < RT; j += 256 / RT) {
      const int r = tr * RT + j, c = tc * RT + i;
      if (r >= N || c >= N) continue;
      cplx<double> a = sA[i][j];
      a.im = -a.im;
      if ((r / nb + c / nb) & 1) { a.re = -a.re; a.im = -a.im; }
      want[(size_t)r * N + c] = a;
    }
    __syncthreads();
  }
}

// The same for whole_matrices, `mats` links at a time (as k_export_links_whole).
__global__ __launch_bounds__(256) void k_reconstruct_whole(cplx<double>* __restrict__ links,
                                                           Lat4 lat, int N, int mats,
                                                           int disp_have,
                                                           const int* __restrict__ nbr) {
  extern __shared__ unsigned char smem_raw[];
  cplx<double>* sA = reinterpret_cast<cplx<double>*>(smem_raw);  // [link][r][c], rows N + 1 apart
  const unsigned V = lat.volume(), nb = N / 2, N2 = N * N;
  for (size_t m0 = (size_t)blockIdx.x * mats; m0 < (size_t)4 * V; m0 += (size_t)gridDim.x * mats) {
    const size_t left = (size_t)4 * V - m0;
    const unsigned n = (unsigned)(left < (size_t)mats ? left : mats) * N2;
    for (unsigned i = threadIdx.x; i < n; i += 256) {
      const unsigned q = i / N2;
      const size_t m = m0 + q;  // (mu, x)
      const unsigned mu = (unsigned)(m / V), x = (unsigned)(m - (size_t)mu * V);
      const unsigned ph = disp_have > 0 ? mu : mu + 4, pw = disp_have > 0 ? mu + 4 : mu;
      const unsigned y = nbr[(size_t)x * 8 + pw];
      sA[i + i / N] = links[((size_t)ph * V + y) * N2 + (i - q * N2)];
    }
    __syncthreads();
    for (unsigned i = threadIdx.x; i < n; i += 256) {
      const unsigned q = i / N2, rc = i - q * N2, r = rc / N, c = rc - r * N;
      const size_t m = m0 + q;
      const unsigned mu = (unsigned)(m / V), x = (unsigned)(m - (size_t)mu * V);
      cplx<double> a = sA[(q * N + c) * (N + 1) + r];
      a.im = -a.im;
      if ((r / nb + c / nb) & 1) { a.re = -a.re; a.im = -a.im; }
      links[((size_t)(disp_have > 0 ? mu + 4 : mu) * V + x) * N2 + rc] = a;
    }
    __syncthreads();
  }
}

template <int NB, int TC>
static void launch_coarsen_t(const mgc_aggregation* agg, const mgc_fine_op* fop, const int* plist,
                             int np, cplx<double>* links, hipStream_t s) {
  constexpr int THREADS = 4 * (NB / TC) * (NB / TC);
  k_coarsen<NB, TC><<<agg->Vc * np, THREADS, 0, s>>>(agg->basis64, fop->gauge64, fop->diag64,
                                                      agg->fine, agg->coarse, agg->blk, agg->Vf,
                                                      agg->Vb, plist, np, agg->Vc, links);
  MGC_LAUNCH_CHECK();
}

template <int NB>
static void launch_coarsen_mfma_t(const mgc_aggregation* agg, const mgc_fine_op* fop,
                                  const int* plist, int np, cplx<double>* links, hipStream_t s) {
  // the faces (all points of the list but the last, the self point), then the self point
  k_coarsen_mfma<NB, false><<<agg->Vc * (np - 1), 256, 0, s>>>(
      agg->basis64, fop->gauge64, fop->diag64, agg->fine, agg->coarse, agg->blk, agg->Vf, agg->Vb,
      plist, np - 1, agg->Vc, links);
  MGC_LAUNCH_CHECK();
  k_coarsen_mfma<NB, true><<<agg->Vc, 256, 0, s>>>(
      agg->basis64, fop->gauge64, fop->diag64, agg->fine, agg->coarse, agg->blk, agg->Vf, agg->Vb,
      plist, 1, agg->Vc, links);
  MGC_LAUNCH_CHECK();
}

// build kernel: 0 = FP64 vector form, 1 = FP64 MFMA form; -1 = the default (MFMA)
static int g_coarsen_variant = -1;

static void launch_coarsen(const mgc_aggregation* agg, const mgc_fine_op* fop, const int* plist,
                           int np, cplx<double>* links, hipStream_t s) {
  if (g_coarsen_variant != 0) {
    switch (agg->nb) {
#define CASE(n)                                                    \
  case n:                                                          \
    launch_coarsen_mfma_t<n>(agg, fop, plist, np, links, s);       \
    return;
      CASE(1) CASE(2) CASE(3) CASE(4) CASE(5) CASE(6) CASE(7) CASE(8) CASE(9) CASE(10) CASE(11)
      CASE(12) CASE(13) CASE(14) CASE(15) CASE(16) CASE(17) CASE(18) CASE(19) CASE(20) CASE(21)
      CASE(22) CASE(23) CASE(24) CASE(25) CASE(26) CASE(27) CASE(28) CASE(29) CASE(30) CASE(31)
      CASE(32)
#undef CASE
    }
    throw Error(MGC_ERR_SHAPE, "CoarsenOperator supports nb from 1 to 32");
  }
  switch (agg->nb) {
    case 2: launch_coarsen_t<2, 1>(agg, fop, plist, np, links, s); return;
    case 4: launch_coarsen_t<4, 1>(agg, fop, plist, np, links, s); return;
    case 8: launch_coarsen_t<8, 2>(agg, fop, plist, np, links, s); return;
    case 12: launch_coarsen_t<12, 3>(agg, fop, plist, np, links, s); return;
    case 16: launch_coarsen_t<16, 2>(agg, fop, plist, np, links, s); return;
    case 24: launch_coarsen_t<24, 3>(agg, fop, plist, np, links, s); return;
    case 32: launch_coarsen_t<32, 4>(agg, fop, plist, np, links, s); return;
    case 6: launch_coarsen_t<6, 1>(agg, fop, plist, np, links, s); return;
    case 10: launch_coarsen_t<10, 2>(agg, fop, plist, np, links, s); return;
    case 14: launch_coarsen_t<14, 2>(agg, fop, plist, np, links, s); return;
    case 18: launch_coarsen_t<18, 2>(agg, fop, plist, np, links, s); return;
    case 20: launch_coarsen_t<20, 2>(agg, fop, plist, np, links, s); return;
    case 22: launch_coarsen_t<22, 2>(agg, fop, plist, np, links, s); return;
    case 26: launch_coarsen_t<26, 2>(agg, fop, plist, np, links, s); return;
    case 28: launch_coarsen_t<28, 4>(agg, fop, plist, np, links, s); return;
    case 30: launch_coarsen_t<30, 3>(agg, fop, plist, np, links, s); return;
  }
  throw Error(MGC_ERR_SHAPE,
              "the vector form of CoarsenOperator supports nb = 2 and every even nb from 4 to 32");
}

static void reconstruct(cplx<double>* links, const mgc_coarse_op* cop, int disp_have,
                        hipStream_t s) {
  const int N = cop->N;
  const size_t mats = (size_t)4 * cop->V;
  if (whole_matrices(N)) {
    const int per = std::max(1, 1024 / (N * N));
    k_reconstruct_whole<<<tile_grid((mats + per - 1) / per), 256,
                          (size_t)per * N * (N + 1) * sizeof(cplx<double>), s>>>(
        links, cop->lat, N, per, disp_have, cop->nbr_full);
  } else {
    const int nt = (N + RT - 1) / RT;
    const size_t tiles = mats * nt * nt;
    k_reconstruct<<<tile_grid(tiles), 256, 0, s>>>(links, cop->lat, N, nt, tiles, disp_have,
                                                   cop->nbr_full);
  }
  MGC_LAUNCH_CHECK();
}

static void set_links_or_throw(mgc_coarse_op* cop, const void* links, int invert, hipStream_t s) {
  const int st = mgc_coarse_op_set_links(cop, MGC_LAYOUT_FLAT, links, invert, (void*)s);
  if (st != MGC_OK) throw Error(st, mgc_last_error());
}

// links[p][xc][j][n0 + r] (=, or += when accumulate) proj[xc][r][j], r < nr
__global__ void k_scatter_columns(cplx<double>* __restrict__ links,
                                  const cplx<double>* __restrict__ proj, int Vc, int N, int p,
                                  int n0, int nr, int accumulate) {
  const size_t t = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (t >= (size_t)Vc * nr * N) return;
  const int j = (int)(t % N);
  const size_t q = t / N;
  const int r = (int)(q % nr);
  const size_t xc = q / nr;
  cplx<double>& dst = links[(((size_t)p * Vc + xc) * N + j) * N + n0 + r];
  const cplx<double> v = proj[t];
  if (accumulate) dst = cadd(dst, v);
  else dst = v;
}

static void check_call(int st) {
  if (st != MGC_OK) throw Error(st, mgc_last_error());
}

// Galerkin product of an operator given point by point, in the inner/outer-
// mask form of include/CoarsenedMatrixBaseline.h:609-675: for a batch of nr
// doubled basis columns v_n, W_p = (stencil point p of the operator) v_n for
// p = 0..8 (OpDir / OpDiag), then A_p(xc)[j][n] = sum over the outer sites of
// p of <v_j, W_p> and A_8(xc)[j][n] = sum over the inner sites of every p and
// all sites of W_8, FP64.  apply(p, in, out, nr) acts on FP64 fields
// [site][nr][Ef].  DIRSAVE skips the forward points and rebuilds their links
// by gamma5-hermiticity.
template <typename Apply>
static void coarsen_by_points(mgc_coarse_op* cop2, mgc_aggregation* agg, int mode, int batch,
                              Apply&& apply, hipStream_t s) {
  const int N2 = cop2->N, Vc2 = cop2->V, Vf = agg->Vf, Ef = agg->Ef;
  batch = std::max(1, std::min(batch, N2));
  DevBuf<cplx<double>> links((size_t)9 * Vc2 * N2 * N2), phi((size_t)Vf * batch * Ef),
      mphi((size_t)Vf * batch * Ef), proj((size_t)Vc2 * batch * N2);
  fill_zero(links.p, (size_t)9 * Vc2 * N2 * N2 * sizeof(cplx<double>), s);
  for (int n0 = 0; n0 < N2; n0 += batch) {
    const int nr = std::min(batch, N2 - n0);
    const unsigned g = (unsigned)(((size_t)Vc2 * nr * N2 + 255) / 256);
    agg_extract_doubled(agg, n0, nr, phi.p, s);
    for (int p = 0; p < 9; ++p) {
      apply(p, phi.p, mphi.p, nr);
      // outer sites: link p (DIRSAVE rebuilds the forward links instead)
      if (p < 8 && !(mode == MGC_COARSEN_DIRSAVE && p < 4)) {
        agg_transfer(agg, mphi.p, proj.p, MGC_F64, nr, true, 2, p, s);
        k_scatter_columns<<<g, 256, 0, s>>>(links.p, proj.p, Vc2, N2, p, n0, nr, 0);
        MGC_LAUNCH_CHECK();
      }
      // inner sites of every hop, and every site of the diagonal: the self link
      agg_transfer(agg, mphi.p, proj.p, MGC_F64, nr, true, 1, p, s);
      k_scatter_columns<<<g, 256, 0, s>>>(links.p, proj.p, Vc2, N2, 8, n0, nr, 1);
      MGC_LAUNCH_CHECK();
    }
  }
  if (mode == MGC_COARSEN_DIRSAVE) reconstruct(links.p, cop2, -1, s);
  set_links_or_throw(cop2, links.p, 1, s);
  MGC_HIP(hipStreamSynchronize(s));  // the buffers are freed on return
}

// CoarsenOperator of a coarse operator: one basis column at a time (the
// single-rhs coarse apply)
static void coarsen_coarse(mgc_coarse_op* cop2, mgc_coarse_op* cop1, mgc_aggregation* agg,
                           int mode, hipStream_t s) {
  coarsen_by_points(cop2, agg, mode, 1,
                    [&](int p, const void* in, void* out, int) {
                      if (p == 8) check_call(mgc_coarse_op_Mdiag(cop1, in, out, (void*)s));
                      else
                        check_call(mgc_coarse_op_Mdir(cop1, in, out, p & 3, p < 4 ? 1 : -1,
                                                      (void*)s));
                    },
                    s);
}

// CoarsenOperator of a caller's fine operator, through its point callback
static void coarsen_linop(mgc_coarse_op* cop, const mgc_fine_linop& lop, mgc_aggregation* agg,
                          int mode, hipStream_t s) {
  const int batch = std::max(1, std::min(lop.max_nrhs, 16));
  coarsen_by_points(cop, agg, mode, batch,
                    [&](int p, const void* in, void* out, int nr) {
                      const int st = lop.apply(lop.ctx, p, MGC_F64, in, out, nr, (void*)s);
                      MGC_CHECK(st == MGC_OK, st < 0 ? st : MGC_ERR_ARG,
                                "the fine operator callback failed (point " +
                                    std::to_string(p) + ", status " + std::to_string(st) + ")");
                    },
                    s);
}

}  // namespace mgc

using namespace mgc;

extern "C" {

int mgc_coarsen_operator(mgc_coarse_op* cop, mgc_fine_op* fop, mgc_aggregation* agg, int mode,
                         void* stream) {
  return guarded([&] {
    MGC_CHECK(cop && fop && agg, MGC_ERR_ARG, "null handle");
    MGC_CHECK(mode == MGC_COARSEN_FULL || mode == MGC_COARSEN_DIRSAVE, MGC_ERR_ARG, "bad mode");
    MGC_CHECK(agg->basis_set, MGC_ERR_STATE, "aggregation basis not set");
    MGC_CHECK(fop->gauge_set, MGC_ERR_STATE, "fine gauge field not set");
    MGC_CHECK(agg->Ef == 12, MGC_ERR_SHAPE, "the aggregation must act on Dirac (12-element) sites");
    for (int d = 0; d < 4; ++d) {
      MGC_CHECK(fop->lat.L[d] == agg->fine.L[d], MGC_ERR_SHAPE, "fine lattices differ");
      MGC_CHECK(cop->lat.L[d] == agg->coarse.L[d], MGC_ERR_SHAPE, "coarse lattices differ");
    }
    MGC_CHECK(cop->N == 2 * agg->nb, MGC_ERR_SHAPE, "coarse nbasis must be 2 * nb");
    hipStream_t s = as_stream(stream);
    const int N = cop->N, Vc = cop->V;
    cplx<double>* links = nullptr;
    int* plist = nullptr;
    MGC_HIP(hipMalloc(&links, (size_t)9 * Vc * N * N * sizeof(cplx<double>)));
    MGC_HIP(hipMalloc(&plist, 9 * sizeof(int)));
    try {
      const int full[9] = {0, 1, 2, 3, 4, 5, 6, 7, 8};
      const int dsave[5] = {4, 5, 6, 7, 8};
      const int* pl = mode == MGC_COARSEN_FULL ? full : dsave;
      const int np = mode == MGC_COARSEN_FULL ? 9 : 5;
      MGC_HIP(hipMemcpyAsync(plist, pl, np * sizeof(int), hipMemcpyHostToDevice, s));
      launch_coarsen(agg, fop, plist, np, links, s);
      if (mode == MGC_COARSEN_DIRSAVE) reconstruct(links, cop, -1, s);
      set_links_or_throw(cop, links, 1, s);
    } catch (...) {
      (void)hipStreamSynchronize(s);
      (void)hipFree(links);
      (void)hipFree(plist);
      throw;
    }
    MGC_HIP(hipStreamSynchronize(s));
    MGC_HIP(hipFree(links));
    MGC_HIP(hipFree(plist));
  });
}

int mgc_coarsen_set_variant(int variant) {
  return guarded([&] {
    MGC_CHECK(variant >= -1 && variant <= 1, MGC_ERR_ARG, "unknown CoarsenOperator variant");
    g_coarsen_variant = variant;
  });
}

int mgc_coarsen_operator_linop(mgc_coarse_op* cop, const mgc_fine_linop* lop,
                               mgc_aggregation* agg, int mode, void* stream) {
  return guarded([&] {
    MGC_CHECK(cop && lop && agg && lop->apply, MGC_ERR_ARG, "null handle or callback");
    MGC_CHECK(mode == MGC_COARSEN_FULL || mode == MGC_COARSEN_DIRSAVE, MGC_ERR_ARG, "bad mode");
    MGC_CHECK(mode == MGC_COARSEN_FULL || lop->gamma5_hermitian, MGC_ERR_ARG,
              "DIRSAVE rebuilds forward links by gamma5-hermiticity: the operator must be "
              "gamma5-hermitian");
    MGC_CHECK(lop->precisions & (1 << MGC_F64), MGC_ERR_PRECISION,
              "CoarsenOperator needs an operator that applies in F64");
    MGC_CHECK(lop->max_nrhs >= 1, MGC_ERR_ARG, "max_nrhs < 1");
    MGC_CHECK(agg->basis_set, MGC_ERR_STATE, "aggregation basis not set");
    MGC_CHECK(agg->Ef == 12, MGC_ERR_SHAPE, "the aggregation must act on Dirac (12-element) sites");
    for (int d = 0; d < 4; ++d) {
      MGC_CHECK(lop->dims[d] == agg->fine.L[d], MGC_ERR_SHAPE, "fine lattices differ");
      MGC_CHECK(cop->lat.L[d] == agg->coarse.L[d], MGC_ERR_SHAPE, "coarse lattices differ");
    }
    MGC_CHECK(cop->N == 2 * agg->nb, MGC_ERR_SHAPE, "coarse nbasis must be 2 * nb");
    coarsen_linop(cop, *lop, agg, mode, as_stream(stream));
  });
}

int mgc_coarsen_coarse_operator(mgc_coarse_op* cop2, mgc_coarse_op* cop1, mgc_aggregation* agg,
                                int mode, void* stream) {
  return guarded([&] {
    MGC_CHECK(cop2 && cop1 && agg, MGC_ERR_ARG, "null handle");
    MGC_CHECK(mode == MGC_COARSEN_FULL || mode == MGC_COARSEN_DIRSAVE, MGC_ERR_ARG, "bad mode");
    MGC_CHECK(agg->basis_set, MGC_ERR_STATE, "aggregation basis not set");
    MGC_CHECK(cop1->links_set, MGC_ERR_STATE, "level operator links not set");
    MGC_CHECK(cop1->prec == MGC_F64, MGC_ERR_PRECISION,
              "the operator being coarsened must be an F64 operator");
    MGC_CHECK(agg->Ef == cop1->N, MGC_ERR_SHAPE, "aggregation site elements must equal nbasis");
    for (int d = 0; d < 4; ++d) {
      MGC_CHECK(cop1->lat.L[d] == agg->fine.L[d], MGC_ERR_SHAPE, "fine lattices differ");
      MGC_CHECK(cop2->lat.L[d] == agg->coarse.L[d], MGC_ERR_SHAPE, "coarse lattices differ");
    }
    MGC_CHECK(cop2->N == 2 * agg->nb, MGC_ERR_SHAPE, "coarse nbasis must be 2 * nb");
    coarsen_coarse(cop2, cop1, agg, mode, as_stream(stream));
  });
}

int mgc_coarse_op_construct_remaining_links(mgc_coarse_op* cop, int disp_have, void* stream) {
  return guarded([&] {
    MGC_CHECK(cop, MGC_ERR_ARG, "null handle");
    MGC_CHECK(cop->links_set, MGC_ERR_STATE, "links not set");
    MGC_CHECK(disp_have == 1 || disp_have == -1, MGC_ERR_ARG, "disp_have must be +1 or -1");
    hipStream_t s = as_stream(stream);
    const int N = cop->N, V = cop->V;
    cplx<double>* links = nullptr;
    MGC_HIP(hipMalloc(&links, (size_t)9 * V * N * N * sizeof(cplx<double>)));
    const int st = mgc_coarse_op_get_links(cop, MGC_LAYOUT_FLAT, links, stream);
    if (st != MGC_OK) {
      (void)hipFree(links);
      throw Error(st, mgc_last_error());
    }
    try {
      reconstruct(links, cop, disp_have, s);
      set_links_or_throw(cop, links, cop->inv_set ? 1 : 0, s);
    } catch (...) {
      (void)hipStreamSynchronize(s);
      (void)hipFree(links);
      throw;
    }
    MGC_HIP(hipStreamSynchronize(s));
    MGC_HIP(hipFree(links));
  });
}

}  // extern "C"
