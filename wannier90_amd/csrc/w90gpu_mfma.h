// Matrix-core (MFMA) kernels of libw90gpu: the M rotation
// M(k,b) <- E_k^+ M(k,b) E_{k+b} as two complex products on
// v_mfma_*_16x16x4 tiles (FP64 for the plain path, FP32 with FP32
// accumulation for the mixed bulk phase), and the products of the
// retraction (k_step_panel up to num_wann 96).
//
// num_wann <= 16 (k_rotate_w16): one 16 x 16 tile per block, one wavefront
// per neighbour b.  num_wann 17-48 in FP64 (k_rot_panel): a wavefront per 16
// columns, no barriers.  num_wann 17-64 else (k_rot_fused): a workgroup computes both
// products of one (k, b) block as one GT x GT tile (GT = 32, 48 or 64), T
// kept in LDS between them.  num_wann 65-256 (k_rot_gemm): each product is
// its own launch over up to 4 x 4 tiles of 64 (or 8 x 8 of 32), T through
// a scratch buffer.  Four wavefronts hold a quadrant of a tile each (three
// hold a 48 x 16 strip of a 48 tile), as 16 x 16 fragments; a complex
// fragment product is three real MFMA products per K step (Cfrag, Gauss's
// form).  K runs in chunks staged in LDS with
// coalesced global loads (planar re/im, padded rows), the next chunk
// loaded into registers while the current one is multiplied.  Fragments
// wholly outside num_wann are skipped.  The second product's epilogue
// forms the omega partial sums of the tile (Im ln M_nn, |M_nn|^2,
// sum |M_mn|^2, off-diagonal sum).
//
// MFMA 16x16x4 lane layout (measured on gfx950): lane l holds A[l%16][l/16]
// and B[l/16][l%16]; element i of its result is D[r][l%16] with
// r = 4*(l/16) + i for f32 and r = l/16 + 4*i for f64.
//
// Reference: src/wannierise.F90 internal_new_u_and_m :1737-1748 (the two
// utility_zgemm calls per (k,b)), wann_omega :2034-2090, :2214-2258.
#pragma once

#include "w90gpu_kernels.h"

#ifndef W90_GK
#define W90_GK 16  // K chunk staged in LDS
#endif

typedef double w90_d4 __attribute__((ext_vector_type(4)));
typedef float w90_f4 __attribute__((ext_vector_type(4)));

template <class R>
struct Mfma;
template <>
struct Mfma<double> {
  typedef w90_d4 acc;
  static __device__ __forceinline__ acc mma(double a, double b, acc c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  // row of result element i in lane group lk = l/16
  static __device__ __forceinline__ int row(int lk, int i) { return lk + 4 * i; }
};
template <>
struct Mfma<float> {
  typedef w90_f4 acc;
  static __device__ __forceinline__ acc mma(float a, float b, acc c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lk, int i) { return 4 * lk + i; }
};

// Complex 16 x 16 fragment product accumulated with three real MFMA
// products per K step (Gauss): P1 += ar br, P2 += ai bi,
// P3 += (ar + ai)(br + bi); the product is Re = P1 - P2,
// Im = P3 - P1 - P2.  Three MFMA instructions instead of four.
template <class R>
struct Cfrag {
  typename Mfma<R>::acc p1, p2, p3;
  __device__ __forceinline__ void zero() {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      p1[i] = 0;
      p2[i] = 0;
      p3[i] = 0;
    }
  }
  __device__ __forceinline__ void mma(R ar, R ai, R br, R bi) {
    p1 = Mfma<R>::mma(ar, br, p1);
    p2 = Mfma<R>::mma(ai, bi, p2);
    p3 = Mfma<R>::mma(ar + ai, br + bi, p3);
  }
  __device__ __forceinline__ R re(int i) const { return p1[i] - p2[i]; }
  __device__ __forceinline__ R im(int i) const { return p3[i] - p1[i] - p2[i]; }
};

template <class T2>
struct Real;
template <>
struct Real<cplx> {
  typedef double type;
};
template <>
struct Real<float2> {
  typedef float type;
};


// One GT x GT output tile (row0, col0) of one stage of the rotation of
// block (k, b) by the workgroup (256 threads): operands and scratch as in
// k_rot_gemm, LDS passed in.
template <class T2, int STAGE, int GT>
__device__ __forceinline__ void rot_gemm_tile(const Prob& p, int k, int b, int mate, int tile, int row0, int col0,
                                              int mode, int cur, typename Real<T2>::type (*As)[W90_GK][GT + 1],
                                              typename Real<T2>::type (*Bs)[W90_GK][GT + 1], double* red) {
  constexpr int FR = GT / 32;  // fragments per wavefront along rows and columns
  typedef typename Real<T2>::type R;
  const int nw = p.nw, nn = p.nn;
  const size_t kb = (size_t)k * nn + b;
  const size_t nw2 = p.nw2;
  const int dst = dst_buf(mode, cur);
  T2* Tm = reinterpret_cast<T2*>(p.Tm) + kb * nw2;
  const cplx* Ek = p.E + (size_t)k * nw2;
  const cplx* Ekb = p.E + (size_t)p.nnl[kb] * nw2;
  const T2* src = rot_src<T2>(p, mode, cur) + kb * nw2;

  const int tid = threadIdx.x;
  const int w = tid >> 6, lane = tid & 63;
  const int wr = (w >> 1) * (GT / 2), wc = (w & 1) * (GT / 2);
  const int lr = lane & 15, lk = lane >> 4;
  bool fv_r[FR], fv_c[FR];
#pragma unroll
  for (int f = 0; f < FR; ++f) {
    fv_r[f] = row0 + wr + f * 16 < nw;
    fv_c[f] = col0 + wc + f * 16 < nw;
  }
  Cfrag<R> C[FR][FR];
#pragma unroll
  for (int fi = 0; fi < FR; ++fi)
#pragma unroll
    for (int fj = 0; fj < FR; ++fj) C[fi][fj].zero();

  // K chunks are software-pipelined: the operands of chunk kk + GK are
  // loaded into registers before the products of chunk kk, and stored to
  // LDS after them.  Thread slot e = tid + 256 u of a chunk.
  constexpr int NE = W90_GK * GT / 256;
  static_assert(NE * 256 == W90_GK * GT, "whole chunk per thread slot");
  cplx pa[NE], pb[NE];
  auto load_chunk = [&](int kk) {
#pragma unroll
    for (int u = 0; u < NE; ++u) {
      const int e = tid + 256 * u;
      cplx v = c_make(0.0, 0.0);
      if (STAGE == 1) {
        // A = E_k^+: A[i][l] = conj(E_k[l + i nw]); threads run along l
        const int gi = row0 + e / W90_GK, gl = kk + e % W90_GK;
        if (gi < nw && gl < nw) v = Ek[gl + (size_t)gi * nw];
        v.y = -v.y;
      } else {
        // A = T: A[i][l] = T[i + l nw]; threads run along i
        const int gi = row0 + e % GT, gl = kk + e / GT;
        if (gi < nw && gl < nw) v = c_wide(Tm[gi + (size_t)gl * nw]);
      }
      pa[u] = v;
      // B[l][j] = Bsrc[l + j nw]; threads run along l
      const int gl = kk + e % W90_GK, gj = col0 + e / W90_GK;
      cplx w2 = c_make(0.0, 0.0);
      if (gl < nw && gj < nw) w2 = (STAGE == 1) ? c_wide(src[gl + (size_t)gj * nw]) : Ekb[gl + (size_t)gj * nw];
      pb[u] = w2;
    }
  };
  load_chunk(0);
  for (int kk = 0; kk < nw; kk += W90_GK) {
    __syncthreads();
#pragma unroll
    for (int u = 0; u < NE; ++u) {
      const int e = tid + 256 * u;
      const int la = (STAGE == 1) ? e % W90_GK : e / GT, ia = (STAGE == 1) ? e / W90_GK : e % GT;
      As[0][la][ia] = (R)pa[u].x;
      As[1][la][ia] = (R)pa[u].y;
      const int lb = e % W90_GK, jb = e / W90_GK;
      Bs[0][lb][jb] = (R)pb[u].x;
      Bs[1][lb][jb] = (R)pb[u].y;
    }
    if (kk + W90_GK < nw) load_chunk(kk + W90_GK);
    __syncthreads();
#pragma unroll
    for (int ks = 0; ks < W90_GK; ks += 4) {
      R ar[FR], ai[FR], br[FR], bi[FR];
#pragma unroll
      for (int f = 0; f < FR; ++f) {
        ar[f] = As[0][ks + lk][wr + f * 16 + lr];
        ai[f] = As[1][ks + lk][wr + f * 16 + lr];
        br[f] = Bs[0][ks + lk][wc + f * 16 + lr];
        bi[f] = Bs[1][ks + lk][wc + f * 16 + lr];
      }
#pragma unroll
      for (int fi = 0; fi < FR; ++fi) {
        if (!fv_r[fi]) continue;
#pragma unroll
        for (int fj = 0; fj < FR; ++fj) {
          if (!fv_c[fj]) continue;
          C[fi][fj].mma(ar[fi], ai[fi], br[fj], bi[fj]);
        }
      }
    }
  }

  double od = 0.0, all = 0.0;
  T2* out = (STAGE == 1) ? Tm : mbuf<T2>(p, dst) + kb * nw2;
  T2* outm = mbuf<T2>(p, dst) + (mate >= 0 ? (size_t)mate * nw2 : 0);
#pragma unroll
  for (int fi = 0; fi < FR; ++fi)
#pragma unroll
    for (int fj = 0; fj < FR; ++fj)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = row0 + wr + fi * 16 + Mfma<R>::row(lk, i);
        const int c = col0 + wc + fj * 16 + lr;
        if (r < nw && c < nw) {
          T2 v;
          v.x = C[fi][fj].re(i);
          v.y = C[fi][fj].im(i);
          out[r + (size_t)c * nw] = v;
          if (STAGE == 2) {
            if (mate >= 0) outm[c + (size_t)r * nw] = c_conj(v);
            const cplx vw = c_wide(v);
            const double a2 = c_abs2(vw);
            all += a2;
            if (r != c) {
              od += a2;
            } else {
              const double l = atan2(vw.y, vw.x);
              p.ln[dst][kb * nw + r] = l;
              p.d2[kb * nw + r] = a2;
              if (mate >= 0) {
                p.ln[dst][(size_t)mate * nw + r] = -l;
                p.d2[(size_t)mate * nw + r] = a2;
              }
            }
          }
        }
      }
  if (STAGE == 2) {
    block_sum2(od, all, red);
    if (tid == 0) {
      p.part_od[kb * p.npan + tile] = od;
      p.part_all[kb * p.npan + tile] = all;
      if (mate >= 0) {  // tile (J, I) of the adjoint block
        const int nt1 = (nw + GT - 1) / GT;
        const size_t q = (size_t)mate * p.npan + tile / nt1 + (tile % nt1) * nt1;
        p.part_od[q] = od;
        p.part_all[q] = all;
      }
    }
  }
}

// Two-stage rotation, one launch per stage: workgroup (item, b, tile).
template <class T2, int STAGE, int GT>
__global__ void __launch_bounds__(256, 2) k_rot_gemm(const Prob* probs, const Item* items, int nitems, int mode) {
  typedef typename Real<T2>::type R;
  if (blockIdx.x >= (unsigned)nitems) return;
  const Item it = items[blockIdx.x];
  const Prob& p = probs[it.prob];
  const State* st = p.st;
  const int cur = gate_cur(st, mode);
  if (cur < 0) return;
  const int nw = p.nw, nn = p.nn;
  const int nt1 = (nw + GT - 1) / GT;
  const int ntl = nt1 * nt1;
  const int by = blockIdx.y;
  if (by >= nn * ntl) return;
  const int tile = by % ntl;
  int mate;
  const int b = rot_slot<T2>(p, it.k, by / ntl, &mate);
  if (b < 0) return;
  const int row0 = (tile % nt1) * GT, col0 = (tile / nt1) * GT;
  __shared__ R As[2][W90_GK][GT + 1];  // [re/im][k][row]
  __shared__ R Bs[2][W90_GK][GT + 1];  // [re/im][k][col]
  __shared__ double red[256];
  rot_gemm_tile<T2, STAGE, GT>(p, it.k, b, mate, tile, row0, col0, mode, cur, As, Bs, red);
}

// K chunk of the second product of k_rot_fused (T held in LDS).
#define W90_GK2 8

// Wavefront layout of k_rot_fused by tile edge GT: WR x WC wavefronts, each
// holding (GT / 16 WR) x (GT / 16 WC) fragments of 16 x 16.  A 64 or 32
// tile is split in quadrants over four wavefronts; a 48 tile (num_wann up
// to 48: 3 x 3 fragments, which four wavefronts cannot share evenly) in
// three column strips of 48 x 16 over three wavefronts.
template <int GT>
struct FusedWaves {
  static constexpr int WR = GT == 48 ? 1 : 2, WC = GT == 48 ? 3 : 2;
  static constexpr int NT = 64 * WR * WC;
  static constexpr int FRR = GT / (16 * WR), FRC = GT / (16 * WC);
  static constexpr int MINB = GT == 48 ? 3 : 2;  // workgroups per CU the registers allow
};

// LDS elements (storage-precision reals) of k_rot_fused: the staging of the
// first product (A and B chunks) and, after it, T with the B chunks of the
// second product share one buffer.
template <class R, int GT>
__host__ __device__ constexpr int rot_fused_elems() {
  return (4 * W90_GK * (GT + 1)) > (2 * GT * (GT + 1) + 2 * W90_GK2 * (GT + 1))
             ? 4 * W90_GK * (GT + 1)
             : 2 * GT * (GT + 1) + 2 * W90_GK2 * (GT + 1);
}

// Both products of the rotation of block (k, b) by one workgroup, when one
// GT x GT tile covers the block (num_wann <= GT).  T = E_k^+ src is formed
// as in k_rot_gemm stage 1, then written from the accumulators into LDS
// (planar, k-major: T[i][l] at Ts[p][l][i], zero outside num_wann) over the
// staging buffers of the first product; R = T E_{k+b} takes its A
// fragments from there and its B operand in chunks of W90_GK2 rows of
// E_{k+b}, loaded one chunk ahead.  The epilogue is that of stage 2.
template <class T2, int GT>
__device__ __forceinline__ void rot_fused_tile(const Prob& p, int k, int b, int mate, int mode, int cur,
                                               typename Real<T2>::type* lds, double* red) {
  typedef FusedWaves<GT> WL;
  constexpr int FRR = WL::FRR, FRC = WL::FRC, FRM = FRR > FRC ? FRR : FRC, NT = WL::NT;
  constexpr int LDA = GT + 1;
  typedef typename Real<T2>::type R;
  const int nw = p.nw, nn = p.nn;
  const size_t kb = (size_t)k * nn + b;
  const size_t nw2 = p.nw2;
  const int dst = dst_buf(mode, cur);
  const cplx* Ek = p.E + (size_t)k * nw2;
  const cplx* Ekb = p.E + (size_t)p.nnl[kb] * nw2;
  const T2* src = rot_src<T2>(p, mode, cur) + kb * nw2;
  T2* out = mbuf<T2>(p, dst) + kb * nw2;
  T2* outm = mbuf<T2>(p, dst) + (mate >= 0 ? (size_t)mate * nw2 : 0);
  double* lnd = p.ln[dst] + kb * nw;
  double* d2d = p.d2 + kb * nw;
  double* pod = p.part_od + kb * p.npan;
  double* pall = p.part_all + kb * p.npan;
  R* As = lds;                     // [2][GK][LDA]   first product
  R* Bs = lds + 2 * W90_GK * LDA;  // [2][GK][LDA]   first product
  R* Ts = lds;                     // [2][GT][LDA]   T, k-major
  R* B2 = lds + 2 * GT * LDA;      // [2][GK2][LDA]  second product

  const int tid = threadIdx.x;
  const int w = tid >> 6, lane = tid & 63;
  const int wr = (w / WL::WC) * (GT / WL::WR), wc = (w % WL::WC) * (GT / WL::WC);
  const int lr = lane & 15, lk = lane >> 4;
  Cfrag<R> C[FRR][FRC];
#pragma unroll
  for (int fi = 0; fi < FRR; ++fi)
#pragma unroll
    for (int fj = 0; fj < FRC; ++fj) C[fi][fj].zero();

  // ---- T = E_k^+ src, K chunks of GK loaded one chunk ahead
  constexpr int NE = W90_GK * GT / NT;
  static_assert(NE * NT == W90_GK * GT, "whole chunk per thread slot");
  cplx pa[NE], pb[NE];
  auto load1 = [&](int kk) {
#pragma unroll
    for (int u = 0; u < NE; ++u) {
      const int e = tid + NT * u;
      const int l = e % W90_GK, x = e / W90_GK;
      const int gl = kk + l;
      cplx v = c_make(0.0, 0.0), v2 = c_make(0.0, 0.0);
      if (x < nw && gl < nw) {
        v = Ek[gl + (size_t)x * nw];  // A[x][l] = conj(E_k[l + x nw])
        v2 = c_wide(src[gl + (size_t)x * nw]);  // B[l][x] = src[l + x nw]
      }
      v.y = -v.y;
      pa[u] = v;
      pb[u] = v2;
    }
  };
  load1(0);
  for (int kk = 0; kk < nw; kk += W90_GK) {
    __syncthreads();
#pragma unroll
    for (int u = 0; u < NE; ++u) {
      const int e = tid + NT * u;
      const int l = e % W90_GK, x = e / W90_GK;
      As[(0 * W90_GK + l) * LDA + x] = (R)pa[u].x;
      As[(1 * W90_GK + l) * LDA + x] = (R)pa[u].y;
      Bs[(0 * W90_GK + l) * LDA + x] = (R)pb[u].x;
      Bs[(1 * W90_GK + l) * LDA + x] = (R)pb[u].y;
    }
    if (kk + W90_GK < nw) load1(kk + W90_GK);
    __syncthreads();
#pragma unroll
    for (int ks = 0; ks < W90_GK; ks += 4) {
      R ar[FRR], ai[FRR], br[FRC], bi[FRC];
#pragma unroll
      for (int f = 0; f < FRM; ++f) {
        if (f < FRR) {
          ar[f] = As[(0 * W90_GK + ks + lk) * LDA + wr + f * 16 + lr];
          ai[f] = As[(1 * W90_GK + ks + lk) * LDA + wr + f * 16 + lr];
        }
        if (f < FRC) {
          br[f] = Bs[(0 * W90_GK + ks + lk) * LDA + wc + f * 16 + lr];
          bi[f] = Bs[(1 * W90_GK + ks + lk) * LDA + wc + f * 16 + lr];
        }
      }
#pragma unroll
      for (int fi = 0; fi < FRR; ++fi)
#pragma unroll
        for (int fj = 0; fj < FRC; ++fj) C[fi][fj].mma(ar[fi], ai[fi], br[fj], bi[fj]);
    }
  }
  // every wavefront is done with the staging buffers before T overwrites them
  __syncthreads();
#pragma unroll
  for (int fi = 0; fi < FRR; ++fi)
#pragma unroll
    for (int fj = 0; fj < FRC; ++fj)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = wr + fi * 16 + Mfma<R>::row(lk, i);
        const int c = wc + fj * 16 + lr;
        Ts[(0 * GT + c) * LDA + r] = C[fi][fj].re(i);
        Ts[(1 * GT + c) * LDA + r] = C[fi][fj].im(i);
      }
#pragma unroll
  for (int fi = 0; fi < FRR; ++fi)
#pragma unroll
    for (int fj = 0; fj < FRC; ++fj) C[fi][fj].zero();

  // ---- R = T E_{k+b}, K chunks of GK2 rows of E_{k+b} loaded one ahead
  constexpr int NE2 = W90_GK2 * GT / NT;
  static_assert(NE2 * NT == W90_GK2 * GT, "whole chunk per thread slot");
  cplx pc[NE2];
  auto load2 = [&](int kk) {
#pragma unroll
    for (int u = 0; u < NE2; ++u) {
      const int e = tid + NT * u;
      const int l = e % W90_GK2, j = e / W90_GK2;
      const int gl = kk + l;
      cplx v = c_make(0.0, 0.0);
      if (j < nw && gl < nw) v = Ekb[gl + (size_t)j * nw];
      pc[u] = v;
    }
  };
  load2(0);
  for (int kk = 0; kk < nw; kk += W90_GK2) {
    __syncthreads();
#pragma unroll
    for (int u = 0; u < NE2; ++u) {
      const int e = tid + NT * u;
      const int l = e % W90_GK2, j = e / W90_GK2;
      B2[(0 * W90_GK2 + l) * LDA + j] = (R)pc[u].x;
      B2[(1 * W90_GK2 + l) * LDA + j] = (R)pc[u].y;
    }
    if (kk + W90_GK2 < nw) load2(kk + W90_GK2);
    __syncthreads();
#pragma unroll
    for (int ks = 0; ks < W90_GK2; ks += 4) {
      R ar[FRR], ai[FRR], br[FRC], bi[FRC];
#pragma unroll
      for (int f = 0; f < FRM; ++f) {
        if (f < FRR) {
          ar[f] = Ts[(0 * GT + kk + ks + lk) * LDA + wr + f * 16 + lr];
          ai[f] = Ts[(1 * GT + kk + ks + lk) * LDA + wr + f * 16 + lr];
        }
        if (f < FRC) {
          br[f] = B2[(0 * W90_GK2 + ks + lk) * LDA + wc + f * 16 + lr];
          bi[f] = B2[(1 * W90_GK2 + ks + lk) * LDA + wc + f * 16 + lr];
        }
      }
#pragma unroll
      for (int fi = 0; fi < FRR; ++fi)
#pragma unroll
        for (int fj = 0; fj < FRC; ++fj) C[fi][fj].mma(ar[fi], ai[fi], br[fj], bi[fj]);
    }
  }

  // ---- epilogue: R to the other buffer, diagonal phases and tile sums
  double od = 0.0, all = 0.0;
#pragma unroll
  for (int fi = 0; fi < FRR; ++fi)
#pragma unroll
    for (int fj = 0; fj < FRC; ++fj)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = wr + fi * 16 + Mfma<R>::row(lk, i);
        const int c = wc + fj * 16 + lr;
        if (r < nw && c < nw) {
          T2 v;
          v.x = C[fi][fj].re(i);
          v.y = C[fi][fj].im(i);
          out[r + (size_t)c * nw] = v;
          if (mate >= 0) outm[c + (size_t)r * nw] = c_conj(v);
          const cplx vw = c_wide(v);
          const double a2 = c_abs2(vw);
          all += a2;
          if (r != c) {
            od += a2;
          } else {
            const double l = atan2(vw.y, vw.x);
            lnd[r] = l;
            d2d[r] = a2;
            if (mate >= 0) {
              p.ln[dst][(size_t)mate * nw + r] = -l;
              p.d2[(size_t)mate * nw + r] = a2;
            }
          }
        }
      }
  block_sum2(od, all, red);
  if (tid == 0) {
    pod[0] = od;
    pall[0] = all;
    if (mate >= 0) {
      p.part_od[(size_t)mate * p.npan] = od;
      p.part_all[(size_t)mate * p.npan] = all;
    }
  }
}

// The rotation for num_wann <= GT (one tile per block) in FP32, and in FP64 above
// W90_ROT_PANEL_MAX bands, both products in one workgroup per (item, b) with T in LDS (rot_fused_tile).  Workgroups
// are placed XCD-aware: a one-dimensional grid of 8 * ceil(nitems / 8) *
// nnmax workgroups, where workgroup w runs on XCD w % 8 (round-robin
// dispatch) and takes item 8 t + w % 8 and neighbour b with
// (t, b) = divmod(w / 8, nnmax): the nnmax workgroups of one k run back to
// back on one XCD and share E_k through its L2.
template <class T2, int GT>
__global__ void __launch_bounds__(FusedWaves<GT>::NT, FusedWaves<GT>::MINB) k_rot_fused(const Prob* probs, const Item* items, int nitems,
                                                                     int nnmax, int mode) {
  typedef typename Real<T2>::type R;
  const int w = blockIdx.x;
  const int r = w >> 3;
  const int item = 8 * (r / nnmax) + (w & 7);
  if (item >= nitems) return;
  const Item it = items[item];
  const Prob& p = probs[it.prob];
  const State* st = p.st;
  if (sizeof(T2) == sizeof(cplx) && p.nw <= W90_ROT_PANEL_MAX) return;  // k_rot_panel's
  const int cur = gate_cur(st, mode);
  if (cur < 0) return;
  int mate;
  const int b = rot_slot<T2>(p, it.k, r % nnmax, &mate);
  if (b < 0) return;
  __shared__ R lds[rot_fused_elems<R, GT>()];
  __shared__ double red[256];
  rot_fused_tile<T2, GT>(p, it.k, b, mate, mode, cur, lds, red);
}

// ------------------------------------------------ rotation, direct operands

// K steps of global operands in flight per wavefront in k_rot_direct.
#ifndef W90_RD_PF
#define W90_RD_PF 4
#endif

// The rotation of block (k, b) for num_wann <= 64 by one workgroup, with
// every global operand loaded straight into MFMA fragments, coalesced:
// the products are taken in the order P = M(k,b) E_{k+b}, then
// R = E_k^+ P, so that M (column-major) is the A operand, whose fragment
// rows are consecutive in memory, and E enters through its transpose ET
// (rows of E consecutive: the B operand of the first product, the
// conjugated A operand of the second).  Operands of W90_RD_PF K steps are
// in flight ahead of the MFMA products; P goes to LDS once (planar,
// row-major), the only barrier between the products; R goes through the
// same LDS for column-major stores of whole blocks.  Rows and columns
// outside num_wann are read at clamped (valid) addresses and zeroed.
// Epilogue as k_rot_fused: Im ln M_nn, |M_nn|^2, sum |M_mn|^2 and the
// off-diagonal sum of the block.
template <class T2>
__device__ __forceinline__ void rot_direct_tile(const Prob& p, int k, int b, int mate, int mode, int cur,
                                                typename Real<T2>::type* Ps, double* red) {
  constexpr int GT = 64, LD = GT + 1, FR = 2, PF = W90_RD_PF;
  typedef typename Real<T2>::type R;
  const int nw = p.nw, nn = p.nn;
  const size_t kb = (size_t)k * nn + b;
  const size_t nw2 = p.nw2;
  const int dst = dst_buf(mode, cur);
  const cplx* ETk = p.ET + (size_t)k * nw2;
  const cplx* ETkb = p.ET + (size_t)p.nnl[kb] * nw2;
  const T2* src = rot_src<T2>(p, mode, cur) + kb * nw2;
  T2* out = mbuf<T2>(p, dst) + kb * nw2;
  T2* outm = mbuf<T2>(p, dst) + (mate >= 0 ? (size_t)mate * nw2 : 0);
  double* lnd = p.ln[dst] + kb * nw;
  double* d2d = p.d2 + kb * nw;

  const int tid = threadIdx.x;
  const int w = tid >> 6, lane = tid & 63;
  const int wr = (w >> 1) * 32, wc = (w & 1) * 32;
  const int lr = lane & 15, lk = lane >> 4;
  const int nks = (nw + 3) >> 2;
  // this lane's A rows and B columns, clamped into the block
  int ri[FR], ci[FR];
  bool rv[FR], cv[FR];
#pragma unroll
  for (int f = 0; f < FR; ++f) {
    const int r = wr + 16 * f + lr, c = wc + 16 * f + lr;
    rv[f] = r < nw;
    cv[f] = c < nw;
    ri[f] = rv[f] ? r : 0;
    ci[f] = cv[f] ? c : 0;
  }
  Cfrag<R> C[FR][FR];
#pragma unroll
  for (int fi = 0; fi < FR; ++fi)
#pragma unroll
    for (int fj = 0; fj < FR; ++fj) C[fi][fj].zero();

  // ---- P = M E_{k+b}: A[r][l] = src[r + l nw], B[l][c] = ETkb[c + l nw]
  T2 qa[PF][FR];
  cplx qb[PF][FR];
#pragma unroll
  for (int j = 0; j < PF; ++j) {
    const int l = 4 * j + lk;
    const size_t lo = (size_t)(l < nw ? l : 0) * nw;
#pragma unroll
    for (int f = 0; f < FR; ++f) {
      qa[j][f] = src[ri[f] + lo];
      qb[j][f] = ETkb[ci[f] + lo];
    }
  }
  for (int s0 = 0; s0 < nks; s0 += PF) {
#pragma unroll
    for (int j = 0; j < PF; ++j) {
      const int s = s0 + j;
      if (s < nks) {
        const bool lv = 4 * s + lk < nw;
        R ar[FR], ai[FR], br[FR], bi[FR];
#pragma unroll
        for (int f = 0; f < FR; ++f) {
          const bool va = lv && rv[f], vb = lv && cv[f];
          ar[f] = va ? (R)qa[j][f].x : (R)0;
          ai[f] = va ? (R)qa[j][f].y : (R)0;
          br[f] = vb ? (R)qb[j][f].x : (R)0;
          bi[f] = vb ? (R)qb[j][f].y : (R)0;
        }
        const int sn = s + PF;
        if (sn < nks) {
          const int l = 4 * sn + lk;
          const size_t lo = (size_t)(l < nw ? l : 0) * nw;
#pragma unroll
          for (int f = 0; f < FR; ++f) {
            qa[j][f] = src[ri[f] + lo];
            qb[j][f] = ETkb[ci[f] + lo];
          }
        }
#pragma unroll
        for (int fi = 0; fi < FR; ++fi)
#pragma unroll
          for (int fj = 0; fj < FR; ++fj) C[fi][fj].mma(ar[fi], ai[fi], br[fj], bi[fj]);
      }
    }
  }
  // P to LDS, row-major: P[r][c] at Ps[(part * GT + r) * LD + c]
#pragma unroll
  for (int fi = 0; fi < FR; ++fi)
#pragma unroll
    for (int fj = 0; fj < FR; ++fj)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = wr + fi * 16 + Mfma<R>::row(lk, i);
        const int c = wc + fj * 16 + lr;
        Ps[(0 * GT + r) * LD + c] = C[fi][fj].re(i);
        Ps[(1 * GT + r) * LD + c] = C[fi][fj].im(i);
      }
#pragma unroll
  for (int fi = 0; fi < FR; ++fi)
#pragma unroll
    for (int fj = 0; fj < FR; ++fj) C[fi][fj].zero();

  // ---- R = E_k^+ P: A[r][l] = conj(ETk[r + l nw]), B[l][c] = P[l][c]
  cplx qe[PF][FR];
#pragma unroll
  for (int j = 0; j < PF; ++j) {
    const int l = 4 * j + lk;
    const size_t lo = (size_t)(l < nw ? l : 0) * nw;
#pragma unroll
    for (int f = 0; f < FR; ++f) qe[j][f] = ETk[ri[f] + lo];
  }
  __syncthreads();
  for (int s0 = 0; s0 < nks; s0 += PF) {
#pragma unroll
    for (int j = 0; j < PF; ++j) {
      const int s = s0 + j;
      if (s < nks) {
        const int l = 4 * s + lk;
        const bool lv = l < nw;
        R ar[FR], ai[FR], br[FR], bi[FR];
#pragma unroll
        for (int f = 0; f < FR; ++f) {
          const bool va = lv && rv[f];
          ar[f] = va ? (R)qe[j][f].x : (R)0;
          ai[f] = va ? -(R)qe[j][f].y : (R)0;
          br[f] = Ps[(0 * GT + l) * LD + wc + 16 * f + lr];
          bi[f] = Ps[(1 * GT + l) * LD + wc + 16 * f + lr];
        }
        const int sn = s + PF;
        if (sn < nks) {
          const int ln = 4 * sn + lk;
          const size_t lo = (size_t)(ln < nw ? ln : 0) * nw;
#pragma unroll
          for (int f = 0; f < FR; ++f) qe[j][f] = ETk[ri[f] + lo];
        }
#pragma unroll
        for (int fi = 0; fi < FR; ++fi)
#pragma unroll
          for (int fj = 0; fj < FR; ++fj) C[fi][fj].mma(ar[fi], ai[fi], br[fj], bi[fj]);
      }
    }
  }

  // ---- epilogue: phases, moduli and sums from the accumulators; R through
  // LDS (column-major) for whole-block stores
  double od = 0.0, all = 0.0;
#pragma unroll
  for (int fi = 0; fi < FR; ++fi)
#pragma unroll
    for (int fj = 0; fj < FR; ++fj)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = wr + fi * 16 + Mfma<R>::row(lk, i);
        const int c = wc + fj * 16 + lr;
        if (r < nw && c < nw) {
          T2 v;
          v.x = C[fi][fj].re(i);
          v.y = C[fi][fj].im(i);
          const cplx vw = c_wide(v);
          const double a2 = c_abs2(vw);
          all += a2;
          if (mate >= 0) outm[c + (size_t)r * nw] = c_conj(v);
          if (r != c) {
            od += a2;
          } else {
            const double l = atan2(vw.y, vw.x);
            lnd[r] = l;
            d2d[r] = a2;
            if (mate >= 0) {
              p.ln[dst][(size_t)mate * nw + r] = -l;
              p.d2[(size_t)mate * nw + r] = a2;
            }
          }
        }
      }
  __syncthreads();  // every wavefront has read its last B fragment of P
#pragma unroll
  for (int fi = 0; fi < FR; ++fi)
#pragma unroll
    for (int fj = 0; fj < FR; ++fj)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = wr + fi * 16 + Mfma<R>::row(lk, i);
        const int c = wc + fj * 16 + lr;
        Ps[(0 * GT + c) * LD + r] = C[fi][fj].re(i);
        Ps[(1 * GT + c) * LD + r] = C[fi][fj].im(i);
      }
  __syncthreads();
  for (int e = tid; e < (int)nw2; e += 256) {
    const int r = e % nw, c = e / nw;
    T2 v;
    v.x = Ps[(0 * GT + c) * LD + r];
    v.y = Ps[(1 * GT + c) * LD + r];
    out[e] = v;
  }
  block_sum2(od, all, red);
  if (tid == 0) {
    p.part_od[kb * p.npan] = od;
    p.part_all[kb * p.npan] = all;
    if (mate >= 0) {
      p.part_od[(size_t)mate * p.npan] = od;
      p.part_all[(size_t)mate * p.npan] = all;
    }
  }
}

// The rotation for 32 < num_wann <= 64 with direct operand loads
// (rot_direct_tile); workgroup placement as k_rot_fused (the nnmax
// workgroups of one k back to back on one XCD, sharing ET_k in its L2).
template <class T2>
__global__ void __launch_bounds__(256, 2) k_rot_direct(const Prob* probs, const Item* items, int nitems,
                                                       int nnmax, int mode) {
  typedef typename Real<T2>::type R;
  const int w = blockIdx.x;
  const int r = w >> 3;
  const int item = 8 * (r / nnmax) + (w & 7);
  if (item >= nitems) return;
  const Item it = items[item];
  const Prob& p = probs[it.prob];
  const State* st = p.st;
  if (sizeof(T2) == sizeof(cplx) && p.nw <= W90_ROT_PANEL_MAX) return;  // k_rot_panel's
  const int cur = gate_cur(st, mode);
  if (cur < 0) return;
  int mate;
  const int b = rot_slot<T2>(p, it.k, r % nnmax, &mate);
  if (b < 0) return;
  __shared__ R Ps[2 * 64 * 65];
  __shared__ double red[256];
  rot_direct_tile<T2>(p, it.k, b, mate, mode, cur, Ps, red);
}

// Omega partial sums of the current M by GEMM tile (MODE_INIT of the MFMA
// class): the layout the stage-2 epilogue writes, without a rotation.
template <class T2, int GT>
__global__ void __launch_bounds__(256) k_reduce_tiles(const Prob* probs, const Item* items, int nitems, int mode) {
  if (blockIdx.x >= (unsigned)nitems) return;
  const Item it = items[blockIdx.x];
  const Prob& p = probs[it.prob];
  const State* st = p.st;
  const int cur = gate_cur(st, mode);
  if (cur < 0) return;
  const int nw = p.nw, nn = p.nn;
  const int nt1 = (nw + GT - 1) / GT;
  const int ntl = nt1 * nt1;
  const int by = blockIdx.y;
  if (by >= nn * ntl) return;
  const int b = by / ntl, tile = by % ntl;
  const int row0 = (tile % nt1) * GT, col0 = (tile / nt1) * GT;
  const size_t kb = (size_t)it.k * nn + b;
  const int dst = dst_buf(mode, cur);
  const T2* m = mbuf<T2>(p, cur) + kb * p.nw2;
  __shared__ double red[256];
  double od = 0.0, all = 0.0;
  for (int e = threadIdx.x; e < GT * GT; e += blockDim.x) {
    const int r = row0 + e % GT, c = col0 + e / GT;
    if (r >= nw || c >= nw) continue;
    const cplx v = c_wide(m[r + (size_t)c * nw]);
    const double a2 = c_abs2(v);
    all += a2;
    if (r != c) {
      od += a2;
    } else {
      p.ln[dst][kb * nw + r] = atan2(v.y, v.x);
      p.d2[kb * nw + r] = a2;
    }
  }
  block_sum2(od, all, red);
  if (threadIdx.x == 0) {
    p.part_od[kb * p.npan + tile] = od;
    p.part_all[kb * p.npan + tile] = all;
    // slots that only the FP64 rotation fills (one per 16 columns)
    if (tile == 0)
      for (int q = ntl; q < p.npan; ++q) p.part_od[kb * p.npan + q] = p.part_all[kb * p.npan + q] = 0.0;
  }
}

// ---------------------------------------------------------- retraction

#define W90_STEP_N 64

// Matrices of 16 TN x 16 TN in k_step_panel: column panel w (16 columns) is
// held by wavefront w in the result layout of the MFMA, element q of row
// tile t = row 16 t + 4 q + l / 16, column 16 w + l % 16, which is also the
// layout of the B operand of K step 4 t + q; a matrix that is an A operand
// goes to LDS as 16 x 16 tiles, row-major with the column XORed by the row
// (the store runs along rows and the operand load along columns, both
// without bank conflicts).
template <int TN>
struct Panel {
  double r[TN][4], i[TN][4];
};
constexpr int kStepWaves(int tn) { return tn == 1 ? 4 : tn == 2 ? 3 : 2; }  // wavefronts per SIMD the registers allow

// LDS place of the lane's element (t, q) of its panel
template <int TN>
__device__ __forceinline__ int panel_at(int t, int q) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, lr = lane & 15, row = 4 * q + (lane >> 4);
  return (t * TN + w) * 256 + row * 16 + (lr ^ row);
}
template <int TN>
__device__ __forceinline__ void panel_to_lds(cplx* L, const Panel<TN>& P) {
#pragma unroll
  for (int t = 0; t < TN; ++t)
#pragma unroll
    for (int q = 0; q < 4; ++q) L[panel_at<TN>(t, q)] = c_make(P.r[t][q], P.i[t][q]);
}

// Row tiles of A B (ADJ: A^+ B) for the wavefront's column panel: A in LDS,
// element (t, q) of B from get(t, q, re, im); row tile i of the product to
// out(i, acc).
template <int TN, bool ADJ = false, class Get, class Out>
__device__ __forceinline__ void panel_product(const cplx* L, Get get, Out out) {
  const int lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4;
  int off[4];  // A[l % 16][4 q + l / 16] of a tile, or (ADJ) A[4 q + l / 16][l % 16]
#pragma unroll
  for (int q = 0; q < 4; ++q) off[q] = ADJ ? (4 * q + lk) * 16 + (lr ^ (4 * q + lk)) : lr * 16 + ((4 * q + lk) ^ lr);
#pragma unroll
  for (int i = 0; i < TN; ++i) {
    Cfrag<double> acc;
    acc.zero();
#pragma unroll
    for (int t = 0; t < TN; ++t) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const cplx a = L[(ADJ ? t * TN + i : i * TN + t) * 256 + off[q]];
        double br, bi;
        get(t, q, br, bi);
        acc.mma(a.x, ADJ ? -a.y : a.y, br, bi);
      }
      // no LDS reads of later tiles ahead of the products: their registers
      // would push the panels out
      __builtin_amdgcn_sched_barrier(0);
    }
    out(i, acc);
  }
}

// ------------------------------------------------ rotation by column panels

// The FP64 rotation for num_wann 17-48: R = E_k^+ (M(k,b) E_{k+b}) with one
// wavefront per 16 columns, TN = ceil(num_wann / 16) of them.  E_k^+ is the A
// operand of the second product for every b of the k: a workgroup stages it in
// LDS once and takes up to bchunk blocks of the k.  The first product's A operand
// is M itself, read from memory in operand order (rows along the lanes), kRotPF
// K steps ahead, with a row tile ahead of that touched for L2; its B operand, the
// wavefront's columns of E_{k+b}, and its result, which is the B operand of the
// second product as it stands, stay in registers.  No barrier between the
// products or blocks: wavefronts drift apart and cover each other's loads.  The
// next block's columns of E and first operands of M arrive during the second
// product.
//
// Epilogue: R to the other buffer (and its adjoint to the pair's block), the
// sums of |M|^2 of the wavefront's columns (TN partial sums per block), and the
// diagonal to LDS: Im ln M_nn and |M_nn|^2 follow at the end, for inside the loop
// the compiler keeps atan2's constants in 40 registers over the products.
// Items with another TN are left out.  Placement as k_rot_fused (the workgroups
// of a k back to back on one XCD).
//
// Per block two products of 48 TN^3 MFMA instructions, 64 cycles each: 23 us of
// the 61 at 44 bands; the rest are the chain of tables, E_k and first operands
// before a workgroup's products (7 us) and, at TN = 3, three wavefronts to four
// SIMDs.  Measured per rotation by pairs against a workgroup per block with both
// products staged through LDS in K chunks, two barriers a chunk (k_rot_fused):
//   27 bands, 216 k, nntot 12: 27.2 -> 21.8 us   32, 512 k, 6: 30.4 -> 25.2 us
//   44 bands, 343 k, nntot 8: 69.0 -> 61.0 us    48, 216 k, 12: 71.0 -> 64 us
// With four panels the two operand panels, the accumulators and the loads in
// flight pass the 256 registers: 76 -> 76 us at 52 bands and 404 -> 382 at 64
// with scratch traffic, so 49-64 bands stay with k_rot_fused and k_rot_direct.
constexpr int kRotPF = 4;  // K steps of M in flight

// A pointer that is the same in every lane (said to the compiler here).
template <class T>
__device__ __forceinline__ T* uniform(T* q) {
  const unsigned long long u = (unsigned long long)q;
  const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)u), hi = __builtin_amdgcn_readfirstlane((unsigned)(u >> 32));
  return (T*)(((unsigned long long)hi << 32) | lo);
}

// A matrix of `bytes` bytes as a buffer: offsets past it read zero, writes there
// are dropped.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf_rsrc(const cplx* base, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)uniform(base), 0, __builtin_amdgcn_readfirstlane(bytes), 0x00020000);
}
__device__ __forceinline__ cplx buf_load(__amdgpu_buffer_rsrc_t r, unsigned byte) {
  return __builtin_bit_cast(cplx, __builtin_amdgcn_raw_buffer_load_b128(r, byte, 0, 0));
}
__device__ __forceinline__ void buf_store(__amdgpu_buffer_rsrc_t r, unsigned byte, cplx v) {
  typedef unsigned v4u __attribute__((ext_vector_type(4)));
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u, v), r, byte, 0, 0);
}

// What the rotation reads of a problem, in scalar registers: read after a store
// it would wait for the store.
struct RotProb {
  const cplx *E, *src;
  cplx* out;
  double *od, *all;
  int nw, nn, npan;
  __device__ __forceinline__ void read(const Prob& p, int mode, int cur) {
    E = uniform((const cplx*)p.E);
    src = uniform(rot_src<cplx>(p, mode, cur));
    out = uniform(p.M[dst_buf(mode, cur)]);
    od = uniform(p.part_od);
    all = uniform(p.part_all);
    nw = __builtin_amdgcn_readfirstlane(p.nw);
    nn = __builtin_amdgcn_readfirstlane(p.nn);
    npan = __builtin_amdgcn_readfirstlane(p.npan);
  }
};

template <int TN>
__global__ void __launch_bounds__(64 * TN, kStepWaves(TN)) k_rot_panel(const Prob* probs, const Item* items,
                                                                      int nitems, int nchunk, int bchunk, int mode) {
  const int wg = blockIdx.x, rr = wg >> 3;
  const int item = 8 * (rr / nchunk) + (wg & 7);
  if (item >= nitems) return;
  const Item it = items[item];
  const Prob& p = probs[it.prob];
  if ((p.nw + 15) / 16 != TN) return;
  const int cur = gate_cur(p.st, mode);
  if (cur < 0) return;
  const int j0 = (rr % nchunk) * bchunk, nu = min(bchunk, (p.npair > 0 ? p.npair : p.nn) - j0);
  if (nu <= 0) return;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lr = lane & 15, lk = lane >> 4, k = it.k;
  __shared__ cplx L[TN * TN * 256];
  __shared__ cplx dg[W90_ROT_SLOTS * 16 * TN];
  __shared__ int slot_b[W90_ROT_SLOTS], slot_mate[W90_ROT_SLOTS], slot_k[W90_ROT_SLOTS];
  if ((int)threadIdx.x < nu) {
    int m;
    const int b = rot_slot<cplx>(p, k, j0 + threadIdx.x, &m);
    slot_b[threadIdx.x] = b;
    slot_mate[threadIdx.x] = m;
    slot_k[threadIdx.x] = p.nnl[(size_t)k * p.nn + b];
  }
  RotProb F;
  F.read(p, mode, cur);
  const int nw = F.nw, nw2 = nw * nw, bytes = 16 * nw2;
  const unsigned ks = 64u * nw;
  const int col = 16 * w + lr;
  auto row_of = [&](int t, int q) { return 16 * t + 4 * q + lk; };
  const unsigned far = 0xc0000000u;  // past any matrix, also with a tile's offset added
  constexpr int NS = 4 * TN;         // K steps of the first product
  auto load_panel = [&](const cplx* E, Panel<TN>& P) {
    const auto r = buf_rsrc(E, bytes);
    const unsigned oc = 16u * (unsigned)(col * nw + lk);
#pragma unroll
    for (int t = 0; t < TN; ++t)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const cplx e = buf_load(r, oc + 16u * (16 * t + 4 * q));
        P.r[t][q] = e.x;
        P.i[t][q] = e.y;
      }
  };
  // a word of every 64 bytes of a row tile of M, the wavefront's columns: the
  // operand loads of all wavefronts, a row tile later, then find it in L2
  unsigned warm = 0;
  auto touch = [&](__amdgpu_buffer_rsrc_t r, int i) {
    warm = __builtin_amdgcn_raw_buffer_load_b32(r, 16u * (unsigned)(col * nw + 4 * lk) + 256u * i, 0, 0);
  };
  cplx a[kRotPF];  // M's operand of K step x % NS, row tile x / NS
  Panel<TN> B, P;
  load_panel(F.E + (size_t)k * nw2, P);
  __syncthreads();
  int b, mate;
  // columns of E and first operands of M of slot u
  auto begin = [&](int u) {
    b = __builtin_amdgcn_readfirstlane(slot_b[u]);
    mate = __builtin_amdgcn_readfirstlane(slot_mate[u]);
    load_panel(F.E + (size_t)__builtin_amdgcn_readfirstlane(slot_k[u]) * nw2, B);
    const auto m = buf_rsrc(F.src + ((size_t)k * F.nn + b) * nw2, bytes);
    const unsigned of = 16u * (unsigned)(lk * nw + lr);
#pragma unroll
    for (int x = 0; x < kRotPF; ++x) a[x] = buf_load(m, of + x * ks);
  };
  begin(0);
#pragma unroll
  for (int t = 0; t < TN; ++t)
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (row_of(t, q) >= nw) P.r[t][q] = P.i[t][q] = 0.0;
  panel_to_lds<TN>(L, P);
  __syncthreads();
  for (int u = 0; u < nu; ++u) {
    const size_t kb = (size_t)k * F.nn + b;
    const auto msrc = buf_rsrc(F.src + kb * nw2, bytes);
    // offsets anew for each block: kept over the loop they take the panels' registers
    unsigned of = 16u * (unsigned)(lk * nw + lr), oc = 16u * (unsigned)(col * nw + lk),
             om = col < nw ? 16u * (unsigned)(lk * nw + col) : far;
    asm volatile("" : "+v"(of), "+v"(oc), "+v"(om));
#pragma unroll
    for (int i = 0; i < TN; ++i) {
      Cfrag<double> acc;
      acc.zero();
      if (i + 1 < TN) touch(msrc, i + 1);
#pragma unroll
      for (int sk = 0; sk < NS; ++sk) {
        const int x = i * NS + sk, y = x + kRotPF;
        const cplx v = a[x % kRotPF];
        if (y < TN * NS) a[x % kRotPF] = buf_load(msrc, of + (y % NS) * ks + 256u * (y / NS));
        acc.mma(v.x, v.y, B.r[sk / 4][sk % 4], B.i[sk / 4][sk % 4]);
        if (sk % 2 == 1) __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        P.r[i][q] = acc.re(q);
        P.i[i][q] = acc.im(q);
        // formed here: left to the compiler the three accumulators stay, half as many registers again
        asm volatile("" : "+v"(P.r[i][q]), "+v"(P.i[i][q]));
      }
      asm volatile("" ::"v"(warm));
      __builtin_amdgcn_sched_barrier(0);
    }
    // the next block's, ahead of this one's stores, which share the wait counter
    const int part = kb * F.npan + w, matep = mate;
    const auto out = buf_rsrc(F.out + kb * nw2, bytes);
    const auto outm = buf_rsrc(F.out + (mate >= 0 ? (size_t)mate * nw2 : 0), mate >= 0 ? bytes : 0);
    if (u + 1 < nu) begin(u + 1);
    __builtin_amdgcn_sched_barrier(0);
    double od = 0.0, all = 0.0;
    panel_product<TN, true>(
        L, [&](int t, int q, double& br, double& bi) { br = P.r[t][q]; bi = P.i[t][q]; },
        [&](int i, const Cfrag<double>& acc) {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const int row = row_of(i, q);
            const cplx v = c_make(acc.re(q), acc.im(q));
            buf_store(out, i < TN - 1 || row < nw ? oc + 16u * (16 * i + 4 * q) : far, v);
            buf_store(outm, om + (4 * i + q) * ks, c_conj(v));
            const double a2 = c_abs2(v);  // zero past num_wann
            all += a2;
            if (i == w) {  // the tile on the diagonal
              od += 4 * q + lk != lr ? a2 : 0.0;
              if (4 * q + lk == lr) dg[u * 16 * TN + col] = v;
            } else {
              od += a2;
            }
          }
          __builtin_amdgcn_sched_barrier(0);
        });
    od = wave_sum(od);
    all = wave_sum(all);
    if (lane == 0) {
      F.od[part] = od;
      F.all[part] = all;
      if (matep >= 0) {
        F.od[matep * F.npan + w] = od;
        F.all[matep * F.npan + w] = all;
      }
    }
  }
  __syncthreads();
  double *ln = p.ln[dst_buf(mode, cur)], *d2 = p.d2;
  for (int e = threadIdx.x; e < nu * 16 * TN; e += 64 * TN) {
    const int u = e / (16 * TN), n = e - u * 16 * TN, m = slot_mate[u];
    if (n >= nw) continue;
    const cplx z = dg[e];
    const size_t at = ((size_t)k * F.nn + slot_b[u]) * nw + n;
    const double l = atan2(z.y, z.x), a2 = c_abs2(z);
    ln[at] = l;
    d2[at] = a2;
    if (m >= 0) {
      ln[(size_t)m * nw + n] = -l;
      d2[(size_t)m * nw + n] = a2;
    }
  }
}

// Retraction of one (problem, k) for num_wann <= W90_PANEL_MAX: forms D (trial step),
// X = scale D, E = exp(X) and U_new = U E, one wavefront per 16 columns, TN =
// ceil(num_wann / 16) of them.  A wavefront's columns of X, X2 and the
// product in hand stay in its registers; only the left factor of each
// product goes through LDS, so a product is MFMA instructions with one LDS
// read per three of them.  ||X||_2 is bounded by ||X2||_F^(1/2) once X2 is
// known: closer than the 1-norm of X, and it saves squarings.  exp(X) of the
// anti-Hermitian X is the unitary internal_new_u_and_m builds from the
// eigenvectors of i X (wannierise.F90:1662-1689, 1729-1734).  Workgroups of
// items with another TN return at once.
//
// What bounds it: three products, the squarings and U E at the rate of the
// FP64 MFMA pipe for 49-64 bands (four of 5 us per CU and k), the loads and
// the search below.  Horner's form took a product per degree, 5 to 11 of
// them, with both factors in LDS.  Averages over the launches of a solve, before
// -> now: 16 bands, 512 k 12.7 -> 10.6 us; 27, 216 k 26.2 -> 16.4; 44, 384 k 70
// -> 47; 64, 800 k 205 -> 159; 91, 216 k 422 -> 200 (from k_step's form, all
// operands in the caches).  Alone, without the search, the read of G and the
// store of D, it takes 6.5, 12.7, 39, 126 and 167 us at these sizes.
template <int TN>
__global__ void __launch_bounds__(64 * TN, kStepWaves(TN)) k_step_panel(const Prob* probs, const Item* items,
                                                                       int nitems, int mode) {
  if (blockIdx.x >= (unsigned)nitems) return;
  const Item it = items[blockIdx.x];
  const Prob& p = probs[it.prob];
  if ((p.nw + 15) / 16 != TN) return;
  const State* st = p.st;
  const int cur = gate_cur(st, mode);
  if (cur < 0) return;
  const int nw = p.nw, nw2 = p.nw2;
  const int k = it.k, lane = threadIdx.x & 63, w = threadIdx.x >> 6, lr = lane & 15, lk = lane >> 4;
  __shared__ cplx L[TN * TN * 256];
  __shared__ double red[256];
  __shared__ State lst;
  const int col = 16 * w + lr;
  // element (t, q) of the panel: row 16 t + 4 q + lk
  auto row_of = [&](int t, int q) { return 16 * t + 4 * q + lk; };
  // a lane's element (t, q) of a block: uniform base, offset o + 16 t + 4 q
  const unsigned o = (unsigned)(col * nw + lk);
  cplx* Dk = p.D + (size_t)k * nw2;
  // G and D are requested before the search, so their latency overlaps it
  Panel<TN> X, G;
  {
    const cplx* Gk = p.G + (size_t)k * nw2;
#pragma unroll
    for (int t = 0; t < TN; ++t)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int row = row_of(t, q);
        cplx g = c_make(0.0, 0.0), d = g;
        if (row < nw && col < nw) {
          if (mode == MODE_TRIAL) g = Gk[o + 16 * t + 4 * q];
          d = Dk[o + 16 * t + 4 * q];
        }
        G.r[t][q] = g.x;
        G.i[t][q] = g.y;
        X.r[t][q] = d.x;
        X.i[t][q] = d.y;
      }
  }
  const State* ss = st;
  if (mode == MODE_TRIAL) {
    search_in_step(p, k, &lst, red);
    ss = &lst;
  }
  const double scale = ss->scale, beta = ss->beta, sign = ss->dir_sign;
#pragma unroll
  for (int t = 0; t < TN; ++t)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      cplx d = c_make(X.r[t][q], X.i[t][q]);
      if (mode == MODE_TRIAL) {
        d = c_scale(c_add(c_make(G.r[t][q], G.i[t][q]), c_scale(d, beta)), sign);
        const int row = row_of(t, q);
        if (row < nw && col < nw) Dk[o + 16 * t + 4 * q] = d;
      }
      X.r[t][q] = d.x * scale;
      X.i[t][q] = d.y * scale;
    }
  panel_to_lds<TN>(L, X);
  __syncthreads();
  Panel<TN> Y;  // X2
  double f2 = 0.0;
  panel_product<TN>(
      L, [&](int t, int q, double& br, double& bi) { br = X.r[t][q]; bi = X.i[t][q]; },
      [&](int i, const Cfrag<double>& acc) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const double a = acc.re(q), b = acc.im(q);
          Y.r[i][q] = a;
          Y.i[i][q] = b;
          f2 = fma(a, a, fma(b, b, f2));
        }
      });
  // ||X2||_F^2 over the wavefronts in order; every read of X in LDS is done
  f2 = wave_sum(f2);
  if (lane == 0) red[w] = f2;
  __syncthreads();
  f2 = 0.0;
#pragma unroll
  for (int v = 0; v < TN; ++v) f2 += red[v];
  const int sq = squarings(sqrt(sqrt(f2)));
  const double f = ldexp(1.0, -sq), ff = f * f;
#pragma unroll
  for (int t = 0; t < TN; ++t)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      X.r[t][q] *= f;
      X.i[t][q] *= f;
      Y.r[t][q] *= ff;
      Y.i[t][q] *= ff;
    }
  panel_to_lds<TN>(L, Y);
  __syncthreads();
  Panel<TN> A;  // A4; the panel of X2 is read back from LDS (three panels and
                // the accumulators do not fit the registers at TN = 4)
  panel_product<TN>(
      L,
      [&](int t, int q, double& br, double& bi) {
        const cplx y = L[panel_at<TN>(t, q)];
        br = fma(kT8x2, y.x, kT8x1 * X.r[t][q]);
        bi = fma(kT8x2, y.y, kT8x1 * X.i[t][q]);
      },
      [&](int i, const Cfrag<double>& acc) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          A.r[i][q] = acc.re(q);
          A.i[i][q] = acc.im(q);
        }
      });
#pragma unroll
  for (int t = 0; t < TN; ++t)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const cplx y = L[panel_at<TN>(t, q)];
      Y.r[t][q] = y.x;
      Y.i[t][q] = y.y;
    }
  __syncthreads();
  // the factors of the last product, and 1 + X + y2 X2 into X
#pragma unroll
  for (int t = 0; t < TN; ++t)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const double one = row_of(t, q) == col ? 1.0 : 0.0;
      const double xr = X.r[t][q], xi = X.i[t][q], yr = Y.r[t][q], yi = Y.i[t][q], ar = A.r[t][q], ai = A.i[t][q];
      L[panel_at<TN>(t, q)] = c_make(fma(kT8x3, yr, ar), fma(kT8x3, yi, ai));
      Y.r[t][q] = fma(kT8x7, ar, fma(kT8x6, yr, fma(kT8x5, xr, kT8x4 * one)));
      Y.i[t][q] = fma(kT8x7, ai, fma(kT8x6, yi, kT8x5 * xi));
      X.r[t][q] = one + fma(kT8y2, yr, xr);
      X.i[t][q] = fma(kT8y2, yi, xi);
    }
  __syncthreads();
  panel_product<TN>(
      L, [&](int t, int q, double& br, double& bi) { br = Y.r[t][q]; bi = Y.i[t][q]; },
      [&](int i, const Cfrag<double>& acc) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          X.r[i][q] += acc.re(q);
          X.i[i][q] += acc.im(q);
        }
      });
  for (int s = 0; s < sq; ++s) {
    __syncthreads();
    panel_to_lds<TN>(L, X);
    __syncthreads();
    panel_product<TN>(
        L, [&](int t, int q, double& br, double& bi) { br = X.r[t][q]; bi = X.i[t][q]; },
        [&](int i, const Cfrag<double>& acc) {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            Y.r[i][q] = acc.re(q);
            Y.i[i][q] = acc.im(q);
          }
        });
    X = Y;
  }
  // E (and E^T where the rotation reads its operands from it), and U into LDS
  const cplx* Uc = p.U[cur] + (size_t)k * nw2;
#pragma unroll
  for (int t = 0; t < TN; ++t)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int row = row_of(t, q);
      cplx u = c_make(0.0, 0.0);
      if (row < nw && col < nw) u = Uc[o + 16 * t + 4 * q];
      Y.r[t][q] = u.x;
      Y.i[t][q] = u.y;
    }
  cplx* Ek = p.E + (size_t)k * nw2;
#pragma unroll
  for (int t = 0; t < TN; ++t)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int row = row_of(t, q);
      if (row < nw && col < nw) {
        const cplx e = c_make(X.r[t][q], X.i[t][q]);
        Ek[o + 16 * t + 4 * q] = e;
        if (p.want_et) p.ET[(size_t)k * nw2 + col + (size_t)row * nw] = e;
      }
    }
  __syncthreads();
  panel_to_lds<TN>(L, Y);
  __syncthreads();
  cplx* Un = p.U[1 - cur] + (size_t)k * nw2;
  panel_product<TN>(
      L, [&](int t, int q, double& br, double& bi) { br = X.r[t][q]; bi = X.i[t][q]; },
      [&](int i, const Cfrag<double>& acc) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int row = row_of(i, q);
          if (row < nw && col < nw) Un[o + 16 * i + 4 * q] = c_make(acc.re(q), acc.im(q));
        }
      });
}

// C = A B for n x n column-major complex matrices in global memory, held by
// one workgroup: each wavefront takes 16 x 16 output tiles in turn, two at
// a time (independent accumulator chains), on FP64 MFMA with the operand
// fragments loaded straight from memory (the matrices of one k stay in the
// caches: A fragments read along a column, B fragments reuse cache lines
// over consecutive K steps).  With adj, A^+ for A.  Used by the retraction
// above W90_PANEL_MAX bands and by the one-time kernels.
__device__ void wg_gemm_mfma(cplx* C, const cplx* A, const cplx* B, int n, bool adj) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nwv = blockDim.x >> 6;
  const int lr = lane & 15, lk = lane >> 4;
  const int nt = (n + 15) / 16;
  const int ntt = nt * nt;
  for (int t0 = 2 * w; t0 < ntt; t0 += 2 * nwv) {
    const bool two = t0 + 1 < ntt;
    int i0[2], j0[2];
    Cfrag<double> cc[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int t = two ? t0 + u : t0;
      i0[u] = (t % nt) * 16;
      j0[u] = (t / nt) * 16;
      cc[u].zero();
    }
    for (int ks = 0; ks < n; ks += 4) {
      const int kk = ks + lk;
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int r = i0[u] + lr, c = j0[u] + lr;
        const cplx a = (r < n && kk < n) ? A[adj ? kk + (size_t)r * n : r + (size_t)kk * n] : c_make(0.0, 0.0);
        const cplx b = (kk < n && c < n) ? B[kk + (size_t)c * n] : c_make(0.0, 0.0);
        cc[u].mma(a.x, adj ? -a.y : a.y, b.x, b.y);
      }
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      if (u == 1 && !two) break;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = i0[u] + Mfma<double>::row(lk, i), c = j0[u] + lr;
        if (r < n && c < n) C[r + (size_t)c * n] = c_make(cc[u].re(i), cc[u].im(i));
      }
    }
  }
  __syncthreads();
}

// ---------------------------------------------------------- projection

// Lowdin orthonormalisation of overlap_project (src/overlap.F90:758-952)
// for num_bands = num_wann: the unitary polar factor U = A (A^+ A)^-1/2 of
// A(k) (staged in G), which is the Z V^+ built there from the SVD
// A = Z S V^+.  Newton-Schulz iteration X <- X (3 - X^+ X)/2 from
// X = A/||A||_F (all singular values in (0,1]) converges to it for
// non-singular A, quadratically near the end: once X^+ X = 1 to 1e-12 one
// more step reaches rounding level and the iteration stops (at most
// kPolarSteps).  Writes U(k) to E.
constexpr int kPolarSteps = 200;

// Above 64 bands: matrices in global memory, one workgroup per k.
__global__ void __launch_bounds__(W90_STEP_NT) k_polar(const Prob* probs, const Item* items, int nitems) {
  if (blockIdx.x >= (unsigned)nitems) return;
  const Item it = items[blockIdx.x];
  const Prob& p = probs[it.prob];
  const int nw = p.nw, nw2 = p.nw2;
  const int k = it.k;
  cplx* X = p.E + (size_t)k * nw2;
  cplx* Y = p.W1 + (size_t)k * nw2;
  cplx* Z = p.W2 + (size_t)k * nw2;
  __shared__ double red[W90_NT];
  const cplx* Ak = p.G + (size_t)k * nw2;
  double fro = 0.0;
  for (int e = threadIdx.x; e < nw2; e += blockDim.x) fro += c_abs2(Ak[e]);
  fro = sqrt(block_sum(fro, red));
  const double inv = (fro > 0.0 && isfinite(fro)) ? 1.0 / fro : 0.0;
  for (int e = threadIdx.x; e < nw2; e += blockDim.x) X[e] = c_scale(Ak[e], inv);
  __syncthreads();
  for (int iter = 0; iter < kPolarSteps; ++iter) {
    wg_gemm_mfma(Y, X, X, nw, true);
    double dev = 0.0;
    bool bad = false;
    for (int e = threadIdx.x; e < nw2; e += blockDim.x) {
      cplx y = Y[e];
      const bool diag = e % nw == e / nw;
      const cplx d = c_make(y.x - (diag ? 1.0 : 0.0), y.y);
      const double v = sqrt(c_abs2(d));
      bad |= v != v;
      dev = fmax(dev, v);
      // 3 - X^+ X, halved below
      Y[e] = c_make(-y.x + (diag ? 3.0 : 0.0), -y.y);
    }
    dev = block_max(dev, red);
    if (__syncthreads_or(bad)) break;  // non-finite input: left to the unitarity check
    wg_gemm_mfma(Z, X, Y, nw);
    for (int e = threadIdx.x; e < nw2; e += blockDim.x) X[e] = c_scale(Z[e], 0.5);
    __syncthreads();
    if (dev < 1e-12) break;
  }
}

// Up to 64 bands: X in LDS as the A operand and the panels of the products in
// registers, as in k_step_panel.  32 bands, 216 k: 387 -> 54 us against
// scalar products from global memory.
template <int TN>
__global__ void __launch_bounds__(64 * TN, kStepWaves(TN)) k_polar_panel(const Prob* probs, const Item* items,
                                                                        int nitems) {
  if (blockIdx.x >= (unsigned)nitems) return;
  const Item it = items[blockIdx.x];
  const Prob& p = probs[it.prob];
  if ((p.nw + 15) / 16 != TN) return;
  const int nw = p.nw, nw2 = p.nw2;
  const int k = it.k, lane = threadIdx.x & 63, w = threadIdx.x >> 6, lr = lane & 15, lk = lane >> 4;
  __shared__ cplx L[TN * TN * 256];
  __shared__ double red[2 * TN];
  const int col = 16 * w + lr;
  const unsigned o = (unsigned)(col * nw + lk);
  auto row_of = [&](int t, int q) { return 16 * t + 4 * q + lk; };
  const cplx* Ak = p.G + (size_t)k * nw2;
  Panel<TN> X, Y;
  double fro = 0.0;
#pragma unroll
  for (int t = 0; t < TN; ++t)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      cplx a = c_make(0.0, 0.0);
      if (row_of(t, q) < nw && col < nw) a = Ak[o + 16 * t + 4 * q];
      X.r[t][q] = a.x;
      X.i[t][q] = a.y;
      fro += c_abs2(a);
    }
  fro = wave_sum(fro);
  if (lane == 0) red[w] = fro;
  __syncthreads();
  fro = 0.0;
#pragma unroll
  for (int v = 0; v < TN; ++v) fro += red[v];
  fro = sqrt(fro);
  const double inv = (fro > 0.0 && isfinite(fro)) ? 1.0 / fro : 0.0;
#pragma unroll
  for (int t = 0; t < TN; ++t)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      X.r[t][q] *= inv;
      X.i[t][q] *= inv;
    }
  for (int iter = 0; iter < kPolarSteps; ++iter) {
    __syncthreads();
    panel_to_lds<TN>(L, X);
    __syncthreads();
    // Y = (3 - X^+ X) / 2 and the largest |X^+ X - 1| (NaN kept: the sum below
    // carries it)
    double dev = 0.0, nan = 0.0;
    panel_product<TN, true>(
        L, [&](int t, int q, double& br, double& bi) { br = X.r[t][q]; bi = X.i[t][q]; },
        [&](int i, const Cfrag<double>& acc) {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const double one = row_of(i, q) == col && col < nw ? 1.0 : 0.0;
            const double a = acc.re(q), b = acc.im(q);
            const double v = sqrt((a - one) * (a - one) + b * b);
            dev = fmax(dev, v);
            nan += v - v;
            Y.r[i][q] = 0.5 * (3.0 * one - a);
            Y.i[i][q] = -0.5 * b;
          }
        });
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      dev = fmax(dev, __shfl_xor(dev, off, 64));
      nan += __shfl_xor(nan, off, 64);
    }
    if (lane == 0) {
      red[w] = dev;
      red[TN + w] = nan;
    }
    __syncthreads();
#pragma unroll
    for (int v = 0; v < TN; ++v) {
      dev = fmax(dev, red[v]);
      nan += red[TN + v];
    }
    if (nan != nan) break;  // non-finite input: left to the unitarity check
    panel_product<TN>(
        L, [&](int t, int q, double& br, double& bi) { br = Y.r[t][q]; bi = Y.i[t][q]; },
        [&](int i, const Cfrag<double>& acc) {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            X.r[i][q] = acc.re(q);
            X.i[i][q] = acc.im(q);
          }
        });
    if (dev < 1e-12) break;
  }
  cplx* Ek = p.E + (size_t)k * nw2;
#pragma unroll
  for (int t = 0; t < TN; ++t)
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (row_of(t, q) < nw && col < nw) Ek[o + 16 * t + 4 * q] = c_make(X.r[t][q], X.i[t][q]);
}

// wann_check_unitarity (wannierise.F90:2594-2661): per-k maximum deviation
// of U U^+ and U^+ U from the identity (NaN gives infinity).  Both are
// Hermitian: a wavefront forms tiles of their upper triangles on FP64 MFMA,
// operands from the caches (64 bands, 800 k: 875 -> 135 us against scalar
// dot products of every element).
__global__ void __launch_bounds__(W90_NT) k_unitarity(const Prob* probs, const Item* items, int nitems) {
  if (blockIdx.x >= (unsigned)nitems) return;
  const Item it = items[blockIdx.x];
  const Prob& p = probs[it.prob];
  const int n = p.nw;
  const int k = it.k;
  const cplx* U = p.U[p.st->cur] + (size_t)k * p.nw2;
  __shared__ double red[W90_NT];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nwv = blockDim.x >> 6;
  const int lr = lane & 15, lk = lane >> 4;
  const int nt = (n + 15) / 16;
  double dev = 0.0;
  for (int x = w; x < nt * nt; x += nwv) {
    const int ti = x % nt, tj = x / nt;
    if (ti > tj) continue;
    const int r = 16 * ti + lr, c = 16 * tj + lr;
    Cfrag<double> c1, c2;
    c1.zero();
    c2.zero();
    for (int ks = 0; ks < n; ks += 4) {
      const int kk = ks + lk;
      const bool vr = r < n && kk < n, vc = c < n && kk < n;
      const cplx z = c_make(0.0, 0.0);
      const cplx a1 = vr ? U[r + (size_t)kk * n] : z, b1 = vc ? U[c + (size_t)kk * n] : z;
      const cplx a2 = vr ? U[kk + (size_t)r * n] : z, b2 = vc ? U[kk + (size_t)c * n] : z;
      c1.mma(a1.x, a1.y, b1.x, -b1.y);
      c2.mma(a2.x, -a2.y, b2.x, b2.y);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = 16 * ti + Mfma<double>::row(lk, i);
      if (row >= n || c >= n) continue;
      const double one = row == c ? 1.0 : 0.0;
      const double x1 = c1.re(i) - one, y1 = c1.im(i), x2 = c2.re(i) - one, y2 = c2.im(i);
      const double v1 = sqrt(x1 * x1 + y1 * y1), v2 = sqrt(x2 * x2 + y2 * y2);
      if (v1 != v1 || v2 != v2) dev = INFINITY;
      dev = fmax(dev, fmax(v1, v2));
    }
  }
  dev = block_max(dev, red);
  if (threadIdx.x == 0) p.unit[k] = dev;
}

// ---------------------------------------------------------- small blocks

// LDS bytes of k_rotate_w16 for up to nn neighbours: one padded 16 x 17
// block per wavefront, the diagonal of each rotated block (complex value,
// phase, modulus), the per-wave sums and the k's mesh tables (wb, bk).
template <class T2>
__host__ __device__ constexpr size_t rotate_w16_lds(int nn) {
  return sizeof(T2) * 16 * 17 * (size_t)nn + sizeof(double) * (4 * 16 * (size_t)nn + 6 * (size_t)nn);
}

// M rotation with the omega partial sums for num_wann <= 16: one workgroup
// per (problem, k), one wavefront per neighbour b, each block a single
// 16 x 16 MFMA tile (zero-padded).  T = E_k^+ M(k,b) is formed from operand
// fragments loaded straight from memory, passed through the wavefront's LDS
// block to become the A operand of R = T E_{k+b}; R goes back through the
// same LDS block so that it is stored in column order (coalesced) and its
// diagonal is collected per b; the phases Im ln M_nn of all b are then
// formed in one pass over the workgroup, and threads n < num_wann sum them
// over b in order.  blockDim.x = 64 * (largest nntot of the launch); wavefronts beyond
// the problem's nntot only take part in the barriers, and every sum is
// formed per wavefront and then over b in order, so a problem's result does
// not depend on the other problems of the launch.  MODE_INIT only reduces.
// (internal_new_u_and_m :1737-1748; wann_omega :2034-2090, :2214-2275)
template <class T2>
__global__ void __launch_bounds__(64 * W90GPU_NUM_NNMAX) k_rotate_w16(const Prob* probs, const Item* items,
                                                                      int nitems, int mode) {
  typedef typename Real<T2>::type R;
  if (blockIdx.x >= (unsigned)nitems) return;
  const Item it = items[blockIdx.x];
  const Prob& p = probs[it.prob];
  const State* st = p.st;
  const int cur = gate_cur(st, mode);
  if (cur < 0) return;
  const int nw = p.nw, nw2 = p.nw2, nn = p.nn;
  const int nnl = blockDim.x >> 6;
  const int k = it.k;
  const int tid = threadIdx.x;
  const int b = tid >> 6;
  const bool active = b < nn;
  const int lane = tid & 63, lr = lane & 15, lk = lane >> 4;
  const bool rot = (mode != MODE_INIT);
  const int dst = dst_buf(mode, cur);
  extern __shared__ double lds_w16[];
  T2* Tl = reinterpret_cast<T2*>(lds_w16) + (size_t)b * 16 * 17;  // this wave's block, column-major
  double* lnL = reinterpret_cast<double*>(reinterpret_cast<T2*>(lds_w16) + (size_t)nnl * 16 * 17);
  double* d2L = lnL + nnl * 16;
  double* wod = d2L + nnl * 16;
  double* wall = wod + nnl;
  double* wbL = wall + nnl;
  double* bkL = wbL + nnl;
  double* dRe = bkL + 3 * nnl;  // [b][16] diagonal of the rotated block
  double* dIm = dRe + nnl * 16;
  // mesh tables and the reference centres are loaded with the operands,
  // not inside the loops over b of the epilogue
  kmesh_stage(p, k, wbL, bkL);
  double r0[3];
  if (tid < nw) ref_centre(p, mode, cur, tid, r0);
  const size_t kb = (size_t)k * nn + (active ? b : 0);
  const T2* src = rot_src<T2>(p, mode, cur) + kb * nw2;
  const cplx* Ek = p.E + (size_t)k * nw2;
  const cplx* Ekb = p.E + (size_t)p.nnl[kb] * nw2;
  // output addresses are formed before the first store (the compiler
  // would otherwise reload the problem's pointers after each store)
  T2* out = mbuf<T2>(p, dst) + kb * nw2;
  double* lnd = p.ln[dst] + (size_t)k * nn * nw;
  double* outk = p.kpart + (size_t)k * p.psz;
  Cfrag<R> Racc;
  Racc.zero();
  // every operand fragment of both products is loaded up front, so the
  // global-memory latencies overlap
  cplx fa[4], fm[4], fb[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const int l = 4 * s + lk;
    fa[s] = fm[s] = fb[s] = c_make(0.0, 0.0);
    if (active && rot && l < nw && lr < nw) {
      fa[s] = Ek[l + lr * nw];
      fm[s] = c_wide(src[l + lr * nw]);
      fb[s] = Ekb[l + lr * nw];
    }
  }
  if (active && rot) {
    // T = E_k^+ M: A[i][l] = conj(E_k[l + i nw]), B[l][j] = M[l + j nw]
    Cfrag<R> Tacc;
    Tacc.zero();
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const cplx a = fa[s], v = fm[s];
      Tacc.mma((R)a.x, (R)(-a.y), (R)v.x, (R)v.y);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      T2 t;
      t.x = Tacc.re(i);
      t.y = Tacc.im(i);
      Tl[Mfma<R>::row(lk, i) + lr * 17] = t;
    }
  }
  __syncthreads();
  if (active && rot) {
    // R = T E_{k+b}: A[i][l] = T[i][l] (LDS), B[l][j] = E_{k+b}[l + j nw]
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int l = 4 * s + lk;
      const T2 a = Tl[lr + l * 17];
      Racc.mma(a.x, a.y, (R)fb[s].x, (R)fb[s].y);
    }
    // R replaces T in the wavefront's block (every read of T above feeds
    // the products that produce R)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      T2 t;
      t.x = Racc.re(i);
      t.y = Racc.im(i);
      Tl[Mfma<R>::row(lk, i) + lr * 17] = t;
    }
  }
  __syncthreads();
  double s_od = 0.0, s_all = 0.0;
  if (active) {
    // element e = lane + 64 i of the block: consecutive lanes hold
    // consecutive rows of a column, so the stores are contiguous
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int e = lane + 64 * i;
      const int r = e & 15, c = e >> 4;
      if (r < nw && c < nw) {
        T2 v;
        if (rot) {
          v = Tl[r + c * 17];
          // streamed: the next readers of the block run on other XCDs
          st_stream(&out[r + c * nw], v);
        } else {
          v = src[r + c * nw];
        }
        const cplx vw = c_wide(v);
        const double a2 = c_abs2(vw);
        s_all += a2;
        if (r != c) {
          s_od += a2;
        } else {
          dRe[b * 16 + r] = vw.x;
          dIm[b * 16 + r] = vw.y;
        }
      }
    }
  }
  s_od = wave_sum(s_od);
  s_all = wave_sum(s_all);
  if (active && lane == 0) {
    wod[b] = s_od;
    wall[b] = s_all;
  }
  __syncthreads();
  // Im ln M_nn and |M_nn|^2 of every b in one pass
  for (int t = tid; t < nn * 16; t += blockDim.x) {
    const int bb = t >> 4, n = t & 15;
    if (n < nw) {
      const cplx vw = c_make(dRe[t], dIm[t]);
      const double l = atan2(vw.y, vw.x);
      lnd[bb * nw + n] = l;
      lnL[t] = l;
      d2L[t] = c_abs2(vw);
    }
  }
  __syncthreads();
  if (tid < nw) {
    const int n = tid;
    DiagAcc d = {};
    for (int bb = 0; bb < nn; ++bb)
      diag_add(d, wbL[bb], bkL + bb * 3, lnL[bb * 16 + n], d2L[bb * 16 + n], r0[0], r0[1], r0[2]);
    diag_store(outk, nw, n, d);
  }
  if (tid == 0) {
    double sod = 0.0, sall = 0.0, wsum = 0.0;
    for (int bb = 0; bb < nn; ++bb) {
      const double w = wbL[bb];
      sod += w * wod[bb];
      sall += w * wall[bb];
      wsum += w;
    }
    outk[8 * nw + 0] = sod;
    outk[8 * nw + 1] = (double)nw * wsum - sall;
  }
}
