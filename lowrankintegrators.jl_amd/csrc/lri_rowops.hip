// FP64 kernels on the thin n x r (m x r) factors and the r x r cores.
//
// k_rows is row-parallel over the tall dimension (tiles of 16..256 rows,
// grid-stride over tiles); its products run on FP64 matrix cores and it may
// end in a global reduction C = out' * W (or the Gram out' * out), written as
// one partial per workgroup.  k_reduce sums the partials in a fixed order (so
// results are bitwise reproducible) and k_epilogue runs a small epilogue on C
// in one workgroup: a Cholesky factorisation for CholeskyQR2, the S-step
// update, the Galerkin matrices of the BUG steps.
//
// These replace the LAPACK/BLAS calls of the reference on the factors:
// qr!/Matrix(Q) (projector_splitting.jl:137-138,149-150,174-175,186-187;
// unconventional.jl:141-152; rank_adaptive_unconventional.jl:204-217), the
// U*S / V*S' products (projector_splitting.jl:133,145,170,182), and the r x r
// S-step algebra (projector_splitting.jl:141-142; unconventional.jl:154-156;
// rank_adaptive_unconventional.jl:219-231).
#include <type_traits>

#include "lri_common.h"
#include "lri_kernels.h"

namespace lri {

constexpr int kThreads = 256;
constexpr double kEps = 2.220446049250313e-16;

// ----------------------------------------------------------------------------
// small dense routines on LDS-resident matrices (column-major, ld = k)
// ----------------------------------------------------------------------------

__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ double readlane_f64(double x, int lane) {
  const uint64_t u = __builtin_bit_cast(uint64_t, x);
  const uint32_t lo = __builtin_amdgcn_readlane((int)(uint32_t)u, lane);
  const uint32_t hi = __builtin_amdgcn_readlane((int)(uint32_t)(u >> 32), lane);
  return __builtin_bit_cast(double, (uint64_t(hi) << 32) | lo);
}

// Exponent e (even) with max_diag * 2^-e in [0.5, 2): the Gram matrix is
// scaled by 2^-e (exactly), so R scales by 2^(-e/2) and every pivot stays a
// normal number; zero, NaN and Inf give 0.
__device__ __forceinline__ int chol_scale_exp(double md) {
  int ex = 0;
  if (md > 0.0 && isfinite(md)) frexp(md, &ex);
  return ex & ~1;
}

// Upper Cholesky G = R'R (k <= K <= 64) and R^{-1}, right-looking on the
// augmented system [W | B], W the scaled G and B = L^{-1} (L = R', B starting
// as I): one elimination sweep yields R and R^{-T} together, with no back
// substitution.  G is scaled by 2^-e (exactly; max_i G(i,i) 2^-e in [0.5, 2))
// so that every pivot stays a normal number, and R and R^{-1} are unscaled at
// the end.  A pivot <= tau = 10 eps max_i G(i,i) (scaled) marks column p as
// numerically dependent: dropped[p] = 1, R(p,p) = 1, row p of R is zero and
// row and column p of R^{-1} are zero (so Q gets a zero column there).  R and
// Rinv are written to LDS (column-major, ld k).  Returns the number of
// dropped columns; sets *nonfinite on NaN/Inf.  Called by all threads.
//
// The rows of [W | B] are spread over the first four waves in blocks of four
// (wave w: row blocks w, w + 4, ...; at group g of 16 pivots, slot s of a
// wave's register window holds row 16 (g + s / 4) + 4 w + s % 4, and the
// window shifts by one block after each group) and the columns over the lanes
// (lane j: column j of W and of B).  The wave owning a block factors its four
// pivots in registers, the pivot rows exchanged by readlane, writes the four
// rows R(p, :) and L^{-1}(p, :) into one of two LDS buffers, and after one
// barrier every other wave applies them to its rows (K/4 slots, 2 FMAs each).
// Finished rows read zero multipliers, so no row needs a mask, and the group
// loop is not unrolled.  At k = 32 this takes ~26K cycles, against ~35K with
// one barrier per pivot and ~40K for one wave unrolled over the pivots (LDS
// broadcasts).  G is not modified.
template <int K>
__device__ int chol_inv_waves(const double* __restrict__ G, double* __restrict__ R, double* __restrict__ Rinv, int k,
                              unsigned char* dropped, int* nonfinite) {
  static_assert(K == 16 || K == 32 || K == 64, "K: 16, 32 or 64");
  constexpr int NS = K / 4;
  __shared__ double s_rowR[2][4][128];  // R(p, j) by column j; [K, 128) stays zero (rows past the window)
  __shared__ double s_rowB[2][4][64];   // L^{-1}(p, j)
  __shared__ int s_nfw[4];
  const int t = threadIdx.x, wv = t >> 6, j = t & 63;
  for (int e = t; e < 2 * 4 * 128; e += blockDim.x) (&s_rowR[0][0][0])[e] = 0.0;
  // the scale, found by every wave
  double md = j < k ? G[j + j * k] : 0.0;
  int nf0 = (j < k) && !isfinite(md);
  for (int off = 32; off > 0; off >>= 1) {
    md = fmax(md, __shfl_xor(md, off));
    nf0 |= __shfl_xor(nf0, off);
  }
  const int e2 = chol_scale_exp(md), eh = e2 / 2;
  const double tau = 10.0 * kEps * ldexp(md, -e2);
  double a[NS], b[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    const int tt = 16 * (s / 4) + 4 * wv + (s & 3);
    a[s] = (wv < 4 && tt < k && j < k && tt <= j) ? ldexp(G[tt + j * k], -e2) : 0.0;
    b[s] = (wv < 4 && tt == j && j < k) ? 1.0 : 0.0;
  }
  int nfl = nf0;
  __syncthreads();
  int buf = 0;
  for (int g = 0; 16 * g < k; ++g) {
#pragma unroll
    for (int wp = 0; wp < 4; ++wp) {
      const int p0 = 16 * g + 4 * wp;
      if (p0 < k) {
        if (wv == wp) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int p = p0 + i;
            if (p < k) {
              const double d = readlane_f64(a[i], p);
              const bool fin = isfinite(d);
              const bool keep = (d > tau) && fin;
              const double inv0 = rsqrt_nr(keep ? d : 1.0);
              const double inv = keep ? inv0 : 1.0;
              const double mR = (keep && j > p && j < k) ? a[i] * inv : 0.0;
              const double mB = (keep && j < k) ? b[i] * inv : 0.0;
#pragma unroll
              for (int i2 = i + 1; i2 < 4; ++i2) {
                const double rt = readlane_f64(mR, (p0 + i2) & 63);
                a[i2] = __builtin_fma(-rt, mR, a[i2]);
                b[i2] = __builtin_fma(-rt, mB, b[i2]);
              }
              s_rowR[buf][i][j] = mR;
              s_rowB[buf][i][j] = mB;
              if (j < k) {
                R[p + j * k] = j == p ? (keep ? d * inv : 1.0) : mR;
                Rinv[j + p * k] = mB;
              }
              if (j == p) dropped[p] = keep ? 0 : 1;
              nfl |= !fin;
            } else {
              s_rowR[buf][i][j] = 0.0;
              s_rowB[buf][i][j] = 0.0;
            }
          }
        }
        __syncthreads();
        if (wv < 4) {
          // the owner's own block is done; its later blocks start at slot 4
          const int s0 = wv == wp ? 4 : 0;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const double mRj = s_rowR[buf][i][j], mBj = s_rowB[buf][i][j];
#pragma unroll
            for (int s = 0; s < NS; ++s) {
              if (s >= s0) {
                const double rt = s_rowR[buf][i][16 * (g + s / 4) + 4 * wv + (s & 3)];
                a[s] = __builtin_fma(-rt, mRj, a[s]);
                b[s] = __builtin_fma(-rt, mBj, b[s]);
              }
            }
          }
        }
        buf ^= 1;
      }
    }
#pragma unroll
    for (int s = 0; s + 4 < NS; ++s) {
      a[s] = a[s + 4];
      b[s] = b[s + 4];
    }
#pragma unroll
    for (int s = (NS > 4 ? NS - 4 : 0); s < NS; ++s) {
      a[s] = 0.0;
      b[s] = 0.0;
    }
  }
  if (j == 0 && wv < 4) s_nfw[wv] = nfl;
  __syncthreads();
  // unscale; the rows of R^{-1} of dropped columns are zero (lanes: rows, waves: columns)
  const int nw = blockDim.x >> 6;
  if (j < k)
    for (int c = wv; c < k; c += nw) {
      R[j + c * k] = ldexp(R[j + c * k], eh);
      Rinv[j + c * k] = dropped[j] ? 0.0 : ldexp(Rinv[j + c * k], -eh);
    }
  const int nd = __popcll(__ballot(j < k && dropped[j]));
  if (t == 0 && (s_nfw[0] | s_nfw[1] | s_nfw[2] | s_nfw[3])) *nonfinite = 1;
  __syncthreads();
  return nd;
}

// The same factorisation (same scaling, drop rule and outputs) for k <= K <= 32
// on one wave, blocked by four pivots, with the trailing updates on the FP64
// matrix cores.  The whole scaled G and the running B = L^{-1} stay in
// registers in the v_mfma_f64_16x16x4_f64 result layout: 16 x 16 tiles (T1, T2),
// lane l and item u holding row 16 T1 + 4 u + l / 16, column 16 T2 + l % 16.
// Since G is kept symmetric, the panel of pivot block b (columns 4b .. 4b+3)
// in the operand layout of that instruction (lane l: row 16 t + l % 16, column
// 4b + l / 16) is item b % 4 of tile (b / 4, t) at the same lane: no data moves
// to form it.  Per block:
//  * the 4 x 4 diagonal block D is read by readlane (lane 16 q + 4 (b % 4) + a
//    holds D(a, q)) and factored in uniform registers with the drop rule
//    (keep_q = pivot > tau; inv_q = 1/sqrt(pivot)), giving the multipliers
//    Lb(a, q) and the upper triangular M with L(i, 4b + q) = sum_p A(i, 4b + p) M(p, q):
//    M(:, q) = keep_q inv_q (e_q - sum_{p<q} M(:, p) Lb(q, p));
//  * the panel L = A M takes four cross-lane reads per tile (ds_bpermute);
//  * B's block row becomes M' times itself (rows 4b + a live in item b % 4 of
//    tiles (b / 4, .) at lanes with l / 16 = a);
//  * G -= P P' and B -= P B(block row) on the matrix cores, P the panel with
//    its rows <= 4b + 3 zeroed (finished rows and columns stay untouched).
// The four pivots of a block form the only sequential chain: ~1,000 cycles per
// block against ~770 per pivot for the row-wise forms.  All threads call it;
// the first wave computes, the others wait at the final barrier.
template <int K>
__device__ int chol_inv_mfma(const double* __restrict__ G, double* __restrict__ R, double* __restrict__ Rinv, int k,
                             unsigned char* dropped, int* nonfinite) {
  static_assert(K == 16 || K == 32, "K: 16 or 32");
  constexpr int NT = K / 16, NB = K / 4;
  const int t = threadIdx.x, j = t & 63;
  if (t < 64) {
    const int lr = j & 15, lk = j >> 4;
    double md = j < k ? G[j + j * k] : 0.0;
    int nf0 = (j < k) && !isfinite(md);
    for (int off = 32; off > 0; off >>= 1) {
      md = fmax(md, __shfl_xor(md, off));
      nf0 |= __shfl_xor(nf0, off);
    }
    const int e2 = chol_scale_exp(md), eh = e2 / 2;
    const double tau = 10.0 * kEps * ldexp(md, -e2);
    f64x4_t g[NT][NT], x[NT][NT];
#pragma unroll
    for (int T1 = 0; T1 < NT; ++T1)
#pragma unroll
      for (int T2 = 0; T2 < NT; ++T2)
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int row = 16 * T1 + 4 * u + lk, col = 16 * T2 + lr;
          const bool in = row < k && col < k;
          const int lo = row < col ? row : col, hi = row < col ? col : row;  // the upper triangle
          const double v = G[in ? lo + hi * k : 0];
          g[T1][T2][u] = in ? ldexp(v, -e2) : 0.0;
          x[T1][T2][u] = row == col ? 1.0 : 0.0;
        }
    // one-hot weights of this lane's block column q = l / 16 (selects of uniform
    // values by lane, as multiply-adds: lane-dependent selects compile to branches)
    double w[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) w[q] = lk == q ? 1.0 : 0.0;
    // cross-lane read addresses: lane 16 p + l % 16
    int src[4];
#pragma unroll
    for (int p = 0; p < 4; ++p) src[p] = (16 * p + lr) << 2;
    auto bperm = [](int addr, double v) {
      const uint64_t u = __builtin_bit_cast(uint64_t, v);
      const uint32_t lo = __builtin_amdgcn_ds_bpermute(addr, (int)(uint32_t)u);
      const uint32_t hi = __builtin_amdgcn_ds_bpermute(addr, (int)(uint32_t)(u >> 32));
      return __builtin_bit_cast(double, (uint64_t(hi) << 32) | lo);
    };
    // pivots past k are zero and count as dropped: no mask is needed in the sweep
    uint32_t dm = 0;
    int nfv = 0;
    double rR[NB][NT];
#pragma unroll
    for (int kb = 0; kb < NB; ++kb) {
      const int T = kb >> 2, u0 = kb & 3;
      double P[NT];
#pragma unroll
      for (int tt = 0; tt < NT; ++tt) P[tt] = g[T][tt][u0];
      double W[4][4];
#pragma unroll
      for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int q = 0; q <= a; ++q) W[a][q] = readlane_f64(P[T], 16 * q + 4 * u0 + a);
      // the block's four pivots; a dropped pivot gets inv = 0, which zeroes its
      // multipliers and its column of M
      double Lb[4][4], inv[4], dq[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const double d = W[q][q];
        const bool keep = d > tau && d <= 1.7976931348623157e308;
        nfv |= !(fabs(d) <= 1.7976931348623157e308);
        dm |= keep ? 0u : 1u << (4 * kb + q);
        inv[q] = keep ? rsqrt_nr(d) : 0.0;
        dq[q] = keep ? 0.0 : 1.0;
#pragma unroll
        for (int a = q + 1; a < 4; ++a) Lb[a][q] = W[a][q] * inv[q];
#pragma unroll
        for (int a = q + 1; a < 4; ++a)
#pragma unroll
          for (int b = q + 1; b <= a; ++b) W[a][b] = __builtin_fma(-Lb[a][q], Lb[b][q], W[a][b]);
      }
      double M[4][4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        double c[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) c[i] = i == q ? 1.0 : 0.0;
#pragma unroll
        for (int p = 0; p < q; ++p)
#pragma unroll
          for (int i = 0; i <= p; ++i) c[i] = __builtin_fma(-M[i][p], Lb[q][p], c[i]);
#pragma unroll
        for (int i = 0; i < 4; ++i) M[i][q] = i <= q ? c[i] * inv[q] : 0.0;
      }
      double mq[4];
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        double v = M[p][3] * w[3];
#pragma unroll
        for (int q = 2; q >= p; --q) v = __builtin_fma(M[p][q], w[q], v);
        mq[p] = v;
      }
      const double drq = __builtin_fma(dq[0], w[0], __builtin_fma(dq[1], w[1], __builtin_fma(dq[2], w[2], dq[3] * w[3])));
      double Pm[NT];
#pragma unroll
      for (int tt = 0; tt < NT; ++tt) {
        double acc = bperm(src[0], P[tt]) * mq[0];
#pragma unroll
        for (int p = 1; p < 4; ++p) acc = __builtin_fma(bperm(src[p], P[tt]), mq[p], acc);
        // R(p, row) = L(row, p), p = 4 kb + l / 16: the panel at and below the
        // block's diagonal (1 on the diagonal of a dropped pivot), zero above
        const int row = 16 * tt + lr, a = row - 4 * kb;
        const double rv = a > lk ? acc : 0.0;
        rR[kb][tt] = a == lk ? acc + drq : rv;
        Pm[tt] = row >= 4 * kb + 4 ? acc : 0.0;
      }
      double xn[NT];
#pragma unroll
      for (int t2 = 0; t2 < NT; ++t2) {
        double acc = bperm(src[0], x[T][t2][u0]) * mq[0];
#pragma unroll
        for (int b = 1; b < 4; ++b) acc = __builtin_fma(bperm(src[b], x[T][t2][u0]), mq[b], acc);
        xn[t2] = acc;
      }
#pragma unroll
      for (int t2 = 0; t2 < NT; ++t2) x[T][t2][u0] = xn[t2];
#pragma unroll
      for (int t1 = T; t1 < NT; ++t1) {
#pragma unroll
        for (int t2 = T; t2 < NT; ++t2)
          g[t1][t2] = __builtin_amdgcn_mfma_f64_16x16x4f64(-Pm[t1], Pm[t2], g[t1][t2], 0, 0, 0);
#pragma unroll
        for (int t2 = 0; t2 <= T; ++t2)
          x[t1][t2] = __builtin_amdgcn_mfma_f64_16x16x4f64(-Pm[t1], xn[t2], x[t1][t2], 0, 0, 0);
      }
    }
    // R unscaled; R^{-1} = B' unscaled, the rows of dropped columns zero
#pragma unroll
    for (int kb = 0; kb < NB; ++kb)
#pragma unroll
      for (int tt = 0; tt < NT; ++tt) {
        const int p = 4 * kb + lk, row = 16 * tt + lr;
        if (p < k && row < k) R[p + row * k] = ldexp(rR[kb][tt], eh);
      }
#pragma unroll
    for (int T1 = 0; T1 < NT; ++T1)
#pragma unroll
      for (int T2 = 0; T2 < NT; ++T2)
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int c = 16 * T1 + 4 * u + lk, jj = 16 * T2 + lr;
          if (c < k && jj < k) Rinv[jj + c * k] = ((dm >> jj) & 1) ? 0.0 : ldexp(x[T1][T2][u], -eh);
        }
    if (j < k) dropped[j] = (dm >> j) & 1;
    // a non-finite pivot of a row past k cannot occur (those rows are zero)
    if (t == 0 && (nfv | nf0)) *nonfinite = 1;
  }
  __syncthreads();
  return __popcll(__ballot(j < k && dropped[j]));
}

// CK: the Cholesky variant compiled into an epilogue kernel (16, 32, 64: the
// bound on k): the one-wave matrix-core form up to 32, the four-wave form above.
template <int CK>
__device__ int chol_inv(const double* G, double* R, double* Rinv, int k, unsigned char* dropped, int* nonfinite) {
  if constexpr (CK <= 32) return chol_inv_mfma<CK>(G, R, Rinv, k, dropped, nonfinite);
  else return chol_inv_waves<CK>(G, R, Rinv, k, dropped, nonfinite);
}

// C = op(A) * op(B), k x k, column-major, on the FP64 matrix cores (16 x 16
// blocks over the workgroup's waves).  C must not alias A or B; every thread
// of the workgroup calls it.
__device__ void small_gemm(const double* __restrict__ A, int tA, const double* __restrict__ B, int tB,
                           double* __restrict__ C, int k) {
  // (the transposes select the index, not between two loads: a select of
  // loads compiles to branches)
  wave_gemm(
      k, k, k, 1, [&](int, int i, int l) { return A[tA ? l + i * k : i + l * k]; },
      [&](int, int l, int j) { return B[tB ? j + l * k : l + j * k]; },
      [&](int, int i, int j, double v) { C[i + j * k] = v; });
}

// LDS doubles the epilogue needs beyond C (a x b).
__host__ __device__ inline int epi_scratch_doubles(int kind, int a, int b) {
  int k = a > b ? a : b;
  switch (kind) {
    case EPI_CHOL1:
    case EPI_CHOL2:
    case EPI_CHOL3:
      return 3 * a * a;  // R, R^{-1} and Rtot (C may carry a cross term beyond its first a columns)
    case EPI_BUG_N:
      return 2 * k * k;
    case EPI_RA_N:
      return 2 * k * k;
    default:
      return 0;
  }
}

// ----------------------------------------------------------------------------
// epilogues run by the last workgroup on the reduced C (LDS, a x b)
// ----------------------------------------------------------------------------

// writer: this workgroup stores the results to the state (the epilogue of a
// reduction runs in one workgroup; folded into the prologue of the next row
// kernel, every workgroup computes the factors for itself and workgroup 0
// stores them).  The Cholesky kinds use C's first a columns as the Gram matrix.
//
// The Cholesky kinds.  own_right, own_nd: the factor on the right (LDS) and the first pass's
// dropped count, for a caller that runs all passes in one launch; nd_out receives this
// pass's count.
template <int CK>
__device__ void chol_epilogue(const EpiArgs& E, double* C, int a, double* scr, bool writer,
                              const double* own_right = nullptr, int own_nd = 0, int* nd_out = nullptr) {
  const int t = threadIdx.x;
  SmallState* st = E.small;
  const int k = a;
  __shared__ unsigned char dropped[kMaxAug];
  __shared__ int s_big;
  __shared__ double s_shift;
  if (E.kind == EPI_CHOL1 && E.shift_rows > 0) {
    // shifted CholeskyQR3, first factor: G + s I (Fukaya, Kannan, Nakatsukasa, Yamamoto,
    // Yanagisawa 2020), with ||G||_2 bounded by trace(G)
    if (t < 64) {
      double tr = 0.0;
      for (int i = t; i < k; i += 64) tr += C[i + i * k];
      for (int off = 32; off > 0; off >>= 1) tr += __shfl_xor(tr, off);
      if (t == 0) s_shift = 11.0 * ((double)E.shift_rows * k + (double)k * (k + 1)) * (0.5 * kEps) * tr;
    }
    __syncthreads();
    for (int i = t; i < k; i += blockDim.x) C[i + i * k] += s_shift;
    __syncthreads();
  }
  double* R = scr;
  double* Rinv = scr + k * k;
  int nf = 0, nd = 0;
  // CHOL2/3: the factor on the right of Rtot (R1, or the running Rtot) and
  // the first pass's dropped count were written by an earlier launch on
  // this stream; their loads are issued now, ahead of the factorisation
  // (for CK <= 32; the CK = 64 variant has no registers to spare)
  constexpr int NQ = CK <= 32 ? (CK * CK) / kThreads : 0;
  const double* right = own_right ? own_right : E.kind == EPI_CHOL2 ? st->R1 : st->Rtot;
  double rv[NQ > 0 ? NQ : 1];
  if (E.kind != EPI_CHOL1) {
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const int e = t + kThreads * q;
      rv[q] = e < k * k ? right[e] : 0.0;
    }
  }
  const int nd_first = E.kind == EPI_CHOL1 ? 0 : own_right ? own_nd : st->ndropped;
  // CholeskyQR2's second Gram matrix is I + E with |E| ~ eps cond^2: when
  // max|E| <= 1e-6 (and the first pass dropped nothing), R = I + F with
  // F = F1 + F2, F1 = upper(E) (diagonal halved), F2 = upper(-F1'F1)
  // (diagonal halved), and R^{-1} = I - F + F^2, all exact to O(|E|^3).
  bool pert = false;
  if (E.kind != EPI_CHOL1 && nd_first == 0) {
    if (t == 0) s_big = 0;
    __syncthreads();
    double mx = 0.0;
    for (int e = t; e < k * k; e += blockDim.x) {
      const int i = e % k, jj = e / k;
      const double v = C[e] - (i == jj ? 1.0 : 0.0);
      mx = fmax(mx, isfinite(v) ? fabs(v) : 1e300);
    }
    for (int off = 32; off > 0; off >>= 1) mx = fmax(mx, __shfl_xor(mx, off));
    if ((t & 63) == 0 && mx > 1e-6) atomicOr(&s_big, 1);  // any wave over the bound -> full Cholesky
    __syncthreads();
    pert = (s_big == 0);
  }
  if (pert) {
    double* F1 = Rinv;  // scratch: F1, then F1'F1 into R
    for (int e = t; e < k * k; e += blockDim.x) {
      const int i = e % k, jj = e / k;
      const double v = C[e] - (i == jj ? 1.0 : 0.0);
      F1[e] = i < jj ? v : (i == jj ? 0.5 * v : 0.0);
    }
    __syncthreads();
    small_gemm(F1, 1, F1, 0, R, k);  // R <- F1' F1
    __syncthreads();
    for (int e = t; e < k * k; e += blockDim.x) {  // C <- F = F1 + upper(-F1'F1) (diag halved)
      const int i = e % k, jj = e / k;
      const double f2 = i < jj ? -R[e] : (i == jj ? -0.5 * R[e] : 0.0);
      C[e] = F1[e] + f2;
    }
    __syncthreads();
    small_gemm(C, 0, C, 0, Rinv, k);  // Rinv <- F^2
    __syncthreads();
    for (int e = t; e < k * k; e += blockDim.x) {
      const int i = e % k, jj = e / k;
      const double id = i == jj ? 1.0 : 0.0;
      R[e] = id + C[e];
      Rinv[e] = id - C[e] + Rinv[e];
    }
    if (t < k) dropped[t] = 0;
    __syncthreads();
  } else {
    nd = chol_inv<CK>(C, R, Rinv, k, dropped, &nf);
  }
  if (E.kind == EPI_CHOL1) {
    if (writer)
      for (int e = t; e < k * k; e += blockDim.x) {
        st->R1[e] = R[e];
        st->R1inv[e] = Rinv[e];
      }
  } else {
    // Rtot = R2 * R1 (CHOL2) or R3 * Rtot (CHOL3) into the third scratch
    // matrix; the factor on the right was written by an earlier launch on
    // this stream; C is free now
    double* Rt = scr + 2 * k * k;
    if (own_right && !writer) return;  // a one-launch caller's workgroups need R^{-1} only
    if (writer)
      for (int e = t; e < k * k; e += blockDim.x) st->R2inv[e] = Rinv[e];
    if (NQ > 0) {
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        const int e = t + kThreads * q;
        if (e < k * k) C[e] = rv[q];
      }
    } else {
      for (int e = t; e < k * k; e += blockDim.x) C[e] = right[e];
    }
    __syncthreads();
    small_gemm(R, 0, C, 0, Rt, k);
    __syncthreads();
    if (writer)
      for (int e = t; e < k * k; e += blockDim.x) {
        const int i = e % k, jj = e / k;
        st->Rtot[e] = Rt[e];
        if (E.S) E.S[i + jj * E.ld_s] = E.transpose ? Rt[jj + i * k] : Rt[e];
      }
    if (E.stilde) {
      // C = [Q1'Q1 | Q1'W]: U1 = Q1 R2^{-1}, so U1'W = R2^{-T} (Q1'W) and
      // S~ = Rtot - U1'W; the first k columns of C are free again
      small_gemm(Rinv, 1, C + k * k, 0, C, k);
      __syncthreads();
      if (writer)
        for (int e = t; e < k * k; e += blockDim.x) {
          const int i = e % k, jj = e / k;
          const double v = Rt[e] - C[e];
          if (E.stilde == 2) st->St[jj + i * k] = v;
          else st->St[e] = v;
        }
    }
  }
  if (t == 0 && writer) {
    if (nf) atomicOr(E.flags, FLAG_NONFINITE);
    if (nd && E.breakdown_is_error) atomicOr(E.flags, FLAG_BREAKDOWN);
    if (E.kind == EPI_CHOL1) st->ndropped = nd;
  }
  if (t == 0 && nd_out) *nd_out = nd;
}

// The others (one workgroup).
__device__ void plain_epilogue(const EpiArgs& E, double* C, int a, int b, double* scr) {
  const int t = threadIdx.x;
  SmallState* st = E.small;
  switch (E.kind) {
    case EPI_STILDE: {
      const int k = a;
      for (int e = t; e < k * k; e += blockDim.x) {
        int i = e % k, j = e / k;
        double v = st->Rtot[e] - C[e];
        if (E.transpose) st->St[j + i * k] = v;
        else st->St[e] = v;
      }
      break;
    }
    case EPI_SFINAL: {
      const int k = a;
      for (int e = t; e < k * k; e += blockDim.x) {
        int i = e % k, j = e / k;
        E.S[i + j * E.ld_s] = E.transpose ? st->Rtot[j + i * k] : st->Rtot[e];
      }
      break;
    }
    case EPI_BUG_M: {
      for (int e = t; e < a * b; e += blockDim.x) st->M[e] = C[e];
      break;
    }
    case EPI_BUG_N: {
      // N = C; Sinit = M (S0 N') with S0, then M, staged in the first scratch matrix
      const int k = a;
      double* W = scr;
      double* T = scr + k * k;
      for (int e = t; e < k * k; e += blockDim.x) {
        st->N[e] = C[e];
        W[e] = E.S[(e % k) + (e / k) * E.ld_s];
      }
      __syncthreads();
      small_gemm(W, 0, C, 1, T, k);  // T = S0 N'
      __syncthreads();
      for (int e = t; e < k * k; e += blockDim.x) W[e] = st->M[e];
      __syncthreads();
      small_gemm(W, 0, T, 0, st->Sinit, k);
      break;
    }
    case EPI_BUG_S: {
      const int k = a;
      for (int e = t; e < k * k; e += blockDim.x) {
        int i = e % k, j = e / k;
        E.S[i + j * E.ld_s] = st->Sinit[e] + C[j + i * k];
      }
      break;
    }
    case EPI_RA_M:
    case EPI_RA_N: {
      const int r = a, k2 = 2 * r;
      double* G = (E.kind == EPI_RA_M) ? st->M : st->N;
      for (int e = t; e < k2 * r; e += blockDim.x) {
        int i = e % k2, j = e / k2;
        G[e] = (i < r) ? (i == j ? 1.0 : 0.0) : C[(i - r) + j * r];
      }
      if (E.kind == EPI_RA_M) break;
      __syncthreads();
      double* T = scr;  // M * S0, 2r x r
      for (int e = t; e < k2 * r; e += blockDim.x) {
        int i = e % k2, j = e / k2;
        double s = 0.0;
        for (int l = 0; l < r; ++l) s += st->M[i + l * k2] * E.S[l + j * E.ld_s];
        T[e] = s;
      }
      __syncthreads();
      for (int e = t; e < k2 * k2; e += blockDim.x) {
        int i = e % k2, j = e / k2;
        double s = 0.0;
        for (int l = 0; l < r; ++l) s += T[i + l * k2] * st->N[j + l * k2];
        st->Sinit[e] = s;
      }
      break;
    }
    case EPI_COPYLTU: {
      for (int e = t; e < a * a; e += blockDim.x) {
        const int i = e % a, j = e / a;
        const int p = i >= j ? i : j, q = i >= j ? j : i;  // the lower-triangle entry (p >= q)
        E.dst[e] = (E.S ? E.S[p + q * E.ld_s] : 0.0) - C[p + q * a];
      }
      break;
    }
    case EPI_STORE: {
      for (int e = t; e < a * b; e += blockDim.x) st->Ctmp[e] = C[e];
      break;
    }
    case EPI_COPY: {
      const int ld = E.ld_dst > 0 ? E.ld_dst : (E.transpose ? b : a);
      for (int e = t; e < a * b; e += blockDim.x) {
        const int i = e % a, j = e / a;
        if (E.transpose)
          E.dst[j + i * ld] = C[e];
        else
          E.dst[i + j * ld] = C[e];
      }
      break;
    }
    case EPI_RA_S: {
      const int k2 = a;
      for (int e = t; e < k2 * k2; e += blockDim.x) {
        int i = e % k2, j = e / k2;
        st->Shat[e] = st->Sinit[e] + C[j + i * k2];
      }
      break;
    }
    default:
      break;
  }
}

template <int CK>
__device__ void run_epilogue(const EpiArgs& E, double* C, int a, int b, double* scr, bool writer = true) {
  if (E.kind == EPI_CHOL1 || E.kind == EPI_CHOL2 || E.kind == EPI_CHOL3) chol_epilogue<CK>(E, C, a, scr, writer);
  else plain_epilogue(E, C, a, b, scr);
}

// Partial sums of the per-workgroup reductions: workgroup b of k_reduce sums
// entries [64b, 64b + 64) of the nb partials (each a*b doubles) into C; thread
// (entry e, quarter g) adds partials g, g+4, ... with 16 loads in flight, and the
// four quarters are combined in a fixed order (deterministic).
__device__ __forceinline__ void reduce_entries(const double* __restrict__ gpart, int nb, int ab,
                                               double* __restrict__ C, int bid) {
  __shared__ double q4[4][64];
  const int el = threadIdx.x & 63, g = threadIdx.x >> 6;
  const int e = bid * 64 + el;
  double s = 0.0;
  if (e < ab) {
    int k = g;
    for (; k + 4 * 15 < nb; k += 4 * 16) {
      double v[16];
#pragma unroll
      for (int u = 0; u < 16; ++u) v[u] = gpart[(int64_t)(k + 4 * u) * ab + e];
#pragma unroll
      for (int u = 0; u < 16; ++u) s += v[u];
    }
    for (; k < nb; k += 4) s += gpart[(int64_t)k * ab + e];
  }
  q4[g][el] = s;
  __syncthreads();
  if (g == 0 && e < ab) C[e] = ((q4[0][el] + q4[1][el]) + q4[2][el]) + q4[3][el];
}

__global__ __launch_bounds__(kThreads) void k_reduce(const double* __restrict__ gpart, int nb, int ab,
                                                     double* __restrict__ C) {
  reduce_entries(gpart, nb, ab, C, blockIdx.x);
}

struct ReduceLaunch {
  const double* gpart;
  int nb, ab;
  double* C;
};
__global__ __launch_bounds__(kThreads) void k_reduce_batch(const unsigned char* __restrict__ tab,
                                                           const int* __restrict__ start, int count) {
  const int b = blockIdx.x;
  const int i = batch_member(start, count, b);
  const ReduceLaunch& R = *reinterpret_cast<const ReduceLaunch*>(tab + (size_t)start[count + 1 + i] * kRecArgBytes);
  reduce_entries(R.gpart, R.nb, R.ab, R.C, b - start[i]);
}

// One workgroup: C (a x b, from k_reduce) into LDS, then the epilogue.  (A
// variant where the last k_reduce workgroup ran the epilogue after a
// device-scope release/acquire measured slower than this second launch.)
template <int CK>
__device__ __forceinline__ void epilogue_body(const EpiArgs& E, const double* __restrict__ Cg, int a, int b) {
  extern __shared__ double lds[];
  double* C = lds;
  double* scr = lds + a * b;
  for (int e = threadIdx.x; e < a * b; e += kThreads) C[e] = Cg[e];
  __syncthreads();
  run_epilogue<CK>(E, C, a, b, scr);
}
template <int CK>
__global__ __launch_bounds__(kThreads) void k_epilogue(EpiArgs E, const double* __restrict__ Cg, int a, int b) {
  epilogue_body<CK>(E, Cg, a, b);
}

struct EpiLaunch {
  EpiArgs E;
  const double* Cg;
  int a, b;
};
template <int CK>
__global__ __launch_bounds__(kThreads) void k_epilogue_batch(const unsigned char* __restrict__ tab,
                                                             const int* __restrict__ start, int count) {
  const int i = batch_member(start, count, blockIdx.x);
  const EpiLaunch& L = *reinterpret_cast<const EpiLaunch*>(tab + (size_t)start[count + 1 + i] * kRecArgBytes);
  epilogue_body<CK>(L.E, L.Cg, L.a, L.b);
}


// ----------------------------------------------------------------------------
// the row kernel
//   out[i, c] = (parts ? sum_s part[s][c][i] : 0) + base_sign * op(base)[i, c]
//             + xy_sign * sum_d X[i, d] * op(Y)(d, c)
// and optionally the reduction C = out' * W (W == nullptr: out' * out;
// gram_w: out' * [out | W]).
// A tile has rpb rows.  For loads and stores thread t handles row t % rpb and
// the columns 8*(t / rpb) + 0..7, so every wave reads and writes 64
// consecutive rows of one column.  The tile then goes through LDS (Xt: the X
// rows, Ot: the outputs, Wt: the W rows), where both products run on FP64
// matrix cores (16x16x4): X*Y adds into Ot in place, and the reduction
// accumulates 16x16 blocks of C in registers across tiles (block b belongs to
// wave b % 4), written once per workgroup to gpart[blockIdx.x].
// With a prologue (CK > 0), every workgroup first runs the Cholesky epilogue
// of the previous kernel's reduction on its own LDS copy of C, and Y is that
// epilogue's R^{-1}.
// ----------------------------------------------------------------------------

struct RowsPlan {
  int tpr, rpb;                // threads per row, rows per tile
  int ri4, ro16, rw16;         // padded widths
  int rg16;                    // the out' * out block columns of a gram_w reduction (else 0)
  int ldy, ldxt, ldot, ldwt;   // LDS leading dimensions (doubles; odd against bank conflicts)
  int nxy, nred;               // 16x16 blocks of X*Y per tile, of the reduction
  int ys_off, xt_off, ot_off, wt_off;
  size_t lds_doubles;
};

// threads per row: enough for r_out in groups of 8, and more (fewer rows per
// tile) while the LDS tile would exceed 96 KB (e.g. a narrow output reduced
// against a wide W)
__host__ __device__ inline RowsPlan rows_plan(int ro, int ri, int rw, bool hasX, bool hasW, bool reduce,
                                              bool gramw = false) {
  RowsPlan p;
  p.ri4 = (ri + 3) & ~3;
  p.ro16 = (ro + 15) & ~15;
  p.rw16 = hasW ? ((rw + 15) & ~15) : p.ro16;
  p.rg16 = (hasW && gramw) ? p.ro16 : 0;
  p.ldy = p.ro16 + 1;
  p.ldxt = p.ri4 + 1;
  p.ldot = p.ro16 + 1;
  p.ldwt = p.rw16 + 1;
  int tpr = 1;
  while (8 * tpr < ro) tpr *= 2;
  for (;;) {
    p.tpr = tpr;
    p.rpb = kThreads / tpr;
    int off = 0;
    p.ys_off = off;
    if (hasX) off += p.ri4 * p.ldy;
    p.xt_off = off;
    if (hasX) off += p.rpb * p.ldxt;
    p.ot_off = off;
    if (hasX || reduce) off += p.rpb * p.ldot;
    p.wt_off = off;
    if (hasW && reduce) off += p.rpb * p.ldwt;
    p.lds_doubles = (size_t)off;
    if (p.lds_doubles * sizeof(double) <= 96 * 1024 || tpr >= 16) break;
    tpr *= 2;
  }
  p.nxy = hasX ? (p.rpb / 16) * (p.ro16 / 16) : 0;
  p.nred = reduce ? (p.ro16 / 16) * ((p.rg16 + p.rw16) / 16) : 0;
  return p;
}

// CK > 0: with the prologue of RowArgs::pre (Cholesky variant CK).  bid / nblk:
// this workgroup's index among the nblk of the launch (of its member, batched).
// The arguments are taken by value: bound to a reference into the kernel's
// argument segment, the Cholesky variants spill ~470 bytes per lane to scratch.
// LEAN: fewer loads in flight per thread (2 splits of the partials, 4 X values
// ahead of the Y staging), so that the body fits 256 registers and two
// workgroups share a CU; the arithmetic, and so the result, is the same.
template <typename PT, int NRB, int CK = 0, bool LEAN = false>
__device__ __forceinline__ void rows_body(const RowArgs<PT> A, int bid, int nblk) {
  extern __shared__ double lds[];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int ro = A.r_out, ri = A.r_in;
  const bool hasX = A.X != nullptr;
  const bool hasW = A.W != nullptr;
  const bool reduce = A.reduce != 0;
  const int rw = hasW ? A.rw : ro;
  const RowsPlan p = rows_plan(ro, ri, rw, hasX, hasW, reduce, A.gram_w != 0);
  const int rg = p.rg16 ? ro : 0;  // columns of C before the W part
  const int rpb = p.rpb, tpr = p.tpr;
  const int lrow = t % rpb, cg = t / rpb;
  double* Ys = lds + p.ys_off;
  double* Xt = lds + p.xt_off;
  double* Ot = lds + p.ot_off;
  double* Wt = (hasW && reduce) ? lds + p.wt_off : Ot;
  const int ldwt = (hasW && reduce) ? p.ldwt : p.ldot;
  const bool use_tile = hasX || reduce;
  const int lr = lane & 15, lk = lane >> 4;  // matrix-core lane coordinates

  f64x4_t racc[NRB];
#pragma unroll
  for (int b = 0; b < NRB; ++b) racc[b] = f64x4_t{0.0, 0.0, 0.0, 0.0};

  bool ys_staged = !hasX;
  if constexpr (CK > 0) {
    // the previous reduction's Cholesky epilogue, in the LDS beyond the tile
    const int pa = A.pre_a, pb = A.pre_b;
    double* Cp = lds + p.lds_doubles;
    double* scr = Cp + pa * pb;
    for (int e = t; e < pa * pb; e += kThreads) Cp[e] = A.pre_C[e];
    __syncthreads();
    run_epilogue<CK>(A.pre, Cp, pa, pb, scr, bid == 0);
    __syncthreads();
    // Y = its R^{-1} (pa x pa), staged as below; the tile barrier publishes it
    const double* Ri = scr + pa * pa;
    for (int e = t; e < p.ri4 * p.ro16; e += kThreads) {
      const int c = e % p.ro16, d = e / p.ro16;
      Ys[d * p.ldy + c] = (c < ro && d < ri) ? A.xy_sign * Ri[d + c * pa] : 0.0;
    }
    ys_staged = true;
  }
  const int64_t ntiles = (A.rows + rpb - 1) / rpb;
  for (int64_t tile = bid; tile < ntiles; tile += nblk) {
    const int64_t row0 = tile * rpb;
    const int nrows = (int)min((int64_t)rpb, A.rows - row0);
    const int64_t i = row0 + lrow;
    const bool ok = lrow < nrows;
    double v[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) v[q] = 0.0;
    if (ok) {
      if (A.parts) {
        // the partials were written by the previous launch, mostly into other
        // XCDs' L2: every load is a fabric round trip, so the loads of all 8
        // columns and of PC splits at a time are issued together (addresses
        // clamped into the array, the extra values discarded), then summed in
        // split order
        constexpr int PC = LEAN ? 2 : (sizeof(PT) == 4 ? 8 : 4) / (NRB >= 16 ? 2 : 1);  // (NRB 16 has no registers to spare)
        const int64_t sstride = (int64_t)A.rb * A.rows;
        const int cmax = ro - 1;
        for (int sp0 = 0; sp0 < A.nsplit; sp0 += PC) {
          PT w[8][PC];
#pragma unroll
          for (int q = 0; q < 8; ++q) {
            const int c = min(8 * cg + q, cmax);
#pragma unroll
            for (int u = 0; u < PC; ++u) {
              const int sp = min(sp0 + u, A.nsplit - 1);
              w[q][u] = A.parts[sp * sstride + (int64_t)c * A.rows + i];
            }
          }
#pragma unroll
          for (int q = 0; q < 8; ++q)
#pragma unroll
            for (int u = 0; u < PC; ++u)
              if (sp0 + u < A.nsplit) v[q] += (double)w[q][u];
        }
        if (A.sum_out) {
#pragma unroll
          for (int q = 0; q < 8; ++q) {
            const int c = 8 * cg + q;
            if (c < ro) A.sum_out[i + c * A.ld_sum] = v[q];
          }
        }
      }
      if (A.base) {
        if (A.st_d) {
          // neighbours of row i (with the periodic wrap when asked for)
          const int64_t n = A.rows;
          const bool hasdn = i + 1 < n || A.st_periodic;
          const bool hasup = i > 0 || A.st_periodic;
          const int64_t idn = i + 1 < n ? i + 1 : 0, iup = i > 0 ? i - 1 : n - 1;
          const double dd = A.st_d[i];
          const double edn = hasdn ? A.st_e[i] : 0.0, eup = hasup ? A.st_e[iup] : 0.0;
#pragma unroll
          for (int q = 0; q < 8; ++q) {
            const int c = 8 * cg + q;
            if (c < ro) {
              const double* col = A.base + c * A.ld_base;
              double w = dd * col[i];
              if (hasdn) w += edn * col[idn];
              if (hasup) w += eup * col[iup];
              v[q] += A.base_sign * w;
            }
          }
        } else {
#pragma unroll
          for (int q = 0; q < 8; ++q) {
            const int c = 8 * cg + q;
            if (c < ro) v[q] += A.base_sign * A.base[i + c * A.ld_base];
          }
        }
      }
    }
    // the first XR of this thread's X values, loaded before Y is staged so that
    // both loads are in flight together
    constexpr int XR = LEAN ? 4 : 16;
    double xr[XR];
    if (hasX) {
#pragma unroll
      for (int u = 0; u < XR; ++u) {
        const int d = cg + u * tpr;
        xr[u] = (ok && d < ri) ? A.X[i + d * A.ldx] : 0.0;
      }
    }
    if (!ys_staged) {
      // xy_sign * op(Y) into LDS once, as Ys[d][c] (ri4 x ro16, zero padded);
      // the barrier below publishes it
      for (int e = t; e < p.ri4 * p.ro16; e += kThreads) {
        const int c = e % p.ro16, d = e / p.ro16;
        double y = 0.0;
        if (c < ro && d < ri) y = A.transY ? A.Y[c + d * A.ldy] : A.Y[d + c * A.ldy];
        Ys[d * p.ldy + c] = A.xy_sign * y;
      }
      ys_staged = true;
    }
    if (use_tile) {
      // the tile into LDS: partial outputs, X rows, W rows (zero beyond the data)
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const int c = 8 * cg + q;
        if (c < p.ro16) Ot[lrow * p.ldot + c] = (ok && c < ro) ? v[q] : 0.0;
      }
      for (int c = 8 * tpr + cg; c < p.ro16; c += tpr) Ot[lrow * p.ldot + c] = 0.0;
      if (hasX) {
#pragma unroll
        for (int u = 0; u < XR; ++u) {
          const int d = cg + u * tpr;
          if (d < p.ri4) Xt[lrow * p.ldxt + d] = xr[u];
        }
        for (int d = cg + XR * tpr; d < p.ri4; d += tpr) Xt[lrow * p.ldxt + d] = (ok && d < ri) ? A.X[i + d * A.ldx] : 0.0;
      }
      if (hasW && reduce)
        for (int c = cg; c < p.rw16; c += tpr) Wt[lrow * p.ldwt + c] = (ok && c < rw) ? A.W[i + c * A.ldw] : 0.0;
      __syncthreads();
      if (hasX) {
        // Ot += Xt * Ys, one 16 x 16 output block per wave at a time
        const int nrb = rpb / 16;
        for (int blk = wave; blk < p.nxy; blk += 4) {
          const int r0 = (blk % nrb) * 16, c0 = (blk / nrb) * 16;
          f64x4_t acc;
#pragma unroll
          for (int u = 0; u < 4; ++u) acc[u] = Ot[(r0 + 4 * u + lk) * p.ldot + c0 + lr];
          for (int d0 = 0; d0 < p.ri4; d0 += 4) {
            const double a = Xt[(r0 + lr) * p.ldxt + d0 + lk];
            const double b = Ys[(d0 + lk) * p.ldy + c0 + lr];
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, acc, 0, 0, 0);
          }
#pragma unroll
          for (int u = 0; u < 4; ++u) Ot[(r0 + 4 * u + lk) * p.ldot + c0 + lr] = acc[u];
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          const int c = 8 * cg + q;
          if (c < ro) v[q] = Ot[lrow * p.ldot + c];
        }
      }
    }
    if (ok) {
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const int c = 8 * cg + q;
        if (c < ro) {
          if (A.out) A.out[i + c * A.ldo] = v[q];
          if (A.out2) A.out2[i + c * A.ldo2] = v[q];
          if (A.pk_f64) A.pk_f64[i * A.pk_cols + c] = v[q];
          if (A.pk_f32) A.pk_f32[pk_f32_offset(A.pk_layout, i, c, A.pk_cols)] = (float)v[q];
          if (A.pk_hi) {
            uint32_t hi, lo;
            split_bf16((float)v[q], hi, lo);
            const int64_t off = pk_offset(A.pk_layout, i, c, A.pk_cols);
            A.pk_hi[off] = (uint16_t)hi;
            A.pk_lo[off] = (uint16_t)lo;
          }
        }
      }
      // zero the packed columns beyond the current rank
      for (int c = ro + cg; c < A.pk_cols; c += tpr) {
        if (A.pk_f64) A.pk_f64[i * A.pk_cols + c] = 0.0;
        if (A.pk_f32) A.pk_f32[pk_f32_offset(A.pk_layout, i, c, A.pk_cols)] = 0.0f;
        if (A.pk_hi) {
          const int64_t off = pk_offset(A.pk_layout, i, c, A.pk_cols);
          A.pk_hi[off] = 0;
          A.pk_lo[off] = 0;
        }
      }
    }
    if (reduce) {
      // C += Ot' * Wt over the tile's rows (rows past the data are zero); with
      // gram_w the first rg16 block columns are Ot' * Ot
      const int nbi = p.ro16 / 16;
#pragma unroll
      for (int b = 0; b < NRB; ++b) {
        const int blk = wave + 4 * b;
        if (blk < p.nred) {
          const int c0 = (blk % nbi) * 16, j0 = (blk / nbi) * 16;
          const double* Bt = j0 < p.rg16 ? Ot + j0 : Wt + (j0 - p.rg16);
          const int ldb = j0 < p.rg16 ? p.ldot : ldwt;
          for (int k0 = 0; k0 < rpb; k0 += 4) {
            const double a = Ot[(k0 + lk) * p.ldot + c0 + lr];
            const double bb = Bt[(k0 + lk) * ldb + lr];
            racc[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, bb, racc[b], 0, 0, 0);
          }
        }
      }
    }
    if (use_tile) __syncthreads();  // the next tile overwrites the LDS tile
  }
  if (!reduce) return;
  double* gp = A.gpart + (int64_t)bid * ro * (rg + rw);
  const int nbi = p.ro16 / 16;
#pragma unroll
  for (int b = 0; b < NRB; ++b) {
    const int blk = wave + 4 * b;
    if (blk < p.nred) {
      const int c0 = (blk % nbi) * 16, j0 = (blk / nbi) * 16;
      const bool og = j0 < p.rg16;
      const int jl = (og ? j0 : j0 - p.rg16) + lr;  // column within its part
      const int cj = og ? jl : rg + jl;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int ci = c0 + 4 * u + lk;
        if (ci < ro && jl < (og ? ro : rw)) gp[ci + cj * ro] = racc[b][u];
      }
    }
  }
}

template <typename PT, int NRB, int CK = 0>
__global__ __launch_bounds__(kThreads) void k_rows(RowArgs<PT> A) {
  rows_body<PT, NRB, CK>(A, blockIdx.x, gridDim.x);
}

// The batched form: merged launches cover many narrow members with one tile per
// workgroup, so latency hiding matters more than loads in flight per thread:
// the lean body at two workgroups per CU for NRB <= 2 without a prologue.
template <typename PT, int NRB, int CK>
__global__ __launch_bounds__(kThreads, (NRB <= 2 && CK == 0) ? 2 : 1) void k_rows_batch(
    const unsigned char* __restrict__ tab, const int* __restrict__ start, int count) {
  const int b = blockIdx.x;
  const int i = batch_member(start, count, b);
  const RowArgs<PT>& A = *reinterpret_cast<const RowArgs<PT>*>(tab + (size_t)start[count + 1 + i] * kRecArgBytes);
  rows_body<PT, NRB, CK, (NRB <= 2 && CK == 0)>(A, b - start[i], start[i + 1] - start[i]);
}

template <typename PT>
hipError_t launch_rows(RowArgs<PT> A, hipStream_t st) {
  const bool hasW = A.W != nullptr;
  const int rw = hasW ? A.rw : A.r_out;
  if (A.r_out < 1 || A.r_out > kMaxAug || rw < 1 || rw > kMaxAug || A.r_in < 0 || A.r_in > kMaxAug)
    return hipErrorInvalidValue;
  if (A.X && A.r_in < 1) return hipErrorInvalidValue;
  if (A.gram_w && (!hasW || !A.reduce)) return hipErrorInvalidValue;
  const RowsPlan p = rows_plan(A.r_out, A.r_in, rw, A.X != nullptr, hasW, A.reduce != 0, A.gram_w != 0);
  if (p.tpr > 16) return hipErrorInvalidValue;
  A.tr = p.rpb;
  const int rc = (A.gram_w ? A.r_out : 0) + rw;  // columns of C
  if (A.epi.stilde && (A.epi.kind != EPI_CHOL2 || !A.gram_w || rw != A.r_out)) return hipErrorInvalidValue;
  const bool pre = A.pre.kind != EPI_NONE;
  size_t pre_doubles = 0;
  if (pre) {
    if ((A.pre.kind != EPI_CHOL1 && A.pre.kind != EPI_CHOL2) || !A.pre_C || A.pre_a < 1 || A.pre_a > 32 ||
        A.pre_a != A.r_in || A.pre_a != A.r_out || !A.X || A.transY ||
        (A.pre_b != A.pre_a && A.pre_b != 2 * A.pre_a) || (A.pre.stilde && A.pre_b != 2 * A.pre_a))
      return hipErrorInvalidValue;
    pre_doubles = (size_t)A.pre_a * A.pre_b + epi_scratch_doubles(A.pre.kind, A.pre_a, A.pre_b);
  }
  const size_t lds = sizeof(double) * (p.lds_doubles + pre_doubles);
  const size_t epi_lds = sizeof(double) * ((size_t)A.r_out * rc + epi_scratch_doubles(A.epi.kind, A.r_out, rc));
  // room for the static shared variables (the Cholesky row buffers: 12.3 KB)
  if (lds > 147 * 1024 || epi_lds > 147 * 1024) return hipErrorInvalidValue;
  const int64_t ntiles = (A.rows + p.rpb - 1) / p.rpb;
  int grid = (int)(ntiles < A.max_blocks ? ntiles : A.max_blocks);
  if (grid < 1) grid = 1;
  const int nrb = (p.nred + 3) / 4;
  int nrbv = 0, ckv = 0;
  if (pre) {
    if (!std::is_same<PT, double>::value || nrb > 2) return hipErrorInvalidValue;
    ckv = A.pre_a <= 16 ? 16 : 32;
    nrbv = nrb <= 1 ? 1 : 2;
  } else {
    nrbv = nrb <= 1 ? 1 : (nrb <= 2 ? 2 : (nrb <= 4 ? 4 : (nrb <= 8 ? 8 : 16)));
  }
  const int kid = std::is_same<PT, double>::value ? KID_ROWS_D : KID_ROWS_F;
  if (!record_launch(kid, nrbv * 100 + ckv, (unsigned)grid, kThreads, lds, A)) {
    const dim3 g(grid), b(kThreads);
    switch (nrbv * 100 + ckv) {
      case 116: hipLaunchKernelGGL((k_rows<PT, 1, 16>), g, b, lds, st, A); break;
      case 216: hipLaunchKernelGGL((k_rows<PT, 2, 16>), g, b, lds, st, A); break;
      case 132: hipLaunchKernelGGL((k_rows<PT, 1, 32>), g, b, lds, st, A); break;
      case 232: hipLaunchKernelGGL((k_rows<PT, 2, 32>), g, b, lds, st, A); break;
      case 100: hipLaunchKernelGGL((k_rows<PT, 1>), g, b, lds, st, A); break;
      case 200: hipLaunchKernelGGL((k_rows<PT, 2>), g, b, lds, st, A); break;
      case 400: hipLaunchKernelGGL((k_rows<PT, 4>), g, b, lds, st, A); break;
      case 800: hipLaunchKernelGGL((k_rows<PT, 8>), g, b, lds, st, A); break;
      default: hipLaunchKernelGGL((k_rows<PT, 16>), g, b, lds, st, A); break;
    }
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || !A.reduce) return e;
  const int ab = A.r_out * rc;
  double* Cr = A.epi.small->Cred;
  const ReduceLaunch R{(const double*)A.gpart, grid, ab, Cr};
  if (!record_launch(KID_REDUCE, 0, (unsigned)((ab + 63) / 64), kThreads, 0, R))
    hipLaunchKernelGGL(k_reduce, dim3((ab + 63) / 64), dim3(kThreads), 0, st, R.gpart, R.nb, R.ab, R.C);
  e = hipGetLastError();
  if (e != hipSuccess || A.epi.kind == EPI_NONE || A.defer_epi) return e;
  const bool chol = A.epi.kind == EPI_CHOL1 || A.epi.kind == EPI_CHOL2 || A.epi.kind == EPI_CHOL3;
  const int ck = (chol && A.r_out <= 16) ? 16 : ((chol && A.r_out <= 32) ? 32 : 64);
  const EpiLaunch L{A.epi, (const double*)Cr, A.r_out, rc};
  if (!record_launch(KID_EPILOGUE, ck, 1, kThreads, epi_lds, L)) {
    if (ck == 16)
      hipLaunchKernelGGL(k_epilogue<16>, dim3(1), dim3(kThreads), epi_lds, st, L.E, L.Cg, L.a, L.b);
    else if (ck == 32)
      hipLaunchKernelGGL(k_epilogue<32>, dim3(1), dim3(kThreads), epi_lds, st, L.E, L.Cg, L.a, L.b);
    else
      hipLaunchKernelGGL(k_epilogue<64>, dim3(1), dim3(kThreads), epi_lds, st, L.E, L.Cg, L.a, L.b);
  }
  return hipGetLastError();
}

template hipError_t launch_rows<double>(RowArgs<double>, hipStream_t);
template hipError_t launch_rows<float>(RowArgs<float>, hipStream_t);

// ----------------------------------------------------------------------------
// A whole CholeskyQR2 (or shifted CholeskyQR3) of an n x r matrix, r <= 32, in one
// launch: the formation of the matrix (as k_rows: split partials, a base, X op(Y)),
// the Gram matrices and their factors, the applications of R^{-1}, the packed
// copy and the reduction against W.  At these sizes every step is far below the
// cost of a launch (4 to 5 us each, and each kernel starts by fetching what the one
// before wrote): the chain rows - reduce - rows - reduce - rows took 52 us for 256 x 8 and
// 68 us for 2000 x 21, this launch 27 and 50 us; shifted CholeskyQR3 of 4096 x 32 went
// from 113 to 87 us, of 1000 x 15 from 84 to 38 us (8 us of each pass are the serial
// 32-pivot Cholesky, 4 us at r <= 16).
//
// G <= 64 workgroups keep their rows in LDS from start to end.  A Gram matrix is
// summed over them through memory: every workgroup writes its part with
// write-through stores, waits for them, adds to a counter and waits until all
// have (2 us measured); then each sums all parts in workgroup order (the same bits
// everywhere, whatever the timing) and factors redundantly, as the prologues of
// k_rows do.  One workgroup more, without rows, forms what the step's later kernels
// need (Rtot, S~, the reduction against W) while the others apply R^{-1} and store.
// The workgroups take one CU each and are resident at once on an idle device; with
// other kernels running they become so when those end.  A wait is bounded all
// the same (kQrSpins polls, then FLAG_TIMEOUT and the kernel runs to its end).  The last
// workgroup out resets the counters, so that a captured launch can be replayed.  A
// matrix that one workgroup's LDS holds is done by one alone.
// ----------------------------------------------------------------------------

constexpr int kQrThreads = kThreads, kQrMaxBlocks = 64, kQrDirect = 20, kQrSlots = 4, kQrSpins = 1 << 21;

struct QrShape {
  int blocks, tr;  // workgroups with rows, rows of each (a multiple of 16)
};
// CK = 16 or 32 padded columns
__host__ __device__ inline int qr_max_tile(int ck) { return ck == 16 ? 768 : 256; }
__host__ __device__ inline QrShape qr_shape(int64_t rows, int ck) {
  const int alone = ck == 16 ? 512 : 256, tile = ck == 16 ? 256 : 128;
  if (rows <= alone) return {1, (int)((rows + 15) / 16 * 16)};
  int tr = tile;
  while ((rows + tr - 1) / tr > kQrMaxBlocks) tr += 16;
  return {(int)((rows + tr - 1) / tr), tr};
}
// Two passes over more than 6144 rows stay with the separate kernels at r > 16: exchanging the
// parts of 48 workgroups and more costs what the launches did (16384 x 32: 83 us against
// 85; 2000 x 21: 50 against 68), three passes gain at every size (4096 x 32: 87 against 113).
bool qr_fits(int64_t rows, int r, int passes) {
  if (r < 1 || r > 32) return false;
  const int ck = r <= 16 ? 16 : 32;
  if (passes == 2 && ck == 32 && rows > 6144) return false;
  return rows <= (int64_t)kQrMaxBlocks * qr_max_tile(ck);
}
__host__ __device__ inline int qr_lds_doubles(int tr, int ck) { return tr * (ck + 1) + 4 * ck * (ck + 1) + (2 + 3 + 1) * ck * ck; }

template <typename PT, int CK>
__global__ __launch_bounds__(kQrThreads) void k_qr(QrArgs<PT> Q) {
  extern __shared__ double lds[];
  __shared__ int s_nd;
  constexpr int LD = CK + 1, NT = CK / 16, KS = CK / 4, NW = kQrThreads / 64;
  const RowArgs<PT>& A = Q.form;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, lr = lane & 15, lk = lane >> 4;
  const int r = A.r_out, tr = Q.tr, G = Q.blocks, bid = blockIdx.x;
  const bool rows_wg = bid < G;             // has rows
  const bool scribe = G == 1 || bid == G;   // writes the small results
  const int64_t row0 = (int64_t)bid * tr;
  const int nrows = rows_wg ? (int)min((int64_t)tr, A.rows - row0) : 0;
  double* kt = lds;                 // the tile, kt[row * LD + column], zero beyond the data
  double* red = kt + tr * LD;       // a wave's partial reductions [i + LD j]; operands [k * LD + n]
  double* C = red + NW * CK * LD;   // r x 2r
  double* scr = C + 2 * CK * CK;    // R, R^{-1}, Rtot
  double* Rr = scr + 3 * CK * CK;   // the factor on the right of the next pass
  const int strips = rows_wg ? tr / 16 : 0;  // of 16 rows, wave w taking w, w + NW, ...

  // rows of X (n x r, ld) in operand layout for four of the wave's strips from number si on:
  // lane lr = row, 4 j + lk = column
  auto load_x = [&](double (&x)[4][KS], int si) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int lrow = (wave + NW * (si + q)) * 16 + lr;
#pragma unroll
      for (int j = 0; j < KS; ++j) {
        const int d = 4 * j + lk;
        x[q][j] = lrow < nrows && d < r ? A.X[row0 + lrow + d * A.ldx] : 0.0;
      }
    }
  };
  // rows of W for the reduction: lane lr = column, 4 j + lk = row
  auto load_w = [&](double (&w)[4][4][NT], int si) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int n = 0; n < NT; ++n) {
          const int lrow = (wave + NW * (si + q)) * 16 + 4 * j + lk;
          w[q][j][n] = lrow < nrows && 16 * n + lr < r ? Q.W[row0 + lrow + (16 * n + lr) * Q.ldw] : 0.0;
        }
  };

  // ---- the matrix: split partials + base + X op(Y)
  if (rows_wg) {
    double x[4][KS];
    if (A.X) {
      load_x(x, 0);
      for (int e = t; e < CK * CK; e += kQrThreads) {
        const int d = e % CK, c = e / CK;  // red[d * LD + c] = op(Y)(d, c)
        red[d * LD + c] = d < r && c < r ? (A.transY ? A.Y[c + d * A.ldy] : A.Y[d + c * A.ldy]) : 0.0;
      }
    }
    constexpr int U = CK / NW, B = 2;  // columns of a wave, blocks of 64 rows, loaded together
    const int64_t ss = (int64_t)A.rb * A.rows;
    for (int l0 = lane; l0 < tr; l0 += 64 * B) {
      double v[B][U];
      int64_t i[B];
#pragma unroll
      for (int k = 0; k < B; ++k) {
        i[k] = row0 + (l0 + 64 * k < nrows ? l0 + 64 * k : 0);
#pragma unroll
        for (int u = 0; u < U; ++u) v[k][u] = 0.0;
      }
      if (A.parts) {
        for (int sp = 0; sp < A.nsplit; sp += 4) {
          PT w[B][U][4];
#pragma unroll
          for (int k = 0; k < B; ++k)
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
              for (int q = 0; q < 4; ++q)
                w[k][u][q] = A.parts[min(sp + q, A.nsplit - 1) * ss + (int64_t)min(wave + NW * u, r - 1) * A.rows + i[k]];
#pragma unroll
          for (int k = 0; k < B; ++k)
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
              for (int q = 0; q < 4; ++q)
                if (sp + q < A.nsplit) v[k][u] += (double)w[k][u][q];
        }
      }
      if (A.base) {
        double w[B][U];
#pragma unroll
        for (int k = 0; k < B; ++k)
#pragma unroll
          for (int u = 0; u < U; ++u) w[k][u] = A.base[i[k] + (int64_t)min(wave + NW * u, r - 1) * A.ld_base];
#pragma unroll
        for (int k = 0; k < B; ++k)
#pragma unroll
          for (int u = 0; u < U; ++u) v[k][u] += w[k][u];
      }
#pragma unroll
      for (int k = 0; k < B; ++k)
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int c = wave + NW * u, lrow = l0 + 64 * k;
          const bool ok = c < r && lrow < nrows;
          if (A.sum_out && ok) A.sum_out[i[k] + c * A.ld_sum] = v[k][u];
          if (lrow < tr) kt[lrow * LD + c] = ok ? v[k][u] : 0.0;
        }
    }
    __syncthreads();
    if (A.X) {
      for (int si = 0; wave + NW * si < strips; si += 4) {
        if (si) load_x(x, si);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int s = wave + NW * (si + q);
          if (s < strips)
#pragma unroll
          for (int n = 0; n < NT; ++n) {
            f64x4_t acc;
#pragma unroll
            for (int u = 0; u < 4; ++u) acc[u] = kt[(s * 16 + 4 * u + lk) * LD + 16 * n + lr];
#pragma unroll
            for (int j = 0; j < KS; ++j)
              acc = __builtin_amdgcn_mfma_f64_16x16x4f64(x[q][j], red[(4 * j + lk) * LD + 16 * n + lr], acc, 0, 0, 0);
#pragma unroll
            for (int u = 0; u < 4; ++u) kt[(s * 16 + 4 * u + lk) * LD + 16 * n + lr] = acc[u];
          }
        }
      }
      __syncthreads();
    }
  }
  auto copy_out = [&](double* dst, int64_t ld) {
    for (int lrow = lane; lrow < nrows; lrow += 64)
      for (int c = wave; c < r; c += NW) dst[row0 + lrow + c * ld] = kt[lrow * LD + c];
  };
  if (A.out) copy_out(A.out, A.ldo);

  int arrived = 0;  // reductions over the workgroups so far
  // Stores this workgroup's part (r x r) of a reduction, summed over the waves: into C + at
  // if there is one workgroup, else into its place of `slot`.  sym: only the blocks
  // on and above the diagonal were formed.
  auto store_part = [&](int at, int slot, bool sym) {
    __syncthreads();
    double* gp = Q.gpart + ((int64_t)slot * G + bid) * r * r;
    for (int e = t; e < r * r; e += kQrThreads) {
      int i = e % r, j = e / r;
      if (sym && (i >> 4) > (j >> 4)) {
        const int x = i;
        i = j;
        j = x;
      }
      const int o = i + LD * j;
      double v = red[o];
#pragma unroll
      for (int w = 1; w < NW; ++w) v += red[w * CK * LD + o];
      if (G == 1) C[at + e] = v;
      else __hip_atomic_store(gp + e, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
  };
  auto to_red = [&](int m, int n, const f64x4_t& acc) {
#pragma unroll
    for (int u = 0; u < 4; ++u) red[wave * CK * LD + 16 * m + 4 * u + lk + LD * (16 * n + lr)] = acc[u];
  };
  auto gram = [&](int slot) {  // tile' tile
    f64x4_t acc[NT][NT];
#pragma unroll
    for (int m = 0; m < NT; ++m)
#pragma unroll
      for (int n = 0; n < NT; ++n) acc[m][n] = f64x4_t{0.0, 0.0, 0.0, 0.0};
    for (int s = wave; s < strips; s += NW) {
      double a[4][NT];
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int n = 0; n < NT; ++n) a[j][n] = kt[(s * 16 + 4 * j + lk) * LD + 16 * n + lr];
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int m = 0; m < NT; ++m)
#pragma unroll
          for (int n = m; n < NT; ++n) acc[m][n] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[j][m], a[j][n], acc[m][n], 0, 0, 0);
    }
#pragma unroll
    for (int m = 0; m < NT; ++m)
#pragma unroll
      for (int n = m; n < NT; ++n) to_red(m, n, acc[m][n]);
    store_part(0, slot, true);
  };
  auto cross = [&](double (&w)[4][4][NT], int at, int slot) {  // tile' W; w: load_w(w, 0)
    f64x4_t acc[NT][NT];
#pragma unroll
    for (int m = 0; m < NT; ++m)
#pragma unroll
      for (int n = 0; n < NT; ++n) acc[m][n] = f64x4_t{0.0, 0.0, 0.0, 0.0};
    for (int si = 0; wave + NW * si < strips; si += 4) {
      if (si) load_w(w, si);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int s = wave + NW * (si + q);
        if (s < strips)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int m = 0; m < NT; ++m) {
            const double a = kt[(s * 16 + 4 * j + lk) * LD + 16 * m + lr];
#pragma unroll
            for (int n = 0; n < NT; ++n) acc[m][n] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, w[q][j][n], acc[m][n], 0, 0, 0);
          }
      }
    }
#pragma unroll
    for (int m = 0; m < NT; ++m)
#pragma unroll
      for (int n = 0; n < NT; ++n) to_red(m, n, acc[m][n]);
    store_part(at, slot, false);
  };
  // the stores of this workgroup's parts are done; all workgroups' are when wait returns
  auto arrive = [&]() {
    if (G == 1) return;
    ++arrived;
    if (!rows_wg) return;
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (t == 0) __hip_atomic_fetch_add(Q.sync, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  auto wait = [&]() {
    if (G == 1) return;
    if (t == 0) {
      int n = 0;
      while (__hip_atomic_load(Q.sync, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < arrived * G && ++n < kQrSpins)
        __builtin_amdgcn_s_sleep(1);
      if (n >= kQrSpins) atomicOr(Q.flags, FLAG_TIMEOUT);
    }
    __syncthreads();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  };
  // C + at <- the sum of all workgroups' parts, G <= kQrDirect: every workgroup adds them up
  auto sum = [&](int at, int slot) {
    const double* gp = Q.gpart + (int64_t)slot * G * r * r;
    constexpr int E = CK * CK / kQrThreads;  // entries of a thread
    double s[E];
#pragma unroll
    for (int q = 0; q < E; ++q) s[q] = 0.0;
    for (int g = 0; g < G; g += 8) {  // 8 workgroups' entries in flight together
      double v[8][E];
#pragma unroll
      for (int u = 0; u < 8; ++u)
#pragma unroll
        for (int q = 0; q < E; ++q)
          v[u][q] = gp[(int64_t)min(g + u, G - 1) * r * r + min(t + kQrThreads * q, r * r - 1)];
#pragma unroll
      for (int u = 0; u < 8; ++u)
#pragma unroll
        for (int q = 0; q < E; ++q) s[q] += g + u < G ? v[u][q] : 0.0;
    }
#pragma unroll
    for (int q = 0; q < E; ++q)
      if (t + kQrThreads * q < r * r) C[at + t + kQrThreads * q] = s[q];
    __syncthreads();
  };
  // above that (the parts are 8 KB each at r = 32, and reading 64 of them takes one CU
  // 11 us) a workgroup adds up its share of the entries, thread (entry, quarter) in
  // workgroup order, and the sums are exchanged like the parts
  auto share = [&](int slot, int nslots) {
    const int n = nslots * r * r, len = (n + G - 1) / G;
    const double* gp = Q.gpart + (int64_t)slot * G * r * r;
    double* gs = Q.gpart + (int64_t)(kQrSlots + slot) * G * r * r;
    const int qt = t >> 6;
    for (int x0 = 0; x0 < len; x0 += 64) {  // once, or twice for two parts of r > 25 and G < 32
      const int x = bid * len + x0 + (t & 63);
      const bool mine = rows_wg && x0 + (t & 63) < len && x < n;
      double s = 0.0;
      if (mine) {
        const double* p = gp + (int64_t)(x / (r * r)) * G * r * r + x % (r * r);
        double v[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) v[u] = p[(int64_t)min(qt * 16 + u, G - 1) * r * r];
#pragma unroll
        for (int u = 0; u < 16; ++u) s += qt * 16 + u < G ? v[u] : 0.0;
      }
      red[t] = s;
      __syncthreads();
      if (mine && qt == 0)
        __hip_atomic_store(gs + x, ((red[t] + red[64 + t]) + red[128 + t]) + red[192 + t], __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
      __syncthreads();
    }
    arrive();
    wait();
    for (int e = t; e < (scribe ? n : r * r); e += kQrThreads) C[e] = gs[e];
    __syncthreads();
  };
  // C <- [the reduction of slot | that of slot + 1 (scribe only)] over all workgroups
  auto total = [&](int slot, int nslots) {
    if (G == 1) return;
    arrive();
    wait();
    if (G > kQrDirect) {
      share(slot, nslots);
    } else {
      sum(0, slot);
      if (nslots > 1 && scribe) sum(r * r, slot + 1);
    }
  };
  // tile <- tile * R^{-1}
  auto apply = [&]() {
    const double* Ri = scr + r * r;
    for (int e = t; e < CK * CK; e += kQrThreads) {
      const int d = e % CK, c = e / CK;
      red[d * LD + c] = d < r && c < r ? Ri[d + c * r] : 0.0;
    }
    __syncthreads();
    double b[NT][KS];
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int j = 0; j < KS; ++j) b[n][j] = red[(4 * j + lk) * LD + 16 * n + lr];
    for (int s = wave; s < strips; s += NW) {
      double a[KS];
#pragma unroll
      for (int j = 0; j < KS; ++j) a[j] = kt[(s * 16 + lr) * LD + 4 * j + lk];
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        f64x4_t acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int j = 0; j < KS; ++j) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[j], b[n][j], acc, 0, 0, 0);
#pragma unroll
        for (int u = 0; u < 4; ++u) kt[(s * 16 + 4 * u + lk) * LD + 16 * n + lr] = acc[u];
      }
    }
    __syncthreads();
  };

  int slot = 0, nd = 0;
  for (int pass = 0; pass < Q.passes; ++pass) {
    // by value, from scalars: a reference into the argument segment makes the Cholesky spill
    EpiArgs E;
    E.kind = pass == 0 ? EPI_CHOL1 : pass == 1 ? EPI_CHOL2 : EPI_CHOL3;
    E.breakdown_is_error = pass == 0 ? Q.first_error : Q.later_error;
    E.small = Q.small;
    E.flags = Q.flags;
    E.shift_rows = pass == 0 ? Q.shift_rows : 0;
    E.S = pass == Q.passes - 1 ? Q.S : nullptr;
    E.ld_s = Q.ld_s;
    E.transpose = Q.transpose_s;
    E.stilde = pass == 1 ? Q.stilde : 0;
    const bool with_w = E.stilde != 0;  // C = tile' [tile | W]
    if (rows_wg) {
      if (with_w) {
        double wv[4][4][NT];
        load_w(wv, 0);
        gram(slot);
        cross(wv, r * r, slot + 1);
      } else {
        gram(slot);
      }
    }
    total(slot, with_w ? 2 : 1);
    slot += with_w ? 2 : 1;
    chol_epilogue<CK>(E, C, r, scr, scribe, pass ? Rr : nullptr, nd, &s_nd);
    __syncthreads();
    if (pass == 0) nd = s_nd;
    if (scribe)  // only Rtot needs it
      for (int e = t; e < r * r; e += kQrThreads) Rr[e] = scr[(pass ? 2 * r * r : 0) + e];
    if (rows_wg) apply();
    else __syncthreads();
  }
  // ---- Q, the reduction against W and the packed copy
  if (rows_wg) {
    if (Q.fin.kind != EPI_NONE) {
      double wv[4][4][NT];
      load_w(wv, 0);
      copy_out(Q.q, A.rows);
      cross(wv, 0, slot);
    } else {
      copy_out(Q.q, A.rows);
    }
    if (A.pk_f64) {
      for (int e = t; e < nrows * A.pk_cols; e += kQrThreads) {
        const int c = e % A.pk_cols, lrow = e / A.pk_cols;
        A.pk_f64[(row0 + lrow) * A.pk_cols + c] = c < r ? kt[lrow * LD + c] : 0.0;
      }
    } else if (A.pk_f32 || A.pk_hi) {
      // eight consecutive rows of a column lie together in every layout but pass N's FP32 one
      for (int c = wave; c < A.pk_cols; c += NW)
        for (int g8 = lane; g8 * 8 < nrows; g8 += 64) {
          float v[8];
#pragma unroll
          for (int u = 0; u < 8; ++u) v[u] = c < r ? (float)kt[(g8 * 8 + u) * LD + c] : 0.0f;
          const int64_t i = row0 + g8 * 8;
          const bool whole = g8 * 8 + 8 <= nrows;
          if (A.pk_f32) {
            if (A.pk_layout == 1 && whole) {
              f32x4_t* d = reinterpret_cast<f32x4_t*>(A.pk_f32 + pk_f32_offset(1, i, c, A.pk_cols));
              d[0] = f32x4_t{v[0], v[1], v[2], v[3]};
              d[1] = f32x4_t{v[4], v[5], v[6], v[7]};
            } else {
#pragma unroll
              for (int u = 0; u < 8; ++u)
                if (g8 * 8 + u < nrows) A.pk_f32[pk_f32_offset(A.pk_layout, i + u, c, A.pk_cols)] = v[u];
            }
          }
          if (A.pk_hi) {
            uint32_t hi[8], lo[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) split_bf16(v[u], hi[u], lo[u]);
            const int64_t off = pk_offset(A.pk_layout, i, c, A.pk_cols);
            if (whole) {
              *reinterpret_cast<u32x4_t*>(A.pk_hi + off) = u32x4_t{hi[0] | hi[1] << 16, hi[2] | hi[3] << 16,
                                                                    hi[4] | hi[5] << 16, hi[6] | hi[7] << 16};
              *reinterpret_cast<u32x4_t*>(A.pk_lo + off) = u32x4_t{lo[0] | lo[1] << 16, lo[2] | lo[3] << 16,
                                                                    lo[4] | lo[5] << 16, lo[6] | lo[7] << 16};
            } else {
#pragma unroll
              for (int u = 0; u < 8; ++u)
                if (g8 * 8 + u < nrows) {
                  A.pk_hi[off + u] = (uint16_t)hi[u];
                  A.pk_lo[off + u] = (uint16_t)lo[u];
                }
            }
          }
        }
    }
  }
  if (Q.fin.kind != EPI_NONE) {
    arrive();
    if (scribe) {
      wait();
      if (G > 1) sum(0, slot);
      EpiArgs F = Q.fin;
      plain_epilogue(F, C, r, r, scr);
    }
  }
  if (G > 1) {
    __syncthreads();
    if (t == 0 &&
        __hip_atomic_fetch_add(Q.sync + 1, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == G) {
      // G workgroups and the scribe are past their last wait
      __hip_atomic_store(Q.sync, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(Q.sync + 1, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
}

template <typename PT>
hipError_t launch_qr(QrArgs<PT> Q, hipStream_t st) {
  const int r = Q.form.r_out;
  if (!qr_fits(Q.form.rows, r, Q.passes) || Q.form.rows < 1 || (Q.passes != 2 && Q.passes != 3) || !Q.q || !Q.gpart || !Q.sync ||
      !Q.flags || (Q.form.X && (Q.form.r_in != r || !Q.form.Y)) || (Q.fin.kind != EPI_NONE && !Q.W) ||
      Q.form.st_d || Q.form.xy_sign != 1.0 || Q.form.base_sign != 1.0)
    return hipErrorInvalidValue;
  const int ck = r <= 16 ? 16 : 32;
  const QrShape s = qr_shape(Q.form.rows, ck);
  Q.tr = s.tr;
  Q.blocks = s.blocks;
  const size_t lds = sizeof(double) * qr_lds_doubles(s.tr, ck);
  const dim3 g(s.blocks > 1 ? s.blocks + 1 : 1), b(kQrThreads);
  if (ck == 16) hipLaunchKernelGGL((k_qr<PT, 16>), g, b, lds, st, Q);
  else hipLaunchKernelGGL((k_qr<PT, 32>), g, b, lds, st, Q);
  return hipGetLastError();
}
template hipError_t launch_qr<double>(QrArgs<double>, hipStream_t);
template hipError_t launch_qr<float>(QrArgs<float>, hipStream_t);

// ----------------------------------------------------------------------------
// one-sided (Hestenes) Jacobi SVD of a k x k FP64 matrix, k <= 128, in one
// workgroup, then the truncation rank (rank_adaptive_unconventional.jl:222-223)
// r1 = min{rho >= 1 : sqrt(sum_{j >= rho} sigma_j^2) <= tol}, clipped to rmax.
// Pairs are processed in round-robin (circle-method) order, all at a time.
//
// QR preconditioning (Drmac and Veselic, "New fast and accurate Jacobi SVD
// algorithm", SIAM J. Matrix Anal. Appl. 29, 2008): with S = Q R, the sweeps run on
// R' instead of S.  Its columns are much closer to orthogonal than those of a
// graded S, so the sweeps to convergence drop from 15-30 to 6-11 at k = 16..64.
// With R' J = W (J the accumulated rotations, W = Ur Sigma), S = (Q J) Sigma Ur': the
// left singular vectors are Q J and the right ones the normalised columns of W.
//
// What bounds it is the serial chain of a round: the pair's columns from LDS, three
// dot products, the rotation's square roots, the columns back, a barrier.  Eight
// lanes hold a pair (k <= 8 R: R rows of both columns a lane), so the whole of A
// is one wave per SIMD up to k = 64; the rotations of V, on which the next round does
// not wait, are applied by as many waves more, one round later.  In the QR and in Q J
// eight lanes keep one column in registers.  A k = 40 decomposition takes 181 us; with 16
// lanes a pair in runs over LDS, V on the same lanes and a barrier after every step it
// took 440.  64 merged members: 309 us up to k = 64 and 531 up to 80 (V in LDS up to 96),
// where they took 277 (k <= 32 only, one wave each) and 956.
// ----------------------------------------------------------------------------

// x from lane (lane ^ m) of its row of 16 for the DPP patterns used below
template <int CTRL>
__device__ __forceinline__ double dpp_f64(double x) {
  const uint64_t u = (uint64_t)__double_as_longlong(x);
  const int lo = __builtin_amdgcn_mov_dpp((int)(uint32_t)u, CTRL, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_mov_dpp((int)(uint32_t)(u >> 32), CTRL, 0xF, 0xF, true);
  return __longlong_as_double((long long)(((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo));
}

// Sum over aligned groups of 8 lanes, left in every lane of the group.  Quad swaps
// (quad_perm [1,0,3,2] and [2,3,0,1]) make every quad uniform; the half-row mirror
// (lane i <- 7 - i) then pairs the two quads.
__device__ __forceinline__ double group_sum8(double x) {
  x += dpp_f64<0xB1>(x);
  x += dpp_f64<0x4E>(x);
  x += dpp_f64<0x141>(x);
  return x;
}

// LDS doubles for k <= 8 R.  Column pitches in LDS are odd multiples of 8: neighbouring
// groups' columns then start 8 doubles (16 banks) apart.
constexpr int jacobi_lds_doubles(int R) {
  const int n = 8 * R, ld = n + 8;
  return (R > 12 ? 1 : 2) * n * ld + 5 * n + 2;
}

// 64 R threads (others leave at once).  R = 16: V in P.work, where the reflectors wait too
// (the others keep theirs in registers).
template <int R>
__device__ void jacobi_body(const SvdArgs P, double* lds) {
  constexpr int N = 8 * R, LD = N + 8, LV = R > 12 ? N : LD;
  const int k = P.k, ke = (k + 1) & ~1;
  const int t = threadIdx.x;
  if (t >= 64 * R) return;
  double* A = lds;             // N x N, ld LD
  double* tau = A + N * LD;
  double* sig = tau + N;
  double* sorted = sig + N;
  double2* cs = reinterpret_cast<double2*>(sorted + N);  // rotations of a round (cos, sin), twice N / 2
  int* s_rot = reinterpret_cast<int*>(cs + N);           // a rotation in sweep w: s_rot[w % 3]
  double* Vm = R > 12 ? P.work : sorted + 3 * N + 2;     // N x N, ld LV
  double* H = A;  // the reflectors, ld LD, while A's columns are in registers
  const int c = t >> 3, ln = t & 7;                      // column c, rows ln + 8 u

  // ---- S = Q R, reflector j (H_j = I - tau_j v v', v_j = 1, as LAPACK's dlarfg) in column
  // j of H, formed by column j's lanes as soon as its last update is done
  double x[R], hv[R];  // hv: reflector c
#pragma unroll
  for (int u = 0; u < R; ++u) {
    const int i = ln + 8 * u;
    x[u] = i < k && c < k ? P.S[i + c * P.lds] : 0.0;
    hv[u] = 0.0;
  }
  auto reflector = [&]() {
    double a = 0.0, s2 = 0.0;
#pragma unroll
    for (int u = 0; u < R; ++u) {
      const int i = ln + 8 * u;
      a = i == c ? x[u] : a;
      s2 = i > c ? __builtin_fma(x[u], x[u], s2) : s2;
    }
    a = group_sum8(a);
    s2 = group_sum8(s2);
    double beta = a, tj = 0.0, scale = 0.0;
    if (s2 > 0.0) {
      beta = -copysign(sqrt(__builtin_fma(a, a, s2)), a);
      tj = (beta - a) / beta;
      scale = 1.0 / (a - beta);
    }
#pragma unroll
    for (int u = 0; u < R; ++u) {
      const int i = ln + 8 * u;
      hv[u] = i == c ? 1.0 : i > c ? x[u] * scale : 0.0;
      H[i + c * LD] = hv[u];
      x[u] = i == c ? beta : i > c ? 0.0 : x[u];
    }
    if (ln == 0) tau[c] = tj;
  };
  if (c == 0) reflector();
  if (t < 3) s_rot[t] = 0;
  __syncthreads();
  for (int j = 0; j < k - 1; ++j) {
    if (c > j && c < k) {
      const double tj = tau[j];
      if (tj != 0.0) {
        double h[R], w = 0.0;
#pragma unroll
        for (int u = 0; u < R; ++u) h[u] = H[ln + 8 * u + j * LD];
#pragma unroll
        for (int u = 0; u < R; ++u) w = __builtin_fma(h[u], x[u], w);
        w = group_sum8(w) * tj;
#pragma unroll
        for (int u = 0; u < R; ++u) x[u] = __builtin_fma(-w, h[u], x[u]);
      }
      if (c == j + 1) reflector();
    }
    __syncthreads();
  }
  // A = R', V = I; what is past k stays zero (V: the identity) under the rotations
#pragma unroll
  for (int u = 0; u < R; ++u) {
    const int i = ln + 8 * u;
    A[c + i * LD] = x[u];
    Vm[i + c * LV] = i == c ? 1.0 : 0.0;
    if constexpr (R > 12) P.work[N * N + t + 64 * R * u] = hv[u];
  }
  __syncthreads();

  // ---- the sweeps
  const bool vhalf = t >= 32 * R;
  const int pair = (vhalf ? t - 32 * R : t) >> 3;
  const bool act = pair < ke / 2;
  int pa = pair, pb = pair == 0 ? 1 : ke - pair;
  if (pair) pa = 1 + pair;
  if (pa > ke - 1) pa = 1;
  auto next_pair = [&]() {  // columns 1 .. ke - 1 move round
    if (pair) pa = pa == ke - 1 ? 1 : pa + 1;
    pb = pb == ke - 1 ? 1 : pb + 1;
  };
  auto rotate_v = [&](int b) {
    const double2 r = cs[b * (N / 2) + pair];
    if (act && r.y != 0.0) {
      double u[R], w[R];
#pragma unroll
      for (int q = 0; q < R; ++q) {
        u[q] = Vm[ln + 8 * q + pa * LV];
        w[q] = Vm[ln + 8 * q + pb * LV];
      }
#pragma unroll
      for (int q = 0; q < R; ++q) {
        Vm[ln + 8 * q + pa * LV] = r.x * u[q] - r.y * w[q];
        Vm[ln + 8 * q + pb * LV] = r.y * u[q] + r.x * w[q];
      }
    }
    next_pair();
  };
  int buf = 0;
  for (int sweep = 0; sweep < 60; ++sweep) {
    int rot = 0;
    if (t == 0) s_rot[(sweep + 1) % 3] = 0;
    for (int round = 0; round < ke - 1; ++round) {
      if (!vhalf) {
        if (act) {
          double y[R], al = 0.0, be = 0.0, ga = 0.0;
#pragma unroll
          for (int q = 0; q < R; ++q) {
            x[q] = A[ln + 8 * q + pa * LD];
            y[q] = A[ln + 8 * q + pb * LD];
          }
#pragma unroll
          for (int q = 0; q < R; ++q) {
            al = __builtin_fma(x[q], x[q], al);
            be = __builtin_fma(y[q], y[q], be);
            ga = __builtin_fma(x[q], y[q], ga);
          }
          al = group_sum8(al);
          be = group_sum8(be);
          ga = group_sum8(ga);
          // rotate unless |ga| <= 4 eps sqrt(al be); tan of the angle
          // t = sign(d) 2ga / (|d| + sqrt(d^2 + 4ga^2)), d = be - al (|t| <= 1),
          // through refined hardware reciprocals (column norms are normal numbers)
          double2 r{1.0, 0.0};
          if (ga * ga > 16.0 * kEps * kEps * al * be) {
            const double d = be - al;
            const double g2 = 2.0 * ga;
            const double q2 = __builtin_fma(d, d, g2 * g2);
            const double den = fabs(d) + q2 * rsqrt_nr(q2);
            double tt = g2 * rcp_nr(den);
            if (d < 0.0) tt = -tt;
            r.x = rsqrt_nr(__builtin_fma(tt, tt, 1.0));
            r.y = r.x * tt;
#pragma unroll
            for (int q = 0; q < R; ++q) {
              A[ln + 8 * q + pa * LD] = r.x * x[q] - r.y * y[q];
              A[ln + 8 * q + pb * LD] = r.y * x[q] + r.x * y[q];
            }
            rot = 1;
          }
          if (ln == 0) cs[buf * (N / 2) + pair] = r;
          next_pair();
        }
        if (rot && round == ke - 2) s_rot[sweep % 3] = 1;
      } else if (sweep + round > 0) {
        rotate_v(buf ^ 1);
      }
      buf ^= 1;
      __syncthreads();
    }
    if (!s_rot[sweep % 3]) break;
  }
  if (vhalf) rotate_v(buf ^ 1);  // the last round's, if any
  __syncthreads();

  // ---- column c: the norm, V <- Q J, its place in descending order
  double s2 = 0.0;
#pragma unroll
  for (int u = 0; u < R; ++u) {
    x[u] = A[ln + 8 * u + c * LD];
    s2 = __builtin_fma(x[u], x[u], s2);
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < R; ++u) {
    if constexpr (R > 12) hv[u] = P.work[N * N + t + 64 * R * u];
    H[ln + 8 * u + c * LD] = hv[u];
  }
  __syncthreads();
  double v[R], h[R];
#pragma unroll
  for (int u = 0; u < R; ++u) {
    v[u] = Vm[ln + 8 * u + c * LV];
    h[u] = H[ln + 8 * u + (k - 1) * LD];
  }
  for (int j = k - 1; j >= 0; --j) {
    double g[R], w = 0.0;
    const int jn = j > 0 ? j - 1 : 0;
#pragma unroll
    for (int u = 0; u < R; ++u) g[u] = H[ln + 8 * u + jn * LD];
#pragma unroll
    for (int u = 0; u < R; ++u) w = __builtin_fma(h[u], v[u], w);
    w = group_sum8(w) * tau[j];
#pragma unroll
    for (int u = 0; u < R; ++u) {
      v[u] = __builtin_fma(-w, h[u], v[u]);
      h[u] = g[u];
    }
  }
  const double sg = sqrt(group_sum8(s2));
  if (ln == 0) sig[c] = sg;
  __syncthreads();
  double before = 0.0;
  for (int l = ln; l < k; l += 8) before += (sig[l] > sg) || (sig[l] == sg && l < c) ? 1.0 : 0.0;
  const int pos = (int)group_sum8(before);
  if (c < k) {
    const double inv = sg > 0.0 ? 1.0 / sg : 0.0;
    if (ln == 0) {
      P.sigma[pos] = sg;
      sorted[pos] = sg;
    }
#pragma unroll
    for (int u = 0; u < R; ++u) {
      const int i = ln + 8 * u;
      if (i < k) {
        P.V[i + pos * k] = x[u] * inv;
        P.U[i + pos * k] = v[u];
      }
    }
  }
  __syncthreads();
  // lane j: the tail sum from the smallest value up to sigma_j; the rank is one more than
  // the last j >= 1 whose tail is above tol
  if (t < 64) {
    int rho = 1;
    for (int j0 = 0; j0 < k; j0 += 64) {
      const int j = j0 + t;
      double tail = 0.0;
      for (int l = k - 1; l >= 1; --l) {
        const double q = sorted[l];
        if (l >= j) tail = tail + q * q;
      }
      const unsigned long long above = __ballot(j >= 1 && j < k && !(sqrt(tail) <= P.tol));
      if (above) rho = j0 + 64 - __clzll((long long)above);
    }
    if (rho > P.rmax) rho = (int)P.rmax;
    if (rho < 1) rho = 1;
    if (t == 0) *P.r_out = rho;
  }
}

template <bool kBig>
__device__ void jacobi_dispatch(const SvdArgs P, double* lds) {
  if constexpr (kBig) {
    if (P.k <= 80) jacobi_body<10>(P, lds);
    else if (P.k <= 96) jacobi_body<12>(P, lds);
    else jacobi_body<16>(P, lds);
  } else {
    if (P.k <= 16) jacobi_body<2>(P, lds);
    else if (P.k <= 32) jacobi_body<4>(P, lds);
    else if (P.k <= 48) jacobi_body<6>(P, lds);
    else jacobi_body<8>(P, lds);
  }
}

__global__ __launch_bounds__(kThreads) void k_small_abt(const double* __restrict__ A, const double* __restrict__ B,
                                                        int k, double* __restrict__ C) {
  for (int e = threadIdx.x; e < k * k; e += blockDim.x) {
    const int i = e % k, j = e / k;
    double s = 0.0;
    for (int l = 0; l < k; ++l) s += A[i + l * k] * B[j + l * k];
    C[e] = s;
  }
}

hipError_t launch_small_abt(const double* A, const double* B, int k, double* C, hipStream_t st) {
  if (k < 1 || k > kMaxAug) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_small_abt, dim3(1), dim3(kThreads), 0, st, A, B, k, C);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// r x r parts of the BUG adjoint
// ---------------------------------------------------------------------------

// X1 = R1^{-T} and X2 = R2^{-T} for upper triangular R1, R2 (r x r, ld r, in
// global memory): both are staged in LDS (ws: inv_ws_doubles(r)), thread j of
// wave 0 (R1) or wave 1 (R2) solves R x = e_j by back substitution into column
// j of an LDS block (ld r + 1 against bank conflicts), and the columns of
// R^{-1} are stored as the rows of X.  Called by all threads (>= 128).
__host__ __device__ inline int inv_ws_doubles(int r) { return 2 * r * r + 2 * r * (r + 1); }

__device__ void inv_transpose_upper2(const double* R1, double* X1, const double* R2, double* X2, int r,
                                     double* ws) {
  const int t = threadIdx.x, rr = r * r, lx = r + 1;
  double* R1s = ws;
  double* R2s = ws + rr;
  double* X1s = ws + 2 * rr;
  double* X2s = X1s + r * lx;
  for (int e = t; e < rr; e += blockDim.x) {
    R1s[e] = R1[e];
    R2s[e] = R2[e];
  }
  __syncthreads();
  const int which = t >> 6, j = t & 63;
  if (which < 2 && j < r) {
    const double* Rs = which ? R2s : R1s;
    double* x = (which ? X2s : X1s) + j * lx;
    for (int i = r - 1; i >= 0; --i) {
      double v = (i == j) ? 1.0 : 0.0;
      for (int l = i + 1; l <= j; ++l) v -= Rs[i + l * r] * x[l];  // x[l] = 0 for l > j
      x[i] = (i > j) ? 0.0 : v / Rs[i + i * r];
    }
  }
  __syncthreads();
  for (int e = t; e < rr; e += blockDim.x) {
    const int i = e % r, jj = e / r;  // (R^{-1})_{i jj} -> (R^{-T})_{jj i}
    X1[jj + i * r] = X1s[i + jj * lx];
    X2[jj + i * r] = X2s[i + jj * lx];
  }
}

// LDS of k_bug_adj_pre: r <= 32 stages Sb1, N, M, S0, T1, T2 (6 r^2) and runs
// the products on the matrix cores; larger r keeps T1, T2 only (2 r^2).  Then
// the inverses' workspace reuses it.
__host__ __device__ inline int bug_adj_pre_ws(int r) {
  const int prod = r <= 32 ? 6 * r * r : 2 * r * r;
  return prod > inv_ws_doubles(r) ? prod : inv_ws_doubles(r);
}

__global__ __launch_bounds__(kThreads) void k_bug_adj_pre(BugAdjSmall* A, const double* M, const double* N,
                                                          const double* S0, int lds, int r) {
  extern __shared__ double ws[];
  const int t = threadIdx.x, rr = r * r;
  if (r <= 32) {
    double* sSb = ws;
    double* sN = ws + rr;
    double* sM = ws + 2 * rr;
    double* sS = ws + 3 * rr;
    double* T1 = ws + 4 * rr;
    double* T2 = ws + 5 * rr;
    for (int e = t; e < rr; e += blockDim.x) {
      sSb[e] = A->Sb1[e];
      sN[e] = N[e];
      sM[e] = M[e];
      sS[e] = S0[e % r + (e / r) * lds];
    }
    __syncthreads();
    // T1 = Sb1 N, T2 = M S0
    wave_gemm(
        r, r, r, 2, [&](int b, int i, int l) { return b == 0 ? sSb[i + l * r] : sM[i + l * r]; },
        [&](int b, int l, int jj) { return b == 0 ? sN[l + jj * r] : sS[l + jj * r]; },
        [&](int b, int i, int jj, double v) { (b == 0 ? T1 : T2)[i + jj * r] = v; });
    __syncthreads();
    // Mb = T1 S0', Nb = Sb1' T2, Sb0 = M' T1
    wave_gemm(
        r, r, r, 3,
        [&](int b, int i, int l) { return b == 0 ? T1[i + l * r] : (b == 1 ? sSb[l + i * r] : sM[l + i * r]); },
        [&](int b, int l, int jj) { return b == 0 ? sS[jj + l * r] : (b == 1 ? T2[l + jj * r] : T1[l + jj * r]); },
        [&](int b, int i, int jj, double v) { (b == 0 ? A->Mb : (b == 1 ? A->Nb : A->Sb0))[i + jj * r] = v; });
  } else {
    double* T1 = ws;
    double* T2 = ws + rr;
    for (int e = t; e < rr; e += blockDim.x) {  // T1 = Sb1 N, T2 = M S0
      const int i = e % r, j = e / r;
      double a = 0.0, b = 0.0;
      for (int l = 0; l < r; ++l) {
        a += A->Sb1[i + l * r] * N[l + j * r];
        b += M[i + l * r] * S0[l + j * lds];
      }
      T1[e] = a;
      T2[e] = b;
    }
    __syncthreads();
    for (int e = t; e < rr; e += blockDim.x) {
      const int i = e % r, j = e / r;
      double mb = 0.0, nb = 0.0, sb = 0.0;
      for (int l = 0; l < r; ++l) {
        mb += T1[i + l * r] * S0[j + l * lds];    // (Sb1 N) S0'
        nb += A->Sb1[l + i * r] * T2[l + j * r];  // Sb1' (M S0)
        sb += M[l + i * r] * T1[l + j * r];       // M' (Sb1 N)
      }
      A->Mb[e] = mb;
      A->Nb[e] = nb;
      A->Sb0[e] = sb;
    }
  }
  __syncthreads();
  inv_transpose_upper2(A->RK, A->RKinvT, A->RL, A->RLinvT, r, ws);
}

__global__ __launch_bounds__(kThreads) void k_bug_adj_post(BugAdjSmall* A, int r) {
  for (int e = threadIdx.x; e < r * r; e += blockDim.x) {
    const int i = e % r, j = e / r;
    A->Sb0[e] += A->CK[j + i * r] + A->CL[e];
  }
}

__global__ __launch_bounds__(kThreads) void k_ksl_adj_small(BugAdjSmall* A, int r, int stage) {
  extern __shared__ double ws[];
  const int rr = r * r;
  if (stage == 0) {
    inv_transpose_upper2(A->RK, A->RKinvT, A->RL, A->RLinvT, r, ws);
    for (int e = threadIdx.x; e < rr; e += blockDim.x) {  // Mb = RL Sb1
      const int i = e % r, j = e / r;
      double v = 0.0;
      for (int l = 0; l < r; ++l) v += A->RL[i + l * r] * A->Sb1[l + j * r];
      A->Mb[e] = v;
    }
  } else if (stage == 1) {
    for (int e = threadIdx.x; e < rr; e += blockDim.x) {  // Nb = RK CL'
      const int i = e % r, j = e / r;
      double v = 0.0;
      for (int l = 0; l < r; ++l) v += A->RK[i + l * r] * A->CL[j + l * r];
      A->Nb[e] = v;
    }
  } else {
    for (int e = threadIdx.x; e < rr; e += blockDim.x) A->Sb0[e] = A->CK[(e / r) + (e % r) * r];
  }
}

hipError_t launch_ksl_adj_small(BugAdjSmall* A, int r, int stage, hipStream_t st) {
  if (r < 1 || r > kMaxRank || stage < 0 || stage > 2) return hipErrorInvalidValue;
  const size_t ws = stage == 0 ? sizeof(double) * inv_ws_doubles(r) : 0;
  hipLaunchKernelGGL(k_ksl_adj_small, dim3(1), dim3(kThreads), ws, st, A, r, stage);
  return hipGetLastError();
}

// Reverse of the rank-adaptive step, small parts; one workgroup per stage (see lri_kernels.h).
__global__ __launch_bounds__(kThreads) void k_ra_adj_small(RaAdjSmall* A, const SmallState* st, const double* S0,
                                                           int lds, int r, int r1, int stage) {
  extern __shared__ double ws[];  // stage 0: the inverses' workspace
  const int t = threadIdx.x, nt = blockDim.x, k2 = 2 * r;
  const double* Us = st->Ush;
  const double* Vs = st->Vsh;
  const double* sig = st->sigma;
  const double* M = st->M;  // k2 x r, ld k2
  const double* N = st->N;
  if (stage == 0) {
    for (int e = t; e < k2 * r1; e += nt) {  // Jm = Ush' Ubs, Km = Vsh' Vbs
      const int i = e % k2, j = e / k2;
      double a = 0.0, b = 0.0;
      for (int l = 0; l < k2; ++l) {
        a += Us[l + i * k2] * A->Ubs[l + j * k2];
        b += Vs[l + i * k2] * A->Vbs[l + j * k2];
      }
      A->Jm[e] = a;
      A->Km[e] = b;
    }
    __syncthreads();
    inv_transpose_upper2(A->RU, A->RUinvT, A->RV, A->RVinvT, r, ws);
  } else if (stage == 1) {
    for (int e = t; e < k2 * k2; e += nt) {
      const int i = e % k2, j = e / k2;
      double v = 0.0;
      if (i != j && (i < r1 || j < r1)) {
        const double F = 1.0 / (sig[j] * sig[j] - sig[i] * sig[i]);
        const double jij = j < r1 ? A->Jm[i + j * k2] : 0.0, jji = i < r1 ? A->Jm[j + i * k2] : 0.0;
        const double kij = j < r1 ? A->Km[i + j * k2] : 0.0, kji = i < r1 ? A->Km[j + i * k2] : 0.0;
        v = F * (jij - jji) * sig[j] + sig[i] * F * (kij - kji);
      }
      if (i == j && i < r1) v = A->Sb1[i + i * r1];
      A->core[e] = v;
    }
  } else if (stage == 2) {
    for (int e = t; e < k2 * k2; e += nt) {  // Shb <- core Vsh' (temporarily)
      const int i = e % k2, j = e / k2;
      double v = 0.0;
      for (int l = 0; l < k2; ++l) v += A->core[i + l * k2] * Vs[j + l * k2];
      A->Shb[e] = v;
    }
  } else if (stage == 3) {
    for (int e = t; e < k2 * k2; e += nt) {  // core <- Ush (core Vsh')
      const int i = e % k2, j = e / k2;
      double v = 0.0;
      for (int l = 0; l < k2; ++l) v += Us[i + l * k2] * A->Shb[l + j * k2];
      A->core[e] = v;
    }
  } else {
    // Shb = the cotangent of Shat (in core); Jm <- S0 N' (r x k2), Km <- S0' M' (r x k2), ld r
    for (int e = t; e < k2 * k2; e += nt) A->Shb[e] = A->core[e];
    for (int e = t; e < r * k2; e += nt) {
      const int i = e % r, l = e / r;
      double sn = 0.0, sm = 0.0;
      for (int q = 0; q < r; ++q) {
        sn += S0[i + q * lds] * N[l + q * k2];
        sm += S0[q + i * lds] * M[l + q * k2];
      }
      A->Jm[e] = sn;
      A->Km[e] = sm;
    }
    __syncthreads();
    const double* Sb = A->Shb;
    for (int e = t; e < r * k2; e += nt) {  // G1 = (S0 N') Shb', G2 = (S0' M') Shb  (r x k2)
      const int i = e % r, j = e / r;
      double g1 = 0.0, g2 = 0.0;
      for (int l = 0; l < k2; ++l) {
        g1 += A->Jm[i + l * r] * Sb[j + l * k2];
        g2 += A->Km[i + l * r] * Sb[l + j * k2];
      }
      A->G1[e] = g1;
      A->G2[e] = g2;
    }
    for (int e = t; e < k2 * r; e += nt) {  // G3 = Shb (N S0'), G4 = Shb' (M S0), core <- Shb N  (k2 x r)
      const int i = e % k2, j = e / k2;
      double g3 = 0.0, g4 = 0.0, sn = 0.0;
      for (int l = 0; l < k2; ++l) {
        g3 += Sb[i + l * k2] * A->Jm[j + l * r];
        g4 += Sb[l + i * k2] * A->Km[j + l * r];
        sn += Sb[i + l * k2] * N[l + j * k2];
      }
      A->G3[e] = g3;
      A->G4[e] = g4;
      A->core[e] = sn;
    }
    __syncthreads();
    for (int e = t; e < r * r; e += nt) {  // Sb0 = M' (Shb N)
      const int i = e % r, j = e / r;
      double v = 0.0;
      for (int l = 0; l < k2; ++l) v += M[l + i * k2] * A->core[l + j * k2];
      A->Sb0[e] = v;
    }
  }
}

hipError_t launch_ra_adj_small(RaAdjSmall* A, const SmallState* st, const double* S0, int lds, int r, int r1,
                               int stage, hipStream_t s) {
  if (r < 1 || r > kMaxRank || r1 < 1 || r1 > 2 * r || r1 > kMaxRank || stage < 0 || stage > 4)
    return hipErrorInvalidValue;
  const size_t ws = stage == 0 ? sizeof(double) * inv_ws_doubles(r) : 0;
  hipLaunchKernelGGL(k_ra_adj_small, dim3(1), dim3(kThreads), ws, s, A, st, S0, lds, r, r1, stage);
  return hipGetLastError();
}

hipError_t launch_bug_adj_pre(BugAdjSmall* A, const double* M, const double* N, const double* S0, int lds, int r,
                              hipStream_t st) {
  if (r < 1 || r > kMaxRank) return hipErrorInvalidValue;
  const size_t ws = sizeof(double) * (size_t)bug_adj_pre_ws(r);
  hipLaunchKernelGGL(k_bug_adj_pre, dim3(1), dim3(kThreads), ws, st, A, M, N, S0, lds, r);
  return hipGetLastError();
}

hipError_t launch_bug_adj_post(BugAdjSmall* A, int r, hipStream_t st) {
  if (r < 1 || r > kMaxRank) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_bug_adj_post, dim3(1), dim3(kThreads), 0, st, A, r);
  return hipGetLastError();
}

// workgroup 0 decomposes P0, workgroup 1 (if launched) P1; kBig: 64 < k <= 128
template <bool kBig>
__global__ __launch_bounds__(kBig ? 1024 : 512) void k_jacobi_svd(SvdArgs P0, SvdArgs P1) {
  extern __shared__ double lds[];
  jacobi_dispatch<kBig>(blockIdx.x == 0 ? P0 : P1, lds);
}

// the batched forms: one record holds the one or two decompositions of a launch
struct SvdPair {
  SvdArgs P0, P1;
};
template <bool kBig>
__global__ __launch_bounds__(kBig ? 1024 : 512) void k_jacobi_svd_batch(const unsigned char* __restrict__ tab,
                                                                        const int* __restrict__ start, int count) {
  extern __shared__ double lds[];
  const int i = batch_member(start, count, blockIdx.x);
  const SvdPair& S = *reinterpret_cast<const SvdPair*>(tab + (size_t)start[count + 1 + i] * kRecArgBytes);
  jacobi_dispatch<kBig>(blockIdx.x - start[i] == 0 ? S.P0 : S.P1, lds);
}

static int jacobi_rows(int k) {
  return k <= 16 ? 2 : k <= 32 ? 4 : k <= 48 ? 6 : k <= 64 ? 8 : k <= 80 ? 10 : k <= 96 ? 12 : 16;
}

static hipError_t launch_jacobi(const SvdArgs& P0, const SvdArgs& P1, unsigned count, hipStream_t st) {
  const int k = std::max(P0.k, P1.k), R = jacobi_rows(k);
  const bool big = k > 64;
  for (const SvdArgs* P : {&P0, &P1})
    if (P->k < 1 || P->k > kMaxAug || (big && !P->work)) return hipErrorInvalidValue;
  // R = 12 takes the most: 160 KB to the last 240 bytes
  const size_t lds = sizeof(double) * (k > 96 && std::min(P0.k, P1.k) > 96 ? jacobi_lds_doubles(16)
                                       : k > 96                           ? jacobi_lds_doubles(12)
                                                                          : jacobi_lds_doubles(R));
  // a batch merges all members up to k = 64 into one launch of 512 threads, of which the
  // smaller ones' spare waves leave at once: a launch for every size one after
  // the other would add their times up
  const SvdPair S{P0, P1};
  if (!record_launch(KID_JACOBI, big, count, big ? 1024 : 512, lds, S)) {
    if (big) hipLaunchKernelGGL(k_jacobi_svd<true>, dim3(count), dim3(64 * R), lds, st, P0, P1);
    else hipLaunchKernelGGL(k_jacobi_svd<false>, dim3(count), dim3(64 * R), lds, st, P0, P1);
  }
  return hipGetLastError();
}
hipError_t launch_jacobi_svd(SvdArgs P, hipStream_t st) { return launch_jacobi(P, P, 1, st); }
hipError_t launch_jacobi_svd2(SvdArgs P0, SvdArgs P1, hipStream_t st) { return launch_jacobi(P0, P1, 2, st); }

// ----------------------------------------------------------------------------
// orthonormal completion of dropped CholeskyQR columns (see CompleteArgs)
// ----------------------------------------------------------------------------
constexpr int kCompleteThreads = 256;

// per thread v[0..7]: the workgroup sums into out[0..7] (LDS), visible to all after return
__device__ __forceinline__ void complete_block_sum8(double (&v)[8], double* red, double* out) {
#pragma unroll
  for (int q = 0; q < 8; ++q)
    for (int off = 32; off > 0; off >>= 1) v[q] += __shfl_xor(v[q], off);
  __syncthreads();
  if ((threadIdx.x & 63) == 0)
#pragma unroll
    for (int q = 0; q < 8; ++q) red[(threadIdx.x >> 6) * 8 + q] = v[q];
  __syncthreads();
  if (threadIdx.x < 8) {
    const int q = threadIdx.x;
    out[q] = (red[q] + red[8 + q]) + (red[16 + q] + red[24 + q]);
  }
  __syncthreads();
}

// h[0..n) = Q(:, 0..n)' y over the rows (h in LDS)
__device__ void complete_project(const double* __restrict__ Q, int64_t rows, int n, const double* __restrict__ y,
                                 double* red, double* h) {
  const int t = threadIdx.x;
  for (int c0 = 0; c0 < n; c0 += 8) {
    double v[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int64_t i = t; i < rows; i += kCompleteThreads) {
      const double yi = y[i];
#pragma unroll
      for (int q = 0; q < 8; ++q)
        if (c0 + q < n) v[q] = fma(Q[i + (c0 + q) * rows], yi, v[q]);
    }
    complete_block_sum8(v, red, h + c0);
  }
}

__global__ __launch_bounds__(kCompleteThreads) void k_complete_columns(CompleteArgs A) {
  __shared__ double s_R[kMaxRank * kMaxRank];  // R (k x k, ld k)
  __shared__ double s_h[kMaxAug + 8];
  __shared__ double s_red[32];
  __shared__ int s_dep[kMaxAug];
  __shared__ double s_min[4];
  __shared__ long long s_arg[4];
  const int t = threadIdx.x;
  const int k = A.k;
  const int64_t rows = A.rows;
  double* __restrict__ Q = A.Q;
  // one diagonal entry per thread: the common case (nothing dropped) costs one load
  if (!__syncthreads_or(t < k && (A.Rinv1[t + t * k] == 0.0 || A.Rinv2[t + t * k] == 0.0))) return;
  for (int e = t; e < k * k; e += kCompleteThreads) s_R[e] = 0.0;
  // the largest column norm of X, for the rounding-level threshold
  double cmax = 0.0;
  for (int c0 = 0; c0 < k; c0 += 8) {
    double v[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int64_t i = t; i < rows; i += kCompleteThreads)
#pragma unroll
      for (int q = 0; q < 8; ++q)
        if (c0 + q < k) v[q] = fma(A.X[i + (c0 + q) * rows], A.X[i + (c0 + q) * rows], v[q]);
    complete_block_sum8(v, s_red, s_h);
    for (int q = 0; q < 8 && c0 + q < k; ++q) cmax = fmax(cmax, s_h[q]);
  }
  const double tol = 16.0 * k * kEps * sqrt(cmax);
  // classical Gram-Schmidt, each column projected out twice
  for (int j = 0; j < k; ++j) {
    double* __restrict__ qj = Q + (int64_t)j * rows;
    for (int64_t i = t; i < rows; i += kCompleteThreads) qj[i] = A.X[i + (int64_t)j * rows];
    __syncthreads();
    for (int pass = 0; pass < 2 && j > 0; ++pass) {
      complete_project(Q, rows, j, qj, s_red, s_h);
      for (int64_t i = t; i < rows; i += kCompleteThreads) {
        double v = qj[i];
        for (int c = 0; c < j; ++c) v = fma(-Q[i + c * rows], s_h[c], v);
        qj[i] = v;
      }
      if (t < j) s_R[t + j * k] += s_h[t];
      __syncthreads();
    }
    double v[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int64_t i = t; i < rows; i += kCompleteThreads) v[0] = fma(qj[i], qj[i], v[0]);
    complete_block_sum8(v, s_red, s_h);
    const double nrm = sqrt(s_h[0]);
    const bool dep = !(nrm > tol);
    const double sc = dep ? 0.0 : 1.0 / nrm;
    for (int64_t i = t; i < rows; i += kCompleteThreads) qj[i] *= sc;
    if (t == 0) {
      s_R[j + j * k] = dep ? 0.0 : nrm;
      s_dep[j] = dep ? 1 : 0;
    }
    __syncthreads();
  }
  // orthonormal completion of the dependent columns (their rows of R are zero)
  for (int p = 0; p < k; ++p) {
    if (!s_dep[p]) continue;
    double* __restrict__ q = Q + (int64_t)p * rows;
    double best = 1e300;
    long long bi = 0;
    for (int64_t i = t; i < rows; i += kCompleteThreads) {
      double s2 = 0.0;
      for (int c = 0; c < k; ++c) s2 = fma(Q[i + c * rows], Q[i + c * rows], s2);
      if (s2 < best) {
        best = s2;
        bi = i;
      }
    }
    for (int off = 32; off > 0; off >>= 1) {
      const double ob = __shfl_xor(best, off);
      const long long oi = __shfl_xor(bi, off);
      if (ob < best || (ob == best && oi < bi)) {
        best = ob;
        bi = oi;
      }
    }
    if ((t & 63) == 0) {
      s_min[t >> 6] = best;
      s_arg[t >> 6] = bi;
    }
    __syncthreads();
    if (t == 0)
      for (int w = 1; w < 4; ++w)
        if (s_min[w] < s_min[0] || (s_min[w] == s_min[0] && s_arg[w] < s_arg[0])) {
          s_min[0] = s_min[w];
          s_arg[0] = s_arg[w];
        }
    __syncthreads();
    const int64_t is = s_arg[0];
    if (t < k) s_h[t] = Q[is + t * rows];
    __syncthreads();
    for (int64_t i = t; i < rows; i += kCompleteThreads) {  // column p is zero and takes no part
      double x = i == is ? 1.0 : 0.0;
      for (int c = 0; c < k; ++c) x = fma(-Q[i + c * rows], s_h[c], x);
      q[i] = x;
    }
    __syncthreads();
    for (int pass = 0; pass < 2; ++pass) {
      complete_project(Q, rows, k, q, s_red, s_h);
      if (t == 0) s_h[p] = 0.0;
      __syncthreads();
      for (int64_t i = t; i < rows; i += kCompleteThreads) {
        double x = q[i];
        for (int c = 0; c < k; ++c) x = fma(-Q[i + c * rows], s_h[c], x);
        q[i] = x;
      }
      __syncthreads();
    }
    double v[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int64_t i = t; i < rows; i += kCompleteThreads) v[0] = fma(q[i], q[i], v[0]);
    complete_block_sum8(v, s_red, s_h);
    const double inv = 1.0 / sqrt(s_h[0]);
    for (int64_t i = t; i < rows; i += kCompleteThreads) q[i] *= inv;
    __syncthreads();
  }
  // the packed copy of Q for the next pass
  for (int64_t i = t; i < rows; i += kCompleteThreads)
    for (int p = 0; p < k; ++p) {
      const double x = Q[i + (int64_t)p * rows];
      if (A.pk_f64) A.pk_f64[i * A.pk_cols + p] = x;
      if (A.pk_f32) A.pk_f32[pk_f32_offset(A.pk_layout, i, p, A.pk_cols)] = (float)x;
      if (A.pk_hi) {
        uint32_t hi, lo;
        split_bf16((float)x, hi, lo);
        const int64_t off = pk_offset(A.pk_layout, i, p, A.pk_cols);
        A.pk_hi[off] = (uint16_t)hi;
        A.pk_lo[off] = (uint16_t)lo;
      }
    }
  // the products of R: Z = R (zt: R'), M = R - Q' W (mt: its transpose)
  if (A.Z)
    for (int e = t; e < k * k; e += kCompleteThreads) {
      const int i = e % k, j = e / k;
      if (A.zt) A.Z[j + i * A.ldz] = s_R[e];
      else A.Z[i + j * A.ldz] = s_R[e];
    }
  if (A.M)
    for (int c = 0; c < k; ++c) {
      complete_project(Q, rows, k, A.W + (int64_t)c * A.ldw, s_red, s_h);
      if (t < k) {
        const double x = s_R[t + c * k] - s_h[t];
        if (A.mt) A.M[c + t * A.ldm] = x;
        else A.M[t + c * A.ldm] = x;
      }
      __syncthreads();
    }
}

hipError_t launch_complete_columns(const CompleteArgs& A, hipStream_t st) {
  if (!A.X || !A.Q || A.rows < 1 || A.k < 1 || A.k > kMaxRank || !A.Rinv1 || !A.Rinv2 || (A.M && !A.W))
    return hipErrorInvalidValue;
  if (A.k > A.rows) return hipErrorInvalidValue;  // no room for an orthonormal completion
  hipLaunchKernelGGL(k_complete_columns, dim3(1), dim3(kCompleteThreads), 0, st, A);
  return hipGetLastError();
}

hipError_t launch_rowops_batched(int kid, int variant, const void* tab, const int* start, int count, unsigned total,
                                 unsigned block, size_t lds, hipStream_t st) {
  const unsigned char* t = static_cast<const unsigned char*>(tab);
  const dim3 g(total), b(block);
  switch (kid) {
    case KID_ROWS_D:
    case KID_ROWS_F: {
#define LRI_ROWS_BATCH(PT)                                                                                       \
  switch (variant) {                                                                                             \
    case 100: hipLaunchKernelGGL((k_rows_batch<PT, 1, 0>), g, b, lds, st, t, start, count); break;              \
    case 200: hipLaunchKernelGGL((k_rows_batch<PT, 2, 0>), g, b, lds, st, t, start, count); break;              \
    case 400: hipLaunchKernelGGL((k_rows_batch<PT, 4, 0>), g, b, lds, st, t, start, count); break;              \
    case 800: hipLaunchKernelGGL((k_rows_batch<PT, 8, 0>), g, b, lds, st, t, start, count); break;              \
    case 1600: hipLaunchKernelGGL((k_rows_batch<PT, 16, 0>), g, b, lds, st, t, start, count); break;            \
    default: return hipErrorInvalidValue;                                                                        \
  }
      if (kid == KID_ROWS_F) {
        LRI_ROWS_BATCH(float)
      } else {
        switch (variant) {
          case 116: hipLaunchKernelGGL((k_rows_batch<double, 1, 16>), g, b, lds, st, t, start, count); break;
          case 216: hipLaunchKernelGGL((k_rows_batch<double, 2, 16>), g, b, lds, st, t, start, count); break;
          case 132: hipLaunchKernelGGL((k_rows_batch<double, 1, 32>), g, b, lds, st, t, start, count); break;
          case 232: hipLaunchKernelGGL((k_rows_batch<double, 2, 32>), g, b, lds, st, t, start, count); break;
          default: { LRI_ROWS_BATCH(double) }
        }
      }
#undef LRI_ROWS_BATCH
      break;
    }
    case KID_REDUCE: hipLaunchKernelGGL(k_reduce_batch, g, b, lds, st, t, start, count); break;
    case KID_EPILOGUE:
      if (variant == 16) hipLaunchKernelGGL(k_epilogue_batch<16>, g, b, lds, st, t, start, count);
      else if (variant == 32) hipLaunchKernelGGL(k_epilogue_batch<32>, g, b, lds, st, t, start, count);
      else hipLaunchKernelGGL(k_epilogue_batch<64>, g, b, lds, st, t, start, count);
      break;
    case KID_JACOBI:
      if (variant) hipLaunchKernelGGL(k_jacobi_svd_batch<true>, g, b, lds, st, t, start, count);
      else hipLaunchKernelGGL(k_jacobi_svd_batch<false>, g, b, lds, st, t, start, count);
      break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace lri
