// Matrix-ODE sub-steps for right-hand sides with a quadratic term,
//
//     F(Y) = A Y + Y B' + G H' - (D Y) o Y          (o: elementwise product)
//
// A, B symmetric tridiagonal and D a general tridiagonal acting on the rows
// (e.g. viscous Burgers: A = nu Laplacian, D = central gradient, both
// periodic; each column one parameter sample).  With U, V orthonormal and
// frozen during a sub-step, the reference's default right-hand sides
// (projector_splitting.jl:52-80, unconventional.jl:51-79,
// rank_adaptive_unconventional.jl:59-86) are
//
//     K' = A K + K (V'BV) + G (H'V) - N,  N_ic = sum_ab (D K)_ia K_ib T_abc,
//     L' = B L + L (U'AU) + H (G'U) - Q,  Q_jc = sum_ab L_ja L_jb W_abc,
//     S' = sgn ((U'AU) S + S (V'BV) + (U'G)(H'V)' - P),
//          P_cd = sum_{e f a b} W_efc S_ea S_fb T_abd,
//
// with the third-order tensors T_abc = sum_j V_ja V_jb V_jc and
// W_abc = sum_i (D U)_ia U_ib U_ic.  The sub-problems are no longer linear, so
// every one of the N classical RK4 steps evaluates them: the K and L steps two
// RK4 steps per launch over tiles of rows with a halo, the S step in one
// workgroup.
#include <algorithm>

#include "lri_common.h"
#include "lri_kernels.h"

namespace lri {

namespace {

// RK4 stage weights: y_{s+1} input = y0 + c_s h k_s, accumulation weight w_s
__device__ __forceinline__ double stage_c(int s) { return s == 2 ? 1.0 : 0.5; }
__device__ __forceinline__ double stage_w(int s) { return (s == 1 || s == 2) ? 2.0 : 1.0; }

// row i of X (n x k, ld n), with periodic wrap or zero outside
__device__ __forceinline__ int64_t wrap_row(int64_t i, int64_t n, int periodic, bool* ok) {
  if (i < 0) {
    *ok = periodic != 0;
    return i + n;
  }
  if (i >= n) {
    *ok = periodic != 0;
    return i - n;
  }
  *ok = true;
  return i;
}

}  // namespace

// ----------------------------------------------------------------------------
// Partial third-order tensors: workgroup g sums the rows of chunk g,
//   part[g][c + k (a + k b)] = sum_{r in chunk} X_ra Y_rb Y_rc,
// X = D Y (the tridiagonal D applied to Y) when Q.dd != nullptr, else X = Y.
// ----------------------------------------------------------------------------

constexpr int kTensorRows = 64;

__global__ __launch_bounds__(256) void k_tensor3_part(TensorArgs Q) {
  __shared__ double xs[kTensorRows * kQuadMaxRank];
  __shared__ double ys[kTensorRows * kQuadMaxRank];
  const int k = Q.k, t = threadIdx.x;
  const int64_t r0 = (int64_t)blockIdx.x * kTensorRows;
  for (int e = t; e < kTensorRows * k; e += blockDim.x) {
    const int lr = e % kTensorRows, c = e / kTensorRows;
    const int64_t i = r0 + lr;
    double y = 0.0, x = 0.0;
    if (i < Q.rows) {
      y = Q.Y[i + c * Q.ldy];
      if (Q.dd) {
        bool okl, oku;
        const int64_t il = wrap_row(i - 1, Q.rows, Q.dper, &okl);
        const int64_t iu = wrap_row(i + 1, Q.rows, Q.dper, &oku);
        x = Q.dd[i] * y;
        if (okl) x += Q.dl[i] * Q.Y[il + c * Q.ldy];
        if (oku) x += Q.du[i] * Q.Y[iu + c * Q.ldy];
      } else {
        x = y;
      }
    }
    xs[lr * k + c] = x;
    ys[lr * k + c] = y;
  }
  __syncthreads();
  const int k3 = k * k * k;
  double* out = Q.part + (int64_t)blockIdx.x * k3;
  for (int e = t; e < k3; e += blockDim.x) {
    const int c = e % k, a = (e / k) % k, b = e / (k * k);
    double s = 0.0;
    for (int lr = 0; lr < kTensorRows; ++lr) s += xs[lr * k + a] * ys[lr * k + b] * ys[lr * k + c];
    out[e] = s;
  }
}

// out[e] = sum over chunks, in chunk order
__global__ __launch_bounds__(256) void k_tensor3_sum(const double* __restrict__ part, int nchunks, int k3,
                                                     double* __restrict__ out) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= k3) return;
  double s = 0.0;
  for (int g = 0; g < nchunks; ++g) s += part[(int64_t)g * k3 + e];
  out[e] = s;
}

hipError_t launch_tensor3(const TensorArgs& Q, double* out, hipStream_t st) {
  if (Q.k < 1 || Q.k > kQuadMaxRank || Q.rows < 1 || !Q.part) return hipErrorInvalidValue;
  const int nchunks = (int)((Q.rows + kTensorRows - 1) / kTensorRows);
  hipLaunchKernelGGL(k_tensor3_part, dim3(nchunks), dim3(256), 0, st, Q);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const int k3 = Q.k * Q.k * Q.k;
  hipLaunchKernelGGL(k_tensor3_sum, dim3((k3 + 255) / 256), dim3(256), 0, st, (const double*)Q.part, nchunks, k3,
                     out);
  return hipGetLastError();
}

// ----------------------------------------------------------------------------
// RK4 steps of the K or L sub-problem over a tile of rows, several stages per
// launch.  A stage needs the neighbouring rows of the previous one only, so a
// workgroup holds its kR - 2 kStepHalo rows with kStepHalo more on each side
// and runs up to kStepHalo = 8 stages (two RK4 steps) without leaving the CU:
// each stage makes one more row at either end stale, and after eight the
// workgroup's own rows are still exact.  (One launch per stage was bound by its
// launch latency: 9.4 us at n = 1000, k = 15, against about 0.7 us of FP64
// work; eight stages of both sub-problems of the 1000 x 400 problem now take 19.7 us
// in one launch, 2.5 us a stage: the solve went from 42.6 to 22.3 ms.)
//
//   f_ic = (A X)_ic + (X M)_ic + (g hv)_ic - N_ic,  N_ic = sum_ab (P X)_ia X_ib T_abc
//
// (P = D when Q.dd, else the identity).  X0, the RK4 accumulator and g hv of an
// element stay in its thread's registers; the stage input X and P X are in LDS.
// The quadratic term and X M are one product on the FP64 matrix cores,
//   N - X M = sum_b diag(X_:b) (P X) T_:b:  +  X (-M),
// a sum of k + 1 slabs (k x k each, in the k^2 order of the storage
// T[c + k (a + k b)], the slab b = k holding -M).  A wave keeps its 16 rows of
// P X in registers for the whole stage and scales them by X_:b, so a matrix
// instruction costs one LDS read (of T) and one multiplication.  Wave w takes
// rows 16 (w / 4) .. + 15, column block (w % 4) % nct (nct = ceil(k / 16)) and
// every (4 / nct)-th slab; the slabs' sums meet in LDS in a fixed order.
// ----------------------------------------------------------------------------

constexpr int kStepHalo = 8;

__host__ __device__ inline int quad_steps_pitch(int k) { return k | 1; }
// doubles of LDS; t_lds: the tensor too
__host__ __device__ inline int quad_steps_lds(int R, int k, bool t_lds) {
  return (R + 2) * quad_steps_pitch(k) + R * quad_steps_pitch(k) + (R / 4) * 272 + 6 * R + k * k +
         (t_lds ? k * k * k : 0);
}

// kQ = ceil(k / 4), kT: the tensor in LDS (else read from global memory)
template <int kR, int kQ, bool kT>
__global__ __launch_bounds__(16 * kR) void k_quad_steps(QuadStepsArgs Q0, QuadStepsArgs Q1) {
  extern __shared__ double dyn[];
  const QuadStepsArgs& Q = (int)blockIdx.x < Q0.blocks ? Q0 : Q1;
  const int bid = (int)blockIdx.x - ((int)blockIdx.x < Q0.blocks ? 0 : Q0.blocks);
  constexpr int kNT = 16 * kR, kNct = kQ > 4 ? 2 : 1, kNch = 4 / kNct, kE = kNct;  // kE elements per thread
  constexpr int kOwn = kR - 2 * kStepHalo;
  const int k = Q.k, kp = quad_steps_pitch(k), t = threadIdx.x;
  const int lane = t & 63, wave = t >> 6, lr = lane & 15, lk = lane >> 4;
  const int n = (int)Q.n, r0 = bid * kOwn;
  double* xs = dyn;                  // rows -1 .. kR of the tile: xs[(lrow + 1) * kp + c]
  double* ps = xs + (kR + 2) * kp;   // P X
  double* nl = ps + kR * kp;         // per wave 16 x 16 sums, pitch 17
  double* cf = nl + (kR / 4) * 272;  // stencil coefficients: A lower, diagonal, upper, then P's
  double* ms = cf + 6 * kR;          // -M (the slab b = k)
  double* tl = ms + k * k;           // T
  // row lrow of the tile is row (r0 - halo + lrow) mod n: the wrapped rows are the
  // neighbours of a periodic stencil; without one their coupling is zero
  for (int lrow = t; lrow < kR; lrow += kNT) {
    int i = (r0 - kStepHalo + lrow) % n;
    if (i < 0) i += n;
    const bool first = i == 0, last = i == n - 1;
    double al = 0.0, ad = 0.0, au = 0.0, pl = 0.0, pd = 1.0, pu = 0.0;
    if (Q.st_d) {
      ad = Q.st_d[i];
      al = !first ? Q.st_e[i - 1] : Q.periodic ? Q.st_e[n - 1] : 0.0;
      au = !last ? Q.st_e[i] : Q.periodic ? Q.st_e[n - 1] : 0.0;
    }
    if (Q.dd) {
      pd = Q.dd[i];
      pl = !first || Q.dper ? Q.dl[i] : 0.0;
      pu = !last || Q.dper ? Q.du[i] : 0.0;
    }
    cf[lrow] = al;
    cf[kR + lrow] = ad;
    cf[2 * kR + lrow] = au;
    cf[3 * kR + lrow] = pl;
    cf[4 * kR + lrow] = pd;
    cf[5 * kR + lrow] = pu;
  }
  for (int e = t; e < k * k; e += kNT) ms[e] = Q.M ? -Q.M[(e / k) + (e % k) * k] : 0.0;  // ms[c + k a] = -M(a, c)
  if (kT)
    for (int e = t; e < k * k * k; e += kNT) tl[e] = Q.T[e];
  for (int c = t; c < k; c += kNT) xs[c] = xs[(kR + 1) * kp + c] = 0.0;
  // the thread's elements: row er, columns ec + 16 j
  const int er = t % kR, ec = t / kR;
  int gi = (r0 - kStepHalo + er) % n;
  if (gi < 0) gi += n;
  const bool own = er >= kStepHalo && er < kStepHalo + kOwn && r0 + er - kStepHalo < n;
  double x0[kE], acc[kE], fg[kE];
#pragma unroll
  for (int j = 0; j < kE; ++j) {
    const int c = ec + 16 * j;
    x0[j] = acc[j] = fg[j] = 0.0;
    if (c < k) {
      x0[j] = Q.X[gi + c * Q.ld];
      for (int qq = 0; qq < Q.q; ++qq) fg[j] += Q.g[gi + qq * Q.ldg] * Q.hv[qq + c * Q.q];
      xs[(er + 1) * kp + c] = x0[j];
    }
  }
  __syncthreads();
  const double cal = cf[er], cad = cf[kR + er], cau = cf[2 * kR + er];
  const double cpl = cf[3 * kR + er], cpd = cf[4 * kR + er], cpu = cf[5 * kR + er];
  const int rt = (wave >> 2) * 16, ct = (wave & 3) % kNct, ch = (wave & 3) / kNct;
  const int tc = min(ct * 16 + lr, k - 1);
  const double h = Q.h;
  for (int step = 0; step < Q.nsteps; ++step) {
    if (Q.store && own) {
#pragma unroll
      for (int j = 0; j < kE; ++j)
        if (ec + 16 * j < k) Q.store[step * Q.n * k + gi + (ec + 16 * j) * Q.n] = x0[j];
    }
    for (int s = 0; s < Q.nstages; ++s) {
      double f[kE];
#pragma unroll
      for (int j = 0; j < kE; ++j) {
        const int c = ec + 16 * j;
        f[j] = 0.0;
        if (c < k) {
          const double xm = xs[er * kp + c], xc = xs[(er + 1) * kp + c], xp = xs[(er + 2) * kp + c];
          ps[er * kp + c] = cpl * xm + cpd * xc + cpu * xp;
          f[j] = cal * xm + cad * xc + cau * xp + fg[j];
        }
      }
      __syncthreads();
      {
        double pr[kQ];
        int to[kQ];
#pragma unroll
        for (int j = 0; j < kQ; ++j) {
          const int a = 4 * j + lk;
          to[j] = tc + k * min(a, k - 1);
          pr[j] = a < k ? ps[(rt + lr) * kp + a] : 0.0;
        }
        const double* xr = xs + (rt + lr + 1) * kp;
        f64x4_t a0 = {0.0, 0.0, 0.0, 0.0}, a1 = {0.0, 0.0, 0.0, 0.0};
        for (int b = ch; b < k; b += kNch) {
          const double xb = xr[b];
          const double* tb = (kT ? tl : Q.T) + k * k * b;
          double bv[kQ];
#pragma unroll
          for (int j = 0; j < kQ; ++j) bv[j] = tb[to[j]];
#pragma unroll
          for (int j = 0; j < kQ; ++j) {
            if (j & 1) a1 = __builtin_amdgcn_mfma_f64_16x16x4f64(pr[j] * xb, bv[j], a1, 0, 0, 0);
            else a0 = __builtin_amdgcn_mfma_f64_16x16x4f64(pr[j] * xb, bv[j], a0, 0, 0, 0);
          }
        }
        if (k % kNch == ch) {  // the slab b = k
#pragma unroll
          for (int j = 0; j < kQ; ++j) {
            const double x = 4 * j + lk < k ? xr[min(4 * j + lk, k - 1)] : 0.0;
            a0 = __builtin_amdgcn_mfma_f64_16x16x4f64(x, ms[to[j]], a0, 0, 0, 0);
          }
        }
        a0 += a1;
#pragma unroll
        for (int u = 0; u < 4; ++u) nl[wave * 272 + (4 * u + lk) * 17 + lr] = a0[u];
      }
      __syncthreads();
#pragma unroll
      for (int j = 0; j < kE; ++j) {
        const int c = ec + 16 * j;
        if (c < k) {
          const double* nw = nl + ((er >> 4) * 4 + j) * 272 + (er & 15) * 17 + ec;
#pragma unroll
          for (int u = 0; u < kNch; ++u) f[j] -= nw[u * kNct * 272];
          double x;
          if (s < 3) {
            acc[j] = (s == 0 ? 0.0 : acc[j]) + stage_w(s) * f[j];
            x = x0[j] + stage_c(s) * h * f[j];
            if (Q.stage_out && own) Q.stage_out[s * Q.n * k + gi + c * Q.n] = x;
          } else {
            x = x0[j] = x0[j] + (h / 6.0) * (acc[j] + f[j]);
          }
          xs[(er + 1) * kp + c] = x;
        }
      }
      __syncthreads();
    }
  }
  if (Q.Xn && own) {
#pragma unroll
    for (int j = 0; j < kE; ++j)
      if (ec + 16 * j < k) Q.Xn[gi + (ec + 16 * j) * Q.ld] = x0[j];
  }
}

namespace {

template <int kR, int kQ>
hipError_t run_quad_steps(const QuadStepsArgs& A, const QuadStepsArgs& B, unsigned grid, hipStream_t st) {
  const int k = A.k;
  const bool tl = quad_steps_lds(kR, k, true) <= kQuadStepsLds;
  const size_t lds = sizeof(double) * quad_steps_lds(kR, k, tl);
  if (tl) hipLaunchKernelGGL((k_quad_steps<kR, kQ, true>), dim3(grid), dim3(16 * kR), lds, st, A, B);
  else hipLaunchKernelGGL((k_quad_steps<kR, kQ, false>), dim3(grid), dim3(16 * kR), lds, st, A, B);
  return hipGetLastError();
}

template <int kR>
hipError_t dispatch_quad_steps(const QuadStepsArgs& A, const QuadStepsArgs& B, unsigned grid, hipStream_t st) {
  switch ((A.k + 3) / 4) {
    case 1: return run_quad_steps<kR, 1>(A, B, grid, st);
    case 2: return run_quad_steps<kR, 2>(A, B, grid, st);
    case 3: return run_quad_steps<kR, 3>(A, B, grid, st);
    case 4: return run_quad_steps<kR, 4>(A, B, grid, st);
    case 5: return run_quad_steps<kR, 5>(A, B, grid, st);
    case 6: return run_quad_steps<kR, 6>(A, B, grid, st);
    case 7: return run_quad_steps<kR, 7>(A, B, grid, st);
    default: return run_quad_steps<kR, 8>(A, B, grid, st);
  }
}

}  // namespace

hipError_t launch_quad_steps(QuadStepsArgs A, QuadStepsArgs B, hipStream_t st) {
  for (const QuadStepsArgs* Q : {&A, &B}) {
    if (Q->n == 0 && Q == &B) continue;
    if (Q->k < 1 || Q->k > kQuadMaxRank || Q->n < 1 || Q->n > (1 << 30) || Q->q < 0 || Q->q > kMaxForce || !Q->T ||
        Q->nstages < 1 || Q->nstages > 4 || Q->nsteps < 1 || Q->nsteps * Q->nstages > kStepHalo ||
        (Q->nsteps > 1 && Q->nstages != 4) || Q->X == Q->Xn)
      return hipErrorInvalidValue;
  }
  if (B.n && B.k != A.k) return hipErrorInvalidValue;
  // 32-row tiles (16 own rows) as long as all workgroups are resident at once;
  // above that 64-row tiles, which repeat a third of their rows instead of half
  auto blocks = [](int64_t rows, int own) { return (int)((rows + own - 1) / own); };
  const bool small_tiles = blocks(A.n, 16) + blocks(B.n, 16) <= 512;
  const int own = small_tiles ? 16 : 48;
  A.blocks = blocks(A.n, own);
  B.blocks = B.n ? blocks(B.n, own) : 0;
  const unsigned grid = (unsigned)(A.blocks + B.blocks);
  return small_tiles ? dispatch_quad_steps<32>(A, B, grid, st) : dispatch_quad_steps<64>(A, B, grid, st);
}

// ----------------------------------------------------------------------------
// S sub-step: N RK4 steps of
//   S' = sgn (Ga S + S Gb + cb - P(S)),  P_cd = sum_ab Z_c,ab T_abd,  Z_c = S' W_c S,
// S k x k, W_c = W(c, :, :), in one workgroup of 16 waves: the stages are a serial
// chain, so what counts is the length of a stage.  Wave w takes c = w (and
// c = w + 16 when k > 16): both products of Z_c stay in its registers, the result
// layout of the FP64 matrix instruction (row 4 u + lane / 16, column lane % 16) being
// the operand layout of the next one.  Z goes through LDS once, [a][c][b]; then
// wave w takes a = w (and w + 16) of the contraction with T, and the waves' partial
// sums of P (with slices of -(Ga S + S Gb)) meet in LDS in wave order.  For k <= 16
// W, T, Ga and Gb are in registers for the whole launch, a stage is 12 to 14
// matrix instructions a wave and three barriers: 1.3 us of the pipe's own time on
// the one CU.  Measured with the products as separate passes over LDS (three
// wave_gemm calls and scalar loops) 9.1 us a stage at k = 15; now 2.2 us (a
// launch of 16 RK4 steps: 581 -> 142 us; at k = 24, 30 steps, the whole BUG solve 2.2 times
// as fast together with the row kernel above).
// For k > 16 the slices b < 16 and b >= 16 of Z take turns in LDS and W, T are read
// from L2.
// ----------------------------------------------------------------------------

constexpr int kSZPitch = 17;  // of Z's innermost index and of the partial sums: conflict-free both ways

template <int NB>  // 16-wide blocks: k <= 16 NB
__global__ __launch_bounds__(1024) void k_quad_sstep(QuadSArgs Q) {
  constexpr int NP = 16 * NB, NJ = 4 * NB;  // padded size, 4-deep reduction steps
  __shared__ double sp[NP * (NP + 1)];             // S, zero-padded: sp[i * (NP + 1) + j]
  __shared__ double zs[NP * NP * kSZPitch];        // Z: [(a * NP + c) * 17 + b]
  __shared__ double pp_own[NB == 1 ? 16 * 16 * kSZPitch : 1];
  // partial sums [wave][c][d]; for NB = 2 in zs, a 16-row block of c at a time
  double* pp = NB == 1 ? pp_own : zs;
  const int k = Q.k, t = threadIdx.x, lane = t & 63, wave = t >> 6, lr = lane & 15, lk = lane >> 4;
  constexpr int SP = NP + 1;
  const bool elem = t < NP * NP;
  const int ei = t / NP, ej = t % NP;
  const bool live = elem && ei < k && ej < k;
  double y0 = 0.0, cb = 0.0, acc = 0.0;
  if (live) {
    y0 = Q.transS0 ? Q.S0[ej + ei * Q.lds0] : Q.S0[ei + ej * Q.lds0];
    for (int qq = 0; qq < Q.q; ++qq) cb += Q.gaT[qq + ei * Q.q] * Q.hbT[qq + ej * Q.q];
  }
  if (elem) sp[ei * SP + ej] = y0;
  // W(c, e, f) and T(a, b, d), zero outside
  auto wat = [&](int c, int e, int f) { return c < k && e < k && f < k ? Q.W[c + k * (e + k * f)] : 0.0; };
  auto tat = [&](int a, int b, int d) { return a < k && b < k && d < k ? Q.T[d + k * (a + k * b)] : 0.0; };
  double wr[NB == 1 ? 4 : 1], tr[NB == 1 ? 4 : 1];
  if (NB == 1) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      wr[NB == 1 ? j : 0] = wat(wave, lr, 4 * j + lk);
      tr[NB == 1 ? j : 0] = tat(wave, 4 * j + lk, lr);
    }
  }
  // the linear part: reduction step jl of Ga S (waves 0 .. NJ - 1) or of S Gb (NJ .. 2 NJ - 1)
  const int jl = wave % NJ, lin = wave < NJ ? 1 : wave < 2 * NJ ? 2 : 0;
  double gl[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    const int i = 16 * b + lr, m = 4 * jl + lk;
    gl[b] = lin && i < k && m < k ? -(lin == 1 ? Q.Ga[i + m * k] : Q.Gb[m + i * k]) : 0.0;
  }
  __syncthreads();
  const double h = Q.h;
  for (int64_t step = 0; step < Q.nsub; ++step)
    for (int s = 0; s < 4; ++s) {
      if (Q.store && live) Q.store[(step * 4 + s) * k * k + ei + ej * k] = sp[ei * SP + ej];
      f64x4_t pa[NB][NB];
#pragma unroll
      for (int cbk = 0; cbk < NB; ++cbk)
#pragma unroll
        for (int db = 0; db < NB; ++db) pa[cbk][db] = (f64x4_t){0.0, 0.0, 0.0, 0.0};
      for (int bb = 0; bb < NB; ++bb) {  // columns b of Z
        double sb[NJ];
#pragma unroll
        for (int j = 0; j < NJ; ++j) sb[j] = sp[(4 * j + lk) * SP + 16 * bb + lr];
        for (int c = wave; c < k; c += 16) {
          f64x4_t yc[NB];
#pragma unroll
          for (int eb = 0; eb < NB; ++eb) {  // Y = W_c S, rows 16 eb ..
            f64x4_t a0 = {0.0, 0.0, 0.0, 0.0}, a1 = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
              const double w = NB == 1 ? wr[NB == 1 ? j : 0] : wat(c, 16 * eb + lr, 4 * j + lk);
              if (j & 1) a1 = __builtin_amdgcn_mfma_f64_16x16x4f64(w, sb[j], a1, 0, 0, 0);
              else a0 = __builtin_amdgcn_mfma_f64_16x16x4f64(w, sb[j], a0, 0, 0, 0);
            }
            yc[eb] = a0 + a1;
          }
#pragma unroll
          for (int ab = 0; ab < NB; ++ab) {  // Z_c = S' Y, rows 16 ab ..
            f64x4_t a0 = {0.0, 0.0, 0.0, 0.0}, a1 = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
              const double sa = ab == bb ? sb[j] : sp[(4 * j + lk) * SP + 16 * ab + lr];
              if (j & 1) a1 = __builtin_amdgcn_mfma_f64_16x16x4f64(sa, yc[j / 4][j % 4], a1, 0, 0, 0);
              else a0 = __builtin_amdgcn_mfma_f64_16x16x4f64(sa, yc[j / 4][j % 4], a0, 0, 0, 0);
            }
            a0 += a1;
#pragma unroll
            for (int u = 0; u < 4; ++u) zs[((16 * ab + 4 * u + lk) * NP + c) * kSZPitch + lr] = a0[u];
          }
        }
        if (bb == 0 && lin) {
#pragma unroll
          for (int cbk = 0; cbk < NB; ++cbk)
#pragma unroll
            for (int db = 0; db < NB; ++db) {
              const double sv = lin == 1 ? sp[(4 * jl + lk) * SP + 16 * db + lr] : sp[(16 * cbk + lr) * SP + 4 * jl + lk];
              pa[cbk][db] = lin == 1 ? __builtin_amdgcn_mfma_f64_16x16x4f64(gl[cbk], sv, pa[cbk][db], 0, 0, 0)
                                     : __builtin_amdgcn_mfma_f64_16x16x4f64(sv, gl[db], pa[cbk][db], 0, 0, 0);
            }
        }
        __syncthreads();
        for (int a = wave; a < k; a += 16) {
#pragma unroll
          for (int db = 0; db < NB; ++db)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              const double tv = NB == 1 ? tr[NB == 1 ? j : 0] : tat(a, 16 * bb + 4 * j + lk, 16 * db + lr);
#pragma unroll
              for (int cbk = 0; cbk < NB; ++cbk) {
                const int c = 16 * cbk + lr;
                // the rows c >= k of zs are never written
                const double z = c < k ? zs[(a * NP + c) * kSZPitch + 4 * j + lk] : 0.0;
                pa[cbk][db] = __builtin_amdgcn_mfma_f64_16x16x4f64(z, tv, pa[cbk][db], 0, 0, 0);
              }
            }
        }
        if (NB > 1) __syncthreads();  // zs is free again
      }
      double p = 0.0;
#pragma unroll
      for (int cbk = 0; cbk < NB; ++cbk) {
#pragma unroll
        for (int db = 0; db < NB; ++db)
#pragma unroll
          for (int u = 0; u < 4; ++u)
            pp[((wave * 16 + 4 * u + lk) * NB + db) * kSZPitch + lr] = pa[cbk][db][u];
        __syncthreads();
        if (elem && (ei >> 4) == cbk) {
#pragma unroll
          for (int w = 0; w < 16; ++w) p += pp[((w * 16 + (ei & 15)) * NB + (ej >> 4)) * kSZPitch + (ej & 15)];
        }
        if (NB > 1) __syncthreads();
      }
      if (live) {
        const double f = Q.sgn * (cb - p);
        double x;
        if (s < 3) {
          acc = (s == 0 ? 0.0 : acc) + stage_w(s) * f;
          x = y0 + stage_c(s) * h * f;
        } else {
          x = y0 = y0 + (h / 6.0) * (acc + f);
        }
        sp[ei * SP + ej] = x;
      }
      __syncthreads();
    }
  if (Q.S1 && live) Q.S1[ei + ej * Q.lds1] = y0;
}

hipError_t launch_quad_sstep(const QuadSArgs& Q, hipStream_t st) {
  if (Q.k < 1 || Q.k > kQuadMaxRank || Q.q < 0 || Q.q > kMaxForce || !Q.W || !Q.T || !Q.Ga || !Q.Gb)
    return hipErrorInvalidValue;
  if (Q.k <= 16) hipLaunchKernelGGL(k_quad_sstep<1>, dim3(1), dim3(1024), 0, st, Q);
  else hipLaunchKernelGGL(k_quad_sstep<2>, dim3(1), dim3(1024), 0, st, Q);
  return hipGetLastError();
}

}  // namespace lri
