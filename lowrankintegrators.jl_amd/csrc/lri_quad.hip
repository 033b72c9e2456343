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
//   S' = sgn (Ga S + S Gb + cb - P(S)),  P_cd = sum_{a b} Z_abc T_abd,
//   Z_abc = sum_e S_ea Y_ebc,  Y_ebc = sum_f S_fb W_efc,
// S k x l in LDS, Y (k x l x k) and Z (l x l x k) in global scratch; one workgroup.
// ----------------------------------------------------------------------------

// kLds: the state, its RK4 work, the tensors W, T and the contractions Y, Z all
// in LDS (quad_s_lds_doubles(k, l) <= kQuadSLds), else Y, Z in Q.work and W, T read
// from global memory.
constexpr int kQuadSLds = 20400;  // 159 KB of the 160 KB LDS

__host__ __device__ inline int quad_s_lds_doubles(int k, int l) {
  return 5 * k * l + k * l * k + l * l * k + k * k * k + l * l * l;
}

template <bool kLds>
__global__ __launch_bounds__(1024) void k_quad_sstep(QuadSArgs Q) {
  __shared__ double st_small[kLds ? 1 : 5 * kQuadMaxRank * kQuadMaxRank];
  extern __shared__ double dyn[];
  const int k = Q.k, l = Q.l, t = threadIdx.x, nt = blockDim.x;
  const int kl = k * l;
  double* base = kLds ? dyn : st_small;
  double* y0 = base;
  double* ys = y0 + kl;
  double* acc = ys + kl;
  double* cb = acc + kl;
  double* pv = cb + kl;                          // the quadratic term P of a stage
  double* Y = kLds ? pv + kl : Q.work;           // k x l x k: Y[c + k (e + k b)]
  double* Z = Y + k * l * k;                     // l x l x k: Z[c + k (a + l b)]
  const double* W = Q.W;
  const double* T = Q.T;
  if (kLds && Q.W) {
    double* w = Z + l * l * k;
    double* tt = w + k * k * k;
    for (int e = t; e < k * k * k; e += nt) w[e] = Q.W[e];
    for (int e = t; e < l * l * l; e += nt) tt[e] = Q.T[e];
    W = w;
    T = tt;
  }
  for (int e = t; e < kl; e += nt) {
    const int i = e % k, j = e / k;
    y0[e] = Q.transS0 ? Q.S0[j + i * Q.lds0] : Q.S0[i + j * Q.lds0];
    double s = 0.0;
    for (int qq = 0; qq < Q.q; ++qq) s += Q.gaT[qq + i * Q.q] * Q.hbT[qq + j * Q.q];
    cb[e] = s;
  }
  __syncthreads();
  const double h = Q.h;
  for (int64_t step = 0; step < Q.nsub; ++step) {
    for (int e = t; e < kl; e += nt) ys[e] = y0[e];
    __syncthreads();
    for (int s = 0; s < 4; ++s) {
      if (Q.W) {
        // on the matrix cores: Y_(c + k e), b = sum_f W_(c + k e), f S_fb;  Z_(c, a), b = sum_e Y_(c, e), b S_ea;
        // P_ij = sum_(a + l b) Z_i, (a + l b) T_(a + l b), j  (into pv)
        const int kk2 = k * k;
        wave_gemm(kk2, l, k, 1, [&](int, int m, int f) { return W[m + kk2 * f]; },
                  [&](int, int f, int b) { return ys[f + b * k]; },
                  [&](int, int m, int b, double v) { Y[m + kk2 * b] = v; });
        __syncthreads();
        wave_gemm(k, l, k, l, [&](int b, int c, int e) { return Y[c + k * e + kk2 * b]; },
                  [&](int, int e, int a) { return ys[e + a * k]; },
                  [&](int b, int c, int a, double v) { Z[c + k * a + k * l * b] = v; });
        __syncthreads();
        wave_gemm(k, l, l * l, 1, [&](int, int i, int ab) { return Z[i + k * ab]; },
                  [&](int, int ab, int j) { return T[j + l * ab]; },
                  [&](int, int i, int j, double v) { pv[i + j * k] = v; });
        __syncthreads();
      }
      double fv[(kQuadMaxRank * kQuadMaxRank + 1023) / 1024];
      int cnt = 0;
      for (int e = t; e < kl; e += nt, ++cnt) {
        const int i = e % k, j = e / k;
        double v = cb[e];
        for (int m = 0; m < k; ++m) v += Q.Ga[i + m * k] * ys[m + j * k];
        for (int m = 0; m < l; ++m) v += ys[i + m * k] * Q.Gb[m + j * l];
        if (Q.W) v -= pv[e];
        fv[cnt] = Q.sgn * v;
      }
      __syncthreads();  // every stage input read before it is replaced
      cnt = 0;
      for (int e = t; e < kl; e += nt, ++cnt) {
        const double f = fv[cnt];
        if (s < 3) {
          acc[e] = (s == 0 ? 0.0 : acc[e]) + stage_w(s) * f;
          ys[e] = y0[e] + stage_c(s) * h * f;
        } else {
          y0[e] = y0[e] + (h / 6.0) * (acc[e] + f);
        }
      }
      __syncthreads();
    }
  }
  for (int e = t; e < kl; e += nt) Q.S1[(e % k) + (e / k) * Q.lds1] = y0[e];
}

hipError_t launch_quad_sstep(const QuadSArgs& Q, hipStream_t st) {
  if (Q.k < 1 || Q.l < 1 || Q.k > kQuadMaxRank || Q.l > kQuadMaxRank || Q.q < 0 || Q.q > kMaxForce || !Q.work)
    return hipErrorInvalidValue;
  const int need = quad_s_lds_doubles(Q.k, Q.l);
  if (need <= kQuadSLds)
    hipLaunchKernelGGL(k_quad_sstep<true>, dim3(1), dim3(1024), sizeof(double) * need, st, Q);
  else
    hipLaunchKernelGGL(k_quad_sstep<false>, dim3(1), dim3(1024), 0, st, Q);
  return hipGetLastError();
}

}  // namespace lri
