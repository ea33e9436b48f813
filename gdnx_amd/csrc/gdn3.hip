// GDN3 Kronecker-residual recurrence on gfx950: the fused per-chain forward
// (banded residual window + Kronecker read + periodic compaction), and the
// standalone compaction and Kronecker-read kernels.
//
// Reference semantics (frozen oracle gdn3/_reference_recurrence.py:33-94):
// per chain, state S = sum_r A_r (x) B_r + U Vb^T with a P-slot circular
// residual buffer.  Per token t: gamma = clamp(dec, 0, 1); A, B, Vb *= gamma;
// h = b.k; u = w.v; r = u - S h; alpha = alpha(k.h) (gdn3_upgrade.py:641-648);
// y = S q + alpha (k.q) r; slot t mod P <- (alpha r, k); after token t with
// (t+1) mod K_c == 0 the compaction (_compact_vec, gdn3_upgrade.py:650-719)
// refits A, B from R_mat = sum_r vec(A_r) vec(B_r)^T + rearrange(U Vb^T) by a
// randomized SVD and blends them (A <- s A + (1-s) A_svd, U, Vb unchanged).
//
// Chunked form (one chunk = the P-token window, aligned with the slots).
// With G_i the inclusive log-decay prefix inside the chunk, Gacc the log
// decay since the last compaction, U_old / Vbd the previous chunk's net
// writes and keys (keys decayed to the chunk start):
//   U_i = alpha_i (u_i - e^{2(Gacc+G_i)} Kr(h_i) - e^{G_i} sum_{p>=i} (h_i.Vbd_p) U_old_p)
//         - alpha_i sum_{j<i} e^{G_i-G_j} (h_i.k_j) U_j
//   y_i = e^{2(Gacc+G_i)} Kr(q_i) + e^{G_i} sum_{p>=i} (q_i.Vbd_p) U_old_p
//         + sum_{j<=i} e^{G_i-G_j} (q_i.k_j) U_j
// (slot p of the previous chunk is still visible to token i while p >= i;
// the Kronecker part decays by gamma^2 since A and B each decay by gamma).
// Kr(x) = (sum_r A_r (x) B_r) x is read on MFMA against the materialised
// d x d Kronecker matrix, rebuilt after every compaction.
//
// With a compaction after every window one workgroup per chain carries the
// whole state in LDS (gdn3_fused_kernel); its chunk loop is sequential because
// every compaction depends on the window it closes.  Longer intervals run in
// gdn3_long.hip, with a compaction launch between them.
#include <mutex>

#include "gdn3_common.hpp"
#include "gdnx_internal.hpp"

namespace gdnx {
namespace {

// Sum over the 64 lanes of a wave, the same bits in every lane: DPP row
// rotations by 8, 4, 2, 1 (a butterfly inside each 16-lane row, so all lanes
// of a row form the same sum), then across the four rows.
template <int CTL>
__device__ __forceinline__ double dpp_f64(double x) {
  const long long b = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(b & 0xffffffffll), CTL, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTL, 0xf, 0xf, false);
  return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}
// lane l's x, wave-uniform (l uniform)
__device__ __forceinline__ double readlane_f64(double x, int l) {
  const long long b = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffll), l);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
  return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}
// (the four row sums are read out of lanes 0, 16, 32, 48 and added as
// (r0 + r1) + (r2 + r3): a uniform value, no LDS round trip)
__device__ __forceinline__ double wave_sum_f64(double x) {
  x += dpp_f64<0x128>(x);
  x += dpp_f64<0x124>(x);
  x += dpp_f64<0x122>(x);
  x += dpp_f64<0x121>(x);
  return (readlane_f64(x, 0) + readlane_f64(x, 16)) + (readlane_f64(x, 32) + readlane_f64(x, 48));
}

// Sum of NV doubles over the 256 threads of the block, in a fixed order;
// every thread receives the totals.  red: 4 * NV doubles of LDS.
template <int NV>
__device__ __forceinline__ void block_sum(double (&v)[NV], double* red, int tid) {
#pragma unroll
  for (int e = 0; e < NV; ++e) v[e] = wave_sum_f64(v[e]);
  if ((tid & 63) == 0)
#pragma unroll
    for (int e = 0; e < NV; ++e) red[(tid >> 6) * NV + e] = v[e];
  __syncthreads();
#pragma unroll
  for (int e = 0; e < NV; ++e) v[e] = (red[e] + red[NV + e]) + (red[2 * NV + e] + red[3 * NV + e]);
  __syncthreads();
}

// LDS of one compaction.  STG: the window's writes and keys are staged
// through ut / vt a block of 16 slots at a time (they come from global
// memory); without, they are read where they lie (LDS of the fused kernel).
// Row stride (doubles) of the compaction's row-major [rows][kQ] double arrays:
// where a thread reads or writes a whole row, 9 doubles put the 64 lanes' rows
// on distinct bank pairs (a stride of 8 put 16 lanes on each).
constexpr int kLQ = kQ + 1;

template <int D, int P, bool STG = true>
struct G3Compact {
  static constexpr int m = G3D<D>::m, n = G3D<D>::n;
  static constexpr int ldr = n + 4;                 // R_mat row stride: 16-byte rows, 4 banks apart
  static constexpr int lym = m + 16, lzn = n + 16;  // strides of the column-major fp32 copies
  alignas(16) float rm[m * ldr];          // R_mat
  alignas(16) double y[m * kLQ];          // range basis, rows of kQ (stride kLQ)
  alignas(16) double z[n * kLQ];          // R_mat^T Y, then Bm^T = R_mat^T Q (rows of kQ, stride kLQ)
  alignas(16) float yt[kQ * lym];         // y in fp32, column-major: the B operand of R_mat^T Y
  alignas(16) float zt[kQ * lzn];         // the sketch (zero padded), then z, in fp32 column-major
  alignas(16) float ut[STG ? 16 : 1][D + 4];   // a block of 16 window slots: net writes U_p
  alignas(16) float vt[STG ? 16 : 1][D + 4];   // and keys Vb_p
  double red[4 * 64];
  double rinv[kQ * kQ];                   // the summed Gram Y^T Y of a Cholesky-QR pass (row-major)
  double ev[kQ * kQ];                     // eigenvectors of Bm Bm^T (rows, in rank order)
  double lam[kQ];
  double sig[kRMax];
  double isig[kRMax];                     // 1 / sig (0 where sig is)
  double sgn[kRMax];
};

// Partial Gram X^T X (kQ x kQ) of NR rows of X (rows of kQ doubles, stride
// kLQ) on v_mfma_f64_4x4x4_4b_f64, four rows per step: block b = 2 P + Q is
// the 4 x 4 block (P, Q) of the Gram, so all 64 outputs are live (a 16 x 16
// tile left three quarters of its outputs dead at four times the cycles).
// Lane l = 16 k + 4 b + i supplies X[k][4 P + i] as A[b][i][k] and X[k][4 Q + i]
// as B[b][k][i]; it returns G[4 P + l / 16][4 Q + l % 4], the row-major entry
// gram_entry(l).  Two accumulation chains (even and odd steps) hide the
// MFMA's dependent latency.
__device__ __forceinline__ int gram_entry(int lane) {
  const int b = (lane >> 2) & 3;
  return (4 * (b >> 1) + (lane >> 4)) * kQ + 4 * (b & 1) + (lane & 3);
}
template <int NR>
__device__ __forceinline__ double gram_mfma(const double* x, int lane) {
  static_assert(NR % 8 == 0, "two chains of 4-row steps");
  const int k = lane >> 4, b = (lane >> 2) & 3, i = lane & 3;
  const int ca = 4 * (b >> 1) + i, cb = 4 * (b & 1) + i;
  double acc0 = 0.0, acc1 = 0.0;
#pragma unroll
  for (int r = 0; r < NR; r += 8) {
    acc0 = __builtin_amdgcn_mfma_f64_4x4x4f64(x[(r + k) * kLQ + ca], x[(r + k) * kLQ + cb], acc0, 0, 0, 0);
    acc1 = __builtin_amdgcn_mfma_f64_4x4x4f64(x[(r + 4 + k) * kLQ + ca], x[(r + 4 + k) * kLQ + cb], acc1, 0, 0, 0);
  }
  return acc0 + acc1;
}

// C[M x kQ] = A[M x K] B[K x kQ] on fp32 MFMA: A is R_mat (fp32, row stride
// ldr, a multiple of 4) read as is (TRANS = false, M = m, K = n) or transposed
// (TRANS = true, M = n, K = m); B is fp32 and column-major (column j at bt +
// j ldb, zero where it has no column), so every product is exact and the sums
// are fp32.  v_mfma_f32_4x4x1_16b_f32 (16 blocks of 4 x 4 x 1, a quarter of the
// 16 x 16 x 4 instruction's cycles) takes the kQ = 8 columns as two blocks of
// 4, so no MFMA column is dead (16 x 16 tiles left half of theirs unused).
// Lane l = 4 b + q supplies row q of block b's A operand and column q of its B
// operand and holds D[b][r][q] in element r.  A wave owns RW = M / 4 rows of C; its 16 blocks are RG = RW / 4
// row groups times KP = 64 / RW partitions of k (k = 4 (KP t + p) + s for
// partition p, which puts the lanes of every LDS read on distinct banks),
// summed across the partitions (lane bits 4 and 5) at the end.  C goes to c
// (rows of kQ at stride kLQ, fp64) and, when ct is given, column-major in fp32
// to ct (stride ldc); GR: also this wave's partial Gram C^T C over its rows,
// in the layout of gram_mfma, formed from its rows of c.
template <bool TRANS, int M, int K, int ldr, int ldb, int ldc = 0, bool GR = false>
__device__ __forceinline__ void rm_mfma(const float* rm, const float* bt, double* c, float* ct, int tid,
                                         double* gp = nullptr) {
  constexpr int RW = M / 4, KP = 64 / RW, RG = RW / 4, NG = K / (4 * KP), BATCH = 4;
  static_assert(RW == 16 || RW == 64, "a wave's rows: one or four partitions of k");
  static_assert(NG % BATCH == 0 && ldr % 4 == 0 && ldb % 4 == 0 && ldc % 4 == 0, "whole batches, 16-byte rows");
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int b = lane >> 2, q = lane & 3, kp = b / RG, rg = b % RG;
  const int row = wave * RW + 4 * rg + q;   // the A row this lane supplies
  auto lda = [&](int t) {
    const int k0 = 4 * (KP * t + kp);
    f32x4 x;
    if constexpr (TRANS) {
#pragma unroll
      for (int s4 = 0; s4 < 4; ++s4) x[s4] = rm[(k0 + s4) * ldr + row];
    } else {
      x = *(const f32x4*)&rm[row * ldr + k0];
    }
    return x;
  };
  f32x4 c1 = {0.f, 0.f, 0.f, 0.f}, c2 = {0.f, 0.f, 0.f, 0.f};   // columns q and 4 + q
#pragma unroll
  for (int t0 = 0; t0 < NG; t0 += BATCH) {
    f32x4 av[BATCH], b1[BATCH], b2[BATCH];
#pragma unroll
    for (int u = 0; u < BATCH; ++u) {
      const int k0 = 4 * (KP * (t0 + u) + kp);
      av[u] = lda(t0 + u);
      b1[u] = *(const f32x4*)&bt[q * ldb + k0];
      b2[u] = *(const f32x4*)&bt[(4 + q) * ldb + k0];
    }
    __builtin_amdgcn_sched_barrier(0);   // (the scheduler would interleave them again)
#pragma unroll
    for (int u = 0; u < BATCH; ++u)
#pragma unroll
      for (int s4 = 0; s4 < 4; ++s4) {
        c1 = __builtin_amdgcn_mfma_f32_4x4x1f32(av[u][s4], b1[u][s4], c1, 0, 0, 0);
        c2 = __builtin_amdgcn_mfma_f32_4x4x1f32(av[u][s4], b2[u][s4], c2, 0, 0, 0);
      }
  }
  if constexpr (KP > 1) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      c1[r] = sum_rows4(c1[r]);
      c2[r] = sum_rows4(c2[r]);
    }
  }
  // rows r0 + r of C; with KP = 4 the four partitions' lanes share the stores
  const int r0 = wave * RW + 4 * rg;
  if (KP == 1 || kp == 0)
#pragma unroll
    for (int r = 0; r < 4; ++r) c[(r0 + r) * kLQ + q] = (double)c1[r];
  if (KP == 1 || kp == 1)
#pragma unroll
    for (int r = 0; r < 4; ++r) c[(r0 + r) * kLQ + 4 + q] = (double)c2[r];
  if constexpr (ldc > 0) {
    if (KP == 1 || kp == 2) *(f32x4*)&ct[q * ldc + r0] = c1;
    if (KP == 1 || kp == 3) *(f32x4*)&ct[(4 + q) * ldc + r0] = c2;
  }
  if constexpr (GR) {
    wave_lds_sync();   // the wave's rows of c, written by its lanes above
    *gp = gram_mfma<RW>(c + wave * RW * kLQ, lane);
  }
}

// 1 / sqrt(x) for x > 0 to fp64 rounding: the hardware estimate r0 and the
// Halley-order correction r0 (1 + t/2 + 3 t^2/8), t = 1 - x r0^2 (error
// O(t^3)).  x = 0 gives a NaN (callers select it away).
__device__ __forceinline__ double rsqrt_f64(double x) {
  const double r0 = __builtin_amdgcn_rsq(x);
  const double t = fma(-x * r0, r0, 1.0);
  return fma(r0 * t, fma(t, 0.375, 0.5), r0);
}

// Jacobi rotation zeroing a_pq (Numerical Recipes convention):
// J[p][p] = J[q][q] = c, J[p][q] = s, J[q][p] = -s, with the smaller angle
// t = sgn(th) / (|th| + sqrt(th^2 + 1)), th = (a_qq - a_pp) / (2 a_pq).
// Multiplying through by |2 a_pq| gives it without divisions: with
// d = a_qq - a_pp, e = 2 a_pq, h = sqrt(d^2 + e^2) and w = |d| + h,
// t = sgn(d) e / w, so c = w / sqrt(w^2 + e^2), s = sgn(d) e / sqrt(w^2 + e^2)
// (c^2 + s^2 = 1 by construction; d = +0 counts as positive, and at d = 0
// either sign of the 45-degree rotation zeroes a_pq).
__device__ __forceinline__ void jacobi_rot(double app, double aqq, double apq, double& c, double& s) {
  // the round is bound by its instruction count (one wave issues it), so no
  // selects: h only sets the angle (x times the hardware reciprocal square
  // root, about 2^-23 relative, 0 at x = 0; a rotation that leaves 1e-7 of
  // a_pq behind still converges within the same sweeps), w carries 2^-500,
  // which vanishes against any |d| or h above 2^-447 and makes d = e = 0 give
  // c = 1, s = 0, and sgn(d) e is a sign-bit copy.  c and s are normalised by
  // the refined reciprocal square root, so c^2 + s^2 = 1 to rounding.
  const double d = aqq - app, e = 2.0 * apq;
  const double e2 = e * e;
  const double x = fma(d, d, e2);
  const double h = x * __builtin_amdgcn_rsq(fmax(x, 2.2250738585072014e-308));
  const double w = (fabs(d) + 3.0549363634996047e-151) + h;
  const double r = rsqrt_f64(fma(w, w, e2));
  const long long sb = __double_as_longlong(d) & (long long)0x8000000000000000ull;
  c = w * r;
  s = __longlong_as_double(__double_as_longlong(e) ^ sb) * r;
}

// x as held by lane src of the wave (ds_bpermute, one per 32-bit half)
__device__ __forceinline__ double lane_f64(int src, double x) {
  const long long v = __double_as_longlong(x);
  const unsigned lo = (unsigned)__builtin_amdgcn_ds_bpermute(4 * src, (int)(unsigned)v);
  const unsigned hi = (unsigned)__builtin_amdgcn_ds_bpermute(4 * src, (int)(unsigned)(v >> 32));
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// Round-robin (circle method) partner of index x in round st of 7 for 8 indices.
__device__ __forceinline__ int rr_partner(int x, int st) {
  if (x == 7) return st;
  if (x == st) return 7;
  return (2 * st - x + 14) % 7;
}

// One Cholesky-QR pass leaves Q^T Q - I at about cond(Y)^2 * 1.1e-16 in fp64;
// the pivots' spread (largest / smallest, about cond(Y)^2) below this bound
// makes a second pass unnecessary (Q orthonormal to ~1e-10).
constexpr double kOrthCut = 1e6;
// Pivot spread (about cond(Y)^2) below which an intermediate basis enters the
// next product unnormalised: cond(Y) < 10 costs the fp32 products at most a
// decimal digit in its weakest direction, against their 1e-7
constexpr double kKeepCut = 1e2;

// Y <- Y R^{-1} with Y^T Y = R^T R (Cholesky QR, up to `passes` times: one
// pass keeps the intermediate power-iteration bases well conditioned; the
// final basis takes a second where the first pass's pivots spread by more
// than kOrthCut or a column was dropped); the result also goes column-major in fp32 to yt.  Columns whose pivot falls below 1e-24 of the largest
// diagonal are set to zero.  The Gram runs on fp64 MFMA over 4 row segments;
// each row of Y is then solved against R by forward substitution.
template <int D, int P, int M, bool STG>
__device__ __forceinline__ void orth_rows(G3Compact<D, P, STG>& cs, int tid, int passes, const double* pre = nullptr,
                                          double keep = 0.0) {
  static_assert(M % 16 == 0 && M <= kNT, "rows: 4 segments of whole MFMA steps, one row per thread");
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  constexpr int seg = M / 4;
  for (int pass = 0; pass < passes; ++pass) {
    {   // this wave's partial Gram (the first pass's may come from the product that formed Y)
      const double g = (pass == 0 && pre) ? *pre : gram_mfma<seg>(cs.y + wave * seg * kLQ, lane);
      cs.red[wave * 64 + gram_entry(lane)] = g;
    }
    __syncthreads();
    if (wave == 0)   // the Gram, summed over the segments (rinv holds it row-major)
      cs.rinv[lane] = (cs.red[lane] + cs.red[64 + lane]) + (cs.red[128 + lane] + cs.red[192 + lane]);
    __syncthreads();
    // every thread factors the 8 x 8 Gram itself, in registers (right-looking
    // Cholesky, lower triangle; a dropped column gets rd = 0), and solves its
    // row of Y against R = L^T: no second exchange through LDS
    double L[kQ][kQ], rdv[kQ];
#pragma unroll
    for (int i = 0; i < kQ; ++i)
#pragma unroll
      for (int j = 0; j <= i; ++j) L[i][j] = cs.rinv[i * kQ + j];
    double dmax = 0.0;
#pragma unroll
    for (int k = 0; k < kQ; ++k) dmax = fmax(dmax, L[k][k]);
    const double tol = dmax * 1e-24;
    double pmin = dmax, pmax = 0.0;   // the spread of the pivots
#pragma unroll
    for (int k = 0; k < kQ; ++k) {
      const double akk = L[k][k];
      pmin = fmin(pmin, akk);
      pmax = fmax(pmax, akk);
      const double rq = rsqrt_f64(fmax(akk, 2.2250738585072014e-308));  // unconditional: a select, no branch
      const double rd = (akk > tol && akk > 0.0) ? rq : 0.0;
      rdv[k] = rd;   // 1 / R[k][k] (R[k][k] = akk rd = sqrt(akk))
#pragma unroll
      for (int i = k + 1; i < kQ; ++i) L[i][k] *= rd;
#pragma unroll
      for (int i = k + 1; i < kQ; ++i)
#pragma unroll
        for (int j = k + 1; j <= i; ++j) L[i][j] -= L[i][k] * L[j][k];
    }
    // keep > 0 (an intermediate basis, whose fp32 copy the product wrote):
    // where the pivots spread by less than keep, Y is conditioned well enough
    // to enter the next product as it is (the basis only has to stay well
    // conditioned; its span is what the power iteration carries)
    if (keep > 0.0 && __builtin_amdgcn_readfirstlane(pmin * keep > pmax ? 1 : 0)) return;
    if (tid < M) {
      double x[kQ];
#pragma unroll
      for (int j = 0; j < kQ; ++j) x[j] = cs.y[tid * kLQ + j];
      // x R = y, column by column: x_j = (y_j - sum_{i<j} x_i R[i][j]) / R[j][j], R[i][j] = L[j][i]
#pragma unroll
      for (int j = 0; j < kQ; ++j) {
        double sacc = x[j];
#pragma unroll
        for (int i = 0; i < j; ++i) sacc -= x[i] * L[j][i];
        x[j] = sacc * rdv[j];
      }
#pragma unroll
      for (int j = 0; j < kQ; ++j) {
        cs.y[tid * kLQ + j] = x[j];
        cs.yt[j * cs.lym + tid] = (float)x[j];
      }
    }
    __syncthreads();
    // a later pass only where this one can have lost orthogonality: every
    // thread factored the same Gram, so the test is uniform
    if (pass + 1 < passes && __builtin_amdgcn_readfirstlane(pmin * kOrthCut > pmax ? 1 : 0)) break;
  }
}

// Sums of squares of the first kRMax columns of a row-major [M][kQ] double
// array, into out[0..kRMax) (every thread waits for them).
template <int M>
__device__ __forceinline__ void col_sumsq(const double* y, double* red, double* out, int tid) {
  const int r = tid & (kRMax - 1), lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  double part = 0.0;
  for (int row = tid / kRMax; row < M; row += kNT / kRMax) {
    const double x = y[row * kLQ + r];
    part += x * x;
  }
#pragma unroll
  for (int off = kRMax; off < 64; off <<= 1) part += __shfl_xor(part, off, 64);
  if (lane < kRMax) red[wave * kRMax + lane] = part;
  __syncthreads();
  if (tid < kRMax) out[tid] = (red[tid] + red[kRMax + tid]) + (red[2 * kRMax + tid] + red[3 * kRMax + tid]);
  __syncthreads();
}

struct G3NoOp {
  __device__ void operator()() const {}
};

// Compaction of one chain (gdn3/gdn3_upgrade.py:650-719): ab = [A (R x m) |
// B (R x n)] in LDS as stored (the Kronecker part is decayed by e^{gacc} per
// factor); the window's P net writes U and keys Vb (decayed to now) are read
// from global memory, slot p column d at p u_sp + d u_sd.  Writes the blended A, B back into ab and, from
// thread 0, stats = (|R_mat|^2, sum of the R kept sigma^2).  Sign
// convention: each (u_r, v_r) pair is flipped so that the largest-magnitude
// entry of v_r is positive (first index on ties).
// mode 1 is the reference's 'sketch' / 'sketch_noqr' (both run the same
// branch, gdn3/gdn3_upgrade.py:579-592): no range finder and no SVD, with a
// sketch of qs = R columns, Q = the column-normalised R_mat G,
// Bm = Q^T R_mat, A_svd_r = |Bm_r| Q_r, B_svd_r = Bm_r / |Bm_r| (norms
// clamped at 1e-12); it reports no error (stats = (|R_mat|^2, |R_mat|^2)).
// issue / commit: work of the caller's that uses no compaction state and
// runs in the eigen-solve's shadow (every thread calls issue before it; waves
// 1-3 call commit while wave 0 solves, wave 0 after); 'svd' mode only.
// pre: the sketch entries this thread stages, loaded by the caller (a chain's
// sketch is the same at every compaction), else they are loaded here.
template <int D>
struct G3Sketch {
  static constexpr int N = (G3D<D>::n * kQ + kNT - 1) / kNT;
  float v[N];   // entry e = tid + u kNT: sketch row e / kQ, column e % kQ (zero past its qs columns)
};
template <int D>
__device__ __forceinline__ void g3_sketch_load(G3Sketch<D>& g, const float* __restrict__ sketch, int qs, int tid) {
#pragma unroll
  for (int u = 0; u < G3Sketch<D>::N; ++u) {
    const int e = tid + u * kNT, c = e / kQ, j = e % kQ;
    g.v[u] = (e < G3D<D>::n * kQ && j < qs) ? sketch[c * qs + j] : 0.f;
  }
}
template <int D, int P, bool STG, typename Issue = G3NoOp, typename Commit = G3NoOp>
__device__ __forceinline__ void g3_compact(G3Compact<D, P, STG>& cs, float* ab, const float* __restrict__ U,
                                           const float* __restrict__ Vb, size_t u_sp, size_t u_sd, float gacc,
                                           float sdec, const float* __restrict__ sketch, double* stats, int tid,
                                           int mode = 0, Issue issue = Issue(), Commit commit = Commit(),
                                           const G3Sketch<D>* pre = nullptr) {
  typedef G3D<D> Ge;
  constexpr int R = Ge::R, m = Ge::m, n = Ge::n, q = Ge::q, ak = Ge::ak, bk = Ge::bk;
  constexpr int lbv = Ge::lbv, lbk = Ge::lbk, ln = Ge::ln;
  constexpr int ldr = G3Compact<D, P, STG>::ldr, lym = G3Compact<D, P, STG>::lym, lzn = G3Compact<D, P, STG>::lzn;
  float* A = ab;
  float* Bv = ab + R * m;
  tid = opaque(tid);
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  // the sketch's global loads (unless the caller holds it) are issued first
  // and land in LDS after the residual part (which does not read them)
  constexpr int NGS = G3Sketch<D>::N;
  G3Sketch<D> gs;
  if (pre) gs = *pre;
  else g3_sketch_load<D>(gs, sketch, mode ? R : q, tid);
  double en[1] = {0.0};
  // residual part rearrange(U Vb^T) on fp32 MFMA: out[v][k] = sum_p U_p[v] Vb_p[k]
  // (A[v][p] = U_p[v], B[p][k] = Vb_p[k]), accumulated over the window's
  // blocks of 16 slots staged through LDS; wave w owns the value-row tiles
  // w VTW .. w VTW + VTW - 1 against every key-column tile, and scatters each
  // entry to its rearranged place (iv a_k + ik, jv b_k + jk)
  {
    constexpr int NT16 = D / 16, VTW = NT16 / 4;
    static_assert(NT16 % 4 == 0 && P % 16 == 0, "whole 16x16 tiles on 4 waves, blocks of 16 window slots");
    const int g4 = lane >> 4, n16 = lane & 15;
    f32x4 racc[VTW][NT16];
#pragma unroll
    for (int vi = 0; vi < VTW; ++vi)
#pragma unroll
      for (int kt = 0; kt < NT16; ++kt) racc[vi][kt] = (f32x4){0.f, 0.f, 0.f, 0.f};
    for (int pb = 0; pb < P / 16; ++pb) {
      if constexpr (STG) {
        if (pb > 0) __syncthreads();   // the previous block is consumed
        for (int e = tid; e < 16 * D; e += kNT) {
          const int i = e / D, d = e % D;
          const size_t o = (size_t)(16 * pb + i) * u_sp + (size_t)d * u_sd;
          cs.ut[i][d] = U[o];
          cs.vt[i][d] = Vb[o];
        }
        __syncthreads();
      }
      // slot 16 pb + i, column d
      auto uval = [&](int i, int d) {
        if constexpr (STG) return cs.ut[i][d];
        else return U[(size_t)(16 * pb + i) * u_sp + (size_t)d * u_sd];
      };
      auto vval = [&](int i, int d) {
        if constexpr (STG) return cs.vt[i][d];
        else return Vb[(size_t)(16 * pb + i) * u_sp + (size_t)d * u_sd];
      };
      // every operand read before the MFMAs, behind a scheduling barrier (the
      // compiler, short of registers, waited for each tile's reads); the
      // key fragments serve every value tile
      f32x4 ua[VTW], kb4[NT16];
#pragma unroll
      for (int vi = 0; vi < VTW; ++vi)
#pragma unroll
        for (int s4 = 0; s4 < 4; ++s4) ua[vi][s4] = uval(4 * g4 + s4, (wave * VTW + vi) * 16 + n16);
#pragma unroll
      for (int kt = 0; kt < NT16; ++kt)
#pragma unroll
        for (int s4 = 0; s4 < 4; ++s4) kb4[kt][s4] = vval(4 * g4 + s4, kt * 16 + n16);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int vi = 0; vi < VTW; ++vi)
#pragma unroll
        for (int kt = 0; kt < NT16; ++kt) mma(racc[vi][kt], ua[vi], kb4[kt]);
    }
    // plus the Kronecker part sum_r A_r[iv][ik] B_r[jv][jk] (each factor decayed
    // by e^{gacc}), and the energy |R_mat|^2.  With b_v = b_k = 8 a lane's
    // jk = n16 mod 8 and jv = (4 g4 + i) mod 8 are fixed (its B entries load
    // once), iv = 2 vt + g4 / 2 follows the value tile and ik = 2 kt + n16 / 8
    // the key tile (R A entries per tile pair, 4 addresses per wave)
    static_assert(Ge::bv == 8 && Ge::bk == 8, "lane-fixed Kronecker columns");
    const float sc2 = expf(2.f * gacc);
    float bl[4][kRMax];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int r = 0; r < kRMax; ++r)
        bl[i][r] = r < R ? sc2 * Bv[r * n + ((4 * g4 + i) & 7) * bk + (n16 & 7)] : 0.f;
    double e4[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int vi = 0; vi < VTW; ++vi) {
      const int vt = wave * VTW + vi, iv = 2 * vt + (g4 >> 1);
      float alv[NT16][kRMax];   // (read before use, as above)
#pragma unroll
      for (int kt = 0; kt < NT16; ++kt)
#pragma unroll
        for (int r = 0; r < kRMax; ++r) alv[kt][r] = r < R ? A[r * m + iv * ak + 2 * kt + (n16 >> 3)] : 0.f;
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int kt = 0; kt < NT16; ++kt) {
        const int ik = 2 * kt + (n16 >> 3), jk = n16 & 7, row = iv * ak + ik;
        const float* al = alv[kt];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int jv = (4 * g4 + i) & 7;
          float sv = racc[vi][kt][i];
#pragma unroll
          for (int r = 0; r < kRMax; ++r)
            if (r < R) sv += al[r] * bl[i][r];
          cs.rm[row * ldr + jv * bk + jk] = sv;
          e4[i] += (double)sv * (double)sv;
        }
      }
    }
    en[0] = (e4[0] + e4[1]) + (e4[2] + e4[3]);
  }
#pragma unroll
  for (int u = 0; u < NGS; ++u) {
    const int e = tid + u * kNT;
    if (e < n * kQ) cs.zt[(e % kQ) * lzn + e / kQ] = gs.v[u];
  }
  block_sum<1>(en, cs.red, tid);

  if (mode) {   // 'sketch': one product, column and row normalisation
    rm_mfma<false, m, n, ldr, lzn>(cs.rm, cs.zt, cs.y, nullptr, tid);   // Y = R_mat G (columns >= R are zero)
    __syncthreads();
    col_sumsq<m>(cs.y, cs.red, cs.lam, tid);
    for (int e = tid; e < m * kQ; e += kNT) {
      const int j = e % kQ;
      const double qv = j < R ? cs.y[(e / kQ) * kLQ + j] / fmax(sqrt(cs.lam[j]), 1e-12) : 0.0;   // Q
      cs.y[(e / kQ) * kLQ + j] = qv;
      cs.yt[j * lym + e / kQ] = (float)qv;
    }
    __syncthreads();
    rm_mfma<true, n, m, ldr, lym>(cs.rm, cs.yt, cs.z, nullptr, tid);      // Bm^T = R_mat^T Q
    __syncthreads();
    col_sumsq<n>(cs.z, cs.red, cs.sig, tid);
    const float dk = expf(gacc);
    const float s1 = sdec, s2 = 1.f - sdec;
    for (int e = tid; e < R * m; e += kNT) {
      const int r = e / m, row = e % m;
      const double sv = cs.y[row * kLQ + r] * fmax(sqrt(cs.sig[r]), 1e-12);
      A[e] = s1 * (A[e] * dk) + s2 * (float)sv;
    }
    for (int e = tid; e < R * n; e += kNT) {
      const int r = e / n, col = e % n;
      const double sv = cs.z[col * kLQ + r] / fmax(sqrt(cs.sig[r]), 1e-12);
      Bv[e] = s1 * (Bv[e] * dk) + s2 * (float)sv;
    }
    if (tid == 0 && stats) {
      stats[0] = en[0];
      stats[1] = en[0];
    }
    __syncthreads();
    return;
  }

  // range finder with two power iterations; orthonormalising between the
  // products leaves the final basis unchanged (up to column signs)
  // (each Y = R_mat Z product hands its partial Grams straight to the first
  // Cholesky-QR pass, whose barrier then also publishes Y)
  double gp;
  rm_mfma<false, m, n, ldr, lzn, lym, true>(cs.rm, cs.zt, cs.y, cs.yt, tid, &gp);
  orth_rows<D, P, m, STG>(cs, tid, 1, &gp, kKeepCut);
  for (int it = 0; it < 2; ++it) {
    rm_mfma<true, n, m, ldr, lym, lzn>(cs.rm, cs.yt, cs.z, cs.zt, tid);
    __syncthreads();
    rm_mfma<false, m, n, ldr, lzn, lym, true>(cs.rm, cs.zt, cs.y, cs.yt, tid, &gp);
    orth_rows<D, P, m, STG>(cs, tid, it == 1 ? 2 : 1, &gp, it == 1 ? 0.0 : kKeepCut);
  }
  // Bm^T = R_mat^T Q  [n][kQ]
  rm_mfma<true, n, m, ldr, lym>(cs.rm, cs.yt, cs.z, nullptr, tid);
  __syncthreads();
  {  // W = Bm Bm^T: each wave's partial Gram over a quarter of the rows of Bm^T
    static_assert(n % 32 == 0, "quarters of whole MFMA steps");
    cs.red[wave * 64 + gram_entry(lane)] = gram_mfma<n / 4>(cs.z + wave * (n / 4) * kLQ, lane);
  }
  __syncthreads();
  issue();
  // eigen-decomposition of W = Bm Bm^T by cyclic Jacobi in wave 0: lane
  // (i, j) holds W[i][j] and V[i][j].  Each round rotates 4 disjoint pairs;
  // a lane gathers every operand of its round in one exchange and forms the
  // rotation of its column's pair (that of j); the rotation of i it takes
  // from lane (i, i), whose column pair that is.  The exchange goes through
  // LDS (xa, xv), ordered by wave_lds_sync (the next round's writes depend
  // on this round's reads, so they cannot move above them).
  if (wave == 0) {
    const int i = lane >> 3, j = lane & 7;
    double* xa = cs.rinv;   // 64 doubles each, free after the last Cholesky-QR pass
    double* xv = cs.ev;
    double a;
    {  // the partials summed, upper entry for both (i, j) and (j, i)
      const int e = min(i, j) * kQ + max(i, j);
      a = (cs.red[e] + cs.red[64 + e]) + (cs.red[128 + e] + cs.red[192 + e]);
    }
    double vv = (i == j) ? 1.0 : 0.0;
    // |W|_F^2, which the rotations keep: the diagonal's mass is fro - off
    const double fro = wave_sum_f64(a * a);
    for (int sweep = 0; sweep < 12; ++sweep) {
      if (sweep >= 4) {   // (fewer than four sweeps rarely suffice; extra sweeps over a diagonal W rotate by identities)
        const double off = wave_sum_f64(i != j ? a * a : 0.0);
        // stop at off-diagonal entries ~1e-8 of the diagonal's (in norm): the
        // eigenvectors then sit within ~1e-8 / (relative gap) of W's, an order
        // below what the fp32 products that formed Bm already left in W
        if (!(off > 1e-16 * (fro - off))) break;  // uniform across the wave
      }
#pragma unroll
      for (int st = 0; st < 7; ++st) {
        const int pi = rr_partner(i, st), pj = rr_partner(j, st);
        const int j0 = min(j, pj), j1 = max(j, pj);
        xa[lane] = a;
        xv[lane] = vv;
        wave_lds_sync();
        const double aj0 = xa[9 * j0], aj1 = xa[9 * j1], ajo = xa[8 * j0 + j1];
        const double a_ipj = xa[8 * i + pj], a_pij = xa[8 * pi + j];
        const double a_pipj = xa[8 * pi + pj], v_ipj = xv[8 * i + pj];
        double cj, sj;
        jacobi_rot(aj0, aj1, ajo, cj, sj);
        // J[x][x] = c; J[partner][x] = -s if x < partner else +s
        const double xj = (j < pj) ? -sj : sj;
        // the rotation of i: lane (i, i) formed it as the rotation of its column
        const double ci = lane_f64(9 * i, cj), xi = lane_f64(9 * i, xj);
        a = cj * fma(ci, a, xi * a_pij) + xj * fma(ci, a_ipj, xi * a_pipj);
        vv = vv * cj + v_ipj * xj;
      }
    }
    // (still wave 0 alone, ordered by wave_lds_sync) the rank of eigenvalue j,
    // descending, ties by index; the eigenvectors in rank order,
    // ev[r][i] = component i of the r-th; the kept singular values
    if (i == j) cs.lam[i] = a;
    wave_lds_sync();
    const double lj = cs.lam[j];
    int rk = 0;
#pragma unroll
    for (int k = 0; k < kQ; ++k) rk += (cs.lam[k] > lj || (cs.lam[k] == lj && k < j)) ? 1 : 0;
    cs.ev[rk * kQ + i] = vv;
    if (i == 0 && rk < R) {   // sigma = l / sqrt(l) and 1 / sigma from one refined reciprocal square root
      const double rs = rsqrt_f64(fmax(lj, 2.2250738585072014e-308));
      cs.sig[rk] = lj > 0.0 ? lj * rs : 0.0;
      cs.isig[rk] = lj > 0.0 ? rs : 0.0;
    }
    commit();
  } else {
    commit();
  }
  __syncthreads();
  // leading singular vectors: u_r = Q ev_r (a row per thread, kept in
  // registers for the blend), v_r = Bm^T ev_r / sigma_r
  static_assert(m <= kNT && n <= 64, "left vectors: a row per thread; right vectors: a column per lane of a wave");
  const float dk = expf(gacc);
  const float s1 = sdec, s2 = 1.f - sdec;
  double ur[kRMax];
  if (tid < m) {
    double yv[kQ];
#pragma unroll
    for (int j = 0; j < kQ; ++j) yv[j] = cs.y[tid * kLQ + j];
#pragma unroll
    for (int r = 0; r < kRMax; ++r) {
      double s = 0.0;
#pragma unroll
      for (int j = 0; j < kQ; ++j) s += yv[j] * cs.ev[r * kQ + j];
      ur[r] = s;
    }
  }
  // wave r: v_r (one column per lane) and the pair's canonical sign,
  // argmax_c |v_r[c]| with the first index on ties (an all-reduce by row
  // rotations inside each 16-lane row, then across the rows), then the
  // blend of B's row r, which needs nothing from the other waves
  static_assert(R <= 4, "one factor per wave");
  if (wave < R) {
    const int r = wave, c = lane;
    const bool on = c < n;
    double vr = 0.0;
    if (on) {
      double sv = 0.0;
#pragma unroll
      for (int j = 0; j < kQ; ++j) sv += cs.z[c * kLQ + j] * cs.ev[r * kQ + j];
      vr = cs.sig[r] > 0.0 ? sv * cs.isig[r] : (c == r ? 1.0 : 0.0);
    }
    double bv_ = on ? fabs(vr) : -1.0;
    int bi = on ? c : 0x7fffffff;
    auto take = [&](double ov, int oi) {
      const bool t = (ov > bv_) | ((ov == bv_) & (oi < bi));  // selects, no branches
      bv_ = t ? ov : bv_;
      bi = t ? oi : bi;
    };
    take(dpp_f64<0x128>(bv_), __builtin_amdgcn_update_dpp(0, bi, 0x128, 0xf, 0xf, false));
    take(dpp_f64<0x124>(bv_), __builtin_amdgcn_update_dpp(0, bi, 0x124, 0xf, 0xf, false));
    take(dpp_f64<0x122>(bv_), __builtin_amdgcn_update_dpp(0, bi, 0x122, 0xf, 0xf, false));
    take(dpp_f64<0x121>(bv_), __builtin_amdgcn_update_dpp(0, bi, 0x121, 0xf, 0xf, false));
    // the four rows' results out of lanes 0, 16, 32, 48 (the order does not
    // matter: max value, then least index, is a total order): wave-uniform
    double mv = readlane_f64(bv_, 0);
    int mi = __builtin_amdgcn_readlane(bi, 0);
#pragma unroll
    for (int rr = 1; rr < 4; ++rr) {
      const double ov = readlane_f64(bv_, 16 * rr);
      const int oi = __builtin_amdgcn_readlane(bi, 16 * rr);
      const bool t = (ov > mv) | ((ov == mv) & (oi < mi));
      mv = t ? ov : mv;
      mi = t ? oi : mi;
    }
    const double vb = readlane_f64(vr, mi & 63);
    const double sg = (mi != 0x7fffffff && vb < 0.0) ? -1.0 : 1.0;
    if (lane == 0) cs.sgn[r] = sg;
    if (on) Bv[r * n + c] = s1 * (Bv[r * n + c] * dk) + s2 * (float)(sg * vr);
  }
  __syncthreads();
  // two-timescale blend of the decayed factors with the SVD factors (B above)
  if (tid < m)
#pragma unroll
    for (int r = 0; r < kRMax; ++r)
      if (r < R) {
        const double sv = cs.sgn[r] * cs.sig[r] * ur[r];
        A[r * m + tid] = s1 * (A[r * m + tid] * dk) + s2 * (float)sv;
      }
  if (tid == 0 && stats) {
    double kept = 0.0;
    for (int r = 0; r < R; ++r) kept += cs.sig[r] * cs.sig[r];
    stats[0] = en[0];
    stats[1] = kept;
  }
  __syncthreads();
}

// ---------------------------------------------------------------------------
// fused forward
// ---------------------------------------------------------------------------

template <typename CT> struct W16Of { static constexpr int value = 8 * sizeof(CT) / 16; };

__device__ __forceinline__ void unpack8(const uint4* w, float* f, const bf16*) {
  const unsigned ws[4] = {w[0].x, w[0].y, w[0].z, w[0].w};
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    f[2 * e] = __uint_as_float(ws[e] << 16);
    f[2 * e + 1] = __uint_as_float(ws[e] & 0xffff0000u);
  }
}
__device__ __forceinline__ void unpack8(const uint4* w, float* f, const float*) {
  const unsigned ws[8] = {w[0].x, w[0].y, w[0].z, w[0].w, w[1].x, w[1].y, w[1].z, w[1].w};
#pragma unroll
  for (int e = 0; e < 8; ++e) f[e] = __uint_as_float(ws[e]);
}
__device__ __forceinline__ void store8(bf16* dst, const float* f) {
  *(bf16x8*)dst = (bf16x8){(bf16)f[0], (bf16)f[1], (bf16)f[2], (bf16)f[3],
                           (bf16)f[4], (bf16)f[5], (bf16)f[6], (bf16)f[7]};
}
__device__ __forceinline__ void store8(float* dst, const float* f) {
  *(f32x4*)dst = (f32x4){f[0], f[1], f[2], f[3]};
  *(f32x4*)(dst + 4) = (f32x4){f[4], f[5], f[6], f[7]};
}

// A thread's share of a sub-chunk's token rows as loaded: 8 consecutive
// channels of one token (raw q, k, v; gates and decay as float).  The loads
// always go to an in-bounds token and the validity is applied when the rows
// are committed: loaded registers that branches merge would make the
// prefetch wait for its own loads.
template <typename CT> struct G3Raw {
  uint4 k[W16Of<CT>::value], q[W16Of<CT>::value], v[W16Of<CT>::value];
  f32x4 b0, b1, w0, w1;   // per-channel gates
  float bs, ws, dec;      // scalar gates, decay
  bool ok;                // a token of this call (else zeros and decay 1)
};

// local token t (marked invalid outside [0, T) or for a thread without a
// unit; the loads then read token min(max(t, 0), T - 1))
template <typename CT>
__device__ __forceinline__ void g3_fetch(const G3FwdArgs& p, const G3Tok& o, G3Raw<CT>& r, int t, bool on,
                                         int ud) {
  constexpr int W16 = W16Of<CT>::value;
  r.ok = on && t >= 0 && t < p.T;
  const size_t tc = (size_t)min(max(t, 0), p.T - 1);
  const uint4* kp = (const uint4*)((const CT*)p.k + o.qkv_base + tc * o.qkv_tok + ud);
  const uint4* qp = (const uint4*)((const CT*)p.q + o.qkv_base + tc * o.qkv_tok + ud);
  const uint4* vp = (const uint4*)((const CT*)p.v + o.qkv_base + tc * o.qkv_tok + ud);
#pragma unroll
  for (int w = 0; w < W16; ++w) {
    r.k[w] = kp[w];
    r.q[w] = qp[w];
    r.v[w] = vp[w];
  }
  // both branches define every gate field, so no loaded register is merged
  if (o.gc > 1) {
    const float* bp = p.bg + o.gate_base + tc * o.gate_tok + ud;
    const float* wp = p.wg + o.gate_base + tc * o.gate_tok + ud;
    r.b0 = *(const f32x4*)bp;
    r.b1 = *(const f32x4*)(bp + 4);
    r.w0 = *(const f32x4*)wp;
    r.w1 = *(const f32x4*)(wp + 4);
    r.bs = r.ws = 0.f;
  } else {
    r.bs = p.bg[o.gate_base + tc * o.gate_tok];
    r.ws = p.wg[o.gate_base + tc * o.gate_tok];
    r.b0 = r.b1 = r.w0 = r.w1 = zero4();
  }
  r.dec = p.dec[o.dec_base + tc * o.dec_tok];
}

// the raw q / k vector w of a thread's row, zero for an invalid token
template <typename CT>
__device__ __forceinline__ uint4 g3_raw(const G3Raw<CT>& r, const uint4& x) {
  return r.ok ? x : make_uint4(0u, 0u, 0u, 0u);
}

// h = b o k and u = w o v of the thread's 8 channels (gc: gate channels);
// returns the row sum of k . h over the token's DG threads (consecutive lanes)
template <typename CT, int DG>
__device__ __forceinline__ float g3_unpack(const G3Raw<CT>& r, int gc, float* hf, float* uu) {
  float kf[8], vf[8], bb[8], ww[8];
  unpack8(r.k, kf, (const CT*)nullptr);
  unpack8(r.v, vf, (const CT*)nullptr);
  if (gc > 1) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      bb[e] = r.b0[e];
      bb[4 + e] = r.b1[e];
      ww[e] = r.w0[e];
      ww[4 + e] = r.w1[e];
    }
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      bb[e] = r.bs;
      ww[e] = r.ws;
    }
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) {   // an invalid token commits zeros
    kf[e] = r.ok ? kf[e] : 0.f;
    vf[e] = r.ok ? vf[e] : 0.f;
  }
  float part = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    hf[e] = bb[e] * kf[e];
    uu[e] = ww[e] * vf[e];
    part += kf[e] * hf[e];
  }
  if constexpr (DG == 16) {
    // the 16 lanes of a token row are one DPP row: rotations by 8, 4, 2, 1
    part += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(part), 0x128, 0xf, 0xf, false));
    part += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(part), 0x124, 0xf, 0xf, false));
    part += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(part), 0x122, 0xf, 0xf, false));
    part += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(part), 0x121, 0xf, 0xf, false));
  } else {
#pragma unroll
    for (int off = 1; off < DG; off <<= 1) part += __shfl_xor(part, off, 64);
  }
  return part;
}

// The window LDS a sub-chunk step works on (pointers into one workgroup's
// shared memory)
template <typename CT, int D>
struct G3WinView {
  CT (*x)[D + 8];               // rows: H (0..15), Q (16..31), K (32..47)
  float (*u)[D + 4];            // w (.) v
  float (*kr)[D + 4];           // Kronecker reads of H and Q
  float (*pp)[kSC][kSC + 4];    // [4]: H K^T (then inverse scratch), Aq, T, inverse scratch
  float (*po)[kSC][kSC + 4];    // [2]: Ho, Qo over the slots
  CT (*skron)[D + 8];           // this workgroup's rows of sum_r A_r (x) B_r
  float (*vbd)[D + 4];          // window keys, decayed to now
  CT (*vbx)[D + 8];             // the same in the compute dtype (bf16 IO)
  float *G, *alpha, *lg, *kco, *qco, *gam, *vsc;
};

// The log-decay prefix sums of a sub-chunk (lane i < 16 holds G_i).
template <typename CT, int D>
__device__ __forceinline__ float g3_scan_g(const G3WinView<CT, D>& w, int lane) {
  float gl = lane < kSC ? w.lg[lane] : 0.f;
#pragma unroll
  for (int off = 1; off < kSC; off <<= 1) {
    const float o = __shfl_up(gl, off, 64);
    if (lane >= off) gl += o;
  }
  return gl;
}

// The per-token coefficients of a sub-chunk (one wave): G, e^G, kco = alpha
// e^{2 (gacc + G)}, qco = e^{2 (gacc + G)} and the key scale e^{G_last - G}.
template <typename CT, int D>
__device__ __forceinline__ void g3_scalars(const G3WinView<CT, D>& w, float gl, float gacc, int lane) {
  const float gl_last = __shfl(gl, kSC - 1, 64);
  if (lane < kSC) {
    const float e2 = expf(2.f * (gacc + gl));
    w.G[lane] = gl;
    w.gam[lane] = expf(gl);
    w.kco[lane] = w.alpha[lane] * e2;
    w.qco[lane] = e2;
    w.vsc[lane] = expf(gl_last - gl);
  }
}

// Gram tile ti of a sub-chunk (one wave; 4 tiles):
//   0: H K^T (raw; the inverse turns it into T),  1: Aq = [j <= i] e^{G_i - G_j} q_i.k_j,
//   2: Ho = vis alpha_i e^{G_i} h_i.Vb[j],        3: Qo = vis e^{G_i} q_i.Vb[j]
// with vis = [j >= i or j < lo]
template <typename CT, int D>
__device__ __forceinline__ void g3_gram_tile(const G3WinView<CT, D>& w, int ti, float gl, int lo, int lane) {
  constexpr bool KF = sizeof(CT) == 4;
  const int g4 = lane >> 4, n16 = lane & 15;
  const float gj = __shfl(gl, n16, 64);
  float gi[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) gi[s] = __shfl(gl, 4 * g4 + s, 64);
  const bool isq = ti & 1;
  const CT* arow = &w.x[(isq ? kSC : 0) + n16][0];
  const CT* brow;
  if (ti < 2) brow = &w.x[2 * kSC + n16][0];
  else if constexpr (KF) brow = (const CT*)&w.vbd[n16][0];
  else brow = &w.vbx[n16][0];
  const f32x4 acc = tile_nt<CT, D>(arow, brow, g4);
  const int j = n16;
  if (ti == 0) {
#pragma unroll
    for (int s = 0; s < 4; ++s) w.pp[0][4 * g4 + s][j] = acc[s];
  } else if (ti == 1) {
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int i = 4 * g4 + s;
      w.pp[1][i][j] = (j <= i) ? expf(gi[s] - gj) * acc[s] : 0.f;
    }
  } else {
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int i = 4 * g4 + s;
      const bool vis = j >= i || j < lo;
      const float sc = expf(gi[s]) * (isq ? 1.f : w.alpha[i]);
      w.po[isq ? 1 : 0][i][j] = vis ? sc * acc[s] : 0.f;
    }
  }
}

// T = (I + Lm)^-1 into pp[2] (one wave, the one that formed tile 0 and the
// coefficients: it reads what its own lanes wrote, ordered by the fences).
// Lm[i][j] = alpha_i e^{G_i - G_j} (h_i . k_j), j < i, is strictly lower
// (nilpotent): (I + Lm)^-1 = (I - L)(I + L^2)(I + L^4)(I + L^8), factors that
// commute; squarings and products on fp32 MFMA.  An accumulator tile is a
// k-fragment (B operand); the A operand of each square goes through LDS.
template <typename CT, int D>
__device__ __forceinline__ void g3_inverse(const G3WinView<CT, D>& w, int lane) {
  const int g4 = lane >> 4, n16 = lane & 15;
  wave_lds_sync();
  f32x4 xa, ta;
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const int i = 4 * g4 + s;
    xa[s] = (n16 < i) ? w.alpha[i] * expf(w.G[i] - w.G[n16]) * w.pp[0][i][n16] : 0.f;
    w.pp[3][i][n16] = xa[s];
    ta[s] = (i == n16 ? 1.f : 0.f) - xa[s];
  }
  wave_lds_sync();
  int src = 3;
#pragma unroll
  for (int step = 0; step < 3; ++step) {
    const int dst = step & 1 ? 3 : 0;
    f32x4 sq = zero4();
    mma(sq, *(const f32x4*)&w.pp[src][n16][4 * g4], xa);  // X^2
    xa = sq;
#pragma unroll
    for (int s = 0; s < 4; ++s) w.pp[dst][4 * g4 + s][n16] = sq[s];
    wave_lds_sync();
    mma(ta, *(const f32x4*)&w.pp[dst][n16][4 * g4], ta);  // T += X^2 T
    src = dst;
  }
#pragma unroll
  for (int s = 0; s < 4; ++s) w.pp[2][4 * g4 + s][n16] = ta[s];
}

// The commit of a sub-chunk's prefetched token rows into the window LDS: H =
// b (.) k, the Q and K rows, u = w (.) v, and per token alpha and the log
// decay (thread tid holds load unit (tid / (D / 8), 8 (tid mod (D / 8)))).
template <typename CT, int D>
__device__ __forceinline__ void g3_commit(const G3WinView<CT, D>& w, const G3Tok& tk, const G3Raw<CT>& r, int tid) {
  constexpr int DG = D / 8, W16 = W16Of<CT>::value;
  if (tid >= kSC * DG) return;
  const int ui = tid / DG, ud = 8 * (tid % DG);
  float hf[8], uu[8];
  const float part = g3_unpack<CT, DG>(r, tk.gc, hf, uu);
  store8(&w.x[ui][ud], hf);
#pragma unroll
  for (int q16 = 0; q16 < W16; ++q16) {
    *(uint4*)&w.x[kSC + ui][ud + q16 * (16 / sizeof(CT))] = g3_raw(r, r.q[q16]);
    *(uint4*)&w.x[2 * kSC + ui][ud + q16 * (16 / sizeof(CT))] = g3_raw(r, r.k[q16]);
  }
  *(f32x4*)&w.u[ui][ud] = (f32x4){uu[0], uu[1], uu[2], uu[3]};
  *(f32x4*)&w.u[ui][ud + 4] = (f32x4){uu[4], uu[5], uu[6], uu[7]};
  if (tid % DG == 0) {
    w.alpha[ui] = stable_alpha_f(part);
    w.lg[ui] = log_decay(r.ok ? r.dec : 1.f);
  }
}

// The state-independent half of sub-chunk c's step, formed on waves 1..3
// while wave 0 runs a compaction's eigen-solve (no workgroup barrier can be
// used then): every one of the three waves loads and commits all 16 token
// rows itself (identical values, so the concurrent writes agree), two load
// passes in flight at a time, and reads only what it wrote; then wave 1 forms
// the coefficients, H K^T and the inverse, wave 2 Aq and wave 3 the window
// grams.  The commit's x, u and scalars and the tiles' pp, po must lie in LDS
// the compaction no longer uses.
template <typename CT, int D>
__device__ __forceinline__ void g3_stage_a_shadow(const G3WinView<CT, D>& w, const G3FwdArgs& p,
                                                  const G3Tok& tk, G3Raw<CT>& ra, G3Raw<CT>& rb, int c,
                                                  int wave, int lane) {
  constexpr int DG = D / 8, PASSES = kSC * DG / 64;
  static_assert(PASSES % 2 == 0, "load passes in pairs");
  auto fetch = [&](G3Raw<CT>& r, int pass) {
    const int u = pass * 64 + lane;
    g3_fetch<CT>(p, tk, r, c * kSC + u / DG - p.t0, true, 8 * (u % DG));
  };
#pragma unroll
  for (int pass = 0; pass < PASSES; pass += 2) {
    fetch(ra, pass);
    fetch(rb, pass + 1);
    g3_commit<CT, D>(w, tk, ra, pass * 64 + lane);
    g3_commit<CT, D>(w, tk, rb, (pass + 1) * 64 + lane);
  }
  wave_lds_sync();
  const int lo = max(0, p.t0 - c * kSC);
  const float gl = g3_scan_g(w, lane);
  if (wave == 1) {
    g3_scalars(w, gl, 0.f, lane);
    g3_gram_tile<CT, D>(w, 0, gl, lo, lane);
    g3_inverse(w, lane);
  } else if (wave == 2) {
    g3_gram_tile<CT, D>(w, 1, gl, lo, lane);
  } else {
#pragma unroll
    for (int ti = 2; ti < 4; ++ti) g3_gram_tile<CT, D>(w, ti, gl, lo, lane);
  }
}

// Sub-chunk c of the window recurrence, a chain a workgroup: commit of its
// prefetched token rows, the grams, the inverse, the Kronecker reads, the
// window algebra on the U tiles uo, y and the training stash, then the window
// keys.  committed: its token rows are in LDS already (g3_commit ran earlier).
template <typename CT, int D>
__device__ __forceinline__ void g3_window_step(const G3WinView<CT, D>& w, const G3FwdArgs& p, const G3Tok& tk,
                                               int chain, int c, bool live, float& gacc,
                                               f32x4 (&uo)[(D / 16 + 3) / 4], const G3Raw<CT>& raw, bool committed) {
  constexpr bool KF = sizeof(CT) == 4;
  constexpr int DG = D / 8;  // 8-element load units per token row
  constexpr int W16 = W16Of<CT>::value;
  constexpr int KS = FragT<CT>::KSTEP;
  typedef typename FragT<CT>::type Frag;
  constexpr int NVT = D / 16, VPW = (NVT + 3) / 4;   // value tiles, per wave
  const int tid = opaque(threadIdx.x), lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g4 = lane >> 4, n16 = lane & 15;
  const int T = p.T;
  auto vown = [&](int a) { return wave + 4 * a < NVT; };
  auto vtile = [&](int a) { return wave + 4 * a; };

    // slots [lo, hi) receive this call's tokens; the others (the
    // head a previous call wrote, the tail after the last token) keep the
    // writes they hold and stay visible to every token of the sub-chunk
    const int lo = max(0, p.t0 - c * kSC), hi = min(kSC, p.t0 + T - c * kSC);
    __syncthreads();
    if (!committed) g3_commit<CT, D>(w, tk, raw, tid);
    __syncthreads();
    // per-token scalars | grams and Kronecker reads (MFMA).  Every wave forms
    // the log-decay prefix sums G (lane i holds G_i); wave 0 publishes the
    // per-token coefficients, each wave forms a gram tile, and wave 0
    // forms the inverse while waves 1..3 do the Kronecker reads.  A committed
    // sub-chunk had all of this formed in the previous compaction's shadow.
    if (!committed) {
      const float gl = g3_scan_g(w, lane);
      if (wave == 0) g3_scalars(w, gl, gacc, lane);
      g3_gram_tile<CT, D>(w, wave, gl, lo, lane);
      if (wave == 0) g3_inverse(w, lane);
    }
    if (live && (committed || wave > 0)) {
      // the value tiles over waves 1..3 (wave 0 forms the inverse), or all four
      const int w0 = committed ? wave : wave - 1, ws = committed ? 4 : 3;
      // the H and Q fragments serve every value tile; each tile's Kronecker
      // fragments are read ahead of its MFMAs behind a scheduling barrier (the
      // compiler, short of registers, waited for each MFMA's reads)
      Frag xf[2][D / KS];
#pragma unroll
      for (int rt = 0; rt < 2; ++rt)
#pragma unroll
        for (int kb = 0; kb < D / KS; ++kb) xf[rt][kb] = ld_frag(&w.x[rt * 16 + n16][kb * KS], g4);
      for (int vt = w0; vt < NVT; vt += ws) {
        Frag bf[D / KS];
#pragma unroll
        for (int kb = 0; kb < D / KS; ++kb) bf[kb] = ld_frag(&w.skron[vt * 16 + n16][kb * KS], g4);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) {
          f32x4 acc = zero4();
#pragma unroll
          for (int kb = 0; kb < D / KS; ++kb) mma(acc, xf[rt][kb], bf[kb]);
#pragma unroll
          for (int s = 0; s < 4; ++s) w.kr[rt * 16 + 4 * g4 + s][vt * 16 + n16] = acc[s];
        }
      }
    }
    __syncthreads();
    // window algebra on fp32 MFMA, per wave its VPW value tiles:
    //   Rhs = alpha u - kco KRh - Ho U_old;  U = T Rhs
    //   Y   = qco KRq + Qo U_old + Aq U
    // (an accumulator tile over rows = tokens is directly a k-fragment)
    // (every LDS operand read ahead, behind a scheduling barrier; the
    // coefficient tiles and per-token scalars serve every value tile)
    const f32x4 po0 = *(const f32x4*)&w.po[0][n16][4 * g4], po1 = *(const f32x4*)&w.po[1][n16][4 * g4];
    const f32x4 ptf = *(const f32x4*)&w.pp[2][n16][4 * g4], paf = *(const f32x4*)&w.pp[1][n16][4 * g4];
    float alv[4], kcv[4], qcv[4], uv[VPW][4], khv[VPW][4], kqv[VPW][4];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int i = 4 * g4 + s;
      alv[s] = w.alpha[i];
      kcv[s] = w.kco[i];
      qcv[s] = w.qco[i];
    }
#pragma unroll
    for (int a = 0; a < VPW; ++a)
      if (vown(a)) {
        const int v = vtile(a) * 16 + n16;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const int i = 4 * g4 + s;
          uv[a][s] = w.u[i][v];
          khv[a][s] = w.kr[i][v];
          kqv[a][s] = w.kr[kSC + i][v];
        }
      }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int a = 0; a < VPW; ++a) {
      if (!vown(a)) continue;
      const int v = vtile(a) * 16 + n16;
      f32x4 acc = zero4();
      mma(acc, po0, uo[a]);
      f32x4 rhs;
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        float r = alv[s] * uv[a][s] - acc[s];
        if (live) r -= kcv[s] * khv[a][s];
        rhs[s] = r;
      }
      f32x4 un = zero4();
      mma(un, ptf, rhs);
      f32x4 yv = zero4();
      mma(yv, po1, uo[a]);
      mma(yv, paf, un);
      CT* yp = (CT*)p.y + tk.y_base + v;
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int i = 4 * g4 + s;
        float out = yv[s];
        if (live) out += qcv[s] * kqv[a][s];
        const int t = c * kSC + i - p.t0;
        if (t >= 0 && t < T) yp[(size_t)t * tk.y_tok] = from_f<CT>(out);
      }
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int i = 4 * g4 + s;
        if (i >= lo && i < hi) uo[a][s] = un[s];
      }
      if (p.ts_u) {   // training stash: this sub-chunk's net writes
        float* us = p.ts_u + ((size_t)chain * p.nch + c) * kSC * D + v;
#pragma unroll
        for (int s = 0; s < 4; ++s) us[(size_t)(4 * g4 + s) * D] = un[s];
      }
    }
    if (p.ts_g && tid == 0) p.ts_g[(size_t)chain * p.nch + c] = gacc;
    // the keys for the next sub-chunk: the slots this one wrote take k_j decayed
    // to its end, the others their old keys decayed over it (8 consecutive keys
    // per thread)
    {
      const float olds = expf(w.G[kSC - 1]);
      for (int u8 = tid; u8 < kSC * D / 8; u8 += kNT) {
        const int j = u8 / DG, d = 8 * (u8 % DG);
        uint4 kw[W16];
#pragma unroll
        for (int q16 = 0; q16 < W16; ++q16) kw[q16] = *(const uint4*)&w.x[2 * kSC + j][d + q16 * (16 / sizeof(CT))];
        float kf[8];
        unpack8(kw, kf, (const CT*)nullptr);
        float sc = w.vsc[j];
        if (j < lo || j >= hi) {
          sc = olds;
          const f32x4 o0 = *(const f32x4*)&w.vbd[j][d], o1 = *(const f32x4*)&w.vbd[j][d + 4];
          kf[0] = o0[0], kf[1] = o0[1], kf[2] = o0[2], kf[3] = o0[3];
          kf[4] = o1[0], kf[5] = o1[1], kf[6] = o1[2], kf[7] = o1[3];
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) kf[e] *= sc;
        *(f32x4*)&w.vbd[j][d] = (f32x4){kf[0], kf[1], kf[2], kf[3]};
        *(f32x4*)&w.vbd[j][d + 4] = (f32x4){kf[4], kf[5], kf[6], kf[7]};
        if constexpr (!KF) store8(&w.vbx[j][d], kf);
      }
    }
    gacc += w.G[kSC - 1];
}

// ---------------------------------------------------------------------------
// compaction, one chain per block: the chunked forward's step between
// intervals and the gdnx_gdn3_compact entry point
// ---------------------------------------------------------------------------
template <int D, int P>
struct G3CompactSmem {
  G3Compact<D, P> k;
  alignas(16) float ab[kAB];
};

// sum_r A_r (x) B_r as a [D][D] (v, k) matrix for the window kernel's reads,
// from the factors Af [R][m], Bf [R][n] (LDS), ld the row stride of sk.  With
// p = iv a_k + ik running over A_r's entries and q = jv b_k + jk over B_r's,
// S'^T[q][p] = sum_r B_r[q] A_r[p] is a product with K = R = 4: one fp32 MFMA
// (16x16x4) per 16 x 16 tile.  Lane (g, l) supplies B_g[q0 + l] and A_g[p0 + l]
// and holds q = q0 + 4 g + e (e < 4), p = p0 + l: the entries
// (iv b_v + jv, ik b_k + jk .. jk + 3) of S_kron, one 4-element store.  The
// tiles go round the 4 waves.
template <int D, typename CT>
__device__ __forceinline__ void write_skron(CT* sk, const float* Af, const float* Bf, int tid, int ld = D) {
  typedef G3D<D> Ge;
  constexpr int QT = Ge::n / 16, NT = QT * (Ge::m / 16);
  static_assert(Ge::R == 4 && Ge::bk % 4 == 0 && Ge::m % 16 == 0 && Ge::n % 16 == 0 && NT % 4 == 0,
                "K = R = 4 MFMA tiles, runs of 4 jk");
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), g = lane >> 4, l16 = lane & 15;
  // every tile's operands are loaded before the first MFMA
  float ao[NT / 4], bo[NT / 4];
#pragma unroll
  for (int u = 0; u < NT / 4; ++u) {
    const int t = wave + 4 * u, q0 = (t % QT) * 16, p0 = (t / QT) * 16;
    ao[u] = Bf[g * Ge::n + q0 + l16];
    bo[u] = Af[g * Ge::m + p0 + l16];
  }
  // and every MFMA issued before the first store
  __builtin_amdgcn_sched_barrier(0);
  f32x4 acc[NT / 4];
#pragma unroll
  for (int u = 0; u < NT / 4; ++u) acc[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(ao[u], bo[u], zero4(), 0, 0, 0);
#pragma unroll
  for (int u = 0; u < NT / 4; ++u) {
    const int t = wave + 4 * u, q0 = (t % QT) * 16, p0 = (t / QT) * 16;
    const int p = p0 + l16, q = q0 + 4 * g;
    const int iv = p / Ge::ak, ik = p % Ge::ak, jv = q / Ge::bk, jk = q % Ge::bk;
    st4(sk + (size_t)(iv * Ge::bv + jv) * ld + ik * Ge::bk + jk, acc[u][0], acc[u][1], acc[u][2], acc[u][3]);
  }
}

// ---------------------------------------------------------------------------
// fused forward for the layer's default regime (a compaction after every
// 16-token window: K_c = P = 16): one workgroup per chain walks all of a
// call's windows, each a window step followed by its compaction, with the
// window state, the factors and the Kronecker matrix in LDS (no launch or
// global round trip between the two)
// ---------------------------------------------------------------------------
template <typename CT, int D>
struct G3FusedSmem {
  static constexpr int P = kSC;
  union alignas(16) Phase {
    G3Compact<D, P, false> cs;          // the compaction's scratch
    struct alignas(16) Win {            // the window step's
      CT x[3 * kSC][D + 8];             // x, u and the scalars first: the next window's commit
      float u[kSC][D + 4];              // writes them while the compaction still uses all of
      float G[kSC], alpha[kSC], lg[kSC], kco[kSC], qco[kSC], gam[kSC], vsc[kSC];   // its LDS but R_mat
      alignas(16) float kr[2 * kSC][D + 4];
      float pp[4][kSC][kSC + 4];
      float po[2][kSC][P + 4];
      CT skron[D][D + 8];               // rebuilt from the factors after every compaction
    } w;
  } ph;
  alignas(16) float ab[kAB];            // A | B of this chain
  alignas(16) float uwin[P][D + 4];     // the window's net writes (slot-major)
  alignas(16) float vbd[P][D + 4];      // its keys, decayed to now
  alignas(16) CT vbx[sizeof(CT) == 4 ? 1 : P][D + 8];
};
template <typename CT, int D>
constexpr bool fused_fits() { return sizeof(G3FusedSmem<CT, D>) <= 160 * 1024; }

template <typename CT, int D>
__global__ void __launch_bounds__(kNT) gdn3_fused_kernel(G3FwdArgs p) {
  constexpr int P = kSC;
  typedef G3FusedSmem<CT, D> Sm;
  __shared__ Sm sm;
  static_assert(sizeof(Sm) <= 160 * 1024, "LDS budget");
  typedef G3D<D> Ge;
  constexpr int Rm = Ge::R * Ge::m, Rn = Ge::R * Ge::n, VPW = (D / 16 + 3) / 4;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), g4 = lane >> 4, n16 = lane & 15;
  const int N = p.B * p.H * p.M;
  const int chain = xcd_remap(blockIdx.x, N);
  const G3Tok tk(p, chain, D);
  const int DG = D / 8, ui = tid / DG, ud = 8 * (tid % DG);
  const bool has_unit = tid < kSC * DG;

  // the call's sub-chunks, each its own compaction interval
  const long long tend = (long long)p.t0 + p.T;
  const int cg0 = p.t0 / kSC, cg1 = (int)((tend + kSC - 1) / kSC);
  const bool carried = p.A0 != nullptr;
  G3Raw<CT> raw;
  g3_fetch<CT>(p, tk, raw, cg0 * kSC + ui - p.t0, has_unit, ud);

  // initial state: the carried one (A0, B0 [N][R m|n], U0, Vb0 [N][D][P]) or zero
  const size_t cb = (size_t)chain * D * P;
  for (int e = tid; e < Rm; e += kNT) sm.ab[e] = carried ? p.A0[(size_t)chain * Rm + e] : 0.f;
  for (int e = tid; e < Rn; e += kNT) sm.ab[Rm + e] = carried ? p.B0[(size_t)chain * Rn + e] : 0.f;
  for (int e = tid; e < D * P; e += kNT) {
    const int d = e / P, j = e % P;
    const float uv = carried ? p.U0[cb + e] : 0.f, kv = carried ? p.Vb0[cb + e] : 0.f;
    sm.uwin[j][d] = uv;
    sm.vbd[j][d] = kv;
    if constexpr (sizeof(CT) == 2) sm.vbx[j][d] = from_f<CT>(kv);
  }
  __syncthreads();
  if (carried) write_skron<D, CT>(&sm.ph.w.skron[0][0], sm.ab, sm.ab + Rm, tid, D + 8);
  bool live = carried;
  bool committed = false;   // the window's token rows were committed during the last compaction
  typedef typename Sm::Phase::Win WinT;
  constexpr bool kEarly = offsetof(WinT, skron) <= sizeof(sm.ph.cs.rm);   // x .. po inside R_mat's LDS
  G3Raw<CT> raw2;
  float gacc = 0.f;
  int event = 0;
  const G3WinView<CT, D> w{sm.ph.w.x, sm.ph.w.u, sm.ph.w.kr, sm.ph.w.pp, sm.ph.w.po, sm.ph.w.skron, sm.vbd,
                           sm.vbx, sm.ph.w.G, sm.ph.w.alpha, sm.ph.w.lg, sm.ph.w.kco, sm.ph.w.qco,
                           sm.ph.w.gam, sm.ph.w.vsc};
  f32x4 uo[VPW];
  // the chain's sketch, the same at every compaction, held from here (a load
  // per compaction waited, in order, for the window's output stores before it)
  G3Sketch<D> sk;
  g3_sketch_load<D>(sk, p.sketch + (size_t)chain * Ge::n * (p.cmode ? Ge::R : Ge::q), p.cmode ? Ge::R : Ge::q, tid);
  // (passed through an empty asm here, so that the loop sees register values,
  // not loads it would wait for at every use)
#pragma unroll
  for (int u = 0; u < G3Sketch<D>::N; ++u) sk.v[u] = __int_as_float(opaque(__float_as_int(sk.v[u])));
  for (int c = cg0; c < cg1; ++c) {
    // the window step (its net writes through the registers of their waves)
#pragma unroll
    for (int a = 0; a < VPW; ++a)
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int vt = wave + 4 * a;
        uo[a][s] = vt < D / 16 ? sm.uwin[4 * g4 + s][vt * 16 + n16] : 0.f;
      }
    g3_window_step<CT, D>(w, p, tk, chain, c, live, gacc, uo, raw, committed);
#pragma unroll
    for (int a = 0; a < VPW; ++a)
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int vt = wave + 4 * a;
        if (vt < D / 16) sm.uwin[4 * g4 + s][vt * 16 + n16] = uo[a][s];
      }
    const bool complete = (long long)(c + 1) * kSC <= tend;
    __syncthreads();
    if (!complete) break;   // the tail: no compaction follows
    // its compaction (gdn3/gdn3_upgrade.py:650-719), the factors decayed by e^{gacc}
    const int qs = p.cmode ? Ge::R : Ge::q;
    // the next window's token loads and their commit run in the eigen-solve's
    // shadow when that window's commit targets lie in R_mat's LDS (dead by then)
    const bool pre = kEarly && p.cmode == 0 && c + 1 < cg1;
    // (waves 1..3, all of the next window's state-independent half; nothing
    // is added to the eigen-solve's wave)
    auto issue = [&]() {};
    auto commit = [&]() {
      if (pre && wave > 0) g3_stage_a_shadow<CT, D>(w, p, tk, raw, raw2, c + 1, wave, lane);
    };
    g3_compact<D, P>(sm.ph.cs, sm.ab, &sm.uwin[0][0], &sm.vbd[0][0], (size_t)(D + 4), (size_t)1, gacc, p.sdec,
                     p.sketch + (size_t)chain * Ge::n * qs,
                     p.stats ? p.stats + ((size_t)event * N + chain) * 2 : nullptr, tid, p.cmode, issue, commit, &sk);
    __syncthreads();
    if (p.train_states) {   // the factors after every compaction, for the backward
      const G3Stash ts = g3_stash(p.train_states, N, p.nch, p.T / p.Kc, D, kSC, Ge::RMN);
      for (int e = tid; e < Rm + Rn; e += kNT) ts.ab[((size_t)event * N + chain) * Ge::RMN + e] = sm.ab[e];
    }
    ++event;
    gacc = 0.f;
    live = true;
    if (c + 1 < cg1) {   // the next window's loads (under the Kronecker matrix's rebuild), unless committed
      if (!pre) g3_fetch<CT>(p, tk, raw, (c + 1) * kSC + ui - p.t0, has_unit, ud);
      write_skron<D, CT>(&sm.ph.w.skron[0][0], sm.ab, sm.ab + Rm, tid, D + 8);
    }
    committed = pre;
  }
  __syncthreads();
  // the final state: U, Vb [N][D][P]; A, B (decayed since the last compaction)
  const float dk = expf(gacc);
  for (int e = tid; e < D * P; e += kNT) {
    const int d = e / P, j = e % P;
    if (p.U_out) p.U_out[cb + e] = sm.uwin[j][d];
    if (p.Vb_out) p.Vb_out[cb + e] = sm.vbd[j][d];
  }
  if (p.A_out)
    for (int e = tid; e < Rm; e += kNT) p.A_out[(size_t)chain * Rm + e] = sm.ab[e] * dk;
  if (p.B_out)
    for (int e = tid; e < Rn; e += kNT) p.B_out[(size_t)chain * Rn + e] = sm.ab[Rm + e] * dk;
}

// One chain's compaction; bi indexes the statistics (the chain's row in the
// launch).
template <int D, int P, typename CT>
__device__ __forceinline__ void compact_chain(const G3CompactArgs& p, G3CompactSmem<D, P>& sm, int chain, int bi,
                                              int tid) {
  typedef G3D<D> Ge;
  constexpr int Rm = Ge::R * Ge::m, Rn = Ge::R * Ge::n;
  for (int e = tid; e < Rm; e += kNT) sm.ab[e] = p.A[(size_t)chain * Rm + e];
  for (int e = tid; e < Rn; e += kNT) sm.ab[Rm + e] = p.Bf[(size_t)chain * Rn + e];
  const size_t cb = (size_t)chain * D * P;
  const float gacc = p.gsum ? p.gsum[chain] : 0.f;
  __syncthreads();
  const int qs = p.mode ? Ge::R : Ge::q;   // sketch columns
  g3_compact<D, P>(sm.k, sm.ab, p.U + cb, p.Vb + cb, (size_t)p.u_sp, (size_t)p.u_sd, gacc, p.sdec, p.sketch + (size_t)chain * Ge::n * qs,
                   p.stats ? p.stats + (size_t)bi * 2 : nullptr, tid, p.mode);
  for (int e = tid; e < Rm; e += kNT) {
    p.A_out[(size_t)chain * Rm + e] = sm.ab[e];
    if (p.A_fin) p.A_fin[(size_t)chain * Rm + e] = sm.ab[e];
  }
  for (int e = tid; e < Rn; e += kNT) {
    p.B_out[(size_t)chain * Rn + e] = sm.ab[Rm + e];
    if (p.B_fin) p.B_fin[(size_t)chain * Rn + e] = sm.ab[Rm + e];
  }
  if (p.ab_stash)
    for (int e = tid; e < Rm + Rn; e += kNT) p.ab_stash[(size_t)chain * (Rm + Rn) + e] = sm.ab[e];
  if (p.skron) write_skron<D, CT>((CT*)p.skron + (size_t)chain * D * D, sm.ab, sm.ab + Rm, tid);
}

// A decode batch's positions are read this many rows at a time, four a thread
// in flight (16384 rows of one chain, d = 64, none due: the step 143 us with
// batches of 256, 73 so, 63 with each workgroup checking its own rows only; 1024
// due of them 193, 124, 708).
constexpr int kRowsPer = 4, kRowBatch = 16 * kNT;
static_assert(kRowBatch / 64 == 64, "a lane per 64 rows of a batch");

template <int D, int P, typename CT>
__global__ void __launch_bounds__(kNT) gdn3_compact_kernel(G3CompactArgs p) {
  __shared__ G3CompactSmem<D, P> sm;
  static_assert(sizeof(G3CompactSmem<D, P>) <= 160 * 1024, "LDS budget");
  const int tid = threadIdx.x;
  if (!p.pos) {
    compact_chain<D, P, CT>(p, sm, blockIdx.x, blockIdx.x, tid);
    return;
  }
  // decode batch: only the rows whose token closes a compaction interval.
  // Every workgroup reads all the rows' positions and lists the ones that
  // compact, in row order; the chains of the listed rows go round the grid
  // one by one.  A compaction is ~27 us of latency on a workgroup that holds
  // a CU's LDS, so the launch is as long as the most any workgroup gets:
  // 1024 due chains of 16384 take 4 each on 256 workgroups, 125 us at d =
  // 128 (each workgroup checking its own stride of the chains left all 8 of
  // a stride to one workgroup whenever the rows' positions repeat with a
  // period that divides it: 220 us).
  __shared__ unsigned short rows[kRowBatch];               // of the batch at base
  __shared__ unsigned long long mask[kRowBatch / 64];      // due rows by groups of 64
  const int NS = p.N / p.hm, lane = tid & 63, wave = tid >> 6;
  const unsigned G = gridDim.x;
  unsigned seen = 0;   // due chains of the rows before this batch
  for (int base = 0; base < NS; base += kRowBatch) {
    const int th = opaque(tid);   // (its address arithmetic is not held across the compactions)
    const int ng = min(kRowBatch / 64, (NS - base + 63) / 64);   // groups of 64 rows
#pragma unroll 1
    for (int j = 0; j * (kNT / 64) < ng; j += kRowsPer) {
      int ps[kRowsPer], sl[kRowsPer];
#pragma unroll
      for (int i = 0; i < kRowsPer; ++i) ps[i] = p.pos[min(base + (j + i) * kNT + th, NS - 1)];
#pragma unroll
      for (int i = 0; i < kRowsPer; ++i) sl[i] = p.slots ? p.slots[min(base + (j + i) * kNT + th, NS - 1)] : 0;
#pragma unroll
      for (int i = 0; i < kRowsPer; ++i) {
        const int row = base + (j + i) * kNT + th;
        if (base + (j + i) * kNT >= NS) break;   // (uniform)
        const bool go = row < NS && ps[i] >= 0 && (ps[i] + 1) % p.Kc == 0 &&   // (a negative position is an empty row)
                        (!p.slots || (sl[i] >= 0 && sl[i] < p.nslots));
        const unsigned long long m = __ballot(go);
        if (lane == 0) mask[(j + i) * (kNT / 64) + wave] = m;
      }
    }
    __syncthreads();
    // due rows up to group `lane`, inclusive (whole numbers below 2^24)
    const float upto = lane_prefix<64>(lane < ng ? (float)__popcll(mask[lane]) : 0.f, lane);
    const unsigned cnt = (unsigned)lane_value(upto, 63) * p.hm;
    if (cnt) {   // (uniform)
#pragma unroll 1
      for (int g = wave; g < ng; g += kNT / 64) {
        const unsigned long long m = mask[g];
        const int at = (int)__shfl(upto, g, 64) - __popcll(m) + __popcll(m & ((1ull << lane) - 1));
        if (m >> lane & 1) rows[at] = (unsigned short)(g * 64 + lane);
      }
      __syncthreads();
    }
    for (unsigned e = (blockIdx.x + G - seen % G) % G; e < cnt; e += G) {   // due chain seen + e is this workgroup's
      const int r = base + rows[e / p.hm], ch = (int)(e % p.hm);
      compact_chain<D, P, CT>(p, sm, (p.slots ? p.slots[r] : r) * p.hm + ch, r * p.hm + ch, tid);
      lds_barrier();   // the chain's last LDS reads before the next one's loads (its stores need not have arrived)
    }
    seen += cnt;
    __syncthreads();   // rows and wcnt are read before the next batch writes them
  }
}

// The carried state (A0, B0, U0, Vb0 in the output layouts) in the window
// kernel's workspace form: the factors, their Kronecker matrix, the window's
// writes and keys slot-major, and no decay accumulated since the factors.
template <int D, int P, typename CT>
__global__ void __launch_bounds__(kNT) gdn3_state_in_kernel(G3FwdArgs p) {
  typedef G3D<D> Ge;
  constexpr int Rm = Ge::R * Ge::m, Rn = Ge::R * Ge::n;
  __shared__ float ab[Rm + Rn];
  const int tid = threadIdx.x, chain = blockIdx.x;
  const int N = p.B * p.H * p.M;
  for (int e = tid; e < Rm; e += kNT) {
    const float a = p.A0[(size_t)chain * Rm + e];
    ab[e] = a;
    p.ab[(size_t)chain * Rm + e] = a;
  }
  for (int e = tid; e < Rn; e += kNT) {
    const float b = p.B0[(size_t)chain * Rn + e];
    ab[Rm + e] = b;
    p.ab[(size_t)N * Rm + (size_t)chain * Rn + e] = b;
  }
  // [D][P] -> [P][D]: consecutive threads read consecutive (d, slot) entries
  const size_t cb = (size_t)chain * D * P;
  for (int e = tid; e < D * P; e += kNT) {
    const int d = e / P, j = e % P;
    p.uw[cb + (size_t)j * D + d] = p.U0[cb + e];
    p.vw[cb + (size_t)j * D + d] = p.Vb0[cb + e];
  }
  if (tid == 0) p.gsum[chain] = 0.f;
  __syncthreads();
  write_skron<D, CT>((CT*)p.skron + (size_t)chain * D * D, ab, ab + Rm, tid);
}

__global__ void fill_zero_kernel(float* p, long long n) {
  for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (long long)gridDim.x * blockDim.x)
    p[e] = 0.f;
}

// ---------------------------------------------------------------------------
// Kronecker read S x = vec(sum_r A_r X B_r^T) + U (Vb^T x), X = x as [a_k, b_k]
// (gdn3/gdn3_upgrade.py:626-639; identity of gdn3/kernels.py:7-16)
// ---------------------------------------------------------------------------
template <int D>
__global__ void __launch_bounds__(kNT) kron_read_kernel(KronReadArgs p) {
  __shared__ float xs[D];
  __shared__ float zs[kRMax * kMN];  // Z_r[iv][jk] = sum_ik A_r[iv][ik] X[ik][jk]
  __shared__ float cp[64];           // Vb_p . x
  const int tid = threadIdx.x;
  const int row = blockIdx.x;  // (chain, c)
  const int chain = row / p.C;
  const G3Geom ge = p.ge;
  const int P = p.P;
  const float* x = p.x + (size_t)row * D;
  const float* A = p.A + (size_t)chain * ge.R * ge.m;
  const float* Bf = p.Bf + (size_t)chain * ge.R * ge.n;
  const float* U = p.U + (size_t)chain * D * P;
  const float* Vb = p.Vb + (size_t)chain * D * P;
  if (tid < D) xs[tid] = x[tid];
  __syncthreads();
  const int nz = ge.R * ge.av * ge.bk;
  for (int e = tid; e < nz; e += kNT) {
    const int r = e / (ge.av * ge.bk), rem = e % (ge.av * ge.bk), iv = rem / ge.bk, jk = rem % ge.bk;
    float s = 0.f;
    for (int ik = 0; ik < ge.ak; ++ik) s += A[(r * ge.av + iv) * ge.ak + ik] * xs[ik * ge.bk + jk];
    zs[e] = s;
  }
  for (int pp = tid; pp < P; pp += kNT) {
    float s = 0.f;
    for (int k = 0; k < D; ++k) s += Vb[k * P + pp] * xs[k];
    cp[pp] = s;
  }
  __syncthreads();
  if (tid < D) {
    const int v = tid, iv = v / ge.bv, jv = v % ge.bv;
    float s = 0.f;
    for (int r = 0; r < ge.R; ++r)
      for (int jk = 0; jk < ge.bk; ++jk)
        s += zs[(r * ge.av + iv) * ge.bk + jk] * Bf[(r * ge.bv + jv) * ge.bk + jk];
    for (int pp = 0; pp < P; ++pp) s += U[v * P + pp] * cp[pp];
    p.y[(size_t)row * D + v] = s;
  }
}

int cu_count() {
  static const int n = [] {
    int dev = 0, v = 0;
    return hipGetDevice(&dev) == hipSuccess &&
                   hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && v > 0
               ? v
               : 256;
  }();
  return n;
}

// A decode batch's due chains go round the workgroups that run at once, one a
// CU at d = 128 (LDS), two at d = 64 (registers; LDS alone would take three,
// and with 768 workgroups the last 256 began when the first 512 had done their
// share: 64 rows x 64 chains all due 229 us a step, 191 so).
template <int D, int P, typename CT>
int launch_compact_ct(const G3CompactArgs& a, hipStream_t stream) {
  int grid = a.N;
  if (a.pos) {
    static const int per_cu = [] {
      int v = 0;
      return hipOccupancyMaxActiveBlocksPerMultiprocessor(&v, gdn3_compact_kernel<D, P, CT>, kNT, 0) == hipSuccess && v > 0
                 ? v
                 : 1;
    }();
    const long long fit = (long long)cu_count() * per_cu;
    if (fit < grid) grid = (int)fit;
  }
  hipLaunchKernelGGL((gdn3_compact_kernel<D, P, CT>), dim3(grid), dim3(kNT), 0, stream, a);
  return check_launch("gdn3_compact_kernel");
}

template <int D, int P>
int launch_compact(const G3CompactArgs& a, hipStream_t stream) {
  return a.skron && a.skron_dtype == GDNX_DTYPE_BF16 ? launch_compact_ct<D, P, bf16>(a, stream)
                                                     : launch_compact_ct<D, P, float>(a, stream);
}

int compact_dispatch(const G3CompactArgs& a, hipStream_t stream) {
  if (a.N == 0) return GDNX_OK;
  if (a.D == 128 && a.P == 16) return launch_compact<128, 16>(a, stream);
  if (a.D == 128 && a.P == 32) return launch_compact<128, 32>(a, stream);
  if (a.D == 128 && a.P == 64) return launch_compact<128, 64>(a, stream);
  if (a.D == 64 && a.P == 16) return launch_compact<64, 16>(a, stream);
  if (a.D == 64 && a.P == 32) return launch_compact<64, 32>(a, stream);
  if (a.D == 64 && a.P == 64) return launch_compact<64, 64>(a, stream);
  return set_error(GDNX_ERR_SHAPE, "gdn3_compact: unsupported head_dim %d / P %d", a.D, a.P);
}

inline size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

template <typename CT, int D, int P>
int run_gdn3_fwd(G3FwdArgs a, hipStream_t stream) {
  typedef G3D<D> Ge;
  const int N = a.B * a.H * a.M;
  if constexpr (P == kSC && fused_fits<CT, D>()) {
    if (a.Kc == kSC) {   // the layer's default regime: one fused launch for the whole call
      a.nch = (a.T + kSC - 1) / kSC;
      G3Stash ts{nullptr, nullptr, nullptr};
      if (a.train_states) ts = g3_stash(a.train_states, N, a.nch, a.T / a.Kc, D, kSC, Ge::RMN);
      a.ts_u = ts.u;
      a.ts_g = ts.gacc;
      hipLaunchKernelGGL((gdn3_fused_kernel<CT, D>), dim3(N), dim3(kNT), 0, stream, a);
      return check_launch("gdn3_fused_kernel");
    }
  }
  char* w = (char*)a.workspace;
  a.skron = w;
  w += align256((size_t)N * D * D * sizeof(CT));
  a.ab = (float*)w;
  w += align256((size_t)N * Ge::R * (Ge::m + Ge::n) * 4);
  a.uw = (float*)w;
  w += align256((size_t)N * P * D * 4);
  a.vw = (float*)w;
  w += align256((size_t)N * P * D * 4);
  a.gsum = (float*)w;
  w += align256((size_t)N * 4);
  gdn3_long_carve(a, N, w);
  const bool carried = a.A0 != nullptr;
  int rc;
  if (carried) {
    hipLaunchKernelGGL((gdn3_state_in_kernel<D, P, CT>), dim3(N), dim3(kNT), 0, stream, a);
    rc = check_launch("gdn3_state_in_kernel");
  } else {
    const long long nab = (long long)N * Ge::R * (Ge::m + Ge::n);
    hipLaunchKernelGGL(fill_zero_kernel, dim3((unsigned)((nab + 255) / 256 < 4096 ? (nab + 255) / 256 : 4096)),
                       dim3(256), 0, stream, a.ab, nab);
    rc = check_launch("fill_zero_kernel");
  }
  if (rc) return rc;
  // sub-chunks are global: sub-chunk c covers tokens [16 c, 16 c + 16) of
  // the whole sequence, of which this call holds [t0, t0 + T)
  const long long tend = (long long)a.t0 + a.T;
  const int cg0 = a.t0 / kSC, cg1 = (int)((tend + kSC - 1) / kSC);
  a.nch = (a.T + kSC - 1) / kSC;
  G3Stash ts{nullptr, nullptr, nullptr};
  if (a.train_states) ts = g3_stash(a.train_states, N, a.nch, a.T / a.Kc, D, kSC, Ge::RMN);
  a.ts_u = ts.u;
  a.ts_g = ts.gacc;
  const int per = a.Kc / kSC;
  int event = 0;
  bool first = true;
  for (int c0 = cg0; c0 < cg1;) {
    int c1 = (c0 / per + 1) * per;   // the next compaction boundary
    if (c1 > cg1) c1 = cg1;
    a.c0 = c0;
    a.c1 = c1;
    a.first = first && !carried;     // zero window state
    a.live = !first || carried;      // the Kronecker factors may be nonzero
    a.last = c1 == cg1;
    a.complete = (long long)c1 * kSC <= tend && c1 % per == 0;
    if ((rc = gdn3_long_interval(a, N, stream))) return rc;
    if (a.complete) {
      G3CompactArgs ca{};
      ca.A = a.ab;
      ca.Bf = a.ab + (size_t)N * Ge::R * Ge::m;
      ca.U = a.uw;
      ca.Vb = a.vw;
      ca.sketch = a.sketch;
      ca.A_out = a.ab;
      ca.B_out = a.ab + (size_t)N * Ge::R * Ge::m;
      ca.stats = a.stats ? a.stats + (size_t)event * N * 2 : nullptr;
      ca.ge = a.ge;
      ca.N = N;
      ca.D = D;
      ca.P = P;
      ca.sdec = a.sdec;
      ca.u_sp = D;
      ca.u_sd = 1;
      ca.gsum = a.gsum;
      ca.skron = a.skron;
      ca.skron_dtype = a.dtype;
      ca.A_fin = a.last ? a.A_out : nullptr;
      ca.B_fin = a.last ? a.B_out : nullptr;
      ca.ab_stash = ts.ab ? ts.ab + (size_t)event * N * Ge::RMN : nullptr;
      ca.mode = a.cmode;
      if ((rc = compact_dispatch(ca, stream))) return rc;
      ++event;
    }
    first = false;
    c0 = c1;
  }
  return GDNX_OK;
}

}  // namespace

// Static scratch for gdnx_gdn3_chunk_fwd_state_noalloc: the forward's
// workspace (Kronecker matrices, factors, window state) for callers that
// cannot allocate (graph capture, serving loops).  Each device the library
// runs on holds its own copy for the life of the process; host code reaches
// it only through the address hipGetSymbolAddress returns for that device.
static __device__ __align__(256) unsigned char scratch[kG3ScratchBytes];

namespace {
std::mutex g_scratch_mu;
constexpr int kMaxDevices = 64;
void* g_scratch_ptr[kMaxDevices] = {};
}  // namespace

int gdn3_scratch(void** out) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices)
    return set_error(GDNX_ERR_HIP, "no current HIP device (or device index >= %d)", kMaxDevices);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr)
      return set_error(GDNX_ERR_HIP, "scratch address on device %d: %s", dev, hipGetErrorString(e));
    g_scratch_ptr[dev] = ptr;
  }
  *out = g_scratch_ptr[dev];
  return GDNX_OK;
}

int gdn3_zero_fill(float* p, size_t n, hipStream_t stream) {
  if (n == 0) return GDNX_OK;
  const size_t nb = (n + 255) / 256;
  hipLaunchKernelGGL(fill_zero_kernel, dim3((unsigned)(nb < 4096 ? nb : 4096)), dim3(256), 0, stream, p,
                     (long long)n);
  return check_launch("fill_zero_kernel");
}

size_t gdn3_workspace_bytes(int N, int D, int P, int dtype) {
  const size_t cb = dtype == GDNX_DTYPE_BF16 ? 2 : 4;
  const int R = 4, mn = D == 128 ? 256 + 64 : 64 + 64;
  return align256((size_t)N * D * D * cb) + align256((size_t)N * R * mn * 4) + 2 * align256((size_t)N * P * D * 4) +
         align256((size_t)N * 4) + gdn3_long_bytes(N, D, P);
}

size_t gdn3_train_states_bytes(int N, int T, int D, int P, int Kc) {
  (void)P;   // the stash is kept per 16-token sub-chunk whatever the window
  const int nch = (T + kSC - 1) / kSC, ncomp = T / Kc;
  const int rmn = D == 128 ? G3D<128>::RMN : G3D<64>::RMN;
  return g3_stash_bytes(N, nch, ncomp, D, kSC, rmn);
}

// whether run_gdn3_fwd runs the call as one fused launch, which uses no
// workspace (the layer's default regime, a compaction after every window)
bool gdn3_fwd_fused(int D, int P, int Kc, int dtype) {
  if (P != kSC || Kc != kSC) return false;
  if (dtype == GDNX_DTYPE_BF16) return D == 128 ? fused_fits<bf16, 128>() : D == 64 && fused_fits<bf16, 64>();
  return D == 128 ? fused_fits<float, 128>() : D == 64 && fused_fits<float, 64>();
}

int gdn3_fwd_dispatch(const G3FwdArgs& a, hipStream_t stream) {
  if (a.dtype == GDNX_DTYPE_BF16) {
    if (a.D == 128 && a.P == 16) return run_gdn3_fwd<bf16, 128, 16>(a, stream);
    if (a.D == 128 && a.P == 32) return run_gdn3_fwd<bf16, 128, 32>(a, stream);
    if (a.D == 128 && a.P == 64) return run_gdn3_fwd<bf16, 128, 64>(a, stream);
    if (a.D == 64 && a.P == 16) return run_gdn3_fwd<bf16, 64, 16>(a, stream);
    if (a.D == 64 && a.P == 32) return run_gdn3_fwd<bf16, 64, 32>(a, stream);
    if (a.D == 64 && a.P == 64) return run_gdn3_fwd<bf16, 64, 64>(a, stream);
  } else {
    if (a.D == 128 && a.P == 16) return run_gdn3_fwd<float, 128, 16>(a, stream);
    if (a.D == 128 && a.P == 32) return run_gdn3_fwd<float, 128, 32>(a, stream);
    if (a.D == 128 && a.P == 64) return run_gdn3_fwd<float, 128, 64>(a, stream);
    if (a.D == 64 && a.P == 16) return run_gdn3_fwd<float, 64, 16>(a, stream);
    if (a.D == 64 && a.P == 32) return run_gdn3_fwd<float, 64, 32>(a, stream);
    if (a.D == 64 && a.P == 64) return run_gdn3_fwd<float, 64, 64>(a, stream);
  }
  return set_error(GDNX_ERR_SHAPE, "gdn3: unsupported head_dim %d / P %d (64 or 128 / 16, 32 or 64)", a.D, a.P);
}

int gdn3_compact_dispatch(const G3CompactArgs& a, hipStream_t stream) { return compact_dispatch(a, stream); }

int kron_read_dispatch(const KronReadArgs& a, hipStream_t stream) {
  if ((long long)a.N * a.C == 0) return GDNX_OK;
  if (a.D == 128)
    hipLaunchKernelGGL((kron_read_kernel<128>), dim3(a.N * a.C), dim3(kNT), 0, stream, a);
  else if (a.D == 64)
    hipLaunchKernelGGL((kron_read_kernel<64>), dim3(a.N * a.C), dim3(kNT), 0, stream, a);
  else
    return set_error(GDNX_ERR_SHAPE, "kron_read: unsupported head_dim %d", a.D);
  return check_launch("kron_read_kernel");
}

}  // namespace gdnx
