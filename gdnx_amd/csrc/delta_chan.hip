// Decoupled-erase delta rule with a decay per key channel (gfx950), the
// general KMD-2 scan: per chain (b, h) and token t, with g_t in (0, 1]^dk,
//
//   S <- diag(g_t) S;  r = beta_w v - beta_e S^T k;  S <- S + k r^T;  y = S^T q
//
// (research/kernel_ab/ref_scan.py:37-47, gdn3/kmd2_native.py:109-132, where
// g = exp(g_head + decay_chan) is per key channel).  Chunks of C = 16 tokens,
// float32 throughout.  With the per-channel inclusive prefix G_i = sum_{s<=i}
// log g_s and the chunk's last row G_L:
//
//   M_ij = sum_d x_id k_jd exp(G_id - G_jd)  (j <= i: every exponent <= 0)
//   L = diag(beta_e) M[x=k] (strict),  Aq = M[x=q],  T = (I + L)^-1
//   R = T (diag(beta_w) V - diag(beta_e) (K o e^G) S0)
//   Y = (Q o e^G) S0 + Aq R
//   S = diag(e^{G_L}) S0 + (K o e^{G_L - G})^T R
//
// With a chunk of 16 the decay-weighted grams are formed exactly, channel by
// channel (no sub-chunk factoring whose factors could overflow).  The
// reference's chunked path (gdn3/kmd2_fast_scan.py:198-214) divides keys by
// the cumulative decay product instead, which is valid only at its chunk of
// 16 and moderate decays.  Three kernels, as for the scalar decay: the
// forward state scan, the reverse scan of the state gradient, and the
// per-chunk gradient kernel, here with a prep kernel in front that writes the
// scans' operands chunk by chunk.  One workgroup of D/16 waves per chunk
// (prep, gradients), wave w owning value (and key) columns 16w..16w+15; the
// scans' split is described at their kernels.
#include "delta_common.hpp"
#include "gdnx_internal.hpp"

namespace gdnx {

namespace {

constexpr int CC = 16;        // chunk
constexpr int LDC = CC + 4;   // [*][C] fp32 rows

template <int D>
struct ChD {
  static constexpr int NW = D / 16, NT = 64 * NW, NDT = D / 16, LDD = D + 4;
};

// The chunk's operands in LDS (fp32): q, k, the per-channel prefix G, the
// scalars, the exact grams and T.
template <int D>
struct alignas(16) ChanOps {
  static constexpr int LDD = D + 4;
  float q[CC * LDD];
  float k[CC * LDD];
  float G[CC * LDD];     // raw log-decay on commit, then the clamped prefix
  float L[CC * LDC];     // beta_e,i M_ij (j < i)
  float LT[CC * 20];     // L transposed (the blocked inverse reads it)
  float Td[CC * 20];
  float Aq[CC * LDC];
  float Mk[CC * LDC];    // M_ij[x=k] (j < i), the gram without beta_e
  float T[CC * LDC];     // (I + L)^-1
  float be[CC], bw[CC];
  float eGL[D];          // exp(G_L) per channel
};

// Column prefix of the clamped log-decay (threads t < D, one column each).
template <int D>
__device__ __forceinline__ void chan_prefix(ChanOps<D>& o, int tid) {
  constexpr int LDD = ChD<D>::LDD;
  if (tid < D) {
    float acc = 0.f;
#pragma unroll
    for (int i = 0; i < CC; ++i) {
      acc += fmaxf(fminf(o.G[i * LDD + tid], 0.f), kLogFloor);
      o.G[i * LDD + tid] = acc;
    }
    o.eGL[tid] = __expf(acc);
  }
}

// Exact decay-weighted grams: wave w takes rows i = w, w + NW, ...; lane
// (g, n) takes column j = n and the channel quarter [g D/4, (g+1) D/4).
template <int D>
__device__ __forceinline__ void chan_grams(ChanOps<D>& o, int wave, int lane) {
  constexpr int NW = ChD<D>::NW, LDD = ChD<D>::LDD, DQ = D / 4;
  const int g4 = lane >> 4, j = lane & 15;
  for (int i = wave; i < CC; i += NW) {
    float kk = 0.f, qk = 0.f;
    if (j <= i) {
#pragma unroll 4
      for (int d0 = g4 * DQ; d0 < (g4 + 1) * DQ; d0 += 4) {
        const f32x4 ki = *(const f32x4*)&o.k[i * LDD + d0];
        const f32x4 qi = *(const f32x4*)&o.q[i * LDD + d0];
        const f32x4 Gi = *(const f32x4*)&o.G[i * LDD + d0];
        const f32x4 kj = *(const f32x4*)&o.k[j * LDD + d0];
        const f32x4 Gj = *(const f32x4*)&o.G[j * LDD + d0];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float ex = __expf(Gi[e] - Gj[e]);
          kk += ki[e] * kj[e] * ex;
          qk += qi[e] * kj[e] * ex;
        }
      }
    }
    kk += __shfl_xor(kk, 16, 64);
    kk += __shfl_xor(kk, 32, 64);
    qk += __shfl_xor(qk, 16, 64);
    qk += __shfl_xor(qk, 32, 64);
    if (g4 == 0) {
      const float mk = (j < i) ? kk : 0.f;
      const float l = o.be[i] * mk;
      o.L[i * LDC + j] = l;
      o.LT[j * 20 + i] = l;
      o.Mk[i * LDC + j] = mk;
      o.Aq[i * LDC + j] = (j <= i) ? qk : 0.f;
    }
  }
}

template <int D>
__device__ __forceinline__ void chan_inverse(ChanOps<D>& o, int wave, int lane) {
  invert_unit_lower<CC>(o.L, o.LT, o.Td, wave, lane, [&](int) { return 0; },
                        [&](int i, int jj, float t, int) { o.T[i * LDC + jj] = t; });
}

// Buffer resource over this chain's rows of a [B, T, H, X] fp32 tensor for
// the chunk at token t0 (rows past T read zero / drop stores).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t chunk_rsrc(const float* base, int b, int t0, int T, int H, int h,
                                                             int X) {
  const size_t off = (((size_t)b * T + t0) * H + h) * X;
  return buf_rsrc(base + off, (unsigned)(min(CC, T - t0) * H * X * 4));
}

// per-token scalar (beta) of this chain at t0 + i, zero past T
__device__ __forceinline__ float chunk_scalar(const float* base, int b, int t0, int i, int T, int H, int h) {
  const int t = min(t0 + i, T - 1);
  const float x = base[((size_t)b * T + t) * H + h];
  return (t0 + i < T) ? x : 0.f;
}

}  // namespace

// ---------------------------------------------------------------------------
// per-chunk operand records (state independent, one workgroup per chunk)
//   forward:  U = T diag(beta_w) V, -Wm = -T diag(beta_e) (K o e^G), Q o e^G,
//             (K o e^{G_L - G})^T, Aq, e^{G_L}
//   backward: K o e^{G_L - G}, (Q o e^G)^T, -Wm^T, T^T, Aq^T, e^{G_L}
// so that the scans carry only the state-dependent products.
// ---------------------------------------------------------------------------
template <int D>
struct ChRec {
  static constexpr int CD = CC * D;
  static constexpr int F_U = 0, F_NWM = CD, F_QE = 2 * CD, F_KFT = 3 * CD, F_AQ = 4 * CD, F_EGL = 4 * CD + CC * CC;
  static constexpr int FN = 4 * CD + CC * CC + D;
  static constexpr int B_KF = 0, B_QET = CD, B_NWT = 2 * CD, B_TT = 3 * CD, B_AQT = 3 * CD + CC * CC,
                       B_EGL = 3 * CD + 2 * CC * CC;
  static constexpr int BN = 3 * CD + 2 * CC * CC + D;
  static_assert(FN % 4 == 0 && BN % 4 == 0 && F_EGL % 4 == 0 && B_EGL % 4 == 0, "16-byte aligned records");
};

template <int D>
struct alignas(16) ChanPrepSmem {
  ChanOps<D> o;
  float ket[D * LDC];    // (K o e^G)^T
  float kft[D * LDC];    // (K o e^{G_L - G})^T
  float qet[D * LDC];    // (Q o e^G)^T
  float vt[D * LDC];     // V^T
};

// (registers held to two workgroups a CU at d = 128, 130 -> 128: prep 64 -> 45 us
// at B = 1, T = 2048, H = 16, 36 -> 29 us with the backward's records at 32 chains)
template <int D, bool BWD>
__global__ void __launch_bounds__(64 * (D / 16), D == 128 ? 4 : 3) chan_prep_kernel(ChanArgs p) {
  typedef ChD<D> Cd;
  typedef ChRec<D> Rc;
  constexpr int NT = Cd::NT, LDD = Cd::LDD;
  __shared__ ChanPrepSmem<D> sm;
  ChanOps<D>& o = sm.o;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, g4 = lane >> 4, n16 = lane & 15;
  const int NC = (p.T + CC - 1) / CC;
  const int nchains = p.B * p.H;
  const int blk = xcd_remap(blockIdx.x, nchains * NC);
  const int c = blk % NC, chain = blk / NC;
  const int h = chain % p.H, b = chain / p.H;
  const int t0 = c * CC;
  const size_t rec = rec_index(chain, c, nchains);
  float* fr = p.frec + rec * Rc::FN;
  float* br = BWD ? p.brec + rec * Rc::BN : nullptr;
  const unsigned rsb = (unsigned)((size_t)p.H * D * 4);
  {
    Stage<float, CC, D, 1, NT> sq, sk, sl;
    Stage<float, CC, D, 4, NT> sv;
    sq.fetch(chunk_rsrc(p.q, b, t0, p.T, p.H, h, D), rsb, tid);
    sk.fetch(chunk_rsrc(p.k, b, t0, p.T, p.H, h, D), rsb, tid);
    sl.fetch(chunk_rsrc(p.lg, b, t0, p.T, p.H, h, D), rsb, tid);
    sv.fetch(chunk_rsrc(p.v, b, t0, p.T, p.H, h, D), rsb, tid);
    const float be = chunk_scalar(p.be, b, t0, tid % CC, p.T, p.H, h);
    const float bw = chunk_scalar(p.bw, b, t0, tid % CC, p.T, p.H, h);
    sq.template commit_nat<LDD>(o.q, tid);
    sk.template commit_nat<LDD>(o.k, tid);
    sl.template commit_nat<LDD>(o.G, tid);
    sv.template commit_tr<LDC>(sm.vt, tid);
    if (tid < CC) {
      o.be[tid] = be;
      o.bw[tid] = bw;
    }
  }
  __syncthreads();
  chan_prefix<D>(o, tid);
  __syncthreads();
  chan_grams<D>(o, wave, lane);
  for (int e = tid; e < CC * D; e += NT) {
    const int i = e / D, d = e % D;
    const float G = o.G[i * LDD + d], GL = o.G[(CC - 1) * LDD + d];
    const float E = __expf(G), F = __expf(GL - G), kv = o.k[i * LDD + d], qv = o.q[i * LDD + d] * E;
    fr[Rc::F_QE + e] = qv;
    sm.ket[d * LDC + i] = kv * E;
    sm.kft[d * LDC + i] = kv * F;
    if constexpr (BWD) {
      br[Rc::B_KF + e] = kv * F;
      sm.qet[d * LDC + i] = qv;
    }
  }
  __syncthreads();
  chan_inverse<D>(o, wave, lane);
  __syncthreads();
  {  // -Wm on this wave's key tile: acc[s] = Wm[n][16 wave + 4 g + s]
    const f32x4 bt = frag_scale(ld_frag(&o.T[n16 * LDC], g4), o.be, g4);
    f32x4 acc = zero4();
    mma(acc, ld_frag(&sm.ket[(16 * wave + n16) * LDC], g4), bt);
    *(f32x4*)&fr[Rc::F_NWM + n16 * D + 16 * wave + 4 * g4] = -acc;
    if constexpr (BWD)
#pragma unroll
      for (int s = 0; s < 4; ++s) br[Rc::B_NWT + (16 * wave + 4 * g4 + s) * CC + n16] = -acc[s];
  }
  {  // U = T diag(beta_w) V on value tile wave, stored as rows
    f32x4 acc = zero4();
    mma(acc, frag_scale(ld_frag(&o.T[n16 * LDC], g4), o.bw, g4), ld_frag(&sm.vt[(16 * wave + n16) * LDC], g4));
    *(f32x4*)&fr[Rc::F_U + n16 * D + 16 * wave + 4 * g4] = tile_transpose((float*)nullptr, acc, lane);
  }
  for (int e = tid; e < D * CC; e += NT) {
    const int d = e / CC, i = e % CC;
    fr[Rc::F_KFT + e] = sm.kft[d * LDC + i];
    if constexpr (BWD) {
      br[Rc::B_QET + e] = sm.qet[d * LDC + i];
    }
  }
  for (int e = tid; e < CC * CC; e += NT) {
    const int i = e / CC, j = e % CC;
    fr[Rc::F_AQ + e] = o.Aq[i * LDC + j];
    if constexpr (BWD) {
      br[Rc::B_TT + e] = o.T[j * LDC + i];
      br[Rc::B_AQT + e] = o.Aq[j * LDC + i];
    }
  }
  for (int e = tid; e < D; e += NT) {
    fr[Rc::F_EGL + e] = o.eGL[e];
    if constexpr (BWD) br[Rc::B_EGL + e] = o.eGL[e];
  }
}

// ---------------------------------------------------------------------------
// The scans, per chunk from the record
//   R = U - Wm S0,  Y = (Q o e^G) S0 + Aq R,  S = diag(e^{G_L}) S0 + (K o e^{G_L - G})^T R
// and the reverse below, with a chain's state split over keys as well as
// values: a workgroup of four waves per (chain, NV tiles of 16 value columns),
// wave w carrying the D / 4 keys 16 KT w ... of those columns in registers.
// Per chunk each wave forms its keys' part of Wm S0 (K dS backward); the parts
// are summed through LDS, and every wave updates its own keys with the sum.
// No wave reads another's operands, so the records go from memory straight
// into MFMA fragments, PF chunks ahead, and a step has one barrier.  With few
// chains a step is bound by its latency: the fp32 MFMAs (16 x 16 x 4, 32
// cycles) over D / 4 keys, then the exchange.  d = 128: B = 2, T = 512, H = 16
// with stash, forward / reverse 103 / 90 us with only the value columns split,
// 43 / 45 us so (49 / 51 us while a step could wait for a later chunk's
// loads); B = 1, T = 2048 forward 292 us, then 125 us.
// ---------------------------------------------------------------------------
template <int D>
struct ChSplit {
  static constexpr int KT = D / 64;   // key tiles per wave
  static constexpr int NVT = D / 16;  // value tiles
  // chunks of operands in flight (as the registers of NV value tiles leave room for)
  static constexpr int PF(int nv, bool score) { return nv == 1 ? 4 : nv == 2 ? (score ? 3 : 4) : 2; }
};
// acc0 + acc1 += sum_t A_t B_t: the fp32 MFMAs of a product over all of a
// wave's key tiles as two chains
template <int KT>
__device__ __forceinline__ void mma2(f32x4& acc0, f32x4& acc1, const f32x4 (&a)[KT], const f32x4 (&b)[KT]) {
#pragma unroll
  for (int t = 0; t < KT; ++t)
#pragma unroll
    for (int s = 0; s < 4; s += 2) {
      acc0 = __builtin_amdgcn_mfma_f32_16x16x4f32(a[t][s], b[t][s], acc0, 0, 0, 0);
      acc1 = __builtin_amdgcn_mfma_f32_16x16x4f32(a[t][s + 1], b[t][s + 1], acc1, 0, 0, 0);
    }
}
// Operands of a record: its resource, a lane's byte offset and the wave's
// uniform one, in floats (no vector address is formed).
__device__ __forceinline__ f32x4 rec_load4(__amdgpu_buffer_rsrc_t r, unsigned lane_bytes, int at) {
  return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)lane_bytes, at * 4, 0));
}
__device__ __forceinline__ float rec_load1(__amdgpu_buffer_rsrc_t r, unsigned lane_bytes, int at) {
  return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, (int)lane_bytes, at * 4, 0));
}
// Keeps the loads of a chunk's operands together and after the step that read
// the last ones from the same registers: with the chunks' loads in order, and a
// loop with one exit, a step waits for its own operands only.
__device__ __forceinline__ void load_fence() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}
template <int NV>
struct alignas(16) ChanExchange {
  f32x4 r[2][NV][4][64];   // the waves' parts of R (dR), by chunk parity
  __device__ __forceinline__ f32x4 sum(int c, int v, int lane) const {
    return (r[c & 1][v][0][lane] + r[c & 1][v][1][lane]) + (r[c & 1][v][2][lane] + r[c & 1][v][3][lane]);
  }
};
// x[i] for a uniform i < 4
__device__ __forceinline__ float pick4(const f32x4& x, int i) {
  return i < 2 ? (i == 0 ? x[0] : x[1]) : (i == 2 ? x[2] : x[3]);
}

// SCORE (|r_t| requested): each value tile's sum of squares of a token's net
// write goes to the record's U, at the tile's first column, which only this
// workgroup reads and has read; chan_rnorm_kernel sums them.  A workgroup that
// has all value columns (d = 64, four tiles) writes |r_t| itself.
template <int D, int NV, bool STASH, bool SCORE>
__global__ void __launch_bounds__(256, 2) chan_split_fwd_kernel(ChanArgs p) {
  typedef ChRec<D> Rc;
  typedef ChSplit<D> Sp;
  constexpr int KT = Sp::KT, PF = Sp::PF(NV, SCORE);
  __shared__ ChanExchange<NV> sm, smy;   // parts of R, of Y
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g4 = lane >> 4, n16 = lane & 15;
  const int nchains = p.B * p.H;
  const int work = xcd_remap(blockIdx.x, nchains * (Sp::NVT / NV));   // a chain's workgroups read one record: one XCD
  const int chain = work / (Sp::NVT / NV), V0 = NV * (work % (Sp::NVT / NV));
  const int h = chain % p.H, b = chain / p.H;
  const int NC = (p.T + CC - 1) / CC;
  const size_t NR = (size_t)nchains * NC;
  const unsigned rsb = (unsigned)((size_t)p.H * D * 4);

  f32x4 S[NV][KT];   // S[v][t][i] = S0[16 (KT wave + t) + 4 g + i][16 (V0 + v) + n]
#pragma unroll
  for (int v = 0; v < NV; ++v)
#pragma unroll
    for (int t = 0; t < KT; ++t) {
      S[v][t] = zero4();
      if (p.s0) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          S[v][t][i] = p.s0[(size_t)chain * D * D + ((KT * wave + t) * 16 + 4 * g4 + i) * D + 16 * (V0 + v) + n16];
      }
    }
  struct Ops {
    f32x4 nw[KT], qe[KT], kf[KT], eg[KT], u[NV];
    float aq;   // column 4 g + wave of Aq: each wave takes a quarter of Aq R's sum
  };
  const unsigned orow = (n16 * D + 4 * g4) * 4, ocol = (n16 * CC + 4 * g4) * 4, ou = (4 * g4 * D + n16) * 4, oe = 16 * g4;
  auto fetch = [&](Ops& x, int c) {
    load_fence();
    const float* fr = p.frec + rec_index(chain, c, nchains) * Rc::FN;
    const __amdgpu_buffer_rsrc_t rr = __builtin_amdgcn_make_buffer_rsrc((void*)fr, 0, Rc::FN * 4, 0x00020000);
    const int kw = 16 * KT * wave;
#pragma unroll
    for (int t = 0; t < KT; ++t) {
      x.nw[t] = rec_load4(rr, orow, Rc::F_NWM + 16 * t + kw);
      x.qe[t] = rec_load4(rr, orow, Rc::F_QE + 16 * t + kw);
      x.kf[t] = rec_load4(rr, ocol, Rc::F_KFT + (16 * t + kw) * CC);
      x.eg[t] = rec_load4(rr, oe, Rc::F_EGL + 16 * t + kw);
    }
    x.aq = rec_load1(rr, ocol, Rc::F_AQ + wave);
#pragma unroll
    for (int v = 0; v < NV; ++v)
#pragma unroll
      for (int s = 0; s < 4; ++s) x.u[v][s] = rec_load1(rr, ou, Rc::F_U + s * D + 16 * (V0 + v));
    load_fence();
  };
  // chunk c's output from the waves' parts (one wave a tile, after the barrier that follows them)
  auto y_out = [&](int c, int v) {
    const f32x4 yt = tile_transpose((float*)nullptr, smy.sum(c, v, lane), lane);
    const __amdgpu_buffer_rsrc_t yr = chunk_rsrc((const float*)p.y, b, c * CC, p.T, p.H, h, D);
    buf_store4(yr, (unsigned)n16 * rsb + (16 * (V0 + v) + 4 * g4) * 4, (const float*)nullptr, yt[0], yt[1], yt[2], yt[3]);
  };
  auto step = [&](const Ops& x, int c) {
    const size_t rec = rec_index(chain, c, nchains);
    if constexpr (STASH) {
      float* cst = (float*)p.chunk_states + rec * (D * D);
#pragma unroll
      for (int v = 0; v < NV; ++v)
#pragma unroll
        for (int t = 0; t < KT; ++t)
          *(f32x4*)(cst + stash_tile_offset<float, D>(KT * wave + t, V0 + v, lane)) = S[v][t];
    }
    // this wave's keys of R = U - Wm S0 (U with wave 0) and of (Q o e^G) S0
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      f32x4 r = wave == 0 ? x.u[v] : zero4(), r1 = zero4();
      mma2(r, r1, x.nw, S[v]);
      sm.r[c & 1][v][wave][lane] = r + r1;
    }
    lds_barrier();
    f32x4 y[NV], R[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) {   // (while the parts arrive)
      f32x4 y1 = zero4();
      y[v] = zero4();
      mma2(y[v], y1, x.qe, S[v]);
      y[v] += y1;
    }
    // S = diag(e^{G_L}) S0 + (K o e^{G_L - G})^T R
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      R[v] = sm.sum(c, v, lane);
#pragma unroll
      for (int t = 0; t < KT; ++t) {
        S[v][t] *= x.eg[t];
        mma(S[v][t], x.kf[t], R[v]);
      }
    }
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      smy.r[c & 1][v][wave][lane] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.aq, pick4(R[v], wave), y[v], 0, 0, 0);
      if (c > 0 && wave == ((c + 1 + v) & 3)) y_out(c - 1, v);
      if constexpr (STASH)
        if (wave == ((c + 2 + v) & 3)) {
          float* rst = (float*)p.chunk_states + NR * D * D + rec * (CC * D);
          *(f32x4*)(rst + stash_tile_offset<float, D>(0, V0 + v, lane)) = R[v];
        }
      if constexpr (SCORE && NV < Sp::NVT)
        if (wave == 0) {   // (U's reader)
          float* fr = p.frec + rec * Rc::FN;
          const f32x4 sq = R[v] * R[v];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float n2 = row_prefix16(sq[e]);
            if (n16 == 15) fr[Rc::F_U + (4 * g4 + e) * D + 16 * (V0 + v)] = n2;
          }
        }
    }
    if constexpr (SCORE && NV == Sp::NVT)
      if (wave == (c & 3)) {   // all value columns are here
        f32x4 sq = zero4();
#pragma unroll
        for (int v = 0; v < NV; ++v) sq += R[v] * R[v];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float n2 = row_prefix16(sq[e]);
          const int t = c * CC + 4 * g4 + e;
          if (n16 == 15 && t < p.T) p.r_norm[((size_t)b * p.T + t) * p.H + h] = sqrtf(n2);
        }
      }
  };
  Ops x[PF];
#pragma unroll
  for (int j = 0; j < PF; ++j) {
    fetch(x[j], min(j, NC - 1));   // (in order: a chunk's wait leaves the later ones in flight)
  }
#pragma clang loop unroll(disable)
  for (int c0 = 0; c0 < NC; c0 += PF) {   // (one exit, and the same loads in flight on every path)
#pragma unroll
    for (int j = 0; j < PF; ++j) {
      if (c0 + j < NC) step(x[j], c0 + j);
      fetch(x[j], min(c0 + j + PF, NC - 1));
    }
  }
  lds_barrier();
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    if (NC > 0 && wave == (v & 3)) y_out(NC - 1, v);
    if (p.s_out) {
#pragma unroll
      for (int t = 0; t < KT; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          p.s_out[(size_t)chain * D * D + ((KT * wave + t) * 16 + 4 * g4 + i) * D + 16 * (V0 + v) + n16] = S[v][t][i];
    }
  }
}

template <int D>
__global__ void __launch_bounds__(256) chan_rnorm_kernel(ChanArgs p) {
  typedef ChRec<D> Rc;
  const int nchains = p.B * p.H;
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;   // (chain, token)
  if (i >= (long long)nchains * p.T) return;
  const int t = (int)(i % p.T), chain = (int)(i / p.T), h = chain % p.H, b = chain / p.H;
  const float* u = p.frec + rec_index(chain, t / CC, nchains) * Rc::FN + Rc::F_U + (t % CC) * D;
  float s = 0.f;
#pragma unroll
  for (int V = 0; V < D / 16; ++V) s += u[16 * V];
  p.r_norm[((size_t)b * p.T + t) * p.H + h] = sqrtf(s);
}

// reverse scan of the state gradient:
//   dR = Aq^T dY + (K o e^{G_L - G}) dS,  dB = T^T dR
//   dS0 = diag(e^{G_L}) dS + (Q o e^G)^T dY - (K o e^G)^T diag(beta_e) dB
// where (K o e^G)^T diag(beta_e) T^T = Wm^T, so dS takes dR itself and dB is
// only formed for the stash
template <int D, int NV>
__global__ void __launch_bounds__(256, 2) chan_split_bwd_kernel(ChanBwdArgs p) {
  typedef ChRec<D> Rc;
  typedef ChSplit<D> Sp;
  constexpr int KT = Sp::KT, PF = Sp::PF(NV, false);
  __shared__ ChanExchange<NV> sm;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g4 = lane >> 4, n16 = lane & 15;
  const int nchains = p.B * p.H;
  const int work = xcd_remap(blockIdx.x, nchains * (Sp::NVT / NV));
  const int chain = work / (Sp::NVT / NV), V0 = NV * (work % (Sp::NVT / NV));
  const int h = chain % p.H, b = chain / p.H;
  const int NC = (p.T + CC - 1) / CC;
  const size_t NR = (size_t)nchains * NC;
  const float* brec = (const float*)p.s_stash + NR * ((size_t)D * D + CC * D + Rc::FN);

  f32x4 dS[NV][KT];
#pragma unroll
  for (int v = 0; v < NV; ++v)
#pragma unroll
    for (int t = 0; t < KT; ++t) {
      dS[v][t] = zero4();
      if (p.ds_final) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          dS[v][t][i] = p.ds_final[(size_t)chain * D * D + ((KT * wave + t) * 16 + 4 * g4 + i) * D + 16 * (V0 + v) + n16];
      }
    }
  struct Ops {
    f32x4 kf[KT], qt[KT], nw[KT], eg[KT], tt, dy[NV];
    float at;   // column 4 g + wave of Aq^T: each wave takes a quarter of Aq^T dY's sum
  };
  const unsigned orow = (n16 * D + 4 * g4) * 4, ocol = (n16 * CC + 4 * g4) * 4, oe = 16 * g4;
  auto fetch = [&](Ops& x, int c) {
    load_fence();
    const float* br = brec + rec_index(chain, c, nchains) * Rc::BN;
    const __amdgpu_buffer_rsrc_t rr = __builtin_amdgcn_make_buffer_rsrc((void*)br, 0, Rc::BN * 4, 0x00020000);
    const int kw = 16 * KT * wave;
#pragma unroll
    for (int t = 0; t < KT; ++t) {
      x.kf[t] = rec_load4(rr, orow, Rc::B_KF + 16 * t + kw);
      x.qt[t] = rec_load4(rr, ocol, Rc::B_QET + (16 * t + kw) * CC);
      x.nw[t] = rec_load4(rr, ocol, Rc::B_NWT + (16 * t + kw) * CC);
      x.eg[t] = rec_load4(rr, oe, Rc::B_EGL + 16 * t + kw);
    }
    x.tt = rec_load4(rr, ocol, Rc::B_TT);
    x.at = rec_load1(rr, ocol, Rc::B_AQT + wave);
#pragma unroll
    for (int s = 0; s < 4; ++s) {   // dY as a B operand; rows past T (masked where used) read the last
      const int t = min(c * CC + 4 * g4 + s, p.T - 1);
#pragma unroll
      for (int v = 0; v < NV; ++v) x.dy[v][s] = p.dy[(((size_t)b * p.T + t) * p.H + h) * D + 16 * (V0 + v) + n16];
    }
    load_fence();
  };
  auto step = [&](const Ops& x, int c) {
    const size_t rec = rec_index(chain, c, nchains);
    float* cst = (float*)p.ds_stash + rec * (D * D);
    f32x4 dY[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) {
#pragma unroll
      for (int t = 0; t < KT; ++t)
        *(f32x4*)(cst + stash_tile_offset<float, D>(KT * wave + t, V0 + v, lane)) = dS[v][t];
#pragma unroll
      for (int s = 0; s < 4; ++s) dY[v][s] = c * CC + 4 * g4 + s < p.T ? x.dy[v][s] : 0.f;
      f32x4 r = zero4(), r1 = __builtin_amdgcn_mfma_f32_16x16x4f32(x.at, pick4(dY[v], wave), zero4(), 0, 0, 0);
      mma2(r, r1, x.kf, dS[v]);
      sm.r[c & 1][v][wave][lane] = r + r1;
    }
    lds_barrier();
#pragma unroll
    for (int v = 0; v < NV; ++v)
#pragma unroll
      for (int t = 0; t < KT; ++t) {   // (while the parts arrive)
        dS[v][t] *= x.eg[t];
        mma(dS[v][t], x.qt[t], dY[v]);
      }
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const f32x4 dR = sm.sum(c, v, lane);
#pragma unroll
      for (int t = 0; t < KT; ++t) mma(dS[v][t], x.nw[t], dR);
      if (wave == ((c + v) & 3)) {
        f32x4 dB = zero4();
        mma(dB, x.tt, dR);
        float* bst = (float*)p.ds_stash + NR * D * D + rec * (CC * D);
        *(f32x4*)(bst + stash_tile_offset<float, D>(0, V0 + v, lane)) = dB;
      }
    }
  };
  Ops x[PF];
#pragma unroll
  for (int j = 0; j < PF; ++j) {
    fetch(x[j], max(NC - 1 - j, 0));
  }
#pragma clang loop unroll(disable)
  for (int c0 = NC - 1; c0 >= 0; c0 -= PF) {
#pragma unroll
    for (int j = 0; j < PF; ++j) {
      if (c0 - j >= 0) step(x[j], c0 - j);
      fetch(x[j], max(c0 - j - PF, 0));
    }
  }
  if (p.ds0) {
#pragma unroll
    for (int v = 0; v < NV; ++v)
#pragma unroll
      for (int t = 0; t < KT; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          p.ds0[(size_t)chain * D * D + ((KT * wave + t) * 16 + 4 * g4 + i) * D + 16 * (V0 + v) + n16] = dS[v][t][i];
  }
}

// ---------------------------------------------------------------------------
// per-chunk gradients (one chain per head: no lane sums)
//   P1 = dY S0^T, P2 = dB S0^T, P3 = R dS^T        (wave w: key tile w)
//   dq  = e^G o P1 + [grams],   dk = -beta_e e^G o P2 + e^{G_L - G} o P3 + [grams]
//   dG  = e^G o (q o P1 - beta_e k o P2) - e^{G_L - G} o k o P3 + [grams]
//   dG_L += sum_i e^{G_L - G} o k o P3 + e^{G_L} o rowsum(dS o S0)
//   dlog_g_t = sum_{i >= t} dG_i (zero where the log-decay was clamped)
//   dv = diag(beta_w) dB,  dbeta_w = rowsum(dB o V),
//   dbeta_e = -rowsum(e^G o k o P2) + rowsum(dL o M[x=k])
// with dAq = dY R^T (j <= i), dL = -dB R^T (j < i) entering the grams
// exactly, channel by channel.
// ---------------------------------------------------------------------------
template <int D>
struct alignas(16) ChanGradSmem {
  static constexpr int LDD = D + 4;
  ChanOps<D> o;
  float v[CC * LDD];
  float dy[CC * LDD];
  float R[CC * LDD];
  float dB[CC * LDD];
  float raw[CC * LDD];   // unclamped log-decay (gradient mask)
  float dAq[CC * LDC];
  float dL[CC * LDC];
  float sdot[D];         // rowsum(dS o S0) per key channel
  float red[2][ChD<D>::NW][CC];   // per-wave partial row sums: dbeta_e, dbeta_w
};

// Bound by the latency of its LDS reads and by how many workgroups hide it:
// registers are held to what lets LDS's two (d = 128; three at 64) stay on a CU
// (128 of them; at 138, and with a branch and single LDS reads per pair of
// tokens, one did).  B = 2, T = 512, H = 16, d = 128: 108 -> 80 us.
template <int D>
__global__ void __launch_bounds__(64 * (D / 16), D == 128 ? 4 : 3) chan_grads_kernel(ChanBwdArgs p) {
  typedef ChD<D> Cd;
  constexpr int NW = Cd::NW, NT = Cd::NT, NDT = Cd::NDT, LDD = Cd::LDD;
  __shared__ ChanGradSmem<D> sm;
  ChanOps<D>& o = sm.o;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, g4 = lane >> 4, n16 = lane & 15;
  const int NC = (p.T + CC - 1) / CC;
  const int nchains = p.B * p.H;
  const int blk = xcd_remap(blockIdx.x, nchains * NC);
  const int c = blk % NC, chain = blk / NC;
  const int h = chain % p.H, b = chain / p.H;
  const int t0 = c * CC;
  const size_t NR = (size_t)nchains * NC;
  const size_t rec = rec_index(chain, c, nchains);
  const int d = 16 * wave + n16;   // this lane's key (and value) column
  const unsigned rsb = (unsigned)((size_t)p.H * D * 4);

  // stage the chunk: q, k, v, log-decay, dY (rows), scalars; this wave's R and
  // dB tiles into LDS rows; this wave's key rows of S0 and dS into registers
  f32x4 s0t[NDT], dst[NDT];
  {
    Stage<float, CC, D, 1, NT> sq, sk, sv, sl, sy;
    sq.fetch(chunk_rsrc(p.q, b, t0, p.T, p.H, h, D), rsb, tid);
    sk.fetch(chunk_rsrc(p.k, b, t0, p.T, p.H, h, D), rsb, tid);
    sv.fetch(chunk_rsrc(p.v, b, t0, p.T, p.H, h, D), rsb, tid);
    sl.fetch(chunk_rsrc(p.lg, b, t0, p.T, p.H, h, D), rsb, tid);
    sy.fetch(chunk_rsrc(p.dy, b, t0, p.T, p.H, h, D), rsb, tid);
    const float* srec = (const float*)p.s_stash + rec * (D * D);
    const float* drec = (const float*)p.ds_stash + rec * (D * D);
#pragma unroll
    for (int V = 0; V < NDT; ++V) {
      s0t[V] = *(const f32x4*)(srec + stash_tile_offset<float, D>(wave, V, lane));
      dst[V] = *(const f32x4*)(drec + stash_tile_offset<float, D>(wave, V, lane));
    }
    const f32x4 rt = *(const f32x4*)((const float*)p.s_stash + NR * D * D + rec * (CC * D) +
                                     stash_tile_offset<float, D>(0, wave, lane));
    const f32x4 bt = *(const f32x4*)((const float*)p.ds_stash + NR * D * D + rec * (CC * D) +
                                     stash_tile_offset<float, D>(0, wave, lane));
    const float be = chunk_scalar(p.be, b, t0, tid % CC, p.T, p.H, h);
    const float bw = chunk_scalar(p.bw, b, t0, tid % CC, p.T, p.H, h);
    sq.template commit_nat<LDD>(o.q, tid);
    sk.template commit_nat<LDD>(o.k, tid);
    sv.template commit_nat<LDD>(sm.v, tid);
    sl.template commit_nat<LDD>(o.G, tid);
    sl.template commit_nat<LDD>(sm.raw, tid);
    sy.template commit_nat<LDD>(sm.dy, tid);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      sm.R[(4 * g4 + i) * LDD + d] = rt[i];
      sm.dB[(4 * g4 + i) * LDD + d] = bt[i];
    }
    if (tid < CC) {
      o.be[tid] = be;
      o.bw[tid] = bw;
    }
  }
  {   // rowsum(dS o S0) over this wave's key rows 16 wave + 4 g + i
    f32x4 s = zero4();
#pragma unroll
    for (int V = 0; V < NDT; ++V) s += s0t[V] * dst[V];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float x = s[e];
#pragma unroll
      for (int off = 1; off < 16; off <<= 1) x += __shfl_xor(x, off, 64);
      if (n16 == 0) sm.sdot[16 * wave + 4 * g4 + e] = x;
    }
  }
  __syncthreads();
  chan_prefix<D>(o, tid);
  __syncthreads();
  chan_grams<D>(o, wave, lane);
  if (wave == 0 || wave == 1) {   // dAq = dY R^T (j <= i), dL = -dB R^T (j < i)
    const float* arow = (wave == 0) ? &sm.dy[n16 * LDD] : &sm.dB[n16 * LDD];
    const f32x4 acc = tile_nt<float, D>(arow, &sm.R[n16 * LDD], g4);
#pragma unroll
    for (int ii = 0; ii < 4; ++ii) {
      const int i = 4 * g4 + ii, j = n16;
      if (wave == 0) sm.dAq[i * LDC + j] = (j <= i) ? acc[ii] : 0.f;
      else sm.dL[i * LDC + j] = (j < i) ? -acc[ii] : 0.f;
    }
  }
  __syncthreads();

  // P products on this wave's key tile (S0 / dS rows as fragments over k = v)
  f32x4 P1 = zero4(), P2 = zero4(), P3 = zero4();
#pragma unroll
  for (int kb = 0; kb < NDT; ++kb) {
    const f32x4 Sf = tile_transpose_raw(s0t[kb], lane);
    const f32x4 dSf = tile_transpose_raw(dst[kb], lane);
    mma(P1, ld_frag(&sm.dy[n16 * LDD + kb * 16], g4), Sf);
    mma(P2, ld_frag(&sm.dB[n16 * LDD + kb * 16], g4), Sf);
    mma(P3, ld_frag(&sm.R[n16 * LDD + kb * 16], g4), dSf);
  }
  // lane (g, n): rows i = 4 g + ii of column d
  const float GL = o.G[(CC - 1) * LDD + d];
  float dq[4], dk[4], dG[4], dGLp = 0.f, pbe[4], Gi[4], ki[4], qi[4], bei[4];
#pragma unroll
  for (int ii = 0; ii < 4; ++ii) {
    const int i = 4 * g4 + ii;
    Gi[ii] = o.G[i * LDD + d];
    ki[ii] = o.k[i * LDD + d];
    qi[ii] = o.q[i * LDD + d];
    bei[ii] = o.be[i];
    const float E = __expf(Gi[ii]), F = __expf(GL - Gi[ii]);
    dq[ii] = E * P1[ii];
    dk[ii] = -bei[ii] * E * P2[ii] + F * P3[ii];
    dG[ii] = E * (qi[ii] * P1[ii] - bei[ii] * ki[ii] * P2[ii]) - F * ki[ii] * P3[ii];
    dGLp += F * ki[ii] * P3[ii];
    pbe[ii] = -E * ki[ii] * P2[ii];
  }
  // grams, row i as the query / erase side (j <= i) and as the key side
  // (i <= j).  The prefix never rises, so that one exponential of -|G_i - G_j|
  // serves both; what a row does not take is selected away (a NaN of a later
  // token stays there), so that no lane branches and the LDS reads, four
  // values each, run ahead of the sums.
#pragma unroll 1   // (all blocks' reads at once would spill)
  for (int jb = 0; jb < CC / 4; ++jb) {
    f32x4 ar[4], lr[4];
#pragma unroll
    for (int ii = 0; ii < 4; ++ii) {
      ar[ii] = *(const f32x4*)&sm.dAq[(4 * g4 + ii) * LDC + 4 * jb];
      lr[ii] = *(const f32x4*)&sm.dL[(4 * g4 + ii) * LDC + 4 * jb];
    }
    const f32x4 bej = *(const f32x4*)&o.be[4 * jb];
#pragma unroll
    for (int jj = 0; jj < 4; ++jj) {
      const int j = 4 * jb + jj;
      const float Gj = o.G[j * LDD + d], kj = o.k[j * LDD + d], qj = o.q[j * LDD + d];
      const f32x4 ac = *(const f32x4*)&sm.dAq[j * LDC + 4 * g4], lc = *(const f32x4*)&sm.dL[j * LDC + 4 * g4];
#pragma unroll
      for (int ii = 0; ii < 4; ++ii) {
        const bool lo = j <= 4 * g4 + ii, hi = j >= 4 * g4 + ii;
        const float ex = __expf(-fabsf(Gi[ii] - Gj));
        const float t1 = ar[ii][jj] * ex, t2 = lr[ii][jj] * bei[ii] * ex;
        const float cc = (ac[ii] * qj + lc[ii] * bej[jj] * kj) * ex;
        dq[ii] += lo ? t1 * kj : 0.f;
        dk[ii] += lo ? t2 * kj : 0.f;
        dG[ii] += lo ? (t1 * qi[ii] + t2 * ki[ii]) * kj : 0.f;
        dk[ii] += hi ? cc : 0.f;
        dG[ii] -= hi ? cc * ki[ii] : 0.f;
      }
    }
  }
  // chunk-end decay: the column's dG_L, added to every token's suffix sum
  dGLp += __shfl_xor(dGLp, 16, 64);
  dGLp += __shfl_xor(dGLp, 32, 64);
  const float dGL = dGLp + o.eGL[d] * sm.sdot[d];
  // suffix sums over the chunk's rows (within the lane, then across g)
  float tot = (dG[0] + dG[1]) + (dG[2] + dG[3]);
  const float t1 = __shfl_down(tot, 16, 64), t2 = __shfl_down(tot, 32, 64), t3 = __shfl_down(tot, 48, 64);
  float above = dGL + (g4 < 3 ? t1 : 0.f) + (g4 < 2 ? t2 : 0.f) + (g4 < 1 ? t3 : 0.f);
  float dlg[4];
#pragma unroll
  for (int ii = 3; ii >= 0; --ii) {
    above += dG[ii];
    const float raw = sm.raw[(4 * g4 + ii) * LDD + d];
    dlg[ii] = (raw <= 0.f && raw >= kLogFloor) ? above : 0.f;
  }
  // per-token sums: dbeta_e over the key columns, dbeta_w over the value columns
  float dvv[4];
#pragma unroll
  for (int ii = 0; ii < 4; ++ii) {
    const int i = 4 * g4 + ii;
    const float dbv = sm.dB[i * LDD + d];
    dvv[ii] = o.bw[i] * dbv;
    float xe = pbe[ii], xw = dbv * sm.v[i * LDD + d];
#pragma unroll
    for (int off = 1; off < 16; off <<= 1) {
      xe += __shfl_xor(xe, off, 64);
      xw += __shfl_xor(xw, off, 64);
    }
    if (n16 == 0) {
      sm.red[0][wave][i] = xe;
      sm.red[1][wave][i] = xw;
    }
  }
  // stores: rows past T fall outside the buffer resources
  {
    const __amdgpu_buffer_rsrc_t rq = chunk_rsrc((const float*)p.dq, b, t0, p.T, p.H, h, D);
    const __amdgpu_buffer_rsrc_t rk = chunk_rsrc((const float*)p.dk, b, t0, p.T, p.H, h, D);
    const __amdgpu_buffer_rsrc_t rv = chunk_rsrc((const float*)p.dv, b, t0, p.T, p.H, h, D);
    const __amdgpu_buffer_rsrc_t rg = chunk_rsrc(p.dlg, b, t0, p.T, p.H, h, D);
#pragma unroll
    for (int ii = 0; ii < 4; ++ii) {
      const unsigned off = (unsigned)(4 * g4 + ii) * rsb + d * 4;
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(dq[ii]), rq, (int)off, 0, 0);
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(dk[ii]), rk, (int)off, 0, 0);
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(dvv[ii]), rv, (int)off, 0, 0);
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(dlg[ii]), rg, (int)off, 0, 0);
    }
  }
  __syncthreads();
  if (tid < CC && t0 + tid < p.T) {
    float se = 0.f, sw = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      se += sm.red[0][w][tid];
      sw += sm.red[1][w][tid];
    }
    // the erase coefficient also scales L: + sum_j dL_ij M_ij
#pragma unroll
    for (int j = 0; j < CC; ++j) se += sm.dL[tid * LDC + j] * o.Mk[tid * LDC + j];
    const size_t si = ((size_t)b * p.T + t0 + tid) * p.H + h;
    p.dbe[si] = se;
    p.dbw[si] = sw;
  }
}

// Value tiles per workgroup of the scans: one while each of the 256 CUs
// gets one workgroup at most (the step's latency counts), two up to two full
// rounds of the chip, four beyond (a record is read D / 64 times instead of D / 16, and
// more products stand between two barriers).  The whole call, T = 512, training
// (1 | 2 | 4 tiles) at d = 128: 32 chains 231 | 262 | 331 us, 48: 344 | 322 | 389,
// 64: 423 | 398 | 458, 96: 612 | 586 | 571, 128: 781 | 693 | 673, 256: 1509 | 1337 |
// 1244; at d = 64, 64 chains 182 | 210 | 256, 128: 341 | 321 | 360, 256: 632 | 577 |
// 550.
static int chan_tiles(int nchains, int D) {
  const long long tiles = (long long)nchains * (D / 16);
  return tiles <= 256 ? 1 : tiles < 1024 ? 2 : 4;
}

// Up to this many chunks four tiles a workgroup, which need no launch for |r_t|
// after the scan, are at d = 64 no slower than the narrower split (2 chains, T =
// 16: 86 -> 82 us a scored call; at 128 tokens 84 -> 88, so no more).
constexpr int kScoreChunks = 4;

template <int D, int NV>
static int launch_chan_scan(const ChanArgs& a, hipStream_t stream) {
  const dim3 grid(a.B * a.H * (ChSplit<D>::NVT / NV)), block(256);
  const bool train = a.chunk_states != nullptr;
  if (train && a.r_norm) hipLaunchKernelGGL((chan_split_fwd_kernel<D, NV, true, true>), grid, block, 0, stream, a);
  else if (train) hipLaunchKernelGGL((chan_split_fwd_kernel<D, NV, true, false>), grid, block, 0, stream, a);
  else if (a.r_norm) hipLaunchKernelGGL((chan_split_fwd_kernel<D, NV, false, true>), grid, block, 0, stream, a);
  else hipLaunchKernelGGL((chan_split_fwd_kernel<D, NV, false, false>), grid, block, 0, stream, a);
  return check_launch("chan_split_fwd_kernel");
}

template <int D>
static int launch_chan_fwd(ChanArgs a, hipStream_t stream) {
  typedef ChRec<D> Rc;
  const int nchains = a.B * a.H, NC = (a.T + CC - 1) / CC;
  const size_t NR = (size_t)nchains * NC;
  const bool train = a.chunk_states != nullptr;
  a.frec = train ? (float*)a.chunk_states + NR * ((size_t)D * D + CC * D) : (float*)a.workspace;
  a.brec = train ? a.frec + NR * Rc::FN : nullptr;
  if (train)
    hipLaunchKernelGGL((chan_prep_kernel<D, true>), dim3(nchains * NC), dim3(64 * (D / 16)), 0, stream, a);
  else
    hipLaunchKernelGGL((chan_prep_kernel<D, false>), dim3(nchains * NC), dim3(64 * (D / 16)), 0, stream, a);
  int rc = check_launch("chan_prep_kernel");
  if (rc) return rc;
  int nv = chan_tiles(nchains, D);
  if (a.r_norm && D == 64 && NC <= kScoreChunks) nv = 4;
  rc = nv == 1 ? launch_chan_scan<D, 1>(a, stream)
               : nv == 2 ? launch_chan_scan<D, 2>(a, stream) : launch_chan_scan<D, 4>(a, stream);
  if (rc || !a.r_norm || nv == ChSplit<D>::NVT) return rc;
  const long long n = (long long)nchains * a.T;
  hipLaunchKernelGGL((chan_rnorm_kernel<D>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, a);
  return check_launch("chan_rnorm_kernel");
}

template <int D>
static int launch_chan_bwd(const ChanBwdArgs& a, hipStream_t stream) {
  const int NC = (a.T + CC - 1) / CC;
  const int nv = chan_tiles(a.B * a.H, D);
  const dim3 grid(a.B * a.H * (ChSplit<D>::NVT / nv)), block(256);
  if (nv == 1) hipLaunchKernelGGL((chan_split_bwd_kernel<D, 1>), grid, block, 0, stream, a);
  else if (nv == 2) hipLaunchKernelGGL((chan_split_bwd_kernel<D, 2>), grid, block, 0, stream, a);
  else hipLaunchKernelGGL((chan_split_bwd_kernel<D, 4>), grid, block, 0, stream, a);
  int rc = check_launch("chan_split_bwd_kernel");
  if (rc) return rc;
  hipLaunchKernelGGL((chan_grads_kernel<D>), dim3(a.B * a.H * NC), dim3(64 * (D / 16)), 0, stream, a);
  return check_launch("chan_grads_kernel");
}

int chan_fwd_dispatch(const ChanArgs& a, hipStream_t stream) {
  if (a.D == 128) return launch_chan_fwd<128>(a, stream);
  if (a.D == 64) return launch_chan_fwd<64>(a, stream);
  return set_error(GDNX_ERR_SHAPE, "per-channel decay: head_dim %d unsupported (64 or 128)", a.D);
}

int chan_bwd_dispatch(const ChanBwdArgs& a, hipStream_t stream) {
  if (a.D == 128) return launch_chan_bwd<128>(a, stream);
  if (a.D == 64) return launch_chan_bwd<64>(a, stream);
  return set_error(GDNX_ERR_SHAPE, "per-channel decay: head_dim %d unsupported (64 or 128)", a.D);
}

size_t chan_states_bytes(int nchains, int T, int D) {
  const size_t NR = (size_t)nchains * ((T + CC - 1) / CC);
  const size_t rec = D == 128 ? ChRec<128>::FN + ChRec<128>::BN : ChRec<64>::FN + ChRec<64>::BN;
  return NR * ((size_t)D * D + (size_t)CC * D + rec) * 4;
}

size_t chan_fwd_workspace_bytes(int nchains, int T, int D) {
  const size_t NR = (size_t)nchains * ((T + CC - 1) / CC);
  return NR * (size_t)(D == 128 ? ChRec<128>::FN : ChRec<64>::FN) * 4;
}

}  // namespace gdnx
