// GDN3 Kronecker-residual forward over intervals of many sub-chunks (gfx950).
//
// Between two compactions the Kronecker factors are constants and a token
// sees only the P writes before it, so the recurrence over 16-token
// sub-chunks is, per value column,
//     U_c = X_c - sum_b W_{c,b} U_b,    X_c = T_c (alpha u - kco Kr(h)),    W_{c,b} = T_c Ho_{c,b}
//     y_c = qco Kr(q) + sum_b Qo_{c,b} U_b + Aq_c U_c
// with b over the window's NB = P / 16 blocks and T, Ho, Qo, Aq the 16 x 16
// matrices of gdn3.hip's header: all of a sub-chunk's work but the one 16 x
// 16 product with the blocks' U is independent of the sub-chunks before it,
// and U enters linearly.  So an interval is cut into runs of whole batches
// of four sub-chunks:
//   pass 1 (every run but the last) scans its run from U = 0, and beside the
//     D value columns 16 NB further columns whose X is zero and whose U
//     starts as the identity: the run's map of the window, U_end = U0 + V U_start;
//   pass 2 folds the maps of the runs before it into its own starting window
//     and scans its run for the outputs.
// A workgroup takes a batch at a time.  In the first half wave w forms
// sub-chunk w's matrices from its own loads (no workgroup barrier): the token
// rows go from memory into MFMA fragments, 16 bytes a lane (the k order inside
// a product is free as long as both operands share it).  In the second half
// wave w takes its value tiles through the batch's sub-chunks with U and its
// rows of the Kronecker matrix in registers, which leaves one dependent 16 x
// 16 x 16 product per sub-chunk; H and Q reach it through LDS as fragments.
//
// Bound: the fp32 products of the second half (16 x 16 x 4 MFMA, 512 of the
// ~640 matrix-core cycles per value tile and sub-chunk), then latency.
// Measured at B = 1, T = 32768, H = 16, 4 lanes, d = 128, P = 16, a compaction
// every 2048 (64 chains): see the launch rule below.
#include <utility>

#include "gdn3_common.hpp"
#include "gdnx_internal.hpp"

namespace gdnx {
namespace {

constexpr int kBatch = 4;   // sub-chunks a workgroup prepares at once, one per wave

template <typename CT, int D, int P>
struct G3RunSmem {
  static constexpr int NB = P / kSC, KB = D / FragT<CT>::KSTEP;
  typedef typename FragT<CT>::type Frag;
  Frag hx[kBatch][KB][64];                                  // H rows of the batch as A fragments
  Frag qx[kBatch][KB][64];                                  // Q rows
  alignas(16) float mt[kBatch][2 + 2 * NB][kSC][kSC + 4];   // T, Aq, -W_b, Qo_b
  alignas(16) float al[kBatch][kSC], kco[kBatch][kSC], qco[kBatch][kSC];
  float red[kNT / 64];
  float suf[128];                                           // log decay after a token, to the interval's end
};

// GL: gate layout (1: a scalar per lane, 2: per channel).  FULL: pass 2.
template <typename CT, int D, int P, int GL, bool FULL>
__global__ void __launch_bounds__(kNT) gdn3_run_kernel(G3FwdArgs p) {
  typedef G3RunSmem<CT, D, P> Sm;
  typedef typename FragT<CT>::type Frag;
  typedef G3D<D> Ge;
  constexpr int NB = Sm::NB, KS = FragT<CT>::KSTEP, KB = Sm::KB, EPL = KS / 4;   // elements a lane holds of a k-step
  constexpr int TPW = D / 64;                                                     // value tiles per wave
  static_assert(sizeof(Frag) == 16 && EPL * sizeof(CT) == 16, "a fragment is one 16-byte load");
  static_assert(NB >= 1 && NB <= kBatch && D % 64 == 0, "the decay window holds the last four sub-chunks");
  __shared__ Sm sm;

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g4 = lane >> 4, n16 = lane & 15;
  const int T = p.T, t0 = p.t0, M = p.M;
  const int nr = FULL ? p.nrun : p.nrun - 1;
  // the lanes of a head's run, which share q, k and v, are neighbours on an XCD
  const int work = xcd_remap(blockIdx.x, p.B * p.H * M * nr);
  const int r = (work / M) % nr, chain = (work / M / nr) * M + work % M;
  const int cs = p.c0 + r * p.rlen, ce = min(cs + p.rlen, p.c1);
  const int tlo = max(t0, kSC * p.c0);   // the first token after the state uw, vw stand for
  const long long tend = (long long)t0 + T, tint = min(tend, (long long)kSC * p.c1);
  const G3Tok tk(p, chain, D);
  const CT* kin = (const CT*)p.k + tk.qkv_base;
  const CT* qin = (const CT*)p.q + tk.qkv_base;
  const CT* vin = (const CT*)p.v + tk.qkv_base;
  const float* uw = p.uw + (size_t)chain * P * D;
  const float* vw = p.vw + (size_t)chain * P * D;
  const bool live = p.live;

  // log decay of global token tau, 0 outside this interval and this call
  auto lgtok = [&](int tau) {
    const bool ok = tau >= tlo && tau < tint;
    const int t = min(max(tau - t0, 0), T - 1);
    const float d = p.dec[tk.dec_base + (size_t)t * tk.dec_tok];
    return ok ? log_decay(d) : 0.f;
  };

  // this wave's value rows of the Kronecker matrix
  Frag sk[TPW][KB];
  if (live)
#pragma unroll
    for (int a = 0; a < TPW; ++a)
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
        sk[a][kb] = *(const Frag*)((const CT*)p.skron + ((size_t)chain * D + (wave * TPW + a) * 16 + n16) * D + kb * KS +
                                   g4 * EPL);

  // the window's net writes: [block][tile], the tiles past TPW (pass 1) the
  // wave's virtual one
  constexpr int TU = FULL ? TPW : TPW + 1;
  f32x4 uo[NB][TU];
#pragma unroll
  for (int bl = 0; bl < NB; ++bl) {
#pragma unroll
    for (int a = 0; a < TPW; ++a) {
      uo[bl][a] = zero4();
      if (FULL && !p.first)
#pragma unroll
        for (int e = 0; e < 4; ++e) uo[bl][a][e] = uw[(bl * kSC + 4 * g4 + e) * D + (wave * TPW + a) * 16 + n16];
    }
    if constexpr (!FULL)
#pragma unroll
      for (int e = 0; e < 4; ++e) uo[bl][TPW][e] = (bl == wave && 4 * g4 + e == n16) ? 1.f : 0.f;
  }

  // the log decay since the interval's start, and the window at the run's
  float gacc = 0.f;
  if (r > 0) {
    float s = 0.f;
    for (int tau = kSC * p.c0 + tid; tau < kSC * cs; tau += kNT) s += lgtok(tau);
    s = wave_sum(s);
    if (lane == 0) sm.red[wave] = s;
    __syncthreads();
    gacc = (sm.red[0] + sm.red[1]) + (sm.red[2] + sm.red[3]);
    if constexpr (FULL) {
#pragma unroll 2
      for (int x = 0; x < r; ++x) {
        const float* ru = p.run_u + ((size_t)chain * p.nrun + x) * P * D;
        const float* rv = p.run_v + ((size_t)chain * p.nrun + x) * P * P;
        f32x4 nu[NB][TPW];
#pragma unroll
        for (int bl = 0; bl < NB; ++bl) {
          f32x4 va[NB];
#pragma unroll
          for (int b2 = 0; b2 < NB; ++b2) va[b2] = *(const f32x4*)&rv[(bl * kSC + n16) * P + b2 * kSC + 4 * g4];
#pragma unroll
          for (int a = 0; a < TPW; ++a)
#pragma unroll
            for (int e = 0; e < 4; ++e) nu[bl][a][e] = ru[(bl * kSC + 4 * g4 + e) * D + (wave * TPW + a) * 16 + n16];
#pragma unroll
          for (int b2 = 0; b2 < NB; ++b2)
#pragma unroll
            for (int a = 0; a < TPW; ++a) mma(nu[bl][a], va[b2], uo[b2][a]);
        }
#pragma unroll
        for (int bl = 0; bl < NB; ++bl)
#pragma unroll
          for (int a = 0; a < TPW; ++a) uo[bl][a] = nu[bl][a];
      }
    }
  }

  for (int cb = cs; cb < ce; cb += kBatch) {
    // log-decay prefixes of the batch's sub-chunks (16-lane row x: sub-chunk
    // cb + x) and of the four before it, and their totals
    const float G1 = row_prefix16(lgtok(kSC * cb + lane)), G0 = row_prefix16(lgtok(kSC * (cb - kBatch) + lane));
    float tot[2 * kBatch];
#pragma unroll
    for (int x = 0; x < kBatch; ++x) {
      tot[x] = lane_value(G0, kSC * x + kSC - 1);
      tot[kBatch + x] = lane_value(G1, kSC * x + kSC - 1);
    }
    const int c = cb + wave;
    float u[kBatch][TPW][4];
    if (c < ce) {
      const int tau = kSC * c + n16, t = tau - t0;
      const bool ok = tau >= t0 && tau < tend;
      const size_t tc = (size_t)min(max(t, 0), T - 1);
      const int lo = max(0, t0 - kSC * c);
      Frag kf[KB], qf[KB], hf[KB];
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        kf[kb] = *(const Frag*)(kin + tc * tk.qkv_tok + kb * KS + g4 * EPL);
        if constexpr (FULL) qf[kb] = *(const Frag*)(qin + tc * tk.qkv_tok + kb * KS + g4 * EPL);
      }
      float part = 0.f;
      {
        const float* bp = p.bg + tk.gate_base + tc * tk.gate_tok;
        float b1 = 0.f;
        if constexpr (GL == 1) b1 = *bp;
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
          float bb[EPL];
#pragma unroll
          for (int e = 0; e < EPL; e += 4) {
            f32x4 b4 = {b1, b1, b1, b1};
            if constexpr (GL == 2) b4 = *(const f32x4*)(bp + kb * KS + g4 * EPL + e);
#pragma unroll
            for (int i = 0; i < 4; ++i) bb[e + i] = b4[i];
          }
#pragma unroll
          for (int e = 0; e < EPL; ++e) {   // an invalid token's row is zero
            kf[kb][e] = ok ? kf[kb][e] : from_f<CT>(0.f);
            if constexpr (FULL) qf[kb][e] = ok ? qf[kb][e] : from_f<CT>(0.f);
            const float kv = to_f(kf[kb][e]), h = bb[e] * kv;
            part += kv * h;
            hf[kb][e] = from_f<CT>(h);
          }
          sm.hx[wave][kb][lane] = hf[kb];
          if constexpr (FULL) sm.qx[wave][kb][lane] = qf[kb];
        }
      }
      const float alpha_l = stable_alpha_f(sum_rows4(part));   // of token n16
      const float gl = __shfl(G1, kSC * wave + n16, 64);       // G of token n16
      float gw = gacc;   // the log decay since the last compaction at the sub-chunk's start
#pragma unroll
      for (int x = 0; x < kBatch; ++x) gw += x < wave ? tot[kBatch + x] : 0.f;
      if (lane < kSC) {
        const float e2 = expf(2.f * (gw + gl));
        sm.al[wave][lane] = alpha_l;
        sm.kco[wave][lane] = alpha_l * e2;
        sm.qco[wave][lane] = e2;
      }
      if (FULL && p.ts_g && lane == 0) p.ts_g[(size_t)chain * p.nch + c] = gw;
      float gi[4], ai[4];
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        gi[s] = __shfl(gl, 4 * g4 + s, 64);
        ai[s] = __shfl(alpha_l, 4 * g4 + s, 64);
      }
      float (*mt)[kSC][kSC + 4] = sm.mt[wave];
      // T = (I + Lm)^-1, Lm[i][j] = alpha_i e^{G_i - G_j} (h_i . k_j), j < i:
      // nilpotent, so (I - L)(I + L^2)(I + L^4)(I + L^8), factors that commute;
      // squarings and products on fp32 MFMA, the A operand of each through
      // LDS (in the places that -W and Aq take afterwards)
      {
        f32x4 acc = zero4();
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) mma(acc, hf[kb], kf[kb]);
        f32x4 xa, ta;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const int i = 4 * g4 + s;
          xa[s] = (n16 < i) ? ai[s] * expf(gi[s] - gl) * acc[s] : 0.f;
          mt[1][i][n16] = xa[s];
          ta[s] = (i == n16 ? 1.f : 0.f) - xa[s];
        }
        wave_lds_sync();
#pragma unroll
        for (int step = 0; step < 3; ++step) {
          const int src = 1 + (step & 1), dst = 3 - src;
          f32x4 sq = zero4();
          mma(sq, *(const f32x4*)&mt[src][n16][4 * g4], xa);   // X^2
          xa = sq;
#pragma unroll
          for (int s = 0; s < 4; ++s) mt[dst][4 * g4 + s][n16] = sq[s];
          wave_lds_sync();
          mma(ta, *(const f32x4*)&mt[dst][n16][4 * g4], ta);   // T += X^2 T
        }
#pragma unroll
        for (int s = 0; s < 4; ++s) mt[0][4 * g4 + s][n16] = ta[s];
        wave_lds_sync();
      }
      const f32x4 trow = *(const f32x4*)&mt[0][n16][4 * g4];
      if constexpr (FULL) {   // Aq = [j <= i] e^{G_i - G_j} q_i.k_j
        f32x4 acc = zero4();
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) mma(acc, qf[kb], kf[kb]);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const int i = 4 * g4 + s;
          mt[1][i][n16] = (n16 <= i) ? expf(gi[s] - gl) * acc[s] : 0.f;
        }
      }
      // the window's blocks: slot 16 b + j holds the key of token j of the
      // last sub-chunk before c that writes block b, or the state's key where
      // that token came before the state; decayed from there to c's start
      //   Ho_b = vis alpha_i e^{G_i + off_j} h_i.k_j,  Qo_b = vis e^{G_i + off_j} q_i.k_j,
      // vis: not yet overwritten by sub-chunk c (the block c itself writes)
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const int dist = (c - 1 - b + kBatch * NB) % NB + 1, x = kBatch + wave - dist;
        const int ktau = kSC * (c - dist) + n16;
        const bool st = ktau < tlo;
        float gx = 0.f, tx = 0.f, after = 0.f, all = 0.f;
#pragma unroll
        for (int z = 0; z < 2 * kBatch; ++z) {
          tx = z == x ? tot[z] : tx;
          after += (z > x && z < kBatch + wave) ? tot[z] : 0.f;
          all += z < kBatch + wave ? tot[z] : 0.f;
        }
        {
          const float g0 = __shfl(G0, (kSC * x + n16) & 63, 64), g1 = __shfl(G1, (kSC * x + n16) & 63, 64);
          gx = x < kBatch ? g0 : g1;
        }
        const float off = st ? all : (tx - gx) + after;
        Frag pf[KB];
        const size_t kc = (size_t)min(max(ktau - t0, 0), T - 1);
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) pf[kb] = *(const Frag*)(kin + kc * tk.qkv_tok + kb * KS + g4 * EPL);
        if (kSC * (c - dist) < tlo) {   // (uniform) rows of the state
#pragma unroll
          for (int kb = 0; kb < KB; ++kb)
#pragma unroll
            for (int e = 0; e < EPL; ++e) {
              const float sv = p.first ? 0.f : vw[(kSC * b + n16) * D + kb * KS + g4 * EPL + e];
              pf[kb][e] = st ? from_f<CT>(sv) : pf[kb][e];
            }
        }
        f32x4 ho = zero4(), qo = zero4();
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
          mma(ho, hf[kb], pf[kb]);
          if constexpr (FULL) mma(qo, qf[kb], pf[kb]);
        }
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const int i = 4 * g4 + s;
          const bool vis = dist != NB || n16 >= i || n16 < lo;
          const float sc = vis ? expf(gi[s] + off) : 0.f;
          ho[s] *= sc * ai[s];
          if constexpr (FULL) mt[2 + NB + b][i][n16] = sc * qo[s];
        }
        f32x4 w = zero4();
        mma(w, trow, ho);
#pragma unroll
        for (int s = 0; s < 4; ++s) mt[2 + b][4 * g4 + s][n16] = -w[s];
      }
    }
    // u = w (.) v at the wave's value columns
#pragma unroll
    for (int s = 0; s < kBatch; ++s)
#pragma unroll
      for (int a = 0; a < TPW; ++a)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int t = kSC * (cb + s) + 4 * g4 + e - t0, v = (wave * TPW + a) * 16 + n16;
          const size_t tc = (size_t)min(max(t, 0), T - 1);
          const float vv = to_f(vin[tc * tk.qkv_tok + v]);
          const float wv = p.wg[tk.gate_base + tc * tk.gate_tok + (GL == 2 ? v : 0)];
          u[s][a][e] = (t >= 0 && t < T) ? wv * vv : 0.f;
        }
    lds_barrier();
#pragma unroll
    for (int s = 0; s < kBatch; ++s) {
      const int cc = cb + s;
      if (cc >= ce) break;
      const int beta = cc % NB, lo = max(0, t0 - kSC * cc);
      const int hi = (int)min((long long)kSC, tend - (long long)kSC * cc);
      const float (*mt)[kSC][kSC + 4] = sm.mt[s];
      const f32x4 al = *(const f32x4*)&sm.al[s][4 * g4], kco = *(const f32x4*)&sm.kco[s][4 * g4];
      const f32x4 qco = *(const f32x4*)&sm.qco[s][4 * g4];
      const f32x4 trow = *(const f32x4*)&mt[0][n16][4 * g4];
      f32x4 wrow[NB], qrow[NB], arow = zero4();
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        wrow[b] = *(const f32x4*)&mt[2 + b][n16][4 * g4];
        if constexpr (FULL) qrow[b] = *(const f32x4*)&mt[2 + NB + b][n16][4 * g4];
      }
      if constexpr (FULL) arow = *(const f32x4*)&mt[1][n16][4 * g4];
      f32x4 kh[TPW], kq[TPW];
#pragma unroll
      for (int a = 0; a < TPW; ++a) kh[a] = kq[a] = zero4();
      if (live)
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
          const Frag h = sm.hx[s][kb][lane];
          Frag q;
          if constexpr (FULL) q = sm.qx[s][kb][lane];
#pragma unroll
          for (int a = 0; a < TPW; ++a) {
            mma(kh[a], h, sk[a][kb]);
            if constexpr (FULL) mma(kq[a], q, sk[a][kb]);
          }
        }
      f32x4 un[TU];
#pragma unroll
      for (int a = 0; a < TU; ++a) {
        un[a] = zero4();
        if (a < TPW) {
          f32x4 rhs;
#pragma unroll
          for (int e = 0; e < 4; ++e) rhs[e] = al[e] * u[s][a < TPW ? a : 0][e] - kco[e] * kh[a < TPW ? a : 0][e];
          mma(un[a], trow, rhs);
        }
      }
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int a = 0; a < TU; ++a) mma(un[a], wrow[b], uo[b][a]);
      if constexpr (FULL) {
#pragma unroll
        for (int a = 0; a < TPW; ++a) {
          const int v = (wave * TPW + a) * 16 + n16;
          f32x4 y = qco * kq[a];
#pragma unroll
          for (int b = 0; b < NB; ++b) mma(y, qrow[b], uo[b][a]);
          mma(y, arow, un[a]);
          CT* yp = (CT*)p.y + tk.y_base + v;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int t = kSC * cc + 4 * g4 + e - t0;
            if (t >= 0 && t < T) yp[(size_t)t * tk.y_tok] = from_f<CT>(y[e]);
          }
          if (p.ts_u) {   // training stash: the sub-chunk's net writes
            float* us = p.ts_u + ((size_t)chain * p.nch + cc) * kSC * D + v;
#pragma unroll
            for (int e = 0; e < 4; ++e) us[(size_t)(4 * g4 + e) * D] = un[a][e];
          }
        }
      }
#pragma unroll
      for (int b = 0; b < NB; ++b)
        if (b == beta)
#pragma unroll
          for (int a = 0; a < TU; ++a)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int i = 4 * g4 + e;
              if (i >= lo && i < hi) uo[b][a][e] = un[a][e];
            }
    }
    gacc += (tot[kBatch] + tot[kBatch + 1]) + (tot[kBatch + 2] + tot[kBatch + 3]);
    lds_barrier();
  }

  if constexpr (!FULL) {
    float* ru = p.run_u + ((size_t)chain * p.nrun + r) * P * D;
    float* rv = p.run_v + ((size_t)chain * p.nrun + r) * P * P;
#pragma unroll
    for (int bl = 0; bl < NB; ++bl)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int i = bl * kSC + 4 * g4 + e;
#pragma unroll
        for (int a = 0; a < TPW; ++a) ru[i * D + (wave * TPW + a) * 16 + n16] = uo[bl][a][e];
        if (wave < NB) rv[i * P + wave * kSC + n16] = uo[bl][TPW][e];
      }
    return;
  } else {
    if (ce < p.c1) return;
    // the interval's last run: the window state (and the call's final state)
#pragma unroll
    for (int bl = 0; bl < NB; ++bl)
#pragma unroll
      for (int a = 0; a < TPW; ++a)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int i = bl * kSC + 4 * g4 + e, v = (wave * TPW + a) * 16 + n16;
          p.uw_out[((size_t)chain * P + i) * D + v] = uo[bl][a][e];
          if (p.last && p.U_out) p.U_out[((size_t)chain * D + v) * P + i] = uo[bl][a][e];
        }
    if (wave == 0) {   // suf[x]: the log decay after token 16 c1 - 128 + x
      const float a = lane_prefix<64>(lgtok(kSC * p.c1 - 128 + lane), lane);
      const float b = lane_prefix<64>(lgtok(kSC * p.c1 - 64 + lane), lane);
      const float ta = lane_value(a, 63), tb = lane_value(b, 63);
      sm.suf[lane] = (ta - a) + tb;
      sm.suf[64 + lane] = tb - b;
    }
    __syncthreads();
    for (int e = tid; e < P * D; e += kNT) {
      const int s = e / D, d = e % D, b = s / kSC;
      int tau = kSC * (p.c1 - 1 - (p.c1 - 1 - b + kBatch * NB) % NB) + s % kSC;   // the slot's last writer
      if (tau >= tend) tau -= P;
      const bool st = tau < tlo;
      float kv = 0.f, off = gacc;
      if (!st) {
        kv = to_f(kin[(size_t)(tau - t0) * tk.qkv_tok + d]);
        off = sm.suf[tau - (kSC * p.c1 - 128)];
      } else if (!p.first) {
        kv = vw[e];
      }
      kv *= expf(off);
      p.vw_out[(size_t)chain * P * D + e] = kv;
      if (p.last && p.Vb_out) p.Vb_out[((size_t)chain * D + d) * P + s] = kv;
    }
    if (tid == 0) p.gsum[chain] = gacc;
    if (p.last && !p.complete) {   // no compaction follows: A, B decayed since the last one
      const int N = p.B * p.H * M;
      const float dk = expf(gacc);
      const float* af = p.ab + (size_t)chain * Ge::R * Ge::m;
      const float* bf = p.ab + (size_t)N * Ge::R * Ge::m + (size_t)chain * Ge::R * Ge::n;
      if (p.A_out)
        for (int e = tid; e < Ge::R * Ge::m; e += kNT) p.A_out[(size_t)chain * Ge::R * Ge::m + e] = af[e] * dk;
      if (p.B_out)
        for (int e = tid; e < Ge::R * Ge::n; e += kNT) p.B_out[(size_t)chain * Ge::R * Ge::n + e] = bf[e] * dk;
    }
  }
}

template <typename CT, int D, int P, int GL>
int launch_runs(const G3FwdArgs& a, int N, hipStream_t stream) {
  static_assert(sizeof(G3RunSmem<CT, D, P>) <= 160 * 1024, "LDS budget");
  if (a.nrun > 1) {
    hipLaunchKernelGGL((gdn3_run_kernel<CT, D, P, GL, false>), dim3(N * (a.nrun - 1)), dim3(kNT), 0, stream, a);
    const int rc = check_launch("gdn3_run_kernel");
    if (rc) return rc;
  }
  hipLaunchKernelGGL((gdn3_run_kernel<CT, D, P, GL, true>), dim3(N * a.nrun), dim3(kNT), 0, stream, a);
  return check_launch("gdn3_run_kernel");
}

template <typename CT, int D, int P>
int launch_runs_gl(const G3FwdArgs& a, int N, hipStream_t stream) {
  return a.gate_ch > 1 ? launch_runs<CT, D, P, 2>(a, N, stream) : launch_runs<CT, D, P, 1>(a, N, stream);
}

template <typename CT>
int launch_runs_shape(const G3FwdArgs& a, int N, hipStream_t stream) {
  if (a.D == 128 && a.P == 16) return launch_runs_gl<CT, 128, 16>(a, N, stream);
  if (a.D == 128 && a.P == 32) return launch_runs_gl<CT, 128, 32>(a, N, stream);
  if (a.D == 128 && a.P == 64) return launch_runs_gl<CT, 128, 64>(a, N, stream);
  if (a.D == 64 && a.P == 16) return launch_runs_gl<CT, 64, 16>(a, N, stream);
  if (a.D == 64 && a.P == 32) return launch_runs_gl<CT, 64, 32>(a, N, stream);
  if (a.D == 64 && a.P == 64) return launch_runs_gl<CT, 64, 64>(a, N, stream);
  return set_error(GDNX_ERR_SHAPE, "gdn3: unsupported head_dim %d / P %d", a.D, a.P);
}

// Runs of an interval: enough workgroups over the chains to occupy the CUs
// (kG3RunTarget), each run at least two batches (a run pays its first pass
// and the fold of the runs before it).
constexpr int kMinRun = 2 * kBatch;
int runs_max(int N) { return N >= kG3RunTarget ? 1 : kG3RunTarget / N; }

}  // namespace

// the other copy of the window state and the runs' maps
size_t gdn3_long_bytes(int N, int D, int P) {
  if (N <= 0 || runs_max(N) == 1) return 0;
  const size_t n = (size_t)N * runs_max(N);
  return 2 * g3_align256((size_t)N * P * D * 4) + g3_align256(n * P * D * 4) + g3_align256(n * P * P * 4);
}

void gdn3_long_carve(G3FwdArgs& a, int N, char* w) {
  if (runs_max(N) == 1) return;
  const size_t n = (size_t)N * runs_max(N), win = g3_align256((size_t)N * a.P * a.D * 4);
  a.uw_alt = (float*)w;
  a.vw_alt = (float*)(w + win);
  a.run_u = (float*)(w + 2 * win);
  a.run_v = (float*)(w + 2 * win + g3_align256(n * a.P * a.D * 4));
}

// One interval [c0, c1) of at least three sub-chunks.  With several runs the
// window state is read from a.uw / a.vw by all of them and left in the other
// copy (a.uw_alt / a.vw_alt), which then takes a.uw / a.vw's place; a single
// run updates it in place.
int gdn3_long_interval(G3FwdArgs& a, int N, hipStream_t stream) {
  const int nsub = a.c1 - a.c0;
  int nrun = runs_max(N);
  if (nrun > nsub / kMinRun) nrun = nsub / kMinRun;
  if (nrun < 1) nrun = 1;
  a.rlen = ((nsub + nrun - 1) / nrun + kBatch - 1) / kBatch * kBatch;
  a.nrun = (nsub + a.rlen - 1) / a.rlen;
  a.uw_out = a.nrun > 1 ? a.uw_alt : a.uw;
  a.vw_out = a.nrun > 1 ? a.vw_alt : a.vw;
  const int rc = a.dtype == GDNX_DTYPE_BF16 ? launch_runs_shape<bf16>(a, N, stream)
                                            : launch_runs_shape<float>(a, N, stream);
  if (a.nrun > 1) {
    std::swap(a.uw, a.uw_alt);
    std::swap(a.vw, a.vw_alt);
  }
  return rc;
}

}  // namespace gdnx
