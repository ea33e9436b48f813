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
// The 16 x 16 x 16 algebra (the inverse, W, T X, W U, Qo U, Aq U) and the decays
// are float32 whatever the IO type: where a sub-chunk's keys are alike (repeated
// tokens) the inverse's factors reach (1 + l)^15, l its largest entry, and cancel.
// As hi + lo bf16 parts (2^-17) those products left 5.5e-4 in U for unit keys of one
// direction and 2.4e-2 for |k| = 2; in float32 8e-6 and 5e-4 (the call below
// took 2.00 ms with the parts).
//
// Bound: issue and latency of two waves per SIMD (the token rows of the next
// batch are loaded under the second half of this one).  B = 1, T = 32768, H =
// 16, 4 lanes, d = 128, bf16, a compaction every 2048 tokens (64 chains, 8
// runs), against the walk of the sub-chunks one by one on 8 workgroups per chain
// that this replaced: the call 5.24 -> 2.14 ms.
#include <type_traits>
#include <utility>

#include "gdn3_common.hpp"
#include "gdnx_internal.hpp"

namespace gdnx {
namespace {

constexpr int kBatch = 4;   // sub-chunks a workgroup prepares at once, one per wave

// Where per-channel write gates go: into u = w o v, kept as float32 rows in
// place of V's, their loads ahead with the rows', unless those rows would
// leave LDS (and registers) for one workgroup a CU where two are wanted: bf16, d = 128, all
// value columns in one workgroup.  There they are read inside the step.
template <typename CT, int D, int NVS>
constexpr bool kGatesAhead = sizeof(CT) == 4 || D == 64 || NVS == 2;

template <typename CT, int D, int P, int GL, int NVS>
struct G3RunSmem {
  static constexpr int NB = P / kSC, KB = D / FragT<CT>::KSTEP;
  static constexpr bool AHEAD = GL == 2 && kGatesAhead<CT, D, NVS>;
  typedef typename FragT<CT>::type Frag;
  typedef typename std::conditional<AHEAD, float, CT>::type VT;
  Frag hx[kBatch][KB][64];                                  // H rows of the batch as A fragments
  Frag qx[kBatch][KB][64];                                  // Q rows
  f32x4 mt[kBatch][2 + 2 * NB][64];                         // T, Aq, -W_b, Qo_b as A operands
  alignas(16) VT vx[kBatch][kSC][D / NVS + (sizeof(VT) == 4 ? 4 : 8)];   // V rows (AHEAD: u), this workgroup's columns
  alignas(16) float aw[kBatch][kSC];                        // alpha w (per-channel gates: alpha)
  alignas(16) float kco[kBatch][kSC], qco[kBatch][kSC];     // alpha e^{2 (Gacc + G)}, e^{2 (Gacc + G)}
  float red[kNT / 64];
  float suf[128];                                           // log decay after a token, to the interval's end
};

// GL: gate layout (1: a scalar per lane, 2: per channel).  FULL: pass 2.
// NVS: workgroups a run's value columns go to (2 while each still has a CU).
template <typename CT, int D, int P, int GL, bool FULL, int NVS>
__global__ void __launch_bounds__(kNT) __attribute__((amdgpu_waves_per_eu(2, 2))) gdn3_run_kernel(G3FwdArgs p) {
  typedef G3RunSmem<CT, D, P, GL, NVS> Sm;
  typedef typename FragT<CT>::type Frag;
  typedef G3D<D> Ge;
  constexpr int NB = Sm::NB, KS = FragT<CT>::KSTEP, KB = Sm::KB, EPL = KS / 4;   // elements a lane holds of a k-step
  constexpr int DV = D / NVS, TPW = DV / 64, VK = KB / NVS;   // value columns, tiles per wave, k-steps of a V row
  constexpr bool AHEAD = Sm::AHEAD;
  static_assert(TPW >= 1 && VK * KS == DV, "whole tiles and k-steps");
  static_assert(sizeof(Frag) == 16 && EPL * sizeof(CT) == 16, "a fragment is one 16-byte load");
  static_assert(NB >= 1 && NB <= kBatch && D % 64 == 0, "the decay window holds the last four sub-chunks");
  __shared__ Sm sm;

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g4 = lane >> 4, n16 = lane & 15;
  const int T = p.T, t0 = p.t0, M = p.M;
  const int nr = FULL ? p.nrun : p.nrun - 1;
  // the lanes of a head's run, which share q, k and v, are neighbours on an XCD
  const int bw = xcd_remap(blockIdx.x, p.B * p.H * M * nr * NVS);
  const int vs = bw % NVS, work = bw / NVS, vt0 = (DV / 16) * vs;   // value tiles vt0 + [0, DV / 16)
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

  // A wave's loads for its sub-chunk of a batch: lane (g4, n16) takes 16 bytes
  // of row n16 per k-step (rows outside the call read an end row and are
  // zeroed where they are used), each row at a 32-bit offset from a uniform base
  struct Rows {
    Frag k[KB], q[KB], v[VK], pk[NB == 1 ? KB : 1];
    f32x4 bg[AHEAD ? D / 16 : 1], wg[AHEAD ? DV / 16 : 1];   // per-channel gates
    float d, dp[NB], b, w;
  };
  auto load_steps = [&](const CT* base, int tr, Frag* dst, auto steps) {
    const int tb = min(max(tr, 0), T - 1);
    const unsigned off = (unsigned)((min(max(tr + n16, 0), T - 1) - tb) * (int)tk.qkv_tok + g4 * EPL);
    const CT* src = base + (size_t)tb * tk.qkv_tok;
#pragma unroll
    for (int kb = 0; kb < steps(); ++kb) dst[kb] = *(const Frag*)(src + off + kb * KS);
  };
  auto load_rows = [&](const CT* base, int tr, Frag* dst) {
    load_steps(base, tr, dst, std::integral_constant<int, KB>());
  };
  auto dec_at = [&](int tau) {
    return p.dec[tk.dec_base + (size_t)min(max(tau - t0, 0), T - 1) * tk.dec_tok];
  };
  auto fetch = [&](Rows& x, int cb) {
    const int tr = kSC * (cb + wave) - t0;
    load_rows(kin, tr, x.k);
    if constexpr (FULL) load_rows(qin, tr, x.q);
    load_steps(vin + DV * vs, tr, x.v, std::integral_constant<int, VK>());
    if constexpr (NB == 1) load_rows(kin, tr - kSC, x.pk);
    if constexpr (AHEAD) {
      const size_t go = tk.gate_base + (size_t)min(max(tr + n16, 0), T - 1) * tk.gate_tok + g4 * EPL;
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int e = 0; e < EPL; e += 4) x.bg[(kb * EPL + e) / 4] = *(const f32x4*)(p.bg + go + kb * KS + e);
#pragma unroll
      for (int kb = 0; kb < VK; ++kb)
#pragma unroll
        for (int e = 0; e < EPL; e += 4) x.wg[(kb * EPL + e) / 4] = *(const f32x4*)(p.wg + go + DV * vs + kb * KS + e);
    }
    x.d = dec_at(kSC * cb + lane);
#pragma unroll
    for (int z = 0; z < NB; ++z) x.dp[z] = dec_at(kSC * (cb + wave - 1 - z) + n16);
    if constexpr (GL == 1) {
      const size_t go = tk.gate_base + (size_t)min(max(tr + n16, 0), T - 1) * tk.gate_tok;
      x.b = p.bg[go];
      x.w = p.wg[go];
    }
  };
  auto log_at = [&](float d, int tau) { return tau >= tlo && tau < tint ? log_decay(d) : 0.f; };

  // bf16 rows of the next batch are loaded before the second half of a batch
  // (float32 rows would take twice the registers), the first batch's ahead of
  // everything else: loads retire in order
  constexpr bool PRE = sizeof(CT) == 2;
  Rows x;
  if constexpr (PRE) fetch(x, cs);
  // this wave's value rows of the Kronecker matrix
  Frag sk[TPW][KB];
  if (live)
#pragma unroll
    for (int a = 0; a < TPW; ++a)
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
        sk[a][kb] = *(const Frag*)((const CT*)p.skron + ((size_t)chain * D + (vt0 + wave * TPW + a) * 16 + n16) * D + kb * KS +
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
        for (int e = 0; e < 4; ++e) uo[bl][a][e] = uw[(bl * kSC + 4 * g4 + e) * D + (vt0 + wave * TPW + a) * 16 + n16];
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
        const float* ru = p.run_u + ((size_t)chain * (p.nrun - 1) + x) * P * D;
        const float* rv = p.run_v + ((size_t)chain * (p.nrun - 1) + x) * P * P;
        f32x4 nu[NB][TPW];
#pragma unroll
        for (int bl = 0; bl < NB; ++bl) {
          f32x4 va[NB];
#pragma unroll
          for (int b2 = 0; b2 < NB; ++b2) va[b2] = *(const f32x4*)&rv[(bl * kSC + n16) * P + b2 * kSC + 4 * g4];
#pragma unroll
          for (int a = 0; a < TPW; ++a)
#pragma unroll
            for (int e = 0; e < 4; ++e) nu[bl][a][e] = ru[(bl * kSC + 4 * g4 + e) * D + (vt0 + wave * TPW + a) * 16 + n16];
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

  if (FULL && ce == p.c1 && wave == 3) {   // suf[x]: the log decay after token 16 c1 - 128 + x
    const float a = lane_prefix<64>(lgtok(kSC * p.c1 - 128 + lane), lane);
    const float b = lane_prefix<64>(lgtok(kSC * p.c1 - 64 + lane), lane);
    const float ta = lane_value(a, 63), tb = lane_value(b, 63);
    sm.suf[lane] = (ta - a) + tb;
    sm.suf[64 + lane] = tb - b;
  }
  for (int cb = cs; cb < ce; cb += kBatch) {
    if constexpr (!PRE) fetch(x, cb);
    // log-decay prefixes of the batch (16-lane row z: sub-chunk cb + z)
    const float G1 = row_prefix16(log_at(x.d, kSC * cb + lane));
    const int c = cb + wave;
    if (c < ce) {
      const int tr = kSC * c - t0, lo = max(0, -tr);
      if (tr < 0 || tr + kSC > T) {   // (uniform) rows outside the call are zero
        const bool ok = tr + n16 >= 0 && tr + n16 < T;
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
#pragma unroll
          for (int e = 0; e < EPL; ++e) {
            x.k[kb][e] = ok ? x.k[kb][e] : from_f<CT>(0.f);
            if (kb < VK) x.v[kb < VK ? kb : 0][e] = ok ? x.v[kb < VK ? kb : 0][e] : from_f<CT>(0.f);
            if constexpr (FULL) x.q[kb][e] = ok ? x.q[kb][e] : from_f<CT>(0.f);
          }
      }
      Frag hf[KB];
      float part = 0.f;
      {
        const float* bp = GL == 2 ? p.bg + tk.gate_base + (size_t)min(max(tr + n16, 0), T - 1) * tk.gate_tok + g4 * EPL
                                  : nullptr;
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
          float bb[EPL];
#pragma unroll
          for (int e = 0; e < EPL; e += 4) {
            f32x4 b4 = {x.b, x.b, x.b, x.b};
            if constexpr (AHEAD) b4 = x.bg[(kb * EPL + e) / 4];
            else if constexpr (GL == 2) b4 = *(const f32x4*)(bp + kb * KS + e);
#pragma unroll
            for (int i = 0; i < 4; ++i) bb[e + i] = b4[i];
          }
#pragma unroll
          for (int e = 0; e < EPL; ++e) {
            const float kv = to_f(x.k[kb][e]), h = bb[e] * kv;
            part += kv * h;
            hf[kb][e] = from_f<CT>(h);
          }
          sm.hx[wave][kb][lane] = hf[kb];
          if constexpr (FULL) sm.qx[wave][kb][lane] = x.q[kb];
          if (kb < VK) {
            const Frag vr = x.v[kb < VK ? kb : 0];
            typename Sm::VT* dst = &sm.vx[wave][n16][kb * KS + g4 * EPL];
            if constexpr (AHEAD) {
#pragma unroll
              for (int e = 0; e < EPL; e += 4) {
                f32x4 u;
#pragma unroll
                for (int i = 0; i < 4; ++i) u[i] = x.wg[kb < VK ? (kb * EPL + e) / 4 : 0][i] * to_f(vr[e + i]);
                *(f32x4*)(dst + e) = u;
              }
            } else {
              *(Frag*)dst = vr;
            }
          }
        }
      }
      const float alpha_l = stable_alpha_f(sum_rows4(part));   // of token n16
      const float gl = __shfl(G1, kSC * wave + n16, 64);       // G of token n16
      float gw = gacc;   // the log decay since the last compaction at the sub-chunk's start
#pragma unroll
      for (int z = 0; z < kBatch - 1; ++z) gw += z < wave ? lane_value(G1, kSC * z + kSC - 1) : 0.f;
      if (lane < kSC) {
        const float e2 = expf(2.f * (gw + gl));
        sm.aw[wave][lane] = GL == 1 ? alpha_l * x.w : alpha_l;
        sm.kco[wave][lane] = alpha_l * e2;
        sm.qco[wave][lane] = e2;
      }
      if (FULL && p.ts_g && lane == 0 && vs == 0) p.ts_g[(size_t)chain * p.nch + c] = gw;
      // The 16 x 16 matrices.  A product's accumulator tile (row 4 g + e,
      // column n16) is a B operand as it is, and the A operand of its transpose;
      // so a matrix that is wanted as an A operand is formed transposed, by
      // exchanging the factors, and nothing goes through LDS in between.
      // T = (I + L)^-1, L[i][j] = alpha_i e^{G_i - G_j} (h_i . k_j), j < i, is
      // nilpotent: T = (I - L)(I + L^2)(I + L^4)(I + L^8), factors that commute
      f32x4 xa = zero4(), xt = zero4(), aq = zero4();
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        mma(xa, hf[kb], x.k[kb]);
        mma(xt, x.k[kb], hf[kb]);
        if constexpr (FULL) mma(aq, x.k[kb], x.q[kb]);
      }
      f32x4 gi, ai, tt;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int i = 4 * g4 + e;
        gi[e] = __shfl(gl, i, 64);
        ai[e] = __shfl(alpha_l, i, 64);
        xa[e] = n16 < i ? ai[e] * expf(gi[e] - gl) * xa[e] : 0.f;
        const float dn = n16 >= i ? expf(gl - gi[e]) : 0.f;   // (row j = i here, column the later token)
        xt[e] = n16 > i ? alpha_l * dn * xt[e] : 0.f;
        if constexpr (FULL) aq[e] *= dn;
        tt[e] = (i == n16 ? 1.f : 0.f) - xt[e];                  // T^T, first factor
      }
      if constexpr (FULL) sm.mt[wave][1][lane] = aq;      // Aq = [j <= i] e^{G_i - G_j} q_i.k_j
#pragma unroll
      for (int step = 0; step < 3; ++step) {
        f32x4 s2 = zero4(), s2t = zero4();
        mma(s2, xt, xa);                                         // X^2
        if (step < 2) mma(s2t, xa, xt);                          // (X^2)^T
        mma(tt, s2, tt);                                         // T^T += (X^2)^T T^T
        xa = s2;
        xt = s2t;
      }
      sm.mt[wave][0][lane] = tt;
      // the window's blocks: the one that sub-chunk c - z wrote last (z = 1 ..
      // NB; c itself writes the last of them), its slot j holding the key of
      // that sub-chunk's token j, or the carried state's key where that token
      // came before this call, decayed from there to c's start
      //   Ho_b = vis alpha_i e^{G_i + off_j} h_i.k_j,  Qo_b = vis e^{G_i + off_j} q_i.k_j,
      // vis: not yet overwritten by sub-chunk c; W_b = T Ho_b
      const float el = expf(gl);
      f32x4 ei;
#pragma unroll
      for (int e = 0; e < 4; ++e) ei[e] = __shfl(el, 4 * g4 + e, 64);
      float after = 0.f, all = 0.f;   // log decay from the end of sub-chunk c - z, from the interval's start
#pragma unroll
      for (int z = 1; z <= NB; ++z) {
        const int b = (c - z + kBatch * NB) % NB, t1 = kSC * (c - z);
        const float gp = row_prefix16(t1 + n16 >= t0 ? log_at(x.dp[z - 1], max(t1 + n16, tlo)) : 0.f), total = lane_value(gp, kSC - 1);
        Frag pf[KB];
        if constexpr (NB == 1) {
#pragma unroll
          for (int kb = 0; kb < KB; ++kb) pf[kb] = x.pk[kb];
        } else {
          load_rows(kin, tr - kSC * z, pf);
        }
        float off = (total - gp) + after;
        if (c - z >= p.c0) all += total;
        if (t1 < t0) {   // (uniform) keys of the carried state, as it stands at the interval's start
          const bool st = t1 + n16 < t0;
#pragma unroll
          for (int kb = 0; kb < KB; ++kb)
#pragma unroll
            for (int e = 0; e < EPL; e += 4) {
              const f32x4 sv = p.first ? zero4() : *(const f32x4*)&vw[(kSC * b + n16) * D + kb * KS + g4 * EPL + e];
#pragma unroll
              for (int i = 0; i < 4; ++i) pf[kb][e + i] = st ? from_f<CT>(sv[i]) : pf[kb][e + i];
            }
          if (st) off = all;
        }
        after += total;
        f32x4 ho = zero4(), qt = zero4();
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
          mma(ho, hf[kb], pf[kb]);
          if constexpr (FULL) mma(qt, pf[kb], x.q[kb]);
        }
        const float eo = expf(off);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int i = 4 * g4 + e;
          const bool vis = z != NB || n16 >= i || n16 < lo;       // token i, slot n16
          ho[e] *= vis ? ai[e] * (ei[e] * eo) : 0.f;
          const bool vist = z != NB || i >= n16 || i < lo;        // token n16, slot i
          const float eoi = __shfl(eo, i, 64);   // (every lane takes part)
          if constexpr (FULL) qt[e] *= vist ? el * eoi : 0.f;
        }
        f32x4 wt = zero4();
        mma(wt, ho, tt);                                         // W_b^T = Ho_b^T T^T
        sm.mt[wave][2 + b][lane] = -wt;
        if constexpr (FULL) sm.mt[wave][2 + NB + b][lane] = qt;
      }
    }
    lds_barrier();
    if constexpr (PRE)
      if (cb + kBatch < ce) fetch(x, cb + kBatch);
#pragma unroll 1
    for (int s = 0; s < kBatch && cb + s < ce; ++s) {
      const int cc = cb + s, beta = cc % NB, tr = kSC * cc - t0;
      const bool whole = tr >= 0 && tr + kSC <= T;   // (uniform) every token is of this call
      const f32x4 aw = *(const f32x4*)&sm.aw[s][4 * g4], kco = *(const f32x4*)&sm.kco[s][4 * g4];
      const f32x4 qco = *(const f32x4*)&sm.qco[s][4 * g4];
      const f32x4 trow = sm.mt[s][0][lane];
      f32x4 wrow[NB], qrow[NB], arow;
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        wrow[b] = sm.mt[s][2 + b][lane];
        if constexpr (FULL) qrow[b] = sm.mt[s][2 + NB + b][lane];
      }
      if constexpr (FULL) arow = sm.mt[s][1][lane];
      f32x4 rhs[TPW];
#pragma unroll
      for (int a = 0; a < TPW; ++a)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int v = (wave * TPW + a) * 16 + n16;   // of this workgroup's columns
          float wv = 1.f;
          if constexpr (GL == 2 && !AHEAD)
            wv = p.wg[tk.gate_base + (size_t)min(max(tr + 4 * g4 + e, 0), T - 1) * tk.gate_tok + vt0 * 16 + v];
          rhs[a][e] = aw[e] * (wv * to_f(sm.vx[s][4 * g4 + e][v]));
        }
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
        if (a < TPW) mma(un[a], trow, rhs[a < TPW ? a : 0] - kco * kh[a < TPW ? a : 0]);
      }
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int a = 0; a < TU; ++a) mma(un[a], wrow[b], uo[b][a]);
      if constexpr (FULL) {
        f32x4 y[TPW];
#pragma unroll
        for (int a = 0; a < TPW; ++a) {
          y[a] = qco * kq[a];
#pragma unroll
          for (int b = 0; b < NB; ++b) mma(y[a], qrow[b], uo[b][a]);
          mma(y[a], arow, un[a]);
        }
        CT* yp = (CT*)p.y + tk.y_base + (ptrdiff_t)tr * (ptrdiff_t)tk.y_tok;
        const unsigned yo = (unsigned)(4 * g4 * (int)tk.y_tok + (vt0 + wave * TPW) * 16 + n16);
        if (whole) {
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int a = 0; a < TPW; ++a) (yp + e * tk.y_tok)[yo + a * 16] = from_f<CT>(y[a][e]);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int t = tr + 4 * g4 + e;
            if (t >= 0 && t < T)
#pragma unroll
              for (int a = 0; a < TPW; ++a) (yp + e * tk.y_tok)[yo + a * 16] = from_f<CT>(y[a][e]);
          }
        }
        if (p.ts_u) {   // training stash: the sub-chunk's net writes
          float* us = p.ts_u + ((size_t)chain * p.nch + cc) * kSC * D + (vt0 + wave * TPW) * 16 + n16;
#pragma unroll
          for (int a = 0; a < TPW; ++a)
#pragma unroll
            for (int e = 0; e < 4; ++e) us[(4 * g4 + e) * D + a * 16] = un[a][e];
        }
      }
      // the block sub-chunk cc writes (tokens outside the call leave its slots)
#pragma unroll
      for (int b = 0; b < NB; ++b)
        if (b == beta) {
          if (whole) {
#pragma unroll
            for (int a = 0; a < TU; ++a) uo[b][a] = un[a];
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int t = tr + 4 * g4 + e;
              if (t >= 0 && t < T)
#pragma unroll
                for (int a = 0; a < TU; ++a) uo[b][a][e] = un[a][e];
            }
          }
        }
    }
    gacc += (lane_value(G1, 15) + lane_value(G1, 31)) + (lane_value(G1, 47) + lane_value(G1, 63));
    lds_barrier();
  }

  if constexpr (!FULL) {
    float* ru = p.run_u + ((size_t)chain * (p.nrun - 1) + r) * P * D;
    float* rv = p.run_v + ((size_t)chain * (p.nrun - 1) + r) * P * P;
#pragma unroll
    for (int bl = 0; bl < NB; ++bl)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int i = bl * kSC + 4 * g4 + e;
#pragma unroll
        for (int a = 0; a < TPW; ++a) ru[i * D + (vt0 + wave * TPW + a) * 16 + n16] = uo[bl][a][e];
        if (wave < NB && vs == 0) rv[i * P + wave * kSC + n16] = uo[bl][TPW][e];
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
          const int i = bl * kSC + 4 * g4 + e, v = (vt0 + wave * TPW + a) * 16 + n16;
          p.uw_out[((size_t)chain * P + i) * D + v] = uo[bl][a][e];
          if (p.last && p.U_out) p.U_out[((size_t)chain * D + v) * P + i] = uo[bl][a][e];
        }
    if (vs > 0) return;   // (what follows is the chain's, not the columns')
    for (int e = tid; e < P * D / EPL; e += kNT) {   // 16 bytes of a slot's key
      const int s = e / (D / EPL), d = EPL * (e % (D / EPL)), b = s / kSC;
      int tau = kSC * (p.c1 - 1 - (p.c1 - 1 - b + kBatch * NB) % NB) + s % kSC;   // the slot's last writer
      if (tau >= tend) tau -= P;
      const bool st = tau < tlo;
      float kv[EPL];
      const Frag kr = *(const Frag*)(kin + (size_t)min(max(tau - t0, 0), T - 1) * tk.qkv_tok + d);
      const float sc = expf(st ? gacc : sm.suf[tau - (kSC * p.c1 - 128)]);
#pragma unroll
      for (int i = 0; i < EPL; ++i) kv[i] = to_f(kr[i]);
      if (st)
#pragma unroll
        for (int i = 0; i < EPL; i += 4) {
          const f32x4 o = p.first ? zero4() : *(const f32x4*)&vw[s * D + d + i];
#pragma unroll
          for (int j = 0; j < 4; ++j) kv[i + j] = o[j];
        }
#pragma unroll
      for (int i = 0; i < EPL; i += 4)
        *(f32x4*)&p.vw_out[((size_t)chain * P + s) * D + d + i] =
            (f32x4){kv[i] * sc, kv[i + 1] * sc, kv[i + 2] * sc, kv[i + 3] * sc};
      if (p.last && p.Vb_out)
#pragma unroll
        for (int i = 0; i < EPL; ++i) p.Vb_out[((size_t)chain * D + d + i) * P + s] = kv[i] * sc;
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

template <typename CT, int D, int P, int GL, int NVS>
int launch_passes(const G3FwdArgs& a, int N, hipStream_t stream) {
  static_assert(sizeof(G3RunSmem<CT, D, P, GL, NVS>) <= 160 * 1024, "LDS budget");
  if (a.nrun > 1) {
    hipLaunchKernelGGL((gdn3_run_kernel<CT, D, P, GL, false, NVS>), dim3(N * (a.nrun - 1) * NVS), dim3(kNT), 0, stream, a);
    const int rc = check_launch("gdn3_run_kernel");
    if (rc) return rc;
  }
  hipLaunchKernelGGL((gdn3_run_kernel<CT, D, P, GL, true, NVS>), dim3(N * a.nrun * NVS), dim3(kNT), 0, stream, a);
  return check_launch("gdn3_run_kernel");
}

// Runs of an interval of nsub sub-chunks: as many as the workgroups that run
// at once (slots: two a CU, or one where LDS holds one) leave to a chain, each at
// least a batch, and not so many that folding their maps takes longer than the two
// scans of a run: a fold takes ~0.6 us a block of 16 slots squared, a batch 5
// (bf16) to 9 us, so that sqrt(16 batches / blocks) is about the least sum.
// Under four batches a single run: the second pass would cost what shorter
// runs save.  T = 4096, d = 128, runs of at least two batches up to 512
// workgroups | so | the walk on 8 workgroups: 64 chains, a compaction every 256
// tokens, bf16 967 | 842 | 1112 us, float32 1351 | 1156 | 1629; 16 chains, float32,
// every 320: 1300 | 762 | 1124; P = 64, 64 chains, bf16, every 1024 (one workgroup a
// CU): 847 | 688 | 1141; two chains, T = 32768, none: 1471 | 396 | 6676.
int interval_runs(int nsub, int N, int slots, int blocks) {
  const int nb = (nsub + kBatch - 1) / kBatch;
  if (nb < 4 || N >= slots) return 1;
  int n = slots / N < nb ? slots / N : nb;
  while (n > 1 && (long long)n * n * blocks > 16LL * nb) --n;
  return n;
}

// One interval [c0, c1).  With several workgroups a chain the window state is
// read from a.uw / a.vw by all of them and left in the other copy (a.uw_alt /
// a.vw_alt), which then takes a.uw / a.vw's place; a single one updates it in
// place.
template <typename CT, int D, int P, int GL>
int launch_runs(G3FwdArgs& a, int N, hipStream_t stream) {
  constexpr int slots = sizeof(G3RunSmem<CT, D, P, GL, 1>) * 2 <= 160 * 1024 ? kG3RunTarget : kG3RunTarget / 2;
  const int nsub = a.c1 - a.c0;
  a.nrun = interval_runs(nsub, N, slots, P / kSC);
  a.rlen = ((nsub + a.nrun - 1) / a.nrun + kBatch - 1) / kBatch * kBatch;
  a.nrun = (nsub + a.rlen - 1) / a.rlen;
  // The value columns of a run on two workgroups while each has a CU of its
  // own.  64 chains, T = 4096, d = 128, a compaction every 64 tokens, one workgroup
  // | two (with per-channel gates ahead) | the walk on 8: bf16 2.55 | 2.44 | 2.71
  // ms, per-channel gates 2.79 | 2.57 | 2.79, float32 3.32 | 2.95 | 3.19, with them
  // 3.54 | 3.06 | 3.27.
  const bool split = D == 128 && N * a.nrun <= kG3RunTarget / 4;
  const bool alt = a.nrun > 1 || split;
  a.uw_out = alt ? a.uw_alt : a.uw;
  a.vw_out = alt ? a.vw_alt : a.vw;
  int rc;
  if constexpr (D == 128)
    rc = split ? launch_passes<CT, D, P, GL, 2>(a, N, stream) : launch_passes<CT, D, P, GL, 1>(a, N, stream);
  else
    rc = launch_passes<CT, D, P, GL, 1>(a, N, stream);
  if (alt) {
    std::swap(a.uw, a.uw_alt);
    std::swap(a.vw, a.vw_alt);
  }
  return rc;
}

template <typename CT, int D, int P>
int launch_runs_gl(G3FwdArgs& a, int N, hipStream_t stream) {
  return a.gate_ch > 1 ? launch_runs<CT, D, P, 2>(a, N, stream) : launch_runs<CT, D, P, 1>(a, N, stream);
}

template <typename CT>
int launch_runs_shape(G3FwdArgs& a, int N, hipStream_t stream) {
  if (a.D == 128 && a.P == 16) return launch_runs_gl<CT, 128, 16>(a, N, stream);
  if (a.D == 128 && a.P == 32) return launch_runs_gl<CT, 128, 32>(a, N, stream);
  if (a.D == 128 && a.P == 64) return launch_runs_gl<CT, 128, 64>(a, N, stream);
  if (a.D == 64 && a.P == 16) return launch_runs_gl<CT, 64, 16>(a, N, stream);
  if (a.D == 64 && a.P == 32) return launch_runs_gl<CT, 64, 32>(a, N, stream);
  if (a.D == 64 && a.P == 64) return launch_runs_gl<CT, 64, 64>(a, N, stream);
  return set_error(GDNX_ERR_SHAPE, "gdn3: unsupported head_dim %d / P %d", a.D, a.P);
}

// the runs that any interval of N chains may be cut into
int runs_max(int N) { return N >= kG3RunTarget ? 1 : kG3RunTarget / N; }

}  // namespace

// the other copy of the window state and the maps of all runs but the last.
// At most 256 chains have any: with their states that is 61.3 MiB at d = 128,
// P = 64, float32, so that the workspace fits the static scratch exactly where
// the states do.
size_t gdn3_long_bytes(int N, int D, int P) {
  if (N <= 0 || runs_max(N) == 1) return 0;
  const size_t n = (size_t)N * (runs_max(N) - 1);
  return 2 * g3_align256((size_t)N * P * D * 4) + g3_align256(n * P * D * 4) + g3_align256(n * P * P * 4);
}

void gdn3_long_carve(G3FwdArgs& a, int N, char* w) {
  if (runs_max(N) == 1) return;
  const size_t n = (size_t)N * (runs_max(N) - 1), win = g3_align256((size_t)N * a.P * a.D * 4);
  a.uw_alt = (float*)w;
  a.vw_alt = (float*)(w + win);
  a.run_u = (float*)(w + 2 * win);
  a.run_v = (float*)(w + 2 * win + g3_align256(n * a.P * a.D * 4));
}

int gdn3_long_interval(G3FwdArgs& a, int N, hipStream_t stream) {
  return a.dtype == GDNX_DTYPE_BF16 ? launch_runs_shape<bf16>(a, N, stream) : launch_runs_shape<float>(a, N, stream);
}

}  // namespace gdnx
