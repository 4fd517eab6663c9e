// fp32 path of the recurrent forward (any shape, decay, shared or per-head
// values).  It evaluates the same closed form as the reference's dense-score
// executor (linear.rs:221-400) over state-carry intervals of L tokens:
//   S      = tril(-1)(Q Q^T * d^(r-c))                       [gram]
//   ctx    = S V + (Q * d^r) rho                              [context]
//   rho'   = rho * d^L + (Q * d^(L-r))^T V                     [state]
// with r, c token offsets inside the interval.  Each product is a batched
// fp32 GEMM on the matrix cores (bdh_gemm_f32.h), the masks and decay powers
// in its epilogue or operand loads, and one launch of it covers every
// interval: only the state runs through the intervals in order, and it does
// so inside its launch (a workgroup carries its block of rho over all tokens
// and writes it at each interval's start).  Four products whatever the length:
//   gram     A = B = Q (rows t, k over N), epilogue tril(-1) * d^(r-c)
//   context  A = S (k limited to the causal part of the row block), B = V
//   state    A = Q^T (rows n, k over t, loaded d^(L-t)-scaled), B = V,
//            epilogue acc + rho * d^L (in place when rho_out is rho)
//   readout  A = Q, B = rho at the interval's start, epilogue += acc * d^r
#include <algorithm>

#include "bdh_gemm_f32.h"

namespace bdh {

using namespace gf32;

namespace {

// Most scratch for scores and states between intervals: longer sequences run
// as groups of intervals, each group as above.  (B8 nh4 T4096 N8192 D256: 5
// intervals a group, 1.1 GB of states.)
constexpr int64_t kScoresMax = (int64_t)256 << 20;  // bytes
constexpr int64_t kStatesMax = (int64_t)1 << 30;
// Interval a call falls back to where memory is short.
constexpr int64_t kShortInterval = 256;

struct Intervals {
  int64_t L, n, group;  // tokens of an interval, intervals, intervals of a group
};

// Intervals of at most 512 tokens, of equal length (a multiple of 128) but
// the last: gram work grows with the length, a state write and readout with
// the count.  The f32 C2 shape (T = 512): one interval 1.06 ms, two of 256
// 1.37 ms (then 1.15 in one).
Intervals intervals(const F32Args& a) {
  const int64_t S = a.B * a.H;
  Intervals v;
  if (!a.state) {
    v.L = a.T;
    v.n = v.group = 1;
    return v;
  }
  v.n = (a.T + a.max_len - 1) / a.max_len;
  v.L = v.n == 1 ? a.T : ((a.T + v.n - 1) / v.n + 127) / 128 * 128;
  v.n = (a.T + v.L - 1) / v.L;
  int64_t g = kScoresMax / (S * v.L * v.L * 4);
  g = std::min(g, kStatesMax / (S * a.N * a.D * 4) + 1);
  g = std::min({g, kMaxBatch / S, a.max_group});
  v.group = std::max<int64_t>(1, std::min(g, v.n));
  return v;
}

struct Scratch {
  size_t scores, states, part;  // floats of F32Args' buffers
};

Scratch scratch_of(const F32Args& a) {
  const int64_t S = a.B * a.H;
  const Intervals v = intervals(a);
  Scratch w;
  w.scores = (size_t)(v.group * S * v.L * v.L);
  w.states = (size_t)((v.group - 1) * S * a.N * a.D);
  // Split-K partials: the gram and readout (K = N) and S V (K = L), of the
  // whole groups, the last one and a group's first interval.
  w.part = 0;
  for (const int64_t n : {v.group, v.n % v.group, (int64_t)1}) {
    if (n == 0) continue;
    const int L = (int)v.L;
    for (const size_t p : {split_k_elems(n * S, L, L, (int)a.N), split_k_elems(n * S, L, (int)a.D, (int)a.N),
                           split_k_elems(n * S, L, (int)a.D, L)})
      w.part = std::max(w.part, p);
  }
  return w;
}

}  // namespace

bdh_status f32_path_buffers(F32Args* a, hipStream_t st) {
  for (;;) {
    const Scratch need = scratch_of(*a);
    void *scores = nullptr, *states = nullptr, *part = nullptr;
    bdh_status s = scratch(st, SLOT_SCORES, need.scores * sizeof(float), &scores);
    if (s == BDH_OK && need.states) s = scratch(st, SLOT_SNAP, need.states * sizeof(float), &states);
    a->part_elems = need.part;
    if (s == BDH_OK && need.part) {
      s = scratch(st, SLOT_GEMM_PART, need.part * sizeof(float), &part);
      if (s == BDH_UNSUPPORTED) {  // capturing: fewer split-K ranges in what is there
        a->part_elems = std::min(need.part, scratch_held(st, SLOT_GEMM_PART, &part) / sizeof(float));
        s = BDH_OK;
      }
    }
    a->scores = (float*)scores;
    a->states = (float*)states;
    a->part = (float*)part;
    const bool short_of_memory = scratch_no_memory();
    if (s == BDH_OK || (s != BDH_UNSUPPORTED && !short_of_memory)) return s;
    const Intervals v = intervals(*a);
    if (v.group > 1) {
      a->max_group = v.group / 2;
    } else if (a->state && v.L > kShortInterval) {
      a->max_len = kShortInterval;
      a->max_group = 1;
    } else if (scores && (states || !need.states)) {  // no room for partials alone: unsplit
      a->part = nullptr;
      a->part_elems = 0;
      return BDH_OK;
    } else {
      return s;
    }
    if (short_of_memory) s = scratch_drop(st, {SLOT_SCORES, SLOT_SNAP, SLOT_GEMM_PART});
    if (short_of_memory && s != BDH_OK) return s;
  }
}

hipError_t run_f32_path(const F32Args& a, hipStream_t st, uint64_t* launches) {
  const int64_t S = a.B * a.H, H = a.H, T = a.T, N = a.N, D = a.D;
  const Intervals v = intervals(a);
  const size_t pe = a.part_elems;
  const int64_t L = v.L, sVo = a.Hv * T * D, sVi = a.Hv == 1 ? 0 : T * D;
  const float* rho_cur = a.rho_in;
  uint64_t n = 0;
  for (int64_t i0 = 0; i0 < v.n; i0 += v.group) {
    const int64_t ni = std::min(v.group, v.n - i0), t0 = i0 * L, len = std::min(ni * L, T - t0);
    const int64_t L0 = std::min(L, len), L1 = len - (ni - 1) * L;  // first and last interval
    const float* q = a.q + t0 * N;
    const float* val = a.v + t0 * D;
    float* ctx = a.ctx + t0 * D;
    GemmF32 base{};
    base.H = (int)H;
    base.decay = a.decay;
    base.niv = (int)ni;
    // S = tril(-1)(Q Q^T) * d^(r-c)  ->  scores [ni, S, L, L]
    GemmF32 g = base;
    g.A = g.B = q; g.sAo = g.sBo = H * T * N; g.sAi = g.sBi = T * N; g.sAm = g.sBn = N; g.sAk = g.sBk = 1;
    g.sA3 = g.sB3 = L * N;
    g.C = a.scores; g.sCo = H * L * L; g.sCi = L * L; g.sCm = L; g.sCn = 1; g.sC3 = S * L * L;
    g.M = g.N = (int)L0; g.K = g.K1 = (int)N;
    g.M1 = g.N1 = (int)L1;
    hipError_t e = gemm<E_TRIL_DECAY>(g, S, st, a.part, pe, &n);
    if (e != hipSuccess) return e;
    // ctx = S V
    g = base;
    g.A = a.scores; g.sAo = H * L * L; g.sAi = L * L; g.sAm = L; g.sAk = 1; g.sA3 = S * L * L;
    g.B = val; g.sBo = sVo; g.sBi = sVi; g.sBn = 1; g.sBk = D; g.sB3 = L * D;
    g.C = ctx; g.sCo = H * T * D; g.sCi = T * D; g.sCm = D; g.sCn = 1; g.sC3 = L * D;
    g.M = g.K = (int)L0; g.M1 = g.K1 = (int)L1; g.N = g.N1 = (int)D;
    g.kcausal = 1;
    e = gemm<E_STORE>(g, S, st, a.part, pe, &n);
    if (e != hipSuccess) return e;
    // ctx += (Q * d^r) rho
    GemmF32 r = base;
    r.A = q; r.sAo = H * T * N; r.sAi = T * N; r.sAm = N; r.sAk = 1; r.sA3 = L * N;
    r.sBo = H * N * D; r.sBi = N * D; r.sBn = 1; r.sBk = D; r.sB3 = S * N * D;
    r.C = ctx; r.sCo = H * T * D; r.sCi = T * D; r.sCm = D; r.sCn = 1; r.sC3 = L * D;
    r.M = (int)L0; r.M1 = (int)L1; r.N = r.N1 = (int)D; r.K = r.K1 = (int)N;
    if (rho_cur) {  // the first interval's, before rho_out may replace it
      g = r;
      g.niv = 1;
      g.B = rho_cur;
      e = gemm<E_ROWSCALE_ACC>(g, S, st, a.part, pe, &n);
      if (e != hipSuccess) return e;
    }
    if (!a.state) break;
    // rho' = rho * d^len + (Q * d^(len-t))^T V, rho at the later intervals' starts to states
    g = base;
    g.niv = 1;
    g.A = q; g.sAo = H * T * N; g.sAi = T * N; g.sAm = 1; g.sAk = N;
    g.B = val; g.sBo = sVo; g.sBi = sVi; g.sBn = 1; g.sBk = D;
    g.C = a.rho_out; g.sCo = H * N * D; g.sCi = N * D; g.sCm = D; g.sCn = 1;
    g.src = rho_cur;
    g.M = (int)N; g.N = (int)D; g.K = g.kpow = (int)len;
    g.snap = a.states; g.sSnap = S * N * D;
    g.len = (int)L;
    e = ni > 1 ? gemm<E_CARRY_SNAP, true>(g, S, st, nullptr, 0, &n) : gemm<E_CARRY, true>(g, S, st, nullptr, 0, &n);
    if (e != hipSuccess) return e;
    if (ni > 1) {  // the later intervals' readouts
      r.niv = (int)ni - 1;
      r.A += L * N;
      r.C += L * D;
      if (ni == 2) r.M = r.M1;
      r.B = a.states;
      e = gemm<E_ROWSCALE_ACC>(r, S, st, a.part, pe, &n);
      if (e != hipSuccess) return e;
    }
    rho_cur = a.rho_out;
  }
  if (launches) *launches += n;
  return hipSuccess;
}

}  // namespace bdh
