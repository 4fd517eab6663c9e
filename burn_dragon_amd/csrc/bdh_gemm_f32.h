// Batched fp32 GEMM on gfx950 matrix cores with the epilogues of the
// recurrence's closed form.  Used by the fp32 forward (prefill_f32.hip) and
// the backward (vjp.hip).
//
//   C(m, n) = sum_k A(m, k) B(n, k),  batch b = (b / H, b % H):
//   X(i, j) = X + (b / H) * sXo + (b % H) * sXi + i * sXr + j * sXc
//
// The fp32 MFMAs run at 1/16 of the bf16 rate, so each operand value is split
// into three bf16 parts whose sum is the value itself (24 significant bits
// above 2^-110; x = h + m + l, each part the bf16 nearest to what is left) and the product
// is the six part products down to 2^-16 of the largest:
//   a b = ah bh + (ah bm + am bh) + (am bm + ah bl + al bh)
// on v_mfma_f32_32x32x16_bf16 (exact products, fp32 accumulation).  What is
// left out (am bl + al bm + al bl) is below 2^-24 of the product, the size of
// fp32's own rounding.  ah bh has an accumulator of its own and the five
// small products share a second one, added at the end: in one accumulator
// every small product would be cut to the large sum's last bit.  Measured
// against 64 bits, K = 8192: 4.2e-8 for 5 %-dense ReLU operands, 5.7e-7 for
// normal ones; the fp32 MFMA 7.4e-8 and 1.7e-6; one accumulator 1.4e-7 and
// 1.4e-6.
//
// Workgroups of 256 threads own BT x BT output tiles (BT = 128, or 64 for
// small products), each wave a quarter.  K steps are 16 deep: two steps'
// operands are in flight in registers while a third is multiplied from LDS;
// a thread splits each value it fetched once per tile (6 VALU instructions
// a value with the largest operand's, about half the step's MFMA time) and writes the three parts to
// LDS, double-buffered, so one barrier a step suffices and two workgroups a
// CU overlap one's splitting with the other's MFMAs.
// A long K with few tiles is split into P ranges (split-K): each range's
// workgroup writes its raw sums to a partial buffer, and a reduce kernel
// adds the P partials in range order (deterministic) and applies the
// epilogue.
// Values whose parts do not exist (infinities, NaN, or above bf16's largest)
// and sums past fp32's range make the result not finite, and operands below
// about 2^-110 lose low bits in their parts; a wave that sees a sum that is
// not finite, or one so much smaller than the tile's largest operand that lost
// bits could show (kLost), computes its block again with the fp32 MFMA.  (What
// stays lost: an operand below 2^-134 has no parts, so a sum of products of
// such operands alone is 0.)
// A product with an operand scaled by decay powers multiplies both operands by
// 2^16 instead, which keeps the last part of every fp32 number above bf16's
// smallest: its sums may be as small as the decay makes them.  (Looked at as
// the others, they sent the state of neurons silent while a strong decay
// forgets them to the fp32 MFMA: B1 nh4 T4096 N8192 D128, 1 % active, ALiBi
// decays from 0.78, 3095 us against 1180.  The factor in every product took the
// f32 C2 shape from 1.04 to 1.11 ms: one more instruction for two values.)
#pragma once

#include <type_traits>

#include "bdh_internal.h"
#include "bdh_mfma.h"

namespace bdh {
namespace gf32 {

enum Epi {
  E_STORE = 0,     // C = acc
  E_TRIL_DECAY,    // C = n < m ? acc * d^(m-n) : 0
  E_ROWSCALE,      // C = acc * d^m
  E_ROWSCALE_ACC,  // C += acc * d^m
  E_CARRY,         // C = acc + src * d^kpow (src null: acc)
  E_CARRY_SNAP,    // E_CARRY over a K of several intervals of `len`, the last perhaps shorter, one after
                   // the other; the value at each interval's start but the first goes to snap
  E_ROWREV_ACC,    // C += acc * d^(kpow - m)
  E_SYM_DECAY      // C(m, n) = C(n, m) = acc * d^(m-n) for n < m, C(m, m) = 0; and the decay gradient's
                   // terms ((acc * (m-n)) * src(m, n)) / sd of n < m, summed per tile into dpart
};

struct GemmF32 {
  const float* A;
  const float* B;
  float* C;
  const float* src;     // E_CARRY: addend with C's strides (may equal C); E_SYM_DECAY: the scores, or null (no terms)
  int64_t sAo, sAi, sAm, sAk;   // sAm or sAk is 1
  int64_t sBo, sBi, sBn, sBk;   // sBn or sBk is 1
  int64_t sCo, sCi, sCm, sCn;
  int M, N, K, H;
  int kpow;             // E_CARRY: carry power; KSCALE (decay set): A(m, k) *= d^(kpow - k) (E_CARRY_SNAP: kpow is the end of k's interval)
  int kcausal;          // operand A lower triangular: K of the tile at row m0 limited to m0 + tile
  int klow;             // operand A upper triangular: K of the tile at row m0 from m0's TRI-block on
  const float* decay;   // [H] or null (ones)
  float* part;          // split-K partials [ksplit, batch, M, N] (ksplit > 1)
  int ksplit;
  int64_t batch;        // products of an interval
  // A launch over several intervals (0 and 1: one): interval iv's operands are
  // sA3, sB3, sC3 further each, and the last one's sizes are M1, N1, K1.
  int niv, M1, N1, K1;
  int64_t sA3, sB3, sC3;
  float* snap;          // E_CARRY_SNAP: [intervals - 1] of C's layout, sSnap apart
  int64_t sSnap;
  int len;              // E_CARRY_SNAP: tokens of an interval (a multiple of 2 GK)
  double* dpart;        // E_SYM_DECAY: tile sums [batch, dslots]
  int dslots, dacc;     // (dacc: added to what is there)
  int recurrent_eps;    // E_SYM_DECAY: the recurrent backward's decay guard
  int tri;              // masked square product: only the 128 x 128 blocks on or below the diagonal are computed
};

constexpr int GK = 16;               // k step
constexpr int TRI = 128;             // edge of the blocks a masked product is computed (and written) in
constexpr int DSCALE = 1024;         // KSCALE: most k of one workgroup (LDS table of d^(kpow - k))

// A sum smaller than this share of the tile's largest operand may lack bits:
// an operand's parts end at 2^-133, bf16's smallest, so the sum is off by up
// to sqrt(K) 2^-134 of the largest operand (2^-127.5 at K = 8192), and that
// has to stay below its own 2^-24.
constexpr float kLost = 0x1p-104f;
constexpr float kUp = 0x1p16f;  // KSCALE: the operands' factor

__device__ __forceinline__ float dpowf(float d, int e) { return powf(d, (float)e); }

// The divisor of the decay gradient: the reference's two guards against 0.
__device__ __forceinline__ float decay_sd(float d, int recurrent_eps) {
  if (recurrent_eps) return (d < 1e-8f && d > -1e-8f) ? 1e-8f : d;
  return d + 1e-12f;
}

// Sum of a workgroup's 256 values in a fixed order, in thread 0.
__device__ __forceinline__ double block_sum(double v, double* red) {
  red[threadIdx.x] = v;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  return red[0];
}

// The epilogue's addend: C itself (the accumulating kinds), src (E_CARRY),
// or none.
template <int EPI>
__device__ __forceinline__ const float* epi_addend(const GemmF32& g, int64_t c0) {
  if (EPI == E_ROWSCALE_ACC || EPI == E_ROWREV_ACC) return g.C + c0;
  if ((EPI == E_CARRY || EPI == E_CARRY_SNAP) && g.src) return g.src + c0;
  return nullptr;
}

// Output value of (m, n) from the sum v, the kind's decay power (a function,
// called only where the kind has one and a decay is set) and the addend x
// (when the kind has one).
template <int EPI, class Pow>
__device__ __forceinline__ float epi_value(const GemmF32& g, Pow&& power, float carry, int m, int n, float v, float x) {
  if (EPI == E_TRIL_DECAY) v = n < m ? (g.decay ? v * power(m, n) : v) : 0.0f;
  if ((EPI == E_ROWSCALE || EPI == E_ROWSCALE_ACC || EPI == E_ROWREV_ACC) && g.decay) v *= power(m, n);
  if (EPI == E_ROWSCALE_ACC || EPI == E_ROWREV_ACC) v += x;
  if (EPI == E_CARRY && g.src) v += x * carry;
  if (EPI == E_CARRY_SNAP) v += x * carry;
  return v;
}

// A load of four floats at any float's address.
typedef float floatx4u __attribute__((ext_vector_type(4), aligned(4)));

// One operand's share of a step for thread t of a BT-row tile: E = BT / 16
// values, in fours contiguous in memory (16-byte loads):
//   KC (contiguous along k):    k 4 (t % 4) .. + 3 of rows t / 4 and, BT =
//       128, t / 4 + 64: four lanes read a row's 64 bytes;
//   RC (contiguous along rows): rows 4 (t % (BT / 4)) .. + 3 of the E / 4
//       k's from (t / (BT / 4)) E / 4: a wave reads whole rows of the tile.
// Rows past the operand's end re-read its last row: their sums are never
// written.  k past Kt reads as 0.
template <int BT, bool KC>
struct Loader {
  static constexpr int E = BT / 16;
  const float* p;   // KC: the thread's first row at its first k; RC: the tile's first row at its first k
  const float* p1;  // KC, BT = 128: its second row
  int64_t sk;
  int k0, row, R;   // the thread's first k and row within a step's tile; rows of the tile
  __device__ __forceinline__ void init(const float* X, int64_t sr, int64_t sk_, int R_, int t) {
    sk = sk_;
    R = R_;
    if (KC) {
      k0 = (t & 3) * 4;
      row = t >> 2;
      p = X + (int64_t)min(row, R - 1) * sr + k0;
      p1 = X + (int64_t)min(row + 64, R - 1) * sr + k0;
    } else {
      k0 = t / (BT / 4) * (E / 4);
      row = t % (BT / 4) * 4;
      p = X + (int64_t)k0 * sk;
    }
  }
  // k of value e, relative to the step.
  __device__ __forceinline__ int k_of(int e) const { return k0 + (KC ? e & 3 : e >> 2); }
  __device__ __forceinline__ void load(int kb, int Kt, float (&v)[E]) const {
    const bool fast = kb + GK <= Kt && (KC || R >= BT);
#pragma unroll
    for (int r = 0; r < E / 4; ++r) {
      const float* q = KC ? (r ? p1 : p) + kb : p + (int64_t)(kb + r) * sk + row;
      if (fast) {
        const floatx4u a = *reinterpret_cast<const floatx4u*>(q);
        v[4 * r] = a[0]; v[4 * r + 1] = a[1]; v[4 * r + 2] = a[2]; v[4 * r + 3] = a[3];
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int k = kb + k_of(4 * r + e), kc = min(k, Kt - 1);
          const float x = KC ? (r ? p1 : p)[kc - k0] : p[(int64_t)(kc - k0) * sk + min(row + e, R - 1)];
          v[4 * r + e] = k < Kt ? x : 0.0f;
        }
      }
    }
  }
};

// LDS tile of one part of an operand, every access free of bank conflicts.
//   KC: two halves of 8 k, 16 bytes a row, the second half 128 bytes further
//       (a write's 32 lanes, 8 rows of both halves, cover every bank once);
//       a fragment is one 16-byte read.
//   RC: k rows of BT values, 64 bytes apart beyond their own (a transposing
//       read's 32 lanes, 4 k rows of 64 bytes, cover every bank once); a
//       fragment is two ds_read_b64_tr_b16, 4 k each: lane 4 r + c of 16
//       names 4 values of k row r, lane i receives value i of the 4 rows.
template <int BT>
constexpr int kHalf = BT * 16 + 128;
template <int BT>
constexpr int kPitch = BT * 2 + 64;
template <int BT, bool KC>
constexpr int kPart = KC ? 2 * kHalf<BT> : GK * kPitch<BT>;

// Splits a loader's values into their three bf16 parts and writes them to the
// tiles at `lds`.
template <int BT, bool KC>
__device__ __forceinline__ void split_store(char* lds, const Loader<BT, KC>& l, const float (&v)[BT / 16]) {
  constexpr int E = BT / 16;
  uint32_t w[3][E / 2];
#pragma unroll
  for (int i = 0; i < E / 2; ++i) {
    const float x = v[2 * i], y = v[2 * i + 1];
    // (The pair stays one register: left to itself the compiler converts the
    // low value a second time, 16 more instructions a step of 107.)
    uint32_t h = pack_bf16x2(x, y);
    asm("" : "+v"(h));
    const float rx = x - bf16_lo(h), ry = y - bf16_hi(h);
    uint32_t m = pack_bf16x2(rx, ry);
    asm("" : "+v"(m));
    w[0][i] = h;
    w[1][i] = m;
    w[2][i] = pack_bf16x2(rx - bf16_lo(m), ry - bf16_hi(m));
  }
  char* o = lds + (KC ? (l.k0 >> 3) * kHalf<BT> + l.row * 16 + (l.k0 & 7) * 2 : l.k0 * kPitch<BT> + l.row * 2);
#pragma unroll
  for (int q = 0; q < 3; ++q)
#pragma unroll
    for (int r = 0; r < E / 4; ++r)
      *reinterpret_cast<uint2*>(o + q * kPart<BT, KC> + r * (KC ? 64 * 16 : kPitch<BT>)) =
          make_uint2(w[q][2 * r], w[q][2 * r + 1]);
}

typedef short shortx4 __attribute__((ext_vector_type(4)));

// A 32-row fragment (rows row0 ..) of the part at `lds`; base = frag_base.
template <int BT, bool KC>
__device__ __forceinline__ int frag_base(int lane) {
  if (KC) return (lane >> 5) * kHalf<BT> + (lane & 31) * 16;
  return (8 * (lane >> 5) + ((lane & 15) >> 2)) * kPitch<BT> + (((lane >> 4) & 1) * 16 + (lane & 3) * 4) * 2;
}
template <int BT, bool KC>
__device__ __forceinline__ bf16x8 frag_read(const char* lds, int base, int row0) {
  if constexpr (KC) {
    return *reinterpret_cast<const bf16x8*>(lds + base + row0 * 16);
  } else {
    typedef __attribute__((address_space(3))) shortx4 lds4;
    const char* p = lds + base + row0 * 2;
    struct {
      shortx4 v[2];
    } f = {{__builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4*)p),
            __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4*)(p + 4 * kPitch<BT>))}};
    return __builtin_bit_cast(bf16x8, f);
  }
}

// 256 threads, two workgroups a CU.
template <int EPI, bool KSCALE, bool AKC, bool BKC, int BT>
__global__ __launch_bounds__(256, 2) void gemm_split_kernel(GemmF32 g, int ntx, int nty) {
  constexpr int E = BT / 16, NB = BT / 64;  // values a thread stages; 32 x 32 blocks a wave, each way
  constexpr int PA = kPart<BT, AKC>, PB = kPart<BT, BKC>, STAGE = 3 * (PA + PB);
  __shared__ __attribute__((aligned(16))) char lds[2 * STAGE + (KSCALE ? 4 * (DSCALE + 3 * GK) : 0)];
  __shared__ float wmax[4];  // the waves' largest staged operands
  __shared__ int wask[4];
  const int t = threadIdx.x, lane = t & 63, w = wave_id();
  const int wm = w >> 1, wn = w & 1;
  // Workgroup ids are remapped so that each XCD (id % 8) takes a contiguous
  // range of tiles, the shorter side of the tile grid first: the tiles that
  // share the longer operand's rows then run together on one L2.
  const int nwg = (int)gridDim.x, id = (int)blockIdx.x;
  int wk = (nwg & 7) ? id : (id & 7) * (nwg >> 3) + (id >> 3);
  int tx, ty, slot = 0;
  int64_t z;
  if (g.tri) {
    // TRI-blocks (by, bx <= by) in row order, SUB tiles each.
    constexpr int ED = TRI / BT, SUB = ED * ED;
    const int nbk = (nty + ED - 1) / ED;
    const int per = nbk * (nbk + 1) / 2 * SUB;
    z = wk / per;
    slot = wk - (int)z * per;
    int r = slot / SUB;
    const int sub = slot % SUB;
    ty = 0;
    while (r > ty) {
      r -= ty + 1;
      ++ty;
    }
    ty = ty * ED + sub / ED;
    tx = r * ED + sub % ED;
    if (ty >= nty || tx >= ntx) {
      if (EPI == E_SYM_DECAY && g.src && t == 0 && !g.dacc) g.dpart[z * g.dslots + slot] = 0.0;
      return;
    }
  } else if (ntx < nty) {
    tx = wk % ntx;
    wk /= ntx;
    ty = wk % nty;
    z = wk / nty;
  } else {
    ty = wk % nty;
    wk /= nty;
    tx = wk % ntx;
    z = wk / ntx;
  }
  const int P = g.ksplit > 1 ? g.ksplit : 1;
  const int kp = (int)(z % P);
  const int64_t bz = z / P, iv = g.niv > 1 ? bz / g.batch : 0, b = bz - iv * g.batch, bo = b / g.H, bi = b - bo * g.H;
  const int m0 = ty * BT, n0 = tx * BT;
  const bool lastiv = g.niv > 1 && iv == g.niv - 1;
  const int M = lastiv ? g.M1 : g.M, N = lastiv ? g.N1 : g.N, K = lastiv ? g.K1 : g.K;
  if (m0 >= M || n0 >= N) return;  // a shorter last interval
  const float d = g.decay ? g.decay[bi] : 1.0f;
  const int Kfull = g.kcausal ? min(K, m0 + BT) : K;
  const int kbase = g.klow ? m0 / TRI * TRI : 0;
  const int chunk = ((Kfull - kbase + P - 1) / P + GK - 1) / GK * GK;
  const int k_lo = min(Kfull, kbase + kp * chunk);
  const int Kt = min(Kfull, k_lo + chunk) - k_lo;  // this workgroup's depth, from k_lo
  const int nks = (Kt + GK - 1) / GK;
  const float* A0 = g.A + iv * g.sA3 + bo * g.sAo + bi * g.sAi;
  const float* B0 = g.B + iv * g.sB3 + bo * g.sBo + bi * g.sBi;
  const int64_t c0 = iv * g.sC3 + bo * g.sCo + bi * g.sCi;
  Loader<BT, AKC> la;
  Loader<BT, BKC> lb;
  la.init(A0 + (int64_t)m0 * g.sAm + (int64_t)k_lo * g.sAk, g.sAm, g.sAk, M - m0, t);
  lb.init(B0 + (int64_t)n0 * g.sBn + (int64_t)k_lo * g.sBk, g.sBn, g.sBk, N - n0, t);

  float* sct = reinterpret_cast<float*>(lds + 2 * STAGE);
  constexpr bool SNAP = EPI == E_CARRY_SNAP;
  if (KSCALE) {
    if (SNAP) {
      for (int k = t; k <= g.len; k += 256) sct[k] = dpowf(d, k) * kUp;
    } else {
      for (int k = t; k < (nks + 2) * GK; k += 256) sct[k] = k < Kt ? dpowf(d, g.kpow - (k_lo + k)) * kUp : 0.0f;
    }
    __syncthreads();
  }
  // SNAP: tokens of interval i, and a power of its token k's weight (0 past K).
  auto len_of = [&](int i) { return min(g.len, Kt - i * g.len); };
  int siv = 0, soff = 0;  // the interval and offset of the step staged next

  float va[2][E], vb[2][E];
  float mx = 0.0f;  // the largest operand staged by this thread
  auto load = [&](int s, float (&a)[E], float (&bv)[E]) {
    la.load(s * GK, Kt, a);
    lb.load(s * GK, Kt, bv);
  };
  auto stage = [&](int s, float (&a)[E], float (&bv)[E]) {
    char* o = lds + (s & 1) * STAGE;
    if (KSCALE) {
#pragma unroll
      for (int e = 0; e < E; ++e) a[e] *= sct[SNAP ? max(0, len_of(siv) - soff - la.k_of(e)) : s * GK + la.k_of(e)];
      if (SNAP) {
        soff += GK;
        if (soff == g.len) {
          soff = 0;
          ++siv;
        }
      }
    }
    // (After the splitting where both operands are contiguous along k: the f32
    // C2 shape's gram 398 us against 420; the others' best place is before it.)
    auto largest = [&]() {
#pragma unroll
      for (int e = 0; e < E; ++e) mx = fmaxf(fmaxf(mx, fabsf(a[e])), fabsf(bv[e]));
      asm volatile("" : "+v"(mx));  // here, not where copies of the values would have to live to
    };
    if (KSCALE) {
#pragma unroll
      for (int e = 0; e < E; ++e) bv[e] *= kUp;
    }
    if (!KSCALE && !(AKC && BKC)) largest();
    split_store(o, la, a);
    split_store(o + 3 * PA, lb, bv);
    if (!KSCALE && AKC && BKC) largest();
  };

  floatx16 big[NB][NB], small[NB][NB];
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      big[i][j] = zero16();
      small[i][j] = zero16();
    }
  const int fa = frag_base<BT, AKC>(lane), fb = 3 * PA + frag_base<BT, BKC>(lane);
  auto multiply = [&](int s) {
    const char* o = lds + (s & 1) * STAGE;
    bf16x8 a[3][NB], c[3][NB];
#pragma unroll
    for (int q = 0; q < 3; ++q)
#pragma unroll
      for (int i = 0; i < NB; ++i) {
        a[q][i] = frag_read<BT, AKC>(o + q * PA, fa, wm * 32 * NB + 32 * i);
        c[q][i] = frag_read<BT, BKC>(o + q * PB, fb, wn * 32 * NB + 32 * i);
      }
    auto add = [&](int qa, int qb, floatx16 (&acc)[NB][NB]) {
#pragma unroll
      for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[i][j] = mfma32(a[qa][i], c[qb][j], acc[i][j]);
    };
    add(0, 0, big);
    add(0, 1, small);
    add(1, 0, small);
    add(1, 1, small);
    add(0, 2, small);
    add(2, 0, small);
  };

  const int mw = m0 + wm * 32 * NB, nw = n0 + wn * 32 * NB;  // the wave's block
  // SNAP, at the end of interval i, another one following: the state there is
  // written, and the next interval's sum starts from 0 and is added to it (as
  // an interval's sum always was: one sum over all of them would round to the
  // growing state's last bit).
  const float* X = P > 1 ? nullptr : epi_addend<EPI>(g, c0);
  // Of the sums seen: one is not finite; the smallest that is not 0, as twice
  // its bits less one (0: the largest number there is).
  bool bad = false;
  uint32_t least = ~0u;
  auto look = [&](float v, float& nan) {
    nan = fmaf(v, 0.0f, nan);
    if (!KSCALE) least = min(least, (__builtin_bit_cast(uint32_t, v) << 1) - 1);
  };
  float down = KSCALE ? 1.0f / (kUp * kUp) : 1.0f;
  auto snapshot = [&](int i) {
    float* o = g.snap + i * g.sSnap + c0;
    // (The block's addresses are not kept through the step loop: 64 of them
    // would not fit beside the accumulators.)
    int mo = mw + acc_row(lane, 0);
    asm volatile("" : "+v"(mo));
    const float dl = g.decay ? dpowf(d, len_of(i)) : 1.0f;
    float nan = 0.0f;
#pragma unroll
    for (int i2 = 0; i2 < NB; ++i2)
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        const int n = nw + 32 * j + acc_col(lane);
        const int64_t off = (int64_t)(mo + 32 * i2) * g.sCm + (int64_t)n * g.sCn;
        float x[16];
        if (X != nullptr) {
#pragma unroll
          for (int r = 0; r < 16; ++r)
            x[r] = mo + 32 * i2 + acc_row(0, r) < M && n < N ? X[off + acc_row(0, r) * g.sCm] : 0.0f;
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          float v = big[i2][j][r] + small[i2][j][r];
          look(v, nan);
          if (KSCALE) v *= down;
          if (mo + 32 * i2 + acc_row(0, r) < M && n < N)
            o[off + acc_row(0, r) * g.sCm] = X != nullptr ? v + x[r] * dl : v;
        }
        big[i2][j] = zero16();
        small[i2][j] = zero16();
        __builtin_amdgcn_sched_barrier(0);
      }
    bad |= nan != 0.0f;
    X = o;
  };

  // Step s: its parts are in LDS buffer s & 1, step s + 1's values in
  // register set (s + 1) & 1; the loads of step s + 2 go to the other set.
  // One barrier a step: it ends the writes of step s's buffer and the reads
  // of step s - 1's, which step s + 1's parts replace after it.  The
  // splitting of step s + 1 is spread between the MFMAs of step s, four VALU
  // instructions in the shadow of each.  Steps past the last are zeros (the
  // loop runs an even number, one exit).
  if (nks > 0) {
    load(0, va[0], vb[0]);
    load(1, va[1], vb[1]);
    stage(0, va[0], vb[0]);
    int s = 0, end = SNAP ? min(nks, g.len / GK) : nks, i = 0;
    while (true) {
      do {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          load(s + u + 2, va[u], vb[u]);
          __syncthreads();
          multiply(s + u);
          stage(s + u + 1, va[u ^ 1], vb[u ^ 1]);
          __builtin_amdgcn_sched_group_barrier(0x100, 3 * NB * ((AKC ? 1 : 2) + (BKC ? 1 : 2)), 0);  // fragment reads
#pragma unroll
          for (int k = 0; k < 6 * NB * NB; ++k) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // an MFMA
            __builtin_amdgcn_sched_group_barrier(0x002, NB == 2 ? 4 : 8, 0);  // VALU
          }
        }
        s += 2;
      } while (s < end);
      if (!SNAP || end >= nks) break;
      snapshot(i++);
      end = min(nks, end + g.len / GK);
    }
  }

  float nan = 0.0f;
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        big[i][j][r] += small[i][j][r];
        small[i][j][r] = 0.0f;
        look(big[i][j][r], nan);
        if (KSCALE) big[i][j][r] *= down;
      }
  bad |= nan != 0.0f;
  // A sum below kLost of the largest operand of the workgroup asks for the
  // block again; the largest operand is looked for where one is above kLarge
  // or a sum below its share.
  constexpr float kLarge = 0x1p40f;
  const bool ask = !KSCALE && __any(mx >= kLarge || least < (__builtin_bit_cast(uint32_t, kLarge * kLost) << 1) - 1);
  if (lane == 0) wask[w] = ask;
  __syncthreads();  // also: every wave has read its last fragments
  if (wask[0] || wask[1] || wask[2] || wask[3]) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
    if (lane == 0) wmax[w] = mx;
    __syncthreads();
    const float lost = fmaxf(fmaxf(wmax[0], wmax[1]), fmaxf(wmax[2], wmax[3])) * kLost;
    bad |= least < (__builtin_bit_cast(uint32_t, lost) << 1) - 1;
  }
  if (__any(bad)) {
    // The block again on v_mfma_f32_32x32x2_f32, straight from memory.
    if (SNAP) X = epi_addend<EPI>(g, c0);
    down = 1.0f;
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j) big[i][j] = zero16();
    int i0 = 0;  // SNAP: the interval
    for (int k = 0; k < Kt; k += 2) {
      if (SNAP && k == (i0 + 1) * g.len) snapshot(i0++);
      const int kk = k + (lane >> 5), ka = k_lo + min(kk, Kt - 1);
      float av[NB], bv[NB];
#pragma unroll
      for (int i = 0; i < NB; ++i) {
        av[i] = A0[(int64_t)min(mw + 32 * i + (lane & 31), M - 1) * g.sAm + (int64_t)ka * g.sAk];
        if (KSCALE) av[i] *= dpowf(d, SNAP ? max(0, len_of(i0) - (kk - i0 * g.len)) : g.kpow - ka);
        bv[i] = B0[(int64_t)min(nw + 32 * i + (lane & 31), N - 1) * g.sBn + (int64_t)ka * g.sBk];
        if (kk >= Kt) av[i] = bv[i] = 0.0f;
      }
#pragma unroll
      for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
          big[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[i], bv[j], big[i][j], 0, 0, 0);
    }
  }

  const float carry = !g.decay ? 1.0f
                      : SNAP   ? dpowf(d, len_of((nks - 1) * GK / g.len))
                      : EPI == E_CARRY ? dpowf(d, g.kpow) : 1.0f;
  // The decay powers of the epilogue's m - n (or rows), one powf each for the
  // tile instead of one an element (which took 8 of a C1 product's 16 us).
  constexpr bool DIFF = EPI == E_TRIL_DECAY || EPI == E_SYM_DECAY;
  constexpr bool ROWS = EPI == E_ROWSCALE || EPI == E_ROWSCALE_ACC || EPI == E_ROWREV_ACC;
  float* pw = reinterpret_cast<float*>(lds);
  if ((DIFF || ROWS) && P == 1 && g.decay) {
    if (DIFF && t < 2 * BT) pw[t] = dpowf(d, max(0, m0 - n0 - BT + 1 + t));
    if (ROWS && t < BT) pw[t] = dpowf(d, EPI == E_ROWREV_ACC ? g.kpow - (m0 + t) : m0 + t);
    __syncthreads();
  }
  auto power = [&](int m, int n) {
    if (!(DIFF || ROWS) || !g.decay) return 1.0f;
    return DIFF ? pw[m - n - (m0 - n0 - BT + 1)] : pw[m - m0];
  };
  const int64_t batches = g.batch * (g.niv > 1 ? g.niv : 1);
  float* Pp = P > 1 ? g.part + ((int64_t)kp * batches + bz) * (int64_t)g.M * g.N : nullptr;
  float* C = g.C + c0;
  if constexpr (EPI == E_SYM_DECAY) {
    const float* SC = g.src ? g.src + c0 : nullptr;
    const float sd = decay_sd(d, g.recurrent_eps);
    double sum = 0.0;
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        const int n = nw + 32 * j + acc_col(lane);
        float x[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int m = mw + 32 * i + acc_row(lane, r);
          x[r] = SC && m < M && n < m ? SC[(int64_t)m * g.sCm + n] : 0.0f;
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int m = mw + 32 * i + acc_row(lane, r);
          if (m >= M || n > m) continue;
          const float v = n < m ? big[i][j][r] : 0.0f;
          sum += (double)(((v * (float)(m - n)) * x[r]) / sd);
          const float o = g.decay ? v * power(m, n) : v;
          C[(int64_t)m * g.sCm + n] = o;
          C[(int64_t)n * g.sCm + m] = o;
        }
      }
    if (SC) {
      __syncthreads();
      const double all = block_sum(sum, reinterpret_cast<double*>(lds));
      if (t == 0) {
        double* o = g.dpart + b * g.dslots + slot;
        *o = g.dacc ? *o + all : all;
      }
    }
    return;
  }
  // Out through LDS, 32
  // rows of the wave's block at a time in a region of its own, so that a lane
  // stores 16 bytes and a wave whole 256-byte pieces of rows (from the
  // accumulators' layout, 4 bytes a lane in 128-byte pieces, the 268 MB state
  // of the f32 C2 shape left at 1.6 TB/s).
  constexpr int EP = 32 * NB + 4, LPR = 8 * NB, RPI = 64 / LPR;  // row pitch; lanes a row; rows an access
  float* eb = reinterpret_cast<float*>(lds + 1024) + w * 32 * EP;  // past the power table
  static_assert(1024 + 4 * 32 * EP * 4 <= 2 * STAGE && 2 * BT * 4 <= 1024, "the epilogue's LDS");
  const int er = lane / LPR, n = nw + (lane % LPR) * 4;
  const bool quad = g.sCn == 1 && n + 4 <= N;
#pragma unroll
  for (int i = 0; i < NB; ++i) {
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) eb[acc_row(lane, r) * EP + 32 * j + acc_col(lane)] = big[i][j][r];
    floatx4 v[32 / RPI], x[32 / RPI];
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the wave's lanes have written
#pragma unroll
    for (int q = 0; q < 32 / RPI; ++q) {
      const int m = mw + 32 * i + q * RPI + er;
      v[q] = *reinterpret_cast<const floatx4*>(&eb[(q * RPI + er) * EP + (lane % LPR) * 4]);
      x[q] = zero4();
      // A block's addends are all loaded before its first store.
      if (X == nullptr || m >= M || n >= N) continue;
      const float* xp = X + (int64_t)m * g.sCm + (int64_t)n * g.sCn;
      if (quad) {
        x[q] = *reinterpret_cast<const floatx4u*>(xp);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < N) x[q][e] = xp[e * g.sCn];
      }
    }
#pragma unroll
    for (int q = 0; q < 32 / RPI; ++q) {
      const int m = mw + 32 * i + q * RPI + er;
      if (m >= M || n >= N) continue;
      float* o = P > 1 ? Pp + (int64_t)m * g.N + n : C + (int64_t)m * g.sCm + (int64_t)n * g.sCn;
      floatx4u y;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        y[e] = P > 1 ? v[q][e] : epi_value<EPI>(g, power, carry, m, n + e, v[q][e], x[q][e]);
      if (P > 1 ? n + 4 <= N : quad) {
        if (EPI == E_CARRY || EPI == E_CARRY_SNAP || EPI == E_STORE)
          __builtin_nontemporal_store(y, reinterpret_cast<floatx4u*>(o));
        else
          *reinterpret_cast<floatx4u*>(o) = y;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < N) o[P > 1 ? e : e * g.sCn] = y[e];
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // read before the next 32 rows are written
  }
}

// Split-K: sums the P partials of each (b, m, n) in range order and applies
// the epilogue, four columns a thread (the last thread of a row that is not a
// multiple of four: the rest).  Product blockIdx.y.  A masked
// product's blocks above the diagonal are left out: their partials were not
// written, and their outputs are never read.
template <int EPI>
__global__ __launch_bounds__(256) void gemm_reduce_kernel(GemmF32 g, int n4) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t mi = i / n4;
  if (mi >= g.M) return;
  const int m = (int)mi, n = (int)(i - mi * n4) * 4;
  if (g.tri && n / TRI > m / TRI) return;
  const int64_t bz = blockIdx.y, iv = g.niv > 1 ? bz / g.batch : 0, b = bz - iv * g.batch, bo = b / g.H,
                bi = b - bo * g.H;
  const bool lastiv = g.niv > 1 && iv == g.niv - 1;
  const int M = lastiv ? g.M1 : g.M, N = lastiv ? g.N1 : g.N;
  if (m >= M || n >= N) return;
  const float d = g.decay ? g.decay[bi] : 1.0f;
  const float carry = (EPI == E_CARRY && g.decay) ? dpowf(d, g.kpow) : 1.0f;
  auto power = [&](int m, int n) {
    return dpowf(d, EPI == E_TRIL_DECAY ? m - n : EPI == E_ROWREV_ACC ? g.kpow - m : m);
  };
  const int64_t MN = (int64_t)g.M * g.N, total = (int64_t)gridDim.y * MN;
  const float* P = g.part + bz * MN + (int64_t)m * g.N + n;
  const int64_t c0 = iv * g.sC3 + bo * g.sCo + bi * g.sCi;
  const float* X = epi_addend<EPI>(g, c0);
  const int64_t o = (int64_t)m * g.sCm + (int64_t)n * g.sCn;
  float* C = g.C + c0 + o;
  if (g.sCn == 1 && n + 4 <= N) {
    floatx4 v = zero4(), x = zero4();
    for (int kp = 0; kp < g.ksplit; ++kp) v += *reinterpret_cast<const floatx4u*>(P + kp * total);
    if (X) x = *reinterpret_cast<const floatx4u*>(X + o);
    floatx4u w;
#pragma unroll
    for (int e = 0; e < 4; ++e) w[e] = epi_value<EPI>(g, power, carry, m, n + e, v[e], x[e]);
    *reinterpret_cast<floatx4u*>(C) = w;
    return;
  }
  for (int e = 0; e < 4 && n + e < N; ++e) {
    float v = 0.0f;
    for (int kp = 0; kp < g.ksplit; ++kp) v += P[kp * total + e];
    C[e * g.sCn] = epi_value<EPI>(g, power, carry, m, n + e, v, X ? X[o + e * g.sCn] : 0.0f);
  }
}

// Tiles of a [M, N] product (a masked square one: of its blocks on or below
// the diagonal) in BT x BT tiles.
inline int64_t tile_count(int M, int N, int BT, bool tri) {
  if (tri) {
    const int64_t nb = (M + TRI - 1) / TRI;
    return nb * (nb + 1) / 2 * (TRI / BT) * (TRI / BT);
  }
  return (int64_t)((N + BT - 1) / BT) * ((M + BT - 1) / BT);
}

// Ranges of K for a product of `tiles` 128 x 128 tiles: the count (up to 16,
// each range at least 128 deep) with the least time, in units of one k of a
// round of workgroups (two a CU; 86 ns measured): the rounds' depth, and for
// more than one range the partials' write and read (128 KiB a tile and range
// at 4.5 TB/s: 0.34) and the reduce's launch (5 us).  The masked 512 x 512 x
// 8192 gram of 32 streams, 320 tiles on 512 slots: one range 8192 units, 3
// ranges 5850.  Unsplit with a short K (< 1024) unless the tiles fill under a
// quarter of the CUs.
inline int split_k_ranges(int64_t tiles, int K) {
  const int64_t slots = 2 * (int64_t)device_cus();
  if (K < 1024 && tiles * 4 >= (int64_t)device_cus()) return 1;
  int best = 1;
  double cost = 0;
  for (int p = 1; p <= 16 && (p == 1 || K / p >= 128); ++p) {
    const double c = (double)((tiles * p + slots - 1) / slots) * ((double)K / p) +
                     (p > 1 ? 0.34 * (double)tiles * p + 58.0 : 0.0);
    if (p == 1 || c < cost) {
      best = p;
      cost = c;
    }
  }
  return best;
}

template <int EPI, bool KSCALE, int BT>
hipError_t launch_gemm(const GemmF32& g, int64_t nwg, hipStream_t st) {
  const int ntx = (g.N + BT - 1) / BT, nty = (g.M + BT - 1) / BT;
  const bool akc = g.sAk == 1, bkc = g.sBk == 1;
  if ((!akc && g.sAm != 1) || (!bkc && g.sBn != 1) || nwg > INT32_MAX) return hipErrorInvalidValue;
  const dim3 grid((unsigned)nwg);
  if constexpr (EPI == E_CARRY_SNAP) {  // the state's operands are both contiguous along their rows (at one row or column: along k too)
    if (g.sAm != 1 || g.sBn != 1) return hipErrorInvalidValue;
    hipLaunchKernelGGL((gemm_split_kernel<EPI, KSCALE, false, false, BT>), grid, dim3(256), 0, st, g, ntx, nty);
  } else if (akc && bkc)
    hipLaunchKernelGGL((gemm_split_kernel<EPI, KSCALE, true, true, BT>), grid, dim3(256), 0, st, g, ntx, nty);
  else if (akc)
    hipLaunchKernelGGL((gemm_split_kernel<EPI, KSCALE, true, false, BT>), grid, dim3(256), 0, st, g, ntx, nty);
  else if (bkc)
    hipLaunchKernelGGL((gemm_split_kernel<EPI, KSCALE, false, true, BT>), grid, dim3(256), 0, st, g, ntx, nty);
  else
    hipLaunchKernelGGL((gemm_split_kernel<EPI, KSCALE, false, false, BT>), grid, dim3(256), 0, st, g, ntx, nty);
  return hipGetLastError();
}

constexpr int64_t kMaxBatch = 65535;  // products of a launch (the reduce's grid)

// A product runs on 64 x 64 tiles while its 128 x 128 ones leave CUs idle.
inline bool small_tiles(int64_t tiles, int p) { return tiles * p < (int64_t)device_cus(); }

// Tile sums an unsplit E_SYM_DECAY product of [L, L] writes per batch.
inline int sym_slots(int64_t batch, int L) {
  const int64_t tiles = tile_count(L, L, 128, true);
  return (int)(small_tiles(tiles * batch, 1) ? tile_count(L, L, 64, true) : tiles);
}

// C = epilogue(A B^T) over `batch` products (of each of g.niv intervals).  With `part` (part_elems floats)
// a long K may be split; the partials need ksplit * batch * M * N floats.
template <int EPI, bool KSCALE = false>
hipError_t gemm(GemmF32 g, int64_t batch, hipStream_t st, float* part = nullptr, size_t part_elems = 0,
                uint64_t* launches = nullptr) {
  if (g.M <= 0 || g.N <= 0 || batch <= 0) return hipSuccess;
  if constexpr (KSCALE) {
    if (!g.decay) return gemm<EPI, false>(g, batch, st, part, part_elems, launches);
    if ((EPI == E_CARRY_SNAP ? g.len : g.K) > DSCALE) return hipErrorInvalidValue;
  }
  if (EPI == E_CARRY_SNAP && (part || g.len <= 0 || g.len % (2 * GK) != 0)) return hipErrorInvalidValue;
  g.batch = batch;
  if (g.niv > 1) batch *= g.niv;
  if (batch > kMaxBatch) return hipErrorInvalidValue;
  g.tri = (EPI == E_TRIL_DECAY || EPI == E_SYM_DECAY) && g.M == g.N;
  if (EPI == E_SYM_DECAY && (!g.tri || part)) return hipErrorInvalidValue;
  const size_t per = (size_t)batch * (size_t)g.M * (size_t)g.N;
  const int64_t tiles = tile_count(g.M, g.N, 128, g.tri) * batch;
  int p = part ? split_k_ranges(tiles, g.K) : 1;
  if ((size_t)p * per > part_elems) p = (int)(part_elems / per);
  if (p < 1) p = 1;
  g.ksplit = p;
  g.part = p > 1 ? part : nullptr;
  const hipError_t e = small_tiles(tiles, p)
                           ? launch_gemm<EPI, KSCALE, 64>(g, tile_count(g.M, g.N, 64, g.tri) * batch * p, st)
                           : launch_gemm<EPI, KSCALE, 128>(g, tiles * p, st);
  if (e != hipSuccess) return e;
  if (p > 1 && EPI != E_SYM_DECAY) {
    const int n4 = (g.N + 3) / 4;
    hipLaunchKernelGGL(gemm_reduce_kernel<EPI>, dim3((unsigned)(((int64_t)g.M * n4 + 255) / 256), (unsigned)batch),
                       dim3(256), 0, st, g, n4);
  }
  if (launches) *launches += p > 1 ? 2 : 1;
  return hipGetLastError();
}

// Partial floats the split-K of a [batch, M, N] product at depth K may use.
inline size_t split_k_elems(int64_t batch, int M, int N, int K) {
  // A square product may be the masked one, whose fewer tiles take more ranges.
  const int p = split_k_ranges(tile_count(M, N, 128, M == N) * batch, K);
  return p > 1 ? (size_t)p * (size_t)batch * (size_t)M * (size_t)N : 0;
}

}  // namespace gf32
}  // namespace bdh
