// Chunked WKV7 prefill on gfx950 matrix cores (D = 64, fp32 state carry).
//
// Chunk algebra (L = 16 tokens, rows = tokens, S0 = start-of-chunk state,
// g_t = sum_{s<=t} log w_s inside the chunk, gamma_t = exp(g_t)):
//   A~ = a*gamma_{t-1}, R~ = r*gamma_t, B^ = b/gamma_t, K^ = k/gamma_t
//   Mab = strict_tril(A~ B^T), Mak = strict_tril(A~ K^T)
//   Mrb = tril(R~ B^T),        Mrk = tril(R~ K^T)
//   T = (I - Mab)^-1
//   U (the per-token sa rows) = T (A~ S0 + Mak V)
//   Y = R~ S0 + Mrb U + Mrk V                     (y = scale * Y)
//   S_L = diag(gamma_L) (S0 + B^^T U + K^^T V)
// which is the per-token recurrence
//   sa_t = S_{t-1}^T a_t, S_t = diag(w_t) S_{t-1} + b_t sa_t^T + k_t v_t^T,
//   y_t = scale * S_t^T r_t
// unrolled over the chunk.  Every product runs on
// v_mfma_f32_16x16x32_bf16 with both operands split into bf16 hi + lo
// (hi*hi + hi*lo + lo*hi, fp32 accumulation): fp32-level accuracy.  Raw bf16
// token values (V) are exact and carry no lo part.
//
// Work layout: one 512-thread workgroup per (sequence, head), walking the
// sequence in groups of G = 2 chunks, with two wave roles that run
// concurrently on the 4 SIMDs:
//   key waves (4-7), one (chunk, key half) each, prepare the operators of the
//     NEXT group: token rows loaded straight from HBM (prefetched one group
//     ahead), decays by a 16-lane DPP scan over tokens, operands built in
//     registers, the token-token blocks computed from those registers (each
//     lane's 8 keys are its own MFMA K positions); after the mid-iteration
//     barrier they store the operands for the state waves, and one of the two
//     waves of a chunk forms T by repeated squaring (I+M)(I+M^2)(I+M^4)(I+M^8)
//     (both orientations of every factor in registers);
//   state waves (0-3), state columns [16w, 16w+16) each, run the sequential
//     state path of the CURRENT group, one chunk per half-iteration.  The
//     state never leaves fp32 accumulator registers: accumulator rows are fed
//     to the matrix cores as B-operand K positions directly (the K order of a
//     dot product is free), and the accumulator layout of U is already the
//     B-operand layout of B^^T U.
// Operators are double-buffered in LDS by group parity; outputs are staged in
// LDS and written back as full 128-byte rows by the key waves.
#include "handoff.h"
#include "mfma.h"
#include "recurrent.h"

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstddef>
#include <type_traits>

namespace fr2 {
namespace {

constexpr int D = 64;
constexpr int L = 16;          // tokens per chunk
constexpr int G = 2;           // chunks per group
constexpr int GT = L * G;      // tokens per group
constexpr int NT = 512;        // 8 wavefronts: 4 state + 4 key
constexpr int MPP = L + 4;     // padded row of the partial token-token blocks
constexpr int YP = D + 8;      // padded row of the staged outputs
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kNegExpHalf = -0.6065306597126334f;   // -exp(-1/2)

// Operators of one chunk consumed by the state path.  For bf16 tokens V is
// exact in bf16 (no lo part); fp16 tokens need V's lo part.
//
// Every row array is addressed through the piece swizzles a_col, b_col and
// aop_piece (unswizzled, the same accesses cost ~430 bank-conflict cycles
// per chunk).
template <bool kVExact>
struct alignas(16) ChunkOps {
  static constexpr int RP = D;                      // key row length
  static constexpr int TP = D + 16;                 // token row of B^, K^, V
  float gl[D];                        // gamma_L (read as 16-byte vectors)
  __bf16 at_h[L][RP], at_l[L][RP];    // A~ rows, keys at key_pos()
  __bf16 r_h[L][RP], r_l[L][RP];      // R~ rows, keys at key_pos()
  __bf16 b_h[L][TP], b_l[L][TP];      // B^ rows (natural key order)
  __bf16 k_h[L][TP], k_l[L][TP];      // K^ rows
  __bf16 v_h[L][TP];                  // V rows
  __bf16 v_l[kVExact ? 1 : L][TP];    // V lo part (fp16 tokens only)
  // 16x16 token-token operators in A-operand form: row i, positions
  // 8q..8q+7 = (hi of columns 4q..4q+3, lo of columns 4q..4q+3)
  __bf16 t[L][2 * L];                 // T
  __bf16 mak[L][2 * L], mrb[L][2 * L], mrk[L][2 * L];   // masked Mak, Mrb, Mrk
};
// every 16-byte vector access above needs its array 16-byte aligned
static_assert(offsetof(ChunkOps<true>, at_h) % 16 == 0 && offsetof(ChunkOps<true>, t) % 16 == 0 &&
                  offsetof(ChunkOps<false>, t) % 16 == 0,
              "row arrays must be 16-byte aligned");
static_assert(sizeof(ChunkOps<true>) % 16 == 0 && sizeof(ChunkOps<false>) % 16 == 0,
              "operator blocks must keep 16-byte alignment");

template <bool kVExact>
struct alignas(16) Smem {
  ChunkOps<kVExact> ops[2][G];        // [group parity][chunk]
  // partial token-token blocks, transposed (mpart[..][s][t] = P[t][s]) with
  // rows padded to MPP floats so that both the 16-byte row accesses and the
  // strided column reads spread over the banks
  float mpart[2][G][2][4][L][MPP];    // [group parity][chunk][key half][block][s][t]
  uint16_t yb[2][GT][YP];             // outputs of a group, by parity (padded rows)
  // fused readout: sum over a key half of r k' r_k per token of a group, by
  // group index mod 4 (written by the key waves building group g after the
  // state waves finished g - 2, read by the write-back of group g, which the
  // state waves run after finishing g + 1)
  float rkv[4][2][GT];
  // progress counters, each written by one wave only: groups whose operators
  // key wave w has stored, groups whose part-1 partials it has stored, and
  // groups state wave w has finished / whose output rows it has written back
  int ready[4], part1[4], drained[4], consumed[4];
  int fault;                          // a bounded wait gave up
};

// Column position of key k in the A~ / R~ rows: for each half m = k/32 the 32
// keys are ordered so that lane group q of the state product reads its 8 keys
// (the rows its state accumulators hold) as one contiguous 16-byte run.
__device__ __forceinline__ int key_pos(int k) {
  const int m = k >> 5, kk = k & 31;
  return 32 * m + 8 * ((kk & 15) >> 2) + 4 * (kk >> 4) + (kk & 3);
}

// A operand against the state: row t = lane%16 of X; positions 8q+idx map to
// key (2m + idx/4)*16 + 4q + idx%4, i.e. the rows the lane's state
// accumulators hold.
template <int RP>
__device__ __forceinline__ Sp8 rows_vs_state(const __bf16 (*xh)[RP], const __bf16 (*xl)[RP],
                                             int m, int i, int q) {
  Sp8 s;
  s.hi = *reinterpret_cast<const bf16x8*>(&xh[i][a_col(i, 32 * m + 8 * q)]);
  s.lo = *reinterpret_cast<const bf16x8*>(&xl[i][a_col(i, 32 * m + 8 * q)]);
  return s;
}

__device__ __forceinline__ AOp load_aop(const __bf16 (*x)[2 * L], int i, int q) {
  return *reinterpret_cast<const AOp*>(&x[i][8 * aop_piece(i, q)]);
}
__device__ __forceinline__ void store_aop(__bf16 (*x)[2 * L], int i, int q, const AOp& v) {
  *reinterpret_cast<AOp*>(&x[i][8 * aop_piece(i, q)]) = v;
}

// ---------------------------------------------------------------------------
// key side, part 1: operands of chunk cc (keys 32hh + 8q + e of token i) and
// the partial token-token blocks over this lane's keys.  The operand values
// stay in registers until part 2 stores them for the state waves.
// ---------------------------------------------------------------------------
struct KeyRegs {
  Sp8 As, Rs, Bs, Ks, Vs;
};

// kFull: every token of the chunk is inside the sequence (no masking).
// nbias8 holds -log2(e) * decay_bias for the lane's keys.
// kUnitW: reverse mode, where unit_w marks a lane whose shifted retention
// row lies past the segment (unit retention).
// Per-lane channel parameters of the fused kk / a-gate stage: k_k for the
// lane's keys of both key halves (own first), a0 and k_a for its own keys.
struct KkParams {
  float kk_own[8], kk_other[8], a0[8], ka[8];
};

template <class Io, bool kVExact, bool kFull, bool kUnitW = false, bool kKK = false,
          bool kRO = false>
__device__ __forceinline__ void key_part1(Smem<kVExact>& sm, ChunkOps<kVExact>& op,
                                          const u32x4 (&raw)[6], const float (&nbias8)[8],
                                          bool valid, int mp, int cc, int hh, int i, int q,
                                          KeyRegs& kr, bool unit_w = false,
                                          float kscale = 1.0f, const KkParams* kp = nullptr,
                                          typename Io::raw* new_k_row = nullptr,
                                          const float* rk8 = nullptr, float* rkv_row = nullptr) {
  const int kbase = 32 * hh + 8 * q;
  // tokens past the sequence end (their rows repeat the last token) carry
  // zero operands and a unit retention
  const u32x4 zero4 = {0u, 0u, 0u, 0u};
  auto tok = [&](int j) { return (kFull || valid) ? raw[j] : zero4; };
  float xr[8], xl[8], xk[8], xa[8], xb[8];
  unpack8<Io>(tok(0), xr);
  unpack8<Io>(raw[1], xl);
  unpack8<Io>(tok(2), xk);
  if constexpr (kKK) {
    // Fused producer stage (the kk / a gate of wkv_prepare): raw[4] holds
    // the a-gate logits a12 and raw[5] the same 8 key positions of the other
    // key half, for the kk norm over all 64 keys:
    //   u = k k_k, kk = u / max(|u|, 1e-12), g = sigmoid(a0 + a12),
    //   k' = k (1 + (g - 1) k_a), a = -kk, b = kk g.
    float xo[8], x12[8];
    unpack8<Io>(tok(5), xo);
    unpack8<Io>(tok(4), x12);
    float u[8], ss = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      u[e] = xk[e] * kp->kk_own[e];
      const float w = xo[e] * kp->kk_other[e];
      ss = __builtin_fmaf(u[e], u[e], __builtin_fmaf(w, w, ss));
    }
    // the four lanes of token i (groups q = 0..3) hold all 64 keys
    ss += __shfl_xor(ss, 16);
    ss += __shfl_xor(ss, 32);
    const float inv = __builtin_amdgcn_rcpf(fmaxf(__builtin_sqrtf(ss), 1.0e-12f));
    float nk[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float g = __builtin_amdgcn_rcpf(
          1.0f + __builtin_amdgcn_exp2f(-kLog2e * (kp->a0[e] + x12[e])));
      const float kk = u[e] * inv;
      nk[e] = xk[e] * __builtin_fmaf(g - 1.0f, kp->ka[e], 1.0f);
      xa[e] = -kk;
      xb[e] = kk * g;
    }
    if (new_k_row != nullptr && (kFull || valid)) {
      u32x4 packed;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t lo = __builtin_bit_cast(uint16_t, Io::from_f32(nk[2 * j]));
        const uint32_t hi = __builtin_bit_cast(uint16_t, Io::from_f32(nk[2 * j + 1]));
        packed[j] = lo | (hi << 16);
      }
      *reinterpret_cast<u32x4*>(new_k_row) = packed;
    }
    // the recurrence uses the gated key (masked rows stay zero)
#pragma unroll
    for (int e = 0; e < 8; ++e) xk[e] = (kFull || valid) ? nk[e] : 0.0f;
  } else {
    unpack8<Io>(tok(4), xa);
    unpack8<Io>(tok(5), xb);
  }
  if constexpr (kRO) {
    // the readout's per-token residual weight over this lane's keys, summed
    // over the four lanes of the token: sum r k' r_k with k' as stored
    float part = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float kq = kKK ? Io::to_f32(Io::from_f32(xk[e])) : xk[e];
      part = __builtin_fmaf(xr[e] * kq, rk8[e], part);
    }
    part += __shfl_xor(part, 16);
    part += __shfl_xor(part, 32);
    if (q == 0) rkv_row[i] = part;
  }
  // base-2 log of the retention, log2(w) = c sigmoid(x) with
  // c = -exp(-1/2) log2(e), evaluated as 1 / ((1 + 2^(-log2(e) x)) / c)
  constexpr float kC = kNegExpHalf * kLog2e;
  constexpr float kInvC = 1.0f / kC;
  float at[8], rt[8], bh[8], kh[8];
  // Stage by stage over the lane's eight keys: the eight chains are
  // independent, so each stage's instructions (DPP steps included) issue
  // back to back instead of waiting on one key's dependent chain.
  float g2[8], gm[8], gp[8];
#pragma unroll
  for (int e = 0; e < 8; ++e)
    g2[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(xl[e], -kLog2e, nbias8[e]));
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    float lw2 = __builtin_amdgcn_rcpf(__builtin_fmaf(g2[e], kInvC, kInvC));
    if constexpr (!kFull) lw2 = valid ? lw2 : 0.0f;
    if constexpr (kUnitW) lw2 = unit_w ? 0.0f : lw2;
    g2[e] = lw2;
  }
  // inclusive prefix sum over the 16 tokens (the lanes of a DPP row)
#pragma unroll
  for (int e = 0; e < 8; ++e) g2[e] += row_shr<1>(g2[e]);
#pragma unroll
  for (int e = 0; e < 8; ++e) g2[e] += row_shr<2>(g2[e]);
#pragma unroll
  for (int e = 0; e < 8; ++e) g2[e] += row_shr<4>(g2[e]);
#pragma unroll
  for (int e = 0; e < 8; ++e) g2[e] += row_shr<8>(g2[e]);
#pragma unroll
  for (int e = 0; e < 8; ++e) gm[e] = __builtin_amdgcn_exp2f(g2[e]);      // gamma_t
#pragma unroll
  for (int e = 0; e < 8; ++e) gp[e] = row_prev(gm[e], 1.0f);              // gamma_{t-1}
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float ig = __builtin_amdgcn_exp2f(-g2[e]);                     // 1 / gamma_t
    at[e] = xa[e] * gp[e];
    rt[e] = xr[e] * gm[e];
    bh[e] = xb[e] * ig;
    kh[e] = xk[e] * ig;
    if constexpr (kUnitW) kh[e] *= kscale;   // reverse mode: k is r_t, times scale
  }
  if (i == L - 1) {
    *reinterpret_cast<f32x4*>(&op.gl[kbase]) = f32x4{gm[0], gm[1], gm[2], gm[3]};
    *reinterpret_cast<f32x4*>(&op.gl[kbase + 4]) = f32x4{gm[4], gm[5], gm[6], gm[7]};
  }
  kr.As = split8(at);
  kr.Rs = split8(rt);
  kr.Bs = split8(bh);
  kr.Ks = split8(kh);
  const u32x4 vraw = tok(3);
  if constexpr (kVExact) {
    kr.Vs.hi = __builtin_bit_cast(bf16x8, vraw);       // bf16 values are exact
  } else {
    float xv[8];
    unpack8<Io>(vraw, xv);
    kr.Vs = split8(xv);
  }
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  const f32x4 pab = mma32x3(kr.As, kr.Bs, zero);
  const f32x4 pak = mma32x3(kr.As, kr.Ks, zero);
  // lane (i, q) holds P[4q+e][i]: one 16-byte store per block
  *reinterpret_cast<f32x4*>(&sm.mpart[mp][cc][hh][0][i][4 * q]) = pab;
  *reinterpret_cast<f32x4*>(&sm.mpart[mp][cc][hh][1][i][4 * q]) = pak;
  const f32x4 prb = mma32x3(kr.Rs, kr.Bs, zero);
  const f32x4 prk = mma32x3(kr.Rs, kr.Ks, zero);
  *reinterpret_cast<f32x4*>(&sm.mpart[mp][cc][hh][2][i][4 * q]) = prb;
  *reinterpret_cast<f32x4*>(&sm.mpart[mp][cc][hh][3][i][4 * q]) = prk;
}

// ---------------------------------------------------------------------------
// key side, part 2: store the operands; the wave whose key half hh equals
// the group parity mp forms T, the other one the masked Mak, Mrb, Mrk (the
// T chain is the heavier role: alternating it spreads it over all four SIMDs)
// ---------------------------------------------------------------------------
template <bool kVExact>
__device__ __forceinline__ void key_part2(Smem<kVExact>& sm, ChunkOps<kVExact>& op, int mp,
                                          int cc, int hh, int i, int q, const KeyRegs& kr) {
  const int kbase = 32 * hh + 8 * q;
  {
    // keys kbase..kbase+7 land in two 4-key runs of the permuted rows
    const int p0 = key_pos(kbase), p1 = key_pos(kbase + 4);
    *reinterpret_cast<bf16x4*>(&op.r_h[i][a_col(i, p0)]) = kr.Rs.hi.lo;
    *reinterpret_cast<bf16x4*>(&op.r_h[i][a_col(i, p1)]) = kr.Rs.hi.hi;
    *reinterpret_cast<bf16x4*>(&op.r_l[i][a_col(i, p0)]) = kr.Rs.lo.lo;
    *reinterpret_cast<bf16x4*>(&op.r_l[i][a_col(i, p1)]) = kr.Rs.lo.hi;
    *reinterpret_cast<bf16x4*>(&op.at_h[i][a_col(i, p0)]) = kr.As.hi.lo;
    *reinterpret_cast<bf16x4*>(&op.at_h[i][a_col(i, p1)]) = kr.As.hi.hi;
    *reinterpret_cast<bf16x4*>(&op.at_l[i][a_col(i, p0)]) = kr.As.lo.lo;
    *reinterpret_cast<bf16x4*>(&op.at_l[i][a_col(i, p1)]) = kr.As.lo.hi;
  }
  *reinterpret_cast<bf16x8*>(&op.b_h[i][b_col(i, kbase)]) = kr.Bs.hi;
  *reinterpret_cast<bf16x8*>(&op.b_l[i][b_col(i, kbase)]) = kr.Bs.lo;
  *reinterpret_cast<bf16x8*>(&op.k_h[i][b_col(i, kbase)]) = kr.Ks.hi;
  *reinterpret_cast<bf16x8*>(&op.k_l[i][b_col(i, kbase)]) = kr.Ks.lo;
  *reinterpret_cast<bf16x8*>(&op.v_h[i][b_col(i, kbase)]) = kr.Vs.hi;
  if constexpr (!kVExact) *reinterpret_cast<bf16x8*>(&op.v_l[i][b_col(i, kbase)]) = kr.Vs.lo;
  // P[t][s] of block b, summed over the two key halves, is
  // mp0[0][b][s][t] + mp0[1][b][s][t]
  const float (*mp0)[4][L][MPP] = sm.mpart[mp][cc];
  if (hh == mp) {
    // M[e] = Mab[4q+e][i] (accumulator layout), Mt[e] = Mab[i][4q+e]
    const f32x4 m4 = *reinterpret_cast<const f32x4*>(&mp0[0][0][i][4 * q]) +
                     *reinterpret_cast<const f32x4*>(&mp0[1][0][i][4 * q]);
    f32x4 M, Mt;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int r = 4 * q + e;
      const float mt = mp0[0][0][r][i] + mp0[1][0][r][i];
      M[e] = (r > i) ? m4[e] : 0.f;
      Mt[e] = (i > r) ? mt : 0.f;
    }
    store_aop(op.t, i, q, t_inverse(M, Mt, i, q));
  } else {
    f32x4 mak, mrb, mrk;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int s = 4 * q + e;       // A-operand layout: row i, K = s
      const float v1 = mp0[0][1][s][i] + mp0[1][1][s][i];
      mak[e] = (i > s) ? v1 : 0.f;
      const float v2 = mp0[0][2][s][i] + mp0[1][2][s][i];
      const float v3 = mp0[0][3][s][i] + mp0[1][3][s][i];
      mrb[e] = (i >= s) ? v2 : 0.f;
      mrk[e] = (i >= s) ? v3 : 0.f;
    }
    store_aop(op.mak, i, q, as_a(split4(mak)));
    store_aop(op.mrb, i, q, as_a(split4(mrb)));
    store_aop(op.mrk, i, q, as_a(split4(mrk)));
  }
}

// ---------------------------------------------------------------------------
// state side: one chunk for the columns [16w, 16w+16) held in S.  The
// operand reads of a chunk are separate from its arithmetic so that the
// reads of the next chunk can be issued before this chunk's dependent chain.
// ---------------------------------------------------------------------------
template <bool kVExact>
struct StateOps {
  AOp Ta, Mak, Mrb, Mrk;
  bf16x4 vh, vl;
  Sp8 Aa0, Aa1, Ra0, Ra1;
  AOp Bt[4], Kt[4];
  f32x4 gl[4];
};

// operands the chain needs first: Mak, Mrk, V and the A~ / R~ rows
template <bool kVExact, bool kSum = false>
__device__ __forceinline__ void state_load_early(StateOps<kVExact>& o, const ChunkOps<kVExact>& op,
                                                 int vcol, int i, int q) {
  o.Mak = load_aop(op.mak, i, q);
  if constexpr (!kSum) o.Mrk = load_aop(op.mrk, i, q);
  // transposed operands straight from the token rows (see tr_rows)
  const int trow = 4 * q + (i >> 2), tcol = 4 * (i & 3);
  const int vc0 = 16 * (vcol >> 4) + tcol;
  o.vh = tr_rows(&op.v_h[trow][b_col(trow, vc0)]);                                   // V[4q+e][vcol]
  if constexpr (!kVExact) o.vl = tr_rows(&op.v_l[trow][b_col(trow, vc0)]);
  o.Aa0 = rows_vs_state(op.at_h, op.at_l, 0, i, q);
  o.Aa1 = rows_vs_state(op.at_h, op.at_l, 1, i, q);
  if constexpr (!kSum) {
    o.Ra0 = rows_vs_state(op.r_h, op.r_l, 0, i, q);
    o.Ra1 = rows_vs_state(op.r_h, op.r_l, 1, i, q);
  }
}
// the rest: T, Mrb, B^^T, K^^T and gamma_L
template <bool kVExact, bool kSum = false>
__device__ __forceinline__ void state_load_late(StateOps<kVExact>& o, const ChunkOps<kVExact>& op,
                                                int vcol, int i, int q) {
  (void)vcol;
  o.Ta = load_aop(op.t, i, q);
  if constexpr (!kSum) o.Mrb = load_aop(op.mrb, i, q);
  const int trow = 4 * q + (i >> 2), tcol = 4 * (i & 3);
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) {
    // B^^T, K^^T as A operands: row 16kb+i, K = token
    o.Bt[kb] = __builtin_shufflevector(tr_rows(&op.b_h[trow][b_col(trow, kb * 16 + tcol)]),
                                       tr_rows(&op.b_l[trow][b_col(trow, kb * 16 + tcol)]), 0, 1, 2, 3, 4,
                                       5, 6, 7);
    o.Kt[kb] = __builtin_shufflevector(tr_rows(&op.k_h[trow][b_col(trow, kb * 16 + tcol)]),
                                       tr_rows(&op.k_l[trow][b_col(trow, kb * 16 + tcol)]), 0, 1, 2, 3, 4,
                                       5, 6, 7);
    o.gl[kb] = *reinterpret_cast<const f32x4*>(&op.gl[kb * 16 + 4 * q]);
  }
}
template <bool kVExact, bool kSum = false>
__device__ __forceinline__ StateOps<kVExact> state_load(const ChunkOps<kVExact>& op, int vcol,
                                                        int i, int q) {
  StateOps<kVExact> o;
  state_load_early<kVExact, kSum>(o, op, vcol, i, q);
  state_load_late<kVExact, kSum>(o, op, vcol, i, q);
  return o;
}

// Where the sa rows 4q+e (e = 0..3) of a chunk go: row row0 + dir*e of the
// column pointer col (rows of row_stride floats), except that e = 0 goes to
// row `wrap` when wrap >= 0 (the reverse mode's position 0).  Kept as a few
// integers and formed at the store, so that no per-row pointers stay live
// across the chain.
struct SaRows {
  float* col = nullptr;
  int64_t row_stride = 0;
  int row0 = 0, dir = 1, wrap = -1;
  __device__ __forceinline__ float* at(int e) const {
    const int row = (e == 0 && wrap >= 0) ? wrap : row0 + dir * e;
    return col + static_cast<int64_t>(row) * row_stride;
  }
};

// With kTrain the chunk also writes its per-token sa rows (U, fp32) of tokens
// 4q..4q+3 to sa_rows.at(0..3) and, when bnd_col is set, its post-chunk state
// column to bnd_col[key * D].
// kKeep: writes nothing and leaves U and the scaled outputs of those tokens in
// uy[0] and uy[1].
// kSum (summary pass): the state update only, no outputs; with no_v the
// value rows count as zero (the transition of the chunk).
constexpr int UP = D + 4;   // padded row of a staged sa tile (fp32)
template <class Io, bool kVExact, bool kTrain = false, bool kSum = false, bool kKeep = false>
__device__ __forceinline__ void state_compute(const StateOps<kVExact>& o, f32x4 (&S)[4],
                                              uint16_t (*yrows)[YP], int vcol, int i, int q,
                                              float scale, const SaRows& sa_rows = SaRows{},
                                              float* bnd_col = nullptr, bool no_v = false,
                                              f32x4* uy = nullptr) {
  using raw = typename Io::raw;
  // S split as B operand against the permuted A~ / R~ rows: K positions
  // 8q..8q+7 = rows 32m + 4q + (0..3) then 32m + 16 + 4q + (0..3)
  Sp8 Sb[2];
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    const Split4 a = split4(S[2 * m]), b = split4(S[2 * m + 1]);
    Sb[m].hi = __builtin_bit_cast(bf16x8, u32x4{a.h0, a.h1, b.h0, b.h1});
    Sb[m].lo = __builtin_bit_cast(bf16x8, u32x4{a.l0, a.l1, b.l0, b.l1});
  }
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  // X = A~ S0 + Mak V,  U = T X,  Y = R~ S0 + Mrb U + Mrk V
  f32x4 X, Y;
  auto tokens_out = [&](const f32x4& u, const f32x4& y) {
    if constexpr (kKeep) {
      uy[0] = u;
      uy[1] = scale * y;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if constexpr (kTrain) *sa_rows.at(e) = u[e];
        yrows[4 * q + e][vcol] = __builtin_bit_cast(uint16_t, Io::from_f32(scale * y[e]));
      }
    }
  };
  if constexpr (kSum) {
    // X = A~ S0 + Mak V, U = T X, S_L = diag(gamma_L) (S0 + B^^T U + K^^T V)
    (void)yrows; (void)scale; (void)Y; (void)tokens_out;
    // A x V for the token-indexed A operand (exact bf16 V: one instruction)
    auto times_v = [&](AOp a, f32x4 c) {
      if (no_v) return c;
      if constexpr (kVExact) return mm_ax(a, as_bx(o.vh), c);
      else return mm_ab(a, as_b(o.vh, o.vl), c);
    };
    X = times_v(o.Mak, zero);
    X = mma32x3(o.Aa0, Sb[0], X);
    X = mma32x3(o.Aa1, Sb[1], X);
    const BOp Us = as_b(split4(mm_ab(o.Ta, as_b(split4(X)), zero)));
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      f32x4 acc = mm_ab(o.Bt[kb], Us, S[kb]);
      acc = times_v(o.Kt[kb], acc);
      S[kb] = acc * o.gl[kb];
    }
  } else if constexpr (kVExact) {
    const BX Vx = as_bx(o.vh);
    X = mm_ax(o.Mak, Vx, zero);
    Y = mm_ax(o.Mrk, Vx, zero);
    X = mma32x3(o.Aa0, Sb[0], X);
    X = mma32x3(o.Aa1, Sb[1], X);
    Y = mma32x3(o.Ra0, Sb[0], Y);
    Y = mma32x3(o.Ra1, Sb[1], Y);
    const f32x4 Uf = mm_ab(o.Ta, as_b(split4(X)), zero);
    const BOp Us = as_b(split4(Uf));
    Y = mm_ab(o.Mrb, Us, Y);
    tokens_out(Uf, Y);
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      f32x4 acc = mm_ab(o.Bt[kb], Us, S[kb]);
      acc = mm_ax(o.Kt[kb], Vx, acc);
      S[kb] = acc * o.gl[kb];
      if constexpr (kTrain) {
        // (column stores: a quad transpose to row pieces, on these state
        // waves' chain, measured 0.683 vs 0.662 ms for the forward)
        if (bnd_col != nullptr) {
#pragma unroll
          for (int e = 0; e < 4; ++e) bnd_col[(16 * kb + 4 * q + e) * D] = S[kb][e];
        }
      }
    }
  } else {
    const BOp Vs = as_b(o.vh, o.vl);
    X = mm_ab(o.Mak, Vs, zero);
    Y = mm_ab(o.Mrk, Vs, zero);
    X = mma32x3(o.Aa0, Sb[0], X);
    X = mma32x3(o.Aa1, Sb[1], X);
    Y = mma32x3(o.Ra0, Sb[0], Y);
    Y = mma32x3(o.Ra1, Sb[1], Y);
    const f32x4 Uf = mm_ab(o.Ta, as_b(split4(X)), zero);
    const BOp Us = as_b(split4(Uf));
    Y = mm_ab(o.Mrb, Us, Y);
    tokens_out(Uf, Y);
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      f32x4 acc = mm_ab(o.Bt[kb], Us, S[kb]);
      acc = mm_ab(o.Kt[kb], Vs, acc);
      S[kb] = acc * o.gl[kb];
      if constexpr (kTrain) {
        // (column stores: a quad transpose to row pieces, on these state
        // waves' chain, measured 0.683 vs 0.662 ms for the forward)
        if (bnd_col != nullptr) {
#pragma unroll
          for (int e = 0; e < 4; ++e) bnd_col[(16 * kb + 4 * q + e) * D] = S[kb][e];
        }
      }
    }
  }
}

// Fused readout write-back of group gi (the state waves run it one group
// late, in place of the plain y write-back): thread (o_tok, o_c8) takes 8
// channels of token o_tok of the group's staged y rows.  GroupNorm over the
// head's 64 channels (the 8 consecutive lanes of a token hold 8 channels
// each), the r k' r_k residual whose two key-half sums the key waves left in
// sm.rkv, and the gate:
//   out = (GroupNorm(y) * ln_w + ln_b + (sum r k' r_k) v) * g.
template <class Io, bool kVExact>
__device__ __forceinline__ void readout_write_back(const Smem<kVExact>& sm, const SegArgs& p,
                                                   int gi, int o_tok, int o_c8, int t0,
                                                   int seg_len, int64_t row_stride,
                                                   int64_t head_off) {
  using raw = typename Io::raw;
  // this thread's 8 channels of ln_w / ln_b (read here rather than held in
  // registers across the key waves' loop)
  float ro_w[8], ro_b[8];
  unpack8<Io>(*reinterpret_cast<const u32x4*>(static_cast<const raw*>(p.ro_lnw) + head_off +
                                              o_c8 * 8), ro_w);
  unpack8<Io>(*reinterpret_cast<const u32x4*>(static_cast<const raw*>(p.ro_lnb) + head_off +
                                              o_c8 * 8), ro_b);
  const int pos = gi * GT + o_tok;   // position in the segment
  const bool in_seg = pos < seg_len;
  const int64_t roff =
      static_cast<int64_t>(t0 + min(pos, seg_len - 1)) * row_stride + head_off + o_c8 * 8;
  const u32x4 ypiece = *reinterpret_cast<const u32x4*>(&sm.yb[gi & 1][o_tok][o_c8 * 8]);
  const u32x4 vraw = *reinterpret_cast<const u32x4*>(static_cast<const raw*>(p.v) + roff);
  const u32x4 graw = *reinterpret_cast<const u32x4*>(static_cast<const raw*>(p.ro_g) + roff);
  float yv[8], vv[8], gv[8];
  unpack8<Io>(ypiece, yv);
  unpack8<Io>(vraw, vv);
  unpack8<Io>(graw, gv);
  float s1 = 0.0f;
#pragma unroll
  for (int e = 0; e < 8; ++e) s1 += yv[e];
  s1 += __shfl_xor(s1, 1);
  s1 += __shfl_xor(s1, 2);
  s1 += __shfl_xor(s1, 4);
  const float mean = s1 * (1.0f / D);
  float s2 = 0.0f;
#pragma unroll
  for (int e = 0; e < 8; ++e) s2 = __builtin_fmaf(yv[e] - mean, yv[e] - mean, s2);
  s2 += __shfl_xor(s2, 1);
  s2 += __shfl_xor(s2, 2);
  s2 += __shfl_xor(s2, 4);
  const float inv = 1.0f / __builtin_sqrtf(s2 * (1.0f / D) + 64.0e-5f);
  const float rkv = sm.rkv[gi & 3][0][o_tok] + sm.rkv[gi & 3][1][o_tok];
  u32x4 packed;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    float o2[2];
#pragma unroll
    for (int h2 = 0; h2 < 2; ++h2) {
      const int e = 2 * j + h2;
      o2[h2] = (__builtin_fmaf((yv[e] - mean) * inv, ro_w[e], ro_b[e]) + rkv * vv[e]) * gv[e];
    }
    packed[j] = static_cast<uint32_t>(__builtin_bit_cast(uint16_t, Io::from_f32(o2[0]))) |
                (static_cast<uint32_t>(__builtin_bit_cast(uint16_t, Io::from_f32(o2[1]))) << 16);
  }
  if (in_seg) {
    *reinterpret_cast<u32x4*>(static_cast<raw*>(p.ro_out) + roff) = packed;
    if (p.y != nullptr) *reinterpret_cast<u32x4*>(static_cast<raw*>(p.y) + roff) = ypiece;
  }
}

// kTrain: the training-forward contract (pretrain path) also writes every
// token's sa (p.sa_out) and the post-chunk state of every 16-token chunk
// (p.boundary, [segment, H, boundary_per_seg, D, D]).
template <class Io, bool kTrain, bool kRev = false, bool kKK = false, bool kRO = false>
__global__ __launch_bounds__(NT) void chunk64_kernel(SegArgs p) {
  using raw = typename Io::raw;
  constexpr bool kVExact = !__is_same(Io, IoF16);
  __shared__ Smem<kVExact> sm;

  const int h = blockIdx.x;
  const int seg = blockIdx.y;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  // wave index as a scalar: the role branches below are uniform per wave, so
  // each wave runs only its own role's code (no exec-masked pass through the
  // other role, whose matrix instructions would run regardless of exec)
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i = lane & 15;
  const int q = lane >> 4;
  const int H = p.num_heads;

  if (p.status != nullptr) {
    if (p.status[0] != 0) {
      const int64_t blk = static_cast<int64_t>(seg) * gridDim.x + h;
      const int64_t nblk = static_cast<int64_t>(gridDim.x) * gridDim.y;
      if (!kRO || p.y != nullptr)
        fill_output_nan<Io>(static_cast<raw*>(p.y), p.out_elems, blk, nblk);
      if constexpr (kRO)
        fill_output_nan<Io>(static_cast<raw*>(p.ro_out), p.out_elems, blk, nblk);
      return;
    }
    if (seg >= p.status[2]) return;
  }
  int t0, t1;
  if (p.uniform_len > 0) {
    t0 = seg * p.uniform_len;
    t1 = t0 + p.uniform_len;
  } else if (p.chunk_offsets != nullptr) {
    t0 = p.bounds[p.chunk_offsets[seg]];
    t1 = p.ends[p.chunk_offsets[seg + 1] - 1];
  } else if (p.ends != nullptr) {
    t0 = p.bounds[seg];
    t1 = p.ends[seg];
  } else {
    t0 = p.bounds[seg];
    t1 = p.bounds[seg + 1];
  }
  const int slot = p.slots ? p.slots[seg] : seg;
  const int64_t head_off = static_cast<int64_t>(h) * D;
  const int64_t row_stride = static_cast<int64_t>(H) * D;
  const int ngroups = (t1 - t0 + GT - 1) / GT;
  raw* yout = static_cast<raw*>(p.y);

  if (tid < 17) (&sm.ready[0])[tid] = 0;
  __syncthreads();   // the only workgroup barrier: counters are zero

  // state waves: columns [16wv, 16wv+16)
  const int vcol = 16 * (wv & 3) + i;
  const int64_t sbase = (static_cast<int64_t>(slot) * H + h) * D * D;
  constexpr int kStateThreads = 256;
  if (wv < 4) {
    f32x4 S[4];
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) S[kb] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (p.state_in != nullptr && p.state_bf16) {
      // (bf16-state contract) bf16 widened once; the state stays fp32 for
      // the whole call and is rounded back once at the end.  One branch
      // around each loop: a per-element select compiles to a branch and a
      // wait per load.
      const uint16_t* sinb = static_cast<const uint16_t*>(p.state_in) + sbase + vcol;
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int e = 0; e < 4; ++e) S[kb][e] = IoBF16::to_f32(sinb[(kb * 16 + 4 * q + e) * D]);
    } else if (p.state_in != nullptr) {
      const float* sin = static_cast<const float*>(p.state_in) + sbase + vcol;
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int e = 0; e < 4; ++e) S[kb][e] = sin[(kb * 16 + 4 * q + e) * D];
    }
    // outputs of a finished group: 16-byte pieces of the staged rows, token
    // tid/8, elements 8*(tid%8).. (the four state waves cover the 32 rows)
    const int o_tok = tid >> 3, o_c8 = tid & 7;
    const int seg_len = t1 - t0;
    auto write_out = [&](int gi) {
      if (gi < 0) return;
      wait_min_ge(sm.consumed, gi + 1, p.spin_limit, &sm.fault);   // every state wave staged its columns
      const int pos = gi * GT + o_tok;        // position in processing order
      if constexpr (kRO) {
        readout_write_back<Io, kVExact>(sm, p, gi, o_tok, o_c8, t0, seg_len, row_stride,
                                        head_off);
      } else if (pos < seg_len) {
        const int row = kRev ? t1 - 1 - pos : t0 + pos;
        *reinterpret_cast<u32x4*>(yout + static_cast<int64_t>(row) * row_stride + head_off +
                                  o_c8 * 8) =
            *reinterpret_cast<const u32x4*>(&sm.yb[gi & 1][o_tok][o_c8 * 8]);
      }
      signal(&sm.drained[wv], gi + 1);
    };
    // training outputs: sa column of this lane and the boundary column
    float* const sa_base = kTrain ? p.sa_out + head_off + vcol : nullptr;
    const int nsnap = (p.boundary_per_seg + p.boundary_every - 1) / p.boundary_every;
    float* const bnd_base =
        (kTrain && p.boundary != nullptr)
            ? p.boundary + (static_cast<int64_t>(seg) * H + h) * nsnap * D * D + vcol
            : nullptr;
    auto chunk = [&](const StateOps<kVExact>& o, int gi, int c) {
      const int ci = gi * G + c;   // chunk index within the segment
      SaRows sa_rows;
      if constexpr (kTrain) {
        // forward: rows t0 + pos; reverse: t0 + (n - pos) mod n, which is
        // t1 - pos except at pos = 0
        const int pos0 = ci * L + 4 * q;
        sa_rows.col = sa_base;
        sa_rows.row_stride = row_stride;
        sa_rows.row0 = kRev ? t1 - pos0 : t0 + pos0;
        sa_rows.dir = kRev ? -1 : 1;
        sa_rows.wrap = (kRev && pos0 == 0) ? t0 : -1;
      }
      const int bi = kRev ? p.boundary_per_seg - 1 - ci : ci;
      const bool keep = bnd_base != nullptr && bi % p.boundary_every == 0;
      state_compute<Io, kVExact, kTrain>(
          o, S, &sm.yb[gi & 1][c * L], vcol, i, q, p.scale, sa_rows,
          keep ? bnd_base + static_cast<int64_t>(bi / p.boundary_every) * D * D : nullptr);
    };
    auto group = [&](auto par_c, int gi) {
      constexpr int par = decltype(par_c)::value;
      wait_min_ge(sm.ready, gi + 1, p.spin_limit, &sm.fault);   // operators of group gi stored
      wait_min_ge(sm.drained, gi - 1, p.spin_limit, &sm.fault);   // outputs of group gi-2 written back
      if (!kTrain && t0 + gi * GT + GT <= t1) {
        // both chunks: the second chunk's first-needed operand reads (the
        // S-side rows and V-side blocks) go out before the first chunk's chain
        // (not in training mode, whose extra outputs would then spill)
        const StateOps<kVExact> o0 = state_load(sm.ops[par][0], vcol, i, q);
        StateOps<kVExact> o1;
        state_load_early(o1, sm.ops[par][1], vcol, i, q);
        chunk(o0, gi, 0);
        state_load_late(o1, sm.ops[par][1], vcol, i, q);
        chunk(o1, gi, 1);
      } else {
        chunk(state_load(sm.ops[par][0], vcol, i, q), gi, 0);
        if (t0 + gi * GT + L < t1) chunk(state_load(sm.ops[par][1], vcol, i, q), gi, 1);
      }
      signal(&sm.consumed[wv], gi + 1);
      write_out(gi - 1);
    };
    for (int gi = 0; gi < ngroups; gi += 2) {
      group(std::integral_constant<int, 0>{}, gi);
      if (gi + 1 < ngroups) group(std::integral_constant<int, 1>{}, gi + 1);
    }
    write_out(ngroups - 1);
    // Every wave has left its loop (the key waves meet this barrier at the
    // end of their branch); a raised fault flag means a hand-off wait gave
    // up, so the values computed are not trustworthy: fail closed.
    __syncthreads();
    if (peek(&sm.fault) != 0) {
      if (tid == 0 && p.handoff_fault != nullptr) atomicAdd(p.handoff_fault, 1);
      const float qnan = quiet_nan();
      const raw nanv = Io::from_f32(qnan);
      if (yout != nullptr)
        for (int64_t e = tid; e < static_cast<int64_t>(t1 - t0) * D; e += kStateThreads)
          yout[(t0 + e / D) * row_stride + head_off + e % D] = nanv;
      if constexpr (kRO)
        for (int64_t e = tid; e < static_cast<int64_t>(t1 - t0) * D; e += kStateThreads)
          static_cast<raw*>(p.ro_out)[(t0 + e / D) * row_stride + head_off + e % D] = nanv;
      if constexpr (kTrain) {
        for (int64_t e = tid; e < static_cast<int64_t>(t1 - t0) * D; e += kStateThreads)
          p.sa_out[(t0 + e / D) * row_stride + head_off + e % D] = qnan;
      }
      return;
    }
    if (p.state_out != nullptr && p.state_bf16) {
      uint16_t* soutb = static_cast<uint16_t*>(p.state_out) + sbase + vcol;
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          soutb[(kb * 16 + 4 * q + e) * D] = IoBF16::from_f32(S[kb][e]);
    } else if (p.state_out != nullptr) {
      float* sout = static_cast<float*>(p.state_out) + sbase + vcol;
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int e = 0; e < 4; ++e) sout[(kb * 16 + 4 * q + e) * D] = S[kb][e];
    }
  } else {
    // ---------------- key waves: chunk cc of each group, key half hh
    // The key waves are the pipeline's critical path and share each SIMD
    // with a state wave that has slack: let them win instruction issue.
    __builtin_amdgcn_s_setprio(2);
    const int kw = wv & 3;
    const int cc = kw >> 1;
    const int hh = kw & 1;
    const int partner = kw ^ 1;
    const int kbase = 32 * hh + 8 * q;
    float nbias8[8];
#pragma unroll
    for (int e = 0; e < 8; ++e)
      nbias8[e] = p.bias ? -kLog2e * Io::to_f32(static_cast<const raw*>(p.bias)[head_off + kbase + e])
                         : 0.f;
    const int kbase_other = 32 * (hh ^ 1) + 8 * q;
    float rk8[8];
    if constexpr (kRO) {
      const raw* rk = static_cast<const raw*>(p.ro_rk) + head_off + kbase;
#pragma unroll
      for (int e = 0; e < 8; ++e) rk8[e] = Io::to_f32(rk[e]);
    }
    KkParams kp;
    if constexpr (kKK) {
      const raw* kks = static_cast<const raw*>(p.kk_scale) + head_off;
      const raw* a0 = static_cast<const raw*>(p.a_bias) + head_off;
      const raw* ka = static_cast<const raw*>(p.k_a) + head_off;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        kp.kk_own[e] = Io::to_f32(kks[kbase + e]);
        kp.kk_other[e] = Io::to_f32(kks[kbase_other + e]);
        kp.a0[e] = Io::to_f32(a0[kbase + e]);
        kp.ka[e] = Io::to_f32(ka[kbase + e]);
      }
    }
    // token rows of this lane (token i of chunk cc, keys kbase..+7), as
    // running pointers; the group stride is GT rows
    const int tok0 = t0 + cc * L + i;
    const raw* src[6];
    {
      const int64_t off = static_cast<int64_t>(kRev ? 0 : tok0) * row_stride + head_off + kbase;
      src[0] = static_cast<const raw*>(p.r) + off;
      src[1] = static_cast<const raw*>(p.logits) + off;
      src[2] = static_cast<const raw*>(p.k) + off;
      src[3] = static_cast<const raw*>(p.v) + off;
      src[4] = static_cast<const raw*>(p.a) + off;
      // fused kk / a gate: slot 5 reads the key's other half instead of b
      src[5] = kKK ? static_cast<const raw*>(p.k) + off + (kbase_other - kbase)
                   : static_cast<const raw*>(p.b) + off;
    }
    const int64_t gstride = static_cast<int64_t>(GT) * row_stride;
    // Rows past the sequence end are loaded from the last valid row (always
    // in bounds); key_part1 zeroes them when it consumes them.  A conditional
    // load would compile to a branch whose zeroing path waits for every
    // outstanding memory operation, the previous group's output stores
    // included, and a select right here would wait for the loads themselves.
    auto load_rows = [&](u32x4 (&dst)[6], int gi) {
      if constexpr (kRev) {
        const int pos = cc * L + i + gi * GT;   // position in processing order
#pragma unroll
        for (int j = 0; j < 6; ++j) {
          const int row = min(max(t1 - 1 - pos + ((p.shift_mask >> j) & 1), t0), t1 - 1);
          dst[j] = __builtin_nontemporal_load(
              reinterpret_cast<const u32x4*>(src[j] + static_cast<int64_t>(row) * row_stride));
        }
      } else {
        const int tok = tok0 + gi * GT;
        const int64_t off = static_cast<int64_t>(min(tok, t1 - 1) - tok0) * row_stride;
#pragma unroll
        for (int j = 0; j < 6; ++j)
          dst[j] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(src[j] + off));
      }
    };
    u32x4 rawA[6], rawB[6];
    KeyRegs kr;
    load_rows(rawA, 0);
    // group gn: prefetch the rows of gn + 1, wait until the state waves are
    // done with group gn - 2 (whose operator buffers gn reuses), then build
    // the operators of gn
    auto iter = [&](auto par_c, u32x4 (&cur)[6], u32x4 (&nxt)[6], int gn) {
      constexpr int par = decltype(par_c)::value;   // parity of gn
      if (gn + 1 < ngroups) load_rows(nxt, gn + 1);
      wait_min_ge(sm.consumed, gn - 1, p.spin_limit, &sm.fault);   // group gn-2 no longer read
      const bool active = t0 + gn * GT + cc * L < t1;
      if constexpr (kRev) {
        // position 0 of the segment: the shifted rows lie past its end
        const bool void_row = gn == 0 && cc == 0 && i == 0;
        u32x4 rows[6];
#pragma unroll
        for (int j = 0; j < 6; ++j) {
          const bool z = void_row && ((p.shift_mask >> j) & 1) && j != 1;
          rows[j] = z ? u32x4{0u, 0u, 0u, 0u} : cur[j];
        }
        const bool unit_w = void_row && ((p.shift_mask >> 1) & 1);
        if (t0 + gn * GT + cc * L + L <= t1)
          key_part1<Io, kVExact, true, true>(sm, sm.ops[par][cc], rows, nbias8, true, par, cc,
                                             hh, i, q, kr, unit_w, p.kv_scale);
        else if (active)
          key_part1<Io, kVExact, false, true>(sm, sm.ops[par][cc], rows, nbias8,
                                              t0 + gn * GT + cc * L + i < t1, par, cc, hh, i, q,
                                              kr, unit_w, p.kv_scale);
      } else {
        raw* nk_row = nullptr;
        if constexpr (kKK)
          nk_row = static_cast<raw*>(p.new_k) +
                   static_cast<int64_t>(tok0 + gn * GT) * row_stride + head_off + kbase;
        if (t0 + gn * GT + cc * L + L <= t1)
          key_part1<Io, kVExact, true, false, kKK, kRO>(
              sm, sm.ops[par][cc], cur, nbias8, true, par, cc, hh, i, q, kr, false, 1.0f, &kp,
              nk_row, rk8, &sm.rkv[gn & 3][hh][cc * L]);
        else if (active)
          key_part1<Io, kVExact, false, false, kKK, kRO>(
              sm, sm.ops[par][cc], cur, nbias8, tok0 + gn * GT < t1, par, cc, hh, i, q, kr, false,
              1.0f, &kp, nk_row, rk8, &sm.rkv[gn & 3][hh][cc * L]);
      }
      signal(&sm.part1[kw], gn + 1);
      wait_ge(&sm.part1[partner], gn + 1, p.spin_limit, &sm.fault);
      if (active) key_part2<kVExact>(sm, sm.ops[par][cc], par, cc, hh, i, q, kr);
      if (p.handoff_stall != 1) signal(&sm.ready[kw], gn + 1);
    };
    for (int gn = 0; gn < ngroups; gn += 2) {
      iter(std::integral_constant<int, 0>{}, rawA, rawB, gn);
      if (gn + 1 < ngroups) iter(std::integral_constant<int, 1>{}, rawB, rawA, gn + 1);
    }
    __builtin_amdgcn_s_setprio(0);
    __syncthreads();   // pairs with the state waves' final barrier
  }

}


// ===========================================================================
// Ring variant of the workgroup-per-unit kernel (plain inference contract).
// Each key wave builds WHOLE chunks: key wave w (4..7) takes chunks
// w - 4, w, w + 4, ... of the unit, both key halves one after the other,
// accumulating the token-token blocks over all 64 keys in its own matrix
// accumulators, then forms T and the masked blocks itself.  So no partial
// blocks go through LDS and no key wave waits on a partner.  Operator blocks
// are a ring of R chunks in LDS (chunk c in slot c % R; R = 6 for bf16
// tokens, 5 for fp16), and a key wave may build chunk c as soon as the state
// waves have finished chunk c - R.  A key wave takes about three chunk
// periods to build a chunk, so with R = 4 the state waves waited on the
// ring; with R = 6 the four key waves' throughput sets the period.  The
// state waves run chunk after chunk as in chunk64_kernel.  In inference each
// writes its own 16 output columns, so they never wait on one another; in
// training, whose outputs are ten times the bytes, they leave them in LDS for
// the key waves to write (ChunkOut), which takes one slot of the ring's depth.
// ===========================================================================
// operator slots of the ring kernel (fp16 tokens carry V's lo part and
// fit one slot fewer in the 160 KB of LDS)
template <bool kVExact> constexpr int kRingOf = kVExact ? 6 : 5;
constexpr int kKeyW = 4;   // key waves of the ring kernel
constexpr int NTR = 64 * (4 + kKeyW);
template <bool kVExact>
struct alignas(16) SmemR {
  ChunkOps<kVExact> ops[kRingOf<kVExact>];   // ring by chunk index mod kRing
  uint16_t yb[L][YP];                 // staged output rows of the current chunk
  // progress counters, each written by one wave only: chunks key wave w has
  // built (its chunks are w, w + kKeyW, ...) and chunks state wave w has
  // finished
  int ready[kKeyW], consumed[4];
  int fault;
  int lost;                           // the start state came from a block that failed
};

// A chunk's outputs on their way to memory: the post-chunk state, sa and y, each
// row padded against bank conflicts (the state waves write columns, the key waves
// read 16-byte row pieces).  Chunk c's lie in the operator slot of chunk c - 1,
// between the state waves finishing that chunk and a key wave building chunk
// c - 1 + kRing there.
struct alignas(16) ChunkOut {
  float s[D][UP];
  float u[L][UP];
  uint16_t y[L][YP];
};
static_assert(sizeof(ChunkOut) <= sizeof(ChunkOps<true>) &&
                  sizeof(ChunkOut) <= sizeof(ChunkOps<false>),
              "a chunk's outputs fit an operator slot");
template <bool kVExact>
__device__ __forceinline__ ChunkOut& chunk_out(SmemR<kVExact>& sm, int c) {
  constexpr int kRing = kRingOf<kVExact>;
  return *reinterpret_cast<ChunkOut*>(&sm.ops[(c + kRing - 1) % kRing]);
}

// Token-token products of the whole chunk, accumulated over both key halves:
// ab = Mab in accumulator layout (item e: Mab[4q+e][i]); abt, ak, rb, rk in
// A-operand layout (item e: X[i][4q+e]).
struct KeyAccR {
  f32x4 ab, abt, ak, rb, rk;
};

// One key half hh of chunk operators: as key_part1 (plain contract) plus the
// operand-row stores of key_part2, with the token-token products accumulated.
// kSum (summary pass): no R~ operand, no R-side products.
// Per-lane channel parameters of the fused kk / a-gate stage for the lane's
// eight keys of one key half: the kk scale, the a-gate bias a0 and k_a.
struct KkHalf {
  float kks[8], a0[8], ka[8];
};

// kKK (fused kk / a-gate stage): slot 4 of raw holds the a-gate logits a12,
// slot 5 is unused; kinv = 1 / max(|k k_k|, 1e-12) over the token's 64 keys;
// the gated key k' is stored to nk_row (when the token is in the segment):
//   kk = k k_k kinv, g = sigmoid(a0 + a12), k' = k (1 + (g - 1) k_a),
//   a = -kk, b = kk g.
// kRev (the training backward's value pass): unit_w marks a lane whose
// shifted retention row lies past the segment (unit retention), and K^ is
// scaled by kscale (k is r_t there, times the output scale).
template <class Io, bool kVExact, bool kFull, bool kSum = false, bool kKK = false,
          bool kRev = false>
__device__ __forceinline__ void key_half_ring(ChunkOps<kVExact>& op, const u32x4 (&raw)[6],
                                              const float (&nbias8)[8], bool valid, int hh,
                                              int i, int q, KeyAccR& acc,
                                              const KkHalf* kp = nullptr, float kinv = 0.0f,
                                              typename Io::raw* nk_row = nullptr,
                                              bool unit_w = false, float kscale = 1.0f) {
  const int kbase = 32 * hh + 8 * q;
  const u32x4 zero4 = {0u, 0u, 0u, 0u};
  auto tok = [&](int j) { return (kFull || valid) ? raw[j] : zero4; };
  float xr[8], xl[8], xk[8], xa[8], xb[8];
  if constexpr (!kSum) unpack8<Io>(tok(0), xr);
  unpack8<Io>(raw[1], xl);
  unpack8<Io>(tok(2), xk);
  if constexpr (kKK) {
    float x12[8], nk[8];
    unpack8<Io>(tok(4), x12);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float kk = xk[e] * kp->kks[e] * kinv;
      const float g = __builtin_amdgcn_rcpf(
          1.0f + __builtin_amdgcn_exp2f(-kLog2e * (kp->a0[e] + x12[e])));
      nk[e] = xk[e] * __builtin_fmaf(g - 1.0f, kp->ka[e], 1.0f);
      xa[e] = -kk;
      xb[e] = kk * g;
    }
    if (nk_row != nullptr && (kFull || valid)) {
      u32x4 packed;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t lo = __builtin_bit_cast(uint16_t, Io::from_f32(nk[2 * j]));
        const uint32_t hi = __builtin_bit_cast(uint16_t, Io::from_f32(nk[2 * j + 1]));
        packed[j] = lo | (hi << 16);
      }
      *reinterpret_cast<u32x4*>(nk_row + kbase) = packed;
    }
    // the recurrence uses the gated key (masked rows stay zero)
#pragma unroll
    for (int e = 0; e < 8; ++e) xk[e] = (kFull || valid) ? nk[e] : 0.0f;
  } else {
    unpack8<Io>(tok(4), xa);
    unpack8<Io>(tok(5), xb);
  }
  constexpr float kC = kNegExpHalf * kLog2e;
  constexpr float kInvC = 1.0f / kC;
  float g2[8], gm[8], gp[8], at[8], rt[8], bh[8], kh[8];
#pragma unroll
  for (int e = 0; e < 8; ++e)
    g2[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(xl[e], -kLog2e, nbias8[e]));
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    float lw2 = __builtin_amdgcn_rcpf(__builtin_fmaf(g2[e], kInvC, kInvC));
    if constexpr (!kFull) lw2 = valid ? lw2 : 0.0f;
    if constexpr (kRev) lw2 = unit_w ? 0.0f : lw2;
    g2[e] = lw2;
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) g2[e] += row_shr<1>(g2[e]);
#pragma unroll
  for (int e = 0; e < 8; ++e) g2[e] += row_shr<2>(g2[e]);
#pragma unroll
  for (int e = 0; e < 8; ++e) g2[e] += row_shr<4>(g2[e]);
#pragma unroll
  for (int e = 0; e < 8; ++e) g2[e] += row_shr<8>(g2[e]);
#pragma unroll
  for (int e = 0; e < 8; ++e) gm[e] = __builtin_amdgcn_exp2f(g2[e]);      // gamma_t
#pragma unroll
  for (int e = 0; e < 8; ++e) gp[e] = row_prev(gm[e], 1.0f);              // gamma_{t-1}
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float ig = __builtin_amdgcn_exp2f(-g2[e]);                     // 1 / gamma_t
    at[e] = xa[e] * gp[e];
    if constexpr (!kSum) rt[e] = xr[e] * gm[e];
    bh[e] = xb[e] * ig;
    kh[e] = xk[e] * ig;
    if constexpr (kRev) kh[e] *= kscale;
  }
  if (i == L - 1) {
    *reinterpret_cast<f32x4*>(&op.gl[kbase]) = f32x4{gm[0], gm[1], gm[2], gm[3]};
    *reinterpret_cast<f32x4*>(&op.gl[kbase + 4]) = f32x4{gm[4], gm[5], gm[6], gm[7]};
  }
  Sp8 Rs;
  if constexpr (!kSum) Rs = split8(rt);
  const Sp8 As = split8(at), Bs = split8(bh), Ks = split8(kh);
  Sp8 Vs;
  const u32x4 vraw = tok(3);
  if constexpr (kVExact) {
    Vs.hi = __builtin_bit_cast(bf16x8, vraw);
  } else {
    float xv[8];
    unpack8<Io>(vraw, xv);
    Vs = split8(xv);
  }
  // operand rows for the state waves (keys kbase..kbase+7 land in two 4-key
  // runs of the permuted A~ / R~ rows)
  const int p0 = key_pos(kbase), p1 = key_pos(kbase + 4);
  if constexpr (!kSum) {
    *reinterpret_cast<bf16x4*>(&op.r_h[i][a_col(i, p0)]) = Rs.hi.lo;
    *reinterpret_cast<bf16x4*>(&op.r_h[i][a_col(i, p1)]) = Rs.hi.hi;
    *reinterpret_cast<bf16x4*>(&op.r_l[i][a_col(i, p0)]) = Rs.lo.lo;
    *reinterpret_cast<bf16x4*>(&op.r_l[i][a_col(i, p1)]) = Rs.lo.hi;
  }
  *reinterpret_cast<bf16x4*>(&op.at_h[i][a_col(i, p0)]) = As.hi.lo;
  *reinterpret_cast<bf16x4*>(&op.at_h[i][a_col(i, p1)]) = As.hi.hi;
  *reinterpret_cast<bf16x4*>(&op.at_l[i][a_col(i, p0)]) = As.lo.lo;
  *reinterpret_cast<bf16x4*>(&op.at_l[i][a_col(i, p1)]) = As.lo.hi;
  *reinterpret_cast<bf16x8*>(&op.b_h[i][b_col(i, kbase)]) = Bs.hi;
  *reinterpret_cast<bf16x8*>(&op.b_l[i][b_col(i, kbase)]) = Bs.lo;
  *reinterpret_cast<bf16x8*>(&op.k_h[i][b_col(i, kbase)]) = Ks.hi;
  *reinterpret_cast<bf16x8*>(&op.k_l[i][b_col(i, kbase)]) = Ks.lo;
  *reinterpret_cast<bf16x8*>(&op.v_h[i][b_col(i, kbase)]) = Vs.hi;
  if constexpr (!kVExact) *reinterpret_cast<bf16x8*>(&op.v_l[i][b_col(i, kbase)]) = Vs.lo;
  // mma32x3(X, Y), X, Y in the load layout: item e = X_{4q+e} . Y_i over
  // this lane's keys
  acc.ab = mma32x3(As, Bs, acc.ab);
  acc.abt = mma32x3(Bs, As, acc.abt);
  acc.ak = mma32x3(Ks, As, acc.ak);
  if constexpr (!kSum) {
    acc.rb = mma32x3(Bs, Rs, acc.rb);
    acc.rk = mma32x3(Ks, Rs, acc.rk);
  }
}

// T and the masked Mak, Mrb, Mrk of a chunk from its accumulated products
template <bool kVExact>
__device__ __forceinline__ void key_blocks_ring(ChunkOps<kVExact>& op, const KeyAccR& acc, int i,
                                                int q) {
  f32x4 M, Mt, mak, mrb, mrk;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int r = 4 * q + e;
    M[e] = (r > i) ? acc.ab[e] : 0.f;
    Mt[e] = (i > r) ? acc.abt[e] : 0.f;
    mak[e] = (i > r) ? acc.ak[e] : 0.f;
    mrb[e] = (i >= r) ? acc.rb[e] : 0.f;
    mrk[e] = (i >= r) ? acc.rk[e] : 0.f;
  }
  const AOp t = t_inverse(M, Mt, i, q);
  store_aop(op.t, i, q, t);
  store_aop(op.mak, i, q, as_a(split4(mak)));
  store_aop(op.mrb, i, q, as_a(split4(mrb)));
  store_aop(op.mrk, i, q, as_a(split4(mrk)));
}

// T and the masked Mak of a summary chunk (no R-side blocks)
template <bool kVExact>
__device__ __forceinline__ void key_blocks_ring_sum(ChunkOps<kVExact>& op, const KeyAccR& acc,
                                                    int i, int q) {
  f32x4 M, Mt, mak;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int r = 4 * q + e;
    M[e] = (r > i) ? acc.ab[e] : 0.f;
    Mt[e] = (i > r) ? acc.abt[e] : 0.f;
    mak[e] = (i > r) ? acc.ak[e] : 0.f;
  }
  store_aop(op.t, i, q, t_inverse(M, Mt, i, q));
  store_aop(op.mak, i, q, as_a(split4(mak)));
}

// What the ring kernel writes besides y and the final state, and the order
// it walks a segment in:
//   kInfer  nothing more, first token to last;
//   kFwd    (the training forward) every token's sa (p.sa_out, fp32) and the
//           state after every boundary_every-th chunk (p.boundary);
//   kBwd    (the training backward's value pass) the same outputs with the
//           recurrence run from the segment's last token to its first:
//           tensor j is read one row later when bit j of p.shift_mask is set
//           (a shifted row past the end reads as zero, with unit retention),
//           and y, sa and the snapshots go to the mirrored positions.
// kFwd and kBwd take uniform segments of a multiple of 16 tokens, or (kRows)
// segments of row blocks (see SegArgs); t0, t1, lo and hi below then count
// tokens of the filled-up blocks, from the segment's first.
enum RingMode { kInfer, kFwd, kBwd };
// A segment as a whole, or one of the two launches of a sequence split
// (below): kLead runs a segment's first piece (and, in other blocks, the
// summaries of the later ones), kRest the pieces after the first.
enum RingPhase { kWhole, kLead, kRest };

// One block's stretch of a segment.  "First" and "before" are in processing
// order, so a kBwd piece's rows run from t1 - 1 down to t0.
struct RingPiece {
  int t0, t1;         // token rows of the piece
  int lo, hi;         // token rows of its segment
  int c0 = 0;         // chunks of the segment before the piece
  bool last = true;   // the segment ends with this piece
};

// Token rows of segment seg (see SegArgs); false when the split leaves piece
// `piece` of it empty.
template <RingMode kMode, RingPhase kPhase, bool kRows>
__device__ __forceinline__ bool ring_piece(const SegArgs& p, int seg, int piece, RingPiece& b) {
  if constexpr (kRows) {
    b.lo = 0;
    b.hi = L * (RowBlocks::at(p.seq_blocks, seg + 1) - RowBlocks::at(p.seq_blocks, seg));
  } else if (p.uniform_len > 0) {
    b.lo = seg * p.uniform_len;
    b.hi = b.lo + p.uniform_len;
  } else if (p.chunk_offsets != nullptr) {
    // a sequence's list of contiguous chunks (the rl_infctx forward)
    b.lo = p.bounds[p.chunk_offsets[seg]];
    b.hi = p.ends[p.chunk_offsets[seg + 1] - 1];
  } else if (p.ends != nullptr) {
    b.lo = p.bounds[seg];
    b.hi = p.ends[seg];
  } else {
    b.lo = p.bounds[seg];
    b.hi = p.bounds[seg + 1];
  }
  b.t0 = b.lo;
  b.t1 = b.hi;
  if constexpr (kPhase != kWhole) {
    int start, len, last;
    split_piece(p, b.hi - b.lo, piece, start, len, last);
    if (piece > last) return false;
    b.last = piece == last;
    b.c0 = start / L;
    if constexpr (kMode == kBwd) {
      b.t1 = b.hi - start;
      b.t0 = max(b.t1 - len, b.lo);
    } else {
      b.t0 = b.lo + start;
      b.t1 = min(b.t0 + len, b.hi);
    }
  }
  return true;
}

// A lane's token in a row block: its row (a row of the block where it has no
// such token) and whether it is there.
struct BlockRow {
  int row;
  bool live;
};
__device__ __forceinline__ BlockRow block_row(const SegArgs& p, int block, int token) {
  const int row0 = RowBlocks::at(p.row_blocks, 2 * block);
  const int n = RowBlocks::at(p.row_blocks, 2 * block + 1);
  return {row0 + min(token, n - 1), token < n};
}
// The token after it in the segment whose last block is `end` - 1: an identity
// token inside a short block, the next block's first token after the block's
// sixteenth, nothing after the segment's last.
__device__ __forceinline__ BlockRow block_next_row(const SegArgs& p, int block, int end,
                                                   int token) {
  const int row0 = RowBlocks::at(p.row_blocks, 2 * block);
  const int n = RowBlocks::at(p.row_blocks, 2 * block + 1);
  const bool more = block + 1 < end;
  const int next0 = RowBlocks::at(p.row_blocks, 2 * (more ? block + 1 : block));
  return token == L - 1 ? BlockRow{next0, more}
                        : BlockRow{row0 + min(token + 1, n - 1), token + 1 < n};
}

// Blocks of the split's workspace, D * D floats each: the state at the end of
// segment seg's first piece, and the final state from zero (kind 0, F) or the
// transition (kind 1, Phi) of its piece m >= 1.  The blocks are laid out for
// chain_start_state's reads, 16 bytes per lane and 1 KiB per tile: a state
// block as tile (column block w, row block kb) in accumulator layout, Phi as
// tile (row block rb, column block kb) whose lane (i, q) holds
// Phi[16 rb + i][16 kb + 4 q ..+3], the A operands of four K steps.
__device__ __forceinline__ float* split_first_state(const SegArgs& p, int seg, int h) {
  return p.split_state + (static_cast<int64_t>(seg) * p.num_heads + h) * D * D;
}
__device__ __forceinline__ float* split_summary_of(const SegArgs& p, int seg, int m, int kind,
                                                   int h) {
  const int64_t pair = static_cast<int64_t>(seg) * (p.split_pieces - 2) + (m - 1);
  return p.split_summary + ((pair * 2 + kind) * p.num_heads + h) * D * D;
}
__device__ __forceinline__ f32x4* split_tile(float* blk, int a, int b, int lane) {
  return reinterpret_cast<f32x4*>(blk) + (4 * a + b) * 64 + lane;
}
// The failure words of a split segment: word 0 for its first piece and word m for
// the summary of piece m, written by those blocks (0 or 1), and the last word, which
// the first piece clears for the second launch's blocks.  There, a block whose start
// state is chained from a failed one fails too; and a state updated in place stays
// untouched when another piece of its segment fails, before or after the last piece
// stored it: whichever of the two comes second to the word puts the saved state back.
constexpr int kStateStored = 1, kPieceFailed = 2;
__device__ __forceinline__ int* split_flags_of(const SegArgs& p, int seg, int h) {
  return p.split_flags + (static_cast<int64_t>(seg) * p.num_heads + h) * p.split_pieces;
}
__device__ __forceinline__ float* split_saved_of(const SegArgs& p, int seg, int h) {
  return p.split_saved + (static_cast<int64_t>(seg) * p.num_heads + h) * D * D;
}
// State columns [16 w, 16 w + 16) of the slot at sbase; kThrough: past the XCD's L2,
// so that a block on another XCD may overwrite them.
template <bool kThrough>
__device__ __forceinline__ void store_state(const SegArgs& p, int64_t sbase, int w, int lane,
                                            const f32x4 (&S)[4]) {
  const int64_t at = sbase + (4 * (lane >> 4)) * D + 16 * w + (lane & 15);
  auto put = [](auto* to, auto x) {
    if constexpr (kThrough)
      __hip_atomic_store(to, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else
      *to = x;
  };
  if (p.state_bf16) {
    uint16_t* const to = static_cast<uint16_t*>(p.state_out) + at;
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
      for (int e = 0; e < 4; ++e) put(to + (16 * kb + e) * D, IoBF16::from_f32(S[kb][e]));
  } else {
    float* const to = static_cast<float*>(p.state_out) + at;
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
      for (int e = 0; e < 4; ++e) put(to + (16 * kb + e) * D, S[kb][e]);
  }
}
// (one wave) Adds `mine` to the segment's last word; where `other` came first, the
// saved state goes back to the slot.
__device__ __forceinline__ void settle_state(const SegArgs& p, int seg, int h, int64_t sbase,
                                             int lane, int mine, int other) {
  int seen = 0;
  if (lane == 0)
    seen = __hip_atomic_fetch_or(split_flags_of(p, seg, h) + p.split_pieces - 1, mine,
                                 __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if ((__builtin_amdgcn_readfirstlane(seen) & other) == 0) return;
  float* const saved = split_saved_of(p, seg, h);
  for (int w = 0; w < 4; ++w) {
    f32x4 S[4];
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) S[kb] = *split_tile(saved, w, kb, lane);
    store_state<true>(p, sbase, w, lane, S);
  }
}

// Start state of piece j >= 1 for this wave's 16 columns: the state after
// piece 0, carried over pieces 1..j-1 by S <- Phi_m S + F_m on the fp32 matrix
// instruction (v_mfma_f32_16x16x4_f32: no operand is rounded).  The
// accumulator layout of S is its B operand: K step (kb, e) takes the rows
// 16 kb + 4 q + e that item e of tile kb holds.  The blocks of two pieces are
// in flight, each requested as soon as its registers are free and without a
// branch (requests past the chain's end repeat its last block): a conditional
// request makes the wait in front of the products count the worst path, which
// waited for the requests just issued (2.1 us per piece, 1.6 without).
// Every block of a segment repeats the chain: a combine kernel in between
// (one block per unit, LDS and fp32 FMAs) took 2-3 us per piece plus its own
// launch, and the key waves build their first chunks meanwhile.
__device__ __forceinline__ void chain_start_state(const SegArgs& p, int seg, int piece, int h,
                                                  int w, int lane, f32x4 (&S)[4]) {
  float* s1 = split_first_state(p, seg, h);
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) S[kb] = *split_tile(s1, w, kb, lane);
  if (piece < 2) return;
  struct Step {
    f32x4 phi[4][4], f[4];   // [rb][kb], [rb]
  };
  auto request = [&](Step& st, int m) {
    float* f = split_summary_of(p, seg, min(m, piece - 1), 0, h);
    float* phi = split_summary_of(p, seg, min(m, piece - 1), 1, h);
#pragma unroll
    for (int rb = 0; rb < 4; ++rb) {
      st.f[rb] = *split_tile(f, w, rb, lane);
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) st.phi[rb][kb] = *split_tile(phi, rb, kb, lane);
    }
  };
  auto apply = [&](const Step& st) {
    f32x4 n[4];
#pragma unroll
    for (int rb = 0; rb < 4; ++rb) n[rb] = st.f[rb];
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int rb = 0; rb < 4; ++rb)
          n[rb] = __builtin_amdgcn_mfma_f32_16x16x4f32(st.phi[rb][kb][e], S[kb][e], n[rb], 0, 0, 0);
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) S[kb] = n[kb];
  };
  Step a, b;
  request(a, 1);
  request(b, 2);
  int m = 1;
  for (; m + 1 < piece; m += 2) {
    apply(a);
    request(a, m + 2);
    apply(b);
    request(b, m + 3);
  }
  if (m < piece) apply(a);
}

// The recurrence over one piece (or a whole segment).  kKK: wkv_prepare's
// kk / a-gate stage fused into the key waves' load stage (p.k is the projected
// key, p.a the a-gate logits a12; the gated key goes to p.new_k), as in
// chunk64_kernel.
template <class Io, bool kKK, RingMode kMode, RingPhase kPhase, bool kRows>
__device__ __forceinline__ void ring_real(const SegArgs& p,
                                          SmemR<!__is_same(Io, IoF16)>& sm, int seg, int piece,
                                          int h) {
  using raw = typename Io::raw;
  constexpr bool kVExact = !__is_same(Io, IoF16);
  constexpr bool kTrainOut = kMode != kInfer;
  constexpr bool kRev = kMode == kBwd;
  constexpr int kRing = kRingOf<kVExact>;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i = lane & 15;
  const int q = lane >> 4;
  const int H = p.num_heads;
  RingPiece pc;
  if (!ring_piece<kMode, kPhase, kRows>(p, seg, piece, pc)) return;
  const int t0 = pc.t0, t1 = pc.t1;
  // (kRows) the segment's blocks and the block of the piece's chunk c
  const int blk_lo = kRows ? RowBlocks::at(p.seq_blocks, seg) : 0;
  const int blk_end = kRows ? RowBlocks::at(p.seq_blocks, seg + 1) : 0;
  auto block_of = [&](int c) { return kRev ? blk_lo + t1 / L - 1 - c : blk_lo + t0 / L + c; };
  const int slot = p.slots ? p.slots[seg] : seg;
  const int64_t head_off = static_cast<int64_t>(h) * D;
  const int64_t row_stride = static_cast<int64_t>(H) * D;
  const int nchunks = (t1 - t0 + L - 1) / L;
  raw* yout = static_cast<raw*>(p.y);
  // training outputs: the row of sa position pos of the piece (kBwd: of row
  // t1 - pos, the segment's position 0 wrapping to its first row) and the
  // segment's snapshots
  auto sa_row = [&](int pos) {
    return kMode == kFwd ? t0 + pos : (pc.c0 == 0 && pos == 0) ? pc.lo : t1 - pos;
  };
  float* const sa_base = kTrainOut ? p.sa_out + head_off : nullptr;
  const int nsnap = kTrainOut ? (p.boundary_per_seg + p.boundary_every - 1) / p.boundary_every : 0;
  const int64_t snap_stride = static_cast<int64_t>(kRows ? H : 1) * D * D;
  float* const bnd_base =
      (kTrainOut && p.boundary != nullptr)
          ? p.boundary +
                (kRows ? (static_cast<int64_t>(kRev ? RowBlocks::at(p.seq_spans, seg) : blk_lo) * H + h)
                       : (static_cast<int64_t>(seg) * H + h) * nsnap) * D * D
          : nullptr;
  // index of chunk c's snapshot in the segment, and whether it is kept
  auto snap_at = [&](int c) {
    return kRows ? block_of(c) - blk_lo
           : kRev ? p.boundary_per_seg - 1 - (pc.c0 + c) : pc.c0 + c;
  };
  auto snap_kept = [&](int c) {
    return bnd_base != nullptr && snap_at(c) % p.boundary_every == 0;
  };

  if (tid < kKeyW + 6) (&sm.ready[0])[tid] = 0;
  __syncthreads();   // the only workgroup barrier before the end: counters are zero

  // (split) the state is updated in place, by the last piece
  const bool in_place =
      kPhase != kWhole && p.state_in != nullptr && p.state_out == p.state_in;
  const int vcol = 16 * (wv & 3) + i;
  const int64_t sbase = (static_cast<int64_t>(slot) * H + h) * D * D;
  if (wv < 4) {
    // ---------------- state waves: columns [16wv, 16wv+16)
    f32x4 S[4];
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) S[kb] = f32x4{0.f, 0.f, 0.f, 0.f};
    if constexpr (kPhase == kRest) {
      // (requested in front of the chain's blocks, used when those have arrived)
      const int* const flags = split_flags_of(p, seg, h);
      int lost = flags[min(lane, piece - 1)];
      chain_start_state(p, seg, piece, h, wv, lane, S);
      for (int m = lane + 64; m < piece; m += 64) lost |= flags[m];
      if (lost != 0) {
        raise_fault(&sm.lost);
        raise_fault(&sm.fault);
      }
    } else if (p.state_in != nullptr && p.state_bf16) {
      // (bf16-state contract) widened once; the state stays fp32 for the
      // whole call and is rounded back once at the end
      const uint16_t* sinb = static_cast<const uint16_t*>(p.state_in) + sbase + vcol;
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int e = 0; e < 4; ++e) S[kb][e] = IoBF16::to_f32(sinb[(kb * 16 + 4 * q + e) * D]);
    } else if (p.state_in != nullptr) {
      const float* sin = static_cast<const float*>(p.state_in) + sbase + vcol;
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int e = 0; e < 4; ++e) S[kb][e] = sin[(kb * 16 + 4 * q + e) * D];
    }
    if (kPhase == kLead && in_place && !pc.last) {
      float* const saved = split_saved_of(p, seg, h);
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) *split_tile(saved, wv, kb, lane) = S[kb];
    }
    // Each state wave writes its own 16 output columns: the chunk's rows are
    // staged in the wave's column band of yb (2-byte stores from the
    // accumulators) and read back as 16-byte pieces, lane l < 32 taking
    // row l / 2, columns 16 (wv % 4) + 8 (l % 2) .. + 7.  The band belongs
    // to this wave alone and its LDS accesses complete in order, so no wave
    // waits for another over the output.
    const int y_row = lane >> 1, y_c0 = 16 * (wv & 3) + 8 * (lane & 1);
    for (int c = 0; c < nchunks; ++c) {
      wait_ge(&sm.ready[c % kKeyW], c / kKeyW + 1, p.spin_limit, &sm.fault);   // operators of c
      const StateOps<kVExact> o = state_load(sm.ops[c % kRing], vcol, i, q);
      if constexpr (kTrainOut) {
        // staged for a key wave to write back (ChunkOut)
        const bool keep = snap_kept(c);
        f32x4 uy[2];
        state_compute<Io, kVExact, false, false, true>(o, S, nullptr, vcol, i, q, p.scale, SaRows{},
                                                       nullptr, false, uy);
        wait_min_ge(sm.consumed, c, p.spin_limit, &sm.fault);   // nobody reads chunk c - 1
        ChunkOut& out = chunk_out(sm, c);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          out.u[4 * q + e][vcol] = uy[0][e];
          out.y[4 * q + e][vcol] = __builtin_bit_cast(uint16_t, Io::from_f32(uy[1][e]));
        }
        if (keep) {
#pragma unroll
          for (int kb = 0; kb < 4; ++kb)
#pragma unroll
            for (int e = 0; e < 4; ++e) out.s[16 * kb + 4 * q + e][vcol] = S[kb][e];
        }
      } else {
        state_compute<Io, kVExact>(o, S, &sm.yb[0], vcol, i, q, p.scale);
        const int pos = c * L + y_row;   // position in processing order
        if (lane < 32 && pos < t1 - t0) {
          const u32x4 piece4 = *reinterpret_cast<const u32x4*>(&sm.yb[y_row][y_c0]);
          *reinterpret_cast<u32x4*>(yout + static_cast<int64_t>(t0 + pos) * row_stride + head_off +
                                    y_c0) = piece4;
        }
      }
      signal(&sm.consumed[wv], c + 1);
    }
    __syncthreads();
    const bool failed = peek(&sm.fault) != 0;
    if (kPhase == kLead && !pc.last && tid == 0) {
      int* const flags = split_flags_of(p, seg, h);
      flags[0] = failed;
      flags[p.split_pieces - 1] = 0;
    }
    if (failed) {
      const bool lost = kPhase == kRest && peek(&sm.lost) != 0;
      if (tid == 0 && !lost && p.handoff_fault != nullptr) atomicAdd(p.handoff_fault, 1);
      const float qnan = quiet_nan();
      const raw nanv = Io::from_f32(qnan);
      if (kRev && pc.last && p.state_out != nullptr) {   // (an output of its own there)
        float* const sout = static_cast<float*>(p.state_out) + sbase;
        for (int e = tid; e < D * D; e += 256) sout[e] = qnan;
      }
      if (kPhase == kRest && in_place && !pc.last && !lost && wv == 0)
        settle_state(p, seg, h, sbase, lane, kPieceFailed, kStateStored);
      for (int64_t e = tid; e < static_cast<int64_t>(t1 - t0) * D; e += 256) {
        const int pos = static_cast<int>(e / D), col = static_cast<int>(e % D);
        BlockRow yr{t0 + pos, true}, ur{0, true};
        if constexpr (kRows) {   // (a wave's 64 elements are one row: pos is uniform)
          const int block = block_of(pos / L);
          yr = block_row(p, block, pos % L);
          ur = kRev ? block_next_row(p, block, blk_end, pos % L) : yr;
        } else if constexpr (kTrainOut) {
          ur.row = sa_row(pos);
        }
        if (yr.live) yout[yr.row * row_stride + head_off + col] = nanv;
        if constexpr (kTrainOut) {
          if (ur.live) sa_base[ur.row * row_stride + col] = qnan;
        }
      }
      if (kPhase == kLead && !pc.last) {
        // the pieces that start from this state come out NaN as well
        float* sout = split_first_state(p, seg, h);
        for (int e = tid; e < D * D; e += 256) sout[e] = qnan;
      }
      return;
    }
    if (!pc.last) {
      if constexpr (kPhase == kLead) {
        float* sout = split_first_state(p, seg, h);
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) *split_tile(sout, wv, kb, lane) = S[kb];
      }
    } else if (kPhase == kRest && in_place) {
      store_state<true>(p, sbase, wv, lane, S);
      __atomic_signal_fence(__ATOMIC_SEQ_CST);
      __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0): the stores have landed
      __atomic_signal_fence(__ATOMIC_SEQ_CST);
      __syncthreads();                      // (with the key waves)
      if (wv == 0) settle_state(p, seg, h, sbase, lane, kStateStored, kPieceFailed);
    } else if (p.state_out != nullptr) {
      store_state<false>(p, sbase, wv, lane, S);
    }
  } else {
    // ---------------- key waves: whole chunks kw, kw + 4, ...
    const int kw = wv - 4;
    float nbias[2][8];
#pragma unroll
    for (int hh = 0; hh < 2; ++hh)
#pragma unroll
      for (int e = 0; e < 8; ++e)
        nbias[hh][e] = p.bias ? -kLog2e * Io::to_f32(static_cast<const raw*>(p.bias)[
                                             head_off + 32 * hh + 8 * q + e])
                              : 0.f;
    const raw* src[6] = {
        static_cast<const raw*>(p.r), static_cast<const raw*>(p.logits),
        static_cast<const raw*>(p.k), static_cast<const raw*>(p.v),
        static_cast<const raw*>(p.a), kKK ? nullptr : static_cast<const raw*>(p.b)};
    u32x4 rawc[2][6];
    KkHalf kph[2];
    if constexpr (kKK) {
#pragma unroll
      for (int hh = 0; hh < 2; ++hh)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int64_t ch = head_off + 32 * hh + 8 * q + e;
          kph[hh].kks[e] = Io::to_f32(static_cast<const raw*>(p.kk_scale)[ch]);
          kph[hh].a0[e] = Io::to_f32(static_cast<const raw*>(p.a_bias)[ch]);
          kph[hh].ka[e] = Io::to_f32(static_cast<const raw*>(p.k_a)[ch]);
        }
    }
    // rows past the sequence end are loaded from its last row (in bounds);
    // key_half_ring zeroes them.  (kRows) whether the lane's token and the one
    // after it are there, and the block's token count, of the chunk in rawc
    bool live = true, live_sh = true;
    int blk_n = L;
    auto load_chunk = [&](int c) {
      // reverse: position c L + i reads row t1 - 1 - pos, one row later for
      // the shifted tensors (clamped into the segment; the row past its end
      // is zeroed where it is consumed)
      int row = kRev ? t1 - 1 - (c * L + i) : min(t0 + c * L + i, t1 - 1);
      int row_sh = min(row + 1, pc.hi - 1);
      if constexpr (kRows) {
        const int block = block_of(c);
        const BlockRow own = block_row(p, block, kRev ? L - 1 - i : i);
        row = own.row;
        live = own.live;
        blk_n = RowBlocks::at(p.row_blocks, 2 * block + 1);
        if constexpr (kRev) {
          const BlockRow nxt = block_next_row(p, block, blk_end, L - 1 - i);
          row_sh = nxt.row;
          live_sh = nxt.live;
        }
      }
      const int64_t off = static_cast<int64_t>(row) * row_stride + head_off + 8 * q;
      const int64_t off_sh = static_cast<int64_t>(row_sh) * row_stride + head_off + 8 * q;
#pragma unroll
      for (int hh = 0; hh < 2; ++hh)
#pragma unroll
        for (int j = 0; j < 6; ++j) {
          const int64_t o = (kRev && ((p.shift_mask >> j) & 1)) ? off_sh : off;
          rawc[hh][j] = (kKK && j == 5)   // b is formed from the key
                            ? u32x4{0u, 0u, 0u, 0u}
                            : __builtin_nontemporal_load(
                                  reinterpret_cast<const u32x4*>(src[j] + o + 32 * hh));
        }
    };
    // Writes chunk c's staged outputs to memory in whole rows (128 and 256 bytes),
    // past the caches what the backward reads much later.  The training forward
    // is bound by these bytes (8 x 4 096 tokens, H = 32: 1.48 of 2.28 GB, us):
    // stored by the state waves, 64-byte pieces of their 16 columns on the
    // recurrence's critical path, 728, of which 392 for the snapshots alone;
    // whole rows from here 540; snapshots past the caches 531, sa too 501
    // (4.55 TB/s).  Inference keeps its 2 KB of y per chunk on the state waves:
    // written from here it costs a ring slot, 304 against 289.
    auto write_out = [&](int c) {
      const ChunkOut& out = chunk_out(sm, c);
      const int tok4 = lane >> 4, c4 = 4 * (lane & 15), tok8 = lane >> 3, c8 = 8 * (lane & 7);
      if (snap_kept(c)) {
        float* const snap =
            bnd_base + static_cast<int64_t>(snap_at(c) / p.boundary_every) * snap_stride;
#pragma unroll
        for (int t = 0; t < D / 4; ++t)
          __builtin_nontemporal_store(
              *reinterpret_cast<const f32x4*>(&out.s[4 * t + tok4][c4]),
              reinterpret_cast<f32x4*>(snap + (4 * t + tok4) * D + c4));
      }
#pragma unroll
      for (int t = 0; t < L / 4; ++t) {
        const int tok = 4 * t + tok4;
        BlockRow ur{0, true};
        if constexpr (kRows)
          ur = kRev ? block_next_row(p, block_of(c), blk_end, L - 1 - tok)
                    : block_row(p, block_of(c), tok);
        else
          ur.row = sa_row(c * L + tok);
        if (!kRows || ur.live)
          __builtin_nontemporal_store(
              *reinterpret_cast<const f32x4*>(&out.u[tok][c4]),
              reinterpret_cast<f32x4*>(sa_base + static_cast<int64_t>(ur.row) * row_stride + c4));
      }
#pragma unroll
      for (int t = 0; t < L / 8; ++t) {
        const int tok = 8 * t + tok8, pos = c * L + tok;
        BlockRow yr{kRev ? t1 - 1 - pos : t0 + pos, true};
        if constexpr (kRows) yr = block_row(p, block_of(c), kRev ? L - 1 - tok : tok);
        if (!kRows || yr.live)
          *reinterpret_cast<u32x4*>(yout + static_cast<int64_t>(yr.row) * row_stride + head_off +
                                    c8) = *reinterpret_cast<const u32x4*>(&out.y[tok][c8]);
      }
      // (compiler order only: the wave's LDS accesses complete in order)
      __atomic_signal_fence(__ATOMIC_SEQ_CST);
    };
    if (kw < nchunks) load_chunk(kw);
    // With kTrainOut the wave that builds chunk c writes chunk c - kRing + 1 out
    // first, whose outputs lie in the same slot.
    for (int c = kw; c < nchunks + (kTrainOut ? kRing - 1 : 0); c += kKeyW) {
      // chunk c - kRing no longer read
      wait_min_ge(sm.consumed, min(c - kRing + (kTrainOut ? 2 : 1), nchunks), p.spin_limit,
                  &sm.fault);
      if constexpr (kTrainOut) {
        if (c - kRing + 1 >= 0) write_out(c - kRing + 1);
        if (c >= nchunks) continue;
      }
      ChunkOps<kVExact>& op = sm.ops[c % kRing];
      const bool full = kRows ? blk_n == L : t0 + c * L + L <= t1;
      const bool valid = kRows ? live : t0 + c * L + i < t1;
      KeyAccR acc;
      const f32x4 z = {0.f, 0.f, 0.f, 0.f};
      acc.ab = z; acc.abt = z; acc.ak = z; acc.rb = z; acc.rk = z;
      float kinv = 0.0f;
      raw* nk_row = nullptr;
      if constexpr (kKK) {
        // 1 / |k k_k| over the token's 64 keys (the four lanes of token i
        // hold 16 each)
        float ss = 0.0f;
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) {
          float xk[8];
          unpack8<Io>(rawc[hh][2], xk);
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float u = xk[e] * kph[hh].kks[e];
            ss = __builtin_fmaf(u, u, ss);
          }
        }
        ss += __shfl_xor(ss, 16);
        ss += __shfl_xor(ss, 32);
        kinv = __builtin_amdgcn_rcpf(fmaxf(__builtin_sqrtf(ss), 1.0e-12f));
        nk_row = static_cast<raw*>(p.new_k) +
                 static_cast<int64_t>(t0 + c * L + i) * row_stride + head_off;
      }
      if constexpr (kRev) {
        // position 0 of the segment: its shifted rows lie past the end
        const bool void_row = kRows ? !live_sh : pc.c0 + c == 0 && i == 0;
#pragma unroll
        for (int hh = 0; hh < 2; ++hh)
#pragma unroll
          for (int j = 0; j < 6; ++j)
            if (j != 1 && (((p.shift_mask >> j) & 1) ? void_row : kRows && !live))
              rawc[hh][j] = u32x4{0u, 0u, 0u, 0u};
        const bool unit_w = void_row && ((p.shift_mask >> 1) & 1);
        key_half_ring<Io, kVExact, true, false, false, true>(op, rawc[0], nbias[0], true, 0, i, q,
                                                            acc, nullptr, 0.0f, nullptr, unit_w,
                                                            p.kv_scale);
        key_half_ring<Io, kVExact, true, false, false, true>(op, rawc[1], nbias[1], true, 1, i, q,
                                                            acc, nullptr, 0.0f, nullptr, unit_w,
                                                            p.kv_scale);
      } else if (full) {
        key_half_ring<Io, kVExact, true, false, kKK>(op, rawc[0], nbias[0], true, 0, i, q, acc,
                                                     &kph[0], kinv, nk_row);
        key_half_ring<Io, kVExact, true, false, kKK>(op, rawc[1], nbias[1], true, 1, i, q, acc,
                                                     &kph[1], kinv, nk_row);
      } else {
        key_half_ring<Io, kVExact, false, false, kKK>(op, rawc[0], nbias[0], valid, 0, i, q,
                                                      acc, &kph[0], kinv, nk_row);
        key_half_ring<Io, kVExact, false, false, kKK>(op, rawc[1], nbias[1], valid, 1, i, q,
                                                      acc, &kph[1], kinv, nk_row);
      }
      if (c + kKeyW < nchunks) load_chunk(c + kKeyW);
      key_blocks_ring(op, acc, i, q);
      if (p.handoff_stall != 1 && !(p.handoff_stall == 2 && kPhase == kRest && !pc.last))
        signal(&sm.ready[kw], (c - kw) / kKeyW + 1);
    }
    __syncthreads();   // pairs with the state waves' final barrier
    if (kPhase == kRest && in_place && pc.last && peek(&sm.fault) == 0) __syncthreads();
  }
}

// Summary of piece `piece` >= 1 of a split segment (nothing for its last
// piece).  Four key waves build whole chunks into the operator ring as in
// ring_real, without R~ and the R-side blocks.  Each of the four state waves
// carries, for its 16 columns, both the piece's final state from zero (F) and
// its transition Phi (identity start, V = 0): two independent chains over the
// same operands, read from LDS once.  Writes the two blocks
// split_summary_of(seg, piece, {0: F, 1: Phi}, h) and nothing else.
template <class Io, RingMode kMode, bool kRows>
__device__ __forceinline__ void ring_summary(const SegArgs& p,
                                             SmemR<!__is_same(Io, IoF16)>& sm, int seg,
                                             int piece, int h) {
  using raw = typename Io::raw;
  constexpr bool kVExact = !__is_same(Io, IoF16);
  constexpr bool kRev = kMode == kBwd;
  constexpr int kRing = kRingOf<kVExact>;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i = lane & 15;
  const int q = lane >> 4;
  RingPiece pc;
  if (!ring_piece<kMode, kLead, kRows>(p, seg, piece, pc) || pc.last) return;
  const int t0 = pc.t0, t1 = pc.t1;
  const int blk_lo = kRows ? RowBlocks::at(p.seq_blocks, seg) : 0;
  const int blk_end = kRows ? RowBlocks::at(p.seq_blocks, seg + 1) : 0;
  auto block_of = [&](int c) { return kRev ? blk_lo + t1 / L - 1 - c : blk_lo + t0 / L + c; };
  const int64_t head_off = static_cast<int64_t>(h) * D;
  const int64_t row_stride = static_cast<int64_t>(p.num_heads) * D;
  const int nchunks = (t1 - t0 + L - 1) / L;

  if (tid < kKeyW + 5) (&sm.ready[0])[tid] = 0;
  __syncthreads();   // the only workgroup barrier before the end: counters are zero

  const int vcol = 16 * (wv & 3) + i;
  if (wv < 4) {
    f32x4 F[4], Phi[4];
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        F[kb][e] = 0.0f;
        Phi[kb][e] = (kb * 16 + 4 * q + e == vcol) ? 1.0f : 0.0f;
      }
    for (int c = 0; c < nchunks; ++c) {
      wait_ge(&sm.ready[c % kKeyW], c / kKeyW + 1, p.spin_limit, &sm.fault);   // operators of c
      // every operand is in registers before the slot is released
      const StateOps<kVExact> o = state_load<kVExact, true>(sm.ops[c % kRing], vcol, i, q);
      signal(&sm.consumed[wv], c + 1);
      state_compute<Io, kVExact, false, true>(o, F, nullptr, vcol, i, q, 1.0f, SaRows{},
                                              nullptr, false);
      state_compute<Io, kVExact, false, true>(o, Phi, nullptr, vcol, i, q, 1.0f, SaRows{},
                                              nullptr, true);
    }
    __syncthreads();
    float* sout = split_summary_of(p, seg, piece, 0, h);
    float* pout = split_summary_of(p, seg, piece, 1, h);
    const bool failed = peek(&sm.fault) != 0;
    if (tid == 0) split_flags_of(p, seg, h)[piece] = failed;
    if (failed) {
      // the pieces that start from this summary come out NaN as well
      if (tid == 0 && p.handoff_fault != nullptr) atomicAdd(p.handoff_fault, 1);
      const float qnan = quiet_nan();
      for (int e = tid; e < D * D; e += 256) {
        sout[e] = qnan;
        pout[e] = qnan;
      }
      return;
    }
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      *split_tile(sout, wv, kb, lane) = F[kb];
      // row_piece leaves Phi[16 kb + 4 q + m][16 wv + 4 j..+3] in lane (4j + m, q)
      *split_tile(pout, kb, wv, 16 * (i >> 2) + 4 * q + (i & 3)) = row_piece(Phi[kb], i);
    }
  } else {
    // ---------------- key waves: whole chunks kw, kw + 4, ...
    const int kw = wv - 4;
    float nbias[2][8];
#pragma unroll
    for (int hh = 0; hh < 2; ++hh)
#pragma unroll
      for (int e = 0; e < 8; ++e)
        nbias[hh][e] = p.bias ? -kLog2e * Io::to_f32(static_cast<const raw*>(p.bias)[
                                             head_off + 32 * hh + 8 * q + e])
                              : 0.f;
    const raw* src[6] = {
        nullptr, static_cast<const raw*>(p.logits),
        static_cast<const raw*>(p.k), static_cast<const raw*>(p.v),
        static_cast<const raw*>(p.a), static_cast<const raw*>(p.b)};
    u32x4 rawc[2][6];
    // (a kBwd summary never starts at its segment's position 0, so none of its
    // shifted rows lies past the segment)
    bool live = true, live_sh = true;
    int blk_n = L;
    auto load_chunk = [&](int c) {
      int row = kRev ? t1 - 1 - (c * L + i) : min(t0 + c * L + i, t1 - 1);
      int row_sh = row + 1;
      if constexpr (kRows) {
        const int block = block_of(c);
        const BlockRow own = block_row(p, block, kRev ? L - 1 - i : i);
        row = own.row;
        live = own.live;
        blk_n = RowBlocks::at(p.row_blocks, 2 * block + 1);
        if constexpr (kRev) {
          const BlockRow nxt = block_next_row(p, block, blk_end, L - 1 - i);
          row_sh = nxt.row;
          live_sh = nxt.live;
        }
      }
      const int64_t off = static_cast<int64_t>(row) * row_stride + head_off + 8 * q;
      const int64_t off_sh = static_cast<int64_t>(row_sh) * row_stride + head_off + 8 * q;
#pragma unroll
      for (int hh = 0; hh < 2; ++hh) {
        rawc[hh][0] = u32x4{0u, 0u, 0u, 0u};   // r: not read by the summary
#pragma unroll
        for (int j = 1; j < 6; ++j) {
          const int64_t o = (kRev && ((p.shift_mask >> j) & 1)) ? off_sh : off;
          rawc[hh][j] =
              __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(src[j] + o + 32 * hh));
        }
      }
    };
    if (kw < nchunks) load_chunk(kw);
    for (int c = kw; c < nchunks; c += kKeyW) {
      // chunk c - kRing no longer read
      wait_min_ge(sm.consumed, c - kRing + 1, p.spin_limit, &sm.fault);
      ChunkOps<kVExact>& op = sm.ops[c % kRing];
      const bool full = kRows ? blk_n == L : t0 + c * L + L <= t1;
      const bool valid = kRows ? live : t0 + c * L + i < t1;
      KeyAccR acc;
      const f32x4 z = {0.f, 0.f, 0.f, 0.f};
      acc.ab = z; acc.abt = z; acc.ak = z; acc.rb = z; acc.rk = z;
      if (kRev || full) {
        if constexpr (kRev && kRows) {
#pragma unroll
          for (int hh = 0; hh < 2; ++hh)
#pragma unroll
            for (int j = 2; j < 6; ++j)
              if (((p.shift_mask >> j) & 1) ? !live_sh : !live) rawc[hh][j] = u32x4{0u, 0u, 0u, 0u};
        }
        const bool unit_w = kRev && kRows && !live_sh;
        key_half_ring<Io, kVExact, true, true, false, kRev>(
            op, rawc[0], nbias[0], true, 0, i, q, acc, nullptr, 0.0f, nullptr, unit_w, p.kv_scale);
        key_half_ring<Io, kVExact, true, true, false, kRev>(
            op, rawc[1], nbias[1], true, 1, i, q, acc, nullptr, 0.0f, nullptr, unit_w, p.kv_scale);
      } else {
        key_half_ring<Io, kVExact, false, true>(op, rawc[0], nbias[0], valid, 0, i, q, acc);
        key_half_ring<Io, kVExact, false, true>(op, rawc[1], nbias[1], valid, 1, i, q, acc);
      }
      if (c + kKeyW < nchunks) load_chunk(c + kKeyW);
      key_blocks_ring_sum(op, acc, i, q);
      if (p.handoff_stall != 1 && p.handoff_stall != 3) signal(&sm.ready[kw], (c - kw) / kKeyW + 1);
    }
    __syncthreads();   // pairs with the state waves' final barrier
  }
}

// Grid (H, segments) for whole segments; of a split into P pieces,
// (H, segments * (P - 1)): block y = seg * (P - 1) + j runs piece 0 (j = 0) or
// summarises piece j in the kLead launch, and runs piece j + 1 in the kRest
// launch.
template <class Io, bool kKK = false, RingMode kMode = kInfer, RingPhase kPhase = kWhole,
          bool kRows = false>
__global__ __launch_bounds__(NTR) void chunk64r_kernel(SegArgs p) {
  using raw = typename Io::raw;
  __shared__ SmemR<!__is_same(Io, IoF16)> sm;
  const int h = blockIdx.x;
  const int npc = kPhase == kWhole ? 1 : p.split_pieces - 1;
  const int seg = blockIdx.y / npc, j = blockIdx.y % npc;
  if (p.status != nullptr) {
    if (p.status[0] != 0) {
      if constexpr (kPhase != kLead) {
        const int64_t blk = static_cast<int64_t>(blockIdx.y) * gridDim.x + h;
        const int64_t nblk = static_cast<int64_t>(gridDim.x) * gridDim.y;
        fill_output_nan<Io>(static_cast<raw*>(p.y), p.out_elems, blk, nblk);
      }
      return;
    }
    if (seg >= p.status[2]) return;
  }
  if constexpr (kPhase == kLead) {
    if (j > 0) {
      ring_summary<Io, kMode, kRows>(p, sm, seg, j, h);
      return;
    }
  }
  ring_real<Io, kKK, kMode, kPhase, kRows>(p, sm, seg, kPhase == kRest ? j + 1 : 0, h);
}

}  // namespace

namespace {
// Blocks of the chunked kernels whose wave hand-off gave up, per device (each
// device holds its own copy; read through fr2_handoff_fault_count).
__device__ int g_handoff_faults;
std::atomic<int> g_spin_limit{1 << 20};
std::atomic<int> g_handoff_stall{0};
std::atomic<int> g_chunk_ring{1};
std::atomic<int*> g_fault_ptr[64];
}  // namespace

int* handoff_fault_word() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return nullptr;
  int* ptr = g_fault_ptr[dev].load(std::memory_order_acquire);
  if (ptr == nullptr) {
    if (hipGetSymbolAddress(reinterpret_cast<void**>(&ptr), HIP_SYMBOL(g_handoff_faults)) !=
        hipSuccess)
      return nullptr;
    g_fault_ptr[dev].store(ptr, std::memory_order_release);
  }
  return ptr;
}
int handoff_spin_limit() { return g_spin_limit.load(std::memory_order_relaxed); }
int handoff_stall() { return g_handoff_stall.load(std::memory_order_relaxed); }
bool chunk_ring_enabled() { return g_chunk_ring.load(std::memory_order_relaxed) != 0; }
void set_chunk_ring(int on) { g_chunk_ring.store(on, std::memory_order_relaxed); }
void set_handoff_stall(int mode) { g_handoff_stall.store(mode, std::memory_order_relaxed); }
void set_handoff_spin_limit(int polls) {
  g_spin_limit.store(polls < 0 ? (1 << 20) : polls, std::memory_order_relaxed);
}

// whether an inference call (fp32 or bf16 state, packed, uniform or chunk-list
// segments) runs on the ring variant: all but the fused read-out do, which stays on
// chunk64_kernel, as does everything unsplit with the ring switched off
bool ring_contract(const SegArgs& p) {
  return chunk_ring_enabled() && p.boundary == nullptr && p.sa_out == nullptr &&
         p.ro_out == nullptr;
}

// A unit's share: the state after piece 0, two blocks for each of pieces 1..P-2, the
// saved start state, and P flags (rounded up to 16 bytes).
int64_t split_workspace_floats(int nseg, int H, int pieces) {
  const int64_t units = static_cast<int64_t>(nseg) * H;
  return units * (2 * pieces - 2) * D * D + (units * pieces + 3) / 4 * 4;
}
// Points p's split at its workspace.
static void set_split(SegArgs& p, int nseg, int pieces, int piece_len, int lead_len,
                      float* workspace) {
  const int64_t unit_floats = static_cast<int64_t>(nseg) * p.num_heads * D * D;
  p.split_pieces = pieces;
  p.split_len = piece_len;
  p.split_lead = lead_len;
  p.split_state = workspace;
  p.split_saved = workspace + unit_floats;
  p.split_summary = workspace + 2 * unit_floats;
  p.split_flags = reinterpret_cast<int*>(workspace + (2 * pieces - 2) * unit_floats);
}

namespace {

// The two launches of a sequence split: every segment's piece 0 next to the
// summaries of its pieces 1..P-2, then its pieces 1..P-1, each of which chains
// its own start state (chain_start_state).  A piece 0 on a second stream next
// to a summary launch, and a combine launch between the passes, gave the same
// two phases with two event waits and one more launch: one 1 531-token
// sequence x 32 heads took 0.102 ms (3 pieces; more lost to the fixed cost),
// 0.045 ms here (9 pieces); 65 536 tokens x 64 heads 1.81 -> 1.78 ms.
template <class Io, RingMode kMode, bool kRows = false>
void launch_split_kernels(const SegArgs& p, int nseg, hipStream_t s) {
  const dim3 grid(p.num_heads, nseg * (p.split_pieces - 1));
  hipLaunchKernelGGL((chunk64r_kernel<Io, false, kMode, kLead, kRows>), grid, dim3(NTR), 0, s, p);
  hipLaunchKernelGGL((chunk64r_kernel<Io, false, kMode, kRest, kRows>), grid, dim3(NTR), 0, s, p);
}

// The training modes on row blocks: always on the ring layout, whose chunk period
// is the shorter one where the longest of a few ragged sequences decides (8
// sequences of 300 to 2 048 tokens, H = 32, us: forward 239 against 320 on the
// key-half kernel over the padded grid, reverse 180 to 188 either way).
template <RingMode kMode>
void launch_rows(const SegArgs& p, int nseg, hipStream_t s) {
  if (p.split_pieces > 0)
    launch_split_kernels<IoBF16, kMode, true>(p, nseg, s);
  else
    hipLaunchKernelGGL((chunk64r_kernel<IoBF16, false, kMode, kWhole, true>),
                       dim3(p.num_heads, nseg), dim3(NTR), 0, s, p);
}

}  // namespace

// Pieces (a first one and Q more, of len tokens each, the last one shorter) of
// a sequence split, or 1 where splitting does not pay, from the measured cost
// of a prefill (us, MI355X, bf16, 4-128 units, 256-16 384 tokens):
//   whole:  5.5 + 0.057 T
//   split: 10 + 2 (0.057 + 0.009 blocks / 256) piece + 1.6 (Q - 1)
// 0.057 us per token is the ring kernel's rate with few blocks (0.066 with one
// on every CU), a summary runs at the same rate, and 1.6 us is one step of the
// chain a block carries its start state over.  The split time is least near
// Q = sqrt(2 * 0.057 T / 1.6).  32 units, 1 531 tokens: 0.045 ms (9 pieces)
// against 0.092 ms whole; 512 tokens 0.026 against 0.034; at 256 tokens both
// take 0.020.  128 units (three pieces): 1 024 tokens 0.060 against 0.066,
// 512 tokens 0.040 against 0.037.  The training kernels have their optimum at
// the same counts and gain more, their chunks being slower (forward, 24 units,
// 1 024 tokens: 3 pieces 72 us, 5: 52, 9: 45, 11: 44, whole 88; 32 units,
// 2 048 tokens: 9 pieces 74, whole 191).
constexpr float kSplitTokenUs = 0.057f, kSplitFullTokenUs = 0.009f, kSplitHopUs = 1.6f;
constexpr float kSplitFixedUs = 10.0f, kWholeFixedUs = 5.5f;
int split_rule(int64_t units, int tokens, int& len) {
  if (tokens <= 0 || units <= 0 || units > 128) return 1;
  const float T = static_cast<float>(tokens);
  const int Q = std::min(static_cast<int>(256 / units),
                         static_cast<int>(std::sqrt(2.0f * kSplitTokenUs / kSplitHopUs * T) + 0.5f));
  if (Q < 2) return 1;
  // every piece the same length: the first piece and a summary run at one rate
  len = static_cast<int>((static_cast<int64_t>(tokens) + Q) / (Q + 1) + L - 1) / L * L;
  const int P = static_cast<int>((static_cast<int64_t>(tokens) + len - 1) / len);
  const float token_us =
      kSplitTokenUs + kSplitFullTokenUs * static_cast<float>((P - 1) * units) / 256.0f;
  const float split_us =
      kSplitFixedUs + 2.0f * token_us * static_cast<float>(len) + kSplitHopUs * (P - 2);
  return P < 3 || split_us >= kWholeFixedUs + kSplitTokenUs * T ? 1 : P;
}

int64_t train_split_workspace_floats(int nseg, int T, int H) {
  int len = 0;
  const int P = split_rule(static_cast<int64_t>(nseg) * H, T, len);
  return P < 3 ? 0 : split_workspace_floats(nseg, H, P);
}
void set_train_split(SegArgs& p, int nseg, int T, float* workspace) {
  int len = 0;
  const int P = split_rule(static_cast<int64_t>(nseg) * p.num_heads, T, len);
  if (P < 3 || workspace == nullptr) return;
  set_split(p, nseg, P, len, len, workspace);
}

int launch_chunked(int dtype, const SegArgs& args, int nseg, int max_seqlen, hipStream_t s) {
  (void)max_seqlen;
  SegArgs p = args;
  p.spin_limit = handoff_spin_limit();
  p.handoff_stall = handoff_stall();
  p.handoff_fault = handoff_fault_word();
  const bool train = p.sa_out != nullptr || p.boundary != nullptr || p.reverse;
  const dim3 grid(p.num_heads, nseg);
  if (p.row_blocks != nullptr) {
    if (p.sa_out == nullptr || p.boundary == nullptr || p.boundary_len != L ||
        p.seq_blocks == nullptr || (p.reverse && p.seq_spans == nullptr) ||
        dtype != FR2_DTYPE_BFLOAT16)
      return FR2_ERR_INVALID_ARGUMENT;
    if (p.reverse)
      launch_rows<kBwd>(p, nseg, s);
    else
      launch_rows<kFwd>(p, nseg, s);
  } else if (train) {
    // the training contract: uniform segments whose length is a multiple of
    // the 16-token chunk, both outputs present, bf16 tokens (an initial
    // state, or in reverse mode an initial dL/dS, may be given)
    if (p.sa_out == nullptr || (p.boundary == nullptr && !p.reverse) || p.boundary_len != L ||
        p.uniform_len <= 0 || p.uniform_len % L != 0 || dtype != FR2_DTYPE_BFLOAT16)
      return FR2_ERR_UNSUPPORTED;
    if (p.split_pieces > 0) {
      if (p.reverse)
        launch_split_kernels<IoBF16, kBwd>(p, nseg, s);
      else
        launch_split_kernels<IoBF16, kFwd>(p, nseg, s);
    } else if (p.reverse && chunk_ring_enabled())
      hipLaunchKernelGGL((chunk64r_kernel<IoBF16, false, kBwd>), grid, dim3(NTR), 0, s, p);
    else if (p.reverse)
      hipLaunchKernelGGL((chunk64_kernel<IoBF16, true, true>), grid, dim3(NT), 0, s, p);
    else if (chunk_ring_enabled())
      hipLaunchKernelGGL((chunk64r_kernel<IoBF16, false, kFwd>), grid, dim3(NTR), 0, s, p);
    else
      hipLaunchKernelGGL((chunk64_kernel<IoBF16, true>), grid, dim3(NT), 0, s, p);
  } else if (!ring_contract(p)) {
    if (dtype == FR2_DTYPE_BFLOAT16)
      hipLaunchKernelGGL((chunk64_kernel<IoBF16, false>), grid, dim3(NT), 0, s, p);
    else if (dtype == FR2_DTYPE_FLOAT16)
      hipLaunchKernelGGL((chunk64_kernel<IoF16, false>), grid, dim3(NT), 0, s, p);
    else
      return FR2_ERR_UNSUPPORTED;
  } else if (dtype == FR2_DTYPE_BFLOAT16) {
    hipLaunchKernelGGL((chunk64r_kernel<IoBF16>), grid, dim3(NTR), 0, s, p);
  } else if (dtype == FR2_DTYPE_FLOAT16) {
    hipLaunchKernelGGL((chunk64r_kernel<IoF16>), grid, dim3(NTR), 0, s, p);
  } else {
    return FR2_ERR_UNSUPPORTED;
  }
  return record_launch();
}

int launch_chunked_kk(int dtype, const SegArgs& args, int nseg, hipStream_t s) {
  if (args.sa_out != nullptr || args.boundary != nullptr || args.reverse ||
      args.split_pieces > 0 || args.state_bf16 || args.kk_scale == nullptr ||
      args.a_bias == nullptr || args.k_a == nullptr || args.new_k == nullptr)
    return FR2_ERR_INVALID_ARGUMENT;
  SegArgs p = args;
  p.spin_limit = handoff_spin_limit();
  p.handoff_stall = handoff_stall();
  p.handoff_fault = handoff_fault_word();
  const dim3 grid(p.num_heads, nseg);
  const bool ro = p.ro_out != nullptr;
  if (ro && (p.ro_g == nullptr || p.ro_rk == nullptr || p.ro_lnw == nullptr ||
             p.ro_lnb == nullptr))
    return FR2_ERR_INVALID_ARGUMENT;
  // the fused read-out needs a token's whole output row at the write-back:
  // chunk64_kernel; the kk / a-gate stage alone runs on the ring variant
  const bool ring = !ro && ring_contract(p);
  if (dtype == FR2_DTYPE_BFLOAT16) {
    if (ro)
      hipLaunchKernelGGL((chunk64_kernel<IoBF16, false, false, true, true>), grid,
                         dim3(NT), 0, s, p);
    else if (ring)
      hipLaunchKernelGGL((chunk64r_kernel<IoBF16, true>), grid, dim3(NTR), 0, s, p);
    else
      hipLaunchKernelGGL((chunk64_kernel<IoBF16, false, false, true>), grid, dim3(NT), 0,
                         s, p);
  } else if (dtype == FR2_DTYPE_FLOAT16) {
    if (ro)
      hipLaunchKernelGGL((chunk64_kernel<IoF16, false, false, true, true>), grid, dim3(NT),
                         0, s, p);
    else if (ring)
      hipLaunchKernelGGL((chunk64r_kernel<IoF16, true>), grid, dim3(NTR), 0, s, p);
    else
      hipLaunchKernelGGL((chunk64_kernel<IoF16, false, false, true>), grid, dim3(NT), 0,
                         s, p);
  } else {
    return FR2_ERR_UNSUPPORTED;
  }
  return record_launch();
}

int launch_chunked_split(int dtype, SegArgs p, int nseg, int pieces, int piece_len,
                         int lead_len, float* workspace, hipStream_t s) {
  if (p.sa_out != nullptr || p.boundary != nullptr || p.reverse ||
      p.uniform_len > 0 || p.ends != nullptr || p.chunk_offsets != nullptr)
    return FR2_ERR_UNSUPPORTED;
  if (pieces < 2 || piece_len <= 0 || piece_len % L != 0 || lead_len < 0 ||
      lead_len % L != 0 || workspace == nullptr || p.state_in == nullptr ||
      p.state_out != p.state_in || static_cast<int64_t>(nseg) * pieces > 65535)
    return FR2_ERR_INVALID_ARGUMENT;
  if (dtype != FR2_DTYPE_BFLOAT16 && dtype != FR2_DTYPE_FLOAT16) return FR2_ERR_UNSUPPORTED;
  p.spin_limit = handoff_spin_limit();
  p.handoff_stall = handoff_stall();
  p.handoff_fault = handoff_fault_word();
  set_split(p, nseg, pieces, piece_len, lead_len, workspace);
  if (dtype == FR2_DTYPE_BFLOAT16)
    launch_split_kernels<IoBF16, kInfer>(p, nseg, s);
  else
    launch_split_kernels<IoF16, kInfer>(p, nseg, s);
  return record_launch();
}

}  // namespace fr2
