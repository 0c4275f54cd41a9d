// Gated linear attention (GLA), chunked (chunk size 64), forward and backward, on gfx950.
//
// Recurrence (arXiv:2312.06635; the backbone the reference calls through fla's chunk_gla,
// ccq/ops/ccq_gla/fused_chunk.py:42-45, ccq/ops/ccq_gla/chunk.py:53-58):
//   S <- diag(exp(gk_t)) S + k_t v_t^T;   o_t = S^T (scale q_t)
// Per chunk, with b the in-chunk cumulative sum of gk (per channel) and b_L its last row:
//   O = scale (Q o e^b) S + A V,   A_ts = scale sum_c q_tc k_sc e^{b_tc - b_sc}  (s <= t)
//   S <- diag(e^{b_L}) S + (K o e^{b_L - b})^T V
// Backward (dS: gradient of the state after the chunk; G: cumulative decay over the sequence):
//   dS_prev = diag(e^{b_L}) dS + (scale Q o e^b)^T dO
//   dq = scale e^b o (dO S^T) + [dA (K o e^{-b})] o e^b,       dA = scale (dO V^T), causal
//   dk = e^{b_L - b} o (V dS^T) + [dA^T (Q o e^b)] o e^{-b}
//   dv = A^T dO + (K o e^{b_L - b}) dS
//   dG_t = q_t o dq_t - k_t o dk_t (+ rowsum(dS_final o S_final) at the last token),
//   dgk = suffix sum of dG over the sequence.
// The pairwise factors e^{b_t - b_s} (s <= t) inside a chunk enter the products split at a
// reference row m, e^{b_t - b_m} e^{b_m - b_s}, with decays gk <= 0:
// * between the two 32-row blocks (t >= 32 > s) at m = 32, where both factors are <= 1: exact
//   for any decay;
// * inside a diagonal 32-row block at its middle row (16, 48, clamped to the last valid row), where
//   a factor is > 1 only across half the block: used while the log decay over each half stays above
//   -kSplitRange in every channel of the wave (e^80 < fp32 max); otherwise that block is formed with
//   one exponential per pair, e^{b_t - b_s} <= 1, as a sum over the channels in fp32.
// So every decay gives a finite result; the per-pair form only costs time in the blocks that need it.
//
// Kernels:
//   gla_intra        chunk-parallel: A, and the decayed keys transposed, as operands (where b comes later)
//   gla_state<0>     two wavefronts per (sequence, head, 32 channels, 32 value columns): forward
//                    walk over the chunks, state snapshots (hi/lo bf16) and the final state
//   gla_mix<0>       chunk-parallel: O, and b (written for the backward)
//   gla_xprep        chunk-parallel: the decayed queries transposed, as operands
//   gla_state<1>     reverse walk of the state gradient, snapshots and dh0
//   gla_mix<1>       chunk-parallel: dv
//   gla_bwd_dqk      chunk x 64-channel slabs: dq, dk and dgk
//
// Precision: operands that are exact bf16 inputs (k, v, dO) enter one MFMA; every operand formed
// in fp32 (decay-scaled q and k, A, dA, the states) enters as a hi/lo bf16 pair, so products keep
// about 16 significant bits.
#include "ccq_oper.h"
#include "ccq_params.h"

namespace ccq {

namespace {

constexpr int BT = 64;
constexpr int KS = 64;            // channel slab of the chunk-parallel kernels
constexpr int LDF = KS + 4;       // fp32 slab row stride (LDS)
constexpr int LDH = 64 + 8;       // bf16 64-wide row stride (LDS)
constexpr float kSplitRange = 80.f;   // largest log factor a split decay may carry (e^80 < fp32 max)

// True when the split of the pairwise decay factors at row m of the 32-row block starting at row
// r0 stays below e^kSplitRange for channel column c of b (rows past L - 1 hold b_{L-1}), in every
// lane of the wave; a NaN range counts as unsafe.
__device__ __forceinline__ bool split_ok(const float* b, int ld, int r0, int m, int L, int c) {
  const int first = min(r0, L - 1), last = min(r0 + 31, L - 1);
  const float bm = b[m * ld + c];
  const float r = fmaxf(b[first * ld + c] - bm, bm - b[last * ld + c]);
  return __ballot(!(r <= kSplitRange)) == 0;
}

__device__ __forceinline__ bool gla_chunk(const GlaArgs& a, int gc, int& n, int& c0, long& bos, int& L) {
  if (a.cu) {
    n = a.chunk_idx[2 * gc];
    if (n < 0) return false;
    const int c = a.chunk_idx[2 * gc + 1];
    bos = (long)a.cu[n];
    const int len = (int)(a.cu[n + 1] - a.cu[n]);
    c0 = c * BT;
    L = min(BT, len - c0);
  } else {
    n = gc / a.NT;
    const int c = gc % a.NT;
    bos = (long)n * a.T;
    c0 = c * BT;
    L = min(BT, a.T - c0);
  }
  return true;
}

// 64 rows x 64 columns of fp32 (g32) or bf16 (g16) global rows into fp32 LDS [64][LDF]; rows >= nvalid
// = 0, or (hold_last, fp32 only) a copy of row nvalid - 1 -- for the cumulative decay, which stays at
// its last value past the end of a chunk.
__device__ __forceinline__ void slab_to_f32(float* dst, const float* g32, const bf16* g16, long gstride, int nvalid,
                                            bool hold_last = false) {
  if (g32) {
    for (int idx = threadIdx.x; idx < BT * 16; idx += kThreads) {
      const int r = idx >> 4, c = (idx & 15) * 4;
      f32x4 v;
      if (r < nvalid) v = *(const f32x4*)(g32 + (long)r * gstride + c);
      else if (hold_last) v = *(const f32x4*)(g32 + (long)(nvalid - 1) * gstride + c);
      else v[0] = v[1] = v[2] = v[3] = 0.f;
      *(f32x4*)(dst + r * LDF + c) = v;
    }
  } else {
    for (int idx = threadIdx.x; idx < BT * 8; idx += kThreads) {
      const int r = idx >> 3, c = (idx & 7) * 8;
      bf16x8 v;
      if (r < nvalid) {
        v = *(const bf16x8*)(g16 + (long)r * gstride + c);
      } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = (bf16)0.f;
      }
      f32x4 lo4, hi4;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        lo4[i] = (float)v[i];
        hi4[i] = (float)v[4 + i];
      }
      *(f32x4*)(dst + r * LDF + c) = lo4;
      *(f32x4*)(dst + r * LDF + c + 4) = hi4;
    }
  }
}

// 64 x 64 bf16 tile (rows of a token- or value-major tensor) into LDS [64][LDH], rows >= nvalid = 0.
__device__ __forceinline__ void tile_bf16(bf16* dst, const bf16* g, long gstride, int nvalid) {
  for (int idx = threadIdx.x; idx < BT * 8; idx += kThreads) {
    const int r = idx >> 3, c = (idx & 7) * 8;
    bf16x8 v;
    if (r < nvalid) {
      v = *(const bf16x8*)(g + (long)r * gstride + c);
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = (bf16)0.f;
    }
    *(bf16x8*)(dst + r * LDH + c) = v;
  }
}

// 64 value columns x 64 channels of the state and state-gradient snapshots (operand order, np channel pairs
// per column tile) into LDS rows [v][LDH].  A thread meets the same eight channels in every tile:
// with `dots`, sd[i] += S dS of its value columns, in the order of the lane's slots.
__device__ __forceinline__ void tile_op_pair(bf16* sSh, bf16* sSl, bf16* sDh, bf16* sDl, const GlaArgs& a, long base,
                                             bool dots, float (&sd)[8]) {
  const int np = a.K / 32;
  const bf16* src[4] = {(const bf16*)a.hT + base, (const bf16*)a.hTl + base, (const bf16*)a.dhT + base,
                        (const bf16*)a.dhTl + base};
  bf16* dst[4] = {sSh, sSl, sDh, sDl};
  u32x4 x[2][4];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int idx = threadIdx.x + j * kThreads, l = idx & 63, p = (idx >> 6) & 1, vt = idx >> 7;
#pragma unroll
    for (int f = 0; f < 4; ++f) x[j][f] = *(const u32x4*)(src[f] + ((vt * np + p) * 64 + l) * 8);
  }
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int idx = threadIdx.x + j * kThreads, l = idx & 63, p = (idx >> 6) & 1, vt = idx >> 7;
#pragma unroll
    for (int f = 0; f < 4; ++f) {
      bf16* d = dst[f] + (16 * vt + (l & 15)) * LDH + 32 * p + 4 * (l >> 4);
      *(u32x2*)d = u32x2{x[j][f][0], x[j][f][1]};
      *(u32x2*)(d + 16) = u32x2{x[j][f][2], x[j][f][3]};
    }
    if (dots) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        float y[4];
#pragma unroll
        for (int f = 0; f < 4; ++f)
          y[f] = __builtin_bit_cast(float, (i & 1) ? x[j][f][i >> 1] & 0xffff0000u : x[j][f][i >> 1] << 16);
        sd[i] += (y[0] + y[1]) * (y[2] + y[3]);
      }
    }
  }
}

__device__ __forceinline__ void split8(const float* x, bf16x8& hi, bf16x8& lo) {
  float x8[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) x8[i] = x[i];
  split_vec(x8, hi, lo);
}

// acc += (a_hi + a_lo)(b_hi + b_lo), dropping lo x lo
__device__ __forceinline__ void mfma3(f32x16& acc, const bf16x8& ah, const bf16x8& al, const bf16x8& bh,
                                      const bf16x8& bl) {
  acc = mfma(ah, bh, acc);
  acc = mfma(ah, bl, acc);
  acc = mfma(al, bh, acc);
}

}  // namespace

// Operand tables of one (chunk, head): X^T [K/16 row tiles][q][hi, lo][64 lanes] bf16x8, X the decayed
// keys (DIR 0: k e^{b_L - b}) or queries (DIR 1: scale q e^b) -- channel rows 16 rt + m, tokens 32 q + 4 g
// .. +3 and 32 q + 16 + 4 g .. +3, zero past the chunk.  The queries' table lies in two halves of row tiles
// (qfr, qfr2), each [NTG, H] blocks of K/32 row tiles.  State snapshots hT / dhT (hi) and hTl / dhTl (lo):
// B operands [V/16][K/32][64 lanes] bf16x8, lane 16 g + m holding channels 32 p + 4 g .. +3 and
// 32 p + 16 + 4 g .. +3 of column m.

// row tile rt of one (chunk, head)'s table
template <int DIR>
__device__ __forceinline__ bf16x8* x_table(const GlaArgs& a, long gch, int rt) {
  const int nh = a.K / 32;  // row tiles of half a table
  if (DIR == 0) return (bf16x8*)a.xfr + (gch * 2 * nh + rt) * 256;
  return rt < nh ? (bf16x8*)a.qfr + (gch * nh + rt) * 256 : (bf16x8*)a.qfr2 + (gch * nh + rt - nh) * 256;
}

// the four row tiles of channels s0 .. s0 + 63 from x(token, channel - s0), by the four waves of a workgroup
template <int DIR, class F>
__device__ __forceinline__ void x_slab(const GlaArgs& a, long gch, int s0, F x) {
  const int w = wave_id(), l = lane_id(), g = l >> 4, m = l & 15;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int rt = (w + 4 * j) >> 1, q = w & 1, t = 32 * q + 4 * g;
    f32x4 y, z;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      y[i] = x(t + i, 16 * rt + m);
      z[i] = x(t + 16 + i, 16 * rt + m);
    }
    bf16x8 hi, lo;
    split_pair(y, z, hi, lo);
    bf16x8* xf = x_table<DIR>(a, gch, s0 / 16 + rt) + q * 128 + l;
    *gmem(xf) = hi;
    *gmem(xf + 64) = lo;
  }
}

// ===========================================================================
// gla_intra: grid (NTG, H).  b = in-chunk cumsum of gk, A (to a.A) and the keys' operand table.  The table lies where
// b is kept for the backward (gla_mix<0> writes that, after the walk has read the table).
// Waves 0..2 own the 32x32 blocks (0,0), (1,0), (1,1) of A.  The upper block, which nothing reads as part of A,
// holds the chunk's total decay b_L for the walk: channels 32 r .. +31 at the front of its row r.
// Bound by staging and the split factors' exponentials, three workgroups per CU (53 KiB of LDS, so at most 168
// registers).  With the table in a kernel of its own before the walk, B4 T8192 H4 K128 V256 takes 33 + 88 us
// instead of 65, and every short call a launch more (B1 T300 H4 K128 V256: 91 us instead of 88).
// ===========================================================================
template <int K>
__global__ __launch_bounds__(kThreads, 3) void gla_intra_kernel(const GlaArgs a) {
  __shared__ __attribute__((aligned(16))) float sB[BT * LDF];
  __shared__ __attribute__((aligned(16))) float sQ[BT * LDF];
  __shared__ __attribute__((aligned(16))) float sK[BT * LDF];
  __shared__ float sPart[4 * KS];

  const int tid = threadIdx.x, w = wave_id(), l = lane_id();
  const int gc = blockIdx.x, h = blockIdx.y;
  int n, c0, L;
  long bos;
  if (!gla_chunk(a, gc, n, c0, bos, L)) return;
  const long tok0 = bos + c0;
  const long rsk = (long)a.H * K;
  const int I = (w == 0) ? 0 : 1, J = (w == 2) ? 1 : 0;
  // reference row: the block boundary for the off-diagonal block, the middle of a diagonal block
  // (clamped into the valid rows)
  const bool diag = I == J;
  const int mI = diag ? min(32 * I + 16, L - 1) : min(32, L - 1);

  float* Ag = a.A + ((long)gc * a.H + h) * (BT * BT);
  f32x16 acc = zero16();
#pragma unroll 1
  for (int s0 = 0; s0 < K; s0 += KS) {
    // b for this slab: column c = tid & 63 over the rows of quarter qr = tid >> 6
    {
      const int c = tid & 63, qr = tid >> 6;
      float run = 0.f, vals[16];
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const int t = 16 * qr + j;
        run += (a.gk && t < L) ? a.gk[(tok0 + t) * rsk + (long)h * K + s0 + c] : 0.f;
        vals[j] = run;
      }
      sPart[qr * KS + c] = run;
      __syncthreads();
      float off = 0.f;
      for (int p = 0; p < qr; ++p) off += sPart[p * KS + c];
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const int t = 16 * qr + j;
        sB[t * LDF + c] = vals[j] + off;
      }
      if (qr == 3) Ag[BT * ((s0 + c) >> 5) + 32 + (c & 31)] = vals[15] + off;
    }
    slab_to_f32(sQ, a.q32 ? a.q32 + tok0 * rsk + (long)h * K + s0 : nullptr,
                a.q32 ? nullptr : (const bf16*)a.q16 + tok0 * rsk + (long)h * K + s0, rsk, L);
    slab_to_f32(sK, nullptr, (const bf16*)a.k + tok0 * rsk + (long)h * K + s0, rsk, L);
    __syncthreads();
    x_slab<0>(a, (long)gc * a.H + h, s0, [&](int t, int c) {
      return sK[t * LDF + c] * __expf(sB[(L - 1) * LDF + c] - sB[t * LDF + c]);  // (k is zero past the chunk)
    });
    if (w < 3 && (!diag || split_ok(sB, LDF, 32 * I, mI, L, l))) {
      const int r = 32 * I + (l & 31), s = 32 * J + (l & 31);
      for (int k0 = 0; k0 < KS; k0 += 16) {
        const int kb = k0 + ((l >> 5) << 3);
        float xa[8], xb[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int c = kb + i;
          const float bm = sB[mI * LDF + c];
          xa[i] = sQ[r * LDF + c] * __expf(sB[r * LDF + c] - bm);
          xb[i] = sK[s * LDF + c] * __expf(bm - sB[s * LDF + c]);
        }
        bf16x8 ah, al, bh, bl;
        split8(xa, ah, al);
        split8(xb, bh, bl);
        mfma3(acc, ah, al, bh, bl);
      }
    } else if (w < 3) {
      // a diagonal block whose decay is too steep to split: one exponential per pair (<= 1)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int t = 32 * I + acc_row(i), s = 32 * J + acc_col();
        if (s <= t && t < L) {
          float sum = 0.f;
          for (int c = 0; c < KS; ++c)
            sum += sQ[t * LDF + c] * sK[s * LDF + c] * __expf(sB[t * LDF + c] - sB[s * LDF + c]);
          acc[i] += sum;
        }
      }
    }
    __syncthreads();
  }
  if (w < 3) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int t = 32 * I + acc_row(i), s = 32 * J + acc_col();
      Ag[t * BT + s] = (s <= t && t < L) ? a.scale * acc[i] : 0.f;
    }
  }
}

// ===========================================================================
// gla_xprep: one workgroup per (chunk, head, 64 channels): the queries' table (the keys' is written by gla_intra,
// which has k and b at hand).
// ===========================================================================
__global__ __launch_bounds__(kThreads) void gla_xprep_kernel(const GlaArgs a) {
  __shared__ __attribute__((aligned(16))) float sX[BT * LDF];
  const int tid = threadIdx.x;
  const int gc = blockIdx.x, h = blockIdx.y, s0 = blockIdx.z * KS, K = a.K;
  int n, c0, L;
  long bos;
  if (!gla_chunk(a, gc, n, c0, bos, L)) return;
  const long rsk = (long)a.H * K, o = (bos + c0) * rsk + (long)h * K + s0;
#pragma unroll
  for (int j = 0; j < BT * 16 / kThreads; ++j) {
    const int idx = tid + j * kThreads, t = idx >> 4, c = (idx & 15) * 4;
    f32x4 x = f32x4{0.f, 0.f, 0.f, 0.f};
    if (t < L) {
      const f32x4 b = *(const f32x4*)(a.bcum + o + (long)t * rsk + c);
      if (a.q32) {
        x = *(const f32x4*)(a.q32 + o + (long)t * rsk + c);
      } else {
        const bf16x4 y = *(const bf16x4*)((const bf16*)a.q16 + o + (long)t * rsk + c);
        x = f32x4{(float)y[0], (float)y[1], (float)y[2], (float)y[3]};
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) x[i] *= a.scale * __expf(b[i]);
    }
    *(f32x4*)(sX + t * LDF + c) = x;
  }
  __syncthreads();
  x_slab<1>(a, (long)gc * a.H + h, s0, [&](int t, int c) { return sX[t * LDF + c]; });
}

// ===========================================================================
// gla_state<DIR>: two waves per (sequence, head, 32 channels, 32 value columns), 16 columns each.
//   DIR 0: S_next = diag(e^{b_L}) S + X^T V, snapshots of S at each chunk start.
//   DIR 1: dS_prev = diag(e^{b_L}) dS + X^T dO, walking backwards, snapshots of dS (the gradient of the
//          state after each chunk).
// Every state element evolves independently (diagonal decay), so the walk only streams: 8 KiB of X^T,
// 4 KiB of value rows and the decays per chunk go by direct loads into a ring of LDS buffers, the
// snapshots leave as operands.  A chunk takes about 0.3 us to issue but its loads 3 us to arrive (all
// workgroups of a head ask for the same lines at once), so their depth sets the pace: five chunks ahead is
// what two workgroups per CU have LDS for.  B4 T8192 H4 K128 V256: 147 us; with one wave per workgroup, whose
// operation counter bounds it to three chunks, 186 us, or 154 us at 32 columns per wave (then B2 T777 takes
// 13.8 us instead of 10.9).  Before, every wave staged and decayed the token rows itself and stored its
// snapshots to scattered rows: 283 us forward and 301 us backward.
// ===========================================================================
template <int DIR>
__global__ __launch_bounds__(128) void gla_state_kernel(const GlaArgs a) {
  constexpr int NB = 6;                                          // ring of LDS buffers
  constexpr int kY = 8192, kDec = kY + 4096, kStage = kDec + 256;  // X^T, value rows, decays
  constexpr int NL = 7;                                          // loads of a wave per chunk
  __shared__ __attribute__((aligned(256))) char sIn[NB * kStage];
  const int w = __builtin_amdgcn_readfirstlane(wave_id()), l = lane_id(), g = l >> 4, m = l & 15;
  const int K = a.K, V = a.V, H = a.H, nct = K / 32;
  int unit, split;
  if (!unit_map(blockIdx.x, nct * (V / 32), a.N * H, unit, split)) return;
  const int ct0 = split % nct, v0 = 32 * (split / nct), v = v0 + 16 * w + m;
  const int n = unit / H, h = unit % H;
  long bos;
  int len;
  seq_bounds(a.cu, n, a.T, bos, len);
  const int nc = (len + BT - 1) / BT;
  const int gc0 = a.cu ? a.chunk_off[n] : n * a.NT;
  const int rsv = H * V;

  f32x4 S[2];
  {
    const float* init = DIR == 0 ? a.h0 : a.ds_fin;
#pragma unroll
    for (int rt = 0; rt < 2; ++rt)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        S[rt][i] = init ? init[((long)unit * K + 32 * ct0 + 16 * rt + 4 * g + i) * V + v] : 0.f;
  }
  if (nc > 0) {
    // sources of the next loads and their steps from chunk to chunk
    const int cl = nc - 1, cf = DIR == 0 ? 0 : cl;  // last chunk of the sequence, first of the walk
    const int Ll = len - BT * cl, Lf = DIR == 0 && nc > 1 ? BT : Ll;  // their tokens
    const long gf = (long)(gc0 + cf) * H + h, tf = bos + (long)cf * BT;
    constexpr int sg = DIR == 0 ? 1 : -1;
    const char* xp = (const char*)x_table<DIR>(a, gf, 2 * ct0 + w);
    const char* yp = (const char*)((const bf16*)(DIR == 0 ? a.v : a.dout) + (tf * H + h) * (long)V + v0);
    const char* dp = (const char*)(DIR == 0 ? a.A + gf * (BT * BT) + BT * ct0 + 32
                                            : a.bcum + ((tf + Lf - 1) * H + h) * (long)K + 32 * ct0);
    const long xs = (long)sg * H * K * (DIR == 0 ? 256 : 128), ys = (long)sg * BT * rsv * 2, ds = (long)sg * BT * H * (DIR == 0 ? BT : K) * 4;
    // value rows in LDS: 64 bytes per token, the halves of rows t, t + 2 swapped so that a transposing
    // read's four rows lie in different banks; wave w loads rows 32 w .. +31
    const int yt = 32 * w + (l >> 2), ypc = (l & 3) ^ (2 * ((yt >> 1) & 1));
    unsigned yoff[2];
    auto rows = [&](int L) {
#pragma unroll
      for (int j = 0; j < 2; ++j) yoff[j] = (unsigned)(min(16 * j + yt, L - 1) * rsv * 2 + 16 * ypc);
    };
    rows(Lf);
    const unsigned d0 = lds_addr(sIn);
    unsigned d = d0;
    int ei = 0;  // step whose loads come next
    auto issue = [&]() {
      if (ei >= nc) return;
#pragma unroll
      for (int j = 0; j < 4; ++j) lds_load16(xp, 1024 * j + 16 * l, d + 1024 * (4 * w + j));
#pragma unroll
      for (int j = 0; j < 2; ++j) lds_load16(yp, yoff[j], d + kY + 1024 * (2 * w + j));
      lds_load4(dp, 4 * (l & 31), d + kDec);
      d = d == d0 + (NB - 1) * kStage ? d0 : d + kStage;
      if (++ei < nc) {
        xp += xs;
        yp += ys;
        dp += ds;
        if (DIR == 0 && ei == cl && Ll < BT) rows(Ll);
        if (DIR == 1 && ei == 1 && Ll < BT) {
          rows(BT);
          dp += (long)(BT - Ll) * H * K * 4;
        }
      }
    };
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) settle(S[rt]);
#pragma unroll
    for (int e = 0; e < NB - 1; ++e) issue();
    const char* in = sIn;
    char* hh = (char*)((bf16*)(DIR == 0 ? a.hT : a.dhT) + ((gf * V + v0 + 16 * w) * K + 512 * ct0));
    char* hl = (char*)((bf16*)(DIR == 0 ? a.hTl : a.dhTl) + ((gf * V + v0 + 16 * w) * K + 512 * ct0));
    const long hs = (long)sg * H * V * K * 2;
    for (int e = 0; e < nc; ++e, hh += hs, hl += hs) {
      // (younger than step e's loads: those of the up to NB - 2 steps after it and, from step NB - 1 on, the stores of
      // NB - 1 steps; before that the stores are not counted, which waits for no more than a later step's loads)
      static_assert(NB == 6, "the waits of the last steps");
      const int r = min(nc - 1 - e, NB - 2);
      if (e < NB - 1) {
        if (r == NB - 2)
          wait_loads<(NB - 2) * NL>();
        else
          r == 0 ? wait_loads<0>() : r == 1 ? wait_loads<NL>() : r == 2 ? wait_loads<2 * NL>() : wait_loads<3 * NL>();
      } else if (r == NB - 2) {
        wait_loads<(NB - 2) * NL + 2 * (NB - 1)>();
      } else {
        constexpr int st = 2 * (NB - 1);
        r == 0 ? wait_loads<st>() : r == 1 ? wait_loads<NL + st>() : r == 2 ? wait_loads<2 * NL + st>() : wait_loads<3 * NL + st>();
      }
      lds_barrier();  // both waves' loads of step e are in, and nothing reads step e - 1 any more
      issue();
      bf16x8 x[2][2][2], y[2];
      f32x4 dec[2];
#pragma unroll
      for (int rt = 0; rt < 2; ++rt) {
        dec[rt] = *(const f32x4*)(in + kDec + 64 * rt + 16 * g);
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
          for (int p = 0; p < 2; ++p) x[rt][q][p] = *(const bf16x8*)(in + ((rt * 2 + q) * 2 + p) * 1024 + 16 * l);
      }
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int t = 32 * q + 4 * g + (m >> 2), pc = (2 * w + ((m >> 1) & 1)) ^ (2 * ((t >> 1) & 1));
        const char* r = in + kY + 64 * t + 16 * pc + 8 * (m & 1);
        y[q] = join(read_tr(r), read_tr(r + 16 * 64));
      }
      // snapshot of the current (gradient) state
      bf16x8 sh, sl;
      split_pair(S[0], S[1], sh, sl);
      *at<bf16x8>(hh, 16 * l) = sh;
      *at<bf16x8>(hl, 16 * l) = sl;
#pragma unroll
      for (int rt = 0; rt < 2; ++rt) {
#pragma unroll
        for (int i = 0; i < 4; ++i) S[rt][i] *= __expf(dec[rt][i]);
      }
#pragma unroll
      for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
          for (int rt = 0; rt < 2; ++rt) S[rt] = mfma16(x[rt][q][p], y[q], S[rt]);
      in = in == sIn + (NB - 1) * kStage ? sIn : in + kStage;
    }
    wait_loads<0>();  // no direct load may land after the workgroup's LDS is given back
  }
  float* out = DIR == 0 ? a.s_fin : a.dh0;
  if (out) {
#pragma unroll
    for (int rt = 0; rt < 2; ++rt)
#pragma unroll
      for (int i = 0; i < 4; ++i) out[((long)unit * K + 32 * ct0 + 16 * rt + 4 * g + i) * V + v] = S[rt][i];
  }
}

// ===========================================================================
// gla_mix<K, DIR>: one workgroup of 8 waves per (chunk, head).
//   DIR 0: O = scale (Q o e^b) S + A V            DIR 1: dv = (K o e^{b_L - b}) dS + A^T dO
// The decayed rows go to LDS once as hi/lo rows (operands of every value tile), A or A^T as operands; wave
// w then owns value columns 32 w, 32 w + 256, ..: the snapshots are B operands as they lie in HBM, the
// value rows come through the wave's own LDS tile, by which the results leave as whole pieces.
// DIR 0 forms b from gk on the way (a wave's rows in registers, eight wave totals through LDS): 117 -> 126 us at
// B4 T8192 H4 K128 V256, against the pass before the walk that this saves.
// ===========================================================================
template <int K, int DIR>
__global__ __launch_bounds__(512) void gla_mix_kernel(const GlaArgs a) {
  constexpr int NP = K / 32, LDO = 40;
  __shared__ __attribute__((aligned(1024))) char sXh[BT * K * 2], sXl[BT * K * 2];
  __shared__ __attribute__((aligned(1024))) char sW[8][BT * LDO * 2];  // a wave's value rows, then its output tile
  __shared__ __attribute__((aligned(16))) bf16x8 sA[4][2][2][64];
  __shared__ __attribute__((aligned(16))) float sP[DIR == 0 ? 8 * K : 4];  // decay over the waves' rows
  const int w = __builtin_amdgcn_readfirstlane(wave_id()), l = lane_id(), g = l >> 4, m = l & 15;
  const int gc = blockIdx.x, h = blockIdx.y, H = a.H, V = a.V;
  int n, c0, L;
  long bos;
  if (!gla_chunk(a, gc, n, c0, bos, L)) return;
  const long tok0 = bos + c0, gch = (long)gc * H + h;
  const int rsk = H * K, rsv = H * V;
  const unsigned m0 = lds_addr(sW[w]);
  const int yt = l >> 2, ypc = (l & 3) ^ (2 * ((yt >> 1) & 1));
  auto load_y = [&](int v0) {
    const bf16* ys = (const bf16*)(DIR == 0 ? a.v : a.dout) + (tok0 * H + h) * (long)V + v0;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      lds_load16(ys, (unsigned)(min(16 * j + yt, L - 1) * rsv * 2 + 16 * ypc), m0 + 1024 * j);
  };
  if (32 * w < V) load_y(32 * w);
  {
    // wave w's rows 8 w .. +7: lane group l / LPR takes NR consecutive ones
    constexpr int LPR = K / 4, RPW = 64 / LPR, NR = 8 / RPW;  // lanes per row, rows per wave and load, rows per lane
    const int r0 = 8 * w + NR * (l / LPR), c = 4 * (l & (LPR - 1));
    const long o = (tok0 * H + h) * (long)K + c;
    f32x4 x[NR], b[NR], bl = f32x4{0.f, 0.f, 0.f, 0.f};
    if (DIR == 1) bl = *gmem((const f32x4*)(a.bcum + o + (long)(L - 1) * rsk));
#pragma unroll
    for (int j = 0; j < NR; ++j) {
      const long e = o + (long)min(r0 + j, L - 1) * rsk;
      if (DIR == 0)
        b[j] = a.gk && r0 + j < L ? *gmem((const f32x4*)(a.gk + e)) : f32x4{0.f, 0.f, 0.f, 0.f};
      else
        b[j] = *gmem((const f32x4*)(a.bcum + e));
      if (DIR == 0 && a.q32) {
        x[j] = *gmem((const f32x4*)(a.q32 + e));
      } else {
        const bf16x4 y = *gmem((const bf16x4*)((const bf16*)(DIR == 0 ? a.q16 : a.k) + e));
        x[j] = f32x4{(float)y[0], (float)y[1], (float)y[2], (float)y[3]};
      }
    }
    if (DIR == 0) {
      // the cumulative decay: over the lane's rows, the wave's lane groups, the waves; kept for the backward
#pragma unroll
      for (int j = 1; j < NR; ++j) b[j] += b[j - 1];
      f32x4 off = b[NR - 1];
#pragma unroll
      for (int d = LPR; d < 64; d *= 2)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float y = __shfl_up(off[i], d);
          off[i] += l >= d ? y : 0.f;
        }
      if (l >= 64 - LPR) *(f32x4*)(sP + w * K + c) = off;
#pragma unroll
      for (int i = 0; i < 4; ++i) {  // (of the lane groups before this one)
        const float y = LPR < 64 ? __shfl_up(off[i], LPR) : 0.f;
        off[i] = l >= LPR ? y : 0.f;
      }
      __syncthreads();
      for (int p = 0; p < w; ++p) off += *(const f32x4*)(sP + p * K + c);
#pragma unroll
      for (int j = 0; j < NR; ++j) {
        b[j] += off;
        if (r0 + j < L) *gmem((f32x4*)(a.bcum + o + (long)(r0 + j) * rsk)) = b[j];
      }
    }
#pragma unroll
    for (int j = 0; j < NR; ++j) {
      const int t = r0 + j;
      f32x4 y;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        y[i] = t < L ? (DIR == 0 ? a.scale * x[j][i] * __expf(b[j][i]) : x[j][i] * __expf(bl[i] - b[j][i])) : 0.f;
      u32x2 hi, lo;
      split4(y, hi, lo);
      const int d = t * (2 * K) + (((c >> 3) ^ swz(t)) << 4) + 2 * (c & 4);
      *(u32x2*)(sXh + d) = hi;
      *(u32x2*)(sXl + d) = lo;
    }
  }
  {
    const int tt = w >> 1, q = w & 1;
    const float* Ag = a.A + gch * (BT * BT);
    f32x4 x, y;
    if (DIR == 0) {
      x = *gmem((const f32x4*)(Ag + (16 * tt + m) * BT + 32 * q + 4 * g));
      y = *gmem((const f32x4*)(Ag + (16 * tt + m) * BT + 32 * q + 16 + 4 * g));
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        x[i] = *gmem(Ag + (32 * q + 4 * g + i) * BT + 16 * tt + m);
        y[i] = *gmem(Ag + (32 * q + 16 + 4 * g + i) * BT + 16 * tt + m);
      }
    }
    split_pair(x, y, sA[tt][q][0][l], sA[tt][q][1][l]);
  }
  __syncthreads();
  bf16* so = (bf16*)sW[w];
  for (int v0 = 32 * w; v0 < V; v0 += 256) {
    const bf16x8* hh = (const bf16x8*)((const bf16*)(DIR == 0 ? a.hT : a.dhT) + (gch * V + v0) * K);
    const bf16x8* hl = (const bf16x8*)((const bf16*)(DIR == 0 ? a.hTl : a.dhTl) + (gch * V + v0) * K);
    f32x4 acc[4][2];
#pragma unroll
    for (int tt = 0; tt < 4; ++tt)
#pragma unroll
      for (int ct = 0; ct < 2; ++ct) acc[tt][ct] = f32x4{0.f, 0.f, 0.f, 0.f};
    constexpr int PB = NP < 4 ? NP : 4;  // operand pairs loaded at a time
#pragma unroll
    for (int p0 = 0; p0 < NP; p0 += PB) {
      bf16x8 sh[PB][2], sl[PB][2];
#pragma unroll
      for (int p = 0; p < PB; ++p)
#pragma unroll
        for (int ct = 0; ct < 2; ++ct) {
          sh[p][ct] = *at<const bf16x8>(hh + (ct * NP + p0 + p) * 64, 16 * l);
          sl[p][ct] = *at<const bf16x8>(hl + (ct * NP + p0 + p) * 64, 16 * l);
        }
#pragma unroll
      for (int p = 0; p < PB; ++p)
#pragma unroll
        for (int tt = 0; tt < 4; ++tt) {
          const bf16x8 qh = k_frag<K>(sXh, tt, p0 + p, g, m), ql = k_frag<K>(sXl, tt, p0 + p, g, m);
#pragma unroll
          for (int ct = 0; ct < 2; ++ct) {
            acc[tt][ct] = mfma16(qh, sh[p][ct], acc[tt][ct]);
            acc[tt][ct] = mfma16(qh, sl[p][ct], acc[tt][ct]);
            acc[tt][ct] = mfma16(ql, sh[p][ct], acc[tt][ct]);
          }
        }
    }
    wait_loads<0>();
    bf16x8 y[2][2];
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int ct = 0; ct < 2; ++ct) {
        const int t = 32 * q + 4 * g + (m >> 2), pc = (2 * ct + ((m >> 1) & 1)) ^ (2 * ((t >> 1) & 1));
        const char* r = sW[w] + 64 * t + 16 * pc + 8 * (m & 1);
        y[q][ct] = join(read_tr(r), read_tr(r + 16 * 64));
      }
#pragma unroll
    for (int tt = 0; tt < 4; ++tt)
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        if (DIR == 0 ? q > tt / 2 : q < tt / 2) continue;  // (the other side of A's diagonal)
        const bf16x8 ah = sA[tt][q][0][l], al = sA[tt][q][1][l];
#pragma unroll
        for (int ct = 0; ct < 2; ++ct) {
          acc[tt][ct] = mfma16(ah, y[q][ct], acc[tt][ct]);
          acc[tt][ct] = mfma16(al, y[q][ct], acc[tt][ct]);
        }
      }
    if (DIR == 1 && a.dv32) {
#pragma unroll
      for (int tt = 0; tt < 4; ++tt)
#pragma unroll
        for (int ct = 0; ct < 2; ++ct)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int t = 16 * tt + 4 * g + i;
            if (t < L) a.dv32[((tok0 + t) * H + h) * (long)V + v0 + 16 * ct + m] = acc[tt][ct][i];
          }
    }
    bf16* og = (bf16*)(DIR == 0 ? a.o : a.dv);
    // (the value rows are read: the tile takes the results; rows past the chunk drop)
    if (og) {
#pragma unroll
      for (int tt = 0; tt < 4; ++tt)
#pragma unroll
        for (int ct = 0; ct < 2; ++ct)
#pragma unroll
          for (int i = 0; i < 4; ++i) so[(16 * tt + 4 * g + i) * LDO + 16 * ct + m] = (bf16)acc[tt][ct][i];
      __builtin_amdgcn_wave_barrier();
      asm volatile("" ::: "memory");
      const __amdgpu_buffer_rsrc_t ro = buf_rsrc(og + (tok0 * H + h) * (long)V, ((L - 1) * rsv + V) * 2);
      u32x4 row[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) row[j] = *(const u32x4*)(so + (16 * j + (l >> 2)) * LDO + 8 * (l & 3));
#pragma unroll
      for (int j = 0; j < 4; ++j)
        __builtin_amdgcn_raw_buffer_store_b128(row[j], ro, ((16 * j + (l >> 2)) * rsv + v0 + 8 * (l & 3)) * 2, 0, 0);
    }
    // the next value rows into the same tile, once this pass's LDS reads are complete
    if (v0 + 256 < V) {
      __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
      load_y(v0 + 256);
    }
  }
}

// ===========================================================================
// gla_bwd_dqk: grid NTG * H * (K/64), XCD-mapped.  dq, dk and dgk for one 64-channel slab: dgk is the suffix
// sum of dG = q dq - k dk over the chunk's rows plus that of all later chunks.  The later chunks see this
// one only through its end state, so theirs is sum_v S_end dS_end of the channel, with
//   S_end = e^{b_L} S_start + sum_t e^{b_L - b_t} k_t v_t
//   =>  e^{b_L} sum_v S_start dS_end + sum_t k_t (the inter-chunk part of dk_t),
// both already here (at a sequence's last chunk: the fp32 final state and its gradient).
// Two workgroups per CU wait on their loads, so the dot products cost little: B4 T8192 H4 K128 V256, 290 ->
// 302 us, where a serial carry over the chunks and a pass adding it to dgk took 50 + 35 us.
// ===========================================================================
template <int K>
__global__ __launch_bounds__(kThreads) void gla_bwd_dqk_kernel(const GlaArgs a) {
  // loop phase: dO, V [64][LDH] bf16 and S, dS pieces [v][c] hi/lo; post phase: q (then dG in its
  // place: each element of dG is written by the one thread that last reads that element of q), k,
  // b, dA.  Under 80 KiB, so two workgroups share a CU.
  constexpr long kLoop = 6L * 64 * LDH * 2;
  constexpr long kPost = 3L * BT * LDF * 4 + (long)BT * (BT + 1) * 4;
  __shared__ __attribute__((aligned(16))) char smem[kLoop > kPost ? kLoop : kPost];
  __shared__ float sPart[4 * KS];
  __shared__ float sTerm[KS];
  __shared__ float sSD[2 * KS];    // sum_v S_start dS_end of a channel, two parts
  __shared__ float sKD[2 * KS];    // sum_t k_t (inter-chunk dk_t), the two row blocks
  bf16* sO = (bf16*)smem;
  bf16* sV = sO + 64 * LDH;
  bf16* sSh = sV + 64 * LDH;
  bf16* sSl = sSh + 64 * LDH;
  bf16* sDh = sSl + 64 * LDH;
  bf16* sDl = sDh + 64 * LDH;
  float* sQ = (float*)smem;
  float* sK = sQ + BT * LDF;
  float* sBb = sK + BT * LDF;
  float* sG = sQ;
  float* sdA = sBb + BT * LDF;

  const int tid = threadIdx.x, w = wave_id(), l = lane_id();
  // the K / KS key blocks of a (chunk, head) unit share its operands: one XCD (L2) per unit
  int unit, kb;
  xcd_map(blockIdx.x, K / KS, a.NTG * a.H, unit, kb);
  const int gc = unit / a.H, h = unit % a.H, s0 = kb * KS;
  int n, c0, L;
  long bos;
  if (!gla_chunk(a, gc, n, c0, bos, L)) return;
  const long tok0 = bos + c0;
  const long rsk = (long)a.H * K, rsv = (long)a.H * a.V;
  const int tr = w >> 1, tc = w & 1;
  const int I = (w == 0) ? 0 : 1, J = (w == 2) ? 1 : 0;  // dA block of waves 0..2

  f32x16 dqr = zero16(), dkr = zero16(), dA = zero16();
  float sd[8] = {};
  for (int v0 = 0; v0 < a.V; v0 += 64) {
    const long sbase = (((long)gc * a.H + h) * a.V + v0) * K + 16 * s0;
    tile_bf16(sO, (const bf16*)a.dout + tok0 * rsv + (long)h * a.V + v0, rsv, L);
    tile_bf16(sV, (const bf16*)a.v + tok0 * rsv + (long)h * a.V + v0, rsv, L);
    tile_op_pair(sSh, sSl, sDh, sDl, a, sbase, a.dgk != nullptr, sd);
    __syncthreads();
    for (int k0 = 0; k0 < 64; k0 += 16) {
      const bf16x8 oa = frag_rm(sO + tr * 32 * LDH + k0, LDH);
      const bf16x8 va = frag_rm(sV + tr * 32 * LDH + k0, LDH);
      dqr = mfma(oa, frag32_tr(sSh + k0 * LDH + tc * 32, LDH), dqr);
      dqr = mfma(oa, frag32_tr(sSl + k0 * LDH + tc * 32, LDH), dqr);
      dkr = mfma(va, frag32_tr(sDh + k0 * LDH + tc * 32, LDH), dkr);
      dkr = mfma(va, frag32_tr(sDl + k0 * LDH + tc * 32, LDH), dkr);
      if (w < 3) dA = mfma(frag_rm(sO + I * 32 * LDH + k0, LDH), frag_rm(sV + J * 32 * LDH + k0, LDH), dA);
    }
    __syncthreads();
  }

  // post phase
  if (a.dgk) {
    // the sixteen value columns of a lane group; the wave's channels are 32 (w & 1) + 4 g + (i & 3) + 16 (i >> 2)
#pragma unroll
    for (int i = 0; i < 8; ++i) {
#pragma unroll
      for (int d = 1; d < 16; d <<= 1) sd[i] += __shfl_xor(sd[i], d);
      if ((l & 15) == 0) sSD[(w >> 1) * KS + 32 * (w & 1) + 4 * (l >> 4) + (i & 3) + 16 * (i >> 2)] = sd[i];
    }
  }
  slab_to_f32(sQ, a.q32 ? a.q32 + tok0 * rsk + (long)h * K + s0 : nullptr,
              a.q32 ? nullptr : (const bf16*)a.q16 + tok0 * rsk + (long)h * K + s0, rsk, L);
  slab_to_f32(sK, nullptr, (const bf16*)a.k + tok0 * rsk + (long)h * K + s0, rsk, L);
  slab_to_f32(sBb, a.bcum + tok0 * rsk + (long)h * K + s0, nullptr, rsk, L, true);
  if (w < 3) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int t = 32 * I + acc_row(i), s = 32 * J + acc_col();
      sdA[t * (BT + 1) + s] = (s <= t && t < L) ? a.scale * dA[i] : 0.f;
    }
  } else {
#pragma unroll
    for (int i = 0; i < 16; ++i) sdA[acc_row(i) * (BT + 1) + 32 + acc_col()] = 0.f;
  }
  // final-state term of dG: rowsum over v of dS_final o S_final (last chunk of the sequence only)
  long len_seq;
  {
    long b2;
    int len2;
    seq_bounds(a.cu, n, a.T, b2, len2);
    len_seq = len2;
  }
  const bool last = (c0 + L == len_seq);
  if (last && a.ds_fin && a.s_fin_in && a.dgk) {
    const int c = tid & 63, part = tid >> 6;
    const long base = (((long)n * a.H + h) * K + s0 + c) * a.V;
    float acc_t = 0.f;
    for (int v = part; v < a.V; v += 4) acc_t += a.ds_fin[base + v] * a.s_fin_in[base + v];
    sPart[part * KS + c] = acc_t;
  }
  __syncthreads();
  if (tid < KS) {
    sTerm[tid] = (last && a.ds_fin && a.s_fin_in && a.dgk)
                     ? sPart[tid] + sPart[KS + tid] + sPart[2 * KS + tid] + sPart[3 * KS + tid]
                     : 0.f;
  }

  // intra-chunk parts.  The dq rows of block tr take the keys of block tr (the diagonal block) and,
  // for tr = 1, the keys of block 0; the dk rows (keys) of block tr take the queries of block tr and,
  // for tr = 0, the queries of block 1.  The off-diagonal block (dxo) splits its pairwise factor at
  // row mB = 32, where both factors are <= 1; the diagonal block at its middle row mR while that is
  // safe for this wave's channels (split_ok), else with one exponential per pair, in which case dqi
  // and dki carry their factors whole.
  const int mR = min(32 * tr + 16, L - 1), mB = min(32, L - 1);
  f32x16 dqi = zero16(), dki = zero16(), dxo = zero16();
  const bool fast = split_ok(sBb, LDF, 32 * tr, mR, L, tc * 32 + (l & 31));
  {
    const int c = tc * 32 + (l & 31);
    const float bm = sBb[mR * LDF + c], bb = sBb[mB * LDF + c];
    if (tr == 1) {
      for (int k0 = 0; k0 < 32; k0 += 16) {      // dq: keys of block 0
        bf16x8 ah, al, bh, bl;
        frag_rm_f32(sdA + 32 * (BT + 1) + k0, BT + 1, ah, al);
        float xb[8];
        const int kb = k0 + ((l >> 5) << 3);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int s = kb + i;
          xb[i] = sK[s * LDF + c] * __expf(bb - sBb[s * LDF + c]);
        }
        split8(xb, bh, bl);
        mfma3(dxo, ah, al, bh, bl);
      }
    } else {
      for (int k0 = 32; k0 < BT; k0 += 16) {     // dk: queries of block 1
        bf16x8 ah, al, bh, bl;
        frag_cm_f32(sdA + k0 * (BT + 1), BT + 1, ah, al);
        float xb[8];
        const int kb = k0 + ((l >> 5) << 3);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int t = kb + i;
          xb[i] = sQ[t * LDF + c] * __expf(sBb[t * LDF + c] - bb);
        }
        split8(xb, bh, bl);
        mfma3(dxo, ah, al, bh, bl);
      }
    }
    if (fast) {
      for (int k0 = 32 * tr; k0 < 32 * tr + 32; k0 += 16) {
        bf16x8 ah, al, bh, bl;
        frag_rm_f32(sdA + tr * 32 * (BT + 1) + k0, BT + 1, ah, al);
        float xb[8];
        const int kb = k0 + ((l >> 5) << 3);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int s = kb + i;
          xb[i] = sK[s * LDF + c] * __expf(bm - sBb[s * LDF + c]);
        }
        split8(xb, bh, bl);
        mfma3(dqi, ah, al, bh, bl);
      }
      for (int k0 = 32 * tr; k0 < 32 * tr + 32; k0 += 16) {
        bf16x8 ah, al, bh, bl;
        frag_cm_f32(sdA + tr * 32 + k0 * (BT + 1), BT + 1, ah, al);
        float xb[8];
        const int kb = k0 + ((l >> 5) << 3);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int t = kb + i;
          xb[i] = sQ[t * LDF + c] * __expf(sBb[t * LDF + c] - bm);
        }
        split8(xb, bh, bl);
        mfma3(dki, ah, al, bh, bl);
      }
    } else {
      // dq_r = sum_{s <= r} dA_rs k_s e^{b_r - b_s},  dk_r = sum_{t >= r} dA_tr q_t e^{b_t - b_r}
      // over the block's valid rows, one exponential (<= 1) per pair
      const int cc = tc * 32 + acc_col(), r0 = 32 * tr, r1 = min(32 * tr + 32, L);
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int r = r0 + acc_row(i);
        float sq = 0.f, sk = 0.f;
        if (r < L) {
          const float br = sBb[r * LDF + cc];
          for (int j = r0; j <= r; ++j)
            sq += sdA[r * (BT + 1) + j] * sK[j * LDF + cc] * __expf(br - sBb[j * LDF + cc]);
          for (int j = r; j < r1; ++j)
            sk += sdA[j * (BT + 1) + r] * sQ[j * LDF + cc] * __expf(sBb[j * LDF + cc] - br);
        }
        dqi[i] = sq;
        dki[i] = sk;
      }
    }
  }
  __syncthreads();
  // combine, write dq/dk, form dG
  {
    const int c = tc * 32 + acc_col();
    const float bm = sBb[mR * LDF + c], bb = sBb[mB * LDF + c], bl_ = sBb[(L - 1) * LDF + c];
    float kd = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int t = tr * 32 + acc_row(i);
      const float bt = sBb[t * LDF + c];
      float dq = a.scale * __expf(bt) * dqr[i] + (fast ? __expf(bt - bm) * dqi[i] : dqi[i]);
      const float dke = __expf(bl_ - bt) * dkr[i];
      kd += sK[t * LDF + c] * dke;
      float dk = dke + (fast ? __expf(bm - bt) * dki[i] : dki[i]);
      if (tr == 1) dq += __expf(bt - bb) * dxo[i];
      else dk += __expf(bb - bt) * dxo[i];
      float g = 0.f;
      if (t < L) {
        a.dq32[(tok0 + t) * rsk + (long)h * K + s0 + c] = dq;
        a.dk32[(tok0 + t) * rsk + (long)h * K + s0 + c] = dk;
        g = sQ[t * LDF + c] * dq - sK[t * LDF + c] * dk;
      }
      sG[t * LDF + c] = g;
    }
    kd += __shfl_xor(kd, 32);
    if (l < 32) sKD[tr * KS + c] = kd;
  }
  if (!a.dgk) return;
  __syncthreads();
  // suffix sums over the chunk's rows: column c = tid & 63, quarter qr = tid >> 6 (rows 16 qr ..)
  {
    const int c = tid & 63, qr = tid >> 6;
    float run = 0.f, vals[16];
#pragma unroll
    for (int j = 15; j >= 0; --j) {
      run += sG[(16 * qr + j) * LDF + c];
      vals[j] = run;
    }
    sPart[qr * KS + c] = run;
    __syncthreads();
    float off = last ? sTerm[c] : __expf(sBb[(L - 1) * LDF + c]) * (sSD[c] + sSD[KS + c]) + (sKD[c] + sKD[KS + c]);
    for (int p = qr + 1; p < 4; ++p) off += sPart[p * KS + c];
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const int t = 16 * qr + j;
      if (t < L) a.dgk[(tok0 + t) * rsk + (long)h * K + s0 + c] = vals[j] + off;
    }
  }
}

// ---------------------------------------------------------------------------
// launcher
// ---------------------------------------------------------------------------
template <int K>
hipError_t launch_gla_k(int stage, const GlaArgs& a, hipStream_t st) {
  const dim3 blk(kThreads);
  const int NTG = a.NTG, H = a.H;
  switch (stage) {
    case kGlaIntra:
      hipLaunchKernelGGL(gla_intra_kernel<K>, dim3(NTG, H), blk, 0, st, a);
      break;
    case kGlaFwdState:
      hipLaunchKernelGGL(gla_state_kernel<0>, dim3((a.N * H + 7) / 8 * 8 * (K / 32) * (a.V / 32)), dim3(128), 0, st, a);
      break;
    case kGlaFwdO:
      hipLaunchKernelGGL((gla_mix_kernel<K, 0>), dim3(NTG, H), dim3(512), 0, st, a);
      break;
    case kGlaBwdState:
      hipLaunchKernelGGL(gla_xprep_kernel, dim3(NTG, H, K / KS), blk, 0, st, a);
      hipLaunchKernelGGL(gla_state_kernel<1>, dim3((a.N * H + 7) / 8 * 8 * (K / 32) * (a.V / 32)), dim3(128), 0, st, a);
      break;
    case kGlaBwdDv:
      hipLaunchKernelGGL((gla_mix_kernel<K, 1>), dim3(NTG, H), dim3(512), 0, st, a);
      break;
    case kGlaBwdDqk:
      hipLaunchKernelGGL(gla_bwd_dqk_kernel<K>, dim3(NTG * H * (K / KS)), blk, 0, st, a);
      break;
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_gla_stage(int stage, const GlaArgs& a, hipStream_t st) {
  if (a.NTG <= 0 || a.H <= 0 || a.N <= 0) return hipSuccess;
  switch (a.K) {
    case 64: return launch_gla_k<64>(stage, a, st);
    case 128: return launch_gla_k<128>(stage, a, st);
    case 256: return launch_gla_k<256>(stage, a, st);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace ccq
