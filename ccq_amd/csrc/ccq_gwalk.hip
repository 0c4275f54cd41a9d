// State walks of the gated delta rule (chunk size 64), forward and backward, on gfx950.
//
// A workgroup owns one (sequence, head) and 16 NG state columns and walks the chunks; the state stays
// in the registers of its waves.  The chunk's pseudo-values are U = T diag(beta) (V - diag(gamma) K S)
// (T = (I + A)^-1 of the WY form), so a step needs k, v, T and the gates only:
//   forward   U = Tb V + Tb X,  Tb = T diag(beta),  X = -diag(gamma) K S
//             S <- gamma_L S + K^T diag(gamma_L / gamma) U
//   backward  dU = P^T dO + diag(gamma_L / gamma) K dS'       Y = diag(beta gamma) T^T dU
//             dS <- gamma_L dS' + Qc^T diag(scale gamma) dO - K^T Y
// A walk is a chain of dependent products, one link per chunk, and its time is the chain's latency:
//   * wave w owns state rows [KS w, KS w + KS) as 16x16 accumulator tiles.  Two tiles are a B operand of
//     the next product as they stand (contraction slots 0-3: rows 4 g .. +3 of the first tile, 4-7: of the
//     second, g the lane's 16-lane group), the A operand's slots being read in that order.
//   * products that contract over all state rows (K S, K dS') are summed over the waves through LDS;
//     wave w then owns the 16 token rows of tile w of X and U (dU and Y), which it passes on through
//     LDS in B operand order (8-byte pieces written, 16-byte operands read).  Three exchanges and
//     barriers per step.
//   * consecutive lanes of every load and store are consecutive in memory (a 16-byte access whose lanes lie
//     in different rows is served lane by lane: 35 - 70 cycles instead of 16 per instruction): the state
//     snapshots, U and dU leave in operand and tile order too.
//   * a chunk's k, T, v and gates go to LDS by direct loads (no registers, no conversion: gdn_tprep and
//     gdn_qprep write Tb, T^T, the gates and Qc^T as tables in operand order).  Everything of chunk c is
//     in registers by the second barrier of its step (K^T for the end of the step, and K of chunk c + 1
//     from there on), so two buffers give the loads of chunk c + 2 a whole step to land.
//
// Measured at K = 256, V = 512 (us; before: 32-column walks with the state in LDS, w and u from prep):
//                         prep       forward walk   output     backward walk (+ gdn_qprep)
//   B1 T32768 H6          430 -> 52  3180 -> 948    738 -> 380  4850 -> 1722 + 84
//   B4 T4096 H4           145 -> 28   427 -> 195    245 -> 138   645 -> 466 + 28
//   B1 T1531 H6            36 -> 10   147 -> 48      56 -> 22
// A forward step takes 1.85 us with 16 columns per workgroup: about 0.75 us each of LDS transfers, vector
// and matrix instructions, which one workgroup per CU overlaps little; the chain, not HBM, is the bound.
#include "ccq_oper.h"
#include "ccq_params.h"

#include <type_traits>

namespace ccq {

namespace {

constexpr int BT = 64;

template <int K, int NWV>
struct GwCfg {
  static constexpr int NW = NWV;                       // waves per column group
  static constexpr int KS = K / NW;                    // state rows per wave
  static constexpr int NP = KS / 32;                   // B operands (pairs of tiles) of a column tile
  static constexpr int NRT = KS / 16;                  // row tiles
  static constexpr int TPW = NW < 4 ? 4 / NW : 1;      // token tiles owned by a wave (w < 4): w, w + NW, ..
};

// largest magnitude's bit pattern over the four 16-lane groups (lanes l, l ^ 16, l ^ 32, l ^ 48)
__device__ __forceinline__ unsigned group4_umax(unsigned v) {
  const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
  v = max((unsigned)r[0], (unsigned)r[1]);
  const auto s = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  return max((unsigned)s[0], (unsigned)s[1]);
}

// sequence, first token and length of a chunk; false for the padding entries of a varlen launch
__device__ __forceinline__ bool chunk_of(const GdnArgs& a, int gc, int& n, long& tok0, int& L) {
  if (a.cu) {
    n = a.chunk_idx[2 * gc];
    if (n < 0) return false;
    const int c0 = a.chunk_idx[2 * gc + 1] * BT;
    tok0 = (long)a.cu[n] + c0;
    L = min(BT, (int)(a.cu[n + 1] - a.cu[n]) - c0);
  } else {
    n = gc / a.NT;
    const int c0 = (gc % a.NT) * BT;
    tok0 = (long)n * a.T + c0;
    L = min(BT, a.T - c0);
  }
  return true;
}

// Tb / T^T operand table of one (chunk, head): [2][6 blocks][hi, lo][64 lanes] bf16x8.  Lower-triangle
// blocks (tile tt, contraction half q): Tb (0,0) (1,0) (2,0) (2,1) (3,0) (3,1), T^T (0,0) (0,1) (1,0)
// (1,1) (2,1) (3,1).
constexpr int kTfr = 2 * 6 * 2 * 64;  // bf16x8 per (chunk, head)
constexpr int kTfrBytes = kTfr * 16;
__device__ __forceinline__ int t_blk(int tt, int q) { return tt < 2 ? tt : 2 * (tt - 1) + q; }
__device__ __forceinline__ int tt_blk(int tt, int q) { return tt < 2 ? 2 * tt + q : 2 + tt; }
// gate table of one (chunk, head): rows beta gamma, (free), gamma_L / gamma (0 past the chunk), gamma
// (the last token's past the chunk), 64 floats each
constexpr int kTok = 4 * BT;

// The direct loads of a walk.  A chunk's operands are NPC pieces of 1 KiB -- the k tile, the operand table
// of T (or T^T), a tile of 16 NG value columns, the gates -- at the same places of each LDS buffer; wave wv
// of NWV loads pieces wv, wv + NWV, ...  Source addresses and their step
// from chunk to chunk stay in scalar registers, lane offsets in vector registers: they change only for
// a partial chunk.
template <int K, int NG, int NWV>
struct Feed {
  static constexpr int NK = K / 8, NT = 12, NV = 2 * NG, NPC = NK + NT + NV + 1, N = (NPC + NWV - 1) / NWV;
  static constexpr int kT = NK * 1024, kV = kT + NT * 1024, kTokOff = kV + NV * 1024, kBytes = NPC * 1024;
  const char* src[N];
  long step[N];
  unsigned off[N], m0;
  // sources at the first chunk loaded; dir: +1 or -1 chunks per load; full: the first chunk has 64 tokens
  __device__ __forceinline__ void init(const char* k, const char* t, const char* v, const char* tok, int H, int V, int dir,
                                       char* lds, int wv, int l) {
    m0 = lds_addr(lds) + 1024 * wv;
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const int i = wv + NWV * j;
      if (i < NK) {
        src[j] = k;
        step[j] = (long)dir * BT * H * K * 2;
      } else if (i < NK + NT) {
        src[j] = t + 1024 * (i - NK);
        step[j] = (long)dir * H * (kTfrBytes);
      } else if (i < NK + NT + NV) {
        src[j] = v;
        step[j] = (long)dir * BT * H * V * 2;
      } else {
        src[j] = tok;
        step[j] = (long)dir * H * (kTok * 4);
      }
    }
    rows(H, V, BT, wv, l);
  }
  // lane offsets of a chunk of L tokens
  __device__ __forceinline__ void rows(int H, int V, int L, int wv, int l) {
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const int i = wv + NWV * j;
      off[j] = i < NK ? k_tile_off<K>(i, H * K, L, l)
                      : i >= NK + NT && i < NK + NT + NV ? row_tile_off<16 * NG>(i - NK - NT, H * V, L, l) : 16 * l;
    }
  }
  // The workgroups of a unit walk its chunks together, so a chunk's lines would all be waited for from HBM
  // by every one of them.  Each workgroup therefore touches its share of a later chunk (piece `p` of k, T or
  // the gates, into a scratch KiB of LDS): by the time the chunk is loaded its lines are in the XCD's L2.
  const char* psrc;
  long pstep;
  unsigned poff, pm0;
  bool pf;
  __device__ __forceinline__ void init_prefetch(const char* k, const char* t, const char* tok, int H, int dir, int p,
                                                char* lds, int l) {
    pf = p < NK + NT + 1;
    pm0 = lds_addr(lds);
    psrc = p < NK ? k : p < NK + NT ? t + 1024 * (p - NK) : tok;
    pstep = (long)dir * H * (p < NK ? BT * K * 2 : p < NK + NT ? kTfrBytes : kTok * 4);
    poff = p < NK ? k_tile_off<K>(p, H * K, BT, l) : 16 * l;
  }
  __device__ __forceinline__ void prefetch(int c) {
    if (pf) lds_load16(psrc + c * pstep, poff, pm0);
  }
  // part P of 3 of a chunk's loads (the waves' loads go through one 64-byte path per CU: issued together they
  // would hold each wave for the whole transfer)
  template <int P>
  __device__ __forceinline__ void load(int buf, int wv) {
    const unsigned d = m0 + (buf ? kBytes : 0);
#pragma unroll
    for (int j = P * N / 3; j < (P + 1) * N / 3; ++j) {
      if (NWV * (j + 1) > NPC && wv + NWV * j >= NPC) break;  // (wave-uniform)
      lds_load16(src[j], off[j], d + 1024 * NWV * j);
      src[j] += step[j];
    }
  }
};

// State snapshots hT / dhT of one (chunk, head): B operands [V/16][K/32][64 lanes] of 8 values, lane
// 16 g + m holding rows 32 p + 4 g .. +3 and 32 p + 16 + 4 g .. +3 of column m.  U / dU of one (chunk,
// head): accumulator tiles [V/16][4 token tiles][64 lanes] of four consecutive tokens.

}  // namespace

// ===========================================================================
// gdn_tprep: one wave per (chunk, head).  A = strict_lower(beta_r Gamma_rc (K K^T)_rc) from operands
// loaded straight from k (a row fragment is both A and B operand), T = (I + A)^-1 by 16x16 blocks in
// fp32: the diagonal blocks by forward substitution (one column per lane), the others by distance d,
// T_IJ = -D_I sum_{M=J}^{I-1} A_IM T_MJ, on fp32 MFMAs whose B operand is the accumulator layout as it
// stands (contraction index 4 g + s at step s).  A single wave needs no barrier, and eight of them
// share a CU (LDS), which hides the serial substitution.
// ===========================================================================
template <int K>
__global__ __launch_bounds__(64) void gdn_tprep_kernel(const GdnArgs a) {
  constexpr int LDA = BT + 4;
  __shared__ __attribute__((aligned(16))) float sA[BT * LDA];
  __shared__ __attribute__((aligned(16))) float sG[BT], sB[BT];
  const int l = lane_id(), g = l >> 4, m = l & 15;
  const int gc = blockIdx.x, h = blockIdx.y;
  int n, L;
  long tok0;
  if (!chunk_of(a, gc, n, tok0, L)) return;
  const long gch = (long)gc * a.H + h;
  const int rsk = a.H * K;

  f32x4 acc[10];  // tiles (0,0) (1,0) (1,1) (2,0) ..
#pragma unroll
  for (int i = 0; i < 10; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  const __amdgpu_buffer_rsrc_t rk = buf_rsrc((const bf16*)a.k + (tok0 * a.H + h) * K, ((L - 1) * rsk + K) * 2);
  constexpr int KB = K < 128 ? K : 128;
#pragma unroll
  for (int k0 = 0; k0 < K; k0 += KB) {
    u32x4 f[4][KB / 32];
#pragma unroll
    for (int kk = 0; kk < KB / 32; ++kk)
#pragma unroll
      for (int tt = 0; tt < 4; ++tt)
        f[tt][kk] = __builtin_amdgcn_raw_buffer_load_b128(rk, ((16 * tt + m) * rsk + k0 + 32 * kk + 8 * g) * 2, 0, 0);
#pragma unroll
    for (int kk = 0; kk < KB / 32; ++kk)
#pragma unroll
      for (int tt = 0; tt < 4; ++tt)
#pragma unroll
        for (int ss = 0; ss <= tt; ++ss)
          acc[tt * (tt + 1) / 2 + ss] = mfma16(__builtin_bit_cast(bf16x8, f[tt][kk]), __builtin_bit_cast(bf16x8, f[ss][kk]),
                                               acc[tt * (tt + 1) / 2 + ss]);
  }
  {
    const long t = (tok0 + min(l, L - 1)) * a.H + h;
    const float x = wave_scan_incl((l < L && a.g) ? a.g[t] : 0.f);
    const float be = l < L ? a.beta[t] : 0.f;
    const float xl = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), 63));  // (g = 0 past the chunk)
    sG[l] = x;
    sB[l] = be;
    if (l < L) a.gcum[t] = x;
    float* tk = a.tok + gch * kTok + l;
    tk[0] = be * __expf(x);
    tk[2 * BT] = l < L ? __expf(xl - x) : 0.f;
    tk[3 * BT] = __expf(x);
  }
  __syncthreads();
#pragma unroll
  for (int tt = 0; tt < 4; ++tt) {
    const f32x4 gr = *(const f32x4*)(sG + 16 * tt + 4 * g), br = *(const f32x4*)(sB + 16 * tt + 4 * g);
#pragma unroll
    for (int ss = 0; ss <= tt; ++ss) {
      const float gs = sG[16 * ss + m];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const bool keep = ss < tt || 4 * g + i > m;
        const float e = __expf(keep ? gr[i] - gs : 0.f);
        sA[(16 * tt + 4 * g + i) * LDA + 16 * ss + m] = keep ? br[i] * e * acc[tt * (tt + 1) / 2 + ss][i] : 0.f;
      }
    }
  }
  __syncthreads();
  {
    const float* ap = sA + 16 * g * LDA + 16 * g;
    float x[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      float s = i == m ? 1.f : 0.f;
#pragma unroll
      for (int j = 0; j < i; ++j) s -= ap[i * LDA + j] * x[j];
      x[i] = s;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 16; ++i) sA[(16 * g + i) * LDA + 16 * g + m] = x[i];
  }
  __syncthreads();
  f32x4 T[4][4];
#pragma unroll
  for (int I = 0; I < 4; ++I)
#pragma unroll
    for (int i = 0; i < 4; ++i) T[I][I][i] = sA[(16 * I + 4 * g + i) * LDA + 16 * I + m];
#pragma unroll
  for (int d = 1; d < 4; ++d)
#pragma unroll
    for (int J = 0; J + d < 4; ++J) {
      const int I = J + d;
      f32x4 y = f32x4{0.f, 0.f, 0.f, 0.f}, z = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int M = J; M < I; ++M) {
        const f32x4 am = *(const f32x4*)(sA + (16 * I + m) * LDA + 16 * M + 4 * g);
#pragma unroll
        for (int s = 0; s < 4; ++s) y = __builtin_amdgcn_mfma_f32_16x16x4f32(am[s], T[M][J][s], y, 0, 0, 0);
      }
      const f32x4 di = *(const f32x4*)(sA + (16 * I + m) * LDA + 16 * I + 4 * g);
#pragma unroll
      for (int s = 0; s < 4; ++s) z = __builtin_amdgcn_mfma_f32_16x16x4f32(di[s], y[s], z, 0, 0, 0);
      T[I][J] = -z;
    }
  __syncthreads();
#pragma unroll
  for (int I = 0; I < 4; ++I)
#pragma unroll
    for (int J = 0; J < 4; ++J)
      if (I != J)
#pragma unroll
        for (int i = 0; i < 4; ++i) sA[(16 * I + 4 * g + i) * LDA + 16 * J + m] = J < I ? T[I][J][i] : 0.f;
  __syncthreads();
  float* tg = a.tmat + gch * (BT * BT);
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const int r = 4 * j + g;
    *gmem((f32x4*)(tg + r * BT + 4 * m)) = *(const f32x4*)(sA + r * LDA + 4 * m);
  }
  bf16x8* fr = (bf16x8*)a.tfr + gch * kTfr + l;
#pragma unroll
  for (int tt = 0; tt < 4; ++tt)
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      bf16x8 hi, lo;
      if (q <= tt / 2) {
        const float *p = sA + (16 * tt + m) * LDA + 32 * q + 4 * g, *be = sB + 32 * q + 4 * g;
        split_pair(*(const f32x4*)p * *(const f32x4*)be, *(const f32x4*)(p + 16) * *(const f32x4*)(be + 16), hi, lo);
        *gmem(fr + t_blk(tt, q) * 128) = hi;
        *gmem(fr + t_blk(tt, q) * 128 + 64) = lo;
      }
      if (q >= tt / 2) {
        const float* p = sA + (32 * q + 4 * g) * LDA + 16 * tt + m;
        f32x4 x, y;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          x[i] = p[i * LDA];
          y[i] = p[(16 + i) * LDA];
        }
        split_pair(x, y, hi, lo);
        *gmem(fr + kTfr / 2 + tt_blk(tt, q) * 128) = hi;
        *gmem(fr + kTfr / 2 + tt_blk(tt, q) * 128 + 64) = lo;
      }
    }
}

// ===========================================================================
// forward walk: U rows, int16 state snapshots with a scale per row, final state
// ===========================================================================
template <int K, int NW_, int NG>
__global__ __launch_bounds__(64 * NW_ * NG, 2) void gdn_walk_fwd_kernel(const GdnArgs a, const int V) {
  using C = GwCfg<K, NW_>;
  constexpr int KS = C::KS, NW = C::NW, NP = C::NP, NRT = C::NRT, TPW = C::TPW;
  constexpr bool kAll = NW <= 4;  // every wave owns token tiles (else waves 0 - 3)
  using F = Feed<K, NG, NW * NG>;
  __shared__ __attribute__((aligned(1024))) char sIn[2 * F::kBytes];
  __shared__ __attribute__((aligned(1024))) char sScratch[1024];
  __shared__ __attribute__((aligned(16))) f32x4 sPart[NG][NW][4][64];
  __shared__ __attribute__((aligned(16))) bf16x8 sX[NG][2][2][64], sU[NG][2][2][64];  // [q][hi, lo] operands
  __shared__ unsigned sMax[2][NG][NW][16];  // column maxima of the waves' state rows, by chunk parity

  const int wv = __builtin_amdgcn_readfirstlane(wave_id()), w = wv % NW, gr = wv / NW;
  const int l = lane_id(), g = l >> 4, m = l & 15;
  int unit, vt;
  if (!unit_map(blockIdx.x, V / (16 * NG), a.N * a.H, unit, vt)) return;
  const int n = unit / a.H, h = unit % a.H, H = a.H;
  long bos;
  int len;
  seq_bounds(a.cu, n, a.T, bos, len);
  const int nc = (len + BT - 1) / BT;
  const int gc0 = a.cu ? a.chunk_off[n] : n * a.NT;
  const int v0 = 16 * NG * vt, v = v0 + 16 * gr + m;  // first state column of the workgroup, the lane's column

  f32x4 S[NRT];
#pragma unroll
  for (int rt = 0; rt < NRT; ++rt)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      S[rt][i] = a.s0 ? a.s0[((long)unit * K + KS * w + 16 * rt + 4 * g + i) * V + v] : 0.f;

  F feed;
  feed.init((const char*)((const bf16*)a.k + (bos * H + h) * K), (const char*)((const bf16x8*)a.tfr + ((long)gc0 * H + h) * kTfr),
            (const char*)((const bf16*)a.v + (bos * H + h) * (long)V + v0),
            (const char*)(a.tok + ((long)gc0 * H + h) * kTok), H, V, 1, sIn, wv, l);
  feed.init_prefetch((const char*)((const bf16*)a.k + (bos * H + h) * K), (const char*)((const bf16x8*)a.tfr + ((long)gc0 * H + h) * kTfr),
                     (const char*)(a.tok + ((long)gc0 * H + h) * kTok), H, 1, vt + (V / (16 * NG)) * wv, sScratch, l);
  auto dma = [&](int c, auto P) {
    constexpr int part = decltype(P)::value;
    if (c >= nc) return;
    if (part == 0 && c + 1 == nc && len < BT * nc) feed.rows(H, V, len - BT * c, wv, l);
    feed.template load<part>(c & 1, wv);
  };
  using P0 = std::integral_constant<int, 0>;
  using P1 = std::integral_constant<int, 1>;
  using P2 = std::integral_constant<int, 2>;
  bf16x8 ka[4][NP];  // A operands of K S, read from LDS ahead of the chunk
  auto read_ka = [&](int b) {
#pragma unroll
    for (int q = 0; q < NP; ++q)
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) ka[tt][q] = k_frag<K>(sIn + b * F::kBytes, tt, NP * w + q, g, m);
  };

  if (nc > 0) {
    for (int c = 0; c < 2; ++c) {
      dma(c, P0{});
      dma(c, P1{});
      if (c == 0) dma(c, P2{});
    }
    wait_loads<0>();
  }
  // (values loaded before the loop are settled, or the compiler drains all memory operations at its head)
#pragma unroll
  for (int rt = 0; rt < NRT; ++rt) settle(S[rt]);
  lds_barrier();
  if (nc > 0) read_ka(0);
  float* Uc = a.U + (((long)gc0 * H + h) * V + v0) * BT;
  short* hc = (short*)a.hT + (((long)gc0 * H + h) * V + v0) * K;
  float* hs = (float*)a.hTl + ((long)gc0 * H + h) * V + v0;
  for (int c = 0; c < nc; ++c, Uc += (long)H * V * BT, hc += (long)H * V * K, hs += (long)H * V) {
    const int b0 = c & 1;
    const char* in = sIn + b0 * F::kBytes;
    const float* tok = (const float*)(in + F::kTokOff);
    const bf16x8* sT = (const bf16x8*)(in + F::kT);
    dma(c + 1, P2{});
    // K S over the wave's rows; the column maxima of the snapshot's scales
    f32x4 acc[4];
#pragma unroll
    for (int tt = 0; tt < 4; ++tt) acc[tt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int q = 0; q < NP; ++q) {
      bf16x8 sh, sl;
      split_pair(S[2 * q], S[2 * q + 1], sh, sl);
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) acc[tt] = mfma16(ka[tt][q], sh, acc[tt]);
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) acc[tt] = mfma16(ka[tt][q], sl, acc[tt]);
    }
    {
      unsigned mx = 0;
#pragma unroll
      for (int rt = 0; rt < NRT; ++rt)
#pragma unroll
        for (int i = 0; i < 4; ++i) mx = max(mx, __float_as_uint(S[rt][i]) & 0x7fffffffu);
      mx = group4_umax(mx);
      if (g == 0) sMax[b0][gr][w][m] = mx;
    }
#pragma unroll
    for (int tt = 0; tt < 4; ++tt) sPart[gr][w][tt][l] = acc[tt];
    lds_barrier();
    // own token tiles: X = -gamma (K S).  What the exchange waits for is read first, then the operands of the
    // rest of the step, whose reads overlap it
    bf16x8 kt[NRT][2], Th[TPW][2], Tl[TPW][2], vb[2];
    f32x4 fac[TPW];
    const float gl = tok[kTok - 1];
    auto read_kt = [&]() {
#pragma unroll
      for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int rt = 0; rt < NRT; ++rt) kt[rt][q] = kt_frag<K>(in, NRT * w + rt, q, g, m);
    };
    if (kAll || w < 4) {
      f32x4 part[TPW][NW], ga[TPW];
#pragma unroll
      for (int j = 0; j < TPW; ++j) {
        const int tt = w + NW * j;
#pragma unroll
        for (int ww = 0; ww < NW; ++ww) part[j][ww] = sPart[gr][ww][tt][l];
        ga[j] = *(const f32x4*)(tok + 3 * BT + 16 * tt + 4 * g);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < TPW; ++j) {
        const int tt = w + NW * j;
        fac[j] = *(const f32x4*)(tok + 2 * BT + 16 * tt + 4 * g);
#pragma unroll
        for (int q = 0; q < 2; ++q) {  // (tiles 0 and 1 have one block)
          Th[j][q] = sT[t_blk(tt, min(q, tt / 2)) * 128 + l];
          Tl[j][q] = sT[t_blk(tt, min(q, tt / 2)) * 128 + 64 + l];
        }
      }
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const char* r = in + F::kV + (32 * q + 4 * g + (m >> 2)) * (32 * NG) + 32 * gr + 8 * (m & 3);
        vb[q] = join(read_tr(r), read_tr(r + 16 * 32 * NG));
      }
      read_kt();
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < TPW; ++j) {
        const int tt = w + NW * j;
        f32x4 s = part[j][0], x;
#pragma unroll
        for (int ww = 1; ww < NW; ++ww) s += part[j][ww];
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] = -ga[j][i] * s[i];
        u32x2 hi, lo;
        split4(x, hi, lo);
        *((u32x2*)&sX[gr][tt >> 1][0][l] + (tt & 1)) = hi;
        *((u32x2*)&sX[gr][tt >> 1][1][l] + (tt & 1)) = lo;
      }
    } else {
      read_kt();
    }
    wait_loads<0>();  // chunk c + 1 landed (this wave's share)
    lds_barrier();
    // (nothing reads chunk c's buffers any more: chunk c + 2 goes there)
    // U = Tb V + Tb X to HBM, diag(gamma_L / gamma) U to the other waves.  v enters exactly, as it is: with
    // beta v in X, rounded to a hi/lo pair, the final state was 12 % further off at weak decays and beta
    // near 1.  Its products fill the time in which X's operands come from LDS.
    if (kAll || w < 4) {
      bf16x8 xh[2], xl[2];
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        xh[q] = sX[gr][q][0][l];
        xl[q] = sX[gr][q][1][l];
      }
      __builtin_amdgcn_sched_barrier(0);
      read_ka(b0 ^ 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < TPW; ++j) {
        const int tt = w + NW * j;
        f32x4 u = mfma16(Th[j][0], vb[0], f32x4{0.f, 0.f, 0.f, 0.f});
        f32x4 u2 = mfma16(Tl[j][0], vb[0], f32x4{0.f, 0.f, 0.f, 0.f});
        if (tt >= 2) {
          u = mfma16(Th[j][1], vb[1], u);
          u2 = mfma16(Tl[j][1], vb[1], u2);
        }
        u = mfma16(Th[j][0], xh[0], u);
        u2 = mfma16(Th[j][0], xl[0], u2);
        u = mfma16(Tl[j][0], xh[0], u);
        if (tt >= 2) {
          u2 = mfma16(Th[j][1], xh[1], u2);
          u = mfma16(Th[j][1], xl[1], u);
          u2 = mfma16(Tl[j][1], xh[1], u2);
        }
        u += u2;
        u32x2 hi, lo;
        split4(u * fac[j], hi, lo);
        *((u32x2*)&sU[gr][tt >> 1][0][l] + (tt & 1)) = hi;
        *((u32x2*)&sU[gr][tt >> 1][1][l] + (tt & 1)) = lo;
        *at<f32x4>(Uc, (unsigned)((4 * gr + tt) * 1024 + 16 * l)) = u;
      }
    } else {
      read_ka(b0 ^ 1);
    }
    dma(c + 2, P0{});
    if (c + 5 < nc) feed.prefetch(c + 4);
    lds_barrier();
    // S <- gamma_L S + K^T (fac U); beside it the snapshot of the state before this chunk, one scale per
    // column over all K rows
    dma(c + 2, P1{});
    {
      bf16x8 uh[2], ul[2];
      f32x4 old[NRT];
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        uh[q] = sU[gr][q][0][l];
        ul[q] = sU[gr][q][1][l];
      }
      // (the one LDS read behind the step's last barrier whose words the next step would write before its
      // first one; with a slot per parity they are written two steps on, behind three barriers)
      unsigned mx = sMax[b0][gr][0][m];
#pragma unroll
      for (int ww = 1; ww < NW; ++ww) mx = max(mx, sMax[b0][gr][ww][m]);
      const int e = min(max((int)((mx >> 23) & 0xff) - 127 - 14, -126), 113);
#pragma unroll
      for (int rt = 0; rt < NRT; ++rt) {
        old[rt] = S[rt];
        S[rt] *= gl;
      }
#pragma unroll
      for (int q = 0; q < 2; ++q) {
#pragma unroll
        for (int rt = 0; rt < NRT; ++rt) S[rt] = mfma16(kt[rt][q], uh[q], S[rt]);
#pragma unroll
        for (int rt = 0; rt < NRT; ++rt) S[rt] = mfma16(kt[rt][q], ul[q], S[rt]);
      }
#pragma unroll
      for (int q = 0; q < NP; ++q) {
        s16x8 q8;
#pragma unroll
        for (int i = 0; i < 8; ++i)
          q8[i] = (short)__builtin_amdgcn_fmed3f(rintf(ldexpf(old[2 * q + (i >> 2)][i & 3], -e)), -32767.f, 32767.f);
        *at<s16x8>(hc, (unsigned)((gr * (K / 32) + NP * w + q) * 1024 + 16 * l)) = q8;
      }
      if (w == 0 && g == 0) *at<float>(hs, 4 * (16 * gr + m)) = ldexpf(1.f, e);
    }
  }
  wait_loads<0>();  // no direct load may land after the workgroup's LDS is given back
  if (a.s_fin) {
#pragma unroll
    for (int rt = 0; rt < NRT; ++rt)
#pragma unroll
      for (int i = 0; i < 4; ++i) a.s_fin[((long)unit * K + KS * w + 16 * rt + 4 * g + i) * V + v] = S[rt][i];
  }
}

// ===========================================================================
// gdn_qprep: one workgroup per (chunk, head): operand tables of the backward walk,
//   Q^T  [K/16 row tiles][q][hi, lo][64 lanes]: diag(scale gamma) Qc transposed (rows 16 rt + m, tokens
//        32 q + 4 g .. +3 and 32 q + 16 + 4 g .. +3)
//   P^T  [6 blocks][hi, lo][64 lanes] (blocks as T^T's)
// ===========================================================================
template <int K, bool Q32>
__global__ __launch_bounds__(256) void gdn_qprep_kernel(const GdnArgs a) {
  constexpr int LDQ = K + 4;
  __shared__ __attribute__((aligned(16))) float sQ[BT * LDQ];
  const int tid = threadIdx.x, w = wave_id(), l = lane_id(), g = l >> 4, m = l & 15;
  const int gc = blockIdx.x, h = blockIdx.y, H = a.H;
  int n, L;
  long tok0;
  if (!chunk_of(a, gc, n, tok0, L)) return;
  const long gch = (long)gc * H + h;
  const int rsk = H * K;
  const float* gam = a.tok + gch * kTok + 3 * BT;
  constexpr int VPR = K / 4;
  const __amdgpu_buffer_rsrc_t rq = Q32 ? buf_rsrc(a.qc32 + (tok0 * H + h) * K, ((L - 1) * rsk + K) * 4)
                                        : buf_rsrc((const bf16*)a.qc16 + (tok0 * H + h) * K, ((L - 1) * rsk + K) * 2);
#pragma unroll
  for (int j = 0; j < BT * VPR / 256; ++j) {
    const int idx = tid + 256 * j, t = idx / VPR, c = 4 * (idx % VPR);
    f32x4 x;
    if constexpr (Q32) {
      x = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rq, (t * rsk + c) * 4, 0, 0));
    } else {
      const bf16x4_t y = __builtin_bit_cast(bf16x4_t, __builtin_amdgcn_raw_buffer_load_b64(rq, (t * rsk + c) * 2, 0, 0));
      x = f32x4{(float)y[0], (float)y[1], (float)y[2], (float)y[3]};
    }
    *(f32x4*)(sQ + t * LDQ + c) = x * (a.scale * gam[t]);
  }
  // P^T blocks: wave w the blocks w, w + 4
  const float* pt = a.PT + gch * (BT * BT);
  for (int b = w; b < 6; b += 4) {
    const int tt = b < 4 ? b >> 1 : b - 2, q = b < 4 ? b & 1 : 1;
    const float* p = pt + (16 * tt + m) * BT + 32 * q + 4 * g;
    bf16x8 hi, lo;
    split_pair(*(const f32x4*)p, *(const f32x4*)(p + 16), hi, lo);
    bf16x8* dst = (bf16x8*)a.pfr + (gch * 6 + b) * 128 + l;
    *gmem(dst) = hi;
    *gmem(dst + 64) = lo;
  }
  __syncthreads();
  bf16x8* qf = (bf16x8*)a.qfr + gch * (K / 16) * 256 + l;
  for (int b = w; b < K / 8; b += 4) {
    const int rt = b >> 1, q = b & 1;
    const float* p = sQ + (32 * q + 4 * g) * LDQ + 16 * rt + m;
    f32x4 x, y;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      x[i] = p[i * LDQ];
      y[i] = p[(16 + i) * LDQ];
    }
    bf16x8 hi, lo;
    split_pair(x, y, hi, lo);
    *gmem(qf + b * 128) = hi;
    *gmem(qf + b * 128 + 64) = lo;
  }
}

// ===========================================================================
// backward walk: dU rows, hi/lo state-gradient snapshots (the gradient after each chunk), initial-state
// gradient.  Waves 0-3 own the token tiles; the product Qc^T dO, which depends on no other wave, fills
// the time between the exchanges.
// ===========================================================================
template <int K>
__global__ __launch_bounds__(512, 2) void gdn_walk_bwd_kernel(const GdnArgs a, const int V) {
  using C = GwCfg<K, 8>;
  constexpr int KS = C::KS, NW = C::NW, NP = C::NP, NRT = C::NRT;
  using F = Feed<K, 1, NW>;
  __shared__ __attribute__((aligned(1024))) char sIn[2 * F::kBytes];
  __shared__ __attribute__((aligned(1024))) char sScratch[1024];
  __shared__ __attribute__((aligned(16))) f32x4 sPart[NW][4][64];
  __shared__ __attribute__((aligned(16))) bf16x8 sX[2][2][64], sY[2][2][64];  // [q][hi, lo] operands

  const int w = __builtin_amdgcn_readfirstlane(wave_id()), l = lane_id(), g = l >> 4, m = l & 15;
  int unit, vt;
  if (!unit_map(blockIdx.x, V / 16, a.N * a.H, unit, vt)) return;
  const int n = unit / a.H, h = unit % a.H, H = a.H;
  long bos;
  int len;
  seq_bounds(a.cu, n, a.T, bos, len);
  const int nc = (len + BT - 1) / BT;
  const int gc0 = a.cu ? a.chunk_off[n] : n * a.NT;
  const int v0 = 16 * vt, v = v0 + m;

  f32x4 dS[NRT];
#pragma unroll
  for (int rt = 0; rt < NRT; ++rt)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      dS[rt][i] = a.ds_fin ? a.ds_fin[((long)unit * K + KS * w + 16 * rt + 4 * g + i) * V + v] : 0.f;

  // (chunks are numbered from the end: step e is chunk nc - 1 - e)
  const long lc = gc0 + nc - 1, lt = bos + (long)(nc - 1) * BT;
  F feed;
  {
    const char* kp = (const char*)((const bf16*)a.k + (lt * H + h) * K);
    const char* tp = (const char*)((const bf16x8*)a.tfr + (lc * H + h) * kTfr) + kTfrBytes / 2;
    const char* tk = (const char*)(a.tok + (lc * H + h) * kTok);
    feed.init(kp, tp, (const char*)((const bf16*)a.dout + (lt * H + h) * (long)V + v0), tk, H, V, -1, sIn, w, l);
    feed.init_prefetch(kp, tp, tk, H, -1, vt + (V / 16) * w, sScratch, l);
    if (len < BT * nc) feed.rows(H, V, len - BT * (nc - 1), w, l);
  }
  auto dma = [&](int e, auto P) {
    constexpr int part = decltype(P)::value;
    if (e >= nc) return;
    if (part == 0 && e == 1) feed.rows(H, V, BT, w, l);  // only the last chunk is partial
    feed.template load<part>(e & 1, w);
  };
  using P0 = std::integral_constant<int, 0>;
  using P1 = std::integral_constant<int, 1>;
  using P2 = std::integral_constant<int, 2>;
  bf16x8 ka[4][NP];
  auto read_ka = [&](int b) {
#pragma unroll
    for (int q = 0; q < NP; ++q)
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) ka[tt][q] = k_frag<K>(sIn + b * F::kBytes, tt, NP * w + q, g, m);
  };
  // Qc^T operands of the wave's rows and P^T operands of its token tile, one chunk ahead
  bf16x8 Qh[NRT][2], Ql[NRT][2], Ph[2] = {}, Pl[2] = {};
  auto load_qp = [&](int e) {
    const long gch = (lc - e) * H + h;
    const bf16x8* qf = (const bf16x8*)a.qfr + gch * (K / 16) * 256;
#pragma unroll
    for (int rt = 0; rt < NRT; ++rt)
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        Qh[rt][q] = *at<const bf16x8>(qf + ((NRT * w + rt) * 2 + q) * 128, 16 * l);
        Ql[rt][q] = *at<const bf16x8>(qf + ((NRT * w + rt) * 2 + q) * 128 + 64, 16 * l);
      }
    if (w < 4) {
      const bf16x8* pf = (const bf16x8*)a.pfr + gch * 768;
#pragma unroll
      for (int q = 0; q < 2; ++q) {  // (tiles 2 and 3 have one block)
        Ph[q] = *at<const bf16x8>(pf + tt_blk(w, q) * 128, 16 * l);
        Pl[q] = *at<const bf16x8>(pf + tt_blk(w, q) * 128 + 64, 16 * l);
      }
    }
  };

  if (nc > 0) {
    load_qp(0);
    for (int e = 0; e < 2; ++e) {
      dma(e, P0{});
      dma(e, P1{});
      if (e == 0) dma(e, P2{});
    }
    wait_loads<0>();
  }
#pragma unroll
  for (int rt = 0; rt < NRT; ++rt) {
    settle(dS[rt]);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      settle(Qh[rt][q]);
      settle(Ql[rt][q]);
    }
  }
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    settle(Ph[q]);
    settle(Pl[q]);
  }
  lds_barrier();
  if (nc > 0) read_ka(0);
  float* Uc = a.dU + ((lc * H + h) * V + v0) * BT;
  bf16* hc = (bf16*)a.dhT + ((lc * H + h) * V + v0) * K;
  bf16* hl = (bf16*)a.dhTl + ((lc * H + h) * V + v0) * K;
  for (int e = 0; e < nc; ++e, Uc -= (long)H * V * BT, hc -= (long)H * V * K, hl -= (long)H * V * K) {
    const int b0 = e & 1;
    const char* in = sIn + b0 * F::kBytes;
    const float* tok = (const float*)(in + F::kTokOff);
    const bf16x8* sT = (const bf16x8*)(in + F::kT);
    // K dS' over the wave's rows; the operands are the snapshot as they stand
    f32x4 acc[4];
#pragma unroll
    for (int tt = 0; tt < 4; ++tt) acc[tt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int q = 0; q < NP; ++q) {
      bf16x8 sh, sl;
      split_pair(dS[2 * q], dS[2 * q + 1], sh, sl);
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) acc[tt] = mfma16(ka[tt][q], sh, acc[tt]);
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) acc[tt] = mfma16(ka[tt][q], sl, acc[tt]);
      *at<bf16x8>(hc, (unsigned)((NP * w + q) * 1024 + 16 * l)) = sh;
      *at<bf16x8>(hl, (unsigned)((NP * w + q) * 1024 + 16 * l)) = sl;
    }
#pragma unroll
    for (int tt = 0; tt < 4; ++tt) sPart[w][tt][l] = acc[tt];
    dma(e + 1, P2{});
    lds_barrier();
    bf16x8 kt[NRT][2], dO[2], Th[2], Tl[2];
    f32x4 bg;
    const float gl = tok[kTok - 1];
    auto read_do = [&]() {
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const char* r = in + F::kV + (32 * q + 4 * g + (m >> 2)) * 32 + 8 * (m & 3);
        dO[q] = join(read_tr(r), read_tr(r + 16 * 32));
      }
    };
    auto read_kt = [&]() {
#pragma unroll
      for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int rt = 0; rt < NRT; ++rt) kt[rt][q] = kt_frag<K>(in, NRT * w + rt, q, g, m);
    };
    // own token tile: dU = P^T dO + diag(gamma_L / gamma) K dS'
    if (w < 4) {
      f32x4 part[NW];
#pragma unroll
      for (int ww = 0; ww < NW; ++ww) part[ww] = sPart[ww][w][l];
      const f32x4 fac = *(const f32x4*)(tok + 2 * BT + 16 * w + 4 * g);
      read_do();
      __builtin_amdgcn_sched_barrier(0);
      bg = *(const f32x4*)(tok + 16 * w + 4 * g);
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        Th[q] = sT[tt_blk(w, q) * 128 + l];
        Tl[q] = sT[tt_blk(w, q) * 128 + 64 + l];
      }
      read_kt();
      __builtin_amdgcn_sched_barrier(0);
      f32x4 d = mfma16(Ph[1], dO[1], f32x4{0.f, 0.f, 0.f, 0.f}), d2 = mfma16(Pl[1], dO[1], f32x4{0.f, 0.f, 0.f, 0.f});
      if (w < 2) {
        d = mfma16(Ph[0], dO[0], d);
        d2 = mfma16(Pl[0], dO[0], d2);
      }
      f32x4 s = part[0];
#pragma unroll
      for (int ww = 1; ww < NW; ++ww) s += part[ww];
      d += d2;
#pragma unroll
      for (int i = 0; i < 4; ++i) d[i] += fac[i] * s[i];
      u32x2 hi, lo;
      split4(d, hi, lo);
      *((u32x2*)&sX[w >> 1][0][l] + (w & 1)) = hi;
      *((u32x2*)&sX[w >> 1][1][l] + (w & 1)) = lo;
      *at<f32x4>(Uc, (unsigned)(w * 1024 + 16 * l)) = d;
    } else {
      read_do();
      read_kt();
    }
    // dS <- gamma_L dS' + Qc^T diag(scale gamma) dO (rows past the chunk are zero in Qc^T)
#pragma unroll
    for (int rt = 0; rt < NRT; ++rt) dS[rt] *= gl;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
#pragma unroll
      for (int rt = 0; rt < NRT; ++rt) dS[rt] = mfma16(Qh[rt][q], dO[q], dS[rt]);
#pragma unroll
      for (int rt = 0; rt < NRT; ++rt) dS[rt] = mfma16(Ql[rt][q], dO[q], dS[rt]);
    }
    wait_loads<0>();  // the next chunk landed (this wave's share)
    lds_barrier();
    // -Y = -diag(beta gamma) T^T dU to the other waves
    if (w < 4) {
      bf16x8 xh[2], xl[2];
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        xh[q] = sX[q][0][l];
        xl[q] = sX[q][1][l];
      }
      __builtin_amdgcn_sched_barrier(0);
      read_ka(b0 ^ 1);
      __builtin_amdgcn_sched_barrier(0);
      f32x4 y = mfma16(Th[1], xh[1], f32x4{0.f, 0.f, 0.f, 0.f}), y2 = mfma16(Th[1], xl[1], f32x4{0.f, 0.f, 0.f, 0.f});
      y = mfma16(Tl[1], xh[1], y);
      if (w < 2) {
        y2 = mfma16(Th[0], xh[0], y2);
        y = mfma16(Th[0], xl[0], y);
        y2 = mfma16(Tl[0], xh[0], y2);
      }
      y = -bg * (y + y2);
      u32x2 hi, lo;
      split4(y, hi, lo);
      *((u32x2*)&sY[w >> 1][0][l] + (w & 1)) = hi;
      *((u32x2*)&sY[w >> 1][1][l] + (w & 1)) = lo;
    } else {
      read_ka(b0 ^ 1);
    }
    load_qp(min(e + 1, nc - 1));
    dma(e + 2, P0{});
    if (e + 4 < nc) feed.prefetch(e + 4);
    lds_barrier();
    dma(e + 2, P1{});
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const bf16x8 yh = sY[q][0][l], yl = sY[q][1][l];
#pragma unroll
      for (int rt = 0; rt < NRT; ++rt) dS[rt] = mfma16(kt[rt][q], yh, dS[rt]);
#pragma unroll
      for (int rt = 0; rt < NRT; ++rt) dS[rt] = mfma16(kt[rt][q], yl, dS[rt]);
    }
  }
  wait_loads<0>();  // no direct load may land after the workgroup's LDS is given back
  if (a.ds0) {
#pragma unroll
    for (int rt = 0; rt < NRT; ++rt)
#pragma unroll
      for (int i = 0; i < 4; ++i) a.ds0[((long)unit * K + KS * w + 16 * rt + 4 * g + i) * V + v] = dS[rt][i];
  }
}

// ===========================================================================
// gdn_out: one workgroup of 8 waves per (chunk, head).
//   P = scale (Qc K^T o Gamma), causal (P^T to HBM for the backward);  O = scale diag(gamma) Qc S + P U
// Qc goes to LDS as hi/lo rows with the k tile's swizzle (its A operands are read like k's); wave w then
// owns value tiles w, w + 8, .. two at a time: the state snapshot and U are B operands as they lie in
// HBM, so they never touch LDS.  A column's scale is a power of two and multiplies the result instead.
// O16: o lies on 16 bytes; else its elements are stored one by one (a kernel of its own, since the branch in
// the other one cost it 364 -> 382 us at B1 T32768 H6 V512).
// ===========================================================================
template <int K, bool Q32, bool O16>
__global__ __launch_bounds__(512) void gdn_out_kernel(const GdnArgs a, const int V) {
  constexpr int NP = K / 32, LDO = 40;  // output tile pitch (bf16)
  __shared__ __attribute__((aligned(1024))) char sQh[BT * K * 2], sQl[BT * K * 2];
  __shared__ __attribute__((aligned(1024))) char sKO[BT * K * 2 > 8 * BT * LDO * 2 ? BT * K * 2 : 8 * BT * LDO * 2];  // k, then the output tiles
  __shared__ __attribute__((aligned(16))) bf16x8 sP[4][2][2][64];  // P [tile][q][hi, lo], A operands
  __shared__ __attribute__((aligned(16))) float sGam[BT], sG[BT];
  const int w = __builtin_amdgcn_readfirstlane(wave_id()), l = lane_id(), g = l >> 4, m = l & 15;
  const int gc = blockIdx.x, h = blockIdx.y, H = a.H;
  int n, L;
  long tok0;
  if (!chunk_of(a, gc, n, tok0, L)) return;
  const long gch = (long)gc * H + h;
  const int rsk = H * K, rsv = H * V;
#pragma unroll
  for (int j = 0; j < K / 8 / 8; ++j)
    lds_load16((const bf16*)a.k + (tok0 * H + h) * K, k_tile_off<K>(w + 8 * j, rsk, L, l), lds_addr(sKO) + 1024 * (w + 8 * j));
  // Qc rows (zero past the chunk): wave w rows w, w + 8, ..
  {
    constexpr int LPR = K / 4, RPW = 64 / LPR;  // lanes per row, rows per wave and load
    const int r0 = RPW * w + l / LPR, c = 4 * (l & (LPR - 1));
    const __amdgpu_buffer_rsrc_t rq = Q32 ? buf_rsrc(a.qc32 + (tok0 * H + h) * K, ((L - 1) * rsk + K) * 4)
                                          : buf_rsrc((const bf16*)a.qc16 + (tok0 * H + h) * K, ((L - 1) * rsk + K) * 2);
    f32x4 x[BT / 8 / RPW];
#pragma unroll
    for (int j = 0; j < BT / 8 / RPW; ++j) {
      const int t = r0 + 8 * RPW * j;
      if constexpr (Q32) {
        x[j] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rq, (t * rsk + c) * 4, 0, 0));
      } else {
        const bf16x4_t y = __builtin_bit_cast(bf16x4_t, __builtin_amdgcn_raw_buffer_load_b64(rq, (t * rsk + c) * 2, 0, 0));
        x[j] = f32x4{(float)y[0], (float)y[1], (float)y[2], (float)y[3]};
      }
    }
#pragma unroll
    for (int j = 0; j < BT / 8 / RPW; ++j) {
      const int t = r0 + 8 * RPW * j;
      u32x2 hi, lo;
      split4(x[j], hi, lo);
      const int o = t * (2 * K) + (((c >> 3) ^ swz(t)) << 4) + 2 * (c & 4);
      *(u32x2*)(sQh + o) = hi;
      *(u32x2*)(sQl + o) = lo;
    }
  }
  if (w == 0) {
    const float x = *gmem(a.gcum + (tok0 + min(l, L - 1)) * H + h);
    sG[l] = x;
    sGam[l] = __expf(x);
  }
  wait_loads<0>();
  __syncthreads();
  // P^T tiles (key tile ss, query tile tt >= ss) as K Qc^T: lane = query row, four key rows
  for (int b = w; b < 10; b += 8) {
    const int tt = b < 1 ? 0 : b < 3 ? 1 : b < 6 ? 2 : 3, ss = b - tt * (tt + 1) / 2;
    f32x4 p = f32x4{0.f, 0.f, 0.f, 0.f}, p2 = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int q = 0; q < NP; ++q) {
      const bf16x8 ka = k_frag<K>(sKO, ss, q, g, m);
      p = mfma16(ka, k_frag<K>(sQh, tt, q, g, m), p);
      p2 = mfma16(ka, k_frag<K>(sQl, tt, q, g, m), p2);
    }
    const int t = 16 * tt + m, s0 = 16 * ss + 4 * g;
    const float gt = sG[t];
    const f32x4 gs = *(const f32x4*)(sG + s0);
    f32x4 x;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const bool keep = s0 + i <= t && t < L;
      const float e = __expf(keep ? gt - gs[i] : 0.f);
      x[i] = keep ? a.scale * e * (p[i] + p2[i]) : 0.f;
    }
    u32x2 hi, lo;
    split4(x, hi, lo);
    *((u32x2*)&sP[tt][ss >> 1][0][l] + (ss & 1)) = hi;
    *((u32x2*)&sP[tt][ss >> 1][1][l] + (ss & 1)) = lo;
    float* ptg = a.PT + gch * (BT * BT) + t;
#pragma unroll
    for (int i = 0; i < 4; ++i) *gmem(ptg + (s0 + i) * BT) = x[i];
  }
  // the tiles above the diagonal: zeros (P^T in HBM is a whole matrix; tiles (0, 1) and (2, 3) of P share
  // an operand with a diagonal tile)
  if (w >= 2) {
    const int b = w - 2, tt = b < 3 ? 0 : b < 5 ? 1 : 2, ss = b < 3 ? 1 + b : b < 5 ? b - 1 : 3;
    float* ptg = a.PT + gch * (BT * BT) + 16 * tt + m;
#pragma unroll
    for (int i = 0; i < 4; ++i) *gmem(ptg + (16 * ss + 4 * g + i) * BT) = 0.f;
    if (ss == tt + 1 && (ss & 1)) {
      *((u32x2*)&sP[tt][ss >> 1][0][l] + 1) = u32x2{0u, 0u};
      *((u32x2*)&sP[tt][ss >> 1][1][l] + 1) = u32x2{0u, 0u};
    }
  }
  __syncthreads();
  bf16* so = (bf16*)sKO + w * (BT * LDO);  // this wave's 64 x 32 output tile
  const __amdgpu_buffer_rsrc_t ro = buf_rsrc((const bf16*)a.o + (tok0 * H + h) * (long)V, ((L - 1) * rsv + V) * 2);
  f32x4 gm[4];
#pragma unroll
  for (int tt = 0; tt < 4; ++tt) gm[tt] = *(const f32x4*)(sGam + 16 * tt + 4 * g) * a.scale;
  for (int v0 = 32 * w; v0 < V; v0 += 256) {
    const s16x8* hp = (const s16x8*)((const short*)a.hT + (gch * V + v0) * K);
    const f32x4* up = (const f32x4*)(a.U + (gch * V + v0) * BT);
    s16x8 sv[NP][2];
    f32x4 u[4][2];
    float sc[2];
#pragma unroll
    for (int q = 0; q < NP; ++q)
#pragma unroll
      for (int ct = 0; ct < 2; ++ct) sv[q][ct] = *at<const s16x8>(hp + (ct * NP + q) * 64, 16 * l);
#pragma unroll
    for (int tt = 0; tt < 4; ++tt)
#pragma unroll
      for (int ct = 0; ct < 2; ++ct) u[tt][ct] = *at<const f32x4>(up + (ct * 4 + tt) * 64, 16 * l);
#pragma unroll
    for (int ct = 0; ct < 2; ++ct) sc[ct] = *gmem((const float*)a.hTl + gch * V + v0 + 16 * ct + m);
    f32x4 acc[4][2];
#pragma unroll
    for (int tt = 0; tt < 4; ++tt)
#pragma unroll
      for (int ct = 0; ct < 2; ++ct) acc[tt][ct] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int q = 0; q < NP; ++q) {
      bf16x8 sh[2], sl[2];
#pragma unroll
      for (int ct = 0; ct < 2; ++ct) {
        const s16x8 x = sv[q][ct];
        split_pair(f32x4{(float)x[0], (float)x[1], (float)x[2], (float)x[3]},
                   f32x4{(float)x[4], (float)x[5], (float)x[6], (float)x[7]}, sh[ct], sl[ct]);
      }
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) {
        const bf16x8 qh = k_frag<K>(sQh, tt, q, g, m), ql = k_frag<K>(sQl, tt, q, g, m);
#pragma unroll
        for (int ct = 0; ct < 2; ++ct) {
          acc[tt][ct] = mfma16(qh, sh[ct], acc[tt][ct]);
          acc[tt][ct] = mfma16(qh, sl[ct], acc[tt][ct]);
          acc[tt][ct] = mfma16(ql, sh[ct], acc[tt][ct]);
        }
      }
    }
#pragma unroll
    for (int tt = 0; tt < 4; ++tt)
#pragma unroll
      for (int ct = 0; ct < 2; ++ct) acc[tt][ct] *= gm[tt] * sc[ct];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      bf16x8 uh[2], ul[2];
#pragma unroll
      for (int ct = 0; ct < 2; ++ct) split_pair(u[2 * q][ct], u[2 * q + 1][ct], uh[ct], ul[ct]);
#pragma unroll
      for (int tt = 2 * q; tt < 4; ++tt) {
        const bf16x8 ph = sP[tt][q][0][l], pl = sP[tt][q][1][l];
#pragma unroll
        for (int ct = 0; ct < 2; ++ct) {
          acc[tt][ct] = mfma16(ph, uh[ct], acc[tt][ct]);
          acc[tt][ct] = mfma16(ph, ul[ct], acc[tt][ct]);
          acc[tt][ct] = mfma16(pl, uh[ct], acc[tt][ct]);
        }
      }
    }
    if constexpr (!O16) {
#pragma unroll
      for (int tt = 0; tt < 4; ++tt)
#pragma unroll
        for (int ct = 0; ct < 2; ++ct)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int t = 16 * tt + 4 * g + i;
            if (t < L) *gmem((bf16*)a.o + ((tok0 + t) * H + h) * (long)V + v0 + 16 * ct + m) = (bf16)acc[tt][ct][i];
          }
      continue;
    }
    // rows leave as 16-byte pieces through this wave's LDS tile (range-checked: rows past the chunk drop)
#pragma unroll
    for (int tt = 0; tt < 4; ++tt)
#pragma unroll
      for (int ct = 0; ct < 2; ++ct)
#pragma unroll
        for (int i = 0; i < 4; ++i) so[(16 * tt + 4 * g + i) * LDO + 16 * ct + m] = (bf16)acc[tt][ct][i];
    __builtin_amdgcn_wave_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int t = 16 * j + (l >> 2), c = 8 * (l & 3);
      __builtin_amdgcn_raw_buffer_store_b128(*(const u32x4*)(so + t * LDO + c), ro, (t * rsv + v0 + c) * 2, 0, 0);
    }
    asm volatile("" ::: "memory");
  }
}

// Columns per workgroup: a workgroup of either width fills a CU (LDS), the units are dealt to the eight XCDs, and a
// step takes about 1.42 times as long with 32 columns as with 16 (T1024, 4 units of V512: 53 against 38 us).  So
// 32 where they take less than 2/3 of the rounds: 9 units of V512 or 17 of V256, one round for two, 52 against 62
// and 47 against 59 us; up to 8 units of V512, one round either way, 50 against 37; 24 units of V512, two rounds
// for three, 93 against 90; 9 units of V1024, two for four, 91 against 114.
template <int K>
static hipError_t walk_fwd(const GdnArgs& a, int V, int cus, hipStream_t st) {
  const int units = a.N * a.H, groups = (units + 7) / 8 * 8, per = max(cus / 8, 1);
  const int r16 = (groups / 8 * (V / 16) + per - 1) / per, r32 = (groups / 8 * (V / 32) + per - 1) / per;
  if (3 * r32 < 2 * r16)
    hipLaunchKernelGGL((gdn_walk_fwd_kernel<K, 4, 2>), dim3(groups * (V / 32)), dim3(512), 0, st, a, V);
  else
    hipLaunchKernelGGL((gdn_walk_fwd_kernel<K, 8, 1>), dim3(groups * (V / 16)), dim3(512), 0, st, a, V);
  return hipGetLastError();
}

hipError_t launch_gdn_tprep(const GdnArgs& a, int K, hipStream_t st) {
  switch (K) {
    case 256: hipLaunchKernelGGL(gdn_tprep_kernel<256>, dim3(a.NTG, a.H), dim3(64), 0, st, a); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_gdn_walk_bwd(const GdnArgs& a, int K, int V, hipStream_t st) {
  if (K != 256) return hipErrorInvalidValue;
  if (a.qc32)
    hipLaunchKernelGGL((gdn_qprep_kernel<256, true>), dim3(a.NTG, a.H), dim3(256), 0, st, a);
  else
    hipLaunchKernelGGL((gdn_qprep_kernel<256, false>), dim3(a.NTG, a.H), dim3(256), 0, st, a);
  if (hipError_t e = hipGetLastError()) return e;
  const int groups = (a.N * a.H + 7) / 8 * 8;
  hipLaunchKernelGGL(gdn_walk_bwd_kernel<256>, dim3(groups * (V / 16)), dim3(512), 0, st, a, V);
  return hipGetLastError();
}

hipError_t launch_gdn_out(const GdnArgs& a, int K, int V, hipStream_t st) {
  if (K != 256) return hipErrorInvalidValue;
  const dim3 grid(a.NTG, a.H), blk(512);
  if (((uintptr_t)a.o & 15) == 0) {
    if (a.qc32)
      hipLaunchKernelGGL((gdn_out_kernel<256, true, true>), grid, blk, 0, st, a, V);
    else
      hipLaunchKernelGGL((gdn_out_kernel<256, false, true>), grid, blk, 0, st, a, V);
  } else if (a.qc32) {
    hipLaunchKernelGGL((gdn_out_kernel<256, true, false>), grid, blk, 0, st, a, V);
  } else {
    hipLaunchKernelGGL((gdn_out_kernel<256, false, false>), grid, blk, 0, st, a, V);
  }
  return hipGetLastError();
}

hipError_t launch_gdn_walk_fwd(const GdnArgs& a, int K, int V, int cus, hipStream_t st) {
  switch (K) {
    case 256: return walk_fwd<256>(a, V, cus, st);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace ccq
