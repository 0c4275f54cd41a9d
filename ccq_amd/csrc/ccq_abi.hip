// C ABI of libccq_hip.so: argument checks, buffer carving, kernel launches.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <utility>
#include <vector>

#include "../../include/ccq_hip.h"
#include "ccq_params.h"
#include "ccq_decode_args.h"
#include "ccq_zclean_args.h"
#include "ccq_walk_args.h"

namespace ccq {
hipError_t launch_cwalk(int stage, const WalkArgs& a, hipStream_t st);
hipError_t launch_sum_rows2(const float* partA, float* outA, int colsA, const float* partB, float* outB, int colsB,
                            int nblk, float* red, hipStream_t st);
hipError_t launch_gdn_stage(int stage, const GdnArgs& a, int K, int V, hipStream_t st);
hipError_t launch_l2norm_fwd(const L2NormArgs& a, hipStream_t st);
hipError_t launch_conv(int stage, const ConvArgs& a, int blocks, hipStream_t st);
hipError_t launch_gnorm(int stage, const GNormArgs& a, int blocks, hipStream_t st);
hipError_t launch_decode_prologue(const DecProArgs& a, hipStream_t st);
hipError_t launch_narrow(int stage, const NarrowArgs& a, hipStream_t st);
int narrow_blocks(long M);
hipError_t launch_fill_zero(float* out, long n, hipStream_t st);
hipError_t launch_gla_stage(int stage, const GlaArgs& a, hipStream_t st);
hipError_t launch_decode(const DecodeArgs& a, hipStream_t st);
struct DlConv;
struct DlGate;
hipError_t launch_decode_linear(bool glu, const void* x, long ldx, const void* w, const void* r, long ldr, void* y,
                                long ldy, int M, int K, int N, const void* nw, float eps, int splits, void* ws,
                                const DlConv* conv, hipStream_t st, const DlGate* gate);
hipError_t launch_decode_linear_gnorm(const void* x, long ldx, const void* g, long ldg, const float* gw, int dv,
                                      float geps, const void* w, const void* r, long ldr, void* y, long ldy, int M,
                                      int K, int N, void* ws, hipStream_t st);
hipError_t launch_greedy_embed(const void* logits, long ldl, int M, int N, const void* table, long rows, int D,
                               int64_t* ids, long ldi, void* x, long ldx, hipStream_t st);
hipError_t launch_decode_in_proj(const void* x, long ldx, const void* w, void* y, long ldy, int M, int K, int N,
                                 const void* nw, float eps, int oq, int ok, int ov, int oa, int ob, int Dq, int Dv,
                                 int H, int T, int neg_eig, const void* wq, const void* wk, const void* wv,
                                 const void* bq, const void* bk, const void* bv, void* cq, void* ck, void* cv,
                                 const void* alog, const void* dtb, float* g, float* beta, hipStream_t st);
size_t decode_linear_split_bytes(int N, int splits);
hipError_t launch_cseg(int stage, const WalkArgs& a, hipStream_t st);
int cseg_count(int N, int H, int T, int K);
bool cseg_sums_supported(int K);
bool cseg_supported(int K);
hipError_t decode_scratch(hipStream_t st, void** out);
hipError_t launch_zclean(int stage, const ZCleanArgs& a, hipStream_t st);
hipError_t launch_l2norm_bwd(const L2NormArgs& a, hipStream_t st);
hipError_t launch_chunk_index(const int64_t* cu, int N, int size, int* chunk_off, int* chunk_idx, int cap,
                              hipStream_t st);
}  // namespace ccq

using namespace ccq;

namespace {

thread_local char g_err[512] = "";

int fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

int hip_status(hipError_t e, const char* where) {
  if (e == hipSuccess) return CCQ_OK;
  return fail(CCQ_ERR_HIP, "%s: %s", where, hipGetErrorString(e));
}

bool aligned16(const void* p) { return p == nullptr || (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// The cleaning's buffer sizes (its number of time segments) and the persistent kernels' grids follow
// the CU count of the device that is current when they are queried and launched.  A stream of
// another device would run launches shaped, and buffers sized, for the wrong device: refuse it.
int check_stream_device(void* stream, const char* who) {
  int cur = 0;
  if (hipError_t e = hipGetDevice(&cur); e != hipSuccess) return hip_status(e, who);
  if (!stream) return CCQ_OK;
  hipDevice_t sd = -1;
  if (hipError_t e = hipStreamGetDevice((hipStream_t)stream, &sd); e != hipSuccess) return hip_status(e, who);
  if (sd != cur)
    return fail(CCQ_ERR_DEVICE,
                "%s: the stream belongs to device %d but device %d is current; make the stream's device current "
                "(buffer sizes and launch shapes follow the current device)", who, (int)sd, cur);
  return CCQ_OK;
}

size_t align256(size_t x) { return (x + 255) & ~size_t(255); }

// Consecutive sub-buffers of a caller-provided byte buffer.
struct Slicer {
  char* base;
  size_t off = 0;
  template <typename T>
  T* take(size_t n) {
    T* p = base ? reinterpret_cast<T*>(base + off) : nullptr;
    off += align256(n * sizeof(T));
    return p;
  }
};

int check_common(int B, int T, int H, int N, const int64_t* cu) {
  if (B < 0 || T < 0 || H <= 0 || N < 0) return fail(CCQ_ERR_SHAPE, "negative or zero size (B=%d T=%d H=%d N=%d)", B, T, H, N);
  if (cu && B != 1) return fail(CCQ_ERR_SHAPE, "varlen inputs need B == 1 (got B=%d)", B);
  if (!cu && N != B) return fail(CCQ_ERR_SHAPE, "dense inputs need N == B (got N=%d, B=%d)", N, B);
  return CCQ_OK;
}

int clean_k_ok(int K) { return K == 32 || K == 64 || K == 128 || K == 256; }

// ---- optional kernel timing (measurement only; off unless ccq_timing_enable(1)) ----
struct TimingState {
  std::mutex mu;
  bool on = false;
  std::string only;   // non-empty: time only the kernel of this name
  std::map<std::string, std::vector<std::pair<hipEvent_t, hipEvent_t>>> pending;
  std::map<std::string, std::pair<double, int64_t>> done;
};

TimingState& timing() {
  static TimingState t;
  return t;
}

// Run `launch` between two events recorded on `st` when timing is enabled.
template <typename F>
hipError_t timed(const char* name, hipStream_t st, F&& launch) {
  TimingState& t = timing();
  {
    std::lock_guard<std::mutex> g(t.mu);
    if (!t.on || (!t.only.empty() && t.only != name)) return launch();
  }
  // timing-only events: no system-scope fence on record (that fence writes back and invalidates
  // the caches between every two timed kernels and shows up as idle time before each of them)
  constexpr unsigned kFlags = hipEventDisableSystemFence;
  hipEvent_t a, b;
  if (hipEventCreateWithFlags(&a, kFlags) != hipSuccess) return launch();
  if (hipEventCreateWithFlags(&b, kFlags) != hipSuccess) {
    (void)hipEventDestroy(a);
    return launch();
  }
  (void)hipEventRecord(a, st);
  const hipError_t e = launch();
  (void)hipEventRecord(b, st);
  std::lock_guard<std::mutex> g(t.mu);
  t.pending[name].push_back({a, b});
  return e;
}

void resolve_pending(TimingState& t) {
  for (auto& kv : t.pending) {
    auto& acc = t.done[kv.first];
    for (auto& ev : kv.second) {
      float ms = 0.f;
      if (hipEventSynchronize(ev.second) == hipSuccess && hipEventElapsedTime(&ms, ev.first, ev.second) == hipSuccess) {
        acc.first += ms;
        acc.second += 1;
      }
      (void)hipEventDestroy(ev.first);
      (void)hipEventDestroy(ev.second);
    }
  }
  t.pending.clear();
}

}  // namespace

extern "C" {

int ccq_abi_version(void) { return 1; }

const char* ccq_last_error(void) { return g_err; }

}  // extern "C"

// ---- cleaning: geometry and buffers ----
namespace {

struct WalkGeom {
  int cb;   // tokens per chunk
  int nt;   // chunks per sequence (dense)
  int ntg;  // chunk slots (dense: B * nt; varlen: capacity of the chunk index)
};

WalkGeom walk_geom(int64_t tokens, int B, int T, int N, int K, bool varlen) {
  WalkGeom g;
  g.cb = walk_chunk(K);
  if (varlen) {
    g.nt = 0;
    g.ntg = (int)(tokens / g.cb) + N + 1;
  } else {
    g.nt = (T + g.cb - 1) / g.cb;
    g.ntg = B * g.nt;
  }
  return g;
}

struct WalkSaved {
  int* chunk_idx;
  int* chunk_off;
  float* z;
  float* srow;
  float* mpre;
  float* segD;  // segment walks: per-segment sums of k k^T and of k
  float* segM;
  int nseg;
};

// Time segments of the cleaning walks: the segment walks (K in {64, 128}) always; the column walks
// of K = 256 when more than one segment fits the device; K = 32 walks whole sequences.
int walk_segments(int N, int H, int T, int K) {
  if (!cseg_sums_supported(K)) return 1;
  return cseg_count(N, H, T, K);
}
bool walk_segmented(int N, int H, int T, int K) {
  return cseg_supported(K) || (cseg_sums_supported(K) && walk_segments(N, H, T, K) > 1);
}

// Forward-to-backward buffer of the cleaning: for K in {64, 128} (segment walks) the per-segment
// state totals; otherwise (column walks) the covariance read z, s_t and the chunk-start key sums,
// plus the per-segment totals when the column walks are cut into segments.
size_t carve_walk_saved(char* base, const WalkGeom& g, int64_t tokens, int N, int H, int K, int T, bool varlen,
                        WalkSaved* out) {
  Slicer sl{base};
  WalkSaved t{};
  if (varlen) {
    t.chunk_idx = sl.take<int>((size_t)g.ntg * 2);
    t.chunk_off = sl.take<int>((size_t)N + 1);
  }
  if (walk_segmented(N, H, T, K)) {
    t.nseg = walk_segments(N, H, T, K);
    t.segD = sl.take<float>((size_t)N * H * t.nseg * K * K);
    t.segM = sl.take<float>((size_t)N * H * t.nseg * K);
  }
  if (!cseg_supported(K)) {
    t.z = sl.take<float>((size_t)tokens * H * K);
    t.srow = sl.take<float>((size_t)tokens * H);
    t.mpre = sl.take<float>((size_t)g.ntg * H * K);
  }
  if (out) *out = t;
  return sl.off;
}

struct WalkWork {
  float* sc;
  float* dmsum;
  float* dw_part;
  float* db_part;
  float* red;  // first-pass row sums of dw_part / db_part
  float* segG;  // segment walks: per-segment sums of q dz^T and of dm
  float* segDM;
};

size_t carve_walk_work(char* base, const WalkGeom& g, int64_t tokens, int N, int H, int K, int T, bool gate,
                       WalkWork* out) {
  Slicer sl{base};
  WalkWork t{};
  t.sc = sl.take<float>((size_t)tokens * H * 4);
  if (walk_segmented(N, H, T, K)) {
    const int nseg = walk_segments(N, H, T, K);
    t.segG = sl.take<float>((size_t)N * H * nseg * K * K);
    t.segDM = sl.take<float>((size_t)N * H * nseg * K);
  }
  if (!cseg_supported(K)) t.dmsum = sl.take<float>((size_t)g.ntg * H * K);
  if (gate) {
    t.dw_part = sl.take<float>((size_t)g.ntg * H * K);
    t.db_part = sl.take<float>((size_t)g.ntg * H);
    t.red = sl.take<float>((size_t)kSumSlices * H * (K + 1));
  }
  if (out) *out = t;
  return sl.off;
}

void fill_walk_common(WalkArgs& a, const void* q, const void* k, const float* gate_w, const float* gate_b,
                      const float* h0, const float* m0, const int64_t* cu, const WalkSaved& sv, const WalkGeom& g,
                      int T, int H, int K, int N, int pos_off, int subtract_mean) {
  a.q = q; a.k = k; a.gate_w = gate_w; a.gate_b = gate_b; a.h0 = h0; a.m0 = subtract_mean ? m0 : nullptr;
  a.cu = cu; a.chunk_idx = sv.chunk_idx; a.chunk_off = sv.chunk_off;
  a.z = sv.z; a.srow = sv.srow; a.mpre = sv.mpre; a.segD = sv.segD; a.segM = sv.segM; a.nseg = sv.nseg;
  a.T = T; a.H = H; a.N = N; a.NT = g.nt; a.NTG = g.ntg; a.K = K; a.pos_off = pos_off;
  a.subtract_mean = subtract_mean ? 1 : 0;
}

}  // namespace

extern "C" {

size_t ccq_clean_saved_bytes(int64_t tokens, int B, int T, int N, int H, int K, int varlen) {
  const WalkGeom g = walk_geom(tokens, B, T, N, K, varlen != 0);
  return carve_walk_saved(nullptr, g, tokens, N, H, K, T, varlen != 0, nullptr);
}

size_t ccq_clean_bwd_workspace_bytes(int64_t tokens, int B, int T, int N, int H, int K, int varlen, int gate) {
  const WalkGeom g = walk_geom(tokens, B, T, N, K, varlen != 0);
  return carve_walk_work(nullptr, g, tokens, N, H, K, T, gate != 0, nullptr);
}

int ccq_clean_fwd(const void* q, const void* k, const float* lambda, const float* gate_w, const float* gate_b,
                  float* lambda_out, const float* h0, const float* m0, const int64_t* cu_seqlens, void* saved,
                  void* q_clean, float* q_clean_f32, float* h_final, float* m_final, int B, int T, int H, int K,
                  int N, int position_offset, int subtract_mean, void* stream) {
  if (int s = check_common(B, T, H, N, cu_seqlens)) return s;
  if (!clean_k_ok(K)) return fail(CCQ_ERR_SHAPE, "ccq_clean_fwd: K=%d not in {32, 64, 128, 256}", K);
  if (!q || !k || !saved) return fail(CCQ_ERR_NULL, "ccq_clean_fwd: q, k and saved are required");
  if (!gate_w && !lambda) return fail(CCQ_ERR_NULL, "ccq_clean_fwd: lambda or gate_w is required");
  if (gate_w && !gate_b) return fail(CCQ_ERR_NULL, "ccq_clean_fwd: gate_w needs gate_b");
  if (!q_clean && !q_clean_f32) return fail(CCQ_ERR_NULL, "ccq_clean_fwd: no output (q_clean / q_clean_f32)");
  if (int s = check_stream_device(stream, "ccq_clean_fwd")) return s;
  if (!aligned16(q) || !aligned16(k) || !aligned16(saved))
    return fail(CCQ_ERR_ALIGN, "ccq_clean_fwd: q, k, saved must be 16-byte aligned");
  const bool varlen = cu_seqlens != nullptr;
  const int64_t tokens = (int64_t)B * T;
  const WalkGeom g = walk_geom(tokens, B, T, N, K, varlen);
  WalkSaved sv;
  carve_walk_saved((char*)saved, g, tokens, N, H, K, T, varlen, &sv);
  hipStream_t st = (hipStream_t)stream;
  if (varlen) {
    if (int s = hip_status(launch_chunk_index(cu_seqlens, N, g.cb, sv.chunk_off, sv.chunk_idx, g.ntg, st),
                           "ccq_clean_fwd(index)"))
      return s;
  }
  WalkArgs a{};
  fill_walk_common(a, q, k, gate_w, gate_b, h0, m0, cu_seqlens, sv, g, T, H, K, N, position_offset, subtract_mean);
  a.lam = lambda; a.lam_out = lambda_out; a.qc = q_clean; a.qc32 = q_clean_f32; a.h_fin = h_final;
  a.m_fin = subtract_mean ? m_final : nullptr;
  if (cseg_supported(K)) {
    if (int s = hip_status(timed("clean_fwd_sum", st, [&] { return launch_cseg(kSegSum, a, st); }), "clean_fwd_sum"))
      return s;
    return hip_status(timed("clean_fwd", st, [&] { return launch_cseg(kSegFwd, a, st); }), "ccq_clean_fwd");
  }
  if (sv.segD) {
    if (int s = hip_status(timed("clean_fwd_sum", st, [&] { return launch_cseg(kSegSum, a, st); }), "clean_fwd_sum"))
      return s;
  }
  return hip_status(timed("clean_fwd", st, [&] { return launch_cwalk(kWalkFwd, a, st); }), "ccq_clean_fwd");
}

int ccq_clean_bwd(const void* q, const void* k, const float* lambda, const float* gate_w, const float* gate_b,
                  const float* dq_clean_f32, const void* dq_clean, const float* dk_extra, const float* h0,
                  const float* m0, const int64_t* cu_seqlens, const void* saved, const float* dh_final,
                  const float* dm_final, void* dq, float* dq_f32, void* dk, float* dk_f32, float* dlambda,
                  float* dgate_w, float* dgate_b, float* dh0, float* dm0, void* workspace, int B, int T, int H,
                  int K, int N, int position_offset, int subtract_mean, void* stream) {
  if (int s = check_common(B, T, H, N, cu_seqlens)) return s;
  if (!clean_k_ok(K)) return fail(CCQ_ERR_SHAPE, "ccq_clean_bwd: K=%d not in {32, 64, 128, 256}", K);
  if (!q || !k || !lambda || !saved || !workspace)
    return fail(CCQ_ERR_NULL, "ccq_clean_bwd: q, k, lambda, saved, workspace are required");
  if (!dq_clean_f32 && !dq_clean) return fail(CCQ_ERR_NULL, "ccq_clean_bwd: upstream gradient missing");
  if (!dq && !dq_f32) return fail(CCQ_ERR_NULL, "ccq_clean_bwd: no dq output");
  if (!dk && !dk_f32) return fail(CCQ_ERR_NULL, "ccq_clean_bwd: no dk output");
  if (int s = check_stream_device(stream, "ccq_clean_bwd")) return s;
  const bool gate = gate_w != nullptr;
  if (gate && (!gate_b || !dgate_w || !dgate_b))
    return fail(CCQ_ERR_NULL, "ccq_clean_bwd: gate needs gate_b, dgate_w, dgate_b");
  if (!aligned16(q) || !aligned16(k) || !aligned16(saved) || !aligned16(workspace) ||
      !aligned16(dq_clean_f32 ? (const void*)dq_clean_f32 : dq_clean))
    return fail(CCQ_ERR_ALIGN, "ccq_clean_bwd: q, k, saved, workspace, dq_clean must be 16-byte aligned");
  const bool varlen = cu_seqlens != nullptr;
  const int64_t tokens = (int64_t)B * T;
  const WalkGeom g = walk_geom(tokens, B, T, N, K, varlen);
  WalkSaved sv;
  carve_walk_saved((char*)saved, g, tokens, N, H, K, T, varlen, &sv);
  WalkWork wk;
  carve_walk_work((char*)workspace, g, tokens, N, H, K, T, gate, &wk);
  hipStream_t st = (hipStream_t)stream;
  WalkArgs a{};
  fill_walk_common(a, q, k, gate_w, gate_b, h0, m0, cu_seqlens, sv, g, T, H, K, N, position_offset, subtract_mean);
  a.lam_used = lambda; a.sc = wk.sc; a.dmsum = subtract_mean ? wk.dmsum : nullptr;
  a.segG = wk.segG; a.segDM = wk.segDM;
  a.dw_part = wk.dw_part; a.db_part = wk.db_part;
  a.dqc32 = dq_clean_f32; a.dqc16 = dq_clean_f32 ? nullptr : dq_clean; a.dk_extra = dk_extra;
  a.dh_fin = dh_final; a.dm_fin = subtract_mean ? dm_final : nullptr;
  a.dq = dq; a.dq32 = dq_f32; a.dk = dk; a.dk32 = dk_f32; a.dlam = gate ? nullptr : dlambda; a.dh0 = dh0;
  a.dm0 = subtract_mean ? dm0 : nullptr;
  struct StageName { int stage; const char* name; };
  if (cseg_supported(K)) {
    if (gate && varlen) {
      // the walks write the gate partials of real chunks only: clear the padding entries' too
      if (int s = hip_status(launch_fill_zero(wk.dw_part, (long)g.ntg * H * K, st), "ccq_clean_bwd(dW parts)"))
        return s;
      if (int s = hip_status(launch_fill_zero(wk.db_part, (long)g.ntg * H, st), "ccq_clean_bwd(db parts)"))
        return s;
    }
    const StageName stages[] = {{kSegDq, "clean_bwd_dq"}, {kSegGsum, "clean_bwd_gsum"}, {kSegDk, "clean_bwd_dk"}};
    for (const StageName& sn : stages) {
      if (int s = hip_status(timed(sn.name, st, [&] { return launch_cseg(sn.stage, a, st); }), sn.name)) return s;
    }
  } else {
    const StageName stages[] = {{kWalkRows, "clean_bwd_rows"}, {kWalkDq, "clean_bwd_dq"}, {kWalkDk, "clean_bwd_dk"}};
    for (const StageName& sn : stages) {
      if (sn.stage == kWalkDk && sv.segD) {
        // the dk walk's later segments enter through their totals (from the per-token scalars)
        if (int s = hip_status(timed("clean_bwd_gsum", st, [&] { return launch_cseg(kSegGsum, a, st); }),
                               "clean_bwd_gsum"))
          return s;
      }
      if (int s = hip_status(timed(sn.name, st, [&] { return launch_cwalk(sn.stage, a, st); }), sn.name)) return s;
    }
  }
  if (dm0 && !subtract_mean) {
    if (int s = hip_status(launch_fill_zero(dm0, (long)N * H * K, st), "ccq_clean_bwd(dm0)"))
      return s;
  }
  if (gate) {
    if (int s = hip_status(timed("clean_bwd_gate", st, [&] {
                             return launch_sum_rows2(wk.dw_part, dgate_w, H * K, wk.db_part, dgate_b, H, g.ntg,
                                                     wk.red, st);
                           }),
                           "ccq_clean_bwd(dW, db)"))
      return s;
  }
  return CCQ_OK;
}

int ccq_chunk_index(const int64_t* cu_seqlens, int N, int* chunk_offsets, int* chunk_index, int capacity,
                    void* stream) {
  if (!cu_seqlens || !chunk_offsets || !chunk_index) return fail(CCQ_ERR_NULL, "ccq_chunk_index: null pointer");
  if (N < 0 || capacity < 0) return fail(CCQ_ERR_SHAPE, "ccq_chunk_index: bad sizes");
  return hip_status(launch_chunk_index(cu_seqlens, N, 64, chunk_offsets, chunk_index, capacity, (hipStream_t)stream),
                    "ccq_chunk_index");
}

}  // extern "C"

namespace {

// Snapshot formats (bit 0: the state snapshots hT, bit 1: the state-gradient snapshots dhT): int16
// rows with a power-of-two scale per row (the integers in hT / dhT, one fp32 scale per row in hTl /
// dhTl) where the bit is set, hi/lo bf16 pairs otherwise.  The state snapshots take the int16 form
// wherever their readers do (K = 64 and 256, and K = V = 128); the state-gradient snapshots only at
// K = V = 128: dk is the most sensitive output to them (measured kernel error of dk at K = 256 rose
// from 1.8e-4 to 5.4e-4 with int16 dS', and stayed at 1.8e-4 with int16 S alone).
int gdn_snap16(int K, int V) { return (K == 128 && V == 128) ? 3 : (K == 64 || K == 256) ? 1 : 0; }
// the state part of dk and dw travel from the dq/dk/dw kernel to the WY backward as int16 rows with
// a power-of-two scale per 32 columns where both kernels read and write that form
bool gdn_grad16(int K, int V) { return K == 128 && V == 128; }

// head sizes whose state recurrences run as the register walks of ccq_gwalk.hip
bool gdn_walks(int K) { return K == 256; }

struct GdnSaved {
  float* gcum;
  float* tmat;
  void* w;
  void* wl;
  float* u;
  void* tfr;
  float* tok;
  void* hT;
  void* hTl;
  float* U;
  float* PT;
};

size_t carve_saved(char* base, int64_t tokens, int NTG, int H, int K, int V, GdnSaved* s) {
  Slicer sl{base};
  GdnSaved t;
  t.gcum = sl.take<float>((size_t)tokens * H);
  t.tmat = sl.take<float>((size_t)NTG * H * 64 * 64);
  if (gdn_walks(K)) {  // operand tables of T diag(beta) and T^T and the gates instead of w and u
    t.w = t.wl = nullptr;
    t.u = nullptr;
    t.tfr = sl.take<uint16_t>((size_t)NTG * H * (2 * 6 * 2 * 64 * 8));
    t.tok = sl.take<float>((size_t)NTG * H * 256);
    t.U = sl.take<float>((size_t)NTG * 64 * H * V);  // (whole tiles)
    // (the stated size stays that of w, u and U rows; U's whole tiles take what this form has left of it)
    const size_t rows = (size_t)tokens * H * (4 * K + 8 * V), used = (size_t)NTG * H * (2 * 12288 + 1024 + 256 * V);
    if (rows > used) sl.take<char>(rows - used);
  } else {
    t.w = sl.take<uint16_t>((size_t)tokens * H * K);
    t.wl = sl.take<uint16_t>((size_t)tokens * H * K);
    t.u = sl.take<float>((size_t)tokens * H * V);
    t.tfr = nullptr;
    t.tok = nullptr;
  }
  t.hT = sl.take<uint16_t>((size_t)NTG * H * V * K);
  if (gdn_snap16(K, V) & 1)
    t.hTl = sl.take<float>((size_t)NTG * H * V);
  else
    t.hTl = sl.take<uint16_t>((size_t)NTG * H * V * K);
  if (!gdn_walks(K)) t.U = sl.take<float>((size_t)tokens * H * V);
  t.PT = sl.take<float>((size_t)NTG * H * 64 * 64);
  if (s) *s = t;
  return sl.off;
}

struct GdnWork {
  float* dU;
  void* qfr;
  void* pfr;
  void* dhT;
  void* dhTl;
  float* dkp32;
  float* dw32;
  float* dkp_sc;
  float* dw_sc;
  float* dgp;
};

size_t carve_work(char* base, int64_t tokens, int NTG, int H, int K, int V, GdnWork* s) {
  Slicer sl{base};
  GdnWork t;
  t.dU = sl.take<float>(gdn_walks(K) ? (size_t)NTG * 64 * H * V : (size_t)tokens * H * V);
  t.qfr = t.pfr = nullptr;
  t.dhT = sl.take<uint16_t>((size_t)NTG * H * V * K);
  if (gdn_snap16(K, V) & 2)
    t.dhTl = sl.take<float>((size_t)NTG * H * V);
  else
    t.dhTl = sl.take<uint16_t>((size_t)NTG * H * V * K);
  if (gdn_grad16(K, V)) {
    t.dkp32 = (float*)sl.take<int16_t>((size_t)tokens * H * K);
    t.dw32 = (float*)sl.take<int16_t>((size_t)tokens * H * K);
    t.dkp_sc = sl.take<float>((size_t)tokens * H * (K / 32));
    t.dw_sc = sl.take<float>((size_t)tokens * H * (K / 32));
  } else {
    // (the walk's operand tables lie where dk and dw are written after it)
    const size_t rows = (size_t)tokens * H * K, qt = (size_t)NTG * H * K * 256, pt = (size_t)NTG * H * 12288;
    char* g = (char*)sl.take<char>(gdn_walks(K) ? std::max(8 * rows, qt + pt) : 8 * rows);
    t.dkp32 = (float*)g;
    t.dw32 = t.dkp32 + rows;
    if (gdn_walks(K)) {
      t.qfr = g;
      t.pfr = g + qt;
    }
    t.dkp_sc = t.dw_sc = nullptr;
  }
  t.dgp = sl.take<float>((size_t)(K / 64) * tokens * H);
  if (s) *s = t;
  return sl.off;
}

int gdn_check(const char* who, int B, int T, int H, int K, int V, int N, const int64_t* cu, const int* chunk_index,
              const int* chunk_offsets, int num_chunks) {
  if (int s = check_common(B, T, H, N, cu)) return s;
  if (!(K == 64 || K == 128 || K == 256)) return fail(CCQ_ERR_SHAPE, "%s: K=%d not in {64, 128, 256}", who, K);
  if (V <= 0 || V % 64 != 0 || V > 1024) return fail(CCQ_ERR_SHAPE, "%s: V=%d must be a positive multiple of 64 (<= 1024)", who, V);
  if (cu && (!chunk_index || !chunk_offsets)) return fail(CCQ_ERR_NULL, "%s: varlen needs chunk_index and chunk_offsets", who);
  if (!cu && num_chunks != B * ((T + 63) / 64))
    return fail(CCQ_ERR_SHAPE, "%s: num_chunks=%d, expected B*ceil(T/64)=%d", who, num_chunks, B * ((T + 63) / 64));
  if (cu && num_chunks < 0) return fail(CCQ_ERR_SHAPE, "%s: negative num_chunks", who);
  return CCQ_OK;
}

}  // namespace

extern "C" {

size_t ccq_gdn_saved_bytes(int64_t tokens, int num_chunks, int H, int K, int V) {
  return carve_saved(nullptr, tokens, num_chunks, H, K, V, nullptr);
}

size_t ccq_gdn_bwd_workspace_bytes(int64_t tokens, int num_chunks, int H, int K, int V) {
  return carve_work(nullptr, tokens, num_chunks, H, K, V, nullptr);
}

int ccq_gdn_fwd(const void* q, const float* q_f32, const void* k, const void* v, const float* g, const float* beta,
                const float* initial_state, const int64_t* cu_seqlens, const int* chunk_index,
                const int* chunk_offsets, int num_chunks, void* o, float* final_state, void* saved, int B, int T,
                int H, int K, int V, int N, float scale, void* stream) {
  if (int s = gdn_check("ccq_gdn_fwd", B, T, H, K, V, N, cu_seqlens, chunk_index, chunk_offsets, num_chunks)) return s;
  if ((!q && !q_f32) || !k || !v || !beta || !o || !saved) return fail(CCQ_ERR_NULL, "ccq_gdn_fwd: null input/output");
  if (int s = check_stream_device(stream, "ccq_gdn_fwd")) return s;
  if (!aligned16(q) || !aligned16(q_f32) || !aligned16(k) || !aligned16(v) || !aligned16(saved))
    return fail(CCQ_ERR_ALIGN, "ccq_gdn_fwd: tensors must be 16-byte aligned");
  const int64_t tokens = (int64_t)B * T;
  GdnSaved sv;
  carve_saved((char*)saved, tokens, num_chunks, H, K, V, &sv);
  GdnArgs a{};
  a.qc16 = q_f32 ? nullptr : q; a.qc32 = q_f32; a.k = k; a.v = v; a.g = g; a.beta = beta; a.s0 = initial_state;
  a.cu = cu_seqlens; a.chunk_idx = chunk_index; a.chunk_off = chunk_offsets;
  a.gcum = sv.gcum; a.tmat = sv.tmat; a.w = sv.w; a.wl = sv.wl; a.u = sv.u; a.tfr = sv.tfr; a.tok = sv.tok; a.hT = sv.hT; a.hTl = sv.hTl; a.U = sv.U; a.PT = sv.PT;
  a.o = o; a.s_fin = final_state; a.scale = scale;
  a.T = T; a.H = H; a.N = N; a.NT = (T + 63) / 64; a.NTG = num_chunks;
  a.snap16 = gdn_snap16(K, V);
  hipStream_t st = (hipStream_t)stream;
  static const char* names[] = {"gdn_prep", "gdn_fwd_state", "gdn_fwd_o"};
  const int stages[] = {kGdnPrep, kGdnFwdState, kGdnFwdO};
  // for K <= 128 the forward walk also writes the output (no separate output pass)
  const int nst = K <= 128 ? 2 : 3;
  for (int i = 0; i < nst; ++i) {
    if (int s = hip_status(timed(names[i], st, [&] { return launch_gdn_stage(stages[i], a, K, V, st); }), names[i]))
      return s;
  }
  return CCQ_OK;
}

int ccq_gdn_bwd(const void* q, const float* q_f32, const void* k, const void* v, const float* g, const float* beta,
                const int64_t* cu_seqlens, const int* chunk_index, const int* chunk_offsets, int num_chunks,
                const void* saved, const void* d_o, const float* d_final_state, void* workspace, float* dq_f32,
                float* dk_f32, void* dv, float* dbeta, float* dg, float* d_initial_state, int B, int T, int H, int K,
                int V, int N, float scale, void* stream) {
  if (int s = gdn_check("ccq_gdn_bwd", B, T, H, K, V, N, cu_seqlens, chunk_index, chunk_offsets, num_chunks)) return s;
  if ((!q && !q_f32) || !k || !v || !beta || !saved || !d_o || !workspace || !dq_f32 || !dk_f32 || !dv || !dbeta ||
      !dg)
    return fail(CCQ_ERR_NULL, "ccq_gdn_bwd: null input/output");
  if (int s = check_stream_device(stream, "ccq_gdn_bwd")) return s;
  // the dq/dk/dw kernels read dO with 16-byte direct-to-LDS loads; dv leaves as 16-byte pieces
  if (!aligned16(q) || !aligned16(q_f32) || !aligned16(k) || !aligned16(v) || !aligned16(d_o) || !aligned16(dv) ||
      !aligned16(saved) || !aligned16(workspace) || !aligned16(dq_f32) || !aligned16(dk_f32))
    return fail(CCQ_ERR_ALIGN, "ccq_gdn_bwd: tensors must be 16-byte aligned");
  const int64_t tokens = (int64_t)B * T;
  GdnSaved sv;
  carve_saved((char*)saved, tokens, num_chunks, H, K, V, &sv);
  GdnWork wk;
  carve_work((char*)workspace, tokens, num_chunks, H, K, V, &wk);
  GdnArgs a{};
  a.qc16 = q_f32 ? nullptr : q; a.qc32 = q_f32; a.k = k; a.v = v; a.g = g; a.beta = beta;
  a.cu = cu_seqlens; a.chunk_idx = chunk_index; a.chunk_off = chunk_offsets;
  a.gcum = sv.gcum; a.tmat = sv.tmat; a.w = sv.w; a.wl = sv.wl; a.u = sv.u; a.tfr = sv.tfr; a.tok = sv.tok; a.hT = sv.hT; a.hTl = sv.hTl; a.U = sv.U; a.PT = sv.PT;
  a.dout = d_o; a.ds_fin = d_final_state; a.dU = wk.dU; a.qfr = wk.qfr; a.pfr = wk.pfr; a.dhT = wk.dhT; a.dhTl = wk.dhTl; a.dq32 = dq_f32; a.dkp32 = wk.dkp32;
  a.dw32 = wk.dw32; a.dkp_sc = wk.dkp_sc; a.dw_sc = wk.dw_sc; a.dgp = wk.dgp; a.dk32 = dk_f32; a.dv = dv; a.dbeta = dbeta; a.dg = dg; a.ds0 = d_initial_state;
  a.scale = scale; a.T = T; a.H = H; a.N = N; a.NT = (T + 63) / 64; a.NTG = num_chunks;
  a.snap16 = gdn_snap16(K, V);
  hipStream_t st = (hipStream_t)stream;
  static const char* names[] = {"gdn_bwd_state", "gdn_bwd_dqkw", "gdn_bwd_wy"};
  const int stages[] = {kGdnBwdState, kGdnBwdDqkw, kGdnBwdWy};
  for (int i = 0; i < 3; ++i) {
    if (int s = hip_status(timed(names[i], st, [&] { return launch_gdn_stage(stages[i], a, K, V, st); }), names[i]))
      return s;
  }
  return CCQ_OK;
}

int ccq_l2norm_fwd(const void* x, void* y, float* rstd, int64_t rows, int D, float eps, void* stream) {
  if (!x || !y) return fail(CCQ_ERR_NULL, "ccq_l2norm_fwd: null pointer");
  if (D <= 0 || D > 512 || rows < 0) return fail(CCQ_ERR_SHAPE, "ccq_l2norm_fwd: bad sizes rows=%lld D=%d", (long long)rows, D);
  L2NormArgs a{};
  a.x = x; a.y = y; a.rstd = rstd; a.rows = rows; a.D = D; a.eps = eps;
  return hip_status(launch_l2norm_fwd(a, (hipStream_t)stream), "ccq_l2norm_fwd");
}

int ccq_l2norm_bwd(const void* x, const float* rstd, const float* dy_f32, const void* dy, void* dx, int64_t rows,
                   int D, void* stream) {
  if (!x || !rstd || !dx || (!dy_f32 && !dy)) return fail(CCQ_ERR_NULL, "ccq_l2norm_bwd: null pointer");
  if (D <= 0 || D > 512 || rows < 0) return fail(CCQ_ERR_SHAPE, "ccq_l2norm_bwd: bad sizes");
  L2NormArgs a{};
  a.x = x; a.rstd = const_cast<float*>(rstd); a.dy32 = dy_f32; a.dy16 = dy_f32 ? nullptr : dy; a.dx = dx; a.rows = rows; a.D = D;
  return hip_status(launch_l2norm_bwd(a, (hipStream_t)stream), "ccq_l2norm_bwd");
}

}  // extern "C"

// ---- layer prologue / epilogue: short convolution (+ l2norm), gated RMSNorm ----
namespace {

constexpr int kConvBlocks = 512;   // workgroups of the backward passes (one partial row each)

int conv_blocks(int64_t tokens) { return (int)std::max<int64_t>(1, std::min<int64_t>((tokens + 15) / 16, kConvBlocks)); }
int gnorm_blocks(int64_t rows) { return (int)std::max<int64_t>(1, std::min<int64_t>((rows + 3) / 4, kConvBlocks)); }

struct ConvWork {
  float* dw_part;
  float* db_part;
  float* red;
};
size_t carve_conv_work(char* base, int64_t tokens, int D, int W, ConvWork* out) {
  Slicer sl{base};
  const int nb = conv_blocks(tokens);
  ConvWork t{};
  t.dw_part = sl.take<float>((size_t)nb * D * W);
  t.db_part = sl.take<float>((size_t)nb * D);
  t.red = sl.take<float>((size_t)kSumSlices * D * (W + 1));
  if (out) *out = t;
  return sl.off;
}

int conv_check(const char* who, int B, int T, int N, int D, int W, int head_dim, const int64_t* cu) {
  if (int s = check_common(B, T, 1, N, cu)) return s;
  if (D <= 0 || D % 8 != 0) return fail(CCQ_ERR_SHAPE, "%s: D=%d must be a positive multiple of 8", who, D);
  if (W < 1 || W > 8) return fail(CCQ_ERR_SHAPE, "%s: kernel size W=%d not in [1, 8]", who, W);
  if (head_dim && (head_dim < 8 || head_dim > 512 || (head_dim & (head_dim - 1)) || D % head_dim))
    return fail(CCQ_ERR_SHAPE, "%s: head_dim=%d must be a power of two in [8, 512] dividing D=%d", who, head_dim, D);
  return CCQ_OK;
}

}  // namespace

extern "C" {

size_t ccq_conv_bwd_workspace_bytes(int64_t tokens, int D, int W) {
  return carve_conv_work(nullptr, tokens, D, W, nullptr);
}

int ccq_conv_fwd(const void* x, const float* weight, const float* bias, const float* cache_in,
                 const int64_t* cu_seqlens, void* y, void* y_norm, float* rstd, float* cache_out, int B, int T, int N,
                 int D, int W, int head_dim, int activation, float eps, void* stream) {
  if (int s = conv_check("ccq_conv_fwd", B, T, N, D, W, y_norm ? head_dim : 0, cu_seqlens)) return s;
  if (!x || !weight || (!y && !y_norm)) return fail(CCQ_ERR_NULL, "ccq_conv_fwd: x, weight and an output are required");
  if (y_norm && !rstd) return fail(CCQ_ERR_NULL, "ccq_conv_fwd: y_norm needs rstd");
  if (!aligned16(x) || !aligned16(y) || !aligned16(y_norm))
    return fail(CCQ_ERR_ALIGN, "ccq_conv_fwd: x, y, y_norm must be 16-byte aligned");
  ConvArgs a{};
  a.x = x; a.w = weight; a.bias = bias; a.cache_in = cache_in; a.cu = cu_seqlens; a.y = y; a.yn = y_norm;
  a.rstd = rstd; a.cache_out = cache_out; a.tokens = (long)B * T; a.T = T; a.N = N; a.D = D; a.W = W;
  a.hd = y_norm ? head_dim : 8; a.act = activation ? 1 : 0; a.eps = eps;
  hipStream_t st = (hipStream_t)stream;
  if (cache_out) {
    if (int s = hip_status(launch_conv(2, a, 1, st), "ccq_conv_fwd(cache)")) return s;
  }
  // Tiles of 16 consecutive tokens (one window fill per tile) while that still gives >= 1024
  // tiles; fewer tokens per tile below, down to one token per tile for a decode step, where every
  // token starts its own sequence and a 16-token tile would walk 16 window fills in a row.
  a.tb = (int)std::max<int64_t>(1, std::min<int64_t>(16, a.tokens / 1024));
  return hip_status(timed("conv_fwd", st, [&] {
                      return launch_conv(0, a, (int)std::min<int64_t>((a.tokens + a.tb - 1) / a.tb, 4096), st);
                    }),
                    "ccq_conv_fwd");
}

int ccq_conv_bwd(const void* x, const float* weight, const float* bias, const float* cache_in,
                 const int64_t* cu_seqlens, const void* dy, const void* dy_norm, const float* rstd, void* dx,
                 float* dweight, float* dbias, void* workspace, int B, int T, int N, int D, int W, int head_dim,
                 int activation, void* stream) {
  if (int s = conv_check("ccq_conv_bwd", B, T, N, D, W, dy_norm ? head_dim : 0, cu_seqlens)) return s;
  if (!x || !weight || !dx || !dweight || !workspace || (!dy && !dy_norm))
    return fail(CCQ_ERR_NULL, "ccq_conv_bwd: x, weight, dx, dweight, workspace and a gradient are required");
  if (dy_norm && !rstd) return fail(CCQ_ERR_NULL, "ccq_conv_bwd: dy_norm needs the forward's rstd");
  if (!aligned16(x) || !aligned16(dx) || !aligned16(dy) || !aligned16(dy_norm) || !aligned16(workspace))
    return fail(CCQ_ERR_ALIGN, "ccq_conv_bwd: x, dx, dy, dy_norm, workspace must be 16-byte aligned");
  const int64_t tokens = (int64_t)B * T;
  ConvWork wk;
  carve_conv_work((char*)workspace, tokens, D, W, &wk);
  ConvArgs a{};
  a.x = x; a.w = weight; a.bias = bias; a.cache_in = cache_in; a.cu = cu_seqlens; a.dy = dy; a.dyn = dy_norm;
  a.rstd = const_cast<float*>(rstd); a.dx = dx; a.dw_part = wk.dw_part; a.db_part = dbias ? wk.db_part : nullptr;
  a.tokens = tokens; a.T = T; a.N = N; a.D = D; a.W = W; a.hd = dy_norm ? head_dim : 8;
  a.act = activation ? 1 : 0;
  hipStream_t st = (hipStream_t)stream;
  const int nb = conv_blocks(tokens);
  if (tokens == 0) {
    if (int s = hip_status(launch_fill_zero(dweight, (long)D * W, st), "ccq_conv_bwd(dweight)")) return s;
    return dbias ? hip_status(launch_fill_zero(dbias, (long)D, st), "ccq_conv_bwd(dbias)") : CCQ_OK;
  }
  if (int s = hip_status(timed("conv_bwd", st, [&] { return launch_conv(1, a, nb, st); }), "ccq_conv_bwd")) return s;
  return hip_status(launch_sum_rows2(wk.dw_part, dweight, D * W, dbias ? wk.db_part : nullptr, dbias, dbias ? D : 0,
                                     nb, wk.red, st),
                    "ccq_conv_bwd(dweight, dbias)");
}

size_t ccq_narrow_linear_bwd_workspace_bytes(int64_t rows, int K, int N) {
  Slicer sl{nullptr};
  const int nb = narrow_blocks(rows);
  sl.take<float>((size_t)nb * N * K);
  sl.take<float>((size_t)nb * N);
  sl.take<float>((size_t)kSumSlices * N * (K + 1));
  return sl.off;
}

static int narrow_check(const char* who, int64_t rows, int K, int N, int64_t ldx) {
  if (rows < 0 || N < 1 || N > 16 || K < 32 || K > 2016 || K % 32 || ldx < K || ldx % 8)
    return fail(CCQ_ERR_SHAPE, "%s: rows=%lld K=%d N=%d ldx=%lld (need 1 <= N <= 16, K a multiple of 32 in [32, 2016], "
                "ldx >= K and a multiple of 8)", who, (long long)rows, K, N, (long long)ldx);
  return CCQ_OK;
}

int ccq_narrow_linear_fwd(const void* x, int64_t ldx, const void* weight, const float* bias, void* y, int64_t rows,
                          int K, int N, void* stream) {
  if (int s = narrow_check("ccq_narrow_linear_fwd", rows, K, N, ldx)) return s;
  if (!x || !weight || !y) return fail(CCQ_ERR_NULL, "ccq_narrow_linear_fwd: x, weight, y are required");
  if (!aligned16(x) || !aligned16(weight))
    return fail(CCQ_ERR_ALIGN, "ccq_narrow_linear_fwd: x and weight must be 16-byte aligned");
  hipStream_t st = (hipStream_t)stream;
  if (int s = check_stream_device(st, "ccq_narrow_linear_fwd")) return s;
  NarrowArgs a{};
  a.x = x; a.ldx = ldx; a.w = weight; a.b = bias; a.y = y; a.M = rows; a.K = K; a.N = N;
  return hip_status(timed("narrow_fwd", st, [&] { return launch_narrow(0, a, st); }), "ccq_narrow_linear_fwd");
}

int ccq_narrow_linear_bwd(const void* x, int64_t ldx, const void* weight, const void* dy, void* dx, float* dweight,
                          float* dbias, void* workspace, int64_t rows, int K, int N, void* stream) {
  if (int s = narrow_check("ccq_narrow_linear_bwd", rows, K, N, ldx)) return s;
  if (!x || !weight || !dy || !dweight || !workspace)
    return fail(CCQ_ERR_NULL, "ccq_narrow_linear_bwd: x, weight, dy, dweight and the workspace are required");
  if (!aligned16(x) || !aligned16(weight) || !aligned16(dx) || !aligned16(workspace))
    return fail(CCQ_ERR_ALIGN, "ccq_narrow_linear_bwd: x, weight, dx, workspace must be 16-byte aligned");
  hipStream_t st = (hipStream_t)stream;
  if (int s = check_stream_device(st, "ccq_narrow_linear_bwd")) return s;
  if (rows == 0) {
    if (int s = hip_status(launch_fill_zero(dweight, (long)N * K, st), "ccq_narrow_linear_bwd(dweight)")) return s;
    return dbias ? hip_status(launch_fill_zero(dbias, (long)N, st), "ccq_narrow_linear_bwd(dbias)") : CCQ_OK;
  }
  const int nb = narrow_blocks(rows);
  Slicer sl{(char*)workspace};
  float* dw_part = sl.take<float>((size_t)nb * N * K);
  float* db_part = sl.take<float>((size_t)nb * N);
  float* red = sl.take<float>((size_t)kSumSlices * N * (K + 1));
  NarrowArgs a{};
  a.x = x; a.ldx = ldx; a.w = weight; a.dy = dy; a.dx = dx; a.dw_part = dw_part; a.db_part = dbias ? db_part : nullptr;
  a.M = rows; a.K = K; a.N = N;
  if (int s = hip_status(timed("narrow_bwd", st, [&] { return launch_narrow(1, a, st); }), "ccq_narrow_linear_bwd"))
    return s;
  return hip_status(launch_sum_rows2(dw_part, dweight, N * K, dbias ? db_part : nullptr, dbias, dbias ? N : 0, nb, red,
                                     st),
                    "ccq_narrow_linear_bwd(dweight, dbias)");
}

size_t ccq_gated_rmsnorm_bwd_workspace_bytes(int64_t rows, int dv) {
  Slicer sl{nullptr};
  sl.take<float>((size_t)gnorm_blocks(rows) * dv);
  sl.take<float>((size_t)kSumSlices * dv);
  return sl.off;
}

int ccq_gated_rmsnorm_fwd(const void* x, const void* g, const float* weight, void* y, float* rstd, int64_t rows,
                          int dv, float eps, void* stream) {
  if (!x || !g || !y || !rstd) return fail(CCQ_ERR_NULL, "ccq_gated_rmsnorm_fwd: x, g, y, rstd are required");
  if (rows < 0 || dv <= 0 || dv > 512 || dv % 8)
    return fail(CCQ_ERR_SHAPE, "ccq_gated_rmsnorm_fwd: dv=%d must be a multiple of 8 in [8, 512]", dv);
  if (!aligned16(x) || !aligned16(g) || !aligned16(y))
    return fail(CCQ_ERR_ALIGN, "ccq_gated_rmsnorm_fwd: x, g, y must be 16-byte aligned");
  GNormArgs a{};
  a.x = x; a.g = g; a.w = weight; a.y = y; a.rstd = rstd; a.rows = rows; a.dv = dv; a.eps = eps;
  a.ldg = dv; a.gper = 1;
  hipStream_t st = (hipStream_t)stream;
  return hip_status(timed("gnorm_fwd", st, [&] { return launch_gnorm(0, a, 0, st); }), "ccq_gated_rmsnorm_fwd");
}

int ccq_gated_rmsnorm_fwd_strided(const void* x, const void* g, int64_t ldg, int g_group, const float* weight, void* y,
                                  float* rstd, int64_t rows, int dv, float eps, void* stream) {
  if (!x || !g || !y || !rstd) return fail(CCQ_ERR_NULL, "ccq_gated_rmsnorm_fwd_strided: x, g, y, rstd are required");
  if (rows < 0 || dv <= 0 || dv > 512 || dv % 8)
    return fail(CCQ_ERR_SHAPE, "ccq_gated_rmsnorm_fwd_strided: dv=%d must be a multiple of 8 in [8, 512]", dv);
  if (g_group < 1 || ldg < (int64_t)g_group * dv || ldg % 8)
    return fail(CCQ_ERR_SHAPE, "ccq_gated_rmsnorm_fwd_strided: g_group=%d, ldg=%lld (need ldg >= g_group * dv, a "
                "multiple of 8)", g_group, (long long)ldg);
  if (!aligned16(x) || !aligned16(g) || !aligned16(y))
    return fail(CCQ_ERR_ALIGN, "ccq_gated_rmsnorm_fwd_strided: x, g, y must be 16-byte aligned");
  GNormArgs a{};
  a.x = x; a.g = g; a.w = weight; a.y = y; a.rstd = rstd; a.rows = rows; a.dv = dv; a.eps = eps;
  a.ldg = ldg; a.gper = g_group;
  hipStream_t st = (hipStream_t)stream;
  return hip_status(timed("gnorm_fwd", st, [&] { return launch_gnorm(0, a, 0, st); }),
                    "ccq_gated_rmsnorm_fwd_strided");
}

int ccq_gated_rmsnorm_bwd(const void* x, const void* g, const float* weight, const float* rstd, const void* dy,
                          void* dx, void* dg, float* dweight, void* workspace, int64_t rows, int dv, void* stream) {
  if (!x || !g || !rstd || !dy || !dx || !dg) return fail(CCQ_ERR_NULL, "ccq_gated_rmsnorm_bwd: null pointer");
  if (dweight && !workspace) return fail(CCQ_ERR_NULL, "ccq_gated_rmsnorm_bwd: dweight needs the workspace");
  if (rows < 0 || dv <= 0 || dv > 512 || dv % 8)
    return fail(CCQ_ERR_SHAPE, "ccq_gated_rmsnorm_bwd: dv=%d must be a multiple of 8 in [8, 512]", dv);
  if (!aligned16(x) || !aligned16(g) || !aligned16(dy) || !aligned16(dx) || !aligned16(dg))
    return fail(CCQ_ERR_ALIGN, "ccq_gated_rmsnorm_bwd: x, g, dy, dx, dg must be 16-byte aligned");
  const int nb = gnorm_blocks(rows);
  Slicer sl{(char*)workspace};
  float* part = workspace ? sl.take<float>((size_t)nb * dv) : nullptr;
  float* red = workspace ? sl.take<float>((size_t)kSumSlices * dv) : nullptr;
  GNormArgs a{};
  a.x = x; a.g = g; a.w = weight; a.rstd = const_cast<float*>(rstd); a.dy = dy; a.dx = dx; a.dg = dg;
  a.dw_part = dweight ? part : nullptr; a.rows = rows; a.dv = dv;
  hipStream_t st = (hipStream_t)stream;
  if (rows == 0) return dweight ? hip_status(launch_fill_zero(dweight, dv, st), "ccq_gated_rmsnorm_bwd") : CCQ_OK;
  if (int s = hip_status(timed("gnorm_bwd", st, [&] { return launch_gnorm(1, a, nb, st); }), "ccq_gated_rmsnorm_bwd"))
    return s;
  if (!dweight) return CCQ_OK;
  return hip_status(launch_sum_rows2(part, dweight, dv, nullptr, nullptr, 0, nb, red, st),
                    "ccq_gated_rmsnorm_bwd(dweight)");
}

static int decode_linear_entry(const char* who, bool glu, const void* x, int64_t ldx, const void* weight,
                               const void* residual, int64_t ldr, void* y, int64_t ldy, int M, int K, int N,
                               const void* norm_weight, float norm_eps, void* stream, int splits = 1,
                               void* workspace = nullptr) {
  if (M < 0 || M > 16 || N < 0 || K < 32 || K > 4096 || K % 32 || ldx < K || ldx % 8 || ldy < N ||
      (residual && ldr < N))
    return fail(CCQ_ERR_SHAPE, "%s: M=%d K=%d N=%d ldx=%lld ldy=%lld (need M <= 16, K a multiple of 32 in [32, 4096], "
                "ldx >= K a multiple of 8, ldy >= N, ldr >= N)", who, M, K, N, (long long)ldx, (long long)ldy);
  if (!x || !weight || !y) return fail(CCQ_ERR_NULL, "%s: x, weight, y are required", who);
  if (!aligned16(x) || !aligned16(weight) || !aligned16(norm_weight))
    return fail(CCQ_ERR_ALIGN, "%s: x, the weight and the norm weight must be 16-byte aligned", who);
  return hip_status(launch_decode_linear(glu, x, ldx, weight, residual, ldr, y, ldy, M, K, N, norm_weight, norm_eps,
                                         splits, workspace, nullptr, (hipStream_t)stream, nullptr),
                    who);
}

int ccq_decode_linear_gnorm(const void* x, int64_t ldx, const void* gate, int64_t ldg, const float* norm_weight,
                            int dv, float norm_eps, const void* weight, const void* residual, int64_t ldr, void* y,
                            int64_t ldy, int M, int K, int N, void* workspace, void* stream) {
  const char* who = "ccq_decode_linear_gnorm";
  if (dv < 32 || dv % 32 || K % dv || K / dv > 8)
    return fail(CCQ_ERR_SHAPE, "%s: head width dv=%d must be a multiple of 32 dividing K=%d into at most 8 heads", who,
                dv, K);
  if (M < 0 || M > 16 || N < 0 || K < 32 || K > 4096 || ldx < K || ldx % 8 || ldy < N || (residual && ldr < N))
    return fail(CCQ_ERR_SHAPE, "%s: M=%d K=%d N=%d ldx=%lld ldy=%lld (need M <= 16, K <= 4096, ldx >= K a multiple "
                "of 8, ldy >= N, ldr >= N)", who, M, K, N, (long long)ldx, (long long)ldy);
  if (!x || !gate || !weight || !y) return fail(CCQ_ERR_NULL, "%s: x, gate, weight, y are required", who);
  if (K / dv > 1 && !workspace) return fail(CCQ_ERR_NULL, "%s: more than one head needs the workspace", who);
  if (ldg < K || ldg % 8 || !aligned16(x) || !aligned16(gate) || !aligned16(weight) || !aligned16(norm_weight) ||
      !aligned16(workspace))
    return fail(CCQ_ERR_ALIGN, "%s: x, gate (row stride ldg >= K, a multiple of 8), the weights and the workspace "
                "must be 16-byte aligned", who);
  return hip_status(launch_decode_linear_gnorm(x, ldx, gate, ldg, norm_weight, dv, norm_eps, weight, residual, ldr, y,
                                               ldy, M, K, N, workspace, (hipStream_t)stream),
                    who);
}

int ccq_greedy_embed(const void* logits, int64_t ldl, int M, int N, const void* table, int64_t rows, int D,
                     int64_t* ids, int64_t ldi, void* x, int64_t ldx, void* stream) {
  const char* who = "ccq_greedy_embed";
  if (M < 0 || N < 1 || D < 1 || rows < 1 || ldl < N || ldi < 1 || ldx < D)
    return fail(CCQ_ERR_SHAPE, "%s: M=%d N=%d D=%d rows=%lld ldl=%lld ldi=%lld ldx=%lld (need N, D, rows >= 1, "
                "ldl >= N, ldi >= 1, ldx >= D)", who, M, N, D, (long long)rows, (long long)ldl, (long long)ldi,
                (long long)ldx);
  if (!logits || !table || !ids || !x) return fail(CCQ_ERR_NULL, "%s: logits, table, ids and x are required", who);
  if (((uintptr_t)logits & 1) || ((uintptr_t)table & 1) || ((uintptr_t)x & 1) || ((uintptr_t)ids & 7))
    return fail(CCQ_ERR_ALIGN, "%s: logits, table and x must be 2-byte aligned, ids 8-byte aligned", who);
  return hip_status(launch_greedy_embed(logits, ldl, M, N, table, rows, D, ids, ldi, x, ldx, (hipStream_t)stream), who);
}

int ccq_gdn_decode_in_proj(const void* x, int64_t ldx, const void* weight, void* y, int64_t ldy, int M, int K, int N,
                           const void* norm_weight, float norm_eps, int off_q, int off_k, int off_v, int off_a,
                           int off_b, int H, int Dq, int Dv, int T, const void* wq, const void* wk, const void* wv,
                           const void* bq, const void* bk, const void* bv, void* cq, void* ck, void* cv,
                           const void* A_log, const void* dt_bias, float* g, float* beta, int allow_neg_eigval,
                           void* stream) {
  const char* who = "ccq_gdn_decode_in_proj";
  if (T < 1 || M % T) return fail(CCQ_ERR_SHAPE, "%s: M=%d rows are not whole sequences of T=%d tokens", who, M, T);
  if (H < 1 || Dq < 1 || Dv < 1 || off_q < 0 || off_k < 0 || off_v < 0 || off_a < 0 || off_b < 0 ||
      off_q + Dq > N || off_k + Dq > N || off_v + Dv > N || off_a + H > N || off_b + H > N)
    return fail(CCQ_ERR_SHAPE, "%s: a column block lies outside the N=%d projection columns", who, N);
  if (!wq || !wk || !wv || !cq || !ck || !cv || !A_log || !dt_bias || !g || !beta)
    return fail(CCQ_ERR_NULL, "%s: the convolution weights and caches, A_log, dt_bias, g and beta are required", who);
  if (M < 0 || M > 16 || N < 0 || K < 32 || K > 4096 || K % 32 || ldx < K || ldx % 8 || ldy < N)
    return fail(CCQ_ERR_SHAPE, "%s: M=%d K=%d N=%d ldx=%lld ldy=%lld (need M <= 16, K a multiple of 32 in [32, 4096], "
                "ldx >= K a multiple of 8, ldy >= N)", who, M, K, N, (long long)ldx, (long long)ldy);
  if (!x || !weight || !y) return fail(CCQ_ERR_NULL, "%s: x, weight, y are required", who);
  if (!aligned16(x) || !aligned16(weight) || !aligned16(norm_weight))
    return fail(CCQ_ERR_ALIGN, "%s: x, the weight and the norm weight must be 16-byte aligned", who);
  return hip_status(launch_decode_in_proj(x, ldx, weight, y, ldy, M, K, N, norm_weight, norm_eps, off_q, off_k,
                                          off_v, off_a, off_b, Dq, Dv, H, T, allow_neg_eigval ? 1 : 0, wq, wk, wv,
                                          bq, bk, bv, cq, ck, cv, A_log, dt_bias, g, beta, (hipStream_t)stream),
                    who);
}

size_t ccq_decode_linear_split_workspace_bytes(int N, int splits) {
  return N < 0 || splits < 1 ? 0 : decode_linear_split_bytes(N, splits);
}

int ccq_decode_linear_split(const void* x, int64_t ldx, const void* weight, const void* residual, int64_t ldr, void* y,
                            int64_t ldy, int M, int K, int N, int splits, void* workspace, void* stream) {
  const char* who = "ccq_decode_linear_split";
  if (splits < 1 || splits > 8 || splits > K / 32)
    return fail(CCQ_ERR_SHAPE, "%s: splits=%d not in [1, min(8, K/32)] (K=%d)", who, splits, K);
  if (splits > 1 && !workspace) return fail(CCQ_ERR_NULL, "%s: splits > 1 needs the workspace", who);
  if (!aligned16(workspace)) return fail(CCQ_ERR_ALIGN, "%s: the workspace must be 16-byte aligned", who);
  return decode_linear_entry(who, false, x, ldx, weight, residual, ldr, y, ldy, M, K, N, nullptr, 1e-5f, stream,
                             splits, workspace);
}

int ccq_decode_linear(const void* x, int64_t ldx, const void* weight, const void* residual, int64_t ldr, void* y,
                      int64_t ldy, int M, int K, int N, const void* norm_weight, float norm_eps, void* stream) {
  return decode_linear_entry("ccq_decode_linear", false, x, ldx, weight, residual, ldr, y, ldy, M, K, N, norm_weight,
                             norm_eps, stream);
}

int ccq_decode_linear_glu(const void* x, int64_t ldx, const void* weight, void* y, int64_t ldy, int M, int K, int N,
                          const void* norm_weight, float norm_eps, void* stream) {
  return decode_linear_entry("ccq_decode_linear_glu", true, x, ldx, weight, nullptr, 0, y, ldy, M, K, N, norm_weight,
                             norm_eps, stream);
}

int ccq_gdn_decode_prologue(const void* xq, const void* xk, const void* xv, const void* xa, const void* xb,
                            int64_t ldx, const void* wq, const void* wk, const void* wv, const void* bq,
                            const void* bk, const void* bv, void* cq, void* ck, void* cv, const void* lam_w,
                            const void* lam_b, const void* A_log, const void* dt_bias, void* q, void* k, void* v,
                            float* lam, float* g, float* beta, int B, int T, int H, int K, int V, int W,
                            int allow_neg_eigval, float eps, void* stream) {
  const char* who = "ccq_gdn_decode_prologue";
  if (B < 0 || T < 0) return fail(CCQ_ERR_SHAPE, "%s: negative sizes (B=%d T=%d)", who, B, T);
  if (H < 1 || H > 32) return fail(CCQ_ERR_SHAPE, "%s: H=%d not in [1, 32]", who, H);
  if (K < 8 || K > 512 || (K & (K - 1))) return fail(CCQ_ERR_SHAPE, "%s: K=%d must be a power of two in [8, 512]", who, K);
  if (V <= 0 || V % 8) return fail(CCQ_ERR_SHAPE, "%s: V=%d must be a positive multiple of 8", who, V);
  if (W < 1 || W > 8) return fail(CCQ_ERR_SHAPE, "%s: kernel size W=%d not in [1, 8]", who, W);
  if (ldx < 0 || ldx % 8) return fail(CCQ_ERR_ALIGN, "%s: row stride ldx=%lld must be a multiple of 8", who, (long long)ldx);
  if (!xq || !xk || !xv || !xa || !xb || !wq || !wk || !wv || !A_log || !dt_bias || !q || !k || !v || !g || !beta)
    return fail(CCQ_ERR_NULL, "%s: a required pointer is NULL", who);
  if (lam && !lam_w) return fail(CCQ_ERR_NULL, "%s: the lambda output needs the gate weight", who);
  if (W > 1 && (!cq || !ck || !cv)) return fail(CCQ_ERR_NULL, "%s: W > 1 needs the three caches", who);
  if (H * K > 2048) return fail(CCQ_ERR_SHAPE, "%s: H*K=%d above 2048 (one workgroup holds the whole q row)", who, H * K);
  if (!aligned16(xq) || !aligned16(xk) || !aligned16(xv) || !aligned16(q) || !aligned16(k) || !aligned16(v))
    return fail(CCQ_ERR_ALIGN, "%s: the q, k, v rows and outputs must be 16-byte aligned", who);
  if (!aligned16(wq) || !aligned16(wk) || !aligned16(wv) || !aligned16(bq) || !aligned16(bk) || !aligned16(bv) ||
      !aligned16(cq) || !aligned16(ck) || !aligned16(cv) || !aligned16(lam_w))
    return fail(CCQ_ERR_ALIGN, "%s: the convolution weights, biases, caches and the gate weight must be 16-byte aligned",
                who);
  DecProArgs a{};
  a.xq = xq; a.xk = xk; a.xv = xv; a.xa = xa; a.xb = xb; a.ldx = ldx;
  a.wq = wq; a.wk = wk; a.wv = wv; a.bq = bq; a.bk = bk; a.bv = bv; a.cq = cq; a.ck = ck; a.cv = cv;
  a.lw = lam_w; a.lb = lam_b; a.alog = A_log; a.dtb = dt_bias; a.q = q; a.k = k; a.v = v;
  a.lam = lam; a.g = g; a.beta = beta;
  a.B = B; a.T = T; a.H = H; a.K = K; a.V = V; a.W = W; a.neg_eig = allow_neg_eigval ? 1 : 0; a.eps = eps;
  return hip_status(launch_decode_prologue(a, (hipStream_t)stream), who);
}

}  // extern "C"

extern "C" {

int ccq_timing_enable(int on) {
  TimingState& t = timing();
  std::lock_guard<std::mutex> g(t.mu);
  t.on = on != 0;
  return CCQ_OK;
}

int ccq_timing_select(const char* kernel) {
  TimingState& t = timing();
  std::lock_guard<std::mutex> g(t.mu);
  t.only = kernel ? kernel : "";
  return CCQ_OK;
}

int ccq_timing_reset(void) {
  TimingState& t = timing();
  std::lock_guard<std::mutex> g(t.mu);
  resolve_pending(t);
  t.done.clear();
  return CCQ_OK;
}

int ccq_timing_read(const char* kernel, double* total_ms, int64_t* launches) {
  if (!kernel || !total_ms || !launches) return fail(CCQ_ERR_NULL, "ccq_timing_read: null pointer");
  TimingState& t = timing();
  std::lock_guard<std::mutex> g(t.mu);
  resolve_pending(t);
  auto it = t.done.find(kernel);
  *total_ms = it == t.done.end() ? 0.0 : it->second.first;
  *launches = it == t.done.end() ? 0 : it->second.second;
  return CCQ_OK;
}

}  // extern "C"

// ---- gated linear attention ----
namespace {

struct GlaSaved {
  float* bcum;
  float* A;
  void* xfr;
  void* hT;
  void* hTl;
};

size_t carve_gla_saved(char* base, int64_t tokens, int NTG, int H, int K, int V, GlaSaved* s) {
  Slicer sl{base};
  GlaSaved t;
  // the walk's operand table lies in bcum's place, which is written after the walk (whole chunks fill it exactly)
  t.bcum = (float*)sl.take<char>(std::max((size_t)tokens * H * K * 4, (size_t)NTG * H * K * 256));
  t.xfr = t.bcum;
  t.A = sl.take<float>((size_t)NTG * H * 64 * 64);
  t.hT = sl.take<uint16_t>((size_t)NTG * H * V * K);
  t.hTl = sl.take<uint16_t>((size_t)NTG * H * V * K);
  if (s) *s = t;
  return sl.off;
}

struct GlaWork {
  void* qfr;   // (null: the table's halves lie in dq and dk)
  void* qfr2;
  void* dhT;
  void* dhTl;
};

size_t carve_gla_work(char* base, int64_t tokens, int NTG, int H, int K, int V, GlaWork* s) {
  Slicer sl{base};
  GlaWork t;
  // the walk's operand table: its halves lie in dq and dk, both written after the walk, from their first
  // 16-byte boundary on; chunks less than half full need more than those hold
  const size_t half = (size_t)NTG * H * K * 128;
  const bool out = half + 12 <= (size_t)tokens * H * K * 4;
  t.qfr = out ? nullptr : (void*)sl.take<char>(half);
  t.qfr2 = out ? nullptr : (void*)sl.take<char>(half);
  t.dhT = sl.take<uint16_t>((size_t)NTG * H * V * K);
  t.dhTl = sl.take<uint16_t>((size_t)NTG * H * V * K);
  sl.take<float>((size_t)NTG * H * K);  // (part of the stated size; not used)
  if (s) *s = t;
  return sl.off;
}

int gla_check(const char* who, int B, int T, int H, int K, int V, int N, const int64_t* cu, const int* chunk_index,
              const int* chunk_offsets, int num_chunks) {
  if (int s = check_common(B, T, H, N, cu)) return s;
  if (!(K == 64 || K == 128 || K == 256)) return fail(CCQ_ERR_SHAPE, "%s: K=%d not in {64, 128, 256}", who, K);
  if (V <= 0 || V % 64 != 0 || V > 1024)
    return fail(CCQ_ERR_SHAPE, "%s: V=%d must be a positive multiple of 64 (<= 1024)", who, V);
  if (cu && (!chunk_index || !chunk_offsets))
    return fail(CCQ_ERR_NULL, "%s: varlen needs chunk_index and chunk_offsets", who);
  if (!cu && num_chunks != B * ((T + 63) / 64))
    return fail(CCQ_ERR_SHAPE, "%s: num_chunks=%d, expected B*ceil(T/64)=%d", who, num_chunks, B * ((T + 63) / 64));
  if (cu && num_chunks < 0) return fail(CCQ_ERR_SHAPE, "%s: negative num_chunks", who);
  return CCQ_OK;
}

void fill_gla(GlaArgs& a, const void* q, const float* q_f32, const void* k, const void* v, const float* gk,
              const int64_t* cu, const int* chunk_index, const int* chunk_offsets, int num_chunks, const GlaSaved& sv,
              int B, int T, int H, int K, int V, int N, float scale) {
  a.q16 = q_f32 ? nullptr : q; a.q32 = q_f32; a.k = k; a.v = v; a.gk = gk;
  a.cu = cu; a.chunk_idx = chunk_index; a.chunk_off = chunk_offsets;
  a.bcum = sv.bcum; a.A = sv.A; a.xfr = sv.xfr; a.hT = sv.hT; a.hTl = sv.hTl;
  a.scale = scale; a.T = T; a.H = H; a.N = N; a.NT = (T + 63) / 64; a.NTG = num_chunks; a.K = K; a.V = V;
  (void)B;
}

}  // namespace

extern "C" {

size_t ccq_gla_saved_bytes(int64_t tokens, int num_chunks, int H, int K, int V) {
  return carve_gla_saved(nullptr, tokens, num_chunks, H, K, V, nullptr);
}

size_t ccq_gla_bwd_workspace_bytes(int64_t tokens, int num_chunks, int H, int K, int V) {
  return carve_gla_work(nullptr, tokens, num_chunks, H, K, V, nullptr);
}

int ccq_gla_fwd(const void* q, const float* q_f32, const void* k, const void* v, const float* gk,
                const float* initial_state, const int64_t* cu_seqlens, const int* chunk_index,
                const int* chunk_offsets, int num_chunks, void* o, float* final_state, void* saved, int B, int T,
                int H, int K, int V, int N, float scale, void* stream) {
  if (int s = gla_check("ccq_gla_fwd", B, T, H, K, V, N, cu_seqlens, chunk_index, chunk_offsets, num_chunks)) return s;
  if ((!q && !q_f32) || !k || !v || !o || !saved) return fail(CCQ_ERR_NULL, "ccq_gla_fwd: null input/output");
  if (!aligned16(q) || !aligned16(q_f32) || !aligned16(k) || !aligned16(v) || !aligned16(gk) || !aligned16(o) ||
      !aligned16(saved))
    return fail(CCQ_ERR_ALIGN, "ccq_gla_fwd: tensors must be 16-byte aligned");
  const int64_t tokens = (int64_t)B * T;
  GlaSaved sv;
  carve_gla_saved((char*)saved, tokens, num_chunks, H, K, V, &sv);
  GlaArgs a{};
  fill_gla(a, q, q_f32, k, v, gk, cu_seqlens, chunk_index, chunk_offsets, num_chunks, sv, B, T, H, K, V, N, scale);
  a.h0 = initial_state; a.o = o; a.s_fin = final_state;
  hipStream_t st = (hipStream_t)stream;
  static const char* names[] = {"gla_intra", "gla_fwd_state", "gla_fwd_o"};
  const int stages[] = {kGlaIntra, kGlaFwdState, kGlaFwdO};
  for (int i = 0; i < 3; ++i) {
    if (int s = hip_status(timed(names[i], st, [&] { return launch_gla_stage(stages[i], a, st); }), names[i])) return s;
  }
  return CCQ_OK;
}

int ccq_gla_bwd(const void* q, const float* q_f32, const void* k, const void* v, const float* gk,
                const int64_t* cu_seqlens, const int* chunk_index, const int* chunk_offsets, int num_chunks,
                const void* saved, const void* d_o, const float* d_final_state, const float* final_state,
                void* workspace, float* dq_f32, float* dk_f32, void* dv, float* dv_f32, float* dgk,
                float* d_initial_state, int B, int T, int H, int K, int V, int N, float scale, void* stream) {
  if (int s = gla_check("ccq_gla_bwd", B, T, H, K, V, N, cu_seqlens, chunk_index, chunk_offsets, num_chunks)) return s;
  if ((!q && !q_f32) || !k || !v || !saved || !d_o || !workspace || !dq_f32 || !dk_f32 || (!dv && !dv_f32))
    return fail(CCQ_ERR_NULL, "ccq_gla_bwd: null input/output");
  if (dgk && !gk) return fail(CCQ_ERR_NULL, "ccq_gla_bwd: dgk requested without gk");
  if (d_final_state && dgk && !final_state)
    return fail(CCQ_ERR_NULL, "ccq_gla_bwd: d_final_state with dgk needs the forward's final_state");
  if (!aligned16(q) || !aligned16(q_f32) || !aligned16(k) || !aligned16(v) || !aligned16(d_o) || !aligned16(dv) ||
      !aligned16(saved) || !aligned16(workspace))
    return fail(CCQ_ERR_ALIGN, "ccq_gla_bwd: tensors must be 16-byte aligned");
  const int64_t tokens = (int64_t)B * T;
  GlaSaved sv;
  carve_gla_saved((char*)saved, tokens, num_chunks, H, K, V, &sv);
  GlaWork wk;
  carve_gla_work((char*)workspace, tokens, num_chunks, H, K, V, &wk);
  auto up16 = [](void* p) { return (void*)(((uintptr_t)p + 15) & ~(uintptr_t)15); };
  GlaArgs a{};
  fill_gla(a, q, q_f32, k, v, gk, cu_seqlens, chunk_index, chunk_offsets, num_chunks, sv, B, T, H, K, V, N, scale);
  a.dout = d_o; a.ds_fin = d_final_state; a.s_fin_in = final_state; a.qfr = wk.qfr ? wk.qfr : up16(dq_f32); a.qfr2 = wk.qfr2 ? wk.qfr2 : up16(dk_f32); a.dhT = wk.dhT; a.dhTl = wk.dhTl;
  a.dq32 = dq_f32; a.dk32 = dk_f32; a.dv = dv; a.dv32 = dv_f32; a.dgk = dgk; a.dh0 = d_initial_state;
  hipStream_t st = (hipStream_t)stream;
  static const char* names[] = {"gla_bwd_state", "gla_bwd_dv", "gla_bwd_dqk"};
  const int stages[] = {kGlaBwdState, kGlaBwdDv, kGlaBwdDqk};
  for (int i = 0; i < 3; ++i) {
    if (int s = hip_status(timed(names[i], st, [&] { return launch_gla_stage(stages[i], a, st); }), names[i])) return s;
  }
  return CCQ_OK;
}

}  // extern "C"

// ---- recurrent (decode) step ----
namespace {

size_t carve_decode_work(char* base, int64_t tokens, int H, int K, float** qc, float** kn) {
  Slicer sl{base};
  float* a = sl.take<float>((size_t)tokens * H * K);
  float* b = sl.take<float>((size_t)tokens * H * K);
  if (qc) *qc = a;
  if (kn) *kn = b;
  return sl.off;
}

int decode_common(const char* who, DecodeArgs& a, const void* q, const void* k, const void* v, const float* lambda,
                  const float* gate_w, const float* gate_b, const float* state, const float* cov_state,
                  const float* mean_state, const int64_t* cu_seqlens, void* o, float* state_out,
                  float* cov_state_out, float* mean_state_out, void* workspace, int B, int T, int H, int K, int V,
                  int N, int position_offset, int subtract_mean, int use_l2norm, int enable_ccq, float scale,
                  bool layer = false) {
  if (int s = check_common(B, T, H, N, cu_seqlens)) return s;
  if (!clean_k_ok(K)) return fail(CCQ_ERR_SHAPE, "%s: K=%d not in {32, 64, 128, 256}", who, K);
  if (V <= 0 || V % 64 != 0 || V > 1024)
    return fail(CCQ_ERR_SHAPE, "%s: V=%d must be a positive multiple of 64 (<= 1024)", who, V);
  // (the layer form reads q, k, v from the projection rows and forms lambda itself)
  if ((!layer && (!q || !k || !v)) || !o || !workspace)
    return fail(CCQ_ERR_NULL, "%s: q, k, v, o and workspace are required", who);
  if (!layer && enable_ccq && !lambda && !gate_w) return fail(CCQ_ERR_NULL, "%s: lambda or gate_w is required", who);
  if (gate_w && !gate_b) return fail(CCQ_ERR_NULL, "%s: gate_w needs gate_b", who);
  if (mean_state_out && mean_state_out == mean_state)
    return fail(CCQ_ERR_SHAPE, "%s: mean_state_out may not alias mean_state (every workgroup reads all of it)", who);
  if ((!layer && (!aligned16(q) || !aligned16(k) || !aligned16(v))) || !aligned16(o) || !aligned16(workspace))
    return fail(CCQ_ERR_ALIGN, "%s: tensors must be 16-byte aligned", who);
  // the state slices move as 16-byte pieces of four columns (loads and stores)
  if (!aligned16(state) || !aligned16(cov_state) || !aligned16(state_out) || !aligned16(cov_state_out))
    return fail(CCQ_ERR_ALIGN, "%s: state, cov_state and their outputs must be 16-byte aligned", who);
  const int64_t tokens = (int64_t)B * T;
  carve_decode_work((char*)workspace, tokens, H, K, &a.qc, &a.kn);
  a.q = q; a.k = k; a.v = v; a.lam = lambda; a.gate_w = gate_w; a.gate_b = gate_b;
  a.S_in = state; a.C_in = enable_ccq ? cov_state : nullptr; a.m_in = (enable_ccq && subtract_mean) ? mean_state : nullptr;
  a.S_out = state_out; a.C_out = enable_ccq ? cov_state_out : nullptr;
  a.m_out = enable_ccq ? mean_state_out : nullptr;
  a.o = o; a.cu = cu_seqlens; a.scale = scale;
  a.T = T; a.H = H; a.N = N; a.K = K; a.V = V; a.pos_off = position_offset; a.subtract_mean = subtract_mean ? 1 : 0;
  a.l2norm = use_l2norm ? 1 : 0; a.ccq = enable_ccq ? 1 : 0;
  return CCQ_OK;
}

}  // namespace

extern "C" {

size_t ccq_decode_workspace_bytes(int64_t tokens, int H, int K) {
  return carve_decode_work(nullptr, tokens, H, K, nullptr, nullptr);
}

int ccq_gdn_decode(const void* q, const void* k, const void* v, const float* lambda, const float* gate_w,
                   const float* gate_b, const float* g, const float* beta, const float* gk, const float* gv,
                   const float* state, const float* cov_state,
                   const float* mean_state, const int64_t* cu_seqlens, void* o, float* state_out,
                   float* cov_state_out, float* mean_state_out, void* workspace, int B, int T, int H, int K, int V,
                   int N, int position_offset, int subtract_mean, int use_l2norm, int enable_ccq, float scale,
                   void* stream) {
  DecodeArgs a{};
  if (int s = decode_common("ccq_gdn_decode", a, q, k, v, lambda, gate_w, gate_b, state, cov_state, mean_state,
                            cu_seqlens, o, state_out, cov_state_out, mean_state_out, workspace, B, T, H, K, V, N,
                            position_offset, subtract_mean, use_l2norm, enable_ccq, scale))
    return s;
  if (!beta) return fail(CCQ_ERR_NULL, "ccq_gdn_decode: beta is required");
  if (!aligned16(gv)) return fail(CCQ_ERR_ALIGN, "ccq_gdn_decode: gv must be 16-byte aligned");
  a.g = g; a.beta = beta; a.gk = gk; a.gv = gv; a.gla = 0;
  return hip_status(launch_decode(a, (hipStream_t)stream), "ccq_gdn_decode");
}

static_assert(CCQ_DECODE_SCRATCH_BYTES == ccq::kDecodeScratchBytes, "scratch size in the header and the library");

int ccq_gdn_decode_noalloc(const void* q, const void* k, const void* v, const float* lambda, const float* gate_w,
                           const float* gate_b, const float* g, const float* beta, const float* gk, const float* gv,
                           const float* state,
                           const float* cov_state, const float* mean_state, const int64_t* cu_seqlens, void* o,
                           float* state_out, float* cov_state_out, float* mean_state_out, int B, int T, int H, int K,
                           int V, int N, int position_offset, int subtract_mean, int use_l2norm, int enable_ccq,
                           float scale, void* stream) {
  if (int s = check_common(B, T, H, N, cu_seqlens)) return s;
  if (!clean_k_ok(K)) return fail(CCQ_ERR_SHAPE, "ccq_gdn_decode_noalloc: K=%d not in {32, 64, 128, 256}", K);
  const size_t need = carve_decode_work(nullptr, (int64_t)B * T, H, K, nullptr, nullptr);
  if (need > kDecodeScratchBytes)
    return fail(CCQ_ERR_SHAPE,
                "ccq_gdn_decode_noalloc: %lld tokens x %d heads x K=%d need %zu bytes of scratch, above its "
                "fixed %zu (8 bytes per token, head and key channel); use ccq_gdn_decode with a workspace",
                (long long)B * T, H, K, need, kDecodeScratchBytes);
  void* ws = nullptr;
  if (int s = hip_status(decode_scratch((hipStream_t)stream, &ws), "ccq_gdn_decode_noalloc")) return s;
  return ccq_gdn_decode(q, k, v, lambda, gate_w, gate_b, g, beta, gk, gv, state, cov_state, mean_state, cu_seqlens, o,
                        state_out, cov_state_out, mean_state_out, ws, B, T, H, K, V, N, position_offset,
                        subtract_mean, use_l2norm, enable_ccq, scale, stream);
}

int ccq_gla_decode(const void* q, const void* k, const void* v, const float* lambda, const float* gate_w,
                   const float* gate_b, const float* gk, const float* gv, const float* state, const float* cov_state,
                   const float* mean_state, const int64_t* cu_seqlens, void* o, float* state_out,
                   float* cov_state_out, float* mean_state_out, void* workspace, int B, int T, int H, int K, int V,
                   int N, int position_offset, int subtract_mean, int use_l2norm, int reverse, float scale,
                   void* stream) {
  DecodeArgs a{};
  if (int s = decode_common("ccq_gla_decode", a, q, k, v, lambda, gate_w, gate_b, state, cov_state, mean_state,
                            cu_seqlens, o, state_out, cov_state_out, mean_state_out, workspace, B, T, H, K, V, N,
                            position_offset, subtract_mean, use_l2norm, 1, scale))
    return s;
  if (K > 256) return fail(CCQ_ERR_SHAPE, "ccq_gla_decode: K=%d", K);
  if (!aligned16(gv)) return fail(CCQ_ERR_ALIGN, "ccq_gla_decode: gv must be 16-byte aligned");
  a.gk = gk; a.gv = gv; a.gla = 1; a.reverse = reverse ? 1 : 0;
  return hip_status(launch_decode(a, (hipStream_t)stream), "ccq_gla_decode");
}

// ---- decode step with in-place states and a device-held position (graph capture) ----
size_t ccq_decode_step_workspace_bytes(int B, int T, int H, int K) {
  Slicer sl{nullptr};
  sl.take<char>(carve_decode_work(nullptr, (int64_t)B * T, H, K, nullptr, nullptr));
  sl.take<float>((size_t)B * H * K);
  return sl.off;
}

}  // extern "C"

namespace {

int decode_step(const char* who, bool gla, const void* q, const void* k, const void* v, const float* lambda,
                const float* gate_w, const float* gate_b, const float* g, const float* beta, const float* gk,
                float* state, float* cov_state, float* mean_state, int* position, void* o, void* workspace, int B,
                int T, int H, int K, int V, int subtract_mean, int use_l2norm, int enable_ccq, float scale,
                void* stream, const DecodeLayer* layer = nullptr, long vld = 0) {
  if (!state || !position) return fail(CCQ_ERR_NULL, "%s: state and position are required", who);
  if (enable_ccq && (!cov_state || (subtract_mean && !mean_state)))
    return fail(CCQ_ERR_NULL, "%s: cov_state (and mean_state with subtract_mean) are required", who);
  if (!gla && !beta) return fail(CCQ_ERR_NULL, "%s: beta is required", who);
  DecodeArgs a{};
  // the key sum goes to the workspace tail and is copied back after the step
  Slicer sl{(char*)workspace};
  sl.take<char>(carve_decode_work(nullptr, (int64_t)B * T, H, K, nullptr, nullptr));
  float* m_new = workspace ? sl.take<float>((size_t)B * H * K) : nullptr;
  const bool mean = enable_ccq && subtract_mean;
  if (int s = decode_common(who, a, q, k, v, lambda, gate_w, gate_b, state, cov_state, mean ? mean_state : nullptr,
                            nullptr, o, state, cov_state, mean ? m_new : nullptr, workspace, B, T, H, K, V, B, 0,
                            subtract_mean, use_l2norm, enable_ccq, scale, layer != nullptr))
    return s;
  if (layer) {
    a.lay = *layer;
    a.vld = vld;
  }
  a.pos_dev = position;
  a.pos_adv = position;
  if (mean) {
    a.m_dst = mean_state;
    a.m_src = m_new;
    a.m_count = (long)B * H * K;
  }
  if (gla) {
    a.gk = gk;
    a.gla = 1;
  } else {
    a.g = g;
    a.beta = beta;
  }
  return hip_status(launch_decode(a, (hipStream_t)stream), who);
}

}  // namespace

extern "C" {

int ccq_gdn_decode_step(const void* q, const void* k, const void* v, const float* lambda, const float* gate_w,
                        const float* gate_b, const float* g, const float* beta, float* state, float* cov_state,
                        float* mean_state, int* position, void* o, void* workspace, int B, int T, int H, int K, int V,
                        int subtract_mean, int use_l2norm, int enable_ccq, float scale, void* stream) {
  return decode_step("ccq_gdn_decode_step", false, q, k, v, lambda, gate_w, gate_b, g, beta, nullptr, state,
                     cov_state, mean_state, position, o, workspace, B, T, H, K, V, subtract_mean, use_l2norm,
                     enable_ccq, scale, stream);
}

int ccq_gdn_layer_decode_step(const void* x, int64_t ldx, int off_q, int off_k, int off_v, const void* lam_w,
                              const void* lam_b, const float* g, const float* beta, float* state, float* cov_state,
                              float* mean_state, int* position, void* o, void* workspace, int B, int T, int H, int K,
                              int V, int subtract_mean, int enable_ccq, float scale, float l2_eps, void* stream) {
  const char* who = "ccq_gdn_layer_decode_step";
  if (H * K > kDecodeLayerMaxQ) return fail(CCQ_ERR_SHAPE, "%s: H*K=%d above %d", who, H * K, kDecodeLayerMaxQ);
  if (!x || !lam_w || !g || !beta) return fail(CCQ_ERR_NULL, "%s: x, lam_w, g and beta are required", who);
  if (off_q < 0 || off_k < 0 || off_v < 0 || off_q + (int64_t)H * K > ldx || off_k + (int64_t)H * K > ldx ||
      off_v + (int64_t)H * V > ldx)
    return fail(CCQ_ERR_SHAPE, "%s: a column block lies outside the rows (ldx=%lld)", who, (long long)ldx);
  // the backbone reads v as 8-byte pieces, the clean kernel the q row and the gate weight row as
  // 16-byte pieces of 8 channels
  if ((((uintptr_t)x + 2 * (uintptr_t)off_v) & 7) || (ldx & 3) || (V & 3))
    return fail(CCQ_ERR_ALIGN, "%s: the v rows must be 8-byte aligned", who);
  if (!aligned16(x) || (ldx & 7) || (off_q & 7) || !aligned16(lam_w))
    return fail(CCQ_ERR_ALIGN, "%s: x, lam_w, the row stride and off_q must allow 16-byte pieces (ldx %% 8 == 0)",
                who);
  DecodeLayer lay{};
  lay.x = x;
  lay.ldx = (long)ldx;
  lay.oq = off_q;
  lay.ok = off_k;
  lay.lw = lam_w;
  lay.lb = lam_b;
  lay.l2eps = l2_eps;
  return decode_step(who, false, nullptr, nullptr, (const uint16_t*)x + off_v, nullptr, nullptr, nullptr, g, beta,
                     nullptr, state, cov_state, mean_state, position, o, workspace, B, T, H, K, V, subtract_mean, 0,
                     enable_ccq, scale, stream, &lay, (long)ldx);
}

int ccq_gla_decode_step(const void* q, const void* k, const void* v, const float* lambda, const float* gate_w,
                        const float* gate_b, const float* gk, float* state, float* cov_state, float* mean_state,
                        int* position, void* o, void* workspace, int B, int T, int H, int K, int V, int subtract_mean,
                        int use_l2norm, float scale, void* stream) {
  return decode_step("ccq_gla_decode_step", true, q, k, v, lambda, gate_w, gate_b, nullptr, nullptr, gk, state,
                     cov_state, mean_state, position, o, workspace, B, T, H, K, V, subtract_mean, use_l2norm, 1, scale,
                     stream);
}

}  // extern "C"

// ---- cleaning given a precomputed covariance read z ----
namespace {

int zclean_check(const char* who, int B, int T, int H, int K, int N, const int64_t* cu, const int* chunk_index,
                 const int* chunk_offsets, int num_blocks) {
  if (int s = check_common(B, T, H, N, cu)) return s;
  if (!clean_k_ok(K)) return fail(CCQ_ERR_SHAPE, "%s: K=%d not in {32, 64, 128, 256}", who, K);
  if (cu && (!chunk_index || !chunk_offsets))
    return fail(CCQ_ERR_NULL, "%s: varlen needs chunk_index and chunk_offsets", who);
  if (!cu && num_blocks != B * ((T + 63) / 64))
    return fail(CCQ_ERR_SHAPE, "%s: num_blocks=%d, expected B*ceil(T/64)=%d", who, num_blocks, B * ((T + 63) / 64));
  if (cu && num_blocks < 0) return fail(CCQ_ERR_SHAPE, "%s: negative num_blocks", who);
  return CCQ_OK;
}

void fill_zclean(ZCleanArgs& a, const void* q, const void* k, const void* z, const float* lambda,
                 const int64_t* cu, const int* chunk_index, const int* chunk_offsets, int num_blocks, int T, int H,
                 int K, int N, int position_offset, int subtract_mean) {
  a.q = q; a.k = k; a.z = z; a.lam = lambda; a.cu = cu; a.chunk_idx = chunk_index; a.chunk_off = chunk_offsets;
  a.T = T; a.H = H; a.N = N; a.NT = (T + 63) / 64; a.NB = num_blocks; a.K = K; a.pos_off = position_offset;
  a.subtract_mean = subtract_mean ? 1 : 0;
}

}  // namespace

extern "C" {

size_t ccq_clean_z_saved_bytes(int num_blocks, int H, int K) {
  Slicer sl{nullptr};
  sl.take<float>((size_t)num_blocks * H * K);
  sl.take<float>((size_t)num_blocks * H * K);
  return sl.off;
}

size_t ccq_clean_z_bwd_workspace_bytes(int num_blocks, int H, int K) { return ccq_clean_z_saved_bytes(num_blocks, H, K); }

int ccq_clean_z_fwd(const void* q, const void* k, const void* z, const float* lambda, const float* m0,
                    const int64_t* cu_seqlens, const int* chunk_index, const int* chunk_offsets, int num_blocks,
                    void* saved, void* q_clean, float* m_final, int B, int T, int H, int K, int N, int position_offset,
                    int subtract_mean, void* stream) {
  if (int s = zclean_check("ccq_clean_z_fwd", B, T, H, K, N, cu_seqlens, chunk_index, chunk_offsets, num_blocks))
    return s;
  if (!q || !k || !z || !lambda || !saved || !q_clean)
    return fail(CCQ_ERR_NULL, "ccq_clean_z_fwd: q, k, z, lambda, saved and q_clean are required");
  ZCleanArgs a{};
  fill_zclean(a, q, k, z, lambda, cu_seqlens, chunk_index, chunk_offsets, num_blocks, T, H, K, N, position_offset,
              subtract_mean);
  Slicer sl{(char*)saved};
  a.prefix = sl.take<float>((size_t)num_blocks * H * K);
  a.ksum = sl.take<float>((size_t)num_blocks * H * K);
  a.m0 = m0; a.qc = q_clean; a.m_fin = m_final;
  hipStream_t st = (hipStream_t)stream;
  return hip_status(timed("clean_z_fwd", st, [&] { return launch_zclean(0, a, st); }), "ccq_clean_z_fwd");
}

int ccq_clean_z_bwd(const void* q, const void* k, const void* z, const float* lambda, const int64_t* cu_seqlens,
                    const int* chunk_index, const int* chunk_offsets, int num_blocks, const void* saved,
                    const void* dq_clean, const float* dq_clean_f32, const float* dm_final, void* dq, void* dk,
                    void* dz, float* dlambda, float* dm0, void* workspace, int B, int T, int H, int K, int N,
                    int position_offset, int subtract_mean, void* stream) {
  if (int s = zclean_check("ccq_clean_z_bwd", B, T, H, K, N, cu_seqlens, chunk_index, chunk_offsets, num_blocks))
    return s;
  if (!q || !k || !z || !lambda || !saved || (!dq_clean && !dq_clean_f32) || !dq || !dk || !dz || !workspace)
    return fail(CCQ_ERR_NULL, "ccq_clean_z_bwd: null input/output");
  ZCleanArgs a{};
  fill_zclean(a, q, k, z, lambda, cu_seqlens, chunk_index, chunk_offsets, num_blocks, T, H, K, N, position_offset,
              subtract_mean);
  Slicer sl{(char*)saved};
  a.prefix = sl.take<float>((size_t)num_blocks * H * K);
  Slicer wl{(char*)workspace};
  a.ksum = wl.take<float>((size_t)num_blocks * H * K);
  a.carry = wl.take<float>((size_t)num_blocks * H * K);
  a.dqc16 = dq_clean_f32 ? nullptr : dq_clean; a.dqc32 = dq_clean_f32;
  a.dm_fin = subtract_mean ? dm_final : nullptr; a.dq = dq; a.dk = dk; a.dz = dz; a.dlam = dlambda;
  a.dm0 = dm0;
  hipStream_t st = (hipStream_t)stream;
  return hip_status(timed("clean_z_bwd", st, [&] { return launch_zclean(1, a, st); }), "ccq_clean_z_bwd");
}

}  // extern "C"
