// extern "C" surface of libcastle_hip.so (declared in include/castle_hip.h): argument
// validation, workspace carving and dispatch to the kernel launchers.  No torch types.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/castle_hip.h"
#include <algorithm>
#include <stdlib.h>
#include <initializer_list>
#include "castle_params.h"
#include "castle_gemm.h"
#include "castle_profile.h"
#include "castle_rows.h"
#include "castle_tiles.h"

namespace castle {
int launch_fwd(const FwdArgs& a, int dtype, bool bf16_operands, hipStream_t stream);
int launch_scan(const FwdArgs& a, int dtype, bool bf16_operands, hipStream_t stream);
int launch_short(const FwdArgs& a, int dtype, bool bf16_operands, hipStream_t stream);
int launch_bwd(const BwdArgs& a, int dtype, bool bf16_operands, hipStream_t stream);
int launch_decode(const DecodeArgs& a, int dtype, hipStream_t stream);
int launch_decode_flush(const DecodeArgs& a, int dtype, hipStream_t stream);
int launch_cache_rows(const View4 (&src)[3], const View4 (&dst)[3], int B, int H, int L, int d, int dtype, int rotary, hipStream_t stream);
int launch_rope(const View4& src, const View4& dst, int B, int H, int L, int d, int dtype, int pos0, hipStream_t stream);
int decode_pick_splits(int BH, int t, int rows_per_iteration, int cus);
int decode_static_scratch(float** ptr);
int64_t decode_layer_control_bytes(int B, int H, int d, int es);
bool decode_layer_once_ok(int B, int H, int d, int es, int t, int dim);
int launch_decode_layer(const DecodeArgs& d, const DecodeLinear& in, const DecodeLinear& out, void* control, bool take_over, bool give_up, int dtype, hipStream_t stream);
int launch_small_linear(const void* x, const void* w, void* y, int M, int N, int K, int64_t ldx, int64_t ldw, int64_t ldy,
                        int dtype, const void* norm_w, float eps, int act, const void* res, int64_t ldr, hipStream_t stream, int* clear = nullptr, int clear_n = 0);
int launch_sample(const void* logits, int64_t ld, const float* u, int rows, int V, int k, float inv_temperature, int64_t* out, int64_t out_ld,
                  int64_t* out2, int dtype, hipStream_t stream);
int launch_gather_rows(const void* table, int64_t row_bytes, int64_t ld_bytes, int64_t rows, const int64_t* index, int n, void* y, hipStream_t stream);
}  // namespace castle

namespace {

// compute units of the current device, looked up once per device
int device_cus() {
  static int cus[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
  if (cus[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) return 0;
    cus[dev] = n;
  }
  return cus[dev];
}

using castle::kNB;

int elem_size(int dtype) {
  switch (dtype) {
    case CASTLE_F32: return 4;
    case CASTLE_BF16:
    case CASTLE_F16: return 2;
    default: return 0;
  }
}

bool head_dim_ok(int d) { return d == 16 || d == 32 || d == 64 || d == 128; }

int64_t align_up(int64_t x, int64_t a) { return (x + a - 1) / a * a; }

// upper limit of the dS / dSu tile buffers (they grow with B*H*L^2); beyond it the backward
// falls back to recomputing the score chain in its second kernel
constexpr int64_t kMaxScoreTileBytes = (int64_t)40 << 30;
// CASTLE_MAX_SCORE_TILE_BYTES in the environment overrides the limit (0 = never use the tiles)
// (read once, when the library first needs it, so that castle_bwd_workspace_bytes and castle_bwd
// cannot disagree)
int64_t max_score_tile_bytes() {
  static const int64_t limit = [] {
    const char* e = getenv("CASTLE_MAX_SCORE_TILE_BYTES");
    return e != nullptr ? strtoll(e, nullptr, 10) : kMaxScoreTileBytes;
  }();
  return limit;
}

struct Geometry {
  int Lp, nblk;
  int64_t lse_bytes, tblk_bytes, snap_bytes, mat_bytes, op_bytes;
  int64_t off_lse, off_t, off_tt, off_ttx, off_ops, total;
  int64_t bwd_total;
};
constexpr int64_t kHeaderBytes = 256 + 4 * castle::kAmaxBlocks;   // header + partial maxima, forward and backward alike

Geometry geometry(int B, int H, int L, int d, int es, int flags = 0) {
  Geometry g;
  g.Lp = (int)align_up(L, 128);
  g.nblk = g.Lp / kNB;
  const int64_t BH = (int64_t)B * H;
  g.lse_bytes = align_up(BH * g.Lp * 4, 256);
  g.tblk_bytes = align_up(BH * g.Lp * kNB * es, 256);
  g.snap_bytes = align_up(BH * castle::snap_rows(g.nblk) * d * es, 256);
  // dS / dSu tiles between the two backward kernels
  g.mat_bytes = align_up(BH * g.Lp * g.Lp * es, 256);
  // too long, or the caller asks for it: the query kernel recomputes the scores instead
  if (2 * g.mat_bytes > max_score_tile_bytes() || (flags & CASTLE_FLAG_RECOMPUTE_SCORES)) g.mat_bytes = 0;
  g.off_lse = kHeaderBytes;
  g.off_t = g.off_lse + g.lse_bytes;
  g.off_tt = g.off_t + g.tblk_bytes;
  g.off_ttx = g.off_tt + g.tblk_bytes;
  g.op_bytes = align_up(BH * g.Lp * d * es, 256);   // one operand in the compute type, padded to Lp rows
  g.off_ops = g.off_ttx + g.tblk_bytes;
  g.total = g.off_ops + 6 * g.op_bytes;            // the snapshots live in their own buffer (g.snap_bytes)
  // header, reverse-state snapshots, delta, dO copy, dS / dSu tiles, and the forward snapshots when they are recomputed
  g.bwd_total = kHeaderBytes + g.snap_bytes + g.lse_bytes + g.op_bytes + 2 * g.mat_bytes +
                ((flags & CASTLE_FLAG_RECOMPUTE_STATE) ? g.snap_bytes : 0);
  return g;
}

// pointer and strides must allow 16-byte vector access along d
bool view_ok(const castle_view4* v, int es, bool need_l) {
  if (v == nullptr || v->ptr == nullptr) return false;
  const int64_t q = 16 / es;
  if (reinterpret_cast<uintptr_t>(v->ptr) % 16 != 0) return false;
  if (v->stride_b % q != 0 || v->stride_h % q != 0) return false;
  if (need_l && v->stride_l % q != 0) return false;
  return true;
}

castle::View4 to_view(const castle_view4* v) {
  castle::View4 r;
  if (v == nullptr) {
    r.ptr = nullptr; r.sb = r.sh = r.sl = 0;
  } else {
    r.ptr = v->ptr; r.sb = v->stride_b; r.sh = v->stride_h; r.sl = v->stride_l;
  }
  return r;
}

int check_core(int B, int H, int L, int d, int dtype) {
  if (elem_size(dtype) == 0) return CASTLE_ERR_DTYPE;
  if (B <= 0 || H <= 0 || L <= 0 || !head_dim_ok(d)) return CASTLE_ERR_SHAPE;
  if ((int64_t)B * H > 65535) return CASTLE_ERR_SHAPE;   // grid.y of the small kernels
  if ((int64_t)B * H * ((L + 127) / 128) > 2147483647LL) return CASTLE_ERR_SHAPE;   // 1-D grid
  if (dtype == CASTLE_F32 && d > 64) return CASTLE_ERR_SHAPE;
  return CASTLE_OK;
}

castle::FwdWorkspace carve(void* base, void* state, const Geometry& g) {
  char* p = static_cast<char*>(base);
  castle::FwdWorkspace w;
  w.hdr = reinterpret_cast<castle::WsHeader*>(p);
  w.amax_part = reinterpret_cast<float*>(p + 256);
  w.lse = reinterpret_cast<float*>(p + g.off_lse);
  w.t_blk = p + g.off_t;
  w.tt_blk = p + g.off_tt;
  w.ttx_blk = p + g.off_ttx;
  w.usnap = state;
  w.qc_p = p + g.off_ops;
  w.kc_p = p + g.off_ops + g.op_bytes;
  w.vc_p = p + g.off_ops + 2 * g.op_bytes;
  w.qu_p = p + g.off_ops + 3 * g.op_bytes;
  w.ku_p = p + g.off_ops + 4 * g.op_bytes;
  w.vu_p = p + g.off_ops + 5 * g.op_bytes;
  return w;
}

}  // namespace

constexpr int64_t kMaxRows = (int64_t)1 << 30;   // rows of a launch: the grids stay below 2^31 workgroups

extern "C" {

int castle_abi_version(void) { return CASTLE_ABI_VERSION; }

const char* castle_error_string(int code) {
  switch (code) {
    case CASTLE_OK: return "ok";
    case CASTLE_ERR_DTYPE: return "unknown element type";
    case CASTLE_ERR_SHAPE: return "unsupported shape (head dim must be 16/32/64/128, fp32 needs d <= 64, B*H <= 65535)";
    case CASTLE_ERR_LAUNCH: return "HIP launch or configuration error";
    case CASTLE_ERR_WORKSPACE: return "workspace missing, misaligned or too small";
    case CASTLE_ERR_ARG: return "NULL or misaligned tensor view";
    case CASTLE_ERR_SCRATCH: return "problem too large for the static scratch of the entry point that allocates nothing";
    default: return "unknown error";
  }
}

int64_t castle_fwd_workspace_bytes(int B, int H, int L, int d, int dtype) {
  const int rc = check_core(B, H, L, d, dtype);
  if (rc != CASTLE_OK) return rc;
  return geometry(B, H, L, d, elem_size(dtype)).total;
}

int64_t castle_fwd_state_bytes(int B, int H, int L, int d, int dtype) {
  const int rc = check_core(B, H, L, d, dtype);
  if (rc != CASTLE_OK) return rc;
  const int64_t n = geometry(B, H, L, d, elem_size(dtype)).snap_bytes;
  return n > 0 ? n : 256;   // a single block has no snapshots; keep the buffer non-empty
}

int castle_fwd(const castle_view4* qc, const castle_view4* kc, const castle_view4* vc,
               const castle_view4* qu, const castle_view4* ku, const castle_view4* vu,
               int B, int H, int L, int d, int dtype, float scale, int flags,
               const castle_view4* out, const castle_view4* U,
               void* workspace, int64_t workspace_bytes, void* state, int64_t state_bytes, void* stream) {
  int rc = check_core(B, H, L, d, dtype);
  if (rc != CASTLE_OK) return rc;
  const int es = elem_size(dtype);
  const castle_view4* in[] = {qc, kc, vc, qu, ku, vu, out};
  for (const castle_view4* v : in)
    if (!view_ok(v, es, true)) return CASTLE_ERR_ARG;
  const bool want_U = U != nullptr && U->ptr != nullptr;
  if (want_U && !view_ok(U, es, true)) return CASTLE_ERR_ARG;
  if ((flags & CASTLE_FLAG_U_HALF) && dtype != CASTLE_BF16) return CASTLE_ERR_DTYPE;   // the format replaces bf16 only
  const Geometry g = geometry(B, H, L, d, es);
  if (workspace == nullptr || reinterpret_cast<uintptr_t>(workspace) % 256 != 0 || workspace_bytes < g.total)
    return CASTLE_ERR_WORKSPACE;
  if (state == nullptr || reinterpret_cast<uintptr_t>(state) % 256 != 0 || state_bytes < g.snap_bytes)
    return CASTLE_ERR_WORKSPACE;

  castle::FwdArgs a;
  a.s.B = B; a.s.H = H; a.s.L = L; a.s.d = d; a.s.Lp = g.Lp; a.s.nblk = g.nblk; a.s.scale = scale;
  a.s.rotary = (flags & CASTLE_FLAG_ROTARY) != 0;
  a.s.cus = device_cus();
  a.qc = to_view(qc); a.kc = to_view(kc); a.vc = to_view(vc);
  a.qu = to_view(qu); a.ku = to_view(ku); a.vu = to_view(vu);
  a.out = to_view(out);
  a.U = to_view(want_U ? U : nullptr);
  a.u_half = (flags & CASTLE_FLAG_U_HALF) != 0;
  a.ws = carve(workspace, state, g);
  a.amax_ready = (flags & CASTLE_FLAG_AMAX_READY) != 0;
  if (flags & CASTLE_FLAG_FORWARD_ONLY) {
    rc = castle::launch_short(a, dtype, (flags & CASTLE_FLAG_BF16_OPERANDS) != 0, static_cast<hipStream_t>(stream));
    if (rc != 1) return rc;
  }
  return castle::launch_fwd(a, dtype, (flags & CASTLE_FLAG_BF16_OPERANDS) != 0, static_cast<hipStream_t>(stream));
}

int64_t castle_bwd_workspace_bytes(int B, int H, int L, int d, int dtype, int flags) {
  const int rc = check_core(B, H, L, d, dtype);
  if (rc != CASTLE_OK) return rc;
  const Geometry g = geometry(B, H, L, d, elem_size(dtype), flags);
  return g.bwd_total;
}

int castle_bwd(const castle_view4* qc, const castle_view4* kc, const castle_view4* vc,
               const castle_view4* qu, const castle_view4* ku, const castle_view4* vu,
               const castle_view4* out, const castle_view4* dout,
               int B, int H, int L, int d, int dtype, float scale, int flags,
               const castle_view4* dqc, const castle_view4* dkc, const castle_view4* dvc,
               const castle_view4* dqu, const castle_view4* dku, const castle_view4* dvu,
               const void* fwd_workspace, int64_t fwd_workspace_bytes,
               const void* fwd_state, int64_t fwd_state_bytes,
               void* bwd_workspace, int64_t bwd_workspace_bytes, void* stream) {
  int rc = check_core(B, H, L, d, dtype);
  if (rc != CASTLE_OK) return rc;
  const int es = elem_size(dtype);
  const castle_view4* in[] = {qc, kc, vc, qu, ku, vu, out, dout, dqc, dkc, dvc, dqu, dku, dvu};
  for (const castle_view4* v : in)
    if (!view_ok(v, es, true)) return CASTLE_ERR_ARG;
  if (flags & CASTLE_FLAG_FORWARD_ONLY) return CASTLE_ERR_ARG;
  const Geometry g = geometry(B, H, L, d, es, flags);
  if (fwd_workspace == nullptr || reinterpret_cast<uintptr_t>(fwd_workspace) % 256 != 0 || fwd_workspace_bytes < g.total)
    return CASTLE_ERR_WORKSPACE;
  if (bwd_workspace == nullptr || reinterpret_cast<uintptr_t>(bwd_workspace) % 256 != 0 ||
      bwd_workspace_bytes < g.bwd_total)
    return CASTLE_ERR_WORKSPACE;
  const bool recompute_state = (flags & CASTLE_FLAG_RECOMPUTE_STATE) != 0;
  if (!recompute_state &&
      (fwd_state == nullptr || reinterpret_cast<uintptr_t>(fwd_state) % 256 != 0 || fwd_state_bytes < g.snap_bytes))
    return CASTLE_ERR_WORKSPACE;

  castle::BwdArgs a;
  a.s.B = B; a.s.H = H; a.s.L = L; a.s.d = d; a.s.Lp = g.Lp; a.s.nblk = g.nblk; a.s.scale = scale;
  a.s.rotary = (flags & CASTLE_FLAG_ROTARY) != 0;
  a.s.cus = device_cus();
  a.qc = to_view(qc); a.kc = to_view(kc); a.vc = to_view(vc);
  a.qu = to_view(qu); a.ku = to_view(ku); a.vu = to_view(vu);
  a.out = to_view(out); a.dout = to_view(dout);
  a.dqc = to_view(dqc); a.dkc = to_view(dkc); a.dvc = to_view(dvc);
  a.dqu = to_view(dqu); a.dku = to_view(dku); a.dvu = to_view(dvu);
  char* bw = static_cast<char*>(bwd_workspace);
  // forward snapshots: the caller's, or recomputed into the tail of this call's own workspace
  void* state = recompute_state ? bw + (g.bwd_total - g.snap_bytes) : const_cast<void*>(fwd_state);
  a.ws = carve(const_cast<void*>(fwd_workspace), state, g);
  a.bhdr = reinterpret_cast<castle::BwdHeader*>(bw);
  a.amax_part = reinterpret_cast<float*>(bw + 256);
  a.amax_ready = (flags & CASTLE_FLAG_AMAX_READY) != 0;
  bw += kHeaderBytes;
  a.gsnap = bw;
  a.delta = reinterpret_cast<float*>(bw + g.snap_bytes);
  a.dout_p = bw + g.snap_bytes + g.lse_bytes;
  a.ds_mat = g.mat_bytes ? bw + g.snap_bytes + g.lse_bytes + g.op_bytes : nullptr;
  a.dsu_mat = g.mat_bytes ? bw + g.snap_bytes + g.lse_bytes + g.op_bytes + g.mat_bytes : nullptr;
  if (recompute_state) {   // the scan again, from the operand copies the forward pass left
    castle::FwdArgs f;
    f.s = a.s;
    f.qc = a.qc; f.kc = a.kc; f.vc = a.vc; f.qu = a.qu; f.ku = a.ku; f.vu = a.vu;
    f.out = a.out;
    f.U = to_view(nullptr);
    f.ws = a.ws;
    f.with_t = 0;
    rc = castle::launch_scan(f, dtype, (flags & CASTLE_FLAG_BF16_OPERANDS) != 0, static_cast<hipStream_t>(stream));
    if (rc != 0) return rc;
  }
  return castle::launch_bwd(a, dtype, (flags & CASTLE_FLAG_BF16_OPERANDS) != 0, static_cast<hipStream_t>(stream));
}

int64_t castle_decode_workspace_bytes(int B, int H, int d, int t_max) {
  if (B <= 0 || H <= 0 || !head_dim_ok(d) || t_max < 0) return CASTLE_ERR_SHAPE;
  return align_up((int64_t)B * H * (64 * (d + 2) + 1) * 4, 256);   // partials of up to 64 splits, one arrival count
}

// checks the arguments of a cached step and fills `a`; out may be NULL when the caller sets a.out itself
static int decode_step_args(castle::DecodeArgs& a, const castle_view4* U, const castle_view4* qu_cache,
                              const castle_view4* kc_cache, const castle_view4* vc_cache,
                              int t, const int* t_device, int capacity,
                              const castle_view4* qc, const castle_view4* kc, const castle_view4* vc,
                              const castle_view4* qu, const castle_view4* ku, const castle_view4* vu,
                              int B, int H, int d, int dtype, float scale, int flags,
                              const castle_view4* out, const castle_deferred* deferred,
                              void* workspace, int64_t workspace_bytes, bool static_scratch) {
  const int es = elem_size(dtype);
  if (es == 0) return CASTLE_ERR_DTYPE;
  if ((flags & CASTLE_FLAG_U_HALF) && dtype != CASTLE_BF16) return CASTLE_ERR_DTYPE;
  if (B <= 0 || H <= 0 || t < 0 || capacity <= 0 || !head_dim_ok(d) || (int64_t)B * H > 65535) return CASTLE_ERR_SHAPE;
  if (t_device == nullptr && t >= capacity) return CASTLE_ERR_SHAPE;   // row t would be written past the buffers
  const castle_view4* caches[] = {U, qu_cache, kc_cache, vc_cache};
  for (const castle_view4* v : caches)
    if (!view_ok(v, es, true)) return CASTLE_ERR_ARG;
  const castle_view4* tok[] = {qc, kc, vc, qu, ku, vu};
  for (const castle_view4* v : tok)
    if (!view_ok(v, es, false)) return CASTLE_ERR_ARG;
  if (out != nullptr && !view_ok(out, es, false)) return CASTLE_ERR_ARG;
  if (deferred != nullptr) {
    if (!view_ok(&deferred->vu_ring, es, true) || !view_ok(&deferred->gates, 4, false)) return CASTLE_ERR_ARG;
    if (deferred->base < 0 || (deferred->base_device != nullptr && reinterpret_cast<uintptr_t>(deferred->base_device) % 4 != 0))
      return CASTLE_ERR_ARG;
    // host-side counts: the pending sources must all fit the ring
    if (t_device == nullptr && deferred->base_device == nullptr && deferred->base > t) return CASTLE_ERR_SHAPE;
  }
  // with a device-side count the split must not depend on it: sized for a full cache
  const int splits = castle::decode_pick_splits(B * H, t_device != nullptr ? capacity : t, castle::kThreads * 16 / (d * es), device_cus());
  if (static_scratch) {
    // the per-GPU array replaces the caller's workspace; nothing is allocated on this path
    if ((int64_t)B * H * splits * (d + 2) * 4 > castle::kDecodeStaticScratchBytes) return CASTLE_ERR_SCRATCH;
    float* p = nullptr;
    if (castle::decode_static_scratch(&p) != 0) return CASTLE_ERR_LAUNCH;
    workspace = p;
  } else if (workspace == nullptr || reinterpret_cast<uintptr_t>(workspace) % 256 != 0 ||
             workspace_bytes < castle_decode_workspace_bytes(B, H, d, t)) {
    return CASTLE_ERR_WORKSPACE;
  }

  a.B = B; a.H = H; a.d = d; a.t = t; a.scale = scale;
  a.t_dev = t_device; a.capacity = capacity;
  a.rotary = (flags & CASTLE_FLAG_ROTARY) != 0;
  a.u_half = (flags & CASTLE_FLAG_U_HALF) != 0;
  // the cache alone, where its size is known: 36 x 8 heads x 2080 rows (307 MB) 71 us a layer step, 78 read once; 42 x 8 (358 MB) 90, 86
  a.read_once = (flags & CASTLE_FLAG_READ_ONCE) != 0 || (t_device == nullptr && 4LL * B * H * t * d * es > 320000000);
  a.splits = splits;
  a.U = to_view(U); a.qu_cache = to_view(qu_cache); a.kc_cache = to_view(kc_cache); a.vc_cache = to_view(vc_cache);
  a.qc = to_view(qc); a.kc = to_view(kc); a.vc = to_view(vc);
  a.qu = to_view(qu); a.ku = to_view(ku); a.vu = to_view(vu);
  a.out = to_view(out);
  a.part = static_cast<float*>(workspace);
  a.arrivals = nullptr;
  a.pend_vu = to_view(deferred != nullptr ? &deferred->vu_ring : nullptr);
  a.pend_gate = to_view(deferred != nullptr ? &deferred->gates : nullptr);
  a.base0 = deferred != nullptr ? deferred->base : 0;
  a.base0_dev = deferred != nullptr ? deferred->base_device : nullptr;
  return CASTLE_OK;
}

static int decode_step_common(const castle_view4* U, const castle_view4* qu_cache,
                              const castle_view4* kc_cache, const castle_view4* vc_cache,
                              int t, const int* t_device, int capacity,
                              const castle_view4* qc, const castle_view4* kc, const castle_view4* vc,
                              const castle_view4* qu, const castle_view4* ku, const castle_view4* vu,
                              int B, int H, int d, int dtype, float scale, int flags,
                              const castle_view4* out, const castle_deferred* deferred,
                              void* workspace, int64_t workspace_bytes, bool static_scratch, void* stream) {
  if (out == nullptr) return CASTLE_ERR_ARG;
  castle::DecodeArgs a;
  const int rc = decode_step_args(a, U, qu_cache, kc_cache, vc_cache, t, t_device, capacity, qc, kc, vc, qu, ku, vu, B, H, d, dtype,
                                  scale, flags, out, deferred, workspace, workspace_bytes, static_scratch);
  return rc != CASTLE_OK ? rc : castle::launch_decode(a, dtype, static_cast<hipStream_t>(stream));
}

int castle_decode_step(const castle_view4* U, const castle_view4* qu_cache,
                       const castle_view4* kc_cache, const castle_view4* vc_cache, int t, int capacity,
                       const castle_view4* qc, const castle_view4* kc, const castle_view4* vc,
                       const castle_view4* qu, const castle_view4* ku, const castle_view4* vu,
                       int B, int H, int d, int dtype, float scale, int flags,
                       const castle_view4* out, const castle_deferred* deferred,
                       void* workspace, int64_t workspace_bytes, void* stream) {
  return decode_step_common(U, qu_cache, kc_cache, vc_cache, t, nullptr, capacity, qc, kc, vc, qu, ku, vu,
                            B, H, d, dtype, scale, flags, out, deferred, workspace, workspace_bytes, false, stream);
}

int castle_decode_step_static(const castle_view4* U, const castle_view4* qu_cache,
                              const castle_view4* kc_cache, const castle_view4* vc_cache,
                              int t, const int32_t* t_device, int capacity,
                              const castle_view4* qc, const castle_view4* kc, const castle_view4* vc,
                              const castle_view4* qu, const castle_view4* ku, const castle_view4* vu,
                              int B, int H, int d, int dtype, float scale, int flags,
                              const castle_view4* out, const castle_deferred* deferred, void* stream) {
  if (t_device != nullptr && reinterpret_cast<uintptr_t>(t_device) % 4 != 0) return CASTLE_ERR_ARG;
  return decode_step_common(U, qu_cache, kc_cache, vc_cache, t_device != nullptr ? 0 : t, t_device, capacity,
                            qc, kc, vc, qu, ku, vu, B, H, d, dtype, scale, flags, out, deferred, nullptr, 0, true, stream);
}

int castle_decode_step_device_count(const castle_view4* U, const castle_view4* qu_cache,
                                    const castle_view4* kc_cache, const castle_view4* vc_cache,
                                    const int32_t* t_device, int capacity,
                                    const castle_view4* qc, const castle_view4* kc, const castle_view4* vc,
                                    const castle_view4* qu, const castle_view4* ku, const castle_view4* vu,
                                    int B, int H, int d, int dtype, float scale, int flags,
                                    const castle_view4* out, const castle_deferred* deferred,
                                    void* workspace, int64_t workspace_bytes, void* stream) {
  if (t_device == nullptr || reinterpret_cast<uintptr_t>(t_device) % 4 != 0) return CASTLE_ERR_ARG;
  return decode_step_common(U, qu_cache, kc_cache, vc_cache, 0, t_device, capacity, qc, kc, vc, qu, ku, vu,
                            B, H, d, dtype, scale, flags, out, deferred, workspace, workspace_bytes, false, stream);
}

int64_t castle_decode_layer_control_bytes(int B, int H, int d, int dtype) {
  const int es = elem_size(dtype);
  if (es == 0) return CASTLE_ERR_DTYPE;
  if (B <= 0 || H <= 0 || !head_dim_ok(d) || (int64_t)B * H > 65535) return CASTLE_ERR_SHAPE;
  return align_up(castle::decode_layer_control_bytes(B, H, d, es), 256);
}

int castle_decode_layer_once_ok(int B, int H, int d, int dtype, int t, int dim) {
  const int es = elem_size(dtype);
  return es != 0 && B > 0 && H > 0 && t >= 0 && dim > 0 && head_dim_ok(d) && (int64_t)B * H <= 65535 && castle::decode_layer_once_ok(B, H, d, es, t, dim) ? 1 : 0;
}

static int decode_layer_common(const castle_view4* U, const castle_view4* qu_cache,
                        const castle_view4* kc_cache, const castle_view4* vc_cache,
                        int t, const int32_t* t_device, int capacity,
                        const void* x, int64_t ldx, int dim, const void* norm_weight, float eps,
                        const void* w_in, int64_t ldw_in, const void* w_out, int64_t ldw_out,
                        const void* residual, int64_t ldr, void* y, int64_t ldy, void* proj,
                        int B, int H, int d, int dtype, float scale, int flags, const castle_deferred* deferred,
                        void* workspace, int64_t workspace_bytes, void* control, int64_t control_bytes, void* stream) {
  const int es = elem_size(dtype);
  if (es == 0) return CASTLE_ERR_DTYPE;
  if (B <= 0 || H <= 0 || dim <= 0 || !head_dim_ok(d) || dim % (16 / es) != 0) return CASTLE_ERR_SHAPE;
  const void* p16[] = {x, w_in, w_out, proj};
  for (const void* p : p16)
    if (p == nullptr || reinterpret_cast<uintptr_t>(p) % 16 != 0) return CASTLE_ERR_ARG;
  if (y == nullptr || reinterpret_cast<uintptr_t>(norm_weight) % 16 != 0 || (norm_weight != nullptr && !(eps >= 0.f))) return CASTLE_ERR_ARG;
  const int q = 16 / es;
  if (ldx % q != 0 || ldw_in % q != 0 || ldw_out % q != 0) return CASTLE_ERR_ARG;
  if (t_device != nullptr && reinterpret_cast<uintptr_t>(t_device) % 4 != 0) return CASTLE_ERR_ARG;
  const int inner = H * d, width = 6 * inner;
  castle_view4 tok[6];   // qu, ku, vu, qc, kc, vc
  for (int i = 0; i < 6; ++i) tok[i] = {static_cast<char*>(proj) + (int64_t)i * inner * es, width, d, width};
  castle::DecodeArgs a;
  int rc = decode_step_args(a, U, qu_cache, kc_cache, vc_cache, t_device != nullptr ? 0 : t, t_device, capacity, &tok[3], &tok[4], &tok[5],
                            &tok[0], &tok[1], &tok[2], B, H, d, dtype, scale, flags, nullptr, deferred, workspace, workspace_bytes, false);
  if (rc != CASTLE_OK) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (control != nullptr) {
    if (reinterpret_cast<uintptr_t>(control) % 256 != 0 || control_bytes < castle_decode_layer_control_bytes(B, H, d, dtype)) return CASTLE_ERR_WORKSPACE;
    const castle::DecodeLinear in = {x, w_in, nullptr, B, width, dim, ldx, ldw_in, 0, norm_weight, eps, nullptr, 0};
    const castle::DecodeLinear out = {nullptr, w_out, y, B, dim, inner, 0, ldw_out, ldy, nullptr, 0.f, residual, ldr};
    rc = castle::launch_decode_layer(a, in, out, control, (flags & CASTLE_FLAG_STEP_TAKE_OVER) != 0, (flags & CASTLE_FLAG_STEP_GIVE_UP) != 0, dtype, s);
    if (rc != 1) return rc;
  }
  // the projection clears the arrival counts of the step, which then needs no launch to merge its splits
  a.arrivals = reinterpret_cast<int*>(a.part + (int64_t)B * H * 64 * (d + 2));
  rc = castle::launch_small_linear(x, w_in, proj, B, width, dim, ldx, ldw_in, width, dtype, norm_weight, eps, CASTLE_ACT_NONE, nullptr, 0, s, a.arrivals, B * H);
  a.out = to_view(&tok[0]);   // the attention output goes into the scratch: its token operands are spent by then
  if (rc == 0) rc = castle::launch_decode(a, dtype, s);
  if (rc != 0) return rc;
  return castle::launch_small_linear(proj, w_out, y, B, dim, inner, width, ldw_out, ldy, dtype, nullptr, 0.f, CASTLE_ACT_NONE, residual, ldr, s);
}

int castle_decode_layer(const castle_view4* U, const castle_view4* qu_cache,
                        const castle_view4* kc_cache, const castle_view4* vc_cache,
                        int t, const int32_t* t_device, int capacity,
                        const void* x, int64_t ldx, int dim, const void* norm_weight, float eps,
                        const void* w_in, int64_t ldw_in, const void* w_out, int64_t ldw_out,
                        const void* residual, int64_t ldr, void* y, int64_t ldy, void* proj,
                        int B, int H, int d, int dtype, float scale, int flags, const castle_deferred* deferred,
                        void* workspace, int64_t workspace_bytes, void* stream) {
  return decode_layer_common(U, qu_cache, kc_cache, vc_cache, t, t_device, capacity, x, ldx, dim, norm_weight, eps, w_in, ldw_in, w_out, ldw_out,
                             residual, ldr, y, ldy, proj, B, H, d, dtype, scale, flags, deferred, workspace, workspace_bytes, nullptr, 0, stream);
}

int castle_decode_layer_once(const castle_view4* U, const castle_view4* qu_cache,
                        const castle_view4* kc_cache, const castle_view4* vc_cache,
                        int t, const int32_t* t_device, int capacity,
                        const void* x, int64_t ldx, int dim, const void* norm_weight, float eps,
                        const void* w_in, int64_t ldw_in, const void* w_out, int64_t ldw_out,
                        const void* residual, int64_t ldr, void* y, int64_t ldy, void* proj,
                        int B, int H, int d, int dtype, float scale, int flags, const castle_deferred* deferred,
                        void* workspace, int64_t workspace_bytes, void* control, int64_t control_bytes, void* stream) {
  return decode_layer_common(U, qu_cache, kc_cache, vc_cache, t, t_device, capacity, x, ldx, dim, norm_weight, eps, w_in, ldw_in, w_out, ldw_out,
                             residual, ldr, y, ldy, proj, B, H, d, dtype, scale, flags, deferred, workspace, workspace_bytes, control, control_bytes, stream);
}

int castle_decode_flush(const castle_view4* U, const castle_view4* qu_cache, int t, const castle_deferred* deferred,
                        int B, int H, int d, int dtype, float scale, int flags, void* stream) {
  const int es = elem_size(dtype);
  if (es == 0) return CASTLE_ERR_DTYPE;
  if ((flags & CASTLE_FLAG_U_HALF) && dtype != CASTLE_BF16) return CASTLE_ERR_DTYPE;
  if (B <= 0 || H <= 0 || t < 0 || !head_dim_ok(d) || (int64_t)B * H > 65535) return CASTLE_ERR_SHAPE;
  if (!view_ok(U, es, true) || !view_ok(qu_cache, es, true) || deferred == nullptr) return CASTLE_ERR_ARG;
  if (!view_ok(&deferred->vu_ring, es, true) || !view_ok(&deferred->gates, 4, false)) return CASTLE_ERR_ARG;
  if (deferred->base < 0 || deferred->base > t) return CASTLE_ERR_SHAPE;
  if (t == 0 || castle::decode_base(deferred->base, t) == t) return CASTLE_OK;   // nothing pending
  castle::DecodeArgs a = {};
  a.B = B; a.H = H; a.d = d; a.t = t; a.scale = scale;
  a.U = to_view(U); a.qu_cache = to_view(qu_cache);
  a.pend_vu = to_view(&deferred->vu_ring); a.pend_gate = to_view(&deferred->gates);
  a.base0 = deferred->base;
  a.u_half = (flags & CASTLE_FLAG_U_HALF) != 0;
  return castle::launch_decode_flush(a, dtype, static_cast<hipStream_t>(stream));
}

int castle_rope(const castle_view4* x, const castle_view4* out, int B, int H, int L, int d, int dtype,
                int first_position, void* stream) {
  const int es = elem_size(dtype);
  if (es == 0) return CASTLE_ERR_DTYPE;
  if (B <= 0 || H <= 0 || L <= 0 || first_position < 0 || !head_dim_ok(d) || (int64_t)B * H > 65535) return CASTLE_ERR_SHAPE;
  if (!view_ok(x, es, true) || !view_ok(out, es, true)) return CASTLE_ERR_ARG;
  return castle::launch_rope(to_view(x), to_view(out), B, H, L, d, dtype, first_position, static_cast<hipStream_t>(stream));
}

int castle_cache_rows(const castle_view4* qu, const castle_view4* kc, const castle_view4* vc, const castle_view4* qu_cache,
                      const castle_view4* kc_cache, const castle_view4* vc_cache, int B, int H, int L, int d, int dtype, int flags, void* stream) {
  const int es = elem_size(dtype);
  if (es == 0) return CASTLE_ERR_DTYPE;
  if (B <= 0 || H <= 0 || L <= 0 || !head_dim_ok(d) || (int64_t)B * H > 65535) return CASTLE_ERR_SHAPE;
  const castle_view4* all[] = {qu, kc, vc, qu_cache, kc_cache, vc_cache};
  for (const castle_view4* v : all)
    if (!view_ok(v, es, true)) return CASTLE_ERR_ARG;
  const castle::View4 src[3] = {to_view(qu), to_view(kc), to_view(vc)}, dst[3] = {to_view(qu_cache), to_view(kc_cache), to_view(vc_cache)};
  return castle::launch_cache_rows(src, dst, B, H, L, d, dtype, (flags & CASTLE_FLAG_ROTARY) != 0, static_cast<hipStream_t>(stream));
}

int castle_small_linear_fused(const void* x, const void* w, void* y, int M, int N, int K,
                              int64_t ldx, int64_t ldw, int64_t ldy, int dtype,
                              const void* norm_weight, float eps, int activation,
                              const void* residual, int64_t ldr, void* stream) {
  if (dtype != CASTLE_BF16 && dtype != CASTLE_F16) return CASTLE_ERR_DTYPE;
  if (M <= 0 || N <= 0 || K <= 0 || K % 8 != 0 || N % 2 != 0) return CASTLE_ERR_SHAPE;
  if (x == nullptr || w == nullptr || y == nullptr) return CASTLE_ERR_ARG;
  if (reinterpret_cast<uintptr_t>(x) % 16 != 0 || reinterpret_cast<uintptr_t>(w) % 16 != 0 ||
      reinterpret_cast<uintptr_t>(y) % 4 != 0 || ldx % 8 != 0 || ldw % 8 != 0 || ldy % 2 != 0)
    return CASTLE_ERR_ARG;
  if (activation != CASTLE_ACT_NONE && activation != CASTLE_ACT_GELU) return CASTLE_ERR_ARG;
  if (norm_weight != nullptr && (reinterpret_cast<uintptr_t>(norm_weight) % 16 != 0 || !(eps >= 0.f))) return CASTLE_ERR_ARG;
  if (residual != nullptr && (reinterpret_cast<uintptr_t>(residual) % 4 != 0 || ldr % 2 != 0)) return CASTLE_ERR_ARG;
  return castle::launch_small_linear(x, w, y, M, N, K, ldx, ldw, ldy, dtype, norm_weight, eps, activation, residual, ldr,
                                     static_cast<hipStream_t>(stream));
}

int castle_small_linear(const void* x, const void* w, void* y, int M, int N, int K,
                        int64_t ldx, int64_t ldw, int64_t ldy, int dtype, void* stream) {
  return castle_small_linear_fused(x, w, y, M, N, K, ldx, ldw, ldy, dtype, nullptr, 0.f, CASTLE_ACT_NONE, nullptr, 0, stream);
}

int castle_sample(const void* logits, int64_t ld, const float* uniform, int rows, int vocabulary, int k, float inv_temperature,
                  int64_t* token, int64_t token_ld, int64_t* token_copy, int dtype, void* stream) {
  if (elem_size(dtype) == 0) return CASTLE_ERR_DTYPE;
  if (rows <= 0 || vocabulary <= 0 || k <= 0 || k > vocabulary) return CASTLE_ERR_SHAPE;
  if (logits == nullptr || token == nullptr || reinterpret_cast<uintptr_t>(token) % 8 != 0 || reinterpret_cast<uintptr_t>(token_copy) % 8 != 0 ||
      reinterpret_cast<uintptr_t>(uniform) % 4 != 0)
    return CASTLE_ERR_ARG;
  return castle::launch_sample(logits, ld, uniform, rows, vocabulary, k, inv_temperature, token, token_ld, token_copy, dtype,
                               static_cast<hipStream_t>(stream));
}

int castle_gather_rows(const void* table, int64_t table_rows, int64_t ld, int width, const int64_t* index, int n, void* y, int dtype, void* stream) {
  const int es = elem_size(dtype);
  if (es == 0) return CASTLE_ERR_DTYPE;
  if (table_rows <= 0 || width <= 0 || n <= 0 || (int64_t)width * es % 16 != 0) return CASTLE_ERR_SHAPE;
  if (table == nullptr || index == nullptr || y == nullptr || reinterpret_cast<uintptr_t>(table) % 16 != 0 || reinterpret_cast<uintptr_t>(y) % 16 != 0 ||
      ld * es % 16 != 0 || reinterpret_cast<uintptr_t>(index) % 8 != 0)
    return CASTLE_ERR_ARG;
  return castle::launch_gather_rows(table, (int64_t)width * es, ld * es, table_rows, index, n, y, static_cast<hipStream_t>(stream));
}

static bool row_pieces_ok(int n, int es) { return n > 0 && (int64_t)n * es % 16 == 0; }
static bool aligned16(std::initializer_list<const void*> ps) {
  for (const void* p : ps)
    if (reinterpret_cast<uintptr_t>(p) % 16 != 0) return false;
  return true;
}

int castle_rms_norm(const void* x, const void* delta, const void* weight, void* sum, void* h, float* rstd, int64_t rows, int width, float eps,
                    int dtype, void* stream) {
  const int es = elem_size(dtype);
  if (es == 0) return CASTLE_ERR_DTYPE;
  if (rows <= 0 || rows > kMaxRows || !row_pieces_ok(width, es) || (int64_t)width * es / 16 > castle::kMaxRowPieces) return CASTLE_ERR_SHAPE;
  if (x == nullptr || weight == nullptr || h == nullptr || (delta != nullptr && sum == nullptr) || !(eps >= 0.f) ||
      !aligned16({x, delta, weight, sum, h}) || reinterpret_cast<uintptr_t>(rstd) % 4 != 0)
    return CASTLE_ERR_ARG;
  const castle::NormArgs a = {x, delta, weight, sum, h, rstd, rows, width, eps};
  return castle::launch_norm(a, dtype, static_cast<hipStream_t>(stream));
}

int64_t castle_rms_norm_bwd_workspace_bytes(int64_t rows, int width, int dtype) {
  const int es = elem_size(dtype);
  if (es == 0) return CASTLE_ERR_DTYPE;
  if (rows <= 0 || rows > kMaxRows || !row_pieces_ok(width, es) || (int64_t)width * es / 16 > castle::kMaxRowPieces) return CASTLE_ERR_SHAPE;
  return align_up((int64_t)castle::norm_bwd_groups(rows, width, es) * width * 4, 256);
}

static int norm_bwd_common(castle_sum* dw_sum, const void* dh, const void* x, const void* weight, const float* rstd, const void* dres, void* dx, void* dweight,
                        int64_t rows, int width, int dtype, void* workspace, int64_t workspace_bytes, void* stream) {
  const int64_t need = castle_rms_norm_bwd_workspace_bytes(rows, width, dtype);
  if (need < 0) return (int)need;
  if (dh == nullptr || x == nullptr || weight == nullptr || rstd == nullptr || (dx == nullptr && dweight == nullptr) ||
      !aligned16({dh, x, weight, dres, dx}) || reinterpret_cast<uintptr_t>(rstd) % 4 != 0 ||
      reinterpret_cast<uintptr_t>(dweight) % elem_size(dtype) != 0)
    return CASTLE_ERR_ARG;
  if (dweight != nullptr && (workspace == nullptr || reinterpret_cast<uintptr_t>(workspace) % 16 != 0 || workspace_bytes < need)) return CASTLE_ERR_WORKSPACE;
  const castle::NormBwdArgs a = {dh, x, weight, dres, rstd, dx, dweight != nullptr ? static_cast<float*>(workspace) : nullptr, rows, width};
  castle::PartSum later = {};
  const int rc = castle::launch_norm_bwd(a, dweight, dtype, dw_sum != nullptr ? &later : nullptr, static_cast<hipStream_t>(stream));
  if (rc == 0 && dw_sum != nullptr) *dw_sum = {later.part, later.n, later.out, later.parts, later.columns};
  return rc;
}
int castle_rms_norm_bwd(const void* dh, const void* x, const void* weight, const float* rstd, const void* dres, void* dx, void* dweight,
                        int64_t rows, int width, int dtype, void* workspace, int64_t workspace_bytes, void* stream) {
  return norm_bwd_common(nullptr, dh, x, weight, rstd, dres, dx, dweight, rows, width, dtype, workspace, workspace_bytes, stream);
}
int castle_rms_norm_bwd_parts(const void* dh, const void* x, const void* weight, const float* rstd, const void* dres, void* dx, void* dweight, castle_sum* dw_sum,
                              int64_t rows, int width, int dtype, void* workspace, int64_t workspace_bytes, void* stream) {
  if (dw_sum == nullptr) return CASTLE_ERR_ARG;
  return norm_bwd_common(dw_sum, dh, x, weight, rstd, dres, dx, dweight, rows, width, dtype, workspace, workspace_bytes, stream);
}

int64_t castle_gemm_workspace_bytes(int M, int N, int K, int dtype, int epilogue) {
  const int es = elem_size(dtype);
  if (es == 0) return CASTLE_ERR_DTYPE;
  if (M <= 0 || N <= 0 || K <= 0 || N % (16 / es) != 0 || (int64_t)(M / 64 + 1) * (N / 64 + 1) > (int64_t)1 << 30) return CASTLE_ERR_SHAPE;
  return align_up(castle::gemm_workspace(M, N, K, es, epilogue != CASTLE_GEMM_PLAIN), 256);
}

int castle_gemm_plan(int M, int N, int K, int dtype, int epilogue, int* rows, int* columns, int* ranges, int* groups) {
  const int64_t need = castle_gemm_workspace_bytes(M, N, K, dtype, epilogue);
  if (need < 0) return (int)need;
  if (rows == nullptr || columns == nullptr || ranges == nullptr || groups == nullptr) return CASTLE_ERR_ARG;
  int out[4];
  castle::gemm_plan(M, N, K, elem_size(dtype), epilogue != CASTLE_GEMM_PLAIN, out);
  *rows = out[0]; *columns = out[1]; *ranges = out[2]; *groups = out[3];
  return CASTLE_OK;
}

int castle_gemm_amax_ok(int M, int N, int K, int dtype, int column, int columns) {
  const int es = elem_size(dtype);
  if (es == 0 || M <= 0 || N <= 0 || K <= 0 || column < 0 || columns <= 0 || column + columns > N || column % (16 / es) != 0 || columns % (16 / es) != 0) return 0;
  return castle::gemm_amax_ok(M, N, K, es, column, column + columns);
}

// The kernels form element offsets in 32 bits.  The first step of a range of the contraction, or of the second group of waves in it, may start up to two
// steps (128 rows, 127 of them behind the last one) from the end; places further on are only stepped to, in unsigned numbers, and never read.
int castle_gemm_operand_ok(int64_t rows, int64_t ld) { return rows >= 0 && ld >= 0 && ld < (int64_t)1 << 31 && rows < (int64_t)1 << 31 && (rows + 192) * ld < (int64_t)1 << 31; }

int castle_gemm_norm_ok(int M, int N, int K, int dtype) {
  const int es = elem_size(dtype);
  return es != 0 && M > 0 && N > 0 && K > 0 && K % (16 / es) == 0 && N % (16 / es) == 0 && castle::gemm_norm_ok(M, N, K, es) ? 1 : 0;
}

static int gemm_common(const castle_gemm_norm* norm, const void* a, int64_t lda, int a_free_contiguous, const void* b, int64_t ldb, int b_free_contiguous, void* c, int64_t ldc,
                int M, int N, int K, int dtype, int epilogue, void* aux, const castle_amax* amax, void* workspace, int64_t workspace_bytes, void* stream) {
  const int64_t need = castle_gemm_workspace_bytes(M, N, K, dtype, epilogue);
  if (need < 0) return (int)need;
  static_assert(CASTLE_AMAX_PARTIALS == castle::kAmaxBlocks && CASTLE_GEMM_PLAIN == castle::kGemmPlain && CASTLE_GEMM_GELU == castle::kGemmGelu && CASTLE_GEMM_GELU_SLOPE == castle::kGemmGeluSlope, "");
  const int v = 16 / elem_size(dtype);
  const int a_row = a_free_contiguous ? M : K, b_row = b_free_contiguous ? N : K;
  if (!castle_gemm_operand_ok(a_free_contiguous ? K : M, lda) || !castle_gemm_operand_ok(b_free_contiguous ? K : N, ldb)) return CASTLE_ERR_SHAPE;
  if (a_row % v != 0 || b_row % v != 0 || lda < a_row || ldb < b_row || ldc < N || lda % v != 0 || ldb % v != 0 || ldc % v != 0 ||
      (a_free_contiguous && !b_free_contiguous))
    return CASTLE_ERR_SHAPE;
  if (epilogue < CASTLE_GEMM_PLAIN || epilogue > CASTLE_GEMM_GELU_SLOPE || a == nullptr || b == nullptr || c == nullptr ||
      (epilogue != CASTLE_GEMM_PLAIN && aux == nullptr) || !aligned16({a, b, c, aux}))
    return CASTLE_ERR_ARG;
  if (need > 0 && (ldc != N || (int64_t)M * N % 8 != 0)) return CASTLE_ERR_SHAPE;
  if (need > 0 && (workspace == nullptr || !aligned16({workspace}) || workspace_bytes < need)) return CASTLE_ERR_WORKSPACE;
  castle::GemmArgs args = {a, b, c, aux, M, N, K, lda, ldb, ldc, epilogue, 0, nullptr, nullptr, nullptr, 0, 1, nullptr, 0.f, nullptr, nullptr};
  if (norm != nullptr) {
    if (!castle_gemm_norm_ok(M, N, K, dtype) || a_free_contiguous || b_free_contiguous || epilogue != CASTLE_GEMM_PLAIN) return CASTLE_ERR_SHAPE;
    if (norm->weight == nullptr || !(norm->eps >= 0.f) || !aligned16({norm->h}) || reinterpret_cast<uintptr_t>(norm->weight) % elem_size(dtype) != 0 ||
        reinterpret_cast<uintptr_t>(norm->rstd) % 4 != 0 || (norm->rstd != nullptr && norm->h == nullptr))
      return CASTLE_ERR_ARG;
    args.norm_w = norm->weight;
    args.eps = norm->eps;
    args.h = norm->h;
    args.rstd = norm->rstd;
  }
  if (amax != nullptr) {
    if (!castle_gemm_amax_ok(M, N, K, dtype, amax->column, amax->columns)) return CASTLE_ERR_SHAPE;
    if (amax->partials == nullptr || reinterpret_cast<uintptr_t>(amax->partials) % 4 != 0 || reinterpret_cast<uintptr_t>(amax->status) % 4 != 0) return CASTLE_ERR_ARG;
    args.amax = amax->partials;
    args.amax_status = amax->status;
    args.amax_from = amax->column;
    args.amax_to = amax->column + amax->columns;
  }
  return castle::launch_gemm(args, !a_free_contiguous, !b_free_contiguous, dtype, static_cast<float*>(workspace), static_cast<hipStream_t>(stream));
}

int castle_gemm(const void* a, int64_t lda, int a_free_contiguous, const void* b, int64_t ldb, int b_free_contiguous, void* c, int64_t ldc,
                int M, int N, int K, int dtype, int epilogue, void* aux, const castle_amax* amax, void* workspace, int64_t workspace_bytes, void* stream) {
  return gemm_common(nullptr, a, lda, a_free_contiguous, b, ldb, b_free_contiguous, c, ldc, M, N, K, dtype, epilogue, aux, amax, workspace, workspace_bytes, stream);
}
int castle_gemm_of_norm(const void* a, int64_t lda, const castle_gemm_norm* norm, const void* b, int64_t ldb, void* c, int64_t ldc, int M, int N, int K,
                        int dtype, const castle_amax* amax, void* stream) {
  if (norm == nullptr) return CASTLE_ERR_ARG;
  return gemm_common(norm, a, lda, 0, b, ldb, 0, c, ldc, M, N, K, dtype, CASTLE_GEMM_PLAIN, nullptr, amax, nullptr, 0, stream);
}

int64_t castle_projection_grads_workspace_bytes(int R, int N, int K, int dtype, int epilogue, int with_amax) {
  const int es = elem_size(dtype);
  if (es == 0) return CASTLE_ERR_DTYPE;
  if (R <= 0 || N <= 0 || K <= 0 || N % 8 != 0 || K % 8 != 0 || (int64_t)(std::max(R, N) / 32 + 1) * (std::max(N, K) / 32 + 1) > (int64_t)1 << 30) return CASTLE_ERR_SHAPE;
  if (epilogue != CASTLE_GEMM_PLAIN && epilogue != CASTLE_GEMM_GELU_SLOPE) return CASTLE_ERR_ARG;
  const int64_t n = castle::grads_workspace(R, N, K, es, epilogue, with_amax != 0);
  return n < 0 ? CASTLE_ERR_SHAPE : align_up(n, 256);
}

int castle_projection_grads_plan(int R, int N, int K, int dtype, int epilogue, int with_amax, int* tile, int* waves, int* dw_ranges, int* dx_ranges) {
  const int64_t need = castle_projection_grads_workspace_bytes(R, N, K, dtype, epilogue, with_amax);
  if (need < 0) return (int)need;
  if (tile == nullptr || waves == nullptr || dw_ranges == nullptr || dx_ranges == nullptr) return CASTLE_ERR_ARG;
  const castle::GradsPlan g = castle::grads_plan(R, N, K, elem_size(dtype), epilogue, with_amax != 0);
  *tile = g.tile; *waves = g.waves; *dw_ranges = g.w_splits; *dx_ranges = g.x_splits;
  return CASTLE_OK;
}

int castle_projection_grads(const void* dy, int64_t ld_dy, const void* x, int64_t ld_x, const void* w, int64_t ld_w, void* dw, void* dx, int R, int N, int K,
                            int dtype, int epilogue, const void* aux, const castle_amax* amax, castle_sum* dw_sum, void* workspace, int64_t workspace_bytes, void* stream) {
  const int64_t need = castle_projection_grads_workspace_bytes(R, N, K, dtype, epilogue, amax != nullptr);
  if (need < 0) return (int)need;
  const int v = 16 / elem_size(dtype);
  if (!castle_gemm_operand_ok(R, ld_dy) || !castle_gemm_operand_ok(R, ld_x) || !castle_gemm_operand_ok(N, ld_w) || ld_dy < N || ld_x < K || ld_w < K || ld_dy % v != 0 ||
      ld_x % v != 0 || ld_w % v != 0)
    return CASTLE_ERR_SHAPE;
  if (dy == nullptr || x == nullptr || w == nullptr || dw == nullptr || dx == nullptr || (epilogue != CASTLE_GEMM_PLAIN && aux == nullptr) || !aligned16({dy, x, w, dw, dx, aux}))
    return CASTLE_ERR_ARG;
  if (need > 0 && (workspace == nullptr || !aligned16({workspace}) || workspace_bytes < need)) return CASTLE_ERR_WORKSPACE;
  castle::GradsArgs p = {};
  p.w = {dy, x, dw, nullptr, N, K, R, ld_dy, ld_x, K, castle::kGemmPlain, 0, nullptr, nullptr, nullptr, 0, 1, nullptr, 0.f, nullptr, nullptr};
  p.x = {dy, w, dx, const_cast<void*>(aux), R, K, N, ld_dy, ld_w, K, epilogue, 0, nullptr, nullptr, nullptr, 0, 1, nullptr, 0.f, nullptr, nullptr};
  if (amax != nullptr) {
    if (amax->column < 0 || amax->columns <= 0 || amax->column + amax->columns > K || amax->column % v != 0 || amax->columns % v != 0) return CASTLE_ERR_SHAPE;
    if (amax->partials == nullptr || reinterpret_cast<uintptr_t>(amax->partials) % 4 != 0 || reinterpret_cast<uintptr_t>(amax->status) % 4 != 0) return CASTLE_ERR_ARG;
    p.x.amax = amax->partials;
    p.x.amax_status = amax->status;
    p.x.amax_from = amax->column;
    p.x.amax_to = amax->column + amax->columns;
  }
  castle::PartSum later;
  const int rc = castle::launch_grads(p, dtype, static_cast<float*>(workspace), dw_sum != nullptr ? &later : nullptr, static_cast<hipStream_t>(stream));
  if (rc == 0 && dw_sum != nullptr) {
    if (later.parts > 0) *dw_sum = {later.part, later.n, later.out, later.parts, later.columns};
    else *dw_sum = {nullptr, 0, nullptr, 0, 0};
  }
  return rc;
}

int castle_sum_parts(const float* part, int parts, int64_t n, void* out, int dtype, void* stream) {
  if (elem_size(dtype) == 0) return CASTLE_ERR_DTYPE;
  if (parts <= 0 || n <= 0 || n % 8 != 0 || n / 8 > kMaxRows) return CASTLE_ERR_SHAPE;
  if (part == nullptr || out == nullptr || !aligned16({part, out})) return CASTLE_ERR_ARG;
  return castle::launch_part_sum(part, parts, n, out, dtype, static_cast<hipStream_t>(stream));
}

int castle_sums(const castle_sum* sums, int count, int dtype, void* stream) {
  if (elem_size(dtype) == 0) return CASTLE_ERR_DTYPE;
  static_assert(CASTLE_MAX_SUMS == castle::kMaxSums, "");
  if (sums == nullptr || count <= 0 || count > CASTLE_MAX_SUMS) return CASTLE_ERR_ARG;
  castle::PartSum jobs[CASTLE_MAX_SUMS];
  for (int j = 0; j < count; ++j) {
    const castle_sum& s = sums[j];
    if (s.parts <= 0 || s.n <= 0 || s.n / 8 > kMaxRows || (s.columns ? s.n > 0x7ffffff : s.n % 8 != 0)) return CASTLE_ERR_SHAPE;
    if (s.part == nullptr || s.out == nullptr || (s.columns ? reinterpret_cast<uintptr_t>(s.part) % 4 != 0 || reinterpret_cast<uintptr_t>(s.out) % elem_size(dtype) != 0
                                                            : !aligned16({s.part, s.out})))
      return CASTLE_ERR_ARG;
    jobs[j] = {s.part, s.n, s.out, s.parts, s.columns};
  }
  return castle::launch_sums(jobs, count, dtype, static_cast<hipStream_t>(stream));
}

static int cross_entropy_args(castle::CrossEntropyArgs& a, const void* logits, const int64_t* target, int64_t target_n, int64_t target_ld, int64_t rows,
                              int classes, const float* lse, int dtype) {
  const int es = elem_size(dtype);
  if (es == 0) return CASTLE_ERR_DTYPE;
  if (rows <= 0 || rows > kMaxRows || target_n <= 0 || rows % target_n != 0 || !row_pieces_ok(classes, es)) return CASTLE_ERR_SHAPE;
  if (logits == nullptr || target == nullptr || lse == nullptr || !aligned16({logits}) || reinterpret_cast<uintptr_t>(target) % 8 != 0 ||
      reinterpret_cast<uintptr_t>(lse) % 4 != 0)
    return CASTLE_ERR_ARG;
  a = {logits, target, rows, target_n, target_ld, classes, const_cast<float*>(lse), nullptr};
  return CASTLE_OK;
}

int castle_cross_entropy(const void* logits, const int64_t* target, int64_t target_n, int64_t target_ld, int64_t rows, int classes, void* loss,
                         float* lse, float* inv_count, int dtype, void* workspace, int64_t workspace_bytes, void* stream) {
  castle::CrossEntropyArgs a;
  const int rc = cross_entropy_args(a, logits, target, target_n, target_ld, rows, classes, lse, dtype);
  if (rc != CASTLE_OK) return rc;
  if (loss == nullptr || inv_count == nullptr || reinterpret_cast<uintptr_t>(loss) % elem_size(dtype) != 0 || reinterpret_cast<uintptr_t>(inv_count) % 4 != 0)
    return CASTLE_ERR_ARG;
  if (workspace == nullptr || reinterpret_cast<uintptr_t>(workspace) % 16 != 0 || workspace_bytes < CASTLE_CROSS_ENTROPY_WORKSPACE) return CASTLE_ERR_WORKSPACE;
  static_assert(CASTLE_CROSS_ENTROPY_WORKSPACE >= castle::kCrossEntropyGroups * 8, "two floats a group");
  a.part = static_cast<float*>(workspace);
  return castle::launch_cross_entropy(a, loss, inv_count, dtype, static_cast<hipStream_t>(stream));
}

int castle_cross_entropy_bwd(const void* logits, const int64_t* target, int64_t target_n, int64_t target_ld, int64_t rows, int classes,
                             const float* lse, const float* inv_count, const void* grad, void* dlogits, int dtype, void* stream) {
  castle::CrossEntropyArgs a;
  const int rc = cross_entropy_args(a, logits, target, target_n, target_ld, rows, classes, lse, dtype);
  if (rc != CASTLE_OK) return rc;
  if (inv_count == nullptr || grad == nullptr || dlogits == nullptr || !aligned16({dlogits})) return CASTLE_ERR_ARG;
  return castle::launch_cross_entropy_bwd(a, grad, inv_count, dlogits, dtype, static_cast<hipStream_t>(stream));
}

int64_t castle_embedding_grad_workspace_bytes(int64_t rows, int vocabulary, int width, int dtype) {
  const int es = elem_size(dtype);
  if (es == 0) return CASTLE_ERR_DTYPE;
  // every (vocabulary row, chunk) reads the token numbers of its chunk: above 2^26 of them (0.5 GB, about what the sort of
  // the library's operator costs) this is not the way
  if (rows <= 0 || vocabulary <= 0 || rows > kMaxRows || rows * vocabulary > (int64_t)1 << 26 || !row_pieces_ok(width, es) ||
      (int64_t)width * es / 16 > castle::kMaxRowPieces || castle::embedding_grad_chunks(rows) > 65535)
    return CASTLE_ERR_SHAPE;
  return align_up((int64_t)castle::embedding_grad_chunks(rows) * vocabulary * width * 4, 256);
}

int castle_embedding_grad(const void* dy, const int64_t* index, int64_t index_n, int64_t index_ld, int64_t rows, int vocabulary, int width,
                          void* dweight, int dtype, void* workspace, int64_t workspace_bytes, void* stream) {
  const int64_t need = castle_embedding_grad_workspace_bytes(rows, vocabulary, width, dtype);
  if (need < 0) return (int)need;
  if (index_n <= 0 || rows % index_n != 0 || (int64_t)vocabulary * width % 8 != 0) return CASTLE_ERR_SHAPE;
  if (dy == nullptr || index == nullptr || dweight == nullptr || !aligned16({dy, dweight}) || reinterpret_cast<uintptr_t>(index) % 8 != 0) return CASTLE_ERR_ARG;
  if (workspace == nullptr || reinterpret_cast<uintptr_t>(workspace) % 256 != 0 || workspace_bytes < need) return CASTLE_ERR_WORKSPACE;
  const castle::EmbeddingGradArgs a = {dy, index, rows, index_n, index_ld, vocabulary, width, static_cast<float*>(workspace)};
  return castle::launch_embedding_grad(a, dweight, dtype, static_cast<hipStream_t>(stream));
}

int castle_profile_enable(int on) { return castle::profile_enable(on); }

int castle_profile_read(int* slots, float* ms, int max_records) {
  if (slots == nullptr || ms == nullptr || max_records < 0) return CASTLE_ERR_ARG;
  return castle::profile_read(slots, ms, max_records);
}

}  // extern "C"
