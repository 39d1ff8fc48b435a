// extern "C" boundary of libtriattention_hip.so: argument validation on the host,
// then kernel launches on the caller's stream.  Nothing here allocates or waits.
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <algorithm>
#include <atomic>
#include <climits>
#include <mutex>

#include "tri_common.h"

// Scratch of tri_compress_step_static: one copy per GPU, loaded with the code object.  In host
// code this name is only a handle for hipGetSymbolAddress; the address kernels are given is
// the one that call returns on the device in question.
static __device__ __align__(256) unsigned char scratch[TRI_STATIC_WORKSPACE_BYTES];

namespace {

thread_local char g_err[512] = "";

int fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

int launch_status(hipError_t e, const char* what) {
  if (e == hipSuccess) return TRI_OK;
  return fail(TRI_ERR_LAUNCH, "%s: %s", what, hipGetErrorString(e));
}

bool is_aligned(const void* p, size_t a) { return (reinterpret_cast<uintptr_t>(p) % a) == 0; }

int elem_bytes(int dt) { return dt == TRI_KV_FP8_E4M3 ? 1 : 2; }

int check_layout(const tri_kv_layout* kv, bool need_v) {
  if (!kv) return fail(TRI_ERR_INVALID_ARGUMENT, "kv layout is NULL");
  if (kv->num_layers <= 0 || kv->num_kv_heads <= 0 || kv->num_kv_heads > 256)
    return fail(TRI_ERR_INVALID_ARGUMENT, "bad layer/head count (%d, %d)", kv->num_layers, kv->num_kv_heads);
  if (kv->head_dim != 64 && kv->head_dim != 128 && kv->head_dim != 256)
    return fail(TRI_ERR_UNSUPPORTED, "head_dim %d not in {64,128,256}", kv->head_dim);
  if (kv->block_size <= 0) return fail(TRI_ERR_INVALID_ARGUMENT, "block_size %d", kv->block_size);
  if (kv->kv_dtype != TRI_KV_BF16 && kv->kv_dtype != TRI_KV_FP16 && kv->kv_dtype != TRI_KV_FP8_E4M3)
    return fail(TRI_ERR_INVALID_ARGUMENT, "kv_dtype %d", kv->kv_dtype);
  if (kv->rope_style != TRI_ROPE_HALF && kv->rope_style != TRI_ROPE_INTERLEAVED)
    return fail(TRI_ERR_INVALID_ARGUMENT, "rope_style %d", kv->rope_style);
  const int eb = elem_bytes(kv->kv_dtype);
  const int64_t per16 = 16 / eb;   // elements per 16-byte access
  if (kv->stride_block % per16 || kv->stride_token % per16 || kv->stride_head % per16)
    return fail(TRI_ERR_INVALID_ARGUMENT, "strides must be multiples of %lld elements (16 bytes)", (long long)per16);
  if (kv->stride_head < kv->head_dim && kv->num_kv_heads > 1)
    return fail(TRI_ERR_INVALID_ARGUMENT, "stride_head %lld < head_dim", (long long)kv->stride_head);
  if (!kv->k_layers) return fail(TRI_ERR_INVALID_ARGUMENT, "k_layers is NULL");
  if (need_v && !kv->v_layers) return fail(TRI_ERR_INVALID_ARGUMENT, "v_layers is NULL");
  if (kv->kv_dtype == TRI_KV_FP8_E4M3 && !kv->k_scale_layers)
    return fail(TRI_ERR_INVALID_ARGUMENT, "fp8 cache without k_scale_layers");
  // v_scale_layers may be NULL: the rows then carry no scales of their own (a cache with one
  // scale per tensor) and compaction moves rows only.
  return TRI_OK;
}

int check_batch(const tri_batch* b, bool need_budget) {
  if (!b) return fail(TRI_ERR_INVALID_ARGUMENT, "batch is NULL");
  if (b->num_seqs <= 0) return fail(TRI_ERR_INVALID_ARGUMENT, "num_seqs %d", b->num_seqs);
  if (b->max_seq_len <= 0) return fail(TRI_ERR_INVALID_ARGUMENT, "max_seq_len %d", b->max_seq_len);
  if (!b->seq_lens) return fail(TRI_ERR_INVALID_ARGUMENT, "seq_lens is NULL");
  if (b->block_table && b->block_table_pitch <= 0)
    return fail(TRI_ERR_INVALID_ARGUMENT, "block_table_pitch %d", b->block_table_pitch);
  if (b->seq_lens_host)
    for (int i = 0; i < b->num_seqs; ++i)
      if (b->seq_lens_host[i] < 0 || b->seq_lens_host[i] > b->max_seq_len)
        return fail(TRI_ERR_INVALID_ARGUMENT, "seq_lens_host[%d] = %d not in [0, max_seq_len = %d]", i,
                    b->seq_lens_host[i], b->max_seq_len);
  if (need_budget) {
    if (!b->budgets) return fail(TRI_ERR_INVALID_ARGUMENT, "budgets is NULL");
    if (b->max_budget <= 0) return fail(TRI_ERR_INVALID_ARGUMENT, "max_budget %d", b->max_budget);
  }
  return TRI_OK;
}

int check_score(const tri_kv_layout* kv, const tri_score_params* sp) {
  if (!sp) return fail(TRI_ERR_INVALID_ARGUMENT, "score params are NULL");
  if (sp->num_score_heads <= 0 || sp->num_score_heads % kv->num_kv_heads)
    return fail(TRI_ERR_INVALID_ARGUMENT, "num_score_heads %d is not a multiple of num_kv_heads %d",
                sp->num_score_heads, kv->num_kv_heads);
  if (sp->num_offsets <= 0 || sp->num_offsets > tri::kMaxOffsets)
    return fail(TRI_ERR_INVALID_ARGUMENT, "num_offsets %d not in [1, %d]", sp->num_offsets, tri::kMaxOffsets);
  if (sp->aggregation != TRI_REDUCE_MEAN && sp->aggregation != TRI_REDUCE_MAX)
    return fail(TRI_ERR_INVALID_ARGUMENT, "aggregation %d", sp->aggregation);
  if (!sp->folded || !sp->omega || !sp->offsets)
    return fail(TRI_ERR_INVALID_ARGUMENT, "folded / omega / offsets is NULL");
  if (!is_aligned(sp->folded, 16)) return fail(TRI_ERR_INVALID_ARGUMENT, "folded must be 16-byte aligned");
  return TRI_OK;
}

tri::Workspace plan(const tri_kv_layout* kv, const tri_batch* b, const tri_score_params* sp, int assume_resident = 0,
                    bool allow_resident = true) {
  // Resident kernels: two-byte and fp8 keys go to the matrix-core kernel where the shape has one,
  // and only launches that fill most of the chip take them.  TRI_TUNE_RESIDENT_KERNEL overrides
  // the choice: 1 / 2 take the matrix-core / vector-unit kernel whenever the shape has it (however
  // small the launch), 3 never takes a resident kernel.
  const int64_t force = tri::tuning(TRI_TUNE_RESIDENT_KERNEL);
  const bool f_valu = force == 2;
  const bool f_mfma = force == 1;
  const bool f_off = force == 3;
  // The matrix-core kernel addresses the 16 rows of a step with 32-bit offsets from a scalar base.
  const bool want_mfma = (kv->kv_dtype == TRI_KV_BF16 || kv->kv_dtype == TRI_KV_FP16 || kv->kv_dtype == TRI_KV_FP8_E4M3) &&
                         !f_valu &&
                         kv->stride_token > 0 && kv->stride_token < (1 << 25);
  const int G = sp->num_score_heads / kv->num_kv_heads;
  const bool paged = b->block_table != nullptr;
  // assume_resident > 0: a dry run for a device of that size (tri_describe_plan); no device is asked.
  const int resident = (f_off || !allow_resident) ? 0
                       : (assume_resident > 0 ? assume_resident : tri::fused_resident_workgroups());
  tri::FusedPlan fused{};
  // Small batches are cut by layers as well (TRI_TUNE_LAYER_SPLIT = 0 switches that off, 1 switches
  // it on where the kernel was forced, which otherwise keeps whole-model workgroups).
  const int64_t split_set = tri::tuning(TRI_TUNE_LAYER_SPLIT);
  const bool split = split_set >= 0 ? split_set != 0 : !f_mfma;
  if (want_mfma)
    fused = tri::plan_fused_mfma(b->num_seqs, kv->num_kv_heads, kv->head_dim, G, kv->block_size, paged,
                                 sp->aggregation, b->max_seq_len, resident, f_mfma, kv->kv_dtype, b->seq_lens_host,
                                 kv->num_layers, split);
  if (!fused.eligible && !f_mfma)
    fused = tri::plan_fused(b->num_seqs, kv->num_kv_heads, kv->head_dim, G, kv->block_size, paged, sp->aggregation,
                            b->max_seq_len, resident, f_valu);
  return tri::plan_workspace(b->num_seqs, kv->num_layers, sp->num_score_heads, kv->head_dim / 2, sp->num_offsets,
                             kv->num_kv_heads, b->max_seq_len, fused);
}

int check_workspace(const tri::Workspace& w, void* ws, uint64_t bytes) {
  if (!ws) return fail(TRI_ERR_WORKSPACE, "workspace is NULL");
  if (!is_aligned(ws, 256)) return fail(TRI_ERR_WORKSPACE, "workspace must be 256-byte aligned");
  if (bytes < (uint64_t)w.total)
    return fail(TRI_ERR_WORKSPACE, "workspace has %llu bytes, %lld needed", (unsigned long long)bytes, (long long)w.total);
  return TRI_OK;
}

struct ResidentGate {
  static constexpr int kMaxDevices = 64;
  std::mutex mutex;
  hipEvent_t event[kMaxDevices] = {};
};
ResidentGate& resident_gate() {
  static ResidentGate gate;
  return gate;
}

// Both with the gate's mutex held.  A stream under capture is left alone.
bool gate_applies(hipStream_t s, int& dev) {
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  return hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < ResidentGate::kMaxDevices &&
         hipStreamIsCapturing(s, &cap) == hipSuccess && cap == hipStreamCaptureStatusNone;
}
int gate_enter(ResidentGate& gate, hipStream_t s) {
  int dev = 0;
  if (!gate_applies(s, dev) || !gate.event[dev]) return TRI_OK;
  return launch_status(hipStreamWaitEvent(s, gate.event[dev], 0), "resident chain wait");
}
int gate_leave(ResidentGate& gate, hipStream_t s) {
  int dev = 0;
  if (!gate_applies(s, dev)) return TRI_OK;
  if (!gate.event[dev]) {
    const hipError_t e = hipEventCreateWithFlags(&gate.event[dev], hipEventDisableTiming);
    if (e != hipSuccess) return launch_status(e, "resident chain event");
  }
  return launch_status(hipEventRecord(gate.event[dev], s), "resident chain record");
}

// Process-wide settings (tri_set_tuning).
constexpr int kTunings = 5;
std::atomic<int64_t> g_tuning[kTunings] = {{0}, {0}, {-1}, {0}, {2000000}};

// Device address of `scratch` on the current device, looked up once per device.
struct StaticScratch {
  static constexpr int kMaxDevices = 64;
  std::mutex mutex;
  void* ptr[kMaxDevices] = {};
};
int static_scratch(void** out) {
  static StaticScratch st;
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return launch_status(e, "hipGetDevice");
  if (dev < 0 || dev >= StaticScratch::kMaxDevices) return fail(TRI_ERR_UNSUPPORTED, "device %d out of range", dev);
  std::lock_guard<std::mutex> lock(st.mutex);
  if (!st.ptr[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return launch_status(e, "hipGetSymbolAddress(scratch)");
    if (!p || !is_aligned(p, 256)) return fail(TRI_ERR_WORKSPACE, "static scratch at %p is not 256-byte aligned", p);
    st.ptr[dev] = p;
  }
  *out = st.ptr[dev];
  return TRI_OK;
}

template <typename T>
T* at(void* ws, int64_t off) { return reinterpret_cast<T*>(reinterpret_cast<char*>(ws) + off); }

int do_score(const tri_kv_layout* kv, const tri_batch* batch, const tri_score_params* sp, float* raw,
             int64_t rs_layer, int64_t rs_token, int64_t rs_head, void* ws, const tri::Workspace& w,
             hipStream_t s, int fine, float* partial, uint32_t* status) {
  const int F = kv->head_dim / 2;
  hipError_t e = tri::launch_prepare(sp->folded, sp->omega, sp->offsets, sp->num_offsets, batch->round_start,
                                     batch->num_seqs, kv->num_layers, sp->num_score_heads, F, sp->aggregation,
                                     at<float>(ws, w.coef), at<float>(ws, w.trig), status, s);
  if (e != hipSuccess) return launch_status(e, "prepare");
  tri::ScoreLaunch a{};
  a.B = batch->num_seqs; a.L = kv->num_layers; a.Hkv = kv->num_kv_heads; a.D = kv->head_dim;
  a.block_size = kv->block_size; a.kv_dtype = kv->kv_dtype; a.rope_style = kv->rope_style;
  a.A = sp->num_score_heads; a.G = sp->num_score_heads / kv->num_kv_heads; a.NO = sp->num_offsets;
  a.aggregation = sp->aggregation;
  a.Tmax = batch->max_seq_len; a.fine = fine;
  a.stride_block = kv->stride_block; a.stride_token = kv->stride_token; a.stride_head = kv->stride_head;
  a.k_layers = kv->k_layers; a.k_scale_layers = kv->k_scale_layers;
  a.block_table = batch->block_table; a.block_table_pitch = batch->block_table_pitch;
  a.seq_lens = batch->seq_lens;
  a.coef = at<float>(ws, w.coef); a.trig = at<float>(ws, w.trig); a.partial = partial;
  a.raw = raw; a.raw_stride_layer = rs_layer; a.raw_stride_token = rs_token; a.raw_stride_head = rs_head;
  return launch_status(tri::launch_score(a, s), "score");
}

int check_select(const tri_select_params* sel) {
  if (!sel) return fail(TRI_ERR_INVALID_ARGUMENT, "select params are NULL");
  if (sel->group_reduce != TRI_REDUCE_MEAN && sel->group_reduce != TRI_REDUCE_MAX)
    return fail(TRI_ERR_INVALID_ARGUMENT, "group_reduce %d", sel->group_reduce);
  if (sel->layer_reduce != TRI_REDUCE_MEAN && sel->layer_reduce != TRI_REDUCE_MAX && sel->layer_reduce != -1)
    return fail(TRI_ERR_INVALID_ARGUMENT, "layer_reduce %d", sel->layer_reduce);
  if (sel->window_size < 0) return fail(TRI_ERR_INVALID_ARGUMENT, "window_size %d", sel->window_size);
  if (sel->normalize < 0 || sel->normalize > 2) return fail(TRI_ERR_INVALID_ARGUMENT, "normalize %d", sel->normalize);
  if (sel->normalize == 2 && sel->group_first)
    return fail(TRI_ERR_UNSUPPORTED, "the population-std normalisation is built for the normalise-then-reduce order only");
  return TRI_OK;
}

int do_select(const tri_kv_layout* kv, const tri_batch* batch, const tri_score_params* sp,
              const tri_select_params* sel, const float* raw, int64_t rs_layer, int64_t rs_token,
              int64_t rs_head, float* fin, int32_t* keep, void* ws, const tri::Workspace& w, hipStream_t s,
              int fine, const float* partial, int pass_nan) {
  tri::SelectLaunch a{};
  a.B = batch->num_seqs; a.L = kv->num_layers; a.Hkv = kv->num_kv_heads; a.A = sp->num_score_heads;
  a.G = sp->num_score_heads / kv->num_kv_heads; a.Tmax = batch->max_seq_len; a.fine = fine;
  a.max_budget = batch->max_budget;
  a.normalize = sel->normalize; a.window_size = sel->window_size; a.protect_prefill = sel->protect_prefill;
  a.group_reduce = sel->group_reduce; a.layer_reduce = sel->layer_reduce; a.shared = sel->shared;
  a.group_first = sel->group_first ? 1 : 0;
  a.pass_nan = pass_nan;
  a.seq_lens = batch->seq_lens; a.prefill_lens = batch->prefill_lens; a.budgets = batch->budgets;
  a.partial = partial; a.mustd = at<float>(ws, w.mustd);
  a.raw = raw; a.raw_stride_layer = rs_layer; a.raw_stride_token = rs_token; a.raw_stride_head = rs_head;
  a.fin = fin ? fin : at<float>(ws, w.fin);
  a.keep = keep;
  // Scratch of the chunked statistics: the coefficients (the scorer is done with them) or, where one score per KV head
  // needs no sums of the scorer's tiles, the room planned for those.
  a.group_scratch = at<double>(ws, pass_nan ? w.partial : w.coef);
  a.group_scratch_bytes = pass_nan ? w.mustd - w.partial : w.trig - w.coef;
  return launch_status(tri::launch_select(a, s), "select");
}

// A keep set per layer (layer_reduce -1) of a single layer is the mean over that one layer: same
// rows, same scores (x / 1).  The reference's per-layer modes call their selector once per layer
// (runtime/selector_hf.py:473-747 from the layer loop), so those calls may take a resident kernel.
int layer_reduce_of(const tri_kv_layout* kv, const tri_select_params* sel) {
  return (sel->layer_reduce < 0 && kv->num_layers == 1) ? TRI_REDUCE_MEAN : sel->layer_reduce;
}

bool takes_resident(const tri::Workspace& w, const tri_kv_layout* kv, const tri_select_params* sel) {
  return w.fused.eligible && layer_reduce_of(kv, sel) >= 0 && !sel->shared && !sel->group_first && !sel->no_resident;
}

// Quarter tiles of the two-pass scorer.  Their sums take more room than the workspace plans; they go where the
// selection scores are written later (the statistics are finished by then).
bool takes_quarter_tiles(const tri_kv_layout* kv, int B, int Tmax, int A, int aggregation) {
  const int64_t sums = (int64_t)B * kv->num_layers * A * tri::ceil_div(Tmax, tri::kScoreFineTokens) * 4 * 4;
  const int64_t room = tri::align_up((int64_t)B * kv->num_layers * kv->num_kv_heads * Tmax * 4, 256);   // Workspace::fin
  return sums <= room && tri::score_takes_fine(B, kv->num_layers, kv->num_kv_heads, kv->head_dim, A / kv->num_kv_heads,
                                               Tmax, aggregation);
}

// A few layers of a few requests, where the resident kernel would be taken for them, go through
// tri_score_small.hip: a wave per step of 16 tokens, statistics in the selection's workgroups.  Which of the two is faster goes by
//  - the scorer's workgroups (128 tokens of a KV head of a layer), each of which evaluates the phases again: one round
//    of the chip is 1024 of them, 512 at a head dimension of 256;
//  - the layers, which the selection walks one after the other, the longer the more tokens a thread holds of a row: up to
//    4096 tokens four (one query head per KV head 8192, eight), beyond that twice as many;
//  - what the resident kernel costs: with at most four KV heads its workgroups have four waves and it is about 5 us faster.
// Score + select, called eagerly (the event that chains resident launches is 3 us of theirs; a captured launch has none), us,
// resident / small, `layers x requests x tokens, KV heads x head dimension, workgroups`.  Two to four query heads per KV
// head: 1 x 8 x 1987, 8 x 128, 1024: 31.0 / 24.9; 1 x 4 x 3923, 8 x 256, 992: 41.5 / 34.9; 2 x 1 x 3771, 16 x 128, 960:
// 33.9 / 27.3; 3 x 3 x 1663, 8 x 64, 936: 29.6 / 25.1; 4 x 8 x 415, 8 x 128, 1024: 33.7 / 33.0.  Four KV heads: 2 x 4 x 3495, 4 x 64, 896:
// 27.3 / 22.2; 3 x 8 x 1057, 4 x 128, 864: 28.0 / 26.4, but 3 x 8 x 1075, 4 x 256, 864: 32.1 / 36.4 and 4 x 3 x 2596, 4 x 64, 1008:
// 27.0 / 28.2.  Long rows: 1 x 4 x 7782, 4 x 64, 976: 31.0 / 25.8; 2 x 1 x 7139, 8 x 128, 896: 36.7 / 32.2, but 2 x 3 x 5038, 4 x 128, 960:
// 31.1 / 32.7, 3 x 1 x 5052, 8 x 128, 960: 35.7 / 37.7, 3 x 2 x 5036, 4 x 128, 960: 31.5 / 37.8, 4 x 1 x 4170, 1 x 64, 132: 27.9 / 30.9 and
// 4 x 1 x 7652, 4 x 256, 960: 39.5 / 51.0.  One query head: 4 x 1 x 7964, 4 x 64, 1008: 33.2 / 28.7; 2 x 1 x 14202, 4 x 128, 888:
// 38.7 / 35.4, but 3 x 1 x 8914, 4 x 128, 840: 36.4 / 37.3, 4 x 1 x 14881, 2 x 128, 936: 40.4 / 42.7.  Eight: 1 x 4 x 3821, 8 x 128, 960:
// 32.7 / 30.4; 2 x 2 x 3534, 4 x 128, 448: 27.4 / 25.6, but 1 x 8 x 3770, 4 x 128, 960: 26.7 / 29.9.  Of 830 shapes drawn over 1 to
// 4 layers, 1 to 8 query heads, 1 to 16 KV heads of 64 to 256 and 64 to 1024 workgroups 760 go this way, two of them more than
// 2 % slower (1.04 x), and seven of the others would be more than 2 % faster.
int64_t small_workgroups(int L, int G, int D, int Tmax, bool four_waves) {
  const bool wide = D == 256, long_rows = Tmax > (G == 1 ? 8192 : 4096);
  if (L > (G > 4 ? 2 : 4)) return 0;
  if (G > 4) return std::min(1024 / L, four_waves ? (wide ? 512 : 768) : 1024);
  if (long_rows) return L == 1 ? 1024 : L == 2 ? (four_waves && G > 1 ? 768 : 1024) : L == 3 ? (four_waves ? 512 : 768) : G == 1 ? 512 : 0;
  if (four_waves && G > 1 && L >= 3) return wide ? 512 : L == 4 ? 704 : 1024;
  return 1024;
}
bool takes_small(const tri::Workspace& w, const tri_kv_layout* kv, const tri_batch* batch, const tri_score_params* sp,
                 const tri_select_params* sel) {
  const int G = sp->num_score_heads / kv->num_kv_heads, L = kv->num_layers;
  const int64_t wgs = (int64_t)batch->num_seqs * L * kv->num_kv_heads * tri::ceil_div(batch->max_seq_len, 128);
  return tri::tuning(TRI_TUNE_RESIDENT_KERNEL) == 0 && takes_resident(w, kv, sel) && w.fused.eligible == 2 &&
         kv->kv_dtype != TRI_KV_FP8_E4M3 && tri::select_small_takes(batch->max_seq_len, G) &&
         (int64_t)batch->num_seqs * kv->num_kv_heads <= 256 &&
         wgs <= small_workgroups(L, G, kv->head_dim, batch->max_seq_len, w.fused.waves == 4);
}

// Selection straight from the paged keys: the resident kernel when the shape has one,
// else score into the workspace and select from there.
int do_select_paged(const tri_kv_layout* kv, const tri_batch* batch, const tri_score_params* sp,
                    const tri_select_params* sel, float* fin, int32_t* keep, void* ws, const tri::Workspace& w,
                    hipStream_t s, int pass_nan = 0) {
  if (takes_small(w, kv, batch, sp, sel)) {
    tri::SmallScore c{};
    c.k_layers = kv->k_layers; c.block_table = batch->block_table; c.block_table_pitch = batch->block_table_pitch;
    c.seq_lens = batch->seq_lens; c.round_start = batch->round_start;
    c.folded = sp->folded; c.omega = sp->omega; c.offsets = sp->offsets; c.NO = sp->num_offsets;
    c.raw = at<float>(ws, w.raw); c.raw_pitch = batch->max_seq_len; c.status = at<uint32_t>(ws, w.status);
    c.stride_block = kv->stride_block; c.stride_token = kv->stride_token; c.stride_head = kv->stride_head;
    c.L = kv->num_layers; c.A = sp->num_score_heads; c.G = sp->num_score_heads / kv->num_kv_heads;
    c.Tmax = batch->max_seq_len; c.block_size = kv->block_size;
    hipError_t e = tri::launch_score_small(c, batch->num_seqs, kv->num_kv_heads, kv->head_dim, kv->kv_dtype, kv->rope_style, s);
    if (e != hipSuccess) return launch_status(e, "score_small");
    tri::SmallSelect a{};
    a.raw = c.raw; a.raw_pitch = c.raw_pitch; a.seq_lens = batch->seq_lens; a.prefill_lens = batch->prefill_lens;
    a.budgets = batch->budgets; a.fin = fin; a.keep = keep; a.keep_pitch = batch->max_budget; a.status = c.status;
    a.L = c.L; a.Hkv = kv->num_kv_heads; a.A = c.A; a.G = c.G; a.Tmax = c.Tmax;
    a.normalize = sel->normalize; a.window_size = sel->window_size; a.protect_prefill = sel->protect_prefill;
    a.group_reduce = sel->group_reduce; a.layer_reduce = layer_reduce_of(kv, sel); a.pass_nan = 0;
    return launch_status(tri::launch_select_small(a, batch->num_seqs, s), "select_small");
  }
  const bool fused = takes_resident(w, kv, sel);
  if (!fused) {
    float* raw = at<float>(ws, w.raw);
    const int64_t A = sp->num_score_heads;
    const int64_t rs_layer = (int64_t)batch->max_seq_len * A;
    const int fine = takes_quarter_tiles(kv, batch->num_seqs, batch->max_seq_len, (int)A, sp->aggregation);
    float* partial = at<float>(ws, fine ? w.fin : w.partial);
    // The status word belongs to the resident kernel; on this path it just reads "fine".
    const int rc = do_score(kv, batch, sp, raw, rs_layer, A, 1, ws, w, s, fine, partial, at<uint32_t>(ws, w.status));
    if (rc) return rc;
    return do_select(kv, batch, sp, sel, raw, rs_layer, A, 1, fin, keep, ws, w, s, fine, partial, pass_nan);
  }
  const int F = kv->head_dim / 2;
  hipError_t e = hipSuccess;
  if (w.fused.eligible != 2) {   // the matrix-core kernel has a preparation launch of its own
    e = tri::launch_prepare(sp->folded, sp->omega, sp->offsets, sp->num_offsets, batch->round_start,
                            batch->num_seqs, kv->num_layers, sp->num_score_heads, F, sp->aggregation,
                            at<float>(ws, w.coef), at<float>(ws, w.trig), nullptr, s);
    if (e != hipSuccess) return launch_status(e, "prepare");
  }
  tri::FusedLaunch a{};
  a.B = batch->num_seqs; a.L = kv->num_layers; a.Hkv = kv->num_kv_heads; a.D = kv->head_dim;
  a.block_size = kv->block_size; a.kv_dtype = kv->kv_dtype; a.rope_style = kv->rope_style;
  a.A = sp->num_score_heads; a.G = sp->num_score_heads / kv->num_kv_heads; a.Tmax = batch->max_seq_len;
  a.normalize = sel->normalize; a.window_size = sel->window_size; a.protect_prefill = sel->protect_prefill;
  a.group_reduce = sel->group_reduce; a.layer_reduce = layer_reduce_of(kv, sel);
  a.stride_block = kv->stride_block; a.stride_token = kv->stride_token; a.stride_head = kv->stride_head;
  a.k_layers = kv->k_layers; a.k_scale_layers = kv->k_scale_layers;
  a.block_table = batch->block_table; a.block_table_pitch = batch->block_table_pitch;
  a.seq_lens = batch->seq_lens; a.prefill_lens = batch->prefill_lens;
  a.coef = at<float>(ws, w.coef);
  a.folded = sp->folded; a.omega = sp->omega; a.offsets = sp->offsets; a.NO = sp->num_offsets;
  a.round_start = batch->round_start;
  a.xchg = at<unsigned long long>(ws, w.xchg);
  a.status = at<uint32_t>(ws, w.status);
  a.pack = at<int32_t>(ws, w.pack);
  a.fin = fin ? fin : at<float>(ws, w.fin);
  // Partial results of a layer-split launch live where the two-pass path keeps its raw scores
  // ([B][L][Tmax][A] floats, never smaller than [groups][B][Hkv][Tmax]).
  a.fin_part = at<float>(ws, w.raw);
  a.plan = w.fused;
  // Nobody asked for the selection scores themselves: the groups' partial rows go straight to the
  // top-k, which adds them while it loads (one launch less).
  const bool split = w.fused.eligible == 2 && w.fused.layer_groups > 1;
  a.skip_layer_reduce = split && !fin && keep && batch->max_seq_len <= tri::topk_register_row_limit();
  a.bmat = at<char>(ws, w.bmat);
  if (w.fused.eligible == 2) {
    // The preparation launch writes one 16-byte entry per (sequence, layer, KV head, operand, lane); the region planned for them must hold that.
    const int64_t need = (int64_t)a.B * a.L * a.Hkv * tri::mfma_operands(F, a.G) * 64 * 16;
    if (need > w.total - w.bmat)
      return fail(TRI_ERR_WORKSPACE, "coefficient slabs need %lld bytes, %lld planned", (long long)need,
                  (long long)(w.total - w.bmat));
  }
  {
    // Two resident launches that run at the same time on one device would each hold part of
    // the CUs and wait for the other's workgroups until their waits expire.  Launches of this
    // process are therefore chained: each waits (on the device, not on the host) for the
    // previous one on whatever stream that was.  Streams under graph capture are left alone
    // (whoever replays the graph brackets the replay with tri_resident_gate_enter / _leave).
    ResidentGate& gate = resident_gate();
    std::lock_guard<std::mutex> lock(gate.mutex);
    int rc = gate_enter(gate, s);
    if (rc) return rc;
    e = w.fused.eligible == 2 ? tri::launch_fused_mfma(a, s) : tri::launch_fused_select(a, s);
    if (e != hipSuccess) return launch_status(e, "fused_select");
    rc = gate_leave(gate, s);
    if (rc) return rc;
  }
  if (!keep) return TRI_OK;   // selection scores only
  if (a.skip_layer_reduce)
    return launch_status(tri::launch_topk_rows(a.fin_part, a.Tmax, a.B * a.Hkv, a.seq_lens, batch->budgets, a.Hkv, a.Tmax,
                                               keep, batch->max_budget, s, w.fused.layer_groups,
                                               (int64_t)a.B * a.Hkv * a.Tmax, a.layer_reduce == TRI_REDUCE_MAX),
                         "topk_rows");
  return launch_status(tri::launch_topk_rows(a.fin, a.Tmax, a.B * a.Hkv, a.seq_lens, batch->budgets, a.Hkv, a.Tmax, keep,
                                             batch->max_budget, s),
                       "topk_rows");
}

int fill_compact(const tri_kv_layout* kv, const tri_batch* batch, const int32_t* keep, int keep_per_layer,
                 int shared, tri::CompactLaunch& a) {
  int rc = check_layout(kv, true);
  if (rc) return rc;
  rc = check_batch(batch, true);
  if (rc) return rc;
  if (!batch->block_table) return fail(TRI_ERR_INVALID_ARGUMENT, "compaction needs a block table");
  if (!keep) return fail(TRI_ERR_INVALID_ARGUMENT, "keep is NULL");
  const int eb = elem_bytes(kv->kv_dtype);
  a.B = batch->num_seqs; a.L = kv->num_layers; a.Hkv = kv->num_kv_heads; a.D = kv->head_dim;
  a.block_size = kv->block_size; a.elem_bytes = eb; a.max_budget = batch->max_budget;
  a.keep_per_layer = keep_per_layer ? 1 : 0; a.shared = shared ? 1 : 0;
  a.has_scales = kv->kv_dtype == TRI_KV_FP8_E4M3 && kv->v_scale_layers != nullptr;
  a.stride_block = kv->stride_block; a.stride_token = kv->stride_token; a.stride_head = kv->stride_head;
  a.k_layers = kv->k_layers; a.v_layers = kv->v_layers;
  a.k_scale_layers = kv->k_scale_layers; a.v_scale_layers = kv->v_scale_layers;
  a.block_table = batch->block_table; a.block_table_pitch = batch->block_table_pitch;
  a.seq_lens = batch->seq_lens; a.budgets = batch->budgets; a.keep = keep; a.Tmax = batch->max_seq_len;
  a.staging = nullptr;
  return TRI_OK;
}

}  // namespace

namespace tri {
int64_t tuning(int key) { return key >= 0 && key < kTunings ? g_tuning[key].load(std::memory_order_relaxed) : 0; }
}  // namespace tri

extern "C" {

int tri_abi_version(void) { return TRI_ABI_VERSION; }

const char* tri_last_error(void) { return g_err; }

#ifndef TRI_SOURCE_DIGEST
#define TRI_SOURCE_DIGEST "unknown"
#endif
const char* tri_source_digest(void) {
  static const char digest[] = "TRI_SOURCE_DIGEST=" TRI_SOURCE_DIGEST;
  return digest + sizeof("TRI_SOURCE_DIGEST=") - 1;
}

int tri_set_tuning(int32_t key, int64_t value) {
  switch (key) {
    case TRI_TUNE_RESIDENT_KERNEL:
      if (value < 0 || value > 3) return fail(TRI_ERR_INVALID_ARGUMENT, "TRI_TUNE_RESIDENT_KERNEL takes 0..3, got %lld", (long long)value);
      break;
    case TRI_TUNE_RESIDENT_WORKGROUPS:
      if (value < 0 || value > INT_MAX) return fail(TRI_ERR_INVALID_ARGUMENT, "TRI_TUNE_RESIDENT_WORKGROUPS %lld", (long long)value);
      break;
    case TRI_TUNE_LAYER_SPLIT:
      if (value < -1 || value > 1) return fail(TRI_ERR_INVALID_ARGUMENT, "TRI_TUNE_LAYER_SPLIT takes -1, 0 or 1, got %lld", (long long)value);
      break;
    case TRI_TUNE_MAX_KERNEL:
      if (value < 0 || value > 1) return fail(TRI_ERR_INVALID_ARGUMENT, "TRI_TUNE_MAX_KERNEL takes 0 or 1, got %lld", (long long)value);
      break;
    case TRI_TUNE_RESIDENT_WAIT_US:
      // (the kernels count ticks of a 100 MHz clock in 64 bits)
      if (value > (int64_t)3600 * 1000000) return fail(TRI_ERR_INVALID_ARGUMENT, "TRI_TUNE_RESIDENT_WAIT_US beyond one hour");
      break;
    default:
      return fail(TRI_ERR_INVALID_ARGUMENT, "unknown tuning key %d", key);
  }
  g_tuning[key].store(value, std::memory_order_relaxed);
  return TRI_OK;
}

int64_t tri_get_tuning(int32_t key) {
  if (key < 0 || key >= kTunings) return INT64_MIN;
  return g_tuning[key].load(std::memory_order_relaxed);
}

int tri_resident_gate_enter(void* stream) {
  ResidentGate& gate = resident_gate();
  std::lock_guard<std::mutex> lock(gate.mutex);
  return gate_enter(gate, (hipStream_t)stream);
}

int tri_resident_gate_leave(void* stream) {
  ResidentGate& gate = resident_gate();
  std::lock_guard<std::mutex> lock(gate.mutex);
  return gate_leave(gate, (hipStream_t)stream);
}

int tri_fold_stats(const float* q_mean_real, const float* q_mean_imag, const float* q_abs_mean,
                   const float* freq_scale_sq, int32_t num_layers, int32_t num_score_heads,
                   int32_t num_pairs, int32_t disable_mlr, int32_t disable_trig, float* folded,
                   void* stream) {
  if (!q_mean_real || !q_mean_imag || !q_abs_mean || !freq_scale_sq || !folded)
    return fail(TRI_ERR_INVALID_ARGUMENT, "tri_fold_stats: NULL pointer");
  if (num_layers <= 0 || num_score_heads <= 0 || num_pairs <= 0)
    return fail(TRI_ERR_INVALID_ARGUMENT, "tri_fold_stats: bad sizes (%d, %d, %d)", num_layers, num_score_heads, num_pairs);
  return launch_status(tri::launch_fold_stats(q_mean_real, q_mean_imag, q_abs_mean, freq_scale_sq, num_layers,
                                              num_score_heads, num_pairs, disable_mlr, disable_trig, folded,
                                              (hipStream_t)stream),
                       "fold_stats");
}

uint64_t tri_workspace_bytes(const tri_kv_layout* kv, const tri_batch* batch, const tri_score_params* sp) {
  if (check_layout(kv, false) || check_batch(batch, false) || !sp || sp->num_score_heads <= 0 ||
      sp->num_offsets <= 0)
    return 0;
  return (uint64_t)plan(kv, batch, sp).total;
}

uint64_t tri_workspace_status_offset(const tri_kv_layout* kv, const tri_batch* batch,
                                     const tri_score_params* sp) {
  if (check_layout(kv, false) || check_batch(batch, false) || !sp || sp->num_score_heads <= 0 ||
      sp->num_offsets <= 0)
    return 0;
  return (uint64_t)plan(kv, batch, sp).status;
}

int tri_score_paged(const tri_kv_layout* kv, const tri_batch* batch, const tri_score_params* sp,
                    float* raw, int64_t raw_stride_layer, int64_t raw_stride_token,
                    int64_t raw_stride_head, void* workspace, uint64_t workspace_bytes, void* stream) {
  int rc = check_layout(kv, false);
  if (rc) return rc;
  rc = check_batch(batch, false);
  if (rc) return rc;
  rc = check_score(kv, sp);
  if (rc) return rc;
  if (!batch->round_start) return fail(TRI_ERR_INVALID_ARGUMENT, "round_start is NULL");
  if (!raw) return fail(TRI_ERR_INVALID_ARGUMENT, "raw is NULL");
  const tri::Workspace w = plan(kv, batch, sp);
  rc = check_workspace(w, workspace, workspace_bytes);
  if (rc) return rc;
  return do_score(kv, batch, sp, raw, raw_stride_layer, raw_stride_token, raw_stride_head, workspace, w,
                  (hipStream_t)stream, 0, at<float>(workspace, w.partial), nullptr);
}

int tri_select(const tri_kv_layout* kv, const tri_batch* batch, const tri_score_params* sp,
               const tri_select_params* sel, const float* raw, int64_t raw_stride_layer,
               int64_t raw_stride_token, int64_t raw_stride_head, float* final_scores, int32_t* keep,
               void* workspace, uint64_t workspace_bytes, void* stream) {
  int rc = check_layout(kv, false);
  if (rc) return rc;
  rc = check_batch(batch, true);
  if (rc) return rc;
  if (!sp || sp->num_score_heads <= 0 || sp->num_score_heads % kv->num_kv_heads || sp->num_offsets <= 0)
    return fail(TRI_ERR_INVALID_ARGUMENT, "tri_select: bad score params");
  rc = check_select(sel);
  if (rc) return rc;
  if (!raw || !keep) return fail(TRI_ERR_INVALID_ARGUMENT, "raw / keep is NULL");
  const tri::Workspace w = plan(kv, batch, sp);
  rc = check_workspace(w, workspace, workspace_bytes);
  if (rc) return rc;
  return do_select(kv, batch, sp, sel, raw, raw_stride_layer, raw_stride_token, raw_stride_head, final_scores,
                   keep, workspace, w, (hipStream_t)stream, 0, at<float>(workspace, w.partial), 0);
}

int tri_select_paged(const tri_kv_layout* kv, const tri_batch* batch, const tri_score_params* sp,
                     const tri_select_params* sel, float* final_scores, int32_t* keep, void* workspace,
                     uint64_t workspace_bytes, void* stream) {
  int rc = check_layout(kv, false);
  if (rc) return rc;
  rc = check_batch(batch, true);
  if (rc) return rc;
  rc = check_score(kv, sp);
  if (rc) return rc;
  rc = check_select(sel);
  if (rc) return rc;
  if (!batch->round_start) return fail(TRI_ERR_INVALID_ARGUMENT, "round_start is NULL");
  if (!keep && !final_scores) return fail(TRI_ERR_INVALID_ARGUMENT, "keep and final_scores are both NULL");
  const tri::Workspace w = plan(kv, batch, sp);
  rc = check_workspace(w, workspace, workspace_bytes);
  if (rc) return rc;
  return do_select_paged(kv, batch, sp, sel, final_scores, keep, workspace, w, (hipStream_t)stream);
}

int tri_select_path(const tri_kv_layout* kv, const tri_batch* batch, const tri_score_params* sp,
                    const tri_select_params* sel) {
  if (check_layout(kv, false) || check_batch(batch, false) || check_score(kv, sp) || check_select(sel)) return -1;
  const tri::Workspace w = plan(kv, batch, sp);
  return takes_resident(w, kv, sel) ? w.fused.eligible : 0;
}

int tri_describe_plan(const tri_kv_layout* kv, const tri_batch* batch, const tri_score_params* sp,
                      const tri_select_params* sel, int32_t assume_resident_workgroups, tri_plan_info* out) {
  if (!out) return fail(TRI_ERR_INVALID_ARGUMENT, "tri_describe_plan: out is NULL");
  if (assume_resident_workgroups < 0)
    return fail(TRI_ERR_INVALID_ARGUMENT, "assume_resident_workgroups %d", assume_resident_workgroups);
  int rc = check_layout(kv, false);
  if (!rc) rc = check_batch(batch, false);
  if (!rc) rc = check_score(kv, sp);
  if (!rc) rc = check_select(sel);
  if (rc) return rc;
  const tri::Workspace w = plan(kv, batch, sp, assume_resident_workgroups);
  *out = tri_plan_info{};
  out->workspace_bytes = w.total;
  out->layer_groups = 1;
  out->layers_per_group = kv->num_layers;
  if (!takes_resident(w, kv, sel)) return TRI_OK;
  const tri::FusedPlan& f = w.fused;
  out->path = f.eligible;
  out->tile_tokens = f.tile_tokens;
  out->tiles_per_seq = f.tiles_per_seq;
  out->resident_workgroups = (f.eligible == 2 && f.waves == 4) ? f.resident / 2 : f.resident;
  out->waves_per_workgroup = f.eligible == 2 ? f.waves : 8;
  if (f.eligible == 2 && f.layer_groups > 1) {
    out->layer_groups = f.layer_groups;
    out->layers_per_group = f.layers_per_group;
  }
  if (batch->num_seqs <= f.seqs_per_launch) out->launches = 1;
  else out->launches = f.launches;      // > 0: the planner replayed the packing of the host's lengths
  return TRI_OK;
}

int tri_small_launches(const tri_kv_layout* kv, const tri_batch* batch, const tri_score_params* sp,
                       const tri_select_params* sel, int32_t assume_resident_workgroups) {
  if (check_layout(kv, false) || check_batch(batch, false) || check_score(kv, sp) || check_select(sel)) return -1;
  if (assume_resident_workgroups < 0) {
    fail(TRI_ERR_INVALID_ARGUMENT, "assume_resident_workgroups %d", assume_resident_workgroups);
    return -1;
  }
  return takes_small(plan(kv, batch, sp, assume_resident_workgroups), kv, batch, sp, sel) ? 1 : 0;
}

int32_t tri_score_tile_tokens(const tri_kv_layout* kv, int32_t num_seqs, int32_t max_seq_len, int32_t num_score_heads,
                              int32_t aggregation) {
  if (check_layout(kv, false) || num_seqs <= 0 || max_seq_len <= 0 || num_score_heads <= 0 ||
      num_score_heads % kv->num_kv_heads)
    return 0;
  return takes_quarter_tiles(kv, num_seqs, max_seq_len, num_score_heads, aggregation) ? tri::kScoreFineTokens
                                                                                      : tri::kScoreTileTokens;
}

int tri_topk_rows(const float* scores, int64_t row_pitch, int32_t num_rows, const int32_t* row_lens,
                  const int32_t* row_ks, int32_t rows_per_entry, int32_t max_len, int32_t* keep,
                  int32_t keep_pitch, void* stream) {
  if (!scores || !row_lens || !row_ks || !keep) return fail(TRI_ERR_INVALID_ARGUMENT, "tri_topk_rows: NULL pointer");
  if (num_rows < 0 || rows_per_entry <= 0 || row_pitch < max_len || keep_pitch <= 0 || max_len <= 0)
    return fail(TRI_ERR_INVALID_ARGUMENT, "tri_topk_rows: bad sizes");
  return launch_status(tri::launch_topk_rows(scores, row_pitch, num_rows, row_lens, row_ks, rows_per_entry, max_len, keep,
                                             keep_pitch, (hipStream_t)stream),
                       "topk_rows");
}

namespace {

// Workgroups of 128 tokens and a head up to which a dense call goes through the small launch's kernels (8 heads: 600 tokens
// 38 -> 21 us, 4096 44 -> 21, 9000 56 -> 35, 16384 52 -> 37, of 256 elements 57 -> 49; 128 heads of 256 x 2048 tokens 100 -> 98; longer rows
// do not fit the selection's registers).
constexpr int64_t kDenseSmallWorkgroups = 2048;

// A dense call as the general layout, batch and parameters, on a workspace whose last part holds what those
// point to.
struct DensePlan {
  tri_kv_layout kv{};
  tri_batch batch{};
  tri_score_params sp{};
  tri_select_params sel{};
  tri::Workspace w{};
  int64_t arg_key, arg_words, folded, keep32, total;
};

int plan_dense(const tri_dense_params* p, DensePlan& d) {
  if (!p) return fail(TRI_ERR_INVALID_ARGUMENT, "dense params are NULL");
  if (p->kv_dtype != TRI_KV_BF16 && p->kv_dtype != TRI_KV_FP16)
    return fail(TRI_ERR_UNSUPPORTED, "tri_dense_compress takes two-byte keys, got kv_dtype %d", p->kv_dtype);
  if (p->num_tokens <= 0 || p->budget <= 0 || p->budget > p->num_tokens)
    return fail(TRI_ERR_INVALID_ARGUMENT, "budget %d of %d tokens", p->budget, p->num_tokens);
  if (p->k_stride_head % 2 || p->k_stride_token % 2)
    return fail(TRI_ERR_INVALID_ARGUMENT, "key strides must be whole elements");
  d.kv.num_layers = 1; d.kv.num_kv_heads = p->num_heads; d.kv.head_dim = p->head_dim; d.kv.block_size = p->num_tokens;
  d.kv.kv_dtype = p->kv_dtype; d.kv.rope_style = p->rope_style;
  d.kv.stride_block = p->k_stride_head / 2 * p->num_heads;          // one sequence: never used as a distance
  d.kv.stride_token = p->k_stride_token / 2; d.kv.stride_head = p->k_stride_head / 2;
  d.batch.num_seqs = 1; d.batch.max_seq_len = p->num_tokens; d.batch.max_budget = p->budget;
  d.sp.num_score_heads = p->num_heads; d.sp.num_offsets = p->num_offsets; d.sp.aggregation = p->aggregation;
  d.sel.normalize = p->normalize ? 1 : 0; d.sel.window_size = p->window_size;
  d.sel.group_reduce = TRI_REDUCE_MAX; d.sel.layer_reduce = TRI_REDUCE_MEAN;
  d.sel.group_first = 1; d.sel.no_resident = 1;
  if (p->num_heads <= 0 || p->num_heads > 256 ||
      (p->head_dim != 64 && p->head_dim != 128 && p->head_dim != 256) || p->num_offsets <= 0)
    return fail(TRI_ERR_UNSUPPORTED, "%d heads of %d, %d offsets", p->num_heads, p->head_dim, p->num_offsets);
  d.w = plan(&d.kv, &d.batch, &d.sp, 0, false);
  int64_t off = d.w.total;
  auto take = [&](int64_t bytes) { const int64_t o = off; off = tri::align_up(off + bytes, 256); return o; };
  d.arg_key = take(8);
  d.arg_words = take(12);
  d.folded = take((int64_t)p->num_heads * 3 * (p->head_dim / 2) * 4);
  d.keep32 = take((int64_t)p->num_heads * p->budget * 4);
  d.total = off;
  return TRI_OK;
}

}  // namespace

uint64_t tri_dense_workspace_bytes(const tri_dense_params* params) {
  DensePlan d;
  return plan_dense(params, d) ? 0 : (uint64_t)d.total;
}

int tri_dense_compress(const tri_dense_params* p, void* ws, uint64_t ws_bytes, void* stream) {
  DensePlan d;
  int rc = plan_dense(p, d);
  if (rc) return rc;
  tri::Workspace need = d.w;
  need.total = d.total;
  rc = check_workspace(need, ws, ws_bytes);
  if (rc) return rc;
  if (!p->k || !p->v || !p->q_mean_complex || !p->q_abs_mean || !p->freq_scale_sq || !p->out_k || !p->out_v || !p->out_keep)
    return fail(TRI_ERR_INVALID_ARGUMENT, "tri_dense_compress: NULL pointer");
  if (!is_aligned(p->k, 16) || !is_aligned(p->v, 16) || !is_aligned(p->out_k, 16) || !is_aligned(p->out_v, 16))
    return fail(TRI_ERR_INVALID_ARGUMENT, "tri_dense_compress: bases must be 16-byte aligned");
  if (p->v_row_bytes <= 0 || p->v_row_bytes % 16 || p->v_stride_head % 16 || p->v_stride_token % 16 ||
      p->k_stride_head % 16 || p->k_stride_token % 16)
    return fail(TRI_ERR_INVALID_ARGUMENT, "tri_dense_compress: rows and strides must be multiples of 16 bytes");
  d.kv.k_layers = at<const void*>(ws, d.arg_key);
  int32_t* words = at<int32_t>(ws, d.arg_words);
  d.batch.seq_lens = words; d.batch.round_start = words + 1; d.batch.budgets = words + 2;
  d.sp.folded = at<float>(ws, d.folded); d.sp.omega = p->omega; d.sp.offsets = p->offsets;
  rc = check_layout(&d.kv, false);
  if (!rc) rc = check_batch(&d.batch, true);
  if (!rc) rc = check_score(&d.kv, &d.sp);
  if (!rc) rc = check_select(&d.sel);
  if (rc) return rc;
  tri::DenseLaunch l{};
  l.k = p->k; l.v = p->v;
  l.k_stride_head = p->k_stride_head; l.k_stride_token = p->k_stride_token;
  l.v_stride_head = p->v_stride_head; l.v_stride_token = p->v_stride_token;
  l.k_row_bytes = p->head_dim * 2; l.v_row_bytes = p->v_row_bytes;
  l.H = p->num_heads; l.T = p->num_tokens; l.D = p->head_dim; l.budget = p->budget; l.round_start = p->round_start;
  l.disable_mlr = p->disable_mlr; l.disable_trig = p->disable_trig;
  l.q_mean = p->q_mean_complex; l.q_abs = p->q_abs_mean; l.freq_scale = p->freq_scale_sq;
  l.out_k = p->out_k; l.out_v = p->out_v; l.out_keep = p->out_keep;
  l.folded = at<float>(ws, d.folded); l.arg_key = at<const void*>(ws, d.arg_key); l.arg_words = words;
  l.keep32 = at<int32_t>(ws, d.keep32);
  hipStream_t s = (hipStream_t)stream;
  // (NaN scores stay NaN, the largest of a row or, with the sign set, the smallest: torch's normalisation and
  // tri_topk_rows, which this call stands for, treat them so)
  if (p->aggregation == TRI_REDUCE_MEAN && tri::select_small_takes(p->num_tokens, 1) &&
      (int64_t)p->num_heads * tri::ceil_div(p->num_tokens, 128) <= kDenseSmallWorkgroups) {
    // Three launches: the scorer takes the call's arguments by value and folds the statistics itself.
    tri::SmallScore c{};
    c.k = p->k; c.round = p->round_start;
    c.q_mean = p->q_mean_complex; c.q_abs = p->q_abs_mean; c.freq_scale = p->freq_scale_sq;
    c.disable_mlr = p->disable_mlr; c.disable_trig = p->disable_trig;
    c.omega = p->omega; c.offsets = p->offsets; c.NO = p->num_offsets;
    c.raw = at<float>(ws, d.w.raw); c.raw_pitch = p->num_tokens;
    c.stride_token = d.kv.stride_token; c.stride_head = d.kv.stride_head;
    c.L = 1; c.A = p->num_heads; c.G = 1; c.Tmax = p->num_tokens; c.block_size = p->num_tokens;
    rc = launch_status(tri::launch_score_small(c, 1, p->num_heads, p->head_dim, p->kv_dtype, p->rope_style, s), "score_small");
    if (rc) return rc;
    tri::SmallSelect a{};
    a.raw = c.raw; a.raw_pitch = c.raw_pitch; a.keep = at<int32_t>(ws, d.keep32); a.keep_pitch = p->budget;
    a.L = 1; a.Hkv = p->num_heads; a.A = p->num_heads; a.G = 1; a.Tmax = p->num_tokens;
    a.normalize = d.sel.normalize; a.window_size = d.sel.window_size;
    a.group_reduce = TRI_REDUCE_MAX; a.layer_reduce = TRI_REDUCE_MEAN; a.pass_nan = 1;
    rc = launch_status(tri::launch_select_small(a, 1, s), "select_small");
    if (rc) return rc;
    return launch_status(tri::launch_dense_gather(l, s), "dense gather");
  }
  rc = launch_status(tri::launch_dense_prologue(l, s), "dense prologue");
  if (rc) return rc;
  rc = do_select_paged(&d.kv, &d.batch, &d.sp, &d.sel, nullptr, at<int32_t>(ws, d.keep32), ws, d.w, s, 1);
  if (rc) return rc;
  return launch_status(tri::launch_dense_gather(l, s), "dense gather");
}

int tri_compact_paged(const tri_kv_layout* kv, const tri_batch* batch, const int32_t* keep,
                      int32_t keep_per_layer, int32_t shared, void* stream) {
  tri::CompactLaunch a{};
  const int rc = fill_compact(kv, batch, keep, keep_per_layer, shared, a);
  if (rc) return rc;
  return launch_status(tri::launch_compact(a, (hipStream_t)stream), "compact");
}

uint64_t tri_compact_full_staging_bytes(const tri_kv_layout* kv, const tri_batch* batch) {
  if (check_layout(kv, true) || check_batch(batch, false)) return 0;
  // one layer: K and V of every head row of every logical slot of every sequence
  return (uint64_t)batch->num_seqs * 2 * kv->num_kv_heads * (uint64_t)batch->max_seq_len * kv->head_dim *
         elem_bytes(kv->kv_dtype);
}

int tri_compact_paged_full(const tri_kv_layout* kv, const tri_batch* batch, const int32_t* keep,
                           int32_t keep_per_layer, int32_t shared, void* staging, uint64_t staging_bytes,
                           void* stream) {
  tri::CompactLaunch a{};
  const int rc = fill_compact(kv, batch, keep, keep_per_layer, shared, a);
  if (rc) return rc;
  if (a.has_scales) return fail(TRI_ERR_UNSUPPORTED, "full-permutation compaction of fp8 caches is not built");
  if (!staging || !is_aligned(staging, 16)) return fail(TRI_ERR_WORKSPACE, "staging is NULL or unaligned");
  if (staging_bytes < tri_compact_full_staging_bytes(kv, batch))
    return fail(TRI_ERR_WORKSPACE, "staging has %llu bytes, %llu needed", (unsigned long long)staging_bytes,
                (unsigned long long)tri_compact_full_staging_bytes(kv, batch));
  a.staging = staging;
  return launch_status(tri::launch_compact_full(a, (hipStream_t)stream), "compact_full");
}

int tri_compress_step(const tri_kv_layout* kv, const tri_batch* batch, const tri_score_params* sp,
                      const tri_select_params* sel, int32_t* keep, void* workspace,
                      uint64_t workspace_bytes, void* stream) {
  int rc = check_layout(kv, true);
  if (rc) return rc;
  rc = check_batch(batch, true);
  if (rc) return rc;
  rc = check_score(kv, sp);
  if (rc) return rc;
  rc = check_select(sel);
  if (rc) return rc;
  if (!batch->round_start) return fail(TRI_ERR_INVALID_ARGUMENT, "round_start is NULL");
  if (!batch->block_table) return fail(TRI_ERR_INVALID_ARGUMENT, "tri_compress_step needs a block table");
  if (!keep) return fail(TRI_ERR_INVALID_ARGUMENT, "keep is NULL");
  const tri::Workspace w = plan(kv, batch, sp);
  rc = check_workspace(w, workspace, workspace_bytes);
  if (rc) return rc;
  hipStream_t s = (hipStream_t)stream;
  rc = do_select_paged(kv, batch, sp, sel, nullptr, keep, workspace, w, s);
  if (rc) return rc;
  tri::CompactLaunch c{};
  rc = fill_compact(kv, batch, keep, sel->layer_reduce < 0, sel->shared, c);
  if (rc) return rc;
  // A resident kernel whose bounded wait expired leaves meaningless keep lists and a raised
  // status word: the compaction kernels look at that word and then leave the cache alone.
  c.guard = at<uint32_t>(workspace, w.status);
  return launch_status(tri::launch_compact(c, s), "compact");
}

int tri_compress_step_static(const tri_kv_layout* kv, const tri_batch* batch, const tri_score_params* sp,
                             const tri_select_params* sel, int32_t* keep, const uint32_t** status_out,
                             void* stream) {
  int rc = check_layout(kv, true);
  if (rc) return rc;
  rc = check_batch(batch, true);
  if (rc) return rc;
  rc = check_score(kv, sp);
  if (rc) return rc;
  rc = check_select(sel);
  if (rc) return rc;
  if (!batch->round_start) return fail(TRI_ERR_INVALID_ARGUMENT, "round_start is NULL");
  if (!batch->block_table) return fail(TRI_ERR_INVALID_ARGUMENT, "tri_compress_step_static needs a block table");
  if (!keep) return fail(TRI_ERR_INVALID_ARGUMENT, "keep is NULL");
  // Always the score-then-select kernels, so the scratch is sized for them alone (a resident plan
  // would add its coefficient slabs and exchange words; the status word sits at the same offset).
  const tri::Workspace w = plan(kv, batch, sp, 0, false);
  if ((uint64_t)w.total > (uint64_t)TRI_STATIC_WORKSPACE_BYTES)
    return fail(TRI_ERR_WORKSPACE, "this step needs %lld bytes of scratch, the library's static array holds %llu; "
                "use tri_compress_step with a workspace of the caller's", (long long)w.total,
                (unsigned long long)TRI_STATIC_WORKSPACE_BYTES);
  void* ws = nullptr;
  rc = static_scratch(&ws);
  if (rc) return rc;
  if (status_out) *status_out = at<uint32_t>(ws, w.status);
  tri_select_params two_pass = *sel;
  two_pass.no_resident = 1;   // the resident path chains its launches with an event it creates
  hipStream_t s = (hipStream_t)stream;
  rc = do_select_paged(kv, batch, sp, &two_pass, nullptr, keep, ws, w, s);
  if (rc) return rc;
  tri::CompactLaunch c{};
  rc = fill_compact(kv, batch, keep, sel->layer_reduce < 0, sel->shared, c);
  if (rc) return rc;
  c.guard = at<uint32_t>(ws, w.status);
  c.no_side_stream = 1;
  return launch_status(tri::launch_compact(c, s), "compact");
}

uint64_t tri_qstats_workspace_bytes(int32_t num_heads, int32_t num_tokens, int32_t head_dim) {
  if (num_heads <= 0 || num_tokens <= 0 || (head_dim != 64 && head_dim != 128 && head_dim != 256)) return 0;
  return (uint64_t)tri::qstats_workspace_bytes(num_heads, num_tokens, head_dim);
}

int tri_qstats(const void* q_rot, int64_t stride_head, int64_t stride_token, const void* cos, const void* sin,
               int32_t num_heads, int32_t num_tokens, int32_t head_dim, int32_t dtype, int32_t rope_style,
               float scale, float* out_real, float* out_imag, float* out_abs, void* workspace,
               uint64_t workspace_bytes, void* stream) {
  if (!q_rot || !cos || !sin || !out_real || !out_imag || !out_abs)
    return fail(TRI_ERR_INVALID_ARGUMENT, "tri_qstats: NULL pointer");
  if (num_heads <= 0 || num_tokens <= 0) return fail(TRI_ERR_INVALID_ARGUMENT, "tri_qstats: bad sizes");
  if (head_dim != 64 && head_dim != 128 && head_dim != 256)
    return fail(TRI_ERR_UNSUPPORTED, "head_dim %d not in {64,128,256}", head_dim);
  if (dtype != TRI_KV_BF16 && dtype != TRI_KV_FP16)
    return fail(TRI_ERR_UNSUPPORTED, "tri_qstats: dtype %d (bf16 or fp16 query states)", dtype);
  if (rope_style != TRI_ROPE_HALF && rope_style != TRI_ROPE_INTERLEAVED)
    return fail(TRI_ERR_INVALID_ARGUMENT, "rope_style %d", rope_style);
  if (scale == 0.f) return fail(TRI_ERR_INVALID_ARGUMENT, "attention scaling factor must be non-zero");
  if (stride_token < head_dim || stride_token % 2 || stride_head % 2 || !is_aligned(q_rot, 4) || !is_aligned(cos, 4) ||
      !is_aligned(sin, 4))
    return fail(TRI_ERR_INVALID_ARGUMENT, "tri_qstats: rows must be 4-byte aligned and head_dim contiguous");
  const uint64_t need = tri_qstats_workspace_bytes(num_heads, num_tokens, head_dim);
  if (!workspace || workspace_bytes < need || !is_aligned(workspace, 16))
    return fail(TRI_ERR_WORKSPACE, "tri_qstats: workspace of %llu bytes needed", (unsigned long long)need);
  tri::QStatsLaunch q{};
  q.q_rot = q_rot; q.cos = cos; q.sin = sin;
  q.stride_head = stride_head; q.stride_token = stride_token;
  q.H = num_heads; q.T = num_tokens; q.D = head_dim; q.dtype = dtype; q.rope_style = rope_style;
  q.scale = scale;
  q.out_real = out_real; q.out_imag = out_imag; q.out_abs = out_abs;
  q.workspace = workspace;
  return launch_status(tri::launch_qstats(q, (hipStream_t)stream), "qstats");
}

}  // extern "C"
