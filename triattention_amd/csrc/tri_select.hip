// Score normalisation, guards, head / layer reduction and per-row top-k for gfx950.
//
//  finalize_stats_kernel : per-(sequence, layer, score head) mean and safe std from the
//                          scorer's per-tile sums (runtime/selector_hf.py:896-913).
//  combine_kernel        : z-score, +inf guards, reduce over the query heads of a KV
//                          head, reduce over layers (runtime/selector_hf.py:916-989).
//  group_stats_kernel    : the other order of operations (the reference's SGLang backend,
//                          sglang/scheduler_hooks.py:655-690): reduce over the query heads of
//                          a KV head first, then normalise per (layer, KV head) with
//                          core/utils.py:466-480 (torch mean / unbiased std).
//  topk_rows_kernel      : order-preserving radix select on the monotone integer
//                          image of the float (rows held in registers: one histogram pass
//                          over equal bins of the scores, then exact ranks inside one bin), then
//                          an ordered compaction that emits the kept token indices ascending;
//                          ties at the threshold keep the lowest index (replaces torch.topk + chunk merge +
//                          torch.sort, runtime/selector_hf.py:990-1025).
#include <type_traits>

#include "tri_common.h"

namespace tri {
namespace {

// fine: the sums come per quarter of a tile as (sum of A, sum of B, squares of A, squares of B) and are
// added here in the order in which a whole-tile workgroup adds those of its four waves.
__global__ void finalize_stats_kernel(const float* partial, const int32_t* seq_lens, int B, int L, int A,
                                      int num_tiles, int fine, int normalize, float* mustd) {
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= B * L * A) return;
  const int a = idx % A, bl = idx / A, b = bl / L;
  float mean = 0.f, sd = 1.f;
  if (normalize) {
    const int T = seq_lens[b];
    const int nt = ceil_div(T, kScoreTileTokens);
    double s = 0.0, q = 0.0;
    if (fine) {
      const int nq = ceil_div(T, kScoreFineTokens);
      const float4* p = reinterpret_cast<const float4*>(partial) + (int64_t)bl * num_tiles * A + a;
      for (int t = 0; t < nq; t += 4) {
        float4 x[4];
#pragma unroll
        for (int w = 0; w < 4; ++w) x[w] = p[(int64_t)min(t + w, nq - 1) * A];
        float t1 = 0.f, t2 = 0.f;
#pragma unroll
        for (int w = 0; w < 4; ++w)
          if (t + w < nq) {
            t1 += x[w].x;
            t2 += x[w].z;
            t1 += x[w].y;
            t2 += x[w].w;
          }
        s += (double)t1;
        q += (double)t2;
      }
    } else
      for (int t = 0; t < nt; t += 8) {              // eight tiles requested before the first is added
        const float2* p = reinterpret_cast<const float2*>(partial) + (int64_t)bl * num_tiles * A + a;
        float2 x[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) x[u] = p[(int64_t)min(t + u, nt - 1) * A];
#pragma unroll
        for (int u = 0; u < 8; ++u)
          if (t + u < nt) {
            s += (double)x[u].x;
            q += (double)x[u].y;
          }
      }
    // The reference's formula on fp32 sums (runtime/selector_hf.py:902-909).
    const float sum = (float)s, sumsq = (float)q, cnt = (float)T;
    mean = __fdiv_rn(sum, cnt);
    float var = 0.f;
    if (T > 1) var = __fdiv_rn(__fsub_rn(sumsq, __fmul_rn(cnt, __fmul_rn(mean, mean))), (float)(T - 1));
    var = fmaxf(var, 0.f);
    sd = __fsqrt_rn(var);
    if (sd < 1e-8f) sd = 1.f;
    if (normalize == 2) {
      // The research path's normalisation (methods/triattention.py:255-258): population standard
      // deviation, clamped from below at 1e-6; from the double-precision sums.
      const double m = s / (double)T;
      const double v = q / (double)T - m * m;
      mean = (float)m;
      sd = fmaxf((float)sqrt(v > 0.0 ? v : 0.0), 1e-6f);
    }
  }
  mustd[(int64_t)idx * 2] = mean;
  mustd[(int64_t)idx * 2 + 1] = sd;
}

// Reduce-first order: mean and std over the tokens of m[n] = reduce over the query heads of
// raw[n][h*G .. h*G+G), per (sequence, layer, KV head), with torch's definitions
// (core/utils.py:476-479: mean, unbiased std, std < 1e-8 -> 1).  Sums in double; one
// workgroup per (sequence, layer, KV head).  mustd[(b*L + l)*A*2 + h*2] = (mean, std).
// kPass (SelectLaunch::pass_nan): the one score of a KV head as it is.
template <bool kPass>
__global__ __launch_bounds__(256) void group_stats_kernel(const float* raw, int64_t stride_layer, int64_t stride_token,
                                                          int64_t stride_head, const int32_t* seq_lens, int L, int Hkv,
                                                          int A, int G, int group_reduce, int normalize, float* mustd) {
  __shared__ double red[256][2];
  const int h = blockIdx.x % Hkv;
  const int bl = blockIdx.x / Hkv, b = bl / L;
  float* out = mustd + ((int64_t)bl * A + h) * 2;
  if (!normalize) {
    if (threadIdx.x == 0) { out[0] = 0.f; out[1] = 1.f; }
    return;
  }
  const int T = seq_lens[b];
  const float* base = raw + (int64_t)bl * stride_layer + (int64_t)h * G * stride_head;
  double s = 0.0, q = 0.0;
  for (int n = threadIdx.x; n < T; n += 256) {
    const float* p = base + (int64_t)n * stride_token;
    float m;
    if constexpr (kPass) {
      m = p[0];
    } else {
      m = (group_reduce == TRI_REDUCE_MAX) ? -INFINITY : 0.f;
      for (int g = 0; g < G; ++g) {
        const float x = p[(int64_t)g * stride_head];
        m = (group_reduce == TRI_REDUCE_MAX) ? fmaxf(m, x) : __fadd_rn(m, x);
      }
      if (group_reduce != TRI_REDUCE_MAX) m = __fdiv_rn(m, (float)G);
    }
    s += (double)m;
    q += (double)m * (double)m;
  }
  red[threadIdx.x][0] = s;
  red[threadIdx.x][1] = q;
  __syncthreads();
  for (int off = 128; off > 0; off >>= 1) {
    if (threadIdx.x < off) {
      red[threadIdx.x][0] += red[threadIdx.x + off][0];
      red[threadIdx.x][1] += red[threadIdx.x + off][1];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    const double mean = red[0][0] / (double)T;
    double var = T > 1 ? (red[0][1] - (double)T * mean * mean) / (double)(T - 1) : 0.0;
    if (var < 0.0) var = 0.0;
    float sd = (float)sqrt(var);
    if (sd < 1e-8f) sd = 1.f;     // also a single token, where torch's unbiased std is undefined
    out[0] = (float)mean;
    out[1] = sd;
  }
}

// The same statistics for the usual layout -- four query heads per KV head, raw scores head-contiguous
// ([token][head], 16-byte aligned), a power-of-two number of KV heads -- in two launches that read whole
// token rows: a workgroup takes a chunk of 2048 tokens of one (sequence, layer) with thread = (token,
// KV head), so a wave reads 1 KB of consecutive memory per load where the kernel above reads 16 bytes
// of every 128-byte row eight times over (one request of 16384 tokens x 36 layers: 117 -> 30 us), and
// leaves the chunk's sums in double; the second launch adds the chunks in order.
// A few requests take chunks of down to 256 tokens: one of 2176 tokens x 36 layers is 72 workgroups of 2048
// tokens (27 us) or 324 of 256.
constexpr int kGroupStatsChunk = 2048, kGroupStatsChunkMin = 256;
__global__ __launch_bounds__(256) void group_stats_partial_kernel(const float* raw, int64_t stride_layer,
                                                                  int64_t stride_token, const int32_t* seq_lens, int L,
                                                                  int Hkv, int chunk, int chunks, int group_reduce,
                                                                  double* partial) {
  __shared__ double red[256][2];
  const int c = blockIdx.x, bl = blockIdx.y, b = bl / L;
  const int T = seq_lens[b];
  const int h = threadIdx.x % Hkv, tn = threadIdx.x / Hkv, tstep = 256 / Hkv;
  const int n_end = min(T, (c + 1) * chunk);
  const float* base = raw + (int64_t)bl * stride_layer + h * 4;
  double s = 0.0, q = 0.0;
#pragma unroll 4
  for (int n = c * chunk + tn; n < n_end; n += tstep) {
    const float4 x = *reinterpret_cast<const float4*>(base + (int64_t)n * stride_token);
    float m;
    if (group_reduce == TRI_REDUCE_MAX) m = fmaxf(fmaxf(x.x, x.y), fmaxf(x.z, x.w));
    else m = __fdiv_rn(__fadd_rn(__fadd_rn(__fadd_rn(x.x, x.y), x.z), x.w), 4.f);
    s += (double)m;
    q += (double)m * (double)m;
  }
  red[threadIdx.x][0] = s;
  red[threadIdx.x][1] = q;
  __syncthreads();
  for (int off = 128; off >= Hkv; off >>= 1) {       // threads `off` apart hold the same KV head
    if ((int)threadIdx.x < off) {
      red[threadIdx.x][0] += red[threadIdx.x + off][0];
      red[threadIdx.x][1] += red[threadIdx.x + off][1];
    }
    __syncthreads();
  }
  if ((int)threadIdx.x < Hkv) {
    double* out = partial + (((int64_t)bl * chunks + c) * Hkv + threadIdx.x) * 2;
    out[0] = red[threadIdx.x][0];
    out[1] = red[threadIdx.x][1];
  }
}

// One score per KV head (SelectLaunch::pass_nan), any number of heads up to 256, long rows: thread = (token, head), heads
// padded to a power of two.  group_stats_kernel walks a row in one workgroup, which for 8 rows of 400000 tokens made a whole
// dense call 1695 us (981 in chunks; torch's operators around the scorer 1305).
__global__ __launch_bounds__(256) void single_stats_partial_kernel(const float* raw, int64_t stride_layer,
                                                                   int64_t stride_token, const int32_t* seq_lens, int L,
                                                                   int Hkv, int Hpad, int chunk, int chunks, double* partial) {
  __shared__ double red[256][2];
  const int c = blockIdx.x, bl = blockIdx.y;
  const int T = seq_lens[bl / L];
  const int h = threadIdx.x % Hpad, tn = threadIdx.x / Hpad, tstep = 256 / Hpad;
  const int n_end = min(T, (c + 1) * chunk);
  const float* base = raw + (int64_t)bl * stride_layer + min(h, Hkv - 1);
  double s = 0.0, q = 0.0;
#pragma unroll 4
  for (int n = c * chunk + tn; n < n_end; n += tstep) {
    const float m = base[(int64_t)n * stride_token];
    s += (double)m;
    q += (double)m * (double)m;
  }
  red[threadIdx.x][0] = s;
  red[threadIdx.x][1] = q;
  __syncthreads();
  for (int off = 128; off >= Hpad; off >>= 1) {      // threads `off` apart hold the same KV head
    if ((int)threadIdx.x < off) {
      red[threadIdx.x][0] += red[threadIdx.x + off][0];
      red[threadIdx.x][1] += red[threadIdx.x + off][1];
    }
    __syncthreads();
  }
  if ((int)threadIdx.x < Hkv) {
    double* out = partial + (((int64_t)bl * chunks + c) * Hkv + threadIdx.x) * 2;
    out[0] = red[threadIdx.x][0];
    out[1] = red[threadIdx.x][1];
  }
}

__global__ void group_stats_finish_kernel(const double* partial, const int32_t* seq_lens, int BL, int L, int Hkv, int A,
                                          int chunk, int chunks, float* mustd) {
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= BL * Hkv) return;
  const int h = idx % Hkv, bl = idx / Hkv, b = bl / L;
  const int T = seq_lens[b];
  const int nc = ceil_div(T, chunk);
  double s = 0.0, q = 0.0;
#pragma unroll 8
  for (int c = 0; c < nc; ++c) {
    const double* p = partial + (((int64_t)bl * chunks + c) * Hkv + h) * 2;
    s += p[0];
    q += p[1];
  }
  const double mean = s / (double)T;
  double var = T > 1 ? (q - (double)T * mean * mean) / (double)(T - 1) : 0.0;
  if (var < 0.0) var = 0.0;
  float sd = (float)sqrt(var);
  if (sd < 1e-8f) sd = 1.f;
  float* out = mustd + ((int64_t)bl * A + h) * 2;
  out[0] = (float)mean;
  out[1] = sd;
}

// From where on the row of a KV head's one score takes chunks (single_stats_partial_kernel) instead of one workgroup: a dense
// call of 8 heads x 16384 tokens 68 -> 51 us, x 49152 224 -> 160.  Short rows are one launch less in one workgroup.
constexpr int kSingleStatsTokens = 16384;

struct CombineArgs {
  const float* raw;
  const float* mustd;
  const int32_t* seq_lens;
  const int32_t* prefill_lens;
  float* fin;
  int64_t raw_stride_layer, raw_stride_token, raw_stride_head;
  int B, L, Hkv, A, G, Tmax;
  int window_size, protect_prefill, group_reduce, layer_reduce, shared, pass_nan;
  int rows_per_seq;   // rows per (sequence[, layer]): shared ? 1 : Hkv
  int tokens_per_wg;  // threads / rows_per_seq
};

// z-score of one raw value with the reference's operation order: (x - mean) / std.
__device__ __forceinline__ float zscore(float x, float mean, float sd) {
  return __fdiv_rn(__fsub_rn(x, mean), sd);
}

// The same where a NaN is a score like another (SelectLaunch::pass_nan); its sign says at which end of the order
// it lies, and is kept: that of the score itself, else of the row's mean (the subtraction above would turn it).
// A row with infinite scores and no NaN is NaN throughout too, by inf - inf, with a sign that in torch's reduction
// depends on where the score stood; here it is negative, below the guarded tokens.
__device__ __forceinline__ float passed_zscore(float x, float mean, float sd) {
  const float z = zscore(x, mean, sd);
  if (!__builtin_isnan(z)) return z;
  return __builtin_isnan(x) ? x : (__builtin_isnan(mean) ? mean : __uint_as_float(0xffc00000u));
}

// One thread per (token, output row).  Grid: (token tiles, layers or 1, B).
// NV > 0: groups of 4 * NV query heads (4 or 8), raw scores head-contiguous and 16-byte aligned, read as
// NV 16-byte loads per layer; NV = 0: any layout, one score at a time.
// U (NV > 0): layers a thread requests before it uses the first; GF: group_first, a constant there because a
// branch between the loads made every one of them wait for the one before.
template <int NV, int U, bool GF>
__global__ __launch_bounds__(256) void combine_kernel(CombineArgs a) {
  extern __shared__ float tile[];  // [rows_per_seq][tokens_per_wg]
  const int b = blockIdx.z;
  const int T = a.seq_lens[b];
  const int n0 = blockIdx.x * a.tokens_per_wg;
  if (n0 >= T) return;
  const int R = a.rows_per_seq;
  const int tn = threadIdx.x / R, r = threadIdx.x % R;
  const int n = n0 + tn;
  const bool per_layer = a.layer_reduce < 0;
  const int l_begin = per_layer ? blockIdx.y : 0;
  const int l_end = per_layer ? blockIdx.y + 1 : a.L;

  if (tn < a.tokens_per_wg && n < T) {
    bool guard = false;
    if (a.window_size > 0) guard = n >= T - min(a.window_size, T);
    if (a.protect_prefill && a.prefill_lens) guard = guard || (n < a.prefill_lens[b]);
    const int h_begin = a.shared ? 0 : r;
    const int h_end = a.shared ? a.Hkv : r + 1;
    float acc = 0.f;
    if (NV > 0 && !a.shared) {
      // Default shapes: one KV head per thread, its query heads in NV 16-byte loads; several layers in
      // flight per thread.
      constexpr int NVV = NV > 0 ? NV : 1;
      constexpr int GQ = 4 * NVV;                  // query heads per KV head
      const float* raw0 = a.raw + (int64_t)b * a.L * a.raw_stride_layer + (int64_t)n * a.raw_stride_token + r * GQ;
      // Reduce-first order (group_first): the statistics are those of the KV head's reduced score and
      // sit in entry r of the layer's table; they arrive in m[0].x / m[0].y.
      const float* ms0 = a.mustd + ((int64_t)b * a.L * a.A + (GF ? r : r * GQ)) * 2;
      constexpr int NM = GF ? 1 : 2 * NVV;
      struct LayerIn { float4 x[NVV]; float4 m[NM]; };
      auto load_layer = [&](int l, LayerIn& in) __attribute__((always_inline)) {
        const float* rl = raw0 + (int64_t)l * a.raw_stride_layer;
        const float* ms = ms0 + (int64_t)l * a.A * 2;
#pragma unroll
        for (int i = 0; i < NVV; ++i) in.x[i] = *reinterpret_cast<const float4*>(rl + 4 * i);
        if constexpr (GF) {
          const float2 m = *reinterpret_cast<const float2*>(ms);
          in.m[0] = float4{m.x, m.y, 0.f, 0.f};
        } else {
          // mustd is [head][mean, std]: m[2 i] = (mean, std) of query heads 4 i and 4 i + 1, m[2 i + 1] of the next two.
#pragma unroll
          for (int i = 0; i < NM; ++i) in.m[i] = *reinterpret_cast<const float4*>(ms + 4 * i);
        }
      };
      auto layer_value = [&](const LayerIn& in) __attribute__((always_inline)) {
        float xs[GQ];
#pragma unroll
        for (int i = 0; i < NVV; ++i) { xs[4 * i] = in.x[i].x; xs[4 * i + 1] = in.x[i].y; xs[4 * i + 2] = in.x[i].z; xs[4 * i + 3] = in.x[i].w; }
        float v;
        if constexpr (GF) {
          // (the order of the scalar path below: query heads one after the other)
          float m = xs[0];
#pragma unroll
          for (int q = 1; q < GQ; ++q) m = (a.group_reduce == TRI_REDUCE_MAX) ? fmaxf(m, xs[q]) : __fadd_rn(m, xs[q]);
          if (a.group_reduce != TRI_REDUCE_MAX) m = __fdiv_rn(m, (float)GQ);
          v = zscore(m, in.m[0].x, in.m[0].y);
        } else {
          float z[GQ];
#pragma unroll
          for (int i = 0; i < NM; ++i) {
            z[2 * i] = zscore(xs[2 * i], in.m[i].x, in.m[i].y);
            z[2 * i + 1] = zscore(xs[2 * i + 1], in.m[i].z, in.m[i].w);
          }
          v = z[0];
#pragma unroll
          for (int q = 1; q < GQ; ++q) v = (a.group_reduce == TRI_REDUCE_MAX) ? fmaxf(v, z[q]) : __fadd_rn(v, z[q]);
          if (a.group_reduce != TRI_REDUCE_MAX) v = __fdiv_rn(v, (float)GQ);
        }
        return guard ? INFINITY : v;
      };
      for (int l = l_begin; l < l_end; l += U) {
        LayerIn in[U];
#pragma unroll
        for (int u = 0; u < U; ++u) load_layer(min(l + u, l_end - 1), in[u]);
#pragma unroll
        for (int u = 0; u < U; ++u) {
          if (l + u >= l_end) continue;
          const float v = layer_value(in[u]);
          if (l + u == l_begin) acc = v;
          else acc = (a.layer_reduce == TRI_REDUCE_MAX) ? fmaxf(acc, v) : __fadd_rn(acc, v);
        }
      }
    } else {
      for (int l = l_begin; l < l_end; ++l) {
        const float* raw_l = a.raw + (int64_t)(b * a.L + l) * a.raw_stride_layer + (int64_t)n * a.raw_stride_token;
        const float* ms = a.mustd + (int64_t)(b * a.L + l) * a.A * 2;
        float v = -INFINITY;
        for (int h = h_begin; h < h_end; ++h) {
          if (a.pass_nan) {      // (the maxima below drop a NaN)
            v = passed_zscore(raw_l[(int64_t)h * a.raw_stride_head], ms[h * 2], ms[h * 2 + 1]);
            continue;
          }
          float gv = (a.group_reduce == TRI_REDUCE_MAX) ? -INFINITY : 0.f;
          for (int q = 0; q < a.G; ++q) {
            const int ah = h * a.G + q;
            const float x = raw_l[(int64_t)ah * a.raw_stride_head];
            const float z = GF ? x : zscore(x, ms[ah * 2], ms[ah * 2 + 1]);
            gv = (a.group_reduce == TRI_REDUCE_MAX) ? fmaxf(gv, z) : __fadd_rn(gv, z);
          }
          if (a.group_reduce != TRI_REDUCE_MAX) gv = __fdiv_rn(gv, (float)a.G);
          if (GF) gv = zscore(gv, ms[h * 2], ms[h * 2 + 1]);
          v = fmaxf(v, gv);
        }
        if (guard) v = INFINITY;
        if (l == l_begin) acc = v;
        else acc = (a.layer_reduce == TRI_REDUCE_MAX) ? fmaxf(acc, v) : __fadd_rn(acc, v);
      }
    }
    if (a.layer_reduce == TRI_REDUCE_MEAN) acc = __fdiv_rn(acc, (float)a.L);
    tile[r * a.tokens_per_wg + tn] = acc;
  }
  __syncthreads();
  // Coalesced write of the [rows][tokens] tile.
  const int nvalid = min(a.tokens_per_wg, T - n0);
  const int64_t row0 = per_layer ? ((int64_t)(b * a.L + blockIdx.y) * R) : ((int64_t)b * R);
  for (int i = threadIdx.x; i < R * a.tokens_per_wg; i += (int)blockDim.x) {
    const int rr = i / a.tokens_per_wg, tt = i % a.tokens_per_wg;
    if (tt < nvalid) a.fin[(row0 + rr) * a.Tmax + n0 + tt] = tile[i];
  }
}

// Monotone map float -> uint32: a < b  <=>  key(a) < key(b).
__device__ __forceinline__ uint32_t float_key(float f) {
  const uint32_t u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

constexpr int kTopkThreads = 1024;

// One workgroup per row.
__global__ __launch_bounds__(kTopkThreads) void topk_rows_kernel(const float* scores, int64_t row_pitch,
                                                                const int32_t* row_lens,
                                                                const int32_t* row_ks, int rows_per_entry,
                                                                int32_t* keep, int keep_pitch, int max_len) {
  __shared__ uint32_t hist[256];
  __shared__ uint32_t scan[256];
  __shared__ uint32_t sh_prefix, sh_remaining;
  __shared__ uint32_t cnt_gt[kTopkThreads];
  __shared__ uint32_t cnt_eq[kTopkThreads];

  const int row = blockIdx.x;
  const int entry = row / rows_per_entry;
  // Lengths and budgets live on the device; the host sized rows for max_len scores and
  // keep_pitch indices, and neither is ever exceeded whatever the device arrays say.
  const int T = min(row_lens[entry], max_len);
  int k = min(row_ks[entry], keep_pitch);
  if (k > T) k = T;
  if (k <= 0 || T <= 0) return;
  const float* x = scores + (int64_t)row * row_pitch;
  int32_t* out = keep + (int64_t)row * keep_pitch;
  const int tid = threadIdx.x;

  if (k >= T) {
    for (int i = tid; i < T; i += kTopkThreads) out[i] = i;
    return;
  }

  // ---- radix select of the k-th largest key, 8 bits per pass from the top.
  uint32_t prefix = 0, mask = 0, remaining = (uint32_t)k;
  for (int shift = 24; shift >= 0; shift -= 8) {
    if (tid < 256) hist[tid] = 0;
    __syncthreads();
    for (int i = tid; i < T; i += kTopkThreads) {
      const uint32_t key = float_key(x[i]);
      if ((key & mask) == prefix) atomicAdd(&hist[(key >> shift) & 255u], 1u);
    }
    __syncthreads();
    // suffix[d] = number of candidates with digit >= d (Hillis-Steele over 256 bins).
    if (tid < 256) scan[tid] = hist[tid];
    __syncthreads();
    for (int off = 1; off < 256; off <<= 1) {
      uint32_t v = 0;
      if (tid < 256 && tid + off < 256) v = scan[tid + off];
      __syncthreads();
      if (tid < 256) scan[tid] += v;
      __syncthreads();
    }
    if (tid < 256) {
      const uint32_t ge = scan[tid];
      const uint32_t gt = (tid < 255) ? scan[tid + 1] : 0u;
      if (gt < remaining && remaining <= ge) {   // exactly one digit satisfies this
        sh_prefix = prefix | ((uint32_t)tid << shift);
        sh_remaining = remaining - gt;
      }
    }
    __syncthreads();
    prefix = sh_prefix;
    remaining = sh_remaining;
    mask |= 255u << shift;
    __syncthreads();
  }
  const uint32_t thr = prefix;        // key of the k-th largest element
  const uint32_t need_eq = remaining; // how many elements equal to it are kept (lowest index first)

  // ---- ordered compaction: every thread owns a contiguous chunk of the row.
  const int chunk = ceil_div(T, kTopkThreads);
  const int c0 = min(tid * chunk, T), c1 = min(c0 + chunk, T);
  uint32_t g = 0, e = 0;
  for (int i = c0; i < c1; ++i) {
    const uint32_t key = float_key(x[i]);
    g += key > thr;
    e += key == thr;
  }
  cnt_gt[tid] = g;
  cnt_eq[tid] = e;
  __syncthreads();
  // Exclusive scan of both counters over threads (Hillis-Steele, inclusive then shift).
  for (int off = 1; off < kTopkThreads; off <<= 1) {
    uint32_t vg = 0, ve = 0;
    if (tid >= off) { vg = cnt_gt[tid - off]; ve = cnt_eq[tid - off]; }
    __syncthreads();
    cnt_gt[tid] += vg;
    cnt_eq[tid] += ve;
    __syncthreads();
  }
  uint32_t gt_before = cnt_gt[tid] - g;
  uint32_t eq_before = cnt_eq[tid] - e;
  uint32_t pos = gt_before + min(eq_before, need_eq);
  for (int i = c0; i < c1; ++i) {
    const uint32_t key = float_key(x[i]);
    if (key > thr) {
      out[pos++] = i;
    } else if (key == thr) {
      if (eq_before < need_eq) out[pos++] = i;
      ++eq_before;
    }
  }
}

// Reductions over the 16 lanes of a row and over the wave (every lane gets the result): rotations inside a row, then the
// four rows' results as scalars.
template <int N>
__device__ __forceinline__ uint32_t row_rotate(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x120 + N, 0xf, 0xf, true);
}
template <typename Op>
__device__ __forceinline__ uint32_t row_reduce(uint32_t v, Op op) {
  v = op(v, row_rotate<8>(v));
  v = op(v, row_rotate<4>(v));
  v = op(v, row_rotate<2>(v));
  return op(v, row_rotate<1>(v));
}
template <typename Op>
__device__ __forceinline__ uint32_t wave_reduce(uint32_t v, Op op) {
  v = row_reduce(v, op);
  const uint32_t a = (uint32_t)__builtin_amdgcn_readlane((int)v, 0), b = (uint32_t)__builtin_amdgcn_readlane((int)v, 16);
  const uint32_t c = (uint32_t)__builtin_amdgcn_readlane((int)v, 32), d = (uint32_t)__builtin_amdgcn_readlane((int)v, 48);
  return op(op(a, b), op(c, d));
}
__device__ __forceinline__ uint32_t scalar_of(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }
struct MinOp { __device__ __forceinline__ uint32_t operator()(uint32_t a, uint32_t b) const { return min(a, b); } };
struct MaxOp { __device__ __forceinline__ uint32_t operator()(uint32_t a, uint32_t b) const { return max(a, b); } };
struct SumOp { __device__ __forceinline__ uint32_t operator()(uint32_t a, uint32_t b) const { return a + b; } };
// Inverse of float_key.
__device__ __forceinline__ float key_float(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}
constexpr uint32_t kKeyInf = 0xff800000u;        // float_key(+inf); NaNs of positive sign lie above
constexpr uint32_t kKeyFiniteMin = 0x00800000u;  // float_key(-FLT_MAX); -inf and NaNs of negative sign lie below
constexpr int kTopkBins = 2048;
constexpr int kTopkCand = 128;                   // candidates ranked by counting, one thread each (their square is the time)

// The same selection for rows of at most VPT * 1024 elements: the row is read once into
// registers.  A wave owns 64 * VPT consecutive elements, 64 at a time: loads are whole lines, and the
// ascending emission counts with ballots (a lane's place is the number of kept lanes below it) and
// writes runs of consecutive indices.  (With a thread owning VPT consecutive elements every store of the
// emission went to 64 different lines.)
//
// A few rows on a few CUs: the time is the chain of barriers and LDS round trips, not the
// bytes.  The threshold is found in one histogram pass: the finite scores are
// cut into 2000 bins of equal width between their minimum and maximum ((x - lo) * scale,
// rounded, is monotone in x, so the bins are ordered as the scores are), a scan over all
// threads finds the bin of the k-th largest, and the few scores of that bin are ranked
// against each other, one thread per candidate, on their exact keys.  Guarded tokens (+inf)
// are counted apart, they would stretch the bins.  A bin of more than 128 scores (rows with many equal ones) and rows whose
// range lies far beyond where most scores are (outliers, long tails) are cut by their keys, whose range shrinks by 2^11 a
// pass: a key is a logarithm of the score, so one or two passes take care of those, and equal scores end it.
// Seven barriers, five more a further pass; with radix passes of 8 bits alone it was thirteen, around scans by a single wave.
// us, scores of one size / with an outlier at 1e6, against 27 and 53 of radix passes for the longer ones: 8 rows of 4096
// 6.6 / 6.2 (12.5), 288 rows of 2176 7.7 / 9.2 (15.8: two workgroups a CU, 64 registers a thread), 128 rows of 16384
// 11.3 / 13.5, 8 rows of 32768 19.4 / 23.2 (there the instructions of one CU bound it).  Ranking up to 1024
// candidates took 30 us at 750, radix passes behind the first histogram 57 and 106 with an outlier.
// Key 0 is "no element" (the one NaN pattern whose key it would be shares the next key), so the selection
// never asks for an element's place in the row again.
__device__ __forceinline__ uint32_t row_key(float f) { return max(float_key(f), 1u); }

template <int VPT>
__device__ __forceinline__ void emit_topk(const uint32_t (&key)[VPT], int T, int k, int32_t* out) {
  constexpr int kWaves = kTopkThreads / 64;
  __shared__ uint32_t hist[kTopkBins];
  __shared__ __align__(16) uint32_t cand[kTopkCand];
  __shared__ uint32_t wave_lo[kWaves], wave_hi[kWaves], wave_tot[kWaves];
  __shared__ uint32_t sh_high, sh_ncand, sh_prefix, sh_remaining, sh_count;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int e0 = wave * (64 * VPT) + lane;        // element i of this thread: e0 + 64 * i

  // ---- range of the finite scores, number of scores at or above +inf.
  uint32_t lo_key = 0xffffffffu, hi_key = 0u;
  int high = 0;
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const bool fin = key[i] - kKeyFiniteMin < kKeyInf - kKeyFiniteMin;
    lo_key = min(lo_key, fin ? key[i] : 0xffffffffu);
    hi_key = max(hi_key, fin ? key[i] : 0u);
    high += __popcll(__ballot(key[i] >= kKeyInf));
  }
  lo_key = wave_reduce(lo_key, MinOp());
  hi_key = wave_reduce(hi_key, MaxOp());
  if (lane == 0) {
    wave_lo[wave] = lo_key;
    wave_hi[wave] = hi_key;
    wave_tot[wave] = (uint32_t)high;
  }
  auto clear_hist = [&]() __attribute__((always_inline)) {
    for (int i = tid; i < kTopkBins; i += kTopkThreads) hist[i] = 0;
  };
  clear_hist();
  if (tid == 0) sh_ncand = 0;
  __syncthreads();
  static_assert(kWaves == 16, "a lane of a row reads what one wave left");
  uint32_t above;                                // scores at or above +inf in the row
  uint32_t core_lo, core_hi;                     // a range that every full wave's finite scores reach beyond
  {
    const int w = lane & 15;
    const uint32_t wl = wave_lo[w], wh = wave_hi[w];
    const bool full = (w + 1) * (64 * VPT) <= T && wl <= wh;
    above = scalar_of(row_reduce(wave_tot[w], SumOp()));
    lo_key = scalar_of(row_reduce(wl, MinOp()));
    hi_key = scalar_of(row_reduce(wh, MaxOp()));
    core_lo = scalar_of(row_reduce(full ? wl : 0u, MaxOp()));
    core_hi = scalar_of(row_reduce(full ? wh : 0xffffffffu, MinOp()));
  }
  // A row without a finite score has lo_key > hi_key: everything else then falls into bin 0.
  const float lo = lo_key <= hi_key ? key_float(lo_key) : 0.f;
  const float width = lo_key <= hi_key ? __fsub_rn(key_float(hi_key), lo) : 0.f;
  // (A width beyond the largest float is +inf and makes the scale 0: a score whose distance from lo is still a
  // number falls into bin 0; the largest ones, whose distance is +inf too, give inf * 0 = NaN, which the fminf
  // below drops for the last bin.  Two bins, in order.)
  // (2000 of the 2048 bins: scores on a grid would otherwise fall into bins a power of two apart, counters of one bank)
  const float scale = width > 0.f ? fminf(__fdiv_rn(2000.f, width), 3.0e38f) : 0.f;
  auto bin_of = [&](uint32_t kk) __attribute__((always_inline)) {
    const float t = __fmul_rn(__fsub_rn(key_float(kk), lo), scale);
    const int b = kk < kKeyFiniteMin ? 0 : (int)fminf(t, (float)(kTopkBins - 1));
    return (uint32_t)b;
  };
  // A range far beyond what every wave's scores span (outliers, long tails) would leave most scores in a few bins, and the
  // lanes of a wave adding to one counter one after the other.  Those rows are cut by their keys from the start.  (Scores
  // of one size span 1.5 times the core.)
  const bool skewed = core_lo <= core_hi && core_lo != 0u && !(width <= 16.f * __fsub_rn(key_float(core_hi), key_float(core_lo)));

  // ---- which scores the k-th largest is among, and how many of those are kept.
  uint32_t remaining = (uint32_t)k, count = 0;
  // The bin of the finished histogram that holds the `remaining`-th largest; remaining and count become those of
  // the bin.  Everyone is past the barrier behind the histogram.
  auto find_bin = [&]() __attribute__((always_inline)) {
    constexpr int BPT = kTopkBins / kTopkThreads;   // bins per thread
    uint32_t h[BPT], own = 0;
#pragma unroll
    for (int j = 0; j < BPT; ++j) { h[j] = hist[tid * BPT + j]; own += h[j]; }
    uint32_t suffix = own;                         // scores in the bins of lanes >= this one
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const uint32_t v = __shfl_down(suffix, off);
      if (lane + off < 64) suffix += v;
    }
    if (lane == 0) wave_lo[wave] = suffix;         // (read by everyone before the barrier above)
    __syncthreads();
    uint32_t gt = suffix - own + row_reduce((lane & 15) > wave ? wave_lo[lane & 15] : 0u, SumOp());
#pragma unroll
    for (int j = BPT - 1; j >= 0; --j) {
      const uint32_t ge = gt + h[j];
      if (gt < remaining && remaining <= ge) {     // exactly one bin satisfies this
        sh_prefix = (uint32_t)(tid * BPT + j);
        sh_remaining = remaining - gt;
        sh_count = h[j];
      }
      gt = ge;
    }
    __syncthreads();
    remaining = sh_remaining;
    count = sh_count;
    return sh_prefix;
  };
  // ---- cuts into 2048 bins until few candidates are left or all are equal: the first by score (of a skewed row by the
  // leading bits of the key), the next ones by the range of the keys that are left.
  uint32_t cmask = 0;                            // bit i: element i is a candidate
  if (above >= (uint32_t)k) {                    // (the same for the whole workgroup)
    count = above;
#pragma unroll
    for (int i = 0; i < VPT; ++i) cmask |= (uint32_t)(key[i] >= kKeyInf) << i;
  } else if (skewed) {
    remaining -= above;
#pragma unroll
    for (int i = 0; i < VPT; ++i)
      if (key[i] - 1u < kKeyInf - 1u) atomicAdd(&hist[key[i] >> 21], 1u);
    __syncthreads();
    const uint32_t bin = find_bin();
#pragma unroll
    for (int i = 0; i < VPT; ++i) cmask |= (uint32_t)(key[i] - 1u < kKeyInf - 1u && key[i] >> 21 == bin) << i;
  } else {
    remaining -= above;
    uint32_t bins[VPT / 2];                      // two per register; 0xffff: none
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
      const bool ok = key[i] - 1u < kKeyInf - 1u;
      const uint32_t b = ok ? bin_of(key[i]) : 0xffffu;
      if (ok) atomicAdd(&hist[b], 1u);
      bins[i / 2] = (i & 1) ? bins[i / 2] | (b << 16) : b;
    }
    __syncthreads();
    const uint32_t bin = find_bin();
#pragma unroll
    for (int i = 0; i < VPT; ++i)
      cmask |= (uint32_t)(((bins[i / 2] >> (16 * (i & 1))) & 0xffffu) == bin) << i;
  }
  uint32_t thr = 0, need_eq = 0;                 // key of the k-th largest, how many equal to it are kept (lowest index first)
  bool equal = false;
  while (count > (uint32_t)kTopkCand) {
    uint32_t lo_c = 0xffffffffu, hi_c = 0u;
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
      const bool part = (cmask >> i) & 1u;
      lo_c = min(lo_c, part ? key[i] : 0xffffffffu);
      hi_c = max(hi_c, part ? key[i] : 0u);
    }
    lo_c = wave_reduce(lo_c, MinOp());
    hi_c = wave_reduce(hi_c, MaxOp());
    __syncthreads();                             // (wave_lo and hist are read by everyone before they are written again)
    if (lane == 0) { wave_lo[wave] = lo_c; wave_hi[wave] = hi_c; }
    clear_hist();
    __syncthreads();
    lo_c = scalar_of(row_reduce(wave_lo[lane & 15], MinOp()));
    hi_c = scalar_of(row_reduce(wave_hi[lane & 15], MaxOp()));
    if (lo_c == hi_c) {
      equal = true;
      thr = lo_c;
      need_eq = remaining;
      break;
    }
    const int shift = max(32 - __clz((int)(hi_c - lo_c)) - 11, 0);     // 0: a bin is a key
#pragma unroll
    for (int i = 0; i < VPT; ++i)
      if ((cmask >> i) & 1u) atomicAdd(&hist[(key[i] - lo_c) >> shift], 1u);
    __syncthreads();                             // (wave_lo is free again as well)
    const uint32_t bin = find_bin();
    asm volatile("" : "+v"(lo_c));
#pragma unroll
    for (int i = 0; i < VPT; ++i) cmask &= ~((uint32_t)((key[i] - lo_c) >> shift != bin) << i);
  }

  // ---- the k-th largest among the candidates.
  if (!equal) {
#pragma unroll
    for (int i = 0; i < VPT; ++i)
      if ((cmask >> i) & 1u) cand[atomicAdd(&sh_ncand, 1u)] = key[i];
    __syncthreads();
    if ((uint32_t)tid < count) {
      const uint32_t mine = cand[tid];
      uint32_t gt = 0, ge = 0;
      uint32_t i = 0;
      for (; i + 4 <= count; i += 4) {
        const uint4 c = *reinterpret_cast<const uint4*>(&cand[i]);
        gt += (c.x > mine) + (c.y > mine) + (c.z > mine) + (c.w > mine);
        ge += (c.x >= mine) + (c.y >= mine) + (c.z >= mine) + (c.w >= mine);
      }
      for (; i < count; ++i) { gt += cand[i] > mine; ge += cand[i] >= mine; }
      if (gt < remaining && remaining <= ge) {     // candidates with this very key, and only they
        sh_high = mine;
        sh_count = remaining - gt;
      }
    }
    __syncthreads();
    thr = sh_high;
    need_eq = sh_count;
  }

  // ---- ordered compaction.  Counts of (greater, equal) of the wave packed as (g << 16) | e: a row has
  // at most 32768 elements.  Elements beyond the row hold key 0, which the threshold never is.
  uint32_t mine = 0;
#pragma unroll
  for (int i = 0; i < VPT; ++i)
    mine += ((uint32_t)__popcll(__ballot(key[i] > thr)) << 16) + (uint32_t)__popcll(__ballot(key[i] == thr));
  if (lane == 0) wave_tot[wave] = mine;
  __syncthreads();
  const uint32_t before = scalar_of(row_reduce((lane & 15) < wave ? wave_tot[lane & 15] : 0u, SumOp()));
  uint32_t eq_before = before & 0xffffu;
  uint32_t pos = (before >> 16) + min(eq_before, need_eq);
  auto lanes_below = [](unsigned long long m) __attribute__((always_inline)) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
  };
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    unsigned long long km = __ballot(key[i] > thr);
    bool kept = key[i] > thr;
    const unsigned long long em = __ballot(key[i] == thr);
    if (em != 0) {                               // (wave-uniform, rarely taken)
      const bool eq = key[i] == thr && eq_before + lanes_below(em) < need_eq;
      kept = kept || eq;
      km |= __ballot(eq);
      eq_before += (uint32_t)__popcll(em);
    }
    if (kept) out[pos + lanes_below(km)] = e0 + 64 * i;
    pos += (uint32_t)__popcll(km);
  }
}

template <int VPT>
__global__ __launch_bounds__(kTopkThreads, VPT <= 4 ? 8 : 4) void topk_rows_reg_kernel(const float* scores, int64_t row_pitch,
                                                                    const int32_t* row_lens,
                                                                    const int32_t* row_ks, int rows_per_entry,
                                                                    int32_t* keep, int keep_pitch, int max_len,
                                                                    int groups, int64_t group_stride, int group_max) {
  const int row = blockIdx.x;
  const int entry = row / rows_per_entry;
  // Lengths and budgets live on the device; the host sized rows for max_len scores and
  // keep_pitch indices, and neither is ever exceeded whatever the device arrays say.
  const int T = min(row_lens[entry], max_len);
  int k = min(row_ks[entry], keep_pitch);
  if (k > T) k = T;
  if (k <= 0 || T <= 0) return;
  const float* x = scores + (int64_t)row * row_pitch;
  int32_t* out = keep + (int64_t)row * keep_pitch;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;

  if (k >= T) {
    for (int i = tid; i < T; i += kTopkThreads) out[i] = i;
    return;
  }

  const int e0 = wave * (64 * VPT) + lane;        // element i of this thread: e0 + 64 * i
  const int nvalid = min(max((T - e0 + 63) / 64, 0), VPT);
  uint32_t key[VPT];
  if (groups > 1) {
    // The row arrives as `groups` partial rows `group_stride` floats apart (a resident launch cut
    // by layers): they are added (or maximised) in group order, exactly as
    // fused_layer_reduce_kernel does; the division by the layer count that turns the sum into a
    // mean does not change the order of the scores and is left out.
    // The rows of several groups are requested before the first is added (a thread's loads of one
    // group after the other, each waited for, made 36 groups of a single request take 30 us); the last
    // round repeats the last group where there is none left and leaves it out of the sum.
    constexpr int U = VPT >= 32 ? 1 : (VPT >= 16 ? 3 : (VPT >= 8 ? 6 : 12));   // groups in flight per round
    auto load_row = [&](int g, float (&y)[VPT]) __attribute__((always_inline)) {
      const float* p = x + (int64_t)g * group_stride;
#pragma unroll
      for (int i = 0; i < VPT; ++i) y[i] = p[min(e0 + 64 * i, T - 1)];
    };
    float v[VPT];
    load_row(0, v);
    for (int g = 1; g < groups; g += U) {
      float y[U][VPT];
#pragma unroll
      for (int u = 0; u < U; ++u) load_row(min(g + u, groups - 1), y[u]);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (g + u >= groups) continue;
#pragma unroll
        for (int i = 0; i < VPT; ++i) v[i] = group_max ? fmaxf(v[i], y[u][i]) : __fadd_rn(v[i], y[u][i]);
      }
    }
#pragma unroll
    for (int i = 0; i < VPT; ++i) key[i] = i < nvalid ? row_key(v[i]) : 0u;
  } else {
#pragma unroll
    for (int i = 0; i < VPT; ++i) key[i] = __float_as_uint(x[min(e0 + 64 * i, T - 1)]);
#pragma unroll
    for (int i = 0; i < VPT; ++i) key[i] = i < nvalid ? row_key(__uint_as_float(key[i])) : 0u;
  }
  emit_topk<VPT>(key, T, k, out);
}

// ---- a small launch: statistics, reduction and top-k of the raw scores of one (sequence, KV head) in one workgroup.
// Sum over the 16 lanes of a row (every lane gets it).
template <int N>
__device__ __forceinline__ double row_rotate_f64(double v) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  return __builtin_bit_cast(double, ((uint64_t)row_rotate<N>((uint32_t)(u >> 32)) << 32) | row_rotate<N>((uint32_t)u));
}
__device__ __forceinline__ double row_sum_f64(double v) {
  v += row_rotate_f64<8>(v);
  v += row_rotate_f64<4>(v);
  v += row_rotate_f64<2>(v);
  return v + row_rotate_f64<1>(v);
}
__device__ __forceinline__ double lane_f64(double v, int lane) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  return __builtin_bit_cast(double, ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(u >> 32), lane) << 32) |
                                        (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)u, lane));
}

__device__ __forceinline__ float row_sum_f32(float v) {
  v += __uint_as_float(row_rotate<8>(__float_as_uint(v)));
  v += __uint_as_float(row_rotate<4>(__float_as_uint(v)));
  v += __uint_as_float(row_rotate<2>(__float_as_uint(v)));
  return v + __uint_as_float(row_rotate<1>(__float_as_uint(v)));
}

// The statistics need the whole row, the row is a few thousand scores of a few query heads and the top-k
// holds it in registers anyway: one launch in place of finalize_stats_kernel (or group_stats_kernel) and
// combine_kernel, each 4 to 8 us in front of a 6 us top-k for a microsecond's worth of bytes.  Sixteen waves share a
// CU, so what every wave does counts four times: sums of 64 scores, 128 of rows beyond 4096 tokens, by rows of lanes (fp32, at most as
// many as a resident tile's lanes add up; in double where the reduce-first order has them so), the 64 partial sums of a head in double and its
// statistics in one wave per head.
// GQ: query heads of a KV head, rounded up to 1, 4 or 8.
// A token whose z-scores are NaN ranks as combine_kernel ranks it: below every other (its general form starts each
// maximum from -inf, which drops a NaN), but with four or eight query heads, whose form starts from the first head, as
// the NaN that it is; one score per KV head of a dense call (pass_nan) keeps it too.
template <int VPT, int GQ>
__global__ __launch_bounds__(kTopkThreads, 4) void select_small_kernel(SmallSelect a) {
  constexpr int kWaves = kTopkThreads / 64, NV = 2 * GQ;
  typedef typename std::conditional<GQ == 1, double, float>::type Sum;
  __shared__ Sum red[NV][kWaves * 4];
  __shared__ float2 stats[GQ];               // mean, standard deviation (GQ == 1) or its reciprocal
  const int row = blockIdx.x, b = row / a.Hkv, h = row % a.Hkv;
  const int T = a.seq_lens ? min(a.seq_lens[b], a.Tmax) : a.Tmax;
  if (a.status && a.seq_lens && threadIdx.x == 0 && h == 0 && a.seq_lens[b] > a.Tmax) atomicCAS(a.status, 0u, 3u);
  if (T <= 0) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int e0 = wave * (64 * VPT) + lane;
  const int nvalid = min(max((T - e0 + 63) / 64, 0), VPT);
  const int prefill = (a.protect_prefill && a.prefill_lens) ? a.prefill_lens[b] : 0;
  const int window_from = a.window_size > 0 ? T - min(a.window_size, T) : T;
  float acc[VPT];
  for (int l = 0; l < a.L; ++l) {
    float x[GQ][VPT];
#pragma unroll
    for (int g = 0; g < GQ; ++g) {
      const float* p = a.raw + ((int64_t)(b * a.L + l) * a.A + (int64_t)h * a.G + min(g, a.G - 1)) * a.raw_pitch;
#pragma unroll
      for (int i = 0; i < VPT; ++i) x[g][i] = p[min(e0 + 64 * i, T - 1)];
    }
    float mean[GQ], sd[GQ];
#pragma unroll
    for (int g = 0; g < GQ; ++g) { mean[g] = 0.f; sd[g] = 1.f; }
    if (a.normalize) {
#pragma unroll
      for (int g = 0; g < GQ; ++g) {
        Sum s = 0, q = 0;
#pragma unroll
        for (int i = 0; i < VPT; ++i) {
          const Sum v = i < nvalid ? (Sum)x[g][i] : (Sum)0;
          s += v;
          q = fma(v, v, q);
        }
        if constexpr (GQ == 1) { s = row_sum_f64(s); q = row_sum_f64(q); }
        else { s = row_sum_f32(s); q = row_sum_f32(q); }
        if ((lane & 15) == 0) {
          red[2 * g][wave * 4 + (lane >> 4)] = s;
          red[2 * g + 1][wave * 4 + (lane >> 4)] = q;
        }
      }
      __syncthreads();
      if (wave < GQ) {
        double s = row_sum_f64((double)red[2 * wave][lane]), q = row_sum_f64((double)red[2 * wave + 1][lane]);
        s = ((lane_f64(s, 0) + lane_f64(s, 16)) + lane_f64(s, 32)) + lane_f64(s, 48);
        q = ((lane_f64(q, 0) + lane_f64(q, 16)) + lane_f64(q, 32)) + lane_f64(q, 48);
        float m, e;
        if (a.pass_nan) {                    // (the reduce-first definitions, group_stats_kernel)
          const double mu = s / (double)T;
          double var = T > 1 ? (q - (double)T * mu * mu) / (double)(T - 1) : 0.0;
          if (var < 0.0) var = 0.0;
          e = (float)sqrt(var);
          if (e < 1e-8f) e = 1.f;
          m = (float)mu;
        } else if (a.normalize == 2) {
          const double mu = s / (double)T;
          const double var = q / (double)T - mu * mu;
          m = (float)mu;
          e = fmaxf((float)sqrt(var > 0.0 ? var : 0.0), 1e-6f);
        } else {                             // the reference's formula on fp32 sums (runtime/selector_hf.py:902-909)
          const float sum = (float)s, sumsq = (float)q, cnt = (float)T;
          m = __fdiv_rn(sum, cnt);
          float var = 0.f;
          if (T > 1) var = __fdiv_rn(__fsub_rn(sumsq, __fmul_rn(cnt, __fmul_rn(m, m))), (float)(T - 1));
          var = fmaxf(var, 0.f);
          e = __fsqrt_rn(var);
          if (e < 1e-8f) e = 1.f;
        }
        if (lane == 0) stats[wave] = float2{m, GQ == 1 ? e : __fdiv_rn(1.f, e)};
      }
      __syncthreads();
#pragma unroll
      for (int g = 0; g < GQ; ++g) { mean[g] = stats[g].x; sd[g] = stats[g].y; }
    }
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
      float v;
      if constexpr (GQ == 1) {
        v = a.pass_nan ? passed_zscore(x[0][i], mean[0], sd[0]) : fmaxf(-INFINITY, zscore(x[0][i], mean[0], sd[0]));
      } else {
        // (times the reciprocal, as the resident kernels do it: a division is ten instructions)
        v = __fmul_rn(__fsub_rn(x[0][i], mean[0]), sd[0]);
#pragma unroll
        for (int g = 1; g < GQ; ++g)
          if (g < a.G) {
            const float z = __fmul_rn(__fsub_rn(x[g][i], mean[g]), sd[g]);
            v = (a.group_reduce == TRI_REDUCE_MAX) ? fmaxf(v, z) : __fadd_rn(v, z);
          }
        if (a.group_reduce != TRI_REDUCE_MAX) v = __fdiv_rn(v, (float)a.G);
        if (a.G != GQ) v = fmaxf(-INFINITY, v);
      }
      const int n = e0 + 64 * i;
      if (n >= window_from || n < prefill) v = INFINITY;
      if (l == 0) acc[i] = v;
      else acc[i] = (a.layer_reduce == TRI_REDUCE_MAX) ? fmaxf(acc[i], v) : __fadd_rn(acc[i], v);
    }
  }
  uint32_t key[VPT];
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    if (a.layer_reduce == TRI_REDUCE_MEAN) acc[i] = __fdiv_rn(acc[i], (float)a.L);
    if (a.fin && i < nvalid) a.fin[(int64_t)row * a.Tmax + e0 + 64 * i] = acc[i];
    key[i] = i < nvalid ? row_key(acc[i]) : 0u;
  }
  if (!a.keep) return;
  const int k = min(min(a.budgets ? a.budgets[b] : a.keep_pitch, a.keep_pitch), T);
  int32_t* keep = a.keep + (int64_t)row * a.keep_pitch;
  if (k <= 0) return;
  if (k >= T) {
    for (int i = tid; i < T; i += kTopkThreads) keep[i] = i;
    return;
  }
  emit_topk<VPT>(key, T, k, keep);
}

}  // namespace

bool select_small_takes(int Tmax, int G) {
  return G <= 8 && Tmax <= (G == 1 ? 16 : G <= 4 ? 8 : 4) * kTopkThreads;    // (registers)
}

hipError_t launch_select_small(const SmallSelect& a, int B, hipStream_t s) {
  if (!select_small_takes(a.Tmax, a.G) || (a.pass_nan && a.G != 1)) return hipErrorInvalidValue;
  auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3((unsigned)(B * a.Hkv)), dim3(kTopkThreads), 0, s, a); };
  const int per = ceil_div(a.Tmax, kTopkThreads);
  if (a.G > 4) {
    launch(select_small_kernel<4, 8>);
  } else if (a.G > 1) {
    if (per <= 4) launch(select_small_kernel<4, 4>); else launch(select_small_kernel<8, 4>);
  } else {
    if (per <= 4) launch(select_small_kernel<4, 1>);
    else if (per <= 8) launch(select_small_kernel<8, 1>);
    else launch(select_small_kernel<16, 1>);
  }
  return hipGetLastError();
}

hipError_t launch_topk_rows(const float* scores, int64_t row_pitch, int num_rows,
                            const int32_t* row_lens, const int32_t* row_ks, int rows_per_entry, int max_len,
                            int32_t* keep, int keep_pitch, hipStream_t s, int groups, int64_t group_stride,
                            int group_max) {
  if (num_rows <= 0) return hipSuccess;
  if (max_len > 0 && max_len <= 4 * kTopkThreads)
    hipLaunchKernelGGL(topk_rows_reg_kernel<4>, dim3(num_rows), dim3(kTopkThreads), 0, s, scores, row_pitch, row_lens,
                       row_ks, rows_per_entry, keep, keep_pitch, max_len, groups, group_stride, group_max);
  else if (max_len > 0 && max_len <= 8 * kTopkThreads)
    hipLaunchKernelGGL(topk_rows_reg_kernel<8>, dim3(num_rows), dim3(kTopkThreads), 0, s, scores, row_pitch, row_lens,
                       row_ks, rows_per_entry, keep, keep_pitch, max_len, groups, group_stride, group_max);
  else if (max_len > 0 && max_len <= 16 * kTopkThreads)
    hipLaunchKernelGGL(topk_rows_reg_kernel<16>, dim3(num_rows), dim3(kTopkThreads), 0, s, scores, row_pitch, row_lens,
                       row_ks, rows_per_entry, keep, keep_pitch, max_len, groups, group_stride, group_max);
  else if (max_len > 0 && max_len <= 32 * kTopkThreads)
    hipLaunchKernelGGL(topk_rows_reg_kernel<32>, dim3(num_rows), dim3(kTopkThreads), 0, s, scores, row_pitch, row_lens,
                       row_ks, rows_per_entry, keep, keep_pitch, max_len, groups, group_stride, group_max);
  else if (groups > 1)
    return hipErrorInvalidValue;      // rows beyond the register kernels are reduced by the caller first
  else
    hipLaunchKernelGGL(topk_rows_kernel, dim3(num_rows), dim3(kTopkThreads), 0, s, scores, row_pitch, row_lens,
                       row_ks, rows_per_entry, keep, keep_pitch, max_len);
  return hipGetLastError();
}

// Longest row the register top-k kernels take (they can also add partial rows while loading).
int topk_register_row_limit() { return 32 * kTopkThreads; }

hipError_t launch_select(const SelectLaunch& a, hipStream_t s) {
  const int n = a.B * a.L * a.A;
  // Whole token rows for the usual layout; the chunk sums ([B][L][chunks][Hkv][2] doubles) go
  // into scratch the caller names.
  int chunk = kGroupStatsChunk;
  while (chunk > kGroupStatsChunkMin && (int64_t)ceil_div(a.Tmax, chunk) * a.B * a.L < 1024 &&
         (int64_t)a.B * a.L * ceil_div(a.Tmax, chunk / 2) * a.Hkv * 16 <= a.group_scratch_bytes)
    chunk /= 2;
  const int chunks = ceil_div(a.Tmax, chunk);
  const bool rows = a.group_first && a.normalize && a.G == 4 && a.A == a.Hkv * 4 && a.raw_stride_head == 1 &&
                    a.raw_stride_token % 4 == 0 && a.raw_stride_layer % 4 == 0 &&
                    (reinterpret_cast<uintptr_t>(a.raw) % 16) == 0 && a.Hkv <= 128 && (a.Hkv & (a.Hkv - 1)) == 0 &&
                    a.group_scratch != nullptr &&
                    (int64_t)a.B * a.L * chunks * a.Hkv * 16 <= a.group_scratch_bytes;
  // Long rows of one score per KV head: chunks as well, where the caller's scratch holds their sums.
  const int single_chunks = ceil_div(a.Tmax, kGroupStatsChunk);
  const bool single = a.pass_nan && a.normalize && a.Tmax >= kSingleStatsTokens && a.raw_stride_head == 1 && a.Hkv <= 256 &&
                      a.group_scratch != nullptr && (int64_t)a.B * a.L * single_chunks * a.Hkv * 16 <= a.group_scratch_bytes;
  if (single) {
    int hpad = 1;
    while (hpad < a.Hkv) hpad <<= 1;
    hipLaunchKernelGGL(single_stats_partial_kernel, dim3(single_chunks, a.B * a.L), dim3(256), 0, s, a.raw, a.raw_stride_layer,
                       a.raw_stride_token, a.seq_lens, a.L, a.Hkv, hpad, kGroupStatsChunk, single_chunks, a.group_scratch);
    hipLaunchKernelGGL(group_stats_finish_kernel, dim3(ceil_div(a.B * a.L * a.Hkv, 256)), dim3(256), 0, s, a.group_scratch,
                       a.seq_lens, a.B * a.L, a.L, a.Hkv, a.A, kGroupStatsChunk, single_chunks, a.mustd);
  } else if (rows) {
    double* part = a.group_scratch;
    hipLaunchKernelGGL(group_stats_partial_kernel, dim3(chunks, a.B * a.L), dim3(256), 0, s, a.raw, a.raw_stride_layer,
                       a.raw_stride_token, a.seq_lens, a.L, a.Hkv, chunk, chunks, a.group_reduce, part);
    hipLaunchKernelGGL(group_stats_finish_kernel, dim3(ceil_div(a.B * a.L * a.Hkv, 256)), dim3(256), 0, s, part,
                       a.seq_lens, a.B * a.L, a.L, a.Hkv, a.A, chunk, chunks, a.mustd);
  } else if (a.group_first) {
    auto launch = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3(a.B * a.L * a.Hkv), dim3(256), 0, s, a.raw, a.raw_stride_layer, a.raw_stride_token,
                         a.raw_stride_head, a.seq_lens, a.L, a.Hkv, a.A, a.G, a.group_reduce, a.normalize, a.mustd);
    };
    if (a.pass_nan) launch(group_stats_kernel<true>);
    else launch(group_stats_kernel<false>);
  } else
    hipLaunchKernelGGL(finalize_stats_kernel, dim3(ceil_div(n, 256)), dim3(256), 0, s, a.partial, a.seq_lens,
                       a.B, a.L, a.A, ceil_div(a.Tmax, a.fine ? kScoreFineTokens : kScoreTileTokens), a.fine, a.normalize, a.mustd);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;

  CombineArgs c{};
  c.raw = a.raw;
  c.mustd = a.mustd;
  c.seq_lens = a.seq_lens;
  c.prefill_lens = a.prefill_lens;
  c.fin = a.fin;
  c.raw_stride_layer = a.raw_stride_layer;
  c.raw_stride_token = a.raw_stride_token;
  c.raw_stride_head = a.raw_stride_head;
  c.B = a.B; c.L = a.L; c.Hkv = a.Hkv; c.A = a.A; c.G = a.G; c.Tmax = a.Tmax;
  c.window_size = a.window_size;
  c.protect_prefill = a.protect_prefill;
  c.group_reduce = a.group_reduce;
  c.layer_reduce = a.layer_reduce;
  c.shared = a.shared;
  c.pass_nan = a.pass_nan;
  if (a.pass_nan && (a.G != 1 || a.shared)) return hipErrorInvalidValue;
  c.rows_per_seq = a.shared ? 1 : a.Hkv;
  const bool per_layer = a.layer_reduce < 0;
  // Reducing over the layers, a thread's time is its rounds of loads.  Where few workgroups share the chip
  // nothing hides them: one wave per workgroup (four times as many of them) and three times as many
  // layers requested at once (one request of 2176 tokens x 36 layers, 68 workgroups: 19 -> 8 us; 2 x 8192
  // tokens 32 -> 23).  One layer per thread (a keep set per layer) has nothing to batch.
  const bool vec = (a.G == 4 || a.G == 8) && a.raw_stride_head == 1 && a.raw_stride_token % 4 == 0 &&
                   a.raw_stride_layer % 4 == 0 && (reinterpret_cast<uintptr_t>(a.raw) % 16) == 0 &&
                   (reinterpret_cast<uintptr_t>(a.mustd) % 16) == 0;
  const bool few = vec && !per_layer && c.rows_per_seq <= 64 &&
                   (int64_t)ceil_div(a.Tmax, 256 / c.rows_per_seq) * a.B < 1024;
  const int threads = few ? 64 : 256;
  c.tokens_per_wg = threads / c.rows_per_seq;
  dim3 grid(ceil_div(a.Tmax, c.tokens_per_wg), per_layer ? a.L : 1, a.B);
  const size_t smem = (size_t)c.rows_per_seq * c.tokens_per_wg * sizeof(float);
  auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(threads), smem, s, c); };
  if (!vec) {
    if (a.group_first) launch(combine_kernel<0, 1, true>);
    else launch(combine_kernel<0, 1, false>);
  } else if (a.G == 4) {
    if (per_layer) { if (a.group_first) launch(combine_kernel<1, 1, true>); else launch(combine_kernel<1, 1, false>); }
    else if (few) { if (a.group_first) launch(combine_kernel<1, 12, true>); else launch(combine_kernel<1, 12, false>); }
    else { if (a.group_first) launch(combine_kernel<1, 4, true>); else launch(combine_kernel<1, 4, false>); }
  } else {
    if (per_layer) { if (a.group_first) launch(combine_kernel<2, 1, true>); else launch(combine_kernel<2, 1, false>); }
    else if (few) { if (a.group_first) launch(combine_kernel<2, 6, true>); else launch(combine_kernel<2, 6, false>); }
    else { if (a.group_first) launch(combine_kernel<2, 2, true>); else launch(combine_kernel<2, 2, false>); }
  }
  e = hipGetLastError();
  if (e != hipSuccess) return e;

  if (!a.keep) return hipSuccess;   // selection scores only
  const int rows_per_entry = c.rows_per_seq * (per_layer ? a.L : 1);
  return launch_topk_rows(a.fin, a.Tmax, a.B * rows_per_entry, a.seq_lens, a.budgets, rows_per_entry, a.Tmax, a.keep,
                          a.max_budget, s);
}

}  // namespace tri
