// Scores of a small launch -- few layers of few requests -- in one launch, preparation included: two-byte keys,
// mean aggregation, up to eight query heads per KV head.
//
//   raw[n][q] = sum_e k[n][e] * C[e][q]  +  sum_f |k_f[n]| * E[f][q]
//
// on the matrix cores as in tri_fused_mfma.hip: a step is 16 tokens of one KV head, the A operand of the key
// products is the loaded row as it is, the columns of B are (query head, piece of the coefficient).  What
// differs is what bounds it: one layer of 4096 tokens is 8 MB, 2 us of memory traffic, and the resident
// kernel took 19 us behind 5.5 us of preparation on 32 workgroups that walk eight steps each and then
// wait for each other.  Here a wave takes ONE step: a workgroup is 128 tokens of one (sequence, layer, KV
// head), 256 of them for that layer, every workgroup evaluates the phases, the coefficients of its query
// heads and the operands for itself (in LDS, while its keys are on their way), and the statistics are left
// to the selection (select_small_kernel), which reads the raw scores anyway.  One layer x 4096 tokens, 32 / 8 heads of 128: preparation 5.5 + scorer 18.7
// -> 8.7 us; score + select 32.1 -> 17.5.  The dense call's prologue 2.1 + preparation 3.5 + scorer 17.4 -> 7.3 us.
//
// Nothing is raised or repeated, so fp32's range is kept:
//  - the magnitudes enter as three bf16 pieces of eight bits, cut off and not rounded, which is the whole
//    fp32 value, and so do the magnitude coefficients;
//  - fp16 keys: the coefficients of a query head are scaled by a power of two into fp16's range, and the
//    scores scaled back; with bf16 keys the pieces have fp32's range as they are (below 2^-109 the third one is a
//    subnormal, and a coefficient keeps the bits above 2^-133);
//  - a step in which any score is not finite (keys that are not, products beyond fp32) is evaluated again
//    pair by pair in fp32, so infinities and NaNs come out as a sum of products gives them.
#include "tri_common.h"
#include "tri_mma_device.h"
#include "tri_score_device.h"

namespace tri {
namespace {

constexpr int kMmaThreads = 512;           // eight waves, a step each
constexpr int kMmaTokens = 16 * (kMmaThreads / 64);
constexpr int kMmaRor4 = 0x124, kMmaRor8 = 0x128, kMmaRor12 = 0x12c;    // row_ror:n

// Operands of a KV head: up to four query heads NS key slabs and NS / 2 magnitude slabs, columns (head j % 4,
// piece j / 4); five to eight: key slabs with pieces (1 | 2) of heads j % 8, then with piece 3 beside zeros, and
// the magnitude slabs the same way.
template <int HD, int QG> constexpr int mma_slabs() { return QG * (HD / 32 + HD / 64); }

// Element e of lane block kb in slab s, two-byte rows: 16-byte chunk 4 s + kb.
__device__ __forceinline__ constexpr int mma_elem(int s, int kb, int e) { return (4 * s + kb) * 8 + e; }

// Piece p (0, 1, 2) of x in bf16: what is left after p roundings.
__device__ __forceinline__ uint32_t bf16_piece(float x, int p) {
  uint32_t bits = 0;
  for (int i = 0; i <= p; ++i) {
    bits = (uint32_t)__builtin_bit_cast(unsigned short, (__bf16)x);
    x -= __uint_as_float(bits << 16);
  }
  return bits;
}
__device__ __forceinline__ uint32_t f16_piece(float x, int p) {
  uint32_t bits = 0;
  for (int i = 0; i <= p; ++i) {
    const _Float16 h = (_Float16)x;
    bits = (uint32_t)__builtin_bit_cast(unsigned short, h);
    x -= (float)h;
  }
  return bits;
}

// One lane's 16 bytes of operand o from the coefficients cf[query head][P | R | E][F] (pitch 3 F + 1) and, for fp16
// keys, the heads' scales.
template <int DT, bool IL, int HD, int QG>
__device__ __forceinline__ uint4 mma_operand(const float* cf, const float* scale, int o, int lane, int G) {
  constexpr int F = HD / 2, NS = HD / 32;
  const int j = lane & 15, kb = lane >> 4;
  const bool mag = o >= QG * NS;
  const int within = mag ? o - QG * NS : o, per = mag ? NS / 2 : NS;
  const int slab = within % per;
  int q, piece;
  if constexpr (QG == 1) { q = j & 3; piece = j >> 2; }
  else { q = j & 7; piece = within >= per ? (j < 8 ? 2 : 3) : j >> 3; }
  if (q >= G || piece > 2) return uint4{0, 0, 0, 0};
  const float* c = cf + q * (3 * F + 1);
  const float sc = DT == TRI_KV_FP16 ? scale[q] : 1.f;
  uint32_t w[4];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    int which, pair;
    if (mag) {
      which = 2;
      // interleaved: pairs of slabs 2 * slab and 2 * slab + 1; half: real parts of slab `slab`
      pair = IL ? mma_elem(2 * slab + (e >> 2), kb, 2 * (e & 3)) >> 1 : mma_elem(slab, kb, e) & (F - 1);
    } else {
      const int el = mma_elem(slab, kb, e);
      which = IL ? el & 1 : (el >= F ? 1 : 0);
      pair = IL ? el >> 1 : el & (F - 1);
    }
    const float x = c[which * F + pair] * sc;
    const uint32_t b = (DT == TRI_KV_FP16 && !mag) ? f16_piece(x, piece) : bf16_piece(x, piece);
    w[e >> 1] = (e & 1) ? w[e >> 1] | (b << 16) : b;
  }
  return uint4{w[0], w[1], w[2], w[3]};
}

// Power of two that takes the largest of |P|, |R| of a query head to about 2^13 (fp16 keys), the second and third
// pieces then lie in fp16's range too.  Upwards as far as fp32 goes: beyond 2^126 a coefficient is a subnormal of fp32
// itself.  Down to 2^-40: a larger coefficient overflows, and its steps are evaluated pair by pair.  Called by a whole wave.
template <int F>
__device__ __forceinline__ float fp16_scale(const float* c, int lane) {
  float m = 0.f;
  for (int f = lane; f < 2 * F; f += 64) m = fmaxf(m, fabsf(c[f]));
  for (int d = 32; d > 0; d >>= 1) m = fmaxf(m, __shfl_xor(m, d));
  int e = 0;
  if (m > 0.f && m < INFINITY) (void)frexpf(m, &e);
  else e = 13;
  return ldexpf(1.f, min(max(13 - e, -40), 126));
}

// Means over the offsets of cos and sin of the phases, the way prepare_kernel evaluates them (summed in offset order
// in double).  buf: 2 * NO * F floats.  Ends without a barrier.
template <int HD>
__device__ __forceinline__ void mma_phase_means(const float* omega, const float* offsets, int NO, int round_start, float* buf,
                                                float (*mean_cs)[HD / 2]) {
  constexpr int F = HD / 2;
  const int tid = threadIdx.x, nthreads = blockDim.x;
  const float rs = (float)round_start;
  for (int i = tid; i < NO * F; i += nthreads) {
    const int j = i / F, f = i % F;
    phase_cos_sin(__fmul_rn(__fadd_rn(rs, offsets[j]), omega[f]), buf[j * F + f], buf[(NO + j) * F + f]);
  }
  __syncthreads();
  for (int i = tid; i < 2 * F; i += nthreads) {
    double sum = 0.0;
    for (int j = 0; j < NO; ++j) sum += buf[((i / F) * NO + j) * F + i % F];
    mean_cs[i / F][i % F] = (float)(sum / NO);
  }
}

// Eight fp32 magnitudes as three packed bf16 pieces, eight bits each from the top.
__device__ __forceinline__ void split8_bf16x3(const float (&x)[8], uint4& hi, uint4& mid, uint4& lo) {
  uint32_t h[4], m[4], l[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float a = x[2 * i], b = x[2 * i + 1];
    const float ra = a - __uint_as_float(__float_as_uint(a) & 0xffff0000u), rb = b - __uint_as_float(__float_as_uint(b) & 0xffff0000u);
    const float sa = ra - __uint_as_float(__float_as_uint(ra) & 0xffff0000u), sb = rb - __uint_as_float(__float_as_uint(rb) & 0xffff0000u);
    h[i] = __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
    m[i] = __builtin_amdgcn_perm(__float_as_uint(rb), __float_as_uint(ra), 0x07060302u);
    l[i] = __builtin_amdgcn_perm(__float_as_uint(sb), __float_as_uint(sa), 0x07060302u);
  }
  hi = uint4{h[0], h[1], h[2], h[3]};
  mid = uint4{m[0], m[1], m[2], m[3]};
  lo = uint4{l[0], l[1], l[2], l[3]};
}

// What a lane holds of a step's scores: one group: head j % 4 of token 4 kb + j / 4; two: head j % 8 of tokens
// 4 kb + 2 (j / 8) and the next.
template <int QG> __device__ __forceinline__ int lane_head(int lane) { return lane & (4 * QG - 1); }
template <int QG> __device__ __forceinline__ int lane_token(int lane) {
  const int j = lane & 15, kb = lane >> 4;
  return 4 * kb + (QG == 1 ? j >> 2 : 2 * (j >> 3));
}

// Scores of the 16 rows in A.
template <int DT, bool IL, int HD, int QG>
__device__ __forceinline__ void mma_scores(const uint4 (&A)[HD / 32], const uint4 (&B)[mma_slabs<HD, QG>()], int lane,
                                           float unscale, float (&v)[QG]) {
  constexpr int NS = HD / 32, NK = QG * NS;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int o = 0; o < NK; ++o) acc = mfma_16x16x32<DT>(A[o % NS], B[o], acc);
  uint32_t w[NS][4];
#pragma unroll
  for (int s = 0; s < NS; ++s) { w[s][0] = A[s].x; w[s][1] = A[s].y; w[s][2] = A[s].z; w[s][3] = A[s].w; }
#pragma unroll
  for (int set = 0; set < NS / 2; ++set) {
    float mag[8];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      uint32_t x[4];
      if constexpr (IL) {
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] = w[2 * set + h][i];
      } else {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const uint32_t re = w[set][2 * h + i], im = w[set + NS / 2][2 * h + i];
          x[2 * i] = __builtin_amdgcn_perm(im, re, 0x05040100u);
          x[2 * i + 1] = __builtin_amdgcn_perm(im, re, 0x07060302u);
        }
      }
      magnitudes4<DT>(x, &mag[4 * h]);
    }
    uint4 hi, mid, lo;
    split8_bf16x3(mag, hi, mid, lo);
    acc = mfma_16x16x32<TRI_KV_BF16>(hi, B[NK + set], acc);
    acc = mfma_16x16x32<TRI_KV_BF16>(mid, B[NK + set], acc);
    acc = mfma_16x16x32<TRI_KV_BF16>(lo, B[NK + set], acc);
    if constexpr (QG == 2) {
      acc = mfma_16x16x32<TRI_KV_BF16>(hi, B[NK + NS / 2 + set], acc);
      acc = mfma_16x16x32<TRI_KV_BF16>(mid, B[NK + NS / 2 + set], acc);
    }
  }
  const float x0 = acc[0], x1 = acc[1], x2 = acc[2], x3 = acc[3];
  const bool upper = (lane & 8) != 0;
  // first the two halves of the columns
  const float send0 = upper ? x0 : x2, send1 = upper ? x1 : x3;
  const float y0 = (upper ? x2 : x0) + dpp<kMmaRor8>(send0);
  const float y1 = (upper ? x3 : x1) + dpp<kMmaRor8>(send1);
  if constexpr (QG == 2) {
    v[0] = y0;
    v[1] = y1;
  } else {
    // then columns four apart: of a half the lower quad takes y0, the upper y1
    const bool odd = (lane & 4) != 0;
    const float keep = odd ? y1 : y0, send = odd ? y0 : y1;
    const float below = dpp<kMmaRor4>(send), above = dpp<kMmaRor12>(send);     // (of lane - 4 and of lane + 4)
    v[0] = keep + (odd ? below : above);
  }
  if constexpr (DT == TRI_KV_FP16) {
#pragma unroll
    for (int i = 0; i < QG; ++i) v[i] *= unscale;
  }
}

// The same pair by pair in fp32, for a step with scores that are not finite.  rows: every lane's row (lane % 16 of the
// step); cf + q * pitch: [P | R | E][F] of query head q.
template <int DT, bool IL, int HD, int QG>
__device__ __forceinline__ void plain_scores(const char* row, const float* cf, int pitch, int G, int lane, float (&v)[QG]) {
  constexpr int F = HD / 2;
  for (int i = 0; i < 16; ++i) {
    const uint64_t p = reinterpret_cast<uint64_t>(row);
    const uint64_t r = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(p >> 32), i) << 32) |
                       (uint32_t)__builtin_amdgcn_readlane((int)p, i);
    const unsigned short* k = reinterpret_cast<const unsigned short*>(r);
    for (int q = 0; q < G; ++q) {
      float t = 0.f;
      for (int f = lane; f < F; f += 64) {
        const uint32_t re = k[IL ? 2 * f : f], im = k[IL ? 2 * f + 1 : F + f];
        const float kr = elem_lo<DT>(re), ki = elem_lo<DT>(im);
        const float m = __builtin_amdgcn_sqrtf(fmaf(ki, ki, kr * kr));
        const float* c = cf + q * pitch;
        t = fmaf(kr, c[f], t);
        t = fmaf(ki, c[F + f], t);
        t = fmaf(m, c[2 * F + f], t);
      }
      for (int d = 32; d > 0; d >>= 1) t += __shfl_xor(t, d);
      const int at = i - lane_token<QG>(lane);
      if (lane_head<QG>(lane) == q) {
#pragma unroll
        for (int u = 0; u < QG; ++u)
          if (at == u) v[u] = t;
      }
    }
  }
}

template <int QG>
__device__ __forceinline__ bool all_finite(const float (&v)[QG]) {
  bool bad = !(fabsf(v[0]) < INFINITY);
  if constexpr (QG == 2) bad = bad || !(fabsf(v[1]) < INFINITY);
  return !__any(bad);
}

// Keys of one step: row lane % 16, 16-byte chunks 4 s + lane / 16.
template <int DT, bool IL, int HD, int QG>
__global__ __launch_bounds__(kMmaThreads) __attribute__((amdgpu_waves_per_eu(2, 4)))
void score_small_kernel(SmallScore a) {
  constexpr int NS = HD / 32, NSO = mma_slabs<HD, QG>(), F = HD / 2, NI = (4 * QG * F + kMmaThreads - 1) / kMmaThreads;
  __shared__ __align__(16) float phases[2 * kMaxOffsets * F];
  __shared__ float mean_cs[2][F];
  __shared__ float cf[4 * QG * (3 * F + 1)];
  __shared__ float scale[4 * QG];
  uint4* operands = reinterpret_cast<uint4*>(phases);   // (the phases are spent when the operands are made)
  static_assert(NSO * 64 * 16 <= sizeof(phases), "the operands must fit");
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int head = blockIdx.y, bl = blockIdx.z, b = bl / a.L, l = bl - b * a.L;
  if (a.status && blockIdx.x == 0 && head == 0 && bl == 0 && tid == 0) *a.status = 0u;
  const int T = a.seq_lens ? min(a.seq_lens[b], a.Tmax) : a.Tmax;
  const int n0 = blockIdx.x * kMmaTokens;
  if (n0 >= T) return;                                  // (the whole workgroup)

  // The keys and the statistics are requested first: the phases do not depend on them.
  const int t0 = n0 + 16 * wave;
  const int t = min(t0 + (lane & 15), T - 1);           // rows past the end: the last
  int64_t blk = b;
  int in = t;
  if (a.block_table) {
    const int lb = a.bs_shift >= 0 ? t >> a.bs_shift : t / a.block_size;
    blk = a.block_table[(int64_t)b * a.block_table_pitch + lb];
    in = t - lb * a.block_size;
  }
  const char* k = reinterpret_cast<const char*>(a.k_layers ? a.k_layers[l] : a.k);
  const char* row = k + (blk * a.stride_block + in * a.stride_token + (int64_t)head * a.stride_head) * 2;
  uint4 A[NS];
  {
    GlobalBytes p = (GlobalBytes)(uintptr_t)(row + (lane >> 4) * 16);
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const u32x4 x = *(GlobalU4)(p + s * 64);
      A[s] = uint4{x.x, x.y, x.z, x.w};
    }
  }
  float st[NI][3];
  const int64_t first_head = (int64_t)l * a.A + (int64_t)head * a.G;
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int at = min(tid + i * kMmaThreads, a.G * F - 1);
    if (a.folded) {                                     // head rows [a1 | a2 | e][F]
      const float* p = a.folded + (first_head + at / F) * 3 * F + at % F;
      st[i][0] = p[0]; st[i][1] = p[F]; st[i][2] = p[2 * F];
    } else {                                            // as fold_stats_kernel makes them
      const int64_t o = first_head * F + at;
      const float r = a.q_mean[2 * o], im = a.q_mean[2 * o + 1], s = a.freq_scale[o];
      const float qmag = __fsqrt_rn(__fadd_rn(__fadd_rn(__fmul_rn(r, r), __fmul_rn(im, im)), 1e-8f));
      const float e = a.disable_mlr ? a.q_abs[o] : __fsub_rn(a.q_abs[o], qmag);
      st[i][0] = a.disable_trig ? 0.f : s * r;
      st[i][1] = a.disable_trig ? 0.f : s * im;
      st[i][2] = s * e;
    }
  }
  mma_phase_means<HD>(a.omega, a.offsets, a.NO, a.round_start ? a.round_start[b] : a.round, phases, mean_cs);
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int at = tid + i * kMmaThreads;
    if (at < a.G * F) {
      const int f = at % F;
      const float c = mean_cs[0][f], sn = mean_cs[1][f];
      float* o = cf + at / F * (3 * F + 1) + f;
      o[0] = fmaf(st[i][0], c, -st[i][1] * sn);
      o[F] = fmaf(st[i][1], c, st[i][0] * sn);
      o[2 * F] = st[i][2];
    }
  }
  __syncthreads();
  if constexpr (DT == TRI_KV_FP16) {
    for (int q = wave; q < a.G; q += kMmaThreads / 64) {
      const float s = fp16_scale<F>(cf + q * (3 * F + 1), lane);
      if (lane == 0) scale[q] = s;
    }
    __syncthreads();
  }
  for (int i = tid; i < NSO * 64; i += kMmaThreads) operands[i] = mma_operand<DT, IL, HD, QG>(cf, scale, i >> 6, i & 63, a.G);
  __syncthreads();
  if (t0 >= T) return;                                  // (no barrier below)
  uint4 B[NSO];
#pragma unroll
  for (int o = 0; o < NSO; ++o) B[o] = operands[o * 64 + lane];
  const int q = lane_head<QG>(lane);
  float unscale = 1.f;
  if constexpr (DT == TRI_KV_FP16) unscale = 1.f / scale[min(q, a.G - 1)];
  float v[QG];
  mma_scores<DT, IL, HD, QG>(A, B, lane, unscale, v);
  if (!all_finite<QG>(v)) plain_scores<DT, IL, HD, QG>(row, cf, 3 * F + 1, a.G, lane, v);
  float* out = a.raw + ((int64_t)bl * a.A + (int64_t)head * a.G + q) * a.raw_pitch;
  const int tok = t0 + lane_token<QG>(lane);
#pragma unroll
  for (int i = 0; i < QG; ++i)
    if (q < a.G && tok + i < T) out[tok + i] = v[i];
}

template <int DT, bool IL>
hipError_t launch_small_t(const SmallScore& a, int D, dim3 grid, hipStream_t s) {
  auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(kMmaThreads), 0, s, a); };
  const bool two = a.G > 4;
  switch (D) {
    case 64: if (two) launch(score_small_kernel<DT, IL, 64, 2>); else launch(score_small_kernel<DT, IL, 64, 1>); break;
    case 128: if (two) launch(score_small_kernel<DT, IL, 128, 2>); else launch(score_small_kernel<DT, IL, 128, 1>); break;
    case 256: if (two) launch(score_small_kernel<DT, IL, 256, 2>); else launch(score_small_kernel<DT, IL, 256, 1>); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace

hipError_t launch_score_small(SmallScore a, int B, int Hkv, int D, int kv_dtype, int rope_style, hipStream_t s) {
  if (a.G > 8 || a.NO <= 0 || a.NO > kMaxOffsets) return hipErrorInvalidValue;
  a.bs_shift = -1;
  for (int sft = 0; sft < 31; ++sft)
    if ((1 << sft) == a.block_size) a.bs_shift = sft;
  const dim3 grid((unsigned)ceil_div(a.Tmax, kMmaTokens), (unsigned)Hkv, (unsigned)(B * a.L));
  const bool il = rope_style == TRI_ROPE_INTERLEAVED;
  if (kv_dtype == TRI_KV_BF16) return il ? launch_small_t<TRI_KV_BF16, true>(a, D, grid, s) : launch_small_t<TRI_KV_BF16, false>(a, D, grid, s);
  if (kv_dtype == TRI_KV_FP16) return il ? launch_small_t<TRI_KV_FP16, true>(a, D, grid, s) : launch_small_t<TRI_KV_FP16, false>(a, D, grid, s);
  return hipErrorInvalidValue;
}

}  // namespace tri
