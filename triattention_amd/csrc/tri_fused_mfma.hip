// Resident score + normalise + reduce kernel with the contraction on the matrix cores
// (gfx950, v_mfma_f32_16x16x32_bf16).  Same structure as tri_fused.hip (raw scores of a
// layer stay in LDS, per-layer statistics exchanged through tagged words, one continuous
// stream of key loads), different mapping of the arithmetic:
//
//   raw[n][q] = sum_e k[n][e] * C[e][q]  +  sum_f |k_f[n]| * E[f][q]
//
// with k[n][.] the 128 cached elements of one KV head of token n (bf16, exact), C the P / R
// coefficients laid out per element, E the magnitude coefficients.  One wave owns one KV
// head.  An MFMA multiplies a 16 x 32 coefficient slab whose rows are (query head, split) with a
// 32-element x 16-token slab of keys, taken straight from the 16-byte loads (no
// unpacking): every fp32 coefficient is carried as three bf16 pieces
// c = c1 + c2 + c3, so the products are exact and the sum is an fp32 accumulation of the
// same terms the vector-unit kernel adds.  The magnitudes are evaluated on the vector unit
// in fp32 (sqrt(k_r^2 + k_i^2)), cut into two fp16 pieces and contracted the same way
// (v_mfma_f32_16x16x32_f16 against fp16 pieces of the magnitude coefficients).
// The pieces of a query head are rows of one lane's accumulator and add up there; every
// token's four scores are then spread over the lanes exactly as the ring in LDS wants them.
//
// Per 16 tokens of a head: 8 MFMAs, and vector work only for the magnitudes (about a third
// of the vector-unit kernel's instruction count), so bf16 keys run at the key stream's pace.
// fp8 e4m3 keys are widened to bf16 (exact) in registers and take the same route; the
// per-(token, head) scale multiplies the finished score.
#include <algorithm>
#include <type_traits>
#include <vector>

#include "tri_common.h"
#include "tri_mma_device.h"
#include "tri_score_device.h"
#include "tri_fused_device.h"

namespace tri {
namespace {


// What a lane loads of one (token, head) row per step; the token is lane % 16 of the step,
// kb = lane / 16.  Two-byte keys: the 16-byte chunks 4*s + kb, s = 0..3 (8 elements each,
// MFMA s takes chunk s).  fp8 keys: the 16-byte chunks kb and 4 + kb (16 elements each;
// MFMA s takes half s % 2 of chunk s / 2) and a dequantisation scale: that of token lane / 4 of the
// step; the lane's own token's comes from lane `scale_lane` when the step is scored.
// HD: head dimension, 128 or (two-byte keys only) 64 or 256: half or twice the chunks, MFMAs and pairs.
template <int DT, int HD>
struct StepData {
  uint4 c[DT == TRI_KV_FP8_E4M3 ? 2 : HD / 32];
  float scale;          // fp8 only; of token lane / 4
};

// Index, inside the 128 elements of a head row, of element e of lane block kb in MFMA s.
template <int DT>
__host__ __device__ constexpr int slab_elem(int s, int kb, int e) {
  return DT == TRI_KV_FP8_E4M3 ? (kb + 4 * (s >> 1)) * 16 + (s & 1) * 8 + e : (4 * s + kb) * 8 + e;
}

// Largest of three (the instruction returns the other operands' maximum when one is a NaN, as
// fmaxf does; written out because the compiler canonicalises every operand of fmaxf first).
__device__ __forceinline__ float max3(float a, float b, float c) {
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}

__device__ __forceinline__ float bf16_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }

// Eight fp32 values as two packed fp16 pieces each.  The remainders x - hi are exact in fp32 and rounded to fp16 by
// the same instruction (the mixed-precision fused multiply-add reads and writes halves of packed
// registers): three instructions per two values, which used to be four (no case got measurably faster by it alone).  A half written by one instruction is read by the next but three at
// the earliest: this chip wants one between.  The two idle cycles at the end are what it wants between a vector
// instruction and a matrix instruction that reads its result (the compiler, which keeps that distance elsewhere, does not
// see the instructions of an asm statement).
__device__ __forceinline__ void split8_f16(const float (&x)[8], uint4& hi, uint4& lo) {
  uint32_t h[4], l[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const f32x2 v = {x[2 * i], x[2 * i + 1]};
    h[i] = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, f16x2));
  }
  asm("v_fma_mixlo_f16 %0, %4, -1.0, %8 op_sel_hi:[1,0,0]\n\t"
      "v_fma_mixlo_f16 %1, %5, -1.0, %9 op_sel_hi:[1,0,0]\n\t"
      "v_fma_mixlo_f16 %2, %6, -1.0, %10 op_sel_hi:[1,0,0]\n\t"
      "v_fma_mixlo_f16 %3, %7, -1.0, %11 op_sel_hi:[1,0,0]"
      : "=&v"(l[0]), "=&v"(l[1]), "=&v"(l[2]), "=&v"(l[3])
      : "v"(h[0]), "v"(h[1]), "v"(h[2]), "v"(h[3]), "v"(x[0]), "v"(x[2]), "v"(x[4]), "v"(x[6]));
  asm("v_fma_mixhi_f16 %0, %4, -1.0, %8 op_sel:[1,0,0] op_sel_hi:[1,0,0]\n\t"
      "v_fma_mixhi_f16 %1, %5, -1.0, %9 op_sel:[1,0,0] op_sel_hi:[1,0,0]\n\t"
      "v_fma_mixhi_f16 %2, %6, -1.0, %10 op_sel:[1,0,0] op_sel_hi:[1,0,0]\n\t"
      "v_fma_mixhi_f16 %3, %7, -1.0, %11 op_sel:[1,0,0] op_sel_hi:[1,0,0]\n\t"
      "s_nop 1"
      : "+&v"(l[0]), "+&v"(l[1]), "+&v"(l[2]), "+&v"(l[3])
      : "v"(h[0]), "v"(h[1]), "v"(h[2]), "v"(h[3]), "v"(x[1]), "v"(x[3]), "v"(x[5]), "v"(x[7]));
  hi = uint4{h[0], h[1], h[2], h[3]};
  lo = uint4{l[0], l[1], l[2], l[3]};
}

// Larger halves of two packed fp16 pairs (no quieting of the operands, which costs an instruction each).
__device__ __forceinline__ f16x2 pk_max_f16(f16x2 a, uint32_t b) {
  asm("v_pk_max_f16 %0, %0, %1" : "+v"(a) : "v"(b));
  return a;
}

// Piece `pieces` of x in the operand type: what is left of x after `pieces` roundings.
template <int DT>
__device__ __forceinline__ float coefficient_piece(float x, int pieces) {
  for (int s = 0; s < pieces; ++s) {
    if constexpr (DT == TRI_KV_FP16)
      x = x - (float)(_Float16)x;
    else
      x = x - __uint_as_float((uint32_t)__builtin_bit_cast(unsigned short, (__bf16)x) << 16);
  }
  return x;
}

// Everything the resident kernel needs before it starts, in one launch: workgroup (l, b, z)
//  - clears its share of the exchange words (and workgroup (0, 0, 0) the status word);
//  - evaluates cos / sin of (round_start[b] + offset_j) * omega_f for all offsets and their
//    means over the offsets, the way prepare_kernel does (phase_cos_sin, means summed in offset
//    order in double);
//  - combines the means with the folded statistics of its KV heads of layer l (heads z * heads_per_wg
//    and up) into P = a1*C - a2*S, R = a2*C + a1*S, E and writes them as MFMA A operands:
// bmat[((b*L + l)*Hkv + head)*NSO + o][lane][8] of two bytes.  Lane (j = lane % 16, kb) of an operand holds
// row j, k indices kb*8 .. + 7 of its slab.  Up to four query heads per KV head: operands 0..NS-1 are the
// key slabs, NS/2 magnitude slabs follow; row j = (query head j / 4, piece j % 4).  Five to eight: NS key
// operands with row j = (query head j / 2, piece j % 2), NS more with the third piece in the even rows and
// zeros between, then the magnitude operands the same way.  Piece p of a coefficient x is
// what is left of x after p roundings to the operand type (x = x1 + x2 + x3).
constexpr int kPrepThreads = 1024;
// Query heads whose coefficients are staged at a time, and the pitch of a staged head
// [P | R | E][F] in floats (odd: the four query heads and four k blocks a wave reads at once
// then fall into 16 different banks).
template <int HD> constexpr int prep_heads() { return HD > 128 ? 32 : 64; }
template <int HD> constexpr int prep_pitch() { return 3 * (HD / 2) + 1; }

template <int DT, bool IL, int HD>
__global__ __launch_bounds__(kPrepThreads) void prep_mfma_kernel(const float* folded, const float* omega,
                                                                 const float* offsets, int NO,
                                                                 const int32_t* round_start, int L, int Hkv, int G,
                                                                 int A, uint4* bmat,
                                                                 unsigned long long* xchg, int64_t words,
                                                                 uint32_t* status, int heads_per_wg) {
  // One buffer, used twice: the per-offset cos / sin values, then the coefficients of up to
  // kPrepHeads query heads as [head][P | R | E][F] with a row pitch of 3F + 1 floats.
  constexpr int F = HD / 2;              // frequency pairs
  constexpr int NS = HD / 32;            // key slabs
  const int NSO = mfma_operands(F, G);   // operands of a KV head
  const int NK = G > 4 ? 2 * NS : NS;    // of them key operands, the magnitude operands follow
  constexpr int kPrepHeads = prep_heads<HD>(), kPrepPitch = prep_pitch<HD>();
  __shared__ float buf[kPrepHeads * kPrepPitch];
  __shared__ float mean_cs[2][F];
  static_assert(kPrepHeads * kPrepPitch >= 2 * kMaxOffsets * F, "the trig values must fit the buffer");
  float (*part)[kMaxOffsets][F] = reinterpret_cast<float (*)[kMaxOffsets][F]>(buf);
  const int l = blockIdx.x, b = blockIdx.y, tid = threadIdx.x;
  const int h_begin = blockIdx.z * heads_per_wg, h_end = min(Hkv, h_begin + heads_per_wg);
  const int64_t wg = ((int64_t)blockIdx.z * gridDim.y + b) * gridDim.x + l;
  const int64_t nwg = (int64_t)gridDim.x * gridDim.y * gridDim.z;
  // The first statistics are requested before the phases, on which they do not depend.
  const float* in = folded + ((int64_t)l * A + (int64_t)h_begin * G) * 3 * F;   // [head][a1 | a2 | e][F]
  const int first = min(tid, (h_end - h_begin) * G * F - 1);
  const float* in0 = in + first / F * 3 * F + first % F;
  const float first_a1 = in0[0], first_a2 = in0[F], first_e = in0[2 * F];
  for (int64_t i = wg * kPrepThreads + tid; i < words; i += nwg * kPrepThreads) xchg[i] = 0ull;
  if (wg == 0 && tid == 0) *status = 0u;

  const float rs = (float)round_start[b];
  for (int i = tid; i < NO * F; i += kPrepThreads) {
    const int j = i / F, f = i % F;
    phase_cos_sin(__fmul_rn(__fadd_rn(rs, offsets[j]), omega[f]), part[0][j][f], part[1][j][f]);
  }
  __syncthreads();
  if (tid < 2 * F) {
    const int which = tid / F, f = tid % F;
    double sum = 0.0;
    for (int j = 0; j < NO; ++j) sum += part[which][j][f];
    mean_cs[which][f] = (float)(sum / NO);
  }

  const int heads_per_pass = max(1, kPrepHeads / G);        // whole KV heads
  for (int head0 = h_begin; head0 < h_end; head0 += heads_per_pass) {
    const int nh = min(heads_per_pass, h_end - head0);
    __syncthreads();                                        // means written; buffer free
    // P = a1*C - a2*S, R = a2*C + a1*S, E, of query heads head0*G .. (head0 + nh)*G - 1
    for (int i = tid; i < nh * G * F; i += kPrepThreads) {
      const int q = i / F, f = i % F;
      float a1 = first_a1, a2 = first_a2, e = first_e;
      if (head0 > h_begin || i >= kPrepThreads) {
        const float* p = in + ((int64_t)(head0 - h_begin) * G + q) * 3 * F + f;
        a1 = p[0]; a2 = p[F]; e = p[2 * F];
      }
      const float c = mean_cs[0][f], sn = mean_cs[1][f];
      buf[q * kPrepPitch + f] = fmaf(a1, c, -a2 * sn);
      buf[q * kPrepPitch + F + f] = fmaf(a2, c, a1 * sn);
      buf[q * kPrepPitch + 2 * F + f] = e;
    }
    __syncthreads();
    const int items = nh * NSO * 64;                        // (head, operand, lane)
    uint4* out_base = bmat + (((int64_t)b * L + l) * Hkv + head0) * NSO * 64;
    for (int idx = tid; idx < items; idx += kPrepThreads) {
      const int lane = idx & 63;
      const int o = (idx >> 6) % NSO;
      const int head = idx / (64 * NSO);
      const int j = lane & 15, kb = lane >> 4;
      const bool mag = o >= NK;
      const int slab = mag ? (o - NK) % (NS / 2) : o % NS;
      int q, sp;                                            // query head and piece of row j (piece 3: a zero row)
      if (G > 4) {
        q = j >> 1;
        sp = (mag ? o - NK >= NS / 2 : o >= NS) ? ((j & 1) ? 3 : 2) : j & 1;
      } else {
        q = j >> 2;
        sp = j & 3;
      }
      uint32_t out[4] = {0, 0, 0, 0};
      if (q < G && sp < 3) {
        const float* c = buf + (head * G + q) * kPrepPitch;
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          int which, pair;   // which: 0 = P, 1 = R, 2 = E
          constexpr bool kRegrouped = DT == TRI_KV_FP8_E4M3 && !IL;   // see compute_step
          if (!mag) {
            const int el = slab_elem<DT>(slab, kb, e);
            if (kRegrouped) { which = e & 1; pair = kb * 16 + 4 * slab + (e >> 1); }
            else if (IL) { which = el & 1; pair = el >> 1; }
            else { which = el >= F ? 1 : 0; pair = el & (F - 1); }
          } else {
            which = 2;
            // interleaved: pairs of slabs 2*set and 2*set + 1; half: real parts of slab `set`
            if (kRegrouped) pair = kb * 16 + 4 * (2 * slab + (e >> 2)) + (e & 3);
            else if (IL) pair = slab_elem<DT>(2 * slab + (e >> 2), kb, 2 * (e & 3)) >> 1;
            else pair = slab_elem<DT>(slab, kb, e) & (F - 1);
          }
          // The magnitudes go through the fp16 matrix-core instruction whatever the key type (see
          // compute_step), so the magnitude slabs are fp16 pieces.
          const bool half_slab = DT == TRI_KV_FP16 || mag;
          v[e] = half_slab ? coefficient_piece<TRI_KV_FP16>(c[which * F + pair], sp)
                           : coefficient_piece<TRI_KV_BF16>(c[which * F + pair], sp);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const f32x2 x = {v[2 * e], v[2 * e + 1]};
          if (DT == TRI_KV_FP16 || mag)
            out[e] = __builtin_bit_cast(uint32_t, __builtin_convertvector(x, f16x2));
          else
            out[e] = __builtin_bit_cast(uint32_t, __builtin_convertvector(x, bf16x2));
        }
      }
      out_base[idx] = uint4{out[0], out[1], out[2], out[3]};
    }
  }
}

// QG: groups of four query heads per KV head (1 or 2).
//
// Rows of an operand are ordered so that one lane's four accumulator values are the pieces of its own head (one group) or
// heads (two): they add up in two or four instructions.  With the tokens as rows and (query head, piece) as columns the
// pieces sat in other lanes, 16 and 14 instructions of row rotations and selections a step; the sums are the same bits.
// By itself that is worth 1.4 % at a head dimension of 64 (24 requests of 1500 to 12001 tokens x 36 layers x 64 query heads
// of 64: 1116 -> 1097 us) and nothing where the key stream or the other tiles are waited for (1 x 32768 tokens x 64 layers x 64
// heads of 128: 832 -> 829; what `publish` and the slack give there stands beside them).
//
// Two groups (five to eight query heads): a second operand set per group of four would leave a quarter of the rows
// empty twice.  Instead the rows are (query head, piece 1 | piece 2) and a second operand holds the third pieces beside
// zeros: two accumulators for all eight heads, added at the end -- (piece 1 + piece 3) + piece 2, every sum in the
// order of one group's.  One accumulator and two pieces of the magnitude coefficients (6 and 12 matrix instructions for 8 and
// 16) have the same error, but round differently: a near-tie then shifts a kept list of 12000.
__device__ __forceinline__ int nsteps_of(int ntok) { return (ntok + 15) >> 4; }

// LDS floats in which the sums of a layer meet (`publish`); none where every wave always publishes its own.
constexpr int meeting_floats(int QG, int W) { return QG == 1 || W == 4 ? W * 128 * QG : 0; }

// W: waves per workgroup.  Eight (one workgroup per CU), or four for models with at most four
// KV heads: a workgroup of eight would leave half its waves without a head and the CU with half
// the loads in flight, so two workgroups of four share a CU (half the LDS each; two waves per
// SIMD either way, which the register budget of 256 is for).
template <int DT, bool IL, int TW, int SL, int QG, int NB, int W, int HD>
__global__ __launch_bounds__(W * kWave) __attribute__((amdgpu_waves_per_eu(2, 2)))
void fused_mfma_kernel(FusedArgs a, const uint4* bmat) {
  static_assert(HD == 128 || ((HD == 64 || HD == 256) && DT != TRI_KV_FP8_E4M3), "head dimensions with a kernel");
  constexpr int NS = HD / 32;            // key slabs per step
  constexpr int NK = QG * NS;            // key operands (MFMAs) of a KV head
  constexpr int NSO = QG * (NS + NS / 2);   // all operands
  static_assert(SL % 16 == 0, "the slack must hold whole steps");
  constexpr int kPart = SL / 16 % NB;    // steps by which the slack of a whole tile exceeds whole rotations
  // Token t of layer l sits at (l * ring_stride + t) % RING, ring_stride the tokens of this launch's tiles (at
  // most TW): what a tile leaves free of the ring is slack, down to SL for a whole tile.
  constexpr int RING = TW + SL;
  constexpr int RQ = 4 * QG;                                   // ring floats per token
  extern __shared__ __align__(16) float lds[];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int b, within;
  if (!locate_workgroup(a, a.HC * a.tiles_per_seq, a.HC, reinterpret_cast<int*>(lds), b, within)) return;
  // Layers of this workgroup: all of them, or one group of a layer-split launch, where `b` so far
  // counts (sequence, group) pairs.
  const int lgroup = b % a.layer_groups;
  b /= a.layer_groups;
  const int l_begin = lgroup * a.layers_per_group;
  const int l_end = min(a.L, l_begin + a.layers_per_group);
  const int chunk = within % a.HC;
  const int tile = within / a.HC;
  const int T = checked_seq_len(a.seq_lens, b, a.Tmax, a.status);
  const int n0 = tile * a.tile_tokens;
  if (n0 >= T) return;
  const int n1 = min(n0 + a.tile_tokens, T);
  const int ntok = n1 - n0;
  const int last_tok = n1 - 1;
  const int seq_tiles = ceil_div(T, a.tile_tokens);
  const int heads_here = min(8, a.Hkv - chunk * 8);

  float* ring = lds + wave * (RING * RQ);                      // [QG][RING][4 query heads]
  float* part = lds + W * (RING * RQ);                         // [waves][16 tokens of a step][RQ query heads][2], where sums meet
  float* stats = part + meeting_floats(QG, W);                 // one group: [2][32 score heads][2]
  uint32_t* ctl = reinterpret_cast<uint32_t*>(stats + (QG == 1 ? 128 : 0));  // claimed, ready, arrived; [8..15]: how far each wave is
  if (threadIdx.x < 16) ctl[threadIdx.x] = 0;
  __syncthreads();
  // From here on the waves of the workgroup run independently.
  if (wave >= heads_here) return;
  const int head = chunk * 8 + wave;

  // MFMA column (token of the step) and k block; kb is the output's row block too: this lane ends up with the step's
  // token j, its score of query head kb (one group) or of the heads 2 kb and 2 kb + 1 (two).
  const int j = lane & 15, kb = lane >> 4;

  // Coefficient slabs of the current layer, the A operands.
  uint4 coef[NSO];
  auto load_coefs = [&](int l) __attribute__((always_inline)) {
    const uint4* p = bmat + (((int64_t)(b * a.L + l) * a.Hkv + head) * NSO) * 64 + lane;
#pragma unroll
    for (int o = 0; o < NSO; ++o) coef[o] = p[o * 64];
    {
      // A coefficient beyond fp16's range (65504) arrives as an infinity: the scores of this
      // launch would be meaningless, so the status word is raised (the caller repeats the
      // step on the vector-unit kernels) and every wait of the launch gives up.  fp16 keys:
      // all slabs; otherwise the magnitude slabs.
      uint32_t bad = 0;
#pragma unroll
      for (int o = (DT == TRI_KV_FP16 ? 0 : NK); o < NSO; ++o) {
        const uint32_t w4[4] = {coef[o].x, coef[o].y, coef[o].z, coef[o].w};
#pragma unroll
        for (int i = 0; i < 4; ++i)
          bad |= (uint32_t)((w4[i] & 0x7c00u) == 0x7c00u) | (uint32_t)((w4[i] & 0x7c000000u) == 0x7c000000u);
      }
      if (__any(bad != 0) && lane == 0) atomicExch(a.status, 2u);
    }
  };

  // A step is 16 consecutive tokens starting at a multiple of 16, so with blocks of at
  // least 16 tokens it lies inside one block: lane i keeps the block of step i of the tile
  // (a tile has at most 64 steps), and a step's block is one v_readlane away.  Dense keys:
  // the "block" is the sequence.
  const bool paged = a.block_table_pitch >= 0;
  int step_blk = b;
  if (paged) {
    const int n = min(n0 + 16 * lane, last_tok);
    step_blk = a.block_table[(int64_t)b * a.block_table_pitch + (n >> a.bs_shift)];
  }
  const int bs_mask = paged ? (1 << a.bs_shift) - 1 : -1;

  // Sixteen tokens of layer l starting at local token t (t % 16 == 0).  The address splits
  // into a wave-uniform base (layer, block, first token of the step, head: scalar unit) and
  // a 32-bit lane offset (row lane % 16 of the step, 16-byte chunk lane / 16); rows past the
  // tile's last token re-read that token (loaded, never stored).
  constexpr bool FP8 = DT == TRI_KV_FP8_E4M3;
  constexpr int ES = FP8 ? 1 : 2;
  const uint32_t tok_bytes = (uint32_t)(a.stride_token * ES);
  const uint32_t lane_row = (uint32_t)j * tok_bytes;
  const uint32_t lane_col = (uint32_t)kb * 16u;
  // fp8: four lanes side by side load the scale of one token, so that sixteen lanes touch one line and not four (every
  // lane its own token's: 8 x 16384 tokens x 32 layers 850 -> 900 us); scale_lane is where the scale of this lane's token is.
  const uint32_t lane_scale_row = (uint32_t)(lane >> 2) * (uint32_t)a.Hkv * 4u;
  const int scale_lane = 16 * j;
  struct LayerBase { const char* k; const char* scale; };   // of this wave's head (scalar registers)
  auto layer_base = [&](int l) __attribute__((always_inline)) {
    LayerBase lb;
    lb.k = table_entry(a.k_layers, l) + (int64_t)head * a.stride_head * ES;
    lb.scale = nullptr;
    if constexpr (FP8)
      lb.scale = table_entry(reinterpret_cast<const void* const*>(a.k_scale_layers), l) + head * 4;
    return lb;
  };
  // The address arithmetic of a step is done once per tile: lane i keeps the byte offset of step i's first
  // row from the head's base (the same in every layer) and, for one-byte keys, the index of its first token
  // slot.  (Per step it is 25 scalar instructions in the path of every wave; with one-byte keys, eight step
  // buffers and a scale per row, the compiler kept its operands in lanes of a vector register on top.)
  uint32_t step_off_lo, step_off_hi;
  int step_slot = 0;
  {
    const int nt = min(n0 + 16 * lane, (nsteps_of(ntok) - 1) * 16 + n0);
    const int in_blk = nt & bs_mask;
    const int64_t off = ((int64_t)step_blk * a.stride_block + (int64_t)in_blk * a.stride_token) * ES;
    step_off_lo = (uint32_t)off;
    step_off_hi = (uint32_t)((uint64_t)off >> 32);
    if constexpr (FP8) step_slot = step_blk * a.block_size + in_blk;
  }
  auto load_step = [&](StepData<DT, HD>& d, const LayerBase& lb, int t) __attribute__((always_inline)) {
    const int step = t >> 4;
    const uint32_t rows_left = (uint32_t)(last_tok - (n0 + t));
    const uint64_t row_off = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)step_off_hi, step) << 32) |
                             (uint32_t)__builtin_amdgcn_readlane((int)step_off_lo, step);
    const char* base = reinterpret_cast<const char*>(uniform_ptr(lb.k + row_off));
    const uint32_t off = min(lane_row, rows_left * tok_bytes) + lane_col;
    GlobalBytes p = (GlobalBytes)(uintptr_t)base + off;
#pragma unroll
    for (int s = 0; s < (FP8 ? 2 : NS); ++s) {
      const u32x4 v = *(GlobalU4)(p + s * 64);
      d.c[s] = uint4{v.x, v.y, v.z, v.w};
    }
    if constexpr (FP8) {
      const uint32_t hkv4 = (uint32_t)a.Hkv * 4u;
      const uint64_t slot_off = (uint64_t)(uint32_t)__builtin_amdgcn_readlane(step_slot, step) * hkv4;
      const char* sc = reinterpret_cast<const char*>(uniform_ptr(lb.scale + slot_off));
      d.scale = *(GlobalF32)((GlobalBytes)(uintptr_t)sc + min(lane_scale_row, rows_left * hkv4));
    }
  };

  // Ring of this wave: [group of four query heads][RING tokens][4], so that the 16-byte reads of consecutive
  // tokens are 16 bytes apart, whatever the number of groups.  With one group the 64 lanes of a store (16 tokens x
  // 4 heads) cover 64 consecutive words; with two a lane's pair of heads is one 8-byte store, and either half of the
  // wave covers 64 consecutive words of its group.
  const uint32_t lane_ring = QG == 1 ? (uint32_t)(4 * j + kb) : (uint32_t)(kb >> 1) * (RING * 4) + (uint32_t)(4 * j + 2 * (kb & 1));
  float s1[QG] = {}, s2[QG] = {};       // sums of this lane's i-th head over the steps
  // Largest of a sample of the layer's magnitudes (their first fp16 pieces), per lane; see the check
  // after every layer.
  f16x2 mag_seen = {(_Float16)0.f, (_Float16)0.f};
  // Scores of the 16 tokens of a step: MFMAs over keys and magnitudes, then the pieces of a head, which are rows of
  // one lane's accumulator, are added.
  auto compute_step = [&](const StepData<DT, HD>& raw, float scale, int l, int t, int which) __attribute__((always_inline)) {
    // The keys of the step, the B operands of its MFMAs, as dwords (two elements each): the loaded
    // registers for bf16 keys, one conversion per dword (exact) for fp8 keys.
    uint32_t w[NS][4];
    // One-byte keys in the half-split layout: lane block kb holds the real parts of pairs
    // 16*kb .. 16*kb + 15 in c[0] and their imaginary parts in c[1].  Two byte permutes per
    // dword pair put (real, imaginary) next to each other before the conversion, so every
    // converted dword is a pair: operand s holds pairs 16*kb + 4*s .. + 3, the magnitudes need
    // no regrouping (8 permutes per step instead of 16 after the conversion), and the
    // coefficient slabs are laid out to match.
    constexpr bool kRegrouped = FP8 && !IL;
    if constexpr (kRegrouped) {
      const uint32_t re[4] = {raw.c[0].x, raw.c[0].y, raw.c[0].z, raw.c[0].w};
      const uint32_t im[4] = {raw.c[1].x, raw.c[1].y, raw.c[1].z, raw.c[1].w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t lo = __builtin_amdgcn_perm(im[i], re[i], 0x05010400u);   // (re0, im0, re1, im1)
        const uint32_t hi = __builtin_amdgcn_perm(im[i], re[i], 0x07030602u);   // (re2, im2, re3, im3)
        w[i][0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 1.0f, false));
        w[i][1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 1.0f, true));
        w[i][2] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 1.0f, false));
        w[i][3] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 1.0f, true));
      }
    } else if constexpr (FP8) {
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const uint32_t r[4] = {raw.c[s].x, raw.c[s].y, raw.c[s].z, raw.c[s].w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          uint32_t* o = &w[2 * s + (i >> 1)][(i & 1) * 2];
          o[0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(r[i], 1.0f, false));
          o[1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(r[i], 1.0f, true));
        }
      }
    } else {
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        w[s][0] = raw.c[s].x; w[s][1] = raw.c[s].y; w[s][2] = raw.c[s].z; w[s][3] = raw.c[s].w;
      }
    }
    struct { uint4 c[NS]; } d;
#pragma unroll
    for (int s = 0; s < NS; ++s) d.c[s] = uint4{w[s][0], w[s][1], w[s][2], w[s][3]};
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < NS; ++s) acc = mfma_16x16x32<DT>(coef[s], d.c[s], acc);
    f32x4 acc3 = {0.f, 0.f, 0.f, 0.f};
    if constexpr (QG == 2) {
#pragma unroll
      for (int s = 0; s < NS; ++s) acc3 = mfma_16x16x32<DT>(coef[NS + s], d.c[s], acc3);
    }
#pragma unroll
    for (int set = 0; set < NS / 2; ++set) {
      // |k_f|^2 = k_r^2 + k_i^2 straight from the bf16 pairs (v_dot2_f32_bf16).
      // interleaved: dword e % 4 of operand 2*set + e/4 is the (real, imaginary) pair;
      // half: real parts in operand `set`, imaginary parts in operand `set + 2`, regrouped
      // into (real, imaginary) dwords by two byte permutes per dword.
      float mag[8];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        uint32_t x[4];
        if constexpr (IL || kRegrouped) {
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
      uint4 hi, lo;
      // The magnitudes are cut into two fp16 pieces (22 bits; two bf16 pieces would carry 16) and
      // go through the fp16 matrix-core instruction whatever the key type: the fp16 split is two
      // instructions per pair cheaper than the bf16 one.  Magnitudes of one-byte codes lie in
      // [2^-9, 634]; a two-byte key beyond fp16's range turns its scores into infinities or NaNs,
      // which the check after every layer finds (status word 2: the caller repeats the step on the
      // vector-unit kernels).
      split8_f16(mag, hi, lo);
      if constexpr (!FP8)   // `which` is the step buffer's number: a constant after unrolling
        mag_seen = pk_max_f16(mag_seen, (&hi.x)[which & 3]);
      constexpr int MT = TRI_KV_FP16;                // operand type of the magnitude MFMAs
      acc = mfma_16x16x32<MT>(coef[NK + set], hi, acc);
      acc = mfma_16x16x32<MT>(coef[NK + set], lo, acc);
      if constexpr (QG == 2) {
        acc3 = mfma_16x16x32<MT>(coef[NK + NS / 2 + set], hi, acc3);
        acc3 = mfma_16x16x32<MT>(coef[NK + NS / 2 + set], lo, acc3);
      }
    }
    // v[i]: the score of this lane's token and its i-th head.
    float v[QG];
    if constexpr (QG == 1) {
      v[0] = (acc[0] + acc[2]) + acc[1];
    } else {
      v[0] = (acc[0] + acc3[0]) + acc[1];
      v[1] = (acc[2] + acc3[2]) + acc[3];
    }
    // first ring slot of the step (scalar; a step never straddles the wrap: t and RING are
    // multiples of 16).  The ring has a place for every row of the step and every head slot: rows past the
    // tile's last token and slots beyond the last query head (zero rows) are written too and never read.
    const uint32_t slot0 = (uint32_t)(l * a.ring_stride + t) % RING;
    if (t + 16 > ntok) {                              // (wave-uniform: the last step of a tile)
      asm volatile("");
#pragma unroll
      for (int i = 0; i < QG; ++i)
        if (t + j >= ntok) v[i] = 0.f;
    }
    float score[QG];
#pragma unroll
    for (int i = 0; i < QG; ++i) {
      score[i] = FP8 ? v[i] * scale : v[i];
      s1[i] = FP8 ? fmaf(v[i], scale, s1[i]) : s1[i] + v[i];
      s2[i] = fmaf(score[i], score[i], s2[i]);
    }
    float* entry = ring + slot0 * 4 + lane_ring;
    if constexpr (QG == 1) *entry = score[0];
    else *reinterpret_cast<float2*>(entry) = float2{score[0], score[1]};
  };

  bool aborted = false;
  uint32_t* claimed = ctl;
  uint32_t* ready = ctl + 1;
  uint32_t* arrived = ctl + 2;
  const int items = heads_here * a.G * 2;        // (score head, sum | sum of squares) of this workgroup
  const int ah0 = chunk * 8 * a.G;

  // Publish this wave's sums of layer l.  The sixteen lanes of a row group hold a head's sums over the tokens that share
  // a place in the step; the lane of each of the head's two words adds them in token order.
  //
  // Two groups, eight waves: every wave publishes its own, through the ring slots of the next layer's first two steps (free:
  // of the layer before nothing is left in the ring), which the sums are stored to as scores are.  So a head's words are on
  // their way as soon as its wave is through, where meeting in LDS lets every head wait for the slowest wave of every tile.
  // 1 x 32768 tokens x 64 layers, 64 / 8 heads of 128, both with 64 tokens of slack: 829 -> 783 us; 40, 48, 56 / 8 heads gain
  // as much (with 112: 849 -> 800, 849 -> 793, 854 -> 804).
  //
  // Meeting in LDS, where the last wave of the workgroup adds and publishes all of them:
  //  - One group: one wave fetches the statistics of all heads, so nothing is won by a head that comes early (16 x 16384
  //    tokens x 36 layers 3135 us, 3142 with a publication per wave).
  //  - Two groups, four waves, fewer than eight query heads: a wave's words end inside a 128-byte line that the next
  //    head's wave, and the next tile's workgroup, write too.  24 requests of 2500 to 11000 tokens x 28 layers, us with a
  //    publication per wave | meeting: 898 | 856 for 20 / 4 heads of 128, 923 | 886 for 24 / 4, 935 | 896 for 28 / 4 (the former
  //    with 112 tokens of slack; with 64 no better), but 688 | 691 for 32 / 4 (8 x 16384 tokens, both with 64), whose waves
  //    publish whole lines; heads of 64 (16 x 16384 x 36) 1000 | 943 for 20 / 4, 896 | 916 for 32 / 4.  Padding every wave's
  //    words to a line takes 934 to 908 only, and scratch.
  // Every wave deposits layer l before any deposits layer l + 1 (the last one to arrive has added by the time any wave gets
  // past consuming layer l), so the counter never mixes layers.
  auto publish = [&](int l) __attribute__((always_inline)) {
    if (QG == 1 || (W == 4 && a.G < RQ)) {
      float* mine = part + ((wave * 16 + j) * RQ + kb * QG) * 2;
#pragma unroll
      for (int i = 0; i < QG; ++i) {
        mine[2 * i] = s1[i];
        mine[2 * i + 1] = s2[i];
        s1[i] = s2[i] = 0.f;
      }
      uint32_t prev = 0;
      if (lane == 0) prev = __hip_atomic_fetch_add(arrived, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_WORKGROUP);
      prev = __builtin_amdgcn_readfirstlane(prev);
      if (prev + 1 != (uint32_t)(l - l_begin + 1) * (uint32_t)heads_here) return;
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
      unsigned long long* out = a.xchg + (((int64_t)(b * a.L + l) * a.tiles_per_seq + tile) * a.A + ah0) * 2;
      if (lane < items) {                            // (at most 64: eight waves of four heads, four of seven)
        const int ahl = lane >> 1, w = ahl / a.G, qq = ahl - w * a.G;
        float t = 0.f;
        for (int i = 0; i < 16; ++i) t += part[((w * 16 + i) * RQ + qq) * 2 + (lane & 1)];     // in token order
        xchg_store(out + lane, ((unsigned long long)(uint32_t)(l + 1) << 32) | __float_as_uint(t));
      }
      return;
    }
    const uint32_t slot1 = (uint32_t)((l + 1) * a.ring_stride) % RING, slot2 = (uint32_t)((l + 1) * a.ring_stride + 16) % RING;
    *reinterpret_cast<float2*>(ring + slot1 * 4 + lane_ring) = float2{s1[0], s1[QG - 1]};
    *reinterpret_cast<float2*>(ring + slot2 * 4 + lane_ring) = float2{s2[0], s2[QG - 1]};
#pragma unroll
    for (int i = 0; i < QG; ++i) { s1[i] = 0.f; s2[i] = 0.f; }
    order_lds_of_wave();
    const int qq = lane >> 1, which = lane & 1;                 // lane: (query head, sum | sum of squares)
    if (qq < a.G) {
      const float* p = ring + (qq >> 2) * (RING * 4) + (which ? slot2 : slot1) * 4 + (qq & 3);
      float t = 0.f;
#pragma unroll
      for (int i = 0; i < 16; ++i) t += p[4 * i];
      xchg_store(a.xchg + (((int64_t)(b * a.L + l) * a.tiles_per_seq + tile) * a.A + ah0 + wave * a.G) * 2 + lane,
                 ((unsigned long long)(uint32_t)(l + 1) << 32) | __float_as_uint(t));
    }
    order_lds_of_wave();      // (the next layer's first steps go to the same slots)
  };

  float fin[TW / 64];
#pragma unroll
  for (int k = 0; k < TW / 64; ++k) fin[k] = 0.f;
  const int prefill = (a.protect_prefill && a.prefill_lens) ? a.prefill_lens[b] : 0;
  const int window_from = a.window_size > 0 ? T - min(a.window_size, T) : T;

  // Turn layer l's ring entries into selection-score contributions (lane = token).
  auto consume = [&](int l) __attribute__((always_inline)) {
    float mean[RQ], sd[RQ];
#pragma unroll
    for (int qq = 0; qq < RQ; ++qq) { mean[qq] = 0.f; sd[qq] = 1.f; }
    if (a.normalize) {
      if constexpr (QG == 2) {
        // More than four query heads per KV head: twice the words per tile and tiles half as long,
        // so the gather is four times the work; every wave fetches the words of its own KV head
        // (8 x 32768 tokens x 64 layers, 64 query heads: 7.55 -> 6.82 ms).  With up to four query
        // heads the one wave's gather below hides behind the slack and this form is slower (16 x 16384
        // tokens x 36 layers: 3.29 -> 3.30 ms; fp8 keys 1.72 -> 1.80; 16 x 2176 tokens 0.54 -> 0.62).
        gather_head_stats(a, b, l, seq_tiles, T, (chunk * 8 + wave) * a.G, a.G, mean, sd, lane, aborted);
      } else {
      uint32_t won = 0;
      if (lane == 0) {
        uint32_t expect = (uint32_t)(l - l_begin);
        won = __hip_atomic_compare_exchange_strong(claimed, &expect, (uint32_t)(l - l_begin + 1), __ATOMIC_ACQ_REL,
                                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) ? 1u : 0u;
      }
      won = __builtin_amdgcn_readfirstlane(won);
      if (won) {
        gather_layer_stats(a, b, l, seq_tiles, T, ah0, items, stats + (l & 1) * 64, lane, aborted);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        if (lane == 0)
          __hip_atomic_store(ready, (uint32_t)(l - l_begin + 1), __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
      } else {
        // The claiming wave always finishes (its own waits are bounded).
        while (__hip_atomic_load(ready, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP) < (uint32_t)(l - l_begin + 1))
          __builtin_amdgcn_s_sleep(2);
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
      const float* st = stats + (l & 1) * 64;
#pragma unroll
      for (int qq = 0; qq < RQ; ++qq)
        if (qq < a.G) {
          mean[qq] = st[(wave * a.G + qq) * 2];
          // One division per head and layer; the tokens multiply by the reciprocal (a
          // division per score costs ten vector instructions, 7 % of the kernel's total).
          sd[qq] = __fdiv_rn(1.f, st[(wave * a.G + qq) * 2 + 1]);
        }
      }
    }
    // The usual mode -- every query-head slot of the group in use, maximum over the group, running sum
    // over layers, not the first layer -- without the per-head predicates, the
    // two reduction variants, the lane masks and the modulo per token of the general loop below: a third
    // of its instructions.  (Lanes past the tile's last token take whatever the ring holds there into a sum that
    // nobody reads.)  The guards need no attention here: the first layer of a workgroup goes
    // through the general loop, which sets the guarded tokens to +inf, and a finite contribution leaves
    // them there.  This piece of work sits on every wave's path once per layer (removed altogether, for
    // timing only, it is worth 3.4 % of the kernel on 16 x 16384 tokens x 36 layers, 4.2 % with eight
    // query heads per KV head).
    if (a.G == RQ && a.group_reduce == TRI_REDUCE_MAX && a.layer_reduce == TRI_REDUCE_MEAN && l != l_begin) {
      // This lane's entry of chunk 0 inside the wave's ring; chunk k lies 64 k entries further on, or
      // RING entries back once that passes the ring's end (one compare and one select per chunk, the
      // distance itself goes into the LDS instruction's offset field).
      const uint32_t lane_pos = (uint32_t)(l * a.ring_stride) % RING + (uint32_t)lane;          // below 2 * RING
      uint32_t at = lane_pos * 4, at_wrapped = (lane_pos - RING) * 4;               // in floats
      asm volatile("" : "+v"(at), "+v"(at_wrapped));     // (keeps both in vector registers)
      struct Entry { float4 x[QG]; };
      auto entry = [&](int k) __attribute__((always_inline)) {
        const uint32_t p = (lane_pos >= (uint32_t)(RING - 64 * k)) ? at_wrapped : at;
        Entry e;
#pragma unroll
        for (int g = 0; g < QG; ++g)
          e.x[g] = *reinterpret_cast<const float4*>(ring + p + (64 * 4 * k + g * (RING * 4)));
        return e;
      };
      auto contribution = [&](const Entry& e) __attribute__((always_inline)) {
        float z[RQ];
#pragma unroll
        for (int g = 0; g < QG; ++g) {
          z[4 * g] = __fmul_rn(__fsub_rn(e.x[g].x, mean[4 * g]), sd[4 * g]);
          z[4 * g + 1] = __fmul_rn(__fsub_rn(e.x[g].y, mean[4 * g + 1]), sd[4 * g + 1]);
          z[4 * g + 2] = __fmul_rn(__fsub_rn(e.x[g].z, mean[4 * g + 2]), sd[4 * g + 2]);
          z[4 * g + 3] = __fmul_rn(__fsub_rn(e.x[g].w, mean[4 * g + 3]), sd[4 * g + 3]);
        }
        float v = max3(z[0], z[1], z[2]);
#pragma unroll
        for (int qq = 3; qq + 1 < RQ; qq += 2) v = max3(v, z[qq], z[qq + 1]);
        return max3(v, z[RQ - 1], z[RQ - 1]);
      };
      if (ntok == TW) {
        // a whole tile: straight-line code, the ring entries of four chunks requested before the first is used
        constexpr int kAhead = QG == 1 ? 4 : 2;
#pragma unroll
        for (int k0 = 0; k0 < TW / 64; k0 += kAhead) {
          Entry e[kAhead];
#pragma unroll
          for (int i = 0; i < kAhead; ++i) e[i] = entry(k0 + i);
#pragma unroll
          for (int i = 0; i < kAhead; ++i) fin[k0 + i] = __fadd_rn(fin[k0 + i], contribution(e[i]));
        }
      } else {
#pragma unroll
        for (int k = 0; k < TW / 64; ++k)
          if (64 * k < ntok) fin[k] = __fadd_rn(fin[k], contribution(entry(k)));            // (wave-uniform)
      }
      return;
    }
#pragma unroll
    for (int k = 0; k < TW / 64; ++k) {
      const int tl = lane + 64 * k;
      if (tl >= ntok) continue;
      float xs[RQ];
#pragma unroll
      for (int g = 0; g < QG; ++g) {
        const float4 x = *reinterpret_cast<const float4*>(&ring[(uint32_t)g * (RING * 4) + ((uint32_t)(l * a.ring_stride + tl) % RING) * 4]);
        xs[4 * g] = x.x; xs[4 * g + 1] = x.y; xs[4 * g + 2] = x.z; xs[4 * g + 3] = x.w;
      }
      float v;
      if (a.group_reduce == TRI_REDUCE_MAX) {
        v = -INFINITY;
#pragma unroll
        for (int qq = 0; qq < RQ; ++qq)
          if (qq < a.G) v = fmaxf(v, __fmul_rn(__fsub_rn(xs[qq], mean[qq]), sd[qq]));
      } else {
        v = 0.f;
#pragma unroll
        for (int qq = 0; qq < RQ; ++qq)
          if (qq < a.G) v = __fadd_rn(v, __fmul_rn(__fsub_rn(xs[qq], mean[qq]), sd[qq]));
        v = __fdiv_rn(v, (float)a.G);
      }
      const int n = n0 + tl;
      if (n >= window_from || n < prefill) v = INFINITY;
      if (l == l_begin) fin[k] = v;
      else fin[k] = (a.layer_reduce == TRI_REDUCE_MAX) ? fmaxf(fin[k], v) : __fadd_rn(fin[k], v);
    }
  };

  // ---- one continuous stream of key rows over (layer, step of 16 tokens).  NB step
  // buffers rotate (four of 64 bytes per lane, or eight of 36 for one-byte keys, which keeps
  // the same number of bytes in flight); a buffer is refilled as soon as it has been scored,
  // with the step NB ahead.  A layer is padded to whole rotations (padding steps re-read the
  // last row and are not scored), so the loads of a layer's last rotation are exactly the
  // first NB steps of the next layer; the rotations form inner loops that contain nothing
  // but key loads and scoring, and the work at layer boundaries sits between them (where the slack is no whole number of
  // rotations, one of them is cut in two around the consumption of the layer before).
  const int nsteps = (ntok + 15) >> 4;
  const int rotations = (nsteps + NB - 1) / NB;
  // How far a layer is scored before the layer before it is turned into contributions (a part of a rotation can only lie
  // inside one).
  const int rot_before_consume = kPart ? min(((RING - a.ring_stride) / 16 - kPart) / NB, rotations - 1)
                                       : min((RING - a.ring_stride) / (16 * NB), rotations);
  auto score = [&](const StepData<DT, HD>& d, int l, int slot, int which) __attribute__((always_inline)) {
    // One-byte keys: the scale of this lane's token, from the lane that loaded it (requested in front of the branch, or
    // the compiler asks for it where it is used and waits there).
    float scale = 1.f;
    if constexpr (FP8) scale = __int_as_float(__builtin_amdgcn_ds_bpermute(scale_lane, __float_as_int(d.scale)));
    if (slot < nsteps) compute_step(d, scale, l, slot * 16, which);
  };
  StepData<DT, HD> buf[NB];
  LayerBase base_cur = layer_base(l_begin), base_next = base_cur;
  // The two waves of a SIMD (waves i and i + 4 of a workgroup of eight) compete for its issue slots and
  // the arbiter prefers the older one: left alone, waves 0..3 of every workgroup run ahead, then wait at
  // the next layer's statistics for waves 4..7 of every tile, and the SIMD is half empty meanwhile (with
  // eight query heads per KV head waves 0..3 spent 18 % of their time in that wait, waves 4..7 11 %).
  // So each wave posts how far it is at every rotation and takes the higher priority while it is behind
  // its neighbour (8 x 32768 tokens x 64 layers 6.55 -> 6.48 ms, one-byte keys 1.70 -> 1.63 ms).
  uint32_t* progress = ctl + 8;
  auto balance = [&](int l, int r) __attribute__((always_inline)) {
    if constexpr (W == 8) {
      const uint32_t mine = (uint32_t)((l - l_begin) * rotations + r);
      if (lane == 0) __hip_atomic_store(progress + wave, mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      const uint32_t other = (uint32_t)__builtin_amdgcn_readfirstlane(
          (int)__hip_atomic_load(progress + (wave ^ 4), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
      if (mine < other) __builtin_amdgcn_s_setprio(2);
      else __builtin_amdgcn_s_setprio(0);
    }
  };
  // Steps from .. to - 1 of rotation r (constants: every buffer has its registers).
  auto steps = [&](int l, int r, auto from, auto to) __attribute__((always_inline)) {
    const bool wrap = r + 1 >= rotations;
    const LayerBase lb = {wrap ? base_next.k : base_cur.k, wrap ? base_next.scale : base_cur.scale};
    const int s0 = wrap ? 0 : (r + 1) * NB;
#pragma unroll
    for (int i = decltype(from)::value; i < decltype(to)::value; ++i) {
      score(buf[i], l, r * NB + i, i);
      load_step(buf[i], lb, min(s0 + i, nsteps - 1) * 16);
    }
  };
  constexpr std::integral_constant<int, 0> kFirst{};
  constexpr std::integral_constant<int, kPart> kMiddle{};
  constexpr std::integral_constant<int, NB> kLast{};
  auto rotate = [&](int l, int r0, int r1) __attribute__((always_inline)) {
    for (int r = r0; r < r1; ++r) {
      balance(l, r);
      steps(l, r, kFirst, kLast);
    }
  };
  auto settle = [&]() __attribute__((always_inline)) { __builtin_amdgcn_s_waitcnt(0x0F70); };

  load_coefs(l_begin);
#pragma unroll
  for (int i = 0; i < NB; ++i) load_step(buf[i], base_cur, min(i, nsteps - 1) * 16);
  for (int l = l_begin; l < l_end; ++l) {
    base_cur = base_next;
    base_next = layer_base(min(l + 1, l_end - 1));
    settle();
    rotate(l, 0, rot_before_consume);
    if constexpr (kPart != 0) {
      balance(l, rot_before_consume);
      steps(l, rot_before_consume, kFirst, kMiddle);
    }
    if (l > l_begin) {
      order_lds_of_wave();
      consume(l - 1);
      order_lds_of_wave();
    }
    if constexpr (kPart != 0) steps(l, rot_before_consume, kMiddle, kLast);
    rotate(l, rot_before_consume + (kPart != 0), rotations);
    if constexpr (!FP8) {
      // A magnitude beyond fp16's range (or a key that is not finite) has left an infinity or a NaN
      // in this layer's sums.
      bool bad = false;
#pragma unroll
      for (int i = 0; i < QG; ++i) bad = bad || !(s2[i] < INFINITY);
      // The other end of fp16's range: below 2^-14 the first piece is a subnormal and below 2^-3 the
      // second one is, so magnitudes carry an absolute error of up to 2^-25 whatever their size.
      // Against keys of ordinary size that is nothing (scaled by 2^-10, magnitudes around 2^-9, the
      // selection scores are as close to the fp64 ones as unscaled); keys that are all tiny (scaled by
      // 2^-14: errors of 2e-4 of the largest score) are left to the other kernels: no lane of the
      // wave has seen a magnitude of 2^-9 in this layer (of every step one pair in four is looked at,
      // another one in each of the step buffers, so every frequency pair is among them).
      const bool seen = (float)mag_seen[0] >= 0x1p-9f || (float)mag_seen[1] >= 0x1p-9f;
      mag_seen = f16x2{(_Float16)0.f, (_Float16)0.f};
      if ((__any(bad) || !__any(seen)) && lane == 0) atomicExch(a.status, 2u);
    }
    if (a.normalize) publish(l);
    if (l + 1 < l_end) load_coefs(l + 1);
  }
  order_lds_of_wave();
  consume(l_end - 1);

  if (a.layer_groups > 1) {
    // This group's sum (or maximum) over its layers; fused_layer_reduce_kernel combines the groups.
    const int64_t rows = (int64_t)(a.num_seqs / a.layer_groups) * a.Hkv;
    float* out = a.fin_part + (((int64_t)lgroup * rows + (int64_t)b * a.Hkv + head) * a.Tmax) + n0;
#pragma unroll
    for (int k = 0; k < TW / 64; ++k) {
      const int tl = lane + 64 * k;
      if (tl < ntok) out[tl] = fin[k];
    }
    return;
  }
  float* out = a.fin + ((int64_t)b * a.Hkv + head) * a.Tmax + n0;
#pragma unroll
  for (int k = 0; k < TW / 64; ++k) {
    const int tl = lane + 64 * k;
    if (tl < ntok) out[tl] = (a.layer_reduce == TRI_REDUCE_MEAN) ? __fdiv_rn(fin[k], (float)a.L) : fin[k];
  }
}

// How a batch is cut into launches (from the plan).
struct LaunchShape {
  int seqs_per_launch;   // whole sequences of maximum length one launch holds
  int resident;          // workgroups the device holds at once
  int num_seqs;
  int launches;          // > 0: exactly this many (the planner replayed the device's packing); 0: the worst case
};

template <int TW, int SL, int QG, int W>
constexpr size_t mfma_lds_bytes() {
  return ((size_t)W * (TW + SL) * 4 * QG + meeting_floats(QG, W) + (QG == 1 ? 128 : 0) + 16) * 4;
}

template <int DT, bool IL, int TW, int SL, int QG, int NB, int W = kFusedWaves, int HD = 128>
hipError_t launch_mfma_t(FusedArgs& k, const uint4* bmat, const LaunchShape& shape, hipStream_t s) {
  const int seqs_per_launch = shape.seqs_per_launch, resident = shape.resident, B = shape.num_seqs;
  const int known_launches = shape.launches;
  constexpr size_t lds = mfma_lds_bytes<TW, SL, QG, W>();
  // 8 waves: one workgroup per CU; 4 waves: two (LDS is handed out in blocks of 1280 bytes).
  static_assert(((lds + 1279) / 1280 * 1280) * (kFusedWaves / W) <= (size_t)kFusedLdsLimit, "LDS of a CU");
  const void* fn = reinterpret_cast<const void*>(&fused_mfma_kernel<DT, IL, TW, SL, QG, NB, W, HD>);
  hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return e;
  if (B <= seqs_per_launch) {
    k.packed = 0;
    k.seq_base = 0;
    const int n = B * k.layer_groups;      // (sequence, layer group) pairs; k.num_seqs counts the same
    hipLaunchKernelGGL((fused_mfma_kernel<DT, IL, TW, SL, QG, NB, W, HD>), dim3(n * k.tiles_per_seq * k.HC), dim3(W * kWave), lds, s, k, bmat);
    return hipGetLastError();
  }
  if (k.layer_groups != 1) return hipErrorInvalidValue;   // layer groups exist in single launches only
  // More workgroups than the device holds at once: whole sequences are packed into
  // launches on the device (the host does not know the individual lengths); the host
  // issues as many launches as the worst case needs, surplus ones find no work.
  k.packed = 1;
  const int launches = known_launches > 0 ? known_launches : ceil_div(B, seqs_per_launch);
  hipLaunchKernelGGL(fused_pack_kernel, dim3(1), dim3(256), 0, s, k.seq_lens, B, k.tile_tokens, k.HC, resident,
                     const_cast<int32_t*>(k.seq_launch), const_cast<int32_t*>(k.seq_wg_base), launches, k.Tmax,
                     k.status);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  for (int i = 0; i < launches; ++i) {
    k.launch_idx = i;
    hipLaunchKernelGGL((fused_mfma_kernel<DT, IL, TW, SL, QG, NB, W, HD>), dim3(resident), dim3(W * kWave), lds, s, k, bmat);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace

// Does the current device hold one resident workgroup per CU?  Asked once per device of the
// runtime's occupancy calculator, for the instance with the largest ring (1024 + 192 tokens, eight
// waves, 256 registers a lane): a part with less LDS per CU, or a runtime that gives the kernel
// fewer resources than this file assumes, then takes the two-pass kernels instead of launching
// workgroups that would wait for others that cannot start.
bool fused_mfma_fits_device() {
  const void* fn = reinterpret_cast<const void*>(&fused_mfma_kernel<TRI_KV_BF16, false, 1024, 192, 1, 4, kFusedWaves, 128>);
  constexpr size_t lds = mfma_lds_bytes<1024, 192, 1, kFusedWaves>();
  if (hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  int per_cu = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, kFusedWaves * kWave, lds) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return per_cu >= 1;
}

namespace {

template <int DT, bool IL>
hipError_t launch_mfma_tw(FusedArgs& k, const uint4* bmat, int tw, int waves, int head_dim, const LaunchShape& shape,
                          hipStream_t s) {
  if (head_dim == 256) {
    // Twice the bytes per row: two step buffers hold as many bytes as four do for 128.
    if constexpr (DT != TRI_KV_FP8_E4M3) {
      if (k.G > 4) {
        if (tw != 512) return hipErrorInvalidValue;
        return waves == 4 ? launch_mfma_t<DT, IL, 512, 64, 2, 2, 4, 256>(k, bmat, shape, s)
                          : launch_mfma_t<DT, IL, 512, 64, 2, 2, 8, 256>(k, bmat, shape, s);
      }
      if (tw != 1024) return hipErrorInvalidValue;
      return waves == 4 ? launch_mfma_t<DT, IL, 1024, 128, 1, 2, 4, 256>(k, bmat, shape, s)
                        : launch_mfma_t<DT, IL, 1024, 192, 1, 2, 8, 256>(k, bmat, shape, s);
    }
    return hipErrorInvalidValue;
  }
  if (head_dim == 64) {
    // Half the bytes per row: eight step buffers keep as many bytes in flight (four query heads
    // per KV head; with eight, eight buffers are slower: 24 requests of 1500 to 12001 tokens x 36 layers 1181 us, with four
    // 1087).  One instance per shape, with the largest ring.
    if constexpr (DT != TRI_KV_FP8_E4M3) {
      if (k.G > 4) {
        if (tw != 512) return hipErrorInvalidValue;
        return waves == 4 ? launch_mfma_t<DT, IL, 512, 64, 2, 4, 4, 64>(k, bmat, shape, s)
                          : launch_mfma_t<DT, IL, 512, 64, 2, 4, 8, 64>(k, bmat, shape, s);
      }
      if (tw != 1024) return hipErrorInvalidValue;
      return waves == 4 ? launch_mfma_t<DT, IL, 1024, 128, 1, 8, 4, 64>(k, bmat, shape, s)
                        : launch_mfma_t<DT, IL, 1024, 128, 1, 8, 8, 64>(k, bmat, shape, s);
    }
    return hipErrorInvalidValue;
  }
  if (waves == 4) {
    // Two workgroups per CU: the ring of the largest tile with one rotation of slack less
    // (a smaller tile is a run-time argument inside it).  Five to eight query heads: the 80 tokens that LDS has
    // beside the ring and the sums (28 / 4 heads, 8 x 16384 tokens x 28 layers, bf16: 685 us, with 64 691; 1 x 32768
    // 235 and 236; 3 x 5001 116.0 and 117.5).
    constexpr int NB4 = DT == TRI_KV_FP8_E4M3 ? 8 : 4;
    if (k.G > 4) return tw == 512 ? launch_mfma_t<DT, IL, 512, 80, 2, 4, 4>(k, bmat, shape, s)
                                  : hipErrorInvalidValue;
    return tw == 1024 ? launch_mfma_t<DT, IL, 1024, 128, 1, NB4, 4>(k, bmat, shape, s)
                      : hipErrorInvalidValue;
  }
  if (k.G > 4) {
    // Five to eight query heads per KV head: 32 bytes of ring per token, and slack is what LDS has least of.  Tiles of up to 512:
    // 112 tokens, all there is, in place of 64 (both with `publish` per wave, 64 layers, 64 / 8 heads: 1 x 32768 tokens 783 ->
    // 770 us, 4 x 16384 1460 -> 1445, 13 of 2100 to 8000 2035 -> 2026; one-byte keys the same within 0.6 %: 8 x 16384 1913 and
    // 1925, 1 x 32768 505 and 507).  Tiles of up to 256: 320 tokens, whole rotations and more than a tile; with 368, all there
    // is, a layer would be consumed a step before its end and the code hold a third copy of the steps (5 x 13056 tokens x 64
    // layers 1517 us with 368, 1513 with 320, one-byte keys 1150 and 1121; 17 x 3840 x 64 one-byte keys 1126 and 1113).  Head dimension 64 has whole rotations too: 1087 us with 64 tokens, 1103 with 112 (24 requests of
    // 1500 to 12001 x 36 layers).
    switch (tw) {
      case 512: return launch_mfma_t<DT, IL, 512, 112, 2, 4>(k, bmat, shape, s);
      case 256: return launch_mfma_t<DT, IL, 256, 320, 2, 4>(k, bmat, shape, s);
      default: return hipErrorInvalidValue;
    }
  }
  // One-byte keys: eight step buffers.
  constexpr int NB = DT == TRI_KV_FP8_E4M3 ? 8 : 4;
  // Slack: as much as LDS allows beside the ring of a 1024-token tile, in whole rotations
  // (16 x 16384 tokens x 36 layers, bf16, warm GPU: 3.54 ms with 64, 3.49 with 128, 3.45 with 192).
  // The instances of shorter tiles keep the same ring (one workgroup has the CU's LDS to itself).
  constexpr int SL = DT == TRI_KV_FP8_E4M3 ? 128 : 192;
  switch (tw) {
    case 1024: return launch_mfma_t<DT, IL, 1024, SL, 1, NB>(k, bmat, shape, s);
    case 512: return launch_mfma_t<DT, IL, 512, SL + 512, 1, NB>(k, bmat, shape, s);
    case 256: return launch_mfma_t<DT, IL, 256, SL + 768, 1, NB>(k, bmat, shape, s);
    default: return hipErrorInvalidValue;
  }
}

// What fused_pack_kernel will do with these lengths, on the host: sequences by falling tile
// count, each into the first of the eight most recently opened launches with room.  Returns the
// number of launches.
int host_pack_launches(const int32_t* lens, int B, int tile, int wg_mult, int capacity) {
  std::vector<int> tiles(B);
  for (int i = 0; i < B; ++i) tiles[i] = ceil_div(lens[i], tile);
  std::vector<int> order(B);
  for (int i = 0; i < B; ++i) order[i] = i;
  if (B <= 4096)   // (the kernel sorts up to that many)
    std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return tiles[x] > tiles[y]; });
  int used[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  int first = 0, open = 1;
  for (int i = 0; i < B; ++i) {
    const int n = tiles[order[i]] * wg_mult;
    int pick = -1;
    for (int c = 0; c < open; ++c)
      if (used[c] + n <= capacity) { pick = c; break; }
    if (pick < 0) {
      if (open == 8) {
        for (int c = 0; c < 7; ++c) used[c] = used[c + 1];
        ++first;
        --open;
      }
      pick = open++;
      used[pick] = 0;
    }
    used[pick] += n;
  }
  return first + open;
}

}  // namespace

FusedPlan plan_fused_mfma(int B, int Hkv, int D, int G, int block_size, bool paged, int aggregation, int Tmax,
                          int resident, bool any_fill, int kv_dtype, const int32_t* host_lens, int L,
                          bool split_layers) {
  FusedPlan p{};
  const bool dim_ok = D == 128 || ((D == 64 || D == 256) && kv_dtype != TRI_KV_FP8_E4M3);
  if (resident <= 0 || !dim_ok || G < 1 || G > 8 || aggregation != TRI_REDUCE_MEAN || Tmax <= 0 || B <= 0)
    return p;
  int bs_shift = -1;
  for (int sft = 0; sft < 31; ++sft)
    if ((1 << sft) == block_size) bs_shift = sft;
  if (paged && bs_shift < 4) return p;    // a 16-token step must lie inside one block
  const int HC = ceil_div(Hkv, 8);
  // At most four KV heads: workgroups of four waves, two per CU.
  const int waves = Hkv <= 4 ? 4 : kFusedWaves;
  if (waves == 4) resident *= 2;
  const int tws[3] = {256, 512, 1024};
  const int ntw = G > 4 ? 2 : 3;          // the ring of a 1024-token tile fits LDS for four query heads only
  int tw = tws[ntw - 1];
  if (waves == kFusedWaves && D == 128)   // (four waves, head dimensions 64 and 256: one kernel instance, with the largest ring)
    for (int i = 0; i < ntw; ++i)
      if ((int64_t)B * ceil_div(Tmax, tws[i]) * HC <= resident) { tw = tws[i]; break; }
  int tile = tw, tiles = ceil_div(Tmax, tw);
  if ((int64_t)tiles * HC > resident) return p;
  if ((int64_t)B * tiles * HC <= resident) {
    // The whole batch is one launch: cut the sequences into as many tiles as the chip has
    // room for, in whole rotations of the step buffers (64 tokens, 128 for one-byte keys), so
    // that e.g. 16 sequences of 3072 tokens run as 16 x 16 tiles of 192 instead of 16 x 12 of
    // 256.  Not below 128 tokens and not more than 64 tiles per sequence: smaller tiles pay the
    // per-layer work of a workgroup too often, and every workgroup gathers the statistics of
    // all tiles of its sequence (one sequence of 16384 tokens as 256 tiles of 64 fills the
    // chip and takes 1.14 ms; the two-pass kernels take 0.38).
    const int granule = (kv_dtype == TRI_KV_FP8_E4M3 || (D == 64 && G <= 4)) ? 128 : 64;   // a rotation of the step buffers
    const int tiles_max = min(resident / (B * HC), 64);
    tile = ceil_div(ceil_div(Tmax, tiles_max), granule) * granule;
    tile = min(tw, max(128, tile));
    tiles = ceil_div(Tmax, tile);
  }
  // A launch that fills fewer than ~60 % of the CUs loses to the two-pass kernels, which
  // spread a small problem over the whole chip (16 sequences: even at 2176 tokens = 56 % of
  // the CUs, 10 % ahead at 2560 = 62 %, 21 % ahead at 3072 = 75 %).
  // (Workgroups of four waves: 45 %.  28 query / 4 KV heads, 16 x 2176 tokens, 272 of 512
  // workgroups: 0.40 ms against 0.48 ms on the two-pass kernels.)
  const int64_t need = waves == 4 ? 45 : 60;
  int layer_groups = 1, layers_per_group = L;
  if (split_layers && L > 1 && (int64_t)B * tiles * HC <= resident) {
    // A batch that is one launch: the layers are independent until the reduction over them, so
    // they can be cut into groups, a workgroup running one (sequence, group, tile).  A launch takes
    // as long as its longest workgroup: layers x (tile tokens + the fixed work of a layer, worth
    // ~32 tokens: the exchange of the statistics, the coefficient loads).  Whole-model workgroups
    // of a few requests (the reference's runner compresses one at a time,
    // runtime/runner_compression_actions.py:24) would use a fraction of the chip, 17 of 256 CUs
    // for one request of 2176 tokens x 36 layers: that becomes 36 groups x 7 tiles of 320 tokens
    // = 252 workgroups.  Mid-size batches gain as well: 16 requests of 2176 tokens are 16 x 12
    // tiles of 192 tokens x 36 layers (75 % of the CUs) or, with four groups of nine layers,
    // 16 x 4 x 4 tiles of 576 tokens on every CU, a quarter less per workgroup.  A cut must
    // win 5 % to be taken: the groups' partial sums cost a pass of their own, and a launch that
    // fills the chip already is bound by HBM as much as by its longest workgroup (16 x 8192 tokens
    // as two groups of 1024-token tiles: 1 % slower than whole-model tiles of 512).
    const int granule = (kv_dtype == TRI_KV_FP8_E4M3 || (D == 64 && G <= 4)) ? 128 : 64;
    const int tw_max = tws[ntw - 1];                       // the longest tile any instance of this shape holds
    const bool one_instance = !(waves == kFusedWaves && D == 128);
    constexpr int kLayerFixed = 32;
    int64_t best = (int64_t)L * (tile + kLayerFixed) * 95 / 100;
    for (int lpg = L - 1; lpg >= 1; --lpg) {
      const int groups = ceil_div(L, lpg);
      const int64_t units = (int64_t)B * groups * HC;
      if (units > resident) break;                         // fewer layers per group: more groups still
      const int tiles_max = (int)min((int64_t)64, resident / units);
      int t = ceil_div(ceil_div(Tmax, tiles_max), granule) * granule;
      t = min(tw_max, max(128, t));
      const int nt = ceil_div(Tmax, t);
      if (units * nt > resident) continue;
      const int64_t cost = (int64_t)lpg * (t + kLayerFixed) + groups;
      if (cost >= best) continue;
      best = cost;
      layer_groups = groups;
      layers_per_group = lpg;
      tile = t;
      tiles = nt;
      if (!one_instance)
        for (int i = 0; i < ntw; ++i)
          if (tws[i] >= t) { tw = tws[i]; break; }           // the instance with the smallest ring that holds the tile
    }
  }
  // The rule above is about workgroups that run layer after layer on a chip they do not fill.  With
  // one layer per workgroup the launch is short however few workgroups it has, and the two-pass
  // kernels pay five launches before their first byte: one layer of 1 x 4096 tokens as 32 tiles of
  // 128 takes 0.049 ms (score + select) against 0.079 ms.
  if (!any_fill && layers_per_group > 1 &&
      (int64_t)B * layer_groups * tiles * HC * 100 < (int64_t)resident * need)
    return p;
  p.eligible = 2;
  p.tw = tw;
  p.HC = HC;
  p.tile_tokens = tile;
  p.tiles_per_seq = tiles;
  p.seqs_per_launch = resident / (tiles * HC);
  p.resident = resident;
  p.bs_shift = bs_shift;
  p.waves = waves;
  p.launches = 0;
  p.layer_groups = layer_groups;
  p.layers_per_group = layers_per_group;
  if (layer_groups > 1) p.seqs_per_launch = B;      // one launch by construction
  if (host_lens && (int64_t)B * tiles * HC > resident) {
    // Several launches, and the lengths are known: a launch takes as long as its tiles are
    // long, however many of its workgroups have work, so the tile size that packs the
    // sequences into the fewest tile-lengths wins (64 sequences of 2k-32k tokens, 1.12 M in all:
    // 1124 tiles of 1024 tokens are 4.4 launches' worth and take five, 5 x 1024 tile-lengths;
    // 1777 tiles of 640 fill seven launches to 98 %, 7 x 640).
    const int granule = (kv_dtype == TRI_KV_FP8_E4M3 || (D == 64 && G <= 4)) ? 128 : 64;
    int64_t best_cost = -1;
    for (int cand = tw; cand >= tw / 2 && cand >= 128; cand -= granule) {
      const int per_seq = ceil_div(Tmax, cand) * HC;
      if (per_seq > resident) break;
      const int n = host_pack_launches(host_lens, B, cand, HC, resident);
      const int64_t cost = (int64_t)n * (cand + 32);      // 32 tokens' worth of fixed work per launch and layer
      if (best_cost < 0 || cost < best_cost) {
        best_cost = cost;
        p.tile_tokens = cand;
        p.tiles_per_seq = ceil_div(Tmax, cand);
        p.seqs_per_launch = resident / per_seq;
        p.launches = n;
      }
    }
  }
  return p;
}

hipError_t launch_fused_mfma(const FusedLaunch& a, hipStream_t s) {
  FusedArgs k{};
  k.k_layers = a.k_layers;
  k.k_scale_layers = a.k_scale_layers;
  k.block_table = a.block_table;
  k.seq_lens = a.seq_lens;
  k.prefill_lens = a.prefill_lens;
  k.coef = nullptr;   // this kernel takes its coefficients from bmat
  k.xchg = a.xchg;
  k.fin = a.fin;
  k.status = a.status;
  k.stride_block = a.stride_block; k.stride_token = a.stride_token; k.stride_head = a.stride_head;
  k.L = a.L; k.Hkv = a.Hkv; k.A = a.A; k.G = a.G; k.HC = a.plan.HC;
  k.block_size = a.block_size; k.bs_shift = a.plan.bs_shift;
  k.block_table_pitch = a.block_table ? a.block_table_pitch : -1;
  k.tiles_per_seq = a.plan.tiles_per_seq; k.tile_tokens = a.plan.tile_tokens;
  k.ring_stride = (int)align_up(k.tile_tokens, 16);
  if (k.ring_stride > a.plan.tw) return hipErrorInvalidValue;
  k.layer_groups = a.plan.layer_groups > 1 ? a.plan.layer_groups : 1;
  k.layers_per_group = k.layer_groups > 1 ? a.plan.layers_per_group : a.L;
  k.fin_part = a.fin_part;
  if (k.layer_groups > 1 && (!a.fin_part || (int64_t)k.layer_groups * k.layers_per_group < a.L)) return hipErrorInvalidValue;
  k.seq_base = 0; k.num_seqs = a.B * k.layer_groups; k.Tmax = a.Tmax;
  k.normalize = a.normalize; k.window_size = a.window_size; k.protect_prefill = a.protect_prefill;
  k.group_reduce = a.group_reduce; k.layer_reduce = a.layer_reduce;
  k.spin_ticks = resident_spin_ticks();
  k.seq_launch = a.pack;
  k.seq_wg_base = a.pack + a.B;
  const LaunchShape shape{a.plan.seqs_per_launch, a.plan.resident, a.B, a.plan.launches};
  const int64_t words = (int64_t)a.B * a.L * k.tiles_per_seq * a.A * 2;
  const bool il = a.rope_style == TRI_ROPE_INTERLEAVED;
  uint4* bmat = reinterpret_cast<uint4*>(a.bmat);
  const bool fp8 = a.kv_dtype == TRI_KV_FP8_E4M3;
  const bool fp16 = a.kv_dtype == TRI_KV_FP16;
  if (a.kv_dtype != TRI_KV_BF16 && !fp8 && !fp16) return hipErrorInvalidValue;
  if (a.NO <= 0 || a.NO > kMaxOffsets || (a.D != 128 && a.D != 64 && a.D != 256)) return hipErrorInvalidValue;
  if (a.D != 128 && fp8) return hipErrorInvalidValue;
  // A workgroup takes all KV heads of a layer and request, which evaluates the phases least often, unless that
  // leaves CUs without one: then the heads are halved until there are 256 workgroups.  The launch is a chain of
  // latencies (statistics, phases, slabs), not bytes: the whole step of one layer x 4096 tokens 56.6 -> 53.0 us with eight
  // workgroups in place of one and the statistics requested first; a call on 36 layers x 2176 tokens 267 -> 265.
  int heads_per_wg = a.Hkv;
  while (heads_per_wg > 1 && (int64_t)a.L * a.B * ceil_div(a.Hkv, heads_per_wg) < 256) heads_per_wg = ceil_div(heads_per_wg, 2);
  auto prep_launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)a.L, (unsigned)a.B, (unsigned)ceil_div(a.Hkv, heads_per_wg)),
                       dim3(kPrepThreads), 0, s, a.folded, a.omega, a.offsets, a.NO, a.round_start, a.L, a.Hkv, a.G, a.A,
                       bmat, a.xchg, words, a.status, heads_per_wg);
  };
  if (fp8) {
    if (il) prep_launch(prep_mfma_kernel<TRI_KV_FP8_E4M3, true, 128>);
    else prep_launch(prep_mfma_kernel<TRI_KV_FP8_E4M3, false, 128>);
  } else if (fp16) {
    if (a.D == 64) {
      if (il) prep_launch(prep_mfma_kernel<TRI_KV_FP16, true, 64>);
      else prep_launch(prep_mfma_kernel<TRI_KV_FP16, false, 64>);
    } else if (a.D == 256) {
      if (il) prep_launch(prep_mfma_kernel<TRI_KV_FP16, true, 256>);
      else prep_launch(prep_mfma_kernel<TRI_KV_FP16, false, 256>);
    } else {
      if (il) prep_launch(prep_mfma_kernel<TRI_KV_FP16, true, 128>);
      else prep_launch(prep_mfma_kernel<TRI_KV_FP16, false, 128>);
    }
  } else {
    if (a.D == 64) {
      if (il) prep_launch(prep_mfma_kernel<TRI_KV_BF16, true, 64>);
      else prep_launch(prep_mfma_kernel<TRI_KV_BF16, false, 64>);
    } else if (a.D == 256) {
      if (il) prep_launch(prep_mfma_kernel<TRI_KV_BF16, true, 256>);
      else prep_launch(prep_mfma_kernel<TRI_KV_BF16, false, 256>);
    } else {
      if (il) prep_launch(prep_mfma_kernel<TRI_KV_BF16, true, 128>);
      else prep_launch(prep_mfma_kernel<TRI_KV_BF16, false, 128>);
    }
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  if (fp8)
    e = il ? launch_mfma_tw<TRI_KV_FP8_E4M3, true>(k, bmat, a.plan.tw, a.plan.waves, a.D, shape, s)
           : launch_mfma_tw<TRI_KV_FP8_E4M3, false>(k, bmat, a.plan.tw, a.plan.waves, a.D, shape, s);
  else if (fp16)
    e = il ? launch_mfma_tw<TRI_KV_FP16, true>(k, bmat, a.plan.tw, a.plan.waves, a.D, shape, s)
           : launch_mfma_tw<TRI_KV_FP16, false>(k, bmat, a.plan.tw, a.plan.waves, a.D, shape, s);
  else
    e = il ? launch_mfma_tw<TRI_KV_BF16, true>(k, bmat, a.plan.tw, a.plan.waves, a.D, shape, s)
           : launch_mfma_tw<TRI_KV_BF16, false>(k, bmat, a.plan.tw, a.plan.waves, a.D, shape, s);
  if (e != hipSuccess || k.layer_groups <= 1 || a.skip_layer_reduce) return e;
  const int64_t count = (int64_t)a.B * a.Hkv * a.Tmax;
  hipLaunchKernelGGL(fused_layer_reduce_kernel, dim3((unsigned)ceil_div64(count, 256)), dim3(256), 0, s, a.fin_part, a.fin,
                     count, k.layer_groups, a.layer_reduce, a.L);
  return hipGetLastError();
}

}  // namespace tri
