// Dense varlen multi-head attention for MLA prefill (gfx950, wave64 MFMA):
//
//   out[t, h, :] = softmax(scale * q[t, h, :] . k[j, h, :]^T) v[j, h, :]
//
// over the keys j of token t's sequence (ragged batches given by
// cu_seqlens_q / cu_seqlens_k), causal with the diagonal aligned to the end
// of the key sequence (query i of a q_len-long sequence sees keys
// j <= i + k_len - q_len), or non-causal; lse[h, t] = natural-log
// log-sum-exp, -inf for a query with no key (its output is 0).  This is the
// attention that reference/vllm/v1/attention/backends/mla/prefill/
// sm70_triton.py:54-187 (_varlen_attention) computes per sequence in fp32.
//
// Three kernels: 16-bit inputs at head dims up to (192, 128) (LDS ring, 32
// query rows per wave), 16-bit inputs at (256, 256), whose Q and O rows leave
// no registers for that form, and fp32 inputs.
#include <float.h>

#include "capi_internal.h"
#include "dsa_common.h"

namespace mi355dsa {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef short s16x4v __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4v lds_s16x4v;

constexpr int kVaWaves = 4;
constexpr int kVaThreads = 64 * kVaWaves;

__device__ const __align__(16) uint16_t kVaZero[8] = {};

struct VaArgs {
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* v;
  uint16_t* o;
  float* lse;  // [H, total_q] or null
  const int32_t* cu_q;
  const int32_t* cu_k;
  int64_t q_st, q_sh, k_st, k_sh, v_st, v_sh, o_st, o_sh;  // element strides
  int H, total_q, n_qtiles, causal;
  int o16;    // output rows are 16-byte aligned
  int pairs;  // > 0: 1-D grid in pair-major order over this many (sequence, head) pairs
  float scale_log2;  // softmax scale * log2(e)
  float scale;
};

template <bool BF16>
__device__ __forceinline__ f32x4 mma(const u32x4& a, const u32x4& b, f32x4 c) {
  if constexpr (BF16)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

template <bool BF16>
__device__ __forceinline__ uint16_t to16(float x) {
  if constexpr (BF16) return __builtin_bit_cast(uint16_t, (__bf16)x);
  else return __builtin_bit_cast(uint16_t, (f16)x);
}
template <bool BF16>
__device__ __forceinline__ float from16(uint16_t x) {
  if constexpr (BF16) return (float)__builtin_bit_cast(__bf16, x);
  else return (float)__builtin_bit_cast(f16, x);
}

// K and V rows at a pitch of d / 8 + 2 pieces (two pads): the QK reads (16
// rows x 4 adjacent pieces per instruction) and the V^T transpose reads (8
// rows x 32 bytes per half-wave) are then free of LDS bank conflicts (both
// measured on gfx950; with one pad both conflicted two-way)
template <int DQK, int DV, int KT>
struct VaShape {
  static constexpr int PK = DQK / 8 + 2;  // K row pitch in 16-B pieces
  static constexpr int PV = DV / 8 + 2;
  static constexpr int RK = (KT * PK + kVaThreads - 1) / kVaThreads;  // DMA rounds
  static constexpr int RV = (KT * PV + kVaThreads - 1) / kVaThreads;
  static constexpr int KBYTES = RK * kVaThreads * 16;
  static constexpr int VBYTES = RV * kVaThreads * 16;
  static constexpr int STAGE = KBYTES + VBYTES;
};

template <int N>
__device__ __forceinline__ void va_wait() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// 16-bit inputs at (256, 256).  Workgroup = (query tile of 64 QB rows,
// sequence, head), 4 waves; wave w owns query rows [16 QB w, +16 QB).  Key
// tiles of KT keys stream through two LDS stages by LDS-DMA, the next tile in
// flight while the current one is used.  Per tile and wave: S^T = K Q^T
// (v_mfma_f32_16x16x32, keys the A operand read from LDS, queries resident in
// registers), online softmax per query column, O^T += V^T P^T with P in
// registers and V^T from ds_read_b64_tr_b16.  bf16 P is split into hi + lo.
template <bool BF16, int DQK, int DV, int QB, int KT, int MINB>
__global__ void __launch_bounds__(kVaThreads, MINB) varlen_attn_kernel(VaArgs a) {
  using Sh = VaShape<DQK, DV, KT>;
  constexpr int NKB = KT / 16;  // 16-key blocks per tile
  constexpr int NKH = KT / 32;  // 32-key PV steps per tile
  constexpr int QROWS = 16 * QB * kVaWaves;
  constexpr int NS = DQK / 32;  // QK k-steps
  constexpr int NDT = DV / 16;  // O^T dim tiles
  extern __shared__ __align__(16) unsigned char smem_raw[];

  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int c = lane & 15, g = lane >> 4;
  const int seq = blockIdx.y, h = blockIdx.z;
  const int qs = a.cu_q[seq], q_len = a.cu_q[seq + 1] - qs;
  const int ks = a.cu_k[seq], k_len = a.cu_k[seq + 1] - ks;
  // heaviest (latest) query tiles first under a causal mask
  const int tile = a.causal ? a.n_qtiles - 1 - (int)blockIdx.x : (int)blockIdx.x;
  const int q0 = tile * QROWS;
  if (q0 >= q_len) return;
  const int offset = a.causal ? k_len - q_len : 0;
  const int kend = a.causal ? max(0, min(k_len, q0 + QROWS + offset)) : k_len;
  const int n_kt = (kend + KT - 1) / KT;

  // ---- Q fragments (B operand): row q0 + 16(QB w + qb) + c, dims 32 s + 8 g ----
  u32x4 qf[QB][NS];
#pragma unroll
  for (int qb = 0; qb < QB; qb++) {
    const int i = q0 + 16 * (QB * w + qb) + c;
    const uint16_t* qrow = a.q + (int64_t)(qs + (i < q_len ? i : 0)) * a.q_st + (int64_t)h * a.q_sh +
                           8 * g;
    // rows past q_len read row 0 of the sequence: their MFMA columns and
    // softmax state are their own, and their outputs are not stored
#pragma unroll
    for (int s = 0; s < NS; s++) qf[qb][s] = *reinterpret_cast<const u32x4*>(qrow + 32 * s);
  }

  auto issue_tile = [&](int kt) {
    unsigned char* st = smem_raw + (kt & 1) * Sh::STAGE;
    const int k0 = kt * KT;
#pragma unroll
    for (int u = 0; u < Sh::RK; u++) {
      const int qq = kVaThreads * u + 64 * w + lane;
      const int r = qq / Sh::PK, ch = qq - r * Sh::PK;
      const bool ok = r < KT && ch < DQK / 8 && k0 + r < kend;
      const uint16_t* src = ok ? a.k + (int64_t)(ks + k0 + r) * a.k_st + (int64_t)h * a.k_sh + 8 * ch
                               : kVaZero;
      dma16(src, st + 16 * (kVaThreads * u + 64 * w));
    }
#pragma unroll
    for (int u = 0; u < Sh::RV; u++) {
      const int qq = kVaThreads * u + 64 * w + lane;
      const int r = qq / Sh::PV, ch = qq - r * Sh::PV;
      const bool ok = r < KT && ch < DV / 8 && k0 + r < kend;
      const uint16_t* src = ok ? a.v + (int64_t)(ks + k0 + r) * a.v_st + (int64_t)h * a.v_sh + 8 * ch
                               : kVaZero;
      dma16(src, st + Sh::KBYTES + 16 * (kVaThreads * u + 64 * w));
    }
  };

  f32x4 oacc[NDT][QB];
#pragma unroll
  for (int t = 0; t < NDT; t++)
#pragma unroll
    for (int qb = 0; qb < QB; qb++) oacc[t][qb] = (f32x4){0.f, 0.f, 0.f, 0.f};
  float m_run[QB], l_part[QB];  // raw-score running max (same in the 4 lane groups), partial sums
#pragma unroll
  for (int qb = 0; qb < QB; qb++) {
    m_run[qb] = -1e30f;
    l_part[qb] = 0.f;
  }

  if (n_kt > 0) issue_tile(0);
  // Q completes here, together with tile 0 (one round trip).  The compiler
  // does not count the tile DMAs issued by inline asm, so a wait for Q left
  // to the loop would be vmcnt(0) on every step and drain the next tile.
#pragma unroll
  for (int qb = 0; qb < QB; qb++)
#pragma unroll
    for (int s = 0; s < NS; s++) asm volatile("" ::"v"(qf[qb][s]));
  for (int kt = 0; kt < n_kt; kt++) {
    if (kt + 1 < n_kt) {
      issue_tile(kt + 1);
      va_wait<Sh::RK + Sh::RV>();
    } else {
      va_wait<0>();
    }
    lds_barrier();  // tile kt landed for every wave
    const unsigned char* kst = smem_raw + (kt & 1) * Sh::STAGE;
    const unsigned char* vst = kst + Sh::KBYTES;
    const int k0 = kt * KT;

    // ---- S^T blocks: keys 16 kb + 4 g + r, query column c of block qb ----
    f32x4 sacc[NKB][QB];
#pragma unroll
    for (int kb = 0; kb < NKB; kb++)
#pragma unroll
      for (int qb = 0; qb < QB; qb++) sacc[kb][qb] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < NS; s++) {
#pragma unroll
      for (int kb = 0; kb < NKB; kb++) {
        const u32x4 kf = *reinterpret_cast<const u32x4*>(kst + (16 * kb + c) * Sh::PK * 16 +
                                                         64 * s + 16 * g);
#pragma unroll
        for (int qb = 0; qb < QB; qb++) sacc[kb][qb] = mma<BF16>(kf, qf[qb][s], sacc[kb][qb]);
      }
    }

    // ---- masks and online softmax per query column ----
    u32x4 pb[NKH][QB], pl[NKH][QB];  // P^T operands per 32 keys (hi and, for bf16, lo parts)
#pragma unroll
    for (int qb = 0; qb < QB; qb++) {
      const int i = q0 + 16 * (QB * w + qb) + c;  // query row of this column
      const int jmax = a.causal ? min(kend, i + offset + 1) : kend;  // keys < jmax are valid
      float mt = -1e30f;
#pragma unroll
      for (int kb = 0; kb < NKB; kb++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const int j = k0 + 16 * kb + 4 * g + r;
          if (j >= jmax) sacc[kb][qb][r] = -INFINITY;
          mt = fmaxf(mt, sacc[kb][qb][r]);
        }
      mt = fmaxf(mt, shfl_xor_f(mt, 16));
      mt = fmaxf(mt, shfl_xor_f(mt, 32));
      const float m_new = fmaxf(m_run[qb], mt);
      const float alpha = exp2f((m_run[qb] - m_new) * a.scale_log2);
      m_run[qb] = m_new;
      const float mb = m_new * a.scale_log2;
      float ls = 0.f;
      float pv[NKB][4];
#pragma unroll
      for (int kb = 0; kb < NKB; kb++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const float sv = sacc[kb][qb][r];
          const float p = (sv > -INFINITY) ? exp2f(__builtin_fmaf(sv, a.scale_log2, -mb)) : 0.f;
          pv[kb][r] = p;
          ls += p;
        }
      l_part[qb] = l_part[qb] * alpha + ls;
#pragma unroll
      for (int t = 0; t < NDT; t++) oacc[t][qb] *= alpha;
#pragma unroll
      for (int kh = 0; kh < NKH; kh++) {
        uint16_t hi[8], lo[8];
#pragma unroll
        for (int e = 0; e < 8; e++) {
          const float p = pv[2 * kh + (e >> 2)][e & 3];
          hi[e] = to16<BF16>(p);
          lo[e] = BF16 ? to16<BF16>(p - from16<BF16>(hi[e])) : (uint16_t)0;
        }
#pragma unroll
        for (int e = 0; e < 4; e++) {
          pb[kh][qb][e] = (uint32_t)hi[2 * e] | ((uint32_t)hi[2 * e + 1] << 16);
          pl[kh][qb][e] = (uint32_t)lo[2 * e] | ((uint32_t)lo[2 * e + 1] << 16);
        }
      }
    }

    // ---- O^T += V^T P^T: keys 32 kh + {4g .. 4g+3, 16 + 4g .. 16 + 4g + 3} ----
    // transpose source: lane i of group g points at key 32 kh + 4 g + i / 4
    // (+16 for the second read), dims 16 t + 4 (i % 4) .. +3
    const unsigned char* vsrc = vst + (4 * g + (c >> 2)) * Sh::PV * 16 + 8 * (c & 3);
#pragma unroll
    for (int kh = 0; kh < NKH; kh++) {
#pragma unroll
      for (int t = 0; t < NDT; t++) {
        const s16x4v v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (lds_s16x4v*)(vsrc + (32 * kh) * Sh::PV * 16 + 32 * t));
        const s16x4v v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (lds_s16x4v*)(vsrc + (32 * kh + 16) * Sh::PV * 16 + 32 * t));
        const u32x2 x0 = __builtin_bit_cast(u32x2, v0), x1 = __builtin_bit_cast(u32x2, v1);
        const u32x4 av = {x0[0], x0[1], x1[0], x1[1]};
#pragma unroll
        for (int qb = 0; qb < QB; qb++) {
          oacc[t][qb] = mma<BF16>(av, pb[kh][qb], oacc[t][qb]);
          if constexpr (BF16) oacc[t][qb] = mma<BF16>(av, pl[kh][qb], oacc[t][qb]);
        }
      }
    }
    lds_barrier();  // every wave is done with this stage before it is refilled
  }

  // ---- outputs ----
#pragma unroll
  for (int qb = 0; qb < QB; qb++) {
    float l = l_part[qb];
    l += shfl_xor_f(l, 16);
    l += shfl_xor_f(l, 32);
    const int i = q0 + 16 * (QB * w + qb) + c;
    if (i >= q_len) continue;
    const float inv = l > 0.f ? 1.f / l : 0.f;
    uint16_t* orow = a.o + (int64_t)(qs + i) * a.o_st + (int64_t)h * a.o_sh;
#pragma unroll
    for (int t = 0; t < NDT; t++) {
      u32x2 pk;
      pk[0] = (uint32_t)to16<BF16>(oacc[t][qb][0] * inv) |
              ((uint32_t)to16<BF16>(oacc[t][qb][1] * inv) << 16);
      pk[1] = (uint32_t)to16<BF16>(oacc[t][qb][2] * inv) |
              ((uint32_t)to16<BF16>(oacc[t][qb][3] * inv) << 16);
      *reinterpret_cast<u32x2*>(orow + 16 * t + 4 * g) = pk;
    }
    if (a.lse != nullptr && g == 0)
      a.lse[(int64_t)h * a.total_q + qs + i] =
          l > 0.f ? m_run[qb] * a.scale + logf(l) : -INFINITY;
  }
}

template <bool BF16, int DQK, int DV, int QB, int KT, int MINB>
int launch_va(const VaArgs& a0, int num_seqs, int max_q_len, hipStream_t st) {
  using Sh = VaShape<DQK, DV, KT>;
  constexpr int QROWS = 16 * QB * kVaWaves;
  auto kern = varlen_attn_kernel<BF16, DQK, DV, QB, KT, MINB>;
  const int rc = reserve_lds(reinterpret_cast<const void*>(kern), 2 * Sh::STAGE, "varlen_attention");
  if (rc) return rc;
  VaArgs a = a0;
  a.n_qtiles = (max_q_len + QROWS - 1) / QROWS;
  if (a.n_qtiles == 0) return MI355_DSA_OK;
  kern<<<dim3(a.n_qtiles, num_seqs, a.H), kVaThreads, 2 * Sh::STAGE, st>>>(a);
  return check_launch("varlen_attention");
}

// ---------------------------------------------------------------------------
// 16-bit inputs, head dims (192, 128), (128, 128) and (64, 64).
//
// Workgroup = (query tile of 128 rows, sequence, head), 4 waves of 32 rows;
// two workgroups share a CU.  Steps of 32 keys stream through a four-slot LDS
// ring by LDS-DMA, three steps ahead, one barrier per step.  A wave's step i:
//   * S^T(i+1) = K Q^T (v_mfma_f32_32x32x16: keys the A operand from LDS, the
//     wave's 32 queries the B operand resident in registers) beside the
//     exponentials of step i: independent work for the matrix cores and the
//     VALU in one basic block;
//   * O^T += V^T P^T: the S^T accumulator layout (query = lane % 32, keys
//     8 (e / 4) + 4 (lane / 32) + e % 4) is the B-operand layout of P^T, so P
//     stays in registers; V^T comes from ds_read_b64_tr_b16 transpose reads in
//     the same key order; the maximum of S^T(i+1) is taken beside it.
// A query's 32 scores of a step sit in two lanes, so its maximum is one lane
// swap.  O is rescaled only when a maximum grows by more than kVaLazy binades
// over the one in use (p then stays <= 2^kVaLazy, far inside fp16), and the
// causal / tail masks run only in steps that hold a masked key.
// bf16 inputs keep P as two bf16 parts (p = hi + lo, two PV MFMAs), ~16 bits.
//
// LDS layouts, free of bank conflicts without pads: K as 64-byte blocks
// (4 pieces of 16 B) per key, block-major (block b of key r at 2048 b + 64 r),
// piece p at p ^ ((r >> 2) & 3): the 32 rows of a QK read cover every bank
// once per 16-lane phase.  V rows are whole, 64-byte group u of key r at
// u ^ (r & 3) (DV = 64: u ^ ((r >> 1) & 1)): the 4 keys x 64 bytes of a
// half-wave's transpose read cover the 64 banks.  Both are applied to the
// DMA's source address, so every DMA instruction writes 1 KB in order and
// reads 64-byte or longer runs.
//
// Bound: the matrix cores, with the softmax's VALU work beside them (per step
// and wave 20 MFMAs of 32 clk at (192, 128) fp16, 28 in bf16, against ~120-160
// VALU instructions, 16 of them exponentials at a quarter rate); on short
// sequences the first Q and K reads of each workgroup.  Measured, 64 heads,
// (192, 128), against the two-stage kernel kept for (256, 256): causal 16k
// 11.08 -> 5.66 ms fp16 (972 TFLOP/s; a large library product reaches 1180
// here), 12.90 -> 6.86 ms bf16; causal 800-3203-token prompts, 10007 tokens,
// 1386 -> 815 us fp16, 1460 -> 855 us bf16.  Of that, the 32-row waves, the
// ring and the lazy rescale gave 6.3 ms, whole (sequence, head) pairs per XCD
// 5.9 ms, the grouped MFMA / VALU order 5.66 ms (the compiler's own order put
// the exponentials before the MFMAs).  Measured level: 2 K reads ahead instead
// of 3, two steps per loop iteration, groups of 4-16 query tiles per pair.
// Sequences of one or two steps are all prologue and epilogue.  Addresses of the
// NaN pass and of the outputs kept over the loop spilled 22 registers there, and
// the flags between the waves went by flat loads: 16 x 64 tokens, 64 heads, fp16 22.0
// us with the two-stage kernel, 26.3 so, 21.2 without either (8 x 500 115 -> 106 us;
// one workgroup over 4000 keys 98 -> 100).  A branch around the step past the last one
// slows such long single workgroups by another 4 %.
// ---------------------------------------------------------------------------
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

constexpr float kVaLazy = 8.f;
constexpr int kVaAhead = 3;  // K reads in flight ahead of their MFMA

template <bool BF16>
__device__ __forceinline__ f32x16 mma32x32(const u32x4& a, const u32x4& b, f32x16 c) {
  if constexpr (BF16)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

// two fp32 values as one packed pair of 16-bit values (RNE)
template <bool BF16>
__device__ __forceinline__ uint32_t pack16(float x, float y) {
  if constexpr (BF16) {
    const bf16x2 p = {(__bf16)x, (__bf16)y};
    return __builtin_bit_cast(uint32_t, p);
  } else {
    const f16x2 p = {(f16)x, (f16)y};
    return __builtin_bit_cast(uint32_t, p);
  }
}

template <int DQK, int DV>
struct VaRing {
  static constexpr int KT = 32;              // keys per step
  static constexpr int SLOTS = 4;
  static constexpr int KBYTES = KT * DQK * 2;
  static constexpr int VBYTES = KT * DV * 2;
  static constexpr int SLOT = KBYTES + VBYTES;
  static constexpr int NKD = DQK / 64;       // K DMA instructions per wave and step
  static constexpr int NVD = DV / 64;        // V DMA instructions per wave and step
  static constexpr int ND = NKD + NVD;
};

template <bool BF16, int DQK, int DV>
__global__ void __launch_bounds__(kVaThreads, 2) varlen_attn_ring_kernel(VaArgs a) {
  using R = VaRing<DQK, DV>;
  constexpr int KT = R::KT;
  constexpr int NS = DQK / 16;  // QK k-steps
  constexpr int NDT = DV / 32;  // O^T dim tiles
  constexpr int QROWS = 32 * kVaWaves;
  constexpr int VROWS = 1024 / (2 * DV);  // V rows per DMA instruction
  extern __shared__ __align__(16) unsigned char smem_raw[];

  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int c = lane & 31, hf = lane >> 5;
  int seq = blockIdx.y, h = blockIdx.z, bt = blockIdx.x;
  if (a.pairs > 0) {
    // consecutive workgroups go to the eight XCDs in turn: each XCD takes
    // whole (sequence, head) pairs, one after another, so that the query
    // tiles in flight on it stream the same K and V through its L2
    const int r = blockIdx.x >> 3, pair = 8 * (r / a.n_qtiles) + (blockIdx.x & 7);
    if (pair >= a.pairs) return;
    bt = r % a.n_qtiles;
    seq = pair / a.H;
    h = pair % a.H;
  }
  const int qs = a.cu_q[seq], q_len = a.cu_q[seq + 1] - qs;
  const int ks = a.cu_k[seq], k_len = a.cu_k[seq + 1] - ks;
  // heaviest (latest) query tiles first under a causal mask
  const int tile = a.causal ? a.n_qtiles - 1 - bt : bt;
  const int q0 = tile * QROWS;
  if (q0 >= q_len) return;
  const int offset = a.causal ? k_len - q_len : 0;
  const int kend = a.causal ? max(0, min(k_len, q0 + QROWS + offset)) : k_len;
  const int n = (kend + KT - 1) / KT;

  // ---- Q (B operand): row q0 + 32 w + c, dims 16 s + 8 hf .. +7; rows past
  // q_len read row 0 of the sequence (their columns are not stored) ----
  const int qi = q0 + 32 * w + c;
  u32x4 qf[NS];
  {
    const uint16_t* qrow = a.q + (int64_t)(qs + (qi < q_len ? qi : 0)) * a.q_st +
                           (int64_t)h * a.q_sh + 8 * hf;
#pragma unroll
    for (int s = 0; s < NS; s++) qf[s] = *reinterpret_cast<const u32x4*>(qrow + 16 * s);
  }

  // ---- this wave's share of a step's DMA: K rows 16 (w & 1) + lane / 4 of
  // blocks NKD (w >> 1) .. , V rows VROWS (NVD w + u) + lane / (DV / 8) ----
  const int kr = 16 * (w & 1) + (lane >> 2);
  const int kb0 = R::NKD * (w >> 1);
  const uint16_t* kp = a.k + (int64_t)(ks + kr) * a.k_st + (int64_t)h * a.k_sh + 32 * kb0 +
                       8 * ((lane & 3) ^ ((lane >> 4) & 3));
  const int vl = lane / (DV / 8), vr = VROWS * R::NVD * w + vl;
  const int vsw = DV == 64 ? (vl >> 1) & 1 : vl & 3;
  const uint16_t* vp = a.v + (int64_t)(ks + vr) * a.v_st + (int64_t)h * a.v_sh +
                       8 * ((lane & (DV / 8 - 1)) ^ (4 * vsw));
  unsigned char* const kdst = smem_raw + 2048 * kb0 + 1024 * (w & 1);
  unsigned char* const vdst = smem_raw + R::KBYTES + 1024 * R::NVD * w;

  auto issue = [&](int i) {
    const int so = (i & (R::SLOTS - 1)) * R::SLOT;
    const int k0 = i * KT;
    const uint16_t* kq = kp + (int64_t)k0 * a.k_st;
    const uint16_t* vq = vp + (int64_t)k0 * a.v_st;
    if (k0 + KT <= kend) {
#pragma unroll
      for (int u = 0; u < R::NKD; u++) dma16(kq + 32 * u, kdst + so + 2048 * u);
#pragma unroll
      for (int u = 0; u < R::NVD; u++)
        dma16(vq + (int64_t)(VROWS * u) * a.v_st, vdst + so + 1024 * u);
    } else {  // rows past the last key read zeros
      const bool kok = k0 + kr < kend;
#pragma unroll
      for (int u = 0; u < R::NKD; u++)
        dma16(kok ? kq + 32 * u : kVaZero, kdst + so + 2048 * u);
#pragma unroll
      for (int u = 0; u < R::NVD; u++)
        dma16(k0 + vr + VROWS * u < kend ? vq + (int64_t)(VROWS * u) * a.v_st : kVaZero,
              vdst + so + 1024 * u);
    }
  };

  // ---- LDS read offsets within a slot ----
  const uint32_t lds0 = (uint32_t)(uintptr_t)smem_raw;
  const uint32_t ka0 = 64 * c + 16 * (hf ^ ((c >> 2) & 3));  // QK steps 0, 2, ..; ka0 ^ 32: 1, 3, ..
  const int ti = lane & 15, trow = 4 * hf + (ti >> 2);
  const int tsw = DV == 64 ? (ti >> 3) & 1 : ti >> 2;
  uint32_t va0[NDT];
#pragma unroll
  for (int t = 0; t < NDT; t++)
    va0[t] = R::KBYTES + trow * (2 * DV) + 64 * (t ^ tsw) + 32 * ((lane >> 4) & 1) + 8 * (ti & 3);

  // keys < jmax are visible to this lane's query; steps that end at or below
  // jmin hold no masked key for any query of the wave
  const int jmax = a.causal ? min(kend, qi + offset + 1) : kend;
  const int jmin = a.causal ? min(kend, q0 + 32 * w + offset + 1) : kend;
  const float lazy = kVaLazy / a.scale_log2;

  f32x16 oacc[NDT], s;
  float m_run, l_part;

  auto qk = [&](int i) {
    const uint32_t kb = lds0 + (i & (R::SLOTS - 1)) * R::SLOT + ka0;
    f32x16 acc = {};
#pragma unroll
    for (int t = 0; t < NS; t++) {
      const u32x4 kf = *(const __attribute__((address_space(3))) u32x4*)(
          ((t & 1) ? (kb ^ 32u) : kb) + 2048u * (t >> 1));
      acc = mma32x32<BF16>(kf, qf[t], acc);
    }
    return acc;
  };

  // the ring's first three steps
  auto prologue = [&](int first) {
#pragma unroll
    for (int i = 0; i < 3; i++)
      if (i < n) issue(first + i);
  };
  auto max16 = [&](const f32x16& x) {
    float m = fmaxf(x[0], x[1]);
#pragma unroll
    for (int e = 2; e < 16; e++) m = fmaxf(m, x[e]);
    return xor32_max(m);
  };
  prologue(0);
  // Q completes here, beside the first steps.  The compiler does not count
  // the DMAs issued by inline asm, so a wait for Q left to the loop would
  // drain the steps in flight.
#pragma unroll
  for (int t = 0; t < NS; t++) asm volatile("" : "+v"(qf[t]));

  // NaN scores count as masked.  They show as a NaN row sum, and the tile is
  // then run again with every score tested, so the usual pass tests none.
  for (bool safe = false;; safe = true) {
#pragma unroll
    for (int t = 0; t < NDT; t++) oacc[t] = (f32x16){};
    m_run = -1e30f;
    l_part = 0.f;
    va_wait<0>();
    lds_barrier();
    s = qk(0);
    float mt = max16(s);
    for (int i = 0; i < n; i++) {
      if (i + 2 < n) va_wait<R::ND>();
      else va_wait<0>();
      lds_barrier();  // K(i + 1) and V(i) are in; nobody reads slot (i - 1) any more
      if (i + 3 < n) issue(i + 3);

      const int k0 = i * KT;
      if (k0 + KT > jmin || safe) {
#pragma unroll
        for (int e = 0; e < 16; e++) {
          const int j = k0 + 8 * (e >> 2) + 4 * hf + (e & 3);
          if (j >= jmax || s[e] != s[e]) s[e] = -INFINITY;
        }
        mt = max16(s);
      }
      if (__any(mt > m_run + lazy)) {
        const float m_new = fmaxf(m_run, mt);
        const float alpha = __builtin_amdgcn_exp2f((m_run - m_new) * a.scale_log2);
        m_run = m_new;
        l_part *= alpha;
#pragma unroll
        for (int t = 0; t < NDT; t++) oacc[t] *= alpha;
      }

      // S^T(i + 1) beside p(i), then O(i) beside the row sums and the maximum
      // of S^T(i + 1).  Each group holds one MFMA (pair), the LDS read of a
      // later one and a share of the VALU work; sched_barrier keeps the
      // groups apart.  Past the last step QK multiplies a slot's old keys,
      // and nothing reads the result.
      f32x16 sn = {};
      const float mb = m_run * a.scale_log2;
      u32x4 pb[2], pl[2];
      {
        const uint32_t kb = lds0 + ((i + 1) & (R::SLOTS - 1)) * R::SLOT + ka0;
        auto kread = [&](int t) {
          return *(const __attribute__((address_space(3))) u32x4*)(
              ((t & 1) ? (kb ^ 32u) : kb) + 2048u * (t >> 1));
        };
        u32x4 kf[kVaAhead + 1];
#pragma unroll
        for (int t = 0; t < kVaAhead; t++) kf[t] = kread(t);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < NS; t++) {
          if (t + kVaAhead < NS) kf[(t + kVaAhead) % (kVaAhead + 1)] = kread(t + kVaAhead);
          sn = mma32x32<BF16>(kf[t % (kVaAhead + 1)], qf[t], sn);
#pragma unroll
          for (int e = 16 * t / NS; e < 16 * (t + 1) / NS; e++) {
            s[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[e], a.scale_log2, -mb));
            if (e & 1) {
              const uint32_t hi = pack16<BF16>(s[e - 1], s[e]);
              pb[e >> 3][(e >> 1) & 3] = hi;
              if constexpr (BF16)
                pl[e >> 3][(e >> 1) & 3] =
                    pack16<true>(s[e - 1] - __uint_as_float(hi << 16),
                                 s[e] - __uint_as_float(hi & 0xffff0000u));
            }
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      {
        const uint32_t vb = lds0 + (i & (R::SLOTS - 1)) * R::SLOT;
        auto vread = [&](int u) {
          const int t = u % NDT, t2 = u / NDT;
          const s16x4v v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (lds_s16x4v*)(vb + va0[t] + 32 * DV * t2));
          const s16x4v v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (lds_s16x4v*)(vb + va0[t] + 32 * DV * t2 + 16 * DV));
          const u32x2 x0 = __builtin_bit_cast(u32x2, v0), x1 = __builtin_bit_cast(u32x2, v1);
          return (u32x4){x0[0], x0[1], x1[0], x1[1]};
        };
        constexpr int NP = 2 * NDT;
        u32x4 vf[3];
        vf[0] = vread(0);
        vf[1] = vread(1);
        __builtin_amdgcn_sched_barrier(0);
        float ls[4] = {s[0], s[1], s[2], s[3]};
        mt = -1e30f;
#pragma unroll
        for (int u = 0; u < NP; u++) {
          if (u + 2 < NP) vf[(u + 2) % 3] = vread(u + 2);
          oacc[u % NDT] = mma32x32<BF16>(vf[u % 3], pb[u / NDT], oacc[u % NDT]);
          if constexpr (BF16) oacc[u % NDT] = mma32x32<BF16>(vf[u % 3], pl[u / NDT], oacc[u % NDT]);
          constexpr int H = NP / 2;
#pragma unroll
          for (int e = 4 + 12 * u / NP; e < 4 + 12 * (u + 1) / NP; e++) ls[e & 3] += s[e];
          if (u >= H) {
#pragma unroll
            for (int e = 16 * (u - H) / H; e < 16 * (u - H + 1) / H; e++) mt = fmaxf(mt, sn[e]);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
        l_part += (ls[0] + ls[1]) + (ls[2] + ls[3]);
        mt = xor32_max(mt);
      }
      s = sn;
    }
    if (safe) break;
    // the flags lie past the waves' output rows
    const int bad = __any(l_part != l_part);  // of all 64 lanes
    lds_barrier();  // the ring is idle
    if (lane == 0) *(__attribute__((address_space(3))) int*)(lds0 + 256 * DV + 4 * w) = bad;
    lds_barrier();
    const u32x4 redo = *(const __attribute__((address_space(3))) u32x4*)(lds0 + 256 * DV);
    if (__builtin_amdgcn_readfirstlane(redo[0] | redo[1] | redo[2] | redo[3]) == 0) break;
    lds_barrier();
    // (a first step that the compiler does not know: no address of this rare
    // pass is kept from the first one, in registers that the loop needs)
    int first = 0;
    asm volatile("" : "+s"(first));
    prologue(first);
  }

  // ---- outputs: lane c's query, dims 32 t + 8 u + 4 hf .. +3, turned into
  // whole rows in the wave's part of the idle ring (16-byte piece j of row r
  // at j ^ (r & 7)), so that every store writes full rows ----
  // (an opaque lane, so that no address of the outputs is kept over the loop)
  int ln = lane;
  asm volatile("" : "+v"(ln));
  const int co = ln & 31, ho = ln >> 5, qo = q0 + 32 * w + co;
  float l = l_part;
  l += __shfl_xor(l, 32, 64);
  const float inv = l > 0.f ? 1.f / l : 0.f;
  if (a.lse != nullptr && ho == 0 && qo < q_len)
    a.lse[(int64_t)h * a.total_q + qs + qo] = l > 0.f ? m_run * a.scale + logf(l) : -INFINITY;
  constexpr int NP16 = DV / 8;  // 16-byte pieces of an output row
  unsigned char* const ow = smem_raw + w * (32 * 2 * DV);
#pragma unroll
  for (int t = 0; t < NDT; t++)
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const u32x2 pk = {pack16<BF16>(oacc[t][4 * u] * inv, oacc[t][4 * u + 1] * inv),
                        pack16<BF16>(oacc[t][4 * u + 2] * inv, oacc[t][4 * u + 3] * inv)};
      *reinterpret_cast<u32x2*>(ow + co * (2 * DV) + 16 * ((4 * t + u) ^ (co & 7)) + 8 * ho) = pk;
    }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the wave's own rows
#pragma unroll
  for (int u = 0; u < NP16 / 2; u++) {
    const int r = (64 / NP16) * u + ln / NP16, j = ln % NP16;
    const u32x4 x = *reinterpret_cast<const u32x4*>(ow + r * (2 * DV) + 16 * (j ^ (r & 7)));
    const int i = q0 + 32 * w + r;
    if (i >= q_len) continue;
    uint16_t* dst = a.o + (int64_t)(qs + i) * a.o_st + (int64_t)h * a.o_sh + 8 * j;
    if (a.o16) {
      *reinterpret_cast<u32x4*>(dst) = x;
    } else {  // an output aligned to 8 bytes only
      *reinterpret_cast<u32x2*>(dst) = (u32x2){x[0], x[1]};
      *reinterpret_cast<u32x2*>(dst + 4) = (u32x2){x[2], x[3]};
    }
  }
}

template <bool BF16, int DQK, int DV>
int launch_ring(const VaArgs& a0, int num_seqs, int max_q_len, hipStream_t st) {
  using R = VaRing<DQK, DV>;
  constexpr int QROWS = 32 * kVaWaves;
  auto kern = varlen_attn_ring_kernel<BF16, DQK, DV>;
  const int lds = R::SLOTS * R::SLOT;
  const int rc = reserve_lds(reinterpret_cast<const void*>(kern), lds, "varlen_attention");
  if (rc) return rc;
  VaArgs a = a0;
  // scale 0 (equal weights): a masked score is -inf and needs a factor above 0
  // to stay one (any other score below 1e31 then counts less than 1e-7)
  if (fabsf(a.scale_log2) < FLT_MIN) a.scale_log2 = FLT_MIN;
  a.n_qtiles = (max_q_len + QROWS - 1) / QROWS;
  if (a.n_qtiles == 0) return MI355_DSA_OK;
  // pair-major order where it leaves no XCD idle (a multiple of 8 pairs, or
  // enough of them that the last round is small: at most one pair in nine
  // runs beside idle XCDs) and a 1-D grid can hold it.  Causal 16k, 64 heads:
  // 5.90 against 6.32 ms with consecutive workgroups on different heads.
  const int64_t pairs = (int64_t)num_seqs * a.H, n1 = (pairs + 7) / 8 * 8 * a.n_qtiles;
  const bool by_pair = (pairs % 8 == 0 || pairs >= 64) && n1 <= (1 << 23);
  a.o16 = aligned_to(a.o, 16) && a.o_st % 8 == 0 && a.o_sh % 8 == 0;
  a.pairs = by_pair ? (int)pairs : 0;
  const dim3 grid = by_pair ? dim3((unsigned)n1) : dim3(a.n_qtiles, num_seqs, a.H);
  kern<<<grid, kVaThreads, lds, st>>>(a);
  return check_launch("varlen_attention");
}

template <bool BF16>
int dispatch_va(const VaArgs& a, int d_qk, int d_v, int num_seqs, int max_q_len, hipStream_t st) {
  // (256, 256): the ring kernel would hold 64 + 128 registers of Q and O per
  // wave beside the scores, one wave per SIMD instead of two
  if (d_qk == 192 && d_v == 128) return launch_ring<BF16, 192, 128>(a, num_seqs, max_q_len, st);
  if (d_qk == 128 && d_v == 128) return launch_ring<BF16, 128, 128>(a, num_seqs, max_q_len, st);
  if (d_qk == 64 && d_v == 64) return launch_ring<BF16, 64, 64>(a, num_seqs, max_q_len, st);
  if (d_qk == 256 && d_v == 256) return launch_va<BF16, 256, 256, 1, 32, 2>(a, num_seqs, max_q_len, st);
  return set_error(MI355_DSA_EINVAL,
                   "varlen_attention: head dims (%d, %d) not built; supported (qk, v): "
                   "(192, 128), (128, 128), (64, 64), (256, 256)", d_qk, d_v);
}

// ---------------------------------------------------------------------------
// fp32 inputs: the same attention in fp32 arithmetic throughout, on the fp32
// MFMA (v_mfma_f32_16x16x4_f32), as the reference computes fp32 inputs
// (sm70_triton.py:193 lists fp32; :54-187 runs it in fp32 torch).  Nothing
// is rounded to 16 bits, so the whole fp32 range is accepted.
//
// Workgroup = (query tile of 64 rows, sequence, head), 4 waves; wave w owns
// query rows [16 w, +16).  Key tiles of 32 keys stream through two LDS
// stages by LDS-DMA (rows at a pitch of d + 4 floats: 16 consecutive rows
// then cover all 64 banks).  Per tile and wave:
//   * S^T = K Q^T: K step j of dims 16 u .. 16 u + 15 takes dim 16 u + 4 g +
//     j from lane group g (one 16-byte LDS read per lane feeds 4 MFMAs); Q
//     is resident in registers in the same dim order;
//   * online softmax per query column (exp2, scale folded in), P kept fp32;
//   * O^T += V^T P^T: MFMA step r of a 16-key block takes key 4 g + r from
//     lane group g, which is element r of that lane's own S^T accumulator,
//     so P never moves; V^T[dim 16 t + c][key] is one fp32 LDS read.
// ---------------------------------------------------------------------------
template <int DQK, int DV>
struct VaShape32 {
  static constexpr int KT = 32;
  static constexpr int PK = DQK / 4 + 1;  // row pitch in 16-B pieces (4 floats), one pad
  static constexpr int PV = DV / 4 + 1;
  static constexpr int RK = (KT * PK + kVaThreads - 1) / kVaThreads;  // DMA rounds
  static constexpr int RV = (KT * PV + kVaThreads - 1) / kVaThreads;
  static constexpr int KBYTES = RK * kVaThreads * 16;
  static constexpr int VBYTES = RV * kVaThreads * 16;
  static constexpr int STAGE = KBYTES + VBYTES;
};

__device__ __forceinline__ f32x4 mma32(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

template <int DQK, int DV>
__global__ void __launch_bounds__(kVaThreads) varlen_attn_f32_kernel(VaArgs a) {
  using Sh = VaShape32<DQK, DV>;
  constexpr int KT = Sh::KT;
  constexpr int NKB = KT / 16;
  constexpr int QROWS = 16 * kVaWaves;
  constexpr int NU = DQK / 16;  // 16-dim groups of the QK product
  constexpr int NDT = DV / 16;  // O^T dim tiles
  constexpr int PKF = 4 * Sh::PK, PVF = 4 * Sh::PV;  // row pitches in floats
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const float* qg = reinterpret_cast<const float*>(a.q);
  const float* kg = reinterpret_cast<const float*>(a.k);
  const float* vg = reinterpret_cast<const float*>(a.v);
  float* og = reinterpret_cast<float*>(a.o);

  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int c = lane & 15, g = lane >> 4;
  const int seq = blockIdx.y, h = blockIdx.z;
  const int qs = a.cu_q[seq], q_len = a.cu_q[seq + 1] - qs;
  const int ks = a.cu_k[seq], k_len = a.cu_k[seq + 1] - ks;
  const int tile = a.causal ? a.n_qtiles - 1 - (int)blockIdx.x : (int)blockIdx.x;
  const int q0 = tile * QROWS;
  if (q0 >= q_len) return;
  const int offset = a.causal ? k_len - q_len : 0;
  const int kend = a.causal ? max(0, min(k_len, q0 + QROWS + offset)) : k_len;
  const int n_kt = (kend + KT - 1) / KT;

  // ---- Q (B operand): row q0 + 16 w + c, dims 16 u + 4 g .. +3 ----
  const int qi = q0 + 16 * w + c;
  f32x4 qf[NU];
  {
    const float* qrow = qg + (int64_t)(qs + (qi < q_len ? qi : 0)) * a.q_st + (int64_t)h * a.q_sh +
                        4 * g;
#pragma unroll
    for (int u = 0; u < NU; u++) qf[u] = *reinterpret_cast<const f32x4*>(qrow + 16 * u);
  }

  auto issue_tile = [&](int kt) {
    unsigned char* st = smem_raw + (kt & 1) * Sh::STAGE;
    const int k0 = kt * KT;
#pragma unroll
    for (int u = 0; u < Sh::RK; u++) {
      const int qq = kVaThreads * u + 64 * w + lane;
      const int r = qq / Sh::PK, ch = qq - r * Sh::PK;
      const bool ok = r < KT && ch < DQK / 4 && k0 + r < kend;
      const void* src = ok ? (const void*)(kg + (int64_t)(ks + k0 + r) * a.k_st +
                                           (int64_t)h * a.k_sh + 4 * ch)
                           : (const void*)kVaZero;
      dma16(src, st + 16 * (kVaThreads * u + 64 * w));
    }
#pragma unroll
    for (int u = 0; u < Sh::RV; u++) {
      const int qq = kVaThreads * u + 64 * w + lane;
      const int r = qq / Sh::PV, ch = qq - r * Sh::PV;
      const bool ok = r < KT && ch < DV / 4 && k0 + r < kend;
      const void* src = ok ? (const void*)(vg + (int64_t)(ks + k0 + r) * a.v_st +
                                           (int64_t)h * a.v_sh + 4 * ch)
                           : (const void*)kVaZero;
      dma16(src, st + Sh::KBYTES + 16 * (kVaThreads * u + 64 * w));
    }
  };

  f32x4 oacc[NDT];
#pragma unroll
  for (int t = 0; t < NDT; t++) oacc[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
  float m_run = -1e30f, l_part = 0.f;

  if (n_kt > 0) issue_tile(0);
#pragma unroll
  for (int u = 0; u < NU; u++) asm volatile("" ::"v"(qf[u]));  // Q lands with tile 0
  const int jmax_q = a.causal ? qi + offset + 1 : kend;  // keys < jmax of this column
  for (int kt = 0; kt < n_kt; kt++) {
    if (kt + 1 < n_kt) {
      issue_tile(kt + 1);
      va_wait<Sh::RK + Sh::RV>();
    } else {
      va_wait<0>();
    }
    lds_barrier();  // tile kt landed for every wave
    const float* kst = reinterpret_cast<const float*>(smem_raw + (kt & 1) * Sh::STAGE);
    const float* vst = reinterpret_cast<const float*>(smem_raw + (kt & 1) * Sh::STAGE + Sh::KBYTES);
    const int k0 = kt * KT;

    // ---- S^T blocks: keys 16 kb + 4 g + r, query column c ----
    f32x4 sacc[NKB];
#pragma unroll
    for (int kb = 0; kb < NKB; kb++) {
      sacc[kb] = (f32x4){0.f, 0.f, 0.f, 0.f};
      const float* krow = kst + (16 * kb + c) * PKF + 4 * g;
#pragma unroll
      for (int u = 0; u < NU; u++) {
        const f32x4 kf = *reinterpret_cast<const f32x4*>(krow + 16 * u);
#pragma unroll
        for (int j = 0; j < 4; j++) sacc[kb] = mma32(kf[j], qf[u][j], sacc[kb]);
      }
    }

    // ---- masks and online softmax of column c ----
    const int jmax = min(kend, jmax_q);
    float mt = -1e30f;
#pragma unroll
    for (int kb = 0; kb < NKB; kb++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        if (k0 + 16 * kb + 4 * g + r >= jmax) sacc[kb][r] = -INFINITY;
        mt = fmaxf(mt, sacc[kb][r]);
      }
    mt = fmaxf(mt, shfl_xor_f(mt, 16));
    mt = fmaxf(mt, shfl_xor_f(mt, 32));
    const float m_new = fmaxf(m_run, mt);
    const float alpha = exp2f((m_run - m_new) * a.scale_log2);
    m_run = m_new;
    const float mb = m_new * a.scale_log2;
    float ls = 0.f;
#pragma unroll
    for (int kb = 0; kb < NKB; kb++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const float sv = sacc[kb][r];
        const float pr = (sv > -INFINITY) ? exp2f(__builtin_fmaf(sv, a.scale_log2, -mb)) : 0.f;
        sacc[kb][r] = pr;
        ls += pr;
      }
    l_part = l_part * alpha + ls;
#pragma unroll
    for (int t = 0; t < NDT; t++) oacc[t] *= alpha;

    // ---- O^T += V^T P^T ----
#pragma unroll
    for (int kb = 0; kb < NKB; kb++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const float* vrow = vst + (16 * kb + 4 * g + r) * PVF + c;
#pragma unroll
        for (int t = 0; t < NDT; t++) oacc[t] = mma32(vrow[16 * t], sacc[kb][r], oacc[t]);
      }
    lds_barrier();  // every wave is done with this stage before it is refilled
  }

  // ---- outputs: O^T rows 4 g + r of tile t are dims 16 t + 4 g + r ----
  float l = l_part;
  l += shfl_xor_f(l, 16);
  l += shfl_xor_f(l, 32);
  if (qi >= q_len) return;
  const float inv = l > 0.f ? 1.f / l : 0.f;
  float* orow = og + (int64_t)(qs + qi) * a.o_st + (int64_t)h * a.o_sh + 4 * g;
#pragma unroll
  for (int t = 0; t < NDT; t++) *reinterpret_cast<f32x4*>(orow + 16 * t) = oacc[t] * inv;
  if (a.lse != nullptr && g == 0)
    a.lse[(int64_t)h * a.total_q + qs + qi] = l > 0.f ? m_run * a.scale + logf(l) : -INFINITY;
}

template <int DQK, int DV>
int launch_va32(const VaArgs& a0, int num_seqs, int max_q_len, hipStream_t st) {
  using Sh = VaShape32<DQK, DV>;
  constexpr int QROWS = 16 * kVaWaves;
  auto kern = varlen_attn_f32_kernel<DQK, DV>;
  const int rc = reserve_lds(reinterpret_cast<const void*>(kern), 2 * Sh::STAGE,
                             "varlen_attention_f32");
  if (rc) return rc;
  VaArgs a = a0;
  a.n_qtiles = (max_q_len + QROWS - 1) / QROWS;
  if (a.n_qtiles == 0) return MI355_DSA_OK;
  kern<<<dim3(a.n_qtiles, num_seqs, a.H), kVaThreads, 2 * Sh::STAGE, st>>>(a);
  return check_launch("varlen_attention_f32");
}

int dispatch_va32(const VaArgs& a, int d_qk, int d_v, int num_seqs, int max_q_len,
                  hipStream_t st) {
  if (d_qk == 192 && d_v == 128) return launch_va32<192, 128>(a, num_seqs, max_q_len, st);
  if (d_qk == 128 && d_v == 128) return launch_va32<128, 128>(a, num_seqs, max_q_len, st);
  if (d_qk == 64 && d_v == 64) return launch_va32<64, 64>(a, num_seqs, max_q_len, st);
  if (d_qk == 256 && d_v == 256) return launch_va32<256, 256>(a, num_seqs, max_q_len, st);
  return set_error(MI355_DSA_EINVAL,
                   "varlen_attention: head dims (%d, %d) not built; supported (qk, v): "
                   "(192, 128), (128, 128), (64, 64), (256, 256)", d_qk, d_v);
}

}  // namespace
}  // namespace mi355dsa

using namespace mi355dsa;

extern "C" int mi355_dsa_varlen_attention(
    void* out, float* lse, const void* q, const void* k, const void* v, int dtype, int num_seqs,
    int n_head, int d_qk, int d_v, int64_t q_tok_stride, int64_t q_head_stride,
    int64_t k_tok_stride, int64_t k_head_stride, int64_t v_tok_stride, int64_t v_head_stride,
    int64_t o_tok_stride, int64_t o_head_stride, const int32_t* cu_seqlens_q,
    const int32_t* cu_seqlens_k, int max_q_len, int total_q, float softmax_scale, int causal,
    void* stream) {
  clear_error();
  DSA_CHECK(num_seqs >= 0 && n_head > 0 && max_q_len >= 0 && total_q >= 0, "varlen_attention: bad sizes");
  if (num_seqs == 0 || max_q_len == 0 || total_q == 0) return MI355_DSA_OK;
  DSA_CHECK(out && q && k && v && cu_seqlens_q && cu_seqlens_k, "varlen_attention: null pointer argument");
  DSA_CHECK(dtype >= 0 && dtype <= 2, "varlen_attention: dtype must be 0 (fp16), 1 (bf16) or 2 (fp32)");
  DSA_CHECK(num_seqs <= 65535 && n_head <= 65535, "varlen_attention: too many sequences or heads");
  const bool f32 = dtype == 2;
  DSA_CHECK(aligned_to(q, 16) && aligned_to(k, 16) && aligned_to(v, 16) &&
                aligned_to(out, f32 ? 16 : 8),
            "varlen_attention: q / k / v must be 16-byte and out %d-byte aligned", f32 ? 16 : 8);
  const int64_t sm = f32 ? 4 : 8;  // elements per 16-byte piece
  DSA_CHECK(q_tok_stride % sm == 0 && q_head_stride % sm == 0 && k_tok_stride % sm == 0 &&
                k_head_stride % sm == 0 && v_tok_stride % sm == 0 && v_head_stride % sm == 0 &&
                o_tok_stride % 4 == 0 && o_head_stride % 4 == 0,
            "varlen_attention: strides must be multiples of %d elements (out: 4)", (int)sm);
  VaArgs a{};
  a.q = reinterpret_cast<const uint16_t*>(q);
  a.k = reinterpret_cast<const uint16_t*>(k);
  a.v = reinterpret_cast<const uint16_t*>(v);
  a.o = reinterpret_cast<uint16_t*>(out);
  a.lse = lse;
  a.cu_q = cu_seqlens_q;
  a.cu_k = cu_seqlens_k;
  a.q_st = q_tok_stride;
  a.q_sh = q_head_stride;
  a.k_st = k_tok_stride;
  a.k_sh = k_head_stride;
  a.v_st = v_tok_stride;
  a.v_sh = v_head_stride;
  a.o_st = o_tok_stride;
  a.o_sh = o_head_stride;
  a.H = n_head;
  a.total_q = total_q;
  a.causal = causal ? 1 : 0;
  a.scale = softmax_scale;
  a.scale_log2 = softmax_scale * 1.4426950408889634f;
  hipStream_t st = as_stream(stream);
  if (f32) return dispatch_va32(a, d_qk, d_v, num_seqs, max_q_len, st);
  return dtype == 1 ? dispatch_va<true>(a, d_qk, d_v, num_seqs, max_q_len, st)
                    : dispatch_va<false>(a, d_qk, d_v, num_seqs, max_q_len, st);
}
