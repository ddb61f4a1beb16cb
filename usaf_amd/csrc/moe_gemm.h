// What the grouped GEMM kernels share (moe_gemm.hip, moe_few.hip, moe_dense.hip,
// wgrad.hip): operands, epilogue codes, the 4-bit dequantization of a fragment and
// the MFMA.
#pragma once

#include "common.h"

namespace usaf {

constexpr int BK = 64;                 // contraction elements of one k-step
constexpr int Q_MAX_E = 255;           // experts the per-wave tile lists cover
constexpr int Q_OVL_WORDS = 64;        // overlay entries per 32-row unit and k-step

enum { EPI_STORE = 0, EPI_SWIGLU_FWD = 1, EPI_SWIGLU_BWD = 2 };

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

struct GemmArgs {
  const uint16_t* A;       // activations, 16-bit, row stride lda
  int64_t lda;
  const int32_t* a_rows;   // A row of slot m (nullptr: row m)
  const uint8_t* wq;       // packed codes of the whole [E, w_rows, w_cols] weight
  const uint32_t* wsz;     // per 128-element group: fp16 scale bits | fp16 zero bits << 16
  const uint16_t* w16;     // dense 16-bit weight [E, w_rows, w_cols] (BQ == BQ_DENSE16)
  const int32_t* w_slot;   // dense weights in an arena: expert e's [w_rows, w_cols] block is
  int64_t n_slots;         //   block w_slot[e] (clamped to [0, n_slots)) of w16; nullptr: block e
  int64_t w_rows, w_cols;  // per-expert weight matrix
  int64_t N, K;            // output columns, contraction length
  int64_t inter;           // I (SwiGLU epilogues)
  const int32_t* offsets;  // [E+1]
  int E;
  uint16_t* out;  int64_t ldo;   // STORE: C; SWIGLU_FWD: act; SWIGLU_BWD: dgu
  uint16_t* out2; int64_t ldo2;  // SWIGLU_FWD: gu
  const uint16_t* aux; int64_t ld_aux;  // SWIGLU_BWD: saved gu
  uint16_t* out_t;                // SWIGLU_FWD (4-bit DMA kernel): act also in the blocked slot-major
  const int32_t* blk_table;       //   layout of blk_table (usaf_hip_blocked_layout), or nullptr
  const uint32_t* ovl;            // 4-bit DMA kernel: overlay entries (usaf_hip_overlay_* layout), or nullptr
  int64_t ovl_words;              //   and their count (checked against what the GEMM reads)
  int w_frag;                     // dense weights (DW): 1 = each expert block in the GEMM's fragment order
  int64_t w_blk_elems;            //   (usaf_hip_dequant_q4_slices_frag) of w_blk_elems elements; 0: w_rows * w_cols
};

// Few slots per expert (moe_few.hip): whether a GEMM over S slots goes to that
// kernel, and its launch.  transposed: wq / wsz are a usaf_hip_q4_transpose copy.
bool few_slots(const GemmArgs& g, int epi, bool transposed, int64_t S);
int launch_few(const GemmArgs& g, int epi, bool transposed, int dt, int64_t S, hipStream_t st, const char* what);

// Dense weights and short m-tiles (moe_dense.hip): whether a GEMM over S slots
// goes to that kernel, and its launch.  kn: the weight is [K, N] (grad-input).
bool dense_slots(const GemmArgs& g, int epi, bool kn, int64_t S, int64_t a_rows_total);
int launch_dense(const GemmArgs& g, int epi, bool kn, int dt, int64_t S, hipStream_t st, const char* what);

namespace {

// Workgroup barrier ordering LDS accesses only.  __syncthreads() also orders
// global memory, which makes every wave drain its outstanding global loads
// (s_waitcnt vmcnt(0)) at each barrier and exposes the full memory latency of
// the prefetched k-steps; no thread here communicates through global memory.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Block of the dense weight operand that holds expert e: e itself, or its
// arena slot (clamped, so a stale table can give wrong weights but never an
// access outside the arena).
__device__ __forceinline__ int64_t weight_block(const GemmArgs& g, int e) {
  if (g.w_slot == nullptr) return e;
  const int64_t s = g.w_slot[e];
  return s < 0 ? 0 : (s >= g.n_slots ? g.n_slots - 1 : s);
}

// m-tile mt of the list (experts in order, each in tiles of SLOTS) -> expert,
// first slot, slots; false past the end.  One wave, offsets from global
// memory: lane l counts the tiles of experts 4 l .. 4 l + 3 (E <= 255).
template <int SLOTS>
__device__ __forceinline__ bool slot_tile(const GemmArgs& g, int lane, int mt, int& e, int& m_beg, int& valid) {
  int off[5], c[4], sum = 0;
#pragma unroll
  for (int k = 0; k < 5; ++k) {
    const int i = 4 * lane + k;
    off[k] = g.offsets[i < g.E ? i : g.E];
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    c[k] = (off[k + 1] - off[k] + SLOTS - 1) / SLOTS;
    sum += c[k];
  }
  int incl = sum;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int o = __shfl_up(incl, d, 64);
    if (lane >= d) incl += o;
  }
  const uint64_t past = __ballot(incl > mt);  // lanes at or after the owner
  if (past == 0) return false;
  const int src = __builtin_ctzll(past);
  int j = mt - (incl - sum), ee = 4 * lane, beg = off[0], end = off[1];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    if (ee == 4 * lane + k && j >= c[k]) {  // past expert 4 l + k
      j -= c[k];
      ee = 4 * lane + k + 1;
      beg = off[k + 1];
      end = off[k + 2];
    }
  }
  e = __builtin_amdgcn_readlane(ee, src);
  m_beg = __builtin_amdgcn_readlane(beg + j * SLOTS, src);
  const int rem = __builtin_amdgcn_readlane(end, src) - m_beg;
  valid = rem < SLOTS ? rem : SLOTS;
  return true;
}

__device__ __forceinline__ uint32_t h2_to_bf2(uint32_t h2) {
  const f16x2 h = __builtin_bit_cast(f16x2, h2);
  const f32x2 f = {(float)h.x, (float)h.y};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, bf16x2));
}

// 8 codes of one 32-bit word (code 2i in the low nibble of byte i) -> 8 16-bit
// weights in natural order, bit-identical to dequantize_4bit:
// fp16(fp16(q * s) + z), then RNE bf16 for bf16 operands.
template <int DT>
__device__ __forceinline__ u32x4 dq8(uint32_t w, f16x2 s2, f16x2 z2) {
#pragma clang fp contract(off)
  const f16x2 mul = {(f16)1.0f, (f16)0.0625f};
  const f16x2 sub = {(f16)-1024.0f, (f16)-64.0f};
  uint32_t o[4];
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    // byte p in both halves: the low half keeps code 2p (bits 0-3), the high half
    // code 2p+1 (bits 20-23), as fp16 1024 + q and 1024 + 16 q
    const uint32_t t = __builtin_amdgcn_perm(w, w, 0x0C000C00u | ((uint32_t)p << 16) | (uint32_t)p);
    const uint32_t bits = (t & 0x00F0000Fu) | 0x64006400u;
    const f16x2 q = __builtin_elementwise_fma(__builtin_bit_cast(f16x2, bits), mul, sub);  // exact codes
    const f16x2 m = q * s2;
    const f16x2 v = m + z2;
    o[p] = __builtin_bit_cast(uint32_t, v);
    if constexpr (DT == USAF_BF16) o[p] = h2_to_bf2(o[p]);
  }
  return u32x4{o[0], o[1], o[2], o[3]};
}

// Codes 2p, 2p+1 of a 32-bit code word (byte p) -> their two 16-bit weights
// (dq8 for one pair).  v_perm places byte p under the fp16 exponent byte 0x64 in
// both halves; the mask keeps code 2p in the low half (1024 + q) and code 2p+1
// in the high half (1024 + 16 q).
template <int DT>
__device__ __forceinline__ uint32_t dq_pair(uint32_t w, int p, f16x2 s2, f16x2 z2) {
#pragma clang fp contract(off)
  const f16x2 mul = {(f16)1.0f, (f16)0.0625f};
  const f16x2 sub = {(f16)-1024.0f, (f16)-64.0f};
  const uint32_t t = __builtin_amdgcn_perm(0x64646464u, w, 0x04000400u | ((uint32_t)p << 16) | (uint32_t)p) & 0xFFF0FF0Fu;
  const f16x2 q = __builtin_elementwise_fma(__builtin_bit_cast(f16x2, t), mul, sub);  // exact codes
  const f16x2 m = q * s2;
  const f16x2 v = m + z2;
  uint32_t o = __builtin_bit_cast(uint32_t, v);
  if constexpr (DT == USAF_BF16) o = h2_to_bf2(o);
  return o;
}

// silu(x) = x / (1 + e^-x) with the hardware exp2 and reciprocal (about 1 ulp
// of fp32 each, far below the 16-bit rounding that follows)
__device__ __forceinline__ float silu_fast(float x) {
  return x * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * x));
}

template <int DT>
__device__ __forceinline__ f32x16 mfma32(const u32x4 a, const u32x4 b, f32x16 c) {
  if constexpr (DT == USAF_BF16)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                   0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c,
                                                  0, 0, 0);
}

}  // namespace
}  // namespace usaf
