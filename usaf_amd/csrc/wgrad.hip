// Dense weight gradients of the routed experts:
//   out[e, r, c] = dtype( sum_{slots s of e} fp32(dy[s, r]) * fp32(x[row(s), c]) )
// for every expert (zeros for one without slots): autograd of the reference's
// expert loop for trainable experts (usaf/olmoe_dml.py:22-31).
//
// The contraction is short (tens to hundreds of slots), so the output is what
// bounds it: OLMoE's 64 x 2048 x 2048 bf16 gradient is 537 MB, 90 us at 6 TB/s,
// against 34 GFLOP (22 us at 1.57 PFLOP/s) for 512 tokens.
// * A block computes 128 rows x 128 columns of one expert; its four waves take 32
//   rows each x all columns (64 accumulators a lane).  Blocks of one expert run on
//   one die (when the experts divide evenly), which then holds its 0.5 MB of dy and
//   x in its L2 for all of them.
// * 64 slots at a time, both operands are transposed through LDS (tt_write) into
//   fragments of 8 consecutive slots; the next 64 are in flight meanwhile.  x is
//   the MFMA's A operand: a lane's accumulator holds 4 consecutive columns of one row.
// * 16-bit results leave through LDS as whole 128-byte row segments, stored
//   non-temporally: nothing reads them soon, and kept in the caches they evict the
//   operands the die's other blocks share (dense training pass 742 -> 664 us).
// Measured (kernel trace of a training pass, OLMoE, 512 tokens, bf16, both tensors): 251
// us, 3.2 TB/s written; the per-expert fp32 library products, gathers and casts it
// replaces took 4.3 ms in 770 launches.
#include "moe_gemm.h"

#include <type_traits>

namespace usaf {
namespace {

constexpr int WG_TILE = 128, WG_XCDS = 8;
constexpr int WG_EPW = 72;  // staging row stride, 16-bit elements (64 columns; rows stay 16-byte aligned)
static_assert(4 * 32 * WG_EPW * 2 <= 4 * TT_DWORDS * 4, "the waves' staging tiles fit the operand tiles");

template <int DT, int OT>
__global__ __launch_bounds__(256) void weight_grad_kernel(const uint16_t* __restrict__ dy, const uint16_t* __restrict__ x,
                                                          const int32_t* __restrict__ x_rows,
                                                          const int32_t* __restrict__ offsets, int E, int64_t R,
                                                          int64_t C, int tiles_r, int tiles_c, void* __restrict__ out) {
  __shared__ __align__(16) uint32_t tiles[4][TT_DWORDS];  // dy rows 0-63, 64-127 | x columns 0-63, 64-127
  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, half = lane >> 5, wave = tid >> 6;
  const int per = tiles_r * tiles_c;
  int e, tile;
  if (E % WG_XCDS == 0) {  // blocks are dispatched round-robin over the dies
    const int i = (int)blockIdx.x / WG_XCDS;
    e = i / per * WG_XCDS + (int)blockIdx.x % WG_XCDS;
    tile = i % per;
  } else {
    e = (int)blockIdx.x / per;
    tile = (int)blockIdx.x % per;
  }
  const int64_t r0 = (int64_t)(tile / tiles_c) * WG_TILE, c0 = (int64_t)(tile % tiles_c) * WG_TILE;
  const int s_beg = offsets[e], s_end = offsets[e + 1];
  const int sp = tid >> 3, cg = tid & 7;  // writer cell: slots 2 sp, 2 sp + 1 of 64; 8 features at 8 cg
  f32x16 acc[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) acc[j] = f32x16{};
  uint4 ra[2][2], rb[2][2];  // [64 features][slot of the pair]
  auto load = [&](int s0) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int s = s0 + 2 * sp + u;
      const bool in = s < s_end;
      const int64_t xr = in ? (x_rows ? (int64_t)x_rows[s] : (int64_t)s) : 0;
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int64_t r = r0 + 64 * q + 8 * cg, c = c0 + 64 * q + 8 * cg;
        ra[q][u] = in && r < R ? *reinterpret_cast<const uint4*>(dy + (int64_t)s * R + r) : make_uint4(0, 0, 0, 0);
        rb[q][u] = in && c < C ? *reinterpret_cast<const uint4*>(x + xr * C + c) : make_uint4(0, 0, 0, 0);
      }
    }
  };
  if (s_beg < s_end) load(s_beg);
  for (int s0 = s_beg; s0 < s_end; s0 += 64) {
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      tt_write(tiles[q], sp, cg, ra[q][0], ra[q][1]);
      tt_write(tiles[2 + q], sp, cg, rb[q][0], rb[q][1]);
    }
    __syncthreads();
    if (s0 + 64 < s_end) load(s0 + 64);
    const int row = 32 * wave + l32;  // this lane's row of the tile
#pragma unroll
    for (int kb = 0; kb < 64; kb += 16) {
      const int sg = (kb >> 3) + half;
      const u32x4 b = __builtin_bit_cast(u32x4, tt_read(tiles[row >> 6], row & 63, sg));
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int col = 32 * j + l32;
        const u32x4 a = __builtin_bit_cast(u32x4, tt_read(tiles[2 + (col >> 6)], col & 63, sg));
        acc[j] = mfma32<DT>(a, b, acc[j]);
      }
    }
    __syncthreads();
  }
  // acc[j][4 q + k]: row r0 + 32 wave + l32, column c0 + 32 j + 8 q + 4 half + k
  const int64_t row0 = r0 + 32 * wave;
  if constexpr (OT == USAF_F32) {
    float* const o = reinterpret_cast<float*>(out) + ((int64_t)e * R + row0 + l32) * C + c0;
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int64_t c = 32 * j + 8 * q + 4 * half;
        if (row0 + l32 < R && c0 + c < C)
          *reinterpret_cast<f32x4*>(o + c) =
              f32x4{acc[j][4 * q], acc[j][4 * q + 1], acc[j][4 * q + 2], acc[j][4 * q + 3]};
      }
  } else {
    uint16_t* const ep = reinterpret_cast<uint16_t*>(tiles) + wave * 32 * WG_EPW;  // the wave's own
    uint16_t* const o = reinterpret_cast<uint16_t*>(out) + (int64_t)e * R * C;
#pragma unroll
    for (int p = 0; p < 2; ++p) {  // 64 columns
#pragma unroll
      for (int jj = 0; jj < 2; ++jj)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const f32x16& v = acc[2 * p + jj];
          *reinterpret_cast<uint2*>(ep + l32 * WG_EPW + 32 * jj + 8 * q + 4 * half) =
              make_uint2(pack2<OT>(v[4 * q], v[4 * q + 1]), pack2<OT>(v[4 * q + 2], v[4 * q + 3]));
        }
      __builtin_amdgcn_wave_barrier();  // one wave's LDS operations complete in order
#pragma unroll
      for (int k = 0; k < 4; ++k) {  // lane: 16-byte chunk lane & 7 of rows 8 k + (lane >> 3)
        const int rr = 8 * k + (lane >> 3);
        const int64_t c = c0 + 64 * p + 8 * (lane & 7);
        if (row0 + rr < R && c < C)
          __builtin_nontemporal_store(*reinterpret_cast<const u32x4*>(ep + rr * WG_EPW + 8 * (lane & 7)),
                                      reinterpret_cast<u32x4*>(o + (row0 + rr) * C + c));
      }
      __builtin_amdgcn_wave_barrier();
    }
  }
}

template <int DT, int OT>
void launch_wgrad(const void* dy, const void* x, const int32_t* x_rows, const int32_t* offsets, int64_t E, int64_t R,
                  int64_t C, int64_t tr, int64_t tc, void* out, hipStream_t st) {
  weight_grad_kernel<DT, OT><<<(unsigned)(E * tr * tc), 256, 0, st>>>((const uint16_t*)dy, (const uint16_t*)x, x_rows,
                                                                      offsets, (int)E, R, C, (int)tr, (int)tc, out);
}

}  // namespace
}  // namespace usaf

using namespace usaf;

extern "C" int usaf_hip_moe_weight_grad(const void* dy, const void* x, const int32_t* x_rows, const int32_t* offsets,
                                        int64_t E, int64_t R, int64_t C, int32_t dtype, void* out, int32_t out_dtype,
                                        void* stream) {
  if (E <= 0 || R <= 0 || C <= 0) return set_error(USAF_ERR_INVALID, "moe_weight_grad: bad sizes");
  if (dtype != USAF_F16 && dtype != USAF_BF16)
    return set_error(USAF_ERR_INVALID, "moe_weight_grad: dtype must be fp16 or bf16");
  if (!dy || !x || !offsets || !out) return set_error(USAF_ERR_INVALID, "moe_weight_grad: null pointer");
  if (R % 8 != 0 || C % 8 != 0 || (((uintptr_t)dy | (uintptr_t)x | (uintptr_t)out) & 15))
    return set_error(USAF_ERR_UNSUPPORTED,
                     "moe_weight_grad: needs rows and columns in multiples of 8 and 16-byte aligned operands");
  const int64_t tr = (R + WG_TILE - 1) / WG_TILE, tc = (C + WG_TILE - 1) / WG_TILE;
  if (E > 0x7fffffff || tr > 0x7fffff || tc > 0x7fffff || E * tr * tc > 0x7fffffff)
    return set_error(USAF_ERR_INVALID, "moe_weight_grad: too large");
  hipStream_t st = as_stream(stream);
  auto go = [&](auto dt) -> int {
    constexpr int DT = decltype(dt)::value;
    switch (out_dtype) {
      case USAF_F32: launch_wgrad<DT, USAF_F32>(dy, x, x_rows, offsets, E, R, C, tr, tc, out, st); break;
      case USAF_F16: launch_wgrad<DT, USAF_F16>(dy, x, x_rows, offsets, E, R, C, tr, tc, out, st); break;
      case USAF_BF16: launch_wgrad<DT, USAF_BF16>(dy, x, x_rows, offsets, E, R, C, tr, tc, out, st); break;
      default: return set_error(USAF_ERR_INVALID, "moe_weight_grad: unknown out_dtype %d", (int)out_dtype);
    }
    return check_launch("moe_weight_grad");
  };
  if (dtype == USAF_BF16) return go(std::integral_constant<int, USAF_BF16>{});
  return go(std::integral_constant<int, USAF_F16>{});
}
