// Grouped (per-expert) GEMM on dense 16-bit weights for short m-tiles:
//
//   C[m, n] = sum_k A[row(m), k] * W_e[n, k]   (forward; W_e [N, K] rows or fragment order)
//   C[m, n] = sum_k A[m, k] * W_e[k, n]        (grad-input; W_e [K, N] rows)
//
// With tens of slots per expert the weights are the traffic, and bytes in flight
// set the rate.
// * A block is four waves: 256 weight rows x up to 32 NM slots of one expert.  Two
//   blocks share a CU, each with its own barriers.
// * Weights go straight from global memory into MFMA fragments, a k-step ahead:
//   each element feeds one lane.  A [K, N] weight is read as dwords (two
//   columns) of eight k each, and byte permutes turn a lane's eight dwords into the
//   fragments of its even and its odd column; no transpose through LDS.
// * Activations are staged once per block through two LDS stages.
// * NM = 4 (3 for [K, N], whose raw dwords and fragments would spill at 4: d(act) at
//   64 slots 94 against 68 us).  A k-step (64 KB a CU) in flight does as
//   well as three sets of registers at NM = 2 or 3 (153 against 155, 175 us).
// Measured (kernel trace of a training pass, OLMoE, 512 tokens, bf16, us, gate_up / down /
// d(act) / d(x); floor: the weights at 6 TB/s, 89 / 45 / 45 / 89; before: the persistent
// kernels): 188 / 82 / 124 / 227 -> 117 / 66 / 69 / 105.
#include "moe_gemm.h"

#include <type_traits>

namespace usaf {
namespace {

constexpr int DN_THREADS = 256, DN_WAVES = 4, DN_XCDS = 8;
enum { W_ROWS = 0, W_FRAG = 1, W_KN = 2 };  // [N, K] rows, fragment order (both 32-row units), [K, N] rows

template <int NM, int EPI, int DT, int WM>
__global__ __launch_bounds__(DN_THREADS, 2) void moe_dense_kernel(const GemmArgs g, int per, int chunks) {
  constexpr int SLOTS = 32 * NM, STAGE = SLOTS * BK * 2;
  __shared__ __attribute__((aligned(16))) uint8_t sm[2 * STAGE];
  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // XCD-aware order (blocks are dispatched round-robin over the dies): an m-tile's
  // blocks come in `chunks` runs of `per`, each run on one die
  const int grp = ((int)blockIdx.x / (DN_XCDS * per)) * DN_XCDS + (int)blockIdx.x % DN_XCDS;
  const int mt = grp / chunks;
  const int nb_i = (grp - mt * chunks) * per + (int)blockIdx.x / DN_XCDS % per;
  int e, m_beg, valid;
  if (!slot_tile<SLOTS>(g, lane, mt, e, m_beg, valid)) return;  // block-uniform
  constexpr int UNIT = EPI == EPI_SWIGLU_FWD ? 16 : 32;  // output columns of one 32-row unit
  if ((int64_t)nb_i * DN_WAVES * 2 * UNIT >= g.N) return;  // block-uniform
  // the wave's two units; a wave past the columns reads unit pair 0 and stores nothing
  const int pair = nb_i * DN_WAVES + wave;
  const bool wave_on = (int64_t)pair * 2 * UNIT < g.N;
  const int pw = wave_on ? pair : 0;
  const int nblk = (valid + 31) >> 5;
  const int nk = (int)(g.K / BK);

  // W_ROWS: the blocks start at different k-steps.  Rows of a power-of-two length
  // put one k-step of every row on the same few memory channels, and blocks that
  // walk together all wait for those (OLMoE gate_up, rows of 4 KiB: 182 -> 153 us).
  // The other two orders spread by themselves and lose the L2's sharing of the
  // activations instead (fragment order at 2,048 tokens: 883 -> 948 us a pass).
  const int rot = WM == W_ROWS ? (int)(blockIdx.x % (unsigned)nk) : 0;
  // i-th k-step of the block; past the end the last one again, unused
  auto k_at = [&](int i) {
    const int kt = (i < nk ? i : nk - 1) + rot;
    return kt < nk ? kt : kt - nk;
  };
  const int64_t blk = g.w_blk_elems ? g.w_blk_elems : g.w_rows * g.w_cols;
  const uint8_t* const wb = reinterpret_cast<const uint8_t*>(g.w16) + weight_block(g, e) * blk * 2;
  uint32_t w_off[2];  // lane byte offsets within the block at k-step 0
  const uint32_t n2 = (uint32_t)(g.N * 2);
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    if constexpr (WM == W_KN) w_off[u] = (uint32_t)(32 * half) * n2 + (uint32_t)(pw * 64 + 2 * l32) * 2;
    else if constexpr (WM == W_FRAG) w_off[u] = (uint32_t)(2 * pw + u) * (uint32_t)nk * 4096u + 16u * (uint32_t)lane;
    else {
      int64_t row = (int64_t)(2 * pw + u) * UNIT + l32;
      if constexpr (EPI == EPI_SWIGLU_FWD) row += l32 >= 16 ? g.inter - 16 : 0;
      w_off[u] = (uint32_t)(row * g.K * 2) + 64u * (uint32_t)half;
    }
  }
  // activations: thread t stages chunk t & 7 of rows 32 i + (t >> 3)
  uint32_t a_off[NM];
#pragma unroll
  for (int i = 0; i < NM; ++i) {
    const int r = 32 * i + (tid >> 3);
    const int m = m_beg + (r < valid ? r : valid - 1);
    const uint32_t arow = (uint32_t)(g.a_rows ? g.a_rows[m] : m);
    a_off[i] = arow * (uint32_t)(g.lda * 2) + 16u * (uint32_t)(tid & 7);
  }
  const uint8_t* const A = reinterpret_cast<const uint8_t*>(g.A);
  // rows of 128 bytes whose 16-byte chunk c sits at c ^ ((row >> 1) & 7)
  const int a_lds = (tid >> 3) * 128 + 16 * ((tid & 7) ^ ((tid >> 4) & 7));
  const int swz = (l32 >> 1) & 7;

  u32x4 wf[2][2][4], ar[NM];  // W_KN: the dword of k = 8 j + t is wf[.][t >> 2][j][t & 3]
  auto load_w = [&](auto set, int kt) {
    constexpr int X = decltype(set)::value;
    kt = k_at(kt);
    if constexpr (WM == W_KN) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int t = 0; t < 8; ++t)
          wf[X][t >> 2][j][t & 3] =
              *reinterpret_cast<const uint32_t*>(wb + (int64_t)(kt * BK + 8 * j + t) * n2 + w_off[0]);
    } else {
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          wf[X][u][j] = *reinterpret_cast<const u32x4*>(
              wb + (int64_t)kt * (WM == W_FRAG ? 4096 : BK * 2) + j * (WM == W_FRAG ? 1024 : 16) + w_off[u]);
    }
  };
  auto load_a = [&](int kt) {
    kt = k_at(kt);
#pragma unroll
    for (int i = 0; i < NM; ++i)
      if (i < nblk) ar[i] = *reinterpret_cast<const u32x4*>(A + (int64_t)kt * (BK * 2) + a_off[i]);
  };
  auto store_a = [&](int st) {
#pragma unroll
    for (int i = 0; i < NM; ++i)
      if (i < nblk) *reinterpret_cast<u32x4*>(sm + st * STAGE + 4096 * i + a_lds) = ar[i];
  };

  f32x16 acc[2][NM];
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int i = 0; i < NM; ++i) acc[u][i] = f32x16{};

  // k-step kt: stage kt & 1 and set X hold it, ar the activations of kt + 1.  The
  // other stage was last read before the barrier that ended step kt - 1.
  auto step = [&](auto set, int kt) {
    constexpr int X = decltype(set)::value;
    store_a((kt + 1) & 1);
    load_a(kt + 2);
    load_w(std::integral_constant<int, X ^ 1>{}, kt + 1);
    // the loads stay here, ahead of the products (the scheduler sinks them to their use)
    __builtin_amdgcn_sched_barrier(0);
    u32x4 w[2][4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if constexpr (WM == W_KN) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {  // k = 2 q, 2 q + 1 of the eight
          const uint32_t k0 = wf[X][q >> 1][j][(2 * q) & 3], k1 = wf[X][q >> 1][j][(2 * q + 1) & 3];
          w[0][j][q] = __builtin_amdgcn_perm(k1, k0, 0x05040100u);
          w[1][j][q] = __builtin_amdgcn_perm(k1, k0, 0x07060302u);
        }
      } else {
        w[0][j] = wf[X][0][j];
        w[1][j] = wf[X][1][j];
      }
    }
    const uint8_t* const sa = sm + (kt & 1) * STAGE + 128 * l32;
#pragma unroll
    for (int i = 0; i < NM; ++i) {
      if (i >= nblk) break;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const u32x4 af = *reinterpret_cast<const u32x4*>(sa + 4096 * i + 16 * ((4 * half + j) ^ swz));
        acc[0][i] = mfma32<DT>(w[0][j], af, acc[0][i]);
        acc[1][i] = mfma32<DT>(w[1][j], af, acc[1][i]);
      }
    }
    lds_barrier();
  };
  load_a(0);
  load_w(std::integral_constant<int, 0>{}, 0);
  store_a(0);
  load_a(1);
  lds_barrier();
  for (int kt = 0; kt < nk; kt += 2) {
    step(std::integral_constant<int, 0>{}, kt);
    if (kt + 1 < nk) step(std::integral_constant<int, 1>{}, kt + 1);
  }
  if (!wave_on) return;

  // acc[u][i][4 q + k]: row 8 q + 4 half + k of unit u, slot 32 i + l32
#pragma unroll
  for (int i = 0; i < NM; ++i) {
    if (i >= nblk) break;
    const bool live = 32 * i + l32 < valid;
    const int64_t m = (int64_t)m_beg + 32 * i + l32;
    if constexpr (EPI == EPI_SWIGLU_FWD) {
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const int64_t n = (int64_t)(2 * pair + u) * 16 + 8 * q + 4 * half;
          uint32_t gb[2], ub[2], ab[2];
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            gb[h] = pack2<DT>(acc[u][i][4 * q + 2 * h], acc[u][i][4 * q + 2 * h + 1]);
            ub[h] = pack2<DT>(acc[u][i][8 + 4 * q + 2 * h], acc[u][i][8 + 4 * q + 2 * h + 1]);
            const f32x2 gf = unpack2<DT>(gb[h]), uf = unpack2<DT>(ub[h]);
            const f32x2 sf = unpack2<DT>(pack2<DT>(silu_fast(gf.x), silu_fast(gf.y)));
            ab[h] = pack2<DT>(sf.x * uf.x, sf.y * uf.y);
          }
          if (live) {
            *reinterpret_cast<uint2*>(g.out2 + m * g.ldo2 + n) = uint2{gb[0], gb[1]};
            *reinterpret_cast<uint2*>(g.out2 + m * g.ldo2 + g.inter + n) = uint2{ub[0], ub[1]};
            *reinterpret_cast<uint2*>(g.out + m * g.ldo + n) = uint2{ab[0], ab[1]};
          }
        }
    } else if constexpr (WM == W_KN) {
      // the even columns are unit 0's rows, the odd ones unit 1's: 8 columns in a row
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int64_t n = (int64_t)pair * 64 + 16 * q + 8 * half;
        u32x4 v;
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] = pack2<DT>(acc[0][i][4 * q + k], acc[1][i][4 * q + k]);
        if (!live) continue;
        if constexpr (EPI == EPI_STORE) {
          *reinterpret_cast<u32x4*>(g.out + m * g.ldo + n) = v;
        } else {  // d(act) -> d(gate), d(up) with moe_gemm_kernel's roundings
          const u32x4 gv = *reinterpret_cast<const u32x4*>(g.aux + m * g.ld_aux + n);
          const u32x4 uv = *reinterpret_cast<const u32x4*>(g.aux + m * g.ld_aux + g.inter + n);
          u32x4 dg, du;
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const f32x2 da = unpack2<DT>(v[k]), gt = unpack2<DT>(gv[k]), up = unpack2<DT>(uv[k]);
            const float s0 = 1.0f / (1.0f + expf(-gt.x)), s1 = 1.0f / (1.0f + expf(-gt.y));
            const f32x2 sg = unpack2<DT>(pack2<DT>(gt.x * s0, gt.y * s1));
            const f32x2 ds = unpack2<DT>(pack2<DT>(da.x * up.x, da.y * up.y));
            dg[k] = pack2<DT>((ds.x * s0) * (1.0f + gt.x * (1.0f - s0)), (ds.y * s1) * (1.0f + gt.y * (1.0f - s1)));
            du[k] = pack2<DT>(da.x * sg.x, da.y * sg.y);
          }
          *reinterpret_cast<u32x4*>(g.out + m * g.ldo + n) = dg;
          *reinterpret_cast<u32x4*>(g.out + m * g.ldo + g.inter + n) = du;
        }
      }
    } else {
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int64_t n = (int64_t)(2 * pair + u) * 32 + 8 * q + 4 * half;
          if (live)
            *reinterpret_cast<uint2*>(g.out + m * g.ldo + n) =
                uint2{pack2<DT>(acc[u][i][4 * q], acc[u][i][4 * q + 1]),
                      pack2<DT>(acc[u][i][4 * q + 2], acc[u][i][4 * q + 3])};
        }
    }
  }
}

template <int NM, int EPI, int DT, int WM>
void launch_dense_one(const GemmArgs& g, int64_t S, hipStream_t st) {
  const int64_t cols = DN_WAVES * 2 * (EPI == EPI_SWIGLU_FWD ? 16 : 32);
  const int64_t nb = (g.N + cols - 1) / cols;
  const int64_t m_tiles = (S < g.E ? S : g.E) + S / (32 * NM);
  const int64_t chunks = nb < 2 ? nb : 2, per = (nb + chunks - 1) / chunks;
  const int64_t blocks = (m_tiles * chunks + DN_XCDS - 1) / DN_XCDS * DN_XCDS * per;
  moe_dense_kernel<NM, EPI, DT, WM><<<(unsigned)blocks, DN_THREADS, 0, st>>>(g, (int)per, (int)chunks);
}

template <int EPI, int DT, int WM>
int launch_dense_dt(const GemmArgs& g, int64_t S, hipStream_t st, const char* what) {
  launch_dense_one<WM == W_KN ? 3 : 4, EPI, DT, WM>(g, S, st);
  return check_launch(what);
}

template <int EPI, int WM>
int launch_dense_epi(const GemmArgs& g, int dt, int64_t S, hipStream_t st, const char* what) {
  if (dt == USAF_BF16) return launch_dense_dt<EPI, USAF_BF16, WM>(g, S, st, what);
  if (dt == USAF_F16) return launch_dense_dt<EPI, USAF_F16, WM>(g, S, st, what);
  return set_error(USAF_ERR_INVALID, "%s: dtype must be fp16 or bf16", what);
}

}  // namespace

// The lines against the persistent kernels (moe_gemm.hip), in slots per expert on
// average.  Measured, those kernels / this one, us; a uniform routing, Zipf(1.1):
// * [N, K] rows, gate_up + down with cold weights, 80 slots: OLMoE 244 / 185, 325 / 257,
//   Qwen3 357 / 291, 422 / 378; warm, OLMoE at 128 slots, uniform: 288 / 316 (experts past
//   128 slots take a second m-tile and read their weights again).
// * Fragment order, passes of two Qwen3 layers: 772 / 682, 840 / 716 at 64 slots; at 128
//   849 / 883, 956 / 877 and with another Zipf routing 936 / 933; at 256 1294 / 1321, 1277 / 1201.
//   How the slots spread decides, which their average does not tell: the line stays
//   where both win.
// * [K, N], d(act) + d(x) with cold weights, 128 slots: OLMoE 367 / 304, 469 / 262, Qwen3
//   511 / 447, 624 / 396; warm, OLMoE at 256 slots, uniform: 402 / 475.
// With every token on the same eight experts a 128-slot m-tile reads their weights
// more often than the persistent kernels' 256-slot ones: 640 OLMoE tokens, gate_up +
// down 126 / 159 in rows, 103 / 123 in fragment order.
bool dense_slots(const GemmArgs& g, int epi, bool kn, int64_t S, int64_t a_rows_total) {
  const int64_t lim = kn ? 128 : g.w_frag ? 96 : 80;
  const int64_t cols = epi == EPI_SWIGLU_FWD ? 32 : 64;
  if (S > lim * g.E || g.E > Q_MAX_E || g.N % cols != 0 || g.K % BK != 0) return false;
  if (((uintptr_t)g.A & 15) || g.lda % 8 != 0 || a_rows_total * g.lda * 2 >= ((int64_t)1 << 32)) return false;
  if (kn && g.w_rows * g.w_cols * 2 >= ((int64_t)1 << 32)) return false;
  return ((int64_t)g.E + S / 32 + DN_XCDS) * 2 * (g.N / cols + 2) < ((int64_t)1 << 30);  // blocks of a launch
}

int launch_dense(const GemmArgs& g, int epi, bool kn, int dt, int64_t S, hipStream_t st, const char* what) {
  if (epi == EPI_SWIGLU_BWD) return launch_dense_epi<EPI_SWIGLU_BWD, W_KN>(g, dt, S, st, what);
  if (kn) return launch_dense_epi<EPI_STORE, W_KN>(g, dt, S, st, what);
  if (epi == EPI_SWIGLU_FWD)
    return g.w_frag ? launch_dense_epi<EPI_SWIGLU_FWD, W_FRAG>(g, dt, S, st, what)
                    : launch_dense_epi<EPI_SWIGLU_FWD, W_ROWS>(g, dt, S, st, what);
  return g.w_frag ? launch_dense_epi<EPI_STORE, W_FRAG>(g, dt, S, st, what)
                  : launch_dense_epi<EPI_STORE, W_ROWS>(g, dt, S, st, what);
}

}  // namespace usaf
