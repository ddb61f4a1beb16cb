// Grouped (per-expert) GEMM for few slots per expert: decoding, small batches,
// short training sequences.
//
//   C[m, n] = sum_k A[row(m), k] * W_e[n, k]      (slots m of expert e)
//
// The same product, weights, overlays and epilogues as moe_gemm_q4_kernel
// (moe_gemm.hip), for the sizes at which that kernel is bound by its own
// per-tile costs: a tile of it is 256 weight rows on one CU whatever the slots,
// so eight experts of one token fill 48 of 256 CUs, and a tile of a few slots
// pays the ring, the barriers and the dequantization schedule of a full one.
//
// * A tile is NU units of 32 weight rows of one expert x up to 32 of its slots.
//   ks = 1, 2 or 4 waves of a block split its contraction (in groups of 128);
//   the block's other waves have the next rows.  Partial tiles are summed in LDS
//   in wave order.  Each wave works alone until then: no barrier in its loop.
// * Codes go straight from global memory to registers, a group ahead: a row's 16
//   code bytes are exactly what one lane dequantizes.
// * A wave reads its activation rows in whole 128-byte lines, a k-step ahead, and
//   turns them into MFMA fragments through 4 KiB of LDS of its own.  Rows past
//   the expert's last slot repeat it.
// * The fragment assignment is moe_gemm_q4_kernel's -- lane l32 + 32 h holds
//   k = 32 h + 8 j + [0, 8) of row l32 in register j -- so the overlay tables
//   serve both kernels.
//
// What bounds it: the dequantization and, below it, whole rounds of blocks.  All
// 128 experts of a Qwen3 layer's gate_up are 25 M wave instructions in bf16 (8 a pair
// of weights), 43 us of the VALU, and 33 us of reading 214 MB at 6.5 TB/s; the 97
// experts of 24 tokens take 67 us, all 128 at 256 tokens 86.  Measured with cold
// weights (us, moe_gemm_q4_kernel / this one; gate_up, down, d(act), d(x)):
//   Qwen3, 24 tokens, bf16       116 / 67, 63 / 41, 78 / 48, 110 / 75
//   Qwen3, 320 tokens, bf16      119 / 88, 66 / 48, 81 / 54, 115 / 85
//   Qwen3, 256, fp16, overlay    136 / 103, 73 / 58, 89 / 72, 134 / 110
//   Mixtral, 40 tokens, bf16     311 / 182, 265 / 101, 138 / 99, 431 / 173
// and one token, warm, 36 / 10.6, 17 / 7.3.
#include "moe_gemm.h"

namespace usaf {
namespace {

constexpr int FEW_THREADS = 256, FEW_WAVES = 4;
constexpr int FEW_SLOTS = 32;  // slots of an m-tile: one MFMA column block
constexpr int FEW_XCDS = 8;    // accelerator dies, blocks dispatched round-robin over them
constexpr int FEW_IMG = 4 * 1024 + 128;  // overlay: four fragment images and 128 bytes of discards

// One wave's LDS: activation tiles and overlay images, at the end its partial tile.
template <int NU, bool OVL>
constexpr int few_wave_lds() {
  const int loop = 4096 + (OVL ? FEW_IMG : 0), sum = 4096 * NU;
  return loop > sum ? loop : sum;
}

struct FewTile {
  int e, m_beg, valid, b;  // expert, first slot, slots, block of 32 NU weight rows
};

// One wave's part of a tile: NU units over part `part` of ks of the
// contraction.  sm: the block's LDS.
template <int NU, int EPI, int DT, bool BT, bool OVL>
__device__ __forceinline__ void few_tile_run(const GemmArgs& g, const FewTile& t, uint8_t* sm, int wave, int lane,
                                             int ks, int part) {
  const int l32 = lane & 31, half = lane >> 5, l8 = lane >> 3, c8 = lane & 7;
  const int ng = (int)(g.K / 128);  // groups of two k-steps
  const int g0 = ng * part / ks, g1 = ng * (part + 1) / ks;

  // ---- operand addresses: uniform bases plus 32-bit lane byte offsets ----
  // unit u of the block is 32 weight rows: n = 32 (NU b + u) + r, or (SwiGLU
  // forward) r < 16 gate rows n = 16 (NU b + u) + r and r >= 16 the up rows I + n
  auto unit_row = [&](int u, int r8) -> int64_t {  // weight row of row 8 r8 of unit u
    if constexpr (EPI == EPI_SWIGLU_FWD) return 16 * (NU * t.b + u) + 8 * (r8 & 1) + (r8 >= 2 ? g.inter : 0);
    else return 32 * (NU * t.b + u) + 8 * r8;
  };
  uint32_t c_off[NU], z_off[NU], o_off = 0;
#pragma unroll
  for (int u = 0; u < NU; ++u) {
    const int64_t row = (int64_t)t.e * g.w_rows + unit_row(u, l32 >> 3) + (l32 & 7);
    c_off[u] = (uint32_t)(row * (g.K / 2) + 16 * half);
    if constexpr (BT) {  // {s2, z2} of the lane half's 16 k-pairs; the units share the 128-row group
      z_off[u] = (uint32_t)(((((int64_t)t.e * (g.N / 128) + NU * t.b / 4) * g.K) + 32 * half) * 4);
    } else {
      z_off[u] = (uint32_t)(row * ng * 4);
    }
  }
  const uint32_t o_unit = (uint32_t)(ng * 2 * Q_OVL_WORDS * 4);  // entry words of one unit, bytes
  if constexpr (OVL) {
    // eight units per n-tile of the entry tables
    const int64_t n_nt = EPI == EPI_SWIGLU_FWD ? (g.inter + 127) / 128 : (g.N + 255) / 256;
    o_off = (uint32_t)((int64_t)t.e * n_nt * 8 + NU * t.b) * o_unit + (uint32_t)lane * 4;
  }
  constexpr int AP = FEW_SLOTS / 8;
  uint32_t a_off[AP];  // activations: lane l fetches chunk c8 of rows 8 p + l8
#pragma unroll
  for (int p = 0; p < AP; ++p) {
    const int r = 8 * p + l8;
    const int m = t.m_beg + (r < t.valid ? r : t.valid - 1);
    const uint32_t arow = (uint32_t)(g.a_rows ? g.a_rows[m] : m);
    a_off[p] = arow * (uint32_t)(g.lda * 2) + 16u * (uint32_t)c8;
  }
  const uint8_t* const wsz = reinterpret_cast<const uint8_t*>(g.wsz);
  const uint8_t* const A = reinterpret_cast<const uint8_t*>(g.A);
  const uint8_t* const ent = reinterpret_cast<const uint8_t*>(g.ovl);

  // the wave's LDS: activation tile of one k-step | images.
  // Tiles are rows of 128 bytes whose 16-byte chunk c sits at c ^ ((row >> 1) & 7)
  // (moe_gemm.hip's q_swz: conflict-free fragment reads); one wave's LDS
  // operations complete in order, so a tile is rewritten right behind its reads
  uint8_t* const sa = sm + wave * few_wave_lds<NU, OVL>();
  uint8_t* const img = sa + 4096;
  const int swz_r = (l32 >> 1) & 7;
  // row 8 p + l8 of a tile, chunk c8
  auto tile_at = [&](int p) { return (8 * p + l8) * 128 + 16 * (c8 ^ ((l8 >> 1) | ((p & 1) << 2))); };

  u32x4 cq[NU][2], ar[AP], kz[8];
  uint32_t cz[NU], ce[NU], re[NU];
  // unit u's codes and scale|zero word of group gr (past the wave's range: its last group again)
  auto load_codes = [&](int u, int gr) {
    gr = gr < g1 ? gr : g1 - 1;
#pragma unroll
    for (int s = 0; s < 2; ++s) cq[u][s] = *reinterpret_cast<const u32x4*>(g.wq + gr * 64 + 32 * s + c_off[u]);
    if constexpr (!BT) cz[u] = *reinterpret_cast<const uint32_t*>(wsz + gr * 4 + z_off[u]);
  };
  auto load_acts = [&](int kt) {
    kt = kt < 2 * g1 ? kt : 2 * g1 - 1;
#pragma unroll
    for (int p = 0; p < AP; ++p) ar[p] = *reinterpret_cast<const u32x4*>(A + kt * (BK * 2) + a_off[p]);
  };
  auto store_acts = [&]() {
#pragma unroll
    for (int p = 0; p < AP; ++p) *reinterpret_cast<u32x4*>(sa + tile_at(p)) = ar[p];
  };
  // BT: the {s2, z2} words of the lane half's 16 k-pairs of a k-step
  auto load_kz = [&](int kt) {
    kt = kt < 2 * g1 ? kt : 2 * g1 - 1;
#pragma unroll
    for (int i = 0; i < 8; ++i) kz[i] = *reinterpret_cast<const u32x4*>(wsz + kt * 256 + 16 * i + z_off[0]);
  };
  auto load_entries = [&](int kt) {
    kt = kt < 2 * g1 ? kt : 2 * g1 - 1;
#pragma unroll
    for (int u = 0; u < NU; ++u)
      re[u] = *reinterpret_cast<const uint32_t*>(ent + kt * (Q_OVL_WORDS * 4) + u * o_unit + o_off);
  };

  f32x16 acc[NU];
#pragma unroll
  for (int u = 0; u < NU; ++u) acc[u] = f32x16{};

  // k-step s of group gr: LDS holds its activations, ar (kz, re) the next step's
  auto step = [&](int s, int gr) {
    const int kt = 2 * gr + s;
    u32x4 af[4], kzc[8];
#pragma unroll
    for (int j = 0; j < 4; ++j)
      af[j] = *reinterpret_cast<const u32x4*>(sa + 128 * l32 + 16 * ((4 * half + j) ^ swz_r));
    __builtin_amdgcn_wave_barrier();
    store_acts();
    __builtin_amdgcn_wave_barrier();
    load_acts(kt + 2);
    if constexpr (BT) {
#pragma unroll
      for (int i = 0; i < 8; ++i) kzc[i] = kz[i];
      load_kz(kt + 1);
    }
    if constexpr (OVL) {
#pragma unroll
      for (int u = 0; u < NU; ++u) ce[u] = re[u];
      load_entries(kt + 1);
    }
    // the loads stay here, a step ahead of their use (the scheduler sinks them to it)
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      u32x4 wf[4];
      if constexpr (BT) {
#pragma unroll
        for (int p = 0; p < 16; ++p) {
          const u32x4 w = kzc[p >> 1];
          wf[p >> 2][p & 3] = dq_pair<DT>(cq[u][s][p >> 2], p & 3, __builtin_bit_cast(f16x2, (p & 1) ? w.z : w.x),
                                          __builtin_bit_cast(f16x2, (p & 1) ? w.w : w.y));
        }
      } else {
        const f16x2 s2 = __builtin_bit_cast(f16x2, (cz[u] & 0xFFFFu) * 0x10001u);
        const f16x2 z2 = __builtin_bit_cast(f16x2, (cz[u] >> 16) * 0x10001u);
#pragma unroll
        for (int p = 0; p < 16; ++p) wf[p >> 2][p & 3] = dq_pair<DT>(cq[u][s][p >> 2], p & 3, s2, z2);
      }
      if constexpr (OVL) {
        // trained values over the dequantized ones: the four registers go through
        // their images, each lane storing its entry's 16-bit value on the way (lane
        // l's word is an entry of register l / 16; unused words point past the
        // image and are discarded)
        const uint32_t off = ce[u] & 0xFFFFu;
#pragma unroll
        for (int j = 0; j < 4; ++j) *reinterpret_cast<u32x4*>(img + 1024 * j + 16 * lane) = wf[j];
        __builtin_amdgcn_wave_barrier();
        uint8_t* const dst = img + (off < 1024 ? 1024 * (lane >> 4) + off : 4 * 1024 + 2 * lane);
        *reinterpret_cast<volatile uint16_t*>(dst) = (uint16_t)(ce[u] >> 16);
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int j = 0; j < 4; ++j) wf[j] = *reinterpret_cast<const volatile u32x4*>(img + 1024 * j + 16 * lane);
        __builtin_amdgcn_wave_barrier();
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[u] = mfma32<DT>(wf[j], af[j], acc[u]);
      if (s == 1) load_codes(u, gr + 1);  // its registers are free: the next group's codes
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  if (g0 < g1) {  // wave-uniform
    load_acts(2 * g0);
#pragma unroll
    for (int u = 0; u < NU; ++u) load_codes(u, g0);
    if constexpr (BT) load_kz(2 * g0);
    if constexpr (OVL) load_entries(2 * g0);
    store_acts();
    load_acts(2 * g0 + 1);
    for (int gr = g0; gr < g1; ++gr) {
      step(0, gr);
      step(1, gr);
    }
  }

  // ---- the partial tiles of the ks waves that split the contraction: lane's
  //      accumulator values 4 q .. 4 q + 3 of a unit are rows 8 q + 4 half + [0, 4)
  //      of slot l32.  Each wave parks its own in its LDS, and finishes the
  //      (unit, q & 1) pairs part, part + ks, ... ----
  constexpr int WAVE_LDS = few_wave_lds<NU, OVL>();
  static_assert(WAVE_LDS >= NU * 4096, "a wave's partial tile of one column block fits its LDS");
  uint8_t* const red0 = sm + (wave - part) * WAVE_LDS;  // the first of the ks waves
  if (ks > 1) lds_barrier();
  __builtin_amdgcn_wave_barrier();
  f32x4* const mine = reinterpret_cast<f32x4*>(sm + wave * WAVE_LDS);
#pragma unroll
  for (int u = 0; u < NU; ++u)
#pragma unroll
    for (int q = 0; q < 4; ++q)
      mine[(u * 4 + q) * 64 + lane] =
          f32x4{acc[u][4 * q], acc[u][4 * q + 1], acc[u][4 * q + 2], acc[u][4 * q + 3]};
  __builtin_amdgcn_wave_barrier();
  if (ks > 1) lds_barrier();
  for (int pi = part; pi < 2 * NU; pi += ks) {
    const int eu = pi >> 1;
    auto total = [&](int q) {
      f32x4 s = reinterpret_cast<const f32x4*>(red0)[(eu * 4 + q) * 64 + lane];
      for (int w = 1; w < ks; ++w) {
        const f32x4 p = reinterpret_cast<const f32x4*>(red0 + w * WAVE_LDS)[(eu * 4 + q) * 64 + lane];
        s = f32x4{s.x + p.x, s.y + p.y, s.z + p.z, s.w + p.w};
      }
      return s;
    };
    const bool live = l32 < t.valid;
    const int64_t m = (int64_t)t.m_beg + l32;
    const int unit = NU * t.b + eu;
    if constexpr (EPI == EPI_SWIGLU_FWD) {
      // columns n = 16 unit + 8 q + 4 half + [0, 4), q = pi & 1
      const int q = pi & 1;
      const f32x4 ga = total(q), ua = total(2 + q);
      const int64_t n = 16 * (int64_t)unit + 8 * q + 4 * half;
      uint32_t gb[2], ub[2], ab[2];
#pragma unroll
      for (int h2 = 0; h2 < 2; ++h2) {
        gb[h2] = pack2<DT>(ga[2 * h2], ga[2 * h2 + 1]);
        ub[h2] = pack2<DT>(ua[2 * h2], ua[2 * h2 + 1]);
        const f32x2 gf = unpack2<DT>(gb[h2]), uf = unpack2<DT>(ub[h2]);
        const f32x2 sf = unpack2<DT>(pack2<DT>(silu_fast(gf.x), silu_fast(gf.y)));
        ab[h2] = pack2<DT>(sf.x * uf.x, sf.y * uf.y);
      }
      if (live) {
        *reinterpret_cast<uint2*>(g.out2 + m * g.ldo2 + n) = uint2{gb[0], gb[1]};
        *reinterpret_cast<uint2*>(g.out2 + m * g.ldo2 + g.inter + n) = uint2{ub[0], ub[1]};
        *reinterpret_cast<uint2*>(g.out + m * g.ldo + n) = uint2{ab[0], ab[1]};
      }
      if (g.out_t) {
        // blocked act: feature rows of ld = round_up(se, 16) slots, zero past se
        const int s0 = g.offsets[t.e], se = g.offsets[t.e + 1] - s0, ld = (se + 15) & ~15;
        const int j = t.m_beg - s0 + l32;
        if (j < ld) {
          uint16_t* const dst = g.out_t + g.inter * (int64_t)g.blk_table[t.e] + n * ld + j;
#pragma unroll
          for (int c = 0; c < 4; ++c)
            dst[c * (int64_t)ld] = live ? (uint16_t)(ab[c >> 1] >> (16 * (c & 1))) : (uint16_t)0;
        }
      }
    } else {
#pragma unroll
      for (int qq = 0; qq < 2; ++qq) {
        const int q = 2 * (pi & 1) + qq;
        const f32x4 v = total(q);
        const int64_t n = 32 * (int64_t)unit + 8 * q + 4 * half;
        if (!live) continue;
        if constexpr (EPI == EPI_STORE) {
          *reinterpret_cast<uint2*>(g.out + m * g.ldo + n) = uint2{pack2<DT>(v.x, v.y), pack2<DT>(v.z, v.w)};
        } else {
          // d(act) -> d(gate), d(up) with moe_gemm_q4_kernel's roundings
          const uint2 gv = *reinterpret_cast<const uint2*>(g.aux + m * g.ld_aux + n);
          const uint2 uv = *reinterpret_cast<const uint2*>(g.aux + m * g.ld_aux + g.inter + n);
          const uint32_t gw[2] = {gv.x, gv.y}, uw[2] = {uv.x, uv.y};
          uint32_t dgw[2], duw[2];
#pragma unroll
          for (int h2 = 0; h2 < 2; ++h2) {
            const f32x2 da = unpack2<DT>(pack2<DT>(v[2 * h2], v[2 * h2 + 1]));
            const f32x2 gt = unpack2<DT>(gw[h2]), up = unpack2<DT>(uw[h2]);
            const float s0 = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * gt.x));
            const float s1 = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * gt.y));
            const f32x2 sg = unpack2<DT>(pack2<DT>(gt.x * s0, gt.y * s1));
            const f32x2 dsil = unpack2<DT>(pack2<DT>(da.x * up.x, da.y * up.y));
            dgw[h2] = pack2<DT>((dsil.x * s0) * (1.0f + gt.x * (1.0f - s0)), (dsil.y * s1) * (1.0f + gt.y * (1.0f - s1)));
            duw[h2] = pack2<DT>(da.x * sg.x, da.y * sg.y);
          }
          *reinterpret_cast<uint2*>(g.out + m * g.ldo + n) = uint2{dgw[0], dgw[1]};
          *reinterpret_cast<uint2*>(g.out + m * g.ldo + g.inter + n) = uint2{duw[0], duw[1]};
        }
      }
    }
  }
}

template <int NU, int WPS, int EPI, int DT, bool BT, bool OVL>
__global__ __launch_bounds__(FEW_THREADS, WPS) void moe_few_kernel(const GemmArgs g, int per, int chunks, int ks) {
  __shared__ __attribute__((aligned(16))) uint8_t sm[FEW_WAVES * few_wave_lds<NU, OVL>()];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // XCD-aware order (blocks are dispatched round-robin over the dies): an
  // m-tile's blocks come in `chunks` runs of `per`, each run on one die, so that
  // its activation rows are fetched into one or two L2s instead of all eight
  const int grp = ((int)blockIdx.x / (FEW_XCDS * per)) * FEW_XCDS + (int)blockIdx.x % FEW_XCDS;
  const int mt = grp / chunks, sub = wave / ks, part = wave - sub * ks;
  FewTile t;
  t.b = ((grp - mt * chunks) * per + (int)blockIdx.x / FEW_XCDS % per) * (FEW_WAVES / ks) + sub;
  if (!slot_tile<FEW_SLOTS>(g, lane, mt, t.e, t.m_beg, t.valid)) return;  // block-uniform
  // waves past the weight's rows: all ks of a group together
  if ((int64_t)t.b * (EPI == EPI_SWIGLU_FWD ? 16 : 32) * NU >= g.N) return;
  few_tile_run<NU, EPI, DT, BT, OVL>(g, t, sm, wave, lane, ks, part);
}

// m-tiles at most: full ones, and one partial tile per expert that has slots
int64_t few_m_tiles(const GemmArgs& g, int64_t S) { return (S < g.E ? S : g.E) + S / FEW_SLOTS; }

template <int NU, int WPS, int EPI, int DT, bool BT, bool OVL>
void launch_few_one(const GemmArgs& g, int64_t S, int ks, hipStream_t st) {
  const int64_t rows = (EPI == EPI_SWIGLU_FWD ? 16 : 32) * NU * (FEW_WAVES / ks);
  const int64_t nb = (g.N + rows - 1) / rows;
  const int64_t chunks = nb < 2 ? nb : 2, per = (nb + chunks - 1) / chunks;
  const int64_t blocks = (few_m_tiles(g, S) * chunks + FEW_XCDS - 1) / FEW_XCDS * FEW_XCDS * per;
  moe_few_kernel<NU, WPS, EPI, DT, BT, OVL>
      <<<(unsigned)blocks, FEW_THREADS, 0, st>>>(g, (int)per, (int)chunks, ks);
}

// NU and the split ks of the contraction (cold weights, us).
// * ks: six groups a wave or more, so that its prologue (the m-tile, the first
//   codes: about 3 us) is a small part of it; but four where even that leaves the
//   1,024 SIMDs short of two waves (one token: 10.6 us split four ways, 26 unsplit).
// * NU = 2 keeps three or four blocks a CU (two with a transposed weight) and halves
//   what a last, partly filled round costs against NU = 4.  NU = 4 reads the activations
//   half as often, and a transposed weight's scale words, which its units share.
//   Forward, NU = 4 / 2: gate_up at ks = 2 79 / 67 (24 tokens, Qwen3), 86 / 86 (256), 80 / 72
//   (160, OLMoE, Zipf(1.1)); with the contraction split four ways equal, 182 / 183 (40,
//   Mixtral), and 5 % faster with warm weights.
// * Transposed: NU = 4 needs two full rounds of blocks.  Qwen3 d(x), 1,024 blocks: 84 / 91,
//   Zipf(1.1) 98 / 106; OLMoE d(x), 512 blocks: 58 / 62, but 77 / 72.  With
//   an overlay it takes all 256 registers and spills four (20 bytes a lane).
// * An overlay keeps every wave longer.  Where NU = 2 does not fill two rounds either,
//   ks = 4 evens them out: OLMoE d(act), ks = 2 / 4, 47 / 51, Zipf(1.1) 69 / 61, Qwen3 71 / 72, 84 / 88.
template <int EPI, int DT, bool BT, bool OVL>
void launch_few_dt(const GemmArgs& g, int64_t S, hipStream_t st) {
  const int64_t unit = EPI == EPI_SWIGLU_FWD ? 16 : 32, groups = g.K / 128;
  const int64_t tiles = (S < g.E ? S : g.E) + S / (2 * FEW_SLOTS);  // about as many m-tiles as there will be
  const bool few = tiles * (g.N / (4 * unit)) * 4 < 2048;
  int ks = few || groups >= 24 ? 4 : groups >= 12 ? 2 : 1;
  bool wide = !few && ks == 4;
  if constexpr (BT) {
    // waves' units of an m-tile for each used expert, against two rounds of two blocks a CU
    const int64_t units = (S < g.E ? S : g.E) * (g.N / 32), two = 4 * (int64_t)device_cu_count() * FEW_WAVES;
    wide = units * ks >= two * 4;
    if (OVL && units * ks < two * 2) ks = 4;
  }
  if constexpr (BT || !OVL) {
    if (wide && g.N % (4 * unit) == 0) return launch_few_one<4, 2, EPI, DT, BT, OVL>(g, S, ks, st);
  }
  launch_few_one<2, BT ? 2 : 3, EPI, DT, BT, OVL>(g, S, ks, st);
}

template <int EPI, bool BT>
int launch_few_epi(const GemmArgs& g, int dt, int64_t S, hipStream_t st, const char* what) {
  if (dt == USAF_BF16) {
    if (g.ovl) launch_few_dt<EPI, USAF_BF16, BT, true>(g, S, st);
    else launch_few_dt<EPI, USAF_BF16, BT, false>(g, S, st);
  } else if (dt == USAF_F16) {
    if (g.ovl) launch_few_dt<EPI, USAF_F16, BT, true>(g, S, st);
    else launch_few_dt<EPI, USAF_F16, BT, false>(g, S, st);
  } else {
    return set_error(USAF_ERR_INVALID, "%s: dtype must be fp16 or bf16", what);
  }
  return check_launch(what);
}

}  // namespace

// The lines against moe_gemm_q4_kernel, in slots per expert on average.  Past 32
// slots an expert takes a second m-tile and its codes are dequantized again; with
// a random routing that begins at an average of about 20.  Measured with cold
// weights at the lines (Qwen3 layer, us, that kernel / this one; routings uniform,
// Zipf(1.1), Zipf(2)):
// * forward, 28: gate_up 121 / 108, 153 / 117, 130 / 118, down 68 / 58, 83 / 63, 67 / 67.
// * transposed, 20: d(act) 81 / 54, 86 / 65, 89 / 64, d(x) 114 / 85, 144 / 112, 111 / 95.
// With an overlay (fp16) the same lines where the other kernel, a tile of 256 rows a
// CU, leaves half of its last round or more idle.  Where it fills its rounds:
// * forward 24: at 24 gate_up 139 / 126, 174 / 142, 152 / 137, down 74 / 67, 95 / 75, 74 / 73; at 28
//   141 / 133, 177 / 145, 151 / 154 and 74 / 68, 94 / 76, 75 / 84.
// * transposed, a contraction below 24 groups, 20: d(x) at 20 136 / 111, 171 / 149, 133 / 134 (at
//   16 134 / 110, 143 / 139, 113 / 132); OLMoE d(act) 53 / 52, 65 / 62, 67 / 68.
// * transposed, a longer one, never: Mixtral d(act) at 16 158 / 141, 161 / 198, 163 / 198.
// The host does not see the routing: with every token on the same eight of 128
// experts (448 tokens, 448 slots each) gate_up and down take 74 + 43 us against 60 + 32.
bool few_slots(const GemmArgs& g, int epi, bool transposed, int64_t S) {
  const int64_t rows = epi == EPI_SWIGLU_FWD ? 32 : 64, tile = epi == EPI_SWIGLU_FWD ? 128 : 256;
  int64_t line = transposed ? 20 : 28;
  if (g.ovl) {
    const int64_t cus = device_cu_count(), last = (S < g.E ? S : g.E) * ((g.N + tile - 1) / tile) % cus;
    if (last == 0 || last > cus / 2) line = !transposed ? 24 : g.K >= 24 * 128 ? 0 : 20;
  }
  if (S > line * g.E || g.N % rows != 0) return false;
  return (few_m_tiles(g, S) * 2 + FEW_XCDS) * (g.N / rows + 2) < ((int64_t)1 << 30);  // blocks of a launch
}

int launch_few(const GemmArgs& g, int epi, bool transposed, int dt, int64_t S, hipStream_t st, const char* what) {
  if (epi == EPI_SWIGLU_FWD) return launch_few_epi<EPI_SWIGLU_FWD, false>(g, dt, S, st, what);
  if (epi == EPI_SWIGLU_BWD) return launch_few_epi<EPI_SWIGLU_BWD, true>(g, dt, S, st, what);
  if (transposed) return launch_few_epi<EPI_STORE, true>(g, dt, S, st, what);
  return launch_few_epi<EPI_STORE, false>(g, dt, S, st, what);
}

}  // namespace usaf
