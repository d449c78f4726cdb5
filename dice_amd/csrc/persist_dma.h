// The 64-k pipeline of grouped_gemm_persist.hip for 16-bit operands with its operands copied from memory straight to
// LDS and its products formed 16 x 16 x 32 at a time.  The k-loop is text (persist_dma_asm.inc, written by
// gen_persist_dma_asm.py: why, the order of the pieces and the wait counts are described there); the compiler's share
// is scalar bookkeeping between the statements, the tile switch and the epilogue.  A group's last tile multiplies only
// its live 64-row blocks, and a tile's first products start the sums (as gemm_persist64_asm_body, whose tile order,
// tile table and row table these are).
#pragma once
#include "persist_core.h"

namespace dice {
namespace {

struct PDmaAddr {
  uint32_t ra[2][2];   // LDS address of this lane's activation fragment of 32-k block kb in slot 0 / 1
  uint32_t rb[2][2];   // ... of its weight fragment
  uint32_t va[8];      // byte offsets of this lane's eight activation rows in the tile being copied
  uint32_t vb[8];      // ... of its weight rows
};
#define PDMA_PARAMS \
  f32x32_t (&f)[4], const PDmaAddr &ad, u32x4_t dA, u32x4_t dB0, u32x4_t dB1, uint32_t koff, uint32_t lw
#define PDMA_ARGS f, ad, dA, dB0, dB1, koff, lw
#define PDMA_CONSTRAINTS                                                                                     \
  : "+{v[0:31]}"(f[0]), "+{v[32:63]}"(f[1]), "+{v[64:95]}"(f[2]), "+{v[96:127]}"(f[3])                       \
  : [ra00] "v"(ad.ra[0][0]), [ra01] "v"(ad.ra[0][1]), [ra10] "v"(ad.ra[1][0]), [ra11] "v"(ad.ra[1][1]),      \
    [rb00] "v"(ad.rb[0][0]), [rb01] "v"(ad.rb[0][1]), [rb10] "v"(ad.rb[1][0]), [rb11] "v"(ad.rb[1][1]),      \
    [va0] "v"(ad.va[0]), [va1] "v"(ad.va[1]), [va2] "v"(ad.va[2]), [va3] "v"(ad.va[3]), [va4] "v"(ad.va[4]), \
    [va5] "v"(ad.va[5]), [va6] "v"(ad.va[6]), [va7] "v"(ad.va[7]), [vb0] "v"(ad.vb[0]), [vb1] "v"(ad.vb[1]), \
    [vb2] "v"(ad.vb[2]), [vb3] "v"(ad.vb[3]), [vb4] "v"(ad.vb[4]), [vb5] "v"(ad.vb[5]), [vb6] "v"(ad.vb[6]), \
    [vb7] "v"(ad.vb[7]), [dA] "s"(dA), [dB0] "s"(dB0), [dB1] "s"(dB1), [koff] "s"(koff), [lw] "s"(lw)        \
  : "memory", "m0", "scc"
// fp8: the two 16-byte parts of a lane's fragment have addresses of their own (ra[slot][2 kb + t]).
struct PDma8Addr {
  uint32_t ra[2][4], rb[2][4], va[8], vb[8];
};
#define PDMA8_PARAMS \
  f32x32_t (&f)[4], const PDma8Addr &ad8, u32x4_t dA, u32x4_t dB0, u32x4_t dB1, uint32_t koff, uint32_t lw
#define PDMA8_ARGS f, ad8, dA, dB0, dB1, koff, lw
#define PDMA8_CONSTRAINTS                                                                                        \
  : "+{v[0:31]}"(f[0]), "+{v[32:63]}"(f[1]), "+{v[64:95]}"(f[2]), "+{v[96:127]}"(f[3])                           \
  : [ra00] "v"(ad8.ra[0][0]), [ra01] "v"(ad8.ra[0][1]), [ra02] "v"(ad8.ra[0][2]), [ra03] "v"(ad8.ra[0][3]),      \
    [ra10] "v"(ad8.ra[1][0]), [ra11] "v"(ad8.ra[1][1]), [ra12] "v"(ad8.ra[1][2]), [ra13] "v"(ad8.ra[1][3]),      \
    [rb00] "v"(ad8.rb[0][0]), [rb01] "v"(ad8.rb[0][1]), [rb02] "v"(ad8.rb[0][2]), [rb03] "v"(ad8.rb[0][3]),      \
    [rb10] "v"(ad8.rb[1][0]), [rb11] "v"(ad8.rb[1][1]), [rb12] "v"(ad8.rb[1][2]), [rb13] "v"(ad8.rb[1][3]),      \
    [va0] "v"(ad8.va[0]), [va1] "v"(ad8.va[1]), [va2] "v"(ad8.va[2]), [va3] "v"(ad8.va[3]), [va4] "v"(ad8.va[4]),\
    [va5] "v"(ad8.va[5]), [va6] "v"(ad8.va[6]), [va7] "v"(ad8.va[7]), [vb0] "v"(ad8.vb[0]), [vb1] "v"(ad8.vb[1]),\
    [vb2] "v"(ad8.vb[2]), [vb3] "v"(ad8.vb[3]), [vb4] "v"(ad8.vb[4]), [vb5] "v"(ad8.vb[5]), [vb6] "v"(ad8.vb[6]),\
    [vb7] "v"(ad8.vb[7]), [dA] "s"(dA), [dB0] "s"(dB0), [dB1] "s"(dB1), [koff] "s"(koff), [lw] "s"(lw)           \
  : "memory", "m0", "scc"
#include "persist_dma_asm.inc"

// Epilogue of tile `cp` for one wave: scales, bias and activation, transposition through the wave's LDS staging rows,
// stores of whole row segments.  What tile_epilogue (persist_core.h) does, for kernels that have vector registers to
// spare between tiles: a column's scale and bias are read once per tile, not once per 32-row block, and a band's rows
// are read back from LDS while the next block's values are worked out; no wait stands between the writes and the reads of
// the staging rows, which one wave's LDS operations reach in the order they were issued in.  The matrix pipe
// idles meanwhile, a seventh to a fifth of an fc1 tile's time: cycles per tile, wait for the copies included, before /
// after: SwiGLU fc1 of bf16 rows 8500 / 7470, fc2 on 192 weight rows 5100 / 4200, fp8 SwiGLU fc1 11800 / 9150, fp8 fc2
// 11000 / 8650.  Of the first, some 6200 are vector instructions (8 per value and two transcendental ones).
// ACC16: the sums come from 16 x 16 products: a lane holds, of a block, rows lane % 16 and 16 on, columns
// 4 (lane / 16) .. + 4 and 16 on (value 8 v + 4 u + r: row half v, column half u); else row lane % 32, columns
// 4 (lane / 32) .. + 4 and 8, 16, 24 on.  Row block i of the wave is tile rows wave_row0 + 64 i ..; only the first
// `live` (at least one) hold rows of the group.  Waits for every copy in flight in front of the first store: stores
// retire in another order, and a count would not tell the two apart.
template <int MODE, int TM, int TN, int RESERVE>
struct DmaEpiGeom {
  static constexpr bool SWIGLU = MODE == kFc1Swiglu;
  static constexpr int OUT_BLOCKS = SWIGLU ? TN / 2 : TN, OUT_COLS = OUT_BLOCKS * 32, PITCH = OUT_COLS * 2 + 16;
  // rows staged at a time (RESERVE: bytes of the staging area that other tables take)
  static constexpr int BAND = kQWaves * 32 * PITCH + RESERVE <= kPStageArea ? 32 : 16;
  static constexpr int CHUNKS = OUT_COLS / 8, PASSES = BAND * CHUNKS / kWave;   // 16-byte chunks of a row, stores of a band
  static constexpr int WAVE_BYTES = BAND * PITCH;
  static_assert(PASSES * kWave == BAND * CHUNKS && kQWaves * WAVE_BYTES + RESERVE <= kPStageArea, "whole passes, staging area");
};
template <int MODE, int TM, int TN, int RESERVE, bool HAS_SCALE, bool HAS_ROW, bool HAS_BIAS, int ACC_BLOCK0, bool ACC16>
__device__ __forceinline__ void dma_epilogue(const Tile &cp, unsigned char *stage, int wave_row0, int wave_col0, int lane,
                                             int live, const float *scale_lds, const float *rowscale_lds,
                                             const float *bias_lds) {
  using G = DmaEpiGeom<MODE, TM, TN, RESERVE>;
  constexpr bool SWIGLU = G::SWIGLU;
  constexpr int OUT_BLOCKS = G::OUT_BLOCKS, PITCH = G::PITCH, BAND = G::BAND, PASSES = G::PASSES, BANDS = 32 / BAND;
  static_assert(!HAS_ROW || (HAS_SCALE && !ACC16), "row scales: fp8 rows");
  const int frag_row = ACC16 ? lane & 15 : lane & 31, lane_col = (ACC16 ? lane >> 4 : lane >> 5) * 4;
  // values 4 q .. 4 q + 3 of a block are q_row(q) rows and q_col(q) columns on; NQ different column groups
  auto q_row = [](int q) { return ACC16 ? (q >> 1) * 16 : 0; };
  auto q_col = [](int q) { return ACC16 ? (q & 1) * 16 : q * 8; };
  constexpr int NQ = ACC16 ? 2 : 4;
  const __amdgpu_buffer_rsrc_t crs =
      __builtin_amdgcn_make_buffer_rsrc((void *)uni(cp.c), 0, uni(cp.c_bytes), kRsrcFlags);
  f32x4_t sg[OUT_BLOCKS][NQ], su[OUT_BLOCKS][NQ], sb[OUT_BLOCKS][NQ];
#pragma unroll
  for (int j = 0; j < OUT_BLOCKS; ++j)
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const int c = wave_col0 + j * 32 + lane_col + q_col(q);
      if (HAS_SCALE) sg[j][q] = *reinterpret_cast<const f32x4_t *>(scale_lds + c);
      if (HAS_SCALE && SWIGLU) su[j][q] = *reinterpret_cast<const f32x4_t *>(scale_lds + 128 + c);
      if (HAS_BIAS) sb[j][q] = *reinterpret_cast<const f32x4_t *>(bias_lds + c);
    }
  // where this lane reads the staging rows and stores, pass by pass (chunk 64 ps + lane of the band)
  uint32_t lds_off[PASSES], out_off[PASSES];
#pragma unroll
  for (int ps = 0; ps < PASSES; ++ps) {
    const int at = ps * kWave + lane, r = at / G::CHUNKS, c = at - r * G::CHUNKS, n = cp.n0 + wave_col0 + c * 8;
    lds_off[ps] = (uint32_t)(r * PITCH + c * 16);
    // (columns past the problem's n: an offset that no descriptor covers, whatever row is added)
    out_off[ps] = n < cp.n ? (uint32_t)(wave_row0 + r) * cp.c_pitch + (uint32_t)n * 2 : kOutOfRange;
  }
  u32x4_t rows[PASSES];   // the band read last, not stored yet
  auto store_band = [&](int row_off) {
#pragma unroll
    for (int ps = 0; ps < PASSES; ++ps)
      __builtin_amdgcn_raw_buffer_store_b128(rows[ps], crs, out_off[ps] + (uint32_t)row_off * cp.c_pitch, 0, 0);
  };
  static_for<TM>([&](auto i_c) {
    constexpr int i = decltype(i_c)::value;
    if (i >= live) return;
    float row_scale = 1.0f;
    if (HAS_ROW) row_scale = rowscale_lds[wave_row0 + i * 64 + frag_row];
    h16x4_t packed[OUT_BLOCKS][4];
    static_for<OUT_BLOCKS>([&](auto j_c) {
      constexpr int j = decltype(j_c)::value;
      f32x16_t blk = fixed_acc_block<ACC_BLOCK0 + i * TN + j>(), up;
      if constexpr (SWIGLU) up = fixed_acc_block<ACC_BLOCK0 + i * TN + j + OUT_BLOCKS>();
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        f32x4_t g, u;
        if (HAS_SCALE) {
          g = sg[j][q % NQ];
          if (SWIGLU) u = su[j][q % NQ];
          if (HAS_ROW) {
            g *= row_scale;
            if (SWIGLU) u *= row_scale;
          }
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float v = blk[q * 4 + r];
          if (HAS_SCALE) v *= g[r];
          if (SWIGLU) {
            float w = up[q * 4 + r];
            if (HAS_SCALE) w *= u[r];
            v = silu_fast(v) * w;
          } else {
            if (HAS_BIAS) v += sb[j][q % NQ][r];
            if (MODE == kFc1Gelu) v = gelu_tanh_fast(v);
          }
          packed[j][q][r] = (h16_t)v;
        }
      }
    });
    static_for<BANDS>([&](auto b_c) {
      constexpr int b = decltype(b_c)::value;
      if constexpr (i == 0 && b == 0) pwait_vmcnt<0>();
      else store_band(b > 0 ? i * 64 + (b - 1) * 16 : (i - 1) * 64 + (BANDS - 1) * 16);
#pragma unroll
      for (int j = 0; j < OUT_BLOCKS; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          unsigned char *const dst = stage + (lane_col + j * 32 + q_col(q)) * 2;
          if (BAND == 32) {
            *reinterpret_cast<u32x2_any_t *>(dst + (frag_row + q_row(q)) * PITCH) = __builtin_bit_cast(u32x2_t, packed[j][q]);
          } else if (ACC16) {
            if (q_row(q) == b * 16)
              *reinterpret_cast<u32x2_any_t *>(dst + frag_row * PITCH) = __builtin_bit_cast(u32x2_t, packed[j][q]);
          } else if ((frag_row >> 4) == b) {
            *reinterpret_cast<u32x2_any_t *>(dst + (frag_row & 15) * PITCH) = __builtin_bit_cast(u32x2_t, packed[j][q]);
          }
        }
      asm volatile("" ::: "memory");
#pragma unroll
      for (int ps = 0; ps < PASSES; ++ps) rows[ps] = *reinterpret_cast<const u32x4_any_t *>(stage + lds_off[ps]);
      asm volatile("" ::: "memory");   // (the next band's writes follow in the LDS queue)
    });
  });
  store_band((live - 1) * 64 + (BANDS - 1) * 16);
}

// The tile shapes the generator writes.  GATHER: activation rows may be addressed through a row table.
template <int MODE, bool HAS_BIAS, int BN, bool GATHER>
constexpr bool persist_dma_applies() {
  if (GATHER && MODE == kFc2) return false;
  if (MODE == kFc1Swiglu) return !HAS_BIAS && (BN == 256 || BN == 128);
  if (MODE == kFc1Gelu) return BN == 256;
  return BN == 192 || BN == 128 || (BN == 256 && !HAS_BIAS);
}

// HAS_BIAS: the tile's bias is staged in LDS a tile ahead and added in the epilogue.
template <int MODE, int BN, bool GATHER, bool HAS_BIAS>
__device__ __forceinline__ void gemm_persist_dma_body(const PersistBatch &batch) {
  static_assert(persist_dma_applies<MODE, HAS_BIAS, BN, GATHER>(), "the shapes the generator writes");
  constexpr bool SWIGLU = MODE == kFc1Swiglu;
  constexpr int KIND = SWIGLU ? (BN == 256 ? 0 : 4) : BN == 256 ? 3 : BN == 192 ? 1 : 2;
  constexpr int BN_OUT = SWIGLU ? BN / 2 : BN;
  constexpr int WTN = BN / 2, TM = 4, TN = WTN / 32;
  constexpr int kCopiesA = kPBM / 8 / kQWaves, kCopiesB = BN / 8 / kQWaves;
  constexpr int kAccBlock0 = 16 - TM * TN;
  constexpr int kTableBytes = kTableTurns * kTileWords * 4, kRowSlotBytes = GATHER ? kPBM * 4 : 0;
  // (three bias buffers: the epilogue of a tile reads its bias while the first wave, a little ahead, may already
  // stage that of the tile after the next)
  constexpr int kBiasBufFloats = 256, kBiasBytes = HAS_BIAS ? 3 * kBiasBufFloats * 4 : 0;
  constexpr int kEpiReserve = kTableBytes + kRowSlotBytes + kBiasBytes;
  using Epi = DmaEpiGeom<MODE, TM, TN, kEpiReserve>;
  typedef __attribute__((address_space(3))) unsigned char lds_byte_t;

  __shared__ __attribute__((aligned(1024))) unsigned char lds_slots[2 * kQSlotBytes];
  __shared__ __attribute__((aligned(1024))) unsigned char lds_stage[kPStageArea];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  fixed_acc_declare();

  static_assert(kQWaves * Epi::WAVE_BYTES + kEpiReserve <= kPStageArea, "no room for the tile table");
  uint32_t *const tile_table = reinterpret_cast<uint32_t *>(lds_stage + kPStageArea - kTableBytes);
  int32_t *const lds_row_slots = reinterpret_cast<int32_t *>(lds_stage + kPStageArea - kTableBytes - kRowSlotBytes);
  float *const lds_bias = reinterpret_cast<float *>(lds_stage + kPStageArea - kEpiReserve);
  if (wave == 0) {
    TileWalker<BN_OUT> walk(batch, lane);
    walk.build_table(batch, lane, kQBK, tile_table, false);
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  phase_barrier();
  auto fetch_tile = [&](int turn) {
    return PackedTile{tile_table[(turn & (kTableTurns - 1)) * kTileWords + (lane < kTileWords ? lane : 0)]};
  };

  // ---- addresses the text takes ----
  const int b_row0 = SWIGLU ? wn * (WTN / 2) : wn * WTN;
  const uint32_t slots = (uint32_t)(size_t)(lds_byte_t *)lds_slots;
  PDmaAddr ad;
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      // (row block i of wave row wm = tile rows 64 i + 32 wm ..: the text adds i x 64 rows)
      ad.ra[s][kb] = slots + s * kQSlotBytes + qring_off(wm * 32 + (lane & 15), kb * 4 + (lane >> 4));
      ad.rb[s][kb] = slots + s * kQSlotBytes + kPBM * 128 + qring_off(b_row0 + (lane & 15), kb * 4 + (lane >> 4));
    }
  // A copy lands 64 x 16 consecutive bytes, eight rows of 128: lane l fills position l % 8 of row l / 8, and fetches
  // the chunk that the swizzle puts there.  Copy l of a wave covers rows 32 l + 8 wave ..
  const uint32_t lw = uni(slots + (uint32_t)wave * 1024u);
  const int cp_row0 = wave * 8 + (lane >> 3);
  const uint32_t cp_byte = (uint32_t)(((lane & 7) ^ qswizzle(cp_row0)) << 4);   // (row bits 1..3: the same for every l)
  auto copy_row_slots = [&](const PackedTile &pk) {
    if constexpr (GATHER) {
      const uint64_t ptr = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane(pk.words, 21) << 32) |
                           (uint32_t)__builtin_amdgcn_readlane(pk.words, 20);
      const int rows = __builtin_amdgcn_readlane(pk.words, 23);
      if (wave == 0 && ptr != 0) {
        // (rows past the group's end read as slot 0, a legal row: their products are never stored)
        const u32x4_t rs = {uni((uint32_t)ptr), uni((uint32_t)(ptr >> 32) & 0xffffu), uni((uint32_t)rows * 4u),
                            kRsrcFlags};
        lds_dma_x4_text(rs, (uint32_t)(size_t)(lds_byte_t *)lds_row_slots, (uint32_t)lane * 16u);
      }
    }
  };
  auto copy_bias = [&](const PackedTile &pk, int buf) {
    if constexpr (HAS_BIAS) {
      const uint64_t ptr = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane(pk.words, 9) << 32) |
                           (uint32_t)__builtin_amdgcn_readlane(pk.words, 8);
      const int n0 = __builtin_amdgcn_readlane(pk.words, 16), n = __builtin_amdgcn_readlane(pk.words, 17);
      if (wave == 0) {
        // (a problem without a bias gets zeros: a descriptor that covers no bytes)
        const uint64_t src = ptr != 0 ? ptr + (uint64_t)n0 * 4 : (uint64_t)batch.prob[0].w;
        const u32x4_t rs = {uni((uint32_t)src), uni((uint32_t)(src >> 32) & 0xffffu),
                            uni(ptr != 0 ? (uint32_t)(n - n0) * 4u : 0u), kRsrcFlags};
        lds_dma_x4_text(rs, (uint32_t)(size_t)(lds_byte_t *)(lds_bias + buf * kBiasBufFloats), (uint32_t)lane * 16u);
      }
    }
  };
  // Descriptors of the tile being copied, as plain register values (base, extent, flags).
  u32x4_t dA, dB0, dB1;
  auto set_copy_offsets = [&](const Tile &t) {
    auto desc = [](const unsigned char *base, uint32_t bytes) {
      const uint64_t p = (uint64_t)base;
      return u32x4_t{uni((uint32_t)p), uni((uint32_t)(p >> 32) & 0xffffu), uni(bytes), kRsrcFlags};
    };
    dA = desc(t.a, t.a_bytes);
    dB0 = desc(t.b0, t.b_bytes);
    dB1 = desc(t.b1, t.b_bytes);
#pragma unroll
    for (int i = 0; i < kCopiesA; ++i) {
      const int r = cp_row0 + 32 * i;
      uint32_t off = (uint32_t)r * t.a_pitch + cp_byte;
      if constexpr (GATHER) {
        if (t.a_rows) {
          const uint32_t slot = (uint32_t)lds_row_slots[r];
          // (one slot per source row: 2^32 / 1 does not fit the multiplier, which then reads 0)
          const uint32_t src_row = t.a_magic ? __umulhi(slot, t.a_magic) : slot;
          off = r < t.rows ? src_row * t.a_pitch + cp_byte : kOutOfRange;
        }
      }
      ad.va[i] = off;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int row = cp_row0 + ((SWIGLU && 32 * i >= BN / 2) ? 32 * i - BN / 2 : 32 * i);   // (the up half has its own descriptor)
      ad.vb[i] = i < kCopiesB ? (uint32_t)row * t.b_pitch + cp_byte : 0;
    }
  };

  // ---- pipeline state ----
  // The copies run two steps ahead of the products, so they cross into the next tile once while a tile is multiplied.
  int next_turn = 0;
  PackedTile nxt = fetch_tile(next_turn++);
  Tile ld = unpack_tile(nxt);   // tile being copied
  if (!ld.valid) return;
  int bias_buf = 0;             // buffer of the bias of the tile being multiplied
  if constexpr (GATHER || HAS_BIAS) {
    copy_row_slots(nxt);
    copy_bias(nxt, 0);
    pwait_vmcnt<0>();
    phase_barrier();
  }
  Tile cp = ld;                 // tile being multiplied
  int ld_kt = 0;
  set_copy_offsets(ld);
  nxt = fetch_tile(next_turn++);
  if constexpr (GATHER) {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    phase_barrier();
    copy_row_slots(nxt);
  }
  copy_bias(nxt, 1);
  uint32_t koff = 0;
  auto advance_copy = [&]() {
    if (++ld_kt == ld.steps) {
      ld = unpack_tile(nxt);
      set_copy_offsets(ld);
      ld_kt = 0;
    }
    koff = uni((uint32_t)ld_kt * 128u);
  };
  {
    f32x32_t f[4];
    asm volatile("" : "={v[0:31]}"(f[0]), "={v[32:63]}"(f[1]), "={v[64:95]}"(f[2]), "={v[96:127]}"(f[3]));
    pdma_load_s0<KIND, 4>(PDMA_ARGS);
    advance_copy();
    pdma_load_s1<KIND, 4>(PDMA_ARGS);
  }
  pwait_vmcnt<0>();
  phase_barrier();

  unsigned char *const stage_rows = lds_stage + wave * Epi::WAVE_BYTES;
  const int wave_col0 = SWIGLU ? wn * (WTN / 2) : wn * WTN;

  // The steps of a tile whose rows fill its first LIVE 64-row blocks.
  auto run_tile = [&](auto live_c) {
    constexpr int LIVE = decltype(live_c)::value;
    f32x32_t f[4];   // the fragments: live inside the tile's k-loop only
    asm volatile("" : "={v[0:31]}"(f[0]), "={v[32:63]}"(f[1]), "={v[64:95]}"(f[2]), "={v[96:127]}"(f[3]));
    pdma_read_first<KIND, LIVE>(PDMA_ARGS);
    pdma_t1_s0_v1<KIND, LIVE>(PDMA_ARGS);
    advance_copy();
    pdma_t2_s0_v1<KIND, LIVE>(PDMA_ARGS);
    pdma_t1_s1_v0<KIND, LIVE>(PDMA_ARGS);
    advance_copy();
    pdma_t2_s1_v0<KIND, LIVE>(PDMA_ARGS);
    for (int s = 2; s < cp.steps; s += 2) {   // (every tile has an even number of steps and starts in slot 0)
      pdma_t1_s0_v0<KIND, LIVE>(PDMA_ARGS);
      advance_copy();
      pdma_t2_s0_v0<KIND, LIVE>(PDMA_ARGS);
      pdma_t1_s1_v0<KIND, LIVE>(PDMA_ARGS);
      advance_copy();
      pdma_t2_s1_v0<KIND, LIVE>(PDMA_ARGS);
    }
    // The last reads (of the next tile, which reads them again: the epilogue needs the registers) have landed.
    asm volatile("s_waitcnt lgkmcnt(0)"
                 : "+{v[0:31]}"(f[0]), "+{v[32:63]}"(f[1]), "+{v[64:95]}"(f[2]), "+{v[96:127]}"(f[3])::"memory");
  };

  while (true) {  // one tile per iteration
    const int live = uni((cp.rows + 63) >> 6);   // 64-row blocks of the tile that hold rows of its group
    if (live >= 4) run_tile(template_int<4>{});
    else if (live == 3) run_tile(template_int<3>{});
    else if (live == 2) run_tile(template_int<2>{});
    else run_tile(template_int<1>{});
    fixed_acc_settle();
    dma_epilogue<MODE, TM, TN, kEpiReserve, false, false, HAS_BIAS, kAccBlock0, true>(
        cp, stage_rows, wm * 32, wave_col0, lane, live, nullptr, nullptr, lds_bias + bias_buf * kBiasBufFloats);
    cp = ld;
    if (!cp.valid) break;
    nxt = fetch_tile(next_turn++);
    copy_row_slots(nxt);
    // (the buffer written here was last read a whole tile ago; the copy is older than every one of the
    // coming steps, whose waits therefore cover it)
    bias_buf = bias_buf == 2 ? 0 : bias_buf + 1;          // the tile multiplied next
    copy_bias(nxt, bias_buf == 2 ? 0 : bias_buf + 1);     // the one after it
  }
}

}  // namespace
}  // namespace dice
