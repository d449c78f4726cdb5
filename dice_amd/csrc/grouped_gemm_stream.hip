// Grouped expert GEMMs for small batches, where a launch is the streaming of its
// weights: an expert has few rows (up to about 190 and then one tile, which reads every
// weight once; in layer calls up to 384, two or three tiles, which run side by side on an
// XCD), and what counts is that weight bytes are in flight on every compute unit from the
// first microsecond to the last.  Bound: HBM (this card reads 5.5 to
// 6.9 TB/s whatever the order of the rows, as long as whole 128-byte lines are asked for
// and 48 KB per compute unit are in flight; a copy makes 4.8 of reads and writes).
//
// One workgroup of eight waves per tile of BM grouped rows x BN weight rows; where
// the LDS allows it two workgroups per compute unit, one starting up or writing its
// outputs while the other streams.  Operands go from memory to LDS without passing
// registers (buffer_load_dwordx4 ... lds), 16-byte chunks XOR-swizzled by the row through
// the choice of the chunk a lane fetches.  Activations and weights have rings of
// their own: half of the waves issue the activations' copies (they hit the L2), the
// other half the weights' (they come from HBM, further ahead) - vector loads complete
// in order within a wave, so one wave with both would have to wait for its youngest
// weights whenever it needs its oldest activations.  Waves that share a SIMD hold
// different rows, so that a tile's missing rows are missing on every SIMD alike.
//
// The sums of a tile are formed in the order of the persistent kernels
// (grouped_gemm_persist.hip: ascending k in products of 16, one fp32 accumulator),
// so a whole tile gives the same bits whichever kernel multiplies it.
//
// Measured, layer call, against the persistent kernels: DiT-XL width, fp16, 512
// tokens 144 -> 112 us, DiT-G width with fp8 weights, 512 tokens 441 -> 258 us.  Weights and
// rows in the launches, against that bound: 3.6 TB/s in fc1 (51 us) and 2.9 in fc2 (35 us),
// fp8 weights 3.75 (153 us) and 3.25 (94 us).  What is left: a workgroup's start (row
// ranges, row table, first copies: 4 to 5 us), the last round of workgroups (fc2 at 512
// tokens of DiT-XL width has at most 171 for 256 compute units), and the products, which
// the lockstep of a workgroup's waves hides only in part: the waves wait for 42 to 49 % of
// their cycles with the matrix pipe busy for 20 to 32 %.
//
// Compiled for bf16 and, through grouped_gemm_stream_f16.hip, for fp16.
#include <type_traits>

#include "stream_tiles.h"

#ifndef DICE_STREAM_F16
#define DICE_STREAM_F16 0
#endif

namespace dice {
namespace {

#if DICE_STREAM_F16
typedef f16_t h16_t;
typedef f16x8_t h16x8_t;
typedef _Float16 h16x4_t __attribute__((ext_vector_type(4)));
#define DICE_STREAM_MFMA __builtin_amdgcn_mfma_f32_32x32x16_f16
#define DICE_STREAM_WIDEN __builtin_amdgcn_cvt_scalef32_pk_f16_fp8
#define DICE_STREAM_LAUNCH launch_grouped_gemm_stream_f16
#else
typedef bf16_t h16_t;
typedef bf16x8_t h16x8_t;
typedef bf16x4_t h16x4_t;
#define DICE_STREAM_MFMA __builtin_amdgcn_mfma_f32_32x32x16_bf16
#define DICE_STREAM_WIDEN __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8
#define DICE_STREAM_LAUNCH launch_grouped_gemm_stream
#endif

template <int V> using int_c = std::integral_constant<int, V>;
typedef __attribute__((address_space(3))) unsigned char lds_byte_t;

constexpr uint32_t kRsrc = 0x00020000u;      // raw buffer, 32-bit elements
constexpr uint32_t kNowhere = 0x80000000u;   // an offset no descriptor covers

__device__ __forceinline__ uint32_t uniform(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ u32x4_t descriptor(const void *base, uint32_t bytes) {
  const uint64_t p = (uint64_t)base;
  return u32x4_t{uniform((uint32_t)p), uniform((uint32_t)(p >> 32) & 0xffffu), uniform(bytes), kRsrc};
}
// One copy of 16 bytes per lane, memory -> LDS (lane l to dst + 16 l).  As text: a
// copy that the compiler knows of would have it wait for every copy in flight
// before its next LDS read.
__device__ __forceinline__ void copy_to_lds(u32x4_t rs, uint32_t dst, uint32_t voff, uint32_t soff) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(dst), "v"(voff), "s"(rs),
               "s"(soff)
               : "memory", "m0");
}
// At most N of this wave's copies are still in flight, and its LDS reads are done.
template <int N> __device__ __forceinline__ void wait_copies() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
}

// TM x TN blocks of 32 x 32 per wave, WM x WN waves; KB: bytes of a weight row per
// step (64 or 128).  SwiGLU: a 32-row weight block is a strip of 16 gate and the 16
// matching up rows, so that a lane holds both values of its 16-column outputs.
// W8: the weights are e4m3 bytes with one fp32 scale per output channel (KB k per
// step), widened - exactly - when a fragment is read.
template <bool W8_, int KB_, int TM_, int TN_, int WM_, int WN_, int SA_, int SW_>
struct Shape {
  static constexpr bool W8 = W8_;
  static constexpr int KB = KB_, TM = TM_, TN = TN_, WM = WM_, WN = WN_, SA = SA_, SW = SW_;
};
template <int MODE, typename S>
struct StreamGeom {
  static constexpr bool W8 = S::W8;
  static constexpr int KB = S::KB, TM = S::TM, TN = S::TN, WM = S::WM, WN = S::WN, SA = S::SA, SW = S::SW;
  static constexpr int WAVES = WM * WN, BM = WM * TM * 32, BN = WN * TN * 32;
  static constexpr bool SWIGLU = MODE == kFc1Swiglu;
  static constexpr int BN_OUT = SWIGLU ? BN / 2 : BN;
  static constexpr int STEP_K = W8 ? KB : KB / 2, A_SUB = W8 ? 2 : 1;   // (16-bit rows of KB bytes: A_SUB of them per row and step)
  static constexpr int A_SLOT = BM * KB * A_SUB, W_SLOT = BN * KB;
  static constexpr int CHUNKS = KB / 16, COPY_ROWS = 64 / CHUNKS;
  static constexpr int A_COPIES = BM * A_SUB / COPY_ROWS / (WAVES / 2), W_COPIES = BN / COPY_ROWS / (WAVES / 2);   // per issuing wave per step
  static constexpr int PITCH = BN_OUT * 2 + 16;   // bytes of a staged output row
  static constexpr size_t RINGS = (size_t)SA * A_SLOT + (size_t)SW * W_SLOT, STAGED = (size_t)BM * PITCH;
  static constexpr size_t LDS = RINGS > STAGED ? RINGS : STAGED;
  static_assert(TM == 2 || TM == 3, "what stream_body has a case for");
  static_assert(SW > 2 || SA == 2, "the refill order follows the rings' depth");
  static_assert(SA >= 2 && A_COPIES >= 1 && W_COPIES >= 1 && A_COPIES <= 24 && W_COPIES <= 24, "copies per wave");
  static_assert(A_COPIES * (WAVES / 2) * COPY_ROWS == BM * A_SUB && W_COPIES * (WAVES / 2) * COPY_ROWS == BN, "whole copies");
  static __device__ __forceinline__ int swizzle(int row) { return KB == 128 ? (row >> 1) & 7 : ((row >> 1) & 3) ^ ((row >> 3) & 1); }
};

template <int MODE, typename S>
__device__ __forceinline__ void stream_body(const StreamBatch &b, const StreamTile &t, unsigned char *lds) {
  using G = StreamGeom<MODE, S>;
  constexpr bool SWIGLU = G::SWIGLU, W8 = G::W8;
  constexpr int BM = G::BM, BN = G::BN, BN_OUT = G::BN_OUT, WAVES = G::WAVES, KB = G::KB;
  constexpr int TM = G::TM, TN = G::TN, WM = G::WM, WN = G::WN, SA = G::SA, SW = G::SW;
  const PersistProblem &p = b.prob[t.prob];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = uniform(tid >> 6);
  // (waves w, w + 4, .. share a SIMD: with the row blocks slowest they are of different rows, whose last blocks may be empty)
  const int wm = wave / WN, wn = wave % WN;
  // (constant members of p are read here, once: the kernel arguments sit in scalar memory)
  const int k = p.k, lda = p.lda, n = p.n;
  // this piece's run of steps
  const int all_steps = k / G::STEP_K;
  int step0 = 0, steps = all_steps;
  if (t.pieces > 1) {
    step0 = (int)((unsigned)(all_steps * t.piece) / (unsigned)t.pieces);
    steps = (int)((unsigned)(all_steps * (t.piece + 1)) / (unsigned)t.pieces) - step0;
  }
  steps = uniform(steps);

  // ---- copies ----
  const bool loads_a = wave < WAVES / 2;
  const int issuer = loads_a ? wave : wave - WAVES / 2;
  const uint32_t lds0 = uniform((uint32_t)(size_t)(lds_byte_t *)lds);
  constexpr int COPIES = G::A_COPIES > G::W_COPIES ? G::A_COPIES : G::W_COPIES;
  uint32_t voff[COPIES];
  u32x4_t rs;
  const int copy_row = lane / G::CHUNKS, copy_pos = lane % G::CHUNKS;
  if (loads_a) {
    const uint32_t pitch = (uint32_t)lda * 2;
    // copy i of this wave: COPY_ROWS rows of subtile `sub`
    auto copy_index = [&](int i) { return i * (WAVES / 2) + issuer; };
    auto row_of = [&](int i) { return (copy_index(i) % (BM / G::COPY_ROWS)) * G::COPY_ROWS + copy_row; };
    uint32_t src[G::A_COPIES];
    if (p.a_rows) {
      rs = descriptor(p.a, (uint32_t)p.a_src_rows * pitch);
      const int32_t *rows = p.a_rows + t.row0;
      const uint32_t magic = p.a_div == 1 ? 0u : (uint32_t)(0xffffffffu / (uint32_t)p.a_div + 1u);   // slot / a_div = mulhi(slot, magic)
#pragma unroll
      for (int i = 0; i < G::A_COPIES; ++i) src[i] = (uint32_t)rows[row_of(i) < t.rows ? row_of(i) : 0];
#pragma unroll
      for (int i = 0; i < G::A_COPIES; ++i) src[i] = magic ? __umulhi(src[i], magic) : src[i];
    } else {
      rs = descriptor((const unsigned char *)p.a + (size_t)t.row0 * pitch, (uint32_t)t.rows * pitch);
#pragma unroll
      for (int i = 0; i < G::A_COPIES; ++i) src[i] = (uint32_t)row_of(i);
    }
#pragma unroll
    for (int i = 0; i < G::A_COPIES; ++i) {
      const int r = row_of(i), sub = copy_index(i) / (BM / G::COPY_ROWS);
      const uint32_t off = src[i] * pitch + sub * KB + ((copy_pos ^ G::swizzle(r)) << 4);
      voff[i] = r < t.rows ? off : kNowhere;
    }
  } else {
    const uint32_t pitch = (uint32_t)k * (W8 ? 1 : 2);
    const int up = SWIGLU ? p.up_offset : 0;
    rs = descriptor((const unsigned char *)p.w + (size_t)t.expert * p.w_rows * pitch, (uint32_t)p.w_rows * pitch);
#pragma unroll
    for (int i = 0; i < G::W_COPIES; ++i) {
      const int r = (i * (WAVES / 2) + issuer) * G::COPY_ROWS + copy_row;
      const int col = t.n0 + (SWIGLU ? (r >> 5) * 16 + (r & 15) : r);
      const uint32_t off = (uint32_t)(col + ((r & 16) != 0 ? up : 0)) * pitch + ((copy_pos ^ G::swizzle(r)) << 4);
      voff[i] = col < n ? off : kNowhere;
    }
  }
  // Issues this wave's copies of step s (of this piece) into ring slot `slot`.
  auto issue = [&](int s, int slot) {
    const u32x4_t d = {uniform(rs[0]), uniform(rs[1]), uniform(rs[2]), kRsrc};   // (keeps it in scalar registers)
    const uint32_t koff = uniform((uint32_t)(step0 + s) * (uint32_t)(loads_a ? KB * G::A_SUB : KB));
    if (loads_a) {
      const uint32_t dst = lds0 + slot * G::A_SLOT + issuer * 1024;
#pragma unroll
      for (int i = 0; i < G::A_COPIES; ++i) copy_to_lds(d, uniform(dst + i * (WAVES / 2) * 1024), voff[i], koff);
    } else {
      const uint32_t dst = lds0 + SA * G::A_SLOT + slot * G::W_SLOT + issuer * 1024;
#pragma unroll
      for (int i = 0; i < G::W_COPIES; ++i) copy_to_lds(d, uniform(dst + i * (WAVES / 2) * 1024), voff[i], koff);
    }
  };
  for (int s = 0; s < (loads_a ? SA : SW) && s < steps; ++s) issue(s, s);

  // ---- fragments ----
  const int frag_row = lane & 31, half = lane >> 5;
  // row block i of this wave: tile rows 32 (i WM + wm) ..; weight block j
  const int swz = G::swizzle(frag_row);   // (row blocks are multiples of 32 rows: the same for all)
  const unsigned char *const a_base = lds + (wm * 32 + frag_row) * KB;
  const unsigned char *const w_base = lds + SA * G::A_SLOT + (wn * TN * 32 + frag_row) * KB;

  const int blocks = (t.rows + 31) >> 5;
  const int live = uniform((blocks - wm + WM - 1) / WM);   // row blocks of this wave that hold rows

  auto run = [&](auto live_c) {
    constexpr int LIVE = decltype(live_c)::value;
    f32x16_t acc[LIVE > 0 ? LIVE : 1][TN];
#pragma unroll
    for (int i = 0; i < LIVE; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

    // This wave's copies of the step with `left` younger ones have landed; those of the steps issued behind it may
    // still be in flight.
    constexpr int YA = SW == 2 ? SA - 1 : SA - 2, YW = SW == 2 ? SW - 1 : SW - 2;
    auto landed = [&](int left) {
      if (loads_a) {
        if (YA > 0 && left >= YA) wait_copies<YA * G::A_COPIES>();
        else if (YA > 1 && left >= 1) wait_copies<(YA > 1 ? G::A_COPIES : 0)>();   // (stricter than needed by at most YA - 2 steps)
        else wait_copies<0>();
      } else {
        if (YW > 0 && left >= YW) wait_copies<YW * G::W_COPIES>();
        else if (YW > 1 && left >= 1) wait_copies<(YW > 1 ? G::W_COPIES : 0)>();
        else wait_copies<0>();
      }
    };
    constexpr int KK = G::STEP_K / 16, LV = LIVE > 0 ? LIVE : 1;
    h16x8_t wf[2][TN], af[2][LV];
    auto read_frags = [&](const unsigned char *as, const unsigned char *ws, int kk, int buf) {
      const int ca = ((kk * 2 + half) % G::CHUNKS) ^ swz;   // chunk of a 16-bit row
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        if constexpr (W8) {
          const u32x2_t q = *reinterpret_cast<const u32x2_any_t *>(ws + j * 32 * KB + ((kk ^ swz) << 4) + half * 8);
          u32x4_t w;
          w[0] = __builtin_bit_cast(uint32_t, DICE_STREAM_WIDEN(q[0], 1.0f, false));
          w[1] = __builtin_bit_cast(uint32_t, DICE_STREAM_WIDEN(q[0], 1.0f, true));
          w[2] = __builtin_bit_cast(uint32_t, DICE_STREAM_WIDEN(q[1], 1.0f, false));
          w[3] = __builtin_bit_cast(uint32_t, DICE_STREAM_WIDEN(q[1], 1.0f, true));
          wf[buf][j] = __builtin_bit_cast(h16x8_t, w);
        } else {
          wf[buf][j] = __builtin_bit_cast(h16x8_t, *reinterpret_cast<const u32x4_any_t *>(ws + j * 32 * KB + (ca << 4)));
        }
      }
#pragma unroll
      for (int i = 0; i < LIVE; ++i)
        af[buf][i] = __builtin_bit_cast(h16x8_t, *reinterpret_cast<const u32x4_any_t *>(
                                                     as + (kk * 2 / G::CHUNKS) * (BM * KB) + i * (WM * 32 * KB) + (ca << 4)));
    };
    auto multiply = [&](int buf) {
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int i = 0; i < LIVE; ++i) acc[i][j] = DICE_STREAM_MFMA(wf[buf][j], af[buf][i], acc[i][j], 0, 0, 0);
    };

    int a_slot = 0, w_slot = 0;
    landed(steps - 1);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if constexpr (LIVE > 0) read_frags(a_base, w_base, 0, 0);
    for (int s = 0; s < steps; ++s) {
      if constexpr (LIVE > 0) {
        const unsigned char *as = a_base + a_slot * G::A_SLOT, *ws = w_base + w_slot * G::W_SLOT;
#pragma unroll
        for (int kk = 0; kk < KK - 1; ++kk) {
          read_frags(as, ws, kk + 1, (kk + 1) & 1);
          multiply(kk & 1);
        }
      }
      // Behind the barrier every wave has read step s for the last time (its slots may be refilled) and the copies of
      // step s + 1 have landed.  The last products of step s follow the barrier and the first reads of step s + 1, so
      // that the matrix pipe has work while these arrive.
      if (s + 1 < steps) {
        __builtin_amdgcn_sched_barrier(0);
        const int s_new = s + (loads_a ? SA : SW);
        if constexpr (SW == 2) {
          // (two slots: refill before the wait, or nothing would be in flight when step s + 1 has landed)
          asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
          __builtin_amdgcn_s_barrier();
          if (s_new < steps) issue(s_new, loads_a ? a_slot : w_slot);
          landed(steps - 2 - s);
        } else {
          landed(steps - 2 - s);
        }
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        const int a_next = a_slot == SA - 1 ? 0 : a_slot + 1, w_next = w_slot == SW - 1 ? 0 : w_slot + 1;
        if constexpr (LIVE > 0) read_frags(a_base + a_next * G::A_SLOT, w_base + w_next * G::W_SLOT, 0, KK & 1);
        if constexpr (SW > 2) {
          if (s_new < steps) issue(s_new, loads_a ? a_slot : w_slot);
        }
        a_slot = a_next;
        w_slot = w_next;
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (LIVE > 0) multiply((KK - 1) & 1);
    }

    // ---- epilogue: lane holds row frag_row, columns 8 q + 4 half + {0..3} of each block ----
    // 16-bit outputs are put together in LDS (the rings are done with) and leave as whole row segments: written from
    // here, a store would touch 32 rows with 16 bytes each.
    constexpr int BW = SWIGLU ? 16 : 32;   // output columns of a weight block
    const bool partial = MODE == kFc2 && t.pieces > 1;
    constexpr int PITCH = G::PITCH;
    if (!partial) block_lds_barrier();     // (every wave has read its last fragments)
    if constexpr (LIVE > 0) {
      const float *bias = p.bias ? p.bias + (size_t)t.expert * n : nullptr;
      const float *scale = W8 ? p.w_scale + (size_t)t.expert * p.w_rows : nullptr;
      const int tcol0 = wn * TN * BW + half * 4;
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int q = 0; q < BW / 8; ++q) {
          const int tcol = tcol0 + j * BW + q * 8, col = t.n0 + tcol;
          const int ccol = col < n ? col : 0;
          f32x4_t sg, su, sb;
          if (W8) {
            sg = *reinterpret_cast<const f32x4_t *>(scale + ccol);
            if (SWIGLU) su = *reinterpret_cast<const f32x4_t *>(scale + p.up_offset + ccol);
          }
          if (!SWIGLU) sb = bias && t.piece == 0 ? *reinterpret_cast<const f32x4_t *>(bias + ccol) : f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int i = 0; i < LIVE; ++i) {
            const int m = (i * WM + wm) * 32 + frag_row;
            f32x4_t v;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              float x = acc[i][j][q * 4 + r];
              if (W8) x *= sg[r];
              if (SWIGLU) {
                float u = acc[i][j][8 + q * 4 + r];
                if (W8) u *= su[r];
                x = silu_fast(x) * u;
              } else {
                x += sb[r];
                if (MODE == kFc1Gelu) x = gelu_tanh_fast(x);
              }
              v[r] = x;
            }
            if (partial) {
              if (m < t.rows && col < n)
                *reinterpret_cast<f32x4_t *>((float *)p.c + ((size_t)t.piece * p.max_rows + t.row0 + m) * p.ldc + col) = v;
            } else {
              h16x4_t o;
#pragma unroll
              for (int r = 0; r < 4; ++r) o[r] = (h16_t)v[r];
              *reinterpret_cast<u32x2_any_t *>(lds + m * PITCH + tcol * 2) = __builtin_bit_cast(u32x2_t, o);
            }
          }
        }
    }
    if (!partial) {
      block_lds_barrier();
      constexpr int PER_ROW = BN_OUT / 8;
      const int cols = n - t.n0;
      h16_t *const out = (h16_t *)p.c + (size_t)t.row0 * p.ldc + t.n0;
      for (int i = tid; i < t.rows * PER_ROW; i += WAVES * kWave) {
        const int r = i / PER_ROW, c = (i - r * PER_ROW) * 8;
        if (c < cols)
          *reinterpret_cast<u32x4_any_t *>(out + (size_t)r * p.ldc + c) =
              *reinterpret_cast<const u32x4_any_t *>(lds + r * PITCH + c * 2);
      }
    }
  };
  if constexpr (TM == 3) {
    if (live == 3) return run(int_c<3>{});
  }
  if (live == 2) return run(int_c<2>{});
  if (live >= 1) return run(int_c<1>{});
  run(int_c<0>{});
}

// S0, S1: the tile shapes of the two problems.
template <int MODE, typename S0, typename S1>
__global__ __launch_bounds__(S0::WM *S0::WN *kWave, 2) void grouped_gemm_stream_kernel(StreamBatch b) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char stream_lds[];
  using G0 = StreamGeom<MODE, S0>;
  using G1 = StreamGeom<MODE, S1>;
  const StreamTile t = locate_stream_tile<G0::BM, G0::BN_OUT, G1::BM, G1::BN_OUT>(b);
  if (!t.active) return;
  if constexpr (std::is_same_v<S0, S1>) {
    stream_body<MODE, S0>(b, t, stream_lds);
  } else {
    if (t.prob == 0) stream_body<MODE, S0>(b, t, stream_lds);
    else stream_body<MODE, S1>(b, t, stream_lds);
  }
}

template <int MODE, typename S0, typename S1 = S0>
int launch_shape(const StreamBatch &b, hipStream_t s) {
  using G0 = StreamGeom<MODE, S0>;
  using G1 = StreamGeom<MODE, S1>;
  constexpr size_t lds = G0::LDS > G1::LDS ? G0::LDS : G1::LDS;
  static_assert(lds <= 160 * 1024 && G0::WAVES == G1::WAVES, "LDS; one workgroup size");
  auto kern = grouped_gemm_stream_kernel<MODE, S0, S1>;
  static thread_local bool configured = false;
  if (!configured) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                       (int)lds);
    if (e != hipSuccess) return fail(DICE_ERR_LAUNCH, "streaming expert GEMM: LDS attribute: %s", hipGetErrorString(e));
    configured = true;
  }
  const int64_t grid = stream_grid(b, G0::BM, G0::BN_OUT, G1::BM, G1::BN_OUT);
  hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(G0::WAVES * kWave), lds, s, b);
  return launch_status("grouped_gemm_stream");
}

}  // namespace

#if !DICE_STREAM_F16
// What the kernels take: whole steps of k, 16-byte rows, offsets that fit a descriptor.
bool stream_supported(const StreamBatch &b, int mode) {
  int groups = 0;
  for (int i = 0; i < b.n_problems; ++i) {
    const PersistProblem &p = b.prob[i];
    const bool w8 = p.w_scale != nullptr;
    groups += p.n_experts;
    if (p.a_scale || p.a_block_scale || p.c_block_scale) return false;       // fp8 activations
    if (w8 && i != 0) return false;                                          // (fp8 weights: the first problem's)
    if (p.k % (w8 && mode == kFc2 ? 128 : 64) != 0 || b.pieces[i] < 1 || b.pieces[i] > p.k / 128) return false;
    if (p.n % 8 != 0 || p.lda % 8 != 0 || p.ldc % 8 != 0 || p.up_offset % 4 != 0) return false;
    if ((size_t)p.w_rows * p.k * (w8 ? 1 : 2) >= (1ull << 31)) return false;
    const size_t a_rows = p.a_rows ? (size_t)p.a_src_rows : 256;
    if (a_rows * p.lda * 2 >= (1ull << 31)) return false;
    if (p.a_rows && (p.a_div < 1 || p.a_div > 16 || (int64_t)p.a_src_rows * p.a_div >= (1ll << 28))) return false;
  }
  return groups >= 1 && groups <= kWave;
}
#endif

// Tile shapes, eight waves each.  fc1: two workgroups per compute unit; 16-bit weights
// 128 or 192 rows x 128 weight rows (64 and 80 KB of LDS), fp8 weights (half the bytes
// per product) 128 x 256 with 64-byte steps (80 KB).  fc2, whose tiles are fewer and
// longer: one workgroup per compute unit with deeper rings while all tiles are one
// turn (layer call, deep / shallow rings, us: DiT-XL width 512 tokens 104 / 106,
// width 1408, 16 experts, 1200 tokens 261 / 269); with more tiles two workgroups per
// compute unit, so that the tiles past the first turn start at once instead of
// behind it (DiT-XL width, 700 tokens 135 / 126, GELU 750 tokens 129 / 120; DiT-G
// width with fp8 weights, 512 tokens 278 / 267).
// The 192-row tile where it saves an expert a second tile, whose workgroup
// would read all of the weights again (fc1 54 us against 61).  Four waves per
// workgroup, larger tiles with one workgroup per compute unit (fc1) and 64-byte
// steps of 16-bit weights measured slower: what limits a step is how much
// independent work a compute unit has behind its barriers.
int DICE_STREAM_LAUNCH(const StreamBatch &b, int mode, hipStream_t s) {
  // (Pair..: two workgroups per compute unit, fc1's and those of an fc2 of more than a turn; Deep..: one)
  using Pair = Shape<false, 128, 2, 1, 2, 4, 2, 2>;
  using PairTall = Shape<false, 128, 3, 1, 2, 4, 2, 2>;
  using PairW8Fc1 = Shape<true, 64, 2, 2, 2, 4, 2, 3>;
  using Deep = Shape<false, 128, 2, 1, 2, 4, 3, 5>;
  using DeepTall = Shape<false, 128, 3, 1, 2, 4, 3, 4>;
  using DeepW8 = Shape<true, 128, 2, 1, 2, 4, 3, 4>;
  using PairW8Fc2 = Shape<true, 64, 2, 1, 2, 4, 3, 4>;
  const bool w8 = b.prob[0].w_scale != nullptr;
  switch (mode) {
    case kFc1Swiglu:
      return w8 ? launch_shape<kFc1Swiglu, PairW8Fc1, PairTall>(b, s)
                : b.tall ? launch_shape<kFc1Swiglu, PairTall>(b, s) : launch_shape<kFc1Swiglu, Pair>(b, s);
    case kFc1Gelu:
      return w8 ? launch_shape<kFc1Gelu, PairW8Fc1, PairTall>(b, s)
                : b.tall ? launch_shape<kFc1Gelu, PairTall>(b, s) : launch_shape<kFc1Gelu, Pair>(b, s);
    default:
      if (expected_stream_tiles(b, b.tall && !w8 ? 192 : 128, w8 || b.tall ? 192 : 128, 128) > persist_cu_count())
        return w8 ? launch_shape<kFc2, PairW8Fc2, PairTall>(b, s)
                  : b.tall ? launch_shape<kFc2, PairTall>(b, s) : launch_shape<kFc2, Pair>(b, s);
      return w8 ? launch_shape<kFc2, DeepW8, DeepTall>(b, s)
                : b.tall ? launch_shape<kFc2, DeepTall>(b, s) : launch_shape<kFc2, Deep>(b, s);
  }
}

}  // namespace dice
