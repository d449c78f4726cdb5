// Tile order of the kernels that take one workgroup per tile and up to two problems
// per launch (grouped_gemm_stream.hip, grouped_gemm_split.hip).
#pragma once
#include <cmath>

#include "gemm_common.h"

namespace dice {
namespace {

// What a workgroup multiplies.
struct StreamTile {
  int prob, expert, row0, rows, n0, piece, pieces;
  bool active;
};

// Tile order: XCD x (= blockIdx % 8) takes an eighth of every problem's tiles; within
// an expert the m-tile runs fastest, then the piece of k, then the n-tile, so the
// workgroups that share an L2 and run side by side share weights, then activations.
template <int BM0, int BN0, int BM1, int BN1>
__device__ __forceinline__ StreamTile locate_stream_tile(const StreamBatch &b) {
  const int lane = threadIdx.x & 63;
  int g_prob = 0, g_expert = 0, begin = 0, cnt = 0, nt = 1, groups = 0, bm = BM0;
  for (int pi = 0; pi < b.n_problems; ++pi) {
    const PersistProblem &p = b.prob[pi];
    const int local = lane - groups;
    if (local >= 0 && local < p.n_experts) {
      g_prob = pi;
      g_expert = local;
      begin = p.offsets[local];
      cnt = p.offsets[local + 1] - begin;
      nt = (pi == 0 ? (p.n + BN0 - 1) / BN0 : (p.n + BN1 - 1) / BN1) * b.pieces[pi];
      bm = pi == 0 ? BM0 : BM1;
    }
    groups += p.n_experts;
  }
  const int mt = (int)((unsigned)(cnt + bm - 1) / (unsigned)bm), tiles = mt * nt;
  int inc = tiles;
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    const int up = __shfl_up(inc, o, kWave);
    if (lane >= o) inc += up;
  }
  const int xcd = blockIdx.x % kNumXcd;
  int j = blockIdx.x / kNumXcd, id = -1, first_group = 0;
  for (int pi = 0; pi < b.n_problems; ++pi) {
    const int last = first_group + b.prob[pi].n_experts - 1;
    const int base = __builtin_amdgcn_readlane(inc - tiles, first_group);
    const int total = __builtin_amdgcn_readlane(inc, last) - base;
    const int lo = (int)((unsigned)(total * xcd) / kNumXcd), hi = (int)((unsigned)(total * (xcd + 1)) / kNumXcd);
    if (id < 0 && j < hi - lo) id = base + lo + j;
    j -= hi - lo;
    first_group = last + 1;
  }
  StreamTile t;
  t.active = id >= 0;
  if (!t.active) return t;
  const int g = __builtin_ctzll(__ballot(id >= inc - tiles && id < inc));
  const int r = id - __builtin_amdgcn_readlane(inc - tiles, g);
  const int g_mt = __builtin_amdgcn_readlane(mt, g), g_cnt = __builtin_amdgcn_readlane(cnt, g);
  const int q = (int)((unsigned)r / (unsigned)g_mt), m = r - q * g_mt;
  t.prob = __builtin_amdgcn_readlane(g_prob, g);
  t.expert = __builtin_amdgcn_readlane(g_expert, g);
  const int g_bm = BM0 == BM1 ? BM0 : t.prob == 0 ? BM0 : BM1, g_bn = BN0 == BN1 ? BN0 : t.prob == 0 ? BN0 : BN1;
  t.row0 = __builtin_amdgcn_readlane(begin, g) + m * g_bm;
  t.rows = __builtin_amdgcn_readfirstlane(g_cnt - m * g_bm < g_bm ? g_cnt - m * g_bm : g_bm);
  t.pieces = b.pieces[t.prob];
  const int nq = t.pieces == 1 ? q : (int)((unsigned)q / (unsigned)t.pieces);
  t.piece = __builtin_amdgcn_readfirstlane(q - nq * t.pieces);
  t.n0 = __builtin_amdgcn_readfirstlane(nq * g_bn);
  return t;
}

// Rows of the fuller experts under a uniform routing (1.5 standard deviations).
inline double rows_of_full_expert(int64_t rows, int experts) {
  const double per = (double)rows / experts;
  return per + (experts > 1 ? 1.5 * std::sqrt(per) : 0.0);
}
// Tiles of a launch where every expert is a fuller one: at most as many as compute
// units are one turn of one workgroup each.
inline int64_t expected_stream_tiles(const StreamBatch &b, int bm0, int bm1, int bn) {
  int64_t tiles = 0;
  for (int i = 0; i < b.n_problems; ++i) {
    const PersistProblem &p = b.prob[i];
    const int64_t m_tiles = p.n_experts * (int64_t)std::ceil(rows_of_full_expert(p.max_rows, p.n_experts) / (i == 0 ? bm0 : bm1));
    tiles += m_tiles * ((p.n + bn - 1) / bn) * b.pieces[i];
  }
  return tiles;
}

// Workgroups of a launch: an upper bound (row counts live on the device; surplus workgroups exit at once).
inline int64_t stream_grid(const StreamBatch &b, int bm0, int bn0, int bm1, int bn1) {
  int64_t per_xcd = 0;
  for (int i = 0; i < b.n_problems; ++i) {
    const PersistProblem &p = b.prob[i];
    const int bm = i == 0 ? bm0 : bm1, bn = i == 0 ? bn0 : bn1;
    const int64_t m_tiles = p.n_experts == 1 ? ((int64_t)p.max_rows + bm - 1) / bm : (int64_t)p.max_rows / bm + p.n_experts;
    per_xcd += (m_tiles * ((p.n + bn - 1) / bn) * b.pieces[i] + kNumXcd - 1) / kNumXcd;
  }
  return per_xcd * kNumXcd;
}

}  // namespace
}  // namespace dice
