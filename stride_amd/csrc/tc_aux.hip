// The non-GEMM entry points of stride's tensor-core path for MI355X (gfx950):
// token embedding into fp32 h tiles, RMSNorm from h to bf16 x tiles, paged
// attention over bf16 KV, and lane compaction. They complete the operator
// surface of the reference's src/kernels_tc.h:79-87, so an engine linking this
// library needs no other device code for a decode step.
//
// Each follows the reference's fixed summation trees exactly (the order of every
// fmaf and add, src/kernels_tc.cu:179-340, src/kernel_common.h:84-309), so the
// results do not depend on the batch, the lane position or the launch shape.
// Work is spread over 64-wide wavefronts wherever the tree leaves freedom
// (independent positions, dimensions and lanes); sequential sums stay sequential.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cstddef>
#include <string>

#include "../../include/stride_exact.h"
#include "tc_common.hpp"

namespace stride_tc {

int fail(int code, const std::string& msg);  // tc_gemm.hip

namespace {

// Attention summation page: 64 positions (src/kernels.h:20-21). A numeric
// constant of the tree, independent of the KV storage page size.
constexpr int kAttnPageShift = 6;
constexpr int kAttnPage = 1 << kAttnPageShift;
constexpr int kHeadsPerGroup = 4;  // the reference's float4 query packing

// Maximum over the 64 lanes of a wave, in registers: DPP within each row of 16
// lanes (neighbours in a quad, then rotations by 4 and 8), then the row swaps
// of gfx950 (v_permlane16_swap, v_permlane32_swap; each lane receives its own
// value or its partner row's in the two results, so both are folded in). Each
// step keeps the larger of two values (a strict > pick); scores are sums from a
// +0 start, never -0, so the maximum is the same value whatever the pairing.
template <int CTRL>
__device__ __forceinline__ float dpp_f32(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, false));
}
__device__ __forceinline__ float pick_gt(float o, float m) { return o > m ? o : m; }
__device__ __forceinline__ float wave_max(float m) {
  m = pick_gt(dpp_f32<0xB1>(m), m);   // quad_perm [1,0,3,2]
  m = pick_gt(dpp_f32<0x4E>(m), m);   // quad_perm [2,3,0,1]
  m = pick_gt(dpp_f32<0x124>(m), m);  // row_ror:4
  m = pick_gt(dpp_f32<0x128>(m), m);  // row_ror:8
  const auto r16 = __builtin_amdgcn_permlane16_swap(__float_as_uint(m), __float_as_uint(m), false, false);
  m = pick_gt(__uint_as_float(r16[0]), m);
  m = pick_gt(__uint_as_float(r16[1]), m);
  const auto r32 = __builtin_amdgcn_permlane32_swap(__float_as_uint(m), __float_as_uint(m), false, false);
  m = pick_gt(__uint_as_float(r32[0]), m);
  m = pick_gt(__uint_as_float(r32[1]), m);
  return m;
}

// ---------------------------------------------------------------------------
// Embedding: lane j of the h tiles <- fp32(embed row tokens[j]). The embedding
// is the LM head's weight tiles, so row `token` is slot token % 16 of row tile
// token / 16 (src/kernels_tc.cu:179-203). Thread i moves 8 columns.
__global__ __launch_bounds__(256) void k_embed(StrideTcEmbedParams p) {
  const int b = blockIdx.x;
  const int token = p.tokens[b];
  const int rt = token >> 4, slot = token & 15, lt = b >> 4, jj = b & 15;
  const int col_tiles = p.dim >> 4;
  for (int i = threadIdx.x; i < col_tiles * 2; i += blockDim.x) {
    const int ct = i >> 1, half = i & 1;
    const uint16_t* src = p.embed + (static_cast<int64_t>(rt) * col_tiles + ct) * kTileElems + slot * 16 + half * 8;
    float* dst = p.h + ((static_cast<int64_t>(lt) * col_tiles + ct) * 16 + jj) * 16 + half * 8;
    const u32x4 w = load16(src);
    f32x4 lo, hi;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      lo[2 * k] = f32_of(w[k] << 16);
      lo[2 * k + 1] = f32_of(w[k] & 0xFFFF0000u);
      hi[2 * k] = f32_of(w[k + 2] << 16);
      hi[2 * k + 1] = f32_of(w[k + 2] & 0xFFFF0000u);
    }
    reinterpret_cast<f32x4*>(dst)[0] = lo;
    reinterpret_cast<f32x4*>(dst)[1] = hi;
  }
}

// ---------------------------------------------------------------------------
// RMSNorm, one wave per lane. Lanes 0..31 of the wave compute the reference's
// 32 partials (partial t: fmaf over columns 0..15 of column tiles ct == t mod
// 32, ascending); lane 0 adds them left to right; then x = bf16(g * (v * r))
// (src/kernels_tc.cu:205-271, 276-340). With TPL > 0 (dim == 32 * 16 * TPL)
// each of lanes 0..31 keeps its TPL tiles and their gains in registers, so h
// is read once; TPL == 0 is the general form.
template <int TPL>
__global__ __launch_bounds__(64) void k_norm(StrideTcNormParams p, int per_lane) {
  const int b = blockIdx.x;  // lane index in [0, lane_groups * 16)
  const int lane = threadIdx.x;
  const int lt = b >> 4, j = b & 15;
  const int col_tiles = p.dim >> 4;
  const int64_t row0 = static_cast<int64_t>(lt) * col_tiles * kTileElems + j * 16;
  auto tile = [&](int ct) { return row0 + static_cast<int64_t>(ct) * kTileElems; };
  auto store = [&](int ct, const f32x4* v, const f32x4* g, float r) {
    uint32_t o[8];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const uint32_t b0 = bf16_rne(g[q][0] * (v[q][0] * r)), b1 = bf16_rne(g[q][1] * (v[q][1] * r));
      const uint32_t b2 = bf16_rne(g[q][2] * (v[q][2] * r)), b3 = bf16_rne(g[q][3] * (v[q][3] * r));
      o[2 * q] = b0 | (b1 << 16);
      o[2 * q + 1] = b2 | (b3 << 16);
    }
    u32x4* out = reinterpret_cast<u32x4*>(p.x + tile(ct));
    out[0] = u32x4{o[0], o[1], o[2], o[3]};
    out[1] = u32x4{o[4], o[5], o[6], o[7]};
  };
  if (b >= p.l.rows) {
    if (per_lane) return;
    for (int ct = lane; ct < col_tiles; ct += 64) {
      u32x4* out = reinterpret_cast<u32x4*>(p.x + tile(ct));
      out[0] = u32x4{0u, 0u, 0u, 0u};
      out[1] = u32x4{0u, 0u, 0u, 0u};
    }
    return;
  }
  // The 32 lane partials added left to right, ((p0 + p1) + p2) + ..., from
  // registers (every lane forms the same sum), then r = 1 / sqrt(sum / dim + eps).
  auto inv_rms = [&](float acc) {
    float sum = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(acc), 0));
#pragma unroll
    for (int i = 1; i < 32; ++i) sum = sum + __int_as_float(__builtin_amdgcn_readlane(__float_as_int(acc), i));
    return 1.0f / sqrtf(sum / static_cast<float>(p.dim) + p.eps);
  };
  if constexpr (TPL > 0) {
    f32x4 v[TPL][4], g[TPL][4];
    float acc = 0.0f;
    if (lane < 32) {
#pragma unroll
      for (int k = 0; k < TPL; ++k) {
        const f32x4* src = reinterpret_cast<const f32x4*>(p.h + tile(lane + 32 * k));
        const f32x4* gs = reinterpret_cast<const f32x4*>(p.weight + (lane + 32 * k) * 16);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          v[k][q] = src[q];
          g[k][q] = gs[q];
        }
      }
#pragma unroll
      for (int k = 0; k < TPL; ++k)
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
          for (int c = 0; c < 4; ++c) acc = __builtin_fmaf(v[k][q][c], v[k][q][c], acc);
    }
    const float r = inv_rms(acc);
    if (lane < 32) {
#pragma unroll
      for (int k = 0; k < TPL; ++k) store(lane + 32 * k, v[k], g[k], r);
    }
  } else {
    float acc = 0.0f;
    if (lane < 32) {
      for (int ct = lane; ct < col_tiles; ct += 32) {
        const f32x4* v = reinterpret_cast<const f32x4*>(p.h + tile(ct));
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const f32x4 w = v[q];
#pragma unroll
          for (int c = 0; c < 4; ++c) acc = __builtin_fmaf(w[c], w[c], acc);
        }
      }
    }
    const float r = inv_rms(acc);
    for (int ct = lane; ct < col_tiles; ct += 64) {
      const f32x4* v = reinterpret_cast<const f32x4*>(p.h + tile(ct));
      const f32x4* gv = reinterpret_cast<const f32x4*>(p.weight + ct * 16);
      const f32x4 vv[4] = {v[0], v[1], v[2], v[3]}, gg[4] = {gv[0], gv[1], gv[2], gv[3]};
      store(ct, vv, gg, r);
    }
  }
}

// ---------------------------------------------------------------------------
// Lane compaction: out lane l <- in lane lm_rows[l] (src/kernels_tc.cu:566-587).
__global__ __launch_bounds__(64) void k_compact(StrideTcCompactParams p) {
  const int b = blockIdx.x;
  const int src = p.lm_rows[b];
  const int64_t in0 = static_cast<int64_t>(src >> 4) * p.col_tiles * kTileElems + (src & 15) * 16;
  const int64_t out0 = static_cast<int64_t>(b >> 4) * p.col_tiles * kTileElems + (b & 15) * 16;
  for (int ct = threadIdx.x; ct < p.col_tiles; ct += 64) {
    const u32x4* in = reinterpret_cast<const u32x4*>(p.in + in0 + static_cast<int64_t>(ct) * kTileElems);
    u32x4* out = reinterpret_cast<u32x4*>(p.out + out0 + static_cast<int64_t>(ct) * kTileElems);
    out[0] = in[0];
    out[1] = in[1];
  }
}

// ---------------------------------------------------------------------------
// Attention.

// One row's sums over a page, by one wave. Scores: lane i holds position i, and an
// fmaf chain over the dims in order is a chain of v_mfma_f32_4x4x1_16b_f32, one per dim
// (one fmaf per output; the query column of four heads is block `dim % 16` of the left
// operand, given to all sixteen blocks, which hold four positions each). Mix: lane d
// holds dim d, one MFMA per position with the four heads' weights as the column. The
// four heads cost 8 cycles of the fp32 units a dim or position, against 16 as v_fma_f32.
// Where the KV loads bound the kernel that does not show (bf16, 128 rows of 4-8 pages, 29-30
// us either way), more where they do not (fp32 KV, 32 rows 16.1 -> 13.2 us; bf16, 530 rows of
// 9 pages, each row's read again from L2, 91 -> 69 us).
//
// qa: lane h + 4b holds q[h][16e + b] in qa[e].
template <int D>
__device__ __forceinline__ void load_query(const float* qrow, int lane, float (&qa)[D / 16]) {
#pragma unroll
  for (int e = 0; e < D / 16; ++e) qa[e] = qrow[(lane & 3) * D + 16 * e + (lane >> 2)];
}
template <int D, class KvT>
__device__ __forceinline__ f32x4 page_scores(const u32x4 (&kr)[D * sizeof(KvT) / 16], const float (&qa)[D / 16]) {
  f32x4 a = {0.0f, 0.0f, 0.0f, 0.0f};
  // Eight dims widened ahead of their MFMAs: one that reads a register written just
  // before it waits.
  unroll<D / 8>([&](auto cc) __attribute__((always_inline)) {
    constexpr int c = decltype(cc)::value;
    float k[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      if constexpr (sizeof(KvT) == 2) k[e] = f32_of(e & 1 ? kr[c][e / 2] & 0xFFFF0000u : kr[c][e / 2] << 16);
      else k[e] = f32_of(kr[2 * c + e / 4][e % 4]);
    }
    if constexpr (sizeof(KvT) == 2)
      asm("" : "+v"(k[0]), "+v"(k[1]), "+v"(k[2]), "+v"(k[3]), "+v"(k[4]), "+v"(k[5]), "+v"(k[6]), "+v"(k[7]));
    unroll<8>([&](auto ee) __attribute__((always_inline)) {
      constexpr int e = decltype(ee)::value, d = 8 * c + e;
      a = __builtin_amdgcn_mfma_f32_4x4x1f32(qa[d / 16], k[e], a, 4, d % 16, 0);
    });
  });
  return a;
}
// wt: [head][position] weights; vs: the page's V rows. acc[t][h]: dim lane + 64t of head
// h; den: head lane & 3, its weights added left to right.
template <int D, class KvT>
__device__ __forceinline__ void page_mix(const float* wt, const KvT (*vs)[D], int n, int lane, f32x4 (&acc)[(D + 63) / 64],
                                         float& den) {
  constexpr int T = (D + 63) / 64;
#pragma unroll
  for (int t = 0; t < T; ++t) acc[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  den = 0.0f;
  const float* wh = wt + (lane & 3) * kAttnPage;
  const int d0 = min(lane, D - 1);
  for (int i0 = 0; i0 < n; i0 += 16) {
    const float wa = wh[i0 + (lane >> 2)];  // lane h + 4b: head h, position i0 + b
    f32x4 wd[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) wd[e] = *reinterpret_cast<const f32x4*>(wh + i0 + 4 * e);
    float v[16][T];
#pragma unroll
    for (int b = 0; b < 16; ++b)
#pragma unroll
      for (int t = 0; t < T; ++t) {
        if constexpr (sizeof(KvT) == 2) v[b][t] = f32_of(static_cast<uint32_t>(vs[i0 + b][d0 + 64 * t]) << 16);
        else v[b][t] = vs[i0 + b][d0 + 64 * t];
      }
    auto one = [&](auto bb) __attribute__((always_inline)) {
      constexpr int b = decltype(bb)::value;
      unroll<T>([&](auto tt) {
        constexpr int t = decltype(tt)::value;
        acc[t] = __builtin_amdgcn_mfma_f32_4x4x1f32(wa, v[b][t], acc[t], 4, b, 0);
      });
      den = den + wd[b / 4][b % 4];
    };
    if (i0 + 16 <= n) {
      unroll<16>(one);
    } else {
      unroll<16>([&](auto bb) __attribute__((always_inline)) {
        if (i0 + decltype(bb)::value < n) one(bb);  // n is the same for every lane
      });
    }
  }
}

// One (row, page) item for one KV group (src/kernel_common.h:84-250). The page's
// V rows are fetched with 16-byte loads and parked in LDS, and each lane's K row
// is fetched whole, so both latencies overlap. Lane i scores position p0 + i for
// the four query heads; the page maximum is order-free; the exponentials follow, and
// each lane then mixes the values of its dims over the positions in order.
// KvT is uint16_t (bf16 KV, the tensor-core path) or float (the exact path);
// the arithmetic is the same, on the widened values. Taken by one wave, with LDS of its
// own; LDS accesses of a wave are performed in order, so its phases need no waits.
template <int D, class KvT>
struct PageLds {
  float wt[kHeadsPerGroup * kAttnPage];  // weights [head][position]
  KvT vs[kAttnPage][D];
};
template <int D, class KvT>
__device__ __forceinline__ void page_item(const StrideAttentionParams& p, int page_shift, int j, int slot, int visible, int page,
                                          int g, int lane, PageLds<D, KvT>& lds) {
  constexpr int kEl = 16 / static_cast<int>(sizeof(KvT));  // elements per 16-byte piece
  constexpr int kPer = kAttnPage * D / kEl / 64;  // pieces of one page of V per lane
  constexpr int kKey = D / kEl;                   // pieces of one K row
  const int p0 = page << kAttnPageShift;
  const int n = __builtin_amdgcn_readfirstlane(min(visible - p0, kAttnPage));

  // Positions past the row's last one are clamped to it (their values are never
  // used), so every load is unconditional and stays inside the row's own pages. Lane i
  // reads the KV page number of position p0 + i (src/kernel_common.h:20-25), and the
  // lanes that fetch its V row get it from there, so that two waits come before all of
  // the page's loads. (With a table read per piece of V the compiler, short of registers
  // at head_dim 128 in fp32, waited for every V load before the next table read: 64 rows
  // of 2900 positions, 8 groups, 619 us with the combine against 315.)
  const int last = visible - 1;
  const KvT* base = static_cast<const KvT*>(p.kv.arena) + p.layer * p.kv.layer_elems + g * p.kv.group_elems;
  const int at = min(p0 + lane, last), in_page = (1 << page_shift) - 1;
  const int block = p.kv.table[static_cast<int64_t>(slot) * p.kv.max_blocks + (at >> page_shift)];
  int vblock[kPer];
#pragma unroll
  for (int k = 0; k < kPer; ++k) vblock[k] = __shfl(block, (k * 64 + lane) / (D / kEl));
  __builtin_amdgcn_sched_barrier(0);  // one wait for them all
  u32x4 vr[kPer], kr[kKey];
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int P = k * 64 + lane, i = P / (D / kEl), c = P % (D / kEl);
    vr[k] = ld_kv(base + vblock[k] * p.kv.block_elems + p.kv.which_elems + (min(p0 + i, last) & in_page) * D + c * kEl);
  }
  {
    const KvT* key = base + block * p.kv.block_elems + (at & in_page) * D;
#pragma unroll
    for (int c = 0; c < kKey; ++c) kr[c] = load16(key + kEl * c);
  }
  float qa[D / 16];
  load_query<D>(p.q + static_cast<int64_t>(j) * p.q_stride + static_cast<int64_t>(g * kHeadsPerGroup) * D, lane, qa);
  __builtin_amdgcn_sched_barrier(0);  // every load before the first use
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int P = k * 64 + lane;
    *reinterpret_cast<u32x4*>(&lds.vs[P / (D / kEl)][(P % (D / kEl)) * kEl]) = vr[k];
  }
  const f32x4 a = page_scores<D, KvT>(kr, qa);
  const float neg_inf = f32_of(0xFF800000u);
  f32x4 mx;
#pragma unroll
  for (int h = 0; h < kHeadsPerGroup; ++h) {
    const float sc = lane < n ? a[h] * p.scale : neg_inf;
    mx[h] = wave_max(sc);
    if (lane < n) lds.wt[h * kAttnPage + lane] = det_exp(sc - mx[h]);
  }
  wave_phase();
  float* rec = p.scratch + (static_cast<int64_t>(j * p.n_kv + g) * p.max_pages + page) * p.rec_floats;
  f32x4 acc[(D + 63) / 64];
  float den;
  page_mix<D, KvT>(lds.wt, lds.vs, n, lane, acc, den);
#pragma unroll
  for (int t = 0; t < (D + 63) / 64; ++t)
#pragma unroll
    for (int h = 0; h < kHeadsPerGroup; ++h)
      if (lane + 64 * t < D) rec[8 + h * D + lane + 64 * t] = acc[t][h];
  if (lane < kHeadsPerGroup) {
    rec[lane] = mx[lane];
    rec[4 + lane] = den;
  }
  wave_phase();  // the next item's staging comes after this one's reads
}

// Tiles of kTileRows = 16 consecutive rows (k_attn_tile).
constexpr int kTileRows = 16;

// Where k_attn_tile tells k_attn_page whether it takes the tile of row j0: the first
// output of that row, which the combine overwrites after both.
template <class KvT>
__device__ __forceinline__ auto* tile_taken(const StrideAttentionParams& p, int j0) {
  if constexpr (sizeof(KvT) == 4) return static_cast<uint32_t*>(p.out) + j0;
  else return static_cast<uint16_t*>(p.out) + static_cast<int64_t>(j0 >> 4) * (p.out_cols >> 4) * kTileElems;
}

// Lane l holds row l % 16: its slot, and its visible positions (0 past the last row).
struct TileRow {
  int slot, visible;
};
__device__ __forceinline__ TileRow tile_row(const StrideAttentionParams& p, int j0, int lane) {
  const int nr = min(kTileRows, p.l.rows - j0), row = lane & (kTileRows - 1), j = j0 + min(row, nr - 1);
  const int slot = p.row_slot[j], pos = p.row_pos[j];
  return {slot, row < nr ? pos + 1 : 0};
}

// Do the rows lie in at most two sequences, at neighbouring positions? (Rows far apart
// share few pages that are whole for all of them.)
__device__ __forceinline__ bool tile_shared(TileRow tr) {
  const int first = __builtin_amdgcn_readfirstlane(tr.slot);
  int near = __builtin_amdgcn_readfirstlane(tr.visible);  // the position of this lane's sequence's first row
  const uint64_t others = __ballot(tr.slot != first);
  if (others != 0) {
    const int r = __builtin_ctzll(others), second = __builtin_amdgcn_readlane(tr.slot, r);
    if (__any(tr.slot != first && tr.slot != second)) return false;
    if (tr.slot != first) near = __builtin_amdgcn_readlane(tr.visible, r);
  }
  return !__any(tr.visible > 0 && abs(tr.visible - near) > kAttnPage / 2);
}

// Does the item list hold every page of the tile's rows where the pages of the rows
// before them end (as the engine's list does, src/engine.cpp:93-103)?
__device__ __forceinline__ bool tile_listed(const StrideAttentionParams& p, int j0, int lane, TileRow tr) {
  const int pages = (tr.visible + kAttnPage - 1) >> kAttnPageShift;
  if (__any(pages > p.max_pages)) return false;
  int lo = 0;  // items of the rows before the tile
#pragma unroll 16
  for (int r = lane; r < j0; r += 64) lo += (p.row_pos[r] >> kAttnPageShift) + 1;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) lo += __shfl_xor(lo, off);
  lo = __builtin_amdgcn_readfirstlane(lo);
  int end[kTileRows];  // items of the tile's rows up to each one
  int total = 0;
#pragma unroll
  for (int r = 0; r < kTileRows; ++r) end[r] = total += __builtin_amdgcn_readlane(pages, r);
  if (total > p.item_count - lo) return false;
  bool ok = true;
#pragma unroll 4
  for (int u = lane; u < total; u += 64) {
    int r = 0, c = u;  // item u of the tile: row r, page c
#pragma unroll
    for (int e = 0; e + 1 < kTileRows; ++e)
      if (u >= end[e]) {
        r = e + 1;
        c = u - end[e];
      }
    ok = ok & (p.items[2 * (lo + u)] == j0 + r) & (p.items[2 * (lo + u) + 1] == c);
  }
  return __all(ok);
}

// A tile's pages for one KV group: workgroup (tile, group, walker) takes pages walker,
// walker + walkers, ... of it and stores the records of page_item. Rows of one sequence
// share the pages that they read, and there the fmaf chains run as fp32 MFMAs
// (v_mfma_f32_16x16x4_f32 adds its four products in order, one rounding each: a chain of
// fmaf, bit for bit), K and V of a page being staged once, widened, for the sixteen rows. A wave holds four rows x four heads as the 16 columns i = 4 * row +
// head of the score tile (its rows: 16 positions; lane l holds column l % 16). Position
// 4v + a of a tile is its row 4a + v, so a lane's score register v of quarter a = l / 16
// is the mix's left operand of step v as it stands: the weights never leave their
// registers. They are also multiplied by ones (one more column tile of the mix), which
// adds the denominators in order. Positions past a row's last one must not enter its
// sums at all (a product with a zero weight could turn -0 into +0, or infinity into
// NaN): a page that is not whole for all of the wave's rows takes whole steps as MFMAs
// and its last few positions as fmaf under the row's own bound. Tiles whose rows
// share nothing (decode rows), or whose pages are not all listed, are left to k_attn_page:
// tile_taken() tells it.
//
// Bound by the fp32 units, which the MFMAs (144 of 32 cycles a wave and page) and vector
// instructions (490 of 4 cycles) take in turn: 81 % of them busy at 2048 rows of one
// prompt, 8 groups, head_dim 64 (counted): about 215 us, against 507 us a wave per item on
// the vector pipe alone.
template <int D, class KvT>
__global__ __launch_bounds__(256, D == 64 && sizeof(KvT) == 2 ? 3 : 2) void k_attn_tile(StrideAttentionParams p, int page_shift,
                                                                                     int walkers) {
  constexpr int kEl = 16 / static_cast<int>(sizeof(KvT));  // KV elements per 16-byte piece
  constexpr int kRow = D / kEl;                    // pieces of one K or V row
  constexpr int kPer = kAttnPage * kRow / 256;     // pieces of one page per thread
  constexpr int S4 = D / 4;                        // score steps
  constexpr int KS = D + 4;                        // K row stride in LDS (conflict-free column reads)
  constexpr int NDT = D / 16;                      // output column tiles
  constexpr int VW = D >= 64 ? 4 : 2;              // dims a lane reads of a V row at a time
  typedef float Word __attribute__((ext_vector_type(VW), aligned(4)));
  struct Tile {
    float ks[kAttnPage * KS];  // K: position, then dims 4s + a at a * S4 + s
    float vs[kAttnPage * D];
    float wb[4][16 * 16];      // a wave's weights of 16 positions
  };
  __shared__ __align__(16) Tile lds;
  auto& ks = lds.ks;
  auto& vs = lds.vs;
  auto& wb = lds.wb;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int per_tile = p.n_kv * walkers;
  const int blocks = (p.l.rows + kTileRows - 1) / kTileRows;
  // Later rows of a prompt read more pages: their workgroups start first.
  const int j0 = (blocks - 1 - static_cast<int>(blockIdx.x) / per_tile) * kTileRows;
  const int g = blockIdx.x % p.n_kv, walker = static_cast<int>(blockIdx.x) % per_tile / p.n_kv;
  const int rows4 = wave * 4;
  const TileRow tr = tile_row(p, j0, lane);
  const bool taken = tile_shared(tr) && tile_listed(p, j0, lane, tr);
  if (g == 0 && walker == 0 && tid == 0) *tile_taken<KvT>(p, j0) = taken ? 1 : 0;
  if (!taken || !__any(walker << kAttnPageShift < tr.visible)) return;
  const float neg_inf = f32_of(0xFF800000u);
  const int i = lane & 15, q = lane >> 4;

  // The rows of one sequence at a time (usually all sixteen).
  int slot = __builtin_amdgcn_readfirstlane(tr.slot);
  for (;;) {
    const int mine = tr.slot == slot ? tr.visible : 0;  // 0 for rows that are not the sequence's
    int last = 0;  // last position any of the sequence's rows sees
#pragma unroll
    for (int r = 0; r < kTileRows; ++r) last = max(last, __builtin_amdgcn_readlane(mine, r));
    --last;
    const int pages = (last >> kAttnPageShift) + 1;
    // Visible positions of the wave's rows, the least (of the sequence's) and the most.
    const int n0 = __builtin_amdgcn_readlane(mine, rows4), n1 = __builtin_amdgcn_readlane(mine, rows4 + 1);
    const int n2 = __builtin_amdgcn_readlane(mine, rows4 + 2), n3 = __builtin_amdgcn_readlane(mine, rows4 + 3);
    const int far = p.max_pages * kAttnPage;
    const int lo = min(min(n0 > 0 ? n0 : far, n1 > 0 ? n1 : far), min(n2 > 0 ? n2 : far, n3 > 0 ? n3 : far));
    const int hi = max(max(n0, n1), max(n2, n3));
    // This lane's row as a score column (row i / 4) and as an output row (row q).
    const int vis_i = (i >> 2) < 2 ? ((i >> 2) == 0 ? n0 : n1) : ((i >> 2) == 2 ? n2 : n3);
    const int vis_d = q < 2 ? (q == 0 ? n0 : n1) : (q == 2 ? n2 : n3);
    float qv[S4];
    {
      const int j = min(j0 + rows4 + (i >> 2), p.l.rows - 1);
      const float* src = p.q + static_cast<int64_t>(j) * p.q_stride + static_cast<int64_t>(g * kHeadsPerGroup + (i & 3)) * D + q;
#pragma unroll
      for (int e = 0; e < S4; ++e) qv[e] = src[4 * e];
    }

    // Staging: piece P = k * 256 + tid of a page is piece P % kRow of position P / kRow;
    // the page numbers of the page after next, and the pieces of the next page, are in
    // flight while a page is summed. Positions past `last` are loaded from it.
    // (Many pieces a thread, fp32 at head_dim 128: a page number a lane, of position `lane`
    // of the page, that the threads which fetch it get by lane exchange, and positions formed
    // anew for each page. With numbers and positions for each piece a thread kept some in
    // scratch memory, and waited for its loads to get them back: 2048 rows of one prompt, 8
    // groups, 549 us against 440. Few pieces: 226 us against 220 with the exchange.)
    constexpr bool kOwn = kPer <= 4;
    int blk[kOwn ? kPer : 1];
    u32x4 kr[kPer], vr[kPer];
    const KvT* base = static_cast<const KvT*>(p.kv.arena) + p.layer * p.kv.layer_elems + g * p.kv.group_elems + (tid % kRow) * kEl;
    const int32_t* table = p.kv.table + static_cast<int64_t>(slot) * p.kv.max_blocks;
    auto pos_of = [&](int page, int at) { return min((page << kAttnPageShift) + at, last); };
    auto load_blk = [&](int page) {
#pragma unroll
      for (int k = 0; k < (kOwn ? kPer : 1); ++k) blk[k] = table[pos_of(page, kOwn ? (k * 256 + tid) / kRow : lane) >> page_shift];
    };
    auto fetch = [&](int page) {
      int at0 = tid / kRow;  // of piece 0, in the page
      if constexpr (!kOwn) asm volatile("" : "+v"(at0));
      const int lane_blk = blk[0];
      if constexpr (!kOwn) load_blk(page + walkers);
#pragma unroll
      for (int k = 0; k < kPer; ++k) {
        const int at = at0 + k * (256 / kRow);
        const int64_t block = kOwn ? blk[kOwn ? k : 0] : __shfl(lane_blk, at);
        const KvT* src = base + block * p.kv.block_elems + (pos_of(page, at) & ((1 << page_shift) - 1)) * D;
        kr[k] = load16(src);
        vr[k] = load16(src + p.kv.which_elems);
      }
      if constexpr (kOwn) load_blk(page + walkers);
    };
    auto widen = [&](const u32x4& v, int e) {
      if constexpr (kEl == 8) return f32_of(e & 1 ? v[e >> 1] & 0xFFFF0000u : v[e >> 1] << 16);
      else return f32_of(v[e]);
    };
    load_blk(walker);
    fetch(walker);
    for (int c = walker; c < pages; c += walkers) {
      const int p0 = c << kAttnPageShift;
      lds_barrier();  // the last page has been read
#pragma unroll
      for (int k = 0; k < kPer; ++k) {
        const int pos = (k * 256 + tid) / kRow, d = (tid % kRow) * kEl;
#pragma unroll
        for (int a = 0; a < 4; ++a) {
          float* dst = &ks[pos * KS + a * S4 + d / 4];
          if constexpr (kEl == 8) *reinterpret_cast<f32x2*>(dst) = f32x2{widen(kr[k], a), widen(kr[k], 4 + a)};
          else *dst = widen(kr[k], a);
        }
        f32x4* dst = reinterpret_cast<f32x4*>(&vs[pos * D + d]);
#pragma unroll
        for (int e = 0; e < kEl / 4; ++e)
          dst[e] = f32x4{widen(vr[k], 4 * e), widen(vr[k], 4 * e + 1), widen(vr[k], 4 * e + 2), widen(vr[k], 4 * e + 3)};
      }
      lds_barrier();
      if (c + walkers < pages) fetch(c + walkers);
      if (p0 >= hi) continue;
      // Scores of positions 16t + 4v + q for column i; past the row's last one -inf.
      f32x4 w[4];
      const f32x4* src = reinterpret_cast<const f32x4*>(&ks[(4 * (i & 3) + (i >> 2)) * KS + q * S4]);
      unroll<S4 / 4>([&](auto ee) {
        constexpr int e = decltype(ee)::value;
        f32x4 k4[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) k4[t] = src[t * 4 * KS + e];
        unroll<16>([&](auto xx) {
          constexpr int x = decltype(xx)::value / 4, t = decltype(xx)::value % 4;
          const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
          w[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(k4[t][x], qv[4 * e + x], e == 0 && x == 0 ? zero : w[t], 0, 0, 0);
        });
      });
      const bool partial = p0 + kAttnPage > lo;
      const int n_i = vis_i - p0;
      float mx = neg_inf;
#pragma unroll
      for (int t = 0; t < 4; ++t) w[t] = w[t] * p.scale;
      if (partial) {
        unroll<16>([&](auto ee) {
          constexpr int t = decltype(ee)::value / 4, v = decltype(ee)::value % 4;
          if (16 * t + 4 * v + q >= n_i) w[t][v] = neg_inf;
        });
      }
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int v = 0; v < 4; ++v) mx = fmaxf(mx, w[t][v]);
      {  // over the column's four quarters
        const auto r16 = __builtin_amdgcn_permlane16_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
        mx = fmaxf(__uint_as_float(r16[0]), __uint_as_float(r16[1]));
        const auto r32 = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
        mx = fmaxf(__uint_as_float(r32[0]), __uint_as_float(r32[1]));
      }
      unroll<16>([&](auto ee) {
        constexpr int t = decltype(ee)::value / 4, v = decltype(ee)::value % 4;
        w[t][v] = det_exp(w[t][v] - mx);
      });
      f32x4 mix[NDT], dn = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int t = 0; t < NDT; ++t) mix[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      // Output column of tile t: dim 64 * (t / 4) + 4 * i + t % 4 (D = 32: 2 * i + t).
      auto v_row = [&](int pos, float (&vv)[NDT]) {
#pragma unroll
        for (int hh = 0; hh < NDT / VW; ++hh) {
          const Word x = *reinterpret_cast<const Word*>(&vs[pos * D + 64 * hh + VW * i]);
#pragma unroll
          for (int e = 0; e < VW; ++e) vv[VW * hh + e] = x[e];
        }
      };
      if (!partial) {
        unroll<16>([&](auto ee) __attribute__((always_inline)) {
          constexpr int e = decltype(ee)::value;
          float vv[NDT];
          v_row(4 * e + q, vv);
          const float a = w[e / 4][e % 4];
          dn = __builtin_amdgcn_mfma_f32_16x16x4f32(a, 1.0f, dn, 0, 0, 0);
          unroll<NDT>([&](auto tt) {
            constexpr int t = decltype(tt)::value;
            mix[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, vv[t], mix[t], 0, 0, 0);
          });
        });
      } else {
        // Steps that not all of the wave's rows see whole multiply -0 by 1: a sum plus -0
        // is that sum, whatever it is. (Branches around them would expose every LDS read.)
        const int whole_steps = min(max(lo - p0, 0), kAttnPage) / 4;
        unroll<16>([&](auto ee) __attribute__((always_inline)) {
          constexpr int e = decltype(ee)::value;
          const bool live = e < whole_steps;
          float vv[NDT];
          v_row(4 * e + q, vv);
          const float a = live ? w[e / 4][e % 4] : -0.0f;
          dn = __builtin_amdgcn_mfma_f32_16x16x4f32(a, 1.0f, dn, 0, 0, 0);
          unroll<NDT>([&](auto tt) {
            constexpr int t = decltype(tt)::value;
            mix[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, live ? vv[t] : 1.0f, mix[t], 0, 0, 0);
          });
        });
        const int n_d = vis_d - p0, end = min(hi - p0, kAttnPage);
        for (int c0 = 4 * whole_steps; c0 < end; c0 += 16) {  // usually once
          wave_phase();
          unroll<16>([&](auto ee) __attribute__((always_inline)) {
            constexpr int t = decltype(ee)::value / 4, v = decltype(ee)::value % 4;
            const int at = 16 * t + 4 * v + q - c0;
            if (at >= 0 && at < 16) wb[wave][at * 16 + i] = w[t][v];
          });
          wave_phase();
          for (int pos = c0; pos < min(c0 + 16, end); pos += 4) {
            f32x4 wv[4];
            float vv[4][NDT];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              wv[e] = *reinterpret_cast<const f32x4*>(&wb[wave][(pos - c0 + e) * 16 + 4 * q]);
              v_row(pos + e, vv[e]);
            }
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (pos + e < n_d) {
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                  dn[v] = dn[v] + wv[e][v];
#pragma unroll
                  for (int u = 0; u < NDT; ++u) mix[u][v] = __builtin_fmaf(wv[e][v], vv[e][u], mix[u][v]);
                }
              }
          }
        }
      }
      auto record = [&](int row) {
        return p.scratch + ((static_cast<int64_t>(j0 + rows4 + row) * p.n_kv + g) * p.max_pages + c) * p.rec_floats;
      };
      if (q == 0 && n_i > 0) record(i >> 2)[i & 3] = mx;
      if (p0 < vis_d) {
        float* rec = record(q);
        if (i == 0) {
#pragma unroll
          for (int v = 0; v < 4; ++v) rec[4 + v] = dn[v];
        }
#pragma unroll
        for (int v = 0; v < 4; ++v)
#pragma unroll
          for (int hh = 0; hh < NDT / VW; ++hh) {
            Word x;
#pragma unroll
            for (int e = 0; e < VW; ++e) x[e] = mix[VW * hh + e][v];
            *reinterpret_cast<Word*>(&rec[8 + v * D + 64 * hh + VW * i]) = x;
          }
      }
    }
    // the other sequence's rows, if the first row's have just been done
    const uint64_t others = __ballot(tr.slot != __builtin_amdgcn_readfirstlane(tr.slot));
    if (others == 0 || slot != __builtin_amdgcn_readfirstlane(tr.slot)) break;
    slot = __builtin_amdgcn_readlane(tr.slot, __builtin_ctzll(others));
  }
}

// Items one by one: a wave takes `per_wg` (at most 64) consecutive items of one KV
// group. TILED: those of tiles that k_attn_tile takes are skipped. An item outside the
// record array (page >= max_pages) would write into the next row's records: it is skipped
// (the caller sizes max_pages for its longest row).
template <int D, class KvT, bool TILED>
__global__ __launch_bounds__(64) void k_attn_page(StrideAttentionParams p, int page_shift, int per_wg) {
  __shared__ PageLds<D, KvT> lds;
  const int g = blockIdx.x % p.n_kv, lane = threadIdx.x;
  if constexpr (!TILED) {  // per_wg = 1
    const int one = static_cast<int>(blockIdx.x) / p.n_kv;
    const int j = p.items[2 * one], page = p.items[2 * one + 1];
    if (page >= 0 && page < p.max_pages)
      page_item<D, KvT>(p, page_shift, j, p.row_slot[j], p.row_pos[j] + 1, page, g, lane, lds);
    return;
  }
  const int item = static_cast<int>(blockIdx.x) / p.n_kv * per_wg + lane;  // this lane's
  int row = 0, page = -1;
  if (lane < per_wg && item < p.item_count) {
    row = p.items[2 * item];
    page = p.items[2 * item + 1];
  }
  const bool valid = page >= 0 && page < p.max_pages && row >= 0 && row < p.l.rows;
  row = valid ? row : 0;
  uint64_t todo = __ballot(valid && *tile_taken<KvT>(p, row & ~(kTileRows - 1)) == 0);
  if (todo == 0) return;
  const int slot = p.row_slot[row], visible = p.row_pos[row] + 1;
  for (; todo != 0; todo &= todo - 1) {
    const int n = __builtin_ctzll(todo);
    page_item<D, KvT>(p, page_shift, __builtin_amdgcn_readlane(row, n), __builtin_amdgcn_readlane(slot, n),
                      __builtin_amdgcn_readlane(visible, n), __builtin_amdgcn_readlane(page, n), g, lane, lds);
  }
}

// Ascending-page combine of one row's records for one KV group, written as bf16
// x tiles (src/kernel_common.h:252-309, writer src/kernels_tc.cu:658-666) or,
// for the exact path, as fp32 dim-major out[idx * stride + row] (LaneWriter,
// src/kernels.cu:287-291). Bound by reading the records once. Wave h derives head h's
// page factors, a page per lane; then thread (h, d) folds the weighted values of head h,
// dim d over the pages in order, straight from memory (a page's are 1 KiB at head_dim
// 64), with the denominator beside them. 2048 rows of up to 32 pages, 8 groups: 181 us
// when one thread per head walked the pages and all records went through LDS.
template <int D, bool kExact>
__global__ __launch_bounds__(256) void k_attn_combine(StrideAttentionParams p) {
  extern __shared__ f32x2 fd[];  // [4][pages]: page factor, page denominator
  const int j = blockIdx.x / p.n_kv;
  const int g = blockIdx.x % p.n_kv;
  const int t = threadIdx.x, wave = t >> 6, lane = t & 63;
  const int pages = min((p.row_pos[j] >> kAttnPageShift) + 1, p.max_pages);  // row_pos < 64 * max_pages
  const int64_t rf = p.rec_floats;
  const float* recs = p.scratch + static_cast<int64_t>(j * p.n_kv + g) * p.max_pages * rf;
  // The first pages' values come with their factors' inputs (1000 rows of one page, 8 groups,
  // head_dim 64: 9.7 us, 10.5 with the values read after the factors; 1024 rows of six
  // pages 18.9 / 23.1).
  constexpr int kPer = (kHeadsPerGroup * D + 255) / 256, kAhead = 4;
  float ahead[kPer][kAhead];
#pragma unroll
  for (int e = 0; e < kPer; ++e)
#pragma unroll
    for (int c = 0; c < kAhead; ++c)
      ahead[e][c] = recs[max(min(c, pages - 1), 0) * rf + 8 + min(t + 256 * e, kHeadsPerGroup * D - 1)];
  {
    float m = f32_of(0xFF800000u);
    for (int c = lane; c < pages; c += 64) m = pick_gt(recs[c * rf + wave], m);
    if (pages <= 4) {  // in lanes 0 .. 3, -infinity past the last
      float of[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) of[c] = f32_of(__builtin_amdgcn_readlane(u32_of(m), c));
      m = pick_gt(pick_gt(of[0], of[1]), pick_gt(of[2], of[3]));
    } else {
      m = wave_max(m);
    }
    for (int c = lane; c < pages; c += 64) fd[wave * pages + c] = f32x2{det_exp(recs[c * rf + wave] - m), recs[c * rf + 4 + wave]};
  }
  __syncthreads();
  const int col_tiles = p.out_cols >> 4;
  uint16_t* out = static_cast<uint16_t*>(p.out);
  const int64_t lane0 = static_cast<int64_t>(j >> 4) * col_tiles * kTileElems + (j & 15) * 16;
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    const int hd = t + 256 * u;
    if (hd >= kHeadsPerGroup * D) break;
    const int qh = hd / D, d = hd % D;
    const f32x2* f = fd + qh * pages;
    float acc = 0.0f, dn = 0.0f;
    auto page = [&](int c, float v) {
      const f32x2 e = f[c];
      dn = __builtin_fmaf(e[0], e[1], dn);
      acc = __builtin_fmaf(e[0], v, acc);
    };
#pragma unroll
    for (int c = 0; c < kAhead; ++c)
      if (c < pages) page(c, ahead[u][c]);
    // Eight values in flight, also at the end (the last ones one by one: a row of 74 pages, 2
    // groups, head_dim 128 18.7 us against 17.7).
    float v[8];
    int c0 = kAhead;
    for (; c0 + 8 <= pages; c0 += 8) {
#pragma unroll
      for (int c = 0; c < 8; ++c) v[c] = recs[(c0 + c) * rf + 8 + hd];
#pragma unroll
      for (int c = 0; c < 8; ++c) page(c0 + c, v[c]);
    }
    if (c0 < pages) {
#pragma unroll
      for (int c = 0; c < 8; ++c) v[c] = recs[min(c0 + c, pages - 1) * rf + 8 + hd];
#pragma unroll
      for (int c = 0; c < 8; ++c)
        if (c0 + c < pages) page(c0 + c, v[c]);
    }
    const int idx = (g * kHeadsPerGroup + qh) * D + d;
    if constexpr (kExact) static_cast<float*>(p.out)[static_cast<int64_t>(idx) * p.l.stride + j] = acc / dn;
    else out[lane0 + static_cast<int64_t>(idx >> 4) * kTileElems + (idx & 15)] = static_cast<uint16_t>(bf16_rne(acc / dn));
  }
}

// Pages and combine in one kernel. One workgroup per (row, KV group): its NWV
// waves take the row's 64-position pages round robin, each summing a page
// exactly as k_attn_page does (the same expressions in the same order) into a
// record kept in LDS; after a barrier the workgroup combines the records in
// ascending page order exactly as k_attn_combine does and writes the bf16 x
// tiles (KvT = uint16_t: bf16 KV, the tensor-core path) or the fp32 dim-major
// output (KvT = float, kExact: the exact path's fp32 KV). No second launch is
// needed.
//
// LIST = false: item_count == -1, every page of every row is computed.
// LIST = true: the caller's (row, page) item list decides, with the semantics of
// the page + combine pair (listed pages are summed now, the others are combined
// from the records `scratch` holds). The list the reference's engine builds
// (src/engine.cpp:93-103: rows ascending, each row's pages 0 .. last ascending)
// puts row j's items at offset sum_{i<j} pages_i; the workgroup computes that
// offset from row_pos and checks its row's stretch of the list. When it matches
// (every page listed) the records stay in LDS and scratch is not touched.
// Otherwise the workgroup scans the whole list for its row, sums the listed
// pages, reads the unlisted pages' records from scratch and stores the records
// it summed there, as k_attn_page would.
constexpr int kListMaxPages = 320;  // pages a LIST workgroup tracks (the LDS bound is lower)

template <int D, int NWV, bool LIST, class KvT = uint16_t, bool kExact = false>
__global__ __launch_bounds__(64 * NWV) void k_attn_fused(StrideAttentionParams p, int page_shift) {
  constexpr int kEl = 16 / static_cast<int>(sizeof(KvT));  // KV elements per 16-byte piece
  constexpr int kPer = kAttnPage * D / kEl / 64;  // V pieces per lane
  constexpr int kKey = D / kEl;                 // 16-byte pieces of one K row
  constexpr int RF = 8 + kHeadsPerGroup * D;    // record floats
  extern __shared__ float recs[];  // [max_pages][RF], f[4][max_pages], then the row's KV page numbers
  __shared__ __align__(16) float wt[NWV][kHeadsPerGroup * kAttnPage];  // weights [head][position]
  __shared__ KvT vs[NWV][kAttnPage][D];
  __shared__ uint32_t listed[LIST ? kListMaxPages / 32 : 1];
  __shared__ int part[NWV];
  const int j = blockIdx.x / p.n_kv;
  const int g = blockIdx.x % p.n_kv;
  const int t = threadIdx.x, wave = t >> 6, lane = t & 63;
  const int slot = p.row_slot[j];
  const int visible = p.row_pos[j] + 1;
  const int last = visible - 1;
  // A row must satisfy row_pos < max_pages * 64 (the caller sizes max_pages for
  // its longest row); the clamp keeps a row past it inside this workgroup's LDS.
  const int pages = min((last >> kAttnPageShift) + 1, p.max_pages);
  // The row's KV page numbers, read once: every K/V address below then comes
  // from LDS, so a page's loads never wait on a dependent page-table load.
  int32_t* btab = reinterpret_cast<int32_t*>(recs + p.max_pages * (RF + kHeadsPerGroup));
  const int nblk = min((last >> page_shift) + 1, (p.max_pages * kAttnPage + (1 << page_shift) - 1) >> page_shift);
  for (int i = t; i < nblk; i += 64 * NWV) btab[i] = p.kv.table[static_cast<int64_t>(slot) * p.kv.max_blocks + i];
  const KvT* kv_base = static_cast<const KvT*>(p.kv.arena) + p.layer * p.kv.layer_elems + g * p.kv.group_elems;
  auto kv_at = [&](int which, int pos) {
    return kv_base + btab[pos >> page_shift] * p.kv.block_elems + which * p.kv.which_elems +
           static_cast<int64_t>(pos & ((1 << page_shift) - 1)) * D;
  };
  __syncthreads();
  const float* qrow = p.q + static_cast<int64_t>(j) * p.q_stride + static_cast<int64_t>(g * kHeadsPerGroup) * D;
  float qa[D / 16];
  load_query<D>(qrow, lane, qa);
  const float neg_inf = f32_of(0xFF800000u);
  const int rounds = (pages + NWV - 1) / NWV;  // the same for every wave: barriers stay uniform
  // K and V of the wave's next page are loaded into registers one round ahead:
  // they stream in while the current page is scored and mixed.
  u32x4 vr[kPer], kr[kKey];
  auto fetch = [&](int page) {
    const int p0 = page << kAttnPageShift;
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      const int P = k * 64 + lane, i = P / (D / kEl), c = P % (D / kEl);
      vr[k] = ld_kv(kv_at(1, min(p0 + i, last)) + c * kEl);
    }
    const KvT* key = kv_at(0, min(p0 + lane, last));
#pragma unroll
    for (int c = 0; c < kKey; ++c) kr[c] = load16(key + kEl * c);
  };
  // LIST: does the item list hold row j's pages where the engine's list puts them?
  // (The page counts of the rows before j are loaded before the first page, so
  // the check's loads overlap that page's.)
  int s = 0;
  if constexpr (LIST)
    for (int i = t; i < j; i += 64 * NWV) s += (p.row_pos[i] >> kAttnPageShift) + 1;
  if (wave < pages) fetch(wave);
  // Round 0 runs before the list check completes and sums whichever pages it
  // takes; if the check then fails, the unlisted pages' records are replaced
  // from scratch before anything reads them.
  bool whole = true, checked = !LIST;
  int list_ok = 1, off_list = 0;
  int32_t item_row = 0, item_page = 0;
  auto is_listed = [&](int page) { return !checked || whole || ((listed[page >> 5] >> (page & 31)) & 1u); };
  for (int it = 0; it < rounds; ++it) {
    const int page = it * NWV + wave;
    const bool active = page < pages && is_listed(page);
    const int p0 = page << kAttnPageShift;
    const int n = active ? min(visible - p0, kAttnPage) : 0;
    if (active) {
#pragma unroll
      for (int k = 0; k < kPer; ++k) {
        const int P = k * 64 + lane;
        *reinterpret_cast<u32x4*>(&vs[wave][P / (D / kEl)][(P % (D / kEl)) * kEl]) = vr[k];
      }
    }
    if constexpr (LIST) {
      if (it == 0) {
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
        if (lane == 0) part[wave] = s;
      }
    }
    __syncthreads();  // this wave's V rows
    if constexpr (LIST) {
      if (it == 0) {  // row j's stretch of the list: loads issued now, compared at the end of the round
#pragma unroll
        for (int w = 0; w < NWV; ++w) off_list += part[w];
        list_ok = off_list + pages <= p.item_count;
        if (list_ok && t < pages) {
          item_row = p.items[2 * (off_list + t)];
          item_page = p.items[2 * (off_list + t) + 1];
        } else {
          item_row = j;
          item_page = t;
        }
      }
    }
    f32x4 mx = {0.f, 0.f, 0.f, 0.f};
    float sc[kHeadsPerGroup] = {0.f, 0.f, 0.f, 0.f};
    if (active) {
      const f32x4 a = page_scores<D, KvT>(kr, qa);
#pragma unroll
      for (int h = 0; h < kHeadsPerGroup; ++h) sc[h] = a[h] * p.scale;
    }
    if (page + NWV < pages) fetch(page + NWV);  // registers are free again
    if (active) {
#pragma unroll
      for (int h = 0; h < kHeadsPerGroup; ++h) {
        if (lane >= n) sc[h] = neg_inf;
        mx[h] = wave_max(sc[h]);
        if (lane < n) wt[wave][h * kAttnPage + lane] = det_exp(sc[h] - mx[h]);
      }
    }
    __syncthreads();  // this wave's weights
    if (active) {
      float* rec = recs + page * RF;
      f32x4 acc[(D + 63) / 64];
      float dn;
      page_mix<D, KvT>(wt[wave], vs[wave], __builtin_amdgcn_readfirstlane(n), lane, acc, dn);
#pragma unroll
      for (int t = 0; t < (D + 63) / 64; ++t)
#pragma unroll
        for (int h = 0; h < kHeadsPerGroup; ++h)
          if (lane + 64 * t < D) rec[8 + h * D + lane + 64 * t] = acc[t][h];
      if (lane < kHeadsPerGroup) {
        rec[lane] = mx[lane];
        rec[4 + lane] = dn;
      }
    }
    __syncthreads();  // the staging buffers are reused by the next round
    if constexpr (LIST) {
      if (it == 0) {
        int ok = list_ok && item_row == j && item_page == t;
        for (int c = t + 64 * NWV; ok && c < pages; c += 64 * NWV)  // rows of more pages than threads
          ok = p.items[2 * (off_list + c)] == j && p.items[2 * (off_list + c) + 1] == c;
        whole = __syncthreads_and(ok) != 0;
        checked = true;
        if (!whole) {
          for (int i = t; i < kListMaxPages / 32; i += 64 * NWV) listed[i] = 0u;
          __syncthreads();
          for (int i = t; i < p.item_count; i += 64 * NWV) {
            const int c = p.items[2 * i + 1];
            if (p.items[2 * i] == j && c >= 0 && c < pages) atomicOr(&listed[c >> 5], 1u << (c & 31));
          }
          __syncthreads();
          // unlisted pages: the records an earlier call left in scratch (over
          // whatever round 0 summed for them)
          const float* src = p.scratch + static_cast<int64_t>(j * p.n_kv + g) * p.max_pages * p.rec_floats;
          for (int u = t; u < pages * RF; u += 64 * NWV) {
            const int c = u / RF, e = u % RF;
            if (!((listed[c >> 5] >> (c & 31)) & 1u)) recs[c * RF + e] = src[static_cast<int64_t>(c) * p.rec_floats + e];
          }
          __syncthreads();
        }
      }
    }
  }
  if constexpr (LIST) {
    if (!whole) {  // store the summed records, as the page kernel does
      float* dst = p.scratch + static_cast<int64_t>(j * p.n_kv + g) * p.max_pages * p.rec_floats;
      for (int u = t; u < pages * RF; u += 64 * NWV) {
        const int c = u / RF, e = u % RF;
        if ((listed[c >> 5] >> (c & 31)) & 1u) dst[static_cast<int64_t>(c) * p.rec_floats + e] = recs[c * RF + e];
      }
    }
  }
  // Combine in ascending page order (k_attn_combine's expressions). Each page
  // factor is computed by its own thread; every thread derives the head maximum
  // with the same ascending loop, so all agree; each output thread then forms
  // its head's denominator and its dim's sum over the pages in order.
  float* f = recs + pages * RF;
  for (int u = t; u < kHeadsPerGroup * pages; u += 64 * NWV) {
    const int h = u & 3, c = u >> 2;
    float m = neg_inf;
    for (int c2 = 0; c2 < pages; ++c2) {
      const float mc = recs[c2 * RF + h];
      if (mc > m) m = mc;
    }
    f[h * pages + c] = det_exp(recs[c * RF + h] - m);
  }
  __syncthreads();
  const int col_tiles = p.out_cols >> 4;
  uint16_t* out = static_cast<uint16_t*>(p.out);
  const int64_t lane0 = kExact ? 0 : static_cast<int64_t>(j >> 4) * col_tiles * kTileElems + (j & 15) * 16;
  for (int hd = t; hd < kHeadsPerGroup * D; hd += 64 * NWV) {
    const int qh = hd / D, d = hd % D;
    float acc = 0.0f, dn = 0.0f;
    for (int c = 0; c < pages; ++c) {
      const float e = f[qh * pages + c];
      dn = __builtin_fmaf(e, recs[c * RF + 4 + qh], dn);
      acc = __builtin_fmaf(e, recs[c * RF + 8 + qh * D + d], acc);
    }
    const int idx = (g * kHeadsPerGroup + qh) * D + d;
    if constexpr (kExact) static_cast<float*>(p.out)[static_cast<int64_t>(idx) * p.l.stride + j] = acc / dn;
    else out[lane0 + static_cast<int64_t>(idx >> 4) * kTileElems + (idx & 15)] = static_cast<uint16_t>(bf16_rne(acc / dn));
  }
}

bool lanes_valid(const StrideLanes& l) { return l.rows >= 0 && l.lane_groups == (l.rows + 15) / 16; }

}  // namespace
}  // namespace stride_tc

using namespace stride_tc;

static_assert(sizeof(StrideTcEmbedParams) == 48, "TcEmbedParams layout");
static_assert(sizeof(StrideTcNormParams) == 48, "TcNormParams layout");
static_assert(sizeof(StrideTcCompactParams) == 48, "TcCompactParams layout");
static_assert(offsetof(StrideAttentionParams, kv) == 48 && sizeof(StrideAttentionParams) == 176,
              "AttentionParams layout");

static int launched(const char* what);

// LDS that the one-kernel form may take (160 KiB less a margin). Also the bound on a row's
// records and page factors in every form, so that what a call may ask for does not depend on
// the form that takes it (the page kernels and the combine alone would need 32 bytes of LDS
// a page).
constexpr size_t kRowLdsMax = 159 * 1024;

// One-kernel attention; its static LDS (staging for up to four waves) and the
// row's records share the 160 KiB.
template <int D, int NWV, class KvT>
constexpr size_t fused_static_lds() {
  return NWV * 64 * 16 + NWV * 64 * D * sizeof(KvT) + kListMaxPages / 8 + 4 * NWV;
}

template <int D, int NWV, bool LIST, class KvT, bool kExact>
static int fused_nwv(dim3 grid, size_t lds, hipStream_t st, const StrideAttentionParams& p, int page_shift) {
  if (lds + fused_static_lds<D, NWV, KvT>() > kRowLdsMax)
    return fail(STRIDE_TC_EINVAL, "tc_attention: max_pages too large for the one-kernel form (use an item list)");
  static size_t raised = 64 * 1024;
  if (lds > raised) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_attn_fused<D, NWV, LIST, KvT, kExact>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
    if (e != hipSuccess) return fail(static_cast<int>(e), std::string("tc_attention: raising the LDS limit failed: ") + hipGetErrorString(e));
    raised = lds;
  }
  hipLaunchKernelGGL((k_attn_fused<D, NWV, LIST, KvT, kExact>), grid, dim3(64 * NWV), lds, st, p, page_shift);
  return launched("attention (one kernel)");
}

// Waves per workgroup of the one-kernel form, from measurements of the full
// decode step at position 383 (six pages per row): with many (row, group)
// workgroups (batch 128, 1024 of them) two waves per workgroup (three rounds of
// pages) measured best (30.9 us against 32.4 with three and 33+ with four); with
// fewer (batch 64) four waves finish a row sooner.
template <int D, bool LIST, class KvT = uint16_t, bool kExact = false>
static int fused(dim3 grid, size_t lds, hipStream_t st, const StrideAttentionParams& p, int page_shift) {
  if (grid.x >= 768) return fused_nwv<D, 2, LIST, KvT, kExact>(grid, lds, st, p, page_shift);
  return fused_nwv<D, 4, LIST, KvT, kExact>(grid, lds, st, p, page_shift);
}

// Does the one-kernel form serve a call with this dynamic LDS? (4 waves: the
// larger static staging.)
template <int D, class KvT = uint16_t>
static bool fused_fits(size_t lds) {
  return lds + fused_static_lds<D, 4, KvT>() <= kRowLdsMax;
}

// Item-list calls run the one-kernel form (which checks the list on the device)
// for up to this many rows: each workgroup sums the page counts of the rows
// before its own to find its stretch of the list, which grows with the row count.
constexpr int kListFusedMaxRows = 512;

// Page sums and combine in launches of their own.
template <int D, class KvT, bool kExact>
static int paged(hipStream_t st, const StrideAttentionParams& p, int page_shift) {
  // Tiles for 128 to 8192 rows (a smaller batch that comes here, contexts beyond the
  // one-kernel form's LDS, may as well be decode rows, and each tile adds up the pages of
  // all rows before it) and long lists: finding out what is whose costs two to three
  // launches' latency, which 32768 items and groups are worth (whole attention, tiles
  // against items: 18.5 k 38 against 45 us, 26.6 k 62 / 69, 41.6 k 77 / 100, but 19.7 k, four prompts of
  // 250 rows between other kernels, 60 / 57, and 28.8 k of 600 decode rows, which take
  // both ways, 81 / 70; 82 k 144, 270 k 273 us, against 203 and 695 before there were tiles).
  const int64_t waves = static_cast<int64_t>(p.item_count) * p.n_kv;
  if (waves > 32768 && p.l.rows >= 128 && p.l.rows <= 8192) {
    // Walkers: as many workgroups as the chip holds at once, about four to a CU (1000
    // rows in four prompts, 504 tiles and groups: 36 us with two walkers, 39 with one,
    // 45 with four, which look at the list for one page each).
    const int tiles = (p.l.rows + kTileRows - 1) / kTileRows * p.n_kv;
    const int walkers = std::max(1, std::min(p.max_pages, 1024 / tiles));
    hipLaunchKernelGGL((k_attn_tile<D, KvT>), dim3(tiles * walkers), dim3(256), 0, st, p, page_shift, walkers);
    if (int rc = launched("attention (tiles)")) return rc;
    // Where the tiles take everything the waves below only find that out: several items
    // each, but waves enough for decode rows' items.
    const int per_wg = static_cast<int>(std::max<int64_t>(1, std::min<int64_t>(64, waves / 16384)));
    const dim3 grid((p.item_count + per_wg - 1) / per_wg * p.n_kv);
    hipLaunchKernelGGL((k_attn_page<D, KvT, true>), grid, dim3(64), 0, st, p, page_shift, per_wg);
    if (int rc = launched("attention (pages)")) return rc;
  } else if (p.item_count > 0) {
    hipLaunchKernelGGL((k_attn_page<D, KvT, false>), dim3(p.item_count * p.n_kv), dim3(64), 0, st, p, page_shift, 1);
    if (int rc = launched("attention (pages)")) return rc;
  }
  const size_t lds = static_cast<size_t>(p.max_pages) * kHeadsPerGroup * sizeof(f32x2);
  hipLaunchKernelGGL((k_attn_combine<D, kExact>), dim3(p.l.rows * p.n_kv), dim3(256), lds, st, p);
  return launched("attention (combine)");
}

static int launched(const char* what) {
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(static_cast<int>(e), std::string(what) + " launch failed: " + hipGetErrorString(e));
  return 0;
}

extern "C" {

int stride_tc_embed(const StrideTcEmbedParams* p, void* stream) {
  if (!p || !lanes_valid(p->l) || p->dim <= 0 || p->dim % 16 != 0 || (p->l.rows > 0 && (!p->embed || !p->tokens || !p->h)))
    return fail(STRIDE_TC_EINVAL, "tc_embed: need rows >= 0, lane_groups = ceil(rows/16), dim a positive multiple of 16 and pointers");
  if (p->l.rows == 0) return 0;
  hipLaunchKernelGGL(k_embed, dim3(p->l.rows), dim3(256), 0, static_cast<hipStream_t>(stream), *p);
  return launched("tc_embed");
}

int stride_tc_norm(const StrideTcNormParams* p, int per_lane, void* stream) {
  if (!p || !lanes_valid(p->l) || p->dim <= 0 || p->dim % 16 != 0 ||
      (p->l.rows > 0 && (!p->h || !p->x || !p->weight)))
    return fail(STRIDE_TC_EINVAL, "tc_norm: need rows >= 0, lane_groups = ceil(rows/16), dim a positive multiple of 16 and pointers");
  if (p->l.rows == 0) return 0;
  const dim3 grid(p->l.lane_groups * 16);
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int pl = per_lane ? 1 : 0;
  switch (p->dim) {
    case 512: hipLaunchKernelGGL(k_norm<1>, grid, dim3(64), 0, st, *p, pl); break;
    case 1024: hipLaunchKernelGGL(k_norm<2>, grid, dim3(64), 0, st, *p, pl); break;
    case 2048: hipLaunchKernelGGL(k_norm<4>, grid, dim3(64), 0, st, *p, pl); break;
    case 4096: hipLaunchKernelGGL(k_norm<8>, grid, dim3(64), 0, st, *p, pl); break;
    default: hipLaunchKernelGGL(k_norm<0>, grid, dim3(64), 0, st, *p, pl); break;
  }
  return launched("tc_norm");
}

int stride_tc_compact(const StrideTcCompactParams* p, void* stream) {
  if (!p || p->lm_count < 0 || p->col_tiles <= 0 || (p->lm_count > 0 && (!p->in || !p->out || !p->lm_rows)))
    return fail(STRIDE_TC_EINVAL, "tc_compact: need lm_count >= 0, col_tiles > 0 and pointers");
  if (p->lm_count == 0) return 0;
  hipLaunchKernelGGL(k_compact, dim3(p->lm_count), dim3(64), 0, static_cast<hipStream_t>(stream), *p);
  return launched("tc_compact");
}

}  // extern "C"

// Shared checks and launches of the tensor-core (bf16 KV, bf16 x-tile output)
// and exact (fp32 KV, fp32 dim-major output) attention.
template <bool kExact>
static int attention(const StrideAttentionParams* p, void* stream, const char* name) {
  if (!p) return fail(STRIDE_TC_EINVAL, std::string(name) + ": null parameters");
  const int D = p->head_dim;
  const int64_t page_tokens = D > 0 ? p->kv.group_elems / D : 0;
  int page_shift = 0;
  while (page_shift < 30 && (int64_t{1} << page_shift) < page_tokens) ++page_shift;
  std::string why;
  if (kExact ? (p->l.rows < 0 || p->l.stride < p->l.rows) : !lanes_valid(p->l))
    why = kExact ? "need rows >= 0 and stride >= rows" : "lane_groups must equal ceil(rows/16)";
  else if ((D != 32 && D != 64 && D != 128) || p->kv.head_dim != D) why = "head_dim must be 32, 64 or 128 and match kv.head_dim";
  else if (p->n_q != kHeadsPerGroup) why = "four query heads per KV group are required (the reference packs them in a float4)";
  else if (p->n_kv <= 0 || p->rec_floats < 8 + 4 * D || p->max_pages <= 0 || p->item_count < (kExact ? 0 : -1))
    why = "bad n_kv, rec_floats, max_pages or item_count";
  else if (page_tokens <= 0 || (int64_t{1} << page_shift) != page_tokens) why = "the KV storage page (group_elems / head_dim) must be a power of two";
  else if (!kExact && (p->out_cols % 16 != 0 || p->out_cols < p->n_kv * p->n_q * D)) why = "out_cols must be a multiple of 16 covering every head";
  else if (p->l.rows > 0 && (!p->q || !p->out || !p->kv.arena || !p->kv.table || !p->row_slot || !p->row_pos ||
                             (p->item_count >= 0 && !p->scratch) || (p->item_count > 0 && !p->items)))
    why = "missing pointer";
  else if (static_cast<size_t>(p->max_pages) * (p->rec_floats + kHeadsPerGroup) * sizeof(float) > kRowLdsMax)
    why = "a row's records and factors (max_pages * (rec_floats + 4) floats) must fit in 159 KiB";
  if (!why.empty()) return fail(STRIDE_TC_EINVAL, std::string(name) + ": " + why);
  if (p->l.rows == 0) return 0;
  hipStream_t st = static_cast<hipStream_t>(stream);
  using KvT = typename std::conditional<kExact, float, uint16_t>::type;
  {
    // records and page factors, then the row's KV page numbers
    const size_t blocks = (static_cast<size_t>(p->max_pages) * kAttnPage + page_tokens - 1) / page_tokens;
    const size_t lds = static_cast<size_t>(p->max_pages) * (8 + 4 * D + kHeadsPerGroup) * sizeof(float) + blocks * 4;
    const dim3 grid(p->l.rows * p->n_kv);
    if constexpr (!kExact) {
      if (p->item_count == -1) {
        if (D == 32) return fused<32, false>(grid, lds, st, *p, page_shift);
        if (D == 64) return fused<64, false>(grid, lds, st, *p, page_shift);
        return fused<128, false>(grid, lds, st, *p, page_shift);
      }
    }
    const bool fits = D == 32 ? fused_fits<32, KvT>(lds) : (D == 64 ? fused_fits<64, KvT>(lds) : fused_fits<128, KvT>(lds));
    if (fits && p->max_pages <= kListMaxPages && p->l.rows <= kListFusedMaxRows) {
      if (D == 32) return fused<32, true, KvT, kExact>(grid, lds, st, *p, page_shift);
      if (D == 64) return fused<64, true, KvT, kExact>(grid, lds, st, *p, page_shift);
      return fused<128, true, KvT, kExact>(grid, lds, st, *p, page_shift);
    }
  }
  if (D == 32) return paged<32, KvT, kExact>(st, *p, page_shift);
  if (D == 64) return paged<64, KvT, kExact>(st, *p, page_shift);
  return paged<128, KvT, kExact>(st, *p, page_shift);
}

extern "C" int stride_tc_attention(const StrideAttentionParams* p, void* stream) {
  return attention<false>(p, stream, "tc_attention");
}

// Exact path (src/kernels.cu:474-485): fp32 KV, fp32 dim-major output.
extern "C" int stride_k_attention(const StrideAttentionParams* p, void* stream) {
  return attention<true>(p, stream, "k_attention");
}
