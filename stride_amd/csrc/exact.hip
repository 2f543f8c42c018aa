// The exact path on gfx950: the reference's fused FP32 kernels (src/kernels.cu)
// evaluated on the GPU with the same IEEE operations, in the same order, per
// output element as the reference's CPU exact path, so the two agree bit for bit.
//
// Mapping. The reference runs one 32-thread block per (four-row weight group, lane
// group): thread t owns the 64-byte weight lines l == t mod 32, chaining fmaf over
// their columns in ascending order, and the 32 partial sums are added left to right,
// ((P0 + P1) + P2) + ... + P31. Here one batch lane runs two such blocks side by side
// in a 64-lane wavefront, lane t of a half being the reference's thread t; batches
// run the chains as fp32 MFMAs (below). Built with -ffp-contract=off, so only the
// explicit fmaf calls fuse; division and square root are the correctly rounded ones.
// Nothing here depends on the batch: an output depends on its own weight row and
// batch lane only.
#include <hip/hip_runtime.h>

#include <string>

#include "../../include/stride_exact.h"
#include "exact_lanes.hpp"
#include "tc_common.hpp"

namespace stride_tc {

int fail(int code, const std::string& msg);  // tc_gemm.hip

namespace {

constexpr int kChains = 32;  // partial chains per dot product (src/kernels.h kBlockThreads)

__device__ __forceinline__ float lo_half(uint32_t v) { return f32_of(v << 16); }
__device__ __forceinline__ float hi_half(uint32_t v) { return f32_of(v & 0xFFFF0000u); }

// Chain t of the dot products of one four-row weight group (wg: [col][4] bf16)
// with one row of x: acc[r] for row r. Lines of 8 columns: t, t + 32, ...; each line
// is four 16-byte words, word q holding columns k + 2q (rows 0-3 in its first two
// 32-bit halves' bf16 pairs) and k + 2q + 1 (last two) (src/kernels.cu:22-94).
__device__ __forceinline__ void chain(const uint16_t* wg, const float* x, int cols, int t, float (&acc)[4]) {
#pragma unroll
  for (int e = 0; e < 4; ++e) acc[e] = 0.0f;
  // Line k's weights (four 16-byte words) and x columns k .. k+7.
  struct Line {
    u32x4 v[4];
    f32x4 xc[2];
  };
  auto load = [&](int line, Line& L) {
    const int k = line * 8;
    const u32x4* wl = reinterpret_cast<const u32x4*>(wg + static_cast<int64_t>(k) * 4);
#pragma unroll
    for (int q = 0; q < 4; ++q) L.v[q] = wl[q];
    L.xc[0] = *reinterpret_cast<const f32x4*>(x + k);
    L.xc[1] = *reinterpret_cast<const f32x4*>(x + k + 4);
  };
  auto step = [&](const Line& L) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int c = 2 * q + h;  // column k + c
        const float w[4] = {lo_half(L.v[q][2 * h]), hi_half(L.v[q][2 * h]), lo_half(L.v[q][2 * h + 1]),
                            hi_half(L.v[q][2 * h + 1])};
        const float xc = L.xc[c >> 2][c & 3];
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[r] = __builtin_fmaf(w[r], xc, acc[r]);
      }
    }
  };
  // Lines t, t + 32, ... in ascending order, their loads issued NB lines at a
  // time so that a lane waits one memory round trip per batch, not per line.
  constexpr int NB = 8;
  const int lines = cols / 8;
  int line = t;
  for (; line + (NB - 1) * kChains < lines; line += NB * kChains) {
    Line L[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) load(line + b * kChains, L[b]);
    __builtin_amdgcn_sched_barrier(0);  // every load of the batch before the first use
#pragma unroll
    for (int b = 0; b < NB; ++b) step(L[b]);
  }
  for (; line < lines; line += kChains) {
    Line L;
    load(line, L);
    step(L);
  }
}

// ---------------------------------------------------------------------------
// GEMM-shaped operators: Op supplies the weight group(s) of a block and the
// epilogue on the folded sums y[m][r * J + j].

struct ResidualOp {  // src/kernels.cu:294-325
  using Params = StrideGemmResidualParams;
  static constexpr int kMats = 1;
  static int groups(const Params& p) { return p.m.groups; }
  static int cols(const Params& p) { return p.m.cols; }
  __device__ static const uint16_t* w(const Params& p, int, int group, int& cols) {
    cols = p.m.cols;
    return p.m.w + static_cast<int64_t>(group) * p.m.cols * 4;
  }
  template <int J>
  __device__ static void finish(const Params& p, int group, int lg, int t, const float (*y)[16]) {
    if (t >= 4 * J) return;
    const int r = t / J, jj = t % J;
    float* h = p.h + static_cast<int64_t>(group * 4 + r) * p.l.stride + lg * 4 + jj;
    h[0] = h[0] + y[0][t];
  }
};

struct Mlp13Op {  // src/kernels.cu:329-363
  using Params = StrideMlp13Params;
  static constexpr int kMats = 2;
  static int groups(const Params& p) { return p.w1.groups; }
  static int cols(const Params& p) { return p.w1.cols; }
  __device__ static const uint16_t* w(const Params& p, int m, int group, int& cols) {
    const StrideGemmMat& mm = m == 0 ? p.w1 : p.w3;
    cols = mm.cols;
    return mm.w + static_cast<int64_t>(group) * mm.cols * 4;
  }
  template <int J>
  __device__ static void finish(const Params& p, int group, int lg, int t, const float (*y)[16]) {
    if (t >= 4 * J) return;
    const int r = t / J, jj = t % J;
    p.z[static_cast<int64_t>(group * 4 + r) * p.l.stride + lg * 4 + jj] = det_silu(y[0][t]) * y[1][t];
  }
};

struct LmFullOp {  // src/kernels.cu:427-452
  using Params = StrideLmFullParams;
  static constexpr int kMats = 1;
  static int groups(const Params& p) { return p.m.groups; }
  static int cols(const Params& p) { return p.m.cols; }
  __device__ static const uint16_t* w(const Params& p, int, int group, int& cols) {
    cols = p.m.cols;
    return p.m.w + static_cast<int64_t>(group) * p.m.cols * 4;
  }
  template <int J>
  __device__ static void finish(const Params& p, int group, int lg, int t, const float (*y)[16]) {
    if (t >= 4 * J) return;
    const int r = t / J, jj = t % J;
    p.logits[static_cast<int64_t>(group * 4 + r) * p.l.stride + lg * 4 + jj] = y[0][t];
  }
};

struct LmGreedyOp {  // src/kernels.cu:383-425
  using Params = StrideLmGreedyParams;
  static constexpr int kMats = 1;
  static int groups(const Params& p) { return p.m.groups; }
  static int cols(const Params& p) { return p.m.cols; }
  __device__ static const uint16_t* w(const Params& p, int, int group, int& cols) {
    cols = p.m.cols;
    return p.m.w + static_cast<int64_t>(group) * p.m.cols * 4;
  }
  template <int J>
  __device__ static void finish(const Params& p, int group, int lg, int t, const float (*y)[16]) {
    if (t >= J) return;
    const int lane = lg * 4 + t;
    if (lane >= p.l.rows) return;
    float best = f32_of(0xFF800000u);
    int32_t best_i = -1;
    for (int r = 0; r < 4; ++r) {
      const int index = group * 4 + r;
      if (index >= p.vocab) continue;
      const float v = y[0][r * J + t];
      if (v > best) {
        best = v;
        best_i = index;
      }
    }
    if (best_i >= 0) best_update(&p.best[lane], best, best_i);
  }
};

struct QkvOp {  // src/kernels.cu:204-284
  using Params = StrideQkvParams;
  static constexpr int kMats = 1;
  static int groups(const Params& p) { return p.q.groups + 2 * p.k.groups; }
  static int cols(const Params& p) { return p.q.cols; }
  __device__ static const uint16_t* w(const Params& p, int, int gi, int& cols) {
    const StrideGemmMat& m = gi < p.q.groups ? p.q : (gi < p.q.groups + p.k.groups ? p.k : p.v);
    const int group = gi < p.q.groups ? gi : (gi < p.q.groups + p.k.groups ? gi - p.q.groups : gi - p.q.groups - p.k.groups);
    cols = m.cols;
    return m.w + static_cast<int64_t>(group) * m.cols * 4;
  }
  template <int J>
  __device__ static void finish(const Params& p, int gi, int lg, int t, const float (*y)[16]) {
    if (t >= J) return;
    const int j = lg * 4 + t;
    if (j >= p.l.rows) return;
    const int kind = gi < p.q.groups ? 0 : (gi < p.q.groups + p.k.groups ? 1 : 2);
    const int group = kind == 0 ? gi : (kind == 1 ? gi - p.q.groups : gi - p.q.groups - p.k.groups);
    const int D = p.head_dim, half = D / 2;
    const int head = group / (D / 4);
    const int d0 = 2 * (group % (D / 4));
    const int pos = p.row_pos[j], slot = p.row_slot[j];
    float a0 = y[0][0 * J + t], a1 = y[0][1 * J + t], b0 = y[0][2 * J + t], b1 = y[0][3 * J + t];
    if (kind != 2) {
      const float* cs = p.rope + (static_cast<int64_t>(pos) * half + d0) * 2;
      const float c0 = cs[0], s0 = cs[1], c1 = cs[2], s1 = cs[3];
      const float ra0 = a0 * c0 - b0 * s0, rb0 = b0 * c0 + a0 * s0;
      const float ra1 = a1 * c1 - b1 * s1, rb1 = b1 * c1 + a1 * s1;
      a0 = ra0;
      b0 = rb0;
      a1 = ra1;
      b1 = rb1;
    }
    float* dst;
    if (kind == 0) {
      dst = p.q_out + static_cast<int64_t>(j) * p.q_stride + static_cast<int64_t>(head) * D;
    } else {
      const StrideKvRef& kv = p.kv;
      const int64_t tokens = kv.group_elems / kv.head_dim;  // a power of two (checked on the host)
      const int64_t block = kv.table[static_cast<int64_t>(slot) * kv.max_blocks + pos / tokens];
      dst = static_cast<float*>(kv.arena) + block * kv.block_elems + p.layer * kv.layer_elems +
            (kind - 1) * kv.which_elems + head * kv.group_elems + (pos % tokens) * kv.head_dim;
    }
    dst[d0] = a0;
    dst[d0 + 1] = a1;
    dst[d0 + half] = b0;
    dst[d0 + half + 1] = b1;
  }
};

// The hardware hands workgroup i to XCD i % 8; logical workgroups are numbered so
// that consecutive ones (the lane blocks of one row block) share an XCD and so read
// that block's weights through one L2.
__device__ __forceinline__ int exact_wg_order(int i, int n) {
  const int full = n & ~7;
  if (i >= full) return i;
  return (i & 7) * (full >> 3) + (i >> 3);
}

// One batch lane (J = 1): two reference blocks (weight groups) per 64-lane workgroup,
// group = 2 * (logical workgroup) + half. Bound by the weight stream.
template <class Op>
__global__ __launch_bounds__(64) void k_exact_gemm(typename Op::Params p, int ngroups) {
  constexpr int M = Op::kMats;
  __shared__ float part[2][kChains][M][4];
  __shared__ float ys[2][M][16];
  const int half = threadIdx.x >> 5, t = threadIdx.x & 31;
  const int group = exact_wg_order(blockIdx.x, gridDim.x) * 2 + half;
  const bool live = group < ngroups;
  if (live) {
#pragma unroll
    for (int m = 0; m < M; ++m) {
      int cols = 0;
      const uint16_t* wg = Op::w(p, m, group, cols);
      float acc[4];
      chain(wg, p.x, cols, t, acc);
#pragma unroll
      for (int e = 0; e < 4; ++e) part[half][t][m][e] = acc[e];
    }
  }
  __syncthreads();
  if (live && t < 4) {
#pragma unroll
    for (int m = 0; m < M; ++m) {
      float y = part[half][0][m][t];
      for (int i = 1; i < kChains; ++i) y = y + part[half][i][m][t];
      ys[half][m][t] = y;
    }
  }
  __syncthreads();
  if (live) Op::template finish<1>(p, group, 0, t, ys[half]);
}

// Matrix form (four batch lanes per reference block). v_mfma_f32_16x16x4_f32 adds
// its four products one after the other, k ascending, each with one rounding: the
// same bits as four fmaf calls, denormals, signed zeros and infinities included
// (tests/test_gpu_kat.py checks it on the device). A chain of the reference is
// therefore a chain of MFMAs over its columns, at twice the rate of v_fma_f32
// (155 against 78 TFLOP/s).
//
// A workgroup of WC waves owns NG = 4 * R weight groups (16 * R rows) and 16 * L
// batch lanes. The 32 chains are dealt to the waves, CH neighbours at a time (two
// neighbours read whole 128-byte lines); a wave takes its chains for all rows and
// lanes of the tile, so a weight line and an x column are loaded once per
// workgroup. Every CPR turns of the waves their partials meet in LDS and are added
// left to right, ((P0 + P1) + P2) + ..., by the thread that keeps the output.
//
// Operands. A weight line holds 8 columns x 4 rows of a group (64 bytes): four lanes
// load it, 16 bytes (two columns) each, one batch of four lines ahead. A batch then
// goes through the wave's own LDS slot to reach the operand layout (lane l: row
// l % 16, column 4s + l / 16 of step s); with R row tiles a lane reads its R rows of
// one column as one 2R-byte word, tile r holding row r of the word. x columns are
// loaded in operand layout directly (lane l: column 4s + l / 16, batch lanes
// L * (l % 16) .. + L - 1 as one word, tile b holding lane b of the word).
//
// Bounds: few rows, the weight stream; many, the matrix pipe, which vector
// instructions stall (an fp32 MFMA and a vector instruction share the fp32 units:
// four v_add per four MFMAs take a bare MFMA loop from 154 to 136 TFLOP/s), so
// larger tiles win where there are enough of them. Against fmaf chains on the vector
// pipe, same box: N = 3072, K = 2048 at 8 / 32 / 256 rows 11.8 / 16.1 / 65 -> 7.3 /
// 9.8 / 38 us; 2048 x 8192 34 / 40 / 162 -> 18.1 / 20.0 / 79 us (109 TFLOP/s);
// 2 x 8192 x 2048 22.6 / 54 / 318 -> 18.1 / 27 / 177 us; 128256 x 2048 at 32 rows 354
// -> 184 us.
template <int N>
struct FloatsOf;
template <> struct FloatsOf<1> { typedef float T; };
template <> struct FloatsOf<2> { typedef f32x2 T; };
template <> struct FloatsOf<4> { typedef f32x4 T; };

template <class Op, int R, int L, int WC, int CH, int CPR>
__global__ __launch_bounds__(64 * WC) void k_exact_gemm_m(typename Op::Params p, int nlb, int ngroups) {
  constexpr int M = Op::kMats;
  constexpr int NG = 4 * R;              // weight groups per workgroup
  constexpr int LL = 4 / R;              // lines one wave load covers (NG groups x LL lines x 4 pieces)
  constexpr int RT = R * M;              // row tiles, over the matrices
  constexpr int NL = 4 / CH;             // lines of each chain in a batch
  constexpr int PC = WC * CH * CPR;      // chains folded per round
  constexpr int NT = 64 * WC;
  constexpr int ITEMS = RT * L * 256;    // outputs of the workgroup
  constexpr int PER = (ITEMS + NT - 1) / NT;
  static_assert(kChains % PC == 0, "whole rounds");
  typedef typename FloatsOf<L>::T XV;
  __shared__ u32x4 aw[WC][M * R * 64];
  __shared__ float part[PC][ITEMS];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int w = exact_wg_order(blockIdx.x, gridDim.x);
  const int g0 = (w / nlb) * NG, lg0 = (w % nlb) * 4 * L;
  const int i = lane & 15, q = lane >> 4;

  // This lane's piece of a wave load: group pg, line slot pl, piece kp of the line.
  const int pg = lane / (4 * LL), pl = (lane >> 2) % LL, kp = lane & 3;
  const uint16_t* wp[M];
  int cols = 0;
#pragma unroll
  for (int m = 0; m < M; ++m) wp[m] = Op::w(p, m, min(g0 + pg, ngroups - 1), cols) + kp * 8;
  const int lines = cols / 8;
  const int stride = p.l.stride;
  uint32_t xo[2];  // this lane's byte offset from column 0 of a line: columns q and 4 + q
#pragma unroll
  for (int s = 0; s < 2; ++s)
    xo[s] = 4u * (static_cast<uint32_t>(4 * s + q) * stride + exact_tile_lane(lg0 * 4 + L * i, p.l.lane_groups, L));
  const int per_chain = (lines + kChains - 1) / kChains;  // lines of chain 0, the longest
  const int nb = (per_chain + NL - 1) / NL;               // batches

  // Slot n of a batch: line n / CH of the batch in chain t + n % CH. Slots past a
  // chain's last line are loaded from the matrix's last line and not summed.
  struct Batch {
    u32x4 a[M][R];
    XV x[4][2];
  };
  auto line_of = [&](int t, int b, int n) { return t + n % CH + kChains * (b * NL + n / CH); };
  auto load = [&](int t, int b, Batch& B) __attribute__((always_inline)) {
    unroll<R>([&](auto rr) {
      constexpr int r = decltype(rr)::value;
      const int64_t line = min(line_of(t, b, r * LL + pl), lines - 1);
      unroll<M>([&](auto mm) {
        constexpr int m = decltype(mm)::value;
        B.a[m][r] = load16(wp[m] + line * 32);
      });
    });
    unroll<4>([&](auto nn) {
      constexpr int n = decltype(nn)::value;
      const int64_t line = min(line_of(t, b, n), lines - 1);
      const char* base = reinterpret_cast<const char*>(p.x + line * 8 * stride);
      B.x[n][0] = *reinterpret_cast<const XV*>(base + xo[0]);
      B.x[n][1] = *reinterpret_cast<const XV*>(base + xo[1]);
    });
  };
  f32x4 acc[CH][RT][L];
  auto slot_step = [&](const Batch& B, auto nn) __attribute__((always_inline)) {
    constexpr int n = decltype(nn)::value;
    unroll<2>([&](auto ss) {
      constexpr int s = decltype(ss)::value;
      float av[RT];
#pragma unroll
      for (int m = 0; m < M; ++m) {
        const char* src = reinterpret_cast<const char*>(&aw[wave][m * R * 64 + (n * 4 + 2 * s + (q >> 1)) * NG]) + (q & 1) * 8;
        if constexpr (R == 1) {
          av[m] = lo_half(*reinterpret_cast<const uint16_t*>(src + (i >> 2) * 16 + (i & 3) * 2));
        } else if constexpr (R == 2) {
          const uint32_t v = *reinterpret_cast<const uint32_t*>(src + (i >> 1) * 16 + (i & 1) * 4);
          av[m * R] = lo_half(v);
          av[m * R + 1] = hi_half(v);
        } else {
          const u32x2 v = *reinterpret_cast<const u32x2*>(src + i * 16);
          av[m * R] = lo_half(v[0]);
          av[m * R + 1] = hi_half(v[0]);
          av[m * R + 2] = lo_half(v[1]);
          av[m * R + 3] = hi_half(v[1]);
        }
      }
      unroll<L>([&](auto bb) {
        constexpr int b = decltype(bb)::value;
        float xv;
        if constexpr (L == 1) xv = B.x[n][s];
        else xv = B.x[n][s][b];
        unroll<RT>([&](auto rr) {
          constexpr int r = decltype(rr)::value;
          acc[n % CH][r][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[r], xv, acc[n % CH][r][b], 0, 0, 0);
        });
      });
    });
  };
  // One batch: through the LDS slot (pieces at (line slot, piece, group), so that an
  // operand read touches consecutive words), then eight steps.
  auto sum = [&](const Batch& B, int t, int b) __attribute__((always_inline)) {
    unroll<M * R>([&](auto ee) {
      constexpr int m = decltype(ee)::value / R, r = decltype(ee)::value % R;
      aw[wave][m * R * 64 + ((r * LL + pl) * 4 + kp) * NG + pg] = B.a[m][r];
    });
    wave_phase();  // other lanes' pieces are read from here on
    if (line_of(t, b, 3) < lines) {
      unroll<4>([&](auto n) { slot_step(B, n); });
    } else {
      if (line_of(t, b, 0) < lines) slot_step(B, std::integral_constant<int, 0>{});
      if (line_of(t, b, 1) < lines) slot_step(B, std::integral_constant<int, 1>{});
      if (line_of(t, b, 2) < lines) slot_step(B, std::integral_constant<int, 2>{});
    }
    wave_phase();  // the next batch overwrites the slot
  };
  unroll<CH * RT * L>([&](auto ee) {
    constexpr int e = decltype(ee)::value;
    acc[e / (RT * L)][e / L % RT][e % L] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  });

  // Turn n of a wave: chains (n * WC + wave) * CH ..; a round is CPR turns of every
  // wave, whose partials are then added to the outputs, chains ascending.
  float y[PER];
  constexpr int kTurns = kChains / (WC * CH);
  auto first_chain = [&](int turn) { return (turn * WC + wave) * CH; };
  auto end_turn = [&](int turn) __attribute__((always_inline)) {
    const int in_round = turn % CPR;
    if (turn > 0 && in_round == 0) lds_barrier();  // the last round's partials have been read
    unroll<CH * RT * L>([&](auto ee) {
      constexpr int e = decltype(ee)::value, c = e / (RT * L);
      f32x4& a = acc[c][e / L % RT][e % L];
      reinterpret_cast<f32x4*>(part[(in_round * WC + wave) * CH + c])[e % (RT * L) * 64 + lane] = a;
      a = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    });
    if (in_round != CPR - 1) return;
    lds_barrier();
    unroll<PER>([&](auto uu) {
      constexpr int u = decltype(uu)::value;
      const int e = tid + NT * u;
      if (ITEMS % NT == 0 || e < ITEMS) {
        float v = turn < CPR ? part[0][e] : y[u] + part[0][e];
#pragma unroll
        for (int k = 1; k < PC; ++k) v = v + part[k][e];
        y[u] = v;
      }
    });
  };
  // The next batch's loads are in flight while one is summed.
  Batch B[2];
  load(first_chain(0), 0, B[0]);
  int turn = 0, b = 0;
  auto pass = [&](auto buf) __attribute__((always_inline)) {
    constexpr int k = decltype(buf)::value;
    const bool last = b == nb - 1;
    load(first_chain(min(turn + (last ? 1 : 0), kTurns - 1)), last ? 0 : b + 1, B[k ^ 1]);
    sum(B[k], first_chain(turn), b);
    ++b;
    if (last) {
      end_turn(turn);
      ++turn;
      b = 0;
    }
  };
  while (turn < kTurns) {
    pass(std::integral_constant<int, 0>{});
    if (turn < kTurns) pass(std::integral_constant<int, 1>{});
  }

  // Outputs back to (group, lane group) blocks of sixteen, then the operator's finish.
  lds_barrier();
  float* ys = &part[0][0];  // [NG * 4 * L][M][16]
  unroll<PER>([&](auto uu) {
    constexpr int u = decltype(uu)::value;
    const int e = tid + NT * u;
    if (ITEMS % NT == 0 || e < ITEMS) {
      const int tile = e >> 8, b_ = tile % L, rt = tile / L, m = rt / R, r = rt % R;
      const int ln = (e & 255) >> 2, row = 4 * (ln >> 4) + (e & 3), bl = L * (ln & 15) + b_;
      const int g = row * R / 4, rr = (row * R) % 4 + r;
      ys[((g * 4 * L + (bl >> 2)) * M + m) * 16 + rr * 4 + (bl & 3)] = y[u];
    }
  });
  lds_barrier();
  for (int k = tid >> 4; k < NG * 4 * L; k += NT / 16) {
    const int group = g0 + k / (4 * L), lg = lg0 + k % (4 * L);
    if (group < ngroups && lg < p.l.lane_groups)
      Op::template finish<4>(p, group, lg, tid & 15, reinterpret_cast<const float(*)[16]>(ys + k * M * 16));
  }
}

// Vector form, for up to eight rows of a large weight matrix: two lane groups leave half
// of a matrix tile's sixteen lanes dead, while here every fmaf is of a live lane (of a
// dead one for up to four rows). A workgroup of NWV waves runs NB = 2 * NWV reference
// blocks, i.e. NB consecutive weight groups with the (at most LG) lane groups, so the
// blocks share x. K is taken kSlice columns at a time: slice s holds line 32 * s + t of chain t,
// so each lane chains its lines in ascending order and every output's operations are
// those of chain() (and of the reference). The slice's x is staged once per workgroup in
// LDS (double buffered, the next slice's loads in flight while the current one is
// summed), laid out so that lane t's reads of a column are consecutive 16-byte words;
// each lane loads its own weight line one slice ahead. The matrices of a paired GEMM are
// swept one after the other, each one's partials folded as in k_exact_gemm.
// Bound by the vector pipe and, weights from memory, by their stream: 14336 x 8192, 8
// rows, 42-48 us (4.9-5.6 TB/s) against 51-55 as the best matrix tile of 18.
constexpr int kSlice = 256;  // 32 lines of 8 columns: one line of each chain

template <class Op, int LG, int NWV>
__global__ __launch_bounds__(64 * NWV) void k_exact_gemm_s(typename Op::Params p, int ngroups) {
  constexpr int M = Op::kMats;
  constexpr int NB = 2 * NWV;
  constexpr int NO = 16;                     // outputs per reference block (4 rows x 4 lanes)
  constexpr int XS = kSlice * LG;            // staged f32x4 per slice: one per column and lane group
  constexpr int NT = 64 * NWV;
  constexpr int XPER = (XS + NT - 1) / NT;   // staging loads per thread
  __shared__ f32x4 xs[2 * XS];
  __shared__ float part[NB][kChains][NO * LG];
  __shared__ float ys[NB][LG][M][16];
  const int tid = threadIdx.x, wave = tid >> 6, half = (tid >> 5) & 1, t = tid & 31;
  const int b = wave * 2 + half;
  const int group = exact_wg_order(blockIdx.x, gridDim.x) * NB + b;
  const bool live = group < ngroups;
  const int nlg = p.l.lane_groups;  // at most LG

  // Staging: item q of a slice is column c = q / LG, lane group q % LG (clamped
  // to the last live one); column 8 * l + e (line l, column e of the line) sits
  // at (e * 32 + l) * LG + i.
  f32x4 xr[XPER];
  auto load_x = [&](int sl) {
#pragma unroll
    for (int r = 0; r < XPER; ++r) {
      const int q = tid + r * NT;
      if (q < XS) {
        const int c = q / LG, i = min(q % LG, nlg - 1);
        xr[r] = *reinterpret_cast<const f32x4*>(p.x + static_cast<int64_t>(sl * kSlice + c) * p.l.stride + 4 * i);
      }
    }
  };
  auto store_x = [&](int buf) {
#pragma unroll
    for (int r = 0; r < XPER; ++r) {
      const int q = tid + r * NT;
      if (q < XS) {
        const int c = q / LG, i = q % LG, l = c >> 3, e = c & 7;
        xs[buf * XS + (e * 32 + l) * LG + i] = xr[r];
      }
    }
  };

  unroll<M>([&](auto mm) {
    constexpr int m = decltype(mm)::value;
    int cols = 0;
    const uint16_t* wg = Op::w(p, m, min(group, ngroups - 1), cols);
    const int nsl = cols / kSlice;
    u32x4 wl[2][4];  // this lane's weight line of the current and the next slice
    auto load_w = [&](int sl, auto buf) {
      const u32x4* src = reinterpret_cast<const u32x4*>(wg + static_cast<int64_t>(sl * kChains + t) * 32);
#pragma unroll
      for (int q = 0; q < 4; ++q) wl[decltype(buf)::value][q] = src[q];
    };
    float acc[NO * LG];
#pragma unroll
    for (int e = 0; e < NO * LG; ++e) acc[e] = 0.0f;
    auto step = [&](auto buf) {
      constexpr int c2 = decltype(buf)::value;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int c = 2 * q + h;  // column c of the line
          const float wv[4] = {lo_half(wl[c2][q][2 * h]), hi_half(wl[c2][q][2 * h]), lo_half(wl[c2][q][2 * h + 1]),
                               hi_half(wl[c2][q][2 * h + 1])};
#pragma unroll
          for (int i = 0; i < LG; ++i) {
            const f32x4 xc = xs[c2 * XS + (c * 32 + t) * LG + i];
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
              for (int j = 0; j < 4; ++j) acc[(i * 4 + r) * 4 + j] = __builtin_fmaf(wv[r], xc[j], acc[(i * 4 + r) * 4 + j]);
          }
        }
      }
    };
    load_x(0);
    load_w(0, std::integral_constant<int, 0>{});
    store_x(0);
    __syncthreads();
    // Slices in pairs so that the register and LDS buffers are compile-time.
    // The next slice's loads are issued unconditionally (the last slice's again
    // after it, into buffers nobody reads), so every pass waits on the same loads.
    int sl = 0;
    auto one = [&](auto cur) {
      constexpr int c = decltype(cur)::value;
      const int nx = min(sl + 1, nsl - 1);
      load_x(nx);
      load_w(nx, std::integral_constant<int, c ^ 1>{});
      step(cur);
      store_x(c ^ 1);
      __syncthreads();
      ++sl;
    };
    while (sl < nsl) {
      one(std::integral_constant<int, 0>{});
      if (sl < nsl) one(std::integral_constant<int, 1>{});
    }
    // Partials of this matrix, folded left to right per output.
#pragma unroll
    for (int e = 0; e < NO * LG; ++e) part[b][t][e] = acc[e];
    __syncthreads();
    for (int e = t; e < NO * LG; e += kChains) {
      float y = part[b][0][e];
      for (int i = 1; i < kChains; ++i) y = y + part[b][i][e];
      ys[b][e / NO][m][e % NO] = y;
    }
    __syncthreads();
  });
  if (live)
    for (int i = 0; i < nlg; ++i) Op::template finish<4>(p, group, i, t, ys[b][i]);
}

// ---------------------------------------------------------------------------
// Embedding, RMSNorm, compaction.

// h[k * stride + row] = widen(embed[token][k]); embed in [token/4][dim][4]
// groups (src/kernels.cu:98-117). A thread's kEmbedBatch elements are loaded
// before any is stored, so the row costs one memory round trip per batch, not
// one per element.
constexpr int kEmbedBatch = 8;
__global__ __launch_bounds__(256) void k_exact_embed(StrideEmbedParams p) {
  const int row = blockIdx.x;
  const int token = p.tokens[row];
  const uint16_t* src = p.embed + static_cast<int64_t>(token / 4) * p.dim * 4 + token % 4;
  for (int k0 = threadIdx.x; k0 < p.dim; k0 += 256 * kEmbedBatch) {
    uint16_t v[kEmbedBatch];
#pragma unroll
    for (int i = 0; i < kEmbedBatch; ++i) {
      const int k = min(k0 + 256 * i, p.dim - 1);
      v[i] = src[static_cast<int64_t>(k) * 4];
    }
#pragma unroll
    for (int i = 0; i < kEmbedBatch; ++i) {
      const int k = k0 + 256 * i;
      if (k < p.dim) p.h[static_cast<int64_t>(k) * p.l.stride + row] = f32_of(static_cast<uint32_t>(v[i]) << 16);
    }
  }
}

// RMSNorm over four-dim units (src/kernels.cu:119-200): chain t sums the squares
// of units u == t (mod 32) by fmaf, the 32 partials are added left to right,
// r = 1 / sqrtf(sum / dim + eps), out = w * (v * r). One reference block (lane
// group) per wavefront half.
template <int J>
__global__ __launch_bounds__(64) void k_exact_norm(StrideNormParams p) {
  __shared__ float part[2][kChains][J];
  __shared__ float rs[2][J];
  const int half = threadIdx.x >> 5, t = threadIdx.x & 31;
  const int block = blockIdx.x * 2 + half;
  const bool live = block < p.l.lane_groups;
  const int units = p.dim / 4, stride = p.l.stride;
  const float* in = J == 1 ? p.in : p.in + (live ? block : 0) * 4;
  float* out = J == 1 ? p.out : p.out + (live ? block : 0) * 4;
  // A lane's units u = t, t + 32, ... are loaded NB at a time before their
  // FMAs, so the chain waits one memory round trip per batch, not per unit.
  constexpr int NB = J == 1 ? 8 : 4;
  auto load_unit = [&](int u, f32x4 (&v)[4]) {
    const int k = u * 4;
    if constexpr (J == 1) {
      v[0] = *reinterpret_cast<const f32x4*>(in + k);
    } else {
#pragma unroll
      for (int c = 0; c < 4; ++c) v[c] = *reinterpret_cast<const f32x4*>(in + static_cast<int64_t>(k + c) * stride);
    }
  };
  if (live) {
    float acc[J];
#pragma unroll
    for (int j = 0; j < J; ++j) acc[j] = 0.0f;
    auto sum_unit = [&](const f32x4 (&v)[4]) {
      if constexpr (J == 1) {
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[0] = __builtin_fmaf(v[0][e], v[0][e], acc[0]);
      } else {
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
          for (int j = 0; j < 4; ++j) acc[j] = __builtin_fmaf(v[c][j], v[c][j], acc[j]);
      }
    };
    int u = t;
    for (; u + (NB - 1) * kChains < units; u += NB * kChains) {
      f32x4 v[NB][4];
#pragma unroll
      for (int b = 0; b < NB; ++b) load_unit(u + b * kChains, v[b]);
      __builtin_amdgcn_sched_barrier(0);  // every load of the batch before the first FMA
#pragma unroll
      for (int b = 0; b < NB; ++b) sum_unit(v[b]);
    }
    for (; u < units; u += kChains) {
      f32x4 v[4];
      load_unit(u, v);
      sum_unit(v);
    }
#pragma unroll
    for (int j = 0; j < J; ++j) part[half][t][j] = acc[j];
  }
  __syncthreads();
  if (live && t < J) {
    float sum = part[half][0][t];
    for (int i = 1; i < kChains; ++i) sum = sum + part[half][i][t];
    rs[half][t] = 1.0f / sqrtf(sum / static_cast<float>(p.dim) + p.eps);
  }
  __syncthreads();
  if (!live) return;
  auto scale_unit = [&](int u, const f32x4& w4, const f32x4 (&v)[4]) {
    const int k = u * 4;
    if constexpr (J == 1) {
      const float r = rs[half][0];
      f32x4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = w4[e] * (v[0][e] * r);
      *reinterpret_cast<f32x4*>(out + k) = o;
    } else {
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        f32x4 o;
#pragma unroll
        for (int j = 0; j < 4; ++j) o[j] = w4[c] * (v[c][j] * rs[half][j]);
        *reinterpret_cast<f32x4*>(out + static_cast<int64_t>(k + c) * stride) = o;
      }
    }
  };
  int u = t;
  for (; u + (NB - 1) * kChains < units; u += NB * kChains) {
    f32x4 v[NB][4], w4[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      w4[b] = *reinterpret_cast<const f32x4*>(p.weight + (u + b * kChains) * 4);
      load_unit(u + b * kChains, v[b]);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int b = 0; b < NB; ++b) scale_unit(u + b * kChains, w4[b], v[b]);
  }
  for (; u < units; u += kChains) {
    f32x4 v[4];
    load_unit(u, v);
    scale_unit(u, *reinterpret_cast<const f32x4*>(p.weight + u * 4), v);
  }
}

// The same RMSNorm with one 256-thread workgroup per lane group: every thread
// loads its share of the lane group's inputs (and the gains it will scale them
// with) in one memory round trip, the inputs into LDS; the 32 chains then run
// over LDS in the order above, and all 256 threads scale and store. Serves rows
// of up to kNormLdsItems 16-byte items (dim four-lane columns for J = 4, dim / 4
// units for J = 1): 64 KiB of LDS.
constexpr int kNormPer = 16;
constexpr int kNormLdsItems = 256 * kNormPer;
template <int J>
__global__ __launch_bounds__(256) void k_exact_norm_lds(StrideNormParams p) {
  extern __shared__ f32x4 vsm[];  // item i: unit i (J = 1) or column i's four lanes (J = 4)
  __shared__ float part[kChains][J];
  __shared__ float rs[J];
  const int tid = threadIdx.x, block = blockIdx.x;
  const int units = p.dim / 4, stride = p.l.stride;
  const int items = J == 1 ? units : p.dim;
  const float* in = J == 1 ? p.in : p.in + block * 4;
  float* out = J == 1 ? p.out : p.out + block * 4;
  f32x4 v[kNormPer], w4[J == 1 ? kNormPer : 1];
  float wk[J == 1 ? 1 : kNormPer];
#pragma unroll
  for (int r = 0; r < kNormPer; ++r) {
    const int i = tid + 256 * r;
    if (i < items) {
      if constexpr (J == 1) {
        v[r] = *reinterpret_cast<const f32x4*>(in + 4 * i);
        w4[r] = *reinterpret_cast<const f32x4*>(p.weight + 4 * i);
      } else {
        v[r] = *reinterpret_cast<const f32x4*>(in + static_cast<int64_t>(i) * stride);
        wk[r] = p.weight[i];
      }
    }
  }
#pragma unroll
  for (int r = 0; r < kNormPer; ++r)
    if (tid + 256 * r < items) vsm[tid + 256 * r] = v[r];
  __syncthreads();
  // A thread per chain and lane (four lanes in one thread: 6.6 us against 5.9 at 32 rows
  // of 2048), its LDS reads issued several units ahead.
  if (tid < kChains * J) {
    const int t = tid / J, j = tid % J;
    const float* x = reinterpret_cast<const float*>(vsm) + j;
    float acc = 0.0f;
#pragma unroll 4
    for (int u = t; u < units; u += kChains) {
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const float e = x[(u * 4 + c) * J];
        acc = __builtin_fmaf(e, e, acc);
      }
    }
    part[t][j] = acc;
  }
  __syncthreads();
  if (tid < J) {
    float sum = part[0][tid];
    for (int i = 1; i < kChains; ++i) sum = sum + part[i][tid];
    rs[tid] = 1.0f / sqrtf(sum / static_cast<float>(p.dim) + p.eps);
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kNormPer; ++r) {
    const int i = tid + 256 * r;
    if (i >= items) continue;
    f32x4 o;
    if constexpr (J == 1) {
      const float q = rs[0];
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = w4[r][e] * (v[r][e] * q);
      *reinterpret_cast<f32x4*>(out + 4 * i) = o;
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) o[j] = wk[r] * (v[r][j] * rs[j]);
      *reinterpret_cast<f32x4*>(out + static_cast<int64_t>(i) * stride) = o;
    }
  }
}

// out[k * lm_stride + l] = in[k * stride + lm_rows[l]] (src/kernels.cu:365-380).
__global__ __launch_bounds__(64) void k_exact_compact(StrideCompactParams p) {
  const int k = blockIdx.x * 64 + threadIdx.x;
  if (k >= p.dim) return;
  for (int l = 0; l < p.lm_count; ++l)
    p.out[static_cast<int64_t>(k) * p.lm_stride + l] = p.in[static_cast<int64_t>(k) * p.l.stride + p.lm_rows[l]];
}

// ---------------------------------------------------------------------------
// Host side.

std::string lanes_why(const StrideLanes& l, int J) {
  if (J != 1 && J != 4) return "J must be 1 or 4";
  if (l.rows < 0) return "rows must be >= 0";
  if (J == 1 && (l.rows > 1 || l.lane_groups != 1 || l.stride != 1)) return "J = 1 serves one row with lane_groups 1 and stride 1";
  if (J == 4 && (l.lane_groups != (l.rows + 3) / 4 || l.stride < 4 * l.lane_groups || l.stride % 4 != 0))
    return "J = 4 needs lane_groups = ceil(rows / 4) and a stride that is a multiple of 4 covering them";
  return "";
}

std::string mat_why(const StrideGemmMat& m, const char* name) {
  if (!m.w || m.groups <= 0 || m.cols <= 0 || m.cols % 8 != 0)
    return std::string(name) + ": need a weight pointer, groups > 0 and cols a positive multiple of 8";
  return "";
}

int launched(const char* what) {
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(static_cast<int>(e), std::string(what) + " launch failed: " + hipGetErrorString(e));
  return 0;
}

template <class Op, int R, int L, int WC, int CH, int CPR>
int run_matrix(const typename Op::Params& p, hipStream_t st, const char* what) {
  const int nlb = (p.l.lane_groups + 4 * L - 1) / (4 * L);
  const int nrb = (Op::groups(p) + 4 * R - 1) / (4 * R);
  hipLaunchKernelGGL((k_exact_gemm_m<Op, R, L, WC, CH, CPR>), dim3(nrb * nlb), dim3(64 * WC), 0, st, p, nlb, Op::groups(p));
  return launched(what);
}

template <class Op>
int run_gemm(const typename Op::Params& p, int J, void* stream, const char* what) {
  const int groups = Op::groups(p);
  if (p.l.rows == 0 || groups == 0) return 0;
  hipStream_t st = static_cast<hipStream_t>(stream);
  // One lane: the loads are weight-bound, and the streaming form keeps more of them
  // in flight than a matrix tile with one live lane in sixteen would.
  if (J == 1) {
    hipLaunchKernelGGL((k_exact_gemm<Op>), dim3((groups + 1) / 2), dim3(64), 0, st, p, groups);
    return launched(what);
  }
  // Tile and waves by the number of 16 x 16 output tiles, from a sweep of 18 tile and
  // wave shapes at 2-256 rows, N = 2048, 3072, 2 x 8192 and 128256, K = 2048 and 8192:
  // the workgroups have to fill the 256 CUs, so few tiles get a workgroup of 16 waves
  // each, many get larger tiles (fewer operand loads and vector instructions per MFMA)
  // and smaller workgroups (more of them resident, so that one folds while another
  // multiplies). The other side of each line, measured: 256 tiles 7.2 us at 16 waves
  // per tile against 9.3 at two tiles per workgroup (N = K = 2048, 32 rows); 384 tiles
  // 13.4 against 9.8 (N = 3072, 32 rows); 768 tiles 18.3 at 1 x 2 against 15.5 at 2 x 2;
  // 1536 tiles 28.7 at 2 x 2 x 16 waves against 21.3 (128 rows); 2048 tiles 27.2 at
  // 1 x 2 against 25.1 at 2 x 4, whose four lane tiles have to be live (K = 8192: 91
  // against 79); 3072 tiles 48 at 2 x 4 against 38 (256 rows).
  const int rt = (groups + 3) / 4, lt = (p.l.lane_groups + 3) / 4, cols = Op::cols(p);
  const int64_t tiles = static_cast<int64_t>(rt) * lt;
  auto dealt = [&](int step) { return (rt + step - 1) / step * step; };
  // Up to eight rows, columns in whole slices: the vector form where it is the faster one.
  // That is where columns are many (it folds 32 partials of every output and starts fewer
  // waves), but for row counts that leave its workgroups, 32 rows each and two or three
  // to a CU, poorly dealt. Measured at 8 rows, 24 sizes up to N = 128256 and K = 8192, each
  // with its weights in the last-level cache and from memory (the latter second); vector
  // against the best matrix tile, in us: N = 8192, K = 4096 20.3-22.4 / 18.6-19.5;
  // 11008 x 3072 20.0-22.2 / 20.2-21.1, x 8192 42.6-45.8 / 47.5-48.3; 14336 x 1024 9.3-12.0
  // / 10.4-11.3, x 8192 43.4-48.4 / 52.7-54.5; 28672 x 2048 29.4-34.3 / 29.2-30.6;
  // 36864 x 3072 42-55 / 49-53; 50304 x 1024 28-32 / 30-31, x 2048 44-50 / 49-51; pairs
  // 2 x 14336 x 1024 18.3-18.5 / 18.4-18.8, x 8192 91-90 / 100-101, 2 x 11008 x 8192
  // 91-90 / 81-82, 2 x 28672 x 4096 110-109 / 95-101. (An odd number of lines a chain leaves
  // part of a matrix batch empty: 100000 x 1280 51 / 64. Vocabularies whose 4 x 1 tiles deal
  // evenly: 128256 x 3072 158 / 155, x 4096 190 / 204; 151936 x 3072 187 / 193.)
  if (p.l.lane_groups <= 2 && cols % kSlice == 0) {
    const bool vector = Op::kMats == 2 ? rt >= 832 && rt < 1600 && cols >= 1024
                                       : (rt > 512 && rt < 832 && cols >= 4096) ||
                                             (rt >= 832 && rt <= 1536 && cols >= 1024) ||
                                             (rt >= 2200 && cols >= (cols % (2 * kSlice) == 0 ? 2048 : 768) &&
                                              !(rt >= 6144 && cols < 4096 && 100 * dealt(1024) <= 103 * rt));
    if (vector) {
      constexpr int LG = 2, NWV = 4;
      hipLaunchKernelGGL((k_exact_gemm_s<Op, LG, NWV>), dim3((groups + 2 * NWV - 1) / (2 * NWV)), dim3(64 * NWV), 0, st, p, groups);
      return launched(what);
    }
  }
  // Few columns leave a wave few lines of each chain: it takes four chains at a time, and
  // workgroups are half as large (N = 2048, 8 rows: K = 64 3.2 us against 3.8 with sixteen
  // waves, K = 1024 5.0 / 5.1, K = 2048 7.2 / 7.0).
  if (tiles <= 256)
    return cols < 2048 ? run_matrix<Op, 1, 1, 8, 4, 1>(p, st, what) : run_matrix<Op, 1, 1, 16, 2, 1>(p, st, what);
  // At most a line for every chain: a wave's four chains are one batch, and small workgroups
  // that fold at once (8192 x 256, 33 rows 7.5 us against 13.5 as below and 12.1 for the
  // vector form; 3072 x 64 4.7 / 6.8 / 5.3; pairs of 32000 x 128 34 / 62 / 56; of 216 sizes
  // of more than one lane tile none is slower).
  if (lt > 1 && cols <= 8 * kChains) return run_matrix<Op, 1, 1, 4, 4, 1>(p, st, what);
  if constexpr (Op::kMats == 2) {
    if (lt == 1)  // 2 x 8192 rows, K = 512: 7.1 us against 7.4; K = 2048 18.6 / 18.3; 2 x 14336, K = 64 7.5 / 8.9
      return cols < 2048 ? run_matrix<Op, 1, 1, 8, 4, 1>(p, st, what) : run_matrix<Op, 1, 1, 8, 2, 1>(p, st, what);
    if (tiles <= 512) return run_matrix<Op, 1, 2, 16, 1, 1>(p, st, what);
    return run_matrix<Op, 1, 2, 8, 1, 2>(p, st, what);
  } else {
    if (lt == 1) {
      // One lane tile: the largest row tile that deals the rows about evenly to the CUs (1,
      // 2 or 4 x 256 row tiles at a time; the sweep above). 4 x 1 reads a vocabulary's
      // weights fastest (128256 x 2048: 110-112 us against 116 at 2 x 1 and 126 at 1 x 1;
      // 32000 x 2048 31-32 / 31-35 / 33-36, but 28672 x 1024 18.9-19.3 / 18.3-19.3 /
      // 17.7-18.7). 2 x 1: N = 8192, K = 1024 6.8-7.8 against 7.3-8.4 at 1 x 1, but
      // 11008 x 1024 10.3-10.9 / 9.1-9.6. Less than a line for every chain: small
      // workgroups (32000 x 64: 7.7 us against 8.8).
      if (cols < 8 * kChains && rt > 512) return run_matrix<Op, 1, 1, 4, 4, 1>(p, st, what);
      if (rt >= 1900 && 20 * dealt(1024) <= 23 * rt) return run_matrix<Op, 4, 1, 4, 2, 1>(p, st, what);
      if (rt <= 512 || dealt(512) == dealt(256)) return run_matrix<Op, 2, 1, 8, 4, 1>(p, st, what);
      return run_matrix<Op, 1, 1, 8, 4, 1>(p, st, what);
    }
    if (tiles <= 512) return run_matrix<Op, 1, 2, 16, 2, 1>(p, st, what);
    if (tiles <= 1024)  // 3072 x 512: 33 rows 6.5 us against 8.0, 64 rows 6.7 / 8.0
      return cols <= 512 ? run_matrix<Op, 1, 1, 8, 4, 1>(p, st, what) : run_matrix<Op, 2, 2, 16, 1, 1>(p, st, what);
    if (tiles <= 1536 || (tiles <= 2048 && lt % 4 != 0)) return run_matrix<Op, 1, 2, 8, 1, 2>(p, st, what);
    if (tiles <= 2048) return run_matrix<Op, 2, 4, 8, 1, 1>(p, st, what);
    return run_matrix<Op, 2, 2, 4, 2, 1>(p, st, what);
  }
}

}  // namespace
}  // namespace stride_tc

using namespace stride_tc;

static_assert(sizeof(StrideEmbedParams) == 48, "EmbedParams layout");
static_assert(sizeof(StrideNormParams) == 48, "NormParams layout");
static_assert(offsetof(StrideQkvParams, kv) == 88 && offsetof(StrideQkvParams, rope) == 144 &&
                  sizeof(StrideQkvParams) == 176, "QkvParams layout");
static_assert(sizeof(StrideGemmResidualParams) == 48, "GemmResidualParams layout");
static_assert(sizeof(StrideMlp13Params) == 64, "Mlp13Params layout");
static_assert(sizeof(StrideCompactParams) == 56, "CompactParams layout");
static_assert(offsetof(StrideLmGreedyParams, best) == 48 && sizeof(StrideLmGreedyParams) == 56, "LmGreedyParams layout");
static_assert(sizeof(StrideLmFullParams) == 48, "LmFullParams layout");

extern "C" {

int stride_k_embed(const StrideEmbedParams* p, void* stream) {
  if (!p) return fail(STRIDE_TC_EINVAL, "k_embed: null parameters");
  if (p->l.rows < 0 || p->dim <= 0 || (p->l.rows > 0 && (!p->embed || !p->tokens || !p->h)) ||
      p->l.stride < p->l.rows)
    return fail(STRIDE_TC_EINVAL, "k_embed: need rows >= 0, dim > 0, stride >= rows and pointers");
  if (p->l.rows == 0) return 0;
  hipLaunchKernelGGL(k_exact_embed, dim3(p->l.rows), dim3(256), 0, static_cast<hipStream_t>(stream), *p);
  return launched("k_embed");
}

int stride_k_norm(const StrideNormParams* p, int32_t J, void* stream) {
  if (!p) return fail(STRIDE_TC_EINVAL, "k_norm: null parameters");
  std::string why = lanes_why(p->l, J);
  if (why.empty() && (p->dim <= 0 || p->dim % 4 != 0)) why = "dim must be a positive multiple of 4";
  if (why.empty() && p->l.rows > 0 && (!p->in || !p->out || !p->weight)) why = "missing pointer";
  if (!why.empty()) return fail(STRIDE_TC_EINVAL, "k_norm: " + why);
  if (p->l.rows == 0) return 0;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int items = J == 1 ? p->dim / 4 : p->dim;
  if (items <= kNormLdsItems) {
    const size_t lds = static_cast<size_t>(items) * 16;
    if (J == 1) hipLaunchKernelGGL(k_exact_norm_lds<1>, dim3(p->l.lane_groups), dim3(256), lds, st, *p);
    else hipLaunchKernelGGL(k_exact_norm_lds<4>, dim3(p->l.lane_groups), dim3(256), lds, st, *p);
    return launched("k_norm");
  }
  const dim3 grid((p->l.lane_groups + 1) / 2);
  if (J == 1) hipLaunchKernelGGL(k_exact_norm<1>, grid, dim3(64), 0, st, *p);
  else hipLaunchKernelGGL(k_exact_norm<4>, grid, dim3(64), 0, st, *p);
  return launched("k_norm");
}

int stride_k_qkv(const StrideQkvParams* p, int32_t J, void* stream) {
  if (!p) return fail(STRIDE_TC_EINVAL, "k_qkv: null parameters");
  std::string why = lanes_why(p->l, J);
  const int D = p->head_dim;
  if (why.empty()) why = mat_why(p->q, "q");
  if (why.empty()) why = mat_why(p->k, "k");
  if (why.empty()) why = mat_why(p->v, "v");
  if (why.empty() && (D <= 0 || D % 4 != 0 || p->kv.head_dim != D)) why = "head_dim must be a positive multiple of 4 matching kv.head_dim";
  if (why.empty() && (p->k.groups != p->v.groups || p->q.cols != p->k.cols || p->k.cols != p->v.cols))
    why = "k and v must have the same groups and all three the same cols";
  if (why.empty()) {
    const int64_t tokens = D > 0 ? p->kv.group_elems / D : 0;
    if (tokens <= 0 || (tokens & (tokens - 1)) != 0) why = "the KV block (group_elems / head_dim) must be a power of two";
  }
  if (why.empty() && p->l.rows > 0 && (!p->x || !p->q_out || !p->rope || !p->row_slot || !p->row_pos || !p->kv.arena || !p->kv.table))
    why = "missing pointer";
  if (!why.empty()) return fail(STRIDE_TC_EINVAL, "k_qkv: " + why);
  return run_gemm<QkvOp>(*p, J, stream, "k_qkv");
}

int stride_k_gemm_residual(const StrideGemmResidualParams* p, int32_t J, void* stream) {
  if (!p) return fail(STRIDE_TC_EINVAL, "k_gemm_residual: null parameters");
  std::string why = lanes_why(p->l, J);
  if (why.empty()) why = mat_why(p->m, "m");
  if (why.empty() && p->l.rows > 0 && (!p->x || !p->h)) why = "missing pointer";
  if (!why.empty()) return fail(STRIDE_TC_EINVAL, "k_gemm_residual: " + why);
  return run_gemm<ResidualOp>(*p, J, stream, "k_gemm_residual");
}

int stride_k_mlp13(const StrideMlp13Params* p, int32_t J, void* stream) {
  if (!p) return fail(STRIDE_TC_EINVAL, "k_mlp13: null parameters");
  std::string why = lanes_why(p->l, J);
  if (why.empty()) why = mat_why(p->w1, "w1");
  if (why.empty()) why = mat_why(p->w3, "w3");
  if (why.empty() && (p->w1.groups != p->w3.groups || p->w1.cols != p->w3.cols)) why = "w1 and w3 must have the same shape";
  if (why.empty() && p->l.rows > 0 && (!p->x || !p->z)) why = "missing pointer";
  if (!why.empty()) return fail(STRIDE_TC_EINVAL, "k_mlp13: " + why);
  return run_gemm<Mlp13Op>(*p, J, stream, "k_mlp13");
}

int stride_k_compact(const StrideCompactParams* p, void* stream) {
  if (!p || p->lm_count < 0 || p->dim <= 0 || (p->lm_count > 0 && (!p->in || !p->out || !p->lm_rows)) ||
      p->lm_stride < p->lm_count)
    return fail(STRIDE_TC_EINVAL, "k_compact: need lm_count >= 0, dim > 0, lm_stride >= lm_count and pointers");
  if (p->lm_count == 0) return 0;
  hipLaunchKernelGGL(k_exact_compact, dim3((p->dim + 63) / 64), dim3(64), 0, static_cast<hipStream_t>(stream), *p);
  return launched("k_compact");
}

int stride_k_lm_greedy(const StrideLmGreedyParams* p, int32_t J, void* stream) {
  if (!p) return fail(STRIDE_TC_EINVAL, "k_lm_greedy: null parameters");
  std::string why = lanes_why(p->l, J);
  if (why.empty()) why = mat_why(p->m, "m");
  if (why.empty() && (p->vocab <= 0 || p->vocab > p->m.groups * 4)) why = "vocab must be in (0, 4 * groups]";
  if (why.empty() && p->l.rows > 0 && (!p->x || !p->best)) why = "missing pointer";
  if (!why.empty()) return fail(STRIDE_TC_EINVAL, "k_lm_greedy: " + why);
  return run_gemm<LmGreedyOp>(*p, J, stream, "k_lm_greedy");
}

int stride_k_lm_full(const StrideLmFullParams* p, int32_t J, void* stream) {
  if (!p) return fail(STRIDE_TC_EINVAL, "k_lm_full: null parameters");
  std::string why = lanes_why(p->l, J);
  if (why.empty()) why = mat_why(p->m, "m");
  if (why.empty() && p->l.rows > 0 && (!p->x || !p->logits)) why = "missing pointer";
  if (!why.empty()) return fail(STRIDE_TC_EINVAL, "k_lm_full: " + why);
  return run_gemm<LmFullOp>(*p, J, stream, "k_lm_full");
}

}  // extern "C"
