// Mixture of experts of the layered decoder: a token's `top` experts are those with the largest router logits, weighted by the
// softmax over these logits; an expert is down(g sigmoid(1.702 g) (u + 1)) with g = min(gate(h), limit), u = clamp(up(h)).
//
// Prefill: [choose] a wavefront per token; [plan] the (token, slot) pairs sorted by expert, and the tiles of the grouped
// products; [gate, up + activation] rows gathered, a wavefront's two column blocks are gate and up of the same 32
// columns; [down] weighted rows to [slot][token], which the norm that follows adds to the residual stream. Nothing depends on the
// order in which workgroups run.
// Decode: [norm + choice + gate, up + activation] [down of all chosen experts as one product over their joined columns].
#include <algorithm>
#include <cmath>

#include "w4a32_layered.h"
#include "w4a32_layered_kernels.h"
#include "w4a32_mfma_tile.h"
#include "w4a32_row_prologue.h"

namespace w4 {

namespace {

constexpr float kGluAlpha = 1.702f;
constexpr int kMaxParts = kMoeLogitParts;
constexpr int kLogitRegs = W4A32_LAYERED_MAX_EXPERTS / 64;
static_assert(W4A32_LAYERED_MAX_TOP <= 64, "a lane per chosen expert");

// T: what the result is rounded to. For bf16 the sigmoid comes from the hardware's exponential and reciprocal (1 ulp of f32 each) with
// the product in the exponent carried on in two parts and one Newton step: in the epilogue of a grouped product expf and the
// divide took as long as a fifth of its products. Largest relative error over g in [-51, -10], [-10, -1], [-1, 20]: 1.9e-7, 2.1e-7,
// 1.5e-7; with expf and a divide, whose argument is rounded, 3.9e-6, 1.1e-6, 1.7e-7. Below -51 a sigmoid under 2^-126 is 0.
template <typename T>
__device__ __forceinline__ float clamped_glu(float g, float u, float limit) {
  g = fminf(g, limit);
  u = fminf(fmaxf(u, -limit), limit);
  if constexpr (sizeof(T) == 2) {
    constexpr double kExp = -(double)kGluAlpha * 1.4426950408889634;  // of 2
    constexpr float kHi = (float)kExp, kLo = (float)(kExp - (double)kHi);
    const float t = g * kHi, rest = __fmaf_rn(g, kLo, __fmaf_rn(g, kHi, -t));
    float e = __builtin_amdgcn_exp2f(t);
    e = __fmaf_rn(e, rest * 0.69314718f, e);
    const float d = 1.0f + e, y = __builtin_amdgcn_rcpf(d);
    const float sigmoid = fmaxf(__fmaf_rn(__fmaf_rn(-d, y, 1.0f), y, y), 0.0f);  // d infinite: 0, not the step's NaN
    return g * sigmoid * (u + 1.0f);
  }
  return g * sigmoid_f(kGluAlpha * g) * (u + 1.0f);
}

// The `top` largest of a wavefront's values (value i of lane l belongs to expert 64 i + l; equal ones: the lower expert
// first). Lane t < top returns the t-th expert and its softmax weight.
__device__ __forceinline__ void top_experts(float (&v)[kLogitRegs], int experts, int top, int* expert, float* weight) {
  const int lane = threadIdx.x & 63;
  int pick = 0;
  float mine = 0.0f, first = 0.0f, sum = 0.0f;
  // A value per lane, all of them comparable: each lane counts what comes in front of it, four operations per expert and a few
  // per choice. The rounds below are six exchanges between lanes each, whatever the number of experts. Us of a launch that
  // chooses, counting / rounds, 100 tokens: 4 of 16 experts 2.8 / 4.8, 8 of 64 4.9 / 7.7, 4 of 64 4.6 / 4.7, 2 of 32 3.2 / 3.3; but 1 of 16
  // 2.6 / 2.6, 1 of 64 4.4 / 2.5, 2 of 48 3.8 / 3.3 (one token: 4.0 / 2.2 and 3.5 / 2.9): a round is worth 18 experts.
  if (experts <= min(64, 18 * top - 4) && __popcll(__ballot(v[0] > -INFINITY)) == experts) {
    int rank = 0;
    for (int j = 0; j < experts; ++j) {
      const float x = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v[0]), j));
      rank += x > v[0] || (x == v[0] && j < lane) ? 1 : 0;
    }
    for (int t = 0; t < top; ++t) {
      const int at = __ffsll((unsigned long long)__ballot(rank == t && lane < experts)) - 1;
      const float best = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v[0]), at));
      if (t == 0) first = best;
      const float w = expf(best - first);
      sum += w;
      if (lane == t) {
        pick = at;
        mine = w;
      }
    }
    *expert = pick;
    *weight = mine / sum;
    return;
  }
  for (int t = 0; t < top; ++t) {
    float best = -INFINITY;
    int at = 0x7fffffff;
#pragma unroll
    for (int i = 0; i < kLogitRegs; ++i)
      if (64 * i < experts && v[i] > best) {
        best = v[i];
        at = 64 * i + lane;
      }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
      const float ov = __shfl_xor(best, off, 64);
      const int oa = __shfl_xor(at, off, 64);
      if (ov > best || (ov == best && oa < at)) {
        best = ov;
        at = oa;
      }
    }
    at = min(at, experts - 1);  // (values that do not compare choose the last expert)
#pragma unroll
    for (int i = 0; i < kLogitRegs; ++i)
      if (64 * i + lane == at) v[i] = -INFINITY;
    if (t == 0) first = best;
    const float w = expf(best - first);
    sum += w;
    if (lane == t) {
      pick = at;
      mine = w;
    }
  }
  *expert = pick;
  *weight = mine / sum;
}

// ---------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void moe_choose_kernel(const float* __restrict__ logits, int parts, size_t part_stride,
                                                         int ldl, int M, int experts, int top, int* __restrict__ ids,
                                                         float* __restrict__ wts) {
  const int m = 4 * (int)blockIdx.x + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (m >= M) return;
  float v[kLogitRegs];
#pragma unroll
  for (int i = 0; i < kLogitRegs; ++i) {
    const int e = 64 * i + lane;
    v[i] = -INFINITY;
    if (e < experts) {
      const float* src = logits + (size_t)m * ldl + e;
      float x[kMaxParts], s = 0.0f;
#pragma unroll
      for (int p = 0; p < kMaxParts; ++p) x[p] = src[min(p, parts - 1) * part_stride];  // all requested before the first is used
#pragma unroll
      for (int p = 0; p < kMaxParts; ++p) s += p < parts ? x[p] : 0.0f;
      v[i] = s;
    }
  }
  int e;
  float w;
  top_experts(v, experts, top, &e, &w);
  if (lane < top) {
    ids[(size_t)m * top + lane] = e;
    wts[(size_t)m * top + lane] = w;
  }
}

// A tile of an expert: those of one height all say the same, so that a workgroup needs one of them only, whichever it takes.
struct MoeTile {
  int expert, row0, rows;  // the expert's rows of the sorted list that go in tiles of this height
  int first, tiles;        // the first of these tiles and how many there are
  int pad[3];
};

constexpr int kPlanThreads = 1024, kPlanWaves = kPlanThreads / 64;

// Sum over the workgroup of one int per thread, and of those of lower threads.
__device__ __forceinline__ int block_scan(int x, int* s_w, int* total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int inc = x;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int y = __shfl_up(inc, off, 64);
    if (lane >= off) inc += y;
  }
  __syncthreads();  // s_w of an earlier call
  if (lane == 63) s_w[wave] = inc;
  __syncthreads();
  int before = 0, all = 0;
#pragma unroll
  for (int w = 0; w < kPlanWaves; ++w) {
    before += w < wave ? s_w[w] : 0;
    all += s_w[w];
  }
  *total = all;
  return before + inc - x;
}

// Tiles of bm = 2^log_bm rows, of which an expert's last one has `rest` rows where its rows fit that (0: never).
struct MoeHeights {
  int log_bm, rest;
  // tiles of bm rows that `count` rows go in
  __host__ __device__ int whole(int count) const {
    const int n = count >> log_bm;
    return n + (count - (n << log_bm) > rest ? 1 : 0);
  }
};

// A workgroup per expert: where its run of the sorted list starts (all of them count everything), its pairs in ascending order,
// its tiles in the two products' lists. In a list the tiles of bm rows stand first (n_tiles[0] of them), then those of `rest` rows
// (n_tiles[1]).
__global__ __launch_bounds__(kPlanThreads) void moe_plan_kernel(const int* __restrict__ ids, int n, int experts,
                                                                const MoeHeights up, const MoeHeights down,
                                                                int* __restrict__ order, MoeTile* __restrict__ up_tiles,
                                                                MoeTile* __restrict__ down_tiles, int* __restrict__ n_tiles) {
  __shared__ int s_count[W4A32_LAYERED_MAX_EXPERTS];
  __shared__ int s_w[kPlanWaves], s_sums[2][5];
  const int e = blockIdx.x, tid = threadIdx.x;
  for (int i = tid; i < experts; i += kPlanThreads) s_count[i] = 0;
  __syncthreads();
  // a thread takes a run of pairs, up to eight of them in registers
  constexpr int kRegs = 8;
  const int per = (n + kPlanThreads - 1) / kPlanThreads, lo = min(n, tid * per), hi = min(n, lo + per);
  int mine = 0, id[kRegs];
#pragma unroll
  for (int i = 0; i < kRegs; ++i) id[i] = ids[min(lo + i, n - 1)];
#pragma unroll
  for (int i = 0; i < kRegs; ++i)
    if (lo + i < hi) {
      atomicAdd(&s_count[id[i]], 1);
      mine += id[i] == e;
    }
  for (int i = lo + kRegs; i < hi; ++i) {
    atomicAdd(&s_count[ids[i]], 1);
    mine += ids[i] == e;
  }
  __syncthreads();
  // what comes in front of this expert, and in all: a wavefront adds up each list's tiles
  if (tid < 128) {
    const MoeHeights g = tid < 64 ? up : down;
    int sums[5] = {0, 0, 0, 0, 0};  // rows; whole tiles, rests; the same of all experts
    for (int i = tid & 63; i < experts; i += 64) {
      const int c = s_count[i], whole = g.whole(c), rest = c > whole << g.log_bm ? 1 : 0;
      sums[0] += i < e ? c : 0;
      sums[1] += i < e ? whole : 0;
      sums[2] += i < e ? rest : 0;
      sums[3] += whole;
      sums[4] += rest;
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1)
#pragma unroll
      for (int i = 0; i < 5; ++i) sums[i] += __shfl_xor(sums[i], off, 64);
    if ((tid & 63) == 0)
#pragma unroll
      for (int i = 0; i < 5; ++i) s_sums[tid >> 6][i] = sums[i];
  }
  int count;
  const int before_mine = block_scan(mine, s_w, &count), offset = s_sums[0][0];
  int at = offset + before_mine;
#pragma unroll
  for (int i = 0; i < kRegs; ++i)
    if (lo + i < hi && id[i] == e) order[at++] = lo + i;
  for (int i = lo + kRegs; i < hi; ++i)
    if (ids[i] == e) order[at++] = i;
  if (tid < 128) {  // a wavefront per list
    const int list = tid >> 6, lane = tid & 63;
    const MoeHeights g = list ? down : up;
    MoeTile* tiles = list ? down_tiles : up_tiles;
    const int whole = g.whole(count), in_whole = min(count, whole << g.log_bm), first = s_sums[list][1];
    for (int t = lane; t < whole; t += 64) tiles[first + t] = MoeTile{e, offset, in_whole, first, whole, {0, 0, 0}};
    if (lane == 0 && count > in_whole) {
      const int t = s_sums[list][3] + s_sums[list][2];
      tiles[t] = MoeTile{e, offset + in_whole, count - in_whole, t, 1, {0, 0, 0}};
    }
    if (e == 0 && lane < 2) n_tiles[2 * list + lane] = s_sums[list][3 + lane];
  }
}

// The tile of a workgroup: first those of bm rows, then (kRest) those of fewer, which the CUs take that come free early. An expert's
// tiles are numbered rows fastest, experts one after the other; consecutive numbers on one XCD. `row0` and `rows` become the tile's.
// Returns false past the last one.
template <bool kRest>
__device__ __forceinline__ bool moe_tile(const MoeTile* __restrict__ tiles, const int* __restrict__ n_tiles, int bm, int nt,
                                         MoeTile* tile, int* n, bool* rest) {
  const int whole = n_tiles[0], all = whole + (kRest ? n_tiles[1] : 0);
  int b = blockIdx.x;
  if (b >= all * nt) return false;
  *rest = kRest && b >= whole * nt;
  if (*rest) b -= whole * nt;
  const int t = xcd_tile(b, (*rest ? all - whole : whole) * nt) + (*rest ? whole * nt : 0);
  *tile = tiles[t / nt];
  if (tile->tiles <= 0) return false;
  const int local = t - tile->first * nt, at = local % tile->tiles * bm;
  *n = local / tile->tiles;
  tile->row0 += at;
  tile->rows = min(bm, tile->rows - at);
  return true;
}

template <typename T, int BM, int BN, int WM, int WN, int D>
struct TileOf {
  using Tile = MfmaTile<T, BM, BN, WM, WN, D>;
  static constexpr int kRows = BM, kCols = BN, kWM = WM, kWN = WN, kThreads = Tile::kThreads;
  static constexpr size_t kLds = Tile::kLds;
};

// act [sorted pair][Fp] = glu(h gate^T, h up^T). A wavefront's column blocks are gate and up of the same 32 columns, in turn.
// kFar, here and below: rows too long for 32-bit offsets.
template <typename T, typename Shape, bool kFar>
__device__ __forceinline__ void gate_up_tile(uint8_t* smem, const MoeTile& tile, int n, const T* __restrict__ h,
                                             const T* __restrict__ w, T* __restrict__ act, const int* __restrict__ order, int M,
                                             int top, int Hp, int Fp, float limit) {
  using Tile = typename Shape::Tile;
  constexpr int BM = Shape::kRows, BN = Shape::kCols, WM = Shape::kWM, WN = Shape::kWN;
  static_assert(Tile::FN % 2 == 0, "gate and up in one wavefront");
  const int N = 2 * Fp;
  const int n0 = BN * n, wave = threadIdx.x >> 6, lane = threadIdx.x & 63, nb = min(BN, N - n0);
  RowOffset<kFar> oa[Tile::LA], ob[Tile::LB];
#pragma unroll
  for (int i = 0; i < Tile::LA; ++i)
    oa[i] = (RowOffset<kFar>)sizeof(T) * (order[tile.row0 + min(Tile::row(i), tile.rows - 1)] / top) * Hp + Tile::column();
#pragma unroll
  for (int i = 0; i < Tile::LB; ++i)
    ob[i] = (RowOffset<kFar>)sizeof(T) * (kFar ? min(Tile::row(i), nb - 1) : Tile::row(i)) * Hp + Tile::column();
  f32x16 acc[Tile::FM][Tile::FN];
  Tile::run(smem, tile_rows_at<kFar>(h, sizeof(T) * M * Hp), oa,
            tile_rows_at<kFar>(w + ((size_t)tile.expert * N + n0) * Hp, sizeof(T) * nb * Hp), ob, 0, Hp, acc);
  if constexpr (kFar) {
#pragma unroll
    for (int j = 0; j < Tile::FN; j += 2) {
      const int col = (n0 + BN / WN * (wave % WN) + 32 * j) / 2 + (lane & 31);
#pragma unroll
      for (int i = 0; i < Tile::FM; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int r = BM / WM * (wave / WN) + 32 * i + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
          if (r < tile.rows && col < Fp)
            act[(size_t)(tile.row0 + r) * Fp + col] = (T)clamped_glu<T>(acc[i][j][v], acc[i][j + 1][v], limit);
        }
    }
    return;
  }
  const __amdgpu_buffer_rsrc_t out = rows_buffer(act + (size_t)tile.row0 * Fp, sizeof(T) * tile.rows * Fp);
#pragma unroll
  for (int j = 0; j < Tile::FN; j += 2) {
    const int col = (n0 + BN / WN * (wave % WN) + 32 * j) / 2 + (lane & 31);
#pragma unroll
    for (int i = 0; i < Tile::FM; ++i) {
      const int r = BM / WM * (wave / WN) + 32 * i + 4 * (lane >> 5);
      unsigned off = col < Fp ? (unsigned)sizeof(T) * (r * Fp + col) : kPastEnd;  // past the end: not stored
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        float g = acc[i][j][v], u = acc[i][j + 1][v];
        asm volatile("" : "+v"(g), "+v"(u), "+v"(off));  // one after the other, or all of it is in registers at once
        const T y = (T)clamped_glu<T>(g, u, limit);
        if constexpr (sizeof(T) == 2) __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(unsigned short, y), out, off, 0, 0);
        else __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(y), out, off, 0, 0);
        off += (unsigned)sizeof(T) * (v % 4 == 3 ? 5 : 1) * Fp;
      }
    }
  }
}

template <typename T, typename Big, typename Rest, bool kFar>
__global__ __launch_bounds__(Big::kThreads) void moe_gate_up_kernel(const T* __restrict__ h, const T* __restrict__ w,
                                                                    T* __restrict__ act, const int* __restrict__ order,
                                                                    const MoeTile* __restrict__ tiles,
                                                                    const int* __restrict__ n_tiles, int M, int top, int Hp,
                                                                    int Fp, float limit) {
  extern __shared__ __align__(16) uint8_t smem[];
  MoeTile tile;
  int n;
  bool rest;
  if (!moe_tile<(Rest::kRows < Big::kRows)>(tiles, n_tiles, Big::kRows, (2 * Fp + Big::kCols - 1) / Big::kCols, &tile, &n, &rest)) return;
  if (Rest::kRows < Big::kRows && rest)
    gate_up_tile<T, Rest, kFar>(smem, tile, n, h, w, act, order, M, top, Hp, Fp, limit);
  else
    gate_up_tile<T, Big, kFar>(smem, tile, n, h, w, act, order, M, top, Hp, Fp, limit);
}

// parts [slot][token][Hp] = weight * act down^T; a slot has rows_all tokens
template <typename T, typename Shape, bool kFar>
__device__ __forceinline__ void down_tile(uint8_t* smem, const MoeTile& tile, int n, const T* __restrict__ act,
                                          const T* __restrict__ w, float* __restrict__ parts, const int* __restrict__ order,
                                          const float* __restrict__ wts, int top, int rows_all, int Hp, int Fp) {
  using Tile = typename Shape::Tile;
  constexpr int BM = Shape::kRows, BN = Shape::kCols, WM = Shape::kWM, WN = Shape::kWN;
  const int n0 = BN * n, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  // a row's place and weight, asked for now and handed round through LDS behind the products
  static_assert(BM <= Tile::kThreads, "a thread per row");
  const int own = order[tile.row0 + min((int)threadIdx.x, tile.rows - 1)];
  const int nb = min(BN, Hp - n0);
  RowOffset<kFar> oa[Tile::LA], ob[Tile::LB];
  auto at = [&](int i, int rows) __attribute__((always_inline)) {
    const int r = kFar ? min(Tile::row(i), rows - 1) : Tile::row(i);
    return (RowOffset<kFar>)sizeof(T) * r * Fp + Tile::column();
  };
#pragma unroll
  for (int i = 0; i < Tile::LA; ++i) oa[i] = at(i, tile.rows);
#pragma unroll
  for (int i = 0; i < Tile::LB; ++i) ob[i] = at(i, nb);
  f32x16 acc[Tile::FM][Tile::FN];
  Tile::run(smem, tile_rows_at<kFar>(act + (size_t)tile.row0 * Fp, sizeof(T) * tile.rows * Fp), oa,
            tile_rows_at<kFar>(w + ((size_t)tile.expert * Hp + n0) * Fp, sizeof(T) * nb * Fp), ob, 0, Fp, acc);
  const float weight = wts[own];
  __syncthreads();
  float* s_w = reinterpret_cast<float*>(smem);            // [BM]
  int* s_row = reinterpret_cast<int*>(smem) + BM;         // [BM], row of parts
  if (threadIdx.x < BM) {
    const int m = own / top;
    s_w[threadIdx.x] = weight;
    s_row[threadIdx.x] = (own - m * top) * rows_all + m;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < Tile::FM; ++i)
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int r = BM / WM * (wave / WN) + 32 * i + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
      if (r >= tile.rows) continue;
      const float a = s_w[r];
      float* dst = parts + (size_t)s_row[r] * Hp;
#pragma unroll
      for (int j = 0; j < Tile::FN; ++j) {
        const int col = n0 + BN / WN * (wave % WN) + 32 * j + (lane & 31);
        if (col < Hp) dst[col] = a * acc[i][j][v];
      }
    }
}

template <typename T, typename Big, typename Rest, bool kFar>
__global__ __launch_bounds__(Big::kThreads) void moe_down_kernel(const T* __restrict__ act, const T* __restrict__ w,
                                                                 float* __restrict__ parts, const int* __restrict__ order,
                                                                 const float* __restrict__ wts,
                                                                 const MoeTile* __restrict__ tiles,
                                                                 const int* __restrict__ n_tiles, int top, int rows_all, int Hp,
                                                                 int Fp) {
  extern __shared__ __align__(16) uint8_t smem[];
  MoeTile tile;
  int n;
  bool rest;
  if (!moe_tile<(Rest::kRows < Big::kRows)>(tiles, n_tiles, Big::kRows, (Hp + Big::kCols - 1) / Big::kCols, &tile, &n, &rest)) return;
  if (Rest::kRows < Big::kRows && rest)
    down_tile<T, Rest, kFar>(smem, tile, n, act, w, parts, order, wts, top, rows_all, Hp, Fp);
  else
    down_tile<T, Big, kFar>(smem, tile, n, act, w, parts, order, wts, top, rows_all, Hp, Fp);
}

// ---------------------------------------------------------------------------------------------
// z [slot][Fp] = weight * glu of the chosen experts; a group is P columns of one expert, gate and up row of each. The first
// workgroup leaves the choice for the launch behind. kRouter: every workgroup multiplies the router's rows [experts][Hp] itself,
// else `logits` holds the products.
template <typename WT, int P, int U, bool kRouter>
__global__ __launch_bounds__(kRowThreads) void moe_row_gate_up_kernel(const RowPrologue p, const float* __restrict__ logits,
                                                                      const WT* __restrict__ router,
                                                                      const WT* __restrict__ w, int experts, int top,
                                                                      int Hp, int Fp, float limit, float* __restrict__ z,
                                                                      int* __restrict__ sel) {
  extern __shared__ __align__(16) float s_x[];  // [Hp]
  __shared__ float s_red[3 * kRowWaves], s_logit[64];
  constexpr int R = 2 * P;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int gw = (int)blockIdx.x * kRowWaves + wave, nw = (int)gridDim.x * kRowWaves;
  const int per = Fp / P, groups = top * per;
  int expert = 0;
  float weight = 0.0f;
  auto ptr = [&](int g, int r, int k) {
    const int slot = g / per, c = (g - slot * per) * P + (r >> 1);
    const int row = (c >> 5) * 64 + (r & 1) * 32 + (c & 31);
    return w + ((size_t)__builtin_amdgcn_readlane(expert, slot) * 2 * Fp + row) * Hp + k;
  };
  Raw<WT> cur[R][U];
  float v[kLogitRegs];
  if constexpr (kRouter) {
    auto router_ptr = [&](int g, int, int k) { return router + (size_t)g * Hp + k; };
    Raw<WT> rows[1][U];
    row_prologue<WT, kRowNorm>(p, Hp, s_x, s_red, [&] {
      __builtin_amdgcn_sched_barrier(0);
      if (wave < experts) fetch_rows<WT, 1, U>(rows, wave, 0, Hp, router_ptr);
      __builtin_amdgcn_sched_barrier(0);
    });
    __syncthreads();
    stream_rows<WT, 1, U>(rows, wave, kRowWaves, experts, Hp, s_x, router_ptr, [&](int g, const float (&t)[1]) {
      if (lane == 0) s_logit[g] = t[0];
    });
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kLogitRegs; ++i) v[i] = i == 0 && lane < experts ? s_logit[lane] : -INFINITY;
    top_experts(v, experts, top, &expert, &weight);
    if (gw < groups) fetch_rows<WT, R, U>(cur, gw, 0, Hp, ptr);
  } else {
#pragma unroll
    for (int i = 0; i < kLogitRegs; ++i) v[i] = 64 * i + lane < experts ? logits[64 * i + lane] : -INFINITY;
    row_prologue<WT, kRowNorm>(p, Hp, s_x, s_red, [&] {
      top_experts(v, experts, top, &expert, &weight);
      __builtin_amdgcn_sched_barrier(0);
      if (gw < groups) fetch_rows<WT, R, U>(cur, gw, 0, Hp, ptr);
      __builtin_amdgcn_sched_barrier(0);
    });
    __syncthreads();
  }
  if (blockIdx.x == 0 && wave == 0 && lane < top) sel[lane] = expert;
  stream_rows<WT, R, U>(cur, gw, nw, groups, Hp, s_x, ptr, [&](int g, const float (&t)[R]) {
    const int slot = g / per;
    const float a = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(weight), slot));
#pragma unroll
    for (int i = 0; i < P; ++i)
      if (lane == 0) z[(size_t)g * P + i] = a * clamped_glu<float>(t[2 * i], t[2 * i + 1], limit);
  });
}

// out [Hp] = sum over the chosen experts of z_slot down^T: one product over the joined columns
template <typename WT, int R, int U>
__global__ __launch_bounds__(kRowThreads) void moe_row_down_kernel(const RowPrologue p, const int* __restrict__ sel,
                                                                   const WT* __restrict__ w, int top, int Hp, int Fp,
                                                                   unsigned magic, float* __restrict__ out) {
  extern __shared__ __align__(16) float s_x[];  // [top * Fp]
  __shared__ float s_red[3 * kRowWaves];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int gw = (int)blockIdx.x * kRowWaves + wave, nw = (int)gridDim.x * kRowWaves;
  const int groups = (Hp + R - 1) / R, K = top * Fp;
  const int expert = sel[min(lane, top - 1)];
  auto ptr = [&](int g, int r, int k) {
    const int slot = (int)__umulhi((unsigned)k, magic);  // k / Fp
    const int e = __shfl(expert, slot, 64);
    return w + ((size_t)e * Hp + min(g * R + r, Hp - 1)) * Fp + (k - slot * Fp);
  };
  Raw<WT> cur[R][U];
  row_prologue<WT, kRowPlain>(p, K, s_x, s_red, [&] {
    __builtin_amdgcn_sched_barrier(0);
    if (gw < groups) fetch_rows<WT, R, U>(cur, gw, 0, K, ptr);
    __builtin_amdgcn_sched_barrier(0);
  });
  __syncthreads();
  stream_rows<WT, R, U>(cur, gw, nw, groups, K, s_x, ptr, [&](int g, const float (&t)[R]) {
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (lane == 0 && g * R + r < Hp) out[g * R + r] = t[r];
  });
}

// ---------------------------------------------------------------------------------------------
inline size_t up256(size_t v) { return (v + 255) / 256 * 256; }

// what a portion's experts work in
struct Scratch {
  size_t ids, wts, order, up_tiles, down_tiles, n_tiles, act, bytes;
  int max_tiles;
};
Scratch scratch_of(int dtype, int M, int experts, int top, int Fp) {
  const size_t n = (size_t)M * top, elem = dtype == W4A32_LAYERED_BF16 ? 2 : 4;
  Scratch c;
  c.max_tiles = (int)((n + 63) / 64) + experts;
  size_t o = 0;
  auto take = [&](size_t bytes) {
    const size_t at = o;
    o += up256(bytes);
    return at;
  };
  c.ids = take(4 * n);
  c.wts = take(4 * n);
  c.order = take(4 * n);
  c.up_tiles = take(sizeof(MoeTile) * c.max_tiles);
  c.down_tiles = take(sizeof(MoeTile) * c.max_tiles);
  c.n_tiles = take(4 * 4);
  c.act = take(elem * n * Fp);
  c.bytes = o;
  return c;
}

// The shapes of the grouped products. Rest: the tile of an expert's last rows where they fit it.
template <typename T, int BM, int BN, int WM, int WN, int D, int RM = BM>
struct ShapeOf {
  using Big = TileOf<T, BM, BN, WM, WN, D>;
  using Rest = TileOf<T, RM, BN, WM, WN, D>;
  static_assert(Rest::kLds <= Big::kLds && Rest::kThreads == Big::kThreads);
  static_assert((BM & (BM - 1)) == 0);
  static constexpr MoeHeights heights() { return {BM == 256 ? 8 : BM == 128 ? 7 : 6, RM < BM ? RM : 0}; }
  // workgroups; those past the last tile return
  static unsigned grid(const MoeGeom& g, int M, int N) {
    return (unsigned)((size_t)M * g.top / BM + g.experts) * (unsigned)((N + BN - 1) / BN);
  }
};

template <typename Shape, bool kFar = false, typename T>
hipError_t launch_gate_up(const MoeGeom& g, const T* h, const T* gate_up, int M, uint8_t* ws, const Scratch& c, hipStream_t s) {
  using Big = typename Shape::Big;
  auto kern = moe_gate_up_kernel<T, Big, typename Shape::Rest, kFar>;
  static LdsLimitOnce raised;
  if (Big::kLds > 64 * 1024)
    if (hipError_t e = raised.raise(reinterpret_cast<const void*>(kern), Big::kLds); e != hipSuccess) return e;
  hipLaunchKernelGGL(kern, dim3(Shape::grid(g, M, 2 * g.Fp)), dim3(Big::kThreads), Big::kLds, s, h, gate_up,
                     reinterpret_cast<T*>(ws + c.act), reinterpret_cast<const int*>(ws + c.order),
                     reinterpret_cast<const MoeTile*>(ws + c.up_tiles), reinterpret_cast<const int*>(ws + c.n_tiles), M, g.top,
                     g.Hp, g.Fp, g.limit);
  return hipGetLastError();
}

template <typename Shape, bool kFar = false, typename T>
hipError_t launch_down(const MoeGeom& g, const T* down, int M, int rows_all, float* parts, uint8_t* ws, const Scratch& c,
                       hipStream_t s) {
  using Big = typename Shape::Big;
  auto kern = moe_down_kernel<T, Big, typename Shape::Rest, kFar>;
  static LdsLimitOnce raised;
  if (Big::kLds > 64 * 1024)
    if (hipError_t e = raised.raise(reinterpret_cast<const void*>(kern), Big::kLds); e != hipSuccess) return e;
  hipLaunchKernelGGL(kern, dim3(Shape::grid(g, M, g.Hp)), dim3(Big::kThreads), Big::kLds, s,
                     reinterpret_cast<const T*>(ws + c.act), down, parts, reinterpret_cast<const int*>(ws + c.order),
                     reinterpret_cast<const float*>(ws + c.wts), reinterpret_cast<const MoeTile*>(ws + c.down_tiles),
                     reinterpret_cast<const int*>(ws + c.n_tiles) + 2, g.top, rows_all, g.Hp, g.Fp);
  return hipGetLastError();
}

// A 256 x 256 tile of [2 x 2240][1536] takes 42 us of which its activation and stores are 5: with one workgroup per CU nothing runs under
// them. Whole tiles stand in front of the shorter last rows': mixed, 1501 tokens of 16 experts, 4 per token, took 116 / 57 us (gate and up /
// down) against 106 / 57, as the large ones then end late. 100 tokens, [2 x 2240][1536], 64 x 128: 49 / 23 = 4.5 and 4.9 TB/s of weights, 128 x
// 128 53 / 26.
//
// What the bf16 shapes cost: us per 64 k of a tile with all CUs busy, and per tile for what stands in front of and behind its products, on
// `slots` tiles at once. Fitted for the choice, not for the time (which is 10 to 20 % off: the weights' way from memory is not in it), to 1700
// products of 96 to 2000 rows per expert, 4 to 128 experts, from [2 x 256][512] to [2 x 4736][3584].
struct MoeShape {
  int bm, rest, bn, slots;
  double up_tile_us, down_tile_us, up_us, down_us;
};
constexpr MoeShape kTall = {256, 128, 256, 256, 1.57, 1.57, 6.3, 10.8}, kWide = {128, 0, 256, 256, 0.967, 0.967, 2.2, 4.6},
                   kSmall = {128, 0, 128, 512, 1.13, 1.36, 1.55, 3.0};

// What an expert has where `per` rows come to it by independent choices (standard deviation sqrt(per)): on average, and the
// variance of the whole tiles.
struct MoeTiles {
  double whole, rest, var;
};
MoeTiles expected_tiles(double per, int bm, int rest) {
  const double sd = std::sqrt(per);
  auto more_than = [&](double rows) { return 0.5 * std::erfc((rows + 0.5 - per) / (sd * std::sqrt(2.0))); };
  int n = std::max(0, (int)((per - 5.0 * sd) / bm) - 1);  // so many are whole as good as always
  MoeTiles t{(double)n, 0.0, 0.0};
  for (;; ++n) {
    const double begun = n > 0 ? more_than((double)n * bm) : 1.0, full = n > 0 || rest > 0 ? more_than((double)n * bm + rest) : 1.0;
    if (begun < 1e-4) return t;
    t.whole += full;
    t.rest += begun - full;
    t.var += full * (1.0 - full);
  }
}

// us of `whole` tiles, and with kTall of `rest` lower ones behind them
double moe_rounds_us(const MoeShape& t, double whole, double rest, double tile_us, double rest_us) {
  if (t.rest == 0) whole = std::max(1.0, whole - 0.5);
  const double rounds = std::floor(whole / t.slots), left = whole - rounds * t.slots;
  if (t.slots == 512)  // two tiles per CU: alone on it one takes half as long
    return tile_us * (rounds + (left <= 0.0 ? 0.0 : left <= 256.0 ? 0.53 : 0.53 + 0.47 * std::min(1.0, (left - 256.0) / 14.0)));
  if (t.rest == 0) return tile_us * (rounds + (left > 0.0 ? 1.0 : 0.0));
  // the slots with a tile of the last round and those without one, as the rests come to them
  double free_at[2] = {(rounds + (left >= 1.0 ? 1.0 : 0.0)) * tile_us, rounds * tile_us}, end = (rounds + std::min(1.0, left)) * tile_us;
  const double slots[2] = {left >= 1.0 ? left : 0.0, left >= 1.0 ? t.slots - left : t.slots};
  while (rest > 0.5) {
    const int i = free_at[1] <= free_at[0] || slots[0] <= 0.0 ? 1 : 0;
    rest -= slots[i];
    free_at[i] += rest_us;
    end = std::max(end, free_at[i]);
  }
  return end;
}

double moe_shape_us(const MoeShape& t, const MoeGeom& g, int M, bool up) {
  const int N = up ? 2 * g.Fp : g.Hp, nt = (N + t.bn - 1) / t.bn;
  const double k = (up ? g.Hp : g.Fp) / 64.0, over = up ? t.up_us : t.down_us, tile_us = (up ? t.up_tile_us : t.down_tile_us) * k + over;
  const MoeTiles tiles = expected_tiles((double)M * g.top / g.experts, t.bm, t.rest);
  // a rest's tile beside whole ones takes about as long as kWide's; the more of the time all CUs are at rests, the more they wait for memory
  const double rest_us = (1.03 + 0.49 * std::min(1.0, tiles.rest / std::max(tiles.whole, 1e-9))) * k + over / 2;
  // the number of tiles is not known: a last round that a few of them begin counts as often as it comes
  const double mean = tiles.whole * g.experts * nt, sd = nt * std::sqrt(g.experts * tiles.var), rest = tiles.rest * g.experts * nt;
  auto at = [&](double z) { return moe_rounds_us(t, std::max(0.0, mean + z * sd), rest, tile_us, rest_us); };
  return 0.25 * at(-1.22) + 0.5 * at(0.0) + 0.25 * at(1.22);
}

// The cheapest: 0 kTall, 1 kWide, 2 kSmall. (128 x 256 is one workgroup per CU, 128 x 128 two that fill each other's gaps, which the costs do not
// know: it has to be clearly cheaper.) Over those products that is 1.0 % slower than the best shape; against a shape by rows per expert and
// number of tiles alone 3.8 % quicker, and slower by more than 3 % for 27 of them (16 % at most). Us in 256 x 256 with last rows in 128 x 256 / in
// 128 x 256 / in 128 x 128, and what is chosen, 16 experts, 4 per token:
//   tokens, experts         gate and up                    down
//   900, [2 x 2240][1536]   86.5 89.1 80.7 (128 x 128)     54.0 43.3 49.7 (128 x 256)
//   1501                    103  115  112  (128 x 128)     57.4 77.7 69.3 (256 x 256)
//   2048                    136  140  146  (256 x 256)     62.8 78.9 88.3 (256 x 256)
//   512, [2 x 4736][3584]   257  282  293  (128 x 128)     110  170  165  (256 x 256)
//   2048                    541  628  675  (256 x 256)     285  314  360  (256 x 256)
// (1501 tokens, gate and up: in the whole model 256 x 256 is half a percent of it quicker.)
int moe_shape(const MoeGeom& g, int M, bool up) {
  const double us[3] = {moe_shape_us(kTall, g, M, up), moe_shape_us(kWide, g, M, up) / 0.91, moe_shape_us(kSmall, g, M, up)};
  return (int)(std::min_element(us, us + 3) - us);
}

// rows an expert has on average, too few of them for 128-row tiles
bool moe_few(const MoeGeom& g, int M) { return (long)M * g.top / g.experts < 96; }

template <typename T>
bool experts_far(const MoeGeom& g) {
  return !rows_near(sizeof(T) * (size_t)std::max(g.Hp, g.Fp)) || !results_near(sizeof(T) * (size_t)g.Fp);
}

template <typename Up, typename Down, bool kFar = false, typename T>
hipError_t grouped(const MoeGeom& g, const T* h, const T* gate_up, const T* down, int M, int rows_all, float* parts,
                   uint8_t* ws, const Scratch& c, hipStream_t s) {
  hipLaunchKernelGGL(moe_plan_kernel, dim3(g.experts), dim3(kPlanThreads), 0, s, reinterpret_cast<const int*>(ws + c.ids),
                     M * g.top, g.experts, Up::heights(), Down::heights(), reinterpret_cast<int*>(ws + c.order),
                     reinterpret_cast<MoeTile*>(ws + c.up_tiles), reinterpret_cast<MoeTile*>(ws + c.down_tiles),
                     reinterpret_cast<int*>(ws + c.n_tiles));
  if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
  if (hipError_t e = launch_gate_up<Up, kFar>(g, h, gate_up, M, ws, c, s); e != hipSuccess) return e;
  return launch_down<Down, kFar>(g, down, M, rows_all, parts, ws, c, s);
}

template <typename T>
hipError_t prefill_t(int dtype, const MoeGeom& g, const T* h, const float* logits, int logit_parts, size_t part_stride, int ldl,
                     const T* gate_up, const T* down, int M, int rows_all, float* parts, uint8_t* ws, hipStream_t s) {
  const Scratch c = scratch_of(dtype, M, g.experts, g.top, g.Fp);
  hipLaunchKernelGGL(moe_choose_kernel, dim3((M + 3) / 4), dim3(256), 0, s, logits, logit_parts, part_stride, ldl, M,
                     g.experts, g.top, reinterpret_cast<int*>(ws + c.ids), reinterpret_cast<float*>(ws + c.wts));
  if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
  auto run = [&](auto up, auto down_shape) {
    return grouped<decltype(up), decltype(down_shape)>(g, h, gate_up, down, M, rows_all, parts, ws, c, s);
  };
  if (experts_far<T>(g)) {
    using Far = ShapeOf<T, 64, 128, 2, 2, 2>;
    return grouped<Far, Far, true>(g, h, gate_up, down, M, rows_all, parts, ws, c, s);
  }
  const bool few = moe_few(g, M);
  if constexpr (sizeof(T) == 2) {
    if (few) return run(ShapeOf<T, 64, 128, 2, 2, 4>{}, ShapeOf<T, 64, 128, 2, 4, 4>{});
    auto with = [&](auto up) {
      switch (moe_shape(g, M, false)) {
        case 0: return run(up, ShapeOf<T, 256, 256, 2, 4, 2, 128>{});
        case 1: return run(up, ShapeOf<T, 128, 256, 2, 4, 2>{});
        default: return run(up, ShapeOf<T, 128, 128, 2, 4, 2>{});
      }
    };
    switch (moe_shape(g, M, true)) {
      case 0: return with(ShapeOf<T, 256, 256, 2, 4, 2, 128>{});
      case 1: return with(ShapeOf<T, 128, 256, 2, 4, 2>{});
      default: return with(ShapeOf<T, 128, 128, 2, 2, 2>{});
    }
  } else {
    if (few) return run(ShapeOf<T, 64, 128, 2, 2, 2>{}, ShapeOf<T, 64, 128, 2, 2, 2>{});
    return run(ShapeOf<T, 128, 128, 2, 2, 2>{}, ShapeOf<T, 128, 128, 2, 2, 2>{});
  }
}

// The gathered rows' byte offsets have 32 bits: more rows than that go in several turns, one after the other on the same scratch.
template <typename T>
hipError_t prefill_turns(int dtype, const MoeGeom& g, const T* h, const float* logits, int logit_parts, int ldl,
                         const T* gate_up, const T* down, int M, float* parts, uint8_t* ws, hipStream_t s) {
  if (logit_parts < 1 || logit_parts > kMaxParts) return hipErrorInvalidValue;
  const int turn = experts_far<T>(g) ? M : (int)std::min<size_t>(M, 0xFFFFFFFFu / (sizeof(T) * g.Hp));
  for (int m = 0; m < M; m += turn)
    if (hipError_t e = prefill_t(dtype, g, h + (size_t)m * g.Hp, logits + (size_t)m * ldl, logit_parts, (size_t)M * ldl, ldl,
                                 gate_up, down, std::min(turn, M - m), M, parts + (size_t)m * g.Hp, ws, s);
        e != hipSuccess)
      return e;
  return hipSuccess;
}

template <typename WT>
hipError_t decode_t(const MoeGeom& g, const RowPrologue& pro, const float* logits, const WT* router, const WT* gate_up,
                    const WT* down, float* z, int* sel, float* out, hipStream_t s) {
  {
    // One column at a time, as the rows of w4a32_lin16.hip: bf16, four experts of [2 x 2240][1536]: 15.5 us = 3.6 TB/s (17.0 with
    // the router's products inside, 4.3 of a launch less), two columns 18.1 (4480 groups on 4096 wavefronts); [2 x 576][832]: 5.8 against 6.9; [2 x 4736][3584]: 46.5 against 46.2.
    constexpr int P = 1, U = 3;
    const int groups = g.top * g.Fp / P;
    const dim3 grid(std::min((groups + kRowWaves - 1) / kRowWaves, 512));
    const size_t lds = sizeof(float) * g.Hp;
    auto run = [&](auto kern, LdsLimitOnce* raised) -> hipError_t {  // (both kernels have one type: a limit raised here would be for either)
      if (lds > 60 * 1024)
        if (hipError_t e = raised->raise(reinterpret_cast<const void*>(kern), 159 * 1024); e != hipSuccess) return e;
      hipLaunchKernelGGL(kern, grid, dim3(kRowThreads), lds, s, pro, logits, router, gate_up, g.experts, g.top, g.Hp, g.Fp,
                         g.limit, z, sel);
      return hipGetLastError();
    };
    static LdsLimitOnce raised_router, raised_plain;
    const hipError_t e = moe_routes_itself(sizeof(WT), g) ? run(moe_row_gate_up_kernel<WT, P, U, true>, &raised_router)
                                                          : run(moe_row_gate_up_kernel<WT, P, U, false>, &raised_plain);
    if (e != hipSuccess) return e;
  }
  RowPrologue p{};
  p.K = g.top * g.Fp;
  p.x = z;
  constexpr int U = 6;
  auto kern = moe_row_down_kernel<WT, 1, U>;
  const size_t lds = sizeof(float) * g.top * g.Fp;
  static LdsLimitOnce raised;
  if (lds > 60 * 1024)
    if (hipError_t e = raised.raise(reinterpret_cast<const void*>(kern), 159 * 1024); e != hipSuccess) return e;
  const unsigned magic = (unsigned)(((1ull << 32) + g.Fp - 1) / g.Fp);  // exact quotients below 2^32 / Fp
  hipLaunchKernelGGL(kern, dim3(std::min((g.Hp + kRowWaves - 1) / kRowWaves, 512)), dim3(kRowThreads), lds, s, p, sel, down,
                     g.top, g.Hp, g.Fp, magic, out);
  return hipGetLastError();
}

}  // namespace

int moe_tile_size(int dtype, const MoeGeom& g, int M, bool up) {
  const bool bf16 = dtype == W4A32_LAYERED_BF16;
  if ((bf16 ? experts_far<__bf16>(g) : experts_far<float>(g)) || moe_few(g, M)) return 64 << 16 | 128;
  const int shape = bf16 ? moe_shape(g, M, up) : 2;
  return shape == 0 ? 256 << 16 | 256 : shape == 1 ? 128 << 16 | 256 : 128 << 16 | 128;
}

size_t moe_scratch_bytes(int dtype, int M, int experts, int top, int Fp) { return scratch_of(dtype, M, experts, top, Fp).bytes; }

hipError_t launch_moe_prefill(int dtype, const MoeGeom& g, const void* h, const float* logits, int logit_parts, int ldl,
                              const void* gate_up, const void* down, int M, float* parts, void* scratch, hipStream_t s) {
  uint8_t* ws = static_cast<uint8_t*>(scratch);
  if (dtype == W4A32_LAYERED_BF16)
    return prefill_turns(dtype, g, static_cast<const __bf16*>(h), logits, logit_parts, ldl, static_cast<const __bf16*>(gate_up),
                     static_cast<const __bf16*>(down), M, parts, ws, s);
  return prefill_turns(dtype, g, static_cast<const float*>(h), logits, logit_parts, ldl, static_cast<const float*>(gate_up),
                   static_cast<const float*>(down), M, parts, ws, s);
}

// Up to 96 KB of router a launch of its own costs more than every workgroup's pass over it: per layer of a decode step with four
// experts of [128][width], bf16, [16][1536]: 28.2 -> 26.3 us, [32][1536]: 29.6 -> 28.5, [64][1024]: 30.4 -> 30.7, [64][1536]: 31.7 ->
// 32.6; f32, [16][1536]: 32.0 -> 30.1, [32][1536]: 33.0 -> 32.8, [64][1024]: 32.7 -> 34.9.
bool moe_routes_itself(size_t elem_bytes, const MoeGeom& g) {
  return g.experts <= 64 && (size_t)g.experts * g.Hp * elem_bytes <= 96 * 1024;
}

bool moe_decode_fits(const MoeGeom& g) { return row_linear_fits(g.Hp) && (long)g.top * g.Fp <= 35840; }

hipError_t launch_moe_decode(int dtype, const MoeGeom& g, const RowPrologue& pro, const float* logits, const void* router,
                             const void* gate_up, const void* down, float* z, int* sel, float* out, hipStream_t s) {
  if (!moe_decode_fits(g)) return hipErrorInvalidValue;
  if (dtype == W4A32_LAYERED_BF16)
    return decode_t(g, pro, logits, static_cast<const __bf16*>(router), static_cast<const __bf16*>(gate_up),
                    static_cast<const __bf16*>(down), z, sel, out, s);
  return decode_t(g, pro, logits, static_cast<const float*>(router), static_cast<const float*>(gate_up),
                  static_cast<const float*>(down), z, sel, out, s);
}

}  // namespace w4
