// Linears with bf16 (or f32) weights for the layered decoder.
//
//   matmul_kernel        C = A B^T, bf16 or f32 operands, f32 accumulation, for prefill rows: tiles from 64 x 64 to 256 x 256
//                        (f32: 64 x 128), the k range dealt to several workgroups where the caller adds the parts up.
//   row_linear_kernel    one decode row through [N][K] weights, read once, with the operator that produces the row
//                        in front (residual add + norm + input convolution, merge of the attention's key slices,
//                        per-head norm and gate, PolyNorm, none): HBM-bound, N * K * sizeof(weight) bytes.
//
// The tile of C a workgroup owns and the rows a decode Linear multiplies are in w4a32_mfma_tile.h and w4a32_row_prologue.h.
#include <algorithm>
#include <cmath>

#include "w4a32_layered.h"
#include "w4a32_layered_kernels.h"
#include "w4a32_mfma_tile.h"
#include "w4a32_row_prologue.h"

namespace w4 {

namespace {

// The tile of C from row m0 and column n0 on, over k in [kb, ke). kFar: operands or results whose rows are too long for 32-bit offsets
template <typename T, int BM, int BN, int WM, int WN, int D, typename CT, bool kFar>
__device__ __forceinline__ void matmul_tile(uint8_t* smem, const T* __restrict__ a, const T* __restrict__ b, CT* __restrict__ c,
                                            int M, int N, int K, int ldc, int m0, int n0, int kb, int ke) {
  using Tile = MfmaTile<T, BM, BN, WM, WN, D>;
  constexpr int FM = Tile::FM, FN = Tile::FN;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int wm = (wave / WN) * (BM / WM), wn = (wave % WN) * (BN / WN);

  const int ma = min(M - m0, BM), nb = min(N - n0, BN);
  RowOffset<kFar> oa[Tile::LA], ob[Tile::LB];
  auto at = [&](int i, int rows) __attribute__((always_inline)) {
    const int r = kFar ? min(Tile::row(i), rows - 1) : Tile::row(i);
    return (RowOffset<kFar>)sizeof(T) * r * K + Tile::column();
  };
#pragma unroll
  for (int i = 0; i < Tile::LA; ++i) oa[i] = at(i, ma);
#pragma unroll
  for (int i = 0; i < Tile::LB; ++i) ob[i] = at(i, nb);
  f32x16 acc[FM][FN];
  Tile::run(smem, tile_rows_at<kFar>(a + (size_t)m0 * K, sizeof(T) * ma * K), oa,
            tile_rows_at<kFar>(b + (size_t)n0 * K, sizeof(T) * nb * K), ob, kb, ke, acc);

  c += (size_t)m0 * ldc;
  if constexpr (kFar) {
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int row = wm + 32 * i + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3), col = n0 + wn + 32 * j + (lane & 31);
          if (row < ma && col < N) c[(size_t)row * ldc + col] = (CT)acc[i][j][v];
        }
    return;
  }
  // rows past the last one lie past the buffer's end, columns are sent there: what is stored there is dropped
  const __amdgpu_buffer_rsrc_t out = rows_buffer(c, sizeof(CT) * ma * ldc);
  const unsigned step = (unsigned)sizeof(CT) * ldc;
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const int col = n0 + wn + 32 * j + (lane & 31);
      unsigned off = col < N ? (unsigned)sizeof(CT) * ((wm + 32 * i + 4 * (lane >> 5)) * ldc + col) : kPastEnd;
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        float x = acc[i][j][v];
        asm volatile("" : "+v"(x), "+v"(off));  // or all offsets, and a copy of acc as integers, are made first, and spilled
        if constexpr (sizeof(CT) == 4) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(x), out, off, 0, 0);
        else __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(unsigned short, (CT)x), out, off, 0, 0);
        off += v % 4 == 3 ? 5 * step : step;
      }
    }
}

template <typename T, int BM, int BN, int WM, int WN, int D, typename CT, bool kFar>
__global__ __launch_bounds__(64 * WM * WN) void matmul_kernel(const T* __restrict__ a, const T* __restrict__ b,
                                                              CT* __restrict__ c, int M, int N, int K, int ldc, int mt,
                                                              int nt) {
  extern __shared__ __align__(16) uint8_t smem[];
  // tile number: consecutive ones on one XCD
  const int t = xcd_tile(blockIdx.x, mt * nt);
  // this workgroup's share of the k range, in whole LDS tiles
  constexpr int kBK = MfmaTile<T, BM, BN, WM, WN, D>::kBK;
  const int k_steps = K / kBK;
  const int kb = (int)((long)k_steps * blockIdx.y / gridDim.y) * kBK;
  const int ke = (int)((long)k_steps * (blockIdx.y + 1) / gridDim.y) * kBK;
  matmul_tile<T, BM, BN, WM, WN, D, CT, kFar>(smem, a, b, c + (size_t)blockIdx.y * M * ldc, M, N, K, ldc, (t % mt) * BM, (t / mt) * BN,
                                              kb, ke);
}

// The first `whole` bands of columns in tiles of 256 x 256, the others, behind them, in tiles of 128 x 256: whole rounds of the CUs
// in the large tile, what is left of C in one that takes half as long. [2048][3584] x [18944][3584], 592 large tiles: 259 us, as 512
// and 160 small ones 243; [2048][3584] x [10752][3584]: 164 (256 x 128) and 150; [2048][1536] x [8960][1536]: 68 (128 x 128) and 61.
template <typename CT>
__global__ __launch_bounds__(512) void matmul_two_heights_kernel(const __bf16* __restrict__ a, const __bf16* __restrict__ b,
                                                                 CT* __restrict__ c, int M, int N, int K, int ldc, int nt, int whole) {
  extern __shared__ __align__(16) uint8_t smem[];
  const int mt = (M + 255) / 256, rt = (M + 127) / 128;
  if ((int)blockIdx.x < whole * mt) {
    const int t = xcd_tile(blockIdx.x, whole * mt);
    matmul_tile<__bf16, 256, 256, 2, 4, 2, CT, false>(smem, a, b, c, M, N, K, ldc, t % mt * 256, t / mt * 256, 0, K);
  } else {
    const int t = xcd_tile((int)blockIdx.x - whole * mt, (nt - whole) * rt);
    matmul_tile<__bf16, 128, 256, 2, 4, 2, CT, false>(smem, a, b, c, M, N, K, ldc, t % rt * 128, (whole + t / rt) * 256, 0, K);
  }
}

template <typename T, int BM, int BN, int WM, int WN, int D, typename CT, bool kFar = false>
hipError_t launch_tile_t(const T* a, const T* b, void* c, int M, int N, int K, int ldc, int parts, hipStream_t s) {
  const int mt = (M + BM - 1) / BM, nt = (N + BN - 1) / BN;
  constexpr size_t lds = MfmaTile<T, BM, BN, WM, WN, D>::kLds;
  auto kern = matmul_kernel<T, BM, BN, WM, WN, D, CT, kFar>;
  static LdsLimitOnce raised;
  if (lds > 64 * 1024)
    if (hipError_t e = raised.raise(reinterpret_cast<const void*>(kern), lds); e != hipSuccess) return e;
  // parts <= K / kBK: no share is empty
  hipLaunchKernelGGL(kern, dim3(mt * nt, parts), dim3(64 * WM * WN), lds, s, a, b, static_cast<CT*>(c), M, N, K, ldc, mt, nt);
  return hipGetLastError();
}

template <typename CT>
hipError_t launch_two_heights(const __bf16* a, const __bf16* b, void* c, int M, int N, int K, int ldc, int whole, hipStream_t s) {
  const int mt = (M + 255) / 256, rt = (M + 127) / 128, nt = (N + 255) / 256;
  constexpr size_t lds = MfmaTile<__bf16, 256, 256, 2, 4, 2>::kLds;
  auto kern = matmul_two_heights_kernel<CT>;
  static LdsLimitOnce raised;
  if (hipError_t e = raised.raise(reinterpret_cast<const void*>(kern), lds); e != hipSuccess) return e;
  hipLaunchKernelGGL(kern, dim3(whole * mt + (nt - whole) * rt), dim3(512), lds, s, a, b, static_cast<CT*>(c), M, N, K, ldc, nt, whole);
  return hipGetLastError();
}

// The shapes, and what they cost. A CU that is alone takes tile_us per 64 k of a tile; with all of them busy the chip's clock
// drops and it delivers `tflops`. (Fitted to 16 sizes from [40][1536] x [8960][1536] to [2048][3584] x [14336][3584]; over 59
// other sizes of up to 2048 rows the choice was 0.9 % slower than the best one, 10 % at most.)
struct Shape {
  int bm, bn;
  double tile_us, tflops;
};
constexpr Shape kShapes[] = {
    {256, 256, 1.13, 1270}, {256, 128, 0.70, 1060}, {128, 128, 0.46, 950}, {64, 128, 0.36, 660}, {64, 64, 0.25, 490}};
// The same in f32, per 32 k: bound by the matrix cores (157 TFLOP/s) whatever the shape, so the small one, which fills the CUs
// first, unless there are many ([2000][2048] x [3000][2048]: 224 us, 64 x 128 190 = 130 TFLOP/s, 128 x 128 242). [300][4096] x
// [1024][4096] took 100 us in one part of 64 x 64 without anything requested ahead; in one part of these 64, in four 34.
constexpr Shape kShapesF32[] = {{64, 128, 0.91, 130}, {64, 64, 0.50, 118}};

// Half of the first one, for its last round: not fitted by itself, but priced as 256 x 128, which has as many products and loads. Of 240 products
// of 128 to 8192 rows, [N][K] from [500][256] to [32000][11500], 21 were given to it; they take 0.78 to 1.00 times the best single shape's time.
constexpr Shape kHalf = {128, 256, 0.70, 1060};

// us: rounds of the CUs, and the results' way to memory (and, as partial products, back)
double shape_us(const Shape& t, int M, int N, double k_tiles, double tile_flops, int parts, int c_bytes) {
  const long tiles = (long)((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn) * parts;
  k_tiles /= parts;
  const double flops = tile_flops * t.bm * t.bn * k_tiles;
  auto round_us = [&](long n) { return std::max(t.tile_us * k_tiles, n * flops / (t.tflops * 1e6)); };
  const double out = (double)M * N * c_bytes * (2 * parts - 1) / 5e6;
  return 2.5 + tiles / 256 * round_us(256) + (tiles % 256 ? round_us(tiles % 256) : 0.0) + out;
}

struct Plan {
  int shape, parts;
  int whole;  // bands of 256 columns in tiles of 256 rows, the others in tiles of 128; 0: one shape throughout
};

// us of 256 x 256 tiles whose last, incomplete round is cut into tiles of half the height, and how many bands are left whole
double two_heights_us(int M, int N, double k_tiles, double tile_flops, int c_bytes, int* whole) {
  const Shape& t = kShapes[0];
  const int mt = (M + t.bm - 1) / t.bm, nt = (N + t.bn - 1) / t.bn;
  *whole = (int)((long)mt * nt / 256 * 256 / mt);
  if (*whole < 1 || *whole >= nt) return INFINITY;
  auto round_us = [&](const Shape& s, long n) {
    return std::max(s.tile_us * k_tiles, n * tile_flops * s.bm * s.bn * k_tiles / (s.tflops * 1e6));
  };
  const long rests = (long)(nt - *whole) * ((M + kHalf.bm - 1) / kHalf.bm);
  return 2.5 + (double)*whole * mt / 256 * round_us(t, 256) + rests / 256 * round_us(kHalf, 256) +
         (rests % 256 ? round_us(kHalf, rests % 256) : 0.0) + (double)M * N * c_bytes / 5e6;
}

// The cheapest shape; with most_parts > parts also the number of partial products (parts, twice that, ..) that go with it.
Plan best_plan(bool f32, int M, int N, int K, int parts, int most_parts, int c_bytes) {
  const Shape* shapes = f32 ? kShapesF32 : kShapes;
  const int count = f32 ? sizeof(kShapesF32) / sizeof(Shape) : sizeof(kShapes) / sizeof(Shape), bk = f32 ? 32 : 64;
  Plan best{0, parts, 0};
  double least = INFINITY;
  for (int p = parts; p <= most_parts; p *= 2) {
    if (p > parts && K / p < (f32 ? 128 : 512)) break;
    for (int i = 0; i < count; ++i) {
      const double us = shape_us(shapes[i], M, N, (double)K / bk, 2.0 * bk, p, c_bytes);
      if (us < least) {
        least = us;
        best = {i, p, 0};
      }
    }
  }
  // (3 % cheaper at least: that far the costs of products whose last round is nearly full were seen to be off)
  if (int whole; !f32 && best.parts == 1 && two_heights_us(M, N, K / 64.0, 2.0 * 64, c_bytes, &whole) < 0.97 * least) best = {0, 1, whole};
  return best;
}

template <typename CT>
hipError_t launch_shape(int shape, const __bf16* a, const __bf16* b, void* c, int M, int N, int K, int ldc, int parts,
                        hipStream_t s) {
  switch (shape) {
    case 0: return launch_tile_t<__bf16, 256, 256, 2, 4, 2, CT>(a, b, c, M, N, K, ldc, parts, s);
    case 1: return launch_tile_t<__bf16, 256, 128, 4, 2, 2, CT>(a, b, c, M, N, K, ldc, parts, s);
    case 2: return launch_tile_t<__bf16, 128, 128, 2, 4, 2, CT>(a, b, c, M, N, K, ldc, parts, s);
    case 3: return launch_tile_t<__bf16, 64, 128, 2, 4, 4, CT>(a, b, c, M, N, K, ldc, parts, s);
    default: return launch_tile_t<__bf16, 64, 64, 2, 2, 4, CT>(a, b, c, M, N, K, ldc, parts, s);
  }
}

// Rows of millions of elements: one shape, with 64-bit offsets
template <typename T, typename CT>
hipError_t launch_far(const T* a, const T* b, void* c, int M, int N, int K, int ldc, int parts, hipStream_t s) {
  return launch_tile_t<T, 64, 64, 2, 2, 4, CT, true>(a, b, c, M, N, K, ldc, parts, s);
}
template <typename T, typename CT>
bool product_near(int K, int ldc) { return rows_near(sizeof(T) * (size_t)K) && results_near(sizeof(CT) * (size_t)ldc); }

// ---------------------------------------------------------------------------------------------
template <typename WT, int kKind, int R, int U>
__global__ __launch_bounds__(kRowThreads) void row_linear_kernel(const RowPrologue p, const WT* __restrict__ w, int N,
                                                                 int Kp, float* __restrict__ y,
                                                                 float* __restrict__ amax_val,
                                                                 int* __restrict__ amax_idx) {
  extern __shared__ __align__(16) float s_x[];  // [Kp]
  __shared__ float s_red[3 * kRowWaves];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int gw = (int)blockIdx.x * kRowWaves + wave, nw = (int)gridDim.x * kRowWaves;
  const int groups = (N + R - 1) / R;
  auto ptr = [&](int g, int r, int k) { return w + (size_t)min(g * R + r, N - 1) * Kp + k; };
  Raw<WT> cur[R][U];
  row_prologue<WT, kKind>(p, Kp, s_x, s_red, [&] {
    __builtin_amdgcn_sched_barrier(0);
    if (gw < groups) fetch_rows<WT, R, U>(cur, gw, 0, Kp, ptr);
    __builtin_amdgcn_sched_barrier(0);
  });
  __syncthreads();

  float best_v = -INFINITY;
  int best_n = 0x7fffffff;
  stream_rows<WT, R, U>(cur, gw, nw, groups, Kp, s_x, ptr, [&](int g, const float (&t)[R]) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int n = g * R + r;
      if (n < N) {
        if (lane == 0) y[n] = t[r];
        if (t[r] > best_v || (t[r] == best_v && n < best_n)) {
          best_v = t[r];
          best_n = n;
        }
      }
    }
  });
  if (amax_val && lane == 0) {
    amax_val[gw] = best_v;
    amax_idx[gw] = best_n;
  }
}

// Rows of W a wavefront takes at a time, and workgroups. One row, so that the rows come out even over the wavefronts that fit at
// once (norm: 85 registers, two workgroups per CU, 512 in all). bf16 [8960][1536] behind a norm: 8.6 us = 3.2 TB/s; four rows
// at a time took 11.0 us: 280 workgroups of which only one fits a CU, so that 24 ran behind the others. [6144][1536]: 7.9 -> 6.8
// us, [4632][1536]: 7.3 -> 6.7. Two rows
//  - between 2048 and 4096 of them, where they make one workgroup per CU and single ones one and a half ([2560][2560] behind a
//    gate: 6.8 us against 7.5 with one, [3584][3584]: 9.3 against 9.9, merged 11.3 against 15.6; [2048][2048]: 5.0 against 4.7);
//  - from 12288 on, where the imbalance is small and half the reductions and reads of the row are saved ([18944][3584]: 26.8 us
//    against 27.5, with four rows 28.8).
// A large head is faster with one workgroup per CU, whose prologues are then half as many ([151936][1536]: 77.2 us = 6.0 TB/s
// against 79.6, with four rows 81.7; [100000][2048]: 70.8 against 73.8, but [65536][1024]: 28.9 against 25.2).
int rows_per_group(int N) { return N >= 12288 || (N > 2048 && N <= 4096) ? 2 : 1; }
int row_grid(int N) {
  const int R = rows_per_group(N), groups = (N + R - 1) / R;
  return std::min((groups + kRowWaves - 1) / kRowWaves, N >= 98304 ? 256 : 512);
}

template <typename WT, int kKind, int R, int U>
hipError_t launch_row_r(const RowPrologue& p, const void* w, int N, int Kp, float* y, float* av, int* ai,
                        hipStream_t s) {
  auto kern = row_linear_kernel<WT, kKind, R, U>;
  const size_t lds = sizeof(float) * (Kp + (kKind == kRowMerge ? (size_t)kPoolAttnSlices * p.heads : 0));
  static LdsLimitOnce raised;
  if (lds > 159 * 1024) return hipErrorInvalidValue;
  if (lds > 60 * 1024)
    if (hipError_t e = raised.raise(reinterpret_cast<const void*>(kern), 159 * 1024); e != hipSuccess) return e;
  hipLaunchKernelGGL(kern, dim3(row_grid(N)), dim3(kRowThreads), lds, s, p, static_cast<const WT*>(w), N, Kp, y, av,
                     ai);
  return hipGetLastError();
}

// A short row is requested whole; of a longer one, six kilobytes at a time (bf16 [1536][8960] behind PolyNorm: 9.2 us, with nine
// 9.7, with three 9.4; f32 [1024][4096]: 7.5 us for four, eight or sixteen).
template <typename WT, int kKind>
hipError_t launch_row_k(const RowPrologue& p, const void* w, int N, int Kp, float* y, float* av, int* ai,
                        hipStream_t s) {
  constexpr int kStep = 64 * Raw<WT>::kE;
  const int steps = (Kp + kStep - 1) / kStep;
  if (rows_per_group(N) == 2)
    return steps <= 3 ? launch_row_r<WT, kKind, 2, 3>(p, w, N, Kp, y, av, ai, s)
                      : launch_row_r<WT, kKind, 2, 4>(p, w, N, Kp, y, av, ai, s);
  if (steps <= 3) return launch_row_r<WT, kKind, 1, 3>(p, w, N, Kp, y, av, ai, s);
  if (steps == 4) return launch_row_r<WT, kKind, 1, 4>(p, w, N, Kp, y, av, ai, s);
  if (steps == 7 || steps == 8) return launch_row_r<WT, kKind, 1, 8>(p, w, N, Kp, y, av, ai, s);
  return launch_row_r<WT, kKind, 1, 6>(p, w, N, Kp, y, av, ai, s);
}

template <typename WT>
hipError_t launch_row_t(int kind, const RowPrologue& p, const void* w, int N, int Kp, float* y, float* av, int* ai,
                        hipStream_t s) {
  switch (kind) {
    case kRowNorm: return launch_row_k<WT, kRowNorm>(p, w, N, Kp, y, av, ai, s);
    case kRowMerge: return launch_row_k<WT, kRowMerge>(p, w, N, Kp, y, av, ai, s);
    case kRowGated: return launch_row_k<WT, kRowGated>(p, w, N, Kp, y, av, ai, s);
    case kRowPoly: return launch_row_k<WT, kRowPoly>(p, w, N, Kp, y, av, ai, s);
    case kRowPlain: return launch_row_k<WT, kRowPlain>(p, w, N, Kp, y, av, ai, s);
    case kRowLoop: return launch_row_k<WT, kRowLoop>(p, w, N, Kp, y, av, ai, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

int matmul_parts(int dtype, int M, int N, int K) {
  int most = 8;  // two always fit what the caller has for them
  while (most > 2 && (size_t)most * M * N > kSplitFloats) most /= 2;
  return best_plan(dtype == W4A32_LAYERED_F32, M, N, K, 1, most, 4).parts;
}

hipError_t launch_matmul_bf16(const void* a, const void* b, void* c, int M, int N, int K, int ldc, bool c_bf16,
                              int parts, hipStream_t s) {
  if (K % kPad != 0 || parts < 1 || parts > K / kPad || (parts > 1 && c_bf16)) return hipErrorInvalidValue;
  const __bf16* pa = static_cast<const __bf16*>(a);
  const __bf16* pb = static_cast<const __bf16*>(b);
  if (c_bf16 && !product_near<__bf16, __bf16>(K, ldc)) return launch_far<__bf16, __bf16>(pa, pb, c, M, N, K, ldc, parts, s);
  if (!c_bf16 && !product_near<__bf16, float>(K, ldc)) return launch_far<__bf16, float>(pa, pb, c, M, N, K, ldc, parts, s);
  const Plan plan = best_plan(false, M, N, K, parts, parts, c_bf16 ? 2 : 4);
  if (plan.whole > 0)
    return c_bf16 ? launch_two_heights<__bf16>(pa, pb, c, M, N, K, ldc, plan.whole, s)
                  : launch_two_heights<float>(pa, pb, c, M, N, K, ldc, plan.whole, s);
  const int shape = plan.shape;
  return c_bf16 ? launch_shape<__bf16>(shape, pa, pb, c, M, N, K, ldc, parts, s)
                : launch_shape<float>(shape, pa, pb, c, M, N, K, ldc, parts, s);
}

hipError_t launch_matmul_f32(const float* a, const float* b, float* c, int M, int N, int K, int parts, hipStream_t s) {
  if (K % 32 != 0 || parts < 1 || parts > K / 32) return hipErrorInvalidValue;
  if (!product_near<float, float>(K, N)) return launch_far<float, float>(a, b, c, M, N, K, N, parts, s);
  switch (best_plan(true, M, N, K, parts, parts, 4).shape) {
    case 0: return launch_tile_t<float, 64, 128, 2, 4, 2, float>(a, b, c, M, N, K, N, parts, s);
    default: return launch_tile_t<float, 64, 64, 2, 2, 4, float>(a, b, c, M, N, K, N, parts, s);
  }
}

int row_linear_partials(int N) { return row_grid(N) * kRowWaves; }
// (the slices' weights of a merged attention row lie behind the row)
bool row_linear_fits(int Kp) { return sizeof(float) * (size_t)Kp <= 140 * 1024; }

hipError_t launch_row_linear(int kind, int dtype, const RowPrologue& pro, const void* w, int N, int Kp, float* y,
                             float* amax_val, int* amax_idx, hipStream_t s) {
  if (!row_linear_fits(Kp)) return hipErrorInvalidValue;
  if (dtype == W4A32_LAYERED_BF16) return launch_row_t<__bf16>(kind, pro, w, N, Kp, y, amax_val, amax_idx, s);
  return launch_row_t<float>(kind, pro, w, N, Kp, y, amax_val, amax_idx, s);
}

}  // namespace w4
