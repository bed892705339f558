// The tile of C = A B^T that one workgroup computes: WM x WN wavefronts, each with FM x FN accumulators of 32 x 32. bf16
// operands on v_mfma_f32_32x32x16_bf16, f32 operands on v_mfma_f32_32x32x2_f32. The caller says where the rows lie (a buffer and
// a byte offset per row, so they may be gathered; what lies past the buffer's end reads as zeros) and what becomes of the
// accumulators: lane l of a 32 x 32 block holds column l % 32 and, in register v, row 8 (v / 4) + 4 (l / 32) + v % 4. Every shape
// adds the products of an output in the same order.
//
// Tiles of 128 bytes of k (64 in bf16, 32 in f32), brought in through registers (D tiles requested ahead) and double-buffered in
// LDS as rows of 128 + 16 bytes: that stride puts 16 consecutive rows' 16-byte operands on all 64 banks once. What bounds a shape
// in bf16: a wavefront reads FM + FN kilobytes of LDS for FM x FN products of 32 clocks on its SIMD, all four SIMDs share 128 bytes a
// clock, and the tile's own writes come on top. 128 x 128 on four wavefronts needs 768 LDS clocks for 512 clocks of products,
// 256 x 128 on eight 1152 for 1024, 256 x 256 on eight 2048 for 2048 with two wavefronts to a SIMD that fill each other's gaps.
// The order inside a tile is written out and fenced, as the compiler otherwise moves all LDS reads in front of the products:
// behind each product come the next step's fragments, in the first two steps the next tile's way from registers to LDS, in the
// last two the request for a tile D further on. The one barrier per tile stands in front of the last step's products, whose
// fragments are in registers by then, so that the next tile's first fragments are on their way under them.
// [2048][3584] x [14336][3584]: 128 x 128 on four wavefronts without this order 272 us (775 TFLOP/s), with it 235; 256 x 128
// 213, 256 x 256 185 us (1140 TFLOP/s). Its matrix pipes are busy for 84 % of a wavefront's clocks, LDS has no bank conflicts, and
// the rest is the chip's clock under it: a few launches in a row take 172 us (1.6 GHz), twenty or more 215..229 (1.2..1.3 GHz).
// f32 products take eight times as long for the same bytes: a SIMD with one wavefront is busy once its operands are there.
#pragma once

#include <type_traits>

#include "w4a32_layered_kernels.h"

namespace w4 {

// Workgroups are numbered so that one XCD (number mod 8) gets consecutive tiles: XCD x holds tiles / 8 (+ 1 for the first
// tiles % 8 of them). With rows of C fastest a band of B stays in that XCD's L2 while all of A passes.
__device__ __forceinline__ int xcd_tile(int block, int tiles) {
  const int per = tiles / 8, rem = tiles % 8, x = block & 7, i = block >> 3;
  return x * per + min(x, rem) + i;
}

// `bytes` at base as a buffer; loads past its end give zeros. base and bytes are the same in all lanes.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rows_buffer(const void* base, size_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)(unsigned)bytes, 0x00020000);
}
__device__ __forceinline__ u32x4 load16(__amdgpu_buffer_rsrc_t r, unsigned lane_off, unsigned off) {
  return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, lane_off, off, 0));
}

// Rows that lie further apart than a buffer's 32-bit offsets reach within a tile: plain loads, for which every row must be there.
struct FarRows {
  const uint8_t* base;
};
__device__ __forceinline__ u32x4 load16(FarRows r, size_t lane_off, size_t off) {
  return *reinterpret_cast<const u32x4*>(r.base + lane_off + off);
}
template <bool kFar>
__device__ __forceinline__ auto tile_rows_at(const void* base, size_t bytes) {
  if constexpr (kFar) return FarRows{static_cast<const uint8_t*>(base)};
  else return rows_buffer(base, bytes);
}
template <bool kFar>
using RowOffset = std::conditional_t<kFar, size_t, unsigned>;

// Whether a tile of up to 256 rows of `row_bytes` has them within a buffer; of results also with room for what is sent past the
// buffer's end: from kPastEnd, 27 rows further on at most, without coming round to its start.
constexpr unsigned kPastEnd = 0xF0000000u;
inline bool rows_near(size_t row_bytes) { return 256 * row_bytes <= 0xFFFFFFFFu; }
inline bool results_near(size_t row_bytes) { return 28 * row_bytes <= 0xFFFFFFFFu - kPastEnd; }

// A wavefront's operand of a step, and what a pair of them adds to a block of C: k 8 h .. 8 h + 7 of the step's 16 (bf16) from the
// lanes of half h; of the step's 8 (f32) 4 h .. 4 h + 3, of which one product takes one k from each half.
template <typename T>
struct Frag;
template <>
struct Frag<__bf16> {
  bf16x8 v;
  static __device__ __forceinline__ void product(const Frag& a, const Frag& b, f32x16& c) {
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.v, b.v, c, 0, 0, 0);
  }
};
template <>
struct Frag<float> {
  f32x4 v;
  static __device__ __forceinline__ void product(const Frag& a, const Frag& b, f32x16& c) {
#pragma unroll
    for (int e = 0; e < 4; ++e) c = __builtin_amdgcn_mfma_f32_32x32x2f32(a.v[e], b.v[e], c, 0, 0, 0);
  }
};

template <typename T, int BM, int BN, int WM, int WN, int D>
struct MfmaTile {
  static constexpr int kThreads = 64 * WM * WN;
  static constexpr int FM = BM / WM / 32, FN = BN / WN / 32;            // 32 x 32 blocks of a wavefront
  static constexpr int LA = BM * 8 / kThreads, LB = BN * 8 / kThreads;  // 16-byte pieces a thread brings per tile
  static constexpr int kBK = 128 / (int)sizeof(T), kSteps = 4;          // k per LDS tile and steps of its products
  static constexpr int kLd = kBK + 16 / (int)sizeof(T);                 // LDS row, elements
  static constexpr int kE = 16 / (int)sizeof(T);                        // of a piece
  static constexpr size_t kLds = 2 * (BM + BN) * kLd * sizeof(T);
  // the row of A (B) that this thread's piece i is from, and the piece's first byte in it
  static __device__ __forceinline__ int row(int i) { return ((int)threadIdx.x + kThreads * i) >> 3; }
  static __device__ __forceinline__ unsigned column() { return 16 * (threadIdx.x & 7); }

  // acc = rows of A times rows of B over k in [kb, ke), a range of whole tiles that is not empty; a, b: buffers or FarRows; oa, ob:
  // where the pieces' rows start, with column() added
  template <typename Rows, typename Off>
  static __device__ __forceinline__ void run(uint8_t* smem, Rows a, const Off (&oa)[LA], Rows b, const Off (&ob)[LB], int kb,
                                             int ke, f32x16 (&acc)[FM][FN]) {
    T* s_a = reinterpret_cast<T*>(smem);  // [2][BM][kLd]
    T* s_b = s_a + 2 * BM * kLd;          // [2][BN][kLd]
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int wm = (wave / WN) * (BM / WM), wn = (wave % WN) * (BN / WN);
    constexpr int kPieces = LA + LB, kFrags = FM + FN, kProducts = FM * FN;
    u32x4 ra[D][LA], rb[D][LB];
    Frag<T> fa[2][FM], fb[2][FN];
    T* const sa_w = s_a + (tid >> 3) * kLd + kE * (tid & 7);
    T* const sb_w = s_b + (tid >> 3) * kLd + kE * (tid & 7);
    const T* const sa_r = s_a + (wm + (lane & 31)) * kLd + kE * (lane >> 5);
    const T* const sb_r = s_b + (wn + (lane & 31)) * kLd + kE * (lane >> 5);
    auto fetch = [&](int set, int p, int k) __attribute__((always_inline)) {
      if (p < LA) ra[set][p < LA ? p : 0] = load16(a, oa[p < LA ? p : 0], (Off)sizeof(T) * k);
      else rb[set][p < LA ? 0 : p - LA] = load16(b, ob[p < LA ? 0 : p - LA], (Off)sizeof(T) * k);
    };
    auto stash = [&](int set, int p, int buf) __attribute__((always_inline)) {
      if (p < LA) *reinterpret_cast<u32x4*>(sa_w + (buf * BM + kThreads / 8 * p) * kLd) = ra[set][p < LA ? p : 0];
      else *reinterpret_cast<u32x4*>(sb_w + (buf * BN + kThreads / 8 * (p - LA)) * kLd) = rb[set][p < LA ? 0 : p - LA];
    };
    // fragment r of step ks, in the order of their first use: b0, a0, b1, a1, ..
    auto frag = [&](int r, int set, int buf, int ks) __attribute__((always_inline)) {
      constexpr int kPairs = 2 * (FM < FN ? FM : FN);
      const bool of_b = r < kPairs ? (r & 1) == 0 : FN > FM;
      const int i = r < kPairs ? r / 2 : r - kPairs / 2;
      if (of_b) fb[set][i] = *reinterpret_cast<const Frag<T>*>(sb_r + (buf * BN + 32 * i) * kLd + 2 * kE * ks);
      else fa[set][i] = *reinterpret_cast<const Frag<T>*>(sa_r + (buf * BM + 32 * i) * kLd + 2 * kE * ks);
    };
    // every wavefront's LDS traffic so far is done (loads from memory stay on their way)
    auto barrier = [] __attribute__((always_inline)) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
    };
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;

    const int last = ke - kBK;  // a tile past the end is fetched as the last one again and not used
#pragma unroll
    for (int d = 0; d < D; ++d)
#pragma unroll
      for (int p = 0; p < kPieces; ++p) fetch(d, p, min(kb + d * kBK, last));
#pragma unroll
    for (int p = 0; p < kPieces; ++p) stash(0, p, 0);
#pragma unroll
    for (int p = 0; p < kPieces; ++p) fetch(0, p, min(kb + D * kBK, last));
    barrier();
#pragma unroll
    for (int r = 0; r < kFrags; ++r) frag(r, 0, 0, 0);

    // Tile u (of a turn) out of buffer u % 2; the tile behind it goes from register set (u + 1) % D to the other buffer, and the
    // set takes the tile at k.
    auto tile = [&](int u, int k) __attribute__((always_inline)) {
      const int buf = u & 1, set = (u + 1) % D;
#pragma unroll
      for (int ks = 0; ks < kSteps; ++ks) {
        if (ks == kSteps - 1) barrier();
#pragma unroll
        for (int m = 0; m < kProducts; ++m) {
          const int i = m / FN, j = m % FN;
          Frag<T>::product(fa[ks & 1][i], fb[ks & 1][j], acc[i][j]);
          // the fragments are spread over three quarters of the products
          constexpr int kSlots = kProducts < 4 ? 1 : kProducts * 3 / 4;
#pragma unroll
          for (int r = 0; r < kFrags; ++r)
            if (r * kSlots / kFrags == m) {
              if (ks + 1 < kSteps) frag(r, (ks + 1) & 1, buf, ks + 1);
              else frag(r, 0, buf ^ 1, 0);
            }
#pragma unroll
          for (int p = 0; p < kPieces; ++p)
            if (p * 2 * kProducts / kPieces == (ks & 1) * kProducts + m) {
              if (ks < 2) stash(set, p, buf ^ 1);
              else fetch(set, p, k);
            }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    };
    constexpr int kTurn = D;
    static_assert(D % 2 == 0, "buffers and register sets come round together");
    int k = kb;
    for (; k + (kTurn - 1) * kBK < ke; k += kTurn * kBK) {
#pragma unroll
      for (int u = 0; u < kTurn; ++u) tile(u, min(k + (u + 1 + D) * kBK, last));
    }
#pragma unroll
    for (int u = 0; u < kTurn - 1; ++u)  // (not by leaving the loop: its accumulators would be copied)
      if (k + u * kBK < ke) tile(u, last);
  }
};

}  // namespace w4
