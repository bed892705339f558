// Row operators of the layered decoder's prefill: embedding, layer norm with the input convolution, short
// convolutions with a tail per sequence, PolyNorm, and the rotation table. All bound by HBM.
//
// Convolution tails: a sequence keeps the last inputs of every convolution in a ring of `taps` rows, the row of
// position p in slot p % taps; positions before 0 count as zeros, so a new sequence needs no clearing. In a launch of
// many workgroups only the one that reads the ring (the portion's first tokens) writes it, after its reads.
#include <algorithm>

#include "w4a32_layered.h"
#include "w4a32_layered_kernels.h"

namespace w4 {

namespace {

__global__ __launch_bounds__(256) void fill_zero_kernel(uint4* p, size_t n) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256)
    p[i] = make_uint4(0, 0, 0, 0);
}

template <typename WT>
__global__ __launch_bounds__(256) void embed_rows_kernel(const int64_t* __restrict__ ids, const WT* __restrict__ table,
                                                         float* __restrict__ x, int ld, int vocab) {
  const int64_t id = ids[blockIdx.x];
  const WT* src = table + (size_t)(id < 0 ? 0 : id >= vocab ? vocab - 1 : id) * ld;
  float* dst = x + (size_t)blockIdx.x * ld;
  for (int c = 4 * threadIdx.x; c < ld; c += 1024) store4(dst + c, load4(src + c));
}

// Sums over a workgroup of kWaves wavefronts, in every thread.
template <int kWaves, int N>
__device__ __forceinline__ void workgroup_sums(float (&v)[N], float (*s_part)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i) v[i] = wave_sum64(v[i]);
  __syncthreads();  // s_part of an earlier call
  if ((threadIdx.x & 63) == 0) {
#pragma unroll
    for (int i = 0; i < N; ++i) s_part[threadIdx.x >> 6][i] = v[i];
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < N; ++i) {
    v[i] = 0.0f;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) v[i] += s_part[w][i];
  }
}

// Layer norm (or the norm that takes no mean off) of one row by one wavefront: x + scale * parts -> LDS row s_h (h, zeros past H). The completed residual row goes to
// x_out when that is given. Rows of up to 2048 channels stay in registers on the way.
__device__ __forceinline__ void wave_layer_norm(const float* __restrict__ x, const float* __restrict__ parts,
                                                int n_parts, size_t part_stride, float* __restrict__ x_out,
                                                const float* __restrict__ w, const NormSpec& spec, int H, int ld,
                                                float* __restrict__ s_h) {
  const int lane = threadIdx.x & 63;
  const float inv = 1.0f / (float)H, eps = spec.eps, ps = spec.part_scale;
  auto add = [ps](float4& v, const float4& d) { v.x += ps * d.x; v.y += ps * d.y; v.z += ps * d.z; v.w += ps * d.w; };
  auto clip = [&](float4& v, int c) {
    if (c + 3 >= H) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (c + e >= H) at4(v, e) = 0.0f;
    }
  };
  auto square = [&](float4 v, int c, float mean) {
    float ss = 0.0f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float d = c + e < H ? at4(v, e) - mean : 0.0f;
      ss = __fmaf_rn(d, d, ss);
    }
    return ss;
  };
  constexpr int kRegs = 8;
  if (ld <= 256 * kRegs) {
    // columns past the row are read from its end and count as zeros
    float4 v[kRegs];
#pragma unroll
    for (int i = 0; i < kRegs; ++i) v[i] = load4(x + min(4 * lane + 256 * i, ld - 4));
    float4 ww[kRegs];
#pragma unroll
    for (int i = 0; i < kRegs; ++i) ww[i] = load4(w + min(4 * lane + 256 * i, ld - 4));
#pragma unroll 2
    for (int p = 0; p < n_parts; ++p) {
      float4 d[kRegs];
#pragma unroll
      for (int i = 0; i < kRegs; ++i) d[i] = load4(parts + p * part_stride + min(4 * lane + 256 * i, ld - 4));
#pragma unroll
      for (int i = 0; i < kRegs; ++i) add(v[i], d[i]);
    }
    float sum = 0.0f;
#pragma unroll
    for (int i = 0; i < kRegs; ++i) {
      const int c = 4 * lane + 256 * i;
      clip(v[i], c);
      if (x_out && c < ld) store4(x_out + c, v[i]);
      sum += (v[i].x + v[i].y) + (v[i].z + v[i].w);
    }
    const float mean = spec.rms ? 0.0f : wave_sum64(sum) * inv;
    float ss = 0.0f;
#pragma unroll
    for (int i = 0; i < kRegs; ++i) ss += square(v[i], 4 * lane + 256 * i, mean);
    const float rstd = 1.0f / sqrtf(wave_sum64(ss) * inv + eps);
#pragma unroll
    for (int i = 0; i < kRegs; ++i) {
      const int c = 4 * lane + 256 * i;
      if (c >= ld) continue;
      store4(s_h + c, make_float4((v[i].x - mean) * rstd * ww[i].x, (v[i].y - mean) * rstd * ww[i].y,
                                  (v[i].z - mean) * rstd * ww[i].z, (v[i].w - mean) * rstd * ww[i].w));
    }
    return;
  }
  float sum = 0.0f;
  for (int c = 4 * lane; c < ld; c += 256) {
    float4 v = load4(x + c);
    for (int i = 0; i < n_parts; ++i) add(v, load4(parts + i * part_stride + c));
    clip(v, c);
    if (x_out) store4(x_out + c, v);
    store4(s_h + c, v);
    sum += (v.x + v.y) + (v.z + v.w);
  }
  const float mean = spec.rms ? 0.0f : wave_sum64(sum) * inv;
  float ss = 0.0f;
  for (int c = 4 * lane; c < ld; c += 256) ss += square(load4(s_h + c), c, mean);  // the elements this lane wrote
  const float rstd = 1.0f / sqrtf(wave_sum64(ss) * inv + eps);
  for (int c = 4 * lane; c < ld; c += 256) {
    const float4 v = load4(s_h + c), ww = load4(w + c);
    store4(s_h + c, make_float4((v.x - mean) * rstd * ww.x, (v.y - mean) * rstd * ww.y, (v.z - mean) * rstd * ww.z,
                                (v.w - mean) * rstd * ww.w));
  }
}

constexpr int kNcWaves = 8;

// A workgroup normalises the rows t0 - (TAPS - 1) .. t0 + TR - 1 into LDS, a wavefront per row (rows before the portion
// come from the ring), and convolves its TR rows from there. The first one also leaves the portion's tail in the ring, which no
// other may then read: a portion that has rows in front of it goes in blocks of at least TAPS - 1 rows (kRowsAndTail), or, where
// so many do not fit the LDS, in two launches. (Four taps, 8..100 rows of 1536 in front of position 0 and behind others: 5.8 and 6.4
// us, of 3584 13.7 and 14.6; from 300 rows on blocks are that long anyway.)
enum NormConvPhase { kRowsAndTail, kRowsOnly, kTailOnly };
template <int TAPS, typename YT>
__global__ __launch_bounds__(64 * kNcWaves) void norm_conv_kernel(
    const float* __restrict__ x, const float* __restrict__ parts, int n_parts, float* __restrict__ x_out,
    const float* __restrict__ norm_w, NormSpec spec, const float* __restrict__ conv, float* __restrict__ ring, int M, int H,
    int ld, int pos0, int TR, YT* __restrict__ y, NormConvPhase phase) {
  extern __shared__ __align__(16) float s_h[];  // [halo + TR][ld]
  constexpr int halo = TAPS > 0 ? TAPS - 1 : 0, kRing = TAPS > 0 ? TAPS : 1;
  const int t0 = blockIdx.x * TR, rows = phase == kTailOnly ? 0 : min(TR, M - t0);
  const int wave = threadIdx.x >> 6;
  float4 w[kRing];  // this thread's first columns of the convolution, requested early
#pragma unroll
  for (int j = 0; j < TAPS; ++j) w[j] = load4(conv + (size_t)j * ld + min(4 * (int)threadIdx.x, ld - 4));
  for (int r = wave; r < halo + rows && rows > 0; r += kNcWaves) {
    const int t = t0 - halo + r;
    float* dst = s_h + (size_t)r * ld;
    if (t >= 0) {
      wave_layer_norm(x + (size_t)t * ld, parts + (size_t)t * ld, n_parts, (size_t)M * ld,
                      x_out && r >= halo ? x_out + (size_t)t * ld : nullptr, norm_w, spec, H, ld, dst);
    } else {
      const int q = pos0 + t;
      for (int c = 4 * (threadIdx.x & 63); c < ld; c += 256)
        store4(dst + c, q >= 0 ? load4(ring + (size_t)(q % kRing) * ld + c) : make_float4(0, 0, 0, 0));
    }
  }
  __syncthreads();
  for (int c = 4 * threadIdx.x; c < ld && rows > 0; c += 256 * kNcWaves) {
    float4 win[kRing];  // win[j]: h of the position j before the current one
    if (c >= 256 * kNcWaves) {
#pragma unroll
      for (int j = 0; j < TAPS; ++j) w[j] = load4(conv + (size_t)j * ld + c);
    }
#pragma unroll
    for (int j = 1; j < TAPS; ++j) win[j] = load4(s_h + (size_t)(halo - j) * ld + c);
    for (int r = 0; r < rows; ++r) {
      win[0] = load4(s_h + (size_t)(halo + r) * ld + c);
      float4 v = win[0];
#pragma unroll
      for (int j = TAPS - 1; j >= 0; --j) {
        v.x = __fmaf_rn(w[TAPS - 1 - j].x, win[j].x, v.x);
        v.y = __fmaf_rn(w[TAPS - 1 - j].y, win[j].y, v.y);
        v.z = __fmaf_rn(w[TAPS - 1 - j].z, win[j].z, v.z);
        v.w = __fmaf_rn(w[TAPS - 1 - j].w, win[j].w, v.w);
      }
#pragma unroll
      for (int j = TAPS - 1; j >= 1; --j) win[j] = win[j - 1];
      store4(y + (size_t)(t0 + r) * ld + c, v);
    }
  }
  if (blockIdx.x != 0 || TAPS < 2 || phase == kRowsOnly) return;
  // the tail for the next portion: this workgroup has read the ring, nobody else does
  __syncthreads();
  for (int t = max(0, M - halo) + wave; t < M; t += kNcWaves) {
    // rows past this workgroup's own are normalised once more, into an LDS row in front of its own ones (a wavefront
    // that has one is below `halo`)
    float* row = s_h + (size_t)(halo + t) * ld;
    if (t >= rows) {
      row = s_h + (size_t)wave * ld;
      wave_layer_norm(x + (size_t)t * ld, parts + (size_t)t * ld, n_parts, (size_t)M * ld, nullptr, norm_w, spec, H, ld,
                      row);
    }
    float* dst = ring + (size_t)((pos0 + t) % kRing) * ld;
    for (int c = 4 * (threadIdx.x & 63); c < ld; c += 256) store4(dst + c, load4(row + c));
  }
}
static_assert(kNcWaves >= W4A32_LAYERED_MAX_TAPS - 1, "a wavefront per row of the tail");

// The same for many rows in two launches: statistics (and the completed residual row), then the convolution, whose threads walk
// down the rows with the window in registers. norm_conv_kernel normalises taps - 1 rows for every block of a few again: at
// [2048][3584], four taps and two partial rows it read 220 MB for 88 and took 88 us, these two take 29.
template <int P>
__global__ __launch_bounds__(256) void norm_stats_kernel(const float* __restrict__ x, const float* __restrict__ parts,
                                                         int n_parts, size_t part_stride, float* __restrict__ x_out,
                                                         NormSpec spec, int H, int ld, float2* __restrict__ stats) {
  __shared__ float s_part[4][1];
  const size_t row = (size_t)blockIdx.x * ld;
  float4 v[P];
#pragma unroll
  for (int p = 0; p < P; ++p) v[p] = load4(x + row + min(4 * ((int)threadIdx.x + 256 * p), ld - 4));
#pragma unroll 2
  for (int i = 0; i < n_parts; ++i) {
    float4 d[P];
#pragma unroll
    for (int p = 0; p < P; ++p) d[p] = load4(parts + i * part_stride + row + min(4 * ((int)threadIdx.x + 256 * p), ld - 4));
#pragma unroll
    for (int p = 0; p < P; ++p) {
      v[p].x += spec.part_scale * d[p].x; v[p].y += spec.part_scale * d[p].y;
      v[p].z += spec.part_scale * d[p].z; v[p].w += spec.part_scale * d[p].w;
    }
  }
  float t[1] = {0.0f};
#pragma unroll
  for (int p = 0; p < P; ++p) {
    const int c = 4 * ((int)threadIdx.x + 256 * p);
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (c + e >= H) at4(v[p], e) = 0.0f;
    if (x_out && c < ld) store4(x_out + row + c, v[p]);
    t[0] += (v[p].x + v[p].y) + (v[p].z + v[p].w);
  }
  const float inv = 1.0f / (float)H;
  float mean = 0.0f;
  if (!spec.rms) {
    workgroup_sums<4>(t, s_part);
    mean = t[0] * inv;
  }
  t[0] = 0.0f;
#pragma unroll
  for (int p = 0; p < P; ++p) {
    const int c = 4 * ((int)threadIdx.x + 256 * p);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float d = c + e < H ? at4(v[p], e) - mean : 0.0f;
      t[0] = __fmaf_rn(d, d, t[0]);
    }
  }
  workgroup_sums<4>(t, s_part);
  if (threadIdx.x == 0) stats[blockIdx.x] = make_float2(mean, 1.0f / sqrtf(t[0] * inv + spec.eps));
}

constexpr int kStripRows = 16;
// x: the completed rows (zeros past H). Columns belong to threads: the one that reads a column of the ring writes it.
template <int TAPS, typename YT>
__global__ __launch_bounds__(256) void strip_conv_kernel(const float* __restrict__ x, const float2* __restrict__ stats,
                                                         const float* __restrict__ norm_w, const float* __restrict__ conv,
                                                         float* __restrict__ ring, int M, int H, int ld, int pos0,
                                                         YT* __restrict__ y) {
  const int c = 4 * ((int)blockIdx.x * 256 + (int)threadIdx.x), t0 = blockIdx.y * kStripRows;
  if (c >= ld) return;
  const float4 nw = load4(norm_w + c);
  float4 w[TAPS], win[TAPS];  // win[j]: h of the position j before the current one
#pragma unroll
  for (int j = 0; j < TAPS; ++j) w[j] = load4(conv + (size_t)j * ld + c);
  auto normed = [&](float4 v, float2 st) {
    float4 h, g = nw;
#pragma unroll
    for (int e = 0; e < 4; ++e) at4(h, e) = c + e < H ? (at4(v, e) - st.x) * st.y * at4(g, e) : 0.0f;
    return h;
  };
#pragma unroll
  for (int j = 1; j < TAPS; ++j) {
    const int t = t0 - j, q = pos0 + t;
    if (t >= 0) win[j] = normed(load4(x + (size_t)t * ld + c), stats[t]);
    else win[j] = q >= 0 ? load4(ring + (size_t)(q % TAPS) * ld + c) : make_float4(0, 0, 0, 0);
  }
  constexpr int kAhead = 8;
#pragma unroll
  for (int g = 0; g < kStripRows; g += kAhead) {
    float4 v[kAhead];
#pragma unroll
    for (int i = 0; i < kAhead; ++i) v[i] = load4(x + (size_t)min(t0 + g + i, M - 1) * ld + c);
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      const int t = t0 + g + i;
      if (t >= M) break;
      win[0] = normed(v[i], stats[t]);
      float4 o = win[0];
#pragma unroll
      for (int j = TAPS - 1; j >= 0; --j)
#pragma unroll
        for (int e = 0; e < 4; ++e) at4(o, e) = __fmaf_rn(at4(w[TAPS - 1 - j], e), at4(win[j], e), at4(o, e));
#pragma unroll
      for (int j = TAPS - 1; j >= 1; --j) win[j] = win[j - 1];
      store4(y + (size_t)t * ld + c, o);
    }
  }
  if (blockIdx.y != 0) return;
  for (int t = max(0, M - TAPS + 1); t < M; ++t)
    store4(ring + (size_t)((pos0 + t) % TAPS) * ld + c, normed(load4(x + (size_t)t * ld + c), stats[t]));
}

template <typename YT>
__global__ __launch_bounds__(64) void norm_want_kernel(const float* __restrict__ x, const float* __restrict__ parts,
                                                       int n_parts, const float* __restrict__ norm_w,
                                                       NormSpec spec, const int* __restrict__ want, int M, int H, int ld,
                                                       YT* __restrict__ y) {
  extern __shared__ __align__(16) float s_h[];
  const int t = min(max(want[blockIdx.x], 0), M - 1);
  wave_layer_norm(x + (size_t)t * ld, parts + (size_t)t * ld, n_parts, (size_t)M * ld, nullptr, norm_w, spec, H, ld,
                  s_h);
  for (int c = 4 * threadIdx.x; c < ld; c += 256) store4(y + (size_t)blockIdx.x * ld + c, load4(s_h + c));
}

__global__ __launch_bounds__(256) void add_parts_kernel(const float* x, const float* __restrict__ parts,
                                                        int n_parts, float scale, float* out, size_t n) {
  const size_t i = 4 * ((size_t)blockIdx.x * 256 + threadIdx.x);
  if (i >= n) return;
  float4 v = load4(x + i);
  for (int p = 0; p < n_parts; ++p) {
    const float4 d = load4(parts + p * n + i);
    v.x += scale * d.x; v.y += scale * d.y; v.z += scale * d.z; v.w += scale * d.w;
  }
  store4(out + i, v);
}

template <typename T>
__global__ __launch_bounds__(256) void loop_rows_kernel(const float* __restrict__ x, const float* __restrict__ parts,
                                                        int n_parts, float scale, const int64_t* __restrict__ ids,
                                                        const T* __restrict__ table, int vocab, size_t part_stride,
                                                        int ld, T* __restrict__ y) {
  const size_t row = (size_t)blockIdx.x * ld;
  const int64_t id = ids[blockIdx.x];
  const T* src = table + (size_t)(id < 0 ? 0 : id >= vocab ? vocab - 1 : id) * ld;
  for (int c = 4 * threadIdx.x; c < ld; c += 1024) {
    float4 v = load4(x + row + c);
    for (int p = 0; p < n_parts; ++p) {
      const float4 d = load4(parts + p * part_stride + row + c);
      v.x += scale * d.x; v.y += scale * d.y; v.z += scale * d.z; v.w += scale * d.w;
    }
    store4(y + 2 * row + c, v);
    store4(y + 2 * row + ld + c, load4(src + c));
  }
}

// A row per workgroup, held in registers as it came, P pieces of 16 bytes per thread: the row is read once and the loads are all
// on their way before the first is used. [2048][18944] in bf16, 155 MB: with the row in LDS as f32 (two workgroups per CU, a
// load at a time) 55 us, so 26 us
// (5.9 TB/s); [200][8960]: 7.4 -> 3.6.
// kHalves: bf16 rows that end in half a piece; one check more per piece, 3 % of the time of rows that do not.
template <typename ZT, int kThreads, int P, bool kHalves>
__global__ __launch_bounds__(kThreads) void polynorm_kernel(ZT* __restrict__ z, int F, int ld, const float* __restrict__ act,
                                                            float eps) {
  constexpr int kE = 16 / (int)sizeof(ZT), kWaves = kThreads / 64;
  __shared__ float s_part[kWaves][3];
  // ld is a multiple of four elements: of bf16, rows (and the tensor) start on 8 bytes
  typedef u32x4 Piece __attribute__((aligned(8)));
  typedef uint32_t Half __attribute__((ext_vector_type(2)));
  ZT* row = z + (size_t)blockIdx.x * ld;
  u32x4 raw[P];
#pragma unroll
  for (int p = 0; p < P; ++p) {
    const int c = kE * ((int)threadIdx.x + kThreads * p);
    if constexpr (kHalves) {
      const Half lo = *reinterpret_cast<const Half*>(row + (c < ld ? c : 0));
      const Half hi = *reinterpret_cast<const Half*>(row + (c + 4 < ld ? c + 4 : 0));
      raw[p] = u32x4{lo[0], lo[1], hi[0], hi[1]};
    } else {
      raw[p] = *reinterpret_cast<const Piece*>(row + (c < ld ? c : 0));
    }
  }
  auto get = [](const u32x4& v, int e) __attribute__((always_inline)) {
    if constexpr (sizeof(ZT) == 2) return __uint_as_float(e & 1 ? v[e / 2] & 0xFFFF0000u : v[e / 2] << 16);
    else return __uint_as_float(v[e]);
  };
  float t[3] = {0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int p = 0; p < P; ++p) {
    const int c = kE * ((int)threadIdx.x + kThreads * p);
#pragma unroll
    for (int e = 0; e < kE; ++e) {
      const float x = c + e < F ? get(raw[p], e) : 0.0f, q = x * x;
      t[0] += q;
      t[1] = __fmaf_rn(q, q, t[1]);
      t[2] = __fmaf_rn(q * q, q, t[2]);
    }
  }
  workgroup_sums<kWaves>(t, s_part);
  const float inv = 1.0f / (float)F;
  const float r1 = act[0] / sqrtf(t[0] * inv + eps), r2 = act[1] / sqrtf(t[1] * inv + eps);
  const float r3 = act[2] / sqrtf(t[2] * inv + eps), e0 = act[3];
#pragma unroll
  for (int p = 0; p < P; ++p) {
    const int c = kE * ((int)threadIdx.x + kThreads * p);
    if (c >= ld) continue;
#pragma unroll
    for (int h = 0; h < kE; h += 4) {
      if (kHalves && c + h >= ld) continue;
      float4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float q = get(raw[p], h + e);
        at4(v, e) = c + h + e < F ? q * (r1 + q * (r2 + q * r3)) + e0 : 0.0f;
      }
      store4(row + c + h, v);
    }
  }
}

// One thread per channel and block of kScTok tokens, the last taps - 1 inputs in registers.
constexpr int kScTok = 8;
template <int TAPS>
__global__ __launch_bounds__(256) void short_conv_kernel(const float* __restrict__ x, int ldx, float* __restrict__ y,
                                                         int ldy, const float* __restrict__ w, float* __restrict__ ring,
                                                         int ldw, int channels, int silu, int M, int pos0) {
  const int c = blockIdx.x * 256 + threadIdx.x, t0 = blockIdx.y * kScTok;
  if (c >= channels) return;
  float wt[TAPS], win[TAPS];
#pragma unroll
  for (int j = 0; j < TAPS; ++j) wt[j] = w[(size_t)j * ldw + c];
#pragma unroll
  for (int j = 1; j < TAPS; ++j) {  // win[j]: the input j positions before the current one
    const int t = t0 - j, q = pos0 + t;
    win[j] = t >= 0 ? x[(size_t)t * ldx + c] : q >= 0 ? ring[(size_t)(q % TAPS) * ldw + c] : 0.0f;
  }
  const int te = min(t0 + kScTok, M);
  for (int t = t0; t < te; ++t) {
    win[0] = x[(size_t)t * ldx + c];
    float acc = 0.0f;
#pragma unroll
    for (int j = TAPS - 1; j >= 0; --j) acc = __fmaf_rn(wt[TAPS - 1 - j], win[j], acc);
    y[(size_t)t * ldy + c] = silu ? silu_f(acc) : acc;
#pragma unroll
    for (int j = TAPS - 1; j >= 1; --j) win[j] = win[j - 1];
  }
  if (blockIdx.y == 0) {  // the only block that reads the ring (kScTok >= TAPS - 1)
    for (int t = max(0, M - TAPS + 1); t < M; ++t) ring[(size_t)((pos0 + t) % TAPS) * ldw + c] = x[(size_t)t * ldx + c];
  }
}
static_assert(kScTok >= W4A32_LAYERED_MAX_TAPS - 1, "the second block of tokens must not reach before the portion");

// angle = position * base^(-2 i / dims), in double: a position of many thousands leaves f32 few correct digits
__global__ __launch_bounds__(256) void rot_table_kernel(float* __restrict__ sin_t, float* __restrict__ cos_t,
                                                        int max_pos, int dims, double base) {
  const int half = dims / 2;
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (size_t)max_pos * half) return;
  const int p = (int)(i / half), f = (int)(i % half);
  const double a = (double)p * pow(base, -2.0 * f / dims);
  sin_t[i] = (float)sin(a);
  cos_t[i] = (float)cos(a);
}

constexpr size_t kNcLds = 80 * 1024;  // two workgroups per CU

}  // namespace

hipError_t launch_fill_zero(void* p, size_t bytes, hipStream_t s) {
  const size_t n = bytes / 16;
  hipLaunchKernelGGL(fill_zero_kernel, dim3((unsigned)std::min<size_t>((n + 255) / 256, 8192)), dim3(256), 0, s,
                     static_cast<uint4*>(p), n);
  return hipGetLastError();
}

hipError_t launch_rot_table(float* sin_t, float* cos_t, int max_pos, int dims, double base, hipStream_t s) {
  const size_t n = (size_t)max_pos * (dims / 2);
  hipLaunchKernelGGL(rot_table_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, sin_t, cos_t, max_pos, dims,
                     base);
  return hipGetLastError();
}

hipError_t launch_embed_rows(int dtype, const int64_t* ids, const void* table, int M, int H, int ld, int vocab,
                             float* x, hipStream_t s) {
  (void)H;
  if (dtype == W4A32_LAYERED_BF16) {
    hipLaunchKernelGGL(embed_rows_kernel<__bf16>, dim3(M), dim3(256), 0, s, ids, static_cast<const __bf16*>(table), x,
                       ld, vocab);
  } else {
    hipLaunchKernelGGL(embed_rows_kernel<float>, dim3(M), dim3(256), 0, s, ids, static_cast<const float*>(table), x, ld,
                       vocab);
  }
  return hipGetLastError();
}

static int norm_conv_rows(int M, int ld, int taps) {
  const int halo = taps > 0 ? taps - 1 : 0;
  const int fit = (int)(kNcLds / (sizeof(float) * ld)) - halo;
  const int round = std::max(kNcWaves - halo, 4);  // with its halo, a row per wavefront
  return std::max(1, std::min(std::min(round, (M + 127) / 128), fit));
}

// LDS for the rows and their halo; the tail pass gives every wavefront that has one a row of its own
static size_t norm_conv_lds(int ld, int taps, int rows) {
  const int halo = taps > 0 ? taps - 1 : 0;
  return sizeof(float) * (size_t)ld * (halo + rows);
}

bool norm_conv_fits(int ld, int taps) { return norm_conv_lds(ld, taps, 1) <= 160 * 1024; }

template <int TAPS, typename YT>
static hipError_t norm_conv_t(const float* x, const float* parts, int n_parts, float* x_out, const float* norm_w,
                              const NormSpec& spec, const float* conv, float* ring, int M, int H, int ld, int pos0, YT* y,
                              hipStream_t s) {
  int TR = norm_conv_rows(M, ld, TAPS);
  bool split = false;
  if (constexpr int halo = TAPS > 0 ? TAPS - 1 : 0; pos0 > 0 && TR < halo && TR < M) {
    if (norm_conv_lds(ld, TAPS, halo) <= 160 * 1024) TR = halo;
    else split = true;
  }
  const size_t lds = norm_conv_lds(ld, TAPS, TR);
  auto kern = norm_conv_kernel<TAPS, YT>;
  static LdsLimitOnce raised;
  if (lds > 64 * 1024)
    if (hipError_t e = raised.raise(reinterpret_cast<const void*>(kern), 160 * 1024); e != hipSuccess) return e;
  hipLaunchKernelGGL(kern, dim3((M + TR - 1) / TR), dim3(64 * kNcWaves), lds, s, x, parts, n_parts, x_out, norm_w, spec,
                     conv, ring, M, H, ld, pos0, TR, y, split ? kRowsOnly : kRowsAndTail);
  if (hipError_t e = hipGetLastError(); e != hipSuccess || !split) return e;
  hipLaunchKernelGGL(kern, dim3(1), dim3(64 * kNcWaves), lds, s, x, parts, n_parts, nullptr, norm_w, spec, conv, ring, M, H, ld,
                     pos0, TR, y, kTailOnly);
  return hipGetLastError();
}

template <int TAPS, typename YT>
static hipError_t two_launches_t(const float* x, const float* parts, int n_parts, float* x_out, const float* norm_w,
                                 const NormSpec& spec, const float* conv, float* ring, int M, int H, int ld, int pos0, YT* y,
                                 float2* stats, hipStream_t s) {
  const size_t stride = (size_t)M * ld;
  if (ld <= 4 * 1024)
    hipLaunchKernelGGL(norm_stats_kernel<4>, dim3(M), dim3(256), 0, s, x, parts, n_parts, stride, x_out, spec, H, ld, stats);
  else
    hipLaunchKernelGGL(norm_stats_kernel<8>, dim3(M), dim3(256), 0, s, x, parts, n_parts, stride, x_out, spec, H, ld, stats);
  if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
  hipLaunchKernelGGL((strip_conv_kernel<TAPS, YT>), dim3((ld / 4 + 255) / 256, (M + kStripRows - 1) / kStripRows), dim3(256), 0,
                     s, n_parts > 0 ? x_out : x, stats, norm_w, conv, ring, M, H, ld, pos0, y);
  return hipGetLastError();
}

// Two launches where a row does not fit a wavefront's registers: then norm_conv_kernel reads it from memory several times and few
// rows fit the LDS. us with one and two launches, two partial rows: 2304 channels, 2 / 16 / 64 / 512 / 2048 rows: 14.5, 5.3 / 14.5,
// 10.4 / 14.4, 11.2 / 17.5, 13.9 / 29.7, 22.4; without partial rows 2 / 16 / 64: 9.9, 4.4 / 10.0, 8.3 / 9.9, 8.8; 3584 channels,
// 2 / 64 / 512 / 2048: 20.6, 5.4 / 20.5, 11.4 / 32.0, 15.5 / 88.2, 28.9; 8192, 2 / 64: 42.8, 6.2 / 42.4, 12.5; but 1536 channels, 64 /
// 512 / 2048: 6.9, 10.6 / 8.7, 12.3 / 17.6, 18.1.
static bool two_launches(int ld, int taps) { return taps >= 2 && ld > 2 * 1024 && ld <= 8 * 1024; }

hipError_t launch_norm_conv(const float* x, const float* parts, int n_parts, float* x_out, const float* norm_w,
                            const NormSpec& spec, const float* conv, float* ring, int taps, int M, int H, int ld, int pos0,
                            void* y, bool y_bf16, float2* stats, hipStream_t s) {
  if (!norm_conv_fits(ld, taps)) return hipErrorInvalidValue;
  if (n_parts == 0) x_out = nullptr;  // the residual rows stay where they are
#define W4_NORM_CONV(T)                                                                                            \
  case T:                                                                                                          \
    if constexpr (T >= 2)                                                                                          \
      if (stats && two_launches(ld, T))                                                                         \
        return y_bf16 ? two_launches_t<T>(x, parts, n_parts, x_out, norm_w, spec, conv, ring, M, H, ld, pos0,       \
                                          static_cast<__bf16*>(y), stats, s)                                        \
                      : two_launches_t<T>(x, parts, n_parts, x_out, norm_w, spec, conv, ring, M, H, ld, pos0,       \
                                          static_cast<float*>(y), stats, s);                                        \
    return y_bf16 ? norm_conv_t<T>(x, parts, n_parts, x_out, norm_w, spec, conv, ring, M, H, ld, pos0,              \
                                   static_cast<__bf16*>(y), s)                                                     \
                  : norm_conv_t<T>(x, parts, n_parts, x_out, norm_w, spec, conv, ring, M, H, ld, pos0,              \
                                   static_cast<float*>(y), s)
  switch (taps) {
    W4_NORM_CONV(0); W4_NORM_CONV(1); W4_NORM_CONV(2); W4_NORM_CONV(3); W4_NORM_CONV(4);
    W4_NORM_CONV(5); W4_NORM_CONV(6); W4_NORM_CONV(7); W4_NORM_CONV(8);
    default: return hipErrorInvalidValue;
  }
#undef W4_NORM_CONV
}

hipError_t launch_norm_want(const float* x, const float* parts, int n_parts, const float* norm_w,
                            const NormSpec& spec, const int* want, int n_want, int M, int H, int ld, void* y, bool y_bf16, hipStream_t s) {
  const size_t lds = sizeof(float) * ld;
  if (lds > 160 * 1024) return hipErrorInvalidValue;
  if (y_bf16) {
    static LdsLimitOnce raised;
    if (lds > 64 * 1024)
      if (hipError_t e = raised.raise(reinterpret_cast<const void*>(norm_want_kernel<__bf16>), 160 * 1024);
          e != hipSuccess)
        return e;
    hipLaunchKernelGGL(norm_want_kernel<__bf16>, dim3(n_want), dim3(64), lds, s, x, parts, n_parts, norm_w, spec, want,
                       M, H, ld, static_cast<__bf16*>(y));
  } else {
    static LdsLimitOnce raised;
    if (lds > 64 * 1024)
      if (hipError_t e = raised.raise(reinterpret_cast<const void*>(norm_want_kernel<float>), 160 * 1024);
          e != hipSuccess)
        return e;
    hipLaunchKernelGGL(norm_want_kernel<float>, dim3(n_want), dim3(64), lds, s, x, parts, n_parts, norm_w, spec, want, M,
                       H, ld, static_cast<float*>(y));
  }
  return hipGetLastError();
}

hipError_t launch_loop_rows(int dtype, const float* x, const float* parts, int n_parts, float scale, const int64_t* ids,
                            const void* table, int vocab, int M, int ld, void* y, hipStream_t s) {
  const size_t stride = (size_t)M * ld;
  if (dtype == W4A32_LAYERED_BF16) {
    hipLaunchKernelGGL(loop_rows_kernel<__bf16>, dim3(M), dim3(256), 0, s, x, parts, n_parts, scale, ids,
                       static_cast<const __bf16*>(table), vocab, stride, ld, static_cast<__bf16*>(y));
  } else {
    hipLaunchKernelGGL(loop_rows_kernel<float>, dim3(M), dim3(256), 0, s, x, parts, n_parts, scale, ids,
                       static_cast<const float*>(table), vocab, stride, ld, static_cast<float*>(y));
  }
  return hipGetLastError();
}

hipError_t launch_add_parts(const float* x, const float* parts, int n_parts, float scale, float* out, int M, int ld,
                            hipStream_t s) {
  const size_t n = (size_t)M * ld;
  hipLaunchKernelGGL(add_parts_kernel, dim3((unsigned)((n / 4 + 255) / 256)), dim3(256), 0, s, x, parts, n_parts,
                     scale, out, n);
  return hipGetLastError();
}

bool polynorm_fits(int ld) { return sizeof(float) * (size_t)ld <= 156 * 1024; }

template <typename ZT, bool kHalves = false>
static hipError_t polynorm_t(ZT* z, int M, int F, int ld, const float* act, float eps, hipStream_t s) {
  constexpr int kE = 16 / (int)sizeof(ZT);
  const int pieces = (ld + 512 * kE - 1) / (512 * kE);  // of 512 threads
#define W4_POLY(THREADS, P)                                                                                              \
  do {                                                                                                                  \
    hipLaunchKernelGGL((polynorm_kernel<ZT, THREADS, P, kHalves>), dim3(M), dim3(THREADS), 0, s, z, F, ld, act, eps);    \
    return hipGetLastError();                                                                                           \
  } while (0)
  if (pieces <= 1) W4_POLY(256, 2);
  if (pieces <= 2) W4_POLY(512, 2);
  if (pieces <= 3) W4_POLY(512, 3);
  if (pieces <= 5) W4_POLY(512, 5);
  if (pieces <= 10) W4_POLY(512, 10);
  W4_POLY(512, 20);  // f32 rows of more than 20480; the longest one allowed has 39936
#undef W4_POLY
}

hipError_t launch_polynorm(void* z, bool z_bf16, int M, int F, int ld, const float* act, float eps, hipStream_t s) {
  if (!polynorm_fits(ld)) return hipErrorInvalidValue;
  if (z_bf16 && ld % 8 != 0) return polynorm_t<__bf16, true>(static_cast<__bf16*>(z), M, F, ld, act, eps, s);
  return z_bf16 ? polynorm_t(static_cast<__bf16*>(z), M, F, ld, act, eps, s)
                : polynorm_t(static_cast<float*>(z), M, F, ld, act, eps, s);
}

hipError_t launch_short_conv(const float* x, int ldx, float* y, int ldy, const float* w, float* ring, int ldw, int taps,
                             int channels, bool silu, int M, int pos0, hipStream_t s) {
  const dim3 grid((channels + 255) / 256, (M + kScTok - 1) / kScTok), block(256);
#define W4_SHORT_CONV(T)                                                                                         \
  case T:                                                                                                        \
    hipLaunchKernelGGL(short_conv_kernel<T>, grid, block, 0, s, x, ldx, y, ldy, w, ring, ldw, channels, (int)silu, M, \
                       pos0);                                                                                    \
    break
  switch (taps) {
    W4_SHORT_CONV(1); W4_SHORT_CONV(2); W4_SHORT_CONV(3); W4_SHORT_CONV(4);
    W4_SHORT_CONV(5); W4_SHORT_CONV(6); W4_SHORT_CONV(7); W4_SHORT_CONV(8);
    default: return hipErrorInvalidValue;
  }
#undef W4_SHORT_CONV
  return hipGetLastError();
}

}  // namespace w4
