// Token mixers with a matrix state S [dim][vdim] per head, f32 throughout:
//   gated delta rule   S <- g S;  u = beta (v - S^T k);  S <- S + k u^T;  o = S^T q
//   retention          S <- decay S + k v^T;  o = S^T q        (the same with u = v and a constant g)
//
// Prefill works on chunks of 64 tokens. With G_i the running sum of log g inside the chunk (all exponents below are
// <= 0) and S the state in front of it:
//   (I + L) U = diag(beta) V - diag(beta e^G) K S,   L_ij = beta_i e^(G_i - G_j) k_i . k_j  for j < i
//   o_i = e^(G_i) S^T q_i + sum_(j <= i) e^(G_i - G_j) (q_i . k_j) u_j
//   S'  = e^(G_last) S + sum_j e^(G_last - G_j) k_j u_j^T
//   rec_chunk_kernel   per (chunk, head), independent of the state: norms / rotation, decays, the two Gram matrices, and
//                      forward substitution for W = -(I + L)^-1 diag(beta e^G) K and U0 = (I + L)^-1 diag(beta) V
//   rec_scan_kernel    per (head, 16 value dimensions), chunk after chunk: U = U0 + W S, then the state
//   rec_out_kernel     per (chunk, head): o, its norm, the gate
// All products are v_mfma_f32_16x16x4_f32. An operand's k index is dealt so that lane group l / 16 of a wavefront owns a
// contiguous quarter of k; the scratch holds every operand in the order of its loads, [16-row block][k / 4 of the
// quarter][lane][4], so that each load of a wavefront is one contiguous kilobyte.
//
// State layout in a sequence's state: transposed, [vdim rounded up to 16][D].
#include <algorithm>
#include <type_traits>

#include "w4a32_layered.h"
#include "w4a32_layered_kernels.h"

namespace w4 {

namespace {

constexpr int kC = 64;  // tokens per chunk

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Scratch of one (head, chunk), floats, all in operand order (matrices as rows x k): q e^G [64 x D],
// k e^(G_last - G) [D x 64], weights [64 x 64], W [64 x D], U [dv16 x 64], state in front of the chunk [dv16 x D]; G_last.
struct ChunkOff {
  size_t q, k, a, w, u, s, g, total;
};
__host__ __device__ inline ChunkOff chunk_off(int D, int dv16) {
  ChunkOff o;
  o.q = 0;
  o.k = o.q + (size_t)kC * D;
  o.a = o.k + (size_t)kC * D;
  o.w = o.a + (size_t)kC * kC;
  o.u = o.w + (size_t)kC * D;
  o.s = o.u + (size_t)kC * dv16;
  o.g = o.s + (size_t)D * dv16;
  o.total = o.g + 64;
  return o;
}
// where operand order keeps elements k .. k + 3 (k % 4 == 0) of a row of a matrix with K columns
template <int K>
__device__ __forceinline__ int op_at(int row, int k) {
  constexpr int KQ = K / 4;
  return (((row >> 4) * (KQ / 4) + (k % KQ) / 4) * 64 + (row & 15) + 16 * (k / KQ)) * 4;
}

// One 16 x 16 block of X Y^T from LDS rows (leading dimension ld), k = 0 .. D - 1.
template <int D>
__device__ __forceinline__ f32x4 gram_block(const float* x, const float* y, int ld) {
  const int lane = threadIdx.x & 63;
  const float* px = x + (lane & 15) * ld + (D / 4) * (lane >> 4);
  const float* py = y + (lane & 15) * ld + (D / 4) * (lane >> 4);
  f32x4 a0 = {0, 0, 0, 0}, a1 = {0, 0, 0, 0};
#pragma unroll 4
  for (int s = 0; s < D / 4; s += 4) {
    const float4 u = load4(px + s), v = load4(py + s);
    a0 = mfma4(u.x, v.x, a0);
    a1 = mfma4(u.y, v.y, a1);
    a0 = mfma4(u.z, v.z, a0);
    a1 = mfma4(u.w, v.w, a1);
  }
  return a0 + a1;
}

// LDS of the chunk kernel: k and q rows; the delta rule's L and later W take the q and k rows' place
template <int D>
constexpr size_t chunk_lds() {
  return sizeof(float) * (2 * kC * (D + 4) + 3 * kC) + (D + 4 < kC + 4 ? sizeof(float) * kC * (kC - D) : 0);
}

// grid (chunks, heads), 256 threads
template <int D, bool kDelta>
__global__ __launch_bounds__(256) void rec_chunk_kernel(const RecGeom g, const float* __restrict__ raw,
                                                        const float* __restrict__ cx, int ldcx,
                                                        float* __restrict__ scratch, int M, int pos0, int vec) {
  constexpr int kLdk = D + 4, kLdl = kC + 4;
  extern __shared__ __align__(16) float sm[];
  float* s_g = sm;                      // [64] running log decay
  float* s_b = s_g + kC;                // [64] beta
  float* s_e = s_b + kC;                // [64] e^(running log decay)
  float* s_k = s_e + kC;                // [64][kLdk]
  float* s_q = s_k + kC * kLdk;         // [64][kLdk]
  float* s_l = s_q;                     // [64][kLdl], once the q rows are done with
  const int chunk = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int t0 = chunk * kC, n = min(kC, M - t0);
  const int hk = h / (g.heads / g.kv_heads);
  const int dv16 = (g.vdim + 15) & ~15;
  const ChunkOff off = chunk_off(D, dv16);
  float* out = scratch + ((size_t)h * gridDim.x + chunk) * off.total;
  const float qk_scale = rsqrtf((float)g.dim);

  // rows of q and k: four threads per token
  {
    const int i = tid >> 2, part = tid & 3;
    const bool on = i < n;
    const int ti = t0 + (on ? i : 0);
    const float* src = kDelta ? cx + (size_t)ti * ldcx : raw + (size_t)ti * g.ldr;
    const float* qs = src + g.q_off + hk * g.dim;
    const float* ks = src + g.k_off + hk * g.dim;
    const int half = g.rot_dims / 2;
    const float* st = kDelta ? nullptr : g.sin_t + (size_t)(pos0 + ti) * half;
    const float* ct = kDelta ? nullptr : g.cos_t + (size_t)(pos0 + ti) * half;
    float sq = 0.0f, sk = 0.0f;
    float* dq = s_q + i * kLdk;
    float* dk = s_k + i * kLdk;
    if (vec) {  // four elements at a time
#pragma unroll 4
      for (int d = 4 * part; d < D; d += 16) {
        float4 q = make_float4(0, 0, 0, 0), k = q;
        if (on && d < g.dim) {
          q = load4(qs + d);
          k = load4(ks + d);
          if constexpr (!kDelta) {
            if (d < g.rot_dims) {
              const bool lower = d < half;
              const int f = lower ? d : d - half, other = lower ? d + half : d - half;
              const float4 qo = load4(qs + other), ko = load4(ks + other), c = load4(ct + f);
              float4 s = load4(st + f);
              if (lower) s = make_float4(-s.x, -s.y, -s.z, -s.w);
              q = make_float4(q.x * c.x + qo.x * s.x, q.y * c.y + qo.y * s.y, q.z * c.z + qo.z * s.z,
                              q.w * c.w + qo.w * s.w);
              k = make_float4(k.x * c.x + ko.x * s.x, k.y * c.y + ko.y * s.y, k.z * c.z + ko.z * s.z,
                              k.w * c.w + ko.w * s.w);
            }
            k = make_float4(k.x * qk_scale, k.y * qk_scale, k.z * qk_scale, k.w * qk_scale);
          }
        }
        store4(dq + d, q);
        store4(dk + d, k);
        sq += (q.x * q.x + q.y * q.y) + (q.z * q.z + q.w * q.w);
        sk += (k.x * k.x + k.y * k.y) + (k.z * k.z + k.w * k.w);
      }
    } else {
      for (int d = part; d < D; d += 4) {
        float q = 0.0f, k = 0.0f;
        if (on && d < g.dim) {
          q = qs[d];
          k = ks[d];
          if constexpr (!kDelta) {
            if (d < g.rot_dims) {
              const int f = d < half ? d : d - half, other = d < half ? d + half : d - half;
              const float c = ct[f], s = d < half ? -st[f] : st[f];
              q = q * c + qs[other] * s;
              k = k * c + ks[other] * s;
            }
            k *= qk_scale;
          }
        }
        dq[d] = q;
        dk[d] = k;
        sq = __fmaf_rn(q, q, sq);
        sk = __fmaf_rn(k, k, sk);
      }
    }
    if constexpr (kDelta) {
      sq += __shfl_xor(sq, 1, 64);
      sk += __shfl_xor(sk, 1, 64);
      sq += __shfl_xor(sq, 2, 64);
      sk += __shfl_xor(sk, 2, 64);
      const float rq = qk_scale / sqrtf(sq + 1e-6f), rk = 1.0f / sqrtf(sk + 1e-6f);
      const int step = vec ? 16 : 4;  // the elements this thread wrote
      for (int d = vec ? 4 * part : part; d < D; d += step) {
        for (int e = 0; e < step / 4; ++e) {
          dq[d + e] *= rq;
          dk[d + e] *= rk;
        }
      }
    }
  }
  // decays: one lane per token, tokens past the end leave the state alone
  if (wave == 0) {
    float lg = 0.0f, beta = 0.0f;
    if (lane < n) {
      if constexpr (kDelta) {
        const float* row = raw + (size_t)(t0 + lane) * g.ldr;
        lg = -expf(g.a_log[h]) * softplus_f(row[g.a_off + h] + g.dt_bias[h]);
        beta = sigmoid_f(row[g.b_off + h]);
      } else {
        lg = g.log_decay[h];
      }
    }
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const float up = __shfl_up(lg, o, 64);
      if (lane >= o) lg += up;
    }
    s_g[lane] = lg;
    s_b[lane] = beta;
    s_e[lane] = expf(lg);
    if (lane == 63) out[off.g] = lg;
  }
  // retention: U = V
  if constexpr (!kDelta) {
    for (int it = tid; it < (kC / 4) * dv16; it += 256) {
      const int d = it % dv16, t = 4 * (it / dv16);
      const float* vs = raw + (size_t)t0 * g.ldr + g.v_off + h * g.vdim + d;
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = d < g.vdim && t + e < n ? vs[(size_t)(t + e) * g.ldr] : 0.0f;
      store4(out + off.u + op_at<kC>(d, t), make_float4(v[0], v[1], v[2], v[3]));
    }
  }
  __syncthreads();

  // A = masked, decayed Q K^T; L likewise from K K^T: the blocks on and below the diagonal, dealt to the wavefronts
  constexpr int kTri = 10, kTasks = kDelta ? 2 * kTri : kTri, kMine = (kTasks + 3) / 4;
  f32x4 tile[kMine];
  auto task_of = [&](int t, int& it, int& jt) {  // t-th block of the lower triangle
    it = t >= 6 ? 3 : t >= 3 ? 2 : t >= 1 ? 1 : 0;
    jt = t - it * (it + 1) / 2;
  };
#pragma unroll
  for (int m = 0; m < kMine; ++m) {
    const int t = wave + 4 * m;
    tile[m] = f32x4{0, 0, 0, 0};
    if (t < kTasks) {
      int it, jt;
      task_of(t % kTri, it, jt);
      tile[m] = gram_block<D>((t < kTri ? s_q : s_k) + 16 * it * kLdk, s_k + 16 * jt * kLdk, kLdk);
    }
  }
  // q e^G and k e^(G_last - G)
  for (int u = tid; u < kC * D / 4; u += 256) {
    const int i = u & 63, d = 4 * (u >> 6);  // a wavefront: 64 rows of one k
    const float4 q = load4(s_q + i * kLdk + d);
    const float e = s_e[i];
    store4(out + off.q + op_at<D>(i, d), make_float4(q.x * e, q.y * e, q.z * e, q.w * e));
  }
  {
    const int t = 4 * (tid & 15);
    float w[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) w[e] = expf(s_g[kC - 1] - s_g[t + e]);
    for (int d = tid >> 4; d < D; d += 16) {
      store4(out + off.k + op_at<kC>(d, t),
             make_float4(s_k[t * kLdk + d] * w[0], s_k[(t + 1) * kLdk + d] * w[1], s_k[(t + 2) * kLdk + d] * w[2],
                         s_k[(t + 3) * kLdk + d] * w[3]));
    }
  }
  // the part of A above the diagonal blocks is zero
  for (int u = tid; u < 6 * 64; u += 256) {
    const int b = u >> 6, it = b >= 5 ? 2 : b >= 3 ? 1 : 0, jt = b >= 5 ? 3 : b >= 3 ? b - 1 : b + 1;
    const int i = 16 * it + (u & 15), j = 16 * jt + 4 * ((u >> 4) & 3);
    store4(out + off.a + op_at<kC>(i, j), make_float4(0, 0, 0, 0));
  }
  __syncthreads();  // nobody reads the q rows any more
#pragma unroll
  for (int m = 0; m < kMine; ++m) {
    const int t = wave + 4 * m;
    if (t >= kTasks) continue;
    int it, jt;
    task_of(t % kTri, it, jt);
    const int i0 = 16 * it + 4 * (lane >> 4), j = 16 * jt + (lane & 15);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = i0 + r;
      const float e = j <= i ? expf(s_g[i] - s_g[j]) : 0.0f;
      if (t < kTri) out[off.a + op_at<kC>(i, j & ~3) + (j & 3)] = tile[m][r] * e;
      else s_l[i * kLdl + j] = j < i ? tile[m][r] * e * s_b[i] : 0.0f;
    }
  }
  if constexpr (!kDelta) return;
  __syncthreads();

  // forward substitution, one column of the right-hand side per thread: D columns of diag(beta e^G) K, then V's
  for (int c0 = 0; c0 < D + dv16; c0 += 256) {
    const int c = c0 + tid;
    float x[kC];
    const bool is_k = c < D, is_v = !is_k && c < D + dv16;
    const int d = is_k ? c : c - D;
    if (is_k) {
#pragma unroll
      for (int i = 0; i < kC; ++i) x[i] = s_k[i * kLdk + d] * (s_e[i] * s_b[i]);
    } else {
      const bool on = is_v && d < g.vdim;
      const float* vs = cx + (size_t)t0 * ldcx + g.v_off + h * g.vdim + (on ? d : 0);
      // (beta is 0 from token n on)
#pragma unroll
      for (int i = 0; i < kC; ++i) x[i] = vs[(size_t)min(i, n - 1) * ldcx];
#pragma unroll
      for (int i = 0; i < kC; ++i) x[i] = on ? x[i] * s_b[i] : 0.0f;
    }
#pragma unroll
    for (int i = 1; i < kC; ++i) {
#pragma unroll
      for (int j = 0; j < i; j += 4) {
        const float4 l = load4(s_l + i * kLdl + j);  // zero from column i on
        x[i] = __fmaf_rn(-l.x, x[j], x[i]);
        if (j + 1 < i) x[i] = __fmaf_rn(-l.y, x[j + 1], x[i]);
        if (j + 2 < i) x[i] = __fmaf_rn(-l.z, x[j + 2], x[i]);
        if (j + 3 < i) x[i] = __fmaf_rn(-l.w, x[j + 3], x[i]);
      }
    }
    if (is_v) {
#pragma unroll
      for (int i = 0; i < kC; i += 4)
        store4(out + off.u + op_at<kC>(d, i), make_float4(x[i], x[i + 1], x[i + 2], x[i + 3]));
    }
    if (is_k) {  // W into the k rows' place: nobody else reads this column
#pragma unroll
      for (int i = 0; i < kC; ++i) s_k[i * kLdk + d] = -x[i];
    }
  }
  __syncthreads();
  for (int u = tid; u < kC * D / 4; u += 256) {
    const int i = u & 63, d = 4 * (u >> 6);
    store4(out + off.w + op_at<D>(i, d), load4(s_k + i * kLdk + d));
  }
}

// 256 threads. Wavefront w: tokens 16 w .. of U, and the state's rows (key dimensions) in blocks of 16, NB blocks per
// wavefront. Grid (8, dv16 / 16, ceil(heads / 8)), the first dimension the XCD that consecutive workgroups alternate over: a
// head's workgroups all read its W and K, so they share an XCD's L2. (28 heads of 128 x 128, 32 chunks: retention 45.4 -> 38.3 us, delta
// rule 88.6 -> 86.5, which is bound by its chain: two products with an exchange through LDS behind each, 2.7 us per chunk.)
template <int D, bool kDelta>
__global__ __launch_bounds__(256) void rec_scan_kernel(float* __restrict__ state, float* __restrict__ scratch, int heads,
                                                       int dv16, int chunks, int fresh) {
  constexpr int KQ = D / 4;                          // a lane group's share of k over key dimensions
  constexpr int NB = D >= 64 ? D / 64 : 1;
  constexpr int kGs = KQ * 16 + 16, kGu = 16 * 16 + 16;  // LDS words of a lane group's share (padded)
  __shared__ __align__(16) float s_s[4 * kGs], s_u[4 * kGu];
  const int n0 = 16 * blockIdx.y, h = blockIdx.x + 8 * blockIdx.z, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  if (h >= heads) return;
  const int col = lane & 15, grp = lane >> 4;
  const ChunkOff off = chunk_off(D, dv16);
  float* base = scratch + (size_t)h * chunks * off.total;
  float* st = state + ((size_t)h * dv16 + n0 + col) * D + 4 * grp;  // + 16 * block
  const bool rows_on = D >= 64 || wave < D / 16;

  f32x4 s[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    s[b] = f32x4{0, 0, 0, 0};
    if (!fresh && rows_on) {
      const float4 v = load4(st + 16 * (wave * NB + b));
      s[b] = f32x4{v.x, v.y, v.z, v.w};
    }
  }
  auto publish = [&]() {  // the state's rows to LDS: row d at [d / KQ][d % KQ][col]
    if (!rows_on) return;
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int d = 16 * (wave * NB + b) + 4 * grp + r;
        s_s[(d / KQ) * kGs + (d % KQ) * 16 + col] = s[b][r];
      }
  };
  struct Ops {
    f32x4 w[KQ / 4], k[NB][4], u;
    float gl;
  };
  auto ld = [](const float* p) { return *reinterpret_cast<const f32x4*>(p); };
  auto fetch = [&](int c, Ops& o) __attribute__((always_inline)) {
    const float* p = base + (size_t)min(c, chunks - 1) * off.total;
    if constexpr (kDelta) {
#pragma unroll
      for (int i = 0; i < KQ / 4; ++i) o.w[i] = ld(p + off.w + ((wave * (KQ / 4) + i) * 64 + lane) * 4);
    }
    o.u = ld(p + off.u + op_at<kC>(n0 + col, 16 * wave + 4 * grp));
    if (rows_on) {
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int i = 0; i < 4; ++i) o.k[b][i] = ld(p + off.k + (((wave * NB + b) * 4 + i) * 64 + lane) * 4);
    }
    o.gl = p[off.g];
  };
  auto advance = [&](int c, const Ops& o) __attribute__((always_inline)) {
    float* p = base + (size_t)c * off.total;
    f32x4 acc = o.u;
    if constexpr (kDelta) {
      f32x4 acc1 = {0, 0, 0, 0};
      const float* ps = s_s + grp * kGs + col;
#pragma unroll
      for (int i = 0; i < KQ / 4; ++i) {
        acc = mfma4(o.w[i][0], ps[(4 * i) * 16], acc);
        acc1 = mfma4(o.w[i][1], ps[(4 * i + 1) * 16], acc1);
        acc = mfma4(o.w[i][2], ps[(4 * i + 2) * 16], acc);
        acc1 = mfma4(o.w[i][3], ps[(4 * i + 3) * 16], acc1);
      }
      acc = acc + acc1;
      *reinterpret_cast<f32x4*>(p + off.u + op_at<kC>(n0 + col, 16 * wave + 4 * grp)) = acc;
    }
    // token 16 wave + 4 grp + r is entry (wave, 4 grp + r): its k group is this wavefront's number
#pragma unroll
    for (int r = 0; r < 4; ++r) s_u[wave * kGu + (4 * grp + r) * 16 + col] = acc[r];
    const float decay = expf(o.gl);
    if (rows_on) {
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        *reinterpret_cast<f32x4*>(p + off.s + op_at<D>(n0 + col, 16 * (wave * NB + b) + 4 * grp)) = s[b];
        s[b] *= decay;
      }
    }
    __syncthreads();  // U is complete, and nobody reads the old state any more
    if (rows_on) {
      const float* pu = s_u + grp * kGu + col;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float u0 = pu[(4 * i) * 16], u1 = pu[(4 * i + 1) * 16], u2 = pu[(4 * i + 2) * 16], u3 = pu[(4 * i + 3) * 16];
#pragma unroll
        for (int b = 0; b < NB; ++b) s[b] = mfma4(o.k[b][i][0], u0, s[b]);
#pragma unroll
        for (int b = 0; b < NB; ++b) s[b] = mfma4(o.k[b][i][1], u1, s[b]);
#pragma unroll
        for (int b = 0; b < NB; ++b) s[b] = mfma4(o.k[b][i][2], u2, s[b]);
#pragma unroll
        for (int b = 0; b < NB; ++b) s[b] = mfma4(o.k[b][i][3], u3, s[b]);
      }
    }
    publish();
    __syncthreads();
  };
  // two register sets: a chunk's operands are requested while the one before it runs
  Ops o0, o1;
  fetch(0, o0);
  publish();
  __syncthreads();
  for (int c = 0; c < chunks; c += 2) {
    fetch(c + 1, o1);
    advance(c, o0);
    if (c + 1 >= chunks) break;
    fetch(c + 2, o0);
    advance(c + 1, o1);
  }
  if (rows_on) {
#pragma unroll
    for (int b = 0; b < NB; ++b)
      store4(st + 16 * (wave * NB + b), make_float4(s[b][0], s[b][1], s[b][2], s[b][3]));
  }
}

// grid (chunks, heads), 256 threads; wavefront w: tokens 16 w .. The operands of 16 value dimensions are D / 16 + 4 kilobytes of state and
// U. With kShared they come through LDS once for all four wavefronts, the next ones meanwhile through registers; without it each wavefront
// reads them for itself, into two sets of registers in turn: the same bits, without a barrier and an LDS round trip per step, which nothing
// hides where a workgroup has its CU to itself. 28 heads of 128 x 128 in 32 chunks (129 MB of scratch: 26 us at the rate of a copy) take 45 us
// with kShared, 61 without. (out_shared() says which is launched.)
template <int D, typename T, bool kShared>
__global__ __launch_bounds__(256, !kShared ? 1 : D <= 128 ? 4 : 2) void rec_out_kernel(const RecGeom g, const float* __restrict__ raw,
                                                                                       const float* __restrict__ scratch,
                                                                                       T* __restrict__ out, int ldo, int M) {
  constexpr int KQ = D / 4, NT = D / 16, kPieces = KQ / 4 + 4;
  const int chunk = blockIdx.x, h = blockIdx.y, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int col = lane & 15, grp = lane >> 4;
  const int dv16 = (g.vdim + 15) & ~15;
  const ChunkOff off = chunk_off(D, dv16);
  const float* p = scratch + ((size_t)h * gridDim.x + chunk) * off.total;
  auto ld = [](const float* p) { return *reinterpret_cast<const f32x4*>(p); };
  f32x4 q[KQ / 4], a[4];
  auto fetch_rows = [&] __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < KQ / 4; ++i) q[i] = ld(p + off.q + ((wave * (KQ / 4) + i) * 64 + lane) * 4);
#pragma unroll
    for (int i = 0; i < 4; ++i) a[i] = ld(p + off.a + ((wave * 4 + i) * 64 + lane) * 4);
  };
  f32x4 o[NT];
  float ss[4] = {0, 0, 0, 0};
  auto multiply = [&](auto piece) __attribute__((always_inline)) {
    f32x4 o0 = {0, 0, 0, 0}, o1 = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < kPieces; ++i) {
      const f32x4 x = i < KQ / 4 ? q[i < KQ / 4 ? i : 0] : a[i < KQ / 4 ? 0 : i - KQ / 4], y = piece(i);
      o0 = mfma4(x[0], y[0], o0);
      o1 = mfma4(x[1], y[1], o1);
      o0 = mfma4(x[2], y[2], o0);
      o1 = mfma4(x[3], y[3], o1);
    }
    return o0 + o1;
  };
  auto keep_sum = [&](int nt) __attribute__((always_inline)) {
    const float keep = 16 * nt + col < g.vdim ? 1.0f : 0.0f;
#pragma unroll
    for (int r = 0; r < 4; ++r) ss[r] = __fmaf_rn(o[nt][r] * keep, o[nt][r], ss[r]);
  };

  if constexpr (kShared) {
    constexpr int kPer = (kPieces + 3) / 4;
    __shared__ f32x4 s_op[2][kPieces][64];
    f32x4 piece[kPer];
    auto fetch = [&](int nt) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < kPer; ++i) {
        const int t = min(nt, dv16 / 16 - 1), n = min(wave + 4 * i, kPieces - 1);
        const float* src = n < KQ / 4 ? p + off.s + (size_t)(t * (KQ / 4) + n) * 256 : p + off.u + (size_t)(t * 4 + n - KQ / 4) * 256;
        piece[i] = ld(src + 4 * lane);
      }
    };
    auto stash = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < kPer; ++i)
        if (kPieces % 4 == 0 || wave + 4 * i < kPieces) s_op[buf][wave + 4 * i][lane] = piece[i];
    };
    fetch(0);
    fetch_rows();
    stash(0);
    fetch(1);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      if (16 * nt >= dv16) break;
      // what every wavefront has written and read in LDS so far is done; loads from memory stay on their way
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      const f32x4 sum = multiply([&](int i) { return s_op[nt & 1][i][lane]; });
      if (nt + 1 < NT) {
        stash((nt + 1) & 1);
        if (nt + 2 < NT) fetch(nt + 2);
      }
      o[nt] = sum;
      keep_sum(nt);
    }
  } else {
    f32x4 ops0[kPieces], ops1[kPieces];
    auto fetch = [&](int nt, f32x4(&ops)[kPieces]) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < kPieces; ++i) {
        const int t = min(nt, dv16 / 16 - 1);
        ops[i] = i < KQ / 4 ? ld(p + off.s + ((t * (KQ / 4) + i) * 64 + lane) * 4) : ld(p + off.u + ((t * 4 + i - KQ / 4) * 64 + lane) * 4);
      }
    };
    auto step = [&](int nt, const f32x4(&ops)[kPieces]) __attribute__((always_inline)) {
      o[nt] = multiply([&](int i) { return ops[i]; });
      keep_sum(nt);
    };
    fetch_rows();
    fetch(0, ops0);
#pragma unroll
    for (int nt = 0; nt < NT; nt += 2) {
      if (16 * nt < dv16) {
        fetch(nt + 1, ops1);
        step(nt, ops0);
      }
      if (16 * (nt + 1) < dv16) {
        fetch(nt + 2, ops0);
        step(nt + 1, ops1);
      }
    }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
#pragma unroll
    for (int x = 8; x >= 1; x >>= 1) ss[r] += __shfl_xor(ss[r], x, 64);
    ss[r] = 1.0f / sqrtf(ss[r] / (float)g.vdim + g.eps);
  }
  float gate[4][NT], w[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const int d = min(16 * nt + col, g.vdim - 1);
    w[nt] = g.head_norm ? g.head_norm[d] : 1.0f;
#pragma unroll
    for (int r = 0; r < 4; ++r)
      gate[r][nt] = raw[(size_t)min(chunk * kC + 16 * wave + 4 * grp + r, M - 1) * g.ldr + g.gate_off + h * g.vdim + d];
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int t = chunk * kC + 16 * wave + 4 * grp + r;
    if (t >= M) continue;
    T* row = out + (size_t)t * ldo;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const int d = 16 * nt + col;
      if (d < g.vdim) row[h * g.vdim + d] = (T)(o[nt][r] * ss[r] * w[nt] * silu_f(gate[r][nt]));
    }
    if (h == g.heads - 1)
      for (int c = g.heads * g.vdim + col; c < ldo; c += 16) row[c] = (T)0.0f;
  }
}

// One token. grid (dv16 / 16, heads), 256 threads: a wavefront takes four value rows of the state, D / 64 key
// dimensions per lane. o = g (S^T q) + (k . q) u needs S once: both products with the old state in one pass.
template <int D, bool kDelta>
__global__ __launch_bounds__(256) void rec_decode_kernel(const RecGeom g, const float* __restrict__ raw,
                                                         const float* __restrict__ conv, float* __restrict__ ring,
                                                         float* __restrict__ state, const int* __restrict__ d_pos,
                                                         float* __restrict__ o) {
  constexpr int E = D >= 64 ? D / 64 : 1;
  __shared__ __align__(16) float s_q[D], s_k[D], s_v[16];
  const int n0 = 16 * blockIdx.x, h = blockIdx.y, tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int rep = g.heads / g.kv_heads, hk = h / rep;
  const int dv16 = (g.vdim + 15) & ~15;
  const int pos = *d_pos;
  // the state's rows are requested first
  float s[4][E];
  float* rows = state + ((size_t)h * dv16 + n0 + 4 * wave) * D + E * lane;
  const bool on = E * lane < D;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int e = 0; e < E; ++e) s[i][e] = on && pos > 0 ? rows[(size_t)i * D + e] : 0.0f;

  const float qk_scale = rsqrtf((float)g.dim);
  for (int it = tid; it < 2 * D + 16; it += 256) {
    const bool is_v = it >= 2 * D;
    const int d = is_v ? n0 + it - 2 * D : it % D;
    float y = 0.0f;
    if (d < (is_v ? g.vdim : g.dim)) {
      const int c = is_v ? g.v_off + h * g.vdim + d : (it < D ? g.q_off : g.k_off) + hk * g.dim + d;
      y = raw[c];
      if constexpr (kDelta) {
        const float x = y;
        y = silu_f(conv_step(x, conv, ring, c, g.ldc, g.taps, pos));
        // one workgroup per channel keeps the tail (nobody reads this slot now)
        if (is_v || (blockIdx.x == 0 && h % rep == 0)) ring[(size_t)(pos % g.taps) * g.ldc + c] = x;
      } else if (!is_v) {
        if (d < g.rot_dims) {
          const int half = g.rot_dims / 2, f = d < half ? d : d - half, other = d < half ? c + half : c - half;
          const size_t at = (size_t)min(pos, g.rot_rows - 1) * half + f;
          const float cs = g.cos_t[at], sn = g.sin_t[at];
          y = y * cs + raw[other] * (d < half ? -sn : sn);
        }
        if (it >= D) y *= qk_scale;
      }
    }
    (is_v ? s_v[it - 2 * D] : it < D ? s_q[d] : s_k[d]) = y;
  }
  float decay, beta = 1.0f;
  if constexpr (kDelta) {
    decay = expf(-expf(g.a_log[h]) * softplus_f(raw[g.a_off + h] + g.dt_bias[h]));
    beta = sigmoid_f(raw[g.b_off + h]);
  } else {
    decay = g.decay[h];
  }
  __syncthreads();
  float q[E], k[E], sq = 0.0f, sk = 0.0f, kq = 0.0f;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    q[e] = on ? s_q[E * lane + e] : 0.0f;
    k[e] = on ? s_k[E * lane + e] : 0.0f;
    sq = __fmaf_rn(q[e], q[e], sq);
    sk = __fmaf_rn(k[e], k[e], sk);
  }
  if constexpr (kDelta) {
    const float rq = qk_scale / sqrtf(wave_sum64(sq) + 1e-6f), rk = 1.0f / sqrtf(wave_sum64(sk) + 1e-6f);
#pragma unroll
    for (int e = 0; e < E; ++e) {
      q[e] *= rq;
      k[e] *= rk;
    }
  }
#pragma unroll
  for (int e = 0; e < E; ++e) kq = __fmaf_rn(q[e], k[e], kq);
  kq = wave_sum64(kq);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int d = n0 + 4 * wave + i;
    float dk = 0.0f, dq = 0.0f;
#pragma unroll
    for (int e = 0; e < E; ++e) {
      s[i][e] *= decay;
      if (kDelta) dk = __fmaf_rn(s[i][e], k[e], dk);
      dq = __fmaf_rn(s[i][e], q[e], dq);
    }
    dq = wave_sum64(dq);
    float u = s_v[4 * wave + i];
    if constexpr (kDelta) u = beta * (u - wave_sum64(dk));
#pragma unroll
    for (int e = 0; e < E; ++e) {
      s[i][e] = __fmaf_rn(k[e], u, s[i][e]);
      if (on) rows[(size_t)i * D + e] = s[i][e];
    }
    if (lane == 0 && d < g.vdim) o[h * g.vdim + d] = __fmaf_rn(kq, u, dq);
  }
}

// Whether the output's operands come through LDS: where a CU has more than one of its workgroups. Us through LDS / without, D = 128: 8 heads x 4
// chunks 14.6 / 13.0, 16 x 16 17.4 / 16.1, 48 x 8 24.4 / 32.8, 16 x 32 26.4 / 34.0; D = 256: 16 x 16 41.2 / 37.2, 48 x 8 62.9 / 72.1; D = 64: 28 x
// 2 7.6 / 7.3, 28 x 8 equal, 48 x 8 11.8 / 13.8. D = 32 (two steps): 0.3 to 0.6 us better through LDS throughout.
bool out_shared(int workgroups) { return workgroups > 256; }

template <int D, bool kDelta>
hipError_t prefill_d(int dtype, const RecGeom& g, const float* raw, const float* cx, int ldcx, float* state,
                     float* scratch, void* out, int ldo, int M, int pos0, hipStream_t s) {
  const int chunks = (M + kC - 1) / kC, dv16 = (g.vdim + 15) & ~15;
  auto prep = rec_chunk_kernel<D, kDelta>;
  constexpr size_t lds = chunk_lds<D>();
  const int vec = g.dim % 4 == 0 && (kDelta || g.rot_dims % 8 == 0);
  static LdsLimitOnce raised;
  if (lds > 64 * 1024)
    if (hipError_t e = raised.raise(reinterpret_cast<const void*>(prep), lds); e != hipSuccess) return e;
  hipLaunchKernelGGL(prep, dim3(chunks, g.heads), dim3(256), lds, s, g, raw, cx, ldcx, scratch, M, pos0, vec);
  if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
  hipLaunchKernelGGL((rec_scan_kernel<D, kDelta>), dim3(8, dv16 / 16, (g.heads + 7) / 8), dim3(256), 0, s, state,
                     scratch, g.heads, dv16, chunks, pos0 == 0 ? 1 : 0);
  if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
  auto output = [&](auto* to) {
    using T = std::remove_pointer_t<decltype(to)>;
    auto kern = rec_out_kernel<D, T, true>;
    if constexpr (D >= 64)
      if (!out_shared(chunks * g.heads)) kern = rec_out_kernel<D, T, false>;
    hipLaunchKernelGGL(kern, dim3(chunks, g.heads), dim3(256), 0, s, g, raw, scratch, to, ldo, M);
  };
  if (dtype == W4A32_LAYERED_BF16) output(static_cast<__bf16*>(out));
  else output(static_cast<float*>(out));
  return hipGetLastError();
}

template <int D>
hipError_t decode_d(const RecGeom& g, const float* raw, const float* conv, float* ring, float* state, const int* pos,
                    float* o, hipStream_t s) {
  const dim3 grid((g.vdim + 15) / 16, g.heads);
  if (g.delta) {
    hipLaunchKernelGGL((rec_decode_kernel<D, true>), grid, dim3(256), 0, s, g, raw, conv, ring, state, pos, o);
  } else {
    hipLaunchKernelGGL((rec_decode_kernel<D, false>), grid, dim3(256), 0, s, g, raw, conv, ring, state, pos, o);
  }
  return hipGetLastError();
}

}  // namespace

size_t rec_scratch_floats(int heads, int dim, int vdim, int M) {
  const int chunks = (M + kC - 1) / kC;
  return (size_t)heads * chunks * chunk_off(head_bucket(std::max(dim, vdim)), (vdim + 15) & ~15).total;
}

hipError_t launch_rec_prefill(int dtype, const RecGeom& g, const float* raw, const float* cx, int ldcx, float* state,
                              float* scratch, void* out, int ldo, int M, int pos0, hipStream_t s) {
#define W4_REC(DD)                                                                                              \
  case DD:                                                                                                      \
    return g.delta ? prefill_d<DD, true>(dtype, g, raw, cx, ldcx, state, scratch, out, ldo, M, pos0, s)        \
                   : prefill_d<DD, false>(dtype, g, raw, cx, ldcx, state, scratch, out, ldo, M, pos0, s)
  switch (g.D) {
    W4_REC(32);
    W4_REC(64);
    W4_REC(128);
    W4_REC(256);
    default: return hipErrorInvalidValue;
  }
#undef W4_REC
}

hipError_t launch_rec_decode(const RecGeom& g, const float* raw, const float* conv, float* ring, float* state,
                             const int* pos, float* o, hipStream_t s) {
  switch (g.D) {
    case 32: return decode_d<32>(g, raw, conv, ring, state, pos, o, s);
    case 64: return decode_d<64>(g, raw, conv, ring, state, pos, o, s);
    case 128: return decode_d<128>(g, raw, conv, ring, state, pos, o, s);
    case 256: return decode_d<256>(g, raw, conv, ring, state, pos, o, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace w4
