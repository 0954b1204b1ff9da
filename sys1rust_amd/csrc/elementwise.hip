// Bandwidth-bound kernels of the forward: embedding + LayerNorm, LayerNorm (with or without
// bias), the qkv split + RoPE pass, GeGLU, row gathers and the scorer's final dot product.
// Each row is owned by one wavefront (reductions stay in registers and cross-lane shuffles); every
// global access is a coalesced 16-byte vector per lane.
#include <type_traits>

#include "device.hpp"
#include "kernels.hpp"

namespace s1 {

namespace {

// 8 consecutive floats as two 16-byte loads (parameters are read this way, not element by
// element: scalar loads each wait for the previous one and serialise the row on L2 latency).
__device__ __forceinline__ void load8f(const float* __restrict__ p, float* f) {
  const float4 a = reinterpret_cast<const float4*>(p)[0], b = reinterpret_cast<const float4*>(p)[1];
  f[0] = a.x; f[1] = a.y; f[2] = a.z; f[3] = a.w;
  f[4] = b.x; f[5] = b.y; f[6] = b.z; f[7] = b.w;
}

__device__ __forceinline__ void store8f(float* p, const float* f) {
  reinterpret_cast<float4*>(p)[0] = make_float4(f[0], f[1], f[2], f[3]);
  reinterpret_cast<float4*>(p)[1] = make_float4(f[4], f[5], f[6], f[7]);
}

// 8 results at element o of y: 16-bit of type E, or split f32 times sc where E is Split.
struct Split;
template <class E>
__device__ __forceinline__ void store8(void* y, size_t o, const float* f, float sc) {
  if constexpr (std::is_same<E, Split>::value) {
    uint32_t hi[4], lo[4];
    split_f16<8>(f, sc, hi, lo);
    uint16_t* p = static_cast<uint16_t*>(y) + split_at(o);
    *reinterpret_cast<uint4*>(p) = make_uint4(hi[0], hi[1], hi[2], hi[3]);
    *reinterpret_cast<uint4*>(p + 32) = make_uint4(lo[0], lo[1], lo[2], lo[3]);
  } else {
    *reinterpret_cast<uint4*>(static_cast<uint16_t*>(y) + o) = pack8<E>(f);
  }
}

// A hidden-state row of d floats is owned by one wavefront: lane l holds elements
// [8l + 512c, 8l + 512c + 8) for the NC = ceil(d / 512) passes c, as v[8c .. 8c + 7]. d is a
// multiple of 128, so a pass is either whole for a lane or past the row's end (then the lane
// holds zeros there and leaves them out of every sum).
__device__ __forceinline__ bool in_row(int c, int lane, int d) { return c * 512 + lane * 8 < d; }

// Chunk c of a row for this lane, zeros past the row's end. The load itself is unconditional
// (lanes past the end read the row's first 8 elements and drop them), so every load of a row goes
// out before any is waited on: a branch around each chunk's load made the next chunk's wait for it.
__device__ __forceinline__ void load_chunk_f32(const float* __restrict__ row, int c, int lane, int d, float* f) {
  const bool in = in_row(c, lane, d);
  load8f(row + (in ? c * 512 + lane * 8 : 0), f);
#pragma unroll
  for (int e = 0; e < 8; ++e) f[e] = in ? f[e] : 0.0f;
}
template <class E>
__device__ __forceinline__ void load_chunk_16(const uint16_t* __restrict__ row, int c, int lane, int d, float* f) {
  const bool in = in_row(c, lane, d);
  unpack8<E>(*reinterpret_cast<const uint4*>(row + (in ? c * 512 + lane * 8 : 0)), f);
#pragma unroll
  for (int e = 0; e < 8; ++e) f[e] = in ? f[e] : 0.0f;
}

// Row statistics: mean and 1 / sqrt(biased variance + eps), in f32, every lane the same bits.
template <int NC>
__device__ __forceinline__ void ln_stats(const float* v, int d, int lane, float eps, float& mean, float& rstd) {
  float s = 0.0f;
#pragma unroll
  for (int c = 0; c < NC; ++c)
    if (in_row(c, lane, d)) {
#pragma unroll
      for (int e = 0; e < 8; ++e) s += v[c * 8 + e];
    }
  mean = wave_sum(s) / float(d);
  float q = 0.0f;
#pragma unroll
  for (int c = 0; c < NC; ++c)
    if (in_row(c, lane, d)) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float x = v[c * 8 + e] - mean;
        q += x * x;
      }
    }
  const float var = wave_sum(q) / float(d);
  rstd = 1.0f / sqrtf(var + eps);
}

template <class E, int NC>
__global__ __launch_bounds__(256) void embed_ln_kernel(const uint16_t* __restrict__ emb, const int* __restrict__ ids,
                                                      const float* __restrict__ w, float eps, int T, int d,
                                                      float* __restrict__ h, uint16_t* __restrict__ x) {
  const int row = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (row >= T) return;
  const uint16_t* src = emb + size_t(ids[row]) * d;
  float v[8 * NC], wv[8 * NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    load_chunk_16<E>(src, c, lane, d, v + c * 8);
    load_chunk_f32(w, c, lane, d, wv + c * 8);
  }
  float mean, rstd;
  ln_stats<NC>(v, d, lane, eps, mean, rstd);
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    if (!in_row(c, lane, d)) continue;
    const int o = c * 512 + lane * 8;
    float y[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) y[e] = (v[c * 8 + e] - mean) * rstd * wv[c * 8 + e];
    store8f(h + size_t(row) * d + o, y);
    *reinterpret_cast<uint4*>(x + size_t(row) * d + o) = pack8<E>(y);
  }
}

template <class E, int NC>
__global__ __launch_bounds__(256) void layernorm_kernel(const float* __restrict__ x, const int* __restrict__ rows,
                                                       const float* __restrict__ w, const float* __restrict__ b,
                                                       float eps, int T, int d, void* __restrict__ yb,
                                                       float* __restrict__ yf, const float* __restrict__ addv,
                                                       const int* __restrict__ seg, float* __restrict__ yplus, float ys) {
  const int row = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (row >= T) return;
  const int src_row = rows ? rows[row] : row;
  const float* src = x + size_t(src_row) * d;
  // The row and, loaded while the statistics reduce, this lane's parameters.
  float v[8 * NC], wv[8 * NC], bv[8 * NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    load_chunk_f32(src, c, lane, d, v + c * 8);
    load_chunk_f32(w, c, lane, d, wv + c * 8);
  }
#pragma unroll
  for (int i = 0; i < 8 * NC; ++i) bv[i] = 0.0f;
  if (b) {
#pragma unroll
    for (int c = 0; c < NC; ++c) load_chunk_f32(b, c, lane, d, bv + c * 8);
  }
  float mean, rstd;
  ln_stats<NC>(v, d, lane, eps, mean, rstd);
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    if (!in_row(c, lane, d)) continue;
    const int o = c * 512 + lane * 8;
    float y[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) y[e] = (v[c * 8 + e] - mean) * rstd * wv[c * 8 + e] + bv[c * 8 + e];
    if (yb) store8<E>(yb, size_t(row) * d + o, y, ys);
    if (yf) store8f(yf + size_t(row) * d + o, y);
    if (yplus) {
      float z[8];
      load8f(addv + size_t(seg[row]) * d + o, z);
#pragma unroll
      for (int e = 0; e < 8; ++e) z[e] += y[e];
      store8f(yplus + size_t(row) * d + o, z);
    }
  }
}

// Split-K residual GEMM end + LayerNorm, one wave per row. The sum runs over the splits in
// order from 0.0f, then the bias (or 0.0f), then onto h: the arithmetic of the GEMM's split-K
// epilogue; the statistics and y are layernorm_kernel's on the new h. The row's residual and the
// parameters load first, then the splits SG at a time, all in flight together, so the row waits
// on ceil(splits / SG) load rounds (one at every split count a short request plans for d <= 1024).
template <class E, int NC, int SG = NC == 1 ? 16 : NC == 2 ? 10 : 4>
__global__ __launch_bounds__(256) void splitk_resid_ln_kernel(const float* __restrict__ ws, int splits,
                                                             const float* __restrict__ bias, float* __restrict__ h,
                                                             const float* __restrict__ w, float eps, int T, int d,
                                                             void* __restrict__ y, const float* __restrict__ lnb,
                                                             const float* __restrict__ hsrc,
                                                             const int* __restrict__ hrows, float ys) {
  constexpr int PL = 8 * NC;
  const int row = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (row >= T) return;
  const size_t plane = size_t(T) * d;
  // The residual row (h's own, or row hrows[row] of hsrc: a gather folded into this pass), the
  // GEMM's bias and the LayerNorm's weight and bias (0.0f where absent, as the two-kernel path
  // adds them).
  const float* hin = hsrc ? hsrc + size_t(hrows[row]) * d : h + size_t(row) * d;
  float hb[PL], bb[PL], wv[PL], bv[PL];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    load_chunk_f32(hin, c, lane, d, hb + c * 8);
    load_chunk_f32(w, c, lane, d, wv + c * 8);
  }
#pragma unroll
  for (int i = 0; i < PL; ++i) bb[i] = bv[i] = 0.0f;
  if (bias) {
#pragma unroll
    for (int c = 0; c < NC; ++c) load_chunk_f32(bias, c, lane, d, bb + c * 8);
  }
  if (lnb) {
#pragma unroll
    for (int c = 0; c < NC; ++c) load_chunk_f32(lnb, c, lane, d, bv + c * 8);
  }
  const float* part = ws + size_t(row) * d + lane * 8;
  float x[PL];
#pragma unroll
  for (int i = 0; i < PL; ++i) x[i] = 0.0f;
  for (int s = 0; s < splits; s += SG) {
    float a[SG][PL];
#pragma unroll
    for (int u = 0; u < SG; ++u)
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        if (in_row(c, lane, d)) {
          load8f(part + size_t(min(s + u, splits - 1)) * plane + c * 512, a[u] + c * 8);
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e) a[u][c * 8 + e] = 0.0f;
        }
      }
#pragma unroll
    for (int u = 0; u < SG; ++u)
      if (s + u < splits) {
#pragma unroll
        for (int i = 0; i < PL; ++i) x[i] += a[u][i];
      }
  }
  float v[PL];
#pragma unroll
  for (int i = 0; i < PL; ++i) v[i] = hb[i] + (x[i] + bb[i]);
  float* hr = h + size_t(row) * d + lane * 8;
#pragma unroll
  for (int c = 0; c < NC; ++c)
    if (in_row(c, lane, d)) store8f(hr + c * 512, v + c * 8);
  float mean, rstd;
  ln_stats<NC>(v, d, lane, eps, mean, rstd);
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    if (!in_row(c, lane, d)) continue;
    float o[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = (v[c * 8 + e] - mean) * rstd * wv[c * 8 + e] + bv[c * 8 + e];
    store8<E>(y, size_t(row) * d + c * 512 + lane * 8, o, ys);
  }
}

// The end of the encoder and the start of the decision head, one wave per row: h (plus the last
// residual GEMM's split-K partials when it left them pending, summed as splitk_resid_ln_kernel
// sums them), final_norm, plus type_emb of the row's question type into the head stream hh, and
// then the first head layer's norm1 of hh into x. Every step is the arithmetic of the kernel it
// stands for (the split-K epilogue, layernorm_kernel with its add of type_emb, layernorm_kernel
// with a bias), so the results are the same bits. h itself is not written back: nothing reads
// it after the encoder.
template <class E, int NC, int SG = 4 / NC * 4>
__global__ __launch_bounds__(256) void encoder_end_kernel(const float* __restrict__ ws, int splits,
                                                         const float* __restrict__ h, const float* __restrict__ wf,
                                                         float eps, const float* __restrict__ addv,
                                                         const int* __restrict__ seg, float* __restrict__ hh,
                                                         const float* __restrict__ w1, const float* __restrict__ b1,
                                                         float eps1, uint16_t* __restrict__ x, int T, int d) {
  constexpr int PL = 8 * NC;
  const int row = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (row >= T) return;
  const size_t plane = size_t(T) * d;
  float v[PL], wv[PL], bv[PL], z[PL];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    load_chunk_f32(h + size_t(row) * d, c, lane, d, v + c * 8);
    load_chunk_f32(wf, c, lane, d, wv + c * 8);
    load_chunk_f32(addv + size_t(seg[row]) * d, c, lane, d, z + c * 8);
  }
  if (splits > 1) {
    const float* part = ws + size_t(row) * d + lane * 8;
    float xs[PL];
#pragma unroll
    for (int i = 0; i < PL; ++i) xs[i] = 0.0f;
    for (int s = 0; s < splits; s += SG) {
      float a[SG][PL];
#pragma unroll
      for (int u = 0; u < SG; ++u)
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          if (in_row(c, lane, d)) {
            load8f(part + size_t(min(s + u, splits - 1)) * plane + c * 512, a[u] + c * 8);
          } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) a[u][c * 8 + e] = 0.0f;
          }
        }
#pragma unroll
      for (int u = 0; u < SG; ++u)
        if (s + u < splits) {
#pragma unroll
          for (int i = 0; i < PL; ++i) xs[i] += a[u][i];
        }
    }
    // h + (sum + bias), the residual GEMM having no bias: its reduce adds 0.0f.
    const float nob = 0.0f;
#pragma unroll
    for (int i = 0; i < PL; ++i) v[i] = v[i] + (xs[i] + nob);
  }
#pragma unroll
  for (int i = 0; i < PL; ++i) bv[i] = 0.0f;
  float mean, rstd;
  ln_stats<NC>(v, d, lane, eps, mean, rstd);
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    if (!in_row(c, lane, d)) continue;
    float y[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) y[e] = (v[c * 8 + e] - mean) * rstd * wv[c * 8 + e] + bv[c * 8 + e];
#pragma unroll
    for (int e = 0; e < 8; ++e) z[c * 8 + e] += y[e];
    store8f(hh + size_t(row) * d + c * 512 + lane * 8, z + c * 8);
  }
  if (!x) return;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    load_chunk_f32(w1, c, lane, d, wv + c * 8);
    load_chunk_f32(b1, c, lane, d, bv + c * 8);
  }
  ln_stats<NC>(z, d, lane, eps1, mean, rstd);
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    if (!in_row(c, lane, d)) continue;
    float y[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) y[e] = (z[c * 8 + e] - mean) * rstd * wv[c * 8 + e] + bv[c * 8 + e];
    *reinterpret_cast<uint4*>(x + size_t(row) * d + c * 512 + lane * 8) = pack8<E>(y);
  }
}

// The end of the pruned decision head, one wave per picked row: h (plus the last linear2's
// split-K partials and bias when it left them pending, summed as splitk_resid_ln_kernel sums
// them). A request's picked rows are its row 0, which goes out as the pooled row, then its kmax
// scorer rows, which go out as the scorer's LayerNorm (weight w, bias b) in 16 bits. Bit for bit
// the split-K epilogue, layernorm_kernel over the scorer rows and the gather of the pooled rows.
template <class E, int NC, int SG = 4 / NC * 4>
__global__ __launch_bounds__(256) void head_end_kernel(const float* __restrict__ ws, int splits,
                                                      const float* __restrict__ bias, const float* __restrict__ h,
                                                      int per, const float* __restrict__ w, const float* __restrict__ b,
                                                      float eps, float* __restrict__ pooled, uint16_t* __restrict__ y,
                                                      int P, int d) {
  constexpr int PL = 8 * NC;
  const int row = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (row >= P) return;
  const size_t plane = size_t(P) * d;
  const int req = row / per, slot = row - req * per;
  float v[PL], wv[PL], bv[PL];
#pragma unroll
  for (int c = 0; c < NC; ++c) load_chunk_f32(h + size_t(row) * d, c, lane, d, v + c * 8);
  if (slot) {
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      load_chunk_f32(w, c, lane, d, wv + c * 8);
      load_chunk_f32(b, c, lane, d, bv + c * 8);
    }
  }
  if (splits > 1) {
    const float* part = ws + size_t(row) * d + lane * 8;
    float xs[PL], bb[PL];
#pragma unroll
    for (int i = 0; i < PL; ++i) xs[i] = 0.0f;
    for (int s = 0; s < splits; s += SG) {
      float a[SG][PL];
#pragma unroll
      for (int u = 0; u < SG; ++u)
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          if (in_row(c, lane, d)) {
            load8f(part + size_t(min(s + u, splits - 1)) * plane + c * 512, a[u] + c * 8);
          } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) a[u][c * 8 + e] = 0.0f;
          }
        }
#pragma unroll
      for (int u = 0; u < SG; ++u)
        if (s + u < splits) {
#pragma unroll
          for (int i = 0; i < PL; ++i) xs[i] += a[u][i];
        }
    }
#pragma unroll
    for (int i = 0; i < PL; ++i) bb[i] = 0.0f;
    if (bias) {
#pragma unroll
      for (int c = 0; c < NC; ++c) load_chunk_f32(bias, c, lane, d, bb + c * 8);
    }
#pragma unroll
    for (int i = 0; i < PL; ++i) v[i] = v[i] + (xs[i] + bb[i]);
  }
  if (!slot) {
#pragma unroll
    for (int c = 0; c < NC; ++c)
      if (in_row(c, lane, d)) store8f(pooled + size_t(req) * d + c * 512 + lane * 8, v + c * 8);
    return;
  }
  float mean, rstd;
  ln_stats<NC>(v, d, lane, eps, mean, rstd);
  uint16_t* yr = y + (size_t(req) * (per - 1) + slot - 1) * d;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    if (!in_row(c, lane, d)) continue;
    float o[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = (v[c * 8 + e] - mean) * rstd * wv[c * 8 + e] + bv[c * 8 + e];
    *reinterpret_cast<uint4*>(yr + c * 512 + lane * 8) = pack8<E>(o);
  }
}

// The standalone split + RoPE pass, one workgroup per (64-token block, head), 256 threads:
// thread (token t0 + tid / 4, quarter) takes rotation pairs i0 .. i0 + 7 (i0 = 8 quarter), i.e.
// dims [i0, i0 + 8) and [i0 + 32, i0 + 40) of the head, for q and k. The 4 threads of a token
// read the head's 128 bytes of its qkv row and write them to the head-major q / k, where the
// block's 64 tokens are one contiguous 8 KiB run. v goes through LDS, [token][dim], and leaves
// transposed as 16-byte pieces of 8 tokens: 128-byte rows of [H, 64, ldv].
template <class E>
__global__ __launch_bounds__(256) void split_rope_kernel(const uint16_t* __restrict__ qkv, int T, int d,
                                                        const int* __restrict__ pos, const float* __restrict__ ct,
                                                        const float* __restrict__ stab, uint16_t* __restrict__ q,
                                                        uint16_t* __restrict__ k, uint16_t* __restrict__ v,
                                                        int ldv) {
  constexpr int VP = 64 + 8;  // LDS row pitch of the v block, elements (16 bytes of padding)
  __shared__ __attribute__((aligned(16))) uint16_t sv[64 * VP];
  const int H = d >> 6;
  const int head = blockIdx.x % H;
  const int t0 = (blockIdx.x / H) * 64;
  const int tl = threadIdx.x >> 2, quarter = threadIdx.x & 3;
  const int t = t0 + tl;
  const int i0 = quarter * 8;
  if (t < T) {
    const uint16_t* src = qkv + size_t(t) * 3 * d + head * 64 + i0;
    const size_t dst = (size_t(head) * T + t) * 64 + i0;
    float c[8], s[8];
    const bool rope = ct != nullptr;
    if (rope) {
      const int p = pos[t];
      const float4* cp = reinterpret_cast<const float4*>(ct + p * 32 + i0);
      const float4* sp = reinterpret_cast<const float4*>(stab + p * 32 + i0);
      const float4 c0 = cp[0], c1 = cp[1], s0 = sp[0], s1 = sp[1];
      c[0] = c0.x; c[1] = c0.y; c[2] = c0.z; c[3] = c0.w; c[4] = c1.x; c[5] = c1.y; c[6] = c1.z; c[7] = c1.w;
      s[0] = s0.x; s[1] = s0.y; s[2] = s0.z; s[3] = s0.w; s[4] = s1.x; s[5] = s1.y; s[6] = s1.z; s[7] = s1.w;
    }
#pragma unroll
    for (int part = 0; part < 2; ++part) {
      const uint16_t* sp = src + part * d;
      uint16_t* dp = (part == 0 ? q : k) + dst;
      const uint4 a = *reinterpret_cast<const uint4*>(sp);
      const uint4 b = *reinterpret_cast<const uint4*>(sp + 32);
      if (!rope) {
        *reinterpret_cast<uint4*>(dp) = a;
        *reinterpret_cast<uint4*>(dp + 32) = b;
        continue;
      }
      float x1[8], x2[8], y1[8], y2[8];
      unpack8<E>(a, x1);
      unpack8<E>(b, x2);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        y1[j] = x1[j] * c[j] - x2[j] * s[j];
        y2[j] = x1[j] * s[j] + x2[j] * c[j];
      }
      *reinterpret_cast<uint4*>(dp) = pack8<E>(y1);
      *reinterpret_cast<uint4*>(dp + 32) = pack8<E>(y2);
    }
    const uint16_t* sv_src = src + 2 * d;
    *reinterpret_cast<uint4*>(&sv[tl * VP + i0]) = *reinterpret_cast<const uint4*>(sv_src);
    *reinterpret_cast<uint4*>(&sv[tl * VP + i0 + 32]) = *reinterpret_cast<const uint4*>(sv_src + 32);
  } else {
    // Tokens past T read as zeros: the piece holding token T - 1 writes them into the columns up
    // to the next multiple of 8, which every v writer leaves zero.
    *reinterpret_cast<uint4*>(&sv[tl * VP + i0]) = make_uint4(0, 0, 0, 0);
    *reinterpret_cast<uint4*>(&sv[tl * VP + i0 + 32]) = make_uint4(0, 0, 0, 0);
  }
  __syncthreads();
  const int tend = (T + 7) / 8 * 8;
#pragma unroll
  for (int it = 0; it < 2; ++it) {
    const int p = threadIdx.x + it * 256;
    const int dim = p >> 3, c8 = p & 7;  // tokens t0 + 8 c8 .. + 7 of dim `dim`
    const int tt = t0 + 8 * c8;
    if (tt >= tend) continue;
    uint32_t w[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
      w[j] = uint32_t(sv[(8 * c8 + 2 * j) * VP + dim]) | (uint32_t(sv[(8 * c8 + 2 * j + 1) * VP + dim]) << 16);
    *reinterpret_cast<uint4*>(v + (size_t(head) * 64 + dim) * ldv + tt) = make_uint4(w[0], w[1], w[2], w[3]);
  }
}

template <class E>
__global__ __launch_bounds__(256) void geglu_kernel(const uint16_t* __restrict__ wi, int T, int I,
                                                   uint16_t* __restrict__ act) {
  const long long gid = (long long)blockIdx.x * 256 + threadIdx.x;
  const int per_row = I / 8;
  if (gid >= (long long)T * per_row) return;
  const int t = int(gid / per_row), c = int(gid % per_row) * 8;
  const uint16_t* r = wi + size_t(t) * 2 * I;
  float x[8], g[8], y[8];
  unpack8<E>(*reinterpret_cast<const uint4*>(r + c), x);
  unpack8<E>(*reinterpret_cast<const uint4*>(r + I + c), g);
#pragma unroll
  for (int e = 0; e < 8; ++e) y[e] = gelu_erf(x[e]) * g[e];
  *reinterpret_cast<uint4*>(act + size_t(t) * I + c) = pack8<E>(y);
}

__global__ __launch_bounds__(256) void gather_f32_kernel(const float* __restrict__ x, const int* __restrict__ rows,
                                                        int R, int d, float* __restrict__ out) {
  const int r = blockIdx.x;
  if (r >= R) return;
  const float4* s = reinterpret_cast<const float4*>(x + size_t(rows[r]) * d);
  float4* o = reinterpret_cast<float4*>(out + size_t(r) * d);
  for (int i = threadIdx.x; i < d / 4; i += 256) o[i] = s[i];
}

template <class E>
__global__ __launch_bounds__(256) void rowdot_kernel(const uint16_t* __restrict__ x, const float* __restrict__ w,
                                                    const float* __restrict__ b, int R, int d, float* __restrict__ out) {
  const int row = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (row >= R) return;
  float acc = 0.0f;
  for (int o = lane * 8; o < d; o += 512) {
    float v[8], wv[8];
    unpack8<E>(*reinterpret_cast<const uint4*>(x + size_t(row) * d + o), v);
    load8f(w + o, wv);
#pragma unroll
    for (int e = 0; e < 8; ++e) acc += v[e] * wv[e];
  }
  acc = wave_sum(acc);
  if (lane == 0) out[row] = acc + (b ? b[0] : 0.0f);
}

}  // namespace

// Row kernels run one wave per row and one row per workgroup: a short batch's few rows then spread
// over that many CUs, and at 5686 rows the request ran 1% faster than with four rows per
// workgroup (the per-launch times within noise).
inline int row_waves(int) { return 1; }

// The row kernels' pass count for a hidden size (a multiple of 128 up to 2048): NC = ceil(d / 512).
#define S1_ROWS_BY_NC(d, CALL) \
  switch (((d) + 511) / 512) { \
    case 1: CALL(1); break; \
    case 2: CALL(2); break; \
    case 3: CALL(3); break; \
    default: CALL(4); break; \
  }

template <class E>
void embed_ln_t(const uint16_t* tok_emb, const int* ids, const float* w, float eps, int T, int d, float* h_out,
                uint16_t* x_out, hipStream_t st) {
  const int rw = row_waves(T);
  dim3 grid((T + rw - 1) / rw), block(64 * rw);
#define S1_CALL(NC) hipLaunchKernelGGL((embed_ln_kernel<E, NC>), grid, block, 0, st, tok_emb, ids, w, eps, T, d, h_out, x_out)
  S1_ROWS_BY_NC(d, S1_CALL)
#undef S1_CALL
}

void embed_ln_launch(const uint16_t* tok_emb, const int* ids, const float* w, float eps, int T, int d, float* h_out,
                     uint16_t* x_out, hipStream_t st, int elem) {
  if (T <= 0) return;
  if (elem == ELEM_F16) embed_ln_t<F16>(tok_emb, ids, w, eps, T, d, h_out, x_out, st);
  else embed_ln_t<Bf16>(tok_emb, ids, w, eps, T, d, h_out, x_out, st);
}

template <class E>
void layernorm_t(const float* x, const int* rows, const float* w, const float* b, float eps, int T, int d, void* y,
                 float* y_f32, const float* add_rowvec, const int* seg, float* y_plus, hipStream_t st, float ys) {
  const int rw = row_waves(T);
  dim3 grid((T + rw - 1) / rw), block(64 * rw);
#define S1_CALL(NC)                                                                                              \
  hipLaunchKernelGGL((layernorm_kernel<E, NC>), grid, block, 0, st, x, rows, w, b, eps, T, d, y, y_f32, add_rowvec, \
                     seg, y_plus, ys)
  S1_ROWS_BY_NC(d, S1_CALL)
#undef S1_CALL
}

void layernorm_launch(const float* x, const int* rows, const float* w, const float* b, float eps, int T, int d, void* y,
                      float* y_f32, const float* add_rowvec, const int* seg, float* y_plus, hipStream_t st, int elem,
                      float ys) {
  if (T <= 0) return;
  if (elem == ELEM_F32) layernorm_t<Split>(x, rows, w, b, eps, T, d, y, y_f32, add_rowvec, seg, y_plus, st, ys);
  else if (elem == ELEM_F16) layernorm_t<F16>(x, rows, w, b, eps, T, d, y, y_f32, add_rowvec, seg, y_plus, st, ys);
  else layernorm_t<Bf16>(x, rows, w, b, eps, T, d, y, y_f32, add_rowvec, seg, y_plus, st, ys);
}

template <class E>
void splitk_resid_ln_t(const float* ws, int splits, const float* bias, float* h, const float* w, float eps, int T, int d,
                       void* y, hipStream_t st, const float* lnb, const float* hsrc, const int* hrows, float ys) {
  const int rw = row_waves(T);
  dim3 grid((T + rw - 1) / rw), block(64 * rw);
#define S1_CALL(NC)                                                                                                \
  hipLaunchKernelGGL((splitk_resid_ln_kernel<E, NC>), grid, block, 0, st, ws, splits, bias, h, w, eps, T, d, y, lnb, \
                     hsrc, hrows, ys)
  S1_ROWS_BY_NC(d, S1_CALL)
#undef S1_CALL
}

void splitk_resid_ln_launch(const float* ws, int splits, const float* bias, float* h, const float* w, float eps, int T,
                            int d, void* y, hipStream_t st, int elem, const float* lnb, const float* hsrc,
                            const int* hrows, float ys) {
  if (T <= 0) return;
  if (elem == ELEM_F32) splitk_resid_ln_t<Split>(ws, splits, bias, h, w, eps, T, d, y, st, lnb, hsrc, hrows, ys);
  else if (elem == ELEM_F16) splitk_resid_ln_t<F16>(ws, splits, bias, h, w, eps, T, d, y, st, lnb, hsrc, hrows, ys);
  else splitk_resid_ln_t<Bf16>(ws, splits, bias, h, w, eps, T, d, y, st, lnb, hsrc, hrows, ys);
}

template <class E>
void encoder_end_t(const float* ws, int splits, const float* h, const float* wf, float eps, const float* addv,
                   const int* seg, float* hh, const float* w1, const float* b1, float eps1, uint16_t* x, int T, int d,
                   hipStream_t st) {
  const int rw = row_waves(T);
  dim3 grid((T + rw - 1) / rw), block(64 * rw);
#define S1_CALL(NC)                                                                                                \
  hipLaunchKernelGGL((encoder_end_kernel<E, NC>), grid, block, 0, st, ws, splits, h, wf, eps, addv, seg, hh, w1, b1, \
                     eps1, x, T, d)
  S1_ROWS_BY_NC(d, S1_CALL)
#undef S1_CALL
}

void encoder_end_launch(const float* ws, int splits, const float* h, const float* wf, float eps, const float* addv,
                        const int* seg, float* hh, const float* w1, const float* b1, float eps1, uint16_t* x, int T,
                        int d, hipStream_t st, int elem) {
  if (T <= 0) return;
  if (elem == ELEM_F16) encoder_end_t<F16>(ws, splits, h, wf, eps, addv, seg, hh, w1, b1, eps1, x, T, d, st);
  else encoder_end_t<Bf16>(ws, splits, h, wf, eps, addv, seg, hh, w1, b1, eps1, x, T, d, st);
}

template <class E>
void head_end_t(const float* ws, int splits, const float* bias, const float* h, int per, const float* w, const float* b,
                float eps, float* pooled, uint16_t* y, int P, int d, hipStream_t st) {
  const int rw = row_waves(P);
  dim3 grid((P + rw - 1) / rw), block(64 * rw);
#define S1_CALL(NC) \
  hipLaunchKernelGGL((head_end_kernel<E, NC>), grid, block, 0, st, ws, splits, bias, h, per, w, b, eps, pooled, y, P, d)
  S1_ROWS_BY_NC(d, S1_CALL)
#undef S1_CALL
}

void head_end_launch(const float* ws, int splits, const float* bias, const float* h, int per, const float* w,
                     const float* b, float eps, float* pooled, uint16_t* y, int P, int d, hipStream_t st, int elem) {
  if (P <= 0) return;
  if (elem == ELEM_F16) head_end_t<F16>(ws, splits, bias, h, per, w, b, eps, pooled, y, P, d, st);
  else head_end_t<Bf16>(ws, splits, bias, h, per, w, b, eps, pooled, y, P, d, st);
}

void split_rope_launch(const uint16_t* qkv, int T, int d, const int* pos, const float* cos_t, const float* sin_t,
                       uint16_t* q, uint16_t* k, uint16_t* v, int ldv, hipStream_t st, int elem) {
  if (T <= 0) return;
  const dim3 grid(unsigned((T + 63) / 64 * (d / 64))), block(256);
  if (elem == ELEM_F16)
    hipLaunchKernelGGL(split_rope_kernel<F16>, grid, block, 0, st, qkv, T, d, pos, cos_t, sin_t, q, k, v, ldv);
  else
    hipLaunchKernelGGL(split_rope_kernel<Bf16>, grid, block, 0, st, qkv, T, d, pos, cos_t, sin_t, q, k, v, ldv);
}

void geglu_launch(const uint16_t* wi, int T, int I, uint16_t* act, hipStream_t st, int elem) {
  const long long n = (long long)T * (I / 8);
  if (n <= 0) return;
  const dim3 grid(unsigned((n + 255) / 256)), block(256);
  if (elem == ELEM_F16) hipLaunchKernelGGL(geglu_kernel<F16>, grid, block, 0, st, wi, T, I, act);
  else hipLaunchKernelGGL(geglu_kernel<Bf16>, grid, block, 0, st, wi, T, I, act);
}

void gather_f32_launch(const float* x, const int* rows, int R, int d, float* out, hipStream_t st) {
  if (R <= 0) return;
  hipLaunchKernelGGL(gather_f32_kernel, dim3(R), dim3(256), 0, st, x, rows, R, d, out);
}

void rowdot_launch(const uint16_t* x, const float* w, const float* b, int R, int d, float* out, hipStream_t st,
                   int elem) {
  if (R <= 0) return;
  if (elem == ELEM_F16) hipLaunchKernelGGL(rowdot_kernel<F16>, dim3((R + 3) / 4), dim3(256), 0, st, x, w, b, R, d, out);
  else hipLaunchKernelGGL(rowdot_kernel<Bf16>, dim3((R + 3) / 4), dim3(256), 0, st, x, w, b, R, d, out);
}

}  // namespace s1
