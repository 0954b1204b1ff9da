// Kernels of the dtype=f32 path: the reference's BackendOptions::f32 (f32 weights and compute,
// runtime/crates/laya-core/src/backend.rs:25-27; laya-mlx/tests/parity.rs:54-65 checks it).
// f32 storage and sums throughout; the products take operands of 23 significant bits, each split into
// two f16 (gemm32_kernel says what that costs), attention runs on the f32 matrix instructions, with
// an exact erf GELU and an f32 softmax.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "device.hpp"
#include "kernels.hpp"
#include "lds_load.hpp"

namespace s1 {
namespace {

__device__ __forceinline__ float gelu_exact(float x) { return 0.5f * x * (1.0f + erff(x * 0.70710678118654752f)); }

__device__ __forceinline__ float act32(float v, int act) {
  return act == ACT_RELU ? fmaxf(v, 0.0f) : act == ACT_GELU ? gelu_exact(v) : v;
}

// C[M, N] = A[M, K] . W[N, K]^T of split operands: hi hi + (hi lo + lo hi) / 2048 on
// v_mfma_f32_32x32x16_f16, each of the three exact and summed in f32, the two orders of magnitude in
// accumulators of their own; lo lo, up to 2^-22 of a term, is left out. A term is then off by up to
// 2^-21, 7.9e-8 in the root mean square (an f32 FMA: 2^-24 and 2.5e-8), but the sum is rounded a
// sixteenth as often. Sums of K products of normal values, relative root mean square, here and by one
// FMA after the other (emulated): K 4 8.3e-8, 4.0e-8; 16 8.4e-8, 7.3e-8; 32 8.6e-8, 1.0e-7; 256 1.1e-7, 2.9e-7;
// 1024 1.7e-7, 5.7e-7. So a sum that a few terms outweigh is less exact than by FMAs, and the sums over
// the widths of this model's layers (768 and more) are more exact. Three 16-deep instructions take 96
// clocks of a SIMD where the f32 matrix instruction takes 512; what bounds these products is the power
// that they draw (the same launch on zeros runs 1.4 times as fast). Against v_mfma_f32_32x32x2_f32 on the same tiles, M 5707:
// N 3072, K 1024 330 -> 119 us (302 TFLOP/s); 1024, 1024 112 -> 39; 5248, 1024 524 -> 224; 1024, 2624
// 279 -> 92; 4096, 1024 417 -> 168; 1024, 4096 425 -> 149, and the error against float64 from 5.7e-7 to
// 2.2e-7 at K 1024, 1.2e-6 to 4.3e-7 at 4096 (fewer roundings of the sum). Splitting into three bf16
// and six products, which would hold every operand exactly: 239 us for the first of them.
//
// BM x BN tiles in WM x WN waves, 32-deep k-tiles (128-byte rows, [32 hi | 32 lo]) moved global -> LDS
// by direct loads, STAGES deep, one barrier per k-tile; 16-byte chunk c of row r sits at slot
// c ^ ((r / 2) % 8), so the 16 rows of one fragment read phase start in 16 distinct bank groups. W is
// the first operand (C^T = W . A^T): a lane holds 4 consecutive columns of one row and stores them as
// one float4.
template <int BM, int BN, int WM, int WN, int STAGES>
__global__ __launch_bounds__(WM * WN * 64) void gemm32_kernel(Gemm32Args g) {
  constexpr int NW = WM * WN, TM = BM / WM, TN = BN / WN, FM = TM / 32, FN = TN / 32;
  constexpr int BKF = 32, ROWB = BKF * 4, CH = 8, RG = 8;
  constexpr int AG = BM / RG, WG = BN / RG, LPW = (AG + WG) / NW;
  constexpr int A_BYTES = BM * ROWB, STAGE_BYTES = (BM + BN) * ROWB;
  static_assert(LPW * NW == AG + WG && AG % NW == 0, "a wave's j-th load reads one operand");
  static_assert(TM % 32 == 0 && TN % 32 == 0, "whole fragments");
  __shared__ __attribute__((aligned(1024))) char smem[STAGES * STAGE_BYTES];

  // Tile order as in the 16-bit GEMM: XCD-contiguous runs of 4-row-tile groups across all columns.
  constexpr int GM = 4;
  const int mt = (g.M + BM - 1) / BM, nt = g.N / BN;
  const int bid = xcd_remap(blockIdx.x, gridDim.x);
  const int grp = bid / (GM * nt);
  const int gm = min(GM, mt - grp * GM);
  const int loc = bid - grp * GM * nt;
  const int m0 = (grp * GM + loc % gm) * BM, n0 = loc / gm * BN;
  const int ktiles = g.K / BKF, split = blockIdx.y;
  const int kt0 = int((long long)split * ktiles / g.splits);
  const int NK = int((long long)(split + 1) * ktiles / g.splits) - kt0;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN;

  // Loads: the operands are addressed from the tile's own first row, so 32-bit offsets reach it
  // whatever the matrix spans; rows past M repeat the last one (their results are not stored).
  const int lrow = lane / CH, lslot = lane % CH;
  const int mlast = g.M - 1 - m0;
  uint32_t voff[LPW];
#pragma unroll
  for (int j = 0; j < LPW; ++j) {
    const int gi = wave + j * NW;
    const bool isA = j < AG / NW;
    const int r = (isA ? gi : gi - AG) * RG + lrow;
    const int c = lslot ^ ((r >> 1) & 7);
    voff[j] = (isA ? uint32_t(min(r, mlast)) * uint32_t(g.lda) : uint32_t(r) * uint32_t(g.ldw)) * 4u + c * 16;
  }
  const i32x4 rsrcA = buffer_rsrc(g.A + size_t(m0) * g.lda, uint32_t((size_t(min(BM - 1, mlast)) * g.lda + g.K) * 4));
  const i32x4 rsrcW = buffer_rsrc(g.W + size_t(n0) * g.ldw, uint32_t((size_t(BN - 1) * g.ldw + g.K) * 4));
  auto issue = [&](int stage, int kt, int jlo, int jhi) __attribute__((always_inline)) {  // this wave's loads [jlo, jhi)
    const int koff = __builtin_amdgcn_readfirstlane(kt * ROWB);
    char* sb = smem + stage * STAGE_BYTES + wave * 1024;
#pragma unroll
    for (int j = 0; j < LPW; ++j)
      if (j >= jlo && j < jhi) load16_lds(j < AG / NW ? rsrcA : rsrcW, sb + j * NW * 1024, int(voff[j]), koff);
  };

  f32x16 acc[FM][FN], acx[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = acx[i][j][e] = 0.0f;

#pragma unroll
  for (int s = 0; s < STAGES - 1; ++s)
    if (s < NK) issue(s, kt0 + s, 0, LPW);
  const int lr = lane & 31, lh = lane >> 5;
  int ka[4];  // fragments of k-steps 0 and 1: hi, then lo
#pragma unroll
  for (int c = 0; c < 4; ++c) ka[c] = lr * ROWB + (((c * 2 + lh) ^ ((lr >> 1) & 7)) << 4);
  for (int it = 0; it < NK; ++it) {
    wait_ahead<LPW, STAGES - 2>(min(STAGES - 2, NK - 1 - it));
    // Every wave's loads of k-tile `it` have landed and every wave is done with k-tile it - 1,
    // whose buffer the next issue overwrites.
    barrier_lds();
    const bool pre = it + STAGES - 1 < NK;
    const char* sa = smem + (it % STAGES) * STAGE_BYTES + wm * TM * ROWB;
    const char* sw = smem + (it % STAGES) * STAGE_BYTES + A_BYTES + wn * TN * ROWB;
    typedef typename F16::v8 v8;
    v8 fa[2][2][FM], fb[2][2][FN];
    auto frag = [&](int s) __attribute__((always_inline)) {
#pragma unroll
      for (int p = 0; p < 2; ++p) {
#pragma unroll
        for (int i = 0; i < FM; ++i) fa[s][p][i] = *reinterpret_cast<const v8*>(sa + ka[2 * p + s] + i * 32 * ROWB);
#pragma unroll
        for (int j = 0; j < FN; ++j) fb[s][p][j] = *reinterpret_cast<const v8*>(sw + ka[2 * p + s] + j * 32 * ROWB);
      }
    };
    frag(0);
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      if (pre) issue((it + STAGES - 1) % STAGES, kt0 + it + STAGES - 1, s * LPW / 2, (s + 1) * LPW / 2);
      if (s == 0) frag(1);
      auto mm = [&](int pw, int pa, f32x16 (&c)[FM][FN]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j) c[i][j] = F16::mfma(fb[s][pw][j], fa[s][pa][i], c[i][j]);
      };
      mm(0, 0, acc);
      mm(1, 0, acx);
      mm(0, 1, acx);
    }
  }

  // Lane: row m0 + wm TM + 32 i + l % 32, columns n0 + wn TN + 32 j + 8 q + 4 h .. + 3. A split
  // product leaves its part of the sum in ws[split] for the reduce (splitk32_kernel, or the
  // consumer's own).
  const bool part = g.splits > 1;
  float* out = part ? g.ws + size_t(split) * g.M * g.N : g.C;
  const int ld = part ? g.N : g.ldc;
#pragma unroll
  for (int i = 0; i < FM; ++i) {
    const int row = m0 + wm * TM + i * 32 + lr;
    if (row >= g.M) continue;
    float* orow = out + size_t(row) * ld + n0 + wn * TN + 4 * lh;
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        float4* o = reinterpret_cast<float4*>(orow + j * 32 + q * 8);
        const int4 wexp = *reinterpret_cast<const int4*>(g.wexp + n0 + wn * TN + 4 * lh + j * 32 + q * 8);
        const int ex[4] = {wexp.x + g.aexp, wexp.y + g.aexp, wexp.z + g.aexp, wexp.w + g.aexp};
        float v[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = ldexpf(fmaf(acx[i][j][4 * q + r], 1.0f / 2048.0f, acc[i][j][4 * q + r]), ex[r]);
        if (!part) {
          if (g.bias) {
            const float4 b = *reinterpret_cast<const float4*>(g.bias + n0 + wn * TN + 4 * lh + j * 32 + q * 8);
            v[0] += b.x;
            v[1] += b.y;
            v[2] += b.z;
            v[3] += b.w;
          }
#pragma unroll
          for (int r = 0; r < 4; ++r) v[r] = act32(v[r], g.act);
          if (g.accumulate) {
            const float4 c = *o;
            v[0] += c.x;
            v[1] += c.y;
            v[2] += c.z;
            v[3] += c.w;
          }
          if (g.cs > 0.0f) {
            store4_split(g.C, size_t(row) * ld + n0 + wn * TN + 4 * lh + j * 32 + q * 8, v, g.cs);
            continue;
          }
        }
        *o = make_float4(v[0], v[1], v[2], v[3]);
      }
  }
}

// Four consecutive elements of a product, from C itself (splits 1) or its parts [splits, plane]
// summed in order.
__device__ __forceinline__ float4 sum_parts(const float* p, int splits, size_t plane) {
  float4 s = *reinterpret_cast<const float4*>(p);
  for (int i = 1; i < splits; ++i) {
    const float4 v = *reinterpret_cast<const float4*>(p + size_t(i) * plane);
    s.x += v.x;
    s.y += v.y;
    s.z += v.z;
    s.w += v.w;
  }
  return s;
}

// The end of a split product whose consumer does not sum the parts itself.
__global__ __launch_bounds__(256) void splitk32_kernel(Gemm32Args g) {
  const long long gid = (long long)blockIdx.x * 256 + threadIdx.x;
  const int n4 = g.N / 4;
  if (gid >= (long long)g.M * n4) return;
  const int row = int(gid / n4), c = int(gid % n4) * 4;
  const float4 s = sum_parts(g.ws + size_t(row) * g.N + c, g.splits, size_t(g.M) * g.N);
  const float4 b = g.bias ? *reinterpret_cast<const float4*>(g.bias + c) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  float4* o = reinterpret_cast<float4*>(g.C + size_t(row) * g.ldc + c);
  const float4 old = g.accumulate ? *o : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  const float v[4] = {old.x + act32(s.x + b.x, g.act), old.y + act32(s.y + b.y, g.act), old.z + act32(s.z + b.z, g.act),
                      old.w + act32(s.w + b.w, g.act)};
  if (g.cs > 0.0f) store4_split(g.C, size_t(row) * g.ldc + c, v, g.cs);
  else *o = make_float4(v[0], v[1], v[2], v[3]);
}

// A weight matrix into split f32 in place, each row times the power of two that puts its largest
// element (bounds[2 row]) at 2^14 to 2^15: a wave reads its 64 elements of one row, then writes their
// bytes. wexp[row] is the exponent that undoes the row's scale.
__global__ __launch_bounds__(256) void split_weight_kernel(float* w, size_t n, int K, const float* __restrict__ bounds,
                                                           int* __restrict__ wexp) {
  const size_t e = size_t(blockIdx.x) * 256 + threadIdx.x;
  if (e >= n) return;
  const size_t row = e / K;
  const float m = bounds[2 * row];
  int ex = 0;
  if (m > 0.0f && m < __builtin_huge_valf()) (void)frexpf(m, &ex);
  ex = max(ex, -111) - 15;  // the scale is at most 2^126
  const float sc = ldexpf(1.0f, -ex);
  if (e % K == 0) wexp[row] = ex;
  const float x[2] = {w[e], 0.0f};
  uint32_t hi, lo;
  split_f16<2>(x, sc, &hi, &lo);
  uint16_t* o = reinterpret_cast<uint16_t*>(w) + split_at(e);
  o[0] = uint16_t(hi);
  o[32] = uint16_t(lo);
}

// One wave per row of W (weight_bound_launch): |W_r . (z * lw + lb) + bias| <= sqrt(K) |W_r * lw|_2 +
// |W_r . lb + bias| by the Cauchy-Schwarz inequality. The squares are taken of elements scaled by their largest.
__global__ __launch_bounds__(64) void weight_bound_kernel(const float* __restrict__ W, const float* __restrict__ lw,
                                                          const float* __restrict__ lb, const float* __restrict__ bias, int K,
                                                          float* __restrict__ out) {
  const float* row = W + size_t(blockIdx.x) * K;
  float mx = 0.0f, most = 0.0f, sq = 0.0f, dot = 0.0f;
  for (int k = threadIdx.x; k < K; k += 64) {
    const float w = row[k];
    mx = fmaxf(mx, fabsf(w));
    most = fmaxf(most, fabsf(lw ? w * lw[k] : w));
    if (lb) dot = fmaf(w, lb[k], dot);
  }
  mx = wave_max(mx);
  most = wave_max(most);
  dot = wave_sum(dot);
  int ex = 0;
  if (most > 0.0f && most < __builtin_huge_valf()) (void)frexpf(most, &ex);
  for (int k = threadIdx.x; k < K; k += 64) {
    const float x = ldexpf(lw ? row[k] * lw[k] : row[k], -ex);
    sq = fmaf(x, x, sq);
  }
  sq = wave_sum(sq);
  if (threadIdx.x) return;
  out[2 * blockIdx.x] = mx;
  out[2 * blockIdx.x + 1] = ldexpf(sqrtf(float(K)) * sqrtf(sq), ex) + fabsf(dot + (bias ? bias[blockIdx.x] : 0.0f));
}

// qkv [T, 3d] -> q, k, v [H, T, 64], with the half-split RoPE rotation of q and k at pos[t] when
// the tables are given (split_rope.rs:44-54). qkv comes whole, bias added, or as the parts of a
// split product, which are summed and given the bias here. One thread per (token, head, 4 dim
// pairs i .. i + 3, i + 32 .. i + 35).
__global__ __launch_bounds__(256) void split32_kernel(const float* __restrict__ qkv, int splits, const float* __restrict__ bias,
                                                      int T, int d, const int* __restrict__ pos,
                                                      const float* __restrict__ cs, const float* __restrict__ sn,
                                                      float* __restrict__ q, float* __restrict__ k, float* __restrict__ v) {
  const long long gid = (long long)blockIdx.x * 256 + threadIdx.x;
  const int H = d / 64;
  if (gid >= (long long)T * H * 8) return;
  const int i = int(gid % 8) * 4, h = int((gid / 8) % H), t = int(gid / (8LL * H));
  const size_t plane = size_t(T) * 3 * d;
  const float* row = qkv + size_t(t) * 3 * d + h * 64 + i;
  const size_t o = (size_t(h) * T + t) * 64 + i;
  const bool rot = cs != nullptr;
  float4 c = make_float4(1.0f, 1.0f, 1.0f, 1.0f), s = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  if (rot) {
    c = *reinterpret_cast<const float4*>(cs + size_t(pos[t]) * 32 + i);
    s = *reinterpret_cast<const float4*>(sn + size_t(pos[t]) * 32 + i);
  }
#pragma unroll
  for (int part = 0; part < 3; ++part) {
    float4 x1 = sum_parts(row + part * d, splits, plane), x2 = sum_parts(row + part * d + 32, splits, plane);
    if (bias) {
      const float* bp = bias + part * d + h * 64 + i;
      const float4 b1 = *reinterpret_cast<const float4*>(bp), b2 = *reinterpret_cast<const float4*>(bp + 32);
      x1 = make_float4(x1.x + b1.x, x1.y + b1.y, x1.z + b1.z, x1.w + b1.w);
      x2 = make_float4(x2.x + b2.x, x2.y + b2.y, x2.z + b2.z, x2.w + b2.w);
    }
    float* dst = (part == 0 ? q : part == 1 ? k : v) + o;
    if (rot && part < 2) {
      *reinterpret_cast<float4*>(dst) =
          make_float4(x1.x * c.x - x2.x * s.x, x1.y * c.y - x2.y * s.y, x1.z * c.z - x2.z * s.z, x1.w * c.w - x2.w * s.w);
      *reinterpret_cast<float4*>(dst + 32) =
          make_float4(x1.x * s.x + x2.x * c.x, x1.y * s.y + x2.y * c.y, x1.z * s.z + x2.z * c.z, x1.w * s.w + x2.w * c.w);
    } else {
      *reinterpret_cast<float4*>(dst) = x1;
      *reinterpret_cast<float4*>(dst + 32) = x2;
    }
  }
}

// Attention over packed rows in f32, both products on v_mfma_f32_32x32x2_f32, softmax with an
// online maximum. A wave takes 32 queries of one row and head; the workgroup's four waves are
// 4 / KW groups of 32 queries, and the KW waves of a group take its 32-key tiles in turn, with
// softmax statistics of their own, merged through LDS at the end (KW 1: none to merge).
//
//   S^T[key, q] = K . Q^T: lane (l % 32, h = l / 32) reads 4 consecutive dims 8 j + 4 h of key row
//   l % 32 and of query l % 32 at once, and MFMA u of the four multiplies dims 8 j + u and
//   8 j + 4 + u. The lane then holds query l % 32 and keys 8 g + 4 h + r.
//   O^T[dim, q] += V^T . P^T: step (g, r) takes keys 8 g + r and 8 g + 4 + r, so the operand P is
//   the lane's own accumulator 4 g + r, and the operand V a float per lane of two key rows.
//
// K and V are read straight from memory: the matrix unit needs 4096 clocks for a tile of a wave,
// and its 16 KiB, shared by the waves of the workgroup through L1, are well within what that
// allows, so there is nothing to stage and no barrier in the loop. The next tile's K is loaded
// before this tile's softmax. The weights are exp2 of fma(s, log2 e, -max): the argument is rounded as
// s - max would be, and a weight below 2^-126 of the row's largest is 0. Measured at 5707 tokens in
// 10 rows, 16 heads, against one wave per (query, head) on vector FMAs: global 1720 -> 245 us, local
// 402 -> 74 us.
template <int KW>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void attn32_tile_kernel(Attn32Args a) {
  constexpr float NEG_INF = -__builtin_huge_valf();
  __shared__ float mt[KW > 1 ? 4 * 64 : 1], lt[KW > 1 ? 4 * 64 : 1], ot[KW > 1 ? 4 * 32 * 64 : 1];
  const int lid = xcd_remap(blockIdx.x, gridDim.x);
  const int head = lid / a.n;
  const AttnTile tl = a.tiles[lid - head * a.n];
  const int lane = threadIdx.x & 63, col = lane & 31, hl = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wk = wave % KW;
  const float* __restrict__ Qh = a.q + size_t(head) * a.T * 64;
  const float* __restrict__ Kh = a.k + size_t(head) * a.T * 64;
  const float* __restrict__ Vh = a.v + size_t(head) * a.T * 64;

  const int wq0 = tl.q0 + wave / KW * 32;
  const bool active = wq0 < tl.q1;
  const int qi = wq0 + col, qld = min(qi, tl.q1 - 1);
  const int qk = active ? (a.qkey ? a.qkey[qld] : qld) : tl.k0;  // q row and key index of this query
  int k0 = tl.k0, k1 = tl.k1;
  if (a.window >= 0) {  // no qkey: slots are key indices
    k0 = max(k0, wq0 - a.window);
    k1 = min(k1, min(wq0 + 31, tl.q1 - 1) + a.window + 1);
  }
  if (!active) k1 = k0;
  k0 = __builtin_amdgcn_readfirstlane(k0);
  k1 = __builtin_amdgcn_readfirstlane(k1);
  f32x4 qf[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) qf[j] = *reinterpret_cast<const f32x4*>(Qh + size_t(qk) * 64 + j * 8 + hl * 4);

  const float sl2 = a.scale * 1.4426950408889634f;
  float m = NEG_INF, l = 0.0f;
  f32x16 o[2];
#pragma unroll
  for (int e = 0; e < 16; ++e) o[0][e] = o[1][e] = 0.0f;
  float most = 0.0f;  // the largest |value| met where keys are masked
  f32x4 kf[8];
  auto loadk = [&](int kb) __attribute__((always_inline)) {  // rows past the range repeat its last key
    const float* kr = Kh + size_t(min(kb + col, k1 - 1)) * 64 + hl * 4;
#pragma unroll
    for (int j = 0; j < 8; ++j) kf[j] = *reinterpret_cast<const f32x4*>(kr + j * 8);
  };
  if (k0 + wk * 32 < k1) loadk(k0 + wk * 32);
  for (int kb = k0 + wk * 32; kb < k1; kb += KW * 32) {
    float v[2][16];
    const bool whole = kb + 32 <= k1;
    const float* vr = Vh + size_t(kb + 4 * hl) * 64 + col;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int off = (e >> 2) * 8 + (e & 3);
      const float* p = whole ? vr + off * 64 : Vh + size_t(min(kb + 4 * hl + off, k1 - 1)) * 64 + col;
      v[0][e] = p[0];
      v[1][e] = p[32];
    }
    f32x16 s;
#pragma unroll
    for (int e = 0; e < 16; ++e) s[e] = 0.0f;
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
      for (int u = 0; u < 4; ++u) s = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[j][u], qf[j][u], s, 0, 0, 0);
    if (kb + KW * 32 < k1) loadk(kb + KW * 32);
    // Masks where the tile crosses the range's end or some query's window.
    const int kbase = kb + 4 * hl;
    int lo = 0, hi = k1 - kbase;
    bool edge = !whole;
    if (a.window >= 0) {
      lo = qk - a.window - kbase;
      hi = min(hi, qk + a.window + 1 - kbase);
      edge = edge || kb < wq0 + 31 - a.window || kb + 32 > wq0 + a.window + 1;
    }
    if (edge) {
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int off = (e >> 2) * 8 + (e & 3);
        s[e] = off >= lo && off < hi ? s[e] : NEG_INF;
      }
    }
    float mx = s[0];
#pragma unroll
    for (int e = 1; e < 16; ++e) mx = fmaxf(mx, s[e]);
    const float mn = fmaxf(m, half_max(mx) * sl2);
    const float ms = mn == NEG_INF ? 0.0f : mn;  // nothing visible yet
    const float alpha = __builtin_amdgcn_exp2f(m - ms);
    float psum = 0.0f;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      s[e] = __builtin_amdgcn_exp2f(fmaf(s[e], sl2, -ms));
      psum += s[e];
    }
    l = l * alpha + psum;
    m = mn;
    if (alpha != 1.0f) {
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        o[0][e] *= alpha;
        o[1][e] *= alpha;
      }
    }
    // Where keys are masked, a weight of 0 times a value that is not finite would be NaN: such a value
    // goes into the product as the largest finite one (NaN: the lowest), and to the queries that see
    // its key after the loop.
    if (edge) {
#pragma unroll
      for (int dt = 0; dt < 2; ++dt)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          v[dt][e] = __builtin_amdgcn_fmed3f(v[dt][e], -__FLT_MAX__, __FLT_MAX__);
          most = fmaxf(most, fabsf(v[dt][e]));
        }
    }
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      o[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(v[0][e], s[e], o[0], 0, 0, 0);
      o[1] = __builtin_amdgcn_mfma_f32_32x32x2f32(v[1][e], s[e], o[1], 0, 0, 0);
    }
  }
  uint32_t up = 0, down = 0;  // output elements that a value of +inf, of -inf (NaN: both) reaches
  if (__any(most == __FLT_MAX__)) {
    for (int kb = k0 + wk * 32; kb < k1; kb += KW * 32) {
      for (int key = kb; key < min(kb + 32, k1); ++key) {
        const float* vk = Vh + size_t(key) * 64 + 4 * hl;
        const bool seen = a.window < 0 || abs(key - qk) <= a.window;
        for (int e = 0; e < 32; ++e) {
          const float x = vk[(e >> 2) * 8 + (e & 3)];
          if (!seen || fabsf(x) < -NEG_INF) continue;
          if (x != NEG_INF) up |= 1u << e;
          if (x != -NEG_INF) down |= 1u << e;
        }
      }
    }
  }
  auto reached = [&](int e) __attribute__((always_inline)) {
    return ((up >> e & 1) ? -NEG_INF : 0.0f) + ((down >> e & 1) ? NEG_INF : 0.0f);
  };
  l = half_sum(l);
  float L = l, f[KW];
  if constexpr (KW > 1) {
    mt[wave * 64 + lane] = m;
    lt[wave * 64 + lane] = l;
#pragma unroll
    for (int e = 0; e < 32; ++e) ot[(wave * 32 + e) * 64 + lane] = o[e >> 4][e & 15];
    if (__any((up | down) != 0))
      for (int e = 0; e < 32; ++e) ot[(wave * 32 + e) * 64 + lane] += reached(e);
    __syncthreads();
    if (wk != 0) return;
    float M = m;
#pragma unroll
    for (int w = 1; w < KW; ++w) M = fmaxf(M, mt[(wave + w) * 64 + lane]);
    L = 0.0f;
#pragma unroll
    for (int w = 0; w < KW; ++w) {
      const float mw = mt[(wave + w) * 64 + lane];
      f[w] = mw == NEG_INF ? 0.0f : __builtin_amdgcn_exp2f(mw - M);
      L += lt[(wave + w) * 64 + lane] * f[w];
    }
  }
  if (!active || qi >= tl.q1) return;
  const float inv = 1.0f / L;
  const size_t oe = size_t(qi) * a.ldo + head * 64 + hl * 4;
#pragma unroll
  for (int dt = 0; dt < 2; ++dt)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      float r4[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int e = g * 4 + r;
        float acc = o[dt][e] + reached(dt * 16 + e);
        if constexpr (KW > 1) {
          acc *= f[0];
#pragma unroll
          for (int w = 1; w < KW; ++w) acc += ot[((wave + w) * 32 + dt * 16 + e) * 64 + lane] * f[w];
        }
        r4[r] = acc * inv;
      }
      store4_split(a.out, oe + dt * 32 + g * 8, r4, a.os);
    }
}

// Attention of single queries over a key set each (the padded layout's far padding queries, in the
// entry format of attn_fallback_launch): one wave per (entry, head), 64 keys a step, lane j scoring key j of the step against the query
// held in LDS, lane c accumulating output dim c; softmax with expf.
__global__ __launch_bounds__(64) void attn32_kernel(Attn32Args a) {
  __shared__ float sq[64];
  __shared__ float sp[64];
  const int fi = blockIdx.x / a.heads, head = blockIdx.x % a.heads;
  const int* e = a.entries + size_t(fi) * 8;  // query, a0, a1, b0, b1, lo, hi, zeros
  const int qrow = e[0], a0 = e[1], a1 = e[2], b0 = e[3], b1 = e[4], lo = e[5], hi = e[6], zeros = e[7];
  const int lane = threadIdx.x;
  const float* Qh = a.q + size_t(head) * a.T * 64;
  const float* Kh = a.k + size_t(head) * a.T * 64;
  const float* Vh = a.v + size_t(head) * a.T * 64;
  sq[lane] = Qh[size_t(qrow) * 64 + lane];
  __syncthreads();
  const int khi = (b1 > b0 ? b1 : a1) - 1;
  const float llo = logf(float(1 + lo)), lhi = logf(float(1 + hi));
  float m = -INFINITY, l = 0.0f, o = 0.0f;
  auto keys = [&](int j0, int j1) {
    for (int b = j0; b < j1; b += 64) {
      const int j = b + lane;
      float s = -INFINITY;
      if (j < j1) {
        const float4* kr = reinterpret_cast<const float4*>(Kh + size_t(j) * 64);
        float dot = 0.0f;
#pragma unroll
        for (int c = 0; c < 16; ++c) {
          const float4 kv = kr[c];
          dot = fmaf(sq[4 * c], kv.x, dot);
          dot = fmaf(sq[4 * c + 1], kv.y, dot);
          dot = fmaf(sq[4 * c + 2], kv.z, dot);
          dot = fmaf(sq[4 * c + 3], kv.w, dot);
        }
        s = dot * a.scale + (j == a0 ? llo : 0.0f) + (j == khi ? lhi : 0.0f);
      }
      const float mn = fmaxf(m, wave_max(s));
      const float p = j < j1 ? expf(s - mn) : 0.0f;
      const float alpha = m == -INFINITY ? 0.0f : expf(m - mn);
      l = l * alpha + wave_sum(p);
      o *= alpha;
      m = mn;
      sp[lane] = p;
      __syncthreads();
      const int cnt = min(64, j1 - b);
      for (int t = 0; t < cnt; ++t) o = fmaf(sp[t], Vh[size_t(b + t) * 64 + lane], o);
      __syncthreads();
    }
  };
  keys(a0, a1);
  keys(b0, b1);
  if (zeros > 0) {  // zero slots: score 0, value 0
    const float sz = logf(float(zeros));
    const float mn = fmaxf(m, sz);
    const float alpha = m == -INFINITY ? 0.0f : expf(m - mn);
    l = l * alpha + expf(sz - mn);
    o *= alpha;
  }
  const float r[2] = {o / l, 0.0f};
  uint32_t h16, l16;
  split_f16<2>(r, a.os, &h16, &l16);
  uint16_t* out = reinterpret_cast<uint16_t*>(a.out) + split_at(size_t(qrow) * a.ldo + head * 64 + lane);
  out[0] = uint16_t(h16);
  out[32] = uint16_t(l16);
}

// act[t, i] = gelu(x[t, i]) * x[t, I + i] over x [T, 2I], whole or the parts of a split product.
__global__ __launch_bounds__(256) void geglu32_kernel(const float* __restrict__ x, int splits, int T, int I,
                                                      float* __restrict__ act, float as) {
  const long long gid = (long long)blockIdx.x * 256 + threadIdx.x;
  const int n4 = I / 4;
  if (gid >= (long long)T * n4) return;
  const int t = int(gid / n4), i = int(gid % n4) * 4;
  const float* row = x + size_t(t) * 2 * I + i;
  const size_t plane = size_t(T) * 2 * I;
  const float4 a = sum_parts(row, splits, plane), g = sum_parts(row + I, splits, plane);
  const float v[4] = {gelu_exact(a.x) * g.x, gelu_exact(a.y) * g.y, gelu_exact(a.z) * g.z, gelu_exact(a.w) * g.w};
  store4_split(act, size_t(t) * I + i, v, as);
}

// out[r] = dot(x[r], w) + b over rows of K floats, one wave per row.
__global__ __launch_bounds__(64) void rowdot32_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                      const float* __restrict__ b, int K, float* __restrict__ out) {
  const float* row = x + size_t(blockIdx.x) * K;
  float acc = 0.0f;
  for (int o = threadIdx.x * 4; o < K; o += 256) {
    const float4 v = *reinterpret_cast<const float4*>(row + o), u = *reinterpret_cast<const float4*>(w + o);
    acc = fmaf(v.x, u.x, fmaf(v.y, u.y, fmaf(v.z, u.z, fmaf(v.w, u.w, acc))));
  }
  acc = wave_sum(acc);
  if (threadIdx.x == 0) out[blockIdx.x] = acc + b[0];
}

template <int BM, int BN, int WM, int WN, int STAGES>
void gemm32_t(const Gemm32Args& g, hipStream_t st) {
  const dim3 grid(unsigned((g.M + BM - 1) / BM) * unsigned(g.N / BN), unsigned(g.splits));
  hipLaunchKernelGGL((gemm32_kernel<BM, BN, WM, WN, STAGES>), grid, dim3(WM * WN * 64), 0, st, g);
}

// 64 x 128 tiles in two stages (48 KiB, three workgroups per CU) once there are two for every CU, else
// 64 x 64 in three. At 5707 rows, q|k|v: 64 x 128 119 us, in three stages 129, 192 x 128 119, 128 x 128
// 155, 256 x 128 in 8 waves 138. At 193 rows 32-row tiles gain at most 1 us in 10 and lose as much
// elsewhere.
bool wide32(int M, int N) { return (long long)((M + 63) / 64) * (N / 128) >= 512; }

}  // namespace

const char* gemm32_check(const Gemm32Args& g) {
  if (g.M < 0 || g.N <= 0 || g.K <= 0) return "f32 GEMM: empty shape";
  if (g.K % 32 || g.N % 128 || g.lda % 32 || g.ldw % 32 || g.ldc % 32) return "f32 GEMM: K and leading dimensions must be multiples of 32, N of 128";
  if (g.lda < g.K || g.ldw < g.K) return "f32 GEMM: bad leading dimension";
  if ((reinterpret_cast<uintptr_t>(g.A) | reinterpret_cast<uintptr_t>(g.W) | reinterpret_cast<uintptr_t>(g.C) |
       reinterpret_cast<uintptr_t>(g.bias) | reinterpret_cast<uintptr_t>(g.ws) | reinterpret_cast<uintptr_t>(g.wexp)) % 16)
    return "f32 GEMM: operands must be 16-byte aligned";
  if (size_t(std::max(g.lda, g.ldw)) * 128 * 4 > 0xffffffffu) return "f32 GEMM: a tile's rows must span less than 4 GiB";
  if (g.splits < 1 || g.splits > g.K / 32) return "f32 GEMM: splits must be in 1..K/32";
  if (g.splits > 1 && !g.ws) return "f32 GEMM: a split product needs a workspace";
  return nullptr;
}

int gemm32_splits(int M, int N, int K) {
  if (M <= 0 || wide32(M, N)) return 1;
  const int tiles = (M + 63) / 64 * (N / 64);
  const int kt = K / 32;
  // Three workgroups of 64 x 64 tiles share a CU, and a launch lasts as long as the CU with the most
  // parts of tiles: the split that makes that least, each part at least 4 k-tiles, its start and end
  // counted as 4 more, at most 8 parts, each counted as one k-tile where they are read back. At 193
  // rows of width 1024, against no split: q|k|v 14.0 -> 10.2 us (4 parts), Wo 10.2 -> 5.5 (4), Wo2 20.2 -> 9.0 (8);
  // Wi, 328 tiles, takes two rounds either way.
  int best = 1;
  long long least = 0;
  for (int s = 1; s <= 8 && s <= kt / 4; ++s) {
    const long long t = (long long)((tiles * s + 767) / 768) * ((kt + s - 1) / s + 4) + s;
    if (s == 1 || t < least) {
      best = s;
      least = t;
    }
  }
  return best;
}

void gemm32_launch(const Gemm32Args& g, hipStream_t st) {
  if (g.M <= 0) return;
  if (wide32(g.M, g.N)) gemm32_t<64, 128, 2, 2, 2>(g, st);
  else gemm32_t<64, 64, 2, 2, 3>(g, st);
  if (g.splits > 1 && g.C) {
    const long long n = (long long)g.M * (g.N / 4);
    hipLaunchKernelGGL(splitk32_kernel, dim3(unsigned((n + 255) / 256)), dim3(256), 0, st, g);
  }
}

void split32_launch(const float* qkv, int splits, const float* bias, int T, int d, const int* pos, const float* cos_t,
                    const float* sin_t, float* q, float* k, float* v, hipStream_t st) {
  const long long n = (long long)T * (d / 64) * 8;
  if (n <= 0) return;
  hipLaunchKernelGGL(split32_kernel, dim3(unsigned((n + 255) / 256)), dim3(256), 0, st, qkv, splits, bias, T, d, pos,
                     cos_t, sin_t, q, k, v);
}

int attn32_plan_tiles(const int* row_start, int n, int heads, int window, std::vector<int>& out, const int* q_end,
                      const int* k_end) {
  auto queries = [&](int r) { return (q_end ? q_end[r] : row_start[r + 1]) - row_start[r]; };
  // 128 queries per workgroup while that gives two workgroups per CU or more, else 64 or 32, whose
  // keys two or four waves share: the chain of key tiles is what a short batch waits for.
  int qb = 32;
  for (int c : {128, 64}) {
    long long tiles = 0;
    for (int r = 0; r < n; ++r) tiles += (queries(r) + c - 1) / c;
    if (tiles * heads >= 512) {
      qb = c;
      break;
    }
  }
  for (int r = 0; r < n; ++r) {
    const int rs = row_start[r], qe = rs + queries(r), ke = k_end ? k_end[r] : row_start[r + 1];
    for (int q0 = rs; q0 < qe; q0 += qb) {
      const int t[4] = {q0, std::min(q0 + qb, qe), rs, ke};
      out.insert(out.end(), t, t + 4);
    }
  }
  return qb;
}

void attn32_launch(const Attn32Args& a, hipStream_t st) {
  if (a.n <= 0) return;
  const dim3 grid(unsigned(a.n) * unsigned(a.heads));
  if (a.entries) hipLaunchKernelGGL(attn32_kernel, grid, dim3(64), 0, st, a);
  else if (a.tile_q == 128) hipLaunchKernelGGL(attn32_tile_kernel<1>, grid, dim3(256), 0, st, a);
  else if (a.tile_q == 64) hipLaunchKernelGGL(attn32_tile_kernel<2>, grid, dim3(256), 0, st, a);
  else hipLaunchKernelGGL(attn32_tile_kernel<4>, grid, dim3(256), 0, st, a);
}

void split_weight_launch(float* W, int N, int K, const float* bounds, int* wexp, hipStream_t st) {
  const size_t n = size_t(N) * K;
  hipLaunchKernelGGL(split_weight_kernel, dim3(unsigned((n + 255) / 256)), dim3(256), 0, st, W, n, K, bounds, wexp);
}

void weight_bound_launch(const float* W, const float* lw, const float* lb, const float* bias, int N, int K, float* out,
                         hipStream_t st) {
  hipLaunchKernelGGL(weight_bound_kernel, dim3(unsigned(N)), dim3(64), 0, st, W, lw, lb, bias, K, out);
}

void geglu32_launch(const float* x, int splits, int T, int I, float* act, float as, hipStream_t st) {
  const long long n = (long long)T * (I / 4);
  if (n <= 0) return;
  hipLaunchKernelGGL(geglu32_kernel, dim3(unsigned((n + 255) / 256)), dim3(256), 0, st, x, splits, T, I, act, as);
}

void rowdot32_launch(const float* x, const float* w, const float* b, int R, int K, float* out, hipStream_t st) {
  if (R <= 0) return;
  hipLaunchKernelGGL(rowdot32_kernel, dim3(unsigned(R)), dim3(64), 0, st, x, w, b, K, out);
}

}  // namespace s1
