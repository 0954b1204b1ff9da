// Kernels of the dtype=f32 path: the reference's BackendOptions::f32 (f32 weights and compute,
// runtime/crates/laya-core/src/backend.rs:25-27; laya-mlx/tests/parity.rs:54-65 checks it). Plain
// f32 arithmetic throughout: f32 matrix instructions for the products, an exact erf GELU, f32
// softmax.
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

// C[M, N] = A[M, K] . W[N, K]^T on v_mfma_f32_32x32x2_f32 (64 FLOP per clock and SIMD: the unit
// that bounds these products). BM x BN tiles in WM x WN waves, 32-float k-tiles (128-byte rows)
// moved global -> LDS by direct loads, STAGES deep, one barrier per k-tile; 16-byte chunk c of row
// r sits at slot c ^ ((r / 2) % 8), so the 16 rows of one fragment read phase start in 16 distinct
// bank groups.
//
// A k-step is 8 floats: lane (row l % 32, h = l / 32) reads 4 consecutive floats (chunk 2 ks + h)
// of its row with one access, and MFMA u of the step multiplies element u, i.e. k = 8 ks + u from
// the lanes of half 0 and k = 8 ks + 4 + u from half 1: both operands use the same order, so each
// k is met once. W is the first operand (C^T = W . A^T): a lane holds 4 consecutive columns of one
// row and stores them as one float4.
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
  auto issue = [&](int stage, int kt) __attribute__((always_inline)) {
    const int koff = __builtin_amdgcn_readfirstlane(kt * ROWB);
    char* sb = smem + stage * STAGE_BYTES + wave * 1024;
#pragma unroll
    for (int j = 0; j < LPW; ++j) load16_lds(j < AG / NW ? rsrcA : rsrcW, sb + j * NW * 1024, int(voff[j]), koff);
  };

  f32x16 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

#pragma unroll
  for (int s = 0; s < STAGES - 1; ++s)
    if (s < NK) issue(s, kt0 + s);
  const int lr = lane & 31, lh = lane >> 5;
  int ka[4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) ka[ks] = lr * ROWB + (((ks * 2 + lh) ^ ((lr >> 1) & 7)) << 4);
  for (int it = 0; it < NK; ++it) {
    wait_ahead<LPW, STAGES - 2>(min(STAGES - 2, NK - 1 - it));
    // Every wave's loads of k-tile `it` have landed and every wave is done with k-tile it - 1,
    // whose buffer the next issue overwrites.
    barrier_lds();
    if (it + STAGES - 1 < NK) issue((it + STAGES - 1) % STAGES, kt0 + it + STAGES - 1);
    const char* sa = smem + (it % STAGES) * STAGE_BYTES + wm * TM * ROWB;
    const char* sw = smem + (it % STAGES) * STAGE_BYTES + A_BYTES + wn * TN * ROWB;
    f32x4 fa[2][FM], fb[2][FN];
    auto frag = [&](int ks, int buf) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < FM; ++i) fa[buf][i] = *reinterpret_cast<const f32x4*>(sa + ka[ks] + i * 32 * ROWB);
#pragma unroll
      for (int j = 0; j < FN; ++j) fb[buf][j] = *reinterpret_cast<const f32x4*>(sw + ka[ks] + j * 32 * ROWB);
    };
    frag(0, 0);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      if (ks < 3) frag(ks + 1, (ks + 1) & 1);
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fb[ks & 1][j][u], fa[ks & 1][i][u], acc[i][j], 0, 0, 0);
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
        float v[4] = {acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
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
  *o = make_float4(old.x + act32(s.x + b.x, g.act), old.y + act32(s.y + b.y, g.act), old.z + act32(s.z + b.z, g.act),
                   old.w + act32(s.w + b.w, g.act));
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
// before this tile's softmax. Measured at 5707 tokens in 10 rows, 16 heads, against one wave per
// (query, head) on vector FMAs: global 1720 -> 245 us, local
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
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      o[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(v[0][e], s[e], o[0], 0, 0, 0);
      o[1] = __builtin_amdgcn_mfma_f32_32x32x2f32(v[1][e], s[e], o[1], 0, 0, 0);
    }
  }
  l = half_sum(l);
  float L = l, f[KW];
  if constexpr (KW > 1) {
    mt[wave * 64 + lane] = m;
    lt[wave * 64 + lane] = l;
#pragma unroll
    for (int e = 0; e < 32; ++e) ot[(wave * 32 + e) * 64 + lane] = o[e >> 4][e & 15];
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
  float* orow = a.out + size_t(qi) * a.ldo + head * 64 + hl * 4;
#pragma unroll
  for (int dt = 0; dt < 2; ++dt)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      float r4[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int e = g * 4 + r;
        float acc = o[dt][e];
        if constexpr (KW > 1) {
          acc *= f[0];
#pragma unroll
          for (int w = 1; w < KW; ++w) acc += ot[((wave + w) * 32 + dt * 16 + e) * 64 + lane] * f[w];
        }
        r4[r] = acc * inv;
      }
      *reinterpret_cast<float4*>(orow + dt * 32 + g * 8) = make_float4(r4[0], r4[1], r4[2], r4[3]);
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
  a.out[size_t(qrow) * a.ldo + head * 64 + lane] = o / l;
}

// act[t, i] = gelu(x[t, i]) * x[t, I + i] over x [T, 2I], whole or the parts of a split product.
__global__ __launch_bounds__(256) void geglu32_kernel(const float* __restrict__ x, int splits, int T, int I,
                                                      float* __restrict__ act) {
  const long long gid = (long long)blockIdx.x * 256 + threadIdx.x;
  const int n4 = I / 4;
  if (gid >= (long long)T * n4) return;
  const int t = int(gid / n4), i = int(gid % n4) * 4;
  const float* row = x + size_t(t) * 2 * I + i;
  const size_t plane = size_t(T) * 2 * I;
  const float4 a = sum_parts(row, splits, plane), g = sum_parts(row + I, splits, plane);
  *reinterpret_cast<float4*>(act + size_t(t) * I + i) =
      make_float4(gelu_exact(a.x) * g.x, gelu_exact(a.y) * g.y, gelu_exact(a.z) * g.z, gelu_exact(a.w) * g.w);
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

// Tiles by rows and columns: 64 x 128 once there are two for every CU, else 64 x 64, or 32 x 128
// where those leave fewer rows idle by a tenth of the product or more (193 rows: 224 instead of
// 256). At 5707 rows the 64 x 128 tiles in two stages (48 KiB, three workgroups per CU) run the
// five products of a layer and the head at 128-131 TFLOP/s, 64 x 64 ones at 125, and larger
// tiles, three or four stages, or the next fragments read across the barrier less: what counts is
// waves per SIMD to issue matrix instructions while others wait.
bool rows32(int M) { return ((M + 31) / 32) * 32 * 11 <= ((M + 63) / 64) * 64 * 10; }
bool wide32(int M, int N) { return (long long)((M + 63) / 64) * (N / 128) >= 512; }

}  // namespace

const char* gemm32_check(const Gemm32Args& g) {
  if (g.M < 0 || g.N <= 0 || g.K <= 0) return "f32 GEMM: empty shape";
  if (g.K % 32 || g.N % 128) return "f32 GEMM: K must be a multiple of 32, N of 128";
  if (g.lda < g.K || g.ldw < g.K || g.lda % 4 || g.ldw % 4 || g.ldc % 4) return "f32 GEMM: bad leading dimension";
  if ((reinterpret_cast<uintptr_t>(g.A) | reinterpret_cast<uintptr_t>(g.W) | reinterpret_cast<uintptr_t>(g.C) |
       reinterpret_cast<uintptr_t>(g.bias) | reinterpret_cast<uintptr_t>(g.ws)) % 16)
    return "f32 GEMM: operands must be 16-byte aligned";
  if (size_t(std::max(g.lda, g.ldw)) * 128 * 4 > 0xffffffffu) return "f32 GEMM: a tile's rows must span less than 4 GiB";
  if (g.splits < 1 || g.splits > g.K / 32) return "f32 GEMM: splits must be in 1..K/32";
  if (g.splits > 1 && !g.ws) return "f32 GEMM: a split product needs a workspace";
  return nullptr;
}

int gemm32_splits(int M, int N, int K) {
  if (M <= 0 || wide32(M, N)) return 1;
  const int tiles = rows32(M) ? (M + 31) / 32 * (N / 128) : (M + 63) / 64 * (N / 64);
  const int kt = K / 32;
  // A tile is matrix-unit time, so a launch lasts as long as the CU with the most parts of tiles:
  // the split that makes that least, each part at least 4 k-tiles, its start and end counted as 4
  // more, at most 8 parts (they are written and read back). At 193 rows of width 1024, against no
  // split: q|k|v 26 -> 18 us (3 parts), Wo 25 -> 9.4 (4), Wi 39 -> 30 (3), Wo2 57 -> 18 (4).
  int best = 1;
  long long least = 0;
  for (int s = 1; s <= 8 && s <= kt / 4; ++s) {
    const long long t = (long long)((tiles * s + 255) / 256) * ((kt + s - 1) / s + 4) + 2 * (s > 1);
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
  else if (rows32(g.M)) gemm32_t<32, 128, 1, 4, 2>(g, st);
  else gemm32_t<64, 64, 2, 2, 2>(g, st);
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

void geglu32_launch(const float* x, int splits, int T, int I, float* act, hipStream_t st) {
  const long long n = (long long)T * (I / 4);
  if (n <= 0) return;
  hipLaunchKernelGGL(geglu32_kernel, dim3(unsigned((n + 255) / 256)), dim3(256), 0, st, x, splits, T, I, act);
}

void rowdot32_launch(const float* x, const float* w, const float* b, int R, int K, float* out, hipStream_t st) {
  if (R <= 0) return;
  hipLaunchKernelGGL(rowdot32_kernel, dim3(unsigned(R)), dim3(64), 0, st, x, w, b, K, out);
}

}  // namespace s1
