// Fused attention for gfx950: softmax(q k^T * scale + mask) v over packed variable-length rows,
// one pass over the keys with an online softmax (f32 statistics), both products on MFMA.
//
// Replaces MLX's scaled_dot_product_attention on the encoder's global layers (pad mask only,
// runtime/crates/laya-mlx/src/lib.rs:1653-1656), its local layers (pad + |i - j| <= 64 window,
// lib.rs:1399-1417, 1644-1649; the banded form 1600-1622) and the decision head's attention
// (lib.rs:1710-1712). The reference's additive -1e4 masks give every masked key an exp() of
// exactly 0 in f32 for any query that has one visible key, which every real token has (itself),
// so a hard mask over the row's own keys computes the same values; padding never enters the
// packed layout at all.
//
// Work split: a workgroup of 4 wavefronts takes up to 128 queries of one sequence and one head;
// each wave owns 32 queries (64 in attn_wide_kernel, the global layers of batches that fill
// the GPU). Keys stream through LDS in chunks of 64 (double-buffered on global layers): K as [key][dim] and V as [dim][key], copied with 16-byte accesses from the
// transposed v buffer. On local layers waves skip chunks, and 32-key halves, outside their
// window, and only chunks that cross a window or row edge pay for masking. Short batches (fewer
// tiles than CUs) take 32-query tiles whose keys several waves split and merge at the end
// (attn_ksplit_kernel): all of the row's keys on global layers, the tile's window range on local
// ones.
//
// The products are computed transposed so that every softmax statistic lives in one lane:
//   S^T[key, q] = K . Q^T   (A = K rows from LDS, B = the wave's Q held in registers)
// lane l then holds query l % 32 and keys 8g + 4h + r (h = l / 32), so the row max and sum are a
// lane-local reduction plus one exchange with lane l ^ 32.
//   O^T[dim, q] += V^T . P^T
// reuses P^T straight from the S^T accumulators: within a 16-key MFMA step, operand slot
// 8h + j stands for key 16s + 8(j / 4) + 4h + (j % 4), and the V^T operand is read from LDS with
// the same key order, so no shuffle of P is needed.
//
// Softmax weights are 2^x by the bare v_exp_f32 (__builtin_amdgcn_exp2f): it flushes results
// below 2^-126 to 0, weights far below anything the f32 sums or the bf16 P can hold next to the
// row maximum's 1. exp2f wraps the instruction in a denormal-range fixup of five more VALU
// instructions per weight, and these kernels are VALU-bound.
#include <algorithm>
#include <vector>

#include "device.hpp"
#include "kernels.hpp"
#include "lds_load.hpp"

namespace s1 {

namespace {

constexpr int KC = 64;  // keys per chunk
constexpr float NEG_INF = -__builtin_huge_valf();

// LDS rows of 128 bytes (64 bf16: a K row, or 64 keys of a V^T row) hold 16-byte chunk c of row
// r at slot c ^ ((r / 2) % 8): the 16 rows of one 16-lane read phase then start in 16 distinct
// bank groups, and each 8-row group is one contiguous KiB that a single direct global -> LDS
// load (global_load_lds_dwordx4) fills.
__device__ __forceinline__ int kslot(int r, int c) { return c ^ ((r >> 1) & 7); }

// The launch is one-dimensional, ntiles x heads workgroups; workgroup -> (tile, head) with the
// tile fastest, through xcd_remap, so that consecutive tiles of one head (the query blocks of one
// row, which read the same keys and values, or overlapping windows of them) run on one XCD and
// share its L2.
__device__ __forceinline__ int2 tile_head(int ntiles) {
  const int lid = xcd_remap(blockIdx.x, gridDim.x);
  const int head = lid / ntiles;
  return make_int2(lid - head * ntiles, head);
}

// Three waves per SIMD for the local kernel (register budget 168), four for the global one.
template <class E, bool LOCAL>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(LOCAL ? 3 : 4)))
void attn_kernel(AttnArgs a) {
  typedef typename E::v8 v8;
  constexpr int NW = 4;  // wavefronts
  // K and V^T double buffers, [K0 | K1 | V0 | V1], 8 KiB each.
  __shared__ __attribute__((aligned(1024))) uint16_t smem[4 * KC * 64];
  auto sK = [&](int buf) { return smem + buf * KC * 64; };
  auto sVt = [&](int buf) { return smem + (2 + buf) * KC * 64; };

  const int2 th = tile_head(a.ntiles);
  const AttnTile tl = a.tiles[th.x];
  const int head = th.y;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform: scalar branches
  const int hl = lane >> 5;   // lane half
  const int col = lane & 31;  // query column within the wave

  const uint16_t* __restrict__ Qh = a.q + size_t(head) * a.Tq * 64;
  const uint16_t* __restrict__ Kh = a.k + size_t(head) * a.Tk * 64;
  const uint16_t* __restrict__ Vt = a.v + size_t(head) * 64 * a.ldv;

  const int wq0 = tl.q0 + wave * 32;
  const bool wave_active = wq0 < tl.q1;
  const int qi = wq0 + col;
  const bool qvalid = qi < tl.q1;
  const int qld = min(qi, tl.q1 - 1);
  const int qk = a.qkey ? a.qkey[qld] : qld;  // q row and key index of this query

  // Key range of the workgroup and of this wave.
  int kb0 = tl.k0, kb1 = tl.k1;
  int wk0 = tl.k0, wk1 = tl.k1;
  int wf_key = 0, wl_key = 0;  // key index of the wave's first and last query (local layers)
  if constexpr (LOCAL) {
    const int first = a.qkey ? a.qkey[tl.q0] : tl.q0;
    const int last = a.qkey ? a.qkey[tl.q1 - 1] : tl.q1 - 1;
    kb0 = max(tl.k0, first - a.window);
    kb1 = min(tl.k1, last + a.window + 1);
    if (wave_active) {
      const int wf = a.qkey ? a.qkey[wq0] : wq0;
      const int wlq = min(wq0 + 31, tl.q1 - 1);
      const int wl = a.qkey ? a.qkey[wlq] : wlq;
      wk0 = max(tl.k0, wf - a.window);
      wk1 = min(tl.k1, wl + a.window + 1);
      wf_key = wf;
      wl_key = wl;
    }
  }
  // Chunks start 8-aligned so the V^T rows are read with aligned 16-byte loads; keys before kb0
  // and from kb1 on are masked (and their V entries zeroed in LDS).
  const int cstart = kb0 & ~7;

  // This lane's slice of its query: dims 16kb + 8h .. +7 for kb = 0..3 (MFMA B operand).
  v8 qf[4];
#pragma unroll
  for (int kb = 0; kb < 4; ++kb)
    qf[kb] = *reinterpret_cast<const v8*>(Qh + size_t(qk) * 64 + kb * 16 + hl * 8);

  // A chunk's K goes global -> LDS by direct loads: 8 groups of 8 rows, one KiB each, spread
  // over the waves; rows past kb1 repeat the last key. V^T goes through registers (one 16-byte
  // piece of 8 keys per thread and wave of 64 threads per KiB): loaded with the K loads, stored
  // after the chunk's math. (Direct loads for V^T too make the compiler wait for all of them
  // before the chunk's first V^T read.) V^T pieces from kb1 on load the piece holding key
  // kb1 - 1 (finite values that meet weights of 0); that piece may read up to 7 keys past kb1:
  // the next sequence's, or the zeros every v writer leaves up to the next multiple of 8 tokens.
  const int vlast = cstart + (((kb1 - 1) - cstart) & ~7);
  constexpr int VPT = 64 * 8 / (NW * 64);  // V^T pieces per thread
  static_assert(VPT * NW * 64 == 64 * 8, "V^T pieces split evenly over the threads");
  uint4 vreg[VPT];
  auto stage = [&](int c0, int buf) {
    const int r8 = lane >> 3, slot = lane & 7;
    for (int gi = wave; gi < 8; gi += NW) {
      const int row = gi * 8 + r8;
      const uint16_t* src = Kh + size_t(min(c0 + row, kb1 - 1)) * 64 + kslot(row, slot) * 8;
      __builtin_amdgcn_global_load_lds(src, reinterpret_cast<char*>(sK(buf)) + gi * 1024, 16, 0, 0);
    }
#pragma unroll
    for (int it = 0; it < VPT; ++it) {
      const int p = tid + it * NW * 64;
      const int dim = p >> 3, c = p & 7;
      vreg[it] = *reinterpret_cast<const uint4*>(Vt + size_t(dim) * a.ldv + min(c0 + c * 8, vlast));
    }
  };
  // V^T rows hold each 16-key block's keys in the PV operand order: key 16s + 8a + 4h + r at
  // position 16s + 8h + 4a + r, so a lane's 8 operand keys (4h .. 4h + 3 and 8 + 4h .. 8 + 4h + 3
  // of the block) are one 16-byte chunk (2s + h), read with one access. The 16-byte chunks are
  // then placed by kslot like K's.
  auto vstore = [&](int buf) {
#pragma unroll
    for (int it = 0; it < VPT; ++it) {
      const int p = tid + it * NW * 64;
      const int dim = p >> 3, c = p & 7;  // keys 8c .. 8c + 7 = 16 (c / 2) + 8 (c % 2) + 0 .. 7
      uint16_t* row = sVt(buf) + dim * 64 + (c & 1) * 4;
      *reinterpret_cast<uint2*>(row + kslot(dim, c & ~1) * 8) = make_uint2(vreg[it].x, vreg[it].y);
      *reinterpret_cast<uint2*>(row + kslot(dim, c | 1) * 8) = make_uint2(vreg[it].z, vreg[it].w);
    }
  };
  auto landed = [] { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); };  // this wave's direct loads

  const float sl2 = a.scale * 1.4426950408889634f;  // fold log2(e): exp(x) = exp2(x log2 e)
  float m = NEG_INF, l = 0.0f;
  f32x16 o[2];
#pragma unroll
  for (int e = 0; e < 16; ++e) { o[0][e] = 0.0f; o[1][e] = 0.0f; }

  // Global layers double-buffer the chunks (the next chunk's loads overlap this one's math);
  // local layers visit few chunks per wave and keep the lighter single buffer, which leaves
  // registers for three waves per SIMD.
  constexpr bool DB = !LOCAL;
  if constexpr (DB) {
    stage(cstart, 0);
    vstore(0);
    landed();
    __syncthreads();
  }
  int buf = 0;
  for (int c0 = cstart; c0 < kb1; c0 += KC, buf ^= (DB ? 1 : 0)) {
    const bool more = DB && c0 + KC < kb1;
    if constexpr (DB) {
      if (more) stage(c0 + KC, buf ^ 1);  // the other buffer was last read before the previous barrier
    } else {
      if (c0 != cstart) __syncthreads();  // every wave is done with the previous chunk
      stage(c0, 0);
      vstore(0);
      landed();
      __syncthreads();
    }
    bool work = wave_active;
    if constexpr (LOCAL) work = work && !(c0 + KC <= wk0 || c0 >= wk1);
    if (work) {
      // 32-key tiles of this chunk that hold keys this wave may see (local layers skip the rest).
      bool need[2] = {true, true};
      if constexpr (LOCAL) {
#pragma unroll
        for (int t = 0; t < 2; ++t) need[t] = c0 + 32 * t < wk1 && c0 + 32 * t + 32 > wk0;
      }
      // Masks are needed only where the chunk crosses the key range or some query's window.
      bool edge = c0 < kb0 || c0 + KC > kb1;
      if constexpr (LOCAL) edge = edge || c0 < wl_key - a.window || c0 + KC > wf_key + a.window + 1;
      // S^T for the needed 32-key tiles (raw logits; masked entries -inf): the K fragments of the
      // chunk read first, then the two tiles' k-steps interleaved (two independent MFMA chains).
      f32x16 s[2];
      float mx = NEG_INF;
      v8 kf[2][4];
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const int kr = t * 32 + col;
          if (need[t]) kf[t][kb] = *reinterpret_cast<const v8*>(sK(buf) + kr * 64 + kslot(kr, kb * 2 + hl) * 8);
        }
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) s[t][e] = need[t] ? 0.0f : NEG_INF;
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int t = 0; t < 2; ++t)
          if (need[t]) s[t] = E::mfma(kf[t][kb], qf[kb], s[t]);
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        if (!need[t]) continue;
        if (edge) {
          // Element e of the tile is key kbase + (e / 4) * 8 + e % 4: bounds on that constant
          // offset, one compare per element for each side the chunk crosses.
          const int kbase = c0 + t * 32 + hl * 4;
          if constexpr (LOCAL) {
            const int lo = max(kb0, qk - a.window) - kbase, hi = min(kb1, qk + a.window + 1) - kbase;
#pragma unroll
            for (int e = 0; e < 16; ++e) {
              const int off = (e >> 2) * 8 + (e & 3);
              s[t][e] = off >= lo && off < hi ? s[t][e] : NEG_INF;
            }
          } else {
            if (c0 < kb0) {
              const int lo = kb0 - kbase;
#pragma unroll
              for (int e = 0; e < 16; ++e) s[t][e] = (e >> 2) * 8 + (e & 3) >= lo ? s[t][e] : NEG_INF;
            }
            if (c0 + KC > kb1) {
              const int hi = kb1 - kbase;
#pragma unroll
              for (int e = 0; e < 16; ++e) s[t][e] = (e >> 2) * 8 + (e & 3) < hi ? s[t][e] : NEG_INF;
            }
          }
        }
#pragma unroll
        for (int e = 0; e < 16; ++e) mx = fmaxf(mx, s[t][e]);
      }
      // Online softmax in base 2: p = 2^(s * sl2 - m). sl2 > 0, so the raw max scales.
      mx = half_max(mx);
      const float mn = fmaxf(m, mx * sl2);
      const float ms = mn == NEG_INF ? 0.0f : mn;  // nothing visible yet: every p is exp2(-inf) = 0
      const float alpha = __builtin_amdgcn_exp2f(m - ms);
      float psum = 0.0f;
      v8 pf[2][2];
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int sb = 0; sb < 2; ++sb)
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const float p = __builtin_amdgcn_exp2f(fmaf(s[t][sb * 8 + j], sl2, -ms));
            psum += p;
            pf[t][sb][j] = typename E::scalar(p);
          }
      l = l * alpha + psum;
      m = mn;
      // Once the running maximum settles, alpha is exactly 1 on every lane and the branch (taken
      // by lanes, skipped by the wave when none needs it) saves the 32 multiplies.
      if (alpha != 1.0f) {
#pragma unroll
        for (int e = 0; e < 16; ++e) { o[0][e] *= alpha; o[1][e] *= alpha; }
      }

      // O^T += V^T . P^T over the needed tiles (MFMA k-steps of 16 keys), both 32-dim halves.
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        if (!need[t]) continue;
#pragma unroll
        for (int sb = 0; sb < 2; ++sb) {
#pragma unroll
          for (int dt = 0; dt < 2; ++dt) {
            const int dr = dt * 32 + col;
            const v8 vf = *reinterpret_cast<const v8*>(sVt(buf) + dr * 64 + kslot(dr, (t * 2 + sb) * 2 + hl) * 8);
            o[dt] = E::mfma(vf, pf[t][sb], o[dt]);
          }
        }
      }
    }
    if constexpr (DB) {
      if (more) {
        vstore(buf ^ 1);  // the other buffer was last read before the previous barrier
        landed();
      }
      __syncthreads();
    }
  }

  if (!wave_active) return;
  const float lt = half_sum(l);
  if (!qvalid) return;
  const float inv = 1.0f / lt;
  uint16_t* orow = a.out + size_t(qi) * a.ldo + head * 64;
#pragma unroll
  for (int dt = 0; dt < 2; ++dt)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int dim = dt * 32 + g * 8 + hl * 4;
      uint2 w;
      w.x = E::pack2(o[dt][g * 4 + 0] * inv, o[dt][g * 4 + 1] * inv);
      w.y = E::pack2(o[dt][g * 4 + 2] * inv, o[dt][g * 4 + 3] * inv);
      *reinterpret_cast<uint2*>(orow + dim) = w;
    }
}

// 16 bytes of a result row: a caller's out is aligned to 8 only.
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef u32x4 u32x4_a8 __attribute__((aligned(8)));

// Global layers of batches that fill the GPU: a wave owns 64 queries, as two halves of 32, and a
// workgroup of 4 waves the same 256 queries that 8 waves of 32 would. Each K and V^T fragment read
// from LDS then feeds two MFMAs, and half 1's softmax weights are computed beside half 0's V^T P^T
// products. Two waves per SIMD: by counters a SIMD spends 475k cycles on VALU issue (an exp2 costs
// two FMAs) and 262k on MFMAs at 8192 keys and 16 heads; at equal priority a launch took their
// sum, 709k (counted before V^T went through registers), and takes 592k now. The priority raised
// over the weights and the V^T P^T products lets one wave's vector work go ahead while the other's
// K Q^T products run (raised over K Q^T, or from the row maximum on, it gains nothing). With this
// and the order of the tiles, against 8 waves of 32 queries, 16 heads:
// 8192 keys 336 -> 310 µs (890 TFLOP/s), 10 rows of 547 to 579 tokens 34.1 -> 30.6, 12 of 300 to
// 1100 61.3 -> 51.8, 48 of 215 to 2038 510 -> 481. The same work with 32 queries per wave and four
// waves per SIMD (128 registers, 10 spilled) is 2 to 7% slower, and V^T in its own order in LDS, by direct loads, with a
// lane's 8 keys read as two 8-byte halves, 1 to 6%. For 128-query tiles, about one wave per SIMD,
// attn_kernel is faster (6 rows of 286 to 391 tokens, 12 heads: 11.6 against 13.8 µs with two
// waves of 64).
//
// The next chunk's loads run during this one's math; layouts and sums are attn_kernel's (the same
// bits).
//
// Workgroup b takes head b % heads of tile b / heads; the tiles come longest key range first
// (attn_plan_tiles), so that the short ones fill what the long ones leave at the end. Workgroups
// go round the 8 XCDs, so a head stays on one XCD's L2 (on two where heads are a multiple of 4 only).
constexpr int WQ = 256;  // queries per workgroup
template <class E>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void attn_wide_kernel(AttnArgs a) {
  typedef typename E::v8 v8;
  constexpr int QH = 2;        // query halves of a wave
  constexpr int CB = KC * 64;  // elements of a staged chunk
  __shared__ __attribute__((aligned(1024))) uint16_t smem[4 * CB];  // [K0 | V0 | K1 | V1]

  const AttnTile tl = a.tiles[blockIdx.x / a.heads];
  const int head = blockIdx.x % a.heads;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
  const int hl = lane >> 5, col = lane & 31;
  const uint16_t* __restrict__ Qh = a.q + size_t(head) * a.Tq * 64;
  const uint16_t* __restrict__ Kh = a.k + size_t(head) * a.Tk * 64;
  const uint16_t* __restrict__ Vt = a.v + size_t(head) * 64 * a.ldv;

  const int wq0 = tl.q0 + wave * QH * 32;
  const bool wave_active = wq0 < tl.q1;
  const int kb0 = tl.k0, kb1 = tl.k1;
  const int cstart = kb0 & ~7;  // V^T rows are read in aligned pieces of 8 keys
  const int vlast = cstart + (((kb1 - 1) - cstart) & ~7);

  v8 qf[QH][4];  // dims 16 kb + 8 h .. + 7 of this lane's two queries
#pragma unroll
  for (int qh = 0; qh < QH; ++qh) {
    const int qi = min(wq0 + qh * 32 + col, tl.q1 - 1);
    const uint16_t* qp = Qh + size_t(a.qkey ? a.qkey[qi] : qi) * 64 + hl * 8;
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) qf[qh][kb] = *reinterpret_cast<const v8*>(qp + kb * 16);
  }

  // A chunk's 16 KiB: wave w moves row groups 2w and 2w + 1 of K and of V^T (8 rows of 128 bytes
  // each), K by direct global -> LDS loads, V^T through registers. K rows past kb1 repeat the last key; V^T pieces past it repeat the piece that holds it,
  // which may hold up to 7 keys past kb1: the next row's, or the zeros that every writer of v
  // leaves up to a multiple of 8 tokens. Those meet weights of 0.
  const int r8 = lane >> 3, slot = lane & 7;
  uint4 vreg[2];
  auto stage = [&](int c0, int buf) __attribute__((always_inline)) {
    char* dst = reinterpret_cast<char*>(smem + buf * 2 * CB);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int gi = wave * 2 + i, row = gi * 8 + r8;
      __builtin_amdgcn_global_load_lds(Kh + size_t(min(c0 + row, kb1 - 1)) * 64 + kslot(row, slot) * 8, dst + gi * 1024,
                                       16, 0, 0);
      vreg[i] = *reinterpret_cast<const uint4*>(Vt + size_t(row) * a.ldv + min(c0 + slot * 8, vlast));
    }
  };
  auto vstore = [&](int buf) __attribute__((always_inline)) {
    uint16_t* sv = smem + buf * 2 * CB + CB;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int row = (wave * 2 + i) * 8 + r8;
      uint16_t* p = sv + row * 64 + (slot & 1) * 4;
      *reinterpret_cast<uint2*>(p + kslot(row, slot & ~1) * 8) = make_uint2(vreg[i].x, vreg[i].y);
      *reinterpret_cast<uint2*>(p + kslot(row, slot | 1) * 8) = make_uint2(vreg[i].z, vreg[i].w);
    }
  };

  const float sl2 = a.scale * 1.4426950408889634f;  // exp(x) = exp2(x log2 e)
  float m[QH], l[QH];
  f32x16 o[QH][2];
#pragma unroll
  for (int qh = 0; qh < QH; ++qh) {
    m[qh] = NEG_INF;
    l[qh] = 0.0f;
#pragma unroll
    for (int e = 0; e < 16; ++e) o[qh][0][e] = o[qh][1][e] = 0.0f;
  }

  int fo[4];  // LDS element offsets of this lane's fragments, of K and of V^T alike
#pragma unroll
  for (int i = 0; i < 4; ++i) fo[i] = col * 64 + kslot(col, i * 2 + hl) * 8;

  auto chunk = [&](int c0, int buf) __attribute__((always_inline)) {
    const bool edge = c0 < kb0 || c0 + KC > kb1;
    const uint16_t* sk = smem + buf * 2 * CB;
    const uint16_t* sv = sk + CB;
    v8 kf[2][4];
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
      for (int t = 0; t < 2; ++t) kf[t][kb] = *reinterpret_cast<const v8*>(sk + t * 32 * 64 + fo[kb]);
    f32x16 s[QH][2];
#pragma unroll
    for (int qh = 0; qh < QH; ++qh) {
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) s[qh][t][e] = 0.0f;
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int t = 0; t < 2; ++t) s[qh][t] = E::mfma(kf[t][kb], qf[qh][kb], s[qh][t]);
    }
    if (edge) {  // only the first and the last chunk hold keys outside the range
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const int kbase = c0 + t * 32 + hl * 4, lo = kb0 - kbase, hi = kb1 - kbase;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int off = (e >> 2) * 8 + (e & 3);
          const bool in = off >= lo && off < hi;
#pragma unroll
          for (int qh = 0; qh < QH; ++qh) s[qh][t][e] = in ? s[qh][t][e] : NEG_INF;
        }
      }
    }
    float alpha[QH], ms[QH];
#pragma unroll
    for (int qh = 0; qh < QH; ++qh) {
      float mx = NEG_INF;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) mx = fmaxf(mx, s[qh][t][e]);
      const float mn = fmaxf(m[qh], half_max(mx) * sl2);
      ms[qh] = mn == NEG_INF ? 0.0f : mn;  // nothing visible yet: every p is exp2(-inf) = 0
      alpha[qh] = __builtin_amdgcn_exp2f(m[qh] - ms[qh]);
      m[qh] = mn;
    }
    if (alpha[0] != 1.0f || alpha[QH - 1] != 1.0f) {  // skipped by the wave once its maxima have settled
#pragma unroll
      for (int qh = 0; qh < QH; ++qh) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          o[qh][0][e] *= alpha[qh];
          o[qh][1][e] *= alpha[qh];
        }
      }
    }
    __builtin_amdgcn_s_setprio(1);
    v8 vf[2][4], pf[4];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int dt = 0; dt < 2; ++dt) vf[dt][ks] = *reinterpret_cast<const v8*>(sv + dt * 32 * 64 + fo[ks]);
#pragma unroll
    for (int qh = 0; qh < QH; ++qh) {
      float psum = 0.0f;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const float p = __builtin_amdgcn_exp2f(fmaf(s[qh][t][e], sl2, -ms[qh]));
          psum += p;
          pf[t * 2 + (e >> 3)][e & 7] = typename E::scalar(p);
        }
      l[qh] = l[qh] * alpha[qh] + psum;
#pragma unroll
      for (int ks = 0; ks < 4; ++ks)
#pragma unroll
        for (int dt = 0; dt < 2; ++dt) o[qh][dt] = E::mfma(vf[dt][ks], pf[ks], o[qh][dt]);
    }
    __builtin_amdgcn_s_setprio(0);
  };

  stage(cstart, 0);
  vstore(0);
  wait_vmcnt<0>();
  __syncthreads();
  int buf = 0;
  for (int c0 = cstart; c0 < kb1; c0 += KC, buf ^= 1) {
    const bool more = c0 + KC < kb1;
    if (more) stage(c0 + KC, buf ^ 1);  // that buffer was last read before the last barrier
    if (wave_active) chunk(c0, buf);
    if (more) vstore(buf ^ 1);
    wait_vmcnt<0>();
    __syncthreads();
  }

  if (!wave_active) return;
  // The wave's 64 rows leave through its own 8 KiB of LDS (every wave is past its last read), so
  // that a store writes whole 128-byte rows: chunk c of row r at slot c ^ (r % 8).
  uint16_t* st = smem + wave * QH * 32 * 64;
#pragma unroll
  for (int qh = 0; qh < QH; ++qh) {
    const float inv = 1.0f / half_sum(l[qh]);
#pragma unroll
    for (int dt = 0; dt < 2; ++dt)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const uint2 w = make_uint2(E::pack2(o[qh][dt][g * 4 + 0] * inv, o[qh][dt][g * 4 + 1] * inv),
                                   E::pack2(o[qh][dt][g * 4 + 2] * inv, o[qh][dt][g * 4 + 3] * inv));
        *reinterpret_cast<uint2*>(st + (qh * 32 + col) * 64 + ((dt * 4 + g) ^ (col & 7)) * 8 + hl * 4) = w;
      }
  }
  wave_lds_fence();
#pragma unroll
  for (int i = 0; i < QH * 4; ++i) {
    const int r = i * 8 + r8;
    const u32x4 v = *reinterpret_cast<const u32x4*>(st + r * 64 + (slot ^ (r & 7)) * 8);
    if (wq0 + r < tl.q1) *reinterpret_cast<u32x4_a8*>(a.out + size_t(wq0 + r) * a.ldo + head * 64 + slot * 8) = v;
  }
}

// Local layers with a window of at most 64 keys: a workgroup's 128 queries see at most
// 128 + 2 * 64 keys, so the whole key range is staged in LDS at once (every load of the
// workgroup in flight together, one barrier) and each wave then runs its queries' softmax over
// its own window in a single pass (at most 6 tiles of 32 keys, raw logits kept in registers).
// K and V^T take turns in one LDS buffer (38 KiB): K for the logits, then V^T, loaded while the
// softmax weights are computed. At the 10-request headline that fits four workgroups per CU,
// all 800 tiles in one round, where K and V^T side by side (71 KiB) fit two and took 1.56
// rounds (16.4 -> 15.0 µs per launch, the same bits). The results leave as whole rows through
// LDS: 48 rows of 215 to 2038 tokens 108 -> 92 µs, 10 of 547 to 579 16.5 -> 15.5 (the same bits).
constexpr int LQ = 128;                 // queries per workgroup: 4 waves x 32
constexpr int LMAXW = 64;               // largest window this kernel stages
constexpr int LMAXK = LQ + 2 * LMAXW + 8;  // staged keys: the range plus 8-alignment slack
// V^T rows in LDS: LVC 16-byte chunks of 8 keys (LVC odd, so the 16 rows of one 16-lane read
// phase start in 16 distinct bank groups); LVC x 8 >= LMAXK rounded up to 32 keys, the furthest
// column a tile reads. Each KiB of the 64 rows is filled by one direct global -> LDS load.
constexpr int LVC = 37;
constexpr int LVW = LVC * 8;
constexpr int LTILES = (32 + 2 * LMAXW + 7 + 31) / 32;  // 32-key tiles a wave's window spans
constexpr int LBUF = LMAXK * 64 > 64 * LVW ? LMAXK * 64 : 64 * LVW;  // 16-bit elements of the buffer
static_assert(LVC % 2 == 1 && LVC * 8 >= (LMAXK + 31) / 32 * 32 && 64 * LVC % 64 == 0, "V^T layout");

template <class E>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void attn_local_kernel(AttnArgs a) {
  typedef typename E::v8 v8;
  __shared__ __attribute__((aligned(1024))) uint16_t sbuf[LBUF];
  uint16_t* const sK = sbuf;   // [LMAXK][64] until every wave has its logits
  uint16_t* const sVt = sbuf;  // then [64][LVW]

  const int2 th = tile_head(a.ntiles);
  const AttnTile tl = a.tiles[th.x];
  const int head = th.y;
  const int tid = threadIdx.x, lane = tid & 63;
  // Wave-uniform values go through readfirstlane so the branches on them are scalar branches,
  // not exec-mask regions around every tile.
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hl = lane >> 5, col = lane & 31;
  const int W = a.window;

  const uint16_t* __restrict__ Qh = a.q + size_t(head) * a.Tq * 64;
  const uint16_t* __restrict__ Kh = a.k + size_t(head) * a.Tk * 64;
  const uint16_t* __restrict__ Vt = a.v + size_t(head) * 64 * a.ldv;

  // The workgroup's keys [kb0, kb1), staged from the 8-aligned cstart (keys outside them are
  // masked out of S, so their weights are exactly 0 and their V entries only need be finite).
  const int kb0 = max(tl.k0, tl.q0 - W), kb1 = min(tl.k1, tl.q1 + W);
  const int cstart = kb0 & ~7;
  const int nk8 = (kb1 - cstart + 7) >> 3;  // 8-key groups staged (<= LMAXK / 8)
  const int lim = nk8 * 8;                  // staged keys
  // A wave past the tile's queries computes nothing but takes part in both barriers.
  const int wq0 = tl.q0 + wave * 32;
  const bool wact = wq0 < tl.q1;
  const int qi = wq0 + col;
  const int qk = min(qi, tl.q1 - 1);
  v8 qf[4];
#pragma unroll
  for (int kb = 0; kb < 4; ++kb)
    qf[kb] = *reinterpret_cast<const v8*>(Qh + size_t(qk) * 64 + kb * 16 + hl * 8);
  // K by direct global -> LDS loads: 8-row groups, groups w, w + 4, ... from wave w; rows past
  // kb1 repeat the last key (masked out of S).
  {
    const int r = lane >> 3, slot = lane & 7;
    for (int gi = wave; gi < nk8; gi += 4) {
      const int row = gi * 8 + r;
      const uint16_t* src = Kh + size_t(min(cstart + row, kb1 - 1)) * 64 + kslot(row, slot) * 8;
      __builtin_amdgcn_global_load_lds(src, reinterpret_cast<char*>(sK) + gi * 1024, 16, 0, 0);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's direct loads have landed
  }
  __syncthreads();

  // This wave's window: keys [ws, we) cover every query's |key - q| <= W within the row.
  const int ws = max(kb0, wq0 - W), we = min(kb1, min(wq0 + 31, tl.q1 - 1) + W + 1);
  int t0 = (ws - cstart) & ~7;                 // LDS key offset of the first tile
  const int nt = wact ? __builtin_amdgcn_readfirstlane((we - cstart - t0 + 31) >> 5) : 0;  // tiles (<= LTILES)
  // Shift the tiles left so they end within the staged keys (keys before ws are masked); a range
  // shorter than the tiles starts at 0 and reads up to the zeroed V^T columns.
  if (t0 + 32 * nt > lim) t0 = max(0, lim - 32 * nt);
  t0 = __builtin_amdgcn_readfirstlane(t0);

  // Keys this lane's query sees, as LDS key offsets: [vlo, vhi). Tiles inside the band that every
  // query of the wave sees, [blo, bhi), need no mask.
  const int vlo = max(kb0, qk - W) - cstart, vhi = min(kb1, qk + W + 1) - cstart;
  const int blo = __builtin_amdgcn_readfirstlane(max(kb0, min(wq0 + 31, tl.q1 - 1) - W) - cstart);
  const int bhi = __builtin_amdgcn_readfirstlane(min(kb1, wq0 + W + 1) - cstart);
  f32x16 s[LTILES];
  float mx = NEG_INF;
#pragma unroll
  for (int t = 0; t < LTILES; ++t) {
#pragma unroll
    for (int e = 0; e < 16; ++e) s[t][e] = NEG_INF;
    if (t >= nt) continue;
    f32x16 acc;
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[e] = 0.0f;
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      const int kr = t0 + t * 32 + col;
      const v8 kf = *reinterpret_cast<const v8*>(&sK[kr * 64 + kslot(kr, kb * 2 + hl) * 8]);
      acc = E::mfma(kf, qf[kb], acc);
    }
    const int tb = t0 + t * 32;  // LDS key offset of the tile
    if (tb >= blo && tb + 32 <= bhi) {
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        s[t][e] = acc[e];
        mx = fmaxf(mx, acc[e]);
      }
    } else {
      const int lo = vlo - tb - hl * 4, hi = vhi - tb - hl * 4;  // bounds on (e >> 2) * 8 + (e & 3)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int off = (e >> 2) * 8 + (e & 3);
        s[t][e] = off >= lo && off < hi ? acc[e] : NEG_INF;
        mx = fmaxf(mx, s[t][e]);
      }
    }
  }
  __syncthreads();  // every wave has read K
  // V^T into the same buffer: chunk S of the 64 x LVC chunks is row S / LVC, keys
  // cstart + 8 (S % LVC) .. + 7. Chunks from kb1 on load the chunk holding key kb1 - 1 instead:
  // finite values that meet weights of 0. The chunk holding kb1 - 1 may read up to 7 keys past
  // kb1, which are the next sequence's or the zeros every v writer leaves up to the next
  // multiple of 8 tokens.
  {
    const int last = cstart + (((kb1 - 1) - cstart) & ~7);
    for (int i = wave; i < LVC; i += 4) {
      const int S = i * 64 + lane;
      const int dim = S / LVC, c = S - dim * LVC;
      const int key = min(cstart + 8 * c, last);
      __builtin_amdgcn_global_load_lds(Vt + size_t(dim) * a.ldv + key, reinterpret_cast<char*>(sVt) + i * 1024, 16, 0,
                                       0);
    }
  }
  // The softmax weights while V^T lands. Every real query sees itself, so the row maximum is
  // finite.
  const float sl2 = a.scale * 1.4426950408889634f;
  const float ms = wact ? half_max(mx) * sl2 : 0.0f;
  float psum = 0.0f;
  v8 pf[LTILES][2];
#pragma unroll
  for (int t = 0; t < LTILES; ++t) {
    if (t >= nt) continue;
#pragma unroll
    for (int sb = 0; sb < 2; ++sb)
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float p = __builtin_amdgcn_exp2f(fmaf(s[t][sb * 8 + j], sl2, -ms));
        psum += p;
        pf[t][sb][j] = typename E::scalar(p);
      }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (!wact) return;  // a wave that has ended takes no part in the barrier that follows
  f32x16 o[2];
#pragma unroll
  for (int e = 0; e < 16; ++e) { o[0][e] = 0.0f; o[1][e] = 0.0f; }
#pragma unroll
  for (int t = 0; t < LTILES; ++t) {
    if (t >= nt) continue;
#pragma unroll
    for (int sb = 0; sb < 2; ++sb) {
      const int kbase = t0 + t * 32 + sb * 16 + hl * 4;
#pragma unroll
      for (int dt = 0; dt < 2; ++dt) {
        const uint16_t* vr = &sVt[(dt * 32 + col) * LVW];
        const uint2 lo = *reinterpret_cast<const uint2*>(vr + kbase);
        const uint2 hi = *reinterpret_cast<const uint2*>(vr + kbase + 8);
        const uint4 pk = make_uint4(lo.x, lo.y, hi.x, hi.y);
        const v8 vf = *reinterpret_cast<const v8*>(&pk);
        o[dt] = E::mfma(vf, pf[t][sb], o[dt]);
      }
    }
  }
  // The wave's 32 rows leave through its own 4 KiB of the buffer once every wave has read V^T, so
  // that a store writes whole 128-byte rows: chunk c of row r at slot c ^ (r % 8).
  const float inv = 1.0f / half_sum(psum);
  __syncthreads();
  uint16_t* st = sbuf + wave * 32 * 64;
#pragma unroll
  for (int dt = 0; dt < 2; ++dt)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *reinterpret_cast<uint2*>(st + col * 64 + ((dt * 4 + g) ^ (col & 7)) * 8 + hl * 4) =
          make_uint2(E::pack2(o[dt][g * 4 + 0] * inv, o[dt][g * 4 + 1] * inv),
                     E::pack2(o[dt][g * 4 + 2] * inv, o[dt][g * 4 + 3] * inv));
  wave_lds_fence();
  const int r8 = lane >> 3, slot = lane & 7;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = i * 8 + r8;
    const u32x4 v = *reinterpret_cast<const u32x4*>(st + r * 64 + (slot ^ (r & 7)) * 8);
    if (wq0 + r < tl.q1) *reinterpret_cast<u32x4_a8*>(a.out + size_t(wq0 + r) * a.ldo + head * 64 + slot * 8) = v;
  }
}



// Global attention for a short batch (one request): a workgroup of KW waves takes 32 queries of
// one row and head, and wave w visits the row's key chunks w, w + KW, ... with softmax statistics
// of its own; the KW partial results merge through LDS at the end (the online-softmax
// combination). A short row then runs KW times as many waves, each with 1/KW of the chain of
// dependent chunks. Each wave stages its own chunks in a private 16 KiB of LDS (K rows and V^T
// in the layouts attn_kernel uses), so the chunk loop has no barriers; the next chunk is loaded
// into registers during this one's math and stored after it (a wave's LDS accesses run in
// order), which keeps 4 waves at 64 KiB (two workgroups per CU) and 8 at 128 KiB.
// LOCAL: a local layer's short batch; the tile's keys are its window range, and every key
// outside a query's own window (|key - query| > a.window) is masked.
template <class E, int KW, bool LOCAL>
__global__ __launch_bounds__(KW * 64) __attribute__((amdgpu_waves_per_eu(2))) void attn_ksplit_kernel(AttnArgs a) {
  typedef typename E::v8 v8;
  constexpr int REG = KC * 64;  // 16-bit elements of one 8 KiB K or V^T chunk
  // [wave] x (K | V^T); after the chunk loop the same memory holds the merge tables.
  __shared__ __attribute__((aligned(1024))) uint16_t smem[KW * 2 * REG];

  const int2 th = tile_head(a.ntiles);
  const AttnTile tl = a.tiles[th.x];
  const int head = th.y;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hl = lane >> 5, col = lane & 31;
  const uint16_t* __restrict__ Qh = a.q + size_t(head) * a.Tq * 64;
  const uint16_t* __restrict__ Kh = a.k + size_t(head) * a.Tk * 64;
  const uint16_t* __restrict__ Vt = a.v + size_t(head) * 64 * a.ldv;
  uint16_t* const sK = smem + wave * 2 * REG;
  uint16_t* const sVt = sK + REG;

  const int qi = tl.q0 + col;
  const bool qvalid = qi < tl.q1;
  const int qld = min(qi, tl.q1 - 1);
  const int qk = a.qkey ? a.qkey[qld] : qld;  // q row of this slot
  const int kb0 = tl.k0, kb1 = tl.k1;
  const int cstart = kb0 & ~7;
  const int vlast = cstart + (((kb1 - 1) - cstart) & ~7);
  v8 qf[4];
#pragma unroll
  for (int kb = 0; kb < 4; ++kb)
    qf[kb] = *reinterpret_cast<const v8*>(Qh + size_t(qk) * 64 + kb * 16 + hl * 8);

  // A chunk in registers: 16-byte piece p = lane + 64 it is K row p / 8, slot p % 8 (rows past
  // kb1 repeat the last key), and V^T dim p / 8, keys 8 (p % 8) .. + 7 (from kb1 on, the piece
  // holding key kb1 - 1; it may read up to 7 keys past kb1, the next sequence's or the zeros
  // every v writer leaves up to the next multiple of 8 tokens).
  uint4 kreg[8], vreg[8];
  auto load = [&](int c0) {
#pragma unroll
    for (int it = 0; it < 8; ++it) {
      const int p = lane + it * 64;
      const int r = p >> 3, c = p & 7;
      kreg[it] = *reinterpret_cast<const uint4*>(Kh + size_t(min(c0 + r, kb1 - 1)) * 64 + c * 8);
      vreg[it] = *reinterpret_cast<const uint4*>(Vt + size_t(r) * a.ldv + min(c0 + c * 8, vlast));
    }
  };
  auto store = [&] {  // K rows by kslot; V^T in the PV operand order of attn_kernel
#pragma unroll
    for (int it = 0; it < 8; ++it) {
      const int p = lane + it * 64;
      const int r = p >> 3, c = p & 7;
      const uint4 kv = kreg[it];
      *reinterpret_cast<uint4*>(sK + r * 64 + kslot(r, c) * 8) = make_uint4(kv.x, kv.y, kv.z, kv.w);
      uint16_t* row = sVt + r * 64 + (c & 1) * 4;
      *reinterpret_cast<uint2*>(row + kslot(r, c & ~1) * 8) = make_uint2(vreg[it].x, vreg[it].y);
      *reinterpret_cast<uint2*>(row + kslot(r, c | 1) * 8) = make_uint2(vreg[it].z, vreg[it].w);
    }
  };

  const float sl2 = a.scale * 1.4426950408889634f;
  float m = NEG_INF, l = 0.0f;
  f32x16 o[2];
#pragma unroll
  for (int e = 0; e < 16; ++e) { o[0][e] = 0.0f; o[1][e] = 0.0f; }

  int c0 = cstart + wave * KC;
  if (c0 < kb1) {
    load(c0);
    store();
  }
  for (; c0 < kb1; c0 += KW * KC) {
    const bool more = c0 + KW * KC < kb1;
    if (more) load(c0 + KW * KC);
    f32x16 s[2];
    float mx = NEG_INF;
    // As in attn_kernel: the chunk's K fragments first, the two tiles' k-steps interleaved, and
    // one-sided masks on chunks that cross the key range.
    v8 kf[2][4];
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const int kr = t * 32 + col;
        kf[t][kb] = *reinterpret_cast<const v8*>(sK + kr * 64 + kslot(kr, kb * 2 + hl) * 8);
      }
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int e = 0; e < 16; ++e) s[t][e] = 0.0f;
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
      for (int t = 0; t < 2; ++t) s[t] = E::mfma(kf[t][kb], qf[kb], s[t]);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int kbase = c0 + t * 32 + hl * 4;
      if constexpr (LOCAL) {
        // A 32-query tile's window range is at most 160 keys: every chunk crosses some edge.
        const int lo = max(kb0, qk - a.window) - kbase, hi = min(kb1, qk + a.window + 1) - kbase;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int kk = (e >> 2) * 8 + (e & 3);
          s[t][e] = kk >= lo && kk < hi ? s[t][e] : NEG_INF;
        }
      } else {
      if (c0 < kb0) {
        const int lo = kb0 - kbase;
#pragma unroll
        for (int e = 0; e < 16; ++e) s[t][e] = (e >> 2) * 8 + (e & 3) >= lo ? s[t][e] : NEG_INF;
      }
      if (c0 + KC > kb1) {
        const int hi = kb1 - kbase;
#pragma unroll
        for (int e = 0; e < 16; ++e) s[t][e] = (e >> 2) * 8 + (e & 3) < hi ? s[t][e] : NEG_INF;
      }
      }
#pragma unroll
      for (int e = 0; e < 16; ++e) mx = fmaxf(mx, s[t][e]);
    }
    mx = half_max(mx);
    const float mn = fmaxf(m, mx * sl2);
    const float ms = mn == NEG_INF ? 0.0f : mn;
    const float alpha = __builtin_amdgcn_exp2f(m - ms);
    float psum = 0.0f;
    v8 pf[2][2];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int sb = 0; sb < 2; ++sb)
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float p = __builtin_amdgcn_exp2f(fmaf(s[t][sb * 8 + j], sl2, -ms));
          psum += p;
          pf[t][sb][j] = typename E::scalar(p);
        }
    l = l * alpha + psum;
    m = mn;
    if (alpha != 1.0f) {
#pragma unroll
      for (int e = 0; e < 16; ++e) { o[0][e] *= alpha; o[1][e] *= alpha; }
    }
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int sb = 0; sb < 2; ++sb)
#pragma unroll
        for (int dt = 0; dt < 2; ++dt) {
          const int dr = dt * 32 + col;
          const v8 vf = *reinterpret_cast<const v8*>(sVt + dr * 64 + kslot(dr, (t * 2 + sb) * 2 + hl) * 8);
          o[dt] = E::mfma(vf, pf[t][sb], o[dt]);
        }
    if (more) store();  // after this chunk's reads
  }

  // Merge: wave w leaves (m, l, o) per lane in LDS; wave 0 combines them. A wave that visited no
  // chunk has m = -inf and contributes 0.
  const float lw = half_sum(l);
  __syncthreads();  // every wave is done with its chunk buffers
  float* mt = reinterpret_cast<float*>(smem);  // [KW][64] m, [KW][64] l, [KW][32][64] o
  float* lt = mt + KW * 64;
  float* ot = lt + KW * 64;
  mt[wave * 64 + lane] = m;
  lt[wave * 64 + lane] = lw;
#pragma unroll
  for (int e = 0; e < 32; ++e) ot[(wave * 32 + e) * 64 + lane] = o[e >> 4][e & 15];
  __syncthreads();
  if (wave != 0 || !qvalid) return;
  float M = NEG_INF;
#pragma unroll
  for (int w = 0; w < KW; ++w) M = fmaxf(M, mt[w * 64 + lane]);
  float f[KW], L = 0.0f;
#pragma unroll
  for (int w = 0; w < KW; ++w) {
    const float mw = mt[w * 64 + lane];
    f[w] = mw == NEG_INF ? 0.0f : __builtin_amdgcn_exp2f(mw - M);
    L += lt[w * 64 + lane] * f[w];
  }
  const float inv = 1.0f / L;
  uint16_t* orow = a.out + size_t(qi) * a.ldo + head * 64;
#pragma unroll
  for (int dt = 0; dt < 2; ++dt)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      float v[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int e = dt * 16 + g * 4 + r;
        float acc = 0.0f;
#pragma unroll
        for (int w = 0; w < KW; ++w) acc += ot[(w * 32 + e) * 64 + lane] * f[w];
        v[r] = acc * inv;
      }
      const int dim = dt * 32 + g * 8 + hl * 4;
      *reinterpret_cast<uint2*>(orow + dim) = make_uint2(E::pack2(v[0], v[1]), E::pack2(v[2], v[3]));
    }
}

// Attention of the padded layout's padding queries that the local-attention tiles do not take:
// those whose softmax the reference's masks leave over a key set other than the real keys of
// the window. Each entry names the set, as the host works it out from the masks
// (lib.rs:1241-1310): {query, a0, a1, b0, b1, lo, hi, zeros} = keys [a0, a1) and [b0, b1) (packed
// indices), key a0 counted 1 + lo times, the last key of the last non-empty range 1 + hi times
// (gathered slots clamped to one key), and `zeros` slots of zero key and value (score 0, value 0).
//
// A workgroup takes a tile of up to 32 consecutive entries of one row and one head; its four waves
// take the 32-key tiles of the entries' key ranges (their unions, from the host) in turn and merge
// through LDS, and each lane masks the keys that its own query's entry does not name. The weights
// stay in f32: the scores come from the 16-bit MFMA (S^T = K . Q^T) and the weighted sum from the
// f32 one (v_mfma_f32_32x32x2: step 4g + r takes keys 8g + r and 8g + 4 + r, so its second operand
// is the lane's own weight). Loads go straight to registers: the sets are a few hundred keys that
// the tiles of a row share through L2, and what bounds the kernel is each wave's chain of about
// three key tiles. Measured at 1780 entries of 64 to 320 keys, 16 heads, against one wave per
// (entry, head) on vector FMAs: 156 -> 20.7 us (20.3 without the care for values that are not finite).
template <class E>
__global__ __launch_bounds__(256) void attn_far_kernel(FallbackArgs a) {
  typedef typename E::v8 v8;
  constexpr int KW = 4;
  __shared__ float mt[KW * 64], lt[KW * 64], ot[KW * 32 * 64];
  const int lid = xcd_remap(blockIdx.x, gridDim.x);
  const int head = lid / a.ntiles;
  const int* tile = a.tiles + size_t(lid - head * a.ntiles) * 8;
  const int e0 = tile[0], e1 = tile[1];
  const int lane = threadIdx.x & 63, hl = lane >> 5, col = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ei = min(e0 + col, e1 - 1);
  const int4 f0 = reinterpret_cast<const int4*>(a.far)[2 * ei];      // query, a0, a1, b0
  const int4 f1 = reinterpret_cast<const int4*>(a.far)[2 * ei + 1];  // b1, lo, hi, zeros
  const uint16_t* __restrict__ Qh = a.q + size_t(head) * a.T * 64;
  const uint16_t* __restrict__ Kh = a.k + size_t(head) * a.T * 64;
  const uint16_t* __restrict__ Vt = a.v + size_t(head) * 64 * a.ldv;
  v8 qf[4];
#pragma unroll
  for (int kb = 0; kb < 4; ++kb)
    qf[kb] = *reinterpret_cast<const v8*>(Qh + size_t(f0.x) * 64 + kb * 16 + hl * 8);
  const float sl2 = a.scale * 1.4426950408889634f;
  // Repeated keys: the weight of n copies is exp2(s + log2 n).
  const int klo = f0.y, khi = (f1.x > f0.w ? f1.x : f0.z) - 1;
  const float llo = log2f(float(1 + f1.y)), lhi = log2f(float(1 + f1.z));
  float m = NEG_INF, l = 0.0f;
  f32x16 o[2];
#pragma unroll
  for (int e = 0; e < 16; ++e) o[0][e] = o[1][e] = 0.0f;
  float most = 0.0f;  // the largest |value| met
  // 32-key tiles start 8-aligned, so V^T is read in aligned pieces of 4 keys; pieces past the range
  // repeat the one of its last key (values that meet weights of 0).
  const int first[2] = {tile[2] & ~7, tile[4] & ~7}, end[2] = {tile[3], tile[5]};
  const int na = (end[0] - first[0] + 31) >> 5, nb = (end[1] - first[1] + 31) >> 5;
  for (int t = wave; t < na + nb; t += KW) {
    const bool isb = t >= na;
    const int kb = isb ? first[1] + (t - na) * 32 : first[0] + t * 32, last = (isb ? end[1] : end[0]) - 1;
    const int r0 = isb ? f0.w : f0.y, r1 = isb ? f1.x : f0.z;  // this query's keys of the range
    const uint16_t* kr = Kh + size_t(min(kb + col, last)) * 64 + hl * 8;
    v8 kf[4];
    uint2 vr[2][4];
#pragma unroll
    for (int j = 0; j < 4; ++j) kf[j] = *reinterpret_cast<const v8*>(kr + j * 16);
#pragma unroll
    for (int dt = 0; dt < 2; ++dt)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        vr[dt][g] = *reinterpret_cast<const uint2*>(Vt + size_t(dt * 32 + col) * a.ldv + min(kb + 8 * g + 4 * hl, last & ~3));
    f32x16 s;
#pragma unroll
    for (int e = 0; e < 16; ++e) s[e] = 0.0f;
#pragma unroll
    for (int j = 0; j < 4; ++j) s = E::mfma(kf[j], qf[j], s);
    const int kbase = kb + 4 * hl;
    float mx = NEG_INF;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int key = kbase + (e >> 2) * 8 + (e & 3);
      s[e] = fmaf(s[e], sl2, (key == klo ? llo : 0.0f) + (key == khi ? lhi : 0.0f));
      s[e] = key >= r0 && key < r1 ? s[e] : NEG_INF;
      mx = fmaxf(mx, s[e]);
    }
    const float mn = fmaxf(m, half_max(mx));
    const float ms = mn == NEG_INF ? 0.0f : mn;  // nothing visible yet
    const float alpha = __builtin_amdgcn_exp2f(m - ms);
    float psum = 0.0f;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      s[e] = __builtin_amdgcn_exp2f(s[e] - ms);
      psum += s[e];
    }
    l = l * alpha + psum;
    m = mn;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      o[0][e] *= alpha;
      o[1][e] *= alpha;
    }
    // A weight of 0 times a value that is not finite is NaN: such a value goes into the product as the
    // largest finite one (NaN: the lowest), and to the queries that name its key after the loop.
#pragma unroll
    for (int e = 0; e < 16; ++e) {
#pragma unroll
      for (int dt = 0; dt < 2; ++dt) {
        const uint32_t w = (e & 2) ? vr[dt][e >> 2].y : vr[dt][e >> 2].x;
        const float v = __builtin_amdgcn_fmed3f(E::f32(uint16_t((e & 1) ? w >> 16 : w)), -__FLT_MAX__, __FLT_MAX__);
        most = fmaxf(most, fabsf(v));
        o[dt] = __builtin_amdgcn_mfma_f32_32x32x2f32(v, s[e], o[dt], 0, 0, 0);
      }
    }
  }
  uint32_t up = 0, down = 0;  // output elements that a value of +inf, of -inf (NaN: both) reaches
  if (__any(most == __FLT_MAX__)) {
    for (int t = wave; t < na + nb; t += KW) {
      const bool isb = t >= na;
      const int kb = isb ? first[1] + (t - na) * 32 : first[0] + t * 32, stop = isb ? end[1] : end[0];
      const int r0 = isb ? f0.w : f0.y, r1 = isb ? f1.x : f0.z;
      for (int key = kb; key < min(kb + 32, stop); ++key) {
        const bool seen = key >= r0 && key < r1;
        for (int e = 0; e < 32; ++e) {
          const float v = E::f32(Vt[size_t((e >> 2) * 8 + 4 * hl + (e & 3)) * a.ldv + key]);
          if (!seen || fabsf(v) < __builtin_huge_valf()) continue;
          if (v != NEG_INF) up |= 1u << e;
          if (v != -NEG_INF) down |= 1u << e;
        }
      }
    }
  }
  l = half_sum(l);
  if (wave == 0 && f1.w > 0) {  // zero slots: score 0, value 0, weight `zeros`
    const float sz = log2f(float(f1.w));
    const float mn = fmaxf(m, sz);
    const float alpha = __builtin_amdgcn_exp2f(m - mn);
    l = l * alpha + __builtin_amdgcn_exp2f(sz - mn);
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      o[0][e] *= alpha;
      o[1][e] *= alpha;
    }
    m = mn;
  }
  mt[wave * 64 + lane] = m;
  lt[wave * 64 + lane] = l;
#pragma unroll
  for (int e = 0; e < 32; ++e) ot[(wave * 32 + e) * 64 + lane] = o[e >> 4][e & 15];
  if (__any((up | down) != 0))
    for (int e = 0; e < 32; ++e)
      ot[(wave * 32 + e) * 64 + lane] += ((up >> e & 1) ? -NEG_INF : 0.0f) + ((down >> e & 1) ? NEG_INF : 0.0f);
  __syncthreads();
  // Wave w combines and stores dims 8 w .. 8 w + 7 of both halves' pieces: g = w of each 32 dims.
  if (e0 + col >= e1) return;
  float M = NEG_INF;
#pragma unroll
  for (int w = 0; w < KW; ++w) M = fmaxf(M, mt[w * 64 + lane]);
  float f[KW], L = 0.0f;
#pragma unroll
  for (int w = 0; w < KW; ++w) {
    f[w] = __builtin_amdgcn_exp2f(mt[w * 64 + lane] - M);
    L += lt[w * 64 + lane] * f[w];
  }
  const float inv = 1.0f / L;
  uint16_t* orow = a.out + size_t(f0.x) * a.ldo + head * 64 + wave * 8 + hl * 4;
#pragma unroll
  for (int dt = 0; dt < 2; ++dt) {
    float v[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int e = dt * 16 + wave * 4 + r;
      float acc = 0.0f;
#pragma unroll
      for (int w = 0; w < KW; ++w) acc += ot[(w * 32 + e) * 64 + lane] * f[w];
      v[r] = acc * inv;
    }
    *reinterpret_cast<uint2*>(orow + dt * 32) = make_uint2(E::pack2(v[0], v[1]), E::pack2(v[2], v[3]));
  }
}

}  // namespace

// Query count of row r: up to q_end[r] when given, else the whole row.
static int row_queries(const int* row_start, const int* q_end, int r) {
  return (q_end ? q_end[r] : row_start[r + 1]) - row_start[r];
}

// Local layers: 128-query tiles (attn_local_kernel) while they give at least one workgroup per
// CU; a shorter batch takes 32-query tiles whose keys are the tile's window range, split over 4
// waves (attn_ksplit_kernel<LOCAL>). Windows wider than attn_local_kernel stages keep 128.
static int local_tile(const int* row_start, const int* q_end, int n, int heads, int window) {
  if (window > LMAXW) return LQ;
  long long c = 0;
  for (int r = 0; r < n; ++r) c += (row_queries(row_start, q_end, r) + LQ - 1) / LQ;
  return c * heads >= 256 ? LQ : 32;
}
int attn_local_tile(const int* row_start, int n, int heads, int window) {
  return local_tile(row_start, nullptr, n, heads, window);
}

int attn_row_step(int len, int qb) {
  if (qb <= 32) return qb;
  const int nt = (len + qb - 1) / qb;
  const int wave = qb == WQ ? 64 : 32;  // queries of a wave
  return std::min(qb, ((len + nt - 1) / nt + wave - 1) / wave * wave);
}

// 256-query tiles (attn_wide_kernel, every K/V chunk shared by 256 queries) while they give at
// least one workgroup per CU; then 128 (4 waves) while they give 128 workgroups; a shorter batch takes
// 32-query tiles whose keys are split over 4 waves (attn_ksplit_kernel).
static int global_tile(const int* row_start, const int* q_end, int n, int heads) {
  auto count = [&](int qb) {
    long long c = 0;
    for (int r = 0; r < n; ++r) c += (row_queries(row_start, q_end, r) + qb - 1) / qb;
    return c * heads;
  };
  if (count(256) >= 256) return 256;
  if (count(128) >= 128) return 128;
  return 32;  // attn_ksplit_kernel
}
int attn_global_tile(const int* row_start, int n, int heads) { return global_tile(row_start, nullptr, n, heads); }

int attn_plan_tiles(const int* row_start, int n, int heads, int window, std::vector<int>& out, const int* q_end,
                    const int* k_end) {
  const int qb = window >= 0 ? local_tile(row_start, q_end, n, heads, window) : global_tile(row_start, q_end, n, heads);
  const size_t first = out.size();
  for (int r = 0; r < n; ++r) {
    const int rs = row_start[r], qe = q_end ? q_end[r] : row_start[r + 1], ke = k_end ? k_end[r] : row_start[r + 1];
    const int step = attn_row_step(qe - rs, qb);
    for (int q0 = rs; q0 < qe; q0 += step) {
      const int q1 = std::min(q0 + step, qe);
      const bool win = window >= 0 && qb == 32;
      out.push_back(q0);
      out.push_back(q1);
      out.push_back(win ? std::max(rs, q0 - window) : rs);
      out.push_back(win ? std::min(ke, q1 + window) : ke);
    }
  }
  if (window < 0 && qb == WQ) {  // attn_wide_kernel: most keys first
    std::vector<AttnTile> tiles;
    for (size_t i = first; i < out.size(); i += 4) tiles.push_back({out[i], out[i + 1], out[i + 2], out[i + 3]});
    std::stable_sort(tiles.begin(), tiles.end(),
                     [](const AttnTile& x, const AttnTile& y) { return x.k1 - x.k0 > y.k1 - y.k0; });
    out.resize(first);
    for (const AttnTile& t : tiles) out.insert(out.end(), {t.q0, t.q1, t.k0, t.k1});
  }
  return qb;
}

template <class E>
void attn_launch_t(const AttnArgs& a, hipStream_t st) {
  const dim3 grid(a.ntiles * a.heads);
  if (a.window >= 0 && a.window <= LMAXW && !a.qkey && a.tile_q == 32)
    hipLaunchKernelGGL((attn_ksplit_kernel<E, 4, true>), grid, dim3(256), 0, st, a);
  else if (a.window >= 0 && a.window <= LMAXW && !a.qkey)
    hipLaunchKernelGGL(attn_local_kernel<E>, grid, dim3(256), 0, st, a);  // tiles of <= LQ queries
  else if (a.window >= 0)
    hipLaunchKernelGGL((attn_kernel<E, true>), grid, dim3(256), 0, st, a);
  else if (a.tile_q == 256)
    hipLaunchKernelGGL(attn_wide_kernel<E>, grid, dim3(256), 0, st, a);
  else if (a.tile_q == 128)
    hipLaunchKernelGGL((attn_kernel<E, false>), grid, dim3(256), 0, st, a);
  else if (a.key_waves == 8)  // tile_q 32
    hipLaunchKernelGGL((attn_ksplit_kernel<E, 8, false>), grid, dim3(512), 0, st, a);
  else
    hipLaunchKernelGGL((attn_ksplit_kernel<E, 4, false>), grid, dim3(256), 0, st, a);
}

void attn_launch(const AttnArgs& a, hipStream_t st) {
  if (a.ntiles <= 0) return;
  if (a.elem == ELEM_F16) attn_launch_t<F16>(a, st);
  else attn_launch_t<Bf16>(a, st);
}

void attn_fallback_launch(const FallbackArgs& a, hipStream_t st) {
  if (a.ntiles <= 0) return;
  const dim3 grid(unsigned(a.ntiles) * unsigned(a.heads));
  if (a.elem == ELEM_F16) hipLaunchKernelGGL(attn_far_kernel<F16>, grid, dim3(256), 0, st, a);
  else hipLaunchKernelGGL(attn_far_kernel<Bf16>, grid, dim3(256), 0, st, a);
}

void attn_far_tiles(const std::vector<int>& far, const int* row_far, int n, std::vector<int>& out) {
  for (int r = 0; r < n; ++r)
    for (int e0 = row_far[r]; e0 < row_far[r + 1]; e0 += 32) {
      const int e1 = std::min(e0 + 32, row_far[r + 1]);
      int u[4] = {0, 0, 0, 0};  // union of the entries' non-empty a ranges, then of their b ranges
      for (int i = 0; i < 2; ++i) {
        bool any = false;
        for (int e = e0; e < e1; ++e) {
          const int k0 = far[size_t(e) * 8 + 1 + 2 * i], k1 = far[size_t(e) * 8 + 2 + 2 * i];
          if (k1 <= k0) continue;
          u[2 * i] = any ? std::min(u[2 * i], k0) : k0;
          u[2 * i + 1] = any ? std::max(u[2 * i + 1], k1) : k1;
          any = true;
        }
      }
      const int t[8] = {e0, e1, u[0], u[1], u[2], u[3], 0, 0};
      out.insert(out.end(), t, t + 8);
    }
}

}  // namespace s1
