// Batched (many-token) kernels for gfx950: the prompt is processed as T rows
// at once instead of T decode steps (the reference prefills token by token,
// llama-wgsl-runtime.ts:276-289; the K/V it leaves in the cache and the last
// prompt token's logits are what must match).
//
// Linear layers are dequant-fused GEMMs on the matrix cores (gemm_int.hip; decode
// batches of up to 64 rows below). fp16 MFMA keeps fp32-class accuracy by
// splitting the operands into hi + lo halves:
//   W * 2^ws = Wh + Wl,  x * 2^rs = xh + xl  (per token row),
//   sum W x = 2^-(ws+rs) * (Wh xh + Wh xl + Wl xh)   (Wl xl ~ 2^-22, dropped)
// accumulated in fp32 by gfx950's v_mfma_f32_16x16x32_f16.
#include <hip/hip_runtime.h>
#include <cstdlib>
#include <cstring>

#include <algorithm>

#include "kernel_common.h"
#include "kernels.h"
#include "prefill.h"

namespace chonk {
namespace {

typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef float float2_t __attribute__((ext_vector_type(2)));
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
// gfx950's double-K shape: lane l holds row (or column) l % 16 and 8 consecutive
// k of the 32 (the same k for both operands, so the product is the dot over k)
__device__ __forceinline__ float4_t mfma32(half8_t a, half8_t b, float4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

constexpr int kMaxDeferSplit = 16;  // K split of a deferred GEMM (loads of a sum issued together)

// Elements j[e] (valid columns) of row t of a deferred result: the partials
// are read four splits at a time, every load of a round issued before any is
// added (split indices past ks are clamped to the last split and their sums
// not taken, so no load sits behind a branch: a conditional load makes the
// compiler wait for every outstanding load where the paths join); the sums
// add the partials in split order. With ks <= 4 a call costs one memory round
// trip for all N elements.
// part_gather in two halves, so that the first round's loads can be issued
// early and summed where the values are needed: part_issue loads splits 0..3
// (clamped to the last split) of elements j[e]; part_finish adds them in split
// order and reads any further splits four at a time.
template <int N>
__device__ __forceinline__ void part_issue(const PartSum& P, int t, const int (&j)[N], float (&w)[N][4]) {
  const float* q = P.p + (int64_t)t * P.ld;
#pragma unroll
  for (int e = 0; e < N; ++e)
#pragma unroll
    for (int z = 0; z < 4; ++z) w[e][z] = q[(int64_t)min(z, P.ks - 1) * P.zs + j[e]];
}
template <int N>
__device__ __forceinline__ void part_finish(const PartSum& P, int t, const int (&j)[N], float (&w)[N][4],
                                            float (&v)[N]) {
  const float* q = P.p + (int64_t)t * P.ld;
#pragma unroll
  for (int e = 0; e < N; ++e) {
    v[e] = w[e][0];
#pragma unroll
    for (int z = 1; z < 4; ++z) v[e] = z < P.ks ? v[e] + w[e][z] : v[e];
  }
  for (int z0 = 4; z0 < P.ks; z0 += 4) {
#pragma unroll
    for (int e = 0; e < N; ++e)
#pragma unroll
      for (int z = 0; z < 4; ++z) w[e][z] = q[(int64_t)min(z0 + z, P.ks - 1) * P.zs + j[e]];
#pragma unroll
    for (int e = 0; e < N; ++e)
#pragma unroll
      for (int z = 0; z < 4; ++z) v[e] = z0 + z < P.ks ? v[e] + w[e][z] : v[e];
  }
}

// Elements j[e] (valid columns) of row t of a deferred result: the partials
// are read four splits at a time, every load of a round issued before any is
// added (split indices past ks are clamped to the last split and their sums
// not taken, so no load sits behind a branch: a conditional load makes the
// compiler wait for every outstanding load where the paths join); the sums
// add the partials in split order. With ks <= 4 a call costs one memory round
// trip for all N elements.
template <int N>
__device__ __forceinline__ void part_gather(const PartSum& P, int t, const int (&j)[N], float (&v)[N]) {
  if (P.ks == 1) {
    const float* q = P.p + (int64_t)t * P.ld;
#pragma unroll
    for (int e = 0; e < N; ++e) v[e] = q[j[e]];
    return;
  }
  float w[N][4];
  part_issue<N>(P, t, j, w);
  part_finish<N>(P, t, j, w, v);
}

// ---- per-row glue -----------------------------------------------------------------
//
// TPR threads of a 256-thread workgroup hold a token row in registers, E runs of
// eight consecutive elements each (run c0 + TPR e is elements 8 (c0 + TPR e) ..
// + 7): 16-byte loads and stores throughout, and the planes' 16-byte pieces are
// written whole. With a wave per row (TPR = 64, passes of many rows) the four
// rows of a workgroup write neighbouring pieces, and the row sums need no LDS or
// barrier; short passes spread a row over two or four waves instead.

template <int TPR>
struct RowLane {
  int t, c0, wave;  // token row (clamped), first run, wave of the workgroup
  bool ok;          // false: past the last row (computes along, stores nothing)
  __device__ __forceinline__ explicit RowLane(int rows) {
    const int tid = threadIdx.x, r = (int)blockIdx.x * (kWg / TPR) + tid / TPR;
    t = min(r, rows - 1);
    c0 = tid % TPR;
    wave = tid >> 6;
    ok = r < rows;
  }
};

template <int TPR, bool MAX>
__device__ __forceinline__ float row_reduce(float v, const RowLane<TPR>& L, float* red) {
  v = MAX ? wave_max(v) : wave_sum(v);
  if constexpr (TPR > 64) {
    constexpr int W = TPR / 64;
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[L.wave] = v;
    __syncthreads();
    const float* r = red + L.wave / W * W;
    v = r[0];
#pragma unroll
    for (int w = 1; w < W; ++w) v = MAX ? fmaxf(v, r[w]) : v + r[w];
  }
  return v;
}

__device__ __forceinline__ void load8(const float* p, float (&v)[8]) {
  const float4 a = ldg4f(p), b = ldg4f(p + 4);
  v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w;
  v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
}

// 16-byte loads of the result's rows are aligned (uniform)
__device__ __forceinline__ bool part_aligned(const PartSum& P) {
  return ((P.ld | (int)P.zs) & 3) == 0 && ((uintptr_t)P.p & 15) == 0;
}

// Columns col .. col + 7 of row t of a deferred result, the splits added in
// order, four splits' loads in flight (as part_gather).
__device__ __forceinline__ void part8(const PartSum& P, bool vec, int t, int col, float (&v)[8]) {
  const float* q = P.p + (int64_t)t * P.ld + col;
  auto load = [&](int z, float (&w)[8]) {
    const float* r = q + (int64_t)z * P.zs;
    if (vec) {
      load8(r, w);
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) w[i] = r[i];
    }
  };
  load(0, v);
  for (int z0 = 1; z0 < P.ks; z0 += 4) {
    float w[4][8];
#pragma unroll
    for (int z = 0; z < 4; ++z) load(min(z0 + z, P.ks - 1), w[z]);
#pragma unroll
    for (int z = 0; z < 4; ++z)
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = z0 + z < P.ks ? v[i] + w[z][i] : v[i];
  }
}

// The row's runs of a deferred result from column 0 (zero past its columns).
template <int TPR, int E>
__device__ __forceinline__ void part_row(const PartSum& P, const RowLane<TPR>& L, float (&v)[E][8]) {
  const bool vec = part_aligned(P);
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int col = 8 * (L.c0 + TPR * e);
    part8(P, vec, L.t, min(col, P.n - 8), v[e]);
#pragma unroll
    for (int i = 0; i < 8; ++i) v[e][i] = col < P.n ? v[e][i] : 0.f;
  }
}

// The row v (zero past its end) scaled by a power of two so that |x| < 2^14 and
// split into fp16 hi + lo planes of kpad columns; the sums of its 32-element
// blocks (four threads each), which the block offsets of Q4_K weights multiply,
// go to xs.
template <int TPR, int E>
__device__ __forceinline__ void row_planes(const float (&v)[E][8], const RowLane<TPR>& L, int kpad, _Float16* xh,
                                           _Float16* xl, float* xscale, _Float16* xs, float* red) {
  float mx = 0.f;
#pragma unroll
  for (int e = 0; e < E; ++e)
#pragma unroll
    for (int i = 0; i < 8; ++i) mx = fmaxf(mx, fabsf(v[e][i]));
  mx = row_reduce<TPR, true>(mx, L, red);
  int ex = 0;
  (void)frexpf(mx, &ex);  // mx < 2^ex
  const int rs = max(min(14 - ex, 60), -60);
  const int nb = kpad / 32;
  xs += (size_t)L.t * 2 * nb;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int col = 8 * (L.c0 + TPR * e);
    half8_t h, l;
    float bs = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float sv = ldexpf(v[e][i], rs);
      h[i] = (_Float16)sv;
      l[i] = (_Float16)(sv - (float)h[i]);
      bs += sv;
    }
    bs = group_sum<4>(bs) * 0.03125f;
    if (L.ok && col < kpad) {
      const size_t at = plane_at(L.t, col, kpad);
      *(half8_t*)(xh + at) = h;
      *(half8_t*)(xl + at) = l;
      if ((L.c0 & 3) == 0) {
        const _Float16 bh = (_Float16)bs;
        xs[col / 32] = bh;
        xs[nb + col / 32] = (_Float16)(bs - (float)bh);
      }
    }
  }
  if (L.ok && L.c0 == 0) xscale[L.t] = __builtin_isfinite(mx) ? ldexpf(1.0f, -rs) : __int_as_float(0x7fc00000);
}

// x := (x * inv) * w with the reference's fp32 operation order (RMSNorm)
template <int TPR, int E>
__device__ __forceinline__ void row_rmsnorm(float (&v)[E][8], const RowLane<TPR>& L, const float* w, int k, float eps,
                                            float* red) {
  float ss = 0.f;
#pragma unroll
  for (int e = 0; e < E; ++e)
#pragma unroll
    for (int i = 0; i < 8; ++i) ss += v[e][i] * v[e][i];
  ss = row_reduce<TPR, false>(ss, L, red);
  const float inv = 1.0f / sqrtf(ss / (float)k + eps);
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int col = 8 * (L.c0 + TPR * e);
    float wv[8];
    load8(w + min(col, k - 8), wv);
#pragma unroll
    for (int i = 0; i < 8; ++i) v[e][i] = __fmul_rn(__fmul_rn(v[e][i], inv), col < k ? wv[i] : 0.f);
  }
}

// The pending residual update of a token row, an optional RMSNorm (GPT:
// LayerNorm), then the operand planes.
template <int TPR, int E, bool GPT>
__global__ __launch_bounds__(kWg) void k_pf_split(PfSplitArgs a, int rows) {
  warm_kernarg<(int)(sizeof(PfSplitArgs) + 8)>();  // (dependent argument rounds hit the scalar cache)
  __shared__ float red[4];
  const RowLane<TPR> L(rows);
  float* xw = const_cast<float*>(a.x + (size_t)L.t * a.ldx);
  float v[E][8];
#pragma unroll
  for (int e = 0; e < E; ++e) load8(xw + min(8 * (L.c0 + TPR * e), a.k - 8), v[e]);
#pragma unroll
  for (int e = 0; e < E; ++e)
#pragma unroll
    for (int i = 0; i < 8; ++i) v[e][i] = 8 * (L.c0 + TPR * e) < a.k ? v[e][i] : 0.f;
  if (a.add.p) {
    float d[E][8];
    part_row<TPR, E>(a.add, L, d);
    if constexpr (GPT) {
      // bias, residual add, SANITIZE (gpt-wgsl-runtime.ts:1708-1746)
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const int col = 8 * (L.c0 + TPR * e);
        float b[8];
        load8(a.add_bias + min(col, a.k - 8), b);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const float y = __fadd_rn(v[e][i], __fadd_rn(d[e][i], b[i]));
          v[e][i] = col >= a.k || y != y ? 0.0f : fminf(fmaxf(y, -10000.0f), 10000.0f);
        }
      }
    } else if (a.add_w) {
      // the branch output goes through RMSNorm first (the Gemma-3 sandwich)
      row_rmsnorm<TPR, E>(d, L, a.add_w, a.k, a.eps, red);
#pragma unroll
      for (int e = 0; e < E; ++e)
#pragma unroll
        for (int i = 0; i < 8; ++i) v[e][i] = fminf(fmaxf(__fadd_rn(v[e][i], d[e][i]), -65000.0f), 65000.0f);
    } else {
#pragma unroll
      for (int e = 0; e < E; ++e)
#pragma unroll
        for (int i = 0; i < 8; ++i)
          v[e][i] = __fadd_rn(v[e][i], a.add_scale != 0.f ? __fmul_rn(d[e][i], a.add_scale) : d[e][i]);
    }
    // the updated residual row
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int col = 8 * (L.c0 + TPR * e);
      if (L.ok && col < a.k) {
        *(float4*)(xw + col) = make_float4(v[e][0], v[e][1], v[e][2], v[e][3]);
        *(float4*)(xw + col + 4) = make_float4(v[e][4], v[e][5], v[e][6], v[e][7]);
      }
    }
  }
  if constexpr (GPT) {
    if (a.w) {
      // LAYER_NORM_WGSL (gpt-wgsl-runtime.ts:1658-1706): mean and E[x^2] in one
      // pass, variance max(E[x^2] - mean^2, 0), ((x - mean) * inv_std) * w + b
      float sm = 0.f, sq = 0.f;
#pragma unroll
      for (int e = 0; e < E; ++e)
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          sm += v[e][i];
          sq += v[e][i] * v[e][i];
        }
      sm = row_reduce<TPR, false>(sm, L, red);
      sq = row_reduce<TPR, false>(sq, L, red);
      const float mean = sm / (float)a.k;
      const float var = fmaxf(__fsub_rn(sq / (float)a.k, __fmul_rn(mean, mean)), 0.0f);
      const float inv = 1.0f / sqrtf(var + a.eps);
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const int col = 8 * (L.c0 + TPR * e);
        float w[8], b[8];
        load8(a.w + min(col, a.k - 8), w);
        load8(a.norm_b + min(col, a.k - 8), b);
#pragma unroll
        for (int i = 0; i < 8; ++i)
          v[e][i] = col < a.k ? __fadd_rn(__fmul_rn(__fmul_rn(__fsub_rn(v[e][i], mean), inv), w[i]), b[i]) : 0.f;
      }
    }
  } else if (a.w) {
    row_rmsnorm<TPR, E>(v, L, a.w, a.k, a.eps, red);
  }
  row_planes<TPR, E>(v, L, a.kpad, a.xh, a.xl, a.xscale, a.xs, red);
}

// ---- decode-batch GEMM (at most 64 token rows) ------------------------------------
//
// With 64 or fewer token rows the GEMM streams weights: every weight is used
// by at most 64 products, so staging weight tiles through LDS (k_gemm_int)
// costs more than the products. Here each wave owns 64 weight rows x all 64
// token rows over a quarter of the workgroup's K range, with no LDS for the
// operands: the x planes are loaded straight into MFMA A operands (lane l:
// token l % 16 of each 16-token tile, k 8 (l / 16) .. + 8 of the 32-k step)
// and the weights are dequantized in registers into B operands (lane l: row
// l % 16 of each 16-row tile, the same 8 k), as fp16 hi + lo of W 2^ws; three
// MFMAs per step (Ah Bh + Al Bh + Ah Bl). The lane's weight bytes for its 8 k
// are consecutive in the striped rows: Q4_K sub-blocks 2c and 2c+1 share the
// bytes qs[32c + 8g .. + 8] (low / high nibbles), Q6_K's four 32-k quarters of
// a 128-k half share ql and qh bytes the same way, so the loads of a block
// (64 k of Q4_K, 128 k of Q6_K) are used whole. The four waves' sums meet in
// LDS at the end (in wave order) and the workgroup writes its K split's partial.

constexpr int kSkRows = 64;  // weight rows per wave (and per workgroup)
constexpr int kSkRed = kSkRows + 4;  // k_gemm_sk1's LDS row stride of the per-wave tiles (bank spread)

__device__ __forceinline__ half8_t pack8(const float (&w)[8]) {
  half8_t h;
#pragma unroll
  for (int i = 0; i < 8; ++i) h[i] = (_Float16)w[i];
  return h;
}
// hi = fp16(w), lo = fp16(w - hi)
__device__ __forceinline__ void split8(const float (&w)[8], half8_t& h, half8_t& l) {
  h = pack8(w);
  float r[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) r[i] = w[i] - (float)h[i];
  l = pack8(r);
}
__device__ __forceinline__ float nib(uint32_t w, int i) { return (float)((w >> (4 * i)) & 15u); }

// A block is 64 k: two 32-k steps whose weights the lane reads from one run of
// bytes (Q4_K: sub-blocks 2c and 2c + 1 of qs[32c + 8g .. + 8], low and high
// nibbles; Q6_K: quarters p and p + 2 of a 128-k half, low and high nibbles of
// ql run p, the half's qh bits 2p and 2p + 4).
template <int T>
struct SkBlock;  // the lane's weight bytes of one block for one row
template <>
struct SkBlock<QT_Q4_K> {
  uint2 qs;      // qs[32c + 8g .. + 8]
  uint4 hdr;     // the super-block header (d, dmin, scales)
};
template <>
struct SkBlock<QT_Q6_K> {
  uint2 ql;      // ql[64h + 32p + 8g .. + 8]
  uint2 qh;      // qh[32h + 8g .. + 8]
  uint2 sc;      // the half's 8 scales sc[8h .. + 8]
  uint32_t d;
};
constexpr int kSkBlockK = 64;

// First column of step s2 (0 or 1) of block blk.
template <int T>
__device__ __forceinline__ int sk_col(int blk, int s2) {
  if constexpr (T == QT_Q4_K) return 64 * blk + 32 * s2;
  // Q6_K block blk: super-block blk / 4, half (blk / 2) % 2, run p = blk % 2; quarter p + 2 s2
  return 256 * (blk >> 2) + 128 * ((blk >> 1) & 1) + 32 * ((blk & 1) + 2 * s2);
}

template <int T>
__device__ __forceinline__ SkBlock<T> sk_load(const QMat& w, int row, int blk, int g) {
  const size_t K = (size_t)w.k;
  SkBlock<T> b;
  if constexpr (T == QT_Q4_K) {
    b.qs = ldg2(w.s0 + row * (K / 2) + 32 * blk + 8 * g);
    b.hdr = ldg4(w.s1 + row * (K / 16) + 16 * (blk >> 2));
  } else {
    const int sb = blk >> 2, h = (blk >> 1) & 1, p = blk & 1;
    b.ql = ldg2(w.s0 + row * (K / 2) + 128 * sb + 64 * h + 32 * p + 8 * g);
    b.qh = ldg2(w.s1 + row * (K / 4) + 64 * sb + 32 * h + 8 * g);
    b.sc = ldg2(w.s2 + row * (K / 16) + 16 * sb + 8 * h);
    b.d = ld_u16(w.s3 + 2 * (row * (K / 256) + sb));
  }
  return b;
}

// The lane's 8 weights (times 2^ws) of step s2 of the block.
template <int T>
__device__ __forceinline__ void sk_weights(const SkBlock<T>& b, int blk, int s2, int g, float wsc, float (&w)[8]) {
  if constexpr (T == QT_Q4_K) {
    // sub-block j = 2c + s2 of the super-block: nibble s2 of the lane's bytes
    const int j = ((blk & 3) << 1) + s2;
    uint32_t sc, m;
    scale_min(j, b.hdr.y, b.hdr.z, b.hdr.w, &sc, &m);
    const float dsc = h2f(b.hdr.x) * (float)sc * wsc, dm = h2f(b.hdr.x >> 16) * (float)m * wsc;
    // four codes per word at once: byte i = nibble s2 of the lane's byte i
    const uint32_t c0 = (b.qs.x >> (4 * s2)) & 0x0f0f0f0fu, c1 = (b.qs.y >> (4 * s2)) & 0x0f0f0f0fu;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      w[i] = fmaf(dsc, ub(c0, i), -dm);
      w[4 + i] = fmaf(dsc, ub(c1, i), -dm);
    }
  } else {
    // quarter q = p + 2 s2 of the half: nibble s2 of the ql run, qh bits 2q;
    // the lane's 8 k lie in sub-block 2q + (g >> 1) of the half
    const int q = (blk & 1) + 2 * s2;
    const int si = 2 * q + (g >> 1);
    const uint32_t sw = si < 4 ? b.sc.x : b.sc.y;
    const float dsc = h2f(b.d) * (float)(int8_t)((sw >> (8 * (si & 3))) & 0xffu) * wsc, off = -32.0f * dsc;
    // four 6-bit codes per word at once (byte i: low 4 bits from ql, bits 4-5 from qh)
    const uint32_t c0 = ((b.ql.x >> (4 * s2)) & 0x0f0f0f0fu) | (((b.qh.x >> (2 * q)) & 0x03030303u) << 4);
    const uint32_t c1 = ((b.ql.y >> (4 * s2)) & 0x0f0f0f0fu) | (((b.qh.y >> (2 * q)) & 0x03030303u) << 4);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      w[i] = fmaf(dsc, ub(c0, i), off);
      w[4 + i] = fmaf(dsc, ub(c1, i), off);
    }
  }
}

template <int T>
__global__ __launch_bounds__(kWg, 2) void k_gemm_sk(GemmArgs a) {
  extern __shared__ __align__(16) float ssm[];
  constexpr int BK = kSkBlockK;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * kSkRows;
  const int N = a.n_all ? a.n_all : a.w.n;
  const int seg = a.n_all ? (n0 >= a.n2 ? 2 : (n0 >= a.n1 ? 1 : 0)) : 0;
  const int sb0 = seg == 2 ? a.n2 : (seg == 1 ? a.n1 : 0);
  QMat wm = a.w;
#define CHONK_PICK_W(f) wm.f = seg == 2 ? a.w3.f : (seg == 1 ? a.w2.f : a.w.f)
  CHONK_PICK_W(s0);
  CHONK_PICK_W(s1);
  CHONK_PICK_W(s2);
  CHONK_PICK_W(s3);
  CHONK_PICK_W(n);
#undef CHONK_PICK_W
  // this workgroup's blocks (split blockIdx.z of ksplit), then this wave's quarter
  const int nblk = a.w.k / BK;
  const int z_lo = (int)((int64_t)nblk * blockIdx.z / a.ksplit), z_hi = (int)((int64_t)nblk * (blockIdx.z + 1) / a.ksplit);
  const int b_lo = z_lo + (z_hi - z_lo) * wave / 4, b_hi = z_lo + (z_hi - z_lo) * (wave + 1) / 4;
  const float wsc = ldexpf(1.0f, a.ws);
  // rows of the lane in the matrix (clamped: a ragged tile loads a valid row, its sums are dropped)
  int rows[4];
#pragma unroll
  for (int rt = 0; rt < 4; ++rt) rows[rt] = min(n0 + 16 * rt + r16, N - 1) - sb0;
  // the lane's piece of each token tile's A operands; a tile past a.t loads the
  // last one and its sums are never written
  size_t xo[4];
#pragma unroll
  for (int tt = 0; tt < 4; ++tt) xo[tt] = plane_at(16 * min(tt, (a.t - 1) / 16), 0, a.kpad) + 8 * lane;
  // the epilogue's operand scales, requested up front (read from LDS at the end)
  if (tid < a.t) ssm[4 * 64 * kSkRows + tid] = a.xscale[tid];

  float4_t acc[4][4];  // [token tile][row tile]: lane holds tokens 16 tt + 4 g + i, row 16 rt + r16
#pragma unroll
  for (int tt = 0; tt < 4; ++tt)
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) acc[tt][rt] = float4_t{0.f, 0.f, 0.f, 0.f};

  SkBlock<T> cur[4];
  if (b_lo < b_hi) {
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) cur[rt] = sk_load<T>(wm, rows[rt], b_lo, g);
  }
  for (int blk = b_lo; blk < b_hi; ++blk) {
    // the next block's bytes are requested before this one is reduced (the
    // last block reloads itself, so that the loads stay unconditional)
    SkBlock<T> nxt[4];
    const int bn = min(blk + 1, b_hi - 1);
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) nxt[rt] = sk_load<T>(wm, rows[rt], bn, g);
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2) {
      const int k0 = sk_col<T>(blk, s2);
      half8_t ah[4], al[4];
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) {
        const size_t off = xo[tt] + 16 * k0;  // (512 halves per 32 columns)
        ah[tt] = *gbl((const half8_t*)(a.xh + off));
        al[tt] = *gbl((const half8_t*)(a.xl + off));
      }
#pragma unroll
      for (int rt = 0; rt < 4; ++rt) {
        float w[8];
        sk_weights<T>(cur[rt], blk, s2, g, wsc, w);
        half8_t bh, bl;
        split8(w, bh, bl);
        // (the four token tiles' chains interleaved: no MFMA waits on the one before it)
#pragma unroll
        for (int tt = 0; tt < 4; ++tt) acc[tt][rt] = mfma32(ah[tt], bh, acc[tt][rt]);
#pragma unroll
        for (int tt = 0; tt < 4; ++tt) acc[tt][rt] = mfma32(al[tt], bh, acc[tt][rt]);
#pragma unroll
        for (int tt = 0; tt < 4; ++tt) acc[tt][rt] = mfma32(ah[tt], bl, acc[tt][rt]);
      }
    }
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) cur[rt] = nxt[rt];
  }
  // the four waves' sums, added in wave order: [wave][token][row] floats
  float* red = ssm;
  float* xs = ssm + 4 * 64 * kSkRows;  // the token rows' operand scales
#pragma unroll
  for (int tt = 0; tt < 4; ++tt)
#pragma unroll
    for (int rt = 0; rt < 4; ++rt)
#pragma unroll
      for (int i = 0; i < 4; ++i) red[(wave * 64 + 16 * tt + 4 * g + i) * kSkRows + 16 * rt + r16] = acc[tt][rt][i];
  __syncthreads();
  // thread (tg, r) writes row n0 + r of tokens tg, tg + 4, ...: one coalesced
  // 256-byte run per token and store instruction
  const int r = tid & 63, tg = tid >> 6, n = n0 + r;
  if (n < N) {
    const float wun = ldexpf(1.0f, -a.ws);
    for (int t = tg; t < a.t; t += 4) {
      const int e = t * kSkRows + r;
      const float v = (((red[e] + red[64 * kSkRows + e]) + red[2 * 64 * kSkRows + e]) + red[3 * 64 * kSkRows + e]) *
                      (wun * xs[t]);
      if (a.ksplit > 1 || a.defer) {
        a.part[((size_t)blockIdx.z * a.t + t) * N + n] = v;
      } else if (a.epi == GEMM_ADD) {
        float* y = a.y + (size_t)t * a.ldy + n;
        *y = __fadd_rn(*y, v);
      } else {
        a.y[(size_t)t * a.ldy + n] = v;
      }
    }
  }
}

// The same with exactly one 64-k block per wave (the K split of the decode
// step's layer GEMMs): every load of the wave — its x operands, copied
// straight into its own 16 KiB of LDS, and its weight bytes — is issued at
// entry and awaited once, so the wave pays one memory round trip before its
// two steps of products. LDS per wave: [plane][step][token tile][512 halves].
// NT: token tiles computed, 1, 2 or 4 (up to 16, 32 or 64 rows).
template <int T, int NT>
__global__ __launch_bounds__(kWg, 2) void k_gemm_sk1(GemmArgs a) {
  extern __shared__ __align__(16) float ssm[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * kSkRows;
  const int N = a.n_all ? a.n_all : a.w.n;
  const int seg = a.n_all ? (n0 >= a.n2 ? 2 : (n0 >= a.n1 ? 1 : 0)) : 0;
  const int sb0 = seg == 2 ? a.n2 : (seg == 1 ? a.n1 : 0);
  QMat wm = a.w;
#define CHONK_PICK_W(f) wm.f = seg == 2 ? a.w3.f : (seg == 1 ? a.w2.f : a.w.f)
  CHONK_PICK_W(s0);
  CHONK_PICK_W(s1);
  CHONK_PICK_W(s2);
  CHONK_PICK_W(s3);
  CHONK_PICK_W(n);
#undef CHONK_PICK_W
  // this wave's block: one per wave, the workgroup's four in a row
  const int blk = (int)blockIdx.z * 4 + wave;
  _Float16* xw = (_Float16*)ssm + (size_t)wave * (2 * 2 * NT * 512);  // this wave's x operands
  float* xs = ssm + 4 * 16 * NT * kSkRed;                             // the token rows' operand scales
  // x: 4 NT copies of 1 KiB (a token tile's 32 columns, in operand order; tiles
  // past a.t repeat the last one: their sums are never written)
  {
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2)
#pragma unroll
        for (int i = 0; i < NT; ++i) {
          const _Float16* src =
              (p ? a.xl : a.xh) + plane_at(16 * min(i, (a.t - 1) / 16), sk_col<T>(blk, s2), a.kpad) + 8 * lane;
          __builtin_amdgcn_global_load_lds((gmem_void*)src, (lds_void*)(xw + ((p * 2 + s2) * NT + i) * 512), 16, 0,
                                           0);
        }
  }
  const float wsc = ldexpf(1.0f, a.ws);
  SkBlock<T> bk[4];
#pragma unroll
  for (int rt = 0; rt < 4; ++rt) bk[rt] = sk_load<T>(wm, min(n0 + 16 * rt + r16, N - 1) - sb0, blk, g);
  if (tid < a.t) xs[tid] = a.xscale[tid];
  __builtin_amdgcn_s_waitcnt(0);  // (the copies into LDS land before they are read)
  __syncthreads();
  float4_t acc[NT][4];
#pragma unroll
  for (int tt = 0; tt < NT; ++tt)
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) acc[tt][rt] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s2 = 0; s2 < 2; ++s2) {
    half8_t ah[NT], al[NT];
#pragma unroll
    for (int tt = 0; tt < NT; ++tt) {
      ah[tt] = *(const half8_t*)(xw + ((0 * 2 + s2) * NT + tt) * 512 + 8 * lane);
      al[tt] = *(const half8_t*)(xw + ((1 * 2 + s2) * NT + tt) * 512 + 8 * lane);
    }
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) {
      float w[8];
      sk_weights<T>(bk[rt], blk, s2, g, wsc, w);
      half8_t bh, bl;
      split8(w, bh, bl);
#pragma unroll
      for (int tt = 0; tt < NT; ++tt) acc[tt][rt] = mfma32(ah[tt], bh, acc[tt][rt]);
#pragma unroll
      for (int tt = 0; tt < NT; ++tt) acc[tt][rt] = mfma32(al[tt], bh, acc[tt][rt]);
#pragma unroll
      for (int tt = 0; tt < NT; ++tt) acc[tt][rt] = mfma32(ah[tt], bl, acc[tt][rt]);
    }
  }
  __syncthreads();  // every wave has read its x operands (the area is reused below)
  // the four waves' tiles [wave][token][row] (rows padded to kSkRed floats, so
  // that neither the writes below nor the 16-byte reads after them collide on
  // LDS banks); then thread (token tid / TPT, rows RPT (tid % TPT) .. + RPT - 1) sums
  // its outputs over the waves with 16-byte reads and stores them with 16-byte
  // stores — one pass instead of dependent rounds of single floats
  constexpr int RPT = 4 * NT, TPT = 64 / RPT;
  float* red = ssm;
#pragma unroll
  for (int tt = 0; tt < NT; ++tt)
#pragma unroll
    for (int rt = 0; rt < 4; ++rt)
#pragma unroll
      for (int i = 0; i < 4; ++i) red[(wave * 16 * NT + 16 * tt + 4 * g + i) * kSkRed + 16 * rt + r16] = acc[tt][rt][i];
  __syncthreads();
  const int t = tid / TPT, q = tid % TPT;
  if (t < a.t) {
    const float sc = ldexpf(1.0f, -a.ws) * xs[t];
    float4 v[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const float* e = red + t * kSkRed + RPT * q + 4 * j;
      const float4 w0 = *(const float4*)e, w1 = *(const float4*)(e + 16 * NT * kSkRed);
      const float4 w2 = *(const float4*)(e + 2 * 16 * NT * kSkRed), w3 = *(const float4*)(e + 3 * 16 * NT * kSkRed);
      v[j] = make_float4((((w0.x + w1.x) + w2.x) + w3.x) * sc, (((w0.y + w1.y) + w2.y) + w3.y) * sc,
                         (((w0.z + w1.z) + w2.z) + w3.z) * sc, (((w0.w + w1.w) + w2.w) + w3.w) * sc);
    }
    const int nq = n0 + RPT * q;
    float* dst = a.part + ((size_t)blockIdx.z * a.t + t) * N + nq;
    if (nq + RPT <= N && (N & 3) == 0) {
#pragma unroll
      for (int j = 0; j < NT; ++j) *(float4*)(dst + 4 * j) = v[j];
    } else {
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const float o[4] = {v[j].x, v[j].y, v[j].z, v[j].w};
#pragma unroll
        for (int e2 = 0; e2 < 4; ++e2)
          if (nq + 4 * j + e2 < N) dst[4 * j + e2] = o[e2];
      }
    }
  }
}

// The same for a matrix with many row groups (the lm_head): a workgroup owns
// 4 x 64 weight rows over the whole K, the four waves sharing each 64-k block
// of x operands, copied into LDS one block ahead (two buffers; each wave
// copies a quarter); every wave writes its own rows' results. Per block:
// weights of the next block and its x copies are issued, then this block's
// copies are awaited (s_waitcnt counts the loads issued since) and the waves
// meet at a barrier before the products.
// NT: token tiles computed, as for k_gemm_sk1.
template <int T, int NT>
__global__ __launch_bounds__(kWg, 2) void k_gemm_lm(GemmArgs a) {
  extern __shared__ __align__(16) float ssm[];
  constexpr int W = T == QT_Q4_K ? 8 : 16;  // weight loads per block and wave (4 row tiles)
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * (4 * kSkRows) + wave * kSkRows;  // this wave's rows
  const int N = a.w.n, nblk = a.w.k / kSkBlockK;
  _Float16* xb = (_Float16*)ssm;  // [buffer][plane][step][token tile][512 halves]
  float* xs = (float*)(xb + 2 * (2 * 2 * NT * 512));
  const float wsc = ldexpf(1.0f, a.ws);
  int rows[4];
#pragma unroll
  for (int rt = 0; rt < 4; ++rt) rows[rt] = min(n0 + 16 * rt + r16, N - 1);
  // x of block b into buffer buf: this wave's NT of its 4 NT 1-KiB copies
  auto copy_x = [&](int b, int buf) {
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const int c = wave * NT + j, p = c / (2 * NT), s2 = (c / NT) & 1, i = c % NT;
      const _Float16* src =
          (p ? a.xl : a.xh) + plane_at(16 * min(i, (a.t - 1) / 16), sk_col<T>(b, s2), a.kpad) + 8 * lane;
      __builtin_amdgcn_global_load_lds((gmem_void*)src,
                                       (lds_void*)(xb + ((buf * 4 + p * 2 + s2) * NT + i) * 512), 16, 0, 0);
    }
  };
  if (tid < a.t) xs[tid] = a.xscale[tid];
  SkBlock<T> cur[4];
#pragma unroll
  for (int rt = 0; rt < 4; ++rt) cur[rt] = sk_load<T>(a.w, rows[rt], 0, g);
  __builtin_amdgcn_sched_barrier(0);
  copy_x(0, 0);
  __builtin_amdgcn_sched_barrier(0);
  float4_t acc[NT][4];
#pragma unroll
  for (int tt = 0; tt < NT; ++tt)
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) acc[tt][rt] = float4_t{0.f, 0.f, 0.f, 0.f};
  for (int b = 0; b < nblk; ++b) {
    // the next block's weights, then its x copies into the other buffer (the last
    // block copies itself there, where nothing reads it: the loop body stays
    // branch-free, so every wait counts exactly)
    const int bn = min(b + 1, nblk - 1);
    SkBlock<T> nxt[4];
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) nxt[rt] = sk_load<T>(a.w, rows[rt], bn, g);
    __builtin_amdgcn_sched_barrier(0);
    copy_x(bn, (b + 1) & 1);
    __builtin_amdgcn_sched_barrier(0);
    // this block's copies have landed once at most the loads issued after
    // them are outstanding: the next block's W weight loads and NT copies
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(W + NT));
    // (a bare barrier: __syncthreads would also wait for the loads in flight)
    lds_barrier();
    const _Float16* xc = xb + (size_t)(b & 1) * 4 * NT * 512;
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2) {
      half8_t ah[NT], al[NT];
#pragma unroll
      for (int tt = 0; tt < NT; ++tt) {
        ah[tt] = *(const half8_t*)(xc + ((0 * 2 + s2) * NT + tt) * 512 + 8 * lane);
        al[tt] = *(const half8_t*)(xc + ((1 * 2 + s2) * NT + tt) * 512 + 8 * lane);
      }
#pragma unroll
      for (int rt = 0; rt < 4; ++rt) {
        float w[8];
        sk_weights<T>(cur[rt], b, s2, g, wsc, w);
        half8_t bh, bl;
        split8(w, bh, bl);
#pragma unroll
        for (int tt = 0; tt < NT; ++tt) acc[tt][rt] = mfma32(ah[tt], bh, acc[tt][rt]);
#pragma unroll
        for (int tt = 0; tt < NT; ++tt) acc[tt][rt] = mfma32(al[tt], bh, acc[tt][rt]);
#pragma unroll
        for (int tt = 0; tt < NT; ++tt) acc[tt][rt] = mfma32(ah[tt], bl, acc[tt][rt]);
      }
    }
    lds_barrier();  // every wave has read buffer b & 1 before block b + 2's copies overwrite it
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) cur[rt] = nxt[rt];
  }
  const float wun = ldexpf(1.0f, -a.ws);
  const bool add = a.epi == GEMM_ADD;
#pragma unroll
  for (int tt = 0; tt < NT; ++tt)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int t = 16 * tt + 4 * g + i;
      if (t >= a.t) continue;
      const float sc = wun * xs[t];
#pragma unroll
      for (int rt = 0; rt < 4; ++rt) {
        const int n = n0 + 16 * rt + r16;
        if (n >= N) continue;
        float* y = a.y + (size_t)t * a.ldy + n;
        const float v = acc[tt][rt][i] * sc;
        if (add)
          *y = __fadd_rn(*y, v);
        else
          *y = v;
      }
    }
}

size_t gemm_lm_shared_bytes(int nt) { return sizeof(_Float16) * 2 * (2 * 2 * nt * 512) + sizeof(float) * 64; }

size_t gemm_sk_shared_bytes(int nt = 4) { return sizeof(float) * (4 * 16 * nt * kSkRed + 64); }

// Token tiles a decode-batch launch computes: the four of 64 rows cost a batch of
// a few sequences products, copies and sums it drops (Qwen3-0.6B shape, step of 2,
// 16, 30 and 64 rows: 2.03, 2.12, 2.27, 2.30 ms with four always; 1.83, 1.92, 2.12,
// 2.31 with as many as the rows need).
int gemm_sk_tiles(int rows) { return rows <= 16 ? 1 : rows <= 32 ? 2 : 4; }

// kernel<type, nt> for a decode-batch launch
#define CHONK_SK_LAUNCH(kernel, type, nt, grid, sh, s, a)                                   \
  do {                                                                                      \
    if ((type) == QT_Q4_K) {                                                                \
      if ((nt) == 1) hipLaunchKernelGGL((kernel<QT_Q4_K, 1>), grid, dim3(kWg), sh, s, a);   \
      else if ((nt) == 2) hipLaunchKernelGGL((kernel<QT_Q4_K, 2>), grid, dim3(kWg), sh, s, a); \
      else hipLaunchKernelGGL((kernel<QT_Q4_K, 4>), grid, dim3(kWg), sh, s, a);             \
    } else {                                                                                \
      if ((nt) == 1) hipLaunchKernelGGL((kernel<QT_Q6_K, 1>), grid, dim3(kWg), sh, s, a);   \
      else if ((nt) == 2) hipLaunchKernelGGL((kernel<QT_Q6_K, 2>), grid, dim3(kWg), sh, s, a); \
      else hipLaunchKernelGGL((kernel<QT_Q6_K, 4>), grid, dim3(kWg), sh, s, a);             \
    }                                                                                       \
  } while (0)

// The decode-batch GEMM applies: at most 64 token rows and a K-quant type it covers.
bool gemm_sk_applies(int type, int k, int rows) {
  static const bool off = [] {
    const char* v = std::getenv("CHONK_GEMM");
    return v && std::strcmp(v, "tiles") == 0;
  }();
  return !off && rows >= 1 && rows <= 64 && (type == QT_Q4_K || type == QT_Q6_K) && k % 256 == 0;
}
bool gemm_sk_applies(const GemmArgs& a) { return gemm_sk_applies(a.w.type, a.w.k, a.t) && a.kpad >= a.w.k; }

// K split of a decode-batch GEMM: about 256 workgroups (one per CU), at least
// one block per wave.
int gemm_sk_split(const GemmArgs& a, int row_groups) {
  const int nblk = a.w.k / kSkBlockK;
  int ks = std::max(1, std::min(kMaxDeferSplit, (256 + row_groups - 1) / row_groups));
  while (ks > 1 && nblk / ks < 4) --ks;
  return ks;
}

hipError_t launch_gemm_sk(const GemmArgs& a, int n_rows, hipStream_t s) {
  const dim3 grid((n_rows + kSkRows - 1) / kSkRows, 1, a.ksplit);
  const size_t sh = gemm_sk_shared_bytes();
  if (a.w.type == QT_Q4_K)
    hipLaunchKernelGGL(k_gemm_sk<QT_Q4_K>, grid, dim3(kWg), sh, s, a);
  else
    hipLaunchKernelGGL(k_gemm_sk<QT_Q6_K>, grid, dim3(kWg), sh, s, a);
  return hipGetLastError();
}

// y[t][n] (=|+=) the K-split partial sums, added in split order.
__global__ __launch_bounds__(kWg) void k_gemm_reduce(GemmArgs a) {
  const int64_t total = (int64_t)a.t * a.w.n;
  for (int64_t i = (int64_t)blockIdx.x * kWg + threadIdx.x; i < total; i += (int64_t)gridDim.x * kWg) {
    float v = a.part[i];
    for (int z = 1; z < a.ksplit; ++z) v += a.part[(int64_t)z * total + i];
    const int64_t t = i / a.w.n, n = i - t * a.w.n;
    float* y = a.y + t * a.ldy + n;
    *y = a.epi == GEMM_ADD ? __fadd_rn(*y, v) : v;
  }
}

// ---- per-token glue ---------------------------------------------------------------

// Embedding rows of the prompt tokens times the embedding scale, plus (pos !=
// null) row p0 + t of the learned position table.
__global__ __launch_bounds__(kWg) void k_pf_embed(QMat embed, const int32_t* tok, float scale, const float* pos, int p0,
                                                  int k, float* x) {
  const int t = blockIdx.x;
  const int id = tok[t];
  with_type(embed.type, [&]<int TE>() {
    for (int u = threadIdx.x; u < k / 32; u += kWg) {
      const Frag<TE> f = load_unit<TE>(embed, id, u);
      float v[32];
      dequant_unit<TE>(f, u, v);
#pragma unroll
      for (int e = 0; e < 32; ++e) {
        const int i = unit_col<TE>(u, e);
        const float y = __fmul_rn(v[e], scale);
        x[(size_t)t * k + i] = pos ? __fadd_rn(y, pos[(size_t)(p0 + t) * k + i]) : y;
      }
    }
  });
}

// silu(g) * u, gelu_tanh(g) * u or (GPT-2) gelu_tanh(u + bias) per element (or
// that product as the GEMM left it), then the operand planes.
template <int TPR, int E>
__global__ __launch_bounds__(kWg) void k_pf_glu_split(PfGluArgs a, int rows) {
  warm_kernarg<(int)(sizeof(PfGluArgs) + 8)>();  // (dependent argument rounds hit the scalar cache)
  __shared__ float red[4];
  const RowLane<TPR> L(rows);
  float gv[E][8], v[E][8];
  if (a.act == PF_DONE) {
    part_row<TPR, E>(a.pu, L, v);
    row_planes<TPR, E>(v, L, a.kpad, a.xh, a.xl, a.xscale, a.xs, red);
    return;
  }
  if (a.act != PF_GELU_BIAS) {
    part_row<TPR, E>(a.pg, L, gv);
  } else {
#pragma unroll
    for (int e = 0; e < E; ++e) load8(a.bias + min(8 * (L.c0 + TPR * e), a.k - 8), gv[e]);
  }
  part_row<TPR, E>(a.pu, L, v);
#pragma unroll
  for (int e = 0; e < E; ++e)
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float g = gv[e][i], u = v[e][i];
      const float y = a.act == PF_SWIGLU  ? silu_mul(g, u)
                      : a.act == PF_GEGLU ? __fmul_rn(gelu_tanh(g), u)
                                          : gelu_tanh(__fadd_rn(u, g));
      v[e][i] = 8 * (L.c0 + TPR * e) < a.k ? y : 0.f;
    }
  row_planes<TPR, E>(v, L, a.kpad, a.xh, a.xl, a.xscale, a.xs, red);
}

// ---- lfm2 short convolution ---------------------------------------------------------

// C * (bx[t-2] w0 + bx[t-1] w1 + bx[t] w2) of every channel (CONV_BLOCK_WGSL,
// lfm-wgsl-runtime.ts:1641-1672, each product and sum rounded as the decode
// prologue does), bx = B * x of the in_proj rows, the two rows before the pass
// from the state; then the operand planes.
template <int TPR, int E>
__global__ __launch_bounds__(kWg) void k_pf_conv(PfConvArgs a, int rows) {
  warm_kernarg<(int)(sizeof(PfConvArgs) + 8)>();
  __shared__ float red[4];
  const RowLane<TPR> L(rows);
  const bool vec = part_aligned(a.p) && (a.k & 3) == 0;
  const int t = L.t;
  float v[E][8];
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int col = min(8 * (L.c0 + TPR * e), a.k - 8);
    // B * x of row r, or of a row before the pass
    auto bx = [&](int r, float (&w)[8]) {
      if (r < 0) {
        load8((r == -2 ? a.s1 : a.s2) + col, w);
        return;
      }
      float b[8];
      part8(a.p, vec, r, col, b);
      part8(a.p, vec, r, 2 * a.k + col, w);
#pragma unroll
      for (int i = 0; i < 8; ++i) w[i] = __fmul_rn(b[i], w[i]);
    };
    float p1[8], p2[8], p3[8], c[8], w[24];
    bx(t - 2, p1);
    bx(t - 1, p2);
    bx(t, p3);
    part8(a.p, vec, t, a.k + col, c);
#pragma unroll
    for (int i = 0; i < 24; ++i) w[i] = a.w[3 * (size_t)col + i];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float y = __fadd_rn(__fadd_rn(__fmul_rn(p1[i], w[3 * i]), __fmul_rn(p2[i], w[3 * i + 1])),
                                __fmul_rn(p3[i], w[3 * i + 2]));
      v[e][i] = 8 * (L.c0 + TPR * e) < a.k ? __fmul_rn(c[i], y) : 0.f;
    }
  }
  row_planes<TPR, E>(v, L, a.kpad, a.xh, a.xl, a.xscale, a.xs, red);
}

// s1, s2 = bx of the pass's last two rows (a launch of its own: k_pf_conv's
// rows 0 and 1 read the old state). A thread reads its channel before it writes.
__global__ __launch_bounds__(kWg) void k_pf_conv_state(PfConvArgs a, int rows) {
  const int i = (int)blockIdx.x * kWg + (int)threadIdx.x;
  if (i >= a.k) return;
  const int j[2] = {i, 2 * a.k + i};
  float w[2];
  part_gather<2>(a.p, rows - 1, j, w);
  const float cur = __fmul_rn(w[0], w[1]);
  float prev = a.s2[i];
  if (rows >= 2) {
    part_gather<2>(a.p, rows - 2, j, w);
    prev = __fmul_rn(w[0], w[1]);
  }
  a.s1[i] = prev;
  a.s2[i] = cur;
}

// ---- granitehybrid Mamba2 ------------------------------------------------------------

constexpr int kMbConvRows = 4;   // token rows per thread of k_pf_mamba_conv
constexpr int kMbStates = 128;   // states per channel
constexpr int kMbHd = 32;        // channels per head
constexpr int kMbCh = 8;         // channels per workgroup of the scan
constexpr int kMbSteps = 32;     // token rows staged in LDS at once

// MAMBA_CONV_WGSL (granite-wgsl-runtime.ts:1476-1520) of every row: channel c of
// xBC is silu(((p1 w0 + p2 w1) + p3 w2) + x w3 + bias) over its last four
// inputs, those before row 0 from the window copy of p0's parity; and per head
// dt = softplus(dt_raw + bias) and decay = exp(dt A) as MAMBA_SSM_WGSL forms
// them. A thread walks kMbConvRows rows of one channel.
__global__ __launch_bounds__(kWg) void k_pf_mamba_conv(PfMambaArgs a) {
  warm_kernarg<(int)(sizeof(PfMambaArgs))>();
  const int c = (int)blockIdx.x * kWg + (int)threadIdx.x, t0 = (int)blockIdx.y * kMbConvRows;
  const int nt = min(kMbConvRows, a.rows - t0);
  if (c >= a.conv + a.heads) return;
  const int ld = pf_mamba_ld(a.conv, a.heads);
  const int j[1] = {a.inner + c};
  float x[kMbConvRows + 3];
#pragma unroll
  for (int r = 0; r < kMbConvRows + 3; ++r) {
    float w[1];
    part_gather<1>(a.p, min(max(t0 + r - 3, 0), a.rows - 1), j, w);
    x[r] = w[0];
  }
  if (c >= a.conv) {
    const int n = c - a.conv;
    const float bias = a.dt_bias[n], an = a.a_neg[n];
    for (int r = 0; r < nt; ++r) {
      const float s = __fadd_rn(x[r + 3], bias);
      const float dt = s > 20.0f ? __fadd_rn(s, logf(__fadd_rn(1.0f, expf(-s)))) : logf(__fadd_rn(1.0f, expf(s)));
      float* o = a.xbc + (size_t)(t0 + r) * ld + a.conv;
      o[n] = dt;
      o[a.heads + n] = expf(__fmul_rn(dt, an));
    }
    return;
  }
  if (t0 == 0) {
    const float* cs = a.conv_state + ((size_t)(a.p0 & 1) * a.conv + c) * 3;
#pragma unroll
    for (int r = 0; r < 3; ++r) x[r] = cs[r];
  }
  const float4 w = reinterpret_cast<const float4*>(a.conv_w)[c];
  const float bias = a.conv_b[c];
#pragma unroll
  for (int r = 0; r < kMbConvRows; ++r) {
    if (r >= nt) break;
    const float y = __fadd_rn(__fadd_rn(__fadd_rn(__fadd_rn(__fmul_rn(x[r], w.x), __fmul_rn(x[r + 1], w.y)),
                                                  __fmul_rn(x[r + 2], w.z)),
                                        __fmul_rn(x[r + 3], w.w)),
                              bias);
    a.xbc[(size_t)(t0 + r) * ld + c] = __fdiv_rn(y, __fadd_rn(1.0f, expf(-y)));
  }
}

// MAMBA_SSM_WGSL's recurrence h = h decay + (dt x) B, y = C h + D x over the rows
// of the pass. The chain over the rows is serial per state and its work small
// (two multiplies and two fmas per state and row), so the split is over states:
// a workgroup owns 8 channels of one head, 32 lanes per channel with 4 states
// each in registers, and walks the rows with B, C (shared by every channel),
// x dt, decay and x staged in LDS 32 rows at a time; the next rows' loads are in
// flight while the staged ones are walked. Workgroups of one head and channel
// group also leave the convolution window of the next pass (k_pf_mamba_conv has
// read the old one; a thread reads its channel's window before it writes it).
__global__ __launch_bounds__(kWg) void k_pf_mamba_scan(PfMambaArgs a) {
  warm_kernarg<(int)(sizeof(PfMambaArgs))>();
  __shared__ __align__(16) float sbc[kMbSteps][2 * kMbStates];
  __shared__ float sx[kMbSteps][kMbCh], sxd[kMbSteps][kMbCh], sdec[kMbSteps], sy[kMbSteps][kMbCh];
  const int n = (int)blockIdx.x, c0 = (int)blockIdx.y * kMbCh, tid = (int)threadIdx.x;
  const int h = tid >> 5, l = tid & 31;
  const int ld = pf_mamba_ld(a.conv, a.heads);
  const int nx = n * kMbHd + c0;  // the workgroup's first channel
  float4_t* sp = reinterpret_cast<float4_t*>(a.ssm_state + (size_t)(nx + h) * kMbStates) + l;
  float4_t s = *sp;
  const float dsk = a.d[n];
  // the next window: entry r is the input of row rows - 3 + r, or the old window's
  auto window = [&](int c) {
    const float* co = a.conv_state + ((size_t)(a.p0 & 1) * a.conv + c) * 3;
    float* cn = a.conv_state + ((size_t)((a.p0 + a.rows) & 1) * a.conv + c) * 3;
    const int j[1] = {a.inner + c};
    float v[3];
#pragma unroll
    for (int r = 0; r < 3; ++r) {
      const int t = a.rows - 3 + r;
      float w[1];
      part_gather<1>(a.p, max(t, 0), j, w);
      v[r] = t >= 0 ? w[0] : co[min(3 + t, 2)];
    }
#pragma unroll
    for (int r = 0; r < 3; ++r) cn[r] = v[r];
  };
  if (tid < kMbCh) window(nx + tid);
  if (n == 0 && c0 == 0) window(a.inner + tid);  // B and C: kWg == 2 * kMbStates channels

  // staging roles: thread moves float4 (tid % 64) of rows tid / 64 + 4 i of
  // B | C, and (row tid / 8, channel tid % 8) of x, dt and decay
  float4_t rb[kMbSteps / 4];
  float rx, rdt, rdec;
  auto fetch = [&](int t0) {
#pragma unroll
    for (int i = 0; i < kMbSteps / 4; ++i) {
      const int t = min(t0 + (tid >> 6) + 4 * i, a.rows - 1);
      rb[i] = *reinterpret_cast<const float4_t*>(a.xbc + (size_t)t * ld + a.inner + 4 * (tid & 63));
    }
    const float* r = a.xbc + (size_t)min(t0 + (tid >> 3), a.rows - 1) * ld;
    rx = r[nx + (tid & 7)];
    rdt = r[a.conv + n];
    rdec = r[a.conv + a.heads + n];
  };
  fetch(0);
  for (int t0 = 0; t0 < a.rows; t0 += kMbSteps) {
    __syncthreads();  // the previous rows are consumed, their y written out
#pragma unroll
    for (int i = 0; i < kMbSteps / 4; ++i)
      *reinterpret_cast<float4_t*>(&sbc[(tid >> 6) + 4 * i][4 * (tid & 63)]) = rb[i];
    sx[tid >> 3][tid & 7] = rx;
    // (steps past the last row leave the state as it is)
    const bool live = t0 + (tid >> 3) < a.rows;
    sxd[tid >> 3][tid & 7] = live ? __fmul_rn(rdt, rx) : 0.f;
    if ((tid & 7) == 0) sdec[tid >> 3] = live ? rdec : 1.f;
    __syncthreads();
    fetch(min(t0 + kMbSteps, a.rows - 1));
    const int nt = min(kMbSteps, a.rows - t0);
    // four steps at a time: the next four's LDS reads are in flight, and the four
    // sums over the lanes interleave (a step by itself waits for every read and
    // every lane exchange)
    struct Steps {
      float4_t B[4], C[4];
      float dx[4], dec[4];
    };
    auto load = [&](Steps& g, int tb) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        g.B[u] = *reinterpret_cast<const float4_t*>(&sbc[tb + u][4 * l]);
        g.C[u] = *reinterpret_cast<const float4_t*>(&sbc[tb + u][kMbStates + 4 * l]);
        g.dx[u] = sxd[tb + u][h];
        g.dec[u] = sdec[tb + u];
      }
    };
    auto walk = [&](const Steps& g, int tb) {
      float acc[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
#pragma unroll
        for (int q = 0; q < 4; ++q) s[q] = fmaf(s[q], g.dec[u], g.dx[u] * g.B[u][q]);
        acc[u] = fmaf(s[0], g.C[u][0], s[1] * g.C[u][1]) + fmaf(s[2], g.C[u][2], s[3] * g.C[u][3]);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) acc[u] = group_sum<32>(acc[u]);
      // lane u of the channel's 32 keeps step u
      const float a01 = l == 1 ? acc[1] : acc[0], a23 = l == 3 ? acc[3] : acc[2];
      if (l < 4) sy[tb + l][h] = l < 2 ? a01 : a23;
    };
    Steps g0, g1;
    load(g0, 0);
    for (int tb = 0; tb < nt; tb += 8) {
      load(g1, tb + 4);
      walk(g0, tb);
      load(g0, min(tb + 8, kMbSteps - 4));
      walk(g1, tb + 4);
    }
    __syncthreads();
    const int t = tid >> 3;
    if (t < nt)
      a.y[(size_t)(t0 + t) * a.inner + nx + (tid & 7)] = __fadd_rn(sy[t][tid & 7], __fmul_rn(dsk, sx[t][tid & 7]));
  }
  *sp = s;
}

// MAMBA_GATE_NORM_WGSL (granite-wgsl-runtime.ts:1590-1606) of every row, then
// the operand planes of out_proj.
template <int TPR, int E>
__global__ __launch_bounds__(kWg) void k_pf_gate(PfGateArgs a, int rows) {
  warm_kernarg<(int)(sizeof(PfGateArgs) + 8)>();
  __shared__ float red[4];
  const RowLane<TPR> L(rows);
  float v[E][8], z[E][8];
#pragma unroll
  for (int e = 0; e < E; ++e) load8(a.y + (size_t)L.t * a.k + min(8 * (L.c0 + TPR * e), a.k - 8), v[e]);
  part_row<TPR, E>(a.z, L, z);
#pragma unroll
  for (int e = 0; e < E; ++e)
#pragma unroll
    for (int i = 0; i < 8; ++i)
      v[e][i] = 8 * (L.c0 + TPR * e) < a.k ? __fmul_rn(v[e][i], __fdiv_rn(z[e][i], __fadd_rn(1.0f, expf(-z[e][i])))) : 0.f;
  row_rmsnorm<TPR, E>(v, L, a.w, a.k, a.eps, red);
  row_planes<TPR, E>(v, L, a.kpad, a.xh, a.xl, a.xscale, a.xs, red);
}

__device__ __forceinline__ int row_pos(const KvAddr& k, int t) { return k.row_pos ? k.row_pos[t] : k.p0 + t; }
__device__ __forceinline__ int row_seq(const KvAddr& k, int t) { return k.row_seq ? k.row_seq[t] : k.seq0; }
// element offset of (sequence, kv head, position)'s K/V row
__device__ __forceinline__ size_t kv_row(const KvAddr& k, int kv_heads, int hd, int seq, int kv, int pos) {
  if (!k.pages) return ((size_t)kv * k.ctx + pos) * hd;
  const int page = k.pages[(size_t)seq * k.max_pages + pos / kKvPage];
  return (((size_t)page * kv_heads + kv) * kKvPage + (pos & (kKvPage - 1))) * hd;
}

// (cos, sin) of rotary pair d at a position: from the engine's table (filled with
// this expression on the device) or inline where it keeps none. The inline form
// (two range reductions per pair) held k_pf_rope_kv at 19.8 us per 2047 rows of
// the Qwen3-0.6B shape.
__device__ __forceinline__ float2 rope_cs(const PfRopeArgs& a, int pos, int d, int half) {
  if (a.rope_cs) return a.rope_cs[(size_t)pos * half + d];
  const float ang = __fmul_rn((float)pos, a.rope_inv[d]);
  return make_float2(cosf(ang), sinf(ang));
}

// Per-head q/k RMSNorm and rotary embedding of every prompt row (position
// p0 + t), the new k and v into the cache. One wave per (row, head): workgroup
// (t, y) holds heads 4y .. 4y + 3 of the q heads followed by the kv heads. A
// lane owns rotary pairs p = lane + 64 j and gathers their two elements (and,
// for a kv head, its v dims) straight from the projections' partial sums, every
// load issued at once. Same operation order as the decode attention's phase B.
// The rotated q goes to the q part of the row for the attention kernels.
__global__ __launch_bounds__(kWg) void k_pf_rope_kv(PfRopeArgs a) {
  constexpr int NP = 2;  // pairs per lane: head_dim <= 256
  const int t = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int hh = blockIdx.y * 4 + wave;
  const int nh = a.heads + a.kv_heads;
  if (hh >= nh) return;
  const int pos = row_pos(a.kv, t);
  const int hd = a.hd, half = hd / 2;
  const bool is_k = hh >= a.heads;
  const int kv = hh - a.heads;
  float* row = a.qkv + (size_t)t * a.ld;
  const int col = is_k ? a.heads * hd + kv * hd : hh * hd;  // the head's columns in the q|k|v row
  const PartSum& P = is_k ? a.pk : a.pq;
  const int pcol = is_k ? kv * hd : hh * hd;                 // ... in its projection's result
  int ia[NP], ib[NP];
  float x0[NP], x1[NP];
  float2 cs[NP];
#pragma unroll
  for (int j = 0; j < NP; ++j) {
    const int d = min(lane + 64 * j, half - 1);
    ia[j] = a.interleaved ? 2 * d : d;
    ib[j] = a.interleaved ? 2 * d + 1 : d + half;
    cs[j] = rope_cs(a, pos, d, half);
  }
  if (P.p) {
    // both elements of every pair in one round of loads
    int jj[2 * NP];
    float xx[2 * NP];
#pragma unroll
    for (int j = 0; j < NP; ++j) {
      jj[2 * j] = pcol + ia[j];
      jj[2 * j + 1] = pcol + ib[j];
    }
    part_gather<2 * NP>(P, t, jj, xx);
#pragma unroll
    for (int j = 0; j < NP; ++j) {
      x0[j] = xx[2 * j];
      x1[j] = xx[2 * j + 1];
    }
  } else {
#pragma unroll
    for (int j = 0; j < NP; ++j) {
      x0[j] = row[col + ia[j]];
      x1[j] = row[col + ib[j]];
    }
  }
  if (a.bias) {
#pragma unroll
    for (int j = 0; j < NP; ++j) {
      x0[j] = __fadd_rn(x0[j], a.bias[col + ia[j]]);
      x1[j] = __fadd_rn(x1[j], a.bias[col + ib[j]]);
    }
  }
  float r = 1.0f;
  if (a.qn_w) {
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < NP; ++j)
      if (lane + 64 * j < half) ss += x0[j] * x0[j] + x1[j] * x1[j];
    ss = wave_sum(ss);
    r = 1.0f / sqrtf(ss / (float)hd + a.eps);
  }
  const float* w = is_k ? a.kn_w : a.qn_w;
  size_t base = 0;
  if (is_k) base = kv_row(a.kv, a.kv_heads, hd, row_seq(a.kv, t), kv, pos);
#pragma unroll
  for (int j = 0; j < NP; ++j) {
    const int d = lane + 64 * j;
    if (d >= half) continue;
    float v0 = x0[j], v1 = x1[j];
    if (a.qn_w) {
      v0 = __fmul_rn(__fmul_rn(v0, r), w[ia[j]]);
      v1 = __fmul_rn(__fmul_rn(v1, r), w[ib[j]]);
    }
    const float co = cs[j].x, si = cs[j].y;
    const float y0 = __fsub_rn(__fmul_rn(v0, co), __fmul_rn(v1, si));
    const float y1 = __fadd_rn(__fmul_rn(v0, si), __fmul_rn(v1, co));
    if (is_k) {
      if (a.kv16) {
        ((__half*)a.kv.kc)[base + ia[j]] = __float2half_rn(y0);
        ((__half*)a.kv.kc)[base + ib[j]] = __float2half_rn(y1);
      } else {
        ((float*)a.kv.kc)[base + ia[j]] = y0;
        ((float*)a.kv.kc)[base + ib[j]] = y1;
      }
    } else {
      row[col + ia[j]] = y0;
      row[col + ib[j]] = y1;
    }
  }
  if (is_k) {
    const int vcol = (a.heads + a.kv_heads) * hd + kv * hd;
    // lane's dims lane + 64 i (head_dim <= 256), every load issued at once
    int jv[4];
    float vv[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) jv[i] = min(lane + 64 * i, hd - 1);
    if (a.pv.p) {
#pragma unroll
      for (int i = 0; i < 4; ++i) jv[i] += kv * hd;
      part_gather<4>(a.pv, t, jv, vv);
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) vv[i] = row[vcol + jv[i]];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int d = lane + 64 * i;
      if (d >= hd) continue;
      if (a.bias) vv[i] = __fadd_rn(vv[i], a.bias[vcol + d]);
      if (a.kv16)
        ((__half*)a.kv.vc)[base + d] = __float2half_rn(vv[i]);
      else
        ((float*)a.kv.vc)[base + d] = vv[i];
    }
  }
}

// Causal attention of every prompt row: one workgroup per (token, q head),
// keys [start, p0 + t] of the cache in blocks of 256 (one per thread), an
// online softmax across blocks. q is the rotated row left by k_pf_rope_kv.
__global__ __launch_bounds__(kWg) void k_pf_attn(PfAttnArgs a) {
  __shared__ float qs[256];
  __shared__ float red[8];
  __shared__ float wsh[kWg];
  __shared__ float part[kWg];
  const int t = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
  const int G = a.heads / a.kv_heads, kv = h / G;
  const int hd = a.hd;
  const int pos = row_pos(a.kv, t);
  const int start = (a.window != 0 && pos + 1 > a.window) ? pos + 1 - a.window : 0;
  const float* q = a.qkv + (size_t)t * a.ld + h * hd;
  for (int d = tid; d < hd; d += kWg) qs[d] = q[d];
  __syncthreads();
  const size_t head_base = (size_t)kv * a.kv.ctx * hd;
  float M = -INFINITY, L = 0.f;
  // output dims: thread tid owns dim (tid % hd) for key slice tid / hd
  const int nsl = kWg / hd, my_d = tid % hd, my_sl = tid / hd;
  float o = 0.f;
  for (int b0 = start; b0 <= pos; b0 += kWg) {
    const int p = b0 + tid;
    float s = -INFINITY;
    if (p <= pos) {
      float acc = 0.f;
      if (a.kv16) {
        const __half* kr = (const __half*)a.kv.kc + head_base + (size_t)p * hd;
        for (int d = 0; d < hd; d += 8) {
          const uint4 w4 = *(const uint4*)(kr + d);
          const uint32_t w[4] = {w4.x, w4.y, w4.z, w4.w};
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            acc += qs[d + 2 * i] * h2f(w[i]);
            acc += qs[d + 2 * i + 1] * h2f(w[i] >> 16);
          }
        }
      } else {
        const float* kr = (const float*)a.kv.kc + head_base + (size_t)p * hd;
        for (int d = 0; d < hd; ++d) acc += qs[d] * kr[d];
      }
      s = acc * a.scale;
    }
    float mb = wave_max(s);
    __syncthreads();
    if ((tid & 63) == 0) red[tid >> 6] = mb;
    __syncthreads();
    mb = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    const float e = p <= pos ? expf(s - mb) : 0.f;
    wsh[tid] = e;
    float lb = wave_sum(e);
    __syncthreads();
    if ((tid & 63) == 0) red[4 + (tid >> 6)] = lb;
    __syncthreads();
    lb = (red[4] + red[5]) + (red[6] + red[7]);
    const float Mn = fmaxf(M, mb);
    const float ro = M == -INFINITY ? 0.f : expf(M - Mn), rb = expf(mb - Mn);
    // weighted V of this block for my dim over my slice of the keys
    float ob = 0.f;
    const int nk = min(kWg, pos + 1 - b0);
    for (int kk = my_sl; kk < nk; kk += nsl) {
      const size_t vi = head_base + (size_t)(b0 + kk) * hd + my_d;
      const float vv = a.kv16 ? __half2float(((const __half*)a.kv.vc)[vi]) : ((const float*)a.kv.vc)[vi];
      ob += wsh[kk] * vv;
    }
    part[tid] = ob;
    __syncthreads();
    if (tid < hd) {
      float sb = 0.f;
      for (int sl = 0; sl < nsl; ++sl) sb += part[sl * hd + tid];
      o = o * ro + sb * rb;
    }
    L = L * ro + lb * rb;
    M = Mn;
    __syncthreads();
  }
  if (tid < hd) a.out[(size_t)t * a.ldo + h * hd + tid] = o * (1.0f / L);
}

// Causal attention of the prompt rows on the matrix cores (fp16 K/V cache):
// one workgroup per (block of 64 / G tokens, kv head); its 64 query rows
// (token, q head of the group) are four waves of 16. The products run
// transposed so that no operand needs a shuffle: per block of 64 keys,
//   S^T = K Q^T  (v_mfma 16x16x32: K rows from LDS, q split into fp16 hi + lo),
// whose accumulator layout (lane: query lane % 16, keys 4 (lane / 16) + i of
// each 16-key tile) is a B operand layout with the keys permuted, so
//   O^T += V^T P^T  (P split into hi + lo; V^T staged in LDS, V exact)
// takes P straight from the registers as 16x16x32 products too (twice the rate
// of the 16x16x16 shape): the lane's eight k of a 32-key step are keys 4 quad + i
// of the step's two 16-key tiles, and V^T is staged with its keys in that order, and every lane keeps the running
// maximum, sum and output of its own query. Scores are kept in log2 units
// (scale * log2 e folded into one multiply) and the exponent base is only
// raised when a block's maximum exceeds it by more than 8 (P <= 2^8 stays
// exact enough in fp16 hi + lo and the sums in fp32), so the output rescale
// is skipped by the whole wave on most blocks; blocks that no query of the
// wave sees partly masked skip the masking. The next block's K and V are
// loaded into registers while the current one is multiplied; workgroups
// with the most keys (the last tokens) are dispatched first, and workgroup
// ids step through the kv heads fastest: consecutive ids go to different XCDs
// (id mod 8), so with 8 kv heads each XCD's L2 holds one head's K/V.
constexpr int kFaKeys = 64;

// max / sum over the four lanes of one query (lanes l, l ^ 16, l ^ 32, l ^ 48)
__device__ __forceinline__ float xquad_max(float v) {
  float a, b;
  swap16(v, a, b);
  v = fmaxf(a, b);
  swap32(v, a, b);
  return fmaxf(a, b);
}
__device__ __forceinline__ float xquad_sum(float v) {
  float a, b;
  swap16(v, a, b);
  v = a + b;
  swap32(v, a, b);
  return a + b;
}

template <int HD, bool PAGED>
__global__ __launch_bounds__(kWg, HD <= 128 ? 2 : 1) void k_pf_fattn(PfAttnArgs a) {
  extern __shared__ __align__(16) _Float16 fsm[];
  constexpr int KS = HD + 8, VS = kFaKeys + 8;
  constexpr int NKP = HD / 32;                   // K pieces (8 halves) per thread and block
  constexpr int NVI = HD >= 64 ? HD / 64 : 1;    // V items (2 keys x 8 dims) per thread and block
  constexpr int VITEMS = (kFaKeys / 2) * (HD / 8);
  _Float16* ks = fsm;                  // [64 keys][KS]
  _Float16* vt = ks + kFaKeys * KS;    // [HD dims][VS]   (V transposed)
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // rows of one workgroup share a sequence: one token per workgroup when
  // every row has its own
  const int G = a.heads / a.kv_heads, TW = a.kv.row_seq ? 1 : 64 / G;
  const int ntiles = gridDim.x / a.kv_heads;
  // query tiles in complementary pairs: workgroups q and q + hi (dispatched
  // one dispatch round apart, so that one CU holds both while the grid is two
  // rounds) take tiles ntiles - 1 - q and q, whose causal key ranges sum to a
  // constant
  const int q = (int)blockIdx.x / a.kv_heads, hi = ntiles - ntiles / 2;
  const int kv = blockIdx.x % a.kv_heads, t0 = (q < hi ? ntiles - 1 - q : q - hi) * TW;
  const int col = lane & 15, quad = lane >> 4;
  const int seq = row_seq(a.kv, t0);
  const __half* kc = (const __half*)a.kv.kc;
  const __half* vc = (const __half*)a.kv.vc;

  // this lane's query: row 16 * wave + col of the workgroup (token, head);
  // its B operand of S^T (dims 32 k + 8 quad .. + 8), hi and lo halves
  const int qr = 16 * wave + col, qt = t0 + qr / G;
  const bool qok = qr < TW * G && qt < a.rows;
  half8_t qh[HD / 32], ql[HD / 32];
  {
    const float* q = a.qkv + (size_t)(qok ? qt : t0) * a.ld + (kv * G + qr % G) * HD;
#pragma unroll
    for (int k = 0; k < HD / 32; ++k) {
      float v[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = q[32 * k + 8 * quad + i];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float x = qok ? v[i] : 0.f;
        qh[k][i] = (_Float16)x;
        ql[k][i] = (_Float16)(x - (float)qh[k][i]);
      }
    }
  }
  const int qpos = qok ? row_pos(a.kv, qt) : -1;
  const int qstart = (a.window != 0 && qpos + 1 > a.window) ? qpos + 1 - a.window : 0;
  // the wave's key range seen by every one of its queries (unused rows excluded)
  // (in scalar registers: the masking below is then a branch, not 48 instructions of every block)
  const int wpos_min = __builtin_amdgcn_readfirstlane((int)-wave_max(-(float)(qok ? qpos : 1 << 24)));
  const int wstart_max = __builtin_amdgcn_readfirstlane((int)wave_max((float)(qok ? qstart : 0)));
  const float sl2 = a.scale * 1.44269504088896341f;
  const int t_last = min(t0 + TW, a.rows) - 1;
  const int pos_hi = row_pos(a.kv, t_last), pos_lo = row_pos(a.kv, t0);
  const int st_lo = (a.window != 0 && pos_lo + 1 > a.window) ? pos_lo + 1 - a.window : 0;
  const int kb_lo = st_lo / kFaKeys, kb_hi = pos_hi / kFaKeys;

  // staging: K piece (key, 8 dims) and V item (key pair, 8 dims) of the thread
  uint4 kreg[NKP], vreg[NVI][2];
  // block kb's first K/V row (workgroup-uniform) and the last row of the block
  // that may be addressed (the cache ends inside the block)
  auto block_base = [&](int kb) -> size_t {
    if constexpr (PAGED) {
      const int page = ld_scalar(a.kv.pages + (size_t)seq * a.kv.max_pages + kb);
      return ((size_t)page * a.kv_heads + kv) * kKvPage * HD;
    } else {
      return ((size_t)kv * a.kv.ctx + kb * kFaKeys) * HD;
    }
  };
  auto key_cap = [&](int kb) -> int { return PAGED ? kFaKeys - 1 : min(kFaKeys - 1, a.kv.ctx - 1 - kb * kFaKeys); };
  // Keys past the block's last position were never written (fresh pages can
  // hold NaN bit patterns, and P = 0 times NaN is NaN): staged as zeros.
  auto fetch = [&](int kb) {
    const int k0 = kb * kFaKeys, cap = key_cap(kb);
    const size_t base = block_base(kb);
    const __half* kb0 = kc + base;
    const __half* vb0 = vc + base;
#pragma unroll
    for (int j = 0; j < NKP; ++j) {
      const int piece = tid + kWg * j, key = piece / (HD / 8), d8 = (piece % (HD / 8)) * 8;
      const uint4 v = ldg4(kb0 + (uint32_t)(min(key, cap) * HD + d8));
      kreg[j] = k0 + key <= pos_hi ? v : make_uint4(0u, 0u, 0u, 0u);
    }
#pragma unroll
    for (int j = 0; j < NVI; ++j) {
      const int item = min(tid + kWg * j, VITEMS - 1), kp = item % (kFaKeys / 2), d8 = (item / (kFaKeys / 2)) * 8;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int key = 2 * kp + h;
        const uint4 v = ldg4(vb0 + (uint32_t)(min(key, cap) * HD + d8));
        vreg[j][h] = k0 + key <= pos_hi ? v : make_uint4(0u, 0u, 0u, 0u);
      }
    }
  };
  auto stage = [&]() {
#pragma unroll
    for (int j = 0; j < NKP; ++j) {
      const int piece = tid + kWg * j, key = piece / (HD / 8), d8 = (piece % (HD / 8)) * 8;
      *(uint4*)(ks + key * KS + d8) = kreg[j];
    }
#pragma unroll
    for (int j = 0; j < NVI; ++j) {
      const int item = tid + kWg * j, kp = item % (kFaKeys / 2), d8 = (item / (kFaKeys / 2)) * 8;
      if (item < VITEMS) {
        // dims d8 .. d8 + 7 of keys 2 kp and 2 kp + 1 as eight (key, key + 1) pairs;
        // key 32 s + 16 h + 4 q + i of the block sits at 32 s + 8 q + 4 h + i
        const int key = 2 * kp, at = (key & 32) + 8 * ((key & 15) >> 2) + 4 * ((key >> 4) & 1) + (key & 3);
        const uint32_t* w0 = (const uint32_t*)&vreg[j][0];
        const uint32_t* w1 = (const uint32_t*)&vreg[j][1];
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          *(uint32_t*)(vt + (d8 + 2 * d) * VS + at) = (w0[d] & 0xffffu) | (w1[d] << 16);
          *(uint32_t*)(vt + (d8 + 2 * d + 1) * VS + at) = (w0[d] >> 16) | (w1[d] & 0xffff0000u);
        }
      }
    }
  };

  float m_use = -INFINITY, l_run = 0.f;  // exponent base (log2 units) and running sum of the lane's query
  float4_t o[HD / 16];  // O^T tiles: dims 16 dt + 4 quad + i of the lane's query
#pragma unroll
  for (int d = 0; d < HD / 16; ++d) o[d] = float4_t{0.f, 0.f, 0.f, 0.f};

  fetch(kb_lo);
  for (int kb = kb_lo; kb <= kb_hi; ++kb) {
    const int k0 = kb * kFaKeys;
    __syncthreads();  // the previous block's K / V^T are consumed
    stage();
    __syncthreads();
    fetch(min(kb + 1, kb_hi));  // the next block (the last one again at the end: cache hits)
    // S^T for the block's 64 keys x the wave's 16 queries (four 16 x 16 tiles,
    // their chains interleaved: no MFMA waits on the one before it)
    float4_t sa[4];
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) sa[kt] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < HD / 32; ++k) {
      half8_t kk[4];
#pragma unroll
      for (int kt = 0; kt < 4; ++kt) kk[kt] = *(const half8_t*)(ks + (16 * kt + col) * KS + 32 * k + 8 * quad);
#pragma unroll
      for (int kt = 0; kt < 4; ++kt) sa[kt] = mfma32(kk[kt], qh[k], sa[kt]);
#pragma unroll
      for (int kt = 0; kt < 4; ++kt) sa[kt] = mfma32(kk[kt], ql[k], sa[kt]);
    }
    if (!(k0 >= wstart_max && k0 + kFaKeys - 1 <= wpos_min)) {
      // some query of the wave sees only part of the block
#pragma unroll
      for (int kt = 0; kt < 4; ++kt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int key = k0 + 16 * kt + 4 * quad + i;
          sa[kt][i] = key >= qstart && key <= qpos ? sa[kt][i] : -INFINITY;
        }
    }
    float mb = -INFINITY;
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)
#pragma unroll
      for (int i = 0; i < 4; ++i) mb = fmaxf(mb, sa[kt][i]);
    mb = xquad_max(mb) * sl2;  // (log2 units; the scale is positive)
    const bool upd = mb > m_use + 8.0f;
    const float alpha = !upd ? 1.0f : (m_use == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_use - mb));
    m_use = upd ? mb : m_use;
    const float base = m_use == -INFINITY ? 0.f : m_use;  // masked scores give exp2(-inf) = 0
    float lb = 0.f;
    half8_t ph[2], pl[2];  // of the block's two 32-key steps
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)
#pragma unroll
      for (int i = 0; i < 4; i += 2) {
        // (pairs, for the packed conversion)
        const float2_t p = {__builtin_amdgcn_exp2f(fmaf(sa[kt][i], sl2, -base)),
                            __builtin_amdgcn_exp2f(fmaf(sa[kt][i + 1], sl2, -base))};
        lb += p[0] + p[1];
        const half2_t h = __builtin_convertvector(p, half2_t);
        const float2_t r = {p[0] - (float)h[0], p[1] - (float)h[1]};
        const half2_t lo = __builtin_convertvector(r, half2_t);
        ph[kt >> 1][4 * (kt & 1) + i] = h[0];
        ph[kt >> 1][4 * (kt & 1) + i + 1] = h[1];
        pl[kt >> 1][4 * (kt & 1) + i] = lo[0];
        pl[kt >> 1][4 * (kt & 1) + i + 1] = lo[1];
      }
    l_run = l_run * alpha + xquad_sum(lb);
    if (__builtin_amdgcn_ballot_w64(upd) != 0) {
#pragma unroll
      for (int d = 0; d < HD / 16; ++d) o[d] *= alpha;
    }
    // O^T += V^T P^T over the block's keys (two 32-key steps), DG dim tiles'
    // chains interleaved
    constexpr int DG = HD >= 64 ? 4 : 2;
#pragma unroll
    for (int d = 0; d < HD / 16; d += DG) {
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        half8_t vv[DG];
#pragma unroll
        for (int e = 0; e < DG; ++e) vv[e] = *(const half8_t*)(vt + (16 * (d + e) + col) * VS + 32 * st + 8 * quad);
#pragma unroll
        for (int e = 0; e < DG; ++e) o[d + e] = mfma32(vv[e], ph[st], o[d + e]);
#pragma unroll
        for (int e = 0; e < DG; ++e) o[d + e] = mfma32(vv[e], pl[st], o[d + e]);
      }
    }
  }
  __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));  // the last redundant fetch has returned
  // out[token][head * HD + dim]: the lane's query, dims 16 d + 4 quad .. + 4
  if (qok) {
    float* out = a.out + (size_t)qt * a.ldo + (kv * G + qr % G) * HD;
    const float inv = 1.0f / l_run;
#pragma unroll
    for (int d = 0; d < HD / 16; ++d)
      *(float4*)(out + 16 * d + 4 * quad) = make_float4(o[d][0] * inv, o[d][1] * inv, o[d][2] * inv, o[d][3] * inv);
  }
}

// Decode attention of batch rows over paged K/V. One workgroup per (kv head,
// row, segment) walks a segment of the row's pages [start, pos] with the
// decode attention's layout: a page's K rows in registers (four lanes per
// position), its V rows in registers (wave w holds dims [w*HD/4, (w+1)*HD/4)
// of every position, a lane 2 or 4 dims of every PG-th position); the next
// page's rows are requested before the current page is reduced. The softmax
// runs online over the pages (running maximum and sum per head, the
// accumulators rescaled when the maximum grows). With one segment per row the
// workgroup writes the attention output; otherwise a partial [max, sum,
// acc[hd]] per head for k_bd_merge.
template <int HD, bool ROPE>
__global__ __launch_bounds__(kWg) void k_bd_walk(PfAttnArgs a, float* part, int max_pages, int nseg, PfRopeArgs ra) {
  warm_kernarg<(int)(sizeof(PfAttnArgs) + 2 * sizeof(void*) + sizeof(PfRopeArgs))>();  // (dependent argument rounds hit the scalar cache)
  constexpr int DPT = HD / 4;  // K dims per lane
  constexpr int NKV = DPT / 8;
  constexpr int VD = HD >= 256 ? 4 : 2, VW = VD / 2;
  constexpr int DW = HD / 4 / VD;  // lanes per V position row: 8 or 16
  constexpr int LDW = DW == 8 ? 3 : 4;
  constexpr int PG = 64 / DW, NP = kKvPage / PG;
  static_assert(kKvPage == 64 && (DW == 8 || DW == 16), "page geometry");
  __shared__ __align__(16) float q_s[8 * HD];
  __shared__ float wmx[4][8];
  __shared__ __align__(16) float ew[8][kKvPage];
  __shared__ float lsum[8];
  __shared__ int pt_s[64];  // the segment's page table entries (max_pages <= 64)
  const int kv = blockIdx.x, r = blockIdx.y, sg = blockIdx.z, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int G = a.heads / a.kv_heads;
  // With ROPE, the rotary/K-V write of this (row, kv head) comes first (the
  // arithmetic of k_pf_rope_kv): the G q heads, k and v, gathered from the
  // projections' partial sums, are G + 2 items over the waves; q goes to LDS,
  // k and v to the cache. Item `it`: four elements per lane (q/k: the two
  // elements of the lane's rotary pairs lane and lane + 64; v: dims lane + 64 e),
  // clamped so that every item issues the same loads. The first item's loads
  // go out before anything else.
  constexpr int NPR = 2;  // pairs per lane: head_dim <= 256
  constexpr int HALF = HD / 2;
  int ia[NPR], ib[NPR];
#pragma unroll
  for (int j = 0; j < NPR; ++j) {
    const int d = min(lane + 64 * j, HALF - 1);
    ia[j] = ra.interleaved ? 2 * d : d;
    ib[j] = ra.interleaved ? 2 * d + 1 : d + HALF;
  }
  // item it's partial sums and columns
  auto item_cols = [&](int it, int (&jj)[4]) -> const PartSum& {
    if (it == G + 1) {
#pragma unroll
      for (int e = 0; e < 4; ++e) jj[e] = kv * HD + min(lane + 64 * e, HD - 1);
      return ra.pv;
    }
    const int pcol = it == G ? kv * HD : (kv * G + it) * HD;
#pragma unroll
    for (int j = 0; j < NPR; ++j) {
      jj[2 * j] = pcol + ia[j];
      jj[2 * j + 1] = pcol + ib[j];
    }
    return it == G ? ra.pk : ra.pq;
  };
  const int it0 = min(wave, G + 1);
  int jj0[4];
  float w0[4][4];
  if constexpr (ROPE) part_issue<4>(item_cols(it0, jj0), r, jj0, w0);
  // The row's position and sequence and its page table entries are read
  // through the scalar cache (the scalar load counter is separate: waiting for
  // them never waits for the vector loads in flight), and the segment's
  // entries are staged in LDS for the page loop.
  const int pos = ld_scalar(a.kv.row_pos + r);
  const int start = (a.window != 0 && pos + 1 > a.window) ? pos + 1 - a.window : 0;
  const int j_lo = start / kKvPage, np = pos / kKvPage - j_lo + 1;
  // this segment's pages [p_lo, p_hi) of the row's range
  const int p_lo = j_lo + np * sg / nseg, p_hi = j_lo + np * (sg + 1) / nseg;  // np, nseg <= 64
  const int seq = ld_scalar(a.kv.row_seq + r);
  const int* ptab = a.kv.pages + (size_t)seq * a.kv.max_pages;
  const int jnew = pos / kKvPage;  // the newest page (entries past it may be unassigned)
  const int pt_mine = ptab[min(p_lo + tid, jnew)];
  const int phys0 = ld_scalar(ptab + min(p_lo, jnew));
  const float* q = a.qkv + (size_t)r * a.ld + kv * G * HD;
  const int kp = 16 * wave + (lane >> 2), kd0 = (lane & 3) * DPT;
  const int pg = lane >> LDW, vd = wave * (HD / 4) + VD * (lane & (DW - 1));
  const int ei = (kp % PG) * NP + kp / PG;
  // a page's rows are addressed from a workgroup-uniform base with 32-bit
  // per-lane byte offsets (scalar base + vector offset loads: no 64-bit
  // address arithmetic per load)
  const uint32_t koff = 2u * (uint32_t)(kp * HD + kd0), voff = 2u * (uint32_t)(pg * HD + vd);
  auto load = [&](int phys, uint4 (&kr)[NKV], uint32_t (&vr)[NP][VW]) {
    const size_t pb = ((size_t)__builtin_amdgcn_readfirstlane(phys) * a.kv_heads + kv) * (kKvPage * HD * 2);
    const char* kb = (const char*)a.kv.kc + pb;
    const char* vb = (const char*)a.kv.vc + pb;
#pragma unroll
    for (int v = 0; v < NKV; ++v) kr[v] = ldg4(kb + koff + 16 * v);
#pragma unroll
    for (int t = 0; t < NP; ++t) {
      const char* p = vb + (2 * PG * HD) * t + voff;
      if constexpr (VW == 1) {
        vr[t][0] = ldg1(p);
      } else {
        const uint2 w = ldg2(p);
        vr[t][0] = w.x;
        vr[t][VW - 1] = w.y;
      }
    }
  };
  float mrun[8], o[8][VD];
#pragma unroll
  for (int g = 0; g < 8; ++g) {
    mrun[g] = -INFINITY;
#pragma unroll
    for (int k = 0; k < VD; ++k) o[g][k] = 0.f;
  }
  float lrun[8];  // wave g % 4's running sum of head g
#pragma unroll
  for (int g = 0; g < 8; ++g) lrun[g] = 0.f;
  auto page = [&](int j, uint4 (&kr)[NKV], uint32_t (&vr)[NP][VW]) {
    const int k0 = j * kKvPage;
    const bool valid = k0 + kp >= start && k0 + kp <= pos;
    float s[8];
#pragma unroll
    for (int g = 0; g < 8; ++g) s[g] = 0.f;
#pragma unroll
    for (int v = 0; v < NKV; ++v) {
      const uint32_t w[4] = {kr[v].x, kr[v].y, kr[v].z, kr[v].w};
#pragma unroll
      for (int g = 0; g < 8; ++g) {
        if (g < G) {
          const float4 q0 = *(const float4*)(q_s + g * HD + kd0 + 8 * v);
          const float4 q1 = *(const float4*)(q_s + g * HD + kd0 + 8 * v + 4);
          s[g] = fmaf(q0.x, h2f(w[0]), s[g]);
          s[g] = fmaf(q0.y, h2f(w[0] >> 16), s[g]);
          s[g] = fmaf(q0.z, h2f(w[1]), s[g]);
          s[g] = fmaf(q0.w, h2f(w[1] >> 16), s[g]);
          s[g] = fmaf(q1.x, h2f(w[2]), s[g]);
          s[g] = fmaf(q1.y, h2f(w[2] >> 16), s[g]);
          s[g] = fmaf(q1.z, h2f(w[3]), s[g]);
          s[g] = fmaf(q1.w, h2f(w[3] >> 16), s[g]);
        }
      }
    }
#pragma unroll
    for (int g = 0; g < 8; ++g) {
      if (g < G) {
        const float sc = group_sum<4>(s[g]);
        s[g] = valid ? sc * a.scale : -INFINITY;
        const float mw = wave_max(s[g]);
        if (lane == 0) wmx[wave][g] = mw;
      }
    }
    __syncthreads();  // the page maxima (and the previous page's weights are consumed)
    float alpha[8];
#pragma unroll
    for (int g = 0; g < 8; ++g) {
      if (g < G) {
        const float mp = fmaxf(fmaxf(wmx[0][g], wmx[1][g]), fmaxf(wmx[2][g], wmx[3][g]));
        const float mn = fmaxf(mrun[g], mp);  // finite: every page of the range holds a position
        alpha[g] = exp_fast(mrun[g] - mn);     // 0 on the first page
        mrun[g] = mn;
        const float e = valid ? exp_fast(s[g] - mn) : 0.f;
        if ((lane & 3) == 0) ew[g][ei] = e;
      }
    }
    __syncthreads();  // the page's weights
    if (k0 < start || k0 + kKvPage - 1 > pos) {
#pragma unroll
      for (int t = 0; t < NP; ++t) {
        const int p = k0 + pg + PG * t;
        if (p < start || p > pos)
#pragma unroll
          for (int u = 0; u < VW; ++u) vr[t][u] = 0u;
      }
    }
#pragma unroll
    for (int g = 0; g < 8; ++g) {
      if (g < G) {
        if (g % 4 == wave) lrun[g] = lrun[g] * alpha[g] + wave_sum(ew[g][lane]);
#pragma unroll
        for (int k = 0; k < VD; ++k) o[g][k] *= alpha[g];
#pragma unroll
        for (int t4 = 0; t4 < NP / 4; ++t4) {
          const float4 w4 = *(const float4*)(&ew[g][pg * NP + 4 * t4]);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int t = 4 * t4 + i;
            const float wt = i == 0 ? w4.x : i == 1 ? w4.y : i == 2 ? w4.z : w4.w;
#pragma unroll
            for (int u = 0; u < VW; ++u) {
              o[g][2 * u] = fmaf(wt, h2f(vr[t][u]), o[g][2 * u]);
              o[g][2 * u + 1] = fmaf(wt, h2f(vr[t][u] >> 16), o[g][2 * u + 1]);
            }
          }
        }
      }
    }
  };
  uint4 ka[NKV], kb2[NKV];
  uint32_t va[NP][VW], vb2[NP][VW];
  if constexpr (ROPE) {
    // (one segment) the first page is requested before the rotary work; when
    // it is the newest, it is requested again after the barrier below that
    // publishes the new row
    load(phys0, ka, va);
    const size_t base = (((size_t)ld_scalar(ptab + jnew) * ra.kv_heads + kv) * kKvPage + (pos & (kKvPage - 1))) * HD;
    auto item_do = [&](int it, const float (&xx)[4]) {
      if (it == G + 1) {
#pragma unroll
        for (int e = 0; e < HD / 64; ++e) ((__half*)ra.kv.vc)[base + lane + 64 * e] = __float2half_rn(xx[e]);
        return;
      }
      const bool is_k = it == G;
      const float x0[NPR] = {xx[0], xx[2]}, x1[NPR] = {xx[1], xx[3]};
      float rn = 1.0f;
      if (ra.qn_w) {
        float ss = 0.f;
#pragma unroll
        for (int j = 0; j < NPR; ++j)
          if (lane + 64 * j < HALF) ss += x0[j] * x0[j] + x1[j] * x1[j];
        ss = wave_sum(ss);
        rn = 1.0f / sqrtf(ss / (float)HD + ra.eps);
      }
      const float* w = is_k ? ra.kn_w : ra.qn_w;
#pragma unroll
      for (int j = 0; j < NPR; ++j) {
        const int d = lane + 64 * j;
        if (d >= HALF) continue;
        float v0 = x0[j], v1 = x1[j];
        if (ra.qn_w) {
          v0 = __fmul_rn(__fmul_rn(v0, rn), w[ia[j]]);
          v1 = __fmul_rn(__fmul_rn(v1, rn), w[ib[j]]);
        }
        const float2 cs = rope_cs(ra, pos, d, HALF);
        const float co = cs.x, si = cs.y;
        const float y0 = __fsub_rn(__fmul_rn(v0, co), __fmul_rn(v1, si));
        const float y1 = __fadd_rn(__fmul_rn(v0, si), __fmul_rn(v1, co));
        if (is_k) {
          ((__half*)ra.kv.kc)[base + ia[j]] = __float2half_rn(y0);
          ((__half*)ra.kv.kc)[base + ib[j]] = __float2half_rn(y1);
        } else {
          q_s[it * HD + ia[j]] = y0;
          q_s[it * HD + ib[j]] = y1;
        }
      }
    };
    if (wave < G + 2) {
      float xx[4];
      part_finish<4>(item_cols(it0, jj0), r, jj0, w0, xx);
      item_do(wave, xx);
    }
    for (int it = wave + 4; it < G + 2; it += 4) {  // groups above 2
      int jj[4];
      float xx[4];
      part_gather<4>(item_cols(it, jj), r, jj, xx);
      item_do(it, xx);
    }
    if (tid < 64) pt_s[tid] = pt_mine;
    __syncthreads();  // q and the page table in LDS; the new K/V row visible to this workgroup's loads
    if (p_lo == jnew) load(phys0, ka, va);
  } else {
    // q first: its loads complete before the page's, which stay in flight
    float qv[6];
#pragma unroll
    for (int c = 0; c < 6; ++c) qv[c] = tid + kWg * c < G * HD ? q[tid + kWg * c] : 0.f;
    if (p_lo < p_hi) load(phys0, ka, va);
#pragma unroll
    for (int c = 0; c < 6; ++c)
      if (tid + kWg * c < G * HD) q_s[tid + kWg * c] = qv[c];
    if (tid < 64) pt_s[tid] = pt_mine;
    __syncthreads();
  }
  // The next page's loads are issued unconditionally (the last page requests
  // itself again, a cache hit) so that the loop body has no branch around
  // them: the compiler's load-counter waits then count exactly and page j's
  // reduction waits for page j's rows only.
  for (int j = p_lo; j < p_hi; j += 2) {
    load(pt_s[min(j + 1, p_hi - 1) - p_lo], kb2, vb2);
    __builtin_amdgcn_sched_barrier(0);  // issued before page j's reduction starts
    page(j, ka, va);
    if (j + 1 >= p_hi) break;
    load(pt_s[min(j + 2, p_hi - 1) - p_lo], ka, va);
    __builtin_amdgcn_sched_barrier(0);
    page(j + 1, kb2, vb2);
  }
  __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));  // the last redundant request has returned
#pragma unroll
  for (int g = 0; g < 8; ++g)
    if (g < G)
#pragma unroll
      for (int k = 0; k < VD; ++k) o[g][k] = pg_sum<DW>(o[g][k]);
  // lanes (pg, dw) write item pg + PG * it (head item / VD, dim vd + item % VD)
  if (nseg == 1) {
    if (lane == 0)
#pragma unroll
      for (int g = 0; g < 8; ++g)
        if (g < G && g % 4 == wave) lsum[g] = lrun[g];
    __syncthreads();
    const size_t col = (size_t)kv * G * HD;
    for (int it = 0; it * PG < G * VD; ++it) {
      const int item = it * PG + pg;
      float val = 0.f;
#pragma unroll
      for (int g = 0; g < 8; ++g)
#pragma unroll
        for (int k = 0; k < VD; ++k)
          if (g * VD + k == item) val = o[g][k];
      if (item < G * VD) {
        const size_t i = col + (item / VD) * HD + vd + item % VD;
        const float y = val / lsum[item / VD];
        if (a.oh) {
          // the next GEMM's operand planes at scale 1: hi + lo keeps ~22 bits
          // for |y| >= 2^-3; below that lo is an fp16 subnormal (absolute
          // spacing 2^-24), so the relative error grows to ~2^-24 / |y|
          // (2^-17 at 0.01, 2^-14 at 1e-3), still far inside the 1e-3 logits bar
          const _Float16 h = (_Float16)y;
          const size_t at = plane_at(r, (int)i, a.okpad);
          a.oh[at] = h;
          a.ol[at] = (_Float16)(y - (float)h);
        } else {
          a.out[(size_t)r * a.ldo + i] = y;
        }
      }
    }
    if (a.oh && kv == 0) {
      // the planes past the row's last column are zero; its scale is 1
      for (int i = a.heads * HD + tid; i < a.okpad; i += kWg) {
        a.oh[plane_at(r, i, a.okpad)] = (_Float16)0.f;
        a.ol[plane_at(r, i, a.okpad)] = (_Float16)0.f;
      }
      if (tid == 0) a.oscale[r] = 1.0f;
    }
  } else {
    const int rowf = attn_rowf(G, HD);
    float* out = part + (((size_t)r * a.kv_heads + kv) * max_pages + sg) * rowf;
    for (int it = 0; it * PG < G * VD; ++it) {
      const int item = it * PG + pg;
      float val = 0.f;
#pragma unroll
      for (int g = 0; g < 8; ++g)
#pragma unroll
        for (int k = 0; k < VD; ++k)
          if (g * VD + k == item) val = o[g][k];
      if (item < G * VD) out[(item / VD) * (HD + 2) + 2 + vd + item % VD] = val;
    }
    if (lane == 0)
#pragma unroll
      for (int g = 0; g < 8; ++g)
        if (g < G && g % 4 == wave) {
          out[g * (HD + 2)] = mrun[g];  // -inf for a segment without pages
          out[g * (HD + 2) + 1] = lrun[g];
        }
  }
}

// out row r, heads of kv head blockIdx.x: the segments' partials merged
// (weights exp(m_j - M), normalised by the merged sum).
template <int HD>
__global__ __launch_bounds__(kWg) void k_bd_merge(PfAttnArgs a, const float* part, int max_pages, int nseg) {
  __shared__ float w[8][64];
  __shared__ float inv[8];
  const int kv = blockIdx.x, r = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int G = a.heads / a.kv_heads;
  const int n = nseg;
  const int rowf = attn_rowf(G, HD);
  const float* base = part + ((size_t)r * a.kv_heads + kv) * max_pages * rowf;
  for (int g = wave; g < G; g += 4) {
    float M = -INFINITY;
    for (int j = lane; j < n; j += 64) M = fmaxf(M, base[(size_t)j * rowf + g * (HD + 2)]);
    M = wave_max(M);
    float L = 0.f;
    for (int j = lane; j < n; j += 64) {
      const float mj = base[(size_t)j * rowf + g * (HD + 2)];
      const float f = mj == -INFINITY ? 0.f : expf(mj - M);
      w[g][j] = f;
      L += base[(size_t)j * rowf + g * (HD + 2) + 1] * f;
    }
    L = wave_sum(L);
    if (lane == 0) inv[g] = 1.0f / L;
  }
  __syncthreads();
  for (int i = tid; i < G * HD; i += kWg) {
    const int g = i / HD, d = i - g * HD;
    float acc = 0.f;
    for (int j = 0; j < n; ++j) acc += base[(size_t)j * rowf + g * (HD + 2) + 2 + d] * w[g][j];
    a.out[(size_t)r * a.ldo + (kv * G + g) * HD + d] = acc * inv[g];
  }
}

// Greedy id of each row of logits: the largest value, the lowest index on
// ties, NaN never chosen (argmax's better(), llama-wgsl-runtime.ts:3645-3791).
// Stage 1: kArgParts workgroups per row each reduce a slice to (value, id).
constexpr int kArgParts = 32;

__global__ __launch_bounds__(kWg) void k_row_argmax1(const float* logits, int vocab, float* pv, uint32_t* pi) {
  __shared__ float sv[kWg];
  __shared__ uint32_t si[kWg];
  const float* row = logits + (size_t)blockIdx.x * vocab;
  const int per = (vocab + kArgParts - 1) / kArgParts;
  const int lo = blockIdx.y * per, hi = min(vocab, lo + per);
  float bv = kNegBig;
  uint32_t bi = 0xffffffffu;
  for (int i = lo + threadIdx.x; i < hi; i += kWg) {
    const float v = row[i];
    if (better(v, (uint32_t)i, bv, bi)) {
      bv = v;
      bi = (uint32_t)i;
    }
  }
  sv[threadIdx.x] = bv;
  si[threadIdx.x] = bi;
  __syncthreads();
  for (int stride = kWg / 2; stride >= 1; stride >>= 1) {
    if ((int)threadIdx.x < stride && better(sv[threadIdx.x + stride], si[threadIdx.x + stride], sv[threadIdx.x],
                                            si[threadIdx.x])) {
      sv[threadIdx.x] = sv[threadIdx.x + stride];
      si[threadIdx.x] = si[threadIdx.x + stride];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    pv[blockIdx.x * kArgParts + blockIdx.y] = sv[0];
    pi[blockIdx.x * kArgParts + blockIdx.y] = si[0];
  }
}

// Stage 2: one wave per row over the row's kArgParts candidates.
__global__ __launch_bounds__(64) void k_row_argmax2(const float* pv, const uint32_t* pi, int32_t* out) {
  __shared__ float sv[64];
  __shared__ uint32_t si[64];
  const int r = blockIdx.x, l = threadIdx.x;
  sv[l] = l < kArgParts ? pv[r * kArgParts + l] : kNegBig;
  si[l] = l < kArgParts ? pi[r * kArgParts + l] : 0xffffffffu;
  __syncthreads();
  for (int stride = 32; stride >= 1; stride >>= 1) {
    if (l < stride && better(sv[l + stride], si[l + stride], sv[l], si[l])) {
      sv[l] = sv[l + stride];
      si[l] = si[l + stride];
    }
    __syncthreads();
  }
  if (l == 0) out[r] = si[0] == 0xffffffffu ? 0 : (int32_t)si[0];
}

}  // namespace

// ---- host launchers ----------------------------------------------------------------

bool gemm_needs_sums(int type, int k, int rows) { return gemm_int_sums(type) && !gemm_sk_applies(type, k, rows); }

// the GEMMs address the activation planes with 32-bit byte offsets
bool gemm_planes_fit(const GemmArgs& a) { return a.t >= 1 && (int64_t)plane_rows(a.t) * a.kpad * 2 <= (int64_t)UINT32_MAX; }

size_t fattn_shared_bytes(int hd) {
  return sizeof(_Float16) * ((size_t)kFaKeys * (hd + 8) + (size_t)hd * (kFaKeys + 8));
}

// Tiles and K split of a launch over the integer codes. The larger the tile, the
// less each CU reads and dequantizes per product, as long as the grid covers the
// device; a K split makes up for too few tiles but costs its partial sums twice.
// Measured (us, Q4_K; weight rows x K at token rows: ni, tj, split):
//   4096 x 1024 at 2047: 47.9 (8, 2, 1)  50.7 (4, 2, 1)  55.4 (4, 1, 1)
//   1024 x 2048 at 2047: 26.8 (4, 2, 2)  28.5 (8, 2, 4)  29.9 (4, 1, 1)
//   4096 x 1024 at 1200: 31.4 (8, 2, 2)  41.5 (8, 2, 1)  35.6 (4, 1, 1)
//   4096 x 1024 at 288:  15.4 (4, 1, 1)  16.2 (4, 1, 2)  18.1 (8, 1, 1)
//   1024 x 2048 at 288:  12.2 (4, 1, 4)  13.9 (4, 1, 7)  15.8 (8, 1, 7)
//   1024 x 2048 at 80:    6.6 (4, 1, 8)   7.8 (4, 1, 4)   7.9 (8, 1, 8)
// One row tile (up to 64 rows) has 128 workgroups wanted: prompts of 3, 16 and 64 rows of the
// LFM2.5-350M Q8_0 shape take 0.90, 0.93, 0.99 ms (256: 1.00, 1.04, 1.16), of Granite Q8_0 1.70,
// 1.79, 2.00 (1.73, 1.87, 2.14), of SmolLM2-135M Q8_0 1.34, 1.44, 1.51 (1.32, 1.42, 1.51). (At one
// step of a SmolLM2 run with a 1.3 repetition penalty two ids are 6e-6 apart after it; either
// number has taken the oracle's id there since the block scales left the GEMM's operands.)
struct IntTiles {
  int ni, tj, ks;
};
IntTiles gemm_int_tiles(const GemmArgs& a, int n_rows, int64_t part_cap) {
  auto tiles = [&](int ni, int tj) {
    return ((n_rows + 16 * ni - 1) / (16 * ni)) * ((a.t + 64 * tj - 1) / (64 * tj));
  };
  const int tj = a.t > 512 ? 2 : 1, ni = tj == 2 && tiles(8, 2) >= 256 ? 8 : 4;
  const int n = tiles(ni, tj), want = tj == 2 ? 512 : a.t > 64 ? 256 : 128;
  const int step = gemm_int_step(a.w.type), nst = (a.w.k + step - 1) / step;
  int ks = std::max(1, std::min({(want + n / 2) / n, nst, kMaxDeferSplit}));
  while (ks > 1 && (int64_t)ks * a.t * n_rows > part_cap) --ks;
  return {ni, tj, ks};
}

hipError_t launch_gemm(const GemmArgs& a0, hipStream_t s) {
  GemmArgs a = a0;
  if (!a.n_all && gemm_sk_applies(a) && a.w.n >= 128 * 4 * kSkRows) {
    // many row groups (the lm_head): four per workgroup over the whole K, x shared in LDS
    const dim3 grid((a.w.n + 4 * kSkRows - 1) / (4 * kSkRows));
    const int nt = gemm_sk_tiles(a.t);
    CHONK_SK_LAUNCH(k_gemm_lm, a.w.type, nt, grid, gemm_lm_shared_bytes(nt), s, a);
    return hipGetLastError();
  }
  if (!a.n_all && gemm_sk_applies(a)) {
    const int groups = (a.w.n + kSkRows - 1) / kSkRows;
    int ks = a.part ? gemm_sk_split(a, groups) : 1;
    while (ks > 1 && (int64_t)ks * a.t * a.w.n > a.part_cap) --ks;
    a.ksplit = ks;
    a.defer = 0;
    hipError_t e = launch_gemm_sk(a, a.w.n, s);
    if (e != hipSuccess || ks == 1) return e;
    const int64_t total = (int64_t)a.t * a.w.n;
    const int blocks = (int)std::min<int64_t>((total + kWg - 1) / kWg, 4096);
    hipLaunchKernelGGL(k_gemm_reduce, dim3(blocks), dim3(kWg), 0, s, a);
    return hipGetLastError();
  }
  if (!gemm_planes_fit(a)) return hipErrorInvalidValue;
  const IntTiles it = gemm_int_tiles(a, a.w.n, a.part ? a.part_cap : 0);
  a.ksplit = it.ks;
  const hipError_t e = launch_gemm_int(a, a.w.n, it.ni, it.tj, s);
  if (e != hipSuccess || a.ksplit == 1) return e;
  const int64_t total = (int64_t)a.t * a.w.n;
  const int blocks = (int)std::min<int64_t>((total + kWg - 1) / kWg, 4096);
  hipLaunchKernelGGL(k_gemm_reduce, dim3(blocks), dim3(kWg), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_gemm_deferred(const GemmArgs& a0, float* region, int64_t region_cap, PartSum* out, hipStream_t s) {
  GemmArgs a = a0;
  const int N = a.n_all ? a.n_all : a.w.n;
  if (a.n_all) {
    // fused segments: one type and K, in order, starting at multiples of 64 rows
    // (n2 starts a segment only where there is a third: k of two matrices may end anywhere)
    if (a.n1 <= 0 || a.n1 % kSkRows || a.n2 < a.n1 || (a.n_all > a.n2 && a.n2 % kSkRows) || a.n_all < a.n2 ||
        a.w2.type != a.w.type ||
        a.w3.type != a.w.type || a.w2.k != a.w.k || a.w3.k != a.w.k || a.w.n != a.n1 ||
        (a.n2 > a.n1 && a.w2.n != a.n2 - a.n1) || (a.n_all > a.n2 && a.w3.n != a.n_all - a.n2))
      return hipErrorInvalidValue;
  }
  if ((int64_t)a.t * N > region_cap) return hipErrorInvalidValue;
  if (gemm_sk_applies(a)) {
    // one 64-k block per wave when the partial sums of that split fit
    const int ks1 = a.w.k / kSkBlockK / 4;
    const bool one = ks1 <= kMaxDeferSplit && (int64_t)ks1 * a.t * N <= region_cap;
    int ks = one ? ks1 : gemm_sk_split(a, (N + kSkRows - 1) / kSkRows);
    while (ks > 1 && (int64_t)ks * a.t * N > region_cap) --ks;
    a.ksplit = ks;
    a.part = region;
    a.defer = 1;
    hipError_t e;
    if (one) {
      const dim3 grid((N + kSkRows - 1) / kSkRows, 1, ks);
      const int nt = gemm_sk_tiles(a.t);
      CHONK_SK_LAUNCH(k_gemm_sk1, a.w.type, nt, grid, gemm_sk_shared_bytes(nt), s, a);
      e = hipGetLastError();
    } else {
      e = launch_gemm_sk(a, N, s);
    }
    out->p = region;
    out->n = N;
    out->ld = N;
    out->ks = ks;
    out->zs = (int64_t)a.t * N;
    return e;
  }
  if (!gemm_planes_fit(a)) return hipErrorInvalidValue;
  out->p = region;
  out->n = N;
  out->ld = N;
  out->zs = (int64_t)a.t * N;
  const IntTiles it = gemm_int_tiles(a, N, region_cap);
  a.ksplit = out->ks = it.ks;
  a.part = region;
  a.defer = 1;
  return launch_gemm_int(a, N, it.ni, it.tj, s);
}

hipError_t launch_gemm_glu(const GemmArgs& a0, float* region, int64_t region_cap, PartSum* out, hipStream_t s) {
  GemmArgs a = a0;
  *out = PartSum{};
  if (gemm_sk_applies(a) || !gemm_planes_fit(a)) return hipSuccess;
  const IntTiles it = gemm_int_tiles(a, a.n2, region_cap);
  if (it.ks != 1 || (it.ni == 4 && it.tj == 2) || (int64_t)a.t * a.n1 > region_cap) return hipSuccess;
  a.ksplit = 1;
  a.part = region;
  a.defer = 1;
  const hipError_t e = launch_gemm_int(a, a.n2, it.ni, it.tj, s);
  if (e != hipSuccess) return e;
  out->p = region;
  out->n = out->ld = a.n1;
  out->ks = 1;
  out->zs = (int64_t)a.t * a.n1;
  return hipSuccess;
}

hipError_t init_gemm_attributes() {
  if (const hipError_t e = init_gemm_int_attributes(); e != hipSuccess) return e;
  for (const void* f : {(const void*)k_gemm_sk<QT_Q4_K>, (const void*)k_gemm_sk<QT_Q6_K>,
                        (const void*)k_gemm_sk1<QT_Q4_K, 4>, (const void*)k_gemm_sk1<QT_Q6_K, 4>}) {
    const hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)gemm_sk_shared_bytes());
    if (e != hipSuccess) return e;
  }
  const void* fa[8] = {(const void*)k_pf_fattn<32, false>,  (const void*)k_pf_fattn<64, false>,
                       (const void*)k_pf_fattn<128, false>, (const void*)k_pf_fattn<256, false>,
                       (const void*)k_pf_fattn<32, true>,   (const void*)k_pf_fattn<64, true>,
                       (const void*)k_pf_fattn<128, true>,  (const void*)k_pf_fattn<256, true>};
  const int hds[4] = {32, 64, 128, 256};
  for (int i = 0; i < 8; ++i) {
    const hipError_t e =
        hipFuncSetAttribute(fa[i], hipFuncAttributeMaxDynamicSharedMemorySize, (int)fattn_shared_bytes(hds[i & 3]));
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

// The instance of a per-row kernel for `rows` rows of kpad elements: a wave per
// row once those cover the device a few times over (kRowWave rows), else the
// row over two or four waves.
constexpr int kRowWave = 1024;
#define CHONK_ROW_INST(tpr, e, ...)                              \
  {                                                              \
    constexpr int TPR = tpr, E = e;                              \
    const dim3 grid((rows + kWg / TPR - 1) / (kWg / TPR));       \
    __VA_ARGS__;                                                 \
    return hipGetLastError();                                    \
  }
#define CHONK_ROW_CASE(kpad, ...)                                        \
  do {                                                                   \
    if ((kpad) > kPfRowMax) return hipErrorInvalidValue;                 \
    if (rows >= kRowWave && (kpad) <= 3072) {                            \
      if ((kpad) <= 1024) CHONK_ROW_INST(64, 2, __VA_ARGS__)             \
      if ((kpad) <= 2048) CHONK_ROW_INST(64, 4, __VA_ARGS__)             \
      CHONK_ROW_INST(64, 6, __VA_ARGS__)                                 \
    }                                                                    \
    if ((kpad) <= 1024) CHONK_ROW_INST(128, 1, __VA_ARGS__)              \
    if ((kpad) <= 2048) CHONK_ROW_INST(256, 1, __VA_ARGS__)              \
    if ((kpad) <= 4096) CHONK_ROW_INST(256, 2, __VA_ARGS__)              \
    CHONK_ROW_INST(256, 4, __VA_ARGS__)                                  \
  } while (0)

hipError_t launch_pf_split(const PfSplitArgs& a, int rows, hipStream_t s) {
  if (a.k % 32 != 0 || a.ldx % 4 != 0 || ((uintptr_t)a.x & 15)) return hipErrorInvalidValue;
  if (a.norm_b || a.add_bias) {
    if ((a.w && !a.norm_b) || (a.add.p && !a.add_bias)) return hipErrorInvalidValue;
    CHONK_ROW_CASE(a.kpad, hipLaunchKernelGGL((k_pf_split<TPR, E, true>), grid, dim3(kWg), 0, s, a, rows));
  }
  CHONK_ROW_CASE(a.kpad, hipLaunchKernelGGL((k_pf_split<TPR, E, false>), grid, dim3(kWg), 0, s, a, rows));
}
hipError_t launch_pf_embed(const QMat& embed, const int32_t* tok, float scale, const float* pos, int p0, int k,
                           float* x, int rows, hipStream_t s) {
  hipLaunchKernelGGL(k_pf_embed, dim3(rows), dim3(kWg), 0, s, embed, tok, scale, pos, p0, k, x);
  return hipGetLastError();
}
hipError_t launch_pf_conv(const PfConvArgs& a, int rows, hipStream_t s) {
  if (rows < 1 || a.p.n < 3 * a.k) return hipErrorInvalidValue;
  CHONK_ROW_CASE(a.kpad, hipLaunchKernelGGL((k_pf_conv<TPR, E>), grid, dim3(kWg), 0, s, a, rows));
}
hipError_t launch_pf_conv_state(const PfConvArgs& a, int rows, hipStream_t s) {
  if (rows < 1 || a.p.n < 3 * a.k) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_pf_conv_state, dim3((a.k + kWg - 1) / kWg), dim3(kWg), 0, s, a, rows);
  return hipGetLastError();
}
hipError_t launch_pf_mamba(const PfMambaArgs& a, hipStream_t s) {
  static_assert(kMbSteps % 8 == 0 && kWg == 2 * kMbStates && kWg == kMbSteps * kMbCh && kWg == 32 * kMbCh, "scan geometry");
  if (a.rows < 1 || a.inner != a.heads * kMbHd || a.conv != a.inner + 2 * kMbStates ||
      a.p.n < a.inner + a.conv + a.heads)
    return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_pf_mamba_conv, dim3((a.conv + a.heads + kWg - 1) / kWg, (a.rows + kMbConvRows - 1) / kMbConvRows),
                     dim3(kWg), 0, s, a);
  hipLaunchKernelGGL(k_pf_mamba_scan, dim3(a.heads, kMbHd / kMbCh), dim3(kWg), 0, s, a);
  return hipGetLastError();
}
hipError_t launch_pf_gate(const PfGateArgs& a, int rows, hipStream_t s) {
  CHONK_ROW_CASE(a.kpad, hipLaunchKernelGGL((k_pf_gate<TPR, E>), grid, dim3(kWg), 0, s, a, rows));
}
hipError_t launch_pf_glu_split(const PfGluArgs& a, int rows, hipStream_t s) {
  CHONK_ROW_CASE(a.kpad, hipLaunchKernelGGL((k_pf_glu_split<TPR, E>), grid, dim3(kWg), 0, s, a, rows));
}
hipError_t launch_pf_rope_kv(const PfRopeArgs& a, int rows, hipStream_t s) {
  const int nh = a.heads + a.kv_heads;
  if (a.hd > 256) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_pf_rope_kv, dim3(rows, (nh + 3) / 4), dim3(kWg), 0, s, a);
  return hipGetLastError();
}
hipError_t launch_pf_attn(const PfAttnArgs& a, int rows, hipStream_t s) {
  const int G = a.heads / a.kv_heads;
  if (!a.kv16 || G > 16) {
    if (a.kv.pages || a.kv.row_seq) return hipErrorInvalidValue;  // paged rows need the fp16 cache
    hipLaunchKernelGGL(k_pf_attn, dim3(rows, a.heads), dim3(kWg), 0, s, a);
    return hipGetLastError();
  }
  PfAttnArgs b = a;
  b.rows = rows;
  const int tw = a.kv.row_seq ? 1 : 64 / G;
  const dim3 grid((rows + tw - 1) / tw * a.kv_heads);
  const size_t sh = fattn_shared_bytes(a.hd);
  const bool paged = a.kv.pages != nullptr;
#define CHONK_FA(H)                                                              \
  if (paged)                                                                     \
    hipLaunchKernelGGL((k_pf_fattn<H, true>), grid, dim3(kWg), sh, s, b);        \
  else                                                                           \
    hipLaunchKernelGGL((k_pf_fattn<H, false>), grid, dim3(kWg), sh, s, b);
  switch (a.hd) {
    case 32: CHONK_FA(32) break;
    case 64: CHONK_FA(64) break;
    case 128: CHONK_FA(128) break;
    case 256: CHONK_FA(256) break;
    default: return hipErrorInvalidValue;
  }
#undef CHONK_FA
  return hipGetLastError();
}

}  // namespace chonk

namespace chonk {
hipError_t launch_row_argmax(const float* logits, int vocab, int rows, float* scratch, int32_t* out, hipStream_t s) {
  float* pv = scratch;
  uint32_t* pi = (uint32_t*)(scratch + (size_t)rows * kArgParts);
  hipLaunchKernelGGL(k_row_argmax1, dim3(rows, kArgParts), dim3(kWg), 0, s, logits, vocab, pv, pi);
  hipLaunchKernelGGL(k_row_argmax2, dim3(rows), dim3(64), 0, s, pv, pi, out);
  return hipGetLastError();
}
}  // namespace chonk

namespace chonk {
int bd_attn_segments(int rows, int kv_heads, int max_pages) {
  // enough (kv head, row, segment) workgroups to cover the device; with one
  // segment the walk writes the output (and may do the rotary/K-V write)
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
    return 0;
  return std::max(1, std::min(max_pages, (2 * cus + rows * kv_heads - 1) / std::max(1, rows * kv_heads)));
}

hipError_t launch_bd_attn(const PfAttnArgs& a0, int rows, float* part, int64_t part_cap, hipStream_t s, bool* planes,
                          const PfRopeArgs* rope) {
  PfAttnArgs a = a0;
  a.rows = rows;
  const int G = a.heads / a.kv_heads;
  const int mp = a.kv.max_pages;
  const int nseg = bd_attn_segments(rows, a.kv_heads, mp);
  if (nseg <= 0 || (rope && nseg != 1)) return hipErrorInvalidValue;
  PfRopeArgs ra{};
  if (rope) ra = *rope;
  if (rope && (!ra.pq.p || !ra.pk.p || !ra.pv.p)) return hipErrorInvalidValue;  // the partial sums are read
  if (!a.kv16 || !a.kv.pages || !a.kv.row_seq || !a.kv.row_pos || G > 8 || G * a.hd > 1536 || mp > 64 ||
      (nseg > 1 && (int64_t)rows * a.kv_heads * mp * attn_rowf(G, a.hd) > part_cap))
    return hipErrorInvalidValue;
  if (nseg > 1) a.oh = nullptr;  // the merge writes a.out
  if (a.oh && (!a.ol || !a.oscale || a.okpad < a.heads * a.hd)) return hipErrorInvalidValue;
  *planes = a.oh != nullptr;
  const dim3 g1(a.kv_heads, rows, nseg), g2(a.kv_heads, rows);
#define CHONK_BD_CASE(HH)                                                                     \
  case HH:                                                                                    \
    if (rope)                                                                                 \
      hipLaunchKernelGGL((k_bd_walk<HH, true>), g1, dim3(kWg), 0, s, a, part, mp, nseg, ra);  \
    else                                                                                      \
      hipLaunchKernelGGL((k_bd_walk<HH, false>), g1, dim3(kWg), 0, s, a, part, mp, nseg, ra); \
    if (nseg > 1) hipLaunchKernelGGL(k_bd_merge<HH>, g2, dim3(kWg), 0, s, a, part, mp, nseg); \
    return hipGetLastError();
  switch (a.hd) {
    CHONK_BD_CASE(64)
    CHONK_BD_CASE(128)
    CHONK_BD_CASE(256)
    default: return hipErrorInvalidValue;
  }
#undef CHONK_BD_CASE
}
}  // namespace chonk

