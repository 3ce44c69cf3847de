// Batched (many-token) kernels: operand split, dequant-fused MFMA GEMM and the
// per-token glue of a prompt processed as T rows at once (prefill.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "device_common.h"

namespace chonk {

// GEMM_SWIGLU / GEMM_GEGLU: w is gate and w2 up (n2 = 2 n1), the result is
// silu(gate) * up or gelu_tanh(gate) * up with n1 columns (gemm_int.hip)
enum GemmEpi : int32_t { GEMM_STORE = 0, GEMM_ADD = 1, GEMM_SWIGLU = 2, GEMM_GEGLU = 3 };

// y[t][n] (=|+=) 2^-ws * xscale[t] * sum_k (xh + xl)[t][k] * (W 2^ws)[n][k]
struct GemmArgs {
  QMat w;                 // striped weights, N = w.n rows of K = w.k
  // a fused launch over up to three matrices of one type and K (e.g. q | k | v):
  // output rows [0, n1) come from w, [n1, n2) from w2, [n2, n_all) from w3 (n_all =
  // n2: two matrices); the segment starts are multiples of 64 rows. n_all = 0: w alone.
  QMat w2, w3;
  int32_t n1, n2, n_all, pad0;
  const _Float16* xh;     // activation planes (plane_at), zero past K
  const _Float16* xl;
  const float* xscale;    // [t]
  const _Float16* xs;     // [t][hi | lo][kpad / 32] sums of x over 32 k (pf_split's), or null
  float* y;               // [t][ldy]
  int32_t ldy, t, kpad, epi;
  int32_t ws;             // weight exponent
  int32_t ksplit;         // K partitions (grid z); > 1 needs `part`
  float* part;            // [ksplit][t][w.n] partial sums, reduced in order by the launcher
  int64_t part_cap;       // floats available in part
  int32_t defer;          // 1: always leave partials in part (launch_gemm_deferred)
};

// Where a row batch's K/V live: the engine's contiguous cache
// ([kv_heads][ctx][hd] per layer, pages == null), or pages of 64 positions
// ([page][kv_heads][64][hd]) through a per-sequence page table.
struct KvAddr {
  void *kc, *vc;
  int32_t ctx;
  const int32_t* pages;   // [seq][max_pages] physical page ids, or null
  int32_t max_pages;
  int32_t seq0;           // sequence of every row when row_seq is null
  const int32_t* row_seq; // [rows] per-row sequence, or null
  const int32_t* row_pos; // [rows] per-row position, or null (p0 + row)
  int32_t p0;
};
constexpr int kKvPage = 64;

// A GEMM result left as K-split partial sums: value(t, j) = sum over z < ks
// of p[z * zs + t * n + j], added in z order (the consumer kernel adds them).
struct PartSum {
  const float* p;         // null: absent
  int32_t n, ks;          // valid columns, K splits
  int64_t zs;             // floats between splits
  int32_t ld, pad0;       // floats between rows (>= n: a column range of a fused result)
};

struct PfSplitArgs {
  const float* x;         // [rows][ldx]
  int32_t ldx, k, kpad;
  const float* w;         // RMSNorm weight [k], or null for a plain split
  float eps;
  _Float16 *xh, *xl;      // planes (plane_at)
  float* xscale;          // [rows]
  _Float16* xs;           // [rows][hi | lo][kpad / 32]: sums of the scaled row over 32 k, times 2^-5
  // residual update first (x must then be writable): x += add, or with
  // add_w (the Gemma-3 sandwich) x = clamp(x + RMSNorm(add) * add_w, +-65000)
  PartSum add;
  const float* add_w;
  float add_scale;        // x += add_scale * add when not 0 (granitehybrid)
  // GPT-2: x = sanitize(x + (add + add_bias)), and w / norm_b are a LayerNorm
  const float *add_bias, *norm_b;
};

enum PfAct : int32_t { PF_SWIGLU = 0, PF_GEGLU = 1, PF_GELU_BIAS = 2, PF_DONE = 3 };

struct PfGluArgs {
  PartSum pg, pu;         // gate and up rows [rows][k] (deferred GEMM results)
  const float* bias;      // PF_GELU_BIAS: gelu(up + bias); pg is not read. PF_DONE: pu is the product already
  int32_t k, kpad, act;
  _Float16 *xh, *xl;
  float* xscale;
  _Float16* xs;
};

// lfm2 short convolution over the rows of a pass, in_proj rows B | C | x of k
// channels each, as operand planes; s1 / s2 are B * x two and one positions
// before row 0, and after launch_pf_conv_state those before the next pass.
struct PfConvArgs {
  PartSum p;
  int32_t k, kpad;
  const float* w;         // [k][3] taps
  float *s1, *s2;
  _Float16 *xh, *xl;
  float* xscale;
  _Float16* xs;
};

// granitehybrid Mamba2 layer over the rows of a pass; in_proj rows z | xBC | dt.
struct PfMambaArgs {
  PartSum p;              // in_proj rows (inner + conv + heads columns)
  int32_t rows, inner, conv, heads, p0;
  const float *conv_w, *conv_b, *dt_bias, *a_neg, *d;
  float* conv_state;      // [2][conv][3], indexed by the position's parity
  float* ssm_state;       // [heads][32][128]
  float* xbc;             // [rows][pf_mamba_ld]: silu(conv(xBC)) | dt | decay
  float* y;               // [rows][inner] scan output
};

// floats per row of PfMambaArgs.xbc (16-byte rows for the scan's loads)
constexpr int pf_mamba_ld(int conv, int heads) { return (conv + 2 * heads + 3) / 4 * 4; }

// y * silu(z), RMSNorm, operand planes (the Mamba2 gated norm)
struct PfGateArgs {
  PartSum z;
  const float *y, *w;
  int32_t k, kpad;
  float eps;
  _Float16 *xh, *xl;
  float* xscale;
  _Float16* xs;
};

struct PfRopeArgs {
  float* qkv;             // [rows][ld]: q | k | v (gathered from pq, pk, pv when given)
  PartSum pq, pk, pv;
  int32_t ld, hd, heads, kv_heads, interleaved, kv16;
  const float *qn_w, *kn_w;  // per-head RMSNorm weights (null: none)
  const float* bias;      // [q | k | v] added to the projections first (null: none)
  float eps;
  const float* rope_inv;  // [hd/2]
  const float2* rope_cs;  // [position][hd/2] (cos, sin) of those angles, or null
  KvAddr kv;
};

struct PfAttnArgs {
  const float* qkv;       // rotated q rows
  int32_t ld;
  float* out;             // [rows][ldo]
  int32_t ldo, heads, kv_heads, hd, window, kv16;
  int32_t rows;           // rows of the pass (set by the launcher)
  float scale;
  KvAddr kv;
  // batched decode: the next GEMM's operand planes (plane_at, okpad; hi, lo) and
  // row scales, written instead of `out` when set and the rows are not split
  // into segments (the output of attention needs no scaling: |x| <= max |V|)
  _Float16* oh;
  _Float16* ol;
  float* oscale;
  int32_t okpad;
};

// Widest row the per-row glue kernels hold in registers (four runs of eight
// elements in each of 256 threads).
constexpr int kPfRowMax = 8192;

// Operand planes hold the rows in MFMA operand order: 16 rows x 32 columns are
// 512 consecutive halves, lane l of a wave finding its eight (row l % 16, columns
// 8 (l / 16) .. + 8) at 8 l, so that a wave's operand load is one run of 1 KiB.
// (Row after row, the load touched 64-byte pieces of 16 rows 2 kpad bytes apart:
// the 2047-row Q4_K GEMMs of the Qwen3-0.6B shape took 51.0 us instead of 43.9.)
// Rows are padded to a multiple of 16; the padding rows are never written and
// only reach results that are dropped.
constexpr int plane_rows(int rows) { return (rows + 15) / 16 * 16; }
__host__ __device__ inline size_t plane_at(int row, int col, int kpad) {
  return ((size_t)(row >> 4) * (kpad >> 5) + (col >> 5)) * 512 + ((col >> 3) & 3) * 128 + (row & 15) * 8 + (col & 7);
}

// K padded for the GEMM's activation planes.
constexpr int gemm_kpad(int k) { return (k + 127) / 128 * 128; }

// The GEMM over the weights' integer codes (gemm_int.hip): 16 ni weight rows x
// 64 tj token rows per workgroup ((ni, tj) of (8, 2), (4, 1) or, without a GLU
// epilogue, (4, 2)), a.ksplit and the output
// as set by the caller. K splits are whole steps of gemm_int_step columns; types
// with block offsets (gemm_int_sums) need a.xs.
bool gemm_int_sums(int type);
constexpr int gemm_int_step(int type) { return type == QT_Q4_K || type == QT_Q5_K || type == QT_Q6_K ? 256 : 128; }
hipError_t launch_gemm_int(const GemmArgs& a, int n_rows, int ni, int tj, hipStream_t s);
hipError_t init_gemm_int_attributes();
// Whether a GEMM of `rows` token rows over a matrix of this type and K reads the
// sums of x (GemmArgs.xs) beside the operand planes.
bool gemm_needs_sums(int type, int k, int rows);
hipError_t init_gemm_attributes();
// Picks the K split for a launch (at least ~256 workgroups when the partial
// buffer allows) and launches the GEMM and, when split, the ordered reduction.
hipError_t launch_gemm(const GemmArgs& a, hipStream_t s);
// The GEMM with its result left as partial sums in `region` (capacity in
// floats): the K split is chosen as in launch_gemm within the region, and no
// reduction is launched; *out describes the partials for the consumer.
hipError_t launch_gemm_deferred(const GemmArgs& a, float* region, int64_t region_cap, PartSum* out, hipStream_t s);
// launch_gemm_deferred of gate | up (a.w, a.w2) leaving act(gate) * up; *out with
// p null and nothing launched where the tiles would split K or have no instance.
hipError_t launch_gemm_glu(const GemmArgs& a, float* region, int64_t region_cap, PartSum* out, hipStream_t s);
hipError_t launch_pf_split(const PfSplitArgs& a, int rows, hipStream_t s);
// Embedding rows times scale, plus (pos != null, GPT-2) the rows of the
// position table from position p0 on.
hipError_t launch_pf_embed(const QMat& embed, const int32_t* tok, float scale, const float* pos, int p0, int k,
                           float* x, int rows, hipStream_t s);
hipError_t launch_pf_conv(const PfConvArgs& a, int rows, hipStream_t s);
hipError_t launch_pf_conv_state(const PfConvArgs& a, int rows, hipStream_t s);
hipError_t launch_pf_mamba(const PfMambaArgs& a, hipStream_t s);
hipError_t launch_pf_gate(const PfGateArgs& a, int rows, hipStream_t s);
hipError_t launch_pf_glu_split(const PfGluArgs& a, int rows, hipStream_t s);
hipError_t launch_pf_rope_kv(const PfRopeArgs& a, int rows, hipStream_t s);
hipError_t launch_pf_attn(const PfAttnArgs& a, int rows, hipStream_t s);
// Decode attention of rows with their own sequences (kv.row_seq) over paged
// K/V: per-page partials in `part`, then a merge per (row, kv head).
// Segments per row of the batched decode attention (1: one workgroup walks all
// of a (row, kv head)'s pages; 0: no device).
int bd_attn_segments(int rows, int kv_heads, int max_pages);
// *planes: whether the launch wrote a.oh / a.ol / a.oscale (else a.out). With
// `rope` (only when bd_attn_segments is 1) the attention also does that
// launch's rotary/K-V write, reading q, k and v from the projections.
hipError_t launch_bd_attn(const PfAttnArgs& a, int rows, float* part, int64_t part_cap, hipStream_t s, bool* planes,
                          const PfRopeArgs* rope);
// Greedy id per row of logits [rows][vocab] (the reference's argmax ordering);
// scratch holds 64 floats per row.
hipError_t launch_row_argmax(const float* logits, int vocab, int rows, float* scratch, int32_t* out, hipStream_t s);

}  // namespace chonk
