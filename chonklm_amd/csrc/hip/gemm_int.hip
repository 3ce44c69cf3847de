// Prompt GEMM over the weights' integer codes (Q4_K, Q6_K, Q8_0), gfx950.
//
//   Q4_K  W = d (sc (q - 8)) + c,   c = 8 d sc - dmin m per 32 k
//   Q6_K  W = d (sc (q - 32))
//   Q8_0  W = d q
//
// sc (q - 8) of Q4_K is an integer below 2^9, exact in one fp16 plane, so the
// matrix cores multiply it with the hi and lo activation planes (two products
// per 16x16x32 step where fp16 hi + lo weights take three, and no rounded
// weight): the sums of a 256-k super-block are scaled by d once, and c, which
// is constant over 32 k, meets the sums of x over those 32 k in one more MFMA
// per super-block. sc (q - 32) of Q6_K has 13 bits and d q of Q8_0 up to 19, so
// those keep two planes, split exactly (h = fp16(v), l = v - h by one fma).
// Codes become fp16 by byte permutes under the exponent of 1024 and one or
// two packed fp16 instructions per pair, about 1.5 VALU instructions per weight
// (5 for the fp32 dequantization of k_gemm).
#include <hip/hip_runtime.h>

#include "kernel_common.h"
#include "prefill.h"

namespace chonk {
namespace {

typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));

constexpr int kIK = 128;        // K per stage
constexpr int kIS = kIK + 8;    // LDS row stride in halves (bank spread)

__device__ __forceinline__ float4_t mfma32(half8_t a, half8_t b, float4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ half2_t as_half2(uint32_t v) { return __builtin_bit_cast(half2_t, v); }
__device__ __forceinline__ half2_t splat(float v) {
  const _Float16 h = (_Float16)v;
  return half2_t{h, h};
}
// bytes (0, 1) or (2, 3) of w under the exponent of 1024: 1024 + byte
__device__ __forceinline__ half2_t bytes01(uint32_t w) {
  return as_half2(__builtin_amdgcn_perm(0x64646464u, w, 0x04010400u));
}
__device__ __forceinline__ half2_t bytes23(uint32_t w) {
  return as_half2(__builtin_amdgcn_perm(0x64646464u, w, 0x04030402u));
}
// sixteen halves at dst (16-byte aligned)
__device__ __forceinline__ void put16(_Float16* dst, const half2_t (&v)[8]) {
  uint32_t u[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) u[i] = __builtin_bit_cast(uint32_t, v[i]);
  *(uint4*)dst = make_uint4(u[0], u[1], u[2], u[3]);
  *(uint4*)(dst + 8) = make_uint4(u[4], u[5], u[6], u[7]);
}

// The weight bytes of one thread and stage: NG groups of 32 weights.
template <int T, int NG>
struct Codes;
template <int NG>
struct Codes<QT_Q4_K, NG> {
  uint4 q[NG], hdr;
};
template <int NG>
struct Codes<QT_Q6_K, NG> {
  uint4 ql[NG], qh;
  uint2 sc;
  uint32_t d;
};
template <int NG>
struct Codes<QT_Q8_0, NG> {
  uint4 q[2 * NG];
  uint32_t d[NG];
};

template <int T>
constexpr int gemm_int_planes() { return T == QT_Q4_K ? 1 : 2; }
template <int T, int NI>
constexpr size_t gemm_int_shared() {
  return sizeof(_Float16) * gemm_int_planes<T>() * 16 * NI * kIS + (T == QT_Q4_K ? 16 * NI * 16 * sizeof(_Float16) : 0) +
         (T != QT_Q8_0 ? 16 * NI * sizeof(float) : 0);
}

// 16 NI weight rows x 64 TJ token rows per workgroup; wave w owns token rows
// 16 TJ w .. 16 TJ (w + 1) - 1 against all the weight rows and reads its
// activation operands straight from the planes (each element is read by one
// lane of one wave). At NI = 8, TJ = 2 a 32-k step of the workgroup is 16 KB
// through the vector cache and 32 KB of LDS reads under 512 cycles of MFMA,
// half of what either can move in that time; 64 weight rows would need the
// whole of the vector cache's rate. Codes of the next stage are in flight
// while this one is multiplied.
template <int T, int NI, int TJ>
__global__ __launch_bounds__(kWg, 2) void k_gemm_int(GemmArgs a) {
  extern __shared__ __align__(16) _Float16 gism[];
  constexpr int R = 16 * NI, NP = gemm_int_planes<T>(), NG = NI / 4;
  constexpr bool SB = T != QT_Q8_0;  // sums of a super-block are scaled by d
  _Float16* wp = gism;                                   // [NP][R][kIS]
  _Float16* cs = wp + NP * R * kIS;                      // Q4_K: [R][16], c of eight sub-blocks hi | lo
  float* ds = (float*)(cs + (T == QT_Q4_K ? R * 16 : 0));  // [R] d 2^(ws - 5) (Q6_K: d 2^ws)
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n0 = blockIdx.x * R, t0 = blockIdx.y * 64 * TJ;
  const int N = a.n_all ? a.n_all : a.w.n, K = a.w.k;
  // this workgroup's stages: part blockIdx.z of ksplit, whole super-blocks
  constexpr int SPB = SB ? 2 : 1;
  const int nsb = (K + SPB * kIK - 1) / (SPB * kIK);
  const int s_lo = SPB * (int)((int64_t)nsb * blockIdx.z / a.ksplit);
  const int s_hi = SPB * (int)((int64_t)nsb * (blockIdx.z + 1) / a.ksplit);
  const float wsc = ldexpf(1.0f, a.ws);

  // staging role: row wr, part wq of its 128 k (rows past N repeat the last row)
  constexpr int TPR = kWg / R;  // threads per row
  const int wr = tid / TPR, wq = tid % TPR;
  const int gr = min(n0 + wr, N - 1);
  const int seg = a.n_all ? (gr >= a.n2 ? 2 : (gr >= a.n1 ? 1 : 0)) : 0;
  const size_t row = gr - (seg == 2 ? a.n2 : (seg == 1 ? a.n1 : 0));
#define CHONK_PICK_S(f) (seg == 2 ? a.w3.f : (seg == 1 ? a.w2.f : a.w.f))
  const uint8_t *p0, *p1, *p2 = nullptr, *p3 = nullptr;
  if constexpr (T == QT_Q4_K) {
    p0 = CHONK_PICK_S(s0) + row * (K / 2) + 16 * NG * wq;
    p1 = CHONK_PICK_S(s1) + row * (K / 16);
  } else if constexpr (T == QT_Q6_K) {
    // NI = 8: part wq = l / 16 of every quarter; NI = 4: also one ql run of the two
    p0 = CHONK_PICK_S(s0) + row * (K / 2) + 16 * (wq & 1) + (NG == 1 ? 32 * (wq >> 1) : 0);
    p1 = CHONK_PICK_S(s1) + row * (K / 4) + 16 * (wq & 1);
    p2 = CHONK_PICK_S(s2) + row * (K / 16);
    p3 = CHONK_PICK_S(s3) + row * (K / 256) * 2;
  } else {
    p0 = CHONK_PICK_S(s0) + row * K;
    p1 = CHONK_PICK_S(s1) + row * (K / 32) * 2;
  }
#undef CHONK_PICK_S
  Codes<T, NG> f;
  auto fetch = [&](int s) {
    if constexpr (T == QT_Q4_K) {
#pragma unroll
      for (int g = 0; g < NG; ++g) f.q[g] = ldg4(p0 + 64 * s + 16 * g);
      f.hdr = ldg4(p1 + 16 * (s >> 1));
    } else if constexpr (T == QT_Q6_K) {
#pragma unroll
      for (int g = 0; g < NG; ++g) f.ql[g] = ldg4(p0 + 64 * s + 32 * g);
      f.qh = ldg4(p1 + 32 * s);
      f.sc = ldg2(p2 + 8 * s);
      f.d = ld_u16(p3 + 2 * (s >> 1));
    } else {
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        const int u = min(4 * s + NG * wq + g, (K >> 5) - 1);  // (the last stage may hold fewer units)
        f.q[2 * g] = ldg4(p0 + 32 * u);
        f.q[2 * g + 1] = ldg4(p0 + 32 * u + 16);
        f.d[g] = ld_u16(p1 + 2 * u);
      }
    }
  };
  auto stage = [&](int s) {
    _Float16* rh = wp + wr * kIS;
    _Float16* rl = rh + R * kIS;
    if constexpr (T == QT_Q4_K) {
      const float d = h2f(f.hdr.x) * wsc, dm = h2f(f.hdr.x >> 16) * wsc;
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        // bytes 16 p .. + 16 of sub-blocks 2 c, 2 c + 1 (low and high nibbles)
        const int gi = NG * wq + g, c = gi >> 1, p = gi & 1;
        const int j = 4 * (s & 1) + 2 * c;
        uint32_t sc[2], m[2];
        scale_min(j, f.hdr.y, f.hdr.z, f.hdr.w, &sc[0], &m[0]);
        scale_min(j + 1, f.hdr.y, f.hdr.z, f.hdr.w, &sc[1], &m[1]);
        const uint32_t w[4] = {f.q[g].x, f.q[g].y, f.q[g].z, f.q[g].w};
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          // (1024 + 16 q) sc / 16 - 72 sc = sc (q - 8): every step exact
          const half2_t k = splat((float)sc[h] * 0.0625f), z = splat((float)sc[h] * -72.0f);
          half2_t v[8];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const uint32_t b = (h ? w[i] : w[i] << 4) & 0xf0f0f0f0u;
            v[2 * i] = __builtin_elementwise_fma(bytes01(b), k, z);
            v[2 * i + 1] = __builtin_elementwise_fma(bytes23(b), k, z);
          }
          put16(rh + 64 * c + 32 * h + 16 * p, v);
        }
        if (p == 0) {
          _Float16* cr = cs + wr * 16 + j;
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const float cc = fmaf(8.0f * d, (float)sc[h], -(dm * (float)m[h]));
            const _Float16 ch = (_Float16)cc;
            cr[h] = ch;
            cr[8 + h] = (_Float16)(cc - (float)ch);
          }
        }
      }
      if (wq == 0) ds[wr] = d * 0.03125f;
    } else if constexpr (T == QT_Q6_K) {
      const int p = wq & 1;
      const uint32_t hw[4] = {f.qh.x, f.qh.y, f.qh.z, f.qh.w};
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        const int run = NG == 1 ? wq >> 1 : g;
        const uint32_t w[4] = {f.ql[g].x, f.ql[g].y, f.ql[g].z, f.ql[g].w};
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int q = run + 2 * h;  // quarter of the 128 k
          const int si = 2 * q + p;
          const uint32_t sw = h ? f.sc.y : f.sc.x;
          const half2_t sc = splat((float)(int8_t)((sw >> (8 * (si & 3))) & 0xffu));
          half2_t vh[8], vl[8];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const uint32_t b = ((w[i] >> (4 * h)) & 0x0f0f0f0fu) | (((hw[i] >> (2 * q)) & 0x03030303u) << 4);
            const half2_t x0 = bytes01(b) - half2_t{1056, 1056}, x1 = bytes23(b) - half2_t{1056, 1056};
            vh[2 * i] = x0 * sc;
            vh[2 * i + 1] = x1 * sc;
            vl[2 * i] = __builtin_elementwise_fma(x0, sc, -vh[2 * i]);
            vl[2 * i + 1] = __builtin_elementwise_fma(x1, sc, -vh[2 * i + 1]);
          }
          put16(rh + 32 * q + 16 * p, vh);
          put16(rl + 32 * q + 16 * p, vl);
        }
      }
      if (wq == 0) ds[wr] = h2f(f.d) * wsc;
    } else {
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        const int u = NG * wq + g;
        const half2_t d = splat(4 * s + u < (K >> 5) ? h2f(f.d[g]) * wsc : 0.f);
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          const uint4 q4 = f.q[2 * g + p];
          const uint32_t w[4] = {q4.x, q4.y, q4.z, q4.w};
          half2_t vh[8], vl[8];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const uint32_t b = w[i] ^ 0x80808080u;  // q + 128
            const half2_t x0 = bytes01(b) - half2_t{1152, 1152}, x1 = bytes23(b) - half2_t{1152, 1152};
            vh[2 * i] = x0 * d;
            vh[2 * i + 1] = x1 * d;
            vl[2 * i] = __builtin_elementwise_fma(x0, d, -vh[2 * i]);
            vl[2 * i + 1] = __builtin_elementwise_fma(x1, d, -vh[2 * i + 1]);
          }
          put16(rh + 32 * u + 16 * p, vh);
          put16(rl + 32 * u + 16 * p, vl);
        }
      }
    }
  };

  // operand role: lane l holds row (or token) l % 16 and k 8 (l / 16) .. + 8 of a
  // 32-k step; plane rows as 32-bit byte offsets from the planes' bases, a token
  // row past t reads row t - 1: its products are computed and dropped
  const int col = lane & 15, quad = lane >> 4;
  uint32_t xo[TJ], so[TJ];
#pragma unroll
  for (int j = 0; j < TJ; ++j) {
    const uint32_t t = min(t0 + 16 * (TJ * wave + j) + col, a.t - 1);
    xo[j] = 2u * (t * (uint32_t)a.kpad + 8u * quad);
    // sums of x: [t][hi | lo][kpad / 32]; quads 0, 1: hi, 2: lo (3: times zero)
    so[j] = 2u * (uint32_t)(a.kpad / 32) * (2 * t + (quad == 2 ? 1u : 0u));
  }
  const char* xhb = (const char*)a.xh;
  const char* xlb = (const char*)a.xl;
  const char* xsb = (const char*)a.xs;

  float4_t acc[NI][TJ], tmp[SB ? NI : 1][TJ];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j) acc[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};

  if (s_lo < s_hi) fetch(s_lo);
  for (int s = s_lo; s < s_hi; ++s) {
    // the stage's activation operands: the first steps' ahead of the staging,
    // the others' (when there is no register room for all) ahead of the products
    constexpr int EARLY = TJ == 2 ? 2 : kIK / 32;
    half8_t bh[kIK / 32][TJ], bl[kIK / 32][TJ];
    auto load_x = [&](int k0, int k1) {
#pragma unroll
      for (int ks = k0; ks < k1; ++ks)
#pragma unroll
        for (int j = 0; j < TJ; ++j) {
          const uint32_t o = xo[j] + 2u * (uint32_t)(s * kIK + ks * 32);
          bh[ks][j] = *(const half8_t*)(xhb + o);
          bl[ks][j] = *(const half8_t*)(xlb + o);
        }
    };
    load_x(0, EARLY);
    half8_t xb[TJ];
    if constexpr (T == QT_Q4_K) {
#pragma unroll
      for (int j = 0; j < TJ; ++j) xb[j] = *(const half8_t*)(xsb + so[j] + 16u * (uint32_t)(s >> 1));
    }
    lds_barrier();  // the previous stage's tile is consumed
    stage(s);
    fetch(min(s + 1, s_hi - 1));
    lds_barrier();  // (the codes and operands in flight are not waited for)
    load_x(EARLY, kIK / 32);
    if constexpr (SB) {
      if (!(s & 1)) {
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
          for (int j = 0; j < TJ; ++j) tmp[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};
      }
    }
#pragma unroll
    for (int ks = 0; ks < kIK / 32; ++ks)
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        auto& dst = [&]() -> auto& {
          if constexpr (SB)
            return tmp[i];
          else
            return acc[i];
        }();
        const _Float16* ar = wp + (16 * i + col) * kIS + ks * 32 + 8 * quad;
        const half8_t ah = *(const half8_t*)ar;
#pragma unroll
        for (int j = 0; j < TJ; ++j) dst[j] = mfma32(ah, bh[ks][j], dst[j]);
#pragma unroll
        for (int j = 0; j < TJ; ++j) dst[j] = mfma32(ah, bl[ks][j], dst[j]);
        if constexpr (NP == 2) {
          const half8_t al = *(const half8_t*)(ar + R * kIS);
#pragma unroll
          for (int j = 0; j < TJ; ++j) dst[j] = mfma32(al, bh[ks][j], dst[j]);
        }
      }
    if constexpr (SB) {
      if (s & 1) {
        // the super-block's sums times d, and (Q4_K) its c times the sums of x:
        // k 0..7 c_hi Xh, 8..15 c_lo Xh, 16..23 c_hi Xl, 24..31 nothing
#pragma unroll
        for (int i = 0; i < NI; ++i) {
          const float4_t d4 = *(const float4_t*)(ds + 16 * i + 4 * quad);
          if constexpr (T == QT_Q4_K) {
            half8_t ca = *(const half8_t*)(cs + (16 * i + col) * 16 + (quad == 1 ? 8 : 0));
            if (quad == 3) ca = half8_t{0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
            for (int j = 0; j < TJ; ++j) acc[i][j] = mfma32(ca, xb[j], acc[i][j]);
          }
#pragma unroll
          for (int j = 0; j < TJ; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) acc[i][j][q] = fmaf(d4[q], tmp[i][j][q], acc[i][j][q]);
        }
      }
    }
  }
  // lane holds rows 4 quad + 0..3 of each 16-row tile, token col
  const float wun = ldexpf(1.0f, (T == QT_Q4_K ? 5 : 0) - a.ws);
  const bool part = a.ksplit > 1 || a.defer;
  const bool vec = part && (N & 3) == 0 && ((uintptr_t)a.part & 15) == 0;
#pragma unroll
  for (int j = 0; j < TJ; ++j) {
    const int tt = t0 + 16 * (TJ * wave + j) + col;
    if (tt >= a.t) continue;
    const float sc = wun * a.xscale[tt];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int n = n0 + 16 * i + 4 * quad;
      float* pp = a.part + ((size_t)blockIdx.z * a.t + tt) * N + n;
      if (vec && n + 4 <= N) {
        *(float4*)pp = make_float4(acc[i][j][0] * sc, acc[i][j][1] * sc, acc[i][j][2] * sc, acc[i][j][3] * sc);
        continue;
      }
      float* y = a.y + (size_t)tt * a.ldy + n;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        if (n + q >= N) break;
        const float v = acc[i][j][q] * sc;
        if (part)
          pp[q] = v;
        else
          y[q] = a.epi == GEMM_ADD ? __fadd_rn(y[q], v) : v;
      }
    }
  }
}

template <int T, int NI, int TJ>
hipError_t launch_one(const GemmArgs& a, int n_rows, hipStream_t s) {
  const dim3 grid((n_rows + 16 * NI - 1) / (16 * NI), (a.t + 64 * TJ - 1) / (64 * TJ), a.ksplit);
  hipLaunchKernelGGL((k_gemm_int<T, NI, TJ>), grid, dim3(kWg), (gemm_int_shared<T, NI>()), s, a);
  return hipGetLastError();
}

template <int T>
hipError_t launch_type(const GemmArgs& a, int n_rows, int ni, int tj, hipStream_t s) {
  if (ni == 8) return tj == 2 ? launch_one<T, 8, 2>(a, n_rows, s) : launch_one<T, 8, 1>(a, n_rows, s);
  return tj == 2 ? launch_one<T, 4, 2>(a, n_rows, s) : launch_one<T, 4, 1>(a, n_rows, s);
}

template <int T>
hipError_t init_type() {
  const std::pair<const void*, size_t> f[4] = {{(const void*)k_gemm_int<T, 8, 2>, gemm_int_shared<T, 8>()},
                                               {(const void*)k_gemm_int<T, 8, 1>, gemm_int_shared<T, 8>()},
                                               {(const void*)k_gemm_int<T, 4, 2>, gemm_int_shared<T, 4>()},
                                               {(const void*)k_gemm_int<T, 4, 1>, gemm_int_shared<T, 4>()}};
  for (const auto& p : f) {
    const hipError_t e = hipFuncSetAttribute(p.first, hipFuncAttributeMaxDynamicSharedMemorySize, (int)p.second);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace

bool gemm_int_type(int type) { return type == QT_Q4_K || type == QT_Q6_K || type == QT_Q8_0; }

hipError_t launch_gemm_int(const GemmArgs& a, int n_rows, int ni, int tj, hipStream_t s) {
  if (a.w.type == QT_Q4_K && (!a.xs || a.w.k % 256 != 0)) return hipErrorInvalidValue;
  if (a.w.type == QT_Q6_K && a.w.k % 256 != 0) return hipErrorInvalidValue;
  switch (a.w.type) {
    case QT_Q4_K: return launch_type<QT_Q4_K>(a, n_rows, ni, tj, s);
    case QT_Q6_K: return launch_type<QT_Q6_K>(a, n_rows, ni, tj, s);
    case QT_Q8_0: return launch_type<QT_Q8_0>(a, n_rows, ni, tj, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t init_gemm_int_attributes() {
  for (hipError_t e : {init_type<QT_Q4_K>(), init_type<QT_Q6_K>(), init_type<QT_Q8_0>()})
    if (e != hipSuccess) return e;
  return hipSuccess;
}

}  // namespace chonk
