// Prompt GEMM over the weights' integer codes, gfx950.
//
//   Q4_K, Q5_K  W = d (sc (q - z)) + c,   z = 8, 16,  c = z d sc - dmin m per 32 k
//   Q6_K        W = d (sc (q - 32))
//   Q8_0, Q5_0  W = d q,  d (q - 16) per 32 k
//   Q5_1        W = d q + m, formed in fp32
//
// sc (q - z) of Q4_K and Q5_K is an integer below 2^10, exact in one fp16 plane, so
// the matrix cores multiply it with the hi and lo activation planes (two products
// per 16x16x32 step where fp16 hi + lo weights take three, and no rounded
// weight): the sums of a 256-k super-block are scaled by d once, and c, which
// is constant over 32 k, meets the sums of x over those 32 k in one more MFMA
// per super-block. The codes of Q8_0 and Q5_0 are exact in one plane too; their d
// changes every 32 k, which is one 16x16x32 step: its two products start from
// zero and join the sums of 256 k by one fma with d. sc (q - 32) of Q6_K has 13
// bits and Q5_1's d q + m more, so these keep two planes, split exactly (h =
// fp16(v), l = v - h). Codes become fp16 by byte permutes under the exponent of
// 1024 and one or two packed fp16 instructions per pair, about 1.5 VALU
// instructions per weight.
//
// Chains are kept short: the matrix core rounds several times per step at the
// size of what it adds to. Q8_0 as two planes in one chain over K was 1.6e-7 to
// 3.6e-7 from float64 (8.4e-8 to 9.6e-8 now; 9216 x 1024 at 300 rows 32.7 -> 29.2 us,
// 3376 x 768 at 2047 49.3 -> 48.3, 1024 x 1024 at 200 13.7 -> 13.7), and the logits
// after a Granite or LFM2 Q8_0 prompt (fp32 cache) 1.4e-6 or 2.6e-6, where a prompt
// in decode steps leaves 8.5e-7 or 1.53e-6 (8.5e-7 and 1.53e-6 now).
//
// Against the three-product GEMM over fp32-dequantized hi + lo weights that it
// replaced (MI355X, 2047 token rows): Q4_K 4096 x 1024 95.0 -> 47.9 us, 6144 x 1024
// 139.5 -> 65.2, Q6_K 1024 x 3072 90.6 -> 41.2; error against float64 3.6e-7 -> 1.4e-7
// (Q4_K), 6.2e-7 -> 1.7e-7 (Q6_K). What is left (6144 x 1024, gate * up, 60.4 us): the
// matrix cores are busy 46% of the CUs' busy cycles and LDS 39%, the rest are the
// stages' conversions and barriers.
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
// Orders the LDS accesses of a wave's lanes before and after it. The hardware keeps
// them in order; this keeps the compiler from moving them.
__device__ __forceinline__ void wave_lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
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
struct Codes<QT_Q5_K, NG> {
  uint4 q[NG], qh[NG], hdr;
};
template <int NG>
struct Codes<QT_Q5_0, NG> {
  uint4 q[NG];
  uint32_t qh[NG], d[NG];
};
template <int NG>
struct Codes<QT_Q5_1, NG> {
  Frag<QT_Q5_1> f[NG];
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

// sums of a super-block are scaled by d; block offsets c
template <int T>
constexpr bool gemm_int_sb = T == QT_Q4_K || T == QT_Q5_K || T == QT_Q6_K;
template <int T>
constexpr bool gemm_int_offsets = T == QT_Q4_K || T == QT_Q5_K;
// codes alone in the plane, the sums of a 32-weight block scaled by its d
template <int T>
constexpr bool gemm_int_blocks = T == QT_Q8_0 || T == QT_Q5_0;
template <int T>
constexpr int gemm_int_planes() { return gemm_int_offsets<T> || gemm_int_blocks<T> ? 1 : 2; }
template <int T, int NI>
constexpr size_t gemm_int_shared() {
  return sizeof(_Float16) * gemm_int_planes<T>() * 16 * NI * kIS + (gemm_int_offsets<T> ? 16 * NI * 16 * sizeof(_Float16) : 0) +
         (gemm_int_sb<T> ? 16 * NI * sizeof(float) : 0) + (gemm_int_blocks<T> ? 4 * 16 * NI * sizeof(float) : 0);
}

// 16 NI weight rows x 64 TJ token rows per workgroup; wave w owns token rows
// 16 TJ w .. 16 TJ (w + 1) - 1 against all the weight rows and reads its
// activation operands straight from the planes (each element is read by one
// lane of one wave). At NI = 8, TJ = 2 a 32-k step of the workgroup is 16 KB
// through the vector cache and 32 KB of LDS reads under 512 cycles of MFMA,
// half of what either can move in that time; 64 weight rows would need the
// whole of the vector cache's rate. Codes of the next stage are in flight
// while this one is multiplied, weight fragments are read from LDS three ahead
// of their products, and the results leave through LDS as whole runs of a row
// (64-byte pieces of 16 rows at a time cost 15 us more at 4096 x 1024 x 2047).
// GLU: the first half of the weight rows are gate rows (a.w), the second the same
// rows of up (a.w2).
// (BLK at NI = 4: at most 168 registers, three workgroups per CU; with 198 the 9216 x
// 1024 launch at 300 rows takes 36.5 us instead of 29.9)
template <int T, int NI, int TJ, bool GLU>
__global__ __launch_bounds__(kWg, (gemm_int_blocks<T> && NI == 4 ? 3 : 2)) void k_gemm_int(GemmArgs a) {
  extern __shared__ __align__(16) _Float16 gism[];
  constexpr int R = 16 * NI, NP = gemm_int_planes<T>(), NG = NI / 4;
  constexpr bool SB = gemm_int_sb<T>, OFF = gemm_int_offsets<T>, BLK = gemm_int_blocks<T>;
  _Float16* wp = gism;                                   // [NP][R][kIS]
  _Float16* cs = wp + NP * R * kIS;                      // OFF: [R][16], c of eight sub-blocks hi | lo
  float* ds = (float*)(cs + (OFF ? R * 16 : 0));  // [R] d 2^(ws - 5) (Q6_K: d 2^ws; BLK: [4][R], the stage's blocks)
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
  const int gr = GLU ? min((int)blockIdx.x * (R / 2) + wr % (R / 2), a.n1 - 1) : min(n0 + wr, N - 1);
  const int seg = GLU ? wr / (R / 2) : a.n_all ? (gr >= a.n2 ? 2 : (gr >= a.n1 ? 1 : 0)) : 0;
  const size_t row = GLU ? gr : gr - (seg == 2 ? a.n2 : (seg == 1 ? a.n1 : 0));
#define CHONK_PICK_S(f) (seg == 2 ? a.w3.f : (seg == 1 ? a.w2.f : a.w.f))
  const uint8_t *p0, *p1, *p2 = nullptr, *p3 = nullptr;
  if constexpr (OFF) {
    p0 = CHONK_PICK_S(s0) + row * (K / 2) + 16 * NG * wq;
    p1 = CHONK_PICK_S(s1) + row * (K / 16);
    if constexpr (T == QT_Q5_K) p2 = CHONK_PICK_S(s2) + row * (K / 8) + (NG == 1 ? 16 * (wq & 1) : 0);
  } else if constexpr (T == QT_Q6_K) {
    // NI = 8: part wq = l / 16 of every quarter; NI = 4: also one ql run of the two
    p0 = CHONK_PICK_S(s0) + row * (K / 2) + 16 * (wq & 1) + (NG == 1 ? 32 * (wq >> 1) : 0);
    p1 = CHONK_PICK_S(s1) + row * (K / 4) + 16 * (wq & 1);
    p2 = CHONK_PICK_S(s2) + row * (K / 16);
    p3 = CHONK_PICK_S(s3) + row * (K / 256) * 2;
  } else if constexpr (T == QT_Q8_0) {
    p0 = CHONK_PICK_S(s0) + row * K;
    p1 = CHONK_PICK_S(s1) + row * (K / 32) * 2;
  } else {
    p0 = CHONK_PICK_S(s0) + row * (K / 2);
    p1 = CHONK_PICK_S(s1) + row * (K / 32) * 4;
    p2 = CHONK_PICK_S(s2) + row * (K / 32) * 2;
    if constexpr (T == QT_Q5_1) p3 = CHONK_PICK_S(s3) + row * (K / 32) * 2;
  }
#undef CHONK_PICK_S
  Codes<T, NG> f;
  auto fetch = [&](int s) {
    if constexpr (OFF) {
#pragma unroll
      for (int g = 0; g < NG; ++g) f.q[g] = ldg4(p0 + 64 * s + 16 * g);
      if constexpr (T == QT_Q5_K) {
#pragma unroll
        for (int g = 0; g < NG; ++g) f.qh[g] = ldg4(p2 + 32 * (s >> 1) + 16 * g);
      }
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
        if constexpr (T == QT_Q8_0) {
          f.q[2 * g] = ldg4(p0 + 32 * u);
          f.q[2 * g + 1] = ldg4(p0 + 32 * u + 16);
          f.d[g] = ld_u16(p1 + 2 * u);
        } else if constexpr (T == QT_Q5_0) {
          f.q[g] = ldg4(p0 + 16 * u);
          f.qh[g] = ldg1(p1 + 4 * u);
          f.d[g] = ld_u16(p2 + 2 * u);
        } else {
          f.f[g].qs = ldg4(p0 + 16 * u);
          f.f[g].qh = ldg1(p1 + 4 * u);
          f.f[g].d = ld_u16(p2 + 2 * u);
          f.f[g].m = ld_u16(p3 + 2 * u);
        }
      }
    }
  };
  auto stage = [&]<int PAR>(int s) {
    _Float16* rh = wp + wr * kIS;
    _Float16* rl = rh + R * kIS;
    if constexpr (OFF) {
      const float d = h2f(f.hdr.x) * wsc, dm = h2f(f.hdr.x >> 16) * wsc;
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        // bytes 16 p .. + 16 of sub-blocks 2 c, 2 c + 1 (low and high nibbles)
        const int gi = NG * wq + g, c = gi >> 1, p = gi & 1;
        const int j = 4 * PAR + 2 * c;
        uint32_t sc[2], m[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          // scale_min of sub-block j + h, in the half known here (bytes j, j + 4, j + 8 of the 12)
          const int b = 8 * (2 * c + h);
          if constexpr (PAR == 0) {
            sc[h] = (f.hdr.y >> b) & 63u;
            m[h] = (f.hdr.z >> b) & 63u;
          } else {
            const uint32_t lo = f.hdr.w >> b;
            sc[h] = (lo & 15u) | (((f.hdr.y >> b) >> 2) & 48u);
            m[h] = ((lo >> 4) & 15u) | (((f.hdr.z >> b) >> 2) & 48u);
          }
        }
        const uint32_t w[4] = {f.q[g].x, f.q[g].y, f.q[g].z, f.q[g].w};
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          half2_t v[8];
          if constexpr (T == QT_Q4_K) {
            // (1024 + 16 q) sc / 16 - 72 sc = sc (q - 8): every step exact
            const half2_t k = splat((float)sc[h] * 0.0625f), z = splat((float)sc[h] * -72.0f);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const uint32_t b = (h ? w[i] : w[i] << 4) & 0xf0f0f0f0u;
              v[2 * i] = __builtin_elementwise_fma(bytes01(b), k, z);
              v[2 * i + 1] = __builtin_elementwise_fma(bytes23(b), k, z);
            }
          } else {
            const half2_t k = splat((float)sc[h]);
            const uint32_t hw[4] = {f.qh[g].x, f.qh[g].y, f.qh[g].z, f.qh[g].w};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const uint32_t b = ((w[i] >> (4 * h)) & 0x0f0f0f0fu) | (((hw[i] >> (j + h)) & 0x01010101u) << 4);
              v[2 * i] = (bytes01(b) - half2_t{1040, 1040}) * k;
              v[2 * i + 1] = (bytes23(b) - half2_t{1040, 1040}) * k;
            }
          }
          put16(rh + 64 * c + 32 * h + 16 * p, v);
        }
        if (p == 0) {
          _Float16* cr = cs + wr * 16 + j;
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const float cc = fmaf((T == QT_Q4_K ? 8.0f : 16.0f) * d, (float)sc[h], -(dm * (float)m[h]));
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
    } else if constexpr (T == QT_Q5_1) {
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        const int u = NG * wq + g;
        float v[32];
        dequant_unit<QT_Q5_1>(f.f[g], 4 * s + u, v, 4 * s + u < (K >> 5) ? wsc : 0.f);
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          half2_t vh[8], vl[8];
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            vh[i / 2][i % 2] = (_Float16)v[16 * p + i];
            vl[i / 2][i % 2] = (_Float16)(v[16 * p + i] - (float)vh[i / 2][i % 2]);
          }
          put16(rh + 32 * u + 16 * p, vh);
          put16(rl + 32 * u + 16 * p, vl);
        }
      }
    } else {
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        const int u = NG * wq + g;
        // (odd blocks with both signs turned: the matrix core rounds down on average, and
        // with one sign the products were all low by up to 4e-8 of their rms, in every row alike)
        const float sg = u & 1 ? -1.0f : 1.0f;
        ds[u * R + wr] = 4 * s + u < (K >> 5) ? sg * (h2f(f.d[g]) * wsc) : 0.f;
        const half2_t one = splat(sg), z = splat(sg * (T == QT_Q8_0 ? -1152.0f : -1040.0f));
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          const uint4 q4 = f.q[T == QT_Q8_0 ? 2 * g + p : g];
          const uint32_t w[4] = {q4.x, q4.y, q4.z, q4.w};
          half2_t v[8];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            uint32_t b;
            if constexpr (T == QT_Q8_0) {
              b = w[i] ^ 0x80808080u;  // q + 128
            } else {
              // element 16 p + 4 i + e: nibble p of byte 4 i + e, bit of qh under bit 4 of byte e
              const uint32_t x = (f.qh[g] >> (16 * p + 4 * i)) & 15u;
              b = ((w[i] >> (4 * p)) & 0x0f0f0f0fu) | (((x | x << 7 | x << 14 | x << 21) & 0x01010101u) << 4);
            }
            v[2 * i] = __builtin_elementwise_fma(bytes01(b), one, z);
            v[2 * i + 1] = __builtin_elementwise_fma(bytes23(b), one, z);
          }
          put16(rh + 32 * u + 16 * p, v);
        }
      }
    }
  };

  // operand role: lane l holds row (or token) l % 16 and k 8 (l / 16) .. + 8 of a
  // 32-k step; the lane's pieces as 32-bit byte offsets from the planes' bases, a
  // row tile past the last one reads that: its products are computed and dropped
  const int col = lane & 15, quad = lane >> 4;
  uint32_t xo[TJ], so[TJ];
#pragma unroll
  for (int j = 0; j < TJ; ++j) {
    const uint32_t t = min(t0 + 16 * (TJ * wave + j) + col, a.t - 1);
    xo[j] = 2u * (uint32_t)plane_at(16 * min((t0 + 16 * (TJ * wave + j)) / 16, (a.t - 1) / 16), 0, a.kpad) + 16u * lane;
    // sums of x: [t][hi | lo][kpad / 32]; quads 0, 1: hi, 2: lo (3: times zero)
    so[j] = 2u * (uint32_t)(a.kpad / 32) * (2 * t + (quad == 2 ? 1u : 0u));
  }
  const char* xhb = (const char*)a.xh;
  const char* xlb = (const char*)a.xl;
  const char* xsb = (const char*)a.xs;

  // (tmp: the sums of 256 k; see the merge below)
  float4_t acc[NI][TJ], tmp[NI][TJ];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j) acc[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};

  // The activation operands of 32-k step st sit in slot st % NS, requested LA
  // steps ahead of their use (the last steps request the last one again).
  constexpr int SPS = kIK / 32, NS = TJ == 2 ? 4 : 8, LA = TJ == 2 ? 2 : 6;
  const int st_hi = SPS * s_hi - 1;
  half8_t bh[NS][TJ], bl[NS][TJ];
  auto load_x = [&](int st, int slot) {
#pragma unroll
    for (int j = 0; j < TJ; ++j) {
      const uint32_t o = xo[j] + 1024u * (uint32_t)min(st, st_hi);
      bh[slot][j] = *(const half8_t*)(xhb + o);
      bl[slot][j] = *(const half8_t*)(xlb + o);
    }
  };
  // one stage; PAR: its parity from s_lo on (for super-block types its half)
  auto body = [&]<int PAR>(int s) {
    half8_t xb[TJ];
    if constexpr (OFF && PAR == 1) {
#pragma unroll
      for (int j = 0; j < TJ; ++j) xb[j] = *(const half8_t*)(xsb + so[j] + 16u * (uint32_t)(s >> 1));
    }
    lds_barrier();  // the previous stage's tile is consumed
    stage.template operator()<PAR>(s);
    fetch(min(s + 1, s_hi - 1));
    lds_barrier();  // (the codes and operands in flight are not waited for)
    // the products: weight fragment f is plane f % NP of row tile f / NP % NI and
    // 32-k step f / NP / NI; AD fragments are read from LDS ahead of their use
    // (left alone, the compiler reads one at a time and waits for it)
    constexpr int NF = SPS * NI * NP, AD = BLK && TJ == 2 ? 1 : 3;
    auto frag = [&](int fi) {
      const int p = fi % NP, i = fi / NP % NI, ks = fi / NP / NI;
      return *(const half8_t*)(wp + p * R * kIS + (16 * i + col) * kIS + ks * 32 + 8 * quad);
    };
    half8_t af[AD + 1];
    // BLK: the products of a fragment and their blocks' scales, which join tmp
    // while the next fragment's products are issued
    float4_t us[3][TJ], dv[AD + 1];
    auto scale = [&](int fi) { return *(const float4_t*)(ds + (fi / NI) * R + 16 * (fi % NI) + 4 * quad); };
    auto join = [&](int fi) {
      const int i = fi % NI;
#pragma unroll
      for (int j = 0; j < TJ; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float d = dv[fi % (AD + 1)][q], u = us[fi % 3][j][q];
          tmp[i][j][q] = PAR == 0 && fi < NI ? d * u : fmaf(d, u, tmp[i][j][q]);
        }
    };
    // (the small products first; with one token tile those of the fragment ahead
    // stand between them and the large ones, which add to their result)
    auto small = [&](int fi) {
#pragma unroll
      for (int j = 0; j < TJ; ++j)
        us[fi % 3][j] = mfma32(af[fi % (AD + 1)], bl[(SPS * PAR + fi / NI) % NS][j], float4_t{0.f, 0.f, 0.f, 0.f});
    };
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int fi = 0; fi < AD; ++fi) {
      af[fi] = frag(fi);
      if constexpr (BLK) dv[fi] = scale(fi);
    }
#pragma unroll
    for (int fi = 0; fi < NF; ++fi) {
      const int p = fi % NP, i = fi / NP % NI, ks = fi / NP / NI, sl = (SPS * PAR + ks) % NS;
      if constexpr (BLK) {
        if (fi > 0) join(fi - 1);
        if (fi + AD < NF) dv[(fi + AD) % (AD + 1)] = scale(fi + AD);
      }
      if (fi + AD < NF) af[(fi + AD) % (AD + 1)] = frag(fi + AD);
      if (p == 0 && i == 0) load_x(SPS * s + ks + LA, (SPS * PAR + ks + LA) % NS);
      const half8_t w = af[fi % (AD + 1)];
      if constexpr (BLK) {
        if (TJ == 2 || fi == 0) small(fi);
        if (TJ == 1 && fi + 1 < NF) small(fi + 1);
#pragma unroll
        for (int j = 0; j < TJ; ++j) us[fi % 3][j] = mfma32(w, bh[sl][j], us[fi % 3][j]);
        continue;
      }
      const bool first = (!SB || PAR == 0) && ks == 0 && p == 0;
#pragma unroll
      for (int j = 0; j < TJ; ++j) tmp[i][j] = mfma32(w, bh[sl][j], first ? float4_t{0.f, 0.f, 0.f, 0.f} : tmp[i][j]);
      if (p == 0) {
#pragma unroll
        for (int j = 0; j < TJ; ++j) tmp[i][j] = mfma32(w, bl[sl][j], tmp[i][j]);
      }
    }
    if constexpr (BLK) join(NF - 1);
    // (schedule: AD LDS reads, then per fragment one read and its products; BLK:
    // two reads, the products and, with two token tiles, the fused multiplies of the
    // fragment before. With one they find their own place: 3 rows of the LFM2.5-350M
    // Q8_0 shape take 0.90 ms, 0.945 with a group for them)
    __builtin_amdgcn_sched_group_barrier(0x100, BLK ? 2 * AD : AD, 0);
#pragma unroll
    for (int fi = 0; fi < NF; fi += NP) {
      if (fi % (NP * NI) == 0) __builtin_amdgcn_sched_group_barrier(0x20, 2 * TJ, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, BLK ? 2 : 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x8, 2 * TJ, 0);
      if constexpr (BLK && TJ == 2) __builtin_amdgcn_sched_group_barrier(0x2, 4 * TJ, 0);
      if constexpr (NP == 2) {
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x8, TJ, 0);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (SB && PAR == 1) {
      // the super-block's sums times d, and its c times the sums of x:
      // k 0..7 c_hi Xh, 8..15 c_lo Xh, 16..23 c_hi Xl, 24..31 nothing
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const float4_t d4 = *(const float4_t*)(ds + 16 * i + 4 * quad);
        if constexpr (OFF) {
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
    if constexpr (!SB) {
      // The sums of 256 k (Q5_1: of 128, which are longer chains) join the total in one addition.
      if (!BLK || PAR == 1 || s + 1 >= s_hi) {
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
          for (int j = 0; j < TJ; ++j) acc[i][j] += tmp[i][j];
      }
    }
  };
  if (s_lo < s_hi) {
#pragma unroll
    for (int st = 0; st < LA; ++st) load_x(SPS * s_lo + st, st);
    fetch(s_lo);
  }
  for (int s = s_lo; s < s_hi; s += 2) {
    body.template operator()<0>(s);
    if (SB || s + 1 < s_hi) body.template operator()<1>(s + 1);
  }
  // The lane holds rows 4 quad + 0..3 of each 16-row tile, token col. Each wave
  // turns its 16-token tiles over in LDS, so that a store instruction writes
  // whole runs of a token's row (512 bytes at NI = 8); the GLU launch stores
  // silu(gate) * up (or GELU) of its two halves instead of both.
  constexpr int RO = GLU ? R / 2 : R, NO = GLU ? NI / 2 : NI;  // columns and row tiles stored
  constexpr int OS = RO + 4, LPT = RO / 4;                     // LDS stride; lanes per token row
  const int ncols = GLU ? a.n1 : N, c0 = (int)blockIdx.x * RO;
  const float wun = ldexpf(1.0f, (OFF ? 5 : 0) - a.ws);
  const bool part = a.ksplit > 1 || a.defer;
  const bool vec = part && (ncols & 3) == 0 && ((uintptr_t)a.part & 15) == 0;
  __syncthreads();  // the last stage's tile is consumed
  float* tile = (float*)gism + wave * 16 * OS;
#pragma unroll
  for (int j = 0; j < TJ; ++j) {
    const int tt0 = t0 + 16 * (TJ * wave + j);
    const float sc = wun * a.xscale[min(tt0 + col, a.t - 1)];
#pragma unroll
    for (int i = 0; i < NO; ++i) {
      float4_t v = acc[i][j] * sc;
      if constexpr (GLU) {
        const float4_t u = acc[i + NO][j] * sc;
#pragma unroll
        for (int q = 0; q < 4; ++q)
          v[q] = a.epi == GEMM_GEGLU ? __fmul_rn(gelu_tanh(v[q]), u[q]) : silu_mul(v[q], u[q]);
      }
      *(float4_t*)(tile + col * OS + 16 * i + 4 * quad) = v;
    }
    wave_lds_order();  // the lanes read what other lanes wrote
#pragma unroll
    for (int r = 0; r < 16; r += 64 / LPT) {
      const int tr = r + lane / LPT, cc = 4 * (lane % LPT), tt = tt0 + tr, n = c0 + cc;
      const float4_t v = *(const float4_t*)(tile + tr * OS + cc);
      if (tt >= a.t || n >= ncols) continue;
      float* pp = a.part + ((size_t)blockIdx.z * a.t + tt) * ncols + n;
      if (vec) {
        *(float4_t*)pp = v;
        continue;
      }
      float* y = a.y + (size_t)tt * a.ldy + n;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        if (n + q >= ncols) break;
        if (part)
          pp[q] = v[q];
        else
          y[q] = a.epi == GEMM_ADD ? __fadd_rn(y[q], v[q]) : v[q];
      }
    }
    wave_lds_order();  // the next token tile overwrites them
  }
}

template <int T, int NI, int TJ, bool GLU>
hipError_t launch_one(const GemmArgs& a, int n_rows, hipStream_t s) {
  const dim3 grid((n_rows + 16 * NI - 1) / (16 * NI), (a.t + 64 * TJ - 1) / (64 * TJ), a.ksplit);
  hipLaunchKernelGGL((k_gemm_int<T, NI, TJ, GLU>), grid, dim3(kWg), (gemm_int_shared<T, NI>()), s, a);
  return hipGetLastError();
}

template <int T>
hipError_t launch_type(const GemmArgs& a, int n_rows, int ni, int tj, hipStream_t s) {
  const bool glu = a.epi == GEMM_SWIGLU || a.epi == GEMM_GEGLU;
  if (ni == 8 && tj == 2) return glu ? launch_one<T, 8, 2, true>(a, n_rows, s) : launch_one<T, 8, 2, false>(a, n_rows, s);
  if (ni == 4 && tj == 1) return glu ? launch_one<T, 4, 1, true>(a, n_rows, s) : launch_one<T, 4, 1, false>(a, n_rows, s);
  return ni == 4 && tj == 2 && !glu ? launch_one<T, 4, 2, false>(a, n_rows, s) : hipErrorInvalidValue;
}

template <int T, int NI, int TJ, bool GLU>
hipError_t init_one() {
  return hipFuncSetAttribute((const void*)k_gemm_int<T, NI, TJ, GLU>, hipFuncAttributeMaxDynamicSharedMemorySize,
                             (int)gemm_int_shared<T, NI>());
}
template <int T>
hipError_t init_type() {
  for (hipError_t e : {init_one<T, 8, 2, false>(), init_one<T, 4, 2, false>(), init_one<T, 4, 1, false>(),
                       init_one<T, 8, 2, true>(), init_one<T, 4, 1, true>()})
    if (e != hipSuccess) return e;
  return hipSuccess;
}

}  // namespace

bool gemm_int_sums(int type) { return type == QT_Q4_K || type == QT_Q5_K; }

hipError_t launch_gemm_int(const GemmArgs& a, int n_rows, int ni, int tj, hipStream_t s) {
  if (gemm_int_sums(a.w.type) && !a.xs) return hipErrorInvalidValue;
  if (gemm_int_step(a.w.type) == 256 && a.w.k % 256 != 0) return hipErrorInvalidValue;
  if ((a.epi == GEMM_SWIGLU || a.epi == GEMM_GEGLU) &&
      (a.ksplit != 1 || !a.defer || a.n2 != 2 * a.n1 || n_rows != a.n2 || a.w.n != a.n1 || a.w2.n != a.n1))
    return hipErrorInvalidValue;
  switch (a.w.type) {
    case QT_Q4_K: return launch_type<QT_Q4_K>(a, n_rows, ni, tj, s);
    case QT_Q5_K: return launch_type<QT_Q5_K>(a, n_rows, ni, tj, s);
    case QT_Q6_K: return launch_type<QT_Q6_K>(a, n_rows, ni, tj, s);
    case QT_Q8_0: return launch_type<QT_Q8_0>(a, n_rows, ni, tj, s);
    case QT_Q5_0: return launch_type<QT_Q5_0>(a, n_rows, ni, tj, s);
    case QT_Q5_1: return launch_type<QT_Q5_1>(a, n_rows, ni, tj, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t init_gemm_int_attributes() {
  for (hipError_t e : {init_type<QT_Q4_K>(), init_type<QT_Q5_K>(), init_type<QT_Q6_K>(), init_type<QT_Q8_0>(),
                       init_type<QT_Q5_0>(), init_type<QT_Q5_1>()})
    if (e != hipSuccess) return e;
  return hipSuccess;
}

}  // namespace chonk
