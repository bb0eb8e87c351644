// ConvRot (int8_rot) quantizers: the activation or weight row is rotated by blockdiag(H256) before the
// per-row INT8 quantization, H256 = the 4x4 regular Hadamard [[1,1,1,-1],[1,1,-1,1],[1,-1,1,1],[-1,1,1,1]]
// to the 4th Kronecker power, normalized (triton_fp8.py:70-90).
//
// Activations (triton_fp8.py:102-116, :218-233, :277-351): per 256-column group the prologue values v
// (fp32, same arithmetic as quant.hip) are rounded to bf16 and split into four 64-column chunks X_k;
// Z_k = X_k H64^T (H64 normalized, entries +-1/8) is the fp32 rounding of the exact dot products (the
// reference takes it from a bf16 tensor-core dot with fp32 accumulation, whose summation order is not
// specified; here every product is exact and the 64-term sums are formed exactly in float64, then rounded
// once); the four chunks are combined in fp32 in the reference's order
//   y0 = ((z0 + z1) + z2 - z3) * 0.5,  y1 = ((z0 + z1) - z2 + z3) * 0.5,
//   y2 = ((z0 - z1) + z2 + z3) * 0.5,  y3 = ((z1 + z2) + z3 - z0) * 0.5;
// then s = max(amax / 127, 1e-12), q = rint(clamp(y * (1 / s), -127, 127)).
//
// Weights (kernels.py:52-72, quantize_weight mode int8_rot): w @ blockdiag(H256)^T as the fp32 rounding of
// the exact product (float64 butterflies), then the int8_rowwise quantizer q = rint(w_rot / s).
//
// Layout: activations rotate on the matrix cores, 16 groups of 256 columns per wave (see RotTable below). Weights: one
// wavefront per row; lane l owns the 64-column chunk 64*p + l of pass p, so the H64 part of the transform runs in the
// lane's registers (three radix-4 stages, H4 x = sum(x) - 2 reverse(x), in float64) and the four chunks of a 256-group sit
// in one lane quad, combined through quad DPP broadcasts.
#include "rh3_common.hpp"

namespace rh3 {
namespace {

enum RotKind { ROT_PLAIN = 0, ROT_SWIGLU = 1, ROT_NORMMOD = 2, ROT_HEADS = 3 };

struct RotArgs {
  const uint16_t* x;
  int64_t ldx;       // row stride (PLAIN, SWIGLU, NORMMOD) or token stride (HEADS)
  int64_t ld_head;   // HEADS: head stride
  int64_t M, K;      // K = rotated / quantized width (SWIGLU: F; HEADS: H * 128), K % 256 == 0
  const uint16_t* w; // NORMMOD weight or nullptr
  float eps;
  const int32_t* idx;
  const void* shift;
  const void* scale;
  int64_t ld_tab;
  int8_t* q;
  int64_t ldq;
  float* s;
};

template <typename T> __device__ __forceinline__ float tab_at(const void* p, int64_t i);
template <> __device__ __forceinline__ float tab_at<float>(const void* p, int64_t i) {
  return static_cast<const float*>(p)[i];
}
template <> __device__ __forceinline__ float tab_at<uint16_t>(const void* p, int64_t i) {
  return bf2f(static_cast<const uint16_t*>(p)[i]);
}

typedef __bf16 v2bf_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pk_bf16_hw(float a, float b) {
  const v2bf_t v = {static_cast<__bf16>(a), static_cast<__bf16>(b)};
  return __builtin_bit_cast(uint32_t, v);
}

__device__ __forceinline__ float silu_mul_f(float g, float u) {
  const float sig = 1.0f / (1.0f + __expf(-g));
  return (g * sig) * u;
}

// one radix-4 stage of H64 on the elements i, i+S, i+2S, i+3S of every group (exact in float64 for
// values within 2^38 of each other)
template <int S, int N>
__device__ __forceinline__ void h4_stage(double (&d)[N]) {
#pragma unroll
  for (int g = 0; g < N / 4; ++g) {
    const int i = (g / S) * 4 * S + (g % S);
    const double x0 = d[i], x1 = d[i + S], x2 = d[i + 2 * S], x3 = d[i + 3 * S];
    const double t = ((x0 + x1) + x2) + x3;
    // fma(-2, x, t) rounds t - 2x once, like the subtraction (2x is exact)
    d[i] = fma(-2.0, x3, t);
    d[i + S] = fma(-2.0, x2, t);
    d[i + 2 * S] = fma(-2.0, x1, t);
    d[i + 3 * S] = fma(-2.0, x0, t);
  }
}

__device__ __forceinline__ void h64(double (&d)[64]) {
  h4_stage<1, 64>(d);
  h4_stage<4, 64>(d);
  h4_stage<16, 64>(d);
}

// lane q of every quad receives lane CTRL[2q+1:2q] of the quad (DPP quad_perm; every source lane is inside
// the quad, so bound_ctrl never applies)
template <int CTRL>
__device__ __forceinline__ double quad_d(double v) {
  const uint64_t u = __double_as_longlong(v);
  const uint32_t lo = static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(u & 0xffffffffu), CTRL, 0xf, 0xf, true));
  const uint32_t hi = static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(u >> 32), CTRL, 0xf, 0xf, true));
  return __longlong_as_double(static_cast<long long>((static_cast<uint64_t>(hi) << 32) | lo));
}

// ---------------------------------------------------------------- activations on the matrix cores
typedef float v4f_t __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf_t __attribute__((ext_vector_type(8)));
typedef short v2s_t __attribute__((ext_vector_type(2)));
typedef unsigned short v2us_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ v4f_t mfma_bf16(const uint4 a, const uint4 b, v4f_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf_t, a), __builtin_bit_cast(v8bf_t, b), c, 0, 0, 0);
}

// A 64-lane wave rotates 16 groups of 256 columns at once: H64 of the four 64-column chunks of a group on
// v_mfma_f32_16x16x32_bf16 with the group as the matrix column (lane l: group n = l & 15, quarter g = l >> 4), H64 / 8
// as the constant left operand. In chunk c the lane holds the 16 columns 64 c + 16 g + 8 t + e (t = 0, 1 the two MFMAs
// of k = 32) and receives the outputs 64 c + 16 T + 4 g + r (T = 0..3 the 16-row tiles of H64, r = 0..3).
//
// The sums must be exact before their one rounding to fp32. With E the largest exponent of the group, the bf16 values
// split into hi (exponent >= E - 10) and lo (the rest, exponent >= E - 21): each part's values are multiples of one
// power of two, 2^17 (plus 64 terms) below its largest, so every partial sum of the 64 terms fits 24 bits and the fp32
// accumulation is exact in any order; z = hi + lo is then the correctly rounded sum. A chunk with a nonzero value below
// 2^(E - 21), or a group whose exponents leave that window of normal numbers (E < 48, E > 245, infinities and NaN
// among them), takes the float64 butterflies instead (h64_slow): about 1 in 50 of the wave's chunks for normal values
// with 1 % of the channels x20, 1 in 1000 for normal values.
//
// What bounds it: VALU issue (70-75 % busy at 145,152 x 3072, 4 waves per SIMD), then HBM. VALU instructions per row of 3072,
// with the butterflies of all chunks in float64 and now: RMSNorm + modulation 1,777 and 1,187, head-major 1,097 and 708.
// Measured at 145,152 x 3072: RMSNorm + modulation 0.498 -> 0.397 ms; head-major 22,332 x 7168 0.132 -> 0.102 ms = 4.7 TB/s. The operand table stays in LDS: in registers (32 of them) only 3 waves fit a SIMD (0.495 ms), and a
// workgroup that walks several tiles spills (0.79 ms).
//
// H64 / 8 as that operand: H4[a][b] = -1 where b = 3 - a, +1 elsewhere; row i = 16 T + (l & 15) and column
// k = 16 g + 8 t + e in base 4, for every lane. A table rather than 32 words computed by each wave (a tenth of its
// instructions).
struct RotTable {
  uint32_t w[8][64][4];   // [4 t + T][lane]: the bf16 pairs e = 0..7
};
constexpr RotTable make_rot_table() {
  RotTable r{};
  for (int T = 0; T < 4; ++T)
    for (int t = 0; t < 2; ++t)
      for (int l = 0; l < 64; ++l)
        for (int e = 0; e < 8; ++e) {
          const int i0 = l & 3, i1 = (l >> 2) & 3, g = l >> 4;
          const uint32_t neg = static_cast<uint32_t>(((e & 3) == 3 - i0) ^ ((e >> 2) + 2 * t == 3 - i1) ^ (g == 3 - T));
          r.w[4 * t + T][l][e >> 1] |= (0x3e00u | (neg << 15)) << (16 * (e & 1));
        }
  return r;
}
__device__ constexpr RotTable ROT_TABLE = make_rot_table();

__device__ __forceinline__ uint32_t pk_max_u16(uint32_t a, uint32_t b) {
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(v2us_t, a), __builtin_bit_cast(v2us_t, b)));
}
__device__ __forceinline__ uint32_t pk_min_u16(uint32_t a, uint32_t b) {
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_bit_cast(v2us_t, a), __builtin_bit_cast(v2us_t, b)));
}
__device__ __forceinline__ uint32_t pk_sub_u16(uint32_t a, uint32_t b) {
  return __builtin_bit_cast(uint32_t, static_cast<v2us_t>(__builtin_bit_cast(v2us_t, a) - __builtin_bit_cast(v2us_t, b)));
}
// 0xffff in each half whose 16 bits are negative
__device__ __forceinline__ uint32_t pk_neg_mask(uint32_t a) {
  return __builtin_bit_cast(uint32_t, static_cast<v2s_t>(__builtin_bit_cast(v2s_t, a) >> 15));
}
// the largest of the four lanes l & 15 (+ 16, 32, 48)
__device__ __forceinline__ uint32_t max_quarters(uint32_t v) {
  auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  v = max(r[0], r[1]);
  r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
  return max(r[0], r[1]);
}

// one chunk in float64, every sum in the order of h64: radix-4 stages at strides 1 and 4 on the lane's 16 columns, the
// third across the four quarters by lane shuffles, each result rounded once and then scaled by 1/8 (the rounding of the
// unscaled sum, overflow to infinity included)
__device__ __forceinline__ void h64_slow(const uint32_t (&w)[8], float (&z)[16], int lane) {
  double d[16];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    d[2 * i] = static_cast<double>(__uint_as_float(w[i] << 16));
    d[2 * i + 1] = static_cast<double>(__uint_as_float(w[i] & 0xffff0000u));
  }
  h4_stage<1, 16>(d);
  h4_stage<4, 16>(d);
  const int n = lane & 15, g = lane >> 4;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    double x[4] = {0, 0, 0, 0};   // element 4 g + r of the four quarters
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const double v = __shfl(d[4 * i + r], 16 * k + n, 64);
        x[k] = g == i ? v : x[k];
      }
    const double t = ((x[0] + x[1]) + x[2]) + x[3];
#pragma unroll
    for (int T = 0; T < 4; ++T) z[4 * T + r] = static_cast<float>(fma(-2.0, x[3 - T], t)) * 0.125f;
  }
}

// The rotation of the lane's group, raw[c][4 t + p] = the chunk's bf16 pairs: y[4 q + T][r] = twice output
// 64 q + 16 T + 4 g + r (the reference's final halving is folded into the quantization scale, rot_scale). The H4
// combine of the four chunks is in the reference's order.
__device__ __forceinline__ void rot_group(const uint4* tab, const uint32_t (&raw)[4][8], int lane, float (&y)[16][4]) {
  uint32_t mx = 0;
  uint32_t mn[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    mn[c] = 0xffffffffu;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint32_t t = raw[c][i] & 0x7fff7fffu;
      mx = pk_max_u16(mx, t);
      mn[c] = pk_min_u16(mn[c], pk_sub_u16(t, 0x00010001u));   // zeros wrap to 0xffff
    }
  }
  const uint32_t amax = max_quarters(max(mx >> 16, mx & 0xffffu)), eb = amax & 0x7f80u;
  const uint32_t thr1 = eb - (10u << 7), thr2 = eb - (21u << 7);   // used only where E >= 48
  const bool off = amax != 0 && (eb < (48u << 7) || eb > (245u << 7));
  const uint32_t p1 = amax != 0 ? thr1 * 0x00010001u : 0u;
  float z[4][16];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const uint32_t m = min(mn[c] >> 16, mn[c] & 0xffffu);   // the least nonzero magnitude - 1 (0xffff: all zero)
    if (__builtin_amdgcn_ballot_w64(off || (amax != 0 && m + 1 < thr2)) != 0) {
      h64_slow(raw[c], z[c], lane);
    } else {
      uint32_t hi[8], lo[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const uint32_t s = pk_neg_mask(pk_sub_u16(raw[c][i] & 0x7fff7fffu, p1));
        lo[i] = raw[c][i] & s;
        hi[i] = raw[c][i] & ~s;
      }
      const uint4 h0 = make_uint4(hi[0], hi[1], hi[2], hi[3]), h1 = make_uint4(hi[4], hi[5], hi[6], hi[7]);
      const uint4 l0 = make_uint4(lo[0], lo[1], lo[2], lo[3]), l1 = make_uint4(lo[4], lo[5], lo[6], lo[7]);
#pragma unroll
      for (int T = 0; T < 4; ++T) {
        const v4f_t zero = {0.0f, 0.0f, 0.0f, 0.0f};
        const uint4 a0 = tab[T * 64 + lane], a1 = tab[(4 + T) * 64 + lane];
        const v4f_t zh = mfma_bf16(a1, h1, mfma_bf16(a0, h0, zero));
        const v4f_t zl = mfma_bf16(a1, l1, mfma_bf16(a0, l0, zero));
#pragma unroll
        for (int r = 0; r < 4; ++r) z[c][4 * T + r] = zh[r] + zl[r];
      }
    }
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const float s01 = z[0][i] + z[1][i];
    y[i >> 2][i & 3] = (s01 + z[2][i]) - z[3][i];
    y[4 + (i >> 2)][i & 3] = (s01 - z[2][i]) + z[3][i];
    y[8 + (i >> 2)][i & 3] = ((z[0][i] - z[1][i]) + z[2][i]) + z[3][i];
    y[12 + (i >> 2)][i & 3] = ((z[1][i] + z[2][i]) + z[3][i]) - z[0][i];
  }
}

// Row scale and quantization multiplier from the largest |t| (t = 2 y). With y = t / 2 the reference computes
// s = max(max|y| / 127, 1e-12) and q = rint(clamp(y * (1 / s), +-127)). Halving is exact for every normal t, so
// max|y| = max|t| / 2 and y * inv = t * (inv / 2); where t / 2 would be subnormal (|t| < 2^-125) both products lie
// below 2^-125 * 1e12 and round to the code 0, and a subnormal max|t| / 2 leaves s at its 1e-12 floor either way.
// The clamp never binds: |y * inv| <= 127 (1 + 2^-22) < 127.5.
__device__ __forceinline__ float rot_scale(float amax_t, float* inv_half) {
  const float s = fmaxf((amax_t * 0.5f) / 127.0f, 1e-12f);
  *inv_half = (1.0f / s) * 0.5f;
  return s;
}

// A workgroup of 4 waves holds 64 groups: the K / 256 groups of each of its rows (rot_rows of them), 16 groups per wave.
constexpr int ROT_GROUPS = 64;
// row absmax over the waves that share it, then the codes: rint(t * inv_half) by the magic-number add of pack4_codes
// (|t * inv_half| < 127.5 < 2^22), a 4 x 4 transpose over the quarters (lane g then holds columns 64 q + 16 g .. +15)
// and 16-byte stores
__device__ __forceinline__ void rot_row_max(const float (&y)[16][4], uint32_t* rowmax, int row, bool valid, int lane) {
  float am = 0.0f;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    am = max3_abs(am, y[i][0], y[i][1]);
    am = max3_abs(am, y[i][2], y[i][3]);
  }
  const uint32_t ab = max_quarters(__float_as_uint(am));   // am >= 0 and never NaN: the bits order like the values
  if (valid && lane < 16) atomicMax(rowmax + row, ab);
}
__device__ __forceinline__ void rot_store(const RotArgs& a, const float (&y)[16][4], const uint32_t* rowmax, int64_t m, int row,
                                          int grp, bool valid, int lane) {
  if (!valid) return;
  float inv;
  const float s = rot_scale(__uint_as_float(rowmax[row]), &inv);
  if (grp == 0 && lane < 16) a.s[m] = s;
  int8_t* const qp = a.q + m * a.ldq + grp * 256 + 16 * (lane >> 4);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    uint32_t w[4];
#pragma unroll
    for (int T = 0; T < 4; ++T) {
      float n[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) n[r] = y[4 * q + T][r] * inv;
      w[T] = pack4_codes(n);
    }
    auto r02 = __builtin_amdgcn_permlane32_swap(w[0], w[2], false, false);
    auto r13 = __builtin_amdgcn_permlane32_swap(w[1], w[3], false, false);
    auto lo = __builtin_amdgcn_permlane16_swap(r02[0], r13[0], false, false);
    auto hi = __builtin_amdgcn_permlane16_swap(r02[1], r13[1], false, false);
    // two 8-byte halves: the alignment the entry points require of q
    reinterpret_cast<uint2*>(qp + 64 * q)[0] = make_uint2(lo[0], lo[1]);
    reinterpret_cast<uint2*>(qp + 64 * q)[1] = make_uint2(hi[0], hi[1]);
  }
}

__device__ __forceinline__ void rot_table_to(uint4* tab) {
  const uint4* src = reinterpret_cast<const uint4*>(&ROT_TABLE);
  tab[threadIdx.x] = src[threadIdx.x];
  tab[256 + threadIdx.x] = src[256 + threadIdx.x];
}

// the rows of a workgroup
__host__ __device__ inline int rot_rows(int64_t K) { return static_cast<int>(ROT_GROUPS * 256 / K); }

// Plain, head-major and SwiGLU rows, read straight from global memory: lane (n, g) takes 32 bytes of each 128-byte
// chunk line of its group, four lanes a line.
template <int KIND>
__global__ void __launch_bounds__(256, 4) rot_quant_kernel(const RotArgs a) {
  static_assert(KIND != ROT_NORMMOD, "RMSNorm + modulation runs in rot_normmod_kernel");
  __shared__ uint4 tab[8 * 64];
  __shared__ uint32_t rowmax[ROT_GROUPS];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, n = lane & 15, g = lane >> 4;
  const int G = static_cast<int>(a.K >> 8), R = rot_rows(a.K);
  const int gi = wave * 16 + n, row = gi / G, grp = gi - row * G;
  const int64_t m0 = static_cast<int64_t>(blockIdx.x) * R, m = m0 + row;
  const bool valid = row < R && m < a.M;
  if (threadIdx.x < ROT_GROUPS) rowmax[threadIdx.x] = 0;
  rot_table_to(tab);
  __syncthreads();
  // a lane with no group of its own works on the first group of the workgroup's first row (in bounds) and stores nothing
  const int64_t ml = valid ? m : m0;
  const int gl = valid ? grp : 0;
  uint32_t raw[4][8];
  auto load16 = [&](const uint16_t* p, uint32_t* w) __attribute__((always_inline)) {
    const uint4 u0 = reinterpret_cast<const uint4*>(p)[0], u1 = reinterpret_cast<const uint4*>(p)[1];
    w[0] = u0.x; w[1] = u0.y; w[2] = u0.z; w[3] = u0.w;
    w[4] = u1.x; w[5] = u1.y; w[6] = u1.z; w[7] = u1.w;
  };
  if constexpr (KIND == ROT_SWIGLU) {
    const uint16_t* p = a.x + ml * a.ldx + gl * 256 + 16 * g;
    uint32_t up[4][8];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      load16(p + 64 * c, raw[c]);
      load16(p + 64 * c + a.K, up[c]);
    }
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int i = 0; i < 8; ++i)
        raw[c][i] = pk_bf16_hw(silu_mul_f(__uint_as_float(raw[c][i] << 16), __uint_as_float(up[c][i] << 16)),
                               silu_mul_f(__uint_as_float(raw[c][i] & 0xffff0000u), __uint_as_float(up[c][i] & 0xffff0000u)));
  } else if constexpr (KIND == ROT_HEADS) {
    const uint16_t* p = a.x + 2 * gl * a.ld_head + ml * a.ldx + 16 * g;
#pragma unroll
    for (int c = 0; c < 4; ++c) load16(p + (c >> 1) * a.ld_head + 64 * (c & 1), raw[c]);
  } else {
    const uint16_t* p = a.x + ml * a.ldx + gl * 256 + 16 * g;
#pragma unroll
    for (int c = 0; c < 4; ++c) load16(p + 64 * c, raw[c]);
  }
  float y[16][4];
  rot_group(tab, raw, lane, y);
  rot_row_max(y, rowmax, row, valid, lane);
  __syncthreads();
  rot_store(a, y, rowmax, m, row, grp, valid, lane);
}

// RMSNorm + modulation, rotation and INT8. Phase 1, a wave per row in the coalesced layout of the sum of squares (lane
// l holds columns 512 j + 8 l .. +7, the order of quant.hip): the row, the norm weight and both modulation rows are
// read with whole-wave 16-byte accesses, and the prologue values go to LDS as bf16, group-major, 16-byte unit u of
// group i at u ^ (i & 15), so that both phases' accesses spread over the banks. Phase 2 is the rotation of
// rot_quant_kernel from there.
template <typename TabT, int NCH, bool VEC>
__global__ void __launch_bounds__(256, 4) rot_normmod_kernel(const RotArgs a) {
  extern __shared__ uint4 stage[];   // 32 units of 16 bytes per group of the workgroup's rows
  __shared__ uint4 tab[8 * 64];
  __shared__ uint32_t rowmax[ROT_GROUPS];
  const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int G = static_cast<int>(a.K >> 8), R = min(4, rot_rows(a.K));   // one row per wave
  const int64_t m0 = static_cast<int64_t>(blockIdx.x) * R;
  if (threadIdx.x < ROT_GROUPS) rowmax[threadIdx.x] = 0;
  rot_table_to(tab);
  if (wave < R && m0 + wave < a.M) {
    // every row operand through a buffer resource (the row's base in scalar registers, its size as the range check: lanes
    // past K read zeros), so the loop has fixed 32-bit lane offsets and no branch
    const int64_t m = m0 + wave;
    const int K = static_cast<int>(a.K);
    constexpr int TB = sizeof(TabT);
    const int64_t trow = static_cast<int64_t>(__builtin_amdgcn_readfirstlane(a.idx[m])) * a.ld_tab;
    auto rsrc = [](const void* p, int bytes) __attribute__((always_inline)) {
      return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, BUF_RSRC_WORD3);
    };
    const __amdgpu_buffer_rsrc_t rx = rsrc(a.x + m * a.ldx, 2 * K), rw = rsrc(a.w, a.w ? 2 * K : 0);
    const __amdgpu_buffer_rsrc_t rsc = rsrc(static_cast<const TabT*>(a.scale) + trow, TB * K);
    const __amdgpu_buffer_rsrc_t rsh = rsrc(static_cast<const TabT*>(a.shift) + trow, TB * K);
    auto load16 = [](const __amdgpu_buffer_rsrc_t r, int off, int s) __attribute__((always_inline)) {
      const u32x4_t t = __builtin_amdgcn_raw_buffer_load_b128(r, off, s, 0);
      return make_uint4(t[0], t[1], t[2], t[3]);
    };
    auto load_at = [&](int j) __attribute__((always_inline)) { return load16(rx, 16 * lane, 1024 * j); };
    auto table_at = [&](const __amdgpu_buffer_rsrc_t r, const void* p, int j, float* t) __attribute__((always_inline)) {
      if constexpr (VEC && TB == 4) {
        const uint4 u0 = load16(r, 32 * lane, 2048 * j), u1 = load16(r, 32 * lane + 16, 2048 * j);
        t[0] = __uint_as_float(u0.x); t[1] = __uint_as_float(u0.y); t[2] = __uint_as_float(u0.z); t[3] = __uint_as_float(u0.w);
        t[4] = __uint_as_float(u1.x); t[5] = __uint_as_float(u1.y); t[6] = __uint_as_float(u1.z); t[7] = __uint_as_float(u1.w);
      } else if constexpr (VEC) {
        unpack8(load16(r, 16 * lane, 1024 * j), t);
      } else {  // rows that are not 16-byte aligned
        const int64_t c = 512 * j + 8 * lane;
#pragma unroll
        for (int e = 0; e < 8; ++e) t[e] = c < a.K ? tab_at<TabT>(p, trow + c + e) : 0.0f;
      }
    };
    float ss = 0.0f;
    auto add_squares = [&](const uint4 r) __attribute__((always_inline)) {
      float v[8];
      unpack8(r, v);
#pragma unroll
      for (int e = 0; e < 8; ++e) ss = fmaf(v[e], v[e], ss);  // x * x is exact (bf16 x): = ss + x * x
    };
    float rstd = 0.0f;
    const bool has_w = a.w != nullptr;
    auto modulate = [&](const uint4 r, int j) __attribute__((always_inline)) {
      float v[8], scl[8], shf[8];
      unpack8(r, v);
      table_at(rsc, a.scale, j, scl);
      table_at(rsh, a.shift, j, shf);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = v[e] * rstd;
      if (has_w) {
        float wv[8];
        unpack8(load16(rw, 16 * lane, 1024 * j), wv);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = v[e] * wv[e];
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = v[e] * (1.0f + scl[e]) + shf[e];
      const int i = wave * G + 2 * j + (lane >> 5);
      if (512 * j + 8 * lane < K)
        stage[i * 32 + ((lane & 31) ^ (i & 15))] =
            make_uint4(pk_bf16_hw(v[0], v[1]), pk_bf16_hw(v[2], v[3]), pk_bf16_hw(v[4], v[5]), pk_bf16_hw(v[6], v[7]));
    };
    auto finish = [&]() __attribute__((always_inline)) {
      ss = wave_sum_tree(ss);
      rstd = 1.0f / sqrtf(ss / static_cast<float>(a.K) + a.eps);
    };
    if constexpr (NCH > 0) {
      uint4 r[NCH];
#pragma unroll
      for (int j = 0; j < NCH; ++j) r[j] = load_at(j);
#pragma unroll
      for (int j = 0; j < NCH; ++j) add_squares(r[j]);
      finish();
#pragma unroll
      for (int j = 0; j < NCH; ++j) modulate(r[j], j);
    } else {  // the row does not fit the registers: read twice, the second time from L2
      const int nch = (K + 511) / 512;
#pragma unroll 4
      for (int j = 0; j < nch; ++j) add_squares(load_at(j));
      finish();
#pragma unroll 2
      for (int j = 0; j < nch; ++j) modulate(load_at(j), j);
    }
  }
  __syncthreads();
  const int gi = wave * 16 + n, row = gi / G, grp = gi - row * G;
  const int64_t m = m0 + row;
  const bool valid = row < R && m < a.M;
  const int il = valid ? gi : 0;   // lanes with no group of their own: group 0, nothing stored
  float y[16][4];
  const bool work = wave * 16 < R * G;   // the whole wave's groups may lie past the rows (it still meets the barrier)
  if (work) {
    uint32_t raw[4][8];
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const uint4 u = stage[il * 32 + ((8 * c + 2 * g + t) ^ (il & 15))];
        raw[c][4 * t] = u.x; raw[c][4 * t + 1] = u.y; raw[c][4 * t + 2] = u.z; raw[c][4 * t + 3] = u.w;
      }
    rot_group(tab, raw, lane, y);
    rot_row_max(y, rowmax, row, valid, lane);
  }
  __syncthreads();
  if (work) rot_store(a, y, rowmax, m, row, grp, valid, lane);
}

// ---------------------------------------------------------------- exact H256 rotation of weights
struct ExactArgs {
  const void* x;     // bf16 or fp32 rows
  int64_t ldx;
  int64_t M, K;
  float* y;          // OUT_F32: rotated rows
  int64_t ldy;
  int8_t* q;         // otherwise: int8 codes + per-row scale
  int64_t ldq;
  float* s;
};

// the exactly rotated chunk ch, rounded once to fp32
template <bool IN_F32>
__device__ __forceinline__ void rot_exact_chunk(const ExactArgs& a, int64_t m, int64_t ch, bool valid,
                                                float (&y)[64]) {
  double d[64];
  if (valid) {
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      const int64_t c = ch * 64 + 8 * t;
      float v[8];
      if (IN_F32) {
        const float4* p = reinterpret_cast<const float4*>(static_cast<const float*>(a.x) + m * a.ldx + c);
        const float4 u0 = p[0], u1 = p[1];
        v[0] = u0.x; v[1] = u0.y; v[2] = u0.z; v[3] = u0.w; v[4] = u1.x; v[5] = u1.y; v[6] = u1.z; v[7] = u1.w;
      } else {
        unpack8(*reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(a.x) + m * a.ldx + c), v);
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) d[8 * t + e] = static_cast<double>(v[e]);
    }
  } else {
#pragma unroll
    for (int i = 0; i < 64; ++i) d[i] = 0.0;
  }
  h64(d);
  // the fourth radix-4 stage runs across the lane quad: y_q = sum_k d_k - 2 d_(3-q)
#pragma unroll
  for (int i = 0; i < 64; ++i) {
    const double b0 = quad_d<0x00>(d[i]), b1 = quad_d<0x55>(d[i]), b2 = quad_d<0xAA>(d[i]), b3 = quad_d<0xFF>(d[i]);
    const double mir = quad_d<0x1B>(d[i]);
    const double t = ((b0 + b1) + b2) + b3;
    y[i] = static_cast<float>((t - 2.0 * mir) * 0.0625);
  }
}

template <bool IN_F32, bool OUT_F32, int NP>
__global__ void __launch_bounds__(256) rot_exact_kernel(const ExactArgs a) {
  const int lane = threadIdx.x & 63;
  const int64_t m = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (m >= a.M) return;
  const int64_t nchunks = a.K / 64;
  float y[64];
  if (OUT_F32) {
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const int64_t ch = 64 * p + lane;
      rot_exact_chunk<IN_F32>(a, m, ch, ch < nchunks, y);
      if (ch < nchunks) {
        float4* o = reinterpret_cast<float4*>(a.y + m * a.ldy + 64 * ch);
#pragma unroll
        for (int t = 0; t < 16; ++t) o[t] = make_float4(y[4 * t], y[4 * t + 1], y[4 * t + 2], y[4 * t + 3]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    return;
  }
  float amax = 0.0f;
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const int64_t ch = 64 * p + lane;
    rot_exact_chunk<IN_F32>(a, m, ch, ch < nchunks, y);
#pragma unroll
    for (int i = 0; i < 64; ++i) amax = fmaxf(amax, fabsf(y[i]));
    __builtin_amdgcn_sched_barrier(0);
  }
  amax = wave_max(amax);
  const float s = fmaxf(amax / 127.0f, 1e-12f);
  const float inv = 1.0f / s;
  if (lane == 0) a.s[m] = s;
  // int8_rowwise weight codes: round(w / s) with IEEE quotient semantics (kernels.py:69-71)
  auto emit = [&](int64_t ch) {
    int8_t* q = a.q + m * a.ldq + 64 * ch;
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      uint32_t b[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float r = fminf(fmaxf(rint_div(y[8 * t + e], s, inv), -127.0f), 127.0f);
        b[e] = static_cast<uint32_t>(static_cast<int32_t>(r)) & 0xffu;
      }
      uint2 o;
      o.x = b[0] | (b[1] << 8) | (b[2] << 16) | (b[3] << 24);
      o.y = b[4] | (b[5] << 8) | (b[6] << 16) | (b[7] << 24);
      *reinterpret_cast<uint2*>(q + 8 * t) = o;
    }
  };
  if (NP == 1) {
    if (lane < nchunks) emit(lane);
  } else {
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const int64_t ch = 64 * p + lane;
      rot_exact_chunk<IN_F32>(a, m, ch, ch < nchunks, y);
      if (ch < nchunks) emit(ch);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

template <typename TabT, bool VEC>
void launch_normmod(const RotArgs& a, hipStream_t st) {
  const int64_t R = rot_rows(a.K) < 4 ? rot_rows(a.K) : 4;
  const dim3 grid(static_cast<unsigned>((a.M + R - 1) / R)), block(256);
  const unsigned lds = static_cast<unsigned>(R * (a.K / 256) * 512);
  // the 512-column chunks of a row that a lane holds (wider rows are read twice)
  if (a.K <= 3072) hipLaunchKernelGGL((rot_normmod_kernel<TabT, 6, VEC>), grid, block, lds, st, a);
  else if (a.K <= 6144) hipLaunchKernelGGL((rot_normmod_kernel<TabT, 12, VEC>), grid, block, lds, st, a);
  else hipLaunchKernelGGL((rot_normmod_kernel<TabT, 0, VEC>), grid, block, lds, st, a);
}

template <int KIND>
void launch_rot(const RotArgs& a, hipStream_t st) {
  const int64_t R = rot_rows(a.K);
  hipLaunchKernelGGL((rot_quant_kernel<KIND>), dim3(static_cast<unsigned>((a.M + R - 1) / R)), dim3(256), 0, st, a);
}

template <int KIND, typename TabT>
int launch_act(const RotArgs& a, hipStream_t st, const char* name) {
  if (a.M == 0) return RH3_OK;
  if constexpr (KIND == ROT_NORMMOD) {
    // 16-byte modulation-table loads when every row start is 16-byte aligned
    if (aligned16(a.shift) && aligned16(a.scale) && (a.ld_tab * static_cast<int64_t>(sizeof(TabT))) % 16 == 0)
      launch_normmod<TabT, true>(a, st);
    else
      launch_normmod<TabT, false>(a, st);
  } else {
    launch_rot<KIND>(a, st);
  }
  return launch_status(name);
}

template <bool IN_F32, bool OUT_F32>
void launch_exact(const ExactArgs& a, hipStream_t st) {
  const dim3 grid(static_cast<unsigned>((a.M + 3) / 4)), block(256);
  if (a.K <= 4096) hipLaunchKernelGGL((rot_exact_kernel<IN_F32, OUT_F32, 1>), grid, block, 0, st, a);
  else if (a.K <= 8192) hipLaunchKernelGGL((rot_exact_kernel<IN_F32, OUT_F32, 2>), grid, block, 0, st, a);
  else hipLaunchKernelGGL((rot_exact_kernel<IN_F32, OUT_F32, 4>), grid, block, 0, st, a);
}

int check_rot(const char* name, const void* x, int64_t M, int64_t K, const void* q, int64_t ldq, const void* s) {
  RH3_REQUIRE(M >= 0 && K >= 0, "%s: negative size (M=%lld, K=%lld)", name, (long long)M, (long long)K);
  RH3_REQUIRE(K % 256 == 0, "%s: K=%lld must be a multiple of the rotation group 256", name, (long long)K);
  RH3_REQUIRE(K <= 16384, "%s: K=%lld exceeds the 16384-column limit of the rotation kernels", name, (long long)K);
  if (M == 0) return RH3_OK;
  RH3_REQUIRE(K > 0, "%s: K must be positive", name);
  RH3_REQUIRE(M < (int64_t{1} << 31) * 4, "%s: M=%lld too large", name, (long long)M);
  RH3_REQUIRE(x && q && s, "%s: null pointer", name);
  RH3_REQUIRE(ldq >= K && ldq % 8 == 0, "%s: output row stride %lld (K=%lld) must be >= K and a multiple of 8", name,
              (long long)ldq, (long long)K);
  RH3_REQUIRE(aligned16(x) && (reinterpret_cast<uintptr_t>(q) & 7) == 0, "%s: x must be 16-byte and q 8-byte aligned",
              name);
  return RH3_OK;
}

}  // namespace
}  // namespace rh3

using namespace rh3;

extern "C" int rh3_rot_quant_rows_i8(const uint16_t* x, int64_t ldx, int64_t M, int64_t K, int8_t* q, int64_t ldq,
                                     float* s, hipStream_t stream) {
  clear_error();
  if (int e = check_rot("rot_quant_rows_i8", x, M, K, q, ldq, s)) return e;
  RH3_REQUIRE(M == 0 || (ldx >= K && ldx % 8 == 0), "rot_quant_rows_i8: row stride %lld invalid for K=%lld",
              (long long)ldx, (long long)K);
  RotArgs a{x, ldx, 0, M, K, nullptr, 0.f, nullptr, nullptr, nullptr, 0, q, ldq, s};
  return launch_act<ROT_PLAIN, float>(a, stream, "rot_quant_rows_i8");
}

extern "C" int rh3_swiglu_rot_quant_rows_i8(const uint16_t* x, int64_t ldx, int64_t M, int64_t F, int8_t* q,
                                            int64_t ldq, float* s, hipStream_t stream) {
  clear_error();
  if (int e = check_rot("swiglu_rot_quant_rows_i8", x, M, F, q, ldq, s)) return e;
  RH3_REQUIRE(M == 0 || (ldx >= 2 * F && ldx % 8 == 0), "swiglu_rot_quant_rows_i8: row stride %lld invalid for 2F=%lld",
              (long long)ldx, (long long)(2 * F));
  RotArgs a{x, ldx, 0, M, F, nullptr, 0.f, nullptr, nullptr, nullptr, 0, q, ldq, s};
  return launch_act<ROT_SWIGLU, float>(a, stream, "swiglu_rot_quant_rows_i8");
}

extern "C" int rh3_norm_mod_rot_quant_i8(const uint16_t* x, int64_t ldx, int64_t M, int64_t K, const uint16_t* weight,
                                         float eps, const int32_t* idx, const void* shift, const void* scale,
                                         int tab_dtype, int64_t ld_tab, int8_t* q, int64_t ldq, float* s,
                                         hipStream_t stream) {
  clear_error();
  if (int e = check_rot("norm_mod_rot_quant_i8", x, M, K, q, ldq, s)) return e;
  if (M == 0) return RH3_OK;
  RH3_REQUIRE(ldx >= K && ldx % 8 == 0, "norm_mod_rot_quant_i8: row stride %lld invalid for K=%lld", (long long)ldx,
              (long long)K);
  RH3_REQUIRE(idx && shift && scale, "norm_mod_rot_quant_i8: idx, shift and scale are required");
  RH3_REQUIRE(ld_tab >= K, "norm_mod_rot_quant_i8: table row stride %lld < K=%lld", (long long)ld_tab, (long long)K);
  RH3_REQUIRE(!weight || aligned16(weight), "norm_mod_rot_quant_i8: weight must be 16-byte aligned");
  RH3_REQUIRE(tab_dtype == RH3_DTYPE_F32 || tab_dtype == RH3_DTYPE_BF16, "norm_mod_rot_quant_i8: tab_dtype %d",
              tab_dtype);
  RotArgs a{x, ldx, 0, M, K, weight, eps, idx, shift, scale, ld_tab, q, ldq, s};
  if (tab_dtype == RH3_DTYPE_F32) return launch_act<ROT_NORMMOD, float>(a, stream, "norm_mod_rot_quant_i8");
  return launch_act<ROT_NORMMOD, uint16_t>(a, stream, "norm_mod_rot_quant_i8");
}

extern "C" int rh3_rot_quant_heads_i8(const uint16_t* o, int64_t H, int64_t M, int64_t ld_head, int64_t ld_row,
                                      int8_t* q, int64_t ldq, float* s, hipStream_t stream) {
  clear_error();
  RH3_REQUIRE(H > 0 && H < (int64_t{1} << 24), "rot_quant_heads_i8: H=%lld", (long long)H);
  if (int e = check_rot("rot_quant_heads_i8", o, M, H * 128, q, ldq, s)) return e;
  if (M == 0) return RH3_OK;
  RH3_REQUIRE(ld_head % 8 == 0 && ld_row % 8 == 0 && ld_row >= 0 && ld_head >= 0,
              "rot_quant_heads_i8: strides must be non-negative multiples of 8 elements");
  RotArgs a{o, ld_row, ld_head, M, H * 128, nullptr, 0.f, nullptr, nullptr, nullptr, 0, q, ldq, s};
  return launch_act<ROT_HEADS, float>(a, stream, "rot_quant_heads_i8");
}

extern "C" int rh3_convrot_f32(const void* x, int x_dtype, int64_t ldx, int64_t M, int64_t K, float* y, int64_t ldy,
                               hipStream_t stream) {
  clear_error();
  RH3_REQUIRE(M >= 0 && K >= 0 && K % 256 == 0, "convrot_f32: K=%lld must be a non-negative multiple of 256",
              (long long)K);
  if (M == 0 || K == 0) return RH3_OK;
  RH3_REQUIRE(x && y, "convrot_f32: null pointer");
  RH3_REQUIRE(x_dtype == RH3_DTYPE_BF16 || x_dtype == RH3_DTYPE_F32, "convrot_f32: x_dtype %d", x_dtype);
  RH3_REQUIRE(ldx >= K && ldx % 8 == 0 && ldy >= K && ldy % 4 == 0, "convrot_f32: invalid row strides");
  RH3_REQUIRE(aligned16(x) && aligned16(y), "convrot_f32: x and y must be 16-byte aligned");
  RH3_REQUIRE(K <= 16384, "convrot_f32: K=%lld exceeds the 16384-column limit", (long long)K);
  RH3_REQUIRE(M < (int64_t{1} << 31) * 4, "convrot_f32: M=%lld too large", (long long)M);
  ExactArgs a{x, ldx, M, K, y, ldy, nullptr, 0, nullptr};
  if (x_dtype == RH3_DTYPE_F32) launch_exact<true, true>(a, stream);
  else launch_exact<false, true>(a, stream);
  return launch_status("convrot_f32");
}

extern "C" int rh3_quant_weight_rot_i8(const void* w, int w_dtype, int64_t ldw, int64_t N, int64_t K, int8_t* q,
                                       int64_t ldq, float* s, hipStream_t stream) {
  clear_error();
  if (int e = check_rot("quant_weight_rot_i8", w, N, K, q, ldq, s)) return e;
  if (N == 0) return RH3_OK;
  RH3_REQUIRE(w_dtype == RH3_DTYPE_BF16 || w_dtype == RH3_DTYPE_F32, "quant_weight_rot_i8: w_dtype %d", w_dtype);
  RH3_REQUIRE(ldw >= K && ldw % 8 == 0, "quant_weight_rot_i8: row stride %lld invalid for K=%lld", (long long)ldw,
              (long long)K);
  ExactArgs a{w, ldw, N, K, nullptr, 0, q, ldq, s};
  if (w_dtype == RH3_DTYPE_F32) launch_exact<true, false>(a, stream);
  else launch_exact<false, false>(a, stream);
  return launch_status("quant_weight_rot_i8");
}
