// What the GEMM kernels of librh3 share: the epilogues' names, the argument block, the MFMA forms of the two operand
// types and the LDS row swizzle.
#pragma once

#include <type_traits>

#include "rh3_common.hpp"
#include "attn_layout.hpp"
#include "attn_prologue.hpp"

namespace rh3 {
namespace gemm {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v16f __attribute__((ext_vector_type(16)));

enum Epi { EPI_PLAIN = 0, EPI_SWIGLU = 1, EPI_GATED = 2, EPI_ACC = 3, EPI_QKV = 4, EPI_GATED_ROWS = 5 };

constexpr int BK = 64;  // bytes of K per step

// EPI_QKV operands (pointers into the attention workspace of the chosen numerics)
struct QkvPrep {
  int64_t H, Spad;           // heads, tokens padded to 128
  int mode;                  // 0: one Q scale per (head, 128-token block); 1: per token after the H128 rotation
  int rotate;
  attn::RR rq, rk;           // q / k RMSNorm + RoPE (tab null: none)
  int8_t* q8;                // [H][Spad][128]
  float* qs;                 // mode 0: [H][Spad/128]; mode 1: [H][Spad]
  double* kpart;             // [H][nchunk][128] channel sums of the (RMSNorm + RoPE'd) k
  double* vsum;              // mode 1: [H][nchunk][128]
  float* vmax;
  float* vmin;
};

struct GemmArgs {
  const int8_t* x;  // [M, K] int8 or e4m3 codes
  int64_t ldx;
  const int8_t* w;  // [N, K]
  int64_t ldw;
  const float* xs;
  const float* ws;
  const uint16_t* bias;
  const uint16_t* gate;
  void* out;  // bf16 out / resid / int32 acc
  int64_t ldo;
  int64_t M, N, K;
  int tiles_m, tiles_n;
  QkvPrep qp;
  const int32_t* gidx;  // EPI_GATED_ROWS: gate table row of each output row (the gate is [R, ldg] bf16)
  int64_t ldg;
  int* ctr;  // persistent kernel: per-XCD tile counters (8 ints, zero at launch) or null (fixed tile shares)
};

// 16-byte chunk c (0..3) of LDS row r: rows r, r+1 share a 128-byte line; the XOR keeps 16
// consecutive rows of one chunk column on 16 distinct 16-byte bank groups.
__device__ __forceinline__ int swz(int r, int c) {
  return r * BK + ((c ^ (((r >> 1) & 3) ^ ((r >> 3) & 1))) << 4);
}

// g * sigmoid(g) * u with the sigmoid's reciprocal on v_rcp_f32 (1 ulp) instead of the IEEE division
// sequence (~10 instructions): the exp is approximate on both sides already, so the bf16 result moves by at
// most one ulp on a small fraction of elements, the tolerance the SwiGLU epilogue is held to
__device__ __forceinline__ float silu_mul(float g, float u) {
  const float sig = __builtin_amdgcn_rcpf(1.0f + __expf(-g));
  return (g * sig) * u;
}

// EPI_ACC stores the accumulator registers as they are: int32 values (int8) or fp32 bit patterns (e4m3)
__device__ __forceinline__ int acc_bits(int v) { return v; }
__device__ __forceinline__ int acc_bits(float v) { return __builtin_bit_cast(int, v); }

template <bool FP8>
struct Mma;

template <>
struct Mma<false> {  // int8: 2 MFMAs of k = 32 per 64-byte step, 16-byte fragments
  typedef v16i acc_t;
  static constexpr int KSUB = 2;
  typedef v4i frag_t;
  __device__ static frag_t load(const int8_t* lds, int row, int ks, int g) {
    return *reinterpret_cast<const v4i*>(lds + swz(row, ks * 2 + g));
  }
  __device__ static acc_t mma(frag_t a, frag_t b, acc_t c) {
    return __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, c, 0, 0, 0);
  }
  __device__ static float val(const acc_t& c, int r) { return static_cast<float>(c[r]); }
};

template <>
struct Mma<true> {  // e4m3: 1 MFMA of k = 64 per step, 32-byte fragments (two 16-byte chunks)
  typedef v16f acc_t;
  static constexpr int KSUB = 1;
  typedef v8i frag_t;
  __device__ static frag_t load(const int8_t* lds, int row, int, int g) {
    const v4i lo = *reinterpret_cast<const v4i*>(lds + swz(row, 2 * g));
    const v4i hi = *reinterpret_cast<const v4i*>(lds + swz(row, 2 * g + 1));
    frag_t f;
    f[0] = lo[0]; f[1] = lo[1]; f[2] = lo[2]; f[3] = lo[3];
    f[4] = hi[0]; f[5] = hi[1]; f[6] = hi[2]; f[7] = hi[3];
    return f;
  }
  __device__ static acc_t mma(frag_t a, frag_t b, acc_t c) {
    // cbsz / blgp type 0 = FP8 E4M3 for both operands; zero scale operands select the unscaled form
    return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, b, c, 0, 0, 0, 0, 0, 0);
  }
  __device__ static float val(const acc_t& c, int r) { return c[r]; }
};

// Which tiles a call runs on: `tile` for its rows from `head` on, the 256 x 256 kernels of gemm.hip for the rows before
enum TileId { TILE_256 = 0, TILE_128x64, TILE_128x128, TILE_256x128, TILE_256x192 };
struct TilePlan {
  int tile;
  int64_t head;  // a multiple of 256; 0: every row on `tile`
};
TilePlan plan_tiles(int64_t M, int64_t N, int64_t K, int64_t cus);
// a call on one of the small-tile kernels (gemm_tile.hip); 255 * ldx + 64 and 255 * ldw + 64 must be below 2^32
int run_tile(bool fp8, int epi, int cfg, const GemmArgs& a, hipStream_t stream, const char* name);

}  // namespace gemm
}  // namespace rh3
