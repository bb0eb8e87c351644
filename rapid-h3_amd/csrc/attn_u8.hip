// INT8 flash attention with the reference's production numerics (attn_int8.cu config 80 = attn_fwd8
// :2250-2511; configs 90/94 run the same math on a persistent schedule, and 1xx add the q/k RMSNorm + RoPE
// pre-pass), gfx950, head_dim 128, non-causal.
//
// Pre-pass (HBM-bound; attn_int8.cu:2568-2644):
//   stats_chunk    float64 channel sums of K (after the optional RMSNorm + RoPE), per 256-token chunk
//   vstats_chunk   float64 channel sums, max and min of V, per 256-token chunk
//   kmean_vfinal_kernel  kmean = fp32(sum / Sk) (attn_int8.cu:97-109), vmean = fp32(sum / Sk) (0 without smooth_v),
//                  vscale = max(max(vmax - vmean, vmean - vmin), 1e-6) / 127  (attn_int8.cu:97-109)
//   tokq_rows      per (token, head) row: [RMSNorm + RoPE] -> [- kmean] -> [normalized H128] -> one scale
//                  sc = max(amax, 1e-8) / 127, q = rint(x * (1 / sc))         (attn_int8.cu:113-170, :298-340);
//                  for K also the per-key pair (sc, -1.5*2^23 * sc); padded keys get (0, -inf)
//   vq_tile        per (128-key tile, head): int8 V codes rint((v - vmean) / vscale) (attn_int8.cu:452-475),
//                  transposed to [H][128][Skpad] in the key order of the P.V operand, and the tile's P.V
//                  accumulator start 1.5*2^23 bits + 128 * (sum of its codes) per channel
//   In three launches: pre_a_u8_kernel (both statistics and Q), kmean_vfinal_kernel, pre_b_u8_kernel (K and V).
// Main kernel: per (128-query block, head) workgroup of 4 waves, 32 queries per wave, 128-key tiles.
//   S^T = K8 . Q8^T on v_mfma_i32_32x32x32_i8 (keys on rows, queries on lanes), the accumulator starting at
//   the bits of 1.5*2^23 so that t = fma(float bits, s_j, b_j) is the dequantized score in one instruction;
//   tile max tm, n = max(m, tm), a = 2^((m - n) c), ts = 2^((tm - n) c); P = rint(2^(fma(t, c, log2 255 - tm c)))
//   in [0, 255]; row sums of the integer P; O^T += V8^T . P^T on v_mfma_i32_32x32x32_i8 with P - 128 as the
//   signed operand (the tile's 128 * sum(V codes) is the accumulator start, so the integer result is the
//   reference's u8 x s8 product exactly); O = fma(ts, acc bits, fma(O, a, -ts * 1.5*2^23)); out =
//   bf16(fma(O (1 / l), vscale, vmean)). Text bias (attn_cake.cuh:97-99, :210-240): t += bias*log2(e) / c on
//   keys [0, nbias).
// Configs 60-61 (attn_fwd6 :1786-1962): the same kernel with BK = true and blockk_tile (quant_k_block :404-443)
//   in place of the per-token K quantizer: one K scale per 128-key tile, integer tile max, no per-key dequant.
#include "attn_common.hpp"
#include "attn_layout.hpp"

namespace rh3 {
namespace {

using namespace attn;
using attn_ws::WorkU8;
using attn_ws::layout_u8;

constexpr int TILE = 128;                 // keys per tile (the tile max of the u8 P)
constexpr int SIDE = 2048;                // bytes per (head, tile): 128 (s, b) pairs, 128 int32 starts, pad
constexpr int SIDE_VINIT = 1024;          // byte offset of the accumulator starts inside a side record
constexpr int MAGIC_I = 0x4B400000;       // bits of 1.5 * 2^23
constexpr float MAGIC_F = 12582912.0f;
constexpr float LOG2_255 = 7.99435343685886f;       // attn_int8.cu:24
constexpr float LOG2_448 = 8.807354922057604f;      // attn_int8.cu:1557
constexpr float V_STRETCH = 448.0f / 127.0f;        // attn_int8.cu:468
constexpr float V_UNSTRETCH = 127.0f / 448.0f;      // attn_int8.cu:2642
constexpr float INV_SQRT128 = 0.08838834764831845f;  // attn_int8.cu:127

// ------------------------------------------------------------------ V statistics
// grid (H, nchunk) (heads fastest, so a chunk's token rows are read together), 256 threads = 16 token slots x 16
// lanes (8 channels each)
constexpr int VSTATS_LDS = 16 * D * (8 + 4 + 4);
// max / min of three floats in one instruction (fmaxf and fminf chains get a NaN-quieting max per operand)
__device__ __forceinline__ float max3(float a, float b, float c) {
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}
__device__ __forceinline__ float min3(float a, float b, float c) {
  float r;
  asm("v_min3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}
__device__ __forceinline__ void vstats_chunk(const uint16_t* __restrict__ v, int64_t v_ss, int64_t v_sh, int64_t S,
                                             double* __restrict__ vsum, float* __restrict__ vmax,
                                             float* __restrict__ vmin, int h, int c, int nchunk, void* lds) {
  double(*red)[D] = static_cast<double(*)[D]>(lds);
  float(*rmx)[D] = reinterpret_cast<float(*)[D]>(red + 16);
  float(*rmn)[D] = rmx + 16;
  const int tid = threadIdx.x;
  const int slot = tid >> 4, l16 = tid & 15;
  double acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  float mx[8], mn[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) { mx[e] = -INFINITY; mn[e] = INFINITY; }
  // the rows of four iterations are loaded before any is used (rows past S read row S - 1 and are skipped)
  for (int it0 = 0; it0 < CHUNK / 16; it0 += 4) {
    uint4 rx[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int64_t s = static_cast<int64_t>(c) * CHUNK + (it0 + i) * 16 + slot;
      rx[i] = *reinterpret_cast<const uint4*>(v + (s < S ? s : S - 1) * v_ss + h * v_sh + 8 * l16);
    }
    // max and min two rows at a time, the sums row by row
    auto rows = [&](auto full) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < 4; i += 2) {
        const int64_t s0 = static_cast<int64_t>(c) * CHUNK + (it0 + i) * 16 + slot;
        if (!full && s0 >= S) return;
        const bool two = full || s0 + 16 < S;
        float x[8], y[8];
        unpack8(rx[i], x);
        unpack8(rx[i + 1], y);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float z = two ? y[e] : x[e];
          mx[e] = max3(mx[e], x[e], z);
          mn[e] = min3(mn[e], x[e], z);
          acc[e] += static_cast<double>(x[e]);
          if (two) acc[e] += static_cast<double>(y[e]);
        }
      }
    };
    if (static_cast<int64_t>(c + 1) * CHUNK <= S) rows(std::true_type{});   // uniform: no row of the chunk past S
    else rows(std::false_type{});
  }
  // max3 and min3 skip a quiet NaN, but a signalling one replaces what they held: a lane whose sums met any NaN takes its
  // maxima and minima again, value by value
  bool nan = false;
#pragma unroll
  for (int e = 0; e < 8; ++e) nan |= acc[e] != acc[e];
  if (nan) {
#pragma unroll
    for (int e = 0; e < 8; ++e) { mx[e] = -INFINITY; mn[e] = INFINITY; }
    for (int64_t s = static_cast<int64_t>(c) * CHUNK + slot; s < S && s < static_cast<int64_t>(c + 1) * CHUNK; s += 16) {
      float x[8];
      unpack8(*reinterpret_cast<const uint4*>(v + s * v_ss + h * v_sh + 8 * l16), x);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        mx[e] = fmaxf(mx[e], x[e]);
        mn[e] = fminf(mn[e], x[e]);
      }
    }
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    red[slot][8 * l16 + e] = acc[e];
    rmx[slot][8 * l16 + e] = mx[e];
    rmn[slot][8 * l16 + e] = mn[e];
  }
  __syncthreads();
  if (tid < D) {
    double t = 0.0;
    float a = -INFINITY, b = INFINITY;
    for (int i = 0; i < 16; ++i) {
      t += red[i][tid];
      a = fmaxf(a, rmx[i][tid]);
      b = fminf(b, rmn[i][tid]);
    }
    const int64_t o = (static_cast<int64_t>(h) * nchunk + c) * D + tid;
    vsum[o] = t;
    vmax[o] = a;
    vmin[o] = b;
  }
}

// grid (H, 2), KMEAN_NT threads: y = 0 the K mean (kmean_kernel's fold; zeros without smoothing), y = 1 V's mean and scale:
// group j of 128 channels folds chunks j, j + 8, ..., then the 8 groups (the float64 sums of bf16 values are exact and max /
// min are order-free, so the grouping does not change the result). The first workgroup also clears the work counter.
__global__ void __launch_bounds__(KMEAN_NT) kmean_vfinal_kernel(const WorkU8 w, int nchunk, int64_t S, int smooth_k, int smooth_v) {
  constexpr int G = KMEAN_NT / D;
  __shared__ double rs[G][D];
  __shared__ float rmx[G][D], rmn[G][D];
  const int h = blockIdx.x, d = threadIdx.x % D, j = threadIdx.x / D;
  if (blockIdx.y == 0) {
    if (h == 0 && threadIdx.x == 0) *w.ctr = 0;
    if (!smooth_k) {
      if (j == 0) w.kmean[h * D + d] = 0.0f;
      return;
    }
    kmean_fold(w.kpart + static_cast<int64_t>(h) * nchunk * D + d, nchunk, S, w.kmean + h * D, d, j, rs);
    return;
  }
  double t = 0.0;
  float a = -INFINITY, b = INFINITY;
  for (int c = j; c < nchunk; c += G) {
    const int64_t o = (static_cast<int64_t>(h) * nchunk + c) * D + d;
    t += w.vsum[o];
    a = fmaxf(a, w.vmax[o]);
    b = fminf(b, w.vmin[o]);
  }
  rs[j][d] = t;
  rmx[j][d] = a;
  rmn[j][d] = b;
  __syncthreads();
  if (j != 0) return;
#pragma unroll
  for (int i = 1; i < G; ++i) {
    t += rs[i][d];
    a = fmaxf(a, rmx[i][d]);
    b = fminf(b, rmn[i][d]);
  }
  const float vm = smooth_v ? static_cast<float>(t / static_cast<double>(S)) : 0.0f;
  w.vmean[h * D + d] = vm;
  w.vscale[h * D + d] = fmaxf(fmaxf(a - vm, vm - b), 1e-6f) / 127.0f;
}

// ------------------------------------------------------------------ per-token Q / K quantizer
// 256 threads = 16 groups of 16 lanes; group i = block * 16 + tid / 16 takes the TOKQ_ROWS tokens TOKQ_ROWS (i / H) .. of head
// i % H (heads fastest, so a workgroup's rope-table rows are shared). Bound by VALU: about 260 instructions per 8 values with
// RMSNorm + RoPE, against 522 with one row per group (half of them addresses, norm weights and the division by H) and
// selects in the transform.
constexpr int TOKQ_ROWS = 4;
__device__ __forceinline__ void tokq_rows(const uint16_t* __restrict__ x, int64_t x_ss, int64_t x_sh, int64_t S, int64_t Spad,
                                          int H, const RR& rr, const float* __restrict__ mean, int rotate,
                                          int8_t* __restrict__ codes, float* __restrict__ scales, float* __restrict__ side,
                                          uint32_t block) {
  const int tid = threadIdx.x, lane = tid & 63, l16 = tid & 15;
  const uint32_t i = block * 16 + (tid >> 4), q4 = i / static_cast<uint32_t>(H);   // Spad * H < 2^31
  const int h = static_cast<int>(i - q4 * H);
  const int64_t s0 = static_cast<int64_t>(q4) * TOKQ_ROWS;
  int8_t* co = codes + (h * Spad + s0) * D + 8 * l16;
  float* sc_out = scales + h * Spad + s0;
  // TOKQ_ROWS tokens lie in one tile (TILE is a multiple)
  float2* pair = side ? reinterpret_cast<float2*>(side + (h * (Spad / TILE) + s0 / TILE) * (SIDE / 4)) + s0 % TILE : nullptr;
  // the rows, their rope-table rows and the norm weights are loaded together, before any arithmetic (rows past S read the
  // last one)
  const uint16_t* xp = x + h * x_sh + 8 * l16;
  uint4 rx[TOKQ_ROWS], rt[TOKQ_ROWS][4];
#pragma unroll
  for (int u = 0; u < TOKQ_ROWS; ++u) {
    const int64_t sl = s0 + u < S ? s0 + u : S - 1;
    rx[u] = *reinterpret_cast<const uint4*>(xp + sl * x_ss);
    if (rr.tab) rope_tab8_raw(rr, l16, sl, rt[u]);
  }
  float w[8], m[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  if (rr.tab) load8(rr.w + 8 * l16, w);
  if (mean) {
    const float4 a = *reinterpret_cast<const float4*>(mean + h * D + 8 * l16);
    const float4 b = *reinterpret_cast<const float4*>(mean + h * D + 8 * l16 + 4);
    m[0] = a.x; m[1] = a.y; m[2] = a.z; m[3] = a.w; m[4] = b.x; m[5] = b.y; m[6] = b.z; m[7] = b.w;
  }
#pragma unroll
  for (int u = 0; u < TOKQ_ROWS; ++u) {
    const bool ok = s0 + u < S;   // uniform per 16-lane row
    float v[8];
    unpack8(rx[u], v);
    if (rr.tab) rms_rope8_raw(v, lane, rr, w, rt[u]);
    if (mean) {
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = v[e] - m[e];
    }
    if (rotate) wht128_row(v, l16);
    if (!rr.tab && !mean && !rotate) {   // the raw values: row_amax16 takes no signalling NaN
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = __builtin_canonicalizef(v[e]);
    }
    uint2 o;
    const float sc = token_quant_row(v, o);
    *reinterpret_cast<uint2*>(co + u * D) = ok ? o : make_uint2(0, 0);   // padded rows and keys: zero codes
    if (l16 == 0) {
      sc_out[u] = ok ? sc : 0.0f;
      if (pair) pair[u] = ok ? make_float2(sc, -MAGIC_F * sc) : make_float2(0.0f, -INFINITY);
    }
  }
}
inline unsigned tokq_blocks(int64_t Spad, int64_t H) { return static_cast<unsigned>((Spad / TOKQ_ROWS * H + 15) / 16); }

// ------------------------------------------------------------------ per-block K (configs 60-61)
// grid (H, Skpad / 128) (heads fastest), 256 threads: wave w quantizes tokens 32 w .. 32 w + 31 of the block, four 16-lane rows
// per pass. K - kmean -> [normalized H128] -> one scale per (head, 128-key block) sc = max(amax, 1e-8) / 127,
// codes rint(x * (1 / sc)) (quant_k_block, attn_int8.cu:404-443); sc goes to kbs [H][Skpad/128] and to the first
// float of the block's side record, where the main kernel reads it. Padded tokens are zero rows.
__device__ __forceinline__ void blockk_tile(const uint16_t* __restrict__ k, int64_t k_ss, int64_t k_sh, int64_t S,
                                            int64_t Spad, const float* __restrict__ mean, int rotate,
                                            int8_t* __restrict__ codes, float* __restrict__ kbs, float* __restrict__ side,
                                            int h, int blk, float* wmax) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l16 = lane & 15, sub = lane >> 4;
  float m[8];
  {
    const float4 a = *reinterpret_cast<const float4*>(mean + h * D + 8 * l16);
    const float4 b = *reinterpret_cast<const float4*>(mean + h * D + 8 * l16 + 4);
    m[0] = a.x; m[1] = a.y; m[2] = a.z; m[3] = a.w; m[4] = b.x; m[5] = b.y; m[6] = b.z; m[7] = b.w;
  }
  float v[8][8];
  float amax = 0.0f;
#pragma unroll
  for (int p = 0; p < 8; ++p) {
    const int64_t s = static_cast<int64_t>(blk) * TILE + wave * 32 + p * 4 + sub;
    const bool ok = s < S;  // uniform per 16-lane row
#pragma unroll
    for (int e = 0; e < 8; ++e) v[p][e] = 0.0f;
    if (ok) {
      load8(k + s * k_ss + h * k_sh + 8 * l16, v[p]);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[p][e] = v[p][e] - m[e];
    }
    if (rotate) wht128_row(v[p], l16);  // every lane joins the row shuffles; zero rows stay zero
#pragma unroll
    for (int e = 0; e < 8; ++e) amax = fmaxf(amax, fabsf(v[p][e]));
  }
  amax = wave_max(amax);
  if (lane == 0) wmax[wave] = amax;
  __syncthreads();
  const float bm = fmaxf(fmaxf(wmax[0], wmax[1]), fmaxf(wmax[2], wmax[3]));
  const float sc = fmaxf(bm, 1e-8f) / 127.0f;
  const float inv = 1.0f / sc;
  if (tid == 0) {
    kbs[static_cast<int64_t>(h) * (Spad / TILE) + blk] = sc;
    side[((static_cast<int64_t>(h) * (Spad / TILE) + blk) * SIDE) / 4] = sc;
  }
#pragma unroll
  for (int p = 0; p < 8; ++p) {
    const int64_t s = static_cast<int64_t>(blk) * TILE + wave * 32 + p * 4 + sub;
    uint32_t b[8];
    // |x * inv| <= 127 (1 + 2^-23): rint stays within the int8 range without a clamp
#pragma unroll
    for (int e = 0; e < 8; ++e) b[e] = static_cast<uint32_t>(static_cast<int32_t>(rintf(v[p][e] * inv))) & 0xffu;
    uint2 o;
    o.x = b[0] | (b[1] << 8) | (b[2] << 16) | (b[3] << 24);
    o.y = b[4] | (b[5] << 8) | (b[6] << 16) | (b[7] << 24);
    *reinterpret_cast<uint2*>(codes + (static_cast<int64_t>(h) * Spad + s) * D + 8 * l16) = o;
  }
}

// ------------------------------------------------------------------ V codes, transposed
// Position p of a 32-key block holds key perm_u8(p): p = 16 g + r <-> key 8 (r / 4) + 4 g + r % 4, the key of
// register r of lane group g in the S^T accumulator, so that a lane's 16 P bytes are its P.V B operand.
__device__ __forceinline__ int perm_u8(int p) {
  const int g = p >> 4, r = p & 15;
  return 8 * (r >> 2) + 4 * g + (r & 3);
}

// Position p of a 64-key chunk of the e4m3 layout holds key perm_f8(p): p = 32 g + 16 h + r <-> key 32 h + 8 (r / 4)
// + 4 g + r % 4, the key of register r of 32-key block h in lane group g's S^T accumulator, so that a lane's 32 P
// bytes of the chunk are its B operand of the 64-deep FP8 MFMA.
__device__ __forceinline__ int perm_f8(int p) {
  const int g = p >> 5, hh = (p >> 4) & 1, r = p & 15;
  return 32 * hh + 8 * (r >> 2) + 4 * g + (r & 3);
}

// grid (H, Skpad / 128) (heads fastest), 256 threads. F8 (configs 50-56): e4m3 codes of ((v - vmean) / vscale) *
// fp32(448 / 127) (attn_int8.cu:467-473) in the perm_f8 order, and no accumulator starts.
constexpr int VQ_PITCH = D + 16;  // row pitch of the key-major code tile
template <bool F8>
__device__ __forceinline__ void vq_tile(const uint16_t* __restrict__ v, int64_t v_ss, int64_t v_sh, int64_t S, int64_t Spad,
                                        const float* __restrict__ vmean, const float* __restrict__ vscale,
                                        int8_t* __restrict__ vt, int32_t* __restrict__ side, int h, int blk, int8_t* tile) {
  constexpr int P = VQ_PITCH;
  const int tid = threadIdx.x, l16 = tid & 15;
  const int64_t s0 = static_cast<int64_t>(blk) * TILE;
  float vm[8], vs[8], iv[8];
  {
    const float4 a = *reinterpret_cast<const float4*>(vmean + h * D + 8 * l16);
    const float4 b = *reinterpret_cast<const float4*>(vmean + h * D + 8 * l16 + 4);
    const float4 c = *reinterpret_cast<const float4*>(vscale + h * D + 8 * l16);
    const float4 d = *reinterpret_cast<const float4*>(vscale + h * D + 8 * l16 + 4);
    vm[0] = a.x; vm[1] = a.y; vm[2] = a.z; vm[3] = a.w; vm[4] = b.x; vm[5] = b.y; vm[6] = b.z; vm[7] = b.w;
    vs[0] = c.x; vs[1] = c.y; vs[2] = c.z; vs[3] = c.w; vs[4] = d.x; vs[5] = d.y; vs[6] = d.z; vs[7] = d.w;
#pragma unroll
    for (int e = 0; e < 8; ++e) iv[e] = 1.0f / vs[e];
  }
  // 128 keys x 16 lanes: 8 passes of 16 keys
  for (int r = tid >> 4; r < TILE; r += 16) {
    uint2 o = make_uint2(0, 0);
    if (s0 + r < S) {
      float x[8];
      load8(v + (s0 + r) * v_ss + h * v_sh + 8 * l16, x);
      if constexpr (F8) {
        float y[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) y[e] = fminf(fmaxf(((x[e] - vm[e]) / vs[e]) * V_STRETCH, -448.0f), 448.0f);
        o.x = __builtin_amdgcn_cvt_pk_fp8_f32(y[2], y[3], __builtin_amdgcn_cvt_pk_fp8_f32(y[0], y[1], 0, false), true);
        o.y = __builtin_amdgcn_cvt_pk_fp8_f32(y[6], y[7], __builtin_amdgcn_cvt_pk_fp8_f32(y[4], y[5], 0, false), true);
      } else {
        // rint_div with one wave vote per 8 values: |x * inv| < 128, so the product lies within 2^-15 of the IEEE quotient
        float n[8], d = 0.0f;
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = x[e] - vm[e];
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
          const float t0 = x[e] * iv[e], t1 = x[e + 1] * iv[e + 1];
          n[e] = rintf(t0);
          n[e + 1] = rintf(t1);
          d = max3_abs(d, t0 - n[e], t1 - n[e + 1]);
        }
        if (__builtin_amdgcn_ballot_w64(d > 0.5f - 0x1p-14f) != 0) {
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            float so = vs[e];   // opaque, so that the division's divisor-only steps stay on this path
            asm volatile("" : "+v"(so));
            if (fabsf(x[e] * iv[e] - n[e]) > 0.5f - 0x1p-14f) n[e] = rintf(x[e] / so);
          }
        }
        o = make_uint2(pack4_codes(n), pack4_codes(n + 4));
      }
    }
    *reinterpret_cast<uint2*>(&tile[r * P + 8 * l16]) = o;
  }
  __syncthreads();
  // thread i: channels 4 (i / 8) .. +3, positions 16 (i % 8) .. +15 of the tile, by 4 x 4 byte transposes (four keys' words
  // in, four channels' out)
  const int d0 = 4 * (tid >> 3), pc = (tid & 7) * 16;
  uint32_t w[4][4];   // [channel][position / 4]
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    uint32_t k[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int p = pc + 4 * t + e;
      const int key = F8 ? (p & ~63) + perm_f8(p & 63) : (p & ~31) + perm_u8(p & 31);
      k[e] = *reinterpret_cast<const uint32_t*>(&tile[key * P + d0]);
    }
    // v_perm_b32(hi, lo, sel): selector bytes 0-3 take lo's bytes, 4-7 hi's
    const uint32_t a01 = __builtin_amdgcn_perm(k[1], k[0], 0x05010400u), a23 = __builtin_amdgcn_perm(k[3], k[2], 0x05010400u);
    const uint32_t b01 = __builtin_amdgcn_perm(k[1], k[0], 0x07030602u), b23 = __builtin_amdgcn_perm(k[3], k[2], 0x07030602u);
    w[0][t] = __builtin_amdgcn_perm(a23, a01, 0x05040100u);
    w[1][t] = __builtin_amdgcn_perm(a23, a01, 0x07060302u);
    w[2][t] = __builtin_amdgcn_perm(b23, b01, 0x05040100u);
    w[3][t] = __builtin_amdgcn_perm(b23, b01, 0x07060302u);
  }
#pragma unroll
  for (int c = 0; c < 4; ++c)
    *reinterpret_cast<uint4*>(vt + (static_cast<int64_t>(h) * D + d0 + c) * Spad + s0 + pc) =
        make_uint4(w[c][0], w[c][1], w[c][2], w[c][3]);
  // accumulator starts: 1.5*2^23 bits + 128 * (sum of the tile's codes of channel d), over the 8 threads of a channel; the
  // pad is zeroed
  if constexpr (F8) return;
  int32_t* rec = side + (static_cast<int64_t>(h) * (Spad / TILE) + blk) * (SIDE / 4);
  int sum[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    int t = 0;
#pragma unroll
    for (int u = 0; u < 4; ++u) t = __builtin_amdgcn_sdot4(static_cast<int>(w[c][u]), 0x01010101, t, false);
    t += __builtin_amdgcn_update_dpp(0, t, 0xB1, 0xf, 0xf, true);    // lane ^ 1
    t += __builtin_amdgcn_update_dpp(0, t, 0x4E, 0xf, 0xf, true);    // lane ^ 2
    t += __builtin_amdgcn_update_dpp(0, t, 0x141, 0xf, 0xf, true);   // 7 - lane of the 8: the other four's sum
    sum[c] = MAGIC_I + 128 * t;
  }
  if ((tid & 7) == 0) {
    *reinterpret_cast<int4*>(rec + SIDE_VINIT / 4 + d0) = make_int4(sum[0], sum[1], sum[2], sum[3]);
    *reinterpret_cast<int4*>(rec + SIDE_VINIT / 4 + D + d0) = make_int4(0, 0, 0, 0);
  }
}

// ------------------------------------------------------------------ the pre-pass in three launches
// A: K statistics (smoothing), V statistics and the Q quantizer; kmean_vfinal_kernel: their second level; B: the K quantizer
// and the V codes. The parts of one launch do not depend on each other; run as eight launches of their own, the small ones cost
// more in launch gaps than in work and the memory-bound ones ran beside no arithmetic. Whole pre-pass with RMSNorm + RoPE (us,
// before and now): 1,560 tokens x 24 heads 60 and 42, 5,583 x 56 193 and 168, 22,332 x 56 670 and 611. Both are bound by VALU
// issue (A 79 %, B 74 % busy at 5,583 x 56, both saturated at 145,152 x 24), with 3.1 to 3.8 waves per SIMD.
struct PreU8 {
  const uint16_t *q, *k, *v;
  int64_t q_ss, q_sh, k_ss, k_sh, v_ss, v_sh;
  int64_t Sq, Sk, sqp, skp;
  int H, nchunk, smooth_k, smooth_v, rotate;
  RR rq, rk;
  WorkU8 w;
  unsigned nk, nv;   // workgroups of the first two parts (A: K and V statistics; B: nk of the K quantizer)
};

__global__ void __launch_bounds__(256) pre_a_u8_kernel(const PreU8 a) {
  __shared__ __attribute__((aligned(16))) int8_t lds[VSTATS_LDS];
  static_assert(VSTATS_LDS >= STATS_LDS, "shared by the parts");
  unsigned b = blockIdx.x;
  if (b < a.nk) {
    if (a.rk.tab) stats_chunk<true>(a.k, a.k_ss, a.k_sh, a.Sk, a.rk, a.w.kpart, nullptr, 0, b % a.H, b / a.H, a.nchunk, lds);
    else stats_chunk<false>(a.k, a.k_ss, a.k_sh, a.Sk, a.rk, a.w.kpart, nullptr, 0, b % a.H, b / a.H, a.nchunk, lds);
    return;
  }
  b -= a.nk;
  if (b < a.nv) {
    vstats_chunk(a.v, a.v_ss, a.v_sh, a.Sk, a.w.vsum, a.w.vmax, a.w.vmin, b % a.H, b / a.H, a.nchunk, lds);
    return;
  }
  b -= a.nv;
  tokq_rows(a.q, a.q_ss, a.q_sh, a.Sq, a.sqp, a.H, a.rq, nullptr, a.rotate, a.w.q8, a.w.qs, nullptr, b);
}

// V: 0 int8 codes, 1 e4m3 codes; BLK: K quantized per 128-key block (configs 60-61) instead of per token
template <bool F8, bool BLK>
__global__ void __launch_bounds__(256) pre_b_u8_kernel(const PreU8 a) {
  __shared__ __attribute__((aligned(16))) int8_t tile[TILE * VQ_PITCH];
  const unsigned b = blockIdx.x;
  if (b >= a.nk) {
    const unsigned t = b - a.nk;
    vq_tile<F8>(a.v, a.v_ss, a.v_sh, a.Sk, a.skp, a.w.vmean, a.w.vscale, a.w.vt, reinterpret_cast<int32_t*>(a.w.side), t % a.H,
                t / a.H, tile);
  } else if constexpr (BLK) {
    blockk_tile(a.k, a.k_ss, a.k_sh, a.Sk, a.skp, a.w.kmean, a.rotate, a.w.k8, a.w.ks, reinterpret_cast<float*>(a.w.side),
                b % a.H, b / a.H, reinterpret_cast<float*>(tile));
  } else {
    tokq_rows(a.k, a.k_ss, a.k_sh, a.Sk, a.skp, a.H, a.rk, a.smooth_k ? a.w.kmean : nullptr, a.rotate, a.w.k8, a.w.ks,
              reinterpret_cast<float*>(a.w.side), b);
  }
}

// ------------------------------------------------------------------ main kernel
struct U8Args {
  const int8_t* q8;    // [H][Sqpad][128]
  const float* qs;     // [H][Sqpad]
  const int8_t* k8;    // [H][Skpad][128]
  const int8_t* side;  // [H][Skpad/128][2048 B]: (s, b) pairs, accumulator starts
  const int8_t* vt;    // [H][128][Skpad]
  const float* vscale;  // [H][128]
  const float* vmean;   // [H][128]
  uint16_t* out;
  int64_t o_ss, o_sh;
  int64_t Sq, Sk, Sqpad, Skpad;
  float scale_log2;
  int nbias;
  float bias_log2;
  int nqb;   // query blocks per head; item = h * nqb + qb (query blocks fastest)
  int* ctr;  // work counter, zero at launch: a starting workgroup takes item ctr++
};

// 4 waves (one per SIMD) of 32 queries, two workgroups on a CU: VALU and matrix work of a wave do not overlap, so what fills
// the matrix pipe during one workgroup's softmax is the other workgroup, which no barrier ties to it. (One workgroup of
// 8 waves, half of them held half a tile behind by its barriers, ran 384.8 us against 334.1 for 5,583 tokens x 24 heads,
// 4.49 against 4.27 ms for 22,332 and 43.9 against 43.1 ms for 72,216, same bits; its 256-query items also filled the last
// round worse.)
constexpr int U8_WAVES = 4, U8_NT = U8_WAVES * 64, U8_BQ = U8_WAVES * 32;

typedef __attribute__((address_space(3))) const v4i lds_v4i_u8;
typedef __attribute__((address_space(3))) const float lds_f32_u8;

// Tile j reads K(j), V^T(j) and its side record from ring slot j % 2 and first loads tile j + 1 into the other slot, whose
// last reads returned before the barrier that ended tile j - 1.
// A slot holds K: 128 keys x 128 B (chunk c of row r at c ^ ((r ^ (r >> 3)) & 7)), V^T: 128 channels x 128
// keys (the same swizzle), then the 2 KiB side record. Padded keys carry b = -inf, so every tile runs unmasked.
// BK (configs 60-61, attn_fwd6 :1786-1962): one K scale kb per 128-key tile (the first float of the side record)
// instead of the per-key pairs: the tile max is the integer max ti of the raw accumulators (keys past Sk forced to
// 1.5*2^23 - 2^22 first), cc = c kb, tv = (ti - 1.5*2^23) cc, n = max(m, tv), a = 2^(m - n), ts = 2^(tv - n),
// P = rint(2^(fma(acc bits, cc, fma(-ti bits, cc, log2 255)))); the P.V, row sums and fold are the same.
// MODE 2 (FP8 P.V, configs 50-56, attn_fwd5 :1563-1785): the per-key dequant of MODE 0, then per group of MAXG keys
// (64 or 128, the reference's tile) the group max updates the running max m exactly (O and l scaled by
// 2^((m_old - m) c) when it grows), P = 2^(fma(t, c, fma(-m, c, log2 448))) in e4m3 (v_cvt_pk_fp8_f32: OCP e4m3fn,
// round to nearest even), l += P unquantized, and O^T += V^T . P^T on v_mfma_scale_f32_32x32x64_f8f6f4 (e4m3 V
// from vq_tile<true>) straight into the fp32 accumulators: no per-tile fold.
template <int MODE, int MAXG = 128>
__global__ void __launch_bounds__(U8_NT, 2) attn_u8_kernel(const U8Args a) {
  constexpr bool BK = MODE == 1;
  constexpr int KB = TILE * D, VB = D * TILE, SLOT = KB + VB + SIDE;
  __shared__ __attribute__((aligned(16))) int8_t ring[2 * SLOT];
  // the workgroup runs the item it takes from one work counter when it starts (a fast XCD takes more; see the
  // launch), the (head, query block) pair h * nqb + qb. Per-XCD shares (claim_item) measured 1.6 % slower here
  // (180.3 vs 177.4 ms at C4), so this kernel keeps the single counter.
  __shared__ int item_s;
  if (threadIdx.x == 0) item_s = atomicAdd(a.ctr, 1);
  __syncthreads();
  const int item = __builtin_amdgcn_readfirstlane(item_s);
  if (item >= static_cast<int>(gridDim.y) * a.nqb) return;
  const int h = item / a.nqb, qb = item - h * a.nqb;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, g = lane >> 5;
  const int64_t q = static_cast<int64_t>(qb) * U8_BQ + wave * 32 + l32;
  const int ntiles = static_cast<int>(a.Skpad / TILE);

  // Q operands are padded to 128 queries; a workgroup's last rows may lie past them (computed on zero codes
  // with c = 0 and never stored)
  const bool qin = q < a.Sqpad;
  v4i qf[4];
  {
    const int8_t* qp = a.q8 + (static_cast<int64_t>(h) * a.Sqpad + q) * D + g * 16;
#pragma unroll
    for (int ds = 0; ds < 4; ++ds) qf[ds] = qin ? *reinterpret_cast<const v4i*>(qp + ds * 32) : v4i{0, 0, 0, 0};
  }
  const float c = (qin ? a.qs[static_cast<int64_t>(h) * a.Sqpad + q] : 0.0f) * a.scale_log2;
  const float ib = (a.nbias > 0 && c > 0.0f) ? a.bias_log2 / c : 0.0f;

  // global -> LDS copies (lane l of a wave writes LDS base + 16 l; the swizzle is applied on the global side): copy c of K
  // and of V^T fills rows 8 c .. 8 c + 7 of the slot, row 8 c + l / 8 stored with chunk l % 8 XOR (l / 8 ^ c) & 7; wave w takes
  // copies 4 w .. 4 w + 3 of each, whose lane offsets differ in the XOR with 16 i alone, and waves 0 and 1 a side half
  const int8_t* kbase = a.k8 + static_cast<int64_t>(h) * a.Skpad * D;
  const int8_t* vbase = a.vt + static_cast<int64_t>(h) * D * a.Skpad;
  const int8_t* sbase = a.side + static_cast<int64_t>(h) * ntiles * SIDE;
  const uint32_t sx = ((lane & 7) ^ (((lane >> 3) ^ (4 * wave)) & 7)) << 4;
  const uint32_t ko = (lane >> 3) * D + sx, vo = static_cast<uint32_t>((lane >> 3) * a.Skpad) + sx;
  const uint32_t ring_lds = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(ring));
  auto load_tile = [&](int j) __attribute__((always_inline)) {
    const uint32_t so = static_cast<uint32_t>(j & 1) * SLOT;
    j = min(j, ntiles - 1);  // clamped: a copy past the end lands unread
    const int8_t* kp = kbase + static_cast<int64_t>(j) * KB + wave * 4096;
    const int8_t* vp = vbase + static_cast<int64_t>(j) * TILE + static_cast<int64_t>(wave) * 32 * a.Skpad;
    const uint32_t kd = ring_lds + so + wave * 4096;
#pragma unroll
    for (int i = 0; i < 4; ++i) lds_dma16_s(kp + i * 1024, ko ^ (16 * i), kd + i * 1024);
#pragma unroll
    for (int i = 0; i < 4; ++i) lds_dma16_s(vp + static_cast<int64_t>(i) * 8 * a.Skpad, vo ^ (16 * i), kd + KB + i * 1024);
    if (wave < 2)
      lds_dma16_s(sbase + static_cast<int64_t>(j) * SIDE + wave * 1024, lane * 16, ring_lds + so + KB + VB + wave * 1024);
  };

  // lane parts of the LDS reads inside a slot. K fragment (kb, ds): row 32 kb + l32, chunk 2 ds + g, stored at
  // chunk ^ ((row ^ (row >> 3)) & 7) = (2 ds ^ 4 (kb & 1)) ^ y, y = (g ^ l32 ^ (l32 >> 3)) & 7: lane offsets
  // koff[ds ^ 2 (kb & 1)] plus the immediate 4096 kb. V^T fragment (db, kc) likewise, plus KB.
  uint32_t koff[4];
  {
    const int y = (g ^ l32 ^ (l32 >> 3)) & 7;
#pragma unroll
    for (int i = 0; i < 4; ++i) koff[i] = ring_lds + l32 * 128 + (((2 * i) ^ y) << 4);
  }
  // side record: pairs of keys 32 kb + 8 i + 4 g .. +3 at byte 8 key, accumulator starts of channels
  // 32 db + 8 i + 4 g .. +3 at SIDE_VINIT + 4 d
  const uint32_t soff = ring_lds + KB + VB + 32 * g;
  const uint32_t ioff = ring_lds + KB + VB + SIDE_VINIT + 16 * g;
  // MODE 2: the e4m3 V^T fragment (db, 64-key chunk cc) of lane (l32, g) is logical chunks 4 cc + 2 g + h (h = 0, 1)
  // of row 32 db + l32, stored at chunk ^ ((row ^ (row >> 3)) & 7) = (4 (cc ^ (db & 1)) + 2 g + h) ^ y2
  uint32_t voff8[2][2];
  {
    const int y2 = (l32 ^ (l32 >> 3)) & 7;
#pragma unroll
    for (int c2 = 0; c2 < 2; ++c2)
#pragma unroll
      for (int hh = 0; hh < 2; ++hh) voff8[c2][hh] = ring_lds + KB + l32 * 128 + (((4 * c2 + 2 * g + hh) ^ y2) << 4);
  }

  v16f o[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[i][r] = 0.0f;
  float mx = -INFINITY, lrow = 0.0f;
  v16i magic;
#pragma unroll
  for (int r = 0; r < 16; ++r) magic[r] = MAGIC_I;

  // S^T of tile j: lane (l32, g) of s[kb] holds query l32 and keys 32 kb + 8 (r / 4) + 4 g + r % 4
  v16i s[4];
  auto qk = [&](const int j) __attribute__((always_inline)) {
    const uint32_t so = static_cast<uint32_t>(j & 1) * SLOT;
    uint32_t ka[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) ka[i] = koff[i] + so;
    // key-block outer, so that block kb is complete while the MFMAs of block kb + 1 still run
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
      for (int ds = 0; ds < 4; ++ds) {
        const v4i kf = *reinterpret_cast<lds_v4i_u8*>(static_cast<uintptr_t>(ka[ds ^ (2 * (kb & 1))] + kb * 4096));
        s[kb] = __builtin_amdgcn_mfma_i32_32x32x32_i8(kf, qf[ds], ds == 0 ? magic : s[kb], 0, 0, 0);
      }
    read_ahead<16, 3>();
  };

  auto softmax_pv = [&](const int j) __attribute__((always_inline)) {
    const uint32_t so = static_cast<uint32_t>(j & 1) * SLOT;
    // exponent of P: 2^(fma(t, cx, bb)); u8: t the dequantized score, cx = c; BK: t the accumulator bits, cx = c kb
    float t[4][16];
    float cx, bb, al, ts;
    if constexpr (BK) {
      if ((j + 1) * TILE > a.Sk) {  // the ragged last tile (uniform branch): padded keys far below every score
#pragma unroll
        for (int kb = 0; kb < 4; ++kb)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            if (j * TILE + 32 * kb + 8 * (r >> 2) + 4 * g + (r & 3) >= a.Sk) s[kb][r] = MAGIC_I - (1 << 22);
      }
      int ti = s[0][0];
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int r = 0; r < 16; r += 2) ti = max(ti, max(s[kb][r], s[kb][r + 1]));
      {
        const auto sw = __builtin_amdgcn_permlane32_swap(ti, ti, false, false);
        ti = max(static_cast<int>(sw[0]), static_cast<int>(sw[1]));
      }
      const float kbv = *reinterpret_cast<lds_f32_u8*>(static_cast<uintptr_t>(ring_lds + KB + VB + so));
      cx = c * kbv;
      const float tif = __int_as_float(ti);
      const float tv = (tif - MAGIC_F) * cx;
      const float n = fmaxf(mx, tv);
      al = __builtin_amdgcn_exp2f(mx - n);
      ts = __builtin_amdgcn_exp2f(tv - n);
      mx = n;
      bb = fmaf(-tif, cx, LOG2_255);
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int r = 0; r < 16; ++r) t[kb][r] = __int_as_float(s[kb][r]);
    } else {
    // t = fma(1.5*2^23 + acc, s_key, b_key), in place over the accumulator registers
    float tm = -INFINITY;
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const v4i p01 = *reinterpret_cast<lds_v4i_u8*>(static_cast<uintptr_t>(soff + so + kb * 256 + i * 64));
        const v4i p23 = *reinterpret_cast<lds_v4i_u8*>(static_cast<uintptr_t>(soff + so + kb * 256 + i * 64 + 16));
        const float ps[4] = {__int_as_float(p01[0]), __int_as_float(p01[2]), __int_as_float(p23[0]),
                             __int_as_float(p23[2])};
        const float pb[4] = {__int_as_float(p01[1]), __int_as_float(p01[3]), __int_as_float(p23[1]),
                             __int_as_float(p23[3])};
#pragma unroll
        for (int e = 0; e < 4; ++e) t[kb][4 * i + e] = fmaf(__int_as_float(s[kb][4 * i + e]), ps[e], pb[e]);
      }
    if (a.nbias > j * TILE) {  // text bias on keys [0, nbias) (uniform branch)
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int key = j * TILE + 32 * kb + 8 * (r >> 2) + 4 * g + (r & 3);
          if (key < a.nbias) t[kb][r] = t[kb][r] + ib;
        }
    }
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
      for (int r = 0; r < 16; r += 2) tm = max3(tm, t[kb][r], t[kb][r + 1]);
    {
      const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_int(tm), __float_as_int(tm), false, false);
      tm = fmaxf(__int_as_float(sw[0]), __int_as_float(sw[1]));
    }
    const float n = fmaxf(mx, tm);
    al = __builtin_amdgcn_exp2f((mx - n) * c);
    ts = __builtin_amdgcn_exp2f((tm - n) * c);
    mx = n;
    bb = fmaf(-tm, c, LOG2_255);
    cx = c;
    }
    // P = sat_u8(rint(2^x)) with v_cvt_pk_u8_f32 (round to nearest even, saturating at 0 and 255: the
    // reference's cvt.pack.sat.u8 of __float2int_rn), four per word; the signed operand of the MFMA is P - 128
    uint32_t pw[4][4];
    uint32_t rs = 0;
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        uint32_t x = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e)
          x = __builtin_amdgcn_cvt_pk_u8_f32(__builtin_amdgcn_exp2f(fmaf(t[kb][4 * w + e], cx, bb)), e, x);
        rs = __builtin_amdgcn_udot4(x, 0x01010101u, rs, false);
        pw[kb][w] = x ^ 0x80808080u;
      }
    // l adds the integer row sum of P (the lane's 64 keys)
    lrow = fmaf(ts, static_cast<float>(rs), lrow * al);
    const float nm = -ts * MAGIC_F;
    uint32_t va[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) va[i] = koff[i] + so + KB;
    // O^T[d][query] += V^T . P^T per 32-channel block db, then the fold into fp32
#pragma unroll
    for (int db = 0; db < 4; ++db) {
      v16i acc;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const v4i st = *reinterpret_cast<lds_v4i_u8*>(static_cast<uintptr_t>(ioff + so + db * 128 + i * 32));
        acc[4 * i + 0] = st[0]; acc[4 * i + 1] = st[1]; acc[4 * i + 2] = st[2]; acc[4 * i + 3] = st[3];
      }
#pragma unroll
      for (int kc = 0; kc < 4; ++kc) {
        const v4i vf = *reinterpret_cast<lds_v4i_u8*>(static_cast<uintptr_t>(va[kc ^ (2 * (db & 1))] + db * 4096));
        v4i pf;
        pf[0] = pw[kc][0]; pf[1] = pw[kc][1]; pf[2] = pw[kc][2]; pf[3] = pw[kc][3];
        acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(vf, pf, acc, 0, 0, 0);
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) o[db][r] = fmaf(ts, __int_as_float(acc[r]), fmaf(o[db][r], al, nm));
    }
    // issue order: 8 of the 32 LDS reads (per block: 4 accumulator starts, 4 V^T fragments) first, then each
    // P.V MFMA followed by two more reads, so the reads run ahead of the MFMAs that consume them
    __builtin_amdgcn_sched_group_barrier(0x100, 8, 1);  // 0x100: LDS reads
#pragma unroll
    for (int i = 0; i < 12; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 1);  // 0x008: MFMA
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 1);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, 4, 1);
  };

  auto softmax_pv_f8 = [&](const int j) __attribute__((always_inline)) {
    const uint32_t so = static_cast<uint32_t>(j & 1) * SLOT;
    float t[4][16];
    // t of blocks kb0 .. kb1 - 1 (MAXG 64: per 64-key chunk, so that only one chunk's scores are live at a time)
    auto dequant = [&](const int kb0, const int kb1) __attribute__((always_inline)) {
#pragma unroll
    for (int kb = kb0; kb < kb1; ++kb)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const v4i p01 = *reinterpret_cast<lds_v4i_u8*>(static_cast<uintptr_t>(soff + so + kb * 256 + i * 64));
        const v4i p23 = *reinterpret_cast<lds_v4i_u8*>(static_cast<uintptr_t>(soff + so + kb * 256 + i * 64 + 16));
        const float ps[4] = {__int_as_float(p01[0]), __int_as_float(p01[2]), __int_as_float(p23[0]),
                             __int_as_float(p23[2])};
        const float pb[4] = {__int_as_float(p01[1]), __int_as_float(p01[3]), __int_as_float(p23[1]),
                             __int_as_float(p23[3])};
#pragma unroll
        for (int e = 0; e < 4; ++e) t[kb][4 * i + e] = fmaf(__int_as_float(s[kb][4 * i + e]), ps[e], pb[e]);
      }
    };
    if constexpr (MAXG == 128) dequant(0, 4);
    float bb = 0.0f;
#pragma unroll
    for (int cc = 0; cc < 2; ++cc) {
      if constexpr (MAXG == 64) dequant(2 * cc, 2 * cc + 2);
      if (MAXG == 64 || cc == 0) {
        float tm = -INFINITY;
#pragma unroll
        for (int kb = 2 * cc; kb < 2 * cc + MAXG / 32; ++kb)
#pragma unroll
          for (int r = 0; r < 16; r += 2) tm = max3(tm, t[kb][r], t[kb][r + 1]);
        {
          const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_int(tm), __float_as_int(tm), false, false);
          tm = fmaxf(__int_as_float(sw[0]), __int_as_float(sw[1]));
        }
        if (__builtin_amdgcn_ballot_w64(tm > mx) != 0) {  // a = 1 exactly on the rows whose max stays
          const float n = fmaxf(mx, tm);
          const float al = __builtin_amdgcn_exp2f((mx - n) * c);
          lrow = lrow * al;
#pragma unroll
          for (int db = 0; db < 4; ++db)
#pragma unroll
            for (int r = 0; r < 16; ++r) o[db][r] = o[db][r] * al;
          mx = n;
        }
        bb = fmaf(-mx, c, LOG2_448);
      }
      // P of the chunk's two 32-key blocks in e4m3, four per word: the B operand of the 64-deep MFMA
      v8i pf;
#pragma unroll
      for (int hb = 0; hb < 2; ++hb)
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          const int kb = 2 * cc + hb;
          const float p0 = __builtin_amdgcn_exp2f(fmaf(t[kb][4 * w + 0], c, bb));
          const float p1 = __builtin_amdgcn_exp2f(fmaf(t[kb][4 * w + 1], c, bb));
          const float p2 = __builtin_amdgcn_exp2f(fmaf(t[kb][4 * w + 2], c, bb));
          const float p3 = __builtin_amdgcn_exp2f(fmaf(t[kb][4 * w + 3], c, bb));
          lrow = lrow + (p0 + p1);
          lrow = lrow + (p2 + p3);
          uint32_t x = __builtin_amdgcn_cvt_pk_fp8_f32(p0, p1, 0, false);
          x = __builtin_amdgcn_cvt_pk_fp8_f32(p2, p3, x, true);
          pf[4 * hb + w] = static_cast<int>(x);
        }
#pragma unroll
      for (int db = 0; db < 4; ++db) {
        const uint32_t base = so + db * 4096;
        const v4i lo = *reinterpret_cast<lds_v4i_u8*>(static_cast<uintptr_t>(voff8[cc ^ (db & 1)][0] + base));
        const v4i hi = *reinterpret_cast<lds_v4i_u8*>(static_cast<uintptr_t>(voff8[cc ^ (db & 1)][1] + base));
        v8i vf;
        vf[0] = lo[0]; vf[1] = lo[1]; vf[2] = lo[2]; vf[3] = lo[3];
        vf[4] = hi[0]; vf[5] = hi[1]; vf[6] = hi[2]; vf[7] = hi[3];
        // cbsz / blgp type 0 = FP8 E4M3 for both operands; zero scale operands select the unscaled form
        o[db] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(vf, pf, o[db], 0, 0, 0, 0, 0, 0);
      }
    }
  };

  load_tile(0);
  // vmcnt(0) through the builtin, so the compiler also sees the Q loads above as complete and adds no wait of
  // its own inside the loop (gfx9 s_waitcnt: vmcnt[3:0] | expcnt[6:4] | lgkmcnt[11:8])
  __builtin_amdgcn_s_waitcnt(0x0f70);
  __syncthreads();
  for (int j = 0; j < ntiles; ++j) {
    load_tile(j + 1);
    qk(j);
    if constexpr (MODE == 2) softmax_pv_f8(j);
    else softmax_pv(j);
    // the copies of tile j + 1 have landed and every read of tile j has returned, for every wave past the barrier
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  }

  const float lt = lrow + __shfl_xor(lrow, 32, 64);
  const float il = 1.0f / lt;
  // The wave's 32 rows go through 8 KiB of the idle ring (row r at 256 r, 16-byte chunk c at c ^ (r & 15)), so that a store
  // instruction writes four whole rows; straight from the accumulators it writes 8 bytes to each of 32. Every wave is past
  // the last tile's barrier with no copy in flight; a wave's LDS accesses execute in order.
  const float* vs = a.vscale + h * D;
  const float* vm = a.vmean + h * D;
  const uint32_t st = ring_lds + wave * 8192;
#pragma unroll
  for (int db = 0; db < 4; ++db)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int d = db * 32 + 8 * i + 4 * g, cc = db * 4 + i;
      float4 s4 = *reinterpret_cast<const float4*>(vs + d);
      if constexpr (MODE == 2) {  // the e4m3 V codes were stretched by 448 / 127 (attn_int8.cu:2642)
        s4.x = s4.x * V_UNSTRETCH; s4.y = s4.y * V_UNSTRETCH; s4.z = s4.z * V_UNSTRETCH; s4.w = s4.w * V_UNSTRETCH;
      }
      const float4 m4 = *reinterpret_cast<const float4*>(vm + d);
      lds_write8(st + l32 * 256 + ((cc ^ (l32 & 15)) << 4) + 8 * g,
                 make_uint2(pack_bf2(fmaf(o[db][4 * i + 0] * il, s4.x, m4.x), fmaf(o[db][4 * i + 1] * il, s4.y, m4.y)),
                            pack_bf2(fmaf(o[db][4 * i + 2] * il, s4.z, m4.z), fmaf(o[db][4 * i + 3] * il, s4.w, m4.w))));
    }
  asm volatile("" ::: "memory");
  const int64_t q0 = static_cast<int64_t>(qb) * U8_BQ + wave * 32;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int r = 4 * i + (lane >> 4), cc = lane & 15;
    const v4i w = lds_read16(st + r * 256 + ((cc ^ (r & 15)) << 4));
    if (q0 + r < a.Sq) {   // two 8-byte stores, the alignment the entry points require of out
      uint2* op = reinterpret_cast<uint2*>(a.out + (q0 + r) * a.o_ss + static_cast<int64_t>(h) * a.o_sh + 8 * cc);
      op[0] = make_uint2(static_cast<uint32_t>(w[0]), static_cast<uint32_t>(w[1]));
      op[1] = make_uint2(static_cast<uint32_t>(w[2]), static_cast<uint32_t>(w[3]));
    }
  }
}

// ------------------------------------------------------------------ host
static_assert(TILE == attn_ws::BLK && SIDE == attn_ws::SIDE, "workspace layout constants");
inline int64_t padk(int64_t s) { return attn_ws::pad(s); }

int check_qkv_u8(const char* name, const uint16_t* q, int64_t q_ss, int64_t q_sh, const uint16_t* k, int64_t k_ss,
                 int64_t k_sh, const uint16_t* v, int64_t v_ss, int64_t v_sh, int64_t Sq, int64_t Sk, int64_t H) {
  RH3_REQUIRE(Sq > 0 && Sk > 0 && H > 0, "%s: sizes must be positive (Sq=%lld Sk=%lld H=%lld)", name, (long long)Sq,
              (long long)Sk, (long long)H);
  RH3_REQUIRE(H < 65536 && (Sq + U8_BQ - 1) / U8_BQ < (1ll << 31), "%s: grid too large", name);
  RH3_REQUIRE(padk(Sq) * H < (1ll << 31) && padk(Sk) * H < (1ll << 31), "%s: Spad * H must stay below 2^31", name);
  // the key-side pre-pass grids are (H, key blocks): at most 65,535 blocks of 128 keys
  RH3_REQUIRE(padk(Sk) / TILE < 65536, "%s: Sk=%lld exceeds the 8,388,480-key grid limit", name, (long long)Sk);
  RH3_REQUIRE(q && k && v, "%s: null q/k/v", name);
  RH3_REQUIRE(aligned16(q) && aligned16(k) && aligned16(v), "%s: q/k/v must be 16-byte aligned", name);
  RH3_REQUIRE(q_ss % 8 == 0 && q_sh % 8 == 0 && k_ss % 8 == 0 && k_sh % 8 == 0 && v_ss % 8 == 0 && v_sh % 8 == 0,
              "%s: token/head strides must be multiples of 8 elements", name);
  return RH3_OK;
}

int check_rr_u8(const char* name, const uint16_t* tab, int rot, const uint16_t* qw, const uint16_t* kw) {
  RH3_REQUIRE(tab && qw && kw, "%s: tab, qw and kw are required", name);
  RH3_REQUIRE(rot == 96 || rot == 128, "%s: rot_dim %d (96 or 128 supported)", name, rot);
  RH3_REQUIRE(aligned16(tab) && aligned16(qw) && aligned16(kw), "%s: tab/qw/kw must be 16-byte aligned", name);
  return RH3_OK;
}

// workgroups of the K quantizer
template <bool BLK>
int64_t k_blocks(const PreU8& a) { return BLK ? a.skp / TILE * a.H : tokq_blocks(a.skp, a.H); }

// the merged launches are one-dimensional
template <bool BLK>
int check_grids(const PreU8& a, const char* name) {
  const int64_t ga = static_cast<int64_t>(a.nchunk) * a.H * (a.smooth_k ? 2 : 1) + (a.q ? tokq_blocks(a.sqp, a.H) : 0);
  const int64_t gb = k_blocks<BLK>(a) + a.skp / TILE * a.H;
  RH3_REQUIRE(ga <= MAX_GRID_256 && gb <= MAX_GRID_256, "%s: Sq=%lld Sk=%lld H=%d needs %lld workgroups, beyond the grid limit",
              name, (long long)a.Sq, (long long)a.Sk, a.H, (long long)(ga > gb ? ga : gb));
  return RH3_OK;
}

// the second level of the statistics, then the K quantizer and the V codes
template <bool F8, bool BLK>
int prepass_tail(PreU8& a, hipStream_t st, const char* name) {
  if (int e = check_grids<BLK>(a, name)) return e;
  hipLaunchKernelGGL(kmean_vfinal_kernel, dim3(a.H, 2), dim3(KMEAN_NT), 0, st, a.w, a.nchunk, a.Sk, a.smooth_k, a.smooth_v);
  const unsigned tiles = static_cast<unsigned>(a.skp / TILE * a.H);
  a.nk = static_cast<unsigned>(k_blocks<BLK>(a));
  hipLaunchKernelGGL((pre_b_u8_kernel<F8, BLK>), dim3(a.nk + tiles), dim3(256), 0, st, a);
  return launch_status(name);
}
template <bool F8, bool BLK>
int prepass_all(PreU8& a, hipStream_t st, const char* name) {
  if (int e = check_grids<BLK>(a, name)) return e;
  const unsigned chunks = static_cast<unsigned>(a.nchunk) * a.H;
  a.nk = a.smooth_k ? chunks : 0;
  a.nv = chunks;
  hipLaunchKernelGGL(pre_a_u8_kernel, dim3(a.nk + a.nv + tokq_blocks(a.sqp, a.H)), dim3(256), 0, st, a);
  return prepass_tail<F8, BLK>(a, st, name);
}

int prepass_u8(const uint16_t* q, int64_t q_ss, int64_t q_sh, const uint16_t* k, int64_t k_ss, int64_t k_sh,
               const uint16_t* v, int64_t v_ss, int64_t v_sh, int64_t Sq, int64_t Sk, int64_t H, const RR& rq,
               const RR& rk, int smooth_k, int smooth_v, int rotate, const WorkU8& w, hipStream_t st,
               bool f8 = false) {
  PreU8 a{q, k, v, q_ss, q_sh, k_ss, k_sh, v_ss, v_sh, Sq, Sk, padk(Sq), padk(Sk), static_cast<int>(H),
          static_cast<int>(attn_ws::nchunks(Sk)), smooth_k, smooth_v, rotate, rq, rk, w, 0, 0};
  // configs 50-56: e4m3 V codes (attn_int8.cu:2639-2642)
  return f8 ? prepass_all<true, false>(a, st, "attention_u8 prepass") : prepass_all<false, false>(a, st, "attention_u8 prepass");
}

// Grid of the main kernel, whose workgroups take their (head, query block) items from a work counter: the grid is
// dealt to the XCDs in fixed shares and the XCDs run at different clocks, so the grid holds a quarter more
// workgroups than items (room for the fastest XCD to take a quarter more than its share); the extra ones return
// at once. gridDim.y carries H. The counter is cleared first by a fill kernel (no hipMemsetAsync: graph-safe), unless the
// pre-pass of the same call just did.
dim3 claim_grid(U8Args& f, const WorkU8& w, int64_t Sq, int64_t H, hipStream_t st, bool cleared) {
  f.nqb = static_cast<int>((Sq + U8_BQ - 1) / U8_BQ);
  f.ctr = w.ctr;
  const int64_t per_head = f.nqb + (f.nqb + 3) / 4;
  if (!cleared) hipLaunchKernelGGL(zero_kernel, dim3(1), dim3(64), 0, st, reinterpret_cast<float*>(w.ctr), int64_t{1});
  return dim3(static_cast<uint32_t>(per_head), static_cast<uint32_t>(H));
}

// configs 50-56: the FP8 P.V main kernel; tile = the reference's BN (64 or 128 keys per running-max update)
int forward_f8(const WorkU8& w, int64_t Sq, int64_t Sk, int64_t H, float scale, int tile, uint16_t* out, int64_t o_ss,
               int64_t o_sh, hipStream_t st, bool cleared = false) {
  U8Args f{w.q8, w.qs, w.k8, w.side, w.vt, w.vscale, w.vmean, out, o_ss, o_sh, Sq, Sk, padk(Sq), padk(Sk),
           scale * 1.4426950408889634f, 0, 0.0f};
  const dim3 grid = claim_grid(f, w, Sq, H, st, cleared);  // sets f.nqb and f.ctr: before f is passed
  if (tile == 64) hipLaunchKernelGGL((attn_u8_kernel<2, 64>), grid, dim3(U8_NT), 0, st, f);
  else hipLaunchKernelGGL((attn_u8_kernel<2, 128>), grid, dim3(U8_NT), 0, st, f);
  return launch_status("attention_f8 forward");
}

int forward_u8(const WorkU8& w, int64_t Sq, int64_t Sk, int64_t H, float scale, int nbias, double bias, uint16_t* out,
               int64_t o_ss, int64_t o_sh, hipStream_t st, bool cleared = false) {
  U8Args f{w.q8, w.qs, w.k8, w.side, w.vt, w.vscale, w.vmean, out, o_ss, o_sh, Sq, Sk, padk(Sq), padk(Sk),
           scale * 1.4426950408889634f, nbias, static_cast<float>(bias * 1.4426950408889634)};
  const dim3 grid = claim_grid(f, w, Sq, H, st, cleared);  // sets f.nqb and f.ctr: before f is passed
  hipLaunchKernelGGL(attn_u8_kernel<0>, grid, dim3(U8_NT), 0, st, f);
  return launch_status("attention_u8 forward");
}

// configs 60-61: Q per token as prepass_u8 (no RMSNorm + RoPE: the reference has none for these configs), K one
// scale per 128-key block after the smoothing and the optional H128 (into ks [H][Skpad/128] and the side records),
// V as prepass_u8 (attn_int8.cu:2618-2641)
int prepass_bk(const uint16_t* q, int64_t q_ss, int64_t q_sh, const uint16_t* k, int64_t k_ss, int64_t k_sh,
               const uint16_t* v, int64_t v_ss, int64_t v_sh, int64_t Sq, int64_t Sk, int64_t H, int smooth_k,
               int smooth_v, int rotate, const WorkU8& w, hipStream_t st) {
  const RR none{nullptr, nullptr, 0.f, 0};
  PreU8 a{q, k, v, q_ss, q_sh, k_ss, k_sh, v_ss, v_sh, Sq, Sk, padk(Sq), padk(Sk), static_cast<int>(H),
          static_cast<int>(attn_ws::nchunks(Sk)), smooth_k, smooth_v, rotate, none, none, w, 0, 0};
  return prepass_all<false, true>(a, st, "attention_bk prepass");
}

int forward_bk(const WorkU8& w, int64_t Sq, int64_t Sk, int64_t H, float scale, uint16_t* out, int64_t o_ss,
               int64_t o_sh, hipStream_t st, bool cleared = false) {
  U8Args f{w.q8, w.qs, w.k8, w.side, w.vt, w.vscale, w.vmean, out, o_ss, o_sh, Sq, Sk, padk(Sq), padk(Sk),
           scale * 1.4426950408889634f, 0, 0.0f};
  const dim3 grid = claim_grid(f, w, Sq, H, st, cleared);  // sets f.nqb and f.ctr: before f is passed
  hipLaunchKernelGGL(attn_u8_kernel<1>, grid, dim3(U8_NT), 0, st, f);
  return launch_status("attention_bk forward");
}

int check_out_u8(const char* name, const uint16_t* out, int64_t o_ss, int64_t o_sh) {
  RH3_REQUIRE(out && (reinterpret_cast<uintptr_t>(out) & 7) == 0 && o_ss % 4 == 0 && o_sh % 4 == 0,
              "%s: out must be 8-byte aligned with strides multiple of 4", name);
  return RH3_OK;
}

int check_bias_u8(const char* name, int nbias, int64_t Sk) {
  RH3_REQUIRE(nbias >= 0 && nbias <= Sk, "%s: nbias %d outside [0, Sk=%lld]", name, nbias, (long long)Sk);
  return RH3_OK;
}

}  // namespace
}  // namespace rh3

using namespace rh3;

extern "C" int rh3_attention_workspace_layout(int numerics, int64_t Sq, int64_t Sk, int64_t H, int64_t* offsets) {
  clear_error();
  RH3_REQUIRE(Sq > 0 && Sk > 0 && H > 0 && offsets, "attention_workspace_layout: sizes must be positive, offsets set");
  char* const b = reinterpret_cast<char*>(static_cast<uintptr_t>(256));  // any aligned base; offsets relative
  auto off = [&](const void* p) { return static_cast<int64_t>(static_cast<const char*>(p) - b); };
  if (numerics == 0) {
    const attn_ws::Work w = attn_ws::layout(b, Sq, Sk, H);
    const void* ps[8] = {w.q8, w.qs, w.k8, w.ks, w.kmean, w.part, w.vt, w.kn};
    for (int i = 0; i < 8; ++i) offsets[i] = off(ps[i]);
    offsets[8] = w.bytes;
    return RH3_OK;
  }
  RH3_REQUIRE(numerics == 1, "attention_workspace_layout: numerics %d (0 per-block, 1 production)", numerics);
  const WorkU8 w = layout_u8(b, Sq, Sk, H);
  const void* ps[13] = {w.q8, w.qs, w.k8, w.ks, w.side, w.vt, w.kmean, w.vmean, w.vscale,
                        w.kpart, w.vsum, w.vmax, w.vmin};
  for (int i = 0; i < 13; ++i) offsets[i] = off(ps[i]);
  offsets[13] = w.bytes;
  return RH3_OK;
}

extern "C" int64_t rh3_attention_u8_workspace_bytes(int64_t Sq, int64_t Sk, int64_t H) {
  if (Sq <= 0 || Sk <= 0 || H <= 0) return 0;
  return layout_u8(nullptr, Sq, Sk, H).bytes;
}

extern "C" int rh3_attention_u8_prepass(const uint16_t* q, int64_t q_ss, int64_t q_sh, const uint16_t* k,
                                        int64_t k_ss, int64_t k_sh, const uint16_t* v, int64_t v_ss, int64_t v_sh,
                                        int64_t Sq, int64_t Sk, int64_t H, const uint16_t* tab, int rot,
                                        const uint16_t* qw, const uint16_t* kw, float eps, int smooth_k, int smooth_v,
                                        int rotate, void* workspace, int64_t workspace_bytes, void** ptrs,
                                        hipStream_t stream) {
  clear_error();
  if (int e = check_qkv_u8("attention_u8_prepass", q, q_ss, q_sh, k, k_ss, k_sh, v, v_ss, v_sh, Sq, Sk, H)) return e;
  RH3_REQUIRE(ptrs, "attention_u8_prepass: ptrs required");
  const WorkU8 w = layout_u8(workspace, Sq, Sk, H);
  RH3_REQUIRE(workspace && aligned16(workspace) && workspace_bytes >= w.bytes,
              "attention_u8_prepass: workspace %lld bytes < required %lld", (long long)workspace_bytes,
              (long long)w.bytes);
  RR rq{nullptr, nullptr, 0.f, 0}, rk{nullptr, nullptr, 0.f, 0};
  if (tab) {
    if (int e = check_rr_u8("attention_u8_prepass", tab, rot, qw, kw)) return e;
    RH3_REQUIRE(Sq == Sk, "attention_u8_prepass: RMSNorm+RoPE needs self-attention (Sq == Sk)");
    rq = RR{tab, qw, eps, rot};
    rk = RR{tab, kw, eps, rot};
  }
  if (int e = prepass_u8(q, q_ss, q_sh, k, k_ss, k_sh, v, v_ss, v_sh, Sq, Sk, H, rq, rk, smooth_k, smooth_v, rotate,
                         w, stream))
    return e;
  ptrs[0] = w.q8; ptrs[1] = w.qs; ptrs[2] = w.k8; ptrs[3] = w.ks; ptrs[4] = w.side; ptrs[5] = w.vt;
  ptrs[6] = w.kmean; ptrs[7] = w.vscale; ptrs[8] = w.vmean;
  return RH3_OK;
}

extern "C" int rh3_attention_u8_prepass_qkv(const uint16_t* k, int64_t k_ss, int64_t k_sh, const uint16_t* v,
                                            int64_t v_ss, int64_t v_sh, int64_t S, int64_t H, const uint16_t* tab,
                                            int rot, const uint16_t* kw, float eps, int smooth_k, int smooth_v,
                                            int rotate, void* workspace, int64_t workspace_bytes, void** ptrs,
                                            hipStream_t stream) {
  clear_error();
  if (int e = check_qkv_u8("attention_u8_prepass_qkv", k, k_ss, k_sh, k, k_ss, k_sh, v, v_ss, v_sh, S, S, H)) return e;
  RH3_REQUIRE(ptrs, "attention_u8_prepass_qkv: ptrs required");
  const WorkU8 w = layout_u8(workspace, S, S, H);
  RH3_REQUIRE(workspace && aligned16(workspace) && workspace_bytes >= w.bytes,
              "attention_u8_prepass_qkv: workspace %lld bytes < required %lld", (long long)workspace_bytes,
              (long long)w.bytes);
  RR rk{nullptr, nullptr, 0.f, 0};
  if (tab) {
    RH3_REQUIRE(kw && (rot == 96 || rot == 128) && aligned16(tab) && aligned16(kw),
                "attention_u8_prepass_qkv: kw (16-byte aligned) and rot_dim 96 or 128 required with tab");
    rk = RR{tab, kw, eps, rot};
  }
  // q8, qs and the K / V channel statistics come from rh3_gemm_i8_qkv (numerics 1) on this workspace
  PreU8 a{nullptr, k, v, 0, 0, k_ss, k_sh, v_ss, v_sh, S, S, padk(S), padk(S), static_cast<int>(H),
          static_cast<int>(attn_ws::nchunks(S)), smooth_k, smooth_v, rotate, rk, rk, w, 0, 0};
  if (int e = prepass_tail<false, false>(a, stream, "attention_u8 prepass_qkv")) return e;
  ptrs[0] = w.q8; ptrs[1] = w.qs; ptrs[2] = w.k8; ptrs[3] = w.ks; ptrs[4] = w.side; ptrs[5] = w.vt;
  ptrs[6] = w.kmean; ptrs[7] = w.vscale; ptrs[8] = w.vmean;
  return RH3_OK;
}

extern "C" int rh3_attention_u8_forward(int64_t Sq, int64_t Sk, int64_t H, float scale, int nbias, double bias,
                                        uint16_t* out, int64_t o_ss, int64_t o_sh, void* workspace,
                                        int64_t workspace_bytes, hipStream_t stream) {
  clear_error();
  RH3_REQUIRE(Sq > 0 && Sk > 0 && H > 0, "attention_u8_forward: sizes must be positive");
  if (int e = check_out_u8("attention_u8_forward", out, o_ss, o_sh)) return e;
  if (int e = check_bias_u8("attention_u8_forward", nbias, Sk)) return e;
  const WorkU8 w = layout_u8(workspace, Sq, Sk, H);
  RH3_REQUIRE(workspace && aligned16(workspace) && workspace_bytes >= w.bytes,
              "attention_u8_forward: workspace %lld bytes < required %lld", (long long)workspace_bytes,
              (long long)w.bytes);
  return forward_u8(w, Sq, Sk, H, scale, nbias, bias, out, o_ss, o_sh, stream);
}

extern "C" int rh3_int8_attention_u8(const uint16_t* q, int64_t q_ss, int64_t q_sh, const uint16_t* k, int64_t k_ss,
                                     int64_t k_sh, const uint16_t* v, int64_t v_ss, int64_t v_sh, int64_t Sq,
                                     int64_t Sk, int64_t H, const uint16_t* tab, int rot, const uint16_t* qw,
                                     const uint16_t* kw, float eps, float scale, int nbias, double bias, int smooth_k,
                                     int smooth_v, int rotate, uint16_t* out, int64_t o_ss, int64_t o_sh,
                                     void* workspace, int64_t workspace_bytes, hipStream_t stream) {
  clear_error();
  if (int e = check_qkv_u8("int8_attention_u8", q, q_ss, q_sh, k, k_ss, k_sh, v, v_ss, v_sh, Sq, Sk, H)) return e;
  if (int e = check_out_u8("int8_attention_u8", out, o_ss, o_sh)) return e;
  if (int e = check_bias_u8("int8_attention_u8", nbias, Sk)) return e;
  const WorkU8 w = layout_u8(workspace, Sq, Sk, H);
  RH3_REQUIRE(workspace && aligned16(workspace) && workspace_bytes >= w.bytes,
              "int8_attention_u8: workspace %lld bytes < required %lld", (long long)workspace_bytes,
              (long long)w.bytes);
  RR rq{nullptr, nullptr, 0.f, 0}, rk{nullptr, nullptr, 0.f, 0};
  if (tab) {
    if (int e = check_rr_u8("int8_attention_u8", tab, rot, qw, kw)) return e;
    RH3_REQUIRE(Sq == Sk, "int8_attention_u8: RMSNorm+RoPE needs self-attention (Sq == Sk)");
    rq = RR{tab, qw, eps, rot};
    rk = RR{tab, kw, eps, rot};
  }
  if (int e = prepass_u8(q, q_ss, q_sh, k, k_ss, k_sh, v, v_ss, v_sh, Sq, Sk, H, rq, rk, smooth_k, smooth_v, rotate,
                         w, stream))
    return e;
  return forward_u8(w, Sq, Sk, H, scale, nbias, bias, out, o_ss, o_sh, stream, true);
}

extern "C" int rh3_attention_bk_prepass(const uint16_t* q, int64_t q_ss, int64_t q_sh, const uint16_t* k,
                                        int64_t k_ss, int64_t k_sh, const uint16_t* v, int64_t v_ss, int64_t v_sh,
                                        int64_t Sq, int64_t Sk, int64_t H, int smooth_k, int smooth_v, int rotate,
                                        void* workspace, int64_t workspace_bytes, void** ptrs, hipStream_t stream) {
  clear_error();
  if (int e = check_qkv_u8("attention_bk_prepass", q, q_ss, q_sh, k, k_ss, k_sh, v, v_ss, v_sh, Sq, Sk, H)) return e;
  RH3_REQUIRE(ptrs, "attention_bk_prepass: ptrs required");
  const WorkU8 w = layout_u8(workspace, Sq, Sk, H);
  RH3_REQUIRE(workspace && aligned16(workspace) && workspace_bytes >= w.bytes,
              "attention_bk_prepass: workspace %lld bytes < required %lld", (long long)workspace_bytes,
              (long long)w.bytes);
  if (int e = prepass_bk(q, q_ss, q_sh, k, k_ss, k_sh, v, v_ss, v_sh, Sq, Sk, H, smooth_k, smooth_v, rotate, w, stream))
    return e;
  ptrs[0] = w.q8; ptrs[1] = w.qs; ptrs[2] = w.k8; ptrs[3] = w.ks; ptrs[4] = w.side; ptrs[5] = w.vt;
  ptrs[6] = w.kmean; ptrs[7] = w.vscale; ptrs[8] = w.vmean;
  return RH3_OK;
}

extern "C" int rh3_attention_bk_forward(int64_t Sq, int64_t Sk, int64_t H, float scale, uint16_t* out, int64_t o_ss,
                                        int64_t o_sh, void* workspace, int64_t workspace_bytes, hipStream_t stream) {
  clear_error();
  RH3_REQUIRE(Sq > 0 && Sk > 0 && H > 0, "attention_bk_forward: sizes must be positive");
  if (int e = check_out_u8("attention_bk_forward", out, o_ss, o_sh)) return e;
  const WorkU8 w = layout_u8(workspace, Sq, Sk, H);
  RH3_REQUIRE(workspace && aligned16(workspace) && workspace_bytes >= w.bytes,
              "attention_bk_forward: workspace %lld bytes < required %lld", (long long)workspace_bytes,
              (long long)w.bytes);
  return forward_bk(w, Sq, Sk, H, scale, out, o_ss, o_sh, stream);
}

extern "C" int rh3_int8_attention_bk(const uint16_t* q, int64_t q_ss, int64_t q_sh, const uint16_t* k, int64_t k_ss,
                                     int64_t k_sh, const uint16_t* v, int64_t v_ss, int64_t v_sh, int64_t Sq,
                                     int64_t Sk, int64_t H, float scale, int smooth_k, int smooth_v, int rotate,
                                     uint16_t* out, int64_t o_ss, int64_t o_sh, void* workspace,
                                     int64_t workspace_bytes, hipStream_t stream) {
  clear_error();
  if (int e = check_qkv_u8("int8_attention_bk", q, q_ss, q_sh, k, k_ss, k_sh, v, v_ss, v_sh, Sq, Sk, H)) return e;
  if (int e = check_out_u8("int8_attention_bk", out, o_ss, o_sh)) return e;
  const WorkU8 w = layout_u8(workspace, Sq, Sk, H);
  RH3_REQUIRE(workspace && aligned16(workspace) && workspace_bytes >= w.bytes,
              "int8_attention_bk: workspace %lld bytes < required %lld", (long long)workspace_bytes,
              (long long)w.bytes);
  if (int e = prepass_bk(q, q_ss, q_sh, k, k_ss, k_sh, v, v_ss, v_sh, Sq, Sk, H, smooth_k, smooth_v, rotate, w, stream))
    return e;
  return forward_bk(w, Sq, Sk, H, scale, out, o_ss, o_sh, stream, true);
}

extern "C" int rh3_attention_f8_prepass(const uint16_t* q, int64_t q_ss, int64_t q_sh, const uint16_t* k,
                                        int64_t k_ss, int64_t k_sh, const uint16_t* v, int64_t v_ss, int64_t v_sh,
                                        int64_t Sq, int64_t Sk, int64_t H, const uint16_t* tab, int rot,
                                        const uint16_t* qw, const uint16_t* kw, float eps, int smooth_k, int smooth_v,
                                        int rotate, void* workspace, int64_t workspace_bytes, void** ptrs,
                                        hipStream_t stream) {
  clear_error();
  if (int e = check_qkv_u8("attention_f8_prepass", q, q_ss, q_sh, k, k_ss, k_sh, v, v_ss, v_sh, Sq, Sk, H)) return e;
  RH3_REQUIRE(ptrs, "attention_f8_prepass: ptrs required");
  const WorkU8 w = layout_u8(workspace, Sq, Sk, H);
  RH3_REQUIRE(workspace && aligned16(workspace) && workspace_bytes >= w.bytes,
              "attention_f8_prepass: workspace %lld bytes < required %lld", (long long)workspace_bytes,
              (long long)w.bytes);
  RR rq{nullptr, nullptr, 0.f, 0}, rk{nullptr, nullptr, 0.f, 0};
  if (tab) {
    if (int e = check_rr_u8("attention_f8_prepass", tab, rot, qw, kw)) return e;
    RH3_REQUIRE(Sq == Sk, "attention_f8_prepass: RMSNorm+RoPE needs self-attention (Sq == Sk)");
    rq = RR{tab, qw, eps, rot};
    rk = RR{tab, kw, eps, rot};
  }
  if (int e = prepass_u8(q, q_ss, q_sh, k, k_ss, k_sh, v, v_ss, v_sh, Sq, Sk, H, rq, rk, smooth_k, smooth_v, rotate,
                         w, stream, true))
    return e;
  ptrs[0] = w.q8; ptrs[1] = w.qs; ptrs[2] = w.k8; ptrs[3] = w.ks; ptrs[4] = w.side; ptrs[5] = w.vt;
  ptrs[6] = w.kmean; ptrs[7] = w.vscale; ptrs[8] = w.vmean;
  return RH3_OK;
}

extern "C" int rh3_attention_f8_forward(int64_t Sq, int64_t Sk, int64_t H, float scale, int tile, uint16_t* out,
                                        int64_t o_ss, int64_t o_sh, void* workspace, int64_t workspace_bytes,
                                        hipStream_t stream) {
  clear_error();
  RH3_REQUIRE(Sq > 0 && Sk > 0 && H > 0, "attention_f8_forward: sizes must be positive");
  RH3_REQUIRE(tile == 64 || tile == 128, "attention_f8_forward: tile %d (64 or 128 keys)", tile);
  if (int e = check_out_u8("attention_f8_forward", out, o_ss, o_sh)) return e;
  const WorkU8 w = layout_u8(workspace, Sq, Sk, H);
  RH3_REQUIRE(workspace && aligned16(workspace) && workspace_bytes >= w.bytes,
              "attention_f8_forward: workspace %lld bytes < required %lld", (long long)workspace_bytes,
              (long long)w.bytes);
  return forward_f8(w, Sq, Sk, H, scale, tile, out, o_ss, o_sh, stream);
}

extern "C" int rh3_int8_attention_f8(const uint16_t* q, int64_t q_ss, int64_t q_sh, const uint16_t* k, int64_t k_ss,
                                     int64_t k_sh, const uint16_t* v, int64_t v_ss, int64_t v_sh, int64_t Sq,
                                     int64_t Sk, int64_t H, const uint16_t* tab, int rot, const uint16_t* qw,
                                     const uint16_t* kw, float eps, float scale, int tile, int smooth_k, int smooth_v,
                                     int rotate, uint16_t* out, int64_t o_ss, int64_t o_sh, void* workspace,
                                     int64_t workspace_bytes, hipStream_t stream) {
  void* ptrs[9];
  if (int e = rh3_attention_f8_prepass(q, q_ss, q_sh, k, k_ss, k_sh, v, v_ss, v_sh, Sq, Sk, H, tab, rot, qw, kw, eps,
                                       smooth_k, smooth_v, rotate, workspace, workspace_bytes, ptrs, stream))
    return e;
  return rh3_attention_f8_forward(Sq, Sk, H, scale, tile, out, o_ss, o_sh, workspace, workspace_bytes, stream);
}
