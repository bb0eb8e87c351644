// Small-tile forms of the GEMM (gemm.hip) for calls whose 256 x 256 tiles would leave CUs without work: the same
// operands, epilogues and arithmetic, so the same bits: int32 accumulators are exact in any order, and an e4m3 call adds
// its k-steps one after the other on every tile (KG 1), so a row's result does not depend on the rows beside it.
#include "gemm_common.hpp"

namespace rh3 {
namespace gemm {
namespace {

// TM x TN outputs per workgroup, KG groups of WGM x WGN waves. Group kg runs its share of the k-steps on the whole
// tile through a ring of its own (NST stages of (TM + TN) x 64 bytes); with KG = 2 (int8) the two groups' accumulators are
// added through LDS before the epilogue, each group finishing half of the tile's rows.
template <int TM_, int TN_, int WGM_, int WGN_, int KG_, int NST_>
struct Tile {
  static constexpr int TM = TM_, TN = TN_, WGM = WGM_, WGN = WGN_, KG = KG_, NST = NST_;
  static constexpr int NWG = WGM * WGN, NW = NWG * KG, NT = 64 * NW;
  static constexpr int WM = TM / WGM, WN = TN / WGN, TI = WN / 32, TJ = WM / 32;
  static constexpr int STAGE = (TM + TN) * BK;
  static constexpr int LOADS = (TM + TN) / 16;             // 1 KiB copies per stage
  static constexpr int LW = (LOADS + NWG - 1) / NWG;       // per wave (the last may be short of one)
  static constexpr int RING = KG * NST * STAGE;
  static constexpr int XCHG = KG > 1 ? TM * TN * 4 : 0;    // accumulators handed to the other group
  static constexpr int LDS = RING > XCHG + NW * 2048 ? RING : XCHG + NW * 2048;
  static_assert(WM % 32 == 0 && WN % 32 == 0 && (KG == 1 || TJ % 2 == 0), "wave tile");
  static_assert(LDS + (TM + 2 * TN) * 4 <= 160 * 1024, "LDS");
};

template <int N>
__device__ __forceinline__ void wait_vm_lds() {  // at most N vector memory operations in flight, every LDS read done
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
}

// A 16-pass MFMA (e4m3) needs 20 wait states before its result is read; hipcc (ROCm 7.2) looks back over 19 and can leave a
// read exactly there, which then finds the register of before. Called after the last MFMAs of a path to the epilogue.
__device__ __forceinline__ void mfma_settle() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_nop 15\n\ts_nop 3");
  __builtin_amdgcn_sched_barrier(0);
}

template <bool FP8, int EPI, typename T>
__global__ void __launch_bounds__(T::NT, T::NT == 256 ? 2 : T::NW / 4) gemm_tile_kernel(const GemmArgs a) {
  using MM = Mma<FP8>;
  using acc_t = typename MM::acc_t;
  static_assert(!FP8 || T::KG == 1, "an fp32 sum keeps its order");
  constexpr int TM = T::TM, TN = T::TN, TI = T::TI, TJ = T::TJ, WM = T::WM, WN = T::WN, NST = T::NST, LW = T::LW;
  __shared__ __attribute__((aligned(16))) int8_t ring[T::LDS];
  __shared__ __attribute__((aligned(16))) float rec[TM + 2 * TN];  // xs, ws, bias / gate of the tile

  // tile order as in gemm.hip: XCD x (workgroup b runs on XCD b % 8) takes a contiguous range of the grouped order
  const int nb = a.tiles_m * a.tiles_n, b = blockIdx.x, xcd = b % 8;
  const int lt = xcd * (nb / 8) + min(xcd, nb % 8) + b / 8;
  constexpr int GM = 4;
  const int group = lt / (GM * a.tiles_n), first_m = group * GM;
  const int gsz = min(a.tiles_m - first_m, GM);
  const int64_t m0 = static_cast<int64_t>(first_m + (lt % (GM * a.tiles_n)) % gsz) * TM;
  const int64_t n0 = static_cast<int64_t>((lt % (GM * a.tiles_n)) / gsz) * TN;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kg = wave / T::NWG, wg = wave % T::NWG;
  const int wm = wg / T::WGN, wn = wg % T::WGN;
  const int l32 = lane & 31, g = lane >> 5;

  // the tile's scales (and bias / gate), parked in LDS at the end of the k-loop
  constexpr int NREC = (TM + 2 * TN + T::NT - 1) / T::NT;
  constexpr bool HAS_BG = EPI == EPI_PLAIN || EPI == EPI_GATED;
  const uint16_t* bg = EPI == EPI_GATED ? a.gate : a.bias;
  float rv[NREC];
  if constexpr (EPI != EPI_ACC) {
#pragma unroll
    for (int i = 0; i < NREC; ++i) {
      const int p = i * T::NT + tid;
      rv[i] = 0.0f;
      if (p < TM) {
        if (m0 + p < a.M) rv[i] = a.xs[m0 + p];
      } else if (p < TM + TN) {
        if (n0 + (p - TM) < a.N) rv[i] = a.ws[n0 + (p - TM)];
      } else if (p < TM + 2 * TN) {
        if (HAS_BG && bg && n0 + (p - TM - TN) < a.N) rv[i] = bf2f(bg[n0 + (p - TM - TN)]);
      }
    }
  }

  // global -> LDS copies: copy li of a stage fills its bytes [1024 li, 1024 li + 1024), rows 16 li .. 16 li + 15 of
  // the concatenated (x, w) tile rows; lane l holds row 16 li + l / 4, stored chunk l % 4 (the XOR swizzle applied on
  // the global side). Rows past the operand read its last row.
  const int8_t* const xb = a.x + m0 * a.ldx;
  const int8_t* const wb = a.w + n0 * a.ldw;
  const int rmx = static_cast<int>(min<int64_t>(TM - 1, a.M - 1 - m0));
  const int rmw = static_cast<int>(min<int64_t>(TN - 1, a.N - 1 - n0));
  uint32_t off[LW];
#pragma unroll
  for (int t = 0; t < LW; ++t) {
    const int li = min(t * T::NWG + wg, T::LOADS - 1), r = 16 * li + (lane >> 2);
    const int c = (lane & 3) ^ (((r >> 1) & 3) ^ ((r >> 3) & 1));
    off[t] = 16 * li < TM ? static_cast<uint32_t>(min(r, rmx)) * static_cast<uint32_t>(a.ldx) + c * 16
                          : static_cast<uint32_t>(min(r - TM, rmw)) * static_cast<uint32_t>(a.ldw) + c * 16;
  }
  // group kg runs myn k-steps from klo: nk / KG each, the first group one more of an odd count
  const int nk = static_cast<int>(a.K / BK);
  const int nmin = nk / T::KG, klo = kg * (nk - nmin);
  const uint32_t ring_lds = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(ring)) + kg * NST * T::STAGE;
  // a step past the last is loaded as the last one again, into a stage nobody reads
  auto gload = [&](int s, int stg) __attribute__((always_inline)) {
    const int64_t k0 = static_cast<int64_t>(min(klo + s, nk - 1)) * BK;
    const uint32_t dst = ring_lds + stg * T::STAGE;
#pragma unroll
    for (int t = 0; t < LW; ++t) {
      const int li = t * T::NWG + wg;
      if ((t + 1) * T::NWG <= T::LOADS || li < T::LOADS)
        lds_dma16_s((16 * li < TM ? xb : wb) + k0, off[t], dst + li * 1024);
    }
  };

  acc_t acc[TI][TJ];
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0;

  typename MM::frag_t fa0[TI], fb0[TJ], fa1[TI], fb1[TJ];
  auto load_frags = [&](int stg, const int ks, typename MM::frag_t* fa, typename MM::frag_t* fb)
      __attribute__((always_inline)) {
    const int8_t* const xs_ = ring + (kg * NST + stg) * T::STAGE;
#pragma unroll
    for (int i = 0; i < TI; ++i) fa[i] = MM::load(xs_ + TM * BK, wn * WN + i * 32 + l32, ks, g);
#pragma unroll
    for (int j = 0; j < TJ; ++j) fb[j] = MM::load(xs_, wm * WM + j * 32 + l32, ks, g);
  };
  auto mma_all = [&](const typename MM::frag_t* fa, const typename MM::frag_t* fb) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
      for (int j = 0; j < TJ; ++j) acc[i][j] = MM::mma(fa[i], fb[j], acc[i][j]);
  };
  // issue order: the other fragment set's LDS reads spread between the MFMAs, not after them
  constexpr int NR = (TI + TJ) * (MM::KSUB == 2 ? 1 : 2), NM = TI * TJ, PER = (NR + NM - 2) / (NM - 1);
  auto interleave = [&]() __attribute__((always_inline)) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);    // 0x008: MFMA
#pragma unroll
    for (int i = 0; i < NM - 1; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x100, PER, 0);  // 0x100: LDS reads
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    }
  };
  // every wave's copies of the next step have landed (those of the NST - 2 steps after it stay in flight) and its
  // reads of the ring so far are done
  auto sync_next = [&]() __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (T::LOADS % T::NWG == 0) {
      wait_vm_lds<(NST - 2) * LW>();
    } else {
      if ((LW - 1) * T::NWG + wg < T::LOADS) wait_vm_lds<(NST - 2) * LW>();
      else wait_vm_lds<(NST - 2) * (LW - 1)>();
    }
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  auto next = [](int stg) __attribute__((always_inline)) { return stg == NST - 1 ? 0 : stg + 1; };
  auto prev = [](int stg) __attribute__((always_inline)) { return stg == 0 ? NST - 1 : stg - 1; };
  // Step s reads stage cur = s % NST and first loads step s + NST - 1 into the stage of step s - 1 (every wave passed
  // that step's barrier after its last read of it). int8: the fragments of the step's first half (k = 32) were read at
  // the end of the step before; its second half is read under the first half's MFMAs, the next step's first half under
  // the second's. e4m3 (one MFMA of k = 64 per step): the next step's fragments are read under this step's MFMAs, into
  // the other fragment set, so its steps go in pairs.
  auto step = [&](int s, int cur, auto odd) __attribute__((always_inline)) {
    gload(s + NST - 1, prev(cur));
    if constexpr (MM::KSUB == 2) {
      load_frags(cur, 1, fa1, fb1);
      mma_all(fa0, fb0);
      interleave();
      sync_next();
      load_frags(next(cur), 0, fa0, fb0);
      mma_all(fa1, fb1);
      interleave();
    } else {
      sync_next();
      if constexpr (!decltype(odd)::value) {
        load_frags(next(cur), 0, fa1, fb1);
        mma_all(fa0, fb0);
      } else {
        load_frags(next(cur), 0, fa0, fb0);
        mma_all(fa1, fb1);
      }
      interleave();
    }
  };
  constexpr std::false_type EVEN{};
  constexpr std::true_type ODD{};

  for (int s = 0; s < NST - 1; ++s) gload(s, s);
  sync_next();
  load_frags(0, 0, fa0, fb0);
  int s = 0, cur = 0;
  for (; s + 2 <= nmin; s += 2) {
    step(s, cur, EVEN);
    cur = next(cur);
    step(s + 1, cur, ODD);
    cur = next(cur);
  }
  if constexpr (FP8) mfma_settle();
  if (s < nmin) {
    step(s, cur, EVEN);
    cur = next(cur);
    if constexpr (FP8) mfma_settle();
  }
  if (T::KG > 1 && (nk & 1) && kg == 0) {  // the odd step, already landed: no copy and no barrier of its own
    load_frags(cur, 1, fa1, fb1);
    mma_all(fa0, fb0);
    mma_all(fa1, fb1);
  }
  __builtin_amdgcn_sched_barrier(0);
  wait_vm_lds<0>();  // no copy is in flight and no LDS read pending: the ring is free past the barrier
  if constexpr (EPI != EPI_ACC) {
#pragma unroll
    for (int i = 0; i < NREC; ++i)
      if (i * T::NT + tid < TM + 2 * TN) rec[i * T::NT + tid] = rv[i];
  }
  __syncthreads();

  // KG = 2: group 0 finishes row blocks j < TJ / 2, group 1 the others; each hands the other's blocks over (one 16-byte
  // vector per lane and register quad)
  constexpr int TJO = TJ / T::KG;
  auto xslot = [&](int owner, int j, int i, int rq) __attribute__((always_inline)) {
    return reinterpret_cast<int4*>(ring) + ((((owner * T::NWG + wg) * TJO + j) * TI + i) * 4 + rq) * 64 + lane;
  };
  auto hand_over = [&](auto oc) __attribute__((always_inline)) {
    constexpr int O = decltype(oc)::value;
#pragma unroll
    for (int j = 0; j < TJO; ++j)
#pragma unroll
      for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int rq = 0; rq < 4; ++rq) {
          const acc_t& c = acc[i][O * TJO + j];
          *xslot(O, j, i, rq) = make_int4(c[4 * rq], c[4 * rq + 1], c[4 * rq + 2], c[4 * rq + 3]);
        }
  };
  if constexpr (T::KG == 2) {
    if (kg == 0) hand_over(std::integral_constant<int, 1>{});
    else hand_over(std::integral_constant<int, 0>{});
    __syncthreads();
  }

  // epilogue of the row blocks of owner O: acc[i][j] register r holds m = m0 + wm*WM + j*32 + l32,
  // n = n0 + wn*WN + i*32 + 8*(r/4) + 4*g + (r%4); one 32 x 32 bf16 block at a time goes through a 2 KiB area of the
  // wave (row r at r * 64 B, 16-byte chunk c at c ^ ((r >> 2) & 3)), so global accesses are 64-byte row segments
  int8_t* const ep = ring + T::XCHG + wave * 2048;
  const int chr = lane & 3;
  auto epilogue = [&](auto oc) __attribute__((always_inline)) {
    constexpr int O = decltype(oc)::value;
#pragma unroll
    for (int jo = 0; jo < TJO; ++jo) {
      const int j = O * TJO + jo;
      if constexpr (T::KG == 2) {
#pragma unroll
        for (int i = 0; i < TI; ++i)
#pragma unroll
          for (int rq = 0; rq < 4; ++rq) {
            const int4 v = *xslot(O, jo, i, rq);
            acc[i][j][4 * rq] += v.x;
            acc[i][j][4 * rq + 1] += v.y;
            acc[i][j][4 * rq + 2] += v.z;
            acc[i][j][4 * rq + 3] += v.w;
          }
      }
      if constexpr (EPI == EPI_ACC) {
        const int64_t m = m0 + wm * WM + j * 32 + l32;
#pragma unroll
        for (int i = 0; i < TI; ++i)
#pragma unroll
          for (int rq = 0; rq < 4; ++rq) {
            const int64_t n = n0 + wn * WN + i * 32 + 8 * rq + 4 * g;
            if (m < a.M && n < a.N)
              *reinterpret_cast<int4*>(static_cast<int32_t*>(a.out) + m * a.ldo + n) =
                  make_int4(acc_bits(acc[i][j][4 * rq]), acc_bits(acc[i][j][4 * rq + 1]),
                            acc_bits(acc[i][j][4 * rq + 2]), acc_bits(acc[i][j][4 * rq + 3]));
          }
      } else {
        const float xsm = rec[wm * WM + j * 32 + l32];
        uint4 rres[TI][2];  // the residual segments of this row block, issued before the staging
        if constexpr (EPI == EPI_GATED || EPI == EPI_GATED_ROWS) {
#pragma unroll
          for (int i = 0; i < TI; ++i)
#pragma unroll
            for (int it = 0; it < 2; ++it) {
              const int64_t m = m0 + wm * WM + j * 32 + it * 16 + (lane >> 2);
              const int64_t n = n0 + wn * WN + i * 32 + chr * 8;
              rres[i][it] = (m < a.M && n < a.N)
                                ? *reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(a.out) + m * a.ldo + n)
                                : make_uint4(0, 0, 0, 0);
            }
        }
#pragma unroll
        for (int i = 0; i < TI; ++i) {
#pragma unroll
          for (int rq = 0; rq < 4; ++rq) {
            const int col = wn * WN + i * 32 + 8 * rq + 4 * g;
            const float4 wsn = *reinterpret_cast<const float4*>(rec + TM + col);
            float y[4] = {(MM::val(acc[i][j], 4 * rq + 0) * xsm) * wsn.x, (MM::val(acc[i][j], 4 * rq + 1) * xsm) * wsn.y,
                          (MM::val(acc[i][j], 4 * rq + 2) * xsm) * wsn.z, (MM::val(acc[i][j], 4 * rq + 3) * xsm) * wsn.w};
            if constexpr (EPI == EPI_PLAIN) {
              if (a.bias) {
                const float4 bb = *reinterpret_cast<const float4*>(rec + TM + TN + col);
                y[0] = y[0] + bb.x;
                y[1] = y[1] + bb.y;
                y[2] = y[2] + bb.z;
                y[3] = y[3] + bb.w;
              }
            }
            uint2 o;
            o.x = pack_bf2(y[0], y[1]);
            o.y = pack_bf2(y[2], y[3]);
            *reinterpret_cast<uint2*>(ep + l32 * 64 + ((rq ^ ((l32 >> 2) & 3)) << 4) + 8 * g) = o;
          }
          // each lane reads back what other lanes of its own wave wrote: LDS executes a wave's accesses in order, and
          // the compiler keeps the reads after the writes (same array)
#pragma unroll
          for (int it = 0; it < 2; ++it) {
            const int r = it * 16 + (lane >> 2);
            const uint4 v = *reinterpret_cast<const uint4*>(ep + r * 64 + ((chr ^ ((r >> 2) & 3)) << 4));
            const int64_t m = m0 + wm * WM + j * 32 + r;
            const int64_t n = n0 + wn * WN + i * 32 + chr * 8;
            if (m < a.M && n < a.N) {
              if constexpr (EPI == EPI_PLAIN) {
                *reinterpret_cast<uint4*>(static_cast<uint16_t*>(a.out) + m * a.ldo + n) = v;
              } else if constexpr (EPI == EPI_GATED || EPI == EPI_GATED_ROWS) {
                float gv[8], yv[8], rvv[8];
                if constexpr (EPI == EPI_GATED) {
#pragma unroll
                  for (int e = 0; e < 8; ++e) gv[e] = rec[TM + TN + static_cast<int>(n - n0) + e];
                } else {  // this row's gate row, from global memory (per-token modulation)
                  unpack8(*reinterpret_cast<const uint4*>(a.gate + static_cast<int64_t>(a.gidx[m]) * a.ldg + n), gv);
                }
                unpack8(v, yv);
                unpack8(rres[i][it], rvv);
                uint4 o;
                o.x = pack_bf2(fmaf(yv[0], gv[0], rvv[0]), fmaf(yv[1], gv[1], rvv[1]));
                o.y = pack_bf2(fmaf(yv[2], gv[2], rvv[2]), fmaf(yv[3], gv[3], rvv[3]));
                o.z = pack_bf2(fmaf(yv[4], gv[4], rvv[4]), fmaf(yv[5], gv[5], rvv[5]));
                o.w = pack_bf2(fmaf(yv[6], gv[6], rvv[6]), fmaf(yv[7], gv[7], rvv[7]));
                *reinterpret_cast<uint4*>(static_cast<uint16_t*>(a.out) + m * a.ldo + n) = o;
              } else {  // EPI_SWIGLU: the 8 columns are one [gate 4j..4j+3 | up 4j..4j+3] group of swiglu_perm
                float yv[8];
                unpack8(v, yv);
                uint2 o;
                o.x = pack_bf2(silu_mul(yv[0], yv[4]), silu_mul(yv[1], yv[5]));
                o.y = pack_bf2(silu_mul(yv[2], yv[6]), silu_mul(yv[3], yv[7]));
                *reinterpret_cast<uint2*>(static_cast<uint16_t*>(a.out) + m * a.ldo + n / 2) = o;
              }
            }
          }
        }
      }
    }
  };
  if constexpr (T::KG == 2) {
    if (kg == 0) epilogue(std::integral_constant<int, 0>{});
    else epilogue(std::integral_constant<int, 1>{});
  } else {
    epilogue(std::integral_constant<int, 0>{});
  }
}

template <bool FP8, int EPI, typename T>
int launch(GemmArgs a, hipStream_t st, const char* name) {
  a.tiles_m = static_cast<int>((a.M + T::TM - 1) / T::TM);
  a.tiles_n = static_cast<int>((a.N + T::TN - 1) / T::TN);
  const int64_t nb = static_cast<int64_t>(a.tiles_m) * a.tiles_n;
  hipLaunchKernelGGL((gemm_tile_kernel<FP8, EPI, T>), dim3(static_cast<unsigned>(nb)), dim3(T::NT), 0, st, a);
  return launch_status(name);
}

// The built tiles, small to large. One workgroup of any of them fills a CU's LDS but for the 128 x 128 one (two fit).
// The smallest is bound by its serial k-steps, which two wave groups halve where sums are exact in any order. The e4m3
// form keeps one chain of 4 waves of 32 x 64 outputs (us, two halves of K / one chain: 77 x 3072 -> 9216 9.1 / 10.7,
// 77 x 8192 -> 3072 17.8 / 21.5, 226 x 8192 -> 3072 25.1 / 24.6, 512 x 3072 -> 3072 11.8 / 10.8; 64 x 32 outputs a wave
// 10.8, 23.0, 24.5, 11.1; 8 waves of 32 x 32 12.0, 26.7, 26.7, 12.0).
template <bool FP8>
using T128x64 = std::conditional_t<FP8, Tile<128, 64, 4, 1, 1, 8>, Tile<128, 64, 2, 2, 2, 5>>;
typedef Tile<128, 128, 2, 2, 1, 4> T128x128;
typedef Tile<256, 128, 4, 2, 1, 6> T256x128;
typedef Tile<256, 192, 4, 2, 1, 5> T256x192;

template <bool FP8, int EPI>
int launch_cfg(int cfg, const GemmArgs& a, hipStream_t st, const char* name) {
  switch (cfg) {
    case TILE_128x64: return launch<FP8, EPI, T128x64<FP8>>(a, st, name);
    case TILE_128x128: return launch<FP8, EPI, T128x128>(a, st, name);
    case TILE_256x128: return launch<FP8, EPI, T256x128>(a, st, name);
    default: return launch<FP8, EPI, T256x192>(a, st, name);
  }
}

}  // namespace

// Costs in units of a full round (one 256 x 256 tile on every CU: about 45 us at K = 3072). A tile of its own round
// costs less the smaller it is, but each loads more operand bytes per MFMA, so over many rounds the 256 x 256 kernel is
// the fastest and the small tiles only win where they all run at once. Measured on random sizes (M 64-12,000, eight
// K x N of two model widths; us, 256 x 256 against the tile): one round of 128 x 64 31 -> 11-13 (K = 3072) and
// 68 -> 21-29 (K = 8192), 128 x 128 33 -> 15-20, 256 x 128 35 -> 29, 256 x 192 76 -> 72 (K = 7168). A last round that
// is not full still costs 0.65 of one or more (264 tiles 77 us, 252 tiles 50), so rows just past a full round
// run as a second launch of small tiles (5,442 x 3072 x 3072: 77 -> 61), or all of them as 256 x 192 (964 x 21504 x
// 5376: 144 -> 126). From four rounds on the loss is too small to matter.
TilePlan plan_tiles(int64_t M, int64_t N, int64_t K, int64_t cus) {
  const int64_t nk = K / BK;
  auto tiles = [&](int64_t m, int64_t tm, int64_t tn) { return ((m + tm - 1) / tm) * ((N + tn - 1) / tn); };
  const double launch = 4.8 / static_cast<double>(nk);   // a kernel's fixed time
  // the cheapest tile that runs m rows in one round, or TILE_256
  auto one_round = [&](int64_t m, double* cost) {
    struct { int id, tm, tn; double c; } const t[] = {
        {TILE_128x64, 128, 64, 0.20}, {TILE_128x128, 128, 128, 0.33}, {TILE_256x128, 256, 128, 0.55},
        {TILE_256x192, 256, 192, 0.72}};
    for (const auto& x : t) {
      const int64_t n = tiles(m, x.tm, x.tn);
      // a short K does not carry 256 x 192's longer epilogue on a nearly full chip (4096 x 3072 x 3072 42.5 against 39 us
      // on 256 x 256; x 8192 101 against 103)
      if (x.id == TILE_256x192 && nk < 64 && 4 * n > 3 * cus) continue;
      if (n <= cus) {
        *cost = x.c;
        return x.id;
      }
    }
    *cost = 1.0;
    return static_cast<int>(TILE_256);
  };
  double c1;
  const int small = one_round(M, &c1);
  if (small != TILE_256) return {small, 0};
  const int64_t nt = tiles(M, 256, 256), full = nt / cus, rem = nt % cus;
  if (nt <= cus || full >= 4 || rem == 0) return {TILE_256, 0};
  auto part = [](double a, double b, double frac) { return frac > 0 ? a + b * frac : 0.0; };
  TilePlan best{TILE_256, 0};
  double cost = static_cast<double>(full) + part(0.65, 0.35, static_cast<double>(rem) / cus);
  const int64_t n4 = tiles(M, 256, 192);
  const double c4 = 0.82 * static_cast<double>(n4 / cus) + part(0.60, 0.22, static_cast<double>(n4 % cus) / cus);
  if (c4 < cost) {
    best = {TILE_256x192, 0};
    cost = c4;
  }
  const int64_t head = full * cus / ((N + 255) / 256) * 256;   // rows of the tile rows that fill whole rounds
  if (head > 0 && head < M) {
    double ct;
    const int tail = one_round(M - head, &ct);
    if (tail != TILE_256 && static_cast<double>(full) + launch + ct < cost) best = {tail, head};
  }
  return best;
}

int run_tile(bool fp8, int epi, int cfg, const GemmArgs& a, hipStream_t st, const char* name) {
  if (fp8) return epi == EPI_ACC ? launch_cfg<true, EPI_ACC>(cfg, a, st, name) : launch_cfg<true, EPI_PLAIN>(cfg, a, st, name);
  switch (epi) {
    case EPI_SWIGLU: return launch_cfg<false, EPI_SWIGLU>(cfg, a, st, name);
    case EPI_GATED: return launch_cfg<false, EPI_GATED>(cfg, a, st, name);
    case EPI_GATED_ROWS: return launch_cfg<false, EPI_GATED_ROWS>(cfg, a, st, name);
    case EPI_ACC: return launch_cfg<false, EPI_ACC>(cfg, a, st, name);
    default: return launch_cfg<false, EPI_PLAIN>(cfg, a, st, name);
  }
}

}  // namespace gemm
}  // namespace rh3
