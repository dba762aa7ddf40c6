// fp32 GEMM fed by LDS DMA (gfx950): gemm_fxp_kernel's results, from 16-byte
// aligned operands in either B layout.
//
// What bounds it: the fp32 matrix cores (16x16x4 in 32 cycles: 152 TFLOP/s
// measured on register operands; this kernel reaches 135 at M = 8192,
// N = 14336, K = 4096: 11.45 ms -> 7.10 ms against the register-staged
// 128 x 128 tiles, one wave per SIMD, that it replaced; M = 777: 1.55 ->
// 0.77 ms, N-contiguous B 1.91 -> 0.76 ms; M = 64, N = 6144: 64 -> 39 us).
// One MFMA hides eight VALU instructions, so
// the schedule only has to keep every SIMD's MFMA pipe fed:
//   * tiles small enough in registers (fp32 partials + integer sums) for two
//     or three waves per SIMD, of different workgroups, so one's barrier, LDS
//     latency and quantisation run under another's MFMAs;
//   * stages of 32 k brought straight into LDS (buffer_load ... lds), double
//     buffered, one barrier per stage, no staging registers;
//   * a partial last K-tile peeled off, so the loop has no masked loads.
// LDS rows. K-contiguous operands: 128 bytes per row (32 k), the 16-byte chunk
// c of row r at slot c ^ ((r >> 1) & 7): a fragment read (one element per
// lane: row lane % 16, k = 4 step + lane / 16) touches all 64 banks once.
// N-contiguous B: as loaded, one row per k, chunk c of row k at slot
// c ^ (4 (k % 4)), so the four k rows of a fragment read fall on distinct
// banks and nothing is transposed. Fragment reads are ds_read2st64_b32: two
// 16-row blocks (K-contiguous) or two k steps (N-contiguous) at once.
// The compiler would wait for every DMA in flight before any LDS read it can
// see, so the reads are inline asm with explicit waits (check_lds_reads.py
// scans the generated code for a use before its wait).
#pragma once

#include "gemm_impl.h"

namespace fxpr {
namespace gemm {

typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

template <int BM_, int BN_, int WGM_, int WGN_, int WPE_> struct F32Tile {
  static constexpr int BM = BM_, BN = BN_, WGM = WGM_, WGN = WGN_;
  static constexpr int WPE = WPE_;  // waves per SIMD the register budget is sized for
  static constexpr int WM = BM / WGM, WN = BN / WGN;
  static constexpr int MB = WM / 16, NB = WN / 16;
  static_assert(WGM * WGN == kThreads / 64, "4 waves per workgroup");
  static_assert(MB % 2 == 0 && NB % 2 == 0, "fragments are read two blocks at a time");
};

template <class FT> constexpr size_t f32_lds_bytes() { return size_t(2) * (FT::BM + FT::BN) * 128; }

// two 4-byte elements 256 * OFF0 and 256 * OFF1 bytes past addr
template <int OFF0, int OFF1> __device__ __forceinline__ void lds_read2st64(unsigned addr, u32x2& x) {
  static_assert(OFF0 >= 0 && OFF1 < 256, "8-bit offsets");
  asm volatile("ds_read2st64_b32 %0, %1 offset0:%2 offset1:%3" : "=v"(x) : "v"(addr), "n"(OFF0), "n"(OFF1) : "memory");
}

template <int BITS, class FT, bool BNC, bool SPLIT>
__global__ __launch_bounds__(kThreads, FT::WPE) void gemm_f32_kernel(GemmArgs args) {
  using M_ = Mma<FXPR_DTYPE_F32>;
  using AccT = typename Acc<BITS>::T;
  constexpr int BM = FT::BM, BN = FT::BN, MB = FT::MB, NB = FT::NB, NW = kThreads / 64;
  constexpr int BKS = 32, CH = 4, NP = BKS / 8;  // k per stage, elements per chunk, step pairs per stage
  constexpr int A_SLOT = BM * 128, B_SLOT = BN * 128;  // bytes per stage
  constexpr int B_RING = 2 * A_SLOT;
  constexpr int NIA = BM / 8 / NW, NIB = BN / 8 / NW;  // DMA instructions (1 KB each) per wave per stage
  static_assert(NIA * 8 * NW == BM && NIB * 8 * NW == BN, "tile / wave mismatch");
  constexpr int RB = BN * 4;       // bytes per k row of an N-contiguous stage
  constexpr int CPRB = BN / CH;    // its 16-byte chunks
  static_assert(!BNC || (CPRB % 16 == 0 && CPRB <= 64 && 64 % CPRB == 0), "whole k rows per DMA instruction");

  extern __shared__ __align__(16) unsigned char smem_raw[];
  const unsigned lds0 = static_cast<unsigned>(reinterpret_cast<uintptr_t>(smem_raw));
  const float* A = static_cast<const float*>(args.a);
  const float* B = static_cast<const float*>(args.b);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / FT::WGN, wn = wave % FT::WGN;
  int tm, tn;
  tile_coords(blockIdx.x, gridDim.x, args.tiles_m, args.tiles_n, tm, tn);
  const int64_t m0 = int64_t(tm) * BM, n0 = int64_t(tn) * BN;
  const int split = blockIdx.y;
  const int kt_begin = split * args.tiles_per_split;
  const int kt_end = min(args.ktiles, kt_begin + args.tiles_per_split);
  const bool has_tail = kt_end > kt_begin && int64_t(kt_end) * 64 > args.K;
  const int nfull = max(0, kt_end - kt_begin - (has_tail ? 1 : 0));
  const int64_t kb0 = int64_t(kt_begin) * 64;

  // DMA sources: a fixed 32-bit lane offset per instruction (the host keeps
  // BM and BN rows, and the 32 k rows of an N-contiguous stage, below 2^31
  // bytes) from the tile's first row and the stage's first k. Rows past M and
  // columns past N are clamped: they feed only outputs that are never stored.
  uint32_t va[NIA], vb[NIB];
#pragma unroll
  for (int q = 0; q < NIA; ++q) {
    const int r = 8 * (wave + NW * q) + (lane >> 3);
    const int c = (lane & 7) ^ ((r >> 1) & 7);
    va[q] = uint32_t(((min<int64_t>(m0 + r, args.M - 1) - m0) * args.lda + c * CH) * 4);
  }
#pragma unroll
  for (int q = 0; q < NIB; ++q) {
    const int i = wave + NW * q;
    if constexpr (BNC) {
      const int r = (64 / CPRB) * i + lane / CPRB;
      const int c = (lane % CPRB) ^ ((r & 3) << 2);
      vb[q] = uint32_t((r * args.ldb + (min<int64_t>(n0 + c * CH, args.N - CH) - n0)) * 4);
    } else {
      const int r = 8 * i + (lane >> 3);
      const int c = (lane & 7) ^ ((r >> 1) & 7);
      vb[q] = uint32_t(((min<int64_t>(n0 + r, args.N - 1) - n0) * args.ldb + c * CH) * 4);
    }
  }
  const float* const a_base = A + m0 * args.lda + kb0;
  const float* const b_base = BNC ? B + kb0 * args.ldb + n0 : B + n0 * args.ldb + kb0;
  // stage s (32 k from kb0) into slot s % 2. (The N-contiguous stage offset
  // may pass 2^31 bytes: it goes into the 64-bit base.)
  auto dma = [&](int s, int slot) {
    const __amdgpu_buffer_rsrc_t ar =
        __builtin_amdgcn_make_buffer_rsrc(uniform_ptr(a_base), short(0), -1, kBufferDword3);
    const __amdgpu_buffer_rsrc_t br = __builtin_amdgcn_make_buffer_rsrc(
        uniform_ptr(BNC ? b_base + int64_t(s) * BKS * args.ldb : b_base), short(0), -1, kBufferDword3);
    const int soff = s * (BKS * 4);
#pragma unroll
    for (int q = 0; q < NIA; ++q)
      buffer_to_lds(ar, lds0 + slot * A_SLOT + (wave + NW * q) * 1024, va[q], soff);
#pragma unroll
    for (int q = 0; q < NIB; ++q)
      buffer_to_lds(br, lds0 + B_RING + slot * B_SLOT + (wave + NW * q) * 1024, vb[q], BNC ? 0 : soff);
  };

  f32x4 P[MB][NB];
  AccT I[MB][NB][4];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) I[i][j][r] = 0;
  const f32x4 zero4 = {0.f, 0.f, 0.f, 0.f};

  const int l16 = lane & 15, kg = lane >> 4, sw = l16 >> 1;
  const unsigned arow = lds0 + (wm * FT::WM + l16) * 128 + kg * 4;
  const unsigned brow = lds0 + B_RING + (BNC ? unsigned(kg * RB + (l16 & 3) * 4) : unsigned((wn * FT::WN + l16) * 128 + kg * 4));

  // One stage: 8 steps of 4 k, in pairs. The fragments of a pair: A blocks
  // (2 p, 2 p + 1) of each step; B likewise, or (N-contiguous) block j of both
  // steps. The next pair's reads are issued before the current pair's wait.
  struct Frags {
    u32x2 a[2][MB / 2];
    u32x2 b[NB];
  };
  auto read_pair = [&](int slot, auto uc, Frags& f) __attribute__((always_inline)) {
    constexpr int u = decltype(uc)::value;
    static_for<2>([&](auto hc) {
      constexpr int h = decltype(hc)::value;
      const unsigned x = ((2 * u + h) ^ sw) << 4;
      static_for<MB / 2>([&](auto pc) {
        constexpr int p = decltype(pc)::value;
        lds_read2st64<16 * p, 16 * p + 8>(arow + slot * A_SLOT + x, f.a[h][p]);
      });
      if constexpr (!BNC)
        static_for<NB / 2>([&](auto pc) {
          constexpr int p = decltype(pc)::value;
          lds_read2st64<16 * p, 16 * p + 8>(brow + slot * B_SLOT + x, f.b[h * (NB / 2) + p]);
        });
    });
    if constexpr (BNC)
      static_for<NB>([&](auto jc) {
        constexpr int j = decltype(jc)::value;
        constexpr int SU = 4 * RB / 256;  // 256-byte units per step
        lds_read2st64<2 * u * SU, (2 * u + 1) * SU>(
            brow + slot * B_SLOT + (((wn * (FT::WN / 4) + 4 * j + (l16 >> 2)) ^ (kg << 2)) << 4), f.b[j]);
      });
  };
  // at most N younger LDS operations outstanding; the fragments are bound here
  auto wait_pair = [&](auto nc, Frags& f) __attribute__((always_inline)) {
    asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(decltype(nc)::value) : "memory");
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int p = 0; p < MB / 2; ++p) asm volatile("" : "+v"(f.a[h][p]));
#pragma unroll
    for (int j = 0; j < NB; ++j) asm volatile("" : "+v"(f.b[j]));
  };
  auto mma_pair = [&](const Frags& f, bool first) __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) {
          const float a = __uint_as_float(f.a[h][i / 2][i % 2]);
          const float b = __uint_as_float(BNC ? f.b[j][h] : f.b[h * (NB / 2) + j / 2][j % 2]);
          P[i][j] = M_::mma(a, b, first && h == 0 ? zero4 : P[i][j]);
        }
  };
  auto compute = [&](int slot, bool first) __attribute__((always_inline)) {
    Frags f[2];
    read_pair(slot, std::integral_constant<int, 0>{}, f[0]);
    static_for<NP>([&](auto uc) {
      constexpr int u = decltype(uc)::value;
      if constexpr (u + 1 < NP) {
        read_pair(slot, std::integral_constant<int, u + 1>{}, f[(u + 1) & 1]);
        wait_pair(std::integral_constant<int, MB + NB>{}, f[u & 1]);
      } else {
        wait_pair(std::integral_constant<int, 0>{}, f[u & 1]);
      }
      mma_pair(f[u & 1], first && u == 0);
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  auto quantize = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          I[i][j][r] = wrap_add<BITS>(I[i][j][r], quant<BITS>(__fmul_rn(P[i][j][r], args.scale)));
  };

  // Partial last K-tile first (integer sums do not depend on the order):
  // masked loads into both slots, zero past K.
  if (has_tail) {
    const int64_t kt0 = int64_t(kt_end - 1) * 64;
    const bool whole = args.K % CH == 0;
#pragma unroll 4
    for (int e = tid; e < 2 * BM * 8; e += kThreads) {
      const int st = e / (BM * 8), r = e % (BM * 8) / 8, c = e % 8;
      const int64_t k = kt0 + st * BKS + c * CH, row = m0 + r;
      const int valid = row < args.M && k < args.K ? int(min<int64_t>(CH, args.K - k)) : 0;
      *reinterpret_cast<uint4*>(smem_raw + st * A_SLOT + r * 128 + ((c ^ ((r >> 1) & 7)) << 4)) =
          load_chunk_or_zero(A + (valid ? row * args.lda + k : 0), valid, whole);
    }
#pragma unroll 4
    for (int e = tid; e < 2 * BN * 8; e += kThreads) {
      const int st = e / (BN * 8), w = e % (BN * 8);
      if constexpr (BNC) {
        const int r = w / CPRB, c = w % CPRB;
        const int64_t k = kt0 + st * BKS + r, col = n0 + c * CH;
        const int valid = k < args.K && col < args.N ? CH : 0;  // N is a multiple of CH
        *reinterpret_cast<uint4*>(smem_raw + B_RING + st * B_SLOT + r * RB + ((c ^ ((r & 3) << 2)) << 4)) =
            load_chunk_or_zero(B + (valid ? k * args.ldb + col : 0), valid, true);
      } else {
        const int r = w / 8, c = w % 8;
        const int64_t k = kt0 + st * BKS + c * CH, col = n0 + r;
        const int valid = col < args.N && k < args.K ? int(min<int64_t>(CH, args.K - k)) : 0;
        *reinterpret_cast<uint4*>(smem_raw + B_RING + st * B_SLOT + r * 128 + ((c ^ ((r >> 1) & 7)) << 4)) =
            load_chunk_or_zero(B + (valid ? col * args.ldb + k : 0), valid, whole);
      }
    }
    __syncthreads();
    compute(0, true);
    compute(1, false);
    quantize();
    __syncthreads();
  }

  // Full K-tiles, two stages each. At a stage's start its own DMAs are the
  // only ones in flight: wait for them, barrier (everyone's have landed, and
  // everyone is done reading the other slot), refill the other slot, compute.
  if (nfull > 0) {
    const int nst = 2 * nfull;
    dma(0, 0);
    for (int s = 0; s < nst; s += 2) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      dma(s + 1, 1);
      compute(0, true);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      if (s + 2 < nst) dma(s + 2, 0);  // uniform
      compute(1, false);
      quantize();
    }
  }

  // Epilogue. Lane holds rows 4 kg + r of each 16x16 block, column lane % 16.
  const int64_t row_base = m0 + wm * FT::WM + kg * 4;
  const int64_t col_base = n0 + wn * FT::WN + l16;
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const int64_t n = col_base + j * 16;
    if (n >= args.N) continue;
    const float bv = !SPLIT && args.bias ? args.bias[n] : 0.0f;
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t m = row_base + i * 16 + r;
        if (m >= args.M) continue;
        if constexpr (SPLIT) {
          static_cast<AccT*>(args.ws)[(int64_t(split) * args.M + m) * args.N + n] = I[i][j][r];
        } else {
          float v = acc_to_f32<BITS>(I[i][j][r], args.inv_scale);
          if (args.bias) v = __fadd_rn(v, bv);
          static_cast<float*>(args.c)[m * args.scm + n * args.scn] = v;
        }
      }
  }
}

template <int BITS, class FT, bool BNC>
int launch_f32_tile(GemmArgs a, int splits, hipStream_t st) {
  a.tiles_m = int(cdiv(a.M, FT::BM));
  a.tiles_n = int(cdiv(a.N, FT::BN));
  constexpr size_t lds = f32_lds_bytes<FT>();
  auto go = [&](auto kern) -> int {
    static bool attr_done = false;  // benign race: the attribute is idempotent
    if (!attr_done) {
      hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                         hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
      if (e != hipSuccess) return int(e);
      attr_done = true;
    }
    kern<<<dim3(unsigned(int64_t(a.tiles_m) * a.tiles_n), unsigned(splits)), kThreads, lds, st>>>(a);
    return launch_status();
  };
  if (splits > 1 || a.mode == kPartial) return go(gemm_f32_kernel<BITS, FT, BNC, true>);
  return go(gemm_f32_kernel<BITS, FT, BNC, false>);
}

template <int BITS> int launch_f32(const GemmArgs& a, bool b_ncontig, int splits, hipStream_t st) {
  // 32 x 32 wave tiles in a row of four, or 32 x 64 ones two by two: three
  // workgroups per CU (64-bit sums of the wider one: two)
  using T32 = F32Tile<32, 128, 1, 4, 3>;
  using T64 = F32Tile<64, 128, 2, 2, BITS == 64 ? 2 : 3>;
  const bool small = a.M <= 32 || f32_plan(a.M, a.N, a.ktiles, splits).bm == 32;
  if (small)
    return b_ncontig ? launch_f32_tile<BITS, T32, true>(a, splits, st) : launch_f32_tile<BITS, T32, false>(a, splits, st);
  return b_ncontig ? launch_f32_tile<BITS, T64, true>(a, splits, st) : launch_f32_tile<BITS, T64, false>(a, splits, st);
}

}  // namespace gemm
}  // namespace fxpr
