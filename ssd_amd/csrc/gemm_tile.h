// The main loop of the large-tile bf16 GEMMs (many token rows: prefill): a workgroup owns (WN * NT) 16-row groups of W and (WM * MT)
// 16-row groups of x, its WN x WM waves NT x MT of them each, and leaves the fp32 products in acc[NT][MT].
//
// What bounds it is the matrix cores and the LDS that feeds them: a wave with 4 x 4 accumulator tiles reads 8 KiB of LDS per 16 MFMAs of 16x16x32
// (16 cycles each), so that at full rate the four SIMDs take 32 KiB in 256 cycles, all of the 128 bytes a CU's LDS delivers per cycle; 3 x 3
// tiles ask for a third more than that, 4 x 2 for half as much again.  Both operands therefore travel HBM / L2 -> LDS by DMA (loads to LDS: no
// registers, no LDS write instructions), 1 KiB per instruction, into a ring of STAGES steps of KS x 32 k.  A step's loads are issued
// STAGES - 1 steps ahead, and ONE barrier per step both publishes the step and frees the buffer of the one before.
// In bf16 every accumulator is one chain over the ascending k of the range that its workgroup walks, whatever the tile: where the caller does not cut K
// (gemm_rows.hip), a row's result does not depend on the rows beside it; ssd_gemm_big's K splits go by the number of rows.  fp32: see below.
#pragma once
#include "common.h"

// Buffer descriptor of `bytes` bytes at p (raw, unswizzled; reads past the end return zero).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t tile_rsrc(const void* p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, (int)bytes, 0x00020000);
}

// 64 lanes x 16 bytes: memory at rsrc + voff (per lane) + soff -> LDS at lds (wave-uniform) + 16 * lane.
__device__ __forceinline__ void tile_dma(__amdgpu_buffer_rsrc_t rsrc, uint32_t voff, uint32_t soff, char* lds) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void*)lds, 16, (int)voff, (int)soff, 0, 0);
}
template <int N>
__device__ __forceinline__ void tile_wait() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// fp32 products (mfma 16x16x4: a lane holds ONE k of its row; peak 157 TFLOP/s, twice the vector unit's without packed fp32).  The order of
// a sum is part of what the fp32 mode promises -- a row's result is the same bits whichever kernel computes it -- and is defined here:
// segments of F32_SEG k (the last one shorter), each a chain from zero over its blocks of 16 k, a block being four MFMAs, the e-th over
// k = e, 4 + e, 8 + e, 12 + e (lane q of a row holds 4 consecutive k: one 16-byte load); the segments' sums are added in order, from zero.
constexpr int F32_SEG = 256, F32_SEG_STEPS = F32_SEG / 32;
__device__ __forceinline__ f32x4_t mfma_f32(uint32_t a, uint32_t b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a), __uint_as_float(b), c, 0, 0, 0);
}

// F32: operands are floats, a step is 32 k (KS = 2), `acc` the sum over segments.
template <int WN, int WM, int NT, int MT, int STAGES, int KS = 1, bool F32 = false>
struct TileLoop {
  static constexpr int WAVES = WN * WM, WG = WN * NT, XG = WM * MT;          // waves; 16-row groups of W, of x
  static constexpr int STEP = (WG + XG) * KS * 1024;                              // LDS bytes of a k-step
  static constexpr int PER = (WG + XG) * KS / WAVES;                             // 1 KiB operands each wave fetches per k-step
  static constexpr int LDS = STAGES * STEP;
  static_assert((WG + XG) * KS % WAVES == 0, "every wave fetches as many operands");

  // fetch_one(i, step, lds): KiB i of this wave's PER (KiB wave * PER + i of the workgroup's step: W's groups first, KS each, then x's) of
  // step `step` on its way to LDS.  at[s]: where in a group's KS KiB this lane finds its part of the s-th MFMA operand.
  template <typename Fetch>
  static __device__ __forceinline__ void run(char* smem, int nk, const uint32_t (&at)[KS], f32x4_t (&acc)[NT][MT], const Fetch& fetch_one) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wn = wave / WM, wm = wave % WM;
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int j = 0; j < MT; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    auto fetch = [&](int step, uint32_t buf) {
#pragma unroll
      for (int i = 0; i < PER; ++i) fetch_one(i, step, smem + buf * STEP + (wave * PER + i) * 1024);
    };
#pragma unroll
    for (int s = 0; s < STAGES - 1; ++s) fetch(s < nk ? s : nk - 1, s);
    uint32_t cur = 0;
    f32x4_t part[F32 ? NT : 1][F32 ? MT : 1];
    if constexpr (F32) {
#pragma unroll
      for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) part[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
    for (int k = 0; k < nk; ++k) {
      tile_wait<PER * (STAGES - 2)>();                 // this wave's share of step k is in LDS
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");      // everybody's is, and nobody reads step k - 1 any more
      // (past the end the last step is fetched again: into the buffer nobody reads, so that the count of loads in flight stays static)
      const int ahead = k + STAGES - 1;
      fetch(ahead < nk ? ahead : nk - 1, cur == 0 ? STAGES - 1 : cur - 1);
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const char* a0 = smem + cur * STEP + wn * NT * KS * 1024 + at[s];
        const char* b0 = smem + cur * STEP + (WG + wm * MT) * KS * 1024 + at[s];
        u32x4_t a[NT], b[MT];
#pragma unroll
        for (int j = 0; j < MT; ++j) b[j] = *reinterpret_cast<const u32x4_t*>(b0 + j * KS * 1024);
#pragma unroll
        for (int i = 0; i < NT; ++i) a[i] = *reinterpret_cast<const u32x4_t*>(a0 + i * KS * 1024);
#pragma unroll
        for (int i = 0; i < NT; ++i)
#pragma unroll
          for (int j = 0; j < MT; ++j) {
            if constexpr (!F32) acc[i][j] = mfma16(a[i], b[j], acc[i][j]);
          }
        if constexpr (F32) {
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int i = 0; i < NT; ++i)
#pragma unroll
              for (int j = 0; j < MT; ++j) part[i][j] = mfma_f32(a[i][e], b[j][e], part[i][j]);
        }
      }
      if constexpr (F32) {
        if ((k + 1) % F32_SEG_STEPS == 0 || k + 1 == nk) {
#pragma unroll
          for (int i = 0; i < NT; ++i)
#pragma unroll
            for (int j = 0; j < MT; ++j) { acc[i][j] += part[i][j]; part[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f}; }
        }
      }
      cur = cur + 1 == STAGES ? 0 : cur + 1;
    }
    tile_wait<0>();                                    // nothing may land in LDS after the workgroup has ended
  }
};

// Workgroup -> tile: the 8 XCDs (each with an L2 of its own) take workgroups in turn; every XCD gets one contiguous run of the tile
// list, and the list walks `GM` token tiles for every feature tile, so that the W and x tiles a run shares stay in its L2.
struct TileAt { int n, m; };
__device__ __forceinline__ TileAt tile_at(int bid, int tn, int tm) {
  constexpr int XCDS = 8, GM = 4;
  const int total = tn * tm, per = total / XCDS, rem = total % XCDS;
  const int x = bid % XCDS, i = bid / XCDS;
  const int t = x * per + (x < rem ? x : rem) + i;
  const int band = t / (GM * tn), in = t % (GM * tn);
  const int rows = min(GM, tm - band * GM);
  return TileAt{in / rows, band * GM + in % rows};
}
