// Causal attention of many query rows over the paged cache (varlen prefill; reference ssd/layers/attention.py:90-93): the same products as
// attention.hip -- S^T = K . Q^T and O^T += V^T . P^T on 16x16x32 MFMAs, P as two bf16 terms, so that the weights of the sum keep 2^-17 --
// organised for throughput: a workgroup = 4 waves x 32 rows of one kv head ((token, head of the group) pairs, token-major) shares every
// 64-key tile of K and V through LDS, filled by DMA one tile ahead, one barrier per tile.
//   * What bounds it: 96 MFMAs per wave and tile against 32 scores per lane, each a multiply-add, an exponential, a sum, a maximum and two
//     conversions.  So: no maximum across lanes and no rescaling per tile -- a row keeps its reference maximum until some score exceeds it by
//     2^8 (exact: both numerator and sum carry it), and only tiles that touch the causal edge or the context's end are masked.
//   * LDS: a key's 16-byte chunks are rotated by its index on the way in (K: chunk ^ (key & 7); V: chunk ^ 2 (key & 3)), so that both the
//     8-lane groups of a K read and the 16-lane groups of a V transpose-read hit different banks.
//   * Blocks with the longest scans (the last rows of a sequence) are launched first; blocks of one kv head share an XCD's L2.
// MI355X, attention.hip's form -> this one: 32 heads of 128 in 8 groups, 16384 tokens 10.6 -> 2.81 ms (782 TFLOP/s counting each product once,
// 1170 executed), 2048 tokens 261 -> 73 us, prompts of 1501, 94 and 800 tokens behind 512 cached ones 321 -> 85 us; heads of 64, seven prompts
// of 60 .. 900 tokens 94 -> 31 us.  Error against fp64 unchanged.
#include "common.h"
#include "attention_prefill.h"

namespace {

constexpr int WAVES = 4, RT = PREFILL_ROWS / 16 / WAVES, KEYS = 64;

template <int HD>
__global__ void __launch_bounds__(64 * WAVES, 2)
attn_prefill_kernel(const PrefillAttn p) {
  constexpr int DS = HD / 32, DT = HD / 16, CH = HD / 8;          // k-steps of QK^T, output tiles, 16-byte chunks per key
  constexpr int TILE = KEYS * HD * 2, KPI = 64 / CH, PER = TILE / 1024 / WAVES;    // bytes of a K (V) tile; keys per DMA; DMAs per wave
  __shared__ __attribute__((aligned(1024))) char smem[2][2][TILE];                // [buffer][K, V]
  const int lane = threadIdx.x & 63, r16 = lane & 15, g4 = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int b = blockIdx.x / p.nkv, h = blockIdx.x % p.nkv, G = p.nh / p.nkv;
  const int q0 = p.cu_q ? p.cu_q[b] : b * p.q_per_seq;
  const int Tq = p.cu_q ? p.cu_q[b + 1] - q0 : p.q_per_seq;
  const int rows = Tq * G;
  const int row_wg = (int)(gridDim.y - 1 - blockIdx.y) * PREFILL_ROWS;
  if (row_wg >= rows) return;
  const int ctx = p.context_lens[b];
  const int32_t* bt = p.block_tables + (size_t)b * p.max_blocks;

  // ---- this wave's rows ----
  const int row_w = row_wg + wave * RT * 16;
  u32x4_t qf[RT][DS];
  int lim[RT];                                       // keys [0, lim) are visible
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    const int rho = min(row_w + rt * 16 + r16, rows - 1), tl = rho / G;
    lim[rt] = ctx - (Tq - 1 - tl);
    const bf16_t* qp = p.q + ((size_t)(q0 + tl) * p.nh + h * G + rho % G) * HD + g4 * 8;
#pragma unroll
    for (int ds = 0; ds < DS; ++ds) qf[rt][ds] = *reinterpret_cast<const u32x4_t*>(qp + ds * 32);
  }
  // (Q arrives before the loop: a wait for it inside would be one for the DMA in flight as well)
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int ds = 0; ds < DS; ++ds) asm volatile("" : "+v"(qf[rt][ds]));
  const int kmax = ctx - (Tq - 1 - min(rows - 1, row_wg + PREFILL_ROWS - 1) / G);         // of the workgroup's last row
  const int kmax_w = ctx - (Tq - 1 - min(rows - 1, row_w + RT * 16 - 1) / G);             // of the wave's last, and first, row
  const int kmin_w = ctx - (Tq - 1 - min(rows - 1, row_w) / G);
  const int tiles = (kmax + KEYS - 1) / KEYS;

  // ---- DMA: a wave fetches 16 keys of a tile (one page: pages hold 16 keys or more), KPI per instruction, a lane one chunk of one key into its
  //      rotated place.  Keys past the context are read as its last one: nothing unwritten is touched ----
  const int dkey = lane / CH, dch = lane % CH;
  int pages = 0;                                     // lane i: the page of tile (t & ~63) + i
  auto look_up = [&](int t) { pages = bt[min((t + lane) * KEYS + wave * 16, ctx - 1) >> p.bs_shift]; };
  auto fetch = [&](int t, int buf) {
    const int page = __builtin_amdgcn_readlane(pages, t & 63);
    const int first = min(t * KEYS + wave * 16, ctx - 1) >> p.bs_shift << p.bs_shift;        // the page's first key
    const size_t base = ((((size_t)page * p.nkv + h) << p.bs_shift) - first) * HD;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int key = wave * 16 + i * KPI + dkey;
      const uint32_t row = (uint32_t)min(t * KEYS + key, ctx - 1) * HD;
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(p.kc + base + (row + (dch ^ (key & 7)) * 8)),
                                       (__attribute__((address_space(3))) void*)(smem[buf][0] + (wave * PER + i) * 1024), 16, 0, 0);
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(p.vc + base + (row + (dch ^ ((key & 3) * 2)) * 8)),
                                       (__attribute__((address_space(3))) void*)(smem[buf][1] + (wave * PER + i) * 1024), 16, 0, 0);
    }
  };

  float m[RT], lsum[RT];
  f32x4_t o[RT][DT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    m[rt] = -INFINITY;
    lsum[rt] = 0.f;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) o[rt][dt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }

  if (tiles > 0) {                                   // (no key for any row: a padded sequence, or more rows than keys)
    look_up(0);
    fetch(0, 0);
  }
  for (int t = 0; t < tiles; ++t) {
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");       // tile t is in LDS; nobody reads tile t - 1 any more
    if (t + 1 < tiles) {
      if (((t + 1) & 63) == 0) look_up(t + 1);
      fetch(t + 1, (t + 1) & 1);
    }
    const int k0 = t * KEYS;
    if (k0 >= kmax_w) continue;                      // (a wave past its rows still meets the barriers)
    const char* kl = smem[t & 1][0];
    const char* vl = smem[t & 1][1];
    // -- S^T[key][row] --
    f32x4_t st[KEYS / 16][RT];
#pragma unroll
    for (int kb = 0; kb < KEYS / 16; ++kb) {
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) st[kb][rt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ds = 0; ds < DS; ++ds) {
        const u32x4_t a = *reinterpret_cast<const u32x4_t*>(kl + ((kb * 16 + r16) * CH + ((ds * 4 + g4) ^ (r16 & 7))) * 16);
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) st[kb][rt] = mfma16(a, qf[rt][ds], st[kb][rt]);
      }
    }
    if (k0 + KEYS > kmin_w) {
#pragma unroll
      for (int kb = 0; kb < KEYS / 16; ++kb)
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (k0 + kb * 16 + g4 * 4 + e >= lim[rt]) st[kb][rt][e] = -INFINITY;
    }
    // -- weights against the row's reference maximum --
    u32x4_t ph[KEYS / 32][RT], pl[KEYS / 32][RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      float top = st[0][rt][0];
#pragma unroll
      for (int kb = 0; kb < KEYS / 16; ++kb)
#pragma unroll
        for (int e = 0; e < 4; ++e) top = fmaxf(top, st[kb][rt][e]);
      top *= p.scale_log2e;
      if (__any(top > m[rt] + 8.0f)) {
        top = fmaxf(top, __shfl_xor(top, 16, 64));
        top = fmaxf(m[rt], fmaxf(top, __shfl_xor(top, 32, 64)));
        const float alpha = top == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(m[rt] - top);       // (a row's first key: exp2(-inf) = 0)
        m[rt] = top;
        lsum[rt] *= alpha;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) o[rt][dt] *= alpha;
      }
      const float ref = m[rt] == -INFINITY ? 0.f : m[rt];       // (a row that has seen no key yet: all weights are zero)
      float sum = 0.f;
#pragma unroll
      for (int kb = 0; kb < KEYS / 16; ++kb) {
        float w[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          w[e] = __builtin_amdgcn_exp2f(fmaf(st[kb][rt][e], p.scale_log2e, -ref));
          sum += w[e];
        }
        const uint32_t h0 = pack_bf2(w[0], w[1]), h1 = pack_bf2(w[2], w[3]);
        ph[kb / 2][rt][(kb & 1) * 2] = h0;
        ph[kb / 2][rt][(kb & 1) * 2 + 1] = h1;
        pl[kb / 2][rt][(kb & 1) * 2] = pack_bf2(w[0] - __uint_as_float(h0 << 16), w[1] - __uint_as_float(h0 & 0xffff0000u));
        pl[kb / 2][rt][(kb & 1) * 2 + 1] = pack_bf2(w[2] - __uint_as_float(h1 << 16), w[3] - __uint_as_float(h1 & 0xffff0000u));
      }
      lsum[rt] += sum;
    }
    // -- O^T[d][row] += V^T . P^T: lane (r16, g4) names row 4 g4 + (r16 >> 2), column quad r16 & 3 of a 16 x 16 block and receives column r16 of
    //    rows 4 g4 .. + 3, which are the keys its P holds --
#pragma unroll
    for (int c = 0; c < KEYS / 32; ++c)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        const int key = g4 * 4 + (r16 >> 2);
        const char* a0 = vl + ((c * 32 + key) * CH + ((dt * 2 + ((r16 & 3) >> 1)) ^ ((key & 3) * 2))) * 16 + (r16 & 1) * 8;
        typedef s16x4_t __attribute__((address_space(3))) * lds_v4_t;
        const u32x2_t lo = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4_t)a0));
        const u32x2_t hi = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4_t)(a0 + 16 * CH * 16)));
        const u32x4_t vf = {lo[0], lo[1], hi[0], hi[1]};
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
          o[rt][dt] = mfma16(vf, ph[c][rt], o[rt][dt]);
          o[rt][dt] = mfma16(vf, pl[c][rt], o[rt][dt]);
        }
      }
  }

#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    float l = lsum[rt] + __shfl_xor(lsum[rt], 16, 64);
    l += __shfl_xor(l, 32, 64);
    const int rho = row_w + rt * 16 + r16;
    if (rho >= rows) continue;
    const float inv = l > 0.f ? 1.0f / l : 0.f;
    const int tok = q0 + rho / G, head = h * G + rho % G;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      const int d = dt * 16 + g4 * 4;
      const u32x2_t v = {pack_bf2(o[rt][dt][0] * inv, o[rt][dt][1] * inv), pack_bf2(o[rt][dt][2] * inv, o[rt][dt][3] * inv)};
      if (p.out_rows) *reinterpret_cast<u32x2_t*>(p.out_rows + ((size_t)tok * p.nh + head) * HD + d) = v;
      if (p.out_frag) {
        const int kcol = head * HD + d;
        p.out_frag[frag_chunk(tok, kcol >> 3, (p.nh * HD) >> 5) * 2 + ((kcol >> 2) & 1)] = v;
      }
    }
  }
}

}  // namespace

int attn_prefill_launch(const PrefillAttn& p, int B, int max_q, int hd, hipStream_t st) {
  const dim3 grid(B * p.nkv, (max_q * (p.nh / p.nkv) + PREFILL_ROWS - 1) / PREFILL_ROWS);
  if (hd == 128) hipLaunchKernelGGL(attn_prefill_kernel<128>, grid, dim3(64 * WAVES), 0, st, p);
  else hipLaunchKernelGGL(attn_prefill_kernel<64>, grid, dim3(64 * WAVES), 0, st, p);
  return hipGetLastError() == hipSuccess ? SSD_OK : SSD_ERR_LAUNCH;
}
