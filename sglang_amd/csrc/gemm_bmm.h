// Batched FP8 GEMM with short K (the absorbed products of multi-head latent attention: K = 128 or 512, one small product per
// head), gfx950.
//
// With one to four K blocks there is no loop to pipeline: what a product costs is one trip to memory for its operands, a
// handful of MFMAs and the way out.  The 128x128 tile kernel pays its five-stage LDS ring (160 KB, one workgroup per CU) for
// that: 128 entries of 64 x 512 x 128, two rounds of 512 such workgroups, take it 14.7 us and this kernel 6.2.  Here a workgroup is four waves on a 64(m) x 128(n) tile with two
// 24 KB stages: three workgroups share a CU, and one's loads run under another's write-out.  Operands take the road of the
// tile kernels (buffer_load ... lds, rows past the edge out of the descriptor's range, 16-byte chunk c of row r at position
// c ^ ((r >> 1) & 7)); a wave computes 32 x 64.  The entries of a batch go to the XCDs in turn, all tiles of an entry to one.
#pragma once

#include "gemm_kernels.h"

namespace fp8k {

constexpr int kBmmTileM = 64, kBmmTileN = 128;

template <int OUT_DT>
__global__ __launch_bounds__(256) void gemm_bmm_short_kernel(const GemmArgs p) {
  constexpr int kWOff = kBmmTileM * kTileK, kStage = (kBmmTileM + kBmmTileN) * kTileK;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[2 * kStage];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int wm = w & 1, wn = w >> 1;
  const int per_entry = p.tiles_m * p.tiles_n;
  const int j = (int)(blockIdx.x >> 3);
  const int entry = j / per_entry * 8 + (int)(blockIdx.x & 7), t = j % per_entry;
  if (entry >= p.batch) return;
  const int m0 = t % p.tiles_m * kBmmTileM, n0 = t / p.tiles_m * kBmmTileN;
  const int nkb = p.K / kTileK;

  // ---- global -> LDS: wave w brings rows [16w, 16w+16) of X and [32w, 32w+32) of W, 1 KB (8 rows) a load
  const int rowsX = min(kBmmTileM, p.M - m0), rowsW = min(kBmmTileN, p.N - n0);
  const rsrc_t rX = make_rsrc(p.X + entry * p.batch_x + (int64_t)m0 * p.ldx, (uint32_t)((rowsX - 1) * p.ldx + p.K));
  const rsrc_t rW = make_rsrc(p.W + entry * p.batch_w + (int64_t)n0 * p.ldw, (uint32_t)((rowsW - 1) * p.ldw + p.K));
  const int rl = lane >> 3, cp = lane & 7;
  auto fetch = [&](int stage, int kb) {
    uint8_t* const base = smem + stage * kStage;
    const uint32_t ko = (uint32_t)kb * kTileK;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int c = cp ^ ((i * 4 + (rl >> 1)) & 7);
      buf_load16_to_lds(rX, (uint32_t)((w * 16 + i * 8 + rl) * p.ldx + c * 16) + ko, 0, base + (w * 16 + i * 8) * kTileK);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int c = cp ^ ((i * 4 + (rl >> 1)) & 7);
      buf_load16_to_lds(rW, (uint32_t)((w * 32 + i * 8 + rl) * p.ldw + c * 16) + ko, 0, base + kWOff + (w * 32 + i * 8) * kTileK);
    }
  };

  // ---- LDS -> matrix core
  const int lr = lane & 31, h = lane >> 5, swz = (lr >> 1) & 7;
  auto frag = [&](const uint8_t* rows, int ks) -> v8i {  // row lr of a 32-row group, K half ks
    const v4i lo = *reinterpret_cast<const v4i*>(rows + lr * kTileK + (((ks * 4 + h * 2) ^ swz) << 4));
    const v4i hi = *reinterpret_cast<const v4i*>(rows + lr * kTileK + (((ks * 4 + h * 2 + 1) ^ swz) << 4));
    v8i r;
    r[0] = lo[0]; r[1] = lo[1]; r[2] = lo[2]; r[3] = lo[3];
    r[4] = hi[0]; r[5] = hi[1]; r[6] = hi[2]; r[7] = hi[3];
    return r;
  };
  v16f acc[2];
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[0][r] = acc[1][r] = 0.f;

  fetch(0, 0);
  if (nkb > 1) fetch(1, 1);
  for (int kb = 0; kb < nkb; ++kb) {
    if (kb + 1 < nkb) lds_barrier<6>();  // block kb has landed, the six loads of block kb+1 may be on their way
    else lds_barrier<0>();
    const uint8_t* const st = smem + (kb & 1) * kStage;
    const uint8_t *const xr = st + wm * 32 * kTileK, *const wr = st + kWOff + wn * 64 * kTileK;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const v8i x = frag(xr, ks);
      acc[0] = mfma_32x32x64(frag(wr, ks), x, acc[0]);
      acc[1] = mfma_32x32x64(frag(wr + 32 * kTileK, ks), x, acc[1]);
    }
    if (kb + 2 < nkb) {
      lds_barrier<6>();  // every wave has taken block kb's operands
      fetch(kb & 1, kb + 2);
    }
  }

  const int m_own = m0 + wm * 32 + lr, nw = n0 + wn * 64;
  const float sa[1] = {m_own < p.M ? row_scale(p, m_own) : 1.f};
  finish_rows<8, 1, FP8K_F32>(p, sa, [&](int q) { return nw + (q >> 2) * 32 + (q & 3) * 8 + h * 4; },
                              [&](int q, int, int i, auto f) { acc[q >> 2][(q & 3) * 4 + i] = f(acc[q >> 2][(q & 3) * 4 + i]); });
  // through 4 KB of LDS per wave, 16-byte chunks XOR-swizzled by the row, so that a store covers 128-byte row segments
  u16* const C = (u16*)p.C + entry * p.batch_c;
  const bool wide = (p.ldc & 7) == 0 && (reinterpret_cast<uintptr_t>(C) & 15) == 0;
  // the slot lies in the stage that the last block did not use: with two and more blocks another wave may still be reading
  // operands of the last one
  uint8_t* const ep = smem + (nkb & 1) * kStage + w * 4096;
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const int i = (q & 3) * 4;
    float v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = acc[q >> 2][i + k];
    uint2 o;
    if (OUT_DT == FP8K_BF16) o = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
    else o = make_uint2(f32_to_f16_bits(v[0]) | (f32_to_f16_bits(v[1]) << 16), f32_to_f16_bits(v[2]) | (f32_to_f16_bits(v[3]) << 16));
    const int n = nw + (q >> 2) * 32 + (q & 3) * 8 + h * 4;
    if (wide) *reinterpret_cast<uint2*>(ep + lr * 128 + ((q ^ (lr & 7)) << 4) + h * 8) = o;
    else if (m_own < p.M && n < p.N) *reinterpret_cast<uint2*>(C + (int64_t)m_own * p.ldc + n) = o;
  }
  if (!wide) return;
  __builtin_amdgcn_wave_barrier();  // one wave's LDS accesses complete in order
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = i * 8 + rl, m = m0 + wm * 32 + r, n = nw + (cp << 3);
    const uint4 o = *reinterpret_cast<const uint4*>(ep + r * 128 + ((cp ^ (r & 7)) << 4));
    if (m < p.M && n < p.N) *reinterpret_cast<uint4*>(C + (int64_t)m * p.ldc + n) = o;
  }
}

}  // namespace fp8k
