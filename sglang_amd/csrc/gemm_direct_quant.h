// gemm_wavek_kernel with the quantisation of its activations in front: a decode linear of a few rows in one launch.
//
// Such a linear is two launches of latency: the quant kernel (3 us for 14 KB) and a GEMM whose weights cannot be requested
// before it ends, while the second launch costs the host as much again.  Here every workgroup quantises all M x K
// activations for itself - they are few, they hit the L2, and the vector units have nothing else to do while the first
// weight lines travel - and keeps the bytes and the scales in LDS, in the order the matrix core wants them.  The weight
// requests of the first D K blocks go out between the activation loads and their use, so the two memory latencies overlap.
// The price is the quantisation once per workgroup, about 6 vector instructions per element: kQuantFuseMax says up to which
// M * K it stays under the launch it replaces.
//
// Whole linear, bf16, two launches -> this one, one weight: M = 1: 4608 x 7168 13.5 -> 8.7 us (33 MB: 5.3 us at the read ceiling),
// 6144 x 4096 10.9 -> 7.4, 7168 x 18432 28.9 -> 22.1, 1024 x 1024 9.7 -> 5.2 (the host's time for one launch); M = 8, at the limit
// of M * K: 6144 x 4096 11.7 -> 8.8, per-token 11.1 -> 9.1.  With the weights rotated over 600 MB, so that none comes out of the
// memory-side cache: 9.4, 8.2, 22.4, 5.3; 9.6, 9.9.  Per token the row's scale is one more serial step; with the maxima of all rows
// taken at once, 32 lanes to a row, rather than 64 lanes to two rows in turn, 13 x 3456 x 1152 6.2 -> 5.7 us (replayed from a graph),
// 16 x 896 x 640 5.6 -> 5.2, 11 x 8640 x 2048 8.8 -> 8.4, 8 x 4096 x 2048 6.4 -> 6.2, 1 x 4608 x 7168 9.2 level.
//
// Split of the work, K order, LDS re-layout of the weights and summation are gemm_wavek_kernel's, and the quantisation is
// that of group_quant_kernel (block mode) or token_quant_kernel (row mode), so results are those of the two launches bit for
// bit.
#pragma once

#include "gemm_direct.h"
#include "quant_math.h"

namespace fp8k {

constexpr int kQuantFuseMax = 32768;    // elements of X a workgroup quantises for itself
constexpr int kWqGroups = kQuantFuseMax / 128;

// bytes of LDS for the quantised rows, padded so that the rows of an operand fetch fall into different banks
__host__ __device__ constexpr int wq_row_bytes(int K) { return K + 16; }

// p.X: the 16-bit activations [M, K], contiguous; P: pieces of 8 elements per lane (M * K <= P * 512 * 8); D: K blocks of
// weights in flight per wave.  The two share 128 registers, so that two workgroups fit a CU.
template <int P, int D, int MODE, int OUT_DT, int BIAS_DT>
__global__ __launch_bounds__(512, 4) void gemm_wavek_quant_kernel(const GemmArgs p) {
  static_assert(MODE == kModeBlock || MODE == kModeRow, "float scales only");
  extern __shared__ __attribute__((aligned(16))) uint8_t xq[];                // [M][K + 16]
  __shared__ __attribute__((aligned(16))) uint8_t wl[8][16 * kTileK];         // per wave: one K block of its 16 weight rows
  __shared__ float sgrp[kWqGroups];  // of group m * kb_all + kb - block mode: its scale, row mode: its maximum
  __shared__ float sblk[kWqGroups];  // block mode: the weight scales (all 16 * NW rows of a workgroup lie in one scale block)
  __shared__ float srow[16], sinv[16];  // row mode: the rows' scales and their reciprocals

  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, kq = lane >> 4;
  const int NW = p.wk_nw, nw = w % NW, ks = w / NW;
  const int n0w = (blockIdx.x * NW + nw) * 16;
  const int kb_all = p.K / kTileK;
  const int kb0 = ks * p.kb_per_split;
  const int nkb = n0w < p.N ? max(min(kb_all, kb0 + p.kb_per_split) - kb0, 0) : 0;
  const uint32_t kbytes = (uint32_t)nkb * kTileK;
  const int xrow = wq_row_bytes(p.K);

  // ---- activations: wave w takes groups [4 P w, 4 P (w + 1)) of X, piece j of a lane is 8 elements of group base + 4 j
  const int groups = p.M * kb_all;
  const int base = w * (4 * P) + (lane >> 4), l8 = (lane & 15) * 8;
  const float inv_kb = 1.0f / (float)kb_all;
  auto row_of = [&](int g) { return (int)(((float)g + 0.5f) * inv_kb); };  // g / kb_all, exact: g < 2^8
  Raw8<OUT_DT> raw[P];
#pragma unroll
  for (int j = 0; j < P; ++j)  // past the end: the last group again, whose bytes nobody stores
    raw[j].load(p.X, (int64_t)min(base + 4 * j, groups - 1) * 128 + l8);
  float wscale = 0.f;
  if (MODE == kModeBlock && tid < kb_all)
    wscale = p.sw[(int64_t)(min((int)(blockIdx.x * NW * 16), p.N - 1) >> 7) * p.sw_n + (int64_t)tid * p.sw_k];
  __builtin_amdgcn_sched_barrier(0);

  // ---- weights: line-shaped loads, re-laid out through the wave's LDS slot (as in gemm_wavek_kernel)
  const int rowsW = min(16, p.N - n0w);
  const rsrc_t rW = make_rsrc(p.W + (int64_t)n0w * p.ldw + (int64_t)kb0 * kTileK,
                              (rowsW > 0 && nkb > 0) ? (uint32_t)((rowsW - 1) * p.ldw) + kbytes : 0u);
  const int wrow = lane >> 3, wc = lane & 7;
  const uint32_t voW0 = (uint32_t)(wrow * p.ldw + wc * 16), voW1 = (uint32_t)((wrow + 8) * p.ldw + wc * 16);
  uint8_t* const wslot = wl[w];
  const uint32_t wst0 = (uint32_t)(wrow * kTileK + ((wc ^ ((wrow >> 1) & 7)) << 4));
  const uint32_t wst1 = (uint32_t)((wrow + 8) * kTileK + ((wc ^ (((wrow + 8) >> 1) & 7)) << 4));
  const uint32_t wrd0 = (uint32_t)(r * kTileK + ((kq ^ ((r >> 1) & 7)) << 4));
  const uint32_t wrd1 = (uint32_t)(r * kTileK + (((4 + kq) ^ ((r >> 1) & 7)) << 4));
  v4i wreg[D][2];
  auto issue = [&](int slot, int kb) {
    const bool ok = kb < nkb;
    const uint32_t ko = (uint32_t)kb * kTileK;
    wreg[slot][0] = buf_load16_stream(rW, ok ? voW0 + ko : kOutOfRange);
    wreg[slot][1] = buf_load16_stream(rW, ok ? voW1 + ko : kOutOfRange);
  };
#pragma unroll
  for (int d = 0; d < D; ++d) issue(d, d);
  __builtin_amdgcn_sched_barrier(0);

  // ---- quantise: bytes to LDS; the LDS-only barriers leave the weight requests in flight
  if (MODE == kModeBlock && tid < kb_all) sblk[tid] = wscale;
  if (MODE == kModeRow) {
#pragma unroll
    for (int j = 0; j < P; ++j) {
      float a[8];
      raw[j].unpack(a);
      const float m = group_max<16>(absmax8(a));
      if (l8 == 0 && base + 4 * j < groups) sgrp[base + 4 * j] = m;
    }
    lds_barrier();
    if (const int m = tid >> 5; m < p.M) {  // 32 lanes to a row, all 16 at once (64: two in turn)
      float mx = 0.f;
      for (int g = lane & 31; g < kb_all; g += 32) mx = fmaxf(mx, sgrp[m * kb_all + g]);
      const float sc = group_max<32>(mx) / kFp8Max;
      if ((lane & 31) == 0) {
        srow[m] = sc;
        sinv[m] = sc == 0.f ? 0.f : 1.0f / sc;
      }
    }
    lds_barrier();
  }
#pragma unroll
  for (int j = 0; j < P; ++j) {
    const int g = base + 4 * j;
    if (g < groups) {
      const int m = row_of(g);
      float a[8];
      raw[j].unpack(a);
      uint2 o;
      if (MODE == kModeBlock) {
        const float amax = fmaxf(group_max<16>(absmax8(a)), p.q_eps);
        const float sc = div448<true>(amax);
        bool redo;
        o = quant8_bracket<true>(a, sc, amax, redo);
        if (__builtin_expect(redo, 0)) o = quant8_divide(a, sc);
        if (l8 == 0) sgrp[g] = sc;
      } else {
        const float inv = sinv[m];
        float y[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) y[i] = fmaxf(fminf(a[i] * inv, kFp8Max), -kFp8Max);
        o = make_uint2(cvt4_fp8(y[0], y[1], y[2], y[3]), cvt4_fp8(y[4], y[5], y[6], y[7]));
      }
      *reinterpret_cast<uint2*>(xq + m * xrow + (g - m * kb_all) * kTileK + l8) = o;
    }
  }
  lds_barrier();

  // ---- K loop of the wave: rows past M repeat the last one (their columns of the product are not stored)
  v4f acc = {0.f, 0.f, 0.f, 0.f};
  const int mr = min(r, p.M - 1);
  const uint8_t* const xrd = xq + mr * xrow + kb0 * kTileK + kq * 16;
  const float* const srd = sgrp + mr * kb_all + kb0;
  const float* const swd = sblk + kb0;
  for (int k0 = 0; k0 < nkb; k0 += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      if (k0 + d >= nkb) break;
      *reinterpret_cast<v4i*>(wslot + wst0) = wreg[d][0];
      *reinterpret_cast<v4i*>(wslot + wst1) = wreg[d][1];
      const v8i wa = join(*reinterpret_cast<const v4i*>(wslot + wrd0), *reinterpret_cast<const v4i*>(wslot + wrd1));
      const uint8_t* const xp = xrd + (k0 + d) * kTileK;
      const v8i xa = join(*reinterpret_cast<const v4i*>(xp), *reinterpret_cast<const v4i*>(xp + 64));
      issue(d, k0 + d + D);
      if (MODE == kModeBlock) {
        const float sc = srd[k0 + d] * swd[k0 + d];
        const v4f t = mfma_16x16x128(wa, xa, v4f{0.f, 0.f, 0.f, 0.f});
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] = __builtin_fmaf(t[i], sc, acc[i]);
      } else {
        acc = mfma_16x16x128(wa, xa, acc);
      }
    }
  }
  // ---- the K ranges meet, as in gemm_wavek_kernel; a wave's sums take the place of its weight slot
  *reinterpret_cast<v4f*>(wslot + lane * 16) = acc;
  __syncthreads();
  if (ks != 0) return;
  const int KS = 8 / NW;
  const int n = n0w + kq * 4;
  if (n >= p.N || r >= p.M) return;
  v4f s = acc;
  for (int k = 1; k < KS; ++k) {
    const v4f o = *reinterpret_cast<const v4f*>(wl[k * NW + nw] + lane * 16);
    s[0] += o[0]; s[1] += o[1]; s[2] += o[2]; s[3] += o[3];
  }
  float v[4] = {s[0], s[1], s[2], s[3]};
  finish4<MODE, OUT_DT, BIAS_DT>(p, n, MODE == kModeRow ? srow[r] : 1.f, v);
  store4<OUT_DT>(p.C, (int64_t)r * p.ldc + n, v[0], v[1], v[2], v[3]);
}

}  // namespace fp8k
