// Weight-streaming FP8 GEMM for at most 32 activation rows per block (decode and small-batch MoE), gfx950.
//
// With so few activation rows the GEMM is an HBM stream of the weight matrix (2*TM FLOP per weight byte, far under
// the chip's ridge), so everything is arranged around the weight loads.  A wavefront owns 16 weight rows and keeps
// eight K blocks (16 KB; four in the grouped GEMM) of them in flight in registers: two non-temporal 16-byte loads per
// lane and K block, each instruction covering 8 whole 128-byte lines (lane l: row l/8, 16-byte chunk l%8) - whole-line
// requests measured 25 % more HBM bandwidth here than the half-line requests that loading straight into the matrix-core
// operand layout would make.  The move into that layout (operand "A" of v_mfma_f32_16x16x128_f8f6f4: lane l holds 32 bytes
// of row l%16) is a round trip through a 2 KB LDS slot private to the wave: LDS operations of one wave execute in
// order, so it needs no barrier and no wait beyond the register dependency.  The matrix core only sums over K, so
// the K order inside a 128-byte block is free as long as both operands agree: lane (row, q = l/16) takes chunks
// q and 4+q of the block.
//
// The activation rows (shared by the 8 waves = 128 weight rows of a workgroup) are staged through LDS in chunks
// of as many K blocks: registers -> ds_write one chunk ahead, one barrier per chunk (an LDS-only barrier: the weight
// loads stay in flight across it), rows padded by 16 bytes so the 16 rows of an operand fetch fall into different
// banks.  In block mode the chunk also carries as[m,kb]*bs[nb,kb] (a workgroup spans exactly one 128-row weight
// scale block), zero past the K range, so the K tail needs no branch.  (Every wave re-reads all activation rows
// of the block from LDS, which is why blocks of 64 and 128 rows measured slower here than through
// gemm_stream_kernel.)
//
// The grouped GEMM keeps four K blocks in flight instead of eight: at most 109 registers and 50 KB of LDS let two workgroups
// share a CU (eight took 174 registers: one), so the start and the write-out of one block hide behind the stream of
// another, and a short K (an expert's intermediate size) pads to less.  Bytes in flight per CU stay the same.  Measured
// on the whole layer with 32-row blocks: 128 experts x 4096 x 256 at 384 slots 1.05x, x 1024 1.05x, 64 x 7168 x 1024
// 1.03x; with 16-row blocks 1.00 .. 1.05x.  The linears keep eight: their grid leaves one workgroup per CU.
#pragma once

#include "gemm_kernels.h"

namespace fp8k {

constexpr int kDirTileN = 128;                   // 8 waves x 16 weight rows
constexpr int kDirDepth = 8;                     // of a linear: weight prefetch depth in K blocks = K blocks per activation chunk
constexpr uint32_t kOutOfRange = 0xF0000000u;    // buffer offset past every descriptor range: reads zero

__device__ __forceinline__ v4i buf_load16(rsrc_t r, uint32_t voff) {
  return __builtin_amdgcn_raw_buffer_load_b128(r, voff, 0, 0);
}
__device__ __forceinline__ v4i buf_load16_stream(rsrc_t r, uint32_t voff) {  // non-temporal: used once
  return __builtin_amdgcn_raw_buffer_load_b128(r, voff, 0, 2);
}
template <int TM, int MODE, int OUT_DT, int BIAS_DT, bool SPLIT, bool MOE>
__global__ __launch_bounds__(512, MOE ? 4 : 2) void gemm_direct_kernel(const GemmArgs p) {
  static_assert(TM == 16 || TM == 32, "gemm_direct_kernel: 16 or 32 rows per block (more rows are LDS-read bound here)");
  constexpr int MS = TM / 16;                 // 16-row activation sub-tiles
  constexpr int KC = MOE ? kDirDepth / 2 : kDirDepth;  // K blocks per activation chunk = weight prefetch depth
  constexpr int RB = KC * kTileK;             // bytes of one activation row in a chunk
  constexpr int XROW = RB + 16;               // LDS row stride
  constexpr int LPR = RB / 16;                // lanes per staged row
  constexpr int RPI = 64 / LPR;               // rows per staging load
  constexpr int XI = TM / 8 / RPI;            // staging loads per wave per chunk
  static_assert(TM * KC <= 512, "one scale product per lane and chunk");
  __shared__ __attribute__((aligned(16))) uint8_t xs[2][TM * XROW];
  __shared__ float scs[2][KC][TM];
  __shared__ __attribute__((aligned(16))) uint8_t wl[8][16 * kTileK];  // per wave: one K block of its 16 weight rows

  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int r = lane & 15, kq = lane >> 4;

  // ---- work item (same walk as gemm_stream_kernel)
  int bid = blockIdx.x;
  int split = 0;
  int mb, tile_n;
  if (MOE) {
    const int used = p.num_post_pad[0] / p.block_m;
    const int per_xcd = (used + 7) >> 3;
    const int j = bid >> 3;
    const int mbl = j / p.tiles_n;
    if (mbl >= per_xcd) return;
    mb = (bid & 7) * per_xcd + mbl;
    if (mb >= used || mb >= p.m_blocks) return;
    tile_n = j - mbl * p.tiles_n;
  } else {
    if (SPLIT) { split = bid % p.splits; bid /= p.splits; }
    if (bid >= p.tiles_n * p.m_blocks) return;
    mb = bid % p.m_blocks;
    tile_n = bid / p.m_blocks;
  }
  const int block_m = MOE ? p.block_m : TM;
  const int slot0 = mb * block_m;
  const int expert = MOE ? p.expert_ids[mb] : 0;
  const int nrows = MOE ? p.num_valid : p.M;
  const int n0 = tile_n * kDirTileN;
  const int n0w = n0 + w * 16;

  const int kb_begin = SPLIT ? split * p.kb_per_split : 0;
  const int kb_end = SPLIT ? min(p.K / kTileK, kb_begin + p.kb_per_split) : p.K / kTileK;
  // an expert that lives on another rank contributes zeros: run no K block, the epilogue stores them
  const int nkb = (MOE && expert < 0) ? 0 : max(kb_end - kb_begin, 0);
  const int nch = (nkb + KC - 1) / KC;
  const uint32_t kbytes = (uint32_t)nkb * kTileK;   // bytes of this K range per row

  auto slot_of = [&](int i) -> int {   // row slot of block row i, or nrows when the row is padding
    if (i >= block_m) return nrows;
    const int s = MOE ? p.sorted_ids[slot0 + i] : slot0 + i;
    return s < nrows ? s : nrows;
  };

  // ---- weights: 16 rows of this wave, straight into MFMA operand registers
  const uint8_t* Wb = p.W + (MOE && expert >= 0 ? (int64_t)expert * p.w_expert_stride : 0);
  const int rowsW = min(16, p.N - n0w);
  const rsrc_t rW = make_rsrc(Wb + (int64_t)n0w * p.ldw + (int64_t)kb_begin * kTileK,
                              rowsW > 0 ? (uint32_t)((rowsW - 1) * p.ldw) + kbytes : 0u);
  // load j of a K block: row j*8 + lane/8, chunk lane%8; in LDS chunk c of row i sits at position c ^ ((i>>1)&7),
  // which keeps both the line-shaped writes and the operand-shaped reads free of bank conflicts
  const int wrow = lane >> 3, wc = lane & 7;
  const uint32_t voW0 = (uint32_t)(wrow * p.ldw + wc * 16), voW1 = (uint32_t)((wrow + 8) * p.ldw + wc * 16);
  uint8_t* const wslot = wl[w];
  const uint32_t wst0 = (uint32_t)(wrow * kTileK + ((wc ^ ((wrow >> 1) & 7)) << 4));
  const uint32_t wst1 = (uint32_t)((wrow + 8) * kTileK + ((wc ^ (((wrow + 8) >> 1) & 7)) << 4));
  const uint32_t wrd0 = (uint32_t)(r * kTileK + ((kq ^ ((r >> 1) & 7)) << 4));
  const uint32_t wrd1 = (uint32_t)(r * kTileK + (((4 + kq) ^ ((r >> 1) & 7)) << 4));
  v4i wreg[KC][2];
  auto load_w = [&](int slot, int kb) {
    const bool ok = kb < nkb;
    wreg[slot][0] = buf_load16_stream(rW, ok ? voW0 + (uint32_t)kb * kTileK : kOutOfRange);
    wreg[slot][1] = buf_load16_stream(rW, ok ? voW1 + (uint32_t)kb * kTileK : kOutOfRange);
  };
  auto weight_operand = [&](int slot) -> v8i {  // registers (line layout) -> LDS -> registers (operand layout)
    *reinterpret_cast<v4i*>(wslot + wst0) = wreg[slot][0];
    *reinterpret_cast<v4i*>(wslot + wst1) = wreg[slot][1];
    return join(*reinterpret_cast<const v4i*>(wslot + wrd0), *reinterpret_cast<const v4i*>(wslot + wrd1));
  };

  // ---- activations: wave w stages rows w*TM/8 .. of the block, RB bytes per row and chunk;
  // staging load j of a lane covers row w*TM/8 + j*RPI + lane/LPR, bytes (lane%LPR)*16 ..
  const int64_t xrows = MOE ? (int64_t)((p.num_valid + p.top_k - 1) / p.top_k) : (int64_t)p.M;
  const rsrc_t rX = make_rsrc(p.X + (int64_t)kb_begin * kTileK, (uint32_t)((xrows - 1) * p.ldx) + kbytes);
  const int xcol = (lane % LPR) * 16;
  uint32_t voX[XI];
#pragma unroll
  for (int j = 0; j < XI; ++j) {
    const int s = slot_of(w * (TM / 8) + j * RPI + lane / LPR);
    const int64_t xr = MOE ? s / p.top_k : s;
    voX[j] = s < nrows ? (uint32_t)(xr * p.ldx) + xcol : kOutOfRange;
  }
  v4i xreg[XI];
  // ---- block mode: lane t < TM*KC stages as[m,kb]*bs[nb,kb] of (m = t % TM, kb = chunk*KC + t / TM)
  const int sm = threadIdx.x % TM, skb = threadIdx.x / TM;
  const bool stager = MODE == kModeBlock && (int)threadIdx.x < TM * KC;
  const float* sxp = p.sx;
  const float* swp = p.sw;
  bool srow_ok = false;
  if (stager) {
    const int s = slot_of(sm);
    srow_ok = s < nrows;
    const int64_t xr = srow_ok ? (MOE ? s / p.top_k : s) : 0;
    sxp = p.sx + xr * p.sx_m + (int64_t)kb_begin * p.sx_k;
    swp = p.sw + (MOE && expert >= 0 ? (int64_t)expert * p.sw_expert_stride : 0) +
          (int64_t)(min(n0, p.N - 1) >> 7) * p.sw_n + (int64_t)kb_begin * p.sw_k;
  }
  float sreg_x = 0.f, sreg_w = 0.f;  // multiplied at store time: using them here would wait for every load in flight
  auto stage_load = [&](int c) {
    const uint32_t k0 = (uint32_t)c * RB;
#pragma unroll
    for (int j = 0; j < XI; ++j) {
      const bool ok = voX[j] != kOutOfRange && k0 + xcol < kbytes;
      xreg[j] = buf_load16(rX, ok ? voX[j] + k0 : kOutOfRange);
    }
    if (MODE == kModeBlock) {
      const int kb = c * KC + skb;
      sreg_x = 0.f;
      sreg_w = 0.f;
      if (stager && srow_ok && kb < nkb) {
        sreg_x = sxp[(int64_t)kb * p.sx_k];
        sreg_w = swp[(int64_t)kb * p.sw_k];
      }
    }
  };
  auto stage_store = [&](int buf) {
#pragma unroll
    for (int j = 0; j < XI; ++j)
      *reinterpret_cast<v4i*>(&xs[buf][(w * (TM / 8) + j * RPI + lane / LPR) * XROW + xcol]) = xreg[j];
    if (stager) scs[buf][skb][sm] = sreg_x * sreg_w;
  };

  v4f acc[MS];
#pragma unroll
  for (int ms = 0; ms < MS; ++ms) acc[ms] = v4f{0.f, 0.f, 0.f, 0.f};

  // ---- prologue: chunks 0 and 1 requested, then the weights of K blocks 0..7, then chunk 0 into LDS.  The loop
  // keeps the same age order (staging loads older than the weight loads issued after them), so that the wait
  // for a staged chunk never has to drain the weight prefetch.
  stage_load(0);
  v4i xreg0[XI];
#pragma unroll
  for (int j = 0; j < XI; ++j) xreg0[j] = xreg[j];
  const float s0x = sreg_x, s0w = sreg_w;
  stage_load(1);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int d = 0; d < KC; ++d) load_w(d, d);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int j = 0; j < XI; ++j)
    *reinterpret_cast<v4i*>(&xs[0][(w * (TM / 8) + j * RPI + lane / LPR) * XROW + xcol]) = xreg0[j];
  if (stager) scs[0][skb][sm] = s0x * s0w;

  const uint32_t xrd = (uint32_t)(r * XROW + kq * 16);
  for (int c = 0; c < nch; ++c) {
    const int buf = c & 1;
    lds_barrier();                // chunk c is visible; every wave is done with chunk c-1 (weight loads stay in flight)
    stage_store(buf ^ 1);         // chunk c+1
    stage_load(c + 2);
    // memory operations retire in order: the staging loads must stay OLDER than this trip's weight loads, or
    // the wait for them at the next barrier would drain the weight prefetch
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int kbl = 0; kbl < KC; ++kbl) {
      const v8i wa = weight_operand(kbl);
      load_w(kbl, (c + 1) * KC + kbl);
#pragma unroll
      for (int ms = 0; ms < MS; ++ms) {
        const uint8_t* xp = &xs[buf][ms * 16 * XROW + xrd + kbl * kTileK];
        const v8i xa = join(*reinterpret_cast<const v4i*>(xp), *reinterpret_cast<const v4i*>(xp + 64));
        if (MODE == kModeBlock) {
          const v4f t = mfma_16x16x128(wa, xa, v4f{0.f, 0.f, 0.f, 0.f});
          const float sc = scs[buf][kbl][ms * 16 + r];
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[ms][i] = __builtin_fmaf(t[i], sc, acc[ms][i]);
        } else {
          acc[ms] = mfma_16x16x128(wa, xa, acc[ms]);
        }
      }
    }
  }
  // ---- epilogue: lane holds n = n0w + kq*4 .. +3 of activation row ms*16 + r
  const int n = n0w + kq * 4;
  if (n >= p.N) return;
#pragma unroll
  for (int ms = 0; ms < MS; ++ms) {
    const int s = slot_of(ms * 16 + r);
    if (s >= nrows) continue;
    const int64_t orow = s;
    float v[4] = {acc[ms][0], acc[ms][1], acc[ms][2], acc[ms][3]};
    if (SPLIT) {
      *reinterpret_cast<float4*>(p.partial + ((int64_t)split * p.M + orow) * p.N + n) = make_float4(v[0], v[1], v[2], v[3]);
      continue;
    }
    if (!MOE) {
      finish4<MODE, OUT_DT, BIAS_DT>(p, n, MODE == kModeRow ? row_scale(p, orow) : 1.f, v);
    } else if (p.topk_w) {
      const float tw = p.topk_w[orow];
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] *= tw;
    }
    store4<OUT_DT>(p.C, orow * p.ldc + n, v[0], v[1], v[2], v[3]);
  }
}

// ------------------------------------------------------------------------------------------------
// The same weight stream for matrices with too few 128-row tiles to fill the chip (N below about 16 K rows): the K
// range is cut across the WAVES of a workgroup instead of across workgroups, so the partial sums meet in LDS and
// neither float partials in memory nor a reduction launch are needed.  A workgroup owns 16 * NW weight rows; its 8
// waves are NW (along n) x KS (along k), NW * KS = 8; wave (nw, ks) streams rows nw*16.. of K blocks
// [ks * kbw, (ks+1) * kbw).  No wave shares an activation K range with another (NW = 1) or only with NW - 1 others,
// so the activations skip LDS: a lane fetches its 32 bytes of a row and K block in matrix-core operand form straight
// from memory (they are L2 hits: every workgroup reads the same few rows).  The K loop has no barrier; each wave keeps
// D K blocks of weights, activations and scales in flight.  At the end the 8 accumulator sets are summed through LDS
// in ascending ks (a fixed order: results do not depend on timing) and the ks = 0 waves write the output.
// ------------------------------------------------------------------------------------------------
template <int MODE, int OUT_DT, int BIAS_DT>
__global__ __launch_bounds__(512, 2) void gemm_wavek_kernel(const GemmArgs p) {
  constexpr int MS = 1;  // up to 16 rows
  constexpr int D = 4;  // K blocks in flight per wave
  __shared__ __attribute__((aligned(16))) uint8_t wl[8][16 * kTileK];  // per wave: one K block of its 16 weight rows
  __shared__ __attribute__((aligned(16))) float red[8][MS][64][4];

  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int r = lane & 15, kq = lane >> 4;
  const int NW = p.wk_nw, nw = w % NW, ks = w / NW;
  const int n0w = (blockIdx.x * NW + nw) * 16;
  const int kb_all = p.K / kTileK;
  const int kb0 = ks * p.kb_per_split;
  const int nkb = n0w < p.N ? max(min(kb_all, kb0 + p.kb_per_split) - kb0, 0) : 0;
  const uint32_t kbytes = (uint32_t)nkb * kTileK;

  // ---- weights: line-shaped loads, re-laid out through the wave's LDS slot (as in gemm_direct_kernel)
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
  // ---- activations: lane (r, kq) takes chunks kq and 4 + kq of row ms*16 + r, the K order the weight operand has
  const rsrc_t rX = make_rsrc(p.X + (int64_t)kb0 * kTileK, nkb > 0 ? (uint32_t)((p.M - 1) * p.ldx) + kbytes : 0u);
  uint32_t voX[MS];
#pragma unroll
  for (int ms = 0; ms < MS; ++ms) {
    const int m = ms * 16 + r;
    voX[ms] = m < p.M ? (uint32_t)(m * p.ldx) + kq * 16 : kOutOfRange;
  }
  // ---- block scales: one activation scale per lane row and K block, one weight scale per K block
  const float* sxp[MS];
  const float* swp = p.sw;
  if (MODE == kModeBlock) {
#pragma unroll
    for (int ms = 0; ms < MS; ++ms) sxp[ms] = p.sx + (int64_t)min(ms * 16 + r, p.M - 1) * p.sx_m + (int64_t)kb0 * p.sx_k;
    swp = p.sw + (int64_t)(min(n0w, p.N - 1) >> 7) * p.sw_n + (int64_t)kb0 * p.sw_k;
  }

  v4i wreg[D][2], xreg[D][MS][2];
  float sxr[D][MS], swr[D];
  auto issue = [&](int slot, int kb) {
    const bool ok = kb < nkb;
    const uint32_t ko = (uint32_t)kb * kTileK;
    wreg[slot][0] = buf_load16_stream(rW, ok ? voW0 + ko : kOutOfRange);
    wreg[slot][1] = buf_load16_stream(rW, ok ? voW1 + ko : kOutOfRange);
#pragma unroll
    for (int ms = 0; ms < MS; ++ms) {
      const bool okx = ok && voX[ms] != kOutOfRange;
      xreg[slot][ms][0] = buf_load16(rX, okx ? voX[ms] + ko : kOutOfRange);
      xreg[slot][ms][1] = buf_load16(rX, okx ? voX[ms] + ko + 64 : kOutOfRange);
    }
    if (MODE == kModeBlock) {
      const int kc = min(kb, max(nkb - 1, 0));  // past the range the products are zero: any finite scale will do
#pragma unroll
      for (int ms = 0; ms < MS; ++ms) sxr[slot][ms] = sxp[ms][(int64_t)kc * p.sx_k];
      swr[slot] = swp[(int64_t)kc * p.sw_k];
    }
  };

  v4f acc[MS];
#pragma unroll
  for (int ms = 0; ms < MS; ++ms) acc[ms] = v4f{0.f, 0.f, 0.f, 0.f};

  if (nkb > 0) {
#pragma unroll
    for (int d = 0; d < D; ++d) issue(d, d);
    for (int k0 = 0; k0 < nkb; k0 += D) {
#pragma unroll
      for (int d = 0; d < D; ++d) {
        *reinterpret_cast<v4i*>(wslot + wst0) = wreg[d][0];
        *reinterpret_cast<v4i*>(wslot + wst1) = wreg[d][1];
        const v8i wa = join(*reinterpret_cast<const v4i*>(wslot + wrd0), *reinterpret_cast<const v4i*>(wslot + wrd1));
        v8i xa[MS];
        float sc[MS];
#pragma unroll
        for (int ms = 0; ms < MS; ++ms) {
          xa[ms] = join(xreg[d][ms][0], xreg[d][ms][1]);
          if (MODE == kModeBlock) sc[ms] = sxr[d][ms] * swr[d];
        }
        issue(d, k0 + d + D);
#pragma unroll
        for (int ms = 0; ms < MS; ++ms) {
          if (MODE == kModeBlock) {
            const v4f t = mfma_16x16x128(wa, xa[ms], v4f{0.f, 0.f, 0.f, 0.f});
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[ms][i] = __builtin_fmaf(t[i], sc[ms], acc[ms][i]);
          } else {
            acc[ms] = mfma_16x16x128(wa, xa[ms], acc[ms]);
          }
        }
      }
    }
  }
  // ---- the K ranges meet: every wave leaves its sums in LDS, the ks = 0 waves add them up in ascending ks
#pragma unroll
  for (int ms = 0; ms < MS; ++ms) *reinterpret_cast<v4f*>(red[w][ms][lane]) = acc[ms];
  __syncthreads();
  if (ks != 0) return;
  const int KS = 8 / NW;
  const int n = n0w + kq * 4;
  if (n >= p.N) return;
#pragma unroll
  for (int ms = 0; ms < MS; ++ms) {
    const int m = ms * 16 + r;
    if (m >= p.M) continue;
    v4f s = acc[ms];
    for (int k = 1; k < KS; ++k) {
      const v4f o = *reinterpret_cast<const v4f*>(red[k * NW + nw][ms][lane]);
      s[0] += o[0]; s[1] += o[1]; s[2] += o[2]; s[3] += o[3];
    }
    float v[4] = {s[0], s[1], s[2], s[3]};
    finish4<MODE, OUT_DT, BIAS_DT>(p, n, MODE == kModeRow ? row_scale(p, m) : 1.f, v);
    store4<OUT_DT>(p.C, (int64_t)m * p.ldc + n, v[0], v[1], v[2], v[3]);
  }
}

// ------------------------------------------------------------------------------------------------
// The same for a grouped launch of few 16-slot blocks (the first GEMM of a decode step that hits few experts of a small or sharded
// intermediate size): tiles of 128 weight rows, a wave per 16 of them over all of K, leave most CUs idle, and those at work stream
// 128 x K bytes each.  Here a workgroup owns 16 * NW rows of a block's expert and its waves cut K.  The block's rows and the slots
// they go to come from the slot table; workgroups of a block are dealt over all XCDs, so a weight line is read once per block of its
// expert.  Bound by the latency of the first lines and by launch: the first GEMM of one token, 8 experts of 512 x 7168 (29 MB, 5 us at
// the copy rate) 21.0 -> 8.8 us, 4 experts of 1024 x 4096 13.4 -> 7.3, weights out of HBM.  Eight K blocks in flight per wave are level to
// 10 % slower.
// The grid is sized for the blocks that a table aligned over the launch's own experts can have in use; a table may have more (blocks of
// other ranks' experts, blocks without slots), so a workgroup goes on by that number of blocks.  The loop costs 2 % (0.1 - 0.2 us).
// ------------------------------------------------------------------------------------------------
template <int OUT_DT>
__global__ __launch_bounds__(512, 4) void moe_wavek_kernel(const GemmArgs p) {
  constexpr int D = 4;  // K blocks in flight per wave
  __shared__ __attribute__((aligned(16))) uint8_t wl[8][16 * kTileK];  // per wave: one K block of its 16 weight rows
  __shared__ __attribute__((aligned(16))) float red[8][64][4];

  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int NW = p.wk_nw, nw = w % NW, ks = w / NW;
  const int first = (int)blockIdx.x / p.tiles_n, tile_n = (int)blockIdx.x - first * p.tiles_n;
  const int n0w = (tile_n * NW + nw) * 16;
  const int used = min(as_const_ints(p.num_post_pad)[0] / 16, p.m_blocks);
  for (int mb = first; mb < used; mb += p.walkers) {
    int lane = threadIdx.x & 63;
    asm volatile("" : "+v"(lane));  // what hangs on it is found again per block: kept across the loop the kernel took 2 - 4 % longer
    const int r = lane & 15, kq = lane >> 4;
    const int expert = as_const_ints(p.expert_ids)[mb];
    const int slot = p.sorted_ids[mb * 16 + r];
    const bool real = slot < p.num_valid;
    const int row = real ? slot / p.top_k : 0;
    const int kb_all = p.K / kTileK, kb0 = ks * p.kb_per_split;
    // an expert of another rank: no K block, zeros are stored
    const int nkb = n0w < p.N && expert >= 0 ? max(min(kb_all, kb0 + p.kb_per_split) - kb0, 0) : 0;
    const uint32_t kbytes = (uint32_t)nkb * kTileK;

    const uint8_t* const Wb = p.W + (int64_t)max(expert, 0) * p.w_expert_stride;
    const int rowsW = min(16, p.N - n0w);
    const rsrc_t rW = make_rsrc(Wb + (int64_t)n0w * p.ldw + (int64_t)kb0 * kTileK, nkb > 0 ? (uint32_t)((rowsW - 1) * p.ldw) + kbytes : 0u);
    const int wrow = lane >> 3, wc = lane & 7;
    const uint32_t voW0 = (uint32_t)(wrow * p.ldw + wc * 16), voW1 = (uint32_t)((wrow + 8) * p.ldw + wc * 16);
    uint8_t* const wslot = wl[w];
    const uint32_t wst0 = (uint32_t)(wrow * kTileK + ((wc ^ ((wrow >> 1) & 7)) << 4));
    const uint32_t wst1 = (uint32_t)((wrow + 8) * kTileK + ((wc ^ (((wrow + 8) >> 1) & 7)) << 4));
    const uint32_t wrd0 = (uint32_t)(r * kTileK + ((kq ^ ((r >> 1) & 7)) << 4));
    const uint32_t wrd1 = (uint32_t)(r * kTileK + (((4 + kq) ^ ((r >> 1) & 7)) << 4));
    const int64_t xrows = (p.num_valid + p.top_k - 1) / p.top_k;
    const rsrc_t rX = make_rsrc(p.X + (int64_t)kb0 * kTileK, nkb > 0 ? (uint32_t)((xrows - 1) * p.ldx) + kbytes : 0u);
    const uint32_t voX = (uint32_t)((int64_t)row * p.ldx) + kq * 16;
    const float* const sxp = p.sx + (int64_t)row * p.sx_m + (int64_t)kb0 * p.sx_k;
    // constant like the tables: behind a store of the loop the compiler would take vector loads for these
    const const_floats swp = (const_floats)(uintptr_t)(p.sw + (int64_t)max(expert, 0) * p.sw_expert_stride + (int64_t)(min(n0w, p.N - 1) >> 7) * p.sw_n + (int64_t)kb0 * p.sw_k);

    v4i wreg[D][2], xreg[D][2];
    float sxr[D], swr[D];
    auto issue = [&](int d, int kb) {
      const bool ok = kb < nkb, okx = ok && real;
      const uint32_t ko = (uint32_t)kb * kTileK;
      wreg[d][0] = buf_load16_stream(rW, ok ? voW0 + ko : kOutOfRange);
      wreg[d][1] = buf_load16_stream(rW, ok ? voW1 + ko : kOutOfRange);
      xreg[d][0] = buf_load16(rX, okx ? voX + ko : kOutOfRange);
      xreg[d][1] = buf_load16(rX, okx ? voX + ko + 64 : kOutOfRange);
      const int kc = min(kb, max(nkb - 1, 0));  // past the range the products are zero: any finite scale will do
      sxr[d] = sxp[(int64_t)kc * p.sx_k];
      swr[d] = swp[(int64_t)kc * p.sw_k];
    };
    v4f acc = {0.f, 0.f, 0.f, 0.f};
    if (nkb > 0) {
#pragma unroll
      for (int d = 0; d < D; ++d) issue(d, d);
      for (int k0 = 0; k0 < nkb; k0 += D) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
          *reinterpret_cast<v4i*>(wslot + wst0) = wreg[d][0];
          *reinterpret_cast<v4i*>(wslot + wst1) = wreg[d][1];
          const v8i wa = join(*reinterpret_cast<const v4i*>(wslot + wrd0), *reinterpret_cast<const v4i*>(wslot + wrd1));
          const v8i xa = join(xreg[d][0], xreg[d][1]);
          const float sc = sxr[d] * swr[d];
          const bool live = k0 + d < nkb;
          issue(d, k0 + d + D);
          const v4f t = mfma_16x16x128(wa, xa, v4f{0.f, 0.f, 0.f, 0.f});
          if (live) {
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[i] = __builtin_fmaf(t[i], sc, acc[i]);
          }
        }
      }
    }
    *reinterpret_cast<v4f*>(red[w][lane]) = acc;
    __syncthreads();
    const int n = n0w + kq * 4;
    if (ks == 0 && n < p.N && real) {
      for (int k = 1; k < 8 / NW; ++k) {
        const v4f o = *reinterpret_cast<const v4f*>(red[k * NW + nw][lane]);
        acc[0] += o[0]; acc[1] += o[1]; acc[2] += o[2]; acc[3] += o[3];
      }
      float v[4] = {acc[0], acc[1], acc[2], acc[3]};
      if (p.topk_w) {
        const float tw = p.topk_w[slot];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] *= tw;
      }
      store4<OUT_DT>(p.C, (int64_t)slot * p.ldc + n, v[0], v[1], v[2], v[3]);
    }
    if (mb + p.walkers < used) __syncthreads();  // the sums are read before the next block's are written
  }
}

}  // namespace fp8k
