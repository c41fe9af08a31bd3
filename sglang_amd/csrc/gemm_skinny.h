// FP8 GEMM for decode batches (9 .. 64 activation rows), gfx950: no float partials, no reduction launch.
//
// The weights are a stream from HBM that has to be spread over all CUs.  With narrow strips of weight rows per workgroup (16 or
// 32: one or two to a CU) every workgroup can run over the whole of K and write finished rows; the price is that each of them
// reads ALL activations, M x K bytes against 16 .. 64 x K bytes of weights.  They are L2 hits, and the CU's load path (64 bytes a
// clock, five times the CU's share of HBM) has room for them - if they come as whole lines and if waiting for them does not
// empty the weight stream.  Loads of a wave return in order, so a wave that waits for an activation line also waits for every
// weight line it asked for before.  Hence two kinds of waves:
//
//   * eight streaming waves, NW along n (16 weight rows each) x KS = 8 / NW along k.  A trip covers eight K blocks,
//     U consecutive ones per wave; a wave keeps its next D K blocks of weights in flight in registers (whole-line loads, re-laid
//     out through a private LDS slot as in gemm_direct_kernel) and takes its activations from LDS.  It never waits for a load
//     of anybody else's.
//   * NL loading waves, which bring the activations of a trip - [rows][1 KB], 1 KB per instruction straight into LDS - one
//     or two trips ahead and wait for them in front of the trip's barrier.
//
// One LDS-only barrier per trip.  The 16-byte chunk c of row r lies at chunk c ^ (r & 15) of its row, which spreads the 16 rows of
// an operand fetch over all banks.  At the end the KS partial sums meet in LDS in ascending order, as in gemm_wavek_kernel.
//
// GEMM alone, bf16, against what ran before (K cut across workgroups with partials, or across the waves of one whose lanes fetched
// their own activations), weights rotated over 600 MB: 32 x 4096 x 4096 10.6 -> 7.6 us, 24 x 7168 x 16384 32.4 -> 26.7 (117 MB: 4.4
// TB/s), 64 x 4096 x 4096 15.2 -> 10.3, 13 x 12224 x 3968 19.4 -> 11.8.
#pragma once

#include "gemm_direct.h"

namespace fp8k {

constexpr int kSkinnyMaxM = 64;
constexpr int kSkinnyTrip = 8;  // K blocks of a trip

template <int TM, int NW, int MODE, int OUT_DT, int BIAS_DT>
__global__ __launch_bounds__(TM <= 32 ? 640 : 768) void gemm_skinny_kernel(const GemmArgs p) {
  static_assert(TM == 16 || TM == 32 || TM == 64, "16, 32 or 64 rows");
  constexpr int TRIP = kSkinnyTrip, ROW = TRIP * kTileK;  // K blocks of a trip, bytes of a staged row
  static_assert((NW == 1 || NW == 2 || NW == 4) && TRIP * NW % 8 == 0, "waves along n");
  constexpr int MS = TM / 16, KS = 8 / NW, U = TRIP / KS;  // U: K blocks of a trip per wave
  // K blocks of weights in flight per wave (whole trips): more is slower, 24 x 7168 x 16384 25.2 us with 8 against 24.6
  constexpr int D = NW == 1 ? 2 : 4;
  constexpr int NL = TM <= 32 ? 2 : 4;       // loading waves
  constexpr int NI = TM * ROW / 1024 / NL;   // instructions of a trip per loading wave
  constexpr int STAGE = TM * ROW;
  constexpr int NST = 3 * STAGE + 8 * 2048 <= 160 * 1024 ? 3 : 2;  // trips' worth of activations beside the weight slots
  __shared__ __attribute__((aligned(16))) uint8_t xs[NST * STAGE];     // the sums at the end
  __shared__ __attribute__((aligned(16))) uint8_t wl[8][16 * kTileK];  // per streaming wave: one K block of its 16 weight rows
  static_assert(MS * 8 * 1024 <= NST * STAGE, "room for the sums");

  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int kb_all = p.K / kTileK, trips = (kb_all + TRIP - 1) / TRIP;
  // an XCD (workgroup id mod 8) takes a contiguous run of strips: neighbours complete each other's output lines in its L2
  const int per_xcd = (p.tiles_n + 7) >> 3;
  const int strip = ((int)blockIdx.x & 7) * per_xcd + ((int)blockIdx.x >> 3);
  if (((int)blockIdx.x >> 3) >= per_xcd || strip >= p.tiles_n) return;

  if (w >= 8) {
    // ---- loading wave: instruction i brings rows [i R, (i + 1) R) of the stage, the lane at chunk c of a row its chunk c ^ (row & 15)
    constexpr int LR = ROW / 16, R = 64 / LR;  // lanes per row, rows per instruction
    const int i0 = (w - 8) * NI;
    const int sub = lane / LR, pos = lane % LR;
    const rsrc_t rX = make_rsrc(p.X, (uint32_t)((p.M - 1) * p.ldx + p.K));
    auto load = [&](int c) {
      uint8_t* const st = xs + (c % NST) * STAGE;
#pragma unroll
      for (int j = 0; j < NI; ++j) {
        const int row = (i0 + j) * R + sub;
        const uint32_t k = (uint32_t)c * (uint32_t)ROW + (uint32_t)(pos ^ (row & 15)) * 16u;
        buf_load16_to_lds(rX, row < p.M && k < (uint32_t)p.K ? (uint32_t)(row * p.ldx) + k : kOutOfRange, 0, st + (i0 + j) * 1024);
      }
    };
    load(0);
    if (NST == 3 && trips > 1) load(1);
    for (int c = 0; c < trips; ++c) {
      // everything but the youngest trip's loads (three stages) has to be there; past the last trip nothing younger exists
      if (NST == 2 || c + 1 >= trips) lds_barrier<0>();
      else lds_barrier<NI>();
      if (c + NST - 1 < trips) load(c + NST - 1);
    }
    lds_barrier();
    lds_barrier();
    return;
  }

  // ---- streaming wave
  const int r = lane & 15, kq = lane >> 4;
  const int nw = w % NW, ks = w / NW;
  const int n0w = (strip * NW + nw) * 16;
  const int rowsW = min(16, p.N - n0w);
  const rsrc_t rW = make_rsrc(p.W + (int64_t)n0w * p.ldw, rowsW > 0 ? (uint32_t)((rowsW - 1) * p.ldw + p.K) : 0u);
  const int wrow = lane >> 3, wc = lane & 7;
  const uint32_t voW0 = (uint32_t)(wrow * p.ldw + wc * 16), voW1 = (uint32_t)((wrow + 8) * p.ldw + wc * 16);
  uint8_t* const wslot = wl[w];
  const uint32_t wst0 = (uint32_t)(wrow * kTileK + ((wc ^ ((wrow >> 1) & 7)) << 4));
  const uint32_t wst1 = (uint32_t)((wrow + 8) * kTileK + ((wc ^ (((wrow + 8) >> 1) & 7)) << 4));
  const uint32_t wrd0 = (uint32_t)(r * kTileK + ((kq ^ ((r >> 1) & 7)) << 4));
  const uint32_t wrd1 = (uint32_t)(r * kTileK + (((4 + kq) ^ ((r >> 1) & 7)) << 4));
  // operand fetch of K block u: row ms * 16 + r, chunks (ks * U + u) * 8 + kq and + 4, at their swizzled places
  auto xr = [&](int u, int half) { return (uint32_t)(r * ROW + ((((ks * U + u) * 8 + kq + half * 4) ^ r) << 4)); };
  const float* sxp[MS];
  const float* swp = p.sw;
  if (MODE == kModeBlock) {
#pragma unroll
    for (int ms = 0; ms < MS; ++ms) sxp[ms] = p.sx + (int64_t)min(ms * 16 + r, p.M - 1) * p.sx_m;
    swp = p.sw + (int64_t)(min(n0w, p.N - 1) >> 7) * p.sw_n;
  }

  v4i wreg[D][2];
  float sxr[D][MS], swr[D];
  auto issue = [&](int slot, int c, int u) {
    const int kb = c * TRIP + ks * U + u;
    const bool ok = kb < kb_all;
    const uint32_t ko = (uint32_t)kb * kTileK;
    wreg[slot][0] = buf_load16_stream(rW, ok ? voW0 + ko : kOutOfRange);
    wreg[slot][1] = buf_load16_stream(rW, ok ? voW1 + ko : kOutOfRange);
    if (MODE == kModeBlock) {
      const int kc = min(kb, kb_all - 1);  // past the range the products are zero: any finite scale will do
#pragma unroll
      for (int ms = 0; ms < MS; ++ms) sxr[slot][ms] = sxp[ms][(int64_t)kc * p.sx_k];
      swr[slot] = swp[(int64_t)kc * p.sw_k];
    }
  };
  v4f acc[MS];
#pragma unroll
  for (int ms = 0; ms < MS; ++ms) acc[ms] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int d = 0; d < D; ++d) issue(d, d / U, d % U);
  constexpr int UT = D / U;  // trips per turn of the ring
  static_assert(D % U == 0, "whole trips");
  int st = 0;  // stage of the trip
  for (int c0 = 0; c0 < trips; c0 += UT) {
#pragma unroll
    for (int ct = 0; ct < UT; ++ct) {
      if (c0 + ct >= trips) break;
      lds_barrier();  // the trip's activations are there; nobody reads the stage before it any more
      const uint8_t* const xp = xs + st * STAGE;
      st = st + 1 == NST ? 0 : st + 1;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int d = ct * U + u;
        *reinterpret_cast<v4i*>(wslot + wst0) = wreg[d][0];
        *reinterpret_cast<v4i*>(wslot + wst1) = wreg[d][1];
        const v8i wa = join(*reinterpret_cast<const v4i*>(wslot + wrd0), *reinterpret_cast<const v4i*>(wslot + wrd1));
        float sc[MS];
        if (MODE == kModeBlock) {
#pragma unroll
          for (int ms = 0; ms < MS; ++ms) sc[ms] = sxr[d][ms] * swr[d];
        }
        issue(d, c0 + ct + UT, u);
#pragma unroll
        for (int ms = 0; ms < MS; ++ms) {
          const v8i xa = join(*reinterpret_cast<const v4i*>(xp + ms * 16 * ROW + xr(u, 0)), *reinterpret_cast<const v4i*>(xp + ms * 16 * ROW + xr(u, 1)));
          if (MODE == kModeBlock) {
            const v4f t = mfma_16x16x128(wa, xa, v4f{0.f, 0.f, 0.f, 0.f});
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[ms][i] = __builtin_fmaf(t[i], sc[ms], acc[ms][i]);
          } else {
            acc[ms] = mfma_16x16x128(wa, xa, acc[ms]);
          }
        }
      }
    }
  }
  // ---- the K shares meet: every wave leaves its sums where the activations were, the ks = 0 waves add them up in ascending ks
  lds_barrier();
#pragma unroll
  for (int ms = 0; ms < MS; ++ms) *reinterpret_cast<v4f*>(xs + ((w * MS + ms) * 64 + lane) * 16) = acc[ms];
  lds_barrier();
  if (ks != 0) return;
  const int n = n0w + kq * 4;
  if (n >= p.N) return;
#pragma unroll
  for (int ms = 0; ms < MS; ++ms) {
    const int m = ms * 16 + r;
    if (m >= p.M) continue;
    v4f s = acc[ms];
    for (int k = 1; k < KS; ++k) {
      const v4f o = *reinterpret_cast<const v4f*>(xs + (((k * NW + nw) * MS + ms) * 64 + lane) * 16);
      s[0] += o[0]; s[1] += o[1]; s[2] += o[2]; s[3] += o[3];
    }
    float v[4] = {s[0], s[1], s[2], s[3]};
    finish4<MODE, OUT_DT, BIAS_DT>(p, n, MODE == kModeRow ? row_scale(p, m) : 1.f, v);
    store4<OUT_DT>(p.C, (int64_t)m * p.ldc + n, v[0], v[1], v[2], v[3]);
  }
}

}  // namespace fp8k
