// Grouped FP8 GEMM of 16- or 32-slot blocks with a short K (the second GEMM of experts whose intermediate size is sharded or
// small: K = 256 .. 1280), gfx950.
//
// It is a stream of the hit experts' weights, but in tiles of 128 weight rows x K bytes = 32 .. 128 KB: a workgroup per tile
// (gemm_direct_kernel) spends most of its life on what comes before the stream - block table, slot table, activation rows,
// first weight lines, four dependent memory latencies.  Here a workgroup owns a contiguous run of tiles of the launch's whole
// list (blocks outermost, so it changes the activation block at most once every tiles_n tiles), keeps the block's activations
// of ALL of K and their scales in LDS, and its weight stream runs on across tiles and blocks: every wave owns 16 weight rows of
// each tile of the run and keeps D K blocks of them in flight in registers, the next tile's following this tile's last.
// Finished rows are stored without a barrier; the waves meet only where the block changes.  Two workgroups share a CU, so one
// streams while the other changes blocks; that takes LDS for two, which K = 2048 with 32 slots (84 KB) does not leave.
//
// GEMM alone, a workgroup per tile with eight K blocks in flight / with four and two workgroups per CU / here: 128 experts, 4096
// rows, 128 tokens of top 6, K = 256 91 / 47 / 28 us, 16 slots 58 / 38 / 26; 256 experts, 7168 rows, 865 tokens of top 6, K = 512
// (940 MB) 367 / 228 / 224.  Up to which K it is ahead of the second: moe.hip.
//
// ACT: the rows come as the 16-bit output [slots, 2 K] of the first GEMM, and a workgroup forms silu_and_mul and the group
// quantisation of its block's rows when it puts them into LDS - bit for bit the bytes and scales of the kernel that does it
// between the two GEMMs (4.1 - 4.8 us at up to 128 tokens, and a launch).  Whole layers without / with it: 64 experts, H = 2048,
// I = 256 .. 768 1.03 .. 1.11 times, 128 experts, H = 4096, and 256, H = 7168, up to I = 512 1.01 .. 1.08 (128 experts, I = 256,
// 140 tokens 96 -> 92 us); at I = 1024 64 experts still gain 1 - 6 %, the others lose up to 7 % beyond a few tokens (288 -> 268
// without).  A block is staged by the few workgroups whose runs it spans, padding rows cost nothing.
//
// Operand layouts, the LDS round trip of the weights and the order of the K sums are gemm_direct_kernel's.
#pragma once

#include "gemm_direct.h"
#include "quant_math.h"

namespace fp8k {

constexpr int kLdsBytes = 160 * 1024;  // of a CU
constexpr int kMoeShortKMax = 1280, kMoeShortKFew = 512, kMoeShortKAct = 1024;  // with 32 and 16 slots per block (rule: moe.hip); ACT
__host__ __device__ constexpr int moe_shortk_row(int K) { return K + 16; }  // LDS row: rows of an operand fetch fall into different banks
constexpr int moe_shortk_lds(int slots, int K) {  // a workgroup's: activation rows, the waves' weight slots, scales
  return slots * moe_shortk_row(K) + 8 * 16 * kTileK + kMoeShortKMax / kTileK * slots * 4;
}
static_assert(2 * moe_shortk_lds(32, kMoeShortKMax) <= kLdsBytes, "two workgroups share a CU, and the grid has two for each");

template <int TM, int OUT_DT, bool ACT>
__global__ __launch_bounds__(512, 4) void moe_shortk_kernel(const GemmArgs p) {
  static_assert(TM == 16 || TM == 32, "16 or 32 slots per block");
  constexpr int MS = TM / 16, D = 4;
  extern __shared__ __attribute__((aligned(16))) uint8_t xs[];          // [TM][K + 16]
  __shared__ __attribute__((aligned(16))) uint8_t wl[8][16 * kTileK];   // per wave: one K block of its 16 weight rows
  __shared__ float scx[kMoeShortKMax / kTileK][TM];

  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, kq = lane >> 4;
  const int kb = p.K / kTileK, xrow = moe_shortk_row(p.K);

  // ---- the run of this workgroup: neighbours of an XCD (workgroup id mod 8) get neighbouring runs
  const int used = min(p.num_post_pad[0] / TM, p.m_blocks);
  const int64_t tiles = (int64_t)used * p.tiles_n;
  const int grid = gridDim.x;  // a multiple of 8
  const int idx = ((int)blockIdx.x & 7) * (grid >> 3) + ((int)blockIdx.x >> 3);
  const int first = (int)(tiles * idx / grid), last = (int)(tiles * (idx + 1) / grid);
  if (first >= last) return;
  const int steps = (last - first) * kb;

  // ---- weights: 16 rows per wave and tile, line-shaped loads
  const int wrow = lane >> 3, wc = lane & 7;
  const uint32_t vo0 = (uint32_t)((w * 16 + wrow) * p.ldw + wc * 16), vo1 = vo0 + (uint32_t)(8 * p.ldw);
  const uint32_t wbytes = (uint32_t)((int64_t)(p.N - 1) * p.ldw + p.K);  // of an expert; rows past N read as zero
  uint8_t* const wslot = wl[w];
  const uint32_t wst0 = (uint32_t)(wrow * kTileK + ((wc ^ ((wrow >> 1) & 7)) << 4));
  const uint32_t wst1 = (uint32_t)((wrow + 8) * kTileK + ((wc ^ (((wrow + 8) >> 1) & 7)) << 4));
  const uint32_t wrd0 = (uint32_t)(r * kTileK + ((kq ^ ((r >> 1) & 7)) << 4));
  const uint32_t wrd1 = (uint32_t)(r * kTileK + (((4 + kq) ^ ((r >> 1) & 7)) << 4));
  v4i wreg[D][2];
  float swr[D];
  // next request: K block ik of tile itile; an expert of another rank (-1) has no weights, its rows are stored as zeros
  int itile = first, ik = 0, in = first % p.tiles_n;
  rsrc_t rW = make_rsrc(p.W, 0);
  const float* swe = p.sw;
  auto expert_of_issue = [&]() {
    const int e = p.expert_ids[itile / p.tiles_n];
    rW = make_rsrc(p.W + (int64_t)max(e, 0) * p.w_expert_stride, e < 0 ? 0u : wbytes);
    swe = p.sw + (int64_t)max(e, 0) * p.sw_expert_stride;
  };
  expert_of_issue();
  auto issue = [&](int slot) {
    const bool ok = itile < last;
    const uint32_t off = (uint32_t)in * (uint32_t)(kDirTileN * p.ldw) + (uint32_t)ik * kTileK;
    wreg[slot][0] = buf_load16_stream(rW, ok ? vo0 + off : kOutOfRange);
    wreg[slot][1] = buf_load16_stream(rW, ok ? vo1 + off : kOutOfRange);
    swr[slot] = swe[(int64_t)in * p.sw_n + (int64_t)ik * p.sw_k];  // past the run: the last tile's again
    if (!ok) return;
    if (++ik == kb) {
      ik = 0;
      ++itile;
      if (++in == p.tiles_n) {
        in = 0;
        if (itile < last) expert_of_issue();
      }
      if (itile == last) in = 0;
    }
  };

  // ---- activations of a block: rows, scales and the routed weights of its slots
  const int64_t xrows = (int64_t)((p.num_valid + p.top_k - 1) / p.top_k);
  const rsrc_t rX = make_rsrc(p.X, (uint32_t)((xrows - 1) * p.ldx + (ACT ? 4 * p.K : p.K)));  // ldx: bytes
  int slot[MS];
  float tw[MS];
  bool local = true;
  auto slot_of = [&](int mb, int i) { return min(p.sorted_ids[mb * TM + i], p.num_valid); };  // num_valid: padding
  // `between` runs behind the requests: what it requests is younger, so the rows are not waited for together with it
  auto stage = [&](int mb, auto&& between) {
    local = p.expert_ids[mb] >= 0;
    const int per_row = p.K / (ACT ? 8 : 16), total = TM * per_row;  // pieces of 8 elements, of 16 bytes
    constexpr int U = ACT ? 2 : 4;
    const bool scaler = !ACT && tid < TM * kb;
    float sc = 0.f;
    for (int c0 = 0; c0 < total; c0 += U * 512) {  // uniform: every lane takes part in the first round
      v4i x[U], up[ACT ? U : 1];
      bool there[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int i = c0 + u * 512 + tid, row = i / per_row;
        const int s = i < total ? slot_of(mb, row) : p.num_valid;
        there[u] = s < p.num_valid;
        const uint32_t off = there[u] ? (uint32_t)((int64_t)(s / p.top_k) * p.ldx) + (uint32_t)(i - row * per_row) * 16 : kOutOfRange;
        x[u] = buf_load16(rX, off);
        if (ACT) up[u] = buf_load16(rX, there[u] ? off + 2u * (uint32_t)p.K : kOutOfRange);
      }
      if (c0 == 0) {
        if (scaler) {
          const int s = slot_of(mb, tid % TM);
          if (s < p.num_valid) sc = p.sx[(int64_t)(s / p.top_k) * p.sx_m + (int64_t)(tid / TM) * p.sx_k];
        }
#pragma unroll
        for (int ms = 0; ms < MS; ++ms) {
          slot[ms] = slot_of(mb, ms * 16 + r);
          tw[ms] = p.topk_w && slot[ms] < p.num_valid ? p.topk_w[slot[ms]] : 1.f;
        }
        __builtin_amdgcn_sched_barrier(0);
        between();
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int i = c0 + u * 512 + tid, row = i / per_row, piece = i - row * per_row;
        if (i >= total) continue;
        if (!ACT) {
          *reinterpret_cast<v4i*>(xs + row * xrow + piece * 16) = x[u];
          continue;
        }
        // 16 lanes hold a group of 128; rows are multiples of 16 pieces, so a group is there or padding as a whole
        uint2 o = make_uint2(0, 0);
        float scale = 0.f;
        if (there[u]) {
          Raw8<OUT_DT> g, h;
          g.v = __builtin_bit_cast(uint4, x[u]);
          h.v = __builtin_bit_cast(uint4, up[ACT ? u : 0]);
          float a[8];
          silu_mul8<OUT_DT>(g, h, a);
          const float amax = fmaxf(group_max<16>(absmax8(a)), p.q_eps);
          scale = div448<true>(amax);
          bool redo;
          o = quant8_bracket<true>(a, scale, amax, redo);
          if (__builtin_expect(redo, 0)) o = quant8_divide(a, scale);
        }
        *reinterpret_cast<uint2*>(xs + row * xrow + piece * 8) = o;
        if ((piece & 15) == 0) scx[piece >> 4][row] = scale;
      }
    }
    if (scaler) scx[tid / TM][tid % TM] = sc;
    lds_barrier();
  };

  int mb = first / p.tiles_n, tn = first - mb * p.tiles_n, t = first, k = 0;
  stage(mb, [&]() {
#pragma unroll
    for (int d = 0; d < D; ++d) issue(d);
  });

  v4f acc[MS];
#pragma unroll
  for (int ms = 0; ms < MS; ++ms) acc[ms] = v4f{0.f, 0.f, 0.f, 0.f};
  for (int f0 = 0; f0 < steps; f0 += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      if (f0 + d >= steps) break;
      *reinterpret_cast<v4i*>(wslot + wst0) = wreg[d][0];
      *reinterpret_cast<v4i*>(wslot + wst1) = wreg[d][1];
      const v8i wa = join(*reinterpret_cast<const v4i*>(wslot + wrd0), *reinterpret_cast<const v4i*>(wslot + wrd1));
      const float sw = swr[d];
      issue(d);
#pragma unroll
      for (int ms = 0; ms < MS; ++ms) {
        const uint8_t* const xp = xs + (ms * 16 + r) * xrow + k * kTileK + kq * 16;
        const v8i xa = join(*reinterpret_cast<const v4i*>(xp), *reinterpret_cast<const v4i*>(xp + 64));
        const float sc = scx[k][ms * 16 + r] * sw;
        const v4f y = mfma_16x16x128(wa, xa, v4f{0.f, 0.f, 0.f, 0.f});
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[ms][i] = __builtin_fmaf(y[i], sc, acc[ms][i]);
      }
      if (++k < kb) continue;
      // ---- the tile is finished: lane holds n .. n + 3 of activation row ms * 16 + r
      k = 0;
      const int n = tn * kDirTileN + w * 16 + kq * 4;
#pragma unroll
      for (int ms = 0; ms < MS; ++ms) {
        if (n < p.N && slot[ms] < p.num_valid) {
          float v[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) v[i] = local ? (p.topk_w ? acc[ms][i] * tw[ms] : acc[ms][i]) : 0.f;
          store4<OUT_DT>(p.C, (int64_t)slot[ms] * p.ldc + n, v[0], v[1], v[2], v[3]);
        }
        acc[ms] = v4f{0.f, 0.f, 0.f, 0.f};
      }
      ++t;
      if (++tn == p.tiles_n && t < last) {
        tn = 0;
        lds_barrier();  // every wave is done with the old block's rows
        stage(++mb, []() {});
      }
    }
  }
}

}  // namespace fp8k
