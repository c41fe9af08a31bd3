// Grouped (MoE) block-FP8 GEMM of a short K (256 .. 512) for experts with about a hundred and more token slots, gfx950: the second
// GEMM of experts whose intermediate size is sharded or small.
//
// A 256x256 tile of two to four K blocks is mostly set-up and write-out: one workgroup fills a CU, so nothing else runs while it
// waits for its first blocks or re-lays out its result.  Here K is short enough for a wave to hold the activations of ALL of it in
// registers - 32 slots x K bytes, 16 registers per K block - and a workgroup walks a run of weight tiles with them:
//   * four waves, each 32 slots x all 128 weight rows of a tile: an activation byte is fetched once per run and no LDS goes to it;
//   * the weights, the only stream left, pass through a ring of four 16 KB stages that runs on across the tiles of the run, three K
//     blocks ahead;
//   * 64 KB of ring and a private 4 KB per wave for the layout changes (activations in, result out) make 80 KB: two workgroups share
//     a CU, and one's write-out and waits hide behind the other's matrix-core work.
// The stores of a tile are as many for every wave with real slots (padding rows store out of range, which drops them), so that the
// partial vmcnt waits of the next trips can count them and the stream does not drain at a write-out.
//
// GEMM alone, us, 256x256 tiles -> here: 64 experts, 7168 rows, 32000 slots, K = 512 276 -> 212 (235 MB of weights and 459 of results: 108
// at the copy rate); 128 experts, 24000 slots, K = 256 171 -> 122; 64 experts, 4096 rows, 12380 slots, K = 256 58 -> 46.  Taken alone,
// the stores are 45 of the 180 us that the first of these adds to its layer, the products 33, the weight loads 38, the layout change 29,
// the set-up 5: they overlap badly with only two wavefronts to a SIMD, which the registers do not let grow.  Non-temporal stores or
// weight loads are level or slower.
//
// The products, their order and the scaling are moe_stream256_kernel's with float scales: the results are the same bits.
#pragma once

#include "gemm_kernels.h"

namespace fp8k {

// A store to LDS while direct loads to other parts of it are in flight.  The compiler cannot tell the parts apart and would put
// s_waitcnt vmcnt(0) in front of an ordinary one: the weight stream would drain at every write-out.  A wave's LDS accesses complete in
// order, so its own later reads need no wait.
__device__ __forceinline__ void lds_store8(uint32_t p, uint2 v) {
  asm volatile("ds_write_b64 %0, %1" ::"v"(p), "v"((uint64_t)v.x | ((uint64_t)v.y << 32)) : "memory");
}

constexpr int kMoeRegxMaxKb = 4;     // K blocks whose activations fit beside the accumulators
constexpr int kMoeRegxScales = 64;   // weight scales of a run: one per lane

// 256-slot blocks, activation scales in sorted order; p.tiles_n: runs per 128-slot part of a block
template <int KB, int OUT_DT>
__global__ __launch_bounds__(512) void moe_regx_kernel(const GemmArgs p) {  // 256 threads; the bound keeps a wave within 256 registers
  static_assert(KB >= 2 && KB <= kMoeRegxMaxKb, "K blocks");
  constexpr int NS = 4, STAGE = 128 * kTileK, AHEAD = 3, LW = 4, STORES = 8;  // LW: wave loads of a stage; STORES: per tile and wave
  __shared__ __attribute__((aligned(1024))) uint8_t smem[4 * STAGE + 4 * 4096];

  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int lr = lane & 31, h = lane >> 5, rl = lane >> 3, cp = lane & 7;
  const int nrows = p.num_valid;

  // ---- work: the parts of a block are neighbours on an XCD (workgroup id mod 8) and read the same weights
  const int j = (int)blockIdx.x >> 3;
  const MoeItem item = moe_work_item(p, (j >> 1) * 8 + ((int)blockIdx.x & 7));
  if (item.mb < 0) return;
  const const_ints ids = as_const_ints(p.sorted_ids);
  const int s0 = item.mb * p.block_m + (j & 1) * 128, ws0 = s0 + w * 32;
  if (ids[s0] >= nrows) return;             // all padding: real slots come first
  const bool active = ids[ws0] < nrows;
  const int tiles = p.N >> 7;
  const int t_first = (int)((int64_t)tiles * item.tile_n / p.tiles_n), t_last = (int)((int64_t)tiles * (item.tile_n + 1) / p.tiles_n);
  const int nt = t_last - t_first;

  int rid[4];  // slot ids of rows i * 8 + rl: those whose 16-byte chunk cp this lane loads and stores
#pragma unroll
  for (int i = 0; i < 4; ++i) rid[i] = p.sorted_ids[ws0 + i * 8 + rl];
  const rsrc_t rC = make_rsrc(p.C, (uint32_t)(((int64_t)(nrows - 1) * p.ldc + p.N) * 2));
  uint32_t voC[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) voC[i] = rid[i] < nrows ? (uint32_t)((int64_t)rid[i] * p.ldc * 2) + cp * 16u : 0xF0000000u;

  if (item.expert < 0) {  // an expert of another rank: zeros
    for (int n = t_first * 128; n < t_last * 128; n += 64)
#pragma unroll
      for (int i = 0; i < 4; ++i) __builtin_amdgcn_raw_buffer_store_b128(v4i{0, 0, 0, 0}, rC, voC[i], n * 2, 0);
    return;
  }

  // ---- the weight stream: a wave load covers 8 rows (lane: row lane / 8, 16-byte chunk lane % 8, stored at c ^ ((row >> 1) & 7))
  const rsrc_t rW = make_rsrc(p.W + (int64_t)item.expert * p.w_expert_stride + (int64_t)t_first * 128 * p.ldw,
                              (uint32_t)((int64_t)(nt * 128 - 1) * p.ldw + p.K));
  uint32_t voW[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) voW[q] = (uint32_t)((w * 32 + q * 8 + rl) * p.ldw + (cp ^ ((q << 2) + (rl >> 1))) * 16);
  const uint32_t w16 = (uint32_t)(16 * p.ldw), wtile = (uint32_t)(128 * p.ldw);
  auto issue = [&](int t, int kb, int stage) {  // past the run: out of range, nothing moves
    const uint32_t ko = t < nt ? (uint32_t)t * wtile + (uint32_t)kb * kTileK : 0xF0000000u;
    uint8_t* const base = smem + stage * STAGE + w * (LW * 1024);
    asm volatile("" : "+v"(voW[0]), "+v"(voW[1]));  // or the sums with every K block's offset are kept
#pragma unroll
    for (int q = 0; q < LW; ++q) buf_load16_to_lds(rW, t < nt ? voW[q & 1] + (ko + (q >> 1) * w16) : 0xF0000000u, 0, base + q * 1024);
  };
#pragma unroll
  for (int g = 0; g < AHEAD; ++g) issue(g / KB, g % KB, g);
  __builtin_amdgcn_sched_barrier(0);

  // ---- activations and scales of the wave's 32 slots, the weight scales of the run (lane t * KB + kb)
  uint8_t* const own = smem + 4 * STAGE + w * 4096;
  const int swz = (lr >> 1) & 7;
  uint32_t fa = (uint32_t)(lr * kTileK + (((h * 2) ^ swz) << 4));  // lane part of an operand fetch: row lr, chunk h * 2
  auto frag = [&](const uint8_t* grp, int ks) -> v8i {              // 32 bytes of K half ks
    const v4i lo = *reinterpret_cast<const v4i*>(grp + (fa ^ (ks << 6))), hi = *reinterpret_cast<const v4i*>(grp + (fa ^ (ks << 6) ^ 16));
    return v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  };
  // 16-byte chunk cp of row i * 8 + rl of the private 4 KB
  const uint32_t st0 = (uint32_t)(rl * 128 + ((cp ^ (rl >> 1)) << 4));
  auto chunk = [&](int i) -> v4i* { return reinterpret_cast<v4i*>(own + ((st0 ^ ((i & 1) << 6)) + i * 1024)); };
  v8i xa[KB][2];
  float sx[KB], rs = 1.f, swl = 0.f;
  if (active) {
    const rsrc_t rX = make_rsrc(p.X, (uint32_t)((int64_t)((nrows + p.top_k - 1) / p.top_k - 1) * p.ldx + p.K));
    v4i xr[KB][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t vo = rid[i] < nrows ? (uint32_t)((int64_t)(rid[i] / p.top_k) * p.ldx) + cp * 16u : 0xF0000000u;
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) xr[kb][i] = __builtin_amdgcn_raw_buffer_load_b128(rX, vo + kb * kTileK, 0, 0);
    }
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) sx[kb] = p.sx[(int64_t)(ws0 + lr) * p.sx_m + (int64_t)kb * p.sx_k];
    if (p.topk_w) rs = p.topk_w[min((uint32_t)p.sorted_ids[ws0 + lr], (uint32_t)(nrows - 1))];  // padding slots are not stored
    const int tl = min(lane / KB, nt - 1), kl = lane - lane / KB * KB;
    swl = p.sw[(int64_t)item.expert * p.sw_expert_stride + (int64_t)(t_first + tl) * p.sw_n + (int64_t)kl * p.sw_k];
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {  // one wave's LDS accesses complete in order
#pragma unroll
      for (int i = 0; i < 4; ++i) *chunk(i) = xr[kb][i];
      __builtin_amdgcn_wave_barrier();
      xa[kb][0] = frag(own, 0);
      xa[kb][1] = frag(own, 1);
      __builtin_amdgcn_wave_barrier();
    }
  }
  wait_vm0();  // the waits below count from here
  __builtin_amdgcn_sched_barrier(0);

  auto run = [&](auto active_c) {
    constexpr bool ACTIVE = decltype(active_c)::value;
    int stage = 0;
    for (int t = 0; t < nt; ++t) {
      v16f acc[NS], z;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        z[r] = 0.f;
#pragma unroll
        for (int ns = 0; ns < NS; ++ns) acc[ns][r] = 0.f;
      }
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        // Everything but the two youngest weight blocks has landed, and every wave has left the stage of the block before.  The stores of
        // the last tile stand behind this block's request as long as that was made in front of them: in the first three trips of a tile.
        int later = t;
        asm volatile("" : "+s"(later));  // or the first tile gets a copy of the loop, which spills
        if (ACTIVE && kb < AHEAD && later > 0) lds_barrier<(AHEAD - 1) * LW + STORES>();
        else lds_barrier<(AHEAD - 1) * LW>();
        __builtin_amdgcn_sched_barrier(0);
        issue(t + (kb + AHEAD) / KB, (kb + AHEAD) % KB, (stage + AHEAD) & 3);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (ACTIVE) {
          const uint8_t* const sw_ = smem + stage * STAGE;
          asm volatile("" : "+v"(fa));  // as above
          const float sc = sx[kb] * __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, swl), t * KB + kb));
          v16f tq[2];
          v8i wf[2][2];
          wf[0][0] = frag(sw_, 0);
          wf[0][1] = frag(sw_, 1);
          auto fold = [&](int ns) {
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[ns][r] = __builtin_fmaf(tq[ns & 1][r], sc, acc[ns][r]);
          };
#pragma unroll
          for (int ns = 0; ns < NS; ++ns) {  // the next rows' operands and the last product's scaling in the shadow of the matrix core
            if (ns + 1 < NS) {
              wf[(ns + 1) & 1][0] = frag(sw_ + (ns + 1) * 4096, 0);
              wf[(ns + 1) & 1][1] = frag(sw_ + (ns + 1) * 4096, 1);
            }
            tq[ns & 1] = mfma_32x32x64(wf[ns & 1][0], xa[kb][0], z);
            tq[ns & 1] = mfma_32x32x64(wf[ns & 1][1], xa[kb][1], tq[ns & 1]);
            if (ns > 0) fold(ns - 1);
            __builtin_amdgcn_sched_barrier(0);
          }
          fold(NS - 1);
        }
        stage = (stage + 1) & 3;
      }
      if constexpr (ACTIVE) {
        // ---- 32 slots x 64 columns at a time through the private 4 KB: every store instruction writes eight whole lines
        __builtin_amdgcn_sched_barrier(0);
        // 8 bytes of chunk 0 of row lr; opaque, or the eight addresses made from it are kept across the K loop
        uint32_t wr = (uint32_t)(uintptr_t)(lds_ptr_t)own + (uint32_t)(lr * 128 + (swz << 4) + h * 8);
        asm volatile("" : "+v"(wr));
        const uint32_t so = (uint32_t)(t_first + t) * 256u;
#pragma unroll
        for (int ps = 0; ps < 2; ++ps) {
#pragma unroll
          for (int nr = 0; nr < 8; ++nr) {
            const int ns = ps * 2 + (nr >> 2), rg = nr & 3;
            float v[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              v[r] = acc[ns][rg * 4 + r] * rs;
              if (OUT_DT == FP8K_F16) asm("" : "+v"(v[r]));  // rounded to float32 first, as in the other forms (no v_fma_mix)
            }
            lds_store8(wr ^ (uint32_t)(nr << 4), pack4<OUT_DT>(v[0], v[1], v[2], v[3]));
          }
          __builtin_amdgcn_wave_barrier();
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const v4i o = *chunk(i);
            __builtin_amdgcn_raw_buffer_store_b128(o, rC, voC[i], so + ps * 128u, 0);
          }
          __builtin_amdgcn_wave_barrier();
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  if (active) run(std::integral_constant<bool, true>{});
  else run(std::integral_constant<bool, false>{});
  wait_vm0();  // the out-of-range requests of the last trips still point at the ring
}

}  // namespace fp8k
