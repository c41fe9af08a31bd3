// Tiles of 64 weight rows x 64 activation rows, gfx950: products of more than 64 rows with at most about one such tile per CU, whose
// larger tiles leave most of the chip idle or need a K cut across workgroups, with float partials and a reduction launch.
//
// One workgroup of four waves per tile, each on every fourth K block of the whole range: a wave multiplies 64 x 64 (sixteen products of
// 16x16x128 per block, eight operand fragments for them out of LDS), its loads go to LDS that nobody else touches, and no barrier
// stands in the K loop.  The four sums meet in LDS at the end, in ascending order.
//
// Bound: the CU's load path.  A block is 16 KB for 512 clocks of its wave's matrix core, so 128 clocks per block with the four waves at
// work; with one tile per CU it takes 0.24 us (69 bytes a ns: 1024 x 1024 x 4096 / 8192 / 16384 12.1 / 19.8 / 35.0 us), for a tile alone on
// the chip 0.13 (64 x 64: 8.5 / 12.8 / 21.0), where plain loads of such rows out of L2 reach 120 - 150.  Measured, and no faster: loads
// straight into operand registers (half lines: 2.4 times the time), eight waves with one block each in LDS, weights two blocks ahead
// instead of one, the operands landing in registers and shared by eight waves through LDS (a barrier per four blocks).
//
// LDS, per wave: two slots of [W 64 rows x 128 B | X 64 rows x 128 B], 16-byte chunk c of row r at position c ^ ((r >> 1) & 7) as in the
// larger tiles.  The operands of a block are in registers before its products begin; behind the first of them its slot takes the
// block after next, and behind the last ones the registers, as they fall free, the next block.
#pragma once

#include "gemm_kernels.h"

namespace fp8k {

constexpr int kT64 = 64;

// all but the wave's N youngest vector-memory operations have completed
template <int N>
__device__ __forceinline__ void wait_vm() {
  static_assert(N >= 0 && N < 64, "vmcnt is a 6-bit counter");
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
  asm volatile("" ::: "memory");
}

// 256 threads; the bound of 512 keeps the kernel within 256 registers, all of which vector instructions can address
template <int MODE, int OUT_DT, int BIAS_DT, bool SPLIT>
__global__ __launch_bounds__(512) void gemm_tile64_kernel(const GemmArgs p) {
  constexpr int kOps = kT64 * kTileK;  // bytes of one operand of a K block
  constexpr int kSlot = 2 * kOps;      // weights, then activations
  constexpr int kWave = 2 * kSlot;
  constexpr uint32_t kPast = 0x80000000u;  // past every descriptor's range (64 rows of less than 8 MiB), and so with any offset added
  __shared__ __attribute__((aligned(1024))) uint8_t smem[4 * kWave];

  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  // workgroup -> (tile, K run): each XCD (workgroup id mod 8) walks a contiguous run of the work list
  int t, split;
  {
    const int ntiles = p.tiles_m * p.tiles_n;
    const int total = ntiles * p.splits;
    const int per_xcd = (total + 7) >> 3;
    const int idx = ((int)blockIdx.x & 7) * per_xcd + ((int)blockIdx.x >> 3);
    if (((int)blockIdx.x >> 3) >= per_xcd || idx >= total) return;
    split = idx / ntiles;
    t = idx - split * ntiles;
  }
  int tile_m, tile_n;
  tile_coords(t, p.tiles_m, p.tiles_n, tile_m, tile_n);
  const int m0 = tile_m * kT64, n0 = tile_n * kT64;
  const int kb_begin = SPLIT ? split * p.kb_per_split : 0;
  const int kb_end = SPLIT ? min(p.K / kTileK, kb_begin + p.kb_per_split) : p.K / kTileK;
  const int nkb = kb_end - kb_begin;
  if (nkb <= 0) return;

  // ---- global -> LDS, 1 KB (8 rows) a load
  const int rowsW = min(kT64, p.N - n0), rowsX = min(kT64, p.M - m0);
  const int kbytes = nkb * kTileK;
  const rsrc_t rW = make_rsrc(p.W + (int64_t)n0 * p.ldw + (int64_t)kb_begin * kTileK, (uint32_t)((rowsW - 1) * p.ldw + kbytes));
  const rsrc_t rX = make_rsrc(p.X + (int64_t)m0 * p.ldx + (int64_t)kb_begin * kTileK, (uint32_t)((rowsX - 1) * p.ldx + kbytes));
  uint8_t* const own = smem + w * kWave;
  const int rl = lane >> 3, cp = lane & 7;
  uint32_t voW[2], voX[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {  // chunk c of row r at position c ^ ((r >> 1) & 7)
    const int c = cp ^ ((j << 2) + (rl >> 1));
    voW[j] = (uint32_t)((j * 8 + rl) * p.ldw + c * 16);
    voX[j] = (uint32_t)((j * 8 + rl) * p.ldx + c * 16);
  }
  const uint32_t stW = (uint32_t)(16 * p.ldw), stX = (uint32_t)(16 * p.ldx);
  auto load = [&](uint8_t* slot, int kb, int g) {  // load g of block kb's sixteen: weights, then activations
    const uint32_t ko = kb < nkb ? (uint32_t)kb * kTileK : kPast;
    if (g < 8) buf_load16_to_lds(rW, voW[g & 1] + (ko + (g >> 1) * stW), 0, slot + g * 1024);
    else buf_load16_to_lds(rX, voX[g & 1] + (ko + ((g - 8) >> 1) * stX), 0, slot + g * 1024);
  };
  const int lr = lane & 15, kq = lane >> 4;
  const uint32_t fa0 = (uint32_t)(lr * kTileK + ((kq ^ ((lr >> 1) & 7)) << 4)), fa1 = fa0 ^ 64u;
  auto frag = [&](const uint8_t* grp) -> v8i {
    return join(*reinterpret_cast<const v4i*>(grp + fa0), *reinterpret_cast<const v4i*>(grp + fa1));
  };

  const uint32_t* const sx32 = reinterpret_cast<const uint32_t*>(p.sx);
  const uint32_t sxo = (uint32_t)((int64_t)min(m0 + lane, p.M - 1) * p.sx_m), sxk = (uint32_t)p.sx_k;
  const float* const swp = p.sw + (int64_t)(min(n0, p.N - 1) >> 7) * p.sw_n + (int64_t)kb_begin * p.sw_k;
  struct Scales { uint32_t x; float w; } sa, sb;
  constexpr int kScaleLoads = MODE == kModeRow ? 0 : 2;
  auto load_scales = [&](Scales& c, int kb) {
    if (MODE == kModeRow) return;
    int kc = min(kb, nkb - 1);
    asm volatile("" : "+v"(kc));  // vector loads both: the partial waits count them
    c.x = sx32[sxo + (uint32_t)(MODE == kModeScaled ? (kb_begin + kc) >> 2 : kb_begin + kc) * sxk];
    c.w = swp[(int64_t)kc * p.sw_k];
  };

  v4f acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
  v8i W[4], X[4];
  auto read_w = [&](const uint8_t* slot, int i) { W[i] = frag(slot + i * 2048); };
  auto read_x = [&](const uint8_t* slot, int i) { X[i] = frag(slot + kOps + i * 2048); };
  // The products of block kb, whose operands are in W and X.  Its slot takes block kb + 8, the operand registers, as they fall free, block
  // kb + 4 out of the other one.
  auto trip = [&](uint8_t* slot, const uint8_t* other, Scales& c, int kb) {
    uint32_t s[4] = {127, 127, 127, 127};
    int ew = 127;
    if (MODE == kModeBlock) spread_rows(__float_as_uint(__uint_as_float(c.x) * c.w), s);
    if (MODE == kModeScaled) {
      spread_rows(c.x >> (((kb_begin + kb) & 3) * 8), s);
      ew = (int)(__float_as_uint(c.w) >> 23);
    }
    asm volatile("" : "+v"(s[0]), "+v"(s[1]), "+v"(s[2]), "+v"(s[3]), "+v"(ew));
    SB();
    load_scales(c, kb + 8);
    SB();
    v4f tq[4];
#pragma unroll
    for (int k = 0; k < 20; ++k) {
      if (MODE == kModeBlock && k >= 4) {  // the products of four MFMAs wait for their scale FMAs
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[(k - 4) >> 2][k & 3][i] = __builtin_fmaf(tq[k & 3][i], __uint_as_float(s[k & 3]), acc[(k - 4) >> 2][k & 3][i]);
        SB();
      }
      if (k < 16) {
        const int ns = k >> 2, ms = k & 3;
        if (MODE == kModeBlock) tq[ms] = mfma_16x16x128(W[ns], X[ms], v4f{0.f, 0.f, 0.f, 0.f});
        else if (MODE == kModeScaled) acc[ns][ms] = mfma_16x16x128_scaled(W[ns], X[ms], acc[ns][ms], ew, (int)s[ms]);
        else acc[ns][ms] = mfma_16x16x128(W[ns], X[ms], acc[ns][ms]);
        SB();
        if (k == 2) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // every operand is out of its slot
        if (k >= 2 && k < 10) { load(slot, kb + 8, 2 * (k - 2)); load(slot, kb + 8, 2 * (k - 2) + 1); }
        SB();
        if (k == 9) wait_vm<kScaleLoads + 16>();  // block kb + 4 has landed: younger are this trip's requests
        if (k == 10) read_w(other, 0);
        if (k == 11) { read_w(other, 1); read_w(other, 2); }
        if (k >= 12) read_x(other, k - 12);
        if (k == 15) read_w(other, 3);
        SB();
      }
    }
  };
  // ---- wave w works on K blocks w, w + 4, ..
  load_scales(sa, w);
  SB();
#pragma unroll
  for (int g = 0; g < 16; ++g) load(own, w, g);
  SB();
  load_scales(sb, w + 4);
  SB();
#pragma unroll
  for (int g = 0; g < 16; ++g) load(own + kSlot, w + 4, g);
  SB();
  wait_vm<kScaleLoads + 16>();
#pragma unroll
  for (int i = 0; i < 4; ++i) { read_x(own, i); read_w(own, i); }
  SB();
  for (int kb = w; kb < nkb; kb += 8) {
    trip(own, own + kSlot, sa, kb);
    if (kb + 4 < nkb) trip(own + kSlot, own, sb, kb + 4);
  }
  wait_vm0_lgkm0();  // requests past the last block must not land on the sums

  // ---- the K shares meet in LDS: [wave][row 64][16-byte chunk c at c ^ (row & 15)]
  asm volatile("" ::: "memory");
#pragma unroll
  for (int ms = 0; ms < 4; ++ms)
#pragma unroll
    for (int ns = 0; ns < 4; ++ns) *reinterpret_cast<v4f*>(own + (ms * 16 + lr) * 256 + (((ns * 4 + kq) ^ lr) << 4)) = acc[ns][ms];
  __syncthreads();
  // wave w finishes rows 16 w .. 16 w + 15, eight at a time: lane -> row lane / 8, eight columns
  const int pc = lane & 7, n = n0 + pc * 8;
  const bool wide = (p.ldc & 7) == 0 && (reinterpret_cast<uintptr_t>(p.C) & 15) == 0;
#pragma unroll
  for (int half = 0; half < 2; ++half) {
    const int row = w * 16 + half * 8 + (lane >> 3), m = m0 + row;
    float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint8_t* const q = smem + k * kWave + row * 256;
      const v4f lo = *reinterpret_cast<const v4f*>(q + (((2 * pc) ^ (row & 15)) << 4));
      const v4f hi = *reinterpret_cast<const v4f*>(q + (((2 * pc + 1) ^ (row & 15)) << 4));
#pragma unroll
      for (int i = 0; i < 4; ++i) { v[i] += lo[i]; v[4 + i] += hi[i]; }
    }
    if (m >= p.M || n >= p.N) continue;
    if (SPLIT) {
      float* const o = p.partial + ((int64_t)split * p.M + m) * p.N + n;
      *reinterpret_cast<float4*>(o) = make_float4(v[0], v[1], v[2], v[3]);
      *reinterpret_cast<float4*>(o + 4) = make_float4(v[4], v[5], v[6], v[7]);
      continue;
    }
    float lo[4] = {v[0], v[1], v[2], v[3]}, hi[4] = {v[4], v[5], v[6], v[7]};
    const float sm = MODE == kModeRow ? row_scale(p, m) : 1.f;
    finish4<MODE, OUT_DT, BIAS_DT>(p, n, sm, lo);
    finish4<MODE, OUT_DT, BIAS_DT>(p, n + 4, sm, hi);
    u16* const o = (u16*)p.C + (int64_t)m * p.ldc + n;
    const uint2 ol = pack4<OUT_DT>(lo[0], lo[1], lo[2], lo[3]), oh = pack4<OUT_DT>(hi[0], hi[1], hi[2], hi[3]);
    if (wide) {
      *reinterpret_cast<uint4*>(o) = make_uint4(ol.x, ol.y, oh.x, oh.y);
    } else {
      *reinterpret_cast<uint2*>(o) = ol;
      *reinterpret_cast<uint2*>(o + 4) = oh;
    }
  }
}

}  // namespace fp8k
