// Tiles of 128 weight rows x 128 or 64 activation rows x 128 (k) for the shapes between the weight-streaming kernels and the
// 256x256 tile kernel: 33 .. some thousand activation rows whose 256x256 tiles are fewer than the chip has CUs.
//
// What bounds them is the serial chain of a K block - barrier, operands out of LDS, MFMAs, every wave issuing some hundred
// instructions at eight to nine clocks each with two waves to a SIMD - more than any unit's throughput: with 128 activation rows a
// block takes 0.38 us from L2-resident operands, 0.43 - 0.50 with weights out of HBM, for 0.21 us of matrix-core time; with 64
// rows 0.30 and 0.35 - 0.45 for half the work.  So, against the form before (32x32x64 products, four stages, the scales of every
// block through LDS; 128 rows only): half-height tiles where they bring more workgroups (us, block scales, weights of 1 GB
// in turn: 156 x 4544 x 3968 15.2 -> 12.5, 709 x 704 x 3840 15.4 -> 12.2, 432 x 4224 x 11776 47.7 -> 42.4, 200 x 7168 x 2304 11.2 -> 9.2),
// 16x16x128 products, and fewer instructions per block: the scales come for four K blocks at once.
//
// 8 wavefronts, 2 along n x 4 along m (64 x 32 each), or 4 x 2 (32 x 32) with 64 rows.  LDS: five stages of [W 128 rows x 128 B |
// X 128 rows x 128 B], six with 64 rows - so that three or four K blocks are in flight per CU: these shapes read every weight line
// from HBM exactly once.  (Rings of their own for weights and activations, loaded by waves of their own so that the weights could
// run five or six blocks ahead, were no faster.)  The operands take the same road as in gemm_tile256_kernel (buffer_load ... lds
// with the complete offset in the range-checked per-lane operand, 16-byte chunk c of row r at chunk position c ^ ((r >> 1) & 7)).
//
// One barrier per K block, which waits for loads only.  After the barrier of block `it` a wave issues the MFMAs of block it-1 from
// one of two register sets, and between them fetches its operands of block `it` from LDS into the other set and refills the
// stage of block it-2, whose operands every wave has used by then.
//
// SPLIT: the K range is cut into p.splits runs, every (tile, run) pair is one workgroup, float partials go to
// the workspace [split][M][N] for splitk_reduce_kernel.
#pragma once

#include "gemm_kernels.h"

namespace fp8k {

constexpr int kT128 = 128;  // weight rows of a tile, and activation rows of the larger one
// activation rows TM of a tile: 128 or 64; LDS stages (the whole LDS) and the bytes of one: W rows, X rows
constexpr int t128_stages(int tm) { return tm == 128 ? 5 : 6; }
constexpr int t128_stage(int tm) { return (kT128 + tm) * kTileK; }

template <int MODE, int OUT_DT, int BIAS_DT, bool SPLIT, int TM>
__global__ __launch_bounds__(512, 1) void gemm_tile128_kernel(const GemmArgs p) {
  static_assert(TM == 64 || TM == 128, "activation rows of a tile");
  constexpr int NST = t128_stages(TM), kStage = t128_stage(TM), kXOff = kT128 * kTileK;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[NST * kStage];
  constexpr int XL = TM / 64, LPB = 2 + XL;  // activation loads, all loads of a wave per K block
  // waves along n x along m: 2 x 4 (64 x 32 each) or 4 x 2 (32 x 32 each), in 16 x 16 products
  constexpr int NWN = TM == 128 ? 2 : 4, NT = kT128 / NWN / 16, MT = 2, NM = NT * MT;

  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int wn = w % NWN, wm = w / NWN;
  const int wrow = wn * (NT * 16), xrow = wm * 32;

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
  const int m0 = tile_m * TM, n0 = tile_n * kT128;

  const int kb_begin = SPLIT ? split * p.kb_per_split : 0;
  const int kb_end = SPLIT ? min(p.K / kTileK, kb_begin + p.kb_per_split) : p.K / kTileK;
  const int nkb = kb_end - kb_begin;
  if (nkb <= 0) return;

  // ---- global -> LDS: wave w brings rows [16w, 16w+16) of W and [8 XL w, 8 XL (w+1)) of X, 1 KB (8 rows) a load
  const int rowsW = min(kT128, p.N - n0), rowsX = min(TM, p.M - m0);
  const int kbytes = p.K - kb_begin * kTileK;
  // batched launches (grid y): every batch entry has its own operands and output, the scales are shared
  const uint8_t* const Wb = p.W + (int64_t)blockIdx.y * p.batch_w;
  const uint8_t* const Xb = p.X + (int64_t)blockIdx.y * p.batch_x;
  u16* const Cb = (u16*)p.C + (int64_t)blockIdx.y * p.batch_c;
  const rsrc_t rW = make_rsrc(Wb + (int64_t)n0 * p.ldw + (int64_t)kb_begin * kTileK, (uint32_t)((rowsW - 1) * p.ldw + kbytes));
  const rsrc_t rX = make_rsrc(Xb + (int64_t)m0 * p.ldx + (int64_t)kb_begin * kTileK, (uint32_t)((rowsX - 1) * p.ldx + kbytes));
  const int rl = lane >> 3, cp = lane & 7;
  uint32_t voW[2], voX[XL];
#pragma unroll
  for (int j = 0; j < 2; ++j) voW[j] = (uint32_t)((w * 16 + j * 8 + rl) * p.ldw + (cp ^ ((j << 2) + (rl >> 1))) * 16);
#pragma unroll
  for (int j = 0; j < XL; ++j) {  // swizzle key of row r: (r >> 1) & 7
    const int r = (w * XL + j) * 8 + rl;
    voX[j] = (uint32_t)(r * p.ldx + (cp ^ ((r >> 1) & 7)) * 16);
  }
  auto load_block = [&](int stage, int kstep, int j) {  // j: 0, 1 weights; 2 .. LPB-1 activations
    const uint32_t ko = (uint32_t)kstep * kTileK;
    if (j < 2) buf_load16_to_lds(rW, voW[j] + ko, 0, smem + stage + w * 2048 + j * 1024);
    else buf_load16_to_lds(rX, voX[j - 2] + ko, 0, smem + stage + kXOff + (w * XL + j - 2) * 1024);
  };

  // ---- LDS -> MFMA operands: row lr of a 16-row group, 16-byte chunks kq and kq + 4 at their swizzled places
  const int lr = lane & 15, kq = lane >> 4;
  const uint32_t fa0 = (uint32_t)(lr * kTileK + ((kq ^ ((lr >> 1) & 7)) << 4)), fa1 = fa0 ^ 64u;
  auto frag = [&](const uint8_t* grp) -> v8i {
    return join(*reinterpret_cast<const v4i*>(grp + fa0), *reinterpret_cast<const v4i*>(grp + fa1));
  };

  v4f acc[NT][MT];
#pragma unroll
  for (int ns = 0; ns < NT; ++ns)
#pragma unroll
    for (int ms = 0; ms < MT; ++ms) acc[ns][ms] = v4f{0.f, 0.f, 0.f, 0.f};

  // ---- scales, four K blocks (a group) at a time: lane (lr, kq) fetches those of its two activation rows for block 4c + kq, lane l
  // the weight scale of block 4c + l % 4, one group ahead; at the start of a group the activation scales are handed round.
  uint32_t sxo[MT];
#pragma unroll
  for (int ms = 0; ms < MT; ++ms) sxo[ms] = (uint32_t)((int64_t)min(m0 + xrow + ms * 16 + lr, p.M - 1) * p.sx_m);
  const float* const swp = p.sw + (int64_t)(min(n0, p.N - 1) >> 7) * p.sw_n;
  uint32_t sxr[MT] = {0, 0}, sx[MT][4];
  float swr = 0.f, sw = 0.f;
  auto request_scales = [&](int c) {
    if (MODE == kModeRow) return;
    const int kx = kb_begin + min(4 * c + kq, nkb - 1), kw = kb_begin + min(4 * c + (lane & 3), nkb - 1);
    // scaled mode: int32 words of four UE8M0 bytes (K blocks 4j..4j+3 of a row), sx_k = word stride
    const uint32_t k = (uint32_t)(MODE == kModeScaled ? kx >> 2 : kx) * (uint32_t)p.sx_k;
#pragma unroll
    for (int ms = 0; ms < MT; ++ms) sxr[ms] = reinterpret_cast<const uint32_t*>(p.sx)[sxo[ms] + k];
    swr = swp[(int64_t)kw * p.sw_k];
  };
  auto take_scales = [&](int c) {
    if (MODE == kModeRow) return;
    const int kx = kb_begin + min(4 * c + kq, nkb - 1);
#pragma unroll
    for (int ms = 0; ms < MT; ++ms) spread_rows(MODE == kModeScaled ? sxr[ms] >> ((kx & 3) * 8) : sxr[ms], sx[ms]);
    sw = swr;
    // formed here, in front of the next request: moved behind it, the copies would wait for it
    asm volatile("" : "+v"(sw));
#pragma unroll
    for (int ms = 0; ms < MT; ++ms) asm volatile("" : "+v"(sx[ms][0]), "+v"(sx[ms][1]), "+v"(sx[ms][2]), "+v"(sx[ms][3]));
  };

  struct Operands { v8i W[NT], X[MT]; };  // of one K block
  Operands oa, ob;
  // MFMA k of a K block: weight group k / 2, activation group k % 2.  Block mode: the product waits in tq[k % 4] and is folded into its
  // accumulator in front of MFMA k + 4, the last four of a block with that block's scales (sp) during the next one.
  v4f tq[4];
  float sp[MT] = {0.f, 0.f};
#pragma unroll
  for (int i = 0; i < 4; ++i) tq[i] = v4f{0.f, 0.f, 0.f, 0.f};
  auto F = [&](int k) {
    if (MODE == kModeBlock) {
      const int ns = k / MT, ms = k % MT;
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[ns][ms][i] = __builtin_fmaf(tq[k & 3][i], sp[ms], acc[ns][ms][i]);
    }
  };
  // the MFMAs of a K block, number q of its group; between(k) runs behind MFMA k
  auto compute = [&](auto q_c, const Operands& o, auto&& between) {
    constexpr int q = decltype(q_c)::value;
    const float swq = MODE == kModeRow ? 1.f : __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, sw), q * 0x55, 0xf, 0xf, true));
    const int sqw = (int)(__float_as_uint(swq) >> 23);
#pragma unroll
    for (int k = 0; k < NM; ++k) {
      const int ns = k / MT, ms = k % MT;
      F((k + NM - 4) % NM);
      SB();
      if (MODE == kModeBlock) tq[k & 3] = mfma_16x16x128(o.W[ns], o.X[ms], v4f{0.f, 0.f, 0.f, 0.f});
      else if (MODE == kModeScaled) acc[ns][ms] = mfma_16x16x128_scaled(o.W[ns], o.X[ms], acc[ns][ms], sqw, (int)sx[ms][q]);
      else acc[ns][ms] = mfma_16x16x128(o.W[ns], o.X[ms], acc[ns][ms]);
      SB();
      if (k == 3 && MODE == kModeBlock) {
#pragma unroll
        for (int j = 0; j < MT; ++j) sp[j] = __uint_as_float(sx[j][q]) * swq;
      }
      between(k);
      SB();
    }
  };
  // fragment f of a K block: the activation groups, then the weight groups
  auto read_frag = [&](Operands& o, const uint8_t* st, int f) {
    if (f < MT) o.X[f] = frag(st + kXOff + (xrow + f * 16) * kTileK);
    else o.W[f - MT] = frag(st + (wrow + (f - MT) * 16) * kTileK);
  };
  int st_rd = 0, st_fill = (NST - 2) * kStage;  // stage of block `it`, stage that block it + NST - 2 goes to
  auto next = [&](int st) { return st == (NST - 1) * kStage ? 0 : st + kStage; };
  // trip `it` (u = it % 4): block `it` has landed everywhere; its operands from LDS into `rd`, the MFMAs of block it-1 from `use`, and
  // the loads of block it + NST - 2 into the stage of block it-2.  Every wave has used that block's operands by now, so the barrier
  // does not have to wait for LDS reads: they run on across it.
  auto trip = [&](auto u_c, int it, Operands& rd, const Operands& use) {
    constexpr int u = decltype(u_c)::value;
    constexpr bool first = u == 1;  // block it-1 starts a group of scales
    // younger than block it's loads: those of the blocks behind it, and a group's scales if requested meanwhile
    constexpr int back = NST - 3, scale_ops = MODE != kModeRow && ((u + 3) & 3) >= 1 && ((u + 3) & 3) <= back ? MT + 1 : 0;
    const uint8_t* const st = smem + st_rd;
    const int kf = it + NST - 2, fill = st_fill;
    SB();  // the MFMAs issued before stay in front of this wait
    vm_barrier<back * LPB + scale_ops>();
    if (first) {
      take_scales(it >> 2);
      request_scales((it >> 2) + 1);
      SB();
    }
    compute(std::integral_constant<int, (u + 3) & 3>{}, use, [&](int i) {
      if (i * 2 < NT + MT) { read_frag(rd, st, i * 2); read_frag(rd, st, i * 2 + 1); }
      if (NM == 8 ? i >= 3 && i - 3 < LPB : i >= 1) load_block(fill, kf, NM == 8 ? i - 3 : i - 1);
    });
    st_rd = next(st_rd);
    st_fill = next(st_fill);
  };
  const std::integral_constant<int, 0> c0{};
  const std::integral_constant<int, 1> c1{};
  const std::integral_constant<int, 2> c2{};
  const std::integral_constant<int, 3> c3{};

  // ---- prologue: blocks 0 .. NST-3 and one more into their stages, block 0's operands into `oa`
  request_scales(0);
  SB();
#pragma unroll
  for (int s = 0; s < NST - 2; ++s)
#pragma unroll
    for (int j = 0; j < LPB; ++j) load_block(s * kStage, s, j);
  SB();
  vm_barrier<(NST - 3) * LPB>();
#pragma unroll
  for (int j = 0; j < LPB; ++j) load_block((NST - 2) * kStage, NST - 2, j);
#pragma unroll
  for (int f = 0; f < NT + MT; ++f) read_frag(oa, smem, f);
  st_rd = kStage;
  st_fill = (NST - 1) * kStage;
  // ---- block b is fetched in trip b and multiplied in trip b+1; even blocks live in `oa`, odd ones in `ob`
  auto nothing = [](int) {};
  int it = 1;
  for (; it + 3 < nkb; it += 4) {
    trip(c1, it, ob, oa);
    trip(c2, it + 1, oa, ob);
    trip(c3, it + 2, ob, oa);
    trip(c0, it + 3, oa, ob);
  }
  if (it >= nkb) {
    take_scales(it >> 2);
    compute(c0, oa, nothing);
  } else {
    trip(c1, it, ob, oa);
    if (it + 1 >= nkb) {
      compute(c1, ob, nothing);
    } else {
      trip(c2, it + 1, oa, ob);
      if (it + 2 >= nkb) {
        compute(c2, oa, nothing);
      } else {
        trip(c3, it + 2, ob, oa);
        compute(c3, ob, nothing);
      }
    }
  }
#pragma unroll
  for (int k = NM - 4; k < NM; ++k) F(k);

  const int nrows = p.M;
  const auto col_of = [&](int ns) { return n0 + wrow + ns * 16 + kq * 4; };
  const auto row_of = [&](int ms) { return m0 + xrow + ms * 16 + lr; };
  if (SPLIT) {
    wait_vm0();  // the unread loads past the last block must not land in LDS after the workgroup has gone
    float* part = p.partial + (int64_t)split * p.M * p.N;
#pragma unroll
    for (int ms = 0; ms < MT; ++ms)
#pragma unroll
      for (int ns = 0; ns < NT; ++ns) {
        const int m = row_of(ms), n = col_of(ns);
        if (m >= nrows || n >= p.N) continue;
        *reinterpret_cast<float4*>(part + (int64_t)m * p.N + n) = make_float4(acc[ns][ms][0], acc[ns][ms][1], acc[ns][ms][2], acc[ns][ms][3]);
      }
    return;
  }

  if (MODE == kModeRow) {
    float sa[MT];
#pragma unroll
    for (int ms = 0; ms < MT; ++ms) sa[ms] = row_of(ms) < nrows ? row_scale(p, row_of(ms)) : 1.f;
    finish_rows<NT, MT, BIAS_DT>(p, sa, [&](int j) { return col_of(j); }, [&](int j, int ms, int q, auto f) { acc[j][ms][q] = f(acc[j][ms][q]); });
  }
  // conversion of one run of 4 n
  auto out_quad = [&](int ns, int ms) -> uint2 {
    const v4f v = acc[ns][ms];
    uint2 o;
    if (OUT_DT == FP8K_BF16) {
      o.x = pack_bf16x2(v[0], v[1]);
      o.y = pack_bf16x2(v[2], v[3]);
    } else {
      o.x = f32_to_f16_bits(v[0]) | (f32_to_f16_bits(v[1]) << 16);
      o.y = f32_to_f16_bits(v[2]) | (f32_to_f16_bits(v[3]) << 16);
    }
    return o;
  };

  // Finished tiles leave through LDS so that a store instruction writes whole 128- or 64-byte row segments: each wave
  // re-lays its 32 rows out in a private slot, 16-byte chunks XOR-swizzled by the row.
  const bool wide = (p.ldc & 7) == 0 && (reinterpret_cast<uintptr_t>(Cb) & 15) == 0;
  if (wide) {
    wait_vm0_lgkm0();                // own stray loads have landed ...
    __builtin_amdgcn_s_barrier();    // ... and so have everyone's; every wave has taken its last operands
    asm volatile("" ::: "memory");
    constexpr int CPR = NT * 2, RPI = 64 / CPR;  // 16-byte chunks of a row, rows per store instruction
    const int rr = lane / CPR, pc = lane % CPR;
    float bias8[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (MODE == kModeBlock && p.bias) load_bias8<BIAS_DT>(p.bias, min(n0 + wrow + (pc << 3), p.N - 8), bias8);
    uint8_t* const ep = smem + w * (32 * CPR * 16);
#pragma unroll
    for (int ms = 0; ms < MT; ++ms)
#pragma unroll
      for (int ns = 0; ns < NT; ++ns)
        *reinterpret_cast<uint2*>(ep + (ms * 16 + lr) * (CPR * 16) + (((ns * 2 + (kq >> 1)) ^ (lr & (CPR - 1))) << 4) + (kq & 1) * 8) = out_quad(ns, ms);
    __builtin_amdgcn_wave_barrier();  // one wave's LDS accesses complete in order
#pragma unroll
    for (int i = 0; i < 32 / RPI; ++i) {
      const int r = i * RPI + rr;
      uint4 o = *reinterpret_cast<const uint4*>(ep + r * (CPR * 16) + ((pc ^ (r & (CPR - 1))) << 4));
      if (MODE == kModeBlock && p.bias) o = add_bias8<OUT_DT>(o, bias8);
      const int m = m0 + xrow + r;
      const int n = n0 + wrow + (pc << 3);
      if (m < nrows && n < p.N) *reinterpret_cast<uint4*>(Cb + (int64_t)m * p.ldc + n) = o;
    }
    return;
  }

  wait_vm0();
#pragma unroll
  for (int ms = 0; ms < MT; ++ms)
#pragma unroll
    for (int ns = 0; ns < NT; ++ns) {
      const int m = row_of(ms), n = col_of(ns);
      if (m >= nrows || n >= p.N) continue;
      if (MODE == kModeBlock && p.bias) {
        float v[4] = {acc[ns][ms][0], acc[ns][ms][1], acc[ns][ms][2], acc[ns][ms][3]};
        finish4<MODE, OUT_DT, BIAS_DT>(p, n, 1.f, v);
        store4<OUT_DT>(Cb, (int64_t)m * p.ldc + n, v[0], v[1], v[2], v[3]);
        continue;
      }
      *reinterpret_cast<uint2*>(Cb + (int64_t)m * p.ldc + n) = out_quad(ns, ms);
    }
}

}  // namespace fp8k
