// FP8 (OCP e4m3fn) quantisation kernels for gfx950: per-token-group, per-token, per-tensor.
//
// All three are HBM-bound streaming kernels: 16-byte loads, 8/16-byte stores, one pass over the
// input held in registers, amax by DPP lane exchange inside the wavefront.
#include <algorithm>

#include "fp8k_common.h"
#include "quant_math.h"

namespace fp8k {

// ------------------------------------------------------------------------------------------------
// per-token-group quant
//
// The unit of work is a 1 KB "segment" (64 lanes x 8 elements = 512 columns of one row, i.e.
// GPW = 512/GROUP groups; LPG = GROUP/8 adjacent lanes form a group).  A wavefront owns SEG segments:
// SEG consecutive ones of the flat input (contiguous memory whenever K is a multiple of 512) for
// row-major scales, or the same segment of SEG consecutive rows (ROWFAST) for scale layouts whose rows
// are the contiguous direction.  It loads them all with 16-byte nontemporal loads before touching the
// first, and writes each back as one 8-byte store per lane.  Both streams are used once, so they
// bypass cache retention.
// ------------------------------------------------------------------------------------------------
__device__ __forceinline__ uint4 load16_stream(const void* p) {
  const v4i v = __builtin_nontemporal_load(reinterpret_cast<const v4i*>(p));
  return make_uint4((uint32_t)v[0], (uint32_t)v[1], (uint32_t)v[2], (uint32_t)v[3]);
}
__device__ __forceinline__ void store8_stream(void* p, uint2 o) {
  v2i v;
  v[0] = (int)o.x;
  v[1] = (int)o.y;
  __builtin_nontemporal_store(v, reinterpret_cast<v2i*>(p));
}

template <int DT>
__device__ __forceinline__ void load_stream(Raw8<DT>& r, const void* base, int64_t elem) {
  if constexpr (DT == FP8K_F32) {
    const float* p = (const float*)base + elem;
    const uint4 a = load16_stream(p), b = load16_stream(p + 4);
    r.lo = make_float4(__uint_as_float(a.x), __uint_as_float(a.y), __uint_as_float(a.z), __uint_as_float(a.w));
    r.hi = make_float4(__uint_as_float(b.x), __uint_as_float(b.y), __uint_as_float(b.z), __uint_as_float(b.w));
  } else {
    r.v = load16_stream((const u16*)base + elem);
  }
}

// MASKED: the M rows are E experts x m_max slots; only the first masked_m[e] slots of expert e are quantised
// (the others are neither read nor written), and the scale of slot i of expert e sits at e*se + i*sm + g*sg.
template <int DT, int GROUP, int KIND, int SEG, bool ROWFAST, bool FUSE, bool MASKED>
__global__ __launch_bounds__(256) void group_quant_kernel(const void* __restrict__ x, uint8_t* __restrict__ q,
                                                          void* __restrict__ s, int M, int G, int64_t K,
                                                          int nseg_row, float eps, int64_t sm, int64_t sg,
                                                          const int32_t* __restrict__ masked_m, int m_max, int64_t se) {
  const int64_t XK = FUSE ? 2 * K : K;  // elements per input row
  auto scale_row = [&](int r) -> int64_t {  // offset of the scales of row r
    if (!MASKED) return (int64_t)r * sm;
    const int e = r / m_max;
    return (int64_t)e * se + (int64_t)(r - e * m_max) * sm;
  };
  constexpr int LPG = GROUP / 8;
  constexpr int GPW = 64 / LPG;
  static_assert(KIND != FP8K_SCALE_UE8M0_PACKED || GROUP == 128, "packed UE8M0 scales need 128-element groups");

  const int lane = threadIdx.x & 63;
  const int lg = lane / LPG, li = lane % LPG;
  // A wave owns SEG tasks (row, segment-in-row).  Row-major scales: SEG consecutive segments, i.e. contiguous
  // memory and SEG*GPW consecutive scales.  ROWFAST (scales whose rows are contiguous: column-major float,
  // packed UE8M0): the same segment of SEG consecutive rows, so that the SEG scales of a group column are
  // adjacent words that leave the wave together.
  const unsigned wave = blockIdx.x * 4u + (unsigned)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const unsigned total = (unsigned)M * (unsigned)nseg_row;
  int row, sr;
  if (ROWFAST) {
    row = (int)(wave / (unsigned)nseg_row) * SEG;
    sr = (int)(wave % (unsigned)nseg_row);
    if (row >= M) return;
  } else {
    if (wave * SEG >= total) return;
    row = (int)(wave * SEG / (unsigned)nseg_row);
    sr = (int)(wave * SEG - (unsigned)row * (unsigned)nseg_row);
  }

  Raw8<DT> raw[SEG], up[FUSE ? SEG : 1];
  int rows[SEG], segs[SEG];
  bool act[SEG];  // wave-uniform: task j exists
  float scv[SEG];
  uint32_t redo_mask = 0;
#pragma unroll
  for (int j = 0; j < SEG; ++j) {
    rows[j] = row;
    segs[j] = sr;
    act[j] = ROWFAST ? row < M : wave * SEG + j < total;
    if (MASKED && act[j]) {
      const int e = row / m_max;
      act[j] = row - e * m_max < masked_m[e];
    }
    if (act[j]) {
      const int g = sr * GPW + lg;
      // lanes past the last group of the row re-read the last group and store nothing
      const int64_t col = (int64_t)(g < G ? g : G - 1) * GROUP + li * 8;
      load_stream<DT>(raw[j], x, (int64_t)row * XK + col);
      if (FUSE) load_stream<DT>(up[j], x, (int64_t)row * XK + K + col);
    }
    if (ROWFAST) {
      ++row;
    } else if (++sr == nseg_row) {
      sr = 0;
      ++row;
    }
  }
#pragma unroll
  for (int j = 0; j < SEG; ++j) {
    if (act[j]) {  // wave-uniform
      const int g = segs[j] * GPW + lg;
      const bool valid = g < G;
      float a[8];
      if (FUSE) silu_mul8<DT>(raw[j], up[FUSE ? j : 0], a);
      else raw[j].unpack(a);
      const float amax = fmaxf(group_max<LPG>(absmax8(a)), eps);
      const float sc = div448<DT != FP8K_F32>(amax);
      uint2 out;
      if (KIND == FP8K_SCALE_UE8M0_PACKED) {
        // round the scale up to a power of two; x / 2^e == x * 2^-e exactly
        const uint32_t b = __float_as_uint(fmaxf(sc, 1e-10f));
        const uint32_t e = (b >> 23) + ((b & 0x7fffffu) != 0u);
        const float rinv = __uint_as_float((254u - e) << 23);
        out.x = cvt4_fp8(a[0] * rinv, a[1] * rinv, a[2] * rinv, a[3] * rinv);
        out.y = cvt4_fp8(a[4] * rinv, a[5] * rinv, a[6] * rinv, a[7] * rinv);
        const uint32_t eb = valid ? e : 0u;  // bytes of groups past the row end stay zero
        const uint32_t w = (uint32_t)__builtin_amdgcn_readlane((int)eb, 0) |
                           ((uint32_t)__builtin_amdgcn_readlane((int)eb, 16) << 8) |
                           ((uint32_t)__builtin_amdgcn_readlane((int)eb, 32) << 16) |
                           ((uint32_t)__builtin_amdgcn_readlane((int)eb, 48) << 24);
        if (lane == 0) reinterpret_cast<uint32_t*>(s)[(int64_t)segs[j] * sg + scale_row(rows[j])] = w;
      } else if (KIND == FP8K_SCALE_UE8M0_F32) {
        // the same power of two, stored as a float at the place of a float scale
        const uint32_t b = __float_as_uint(fmaxf(sc, 1e-10f));
        const uint32_t e = (b >> 23) + ((b & 0x7fffffu) != 0u);
        const float rinv = __uint_as_float((254u - e) << 23);
        out.x = cvt4_fp8(a[0] * rinv, a[1] * rinv, a[2] * rinv, a[3] * rinv);
        out.y = cvt4_fp8(a[4] * rinv, a[5] * rinv, a[6] * rinv, a[7] * rinv);
        if (valid && li == 0) reinterpret_cast<float*>(s)[scale_row(rows[j]) + (int64_t)g * sg] = __uint_as_float(e << 23);
      } else {
        bool redo;
        out = quant8_bracket<DT != FP8K_F32>(a, sc, amax, redo);
        redo_mask |= (redo & valid) ? (1u << j) : 0u;
        scv[j] = sc;
        if (valid && li == 0) reinterpret_cast<float*>(s)[scale_row(rows[j]) + (int64_t)g * sg] = sc;
      }
      if (valid) store8_stream(q + (int64_t)rows[j] * K + (int64_t)g * GROUP + li * 8, out);
    }
  }
  // cold: lanes whose bracket was inconclusive reload their 8 values (still in cache) and divide
  if (KIND == FP8K_SCALE_F32 && __builtin_expect(redo_mask != 0, 0)) {
#pragma unroll 1
    for (int j = 0; j < SEG; ++j) {
      if (redo_mask & (1u << j)) {
        float sc = scv[0];
#pragma unroll
        for (int i = 1; i < SEG; ++i) sc = j == i ? scv[i] : sc;
        int row = rows[0], seg = segs[0];
#pragma unroll
        for (int i = 1; i < SEG; ++i) { row = j == i ? rows[i] : row; seg = j == i ? segs[i] : seg; }
        const int64_t col = (int64_t)(seg * GPW + lg) * GROUP + li * 8;
        Raw8<DT> again;
        again.load(x, (int64_t)row * XK + col);
        float a[8];
        if (FUSE) {
          Raw8<DT> again_up;
          again_up.load(x, (int64_t)row * XK + K + col);
          silu_mul8<DT>(again, again_up, a);
        } else {
          again.unpack(a);
        }
        store8_stream(q + (int64_t)row * K + col, quant8_divide(a, sc));
      }
    }
  }
}

// Segments per wave: four keep enough bytes in flight to stream a large input; up to a wave per wave slot of the chip (8192 segments,
// 4 M elements) what counts is that the latency of one segment, not of four, stands in front of the product.  Whole linears,
// quantisation and product, us, four / one: 32 x 4096 x 4096 10.7 / 9.5, 64 x 4096 x 4096 13.5 / 12.6, 200 x 7168 x 2304 15.0 / 14.1,
// 128 x 7168 x 16384 41.3 / 40.5, 1000 x 24576 x 1536 50.6 / 49.8; level above (2048 x 7168 x 2304 41.2 / 41.2).
// The kernel alone, row-major / column-major / packed UE8M0 scales: 32 x 4096 3.16 / 2.21, 3.23 / 2.33, 3.05 / 2.28; 512 x 8192 (8192
// segments) 5.02 / 4.03, 4.94 / 4.06, 4.63 / 3.88; with silu_and_mul in front, which loads two streams, 32 x 4096 4.41 / 2.68, 4.38 /
// 2.70, 4.23 / 2.69 and 512 x 8192 7.84 / 6.05, 7.70 / 6.07, 7.17 / 5.72; one segment in all is level in every form.
constexpr int64_t kFewSegments = 8192;
template <int DT, int GROUP, int KIND, int SEG, bool FUSE, bool MASKED>
static int launch_group_quant_seg(const void* x, void* q, void* s, int64_t M, int64_t K, float eps, int64_t sm, int64_t sg,
                                  hipStream_t st, const int32_t* masked_m, int m_max, int64_t se) {
  constexpr int GPW = 64 / (GROUP / 8);
  const int G = (int)(K / GROUP);
  const int nseg_row = (G + GPW - 1) / GPW;
  const int64_t total = M * nseg_row;
  if (total > 0x7fffffffLL / SEG) return fail(FP8K_ERR_INVALID, "group_quant: input too large for one launch");
  const bool rowfast = KIND == FP8K_SCALE_UE8M0_PACKED || sm < sg;  // rows of the scale tensor are contiguous
  const int64_t waves = rowfast ? (M + SEG - 1) / SEG * nseg_row : (total + SEG - 1) / SEG;
  const dim3 grid((unsigned)((waves + 3) / 4)), block(256);
  if (rowfast)
    hipLaunchKernelGGL((group_quant_kernel<DT, GROUP, KIND, SEG, true, FUSE, MASKED>), grid, block, 0, st, x, (uint8_t*)q, s,
                       (int)M, G, K, nseg_row, eps, sm, sg, masked_m, m_max, se);
  else
    hipLaunchKernelGGL((group_quant_kernel<DT, GROUP, KIND, SEG, false, FUSE, MASKED>), grid, block, 0, st, x, (uint8_t*)q, s,
                       (int)M, G, K, nseg_row, eps, sm, sg, masked_m, m_max, se);
  return check_launch("group_quant");
}
template <int DT, int GROUP, int KIND, bool FUSE = false, bool MASKED = false>
static int launch_group_quant(const void* x, void* q, void* s, int64_t M, int64_t K, float eps, int64_t sm, int64_t sg,
                              hipStream_t st, const int32_t* masked_m = nullptr, int m_max = 1, int64_t se = 0) {
  if constexpr (GROUP == 128 && DT != FP8K_F32 && !MASKED) {
    if (M * ((K / GROUP + 3) / 4) <= kFewSegments)
      return launch_group_quant_seg<DT, GROUP, KIND, 1, FUSE, MASKED>(x, q, s, M, K, eps, sm, sg, st, masked_m, m_max, se);
  }
  return launch_group_quant_seg<DT, GROUP, KIND, 4, FUSE, MASKED>(x, q, s, M, K, eps, sm, sg, st, masked_m, m_max, se);
}

template <int DT, int KIND>
static int dispatch_group(const void* x, void* q, void* s, int64_t M, int64_t K, int64_t group, float eps, int64_t sm,
                          int64_t sg, hipStream_t st) {
  if (KIND == FP8K_SCALE_UE8M0_PACKED) {
    if (group != 128) return fail(FP8K_ERR_INVALID, "group_quant: packed UE8M0 scales require group_size 128");
    return launch_group_quant<DT, 128, KIND>(x, q, s, M, K, eps, sm, sg, st);
  }
  switch (group) {
    case 16: return launch_group_quant<DT, 16, FP8K_SCALE_F32>(x, q, s, M, K, eps, sm, sg, st);
    case 32: return launch_group_quant<DT, 32, FP8K_SCALE_F32>(x, q, s, M, K, eps, sm, sg, st);
    case 64: return launch_group_quant<DT, 64, FP8K_SCALE_F32>(x, q, s, M, K, eps, sm, sg, st);
    case 128: return launch_group_quant<DT, 128, FP8K_SCALE_F32>(x, q, s, M, K, eps, sm, sg, st);
    case 256: return launch_group_quant<DT, 256, FP8K_SCALE_F32>(x, q, s, M, K, eps, sm, sg, st);
    case 512: return launch_group_quant<DT, 512, FP8K_SCALE_F32>(x, q, s, M, K, eps, sm, sg, st);
  }
  return fail(FP8K_ERR_INVALID, "group_quant: group_size %lld not in {16,32,64,128,256,512}", (long long)group);
}

// ------------------------------------------------------------------------------------------------
// per-token quant: WPR waves to a row, the row held in registers between the amax and the cast
// ------------------------------------------------------------------------------------------------
// Bound by the latency of one row: load, maximum, store (large inputs by HBM: 8192 x 4096 runs at 5.9 TB/s).  The loads of a row
// are all in flight together; issued one by one behind the use of the one before, as conditional loads are, a row of 14336
// columns waited for memory seven times.  HOLD is what the row needs, no more: empty turns cost up to 30 % on short rows.
template <int DT, int WPR, int HOLD>
__global__ __launch_bounds__(256) void token_quant_kernel(const void* __restrict__ x, uint8_t* __restrict__ q,
                                                          float* __restrict__ s, int M, int64_t K) {
  static_assert(WPR == 1 || WPR == 4, "a wave or a workgroup to a row");
  constexpr int LANES = WPR * 64;  // HOLD chunks x LANES x 8 elements stay in registers
  __shared__ float red[4];
  const int tid = (int)threadIdx.x % LANES;
  const int64_t row = (int64_t)blockIdx.x * (4 / WPR) + (int)threadIdx.x / LANES;
  const int nchunk = row < M ? (int)(K / 8) : 0;  // lanes of a row past the end take part in the barrier only
  Raw8<DT> raw[HOLD];
  // every load of the row is on its way before the first value is looked at
#pragma unroll
  for (int c = 0; c < HOLD; ++c) {
    const int ch = c * LANES + tid;
    raw[c].zero();
    if (ch < nchunk) raw[c].load(x, row * K + (int64_t)ch * 8);
  }
  float m = 0.f;
#pragma unroll
  for (int c = 0; c < HOLD; ++c) {
    float a[8];
    raw[c].unpack(a);
    m = fmaxf(m, absmax8(a));
  }
  for (int ch = HOLD * LANES + tid; ch < nchunk; ch += LANES) {
    Raw8<DT> t;
    t.load(x, row * K + (int64_t)ch * 8);
    float a[8];
    t.unpack(a);
    m = fmaxf(m, absmax8(a));
  }
  m = group_max<64>(m);
  if constexpr (WPR > 1) {
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  }
  const float sc = m / kFp8Max;
  if (tid == 0 && row < M) s[row] = sc;
  const float inv = (sc == 0.f) ? 0.f : 1.0f / sc;
  auto emit = [&](const float(&a)[8], int ch) {
    float y[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) y[i] = fmaxf(fminf(a[i] * inv, kFp8Max), -kFp8Max);
    uint2 o;
    o.x = cvt4_fp8(y[0], y[1], y[2], y[3]);
    o.y = cvt4_fp8(y[4], y[5], y[6], y[7]);
    *reinterpret_cast<uint2*>(q + row * K + (int64_t)ch * 8) = o;
  };
#pragma unroll
  for (int c = 0; c < HOLD; ++c) {
    const int ch = c * LANES + tid;
    if (ch < nchunk) {
      float a[8];
      raw[c].unpack(a);
      emit(a, ch);
    }
  }
  for (int ch = HOLD * LANES + tid; ch < nchunk; ch += LANES) {
    Raw8<DT> t;
    t.load(x, row * K + (int64_t)ch * 8);
    float a[8];
    t.unpack(a);
    emit(a, ch);
  }
}

// A wave to a row where that fills its lanes with two chunks, four with many rows; else a workgroup.  us, one workgroup with eight
// conditional loads (before) / a workgroup / a wave: 1 x 4096 2.35 / 2.10 / 2.66, 200 x 18432 6.18 / 5.02 / -, 2048 x 4096 6.66 / 6.03
// / 6.55, 500 x 2048 2.56 / 2.37 / 2.52, 8192 x 2048 11.86 / 11.15 / 10.16, 64 x 1024 2.38 / 2.17 / 2.12, 8192 x 1024 8.60 / 7.78
// / 6.06, 4096 x 512 4.73 / 4.41 / 3.14.
template <int DT>
static void launch_token_quant(const void* x, uint8_t* q, float* s, int64_t M, int64_t K, hipStream_t st) {
#define FP8K_TOKEN(WPR, HOLD) \
  hipLaunchKernelGGL((token_quant_kernel<DT, WPR, HOLD>), dim3((unsigned)((M + 4 / WPR - 1) / (4 / WPR))), dim3(256), 0, st, x, q, s, (int)M, K)
  if (K <= 1024) FP8K_TOKEN(1, 2);
  else if (K <= 2048 && M >= 1024) FP8K_TOKEN(1, 4);
  else if (K <= 2048) FP8K_TOKEN(4, 1);
  else if (K <= 4096) FP8K_TOKEN(4, 2);
  else if (K <= 8192) FP8K_TOKEN(4, 4);
  else FP8K_TOKEN(4, 8);
#undef FP8K_TOKEN
}

__device__ __forceinline__ float block_max_256(float v, float* red) {
  v = group_max<64>(v);
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) red[w] = v;
  __syncthreads();
  v = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  __syncthreads();
  return v;
}

// ------------------------------------------------------------------------------------------------
// per-tensor quant: grid-stride absmax with one atomic max per workgroup, then the cast
// ------------------------------------------------------------------------------------------------
template <int DT>
__device__ __forceinline__ float load1(const void* x, int64_t i) {
  if (DT == FP8K_F32) return ((const float*)x)[i];
  if (DT == FP8K_BF16) return __uint_as_float((uint32_t)((const u16*)x)[i] << 16);
  return f16_bits_to_f32(((const u16*)x)[i]);
}

template <int DT>
__global__ __launch_bounds__(256) void tensor_absmax_kernel(const void* __restrict__ x, float* __restrict__ s,
                                                            int64_t numel) {
  __shared__ float red[4];
  const int64_t nchunk = numel / 8;
  const int64_t stride = (int64_t)gridDim.x * 256;
  float m = 0.f;
  for (int64_t ch = (int64_t)blockIdx.x * 256 + threadIdx.x; ch < nchunk; ch += stride) {
    Raw8<DT> t;
    t.load(x, ch * 8);
    float a[8];
    t.unpack(a);
    m = fmaxf(m, absmax8(a));
  }
  for (int64_t i = nchunk * 8 + (int64_t)blockIdx.x * 256 + threadIdx.x; i < numel; i += stride)
    m = fmaxf(m, fabsf(load1<DT>(x, i)));
  m = block_max_256(m, red);
  // non-negative floats order like their bit patterns
  if (threadIdx.x == 0) atomicMax(reinterpret_cast<unsigned int*>(s), __float_as_uint(m / kFp8Max));
}

template <int DT>
__global__ __launch_bounds__(256) void tensor_quant_kernel(const void* __restrict__ x, uint8_t* __restrict__ q,
                                                           const float* __restrict__ s, int64_t numel) {
  const float inv = 1.0f / s[0];
  const int64_t nchunk = numel / 8;
  const int64_t stride = (int64_t)gridDim.x * 256;
  for (int64_t ch = (int64_t)blockIdx.x * 256 + threadIdx.x; ch < nchunk; ch += stride) {
    Raw8<DT> t;
    t.load(x, ch * 8);
    float a[8], y[8];
    t.unpack(a);
#pragma unroll
    for (int i = 0; i < 8; ++i) y[i] = fmaxf(fminf(a[i] * inv, kFp8Max), -kFp8Max);
    uint2 o;
    o.x = cvt4_fp8(y[0], y[1], y[2], y[3]);
    o.y = cvt4_fp8(y[4], y[5], y[6], y[7]);
    *reinterpret_cast<uint2*>(q + ch * 8) = o;
  }
  for (int64_t i = nchunk * 8 + (int64_t)blockIdx.x * 256 + threadIdx.x; i < numel; i += stride) {
    float y = fmaxf(fminf(load1<DT>(x, i) * inv, kFp8Max), -kFp8Max);
    q[i] = (uint8_t)(cvt_pk_fp8_lo(y, 0.f, 0) & 0xff);
  }
}

// ------------------------------------------------------------------------------------------------
// per-tensor quant of a strided [H, S, D] tensor into a contiguous one (the MLA absorbed products): 8 elements (a chunk) a
// lane, four chunks in flight, in grid-stride.  The maxima queue up at one atomic, so a workgroup of the maximum pass takes four chunks
// per lane before a second one's atomic is taken, and above kMlaMaxWide chunks (2 MB of 16-bit input) it has 1024 threads, one per CU at
// most: both passes, us, up to 512 workgroups of 256 threads / 1024 threads: 3.1 MB 7.0 / 6.6, 5.9 MB 9.7 / 7.7, 10.9 MB 12.8 / 9.7,
// 20 MB 15.6 / 13.2, 36 MB 20.3 / 18.7; 2.1 MB 6.16 / 6.14, and below, where the chip is idle, the many small ones are ahead: 1.4 MB 5.6 /
// 6.0, 0.5 MB 4.9 / 5.8, 0.1 MB 4.5 / 5.5.  IDX is 32-bit wherever the chunks can be counted so, because the two divisions per
// chunk (row, then head) are the arithmetic of this kernel.
// ------------------------------------------------------------------------------------------------
constexpr int64_t kMlaMaxWide = 131072;
template <int DT, int T, bool QUANT, typename IDX>
__global__ __launch_bounds__(T) void rows_tensor_quant_kernel(const void* __restrict__ x, uint8_t* __restrict__ q,
                                                                float* __restrict__ s, int64_t rows, int S, int D,
                                                                int64_t stride_h, int64_t stride_s, float eps) {
  __shared__ float red[16];
  const IDX chunks = (IDX)(D / 8);          // per row; the host checks D % 8 == 0 and the alignment of every row
  const IDX total = (IDX)rows * chunks;
  const IDX step = (IDX)gridDim.x * T;
  const float inv = QUANT ? 1.0f / s[0] : 0.f;
  float m = 0.f;
  constexpr int U = 4;
  for (IDX i0 = (IDX)blockIdx.x * T + threadIdx.x; i0 < total; i0 += U * step) {
    Raw8<DT> t[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const IDX i = i0 + u * step;
      if (i < total) {
        const IDX row = i / chunks, c = i - row * chunks;
        const IDX hh = row / (IDX)S, ss = row - hh * (IDX)S;
        t[u].load(x, (int64_t)hh * stride_h + (int64_t)ss * stride_s + (int64_t)c * 8);
      } else {
        t[u].zero();
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      float a[8];
      t[u].unpack(a);
      if (!QUANT) {
        m = fmaxf(m, absmax8(a));
      } else if (const IDX i = i0 + u * step; i < total) {
        float y[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) y[j] = fmaxf(fminf(a[j] * inv, kFp8Max), -kFp8Max);
        uint2 o;
        o.x = cvt4_fp8(y[0], y[1], y[2], y[3]);
        o.y = cvt4_fp8(y[4], y[5], y[6], y[7]);
        *reinterpret_cast<uint2*>(q + (int64_t)i * 8) = o;  // the output is contiguous
      }
    }
  }
  if (!QUANT) {
    m = group_max<64>(fmaxf(m, eps));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < T / 64; ++i) m = fmaxf(m, red[i]);
    // non-negative floats order like their bit patterns
    if (threadIdx.x == 0) atomicMax(reinterpret_cast<unsigned int*>(s), __float_as_uint(m / kFp8Max));
  }
}

// The same for a tensor that one workgroup can hold in its registers (kMlaSmallChunks x 8 elements): one launch instead of
// two, no atomic.  4.9 us of two launches -> 3.1 us at 1 KB, 3.7 at 16 KB, 5.1 at 64 KB, where the line lies: with more, the
// one CU's load path (64 bytes a clock) takes longer than the second launch (7.2 us at 128 KB).
constexpr int kMlaHold = 4, kMlaSmallChunks = 1024 * kMlaHold;
template <int DT>
__global__ __launch_bounds__(1024) void rows_tensor_quant_small_kernel(const void* __restrict__ x, uint8_t* __restrict__ q, float* __restrict__ s,
                                                                       uint32_t total, uint32_t chunks, uint32_t S, int64_t stride_h,
                                                                       int64_t stride_s, float eps) {
  __shared__ float red[16];
  Raw8<DT> t[kMlaHold];
#pragma unroll
  for (int u = 0; u < kMlaHold; ++u) {
    const uint32_t i = u * 1024 + threadIdx.x;
    if (i < total) {
      const uint32_t row = i / chunks, c = i - row * chunks, hh = row / S, ss = row - hh * S;
      t[u].load(x, (int64_t)hh * stride_h + (int64_t)ss * stride_s + (int64_t)c * 8);
    } else {
      t[u].zero();
    }
  }
  float m = eps;
#pragma unroll
  for (int u = 0; u < kMlaHold; ++u) {
    float a[8];
    t[u].unpack(a);
    m = fmaxf(m, absmax8(a));
  }
  m = group_max<64>(m);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 16; ++i) m = fmaxf(m, red[i]);
  const float sc = fmaxf(m / kFp8Max, s[0]);  // accumulates onto what the scale holds, as the atomic form does
  const float inv = 1.0f / sc;
#pragma unroll
  for (int u = 0; u < kMlaHold; ++u) {
    const uint32_t i = u * 1024 + threadIdx.x;
    if (i < total) {
      float a[8], y[8];
      t[u].unpack(a);
#pragma unroll
      for (int j = 0; j < 8; ++j) y[j] = fmaxf(fminf(a[j] * inv, kFp8Max), -kFp8Max);
      *reinterpret_cast<uint2*>(q + (int64_t)i * 8) = make_uint2(cvt4_fp8(y[0], y[1], y[2], y[3]), cvt4_fp8(y[4], y[5], y[6], y[7]));
    }
  }
  __syncthreads();  // every wave has read the old scale
  if (threadIdx.x == 0) s[0] = sc;
}

// The same in one launch for tensors that the registers of one round of workgroups hold: every workgroup adds its maximum to
// sync[1], counts itself in at sync[0], waits until all have, and quantises what it still holds - the tensor is read once, and the
// host pays for one launch (an absorbed product with its zeroed scale 18.6 -> 14.9 us).  The counting costs a queue at one line per
// workgroup, so they are few and large: 256 of 256 threads took 6 us longer than 64 of 1024 at 2 MB.  The wait is bounded: an idle
// chip with a CU for each holds all of them at once, but work of other streams may keep CUs, so a workgroup that has waited kMlaSpins
// polls takes the maximum of the whole tensor for itself and goes on; nobody depends on another one's progress.  The last to leave
// writes the scale and zeroes the three words for the next launch on them, which must be on the same stream.
// What the wait may cost: a poll takes 0.12 us and the maximum of the whole tensor 22 / 60 / 128 us at 0.5 / 2 / 4 MB, so it ends about
// where going on alone would have cost as much: 52 / 90 / 156 us in all for a count that never comes out (485 / 522 / 576 with 4096
// polls).  Beside 256x256 GEMMs of another stream that hold every CU for 470 us each, 58 calls come through in 60 GEMMs' time (29 of
// the two launches, each of which waits for a gap) and the GEMMs take no longer, 27.3 ms; with 64 polls they take 31.2.
constexpr int kMlaOnceHold = 4, kMlaOnceGroups = 64, kMlaSpins = 256;
template <int DT>
__global__ __launch_bounds__(1024) void rows_tensor_quant_once_kernel(const void* __restrict__ x, uint8_t* __restrict__ q, float* __restrict__ s,
                                                                     uint32_t total, uint32_t chunks, uint32_t S, int64_t stride_h,
                                                                     int64_t stride_s, float eps, uint32_t* __restrict__ sync) {
  __shared__ float red[16];
  __shared__ float found;
  auto at = [&](uint32_t i) -> int64_t {
    const uint32_t row = i / chunks, c = i - row * chunks, hh = row / S, ss = row - hh * S;
    return (int64_t)hh * stride_h + (int64_t)ss * stride_s + (int64_t)c * 8;
  };
  auto block_max = [&](float v) -> float {
    v = group_max<64>(v);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    v = red[0];
#pragma unroll
    for (int i = 1; i < 16; ++i) v = fmaxf(v, red[i]);
    __syncthreads();
    return v;
  };
  Raw8<DT> t[kMlaOnceHold];
  const uint32_t step = gridDim.x * 1024u, i0 = blockIdx.x * 1024u + threadIdx.x;
#pragma unroll
  for (int u = 0; u < kMlaOnceHold; ++u) {
    if (i0 + u * step < total) t[u].load(x, at(i0 + u * step));
    else t[u].zero();
  }
  const float old = threadIdx.x == 0 ? __uint_as_float(__hip_atomic_load(reinterpret_cast<uint32_t*>(s), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) : 0.f;
  float m = eps;
#pragma unroll
  for (int u = 0; u < kMlaOnceHold; ++u) {
    float a[8];
    t[u].unpack(a);
    m = fmaxf(m, absmax8(a));
  }
  m = block_max(m);
  if (threadIdx.x == 0) {
    // non-negative floats order like their bit patterns
    __hip_atomic_fetch_max(sync + 1, __float_as_uint(m), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the maximum is there, and the old scale has been read, before the count
    __hip_atomic_fetch_add(sync, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    float all = -1.f;
    for (int n = 0; n < kMlaSpins; ++n) {
      if (__hip_atomic_load(sync, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x) {
        asm volatile("" ::: "memory");
        all = __uint_as_float(__hip_atomic_load(sync + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
        break;
      }
      __builtin_amdgcn_s_sleep(1);
    }
    found = all;
  }
  __syncthreads();
  m = found;
  if (m < 0.f) {  // uniform: the others did not turn up in time
    m = eps;
    for (uint32_t i = threadIdx.x; i < total; i += 1024) {
      Raw8<DT> r;
      r.load(x, at(i));
      float a[8];
      r.unpack(a);
      m = fmaxf(m, absmax8(a));
    }
    m = block_max(m);
  }
  __syncthreads();
  if (threadIdx.x == 0) found = old;
  __syncthreads();
  const float sc = fmaxf(m / kFp8Max, found);  // accumulates onto what the scale holds, as the atomic form does
  const float inv = 1.0f / sc;
#pragma unroll
  for (int u = 0; u < kMlaOnceHold; ++u) {
    const uint32_t i = i0 + u * step;
    if (i < total) {
      float a[8], y[8];
      t[u].unpack(a);
#pragma unroll
      for (int j = 0; j < 8; ++j) y[j] = fmaxf(fminf(a[j] * inv, kFp8Max), -kFp8Max);
      *reinterpret_cast<uint2*>(q + (int64_t)i * 8) = make_uint2(cvt4_fp8(y[0], y[1], y[2], y[3]), cvt4_fp8(y[4], y[5], y[6], y[7]));
    }
  }
  if (threadIdx.x == 0 && __hip_atomic_fetch_add(sync + 2, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1) {
    // every workgroup has read the old scale and is past its wait
    s[0] = sc;
#pragma unroll
    for (int i = 0; i < 3; ++i) __hip_atomic_store(sync + i, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

int quant_for_linear(bool groups, const void* x, void* q, float* s, int64_t M, int64_t K, float eps, int dtype, hipStream_t st) {
  const bool bf = dtype == FP8K_BF16;
  if (groups)
    return bf ? launch_group_quant<FP8K_BF16, 128, FP8K_SCALE_F32>(x, q, s, M, K, quant_eps(eps, dtype), 1, M, st)
              : launch_group_quant<FP8K_F16, 128, FP8K_SCALE_F32>(x, q, s, M, K, quant_eps(eps, dtype), 1, M, st);
  if (bf) launch_token_quant<FP8K_BF16>(x, (uint8_t*)q, s, M, K, st);
  else launch_token_quant<FP8K_F16>(x, (uint8_t*)q, s, M, K, st);
  return check_launch("token_quant");
}

}  // namespace fp8k

using namespace fp8k;

extern "C" int fp8k_group_quant(const void* x, void* q, void* s, int64_t M, int64_t K, int64_t group_size, float eps,
                                float fp8_min, float fp8_max, int in_dtype, int64_t s_stride_m, int64_t s_stride_g,
                                int scale_kind, void* stream) {
  clear_error();
  FP8K_REQUIRE(M >= 0 && K >= 0, "group_quant: negative shape");
  FP8K_REQUIRE(group_size > 0 && K % group_size == 0,
               "group_quant: the last dimension of `x` (%lld) cannot be divisible by `group_size` (%lld)", (long long)K,
               (long long)group_size);
  FP8K_REQUIRE(fp8_max == 448.0f && fp8_min == -448.0f, "group_quant: fp8_min/fp8_max must be -448/448 (OCP e4m3fn)");
  FP8K_REQUIRE(in_dtype == FP8K_F32 || in_dtype == FP8K_F16 || in_dtype == FP8K_BF16, "group_quant: bad input dtype %d",
               in_dtype);
  FP8K_REQUIRE(scale_kind == FP8K_SCALE_F32 || scale_kind == FP8K_SCALE_UE8M0_PACKED, "group_quant: bad scale kind %d",
               scale_kind);
  FP8K_REQUIRE(M <= 0x7fffffffLL && K / group_size <= 0x7fffffffLL, "group_quant: shape too large");
  if (M == 0 || K == 0) return FP8K_OK;
  FP8K_REQUIRE(x && q && s, "group_quant: null pointer");
  FP8K_REQUIRE(aligned(x, 16) && aligned(q, 8) && aligned(s, 4), "group_quant: x must be 16-byte, q 8-byte aligned");
  const int64_t G = K / group_size;
  if (scale_kind == FP8K_SCALE_F32) {
    FP8K_REQUIRE(s_stride_m >= 0 && s_stride_g >= 0 && (M == 1 || s_stride_m > 0) && (G == 1 || s_stride_g > 0),
                 "group_quant: scale strides must be positive");
  } else {
    FP8K_REQUIRE(s_stride_m > 0 && ((G + 3) / 4 == 1 || s_stride_g > 0), "group_quant: packed scale strides must be positive");
  }
  const float eps_eff = quant_eps(eps, in_dtype);
  hipStream_t st = (hipStream_t)stream;
#define FP8K_GQ(DT)                                                                                               \
  (scale_kind == FP8K_SCALE_F32                                                                                   \
       ? dispatch_group<DT, FP8K_SCALE_F32>(x, q, s, M, K, group_size, eps_eff, s_stride_m, s_stride_g, st)       \
       : dispatch_group<DT, FP8K_SCALE_UE8M0_PACKED>(x, q, s, M, K, group_size, eps_eff, s_stride_m, s_stride_g, st))
  switch (in_dtype) {
    case FP8K_BF16: return FP8K_GQ(FP8K_BF16);
    case FP8K_F16: return FP8K_GQ(FP8K_F16);
    default: return FP8K_GQ(FP8K_F32);
  }
#undef FP8K_GQ
}

extern "C" int fp8k_silu_mul_group_quant(const void* x, void* q, void* s, int64_t M, int64_t K, int64_t group_size,
                                         float eps, float fp8_min, float fp8_max, int in_dtype, int64_t s_stride_m,
                                         int64_t s_stride_g, int scale_kind, void* stream) {
  clear_error();
  const char* op = "silu_mul_group_quant";
  FP8K_REQUIRE(M >= 0 && K >= 0, "%s: negative shape", op);
  FP8K_REQUIRE(group_size == 128, "%s: the fused form is built for group_size 128 (got %lld)", op, (long long)group_size);
  FP8K_REQUIRE(K % group_size == 0, "%s: the output width (%lld) cannot be divisible by `group_size` (%lld)", op,
               (long long)K, (long long)group_size);
  FP8K_REQUIRE(fp8_max == 448.0f && fp8_min == -448.0f, "%s: fp8_min/fp8_max must be -448/448 (OCP e4m3fn)", op);
  FP8K_REQUIRE(in_dtype == FP8K_F32 || in_dtype == FP8K_F16 || in_dtype == FP8K_BF16, "%s: bad input dtype %d", op, in_dtype);
  FP8K_REQUIRE(scale_kind == FP8K_SCALE_F32 || scale_kind == FP8K_SCALE_UE8M0_PACKED, "%s: bad scale kind %d", op, scale_kind);
  FP8K_REQUIRE(M <= 0x7fffffffLL && K / group_size <= 0x3fffffffLL, "%s: shape too large", op);
  if (M == 0 || K == 0) return FP8K_OK;
  FP8K_REQUIRE(x && q && s, "%s: null pointer", op);
  FP8K_REQUIRE(aligned(x, 16) && aligned(q, 8) && aligned(s, 4), "%s: x must be 16-byte, q 8-byte aligned", op);
  const int64_t G = K / group_size;
  if (scale_kind == FP8K_SCALE_F32) {
    FP8K_REQUIRE(s_stride_m >= 0 && s_stride_g >= 0 && (M == 1 || s_stride_m > 0) && (G == 1 || s_stride_g > 0),
                 "%s: scale strides must be positive", op);
  } else {
    FP8K_REQUIRE(s_stride_m > 0 && ((G + 3) / 4 == 1 || s_stride_g > 0), "%s: packed scale strides must be positive", op);
  }
  const float eps_eff = quant_eps(eps, in_dtype);
  hipStream_t st = (hipStream_t)stream;
#define FP8K_SGQ(DT)                                                                                                 \
  (scale_kind == FP8K_SCALE_F32                                                                                     \
       ? launch_group_quant<DT, 128, FP8K_SCALE_F32, true>(x, q, s, M, K, eps_eff, s_stride_m, s_stride_g, st)      \
       : launch_group_quant<DT, 128, FP8K_SCALE_UE8M0_PACKED, true>(x, q, s, M, K, eps_eff, s_stride_m, s_stride_g, st))
  switch (in_dtype) {
    case FP8K_BF16: return FP8K_SGQ(FP8K_BF16);
    case FP8K_F16: return FP8K_SGQ(FP8K_F16);
    default: return FP8K_SGQ(FP8K_F32);
  }
#undef FP8K_SGQ
}

extern "C" int fp8k_group_quant_masked(const void* x, void* q, void* s, int64_t E, int64_t m_max, int64_t K,
                                       int64_t group_size, float eps, float fp8_min, float fp8_max, int in_dtype,
                                       int64_t s_stride_e, int64_t s_stride_m, int64_t s_stride_g, int scale_kind,
                                       int fuse_silu_and_mul, const int32_t* masked_m, void* stream) {
  clear_error();
  const char* op = "group_quant_masked";
  FP8K_REQUIRE(E >= 0 && m_max >= 0 && K >= 0, "%s: negative shape", op);
  FP8K_REQUIRE(group_size == 128, "%s: the masked form is built for group_size 128 (got %lld)", op, (long long)group_size);
  FP8K_REQUIRE(K % group_size == 0, "%s: the output width (%lld) cannot be divisible by `group_size` (%lld)", op,
               (long long)K, (long long)group_size);
  FP8K_REQUIRE(fp8_max == 448.0f && fp8_min == -448.0f, "%s: fp8_min/fp8_max must be -448/448 (OCP e4m3fn)", op);
  FP8K_REQUIRE(in_dtype == FP8K_F32 || in_dtype == FP8K_F16 || in_dtype == FP8K_BF16, "%s: bad input dtype %d", op, in_dtype);
  FP8K_REQUIRE(scale_kind == FP8K_SCALE_F32 || scale_kind == FP8K_SCALE_UE8M0_PACKED || scale_kind == FP8K_SCALE_UE8M0_F32,
               "%s: bad scale kind %d", op, scale_kind);
  FP8K_REQUIRE(E * m_max <= 0x7fffffffLL && m_max <= 0x7fffffffLL && K / group_size <= 0x3fffffffLL, "%s: shape too large", op);
  if (E == 0 || m_max == 0 || K == 0) return FP8K_OK;
  FP8K_REQUIRE(x && q && s && masked_m, "%s: null pointer", op);
  FP8K_REQUIRE(aligned(x, 16) && aligned(q, 8) && aligned(s, 4) && aligned(masked_m, 4), "%s: x must be 16-byte, q 8-byte aligned", op);
  FP8K_REQUIRE(s_stride_e >= 0 && s_stride_m >= 0 && s_stride_g >= 0, "%s: negative scale stride", op);
  const float eps_eff = quant_eps(eps, in_dtype);
  hipStream_t st = (hipStream_t)stream;
  const int64_t M = E * m_max;
#define FP8K_MQ3(DT, KIND, FUSE) \
  launch_group_quant<DT, 128, KIND, FUSE, true>(x, q, s, M, K, eps_eff, s_stride_m, s_stride_g, st, masked_m, (int)m_max, s_stride_e)
#define FP8K_MQ2(DT, KIND) (fuse_silu_and_mul ? FP8K_MQ3(DT, KIND, true) : FP8K_MQ3(DT, KIND, false))
#define FP8K_MQ(DT)                                                  \
  (scale_kind == FP8K_SCALE_F32            ? FP8K_MQ2(DT, FP8K_SCALE_F32) \
   : scale_kind == FP8K_SCALE_UE8M0_PACKED ? FP8K_MQ2(DT, FP8K_SCALE_UE8M0_PACKED) \
                                           : FP8K_MQ2(DT, FP8K_SCALE_UE8M0_F32))
  switch (in_dtype) {
    case FP8K_BF16: return FP8K_MQ(FP8K_BF16);
    case FP8K_F16: return FP8K_MQ(FP8K_F16);
    default: return FP8K_MQ(FP8K_F32);
  }
#undef FP8K_MQ
#undef FP8K_MQ2
#undef FP8K_MQ3
}

extern "C" int fp8k_token_quant(const void* x, void* q, float* s, int64_t M, int64_t K, int in_dtype, void* stream) {
  clear_error();
  FP8K_REQUIRE(M >= 0 && K >= 0, "token_quant: negative shape");
  FP8K_REQUIRE(K % 8 == 0, "token_quant: hidden dimension (%lld) must be divisible by 8", (long long)K);
  FP8K_REQUIRE(in_dtype == FP8K_F32 || in_dtype == FP8K_F16 || in_dtype == FP8K_BF16, "token_quant: bad input dtype %d",
               in_dtype);
  FP8K_REQUIRE(M <= 0x7fffffffLL, "token_quant: too many rows");
  if (M == 0 || K == 0) return FP8K_OK;
  FP8K_REQUIRE(x && q && s, "token_quant: null pointer");
  FP8K_REQUIRE(aligned(x, 16) && aligned(q, 8), "token_quant: x must be 16-byte, q 8-byte aligned");
  hipStream_t st = (hipStream_t)stream;
  switch (in_dtype) {
    case FP8K_BF16: launch_token_quant<FP8K_BF16>(x, (uint8_t*)q, s, M, K, st); break;
    case FP8K_F16: launch_token_quant<FP8K_F16>(x, (uint8_t*)q, s, M, K, st); break;
    default: launch_token_quant<FP8K_F32>(x, (uint8_t*)q, s, M, K, st); break;
  }
  return check_launch("token_quant");
}

extern "C" int fp8k_tensor_quant(const void* x, void* q, float* s, int64_t numel, int in_dtype, int is_static,
                                 void* stream) {
  clear_error();
  FP8K_REQUIRE(numel >= 0, "tensor_quant: negative size");
  FP8K_REQUIRE(in_dtype == FP8K_F32 || in_dtype == FP8K_F16 || in_dtype == FP8K_BF16, "tensor_quant: bad input dtype %d",
               in_dtype);
  if (numel == 0) return FP8K_OK;
  FP8K_REQUIRE(x && q && s, "tensor_quant: null pointer");
  FP8K_REQUIRE(aligned(x, 16) && aligned(q, 8), "tensor_quant: x must be 16-byte, q 8-byte aligned");
  hipStream_t st = (hipStream_t)stream;
  const int64_t want = (numel / 8 + 255) / 256;
  dim3 grid((unsigned)(want < 1 ? 1 : (want > 2048 ? 2048 : want))), block(256);
#define FP8K_TQ(DT)                                                                                     \
  do {                                                                                                  \
    if (!is_static) hipLaunchKernelGGL(tensor_absmax_kernel<DT>, grid, block, 0, st, x, s, numel);      \
    hipLaunchKernelGGL(tensor_quant_kernel<DT>, grid, block, 0, st, x, (uint8_t*)q, (const float*)s, numel); \
  } while (0)
  switch (in_dtype) {
    case FP8K_BF16: FP8K_TQ(FP8K_BF16); break;
    case FP8K_F16: FP8K_TQ(FP8K_F16); break;
    default: FP8K_TQ(FP8K_F32); break;
  }
#undef FP8K_TQ
  return check_launch("tensor_quant");
}

extern "C" int fp8k_tensor_quant_mla_takes_sync(int64_t numel) {
  return numel / 8 > kMlaSmallChunks && numel / 8 <= (int64_t)kMlaOnceGroups * 1024 * kMlaOnceHold && num_cu() >= kMlaOnceGroups;
}

static int tensor_quant_mla(const void* x, void* q, float* s, int64_t H, int64_t S, int64_t D, int64_t x_stride_h, int64_t x_stride_s,
                            float eps, int in_dtype, int32_t* sync, void* stream) {
  clear_error();
  const char* op = "per_tensor_quant_mla_fp8";
  FP8K_REQUIRE(H >= 0 && S >= 0 && D >= 0, "%s: negative shape", op);
  FP8K_REQUIRE(in_dtype == FP8K_F32 || in_dtype == FP8K_F16 || in_dtype == FP8K_BF16, "%s: bad input dtype %d", op, in_dtype);
  FP8K_REQUIRE(S <= 0x7fffffffLL && D <= 0x7fffffffLL, "%s: shape too large", op);
  if (H * S * D == 0) return FP8K_OK;
  const int64_t esz = in_dtype == FP8K_F32 ? 4 : 2;
  FP8K_REQUIRE(x && q && s, "%s: null pointer", op);
  FP8K_REQUIRE(D % 8 == 0, "%s: the last dimension (%lld) must be divisible by 8", op, (long long)D);
  FP8K_REQUIRE(x_stride_h >= 0 && x_stride_s >= 0 && (x_stride_h * esz) % 16 == 0 && (x_stride_s * esz) % 16 == 0 && aligned(x, 16) &&
               aligned(q, 8), "%s: rows of x must be 16-byte aligned, q 8-byte aligned", op);
  hipStream_t st = (hipStream_t)stream;
  const int64_t rows = H * S, chunks = rows * (D / 8);
  const bool narrow = chunks < (1LL << 31);  // room for the four steps past the end
  const dim3 block(256);
  const bool wide = chunks > kMlaMaxWide;
  const dim3 grid_max((unsigned)(wide ? std::min<int64_t>(num_cu(), (chunks + 4095) / 4096) : (chunks + 1023) / 1024));
  const dim3 grid_q((unsigned)std::min<int64_t>(2048, (chunks + 255) / 256));
  // one chunk per lane is enough to work on: the more workgroups share it, the shorter the loads
  const dim3 grid_once((unsigned)std::min<int64_t>(kMlaOnceGroups, (chunks + 1023) / 1024));
  FP8K_REQUIRE(!sync || fp8k_tensor_quant_mla_takes_sync(H * S * D), "%s: not a size of the one-launch form", op);
#define FP8K_MLAQ2(DT, IDX)                                                                                                 \
  do {                                                                                                                      \
    if (wide)                                                                                                               \
      hipLaunchKernelGGL((rows_tensor_quant_kernel<DT, 1024, false, IDX>), grid_max, dim3(1024), 0, st, x, (uint8_t*)q, s,  \
                         rows, (int)S, (int)D, x_stride_h, x_stride_s, eps);                                                \
    else                                                                                                                    \
      hipLaunchKernelGGL((rows_tensor_quant_kernel<DT, 256, false, uint32_t>), grid_max, block, 0, st, x, (uint8_t*)q, s,   \
                         rows, (int)S, (int)D, x_stride_h, x_stride_s, eps);                                                \
    hipLaunchKernelGGL((rows_tensor_quant_kernel<DT, 256, true, IDX>), grid_q, block, 0, st, x, (uint8_t*)q, s, rows, (int)S, \
                       (int)D, x_stride_h, x_stride_s, eps);                                                                \
  } while (0)
#define FP8K_MLAQ(DT)                                                                                                          \
  do {                                                                                                                         \
    if (chunks <= kMlaSmallChunks)                                                                                             \
      hipLaunchKernelGGL(rows_tensor_quant_small_kernel<DT>, dim3(1), dim3(1024), 0, st, x, (uint8_t*)q, s, (uint32_t)chunks,  \
                         (uint32_t)(D / 8), (uint32_t)S, x_stride_h, x_stride_s, eps);                                         \
    else if (sync)                                                                                                             \
      hipLaunchKernelGGL(rows_tensor_quant_once_kernel<DT>, grid_once, dim3(1024), 0, st, x, (uint8_t*)q, s, (uint32_t)chunks,      \
                         (uint32_t)(D / 8), (uint32_t)S, x_stride_h, x_stride_s, eps, reinterpret_cast<uint32_t*>(sync));      \
    else if (narrow) FP8K_MLAQ2(DT, uint32_t);                                                                                 \
    else FP8K_MLAQ2(DT, int64_t);             \
  } while (0)
  switch (in_dtype) {
    case FP8K_BF16: FP8K_MLAQ(FP8K_BF16); break;
    case FP8K_F16: FP8K_MLAQ(FP8K_F16); break;
    default: FP8K_MLAQ(FP8K_F32); break;
  }
#undef FP8K_MLAQ
#undef FP8K_MLAQ2
  return check_launch(op);
}

extern "C" int fp8k_tensor_quant_mla(const void* x, void* q, float* s, int64_t H, int64_t S, int64_t D, int64_t x_stride_h,
                                     int64_t x_stride_s, float eps, int in_dtype, void* stream) {
  return tensor_quant_mla(x, q, s, H, S, D, x_stride_h, x_stride_s, eps, in_dtype, nullptr, stream);
}

extern "C" int fp8k_tensor_quant_mla_sync(const void* x, void* q, float* s, int64_t H, int64_t S, int64_t D, int64_t x_stride_h,
                                          int64_t x_stride_s, float eps, int in_dtype, int32_t* sync, void* stream) {
  return tensor_quant_mla(x, q, s, H, S, D, x_stride_h, x_stride_s, eps, in_dtype, sync, stream);
}
