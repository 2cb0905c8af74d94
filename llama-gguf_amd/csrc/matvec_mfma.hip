// matvec_mfma.hip — quantized mat-vec on the int8 matrix cores (v_mfma_i32_16x16x64_i8): Q4_K, Q5_K, Q6_K, Q8_0, Q4_0.
//
// Why MFMA for a mat-VEC.  The VALU formulation (matvec.hip) needs ~3.6 vector instructions per weight
// (byte->f32 convert, FMA, nibble masks); measured on MI355X a wave64 v_cvt_f32_ubyte costs ~2.0 ns and a
// v_fma ~1.2 ns of SIMD time with 4 waves per SIMD (tools/probes/mfma_i8_probe.hip), which made Llama-3-8B
// Q4_K_M decode ISSUE-bound at ~0.76 ms/token — a launch took 21 us whether its 66 MB of weights came from HBM or
// from the Infinity Cache.  The matrix pipe is a separate issue port: one 16x16x64 int8 MFMA multiplies 1024
// weights in ~15 ns, so the multiply-accumulates move there and the VALU only unpacks quants and applies scales.
//
// Arithmetic (the reference keeps x in f32, src/backend/cpu/simd.rs:978-1032; there is no activation quantization
// to mirror): x arrives as XQ records (xq.h) — per 16-element chunk x = s * 2^-30 * I with I = d3*2^24 + d2*2^16 +
// d1*2^8 + d0, balanced int8 digits, exact for every element within 2^6 of the chunk maximum.  The A operand of an
// MFMA is block-diagonal over its four k-chunks (rows 4c..4c+3 = the four digits of chunk c), 16 weight rows x 64
// quants are the B operand, and D holds sum_k q_k * digit_i,k as exact int32 — lane group c gets chunk c.  The four
// digit sums are recombined once in f32 (V = D0*2^24 + D1*2^16 + D2*2^8 + D3) and scaled by d*sc*s*2^-30; min terms
// (Q4_K, Q5_K) and offsets (Q6_K -32, Q4_0 -8) go through the f32 sums of x per chunk, the reference's x_acc.
// Error vs the reference's sequential f32 sum is at f32 rounding level and independent of summation order.
//
// Device layout "tile16" (same bytes as GGUF, rows padded to 16): a tile = 16 rows x one 256-element block = 2304 B.
// The nibbles of MFMA step pp (elements 64pp .. 64pp+63) and k-chunk c (16 elements) of row n belong to lane 16c + n,
// eight bytes per step:  N0, N1 with byte t = w[t] | w[t+4] << 4  (w = elements 0-7 / 8-15 of the chunk), so B-operand
// dwords are N0 & 0x0F.., N0 >> 4 & 0x0F.., N1 & 0x0F.., N1 >> 4 & 0x0F.. and every lane loads only its own nibbles:
//   [0, 1024) lane-major 16 B: N0,N1 of steps 0,1    [1024, 2048) steps 2,3    [2048, 2304) the 16 native 16-byte headers
#include <algorithm>
#include <cstring>
#include <type_traits>

#include "device_utils.h"
#include "mv_epilogue.h"
#include "xq.h"
#include "mvq_core.h"
#include "timeline.h"

LGH_TL_DEFINE(mvq)

namespace lgh {

#ifdef LGH_STAMPS
__device__ unsigned long long g_stamps[8192 * 8];
hipError_t mvq_read_stamps(unsigned long long* host, size_t n) {
  return hipMemcpyFromSymbol(host, HIP_SYMBOL(g_stamps), n * sizeof(unsigned long long));
}
#define LGH_STAMP(i)                                                                             \
  do {                                                                                           \
    if (threadIdx.x == 0 && blockIdx.x < 8192) g_stamps[blockIdx.x * 8 + (i)] = __builtin_amdgcn_s_memrealtime(); \
  } while (0)
// per-WAVE stamps (8 slots): how far apart the waves of a workgroup run and where a wave's prologue goes
__device__ unsigned long long g_wstamps[2048 * 16 * 8];
hipError_t mvq_read_wave_stamps(unsigned long long* host, size_t n) {
  return hipMemcpyFromSymbol(host, HIP_SYMBOL(g_wstamps), n * sizeof(unsigned long long));
}
// first workgroup start / last workgroup end of each of the last 64 launches (slot = MvLaunch::dbg_slot)
__device__ unsigned long long g_span[64 * 2];
hipError_t mvq_spans(unsigned long long* host, int reset) {
  if (reset) {
    unsigned long long init[128];
    for (int i = 0; i < 64; i++) { init[2 * i] = ~0ull; init[2 * i + 1] = 0; }
    return hipMemcpyToSymbol(HIP_SYMBOL(g_span), init, sizeof(init));
  }
  return hipMemcpyFromSymbol(host, HIP_SYMBOL(g_span), 128 * sizeof(unsigned long long));
}
#define LGH_SPAN(i)                                                                              \
  do {                                                                                           \
    if (threadIdx.x == 0) {                                                                      \
      if ((i) == 0) atomicMin(&g_span[A.dbg_slot * 2], (unsigned long long)__builtin_amdgcn_s_memrealtime()); \
      else atomicMax(&g_span[A.dbg_slot * 2 + 1], (unsigned long long)__builtin_amdgcn_s_memrealtime()); \
    }                                                                                            \
  } while (0)
#define LGH_WSTAMP(i)                                                                            \
  do {                                                                                           \
    if ((threadIdx.x & 63) == 0 && blockIdx.x < 2048)                                            \
      g_wstamps[(blockIdx.x * 16 + (threadIdx.x >> 6)) * 8 + (i)] = __builtin_amdgcn_s_memrealtime(); \
  } while (0)
#else
#define LGH_STAMP(i)
#define LGH_WSTAMP(i)
#define LGH_SPAN(i)
#endif

// ------------------------------------------------------------------------------------------------
// native [row][block] Q4_K  ->  tile16
// ------------------------------------------------------------------------------------------------
__global__ void __launch_bounds__(256) repack_q4k_t16_kernel(const uint8_t* __restrict__ raw, uint8_t* __restrict__ dst,
                                                            uint32_t n_rows, uint32_t nblk, uint64_t total) {
  // one thread per (row, block, step pp): idx = ((row * nblk) + b) * 4 + pp.  Elements 64pp .. 64pp+63 of the block live in
  // qs[32pp .. 32pp+31]: low nibbles = the first 32, high nibbles = the second 32 (dequant.rs:232-255).
  for (uint64_t idx = (uint64_t)blockIdx.x * 256 + threadIdx.x; idx < total; idx += (uint64_t)gridDim.x * 256) {
    const uint32_t pp = (uint32_t)(idx & 3);
    const uint64_t rb = idx >> 2;
    const uint32_t row = (uint32_t)(rb / nblk), b = (uint32_t)(rb % nblk);
    const uint32_t rt = row >> 4, n = row & 15;
    uint8_t* tile = dst + ((size_t)rt * nblk + b) * kTileBytes;
    const bool live = row < n_rows;
    const uint8_t* src = raw + ((size_t)row * nblk + b) * 144;
#pragma unroll
    for (uint32_t c = 0; c < 4; c++) {
      uint32_t w[16];
#pragma unroll
      for (uint32_t t = 0; t < 16; t++) {
        const uint32_t byte = live ? src[16 + 32 * pp + 16 * (c & 1) + t] : 0u;
        w[t] = c < 2 ? (byte & 15u) : (byte >> 4);
      }
      uint32_t N0 = 0, N1 = 0;
#pragma unroll
      for (uint32_t t = 0; t < 4; t++) {
        N0 |= (w[t] | w[t + 4] << 4) << (8 * t);
        N1 |= (w[t + 8] | w[t + 12] << 4) << (8 * t);
      }
      uint32_t* nib = reinterpret_cast<uint32_t*>(tile + (pp >> 1) * 1024 + (16 * c + n) * 16 + (pp & 1) * 8);
      nib[0] = N0;
      nib[1] = N1;
    }
    // the native 16-byte header {d, dmin, scales[12]}, one dword per pp-thread
    *reinterpret_cast<uint32_t*>(tile + 2048 + n * 16 + pp * 4) = live ? *reinterpret_cast<const uint32_t*>(src + pp * 4) : 0u;
  }
}

hipError_t repack_q4k_t16_launch(const uint8_t* raw, uint8_t* dst, uint32_t n_rows, uint32_t nblk, hipStream_t st) {
  const uint64_t total = (uint64_t)((n_rows + 15) / 16) * 16 * nblk * 4;
  uint64_t blocks = (total + 255) / 256;
  if (blocks > 65536) blocks = 65536;
  hipLaunchKernelGGL(repack_q4k_t16_kernel, dim3((uint32_t)blocks), dim3(256), 0, st, raw, dst, n_rows, nblk, total);
  return hipGetLastError();
}

// ------------------------------------------------------------------------------------------------
// native [row][block] Q6_K  ->  tile16 (3392 B per 16 rows x 256 elements)
//
// The 6-bit weights q' = ql | qh << 4 (0..63; the reference subtracts 32, dequant.rs:338-341) of MFMA step pp
// (elements 64pp .. 64pp+63) and k-chunk c (16 elements) of row n belong to lane 16c + n.  Per lane and step:
//   N0, N1   byte t = w[t] | w[t+4] << 4          (w = low nibbles of elements 0-7 / 8-15 of the chunk)
//   H        byte t = f[t] | f[t+4] << 2 | f[t+8] << 4 | f[t+12] << 6   (f = the 2 high bits)
// so B-operand dword j (elements 4j..4j+3) = nibbles_j | ((H >> 2j) & 0x03030303) << 4 with plain 32-bit ops.
//   [0    , 1024)  lane-major 16 B: N0,N1 of steps 0 and 1        [1024, 2048)  N0,N1 of steps 2 and 3
//   [2048 , 3072)  lane-major 16 B: H of steps 0..3
//   [3072 , 3328)  row-major 16 B: the 16 int8 sub-block scales    [3328 , 3360)  the 16 rows' f16 d   (+32 B pad)
// ------------------------------------------------------------------------------------------------
__device__ __forceinline__ uint32_t q6_raw(const uint8_t* b, uint32_t i) {   // q' of element i of a native block
  const uint32_t hn = i >> 7, r = i & 127, t = r >> 5, l = r & 31;
  const uint32_t lb = b[hn * 64 + l + 32 * (t & 1)];
  const uint32_t lo = t < 2 ? (lb & 0x0Fu) : (lb >> 4);
  return lo | (((b[128 + hn * 32 + l] >> (2 * t)) & 3u) << 4);
}

__global__ void __launch_bounds__(256) repack_q6k_t16_kernel(const uint8_t* __restrict__ raw, uint8_t* __restrict__ dst,
                                                            uint32_t n_rows, uint32_t nblk, uint64_t total) {
  // one thread per (row, block, step pp): idx = ((row * nblk) + b) * 4 + pp
  for (uint64_t idx = (uint64_t)blockIdx.x * 256 + threadIdx.x; idx < total; idx += (uint64_t)gridDim.x * 256) {
    const uint32_t pp = (uint32_t)(idx & 3);
    const uint64_t rb = idx >> 2;
    const uint32_t row = (uint32_t)(rb / nblk), b = (uint32_t)(rb % nblk);
    const uint32_t rt = row >> 4, n = row & 15;
    uint8_t* tile = dst + ((size_t)rt * nblk + b) * kTileBytesQ6;
    const bool live = row < n_rows;
    const uint8_t* src = raw + ((size_t)row * nblk + b) * 210;
#pragma unroll
    for (uint32_t c = 0; c < 4; c++) {
      uint32_t w[16];
#pragma unroll
      for (uint32_t t = 0; t < 16; t++) w[t] = live ? q6_raw(src, 64 * pp + 16 * c + t) : 0u;
      uint32_t N0 = 0, N1 = 0, H = 0;
#pragma unroll
      for (uint32_t t = 0; t < 4; t++) {
        N0 |= ((w[t] & 15u) | (w[t + 4] & 15u) << 4) << (8 * t);
        N1 |= ((w[t + 8] & 15u) | (w[t + 12] & 15u) << 4) << (8 * t);
        H |= ((w[t] >> 4) | (w[t + 4] >> 4) << 2 | (w[t + 8] >> 4) << 4 | (w[t + 12] >> 4) << 6) << (8 * t);
      }
      const uint32_t lane = 16 * c + n;
      uint32_t* nib = reinterpret_cast<uint32_t*>(tile + (pp >> 1) * 1024 + lane * 16 + (pp & 1) * 8);
      nib[0] = N0;
      nib[1] = N1;
      *reinterpret_cast<uint32_t*>(tile + 2048 + lane * 16 + pp * 4) = H;
    }
    // scales 4pp .. 4pp+3 of the row; d once per (row, block)
    uint32_t sc = 0;
    if (live) sc = (uint32_t)src[192 + 4 * pp] | (uint32_t)src[193 + 4 * pp] << 8 | (uint32_t)src[194 + 4 * pp] << 16 | (uint32_t)src[195 + 4 * pp] << 24;
    *reinterpret_cast<uint32_t*>(tile + 3072 + n * 16 + pp * 4) = sc;
    if (pp == 0) *reinterpret_cast<uint16_t*>(tile + 3328 + n * 2) = live ? (uint16_t)(src[208] | src[209] << 8) : (uint16_t)0;
    if (pp == 1 && n == 0) {   // the pad, so that repacked buffers are fully defined
#pragma unroll
      for (int i = 0; i < 8; i++) *reinterpret_cast<uint32_t*>(tile + 3360 + 4 * i) = 0u;
    }
  }
}

hipError_t repack_q6k_t16_launch(const uint8_t* raw, uint8_t* dst, uint32_t n_rows, uint32_t nblk, hipStream_t st) {
  const uint64_t total = (uint64_t)((n_rows + 15) / 16) * 16 * nblk * 4;
  uint64_t blocks = (total + 255) / 256;
  if (blocks > 65536) blocks = 65536;
  hipLaunchKernelGGL(repack_q6k_t16_kernel, dim3((uint32_t)blocks), dim3(256), 0, st, raw, dst, n_rows, nblk, total);
  return hipGetLastError();
}

// ------------------------------------------------------------------------------------------------
// kernel
// ------------------------------------------------------------------------------------------------

// ------------------------------------------------------------------------------------------------
// Q5_K, Q8_0, Q4_0 -> tile16.  Same lane mapping as above (step pp, k-chunk c, row n -> lane 16c + n).
//   Q5_K (2816 B): the Q4_K tile (nibble words [0,2048), native headers [2048,2304)) + [2304,2816) lane-major 8 B: the fifth
//         bits, one dword per step PAIR: byte t = f[t] | f[t+4]<<1 | f[t+8]<<2 | f[t+12]<<3 of the even step in the low
//         nibble, of the odd step in the high nibble
//   Q8_0 (4352 B): [pp][lane] 16 quants as they are (int8) [0,4096), then per row the 8 f16 d of its 32-element blocks
//   Q4_0 (2304 B): nibble words [0,2048) as Q4_K (unsigned 0..15; the reference's "- 8" goes through the sums of x), then
//         per row the 8 f16 d
// One thread per (row, 256-element block, step).
// ------------------------------------------------------------------------------------------------
template <int F>
__global__ void __launch_bounds__(256) repack_t16_kernel(const uint8_t* __restrict__ raw, uint8_t* __restrict__ dst,
                                                        uint32_t n_rows, uint32_t nblk, uint64_t total) {
  constexpr uint32_t TB = fmt_tile_bytes(F);
  constexpr uint32_t SRC = F == F_Q5K ? 176u : F == F_Q80 ? 8u * 34u : 8u * 18u;   // native bytes of 256 elements
  for (uint64_t idx = (uint64_t)blockIdx.x * 256 + threadIdx.x; idx < total; idx += (uint64_t)gridDim.x * 256) {
    const uint32_t pp = (uint32_t)(idx & 3);
    const uint64_t rb = idx >> 2;
    const uint32_t row = (uint32_t)(rb / nblk), b = (uint32_t)(rb % nblk);
    const uint32_t rt = row >> 4, n = row & 15;
    uint8_t* tile = dst + ((size_t)rt * nblk + b) * TB;
    const bool live = row < n_rows;
    const uint8_t* src = raw + ((size_t)row * nblk + b) * SRC;
    auto quant = [&](uint32_t e) -> uint32_t {   // unsigned quant (Q8_0: the byte) of element e of the 256
      if (!live) return 0u;
      if (F == F_Q5K) {   // dequant.rs:265-316
        const uint32_t g = e >> 6, w = e & 63, l = w & 31, is = 2 * g + (w >> 5);
        const uint32_t byte = src[48 + g * 32 + l];
        return (w < 32 ? (byte & 15u) : (byte >> 4)) | (((src[16 + l] >> is) & 1u) << 4);
      }
      const uint32_t sb = e >> 5, i = e & 31;   // 32-element block and offset
      if (F == F_Q80) return src[sb * 34 + 2 + i];                       // dequant.rs:106-112
      const uint32_t byte = src[sb * 18 + 2 + (i & 15)];               // Q4_0, dequant.rs:16-30
      return i < 16 ? (byte & 15u) : (byte >> 4);
    };
    uint32_t hpair[4] = {0, 0, 0, 0};
#pragma unroll
    for (uint32_t c = 0; c < 4; c++) {
      uint32_t w[16];
#pragma unroll
      for (uint32_t t = 0; t < 16; t++) w[t] = quant(64 * pp + 16 * c + t);
      const uint32_t lane = 16 * c + n;
      if (F == F_Q80) {
        uint32_t* q = reinterpret_cast<uint32_t*>(tile + pp * 1024 + lane * 16);
#pragma unroll
        for (uint32_t j = 0; j < 4; j++) q[j] = w[4 * j] | w[4 * j + 1] << 8 | w[4 * j + 2] << 16 | w[4 * j + 3] << 24;
      } else {
        uint32_t N0 = 0, N1 = 0, H = 0;
#pragma unroll
        for (uint32_t t = 0; t < 4; t++) {
          N0 |= ((w[t] & 15u) | (w[t + 4] & 15u) << 4) << (8 * t);
          N1 |= ((w[t + 8] & 15u) | (w[t + 12] & 15u) << 4) << (8 * t);
          H |= ((w[t] >> 4) | (w[t + 4] >> 4) << 1 | (w[t + 8] >> 4) << 2 | (w[t + 12] >> 4) << 3) << (8 * t);
        }
        uint32_t* nib = reinterpret_cast<uint32_t*>(tile + (pp >> 1) * 1024 + lane * 16 + (pp & 1) * 8);
        nib[0] = N0;
        nib[1] = N1;
        hpair[c] = H;
      }
    }
    if (F == F_Q5K) {
      // the fifth bits of this step go into the low (even step) or high (odd step) nibbles of the pair's dword: two
      // threads (pp, pp^1) write disjoint nibbles of the same dword, so each does a byte-wise read-modify-write of ITS
      // nibbles only -> use 4-bit-disjoint atomicOr on a zero-initialised destination
#pragma unroll
      for (uint32_t c = 0; c < 4; c++)
        atomicOr(reinterpret_cast<uint32_t*>(tile + 2304 + (16 * c + n) * 8 + (pp >> 1) * 4), hpair[c] << (4 * (pp & 1)));
      *reinterpret_cast<uint32_t*>(tile + 2048 + n * 16 + pp * 4) = live ? *reinterpret_cast<const uint32_t*>(src + pp * 4) : 0u;
    } else {
      // two f16 d per step thread: blocks 2pp, 2pp+1
      const uint32_t bs = F == F_Q80 ? 34u : 18u, hoff = F == F_Q80 ? 4096u : 2048u;
      uint32_t d2 = 0;
      if (live) d2 = (uint32_t)(src[(2 * pp) * bs] | src[(2 * pp) * bs + 1] << 8) | (uint32_t)(src[(2 * pp + 1) * bs] | src[(2 * pp + 1) * bs + 1] << 8) << 16;
      *reinterpret_cast<uint32_t*>(tile + hoff + n * 16 + pp * 4) = d2;
    }
  }
}

hipError_t repack_t16_launch(int dev_type, const uint8_t* raw, uint8_t* dst, uint32_t n_rows, uint32_t nblk, hipStream_t st) {
  const uint64_t total = (uint64_t)((n_rows + 15) / 16) * 16 * nblk * 4;
  uint64_t blocks = (total + 255) / 256;
  if (blocks > 65536) blocks = 65536;
  const dim3 g((uint32_t)blocks), t(256);
  switch (fmt_of_dev_type(dev_type)) {
    case F_Q4K: return repack_q4k_t16_launch(raw, dst, n_rows, nblk, st);
    case F_Q6K: return repack_q6k_t16_launch(raw, dst, n_rows, nblk, st);
    case F_Q5K: {
      hipError_t e = hipMemsetAsync(dst, 0, (size_t)((n_rows + 15) / 16) * nblk * fmt_tile_bytes(F_Q5K), st);   // fifth bits are OR-ed in
      if (e != hipSuccess) return e;
      hipLaunchKernelGGL((repack_t16_kernel<F_Q5K>), g, t, 0, st, raw, dst, n_rows, nblk, total);
      break;
    }
    case F_Q80: hipLaunchKernelGGL((repack_t16_kernel<F_Q80>), g, t, 0, st, raw, dst, n_rows, nblk, total); break;
    case F_Q40: hipLaunchKernelGGL((repack_t16_kernel<F_Q40>), g, t, 0, st, raw, dst, n_rows, nblk, total); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

// ------------------------------------------------------------------------------------------------
// stand-alone f32 -> XQ conversion (xq.h): for vectors whose producer cannot write XQ itself (the token embedding, the
// per-op API, pipeline-stage inputs).  One thread per element; with `nw` the record holds x * nw and ssq_part[chunk]
// receives each 16-element chunk's sum of x^2 (the RMSNorm prologue of the consumer).
// ------------------------------------------------------------------------------------------------
__global__ void __launch_bounds__(256) xq_quantize_kernel(const float* __restrict__ x, const float* __restrict__ nw,
                                                          uint8_t* __restrict__ xq, float* __restrict__ ssq_part, uint32_t k) {
  const uint32_t e = blockIdx.x * 256 + threadIdx.x;   // k is a multiple of 256
  const float v = x[e];
  xq_store_chunk(xq, e >> 4, nw ? v * nw[e] : v, ssq_part, v);
}

hipError_t xq_quantize_launch(const float* x, const float* nw, uint8_t* xq, float* ssq_part, uint32_t k, hipStream_t st) {
  if (k == 0 || k % 256) return hipErrorInvalidValue;
  hipLaunchKernelGGL(xq_quantize_kernel, dim3(k / 256), dim3(256), 0, st, x, nw, xq, ssq_part, k);
  return hipGetLastError();
}

constexpr int kWaves = 8;   // waves per workgroup: 2 per SIMD, 256 VGPRs each
constexpr int kDepth = 4;   // weight tiles a wave keeps in flight (4 x 2304 B x 8 waves = 72 KiB per CU)

// Geometry: ONE workgroup per CU.  Its waves are T k-slices x G row-groups; wave (ks, rg) owns blocks
// [ks*nbw, (ks+1)*nbw) of k for the Rg tiles of its row-group, i.e. a private stream of npass x Rg x nbw items
// (item = one 16-row tile x one 256-element block = 2304 B).  Few, fat waves on purpose: the dispatcher starts the waves of a
// grid over ~1 us (measured: the 16 waves of a 1024-thread workgroup began 0.25 / 0.33 / 0.67 / 1.05 us after launch, 4 at a time).
// (The second wave of a SIMD streams slower: done at 11.1 us of a gate | up launch, the first at 9.4.  Shares of 9 : 7 end both at 11.2, and the launch no earlier: the CU's loads are what is full, 28 bytes a ns.)
// A launch is a chain of latencies, and a wave issues one instruction every ~4 cycles (2 ns each where nothing overlaps), so:
//   * what the kernel does with its results is compiled in (KIND), what is launch-uniform is computed on the host and packed into
//     scalars delivered by KERNARG PRELOAD (SGPRs filled at wave launch: -mllvm -amdgpu-kernarg-preload-count=8) or read in two batches of
//     scalar loads: what the first requests need in front of them, what the end needs while the tiles travel.  Read where they are used, behind the last
//     barrier, the end's were a chain of ten waits.
//   * x comes first (behind one tile a wave), for the whole workgroup, one copy in LDS: a CU's loads return in the order they went out, and where every wave asks for its own slice of x in front of its tiles, the second four waves' slices
//     come behind the first four's tiles, from HBM (stamps: 2.3 us after the start, the first four's 1.4).  The barrier between the two costs the 0.15 us that the second four start later.
// Together (all epilogues in one kernel, every wave's own slice of x, scalars where they are used: before; now), logits to the host after every token: TinyLlama-1.1B Q4_K_M 40 rows 612 -> 535 us a token, Llama-3-8B
// Q4_K_M 130 rows 1559 -> 1410, Q5_K_M over 3-bit codes (8 layers) 489 -> 450, Q8_0 3000 rows (8 layers) 570 -> 540, Mixtral Q5_K_M (3 layers) 284 -> 266; a launch of 4096 x 4096 ends 3.8 us after its start instead of 4.0 (median
// workgroup; end behind the last barrier 0.22 us instead of 0.45), gate | up of the 8B model 11.6 instead of 12.3 (0.43 instead of 1.0).
// geom  = T | G << 8 | nbw << 16 | do_norm << 31         geom2 = nblk | Rg << 16        wbpack = wg_begin[1] | wg_begin[2] << 16
// MASK: the formats (1 << F_*) the instantiation handles; with more than one the segment's type decides at run time

// what a launch does with the rows (the epilogues of MvEpilogue that share one instantiation)
enum : int { MK_OUT = 0, MK_PAIR = 1, MK_QKV = 2, MK_MOE_PAIR = 3, MK_MOE_DOWN = 4 };   // store / + residual; SwiGLU; RoPE and the caches; the selected experts'
constexpr int mk_passes(int kind) { return kind == MK_PAIR || kind == MK_MOE_DOWN ? 2 : kind == MK_MOE_PAIR ? 4 : 1; }

struct MvqSeg {
  const uint8_t *w0, *w1;      // tiles of the pass, of the second pass (experts: of the stacks)
  const float *resid, *xq_nw;
  uint32_t n_rows, wg_begin, Rg, type;
  float* out;
  const float* bias;
  uint8_t* xq_out;
  float* xq_ssq;
  uint32_t epi, head_dim, max_seq, pad;
};
struct MvqArgs {
  const uint8_t *xq, *xq1;     // input (second expert's input of a down launch)
  const float* ssq_part;
  const int *sel0, *sel1;      // experts: whose matrices (first two passes or first pass, the rest)
  uint64_t stride0, stride1;
  uint32_t n_ssq, npass, k;
  float eps;
  const int* pos;
  const float* rope_cs;
  const float* moe_w;
  float* out2;
  uint8_t* xq_out2;
  uint64_t dbg_slot;
  MvqSeg seg[3];
};

// a pointer that is in scalar registers from here on (global: behind an asm statement the compiler would take it for any address)
template <class T>
__device__ __forceinline__ T* mvq_here(T* p) {
  auto g = (__attribute__((address_space(1))) T*)p;
  asm volatile("" : "+s"(g));
  return (T*)g;
}
__device__ __forceinline__ void mvq_scalar(uint32_t& v, const int* p) { asm volatile("s_load_dword %0, %1, 0x0\n\ts_waitcnt lgkmcnt(0)" : "=s"(v) : "s"(p) : "memory"); }

template <uint32_t MASK, int KIND>
__device__ __forceinline__ void mvq_body(uint32_t wbpack, uint32_t geom, uint32_t geom2, uint32_t red_off, uint32_t flags, const MvqArgs& A, uint8_t* smem8) {
  constexpr int NP = mk_passes(KIND);
  const uint32_t bid = blockIdx.x;
  const int sg = KIND == MK_QKV ? (int)(bid >= (wbpack & 0xFFFFu)) + (int)(bid >= (wbpack >> 16)) : 0;   // 0xFFFF = no such segment
  const MvqSeg& S = A.seg[sg];
  const uint32_t tid = threadIdx.x, lane = tid & 63;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // ---- the first batch of scalar loads
  const uint8_t *xq = A.xq, *xq1 = KIND == MK_MOE_DOWN ? A.xq1 : nullptr, *w0 = S.w0, *w1 = NP > 1 ? S.w1 : nullptr;
  uint32_t S_nrows = S.n_rows, S_wgb = KIND == MK_QKV ? S.wg_begin : 0u, Rg = KIND == MK_QKV ? S.Rg : geom2 >> 16, L_n_ssq = A.n_ssq, S_type = S.type;
  const float *S_resid = KIND == MK_OUT || KIND == MK_MOE_DOWN ? S.resid : nullptr, *S_nw = KIND == MK_OUT || KIND == MK_MOE_DOWN ? S.xq_nw : nullptr, *L_ssq_part = A.ssq_part;
  asm volatile("" : "+s"(S_nrows), "+s"(S_wgb), "+s"(Rg), "+s"(L_n_ssq), "+s"(S_type));
  xq = mvq_here(xq); w0 = mvq_here(w0); L_ssq_part = mvq_here(L_ssq_part);
  if (KIND == MK_MOE_DOWN) xq1 = mvq_here(xq1);
  if (NP > 1) w1 = mvq_here(w1);
  if (KIND == MK_OUT || KIND == MK_MOE_DOWN) { S_resid = mvq_here(S_resid); S_nw = mvq_here(S_nw); }
  constexpr bool kSingle = (MASK & (MASK - 1)) == 0;
  constexpr int kDp = kDepth;   // weight tiles in flight per wave
  const int fmt = kSingle ? __builtin_ctz(MASK) : fmt_of_dev_type((int)S_type);
  auto is = [&](int f) { return ((MASK >> f) & 1u) != 0 && (kSingle || fmt == f); };   // compile-time false for absent formats
  const uint32_t tb = is(F_Q4K) ? fmt_tile_bytes(F_Q4K) : is(F_Q6K) ? fmt_tile_bytes(F_Q6K) : is(F_Q5K) ? fmt_tile_bytes(F_Q5K)
                      : is(F_Q80) ? fmt_tile_bytes(F_Q80) : fmt_tile_bytes(F_Q40);
  const uint32_t S_T = geom & 0xFFu, S_G = (geom >> 8) & 0xFFu, nbw = (geom >> 16) & 0x3FFFu, S_nblk = geom2 & 0xFFFFu;
  const bool nrm = KIND != MK_MOE_DOWN && (geom >> 31) != 0;
  const uint32_t S_rpw = 16u * Rg * S_G;
  const uint32_t wg = bid - S_wgb;
  const int S_npass = KIND == MK_MOE_PAIR || KIND == MK_MOE_DOWN ? (int)A.npass : NP;
  const uint32_t nw = S_T * S_G;                                  // waves
  LGH_WSTAMP(0);
  LGH_SPAN(0);
  uint32_t ks = wave, rg = 0;                                     // wave = rg * T + ks (at most G - 1 subtractions)
  while (ks >= S_T) { ks -= S_T; rg++; }
  const bool active = rg < S_G;
  const uint32_t blk0 = ks * nbw;
  uint32_t nblk_w = active && blk0 < S_nblk ? min(nbw, S_nblk - blk0) : 0;   // (not const: see below)
  const uint32_t ntiles = (S_nrows + 15) >> 4;
  const uint32_t tile0 = (wg * S_G + rg) * Rg;
  uint32_t ntile_w = active && tile0 < ntiles ? min(Rg, ntiles - tile0) : 0;
  // LDS: the XQ records of x (1280 B per block, xq.h; a down launch of two experts: of both inputs), the partial-sum slots [pass][slice][row], 1 / rms, the rotation's cosines and sines
  const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem8;   // LDS byte address
  const uint32_t xbytes = S_nblk * kXqRecord;
  float* red = reinterpret_cast<float*>(smem8 + red_off);
  float* inv_at = red + (size_t)S_npass * S_T * S_rpw;
  // lane roles inside an MFMA: B operand = weight row n, k-chunk c (16 elements); the A operand is block-diagonal over the
  // four k-chunks — rows 4c'..4c'+3 = the four limbs of chunk c' — because XQ scales every 16 elements; so lane group
  // mq = c of D holds the limb sums of chunk c of weight row n
  const uint32_t n = lane & 15, mq = lane >> 4;

  // RMSNorm: the producer of x left partial sums of x^2; wave 0 gathers up to 256 of them now (oldest loads of the wave,
  // first used after the last tile) and the rest, if any, at the end
  // (four names, not an array: as one value of four registers the second load would wait for the first)
  float ss0 = 0.0f, ss1 = 0.0f, ss2 = 0.0f, ss3 = 0.0f;
  if (nrm && wave == 0) {
    if (lane < L_n_ssq) ss0 = L_ssq_part[lane];
    if (lane + 64 < L_n_ssq) ss1 = L_ssq_part[lane + 64];
    if (lane + 128 < L_n_ssq) ss2 = L_ssq_part[lane + 128];
    if (lane + 192 < L_n_ssq) ss3 = L_ssq_part[lane + 192];
  }
  // the residual element and the next consumer's norm weight of this thread's row
  float pre_res = 0.0f, pre_nw = 1.0f;
  const uint32_t row = wg * S_rpw + tid;
  const bool live = tid < S_rpw && row < S_nrows;
  if ((KIND == MK_OUT || KIND == MK_MOE_DOWN) && live) {
    if (S_resid) pre_res = S_resid[row];
    if (S_nw) pre_nw = S_nw[row];
  }
  LGH_WSTAMP(1);
  LGH_STAMP(0);

  // ---- x into LDS by LDS-DMA (no registers, no vector ALU), 1 KB a transfer.  Inline asm: with the builtin hipcc drains vmcnt to 0 at the next load it issues.
  auto x_request = [&](const uint8_t* src, uint32_t at) {
    for (uint32_t p = wave; p * 1024u < xbytes; p += nw) {
      const uint32_t off = p * 1024u + lane * 16u;
      if (off < xbytes) {
        uint32_t keep;
        asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off\n\ts_mov_b32 m0, %0"
                     : "=&s"(keep) : "v"(src + off), "s"(lds_base + at + p * 1024u) : "memory");
      }
    }
  };
  auto meet = [&]() { asm volatile("s_barrier" : : : "memory"); };

  // the passes' tiles; experts are chosen on the device, by SCALAR loads — vector loads would sit in the same in-order queue as the weight tiles
  const uint64_t woff = ((uint64_t)tile0 * S_nblk + blk0) * tb;
  const uint8_t *pb0 = w0 + woff, *pb1 = w1 + woff, *pb2 = nullptr, *pb3 = nullptr;
  if (KIND == MK_MOE_PAIR) {
    uint32_t e0, e1 = 0;
    mvq_scalar(e0, A.sel0);
    if (S_npass > 2) mvq_scalar(e1, A.sel1);
    pb2 = pb0 + (uint64_t)e1 * A.stride0;
    pb3 = pb1 + (uint64_t)e1 * A.stride1;
    pb0 += (uint64_t)e0 * A.stride0;
    pb1 += (uint64_t)e0 * A.stride1;
  } else if (KIND == MK_MOE_DOWN) {
    uint32_t e0, e1 = 0;
    mvq_scalar(e0, A.sel0);
    if (S_npass > 1) mvq_scalar(e1, A.sel1);
    pb0 += (uint64_t)e0 * A.stride0;
    pb1 += (uint64_t)e1 * A.stride1;
  }
  struct Pos { uint32_t p, tl, b; };
  auto issue = [&](const Pos& q, RawT16& r) {   // fmt_loads_per_tile(format) loads (the wait for x counts on it)
    const uint8_t* base = NP == 1 || q.p == 0 ? pb0 : NP == 2 || q.p == 1 ? pb1 : q.p == 2 ? pb2 : pb3;
    mvq_issue_tile<MASK>(fmt, base + ((size_t)q.tl * S_nblk + q.b) * tb, lane, r);
  };
  // item order: pass-major, then tile, then block (innermost: one accumulator per (pass, tile))
  Pos nx = {0, 0, 0};
  auto advance = [&]() {
    if (++nx.b == nblk_w) { nx.b = 0; if (++nx.tl == ntile_w) { nx.tl = 0; ++nx.p; } }
  };
  float acc = 0.0f;
  auto slot = [&](uint32_t p, uint32_t tl) -> float& { return red[(size_t)(p * S_T + ks) * S_rpw + (rg * Rg + tl) * 16 + n]; };
  // one item = 16 weight rows x 256 elements: four MFMAs (one per 64 elements); lane group c then holds,
  // for weight row n, the four limb sums of chunk 4pp + c, recombined to V = sum_k q_k * I_k (exact int, rounded once to f32).
  auto consume = [&](const Pos& q, const RawT16& r) {
    const uint32_t xat = KIND == MK_MOE_DOWN && q.p == 1 ? xbytes : 0u;
    mvq_consume_tile<MASK>(fmt, r, smem8 + xat + (blk0 + q.b) * kXqRecord, lane, acc);
    if (q.b + 1 == nblk_w) {   // last block of a (pass, tile): the four lane groups -> one partial sum per row
      const float t = swap32_add(swap16_add(acc));
      if (mq == 0) slot(q.p, q.tl) = t;
      acc = 0.0f;
    }
  };

  // ---- the second batch of scalar loads and what hangs on it: while the tiles travel
  float *S_out = nullptr, *S_ssq = nullptr, *L_out2 = nullptr;
  const float *S_bias = nullptr, *L_moe_w = nullptr, *L_cs = nullptr;
  uint8_t *S_xq = nullptr, *S_xq2 = nullptr;
  uint32_t S_epi = 0, S_hd = 0, S_maxseq = 0, L_k = 0, pos = 0;
  float L_eps = 0.0f;
  const uint32_t cs_at = (red_off + (uint32_t)S_npass * S_T * S_rpw * 4u + 16u + 15u) & ~15u;
  bool cs_lds = false;
  auto end_scalars = [&]() {
    S_out = S.out;
    if (KIND != MK_MOE_DOWN) { L_k = A.k; L_eps = A.eps; }
    if (KIND != MK_QKV) S_xq = S.xq_out;
    if (KIND == MK_OUT || KIND == MK_MOE_DOWN) S_ssq = S.xq_ssq;
    if (KIND == MK_OUT || KIND == MK_QKV) S_bias = S.bias;
    if (KIND == MK_QKV) { S_epi = S.epi; S_hd = S.head_dim; S_maxseq = S.max_seq; L_cs = A.rope_cs; }
    if (KIND == MK_MOE_PAIR) { L_out2 = A.out2; S_xq2 = A.xq_out2; }
    if (KIND == MK_MOE_DOWN) { L_out2 = A.out2; L_moe_w = A.moe_w; }
    if (KIND != MK_MOE_DOWN) asm volatile("" : "+s"(L_k), "+s"(L_eps));
    S_out = mvq_here(S_out);
    if (KIND != MK_QKV) S_xq = mvq_here(S_xq);
    if (KIND == MK_OUT || KIND == MK_MOE_DOWN) S_ssq = mvq_here(S_ssq);
    if (KIND == MK_OUT || KIND == MK_QKV) S_bias = mvq_here(S_bias);
    if (KIND == MK_QKV) {
      asm volatile("" : "+s"(S_epi), "+s"(S_hd), "+s"(S_maxseq));
      L_cs = mvq_here(L_cs);
    }
    if (KIND == MK_MOE_PAIR) S_xq2 = mvq_here(S_xq2);
    if (KIND == MK_MOE_PAIR || KIND == MK_MOE_DOWN) L_out2 = mvq_here(L_out2);
    if (KIND == MK_MOE_DOWN) L_moe_w = mvq_here(L_moe_w);
    if (KIND == MK_QKV) {
      mvq_scalar(pos, A.pos);
      cs_lds = (S_epi == EPI_ROPE_Q || S_epi == EPI_ROPE_K) && (flags & 1u) != 0;
    }
  };
  // the position's cosines and sines into LDS (behind the tiles: the compiler's waits for those do not know of it and wait for one load more than they have to)
  auto rotation = [&]() {
    if (KIND == MK_QKV && cs_lds && wave == 0 && lane * 4 < S_hd) {
      const uint8_t* src = reinterpret_cast<const uint8_t*>(L_cs) + (uint64_t)pos * S_hd * 4;
      uint32_t keep;
      asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off\n\ts_mov_b32 m0, %0"
                   : "=&s"(keep) : "v"(src + lane * 16), "s"(lds_base + cs_at) : "memory");
    }
  };

  auto x_all = [&]() {
    x_request(xq, 0);
    if (KIND == MK_MOE_DOWN && S_npass > 1) x_request(xq1, xbytes);
    meet();                                    // all of x is on its way: now the tiles
  };
  {
    // Opaque to the optimizer (the values do not change): otherwise every shape's loop-invariant bookkeeping — ~300
    // scalar instructions, most of them for paths not taken — is hoisted in front of the first load.
    asm volatile("" : "+s"(nblk_w), "+s"(ntile_w));
    const uint32_t nitems = (uint32_t)S_npass * ntile_w * nblk_w;
    auto x_finish = [&](auto n_tiles) {
      constexpr int NT = decltype(n_tiles)::value;
      // n_tiles x fmt_loads_per_tile loads were issued behind the x requests
#define LGH_WAIT_BEHIND(LPT)                                                                      \
  do {                                                                                           \
    if constexpr (NT * (LPT) == 20) asm volatile("s_waitcnt vmcnt(20)" ::: "memory");             \
    else if constexpr (NT * (LPT) == 16) asm volatile("s_waitcnt vmcnt(16)" ::: "memory");        \
    else if constexpr (NT * (LPT) == 15) asm volatile("s_waitcnt vmcnt(15)" ::: "memory");        \
    else if constexpr (NT * (LPT) == 12) asm volatile("s_waitcnt vmcnt(12)" ::: "memory");        \
    else if constexpr (NT * (LPT) == 10) asm volatile("s_waitcnt vmcnt(10)" ::: "memory");        \
    else if constexpr (NT * (LPT) == 9) asm volatile("s_waitcnt vmcnt(9)" ::: "memory");          \
    else if constexpr (NT * (LPT) == 8) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");          \
    else if constexpr (NT * (LPT) == 6) asm volatile("s_waitcnt vmcnt(6)" ::: "memory");          \
    else if constexpr (NT * (LPT) == 5) asm volatile("s_waitcnt vmcnt(5)" ::: "memory");          \
    else if constexpr (NT * (LPT) == 4) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");          \
    else if constexpr (NT * (LPT) == 3) asm volatile("s_waitcnt vmcnt(3)" ::: "memory");          \
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                                         \
  } while (0)
      if (is(F_Q6K) || is(F_Q80)) LGH_WAIT_BEHIND(5);
      else if (is(F_Q5K)) LGH_WAIT_BEHIND(4);
      else LGH_WAIT_BEHIND(3);
#undef LGH_WAIT_BEHIND
      meet();
      LGH_WSTAMP(4);
    };

    RawT16 buf[kDp];
    Pos at[kDp];
    // `run` for a static number of tiles put in flight up front; every path ends with nothing in flight
    auto run = [&](auto n_first) {
      constexpr int NF = decltype(n_first)::value;
      at[0] = nx; issue(nx, buf[0]); advance();   // one tile in front of x: HBM is at work while x comes (8 layers of an 8B model 374.5 -> 371 us a token; two tiles 374, x is late then)
      x_all();
#pragma unroll
      for (int j = 1; j < NF; j++) { at[j] = nx; issue(nx, buf[j]); advance(); }
      LGH_WSTAMP(2);
      end_scalars();
      x_finish(std::integral_constant<int, NF - 1>{});
      rotation();
      LGH_WSTAMP(5);
      if constexpr (NF < kDp) {   // that was everything
#pragma unroll
        for (int j = 0; j < NF; j++) consume(at[j], buf[j]);
      } else {
        uint32_t rem = nitems;       // not yet consumed; kDp of them in flight
        while (rem >= 2 * kDp) {
#pragma unroll
          for (int j = 0; j < kDp; j++) {
            consume(at[j], buf[j]);
            at[j] = nx; issue(nx, buf[j]); advance();
          }
          rem -= kDp;
        }
        const uint32_t unissued = rem - kDp;   // 0 .. kDp-1
#pragma unroll
        for (int j = 0; j < kDp; j++) {
          consume(at[j], buf[j]);
          if ((uint32_t)j < unissued) { at[j] = nx; issue(nx, buf[j]); advance(); }
        }
#pragma unroll
        for (int j = 0; j < kDp - 1; j++)
          if ((uint32_t)j < unissued) consume(at[j], buf[j]);
      }
    };
    if (nitems == 0) {
      if (nblk_w == 0 && ntile_w > 0) {
        // a k-slice beyond the last block (T does not divide the block count): its partial-sum slots must read as zero
        for (uint32_t p = 0; p < (uint32_t)S_npass; p++)
          for (uint32_t tl = 0; tl < ntile_w; tl++)
            if (mq == 0) slot(p, tl) = 0.0f;
      }
      x_all();
      end_scalars();
      x_finish(std::integral_constant<int, 0>{});
      rotation();
    } else if (nitems == 1) {
      run(std::integral_constant<int, 1>{});
    } else if (nitems == 2) {
      run(std::integral_constant<int, 2>{});
    } else if (nitems == 3) {
      run(std::integral_constant<int, 3>{});
    } else {
      run(std::integral_constant<int, kDp>{});
    }
    LGH_STAMP(3);
    LGH_WSTAMP(6);
  }
  if (nrm && wave == 0) {   // the producer's partial sums of x^2 -> 1 / rms (simd.rs:853-855)
    float ss = (ss0 + ss1) + (ss2 + ss3);
    for (uint32_t i = 256 + lane; i < L_n_ssq; i += 64) ss += L_ssq_part[i];
    ss = wave_sum_to_lane63(ss);
    if (lane == 63) inv_at[0] = mv_inv_rms(ss, L_k, L_eps);
  }
  if (KIND == MK_QKV) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // (the rotation's row, long since there)
  __syncthreads();
  LGH_STAMP(4);

  // ---- the end: one thread per row (or per row pair for RoPE)
  const float inv = nrm ? inv_at[0] : 1.0f;
  auto rowval = [&](int p, uint32_t rl) {
    const float* r = red + (size_t)p * S_T * S_rpw + rl;
    float v = 0.0f;
    if (S_T == 8) {
      float t[8];
#pragma unroll
      for (int j = 0; j < 8; j++) t[j] = r[j * S_rpw];
#pragma unroll
      for (int j = 0; j < 8; j++) v += t[j];
    } else {
#pragma nounroll
      for (uint32_t j = 0; j < S_T; j++) v += r[j * S_rpw];
    }
    return v * inv;
  };
  if (KIND == MK_QKV && (S_epi == EPI_ROPE_Q || S_epi == EPI_ROPE_K)) {
    const uint32_t rl = 2 * tid, r0 = wg * S_rpw + rl;
    if (rl < S_rpw && r0 < S_nrows) {
      float x0 = rowval(0, rl), x1 = rowval(0, rl + 1);
      if (S_bias) { x0 += S_bias[r0]; x1 += S_bias[r0 + 1]; }
      const uint32_t head = (S_hd & (S_hd - 1)) == 0 ? r0 >> __builtin_ctz(S_hd) : r0 / S_hd, e = r0 - head * S_hd;   // e even: the pair's first element
      float c, s;
      if (cs_lds) {
        const float* cs = reinterpret_cast<const float*>(smem8 + cs_at) + e;
        c = cs[0]; s = cs[1];
      } else {
        const float* cs = L_cs + (size_t)pos * S_hd + e;
        c = cs[0]; s = cs[1];
      }
      const float y0 = x0 * c - x1 * s, y1 = x0 * s + x1 * c;  // ops.rs:1326-1331
      float* dst = S_epi == EPI_ROPE_Q ? S_out + r0 : S_out + ((size_t)head * S_maxseq + pos) * S_hd + e;
      dst[0] = y0;
      dst[1] = y1;
    }
  } else if (live) {
    float v0 = rowval(0, tid);
    if ((KIND == MK_OUT || KIND == MK_QKV) && S_bias) v0 += S_bias[row];
    if (KIND == MK_QKV) {
      if (S_epi == EPI_V_CACHE) {
        const uint32_t head = (S_hd & (S_hd - 1)) == 0 ? row >> __builtin_ctz(S_hd) : row / S_hd;
        S_out[((size_t)head * S_maxseq + pos) * S_hd + (row - head * S_hd)] = v0;
      } else {
        S_out[row] = v0;
      }
    } else if (KIND == MK_MOE_PAIR) {
#pragma unroll
      for (int e = 0; e < 2; e++) {
        if (2 * e + 1 >= S_npass) break;
        const float g = e == 0 ? v0 : rowval(2, tid), a = silu_f(g) * rowval(2 * e + 1, tid);
        (e == 0 ? S_out : L_out2)[row] = a;
        uint8_t* xo = e == 0 ? S_xq : S_xq2;   // each expert's activation feeds its own down projection
        if (xo) xq_store_chunk(xo, row >> 4, a, nullptr, 0.0f, tid);
      }
    } else {
      float outv;
      if (KIND == MK_PAIR) outv = silu_f(v0) * rowval(1, tid);
      else if (KIND == MK_OUT) outv = S_resid ? v0 + pre_res : v0;
      else {
        // moe.rs:363-368: ONE zero-initialised sum, += weight * expert_out over all selected experts in selection order, then the
        // residual.  The experts run two per launch: a launch continues the running sum the earlier ones left (out2; none: it
        // starts from zero) and only the last one adds the residual (resid; none: the output is the running sum).
        float sum = L_out2 ? L_out2[row] : 0.0f;
        sum += L_moe_w[0] * v0;
        if (S_npass > 1) sum += L_moe_w[1] * rowval(1, tid);
        outv = S_resid ? sum + pre_res : sum;
      }
      S_out[row] = outv;
      // XQ image of the output for a matrix-core consumer (xq.h).  n_rows is a multiple of 16 here (host-checked), so the
      // 16 threads of a chunk are all live; with a norm in front of the consumer the record holds out * norm_weight and each
      // chunk leaves its sum of out^2.
      if (S_xq) xq_store_chunk(S_xq, row >> 4, outv * pre_nw, S_ssq, outv, tid);
    }
  }
  LGH_STAMP(5);
  LGH_WSTAMP(7);
  LGH_SPAN(1);
}

// Q, K and V of a layer (all of the mixes' launches are)
template <uint32_t MASK>
__global__ void __launch_bounds__(kWaves * 64) mvq_kernel(uint32_t wbpack, uint32_t geom, uint32_t geom2, uint32_t red_off, uint32_t flags, const MvqArgs A) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem8[];
  LGH_TL_BEGIN(mvq, lgh::TL_MVQ, geom2);
  mvq_body<MASK, MK_QKV>(wbpack, geom, geom2, red_off, flags, A, smem8);
  LGH_TL_END();
}
// everything else
template <uint32_t MASK, int KIND>
__global__ void __launch_bounds__(kWaves * 64) mvq_rows_kernel(uint32_t wbpack, uint32_t geom, uint32_t geom2, uint32_t red_off, uint32_t flags, const MvqArgs A) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem8[];
  LGH_TL_BEGIN(mvq, lgh::TL_MVQ, geom2);
  mvq_body<MASK, KIND>(wbpack, geom, geom2, red_off, flags, A, smem8);
  LGH_TL_END();
}

// ------------------------------------------------------------------------------------------------
// host: geometry and launch
// ------------------------------------------------------------------------------------------------
hipError_t mvq_plan(uint32_t k, uint32_t n_rows, int npass, MvPlan* plan, uint32_t launch_rows, uint32_t force_tiles) {
  if (k == 0 || k % 256 || n_rows == 0 || npass < 1 || npass > 4) return hipErrorInvalidValue;
  const uint32_t nblk = k / 256, W = kWaves;
  uint32_t T = 1;
  for (uint32_t t = 1; t <= W && t <= nblk; t++)
    if (nblk % t == 0) T = t;                       // largest divisor of nblk that fits the workgroup
  if (T < W / 2 && nblk > W) T = W;                 // awkward block counts: uneven k-slices
  if (T > nblk) T = nblk;
  const uint32_t G = W / T >= 1 ? W / T : 1;
  const uint32_t nbw = (nblk + T - 1) / T;
  if (launch_rows < n_rows) launch_rows = n_rows;
  const uint32_t tiles_launch = (launch_rows + 15) / 16;
  // tiles per workgroup: one workgroup per CU (two or three per CU, each with half / a third of the rows, measured the same
  // to 1 %: 15.5 / 15.6 / 15.7 us for the Llama-3-8B gate-up launch — a launch is bound by its fixed costs, not by waves in flight)
  uint32_t R = force_tiles ? force_tiles : (tiles_launch + kNumCU - 1) / kNumCU;   // (force_tiles: the engine balances mixed-format launches)
  R = (R + G - 1) / G * G;
  const uint32_t threads = T * G * 64;
  const uint32_t rmax = threads / 16 / G * G;         // the epilogue gives every row (pair) a thread
  if (R > rmax) R = rmax;
  plan->units = nbw;
  plan->T = T;
  plan->G = G;
  plan->rows_per_wg = 16 * R;
  plan->n_wg = ((n_rows + 15) / 16 + R - 1) / R;
  plan->threads = threads;
  plan->red_floats = (uint32_t)npass * T * 16 * R;
  return hipSuccess;
}

// LDS of a launch: x (of `n_x` inputs), the partial sums, 1 / rms (and the rotation's row where there is room)
static uint32_t mvq_red_offset(uint32_t nblk, uint32_t n_x) { return nblk * kXqRecord * n_x; }
static size_t mvq_lds_bytes(uint32_t nblk, uint32_t n_x, uint32_t red_floats) { return (size_t)mvq_red_offset(nblk, n_x) + (size_t)red_floats * 4 + 16; }

bool mvq_two_inputs(uint32_t k) { return mvq_lds_bytes((k + 255) / 256, 2, 2 * 8 * kWaves * 16) <= 160 * 1024; }   // (with the partial sums of up to eight tiles a workgroup)

// launch-uniform geometry of one op, packed for the kernel; returns the format mask (0 = not launchable)
uint32_t mvq_pack(const MvLaunch& L, uint32_t n_wg, uint32_t threads, MvGeom* g, size_t* lds_out) {
  const MvSeg& S0 = L.seg[0];
  if (threads == 0 || threads > kWaves * 64 || n_wg == 0 || L.nseg < 1 || L.nseg > 3) return 0;
  const uint32_t n_x = S0.epi == EPI_MOE_DOWN && S0.npass > 1 ? 2 : 1, row = S0.head_dim * 4;
  size_t lds = mvq_lds_bytes(S0.nblk, n_x, L.red_floats);
  if (lds > 160 * 1024) return 0;
  const bool rotation = (S0.epi == EPI_ROPE_Q || S0.epi == EPI_ROPE_K) && row % 16 == 0 && row <= 1024 && lds + 16 + row <= 160 * 1024;   // a transfer of 64 lanes
  if (rotation) lds += 16 + row;
  g->flags = rotation ? 1u : 0u;
  uint32_t mask = 0;
  for (int i = 0; i < L.nseg; i++) {   // the launch-uniform geometry travels as scalars
    const MvSeg& Si = L.seg[i];
    // (rows per workgroup may differ between the segments of one launch: a segment in a format with more bytes per tile
    // gets fewer tiles per workgroup; the kernel reads it per segment)
    if (Si.T != S0.T || Si.G != S0.G || Si.units != S0.units || Si.nblk != S0.nblk || Si.rows_per_wg % (16 * S0.G) ||
        (i > 0 && Si.wg_begin >= 0xFFFFu))
      return 0;
    const int f = fmt_of_dev_type(Si.type);
    if (f < 0) return 0;
    mask |= 1u << f;
  }
  const uint32_t Rg = S0.rows_per_wg / 16 / S0.G;
  if (S0.T > 255 || S0.G > 255 || S0.units > 0x3FFF || S0.nblk > 0xFFFF || Rg > 0xFFFF) return 0;
  g->wbpack = (L.nseg > 1 ? L.seg[1].wg_begin : 0xFFFFu) | (L.nseg > 2 ? L.seg[2].wg_begin : 0xFFFFu) << 16;
  g->geom = S0.T | S0.G << 8 | S0.units << 16 | (L.do_norm ? 1u << 31 : 0u);
  g->geom2 = S0.nblk | Rg << 16;
  g->lds_red_off = mvq_red_offset(S0.nblk, n_x);
  g->n_wg = n_wg;
  *lds_out = lds;
  return mask;
}

// the launch as the kernel takes it; the instantiation (MK_*), or -1 where there is none
static int mvq_args(const MvLaunch& L, MvqArgs* A) {
  std::memset(A, 0, sizeof(*A));
  const MvSeg& S0 = L.seg[0];
  int kind = -1;
  switch (S0.epi) {
    case EPI_STORE: case EPI_RESID: kind = L.nseg == 1 && S0.npass == 1 ? MK_OUT : -1; break;
    case EPI_SWIGLU: kind = L.nseg == 1 && S0.npass == 2 ? MK_PAIR : -1; break;
    case EPI_ROPE_Q: case EPI_ROPE_K: case EPI_V_CACHE: kind = MK_QKV; break;
    case EPI_MOE_SWIGLU: kind = L.nseg == 1 && (S0.npass == 2 || S0.npass == 4) ? MK_MOE_PAIR : -1; break;
    case EPI_MOE_DOWN: kind = L.nseg == 1 && (S0.npass == 1 || S0.npass == 2) ? MK_MOE_DOWN : -1; break;
    default: break;
  }
  if (kind < 0 || (kind == MK_MOE_DOWN && L.do_norm)) return -1;
  const MvPass* P = S0.pass;
  const bool moe = kind == MK_MOE_PAIR || kind == MK_MOE_DOWN;
  const int second = kind == MK_MOE_PAIR ? 2 : 1;   // the second expert's first pass
  for (int p = 0; p < S0.npass; p++) {
    if ((P[p].sel != nullptr) != moe) return -1;
    if (kind != MK_MOE_DOWN && P[p].xq != P[0].xq) return -1;
    if (moe && (P[p].plane[0] != P[p % second].plane[0] || P[p].sel_stride[0] != P[p % second].sel_stride[0] || P[p].sel != P[p / second * second].sel)) return -1;
  }
  A->xq = P[0].xq;
  A->xq1 = S0.npass > 1 ? P[1].xq : P[0].xq;
  A->ssq_part = L.ssq_part;
  A->n_ssq = L.n_ssq_part;
  A->npass = (uint32_t)S0.npass;
  A->k = L.k;
  A->eps = L.eps;
  A->pos = L.pos;
  A->rope_cs = L.rope_cs;
  A->moe_w = S0.moe_w;
  A->out2 = S0.out2;
  A->xq_out2 = S0.xq_out2;
  A->dbg_slot = L.dbg_slot;
  if (moe) {
    A->sel0 = P[0].sel;
    A->sel1 = S0.npass > second ? P[second].sel : P[0].sel;
    A->stride0 = P[0].sel_stride[0];
    A->stride1 = P[S0.npass > 1 ? 1 : 0].sel_stride[0];
  }
  for (int i = 0; i < L.nseg; i++) {
    const MvSeg& S = L.seg[i];
    if (i > 0 && (S.npass != 1 || S.pass[0].sel || S.pass[0].xq != P[0].xq)) return -1;
    if (i > 0 && S.epi != EPI_ROPE_Q && S.epi != EPI_ROPE_K && S.epi != EPI_V_CACHE && S.epi != EPI_STORE) return -1;
    if ((kind == MK_QKV && S.xq_out) || (kind == MK_PAIR && S.xq_nw) || ((moe || kind == MK_PAIR) && S.bias)) return -1;
    MvqSeg& D = A->seg[i];
    D.w0 = S.pass[0].plane[0];
    D.w1 = S.npass > 1 ? S.pass[1].plane[0] : S.pass[0].plane[0];
    D.resid = kind == MK_MOE_DOWN || S.epi == EPI_RESID ? S.resid : nullptr;
    D.xq_nw = S.xq_out ? S.xq_nw : nullptr;
    D.n_rows = S.n_rows;
    D.wg_begin = S.wg_begin;
    D.Rg = S.rows_per_wg / 16 / S.G;
    D.type = (uint32_t)S.type;
    D.out = S.out;
    D.bias = S.bias;
    D.xq_out = S.xq_out;
    D.xq_ssq = S.xq_ssq;
    D.epi = (uint32_t)S.epi;
    D.head_dim = S.head_dim;
    D.max_seq = S.max_seq;
  }
  return kind;
}

typedef void (*MvqKernel)(uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, const MvqArgs);
template <MvqKernel FN>
static hipError_t mvq_go(const MvqArgs& A, const MvGeom& g, uint32_t threads, size_t lds, hipStream_t st) {
  static bool attr_set[64] = {};
  if (hipError_t e = lds_opt_in(reinterpret_cast<const void*>(FN), 160 * 1024, attr_set); e != hipSuccess) return e;
  hipLaunchKernelGGL(FN, dim3(g.n_wg), dim3(threads), lds, st, g.wbpack, g.geom, g.geom2, g.lds_red_off, g.flags, A);
  return hipGetLastError();
}

template <uint32_t MASK>
static hipError_t mvq_kind(int kind, const MvqArgs& A, const MvGeom& g, uint32_t threads, size_t lds, hipStream_t st) {
  if (kind == MK_QKV) return mvq_go<&mvq_kernel<MASK>>(A, g, threads, lds, st);
  if constexpr ((MASK & (MASK - 1)) == 0) {   // (only the fused QKV launch mixes formats)
    switch (kind) {
      case MK_OUT: return mvq_go<&mvq_rows_kernel<MASK, MK_OUT>>(A, g, threads, lds, st);
      case MK_PAIR: return mvq_go<&mvq_rows_kernel<MASK, MK_PAIR>>(A, g, threads, lds, st);
      case MK_MOE_PAIR: return mvq_go<&mvq_rows_kernel<MASK, MK_MOE_PAIR>>(A, g, threads, lds, st);
      case MK_MOE_DOWN: return mvq_go<&mvq_rows_kernel<MASK, MK_MOE_DOWN>>(A, g, threads, lds, st);
      default: break;
    }
  }
  return hipErrorInvalidValue;
}

hipError_t mvq_launch(const MvLaunch& L, uint32_t n_wg, uint32_t threads, hipStream_t st) {
  MvGeom g;
  MvqArgs A;
  size_t lds = 0;
  const uint32_t mask = mvq_pack(L, n_wg, threads, &g, &lds);
  const int kind = mask ? mvq_args(L, &A) : -1;
  if (kind < 0) return hipErrorInvalidValue;
#define LGH_MVQ_CASE(M) case M: return mvq_kind<M>(kind, A, g, threads, lds, st)
  switch (mask) {   // single formats and the two mixes of the "_M" quantisations (fused QKV: V in Q6_K)
    LGH_MVQ_CASE(1u << F_Q4K); LGH_MVQ_CASE(1u << F_Q6K); LGH_MVQ_CASE(1u << F_Q5K); LGH_MVQ_CASE(1u << F_Q80); LGH_MVQ_CASE(1u << F_Q40);
    LGH_MVQ_CASE((1u << F_Q4K) | (1u << F_Q6K)); LGH_MVQ_CASE((1u << F_Q5K) | (1u << F_Q6K));
    default: return hipErrorInvalidValue;   // other mixes: the caller launches one format at a time
  }
#undef LGH_MVQ_CASE
}

uint32_t mvq_tile_bytes(int dev_type) {
  const int f = fmt_of_dev_type(dev_type);
  return f < 0 ? 0u : fmt_tile_bytes(f);
}

uint32_t mvq_format_mask(const MvLaunch& L) {
  uint32_t m = 0;
  for (int i = 0; i < L.nseg; i++) {
    const int f = fmt_of_dev_type(L.seg[i].type);
    if (f < 0) return 0;
    m |= 1u << f;
  }
  return m;
}

}  // namespace lgh
