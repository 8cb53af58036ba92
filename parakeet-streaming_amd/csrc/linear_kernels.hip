// gfx950 linear layers of the encoder (parakeet/modules/feedforward.py:4-26,
// attention.py:92,122, convolution.py:152,158):
//
//   out = act( x W^T + bias )
//
//   lin_tile_kernel  16 x 16 to 256 x 256 outputs a workgroup, both operands
//                    staged in LDS by buffer loads
//   lin_norm_kernel  few rows, with the residual update and LayerNorm (or two)
//                    that make x in the same launch (encoder.py:58-81)
//
// 16-bit operands, fp32 accumulation, one rounding of each output.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "pk_common.h"
#include "pk_device.h"

namespace pk {

template <typename ST>
struct MmaL;
template <>
struct MmaL<_Float16> {
  typedef _Float16 H8 __attribute__((ext_vector_type(8)));
  __device__ static inline f32x4_t k32(u32x4 a, u32x4 b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(H8, a), __builtin_bit_cast(H8, b), c, 0, 0, 0);
  }
};
template <>
struct MmaL<bf16_t> {
  typedef __bf16 H8 __attribute__((ext_vector_type(8)));
  __device__ static inline f32x4_t k32(u32x4 a, u32x4 b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(H8, a), __builtin_bit_cast(H8, b), c, 0, 0, 0);
  }
};

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// kEpiConv: GLU and the causal depthwise convolution with its cache (store_conv)
enum { kEpiNone = 0, kEpiSilu = 1, kEpiConv = 2 };
// what stands before the product: LayerNorm(x); r = x + alpha * branch, then
// LayerNorm(r); the same with a LayerNorm between, y = LayerNorm'(r)
// kProNormSilu: SiLU(LayerNorm(x)) of fp32 rows
enum { kProNorm = 1, kProResNorm = 2, kProResNorm2 = 3, kProNormSilu = 4 };
constexpr int kTaps = 9;  // depthwise taps of kEpiConv

template <typename ST>
struct LinK {
  const ST* x;  // [M][K] rows, stride x_s
  int64_t x_s;
  const ST* br;  // [M][K], stride br_s: the branch added to x (lin_norm_kernel)
  int64_t br_s;
  const ST* lnw;  // [K]: the LayerNorm that the product reads
  const ST* lnb;
  const ST* lnw0;  // [K]: kProResNorm2: the LayerNorm before it
  const ST* lnb0;
  ST* rout;  // [M][K], stride rout_s: r (kProResNorm) or y (kProResNorm2)
  int64_t rout_s;
  float alpha, eps, eps0;
  const ST* w;  // [N][K], stride w_s
  int64_t w_s;
  const ST* bias;  // [N] or nullptr
  ST* out;         // [M][N], stride out_s
  int64_t out_s;
  int32_t M, N, K;
  int32_t mtiles, xm;
  int32_t rpt;      // rows a tile (kEpiConv: whole streams of T frames)
  const float* xf;  // kProNormSilu: [M][K] fp32 rows, stride x_s
  // kEpiConv: rows are [batch][T] frames, W [2 D][K] (values, then gates); y
  // [batch T][D] fp32, the cache as in pk_conv_step
  float* y;
  int64_t y_s;
  ST* cache;
  const int32_t* slots;
  const uint8_t* pad;
  const int64_t* lengths;
  int64_t len_scalar;
  const ST* dw;   // [D][kTaps]
  const ST* dwb;  // [D] or nullptr
  int32_t num_slots, num_layers, layer, T, batch;
  int32_t per;  // streams a tile
};

template <typename ST>
__device__ static inline u32x2 pack4(const float* f) {
  u32x2 v;
  if constexpr (sizeof(ST) == 2 && __is_same(ST, bf16_t)) {
    v.x = bf16_pair_bits(f[0], f[1]);
    v.y = bf16_pair_bits(f[2], f[3]);
  } else {
    v.x = Tr<_Float16>::two(f);
    v.y = Tr<_Float16>::two(f + 2);
  }
  return v;
}

template <int EPI>
__device__ static inline float epi_act(float v) {
  if constexpr (EPI == kEpiSilu) return v / (1.f + __expf(-v));
  return v;
}

// Tile (m, n) of a workgroup: workgroups go to the XCDs in turn in launch order.
// xm > 0: grid (8, row tiles, column tiles of an XCD): the XCDs take an xm x 8/xm
// grid of equal blocks of tiles (the host picks xm, a power of two, so that a
// block's rows and weight columns together are fewest: what each XCD's L2
// fetches).  xm == 0 (the tiles do not divide): grid (tiles), contiguous runs of
// them an XCD, rows fastest.
__device__ static inline void xcd_tile(int mtiles, int xm, int& m, int& n) {
  if (xm > 0) {
    const int x = blockIdx.x, lg = xm == 1 ? 0 : xm == 2 ? 1 : xm == 4 ? 2 : 3;
    m = (x & (xm - 1)) * gridDim.y + blockIdx.y;
    n = (x >> lg) * gridDim.z + blockIdx.z;
    return;
  }
  const int total = gridDim.x, x = blockIdx.x & 7, j = blockIdx.x >> 3;
  const int t = x * (total >> 3) + min(x, total & 7) + j;
  m = t % mtiles;
  n = t / mtiles;
}

// `bytes` readable from base; a read past them gives zeros
__device__ static inline __amdgpu_buffer_rsrc_t bytes_rsrc(const void* base, uint32_t bytes) {
  // word 3 0x00020000: 32-bit data format, the setting untyped loads need on CDNA
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)bytes, 0x00020000);
}

// 16 bytes a lane to lds + 16 lane (lds wave-uniform)
__device__ static inline void load_lds16(const __amdgpu_buffer_rsrc_t r, unsigned char* lds, uint32_t off, int soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)lds, 16, off, soff, 0, 0);
}

// vmcnt(n): at most n of the wave's memory reads still in flight
template <int N>
__device__ static inline void wait_vm() {
  __builtin_amdgcn_s_waitcnt(0x0f70 | (N & 15) | ((N & 0x30) << 10));
}

// The sums of the WK parts of K meet in LDS (at smem + at); waves are numbered
// (wk WM + wm) WN + wn, the waves wk == 0 end with the sums.
template <int BM, int BN, int WMN, int WK, int TM, int TN>
__device__ static inline void sum_parts(unsigned char* smem, int at, f32x4_t (&acc)[TM][TN], int wave, int lane) {
  if constexpr (WK > 1) {
    f32x4_t* const red = reinterpret_cast<f32x4_t*>(smem + at);
    if (wave >= WMN) {
#pragma unroll
      for (int m = 0; m < TM; ++m)
#pragma unroll
        for (int n = 0; n < TN; ++n) red[((wave - WMN) * TM * TN + m * TN + n) * 64 + lane] = acc[m][n];
    }
    __syncthreads();
    if (wave < WMN) {
#pragma unroll
      for (int w = 1; w < WK; ++w)
#pragma unroll
        for (int m = 0; m < TM; ++m)
#pragma unroll
          for (int n = 0; n < TN; ++n) acc[m][n] += red[((wave + (w - 1) * WMN) * TM * TN + m * TN + n) * 64 + lane];
    }
  }
}

// A tile's output: bias and activation, then through LDS to whole 16-byte chunks
// of a row.  smem is free when every wave is here.
template <typename ST, int BM, int BN, int WM, int WN, int WK, int TM, int TN, int EPI>
__device__ static inline void store_tile(const LinK<ST>& p, unsigned char* smem, f32x4_t (&acc)[TM][TN], int row0, int n0,
                                         int wave, int lane) {
  constexpr int NW = WM * WN * WK;
  constexpr int OS = BN + 8;  // LDS row stride of the staged output
  constexpr int kOut = BM * OS * 2;
  const int l16 = lane & 15, kg = lane >> 4;
  const int wk = wave / (WM * WN), wm = (wave / WN) % WM, wn = wave % WN;
  sum_parts<BM, BN, WM * WN, WK>(smem, kOut, acc, wave, lane);
  ST* const os = reinterpret_cast<ST*>(smem);
  if (wk == 0) {
#pragma unroll
    for (int n = 0; n < TN; ++n) {
      const int c = (wn * TN + n) * 16 + kg * 4;
      float b[4] = {0.f, 0.f, 0.f, 0.f};
      if (p.bias) {
#pragma unroll
        for (int e = 0; e < 4; ++e) b[e] = from_st(p.bias[n0 + c + e]);
      }
#pragma unroll
      for (int m = 0; m < TM; ++m) {
        float f[4] = {acc[m][n].x, acc[m][n].y, acc[m][n].z, acc[m][n].w};
#pragma unroll
        for (int e = 0; e < 4; ++e) f[e] = epi_act<EPI>(f[e] + b[e]);
        *reinterpret_cast<u32x2*>(os + ((wm * TM + m) * 16 + l16) * OS + c) = pack4<ST>(f);
      }
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < BM * BN / 8; i += 64 * NW) {
    const int r = i / (BN / 8), c = (i % (BN / 8)) * 8;
    if (row0 + r < p.M) st16(p.out + (int64_t)(row0 + r) * p.out_s + n0 + c, *reinterpret_cast<const u32x4*>(os + r * OS + c));
  }
}

// The first pointwise convolution's tile up to the depthwise convolution
// (convolution.py:37-47,152-155), in place of a launch that reads its output
// back: the weight rows of a tile alternate 16 values and their 16 gates, so a
// lane holds both; GLU in fp32, zero where padded, rounded once to the storage
// type (what the cache holds); then a thread takes 2 channels of a stream: its
// cache rows (loaded before the product, `cw`), the tile's frames, fp32 sums in
// pk_conv_step's order, the next cache in place.  A tile holds whole streams, so
// no other workgroup touches these channels of their caches.  840 rows (60
// streams x 14) x 1024 -> 2048: 12.8 us and 4.8 for the norm after it, against
// 10.8 for the product and 14.8 for the convolution step as launches of their own;
// 256 rows x 512 7.7 (residual and norm in it) against 13 for the three.
struct ConvItem {
  uint32_t cw[kTaps - 1], tw[kTaps];  // 2 channels of the cache rows; 2 x kTaps taps
};
template <typename ST>
__device__ static inline ST* conv_cache(const LinK<ST>& p, int b, int c) {
  const int slot = p.slots ? p.slots[b] : b;
  if ((uint32_t)slot >= (uint32_t)p.num_slots) return nullptr;  // such a stream is left untouched
  return p.cache + ((int64_t)slot * p.num_layers + p.layer) * (kTaps - 1) * (p.N / 2) + c;
}
template <typename ST, int CB>
__device__ static inline void conv_load(const LinK<ST>& p, int i, int mt_i, int c0, ConvItem& it) {
  const int per = p.per;
  const int s = i / (CB / 2), c = c0 + (i % (CB / 2)) * 2, b = mt_i * per + s;
  if (s >= per || b >= p.batch) return;
  const uint32_t* tp = reinterpret_cast<const uint32_t*>(p.dw + (int64_t)c * kTaps);  // c even: 4-byte aligned
#pragma unroll
  for (int k = 0; k < kTaps; ++k) it.tw[k] = tp[k];
  const ST* q = conv_cache(p, b, c);
  if (!q) return;
#pragma unroll
  for (int r = 0; r < kTaps - 1; ++r) it.cw[r] = *reinterpret_cast<const uint32_t*>(q + (int64_t)r * (p.N / 2));
}
template <typename ST>
__device__ static inline void two_of(uint32_t w, float& lo, float& hi) {
  if constexpr (__is_same(ST, bf16_t)) {
    lo = __uint_as_float(w << 16);
    hi = __uint_as_float(w & 0xffff0000u);
  } else {
    float f[2];
    Tr<_Float16>::two(w, f);
    lo = f[0];
    hi = f[1];
  }
}
template <typename ST>
__device__ static inline uint32_t pack2(float lo, float hi) {
  if constexpr (__is_same(ST, bf16_t)) return bf16_pair_bits(lo, hi);
  const float f[2] = {lo, hi};
  return Tr<_Float16>::two(f);
}
template <typename ST, int BM, int BN, int WM, int WN, int WK, int TM, int TN>
__device__ static inline void store_conv(const LinK<ST>& p, unsigned char* smem, f32x4_t (&acc)[TM][TN], int mt_i, int nt_i,
                                         ConvItem& it, int wave, int lane) {
  constexpr int NTH = 64 * WM * WN * WK;
  constexpr int CB = BN / 2, GS = CB + 8;
  constexpr int kOut = BM * GS * 2;
  const int D = p.N / 2, c0 = nt_i * CB, row0 = mt_i * p.rpt;
  const int l16 = lane & 15, kg = lane >> 4;
  const int wm = (wave / WN) % WM, wn = wave % WN;
  sum_parts<BM, BN, WM * WN, WK>(smem, kOut, acc, wave, lane);
  ST* const gl = reinterpret_cast<ST*>(smem);  // [BM][GS] GLU outputs
  if (wave < WM * WN) {
#pragma unroll
    for (int m = 0; m < TM; ++m) {
      const int lr = (wm * TM + m) * 16 + l16, row = min(row0 + lr, p.M - 1);
      const int b = row / p.T, t = row - b * p.T;
      const bool valid = p.pad ? p.pad[row] == 0 : (int64_t)t < (p.lengths ? p.lengths[b] : p.len_scalar);
#pragma unroll
      for (int n = 0; n < TN / 2; ++n) {
        const int c = (wn * (TN / 2) + n) * 16 + kg * 4;
        float f[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float a = acc[m][2 * n][e], g = acc[m][2 * n + 1][e];
          if (p.bias) {
            a += from_st(p.bias[c0 + c + e]);
            g += from_st(p.bias[D + c0 + c + e]);
          }
          f[e] = valid ? a / (1.f + __expf(-g)) : 0.f;
        }
        *reinterpret_cast<u32x2*>(gl + lr * GS + c) = pack4<ST>(f);
      }
    }
  }
  __syncthreads();
  const int per = p.per;
  for (int i = threadIdx.x; i < per * (CB / 2); i += NTH) {
    const int s = i / (CB / 2), cl = (i % (CB / 2)) * 2, c = c0 + cl, b = mt_i * per + s;
    if (b >= p.batch) break;  // streams ascend
    if (i >= NTH) conv_load<ST, CB>(p, i, mt_i, c0, it);  // past the ones loaded ahead
    ST* const q = conv_cache(p, b, c);
    if (!q) continue;
    float w[2][kTaps], win[kTaps][2], bias[2] = {0.f, 0.f};
#pragma unroll
    for (int k = 0; k < kTaps; ++k) {
      // element e of the pair's 2 kTaps taps: channel e / kTaps, tap e % kTaps
      float lo, hi;
      two_of<ST>(it.tw[k], lo, hi);
      w[(2 * k) / kTaps][(2 * k) % kTaps] = lo;
      w[(2 * k + 1) / kTaps][(2 * k + 1) % kTaps] = hi;
    }
    if (p.dwb) {
      bias[0] = from_st(p.dwb[c]);
      bias[1] = from_st(p.dwb[c + 1]);
    }
#pragma unroll
    for (int r = 0; r < kTaps - 1; ++r) two_of<ST>(it.cw[r], win[r][0], win[r][1]);
    float* yp = p.y + (int64_t)b * p.T * p.y_s + c;
    for (int t = 0; t < p.T; ++t) {
      two_of<ST>(*reinterpret_cast<const uint32_t*>(gl + (s * p.T + t) * GS + cl), win[kTaps - 1][0], win[kTaps - 1][1]);
      float2 o = {bias[0], bias[1]};
#pragma unroll
      for (int k = 0; k < kTaps; ++k) {
        o.x = fmaf(w[0][k], win[k][0], o.x);
        o.y = fmaf(w[1][k], win[k][1], o.y);
      }
      *reinterpret_cast<float2*>(yp + t * p.y_s) = o;
#pragma unroll
      for (int k = 0; k < kTaps - 1; ++k) {
        win[k][0] = win[k + 1][0];
        win[k][1] = win[k + 1][1];
      }
    }
#pragma unroll
    for (int r = 0; r < kTaps - 1; ++r)
      *reinterpret_cast<uint32_t*>(q + (int64_t)r * D) = pack2<ST>(win[r][0], win[r][1]);
  }
}

// row of W that a tile's output column n (of BN) multiplies
template <int BN, int EPI>
__device__ static inline int w_row(int nt_i, int n, int N) {
  if constexpr (EPI == kEpiConv) return ((n & 16) ? N / 2 : 0) + nt_i * (BN / 2) + (n >> 5) * 16 + (n & 15);
  return nt_i * BN + n;
}

// Many rows: BM x BN outputs a workgroup, WM x WN x WK waves, both operands
// staged in LDS BK columns a stage (S stages in flight, buffer loads straight to
// LDS).  A row's 16-byte chunks are permuted within each 128 bytes by the row's
// low three bits, so the 16 rows of an operand read fall on distinct banks in stages
// of 64 columns; in longer ones two rows share each bank (40-46% of LDS's active
// cycles in the counters, 11-13% of the launch's time active).
// Small tiles split K over the waves (WK): each staged byte is then read from LDS
// once or twice, and the sum over the waves costs one exchange at the end.
// Bound by: latency up to about one tile a CU (128 x 512 -> 2048 with SiLU 4.2 us,
// torch's GEMM and SiLU 10.2); on the large forms the chain of a stage, its loads and
// barrier, then operand reads, then products, with two waves a SIMD or fewer to
// overlap: counters at 840 x 1024 -> 4096 have the matrix cores busy 19% of the time,
// LDS active 16%, L2 at 7.3 TB/s and the waves waiting 46% of their cycles (3584 rows
// 29%, 13%, 5.7 and 35%).  An operand read straight from memory (16 rows x 64 bytes
// an instruction, half of each 128-byte line) moved 37 GB/s a CU against about 100
// through LDS: 16 rows x 2048 -> 512 6.1 us so, 4.4 staged (torch's GEMM 7.9).
// 840 x 1024 -> 4096 with SiLU 13.6 us (518 TFLOP/s) against
// 21.3, 840 x 4096 -> 1024 17.1 against 19.5 for torch's.
template <typename ST, int BM, int BN, int WM, int WN, int WK, int BK, int S, int EPI>
__global__ void __launch_bounds__(64 * WM * WN * WK) lin_tile_kernel(const LinK<ST> p) {
#pragma clang fp contract(off)
  constexpr int NW = WM * WN * WK;
  constexpr int TM = BM / WM / 16, TN = BN / WN / 16;  // 16x16 products a wave
  constexpr int CH = BK / 8;                           // 16-byte chunks a row
  constexpr int kStage = (BM + BN) * BK * 2;
  constexpr int LPS = kStage / 1024 / NW;  // loads a wave issues a stage
  static_assert(BK % 64 == 0, "the permutation stays within a row's stage: whole groups of 8 chunks");
  static_assert(kStage % (1024 * NW) == 0 && (BM * CH) % 64 == 0, "whole waves of chunks");
  constexpr int KS = BK / 32 / WK;  // 32-column steps a wave does a stage
  constexpr int OS = BN + 8;        // LDS row stride of the staged output
  constexpr int kOut = BM * OS * 2;
  constexpr int kRed = WK > 1 ? (WK - 1) * BM * BN * 4 : 0;
  constexpr int kSmem = S * kStage > kOut + kRed ? S * kStage : kOut + kRed;
  __shared__ __align__(16) unsigned char smem[kSmem];

  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, kg = lane >> 4;
  const int wk = wave / (WM * WN), wm = (wave / WN) % WM, wn = wave % WN;
  int mt_i, nt_i;
  xcd_tile(p.mtiles, p.xm, mt_i, nt_i);
  const int row0 = mt_i * p.rpt, n0 = nt_i * BN;

  // chunk c of a stage: row c / CH of [x rows ; w rows], LDS position c % CH
  const __amdgpu_buffer_rsrc_t rx = bytes_rsrc(p.x, (uint32_t)((p.M - 1) * p.x_s + p.K) * 2u);
  const __amdgpu_buffer_rsrc_t rw = bytes_rsrc(p.w, (uint32_t)((p.N - 1) * p.w_s + p.K) * 2u);
  uint32_t off[LPS];
#pragma unroll
  for (int i = 0; i < LPS; ++i) {
    const int c = (i * NW + wave) * 64 + lane;
    const int r = c / CH, pos = c % CH;
    const int ch = (pos & ~7) | ((pos ^ r) & 7);
    off[i] = r < BM ? (uint32_t)(min(row0 + r, p.M - 1) * p.x_s + ch * 8) * 2u
                    : (uint32_t)(w_row<BN, EPI>(nt_i, r - BM, p.N) * p.w_s + ch * 8) * 2u;
  }
  auto issue = [&](int st, int k) {
#pragma unroll
    for (int i = 0; i < LPS; ++i) {
      const int base = (i * NW + wave) * 64;  // wave-uniform: whole waves of one operand
      load_lds16(base < BM * CH ? rx : rw, smem + st * kStage + base * 16, off[i], k * 2);
    }
  };
  f32x4_t acc[TM][TN];
#pragma unroll
  for (int m = 0; m < TM; ++m)
#pragma unroll
    for (int n = 0; n < TN; ++n) acc[m][n] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  const int iters = p.K / BK;
  ConvItem cv;
  if constexpr (EPI == kEpiConv) {
    conv_load<ST, BN / 2>(p, threadIdx.x, mt_i, nt_i * (BN / 2), cv);
    __builtin_amdgcn_sched_barrier(0);  // ahead of the stages, whose counts the waits below rely on
  }
#pragma unroll
  for (int s = 0; s < S - 1; ++s)
    if (s < iters) issue(s, s * BK);
  int st = 0;
  for (int it = 0; it < iters; ++it) {
    // this stage's loads are in; the later stages' may still be in flight
    if (it + S - 2 < iters)
      wait_vm<(S - 2) * LPS>();
    else
      wait_vm<0>();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();  // every wave's part of the stage; the slot refilled below is read by none
    asm volatile("" ::: "memory");
    if (it + S - 1 < iters) issue(st == 0 ? S - 1 : st - 1, (it + S - 1) * BK);
    const unsigned char* xs = smem + st * kStage;
    const unsigned char* ws = xs + BM * BK * 2;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const int ch = (wk * KS + s) * 4 + kg;
      u32x4 xf[TM], wf[TN];
#pragma unroll
      for (int m = 0; m < TM; ++m) {
        const int r = (wm * TM + m) * 16 + l16;
        xf[m] = *reinterpret_cast<const u32x4*>(xs + r * BK * 2 + ((ch & ~7) | ((ch ^ r) & 7)) * 16);
      }
#pragma unroll
      for (int n = 0; n < TN; ++n) {
        const int r = (wn * TN + n) * 16 + l16;
        wf[n] = *reinterpret_cast<const u32x4*>(ws + r * BK * 2 + ((ch & ~7) | ((ch ^ r) & 7)) * 16);
      }
#pragma unroll
      for (int m = 0; m < TM; ++m)
#pragma unroll
        for (int n = 0; n < TN; ++n) acc[m][n] = MmaL<ST>::k32(wf[n], xf[m], acc[m][n]);
    }
    st = st == S - 1 ? 0 : st + 1;
  }
  __syncthreads();
  if constexpr (EPI == kEpiConv)
    store_conv<ST, BM, BN, WM, WN, WK, TM, TN>(p, smem, acc, mt_i, nt_i, cv, wave, lane);
  else
    store_tile<ST, BM, BN, WM, WN, WK, TM, TN, EPI>(p, smem, acc, row0, n0, wave, lane);
}

// A Conformer layer's residual update and LayerNorm (encoder.py:58-81) in the
// launch of the product that reads it: BM rows x BN outputs a workgroup.  The
// weight stages are on their way (as in lin_tile_kernel) while the waves update
// and normalise the tile's whole rows into LDS; a row's statistics are fp32,
// two passes over the values in registers, and the residual and the norm round
// to the storage type as pk_residual_norm rounds them.  Every workgroup of a row
// tile normalises the same rows again (about 14 vector operations an element,
// 0.8 us a CU for 16 rows x 512), which is less than a launch of its own (4 us)
// until a CU has several tiles: the host takes this form for few rows.
template <typename ST, int KV, int BM, int BN, int WN, int WK, int BK, int S, int PRO, int EPI>
__global__ void __launch_bounds__(64 * WN * WK) lin_norm_kernel(const LinK<ST> p) {
#pragma clang fp contract(off)
  constexpr int K = 512 * KV;
  constexpr int NW = WN * WK;
  constexpr int TM = BM / 16, TN = BN / WN / 16;
  constexpr int CH = BK / 8;
  constexpr int kAct = BM * K * 2;  // the normalised rows, [BM][K], chunks permuted as in a stage
  constexpr int kStage = BN * BK * 2;
  constexpr int LPS = kStage / 1024 / NW;
  constexpr int KS = BK / 32 / WK;
  constexpr int RPW = BM / NW;  // rows a wave normalises
  static_assert(BK % 64 == 0 && K % BK == 0, "whole groups of 8 chunks, whole stages");
  static_assert(kStage % (1024 * NW) == 0 && BM % NW == 0 && KS > 0, "whole waves of chunks and rows");
  constexpr int OS = BN + 8;
  constexpr int kOut = BM * OS * 2;
  constexpr int kRed = (WK - 1) * BM * BN * 4;
  constexpr int kSmem = kAct + S * kStage > kOut + kRed ? kAct + S * kStage : kOut + kRed;
  __shared__ __align__(16) unsigned char smem[kSmem];

  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, kg = lane >> 4;
  const int wk = wave / WN, wn = wave % WN;
  int mt_i, nt_i;
  xcd_tile(p.mtiles, p.xm, mt_i, nt_i);
  const int row0 = mt_i * p.rpt, n0 = nt_i * BN;

  const __amdgpu_buffer_rsrc_t rw = bytes_rsrc(p.w, (uint32_t)((p.N - 1) * p.w_s + p.K) * 2u);
  unsigned char* const ring = smem + kAct;
  uint32_t off[LPS];
#pragma unroll
  for (int i = 0; i < LPS; ++i) {
    const int c = (i * NW + wave) * 64 + lane;
    const int r = c / CH, pos = c % CH;
    off[i] = (uint32_t)(w_row<BN, EPI>(nt_i, r, p.N) * p.w_s + ((pos & ~7) | ((pos ^ r) & 7)) * 8) * 2u;
  }
  auto issue = [&](int st, int k) {
#pragma unroll
    for (int i = 0; i < LPS; ++i) load_lds16(rw, ring + st * kStage + (i * NW + wave) * 1024, off[i], k * 2);
  };

  // the rows first (their use comes first), then the first weight stages
  constexpr bool kRes = PRO == kProResNorm || PRO == kProResNorm2;
  u32x4 xv[RPW][KV], bv[RPW][KV], lwv[KV], lbv[KV], lwv0[KV], lbv0[KV];
  ConvItem cv;
  if constexpr (EPI == kEpiConv) conv_load<ST, BN / 2>(p, threadIdx.x, mt_i, nt_i * (BN / 2), cv);
#pragma unroll
  for (int v = 0; v < KV; ++v) {
    const int c = (lane + 64 * v) * 8;
#pragma unroll
    for (int r = 0; r < RPW; ++r) {
      const int row = min(row0 + wave * RPW + r, p.M - 1);
      if constexpr (PRO == kProNormSilu) {  // 8 fp32 values: 2 chunks
        xv[r][v] = ld16(p.xf + row * p.x_s + c);
        bv[r][v] = ld16(p.xf + row * p.x_s + c + 4);
      } else {
        xv[r][v] = ld16(p.x + row * p.x_s + c);
        if constexpr (kRes) bv[r][v] = ld16(p.br + row * p.br_s + c);
      }
    }
    lwv[v] = ld16(p.lnw + c);
    lbv[v] = ld16(p.lnb + c);
    if constexpr (PRO == kProResNorm2) {
      lwv0[v] = ld16(p.lnw0 + c);
      lbv0[v] = ld16(p.lnb0 + c);
    }
  }
  constexpr int iters = K / BK;
#pragma unroll
  for (int s = 0; s < S - 1; ++s)
    if (s < iters) issue(s, s * BK);
  __builtin_amdgcn_sched_barrier(0);  // all of the above in flight before any use

  const bool scaled = p.alpha != 1.f;
  auto normed = [&](float (&f)[KV][8], const u32x4* lw, const u32x4* lb, float eps) {
    float s = 0.f;
#pragma unroll
    for (int v = 0; v < KV; ++v)
#pragma unroll
      for (int e = 0; e < 8; ++e) s += f[v][e];
    const float mean = group_sum<64>(s) * (1.f / (float)K);
    float q = 0.f;
#pragma unroll
    for (int v = 0; v < KV; ++v)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        f[v][e] -= mean;
        q = fmaf(f[v][e], f[v][e], q);
      }
    const float rstd = rsqrtf(group_sum<64>(q) * (1.f / (float)K) + eps);
#pragma unroll
    for (int v = 0; v < KV; ++v) {
      float w[8], b[8];
      Tr<ST>::unpack(lw[v], w);
      Tr<ST>::unpack(lb[v], b);
#pragma unroll
      for (int e = 0; e < 8; ++e) f[v][e] = fmaf(f[v][e] * rstd, w[e], b[e]);
    }
  };
#pragma unroll
  for (int r = 0; r < RPW; ++r) {
    const int lr = wave * RPW + r;
    const bool write = kRes && nt_i == 0 && lr < p.rpt && row0 + lr < p.M;  // one workgroup of the row tile
    ST* const rout = p.rout + (int64_t)(row0 + lr) * p.rout_s;
    float f[KV][8];
#pragma unroll
    for (int v = 0; v < KV; ++v) {
      if constexpr (PRO == kProNormSilu) {
        Tr<float>::unpack(xv[r][v], f[v]);
        Tr<float>::unpack(bv[r][v], f[v] + 4);
      } else {
        Tr<ST>::unpack(xv[r][v], f[v]);
      }
      if constexpr (kRes) {
        float b[8];
        Tr<ST>::unpack(bv[r][v], b);
#pragma unroll
        for (int e = 0; e < 8; ++e) f[v][e] = round_to<ST>(f[v][e] + (scaled ? round_to<ST>(p.alpha * b[e]) : b[e]));
      }
    }
    if constexpr (PRO == kProResNorm2) {
      normed(f, lwv0, lbv0, p.eps0);
#pragma unroll
      for (int v = 0; v < KV; ++v)
#pragma unroll
        for (int e = 0; e < 8; ++e) f[v][e] = round_to<ST>(f[v][e]);
    }
    if (write) {
#pragma unroll
      for (int v = 0; v < KV; ++v) st16(rout + (lane + 64 * v) * 8, Tr<ST>::pack(f[v]));
    }
    normed(f, lwv, lbv, p.eps);
#pragma unroll
    for (int v = 0; v < KV; ++v) {
      const int c = lane + 64 * v;
      if constexpr (PRO == kProNormSilu) {
#pragma unroll
        for (int e = 0; e < 8; ++e) f[v][e] = epi_act<kEpiSilu>(f[v][e]);
      }
      *reinterpret_cast<u32x4*>(smem + lr * K * 2 + ((c & ~7) | ((c ^ lr) & 7)) * 16) = Tr<ST>::pack(f[v]);
    }
  }

  // the wave's rows are in LDS before the first barrier below (lgkmcnt(0) alone:
  // the weight stages stay in flight)
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt(0xc07f);
  __builtin_amdgcn_sched_barrier(0);

  f32x4_t acc[TM][TN];
#pragma unroll
  for (int m = 0; m < TM; ++m)
#pragma unroll
    for (int n = 0; n < TN; ++n) acc[m][n] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  int st = 0;
#pragma unroll 1
  for (int it = 0; it < iters; ++it) {
    // this stage's loads are in, the later stages' may be in flight (stores of
    // the residual only make the wait longer)
    if (it + S - 2 < iters)
      wait_vm<(S - 2) * LPS>();
    else
      wait_vm<0>();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (it + S - 1 < iters) issue(st == 0 ? S - 1 : st - 1, (it + S - 1) * BK);
    const unsigned char* ws = ring + st * kStage;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const int ch = (wk * KS + s) * 4 + kg, xch = it * CH + ch;
      u32x4 xf[TM], wf[TN];
#pragma unroll
      for (int m = 0; m < TM; ++m) {
        const int r = m * 16 + l16;
        xf[m] = *reinterpret_cast<const u32x4*>(smem + r * K * 2 + ((xch & ~7) | ((xch ^ r) & 7)) * 16);
      }
#pragma unroll
      for (int n = 0; n < TN; ++n) {
        const int r = (wn * TN + n) * 16 + l16;
        wf[n] = *reinterpret_cast<const u32x4*>(ws + r * BK * 2 + ((ch & ~7) | ((ch ^ r) & 7)) * 16);
      }
#pragma unroll
      for (int m = 0; m < TM; ++m)
#pragma unroll
        for (int n = 0; n < TN; ++n) acc[m][n] = MmaL<ST>::k32(wf[n], xf[m], acc[m][n]);
    }
    st = st == S - 1 ? 0 : st + 1;
  }
  __syncthreads();
  if constexpr (EPI == kEpiConv)
    store_conv<ST, BM, BN, 1, WN, WK, TM, TN>(p, smem, acc, mt_i, nt_i, cv, wave, lane);
  else
    store_tile<ST, BM, BN, 1, WN, WK, TM, TN, EPI>(p, smem, acc, row0, n0, wave, lane);
}

// SiLU(LayerNorm(x)) of fp32 rows (convolution.py:156-157), a wave a row, for the
// row counts past lin_norm_kernel: bound by a launch and its 6 bytes an element
// (4.8 us in the trace for 840 rows x 1024, 5.2 for 4096 x 512)
template <typename ST, int KV>
__global__ void __launch_bounds__(256) norm_silu_kernel(const float* x, int64_t x_s, const ST* lnw, const ST* lnb, float eps,
                                                        ST* out, int64_t out_s, int rows) {
#pragma clang fp contract(off)
  constexpr int K = 512 * KV;
  const int lane = threadIdx.x & 63, row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;  // the whole wave: no barrier below
  float f[KV][8];
  u32x4 wv[KV], bv[KV];
  float s = 0.f;
#pragma unroll
  for (int v = 0; v < KV; ++v) {
    const int c = (lane + 64 * v) * 8;
    Tr<float>::unpack(ld16(x + row * x_s + c), f[v]);
    Tr<float>::unpack(ld16(x + row * x_s + c + 4), f[v] + 4);
    wv[v] = ld16(lnw + c);
    bv[v] = ld16(lnb + c);
  }
#pragma unroll
  for (int v = 0; v < KV; ++v)
#pragma unroll
    for (int e = 0; e < 8; ++e) s += f[v][e];
  const float mean = group_sum<64>(s) * (1.f / (float)K);
  float q = 0.f;
#pragma unroll
  for (int v = 0; v < KV; ++v)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      f[v][e] -= mean;
      q = fmaf(f[v][e], f[v][e], q);
    }
  const float rstd = rsqrtf(group_sum<64>(q) * (1.f / (float)K) + eps);
#pragma unroll
  for (int v = 0; v < KV; ++v) {
    float w[8], b[8];
    Tr<ST>::unpack(wv[v], w);
    Tr<ST>::unpack(bv[v], b);
#pragma unroll
    for (int e = 0; e < 8; ++e) f[v][e] = epi_act<kEpiSilu>(fmaf(f[v][e] * rstd, w[e], b[e]));
    st16(out + row * out_s + (lane + 64 * v) * 8, Tr<ST>::pack(f[v]));
  }
}

namespace {

// the split of the XCDs over rows (see xcd_tile)
int xcd_split(int mtiles, int ntiles, int bm, int bn) {
  int best = 0;
  int64_t cost = 0;
  for (int xm = 1; xm <= 8; xm *= 2) {
    if (mtiles % xm != 0 || ntiles % (8 / xm) != 0) continue;
    const int64_t c = (int64_t)(mtiles / xm) * bm + (int64_t)(ntiles / (8 / xm)) * bn;
    if (best == 0 || c < cost) {
      best = xm;
      cost = c;
    }
  }
  return best;
}

template <typename ST>
dim3 tile_grid(LinK<ST>& k, int bm, int bn) {
  k.per = k.T > 0 ? bm / k.T : 0;
  k.rpt = k.T > 0 ? k.per * k.T : bm;
  k.mtiles = (k.M + k.rpt - 1) / k.rpt;
  const int nt = k.N / bn;
  k.xm = xcd_split(k.mtiles, nt, bm, bn);
  if (k.xm > 0 && k.mtiles / k.xm <= 65535 && nt / (8 / k.xm) <= 65535)  // y and z of a grid
    return dim3(8u, (unsigned)(k.mtiles / k.xm), (unsigned)(nt / (8 / k.xm)));
  k.xm = 0;
  return dim3((unsigned)(k.mtiles * nt));
}

template <typename ST, int BM, int BN, int WM, int WN, int WK, int BK, int S, int EPI>
int launch_tile(LinK<ST> k, hipStream_t s) {
  const dim3 grid = tile_grid(k, BM, BN);
  hipLaunchKernelGGL((lin_tile_kernel<ST, BM, BN, WM, WN, WK, BK, S, EPI>), grid, dim3(64 * WM * WN * WK), 0, s, k);
  return check_launch("pk_linear");
}

// The forms without a prologue and what a launch of each takes, fitted to launches
// in a graph with cold weights (K 512 - 4096, 16 - 3584 rows, bf16): `a` us plus `s`
// us a 1024 columns for workgroups that are alone on their CU, `m` of the latter
// for each further one resident with it (`occ` fit), and again a - 2 for each
// further round.  Small tiles read more bytes an output but put more CUs on a
// short launch, and few long stages (up to 512 columns) wait for fewer barriers;
// the large ones reuse a byte more often (the 64 x 64 form reads 12.9 TB/s from L2 at
// 840 x 4096 -> 1024, the 128 x 128 form 7.3 at 840 x 1024 -> 4096).  The cheapest by this model is launched; at the measured shapes it
// is the fastest form or within 6% of it.
struct Form {
  int bm, bn, kmul, occ;
  float a, s, m;
};
constexpr Form kForms[] = {
    {16, 16, 128, 4, 2.8f, 1.2f, 0.25f},   // 0
    {16, 16, 512, 1, 3.0f, 0.7f, 0.f},     // 1
    {16, 16, 256, 2, 2.95f, 0.85f, 0.5f},  // 2
    {16, 32, 128, 3, 3.05f, 1.37f, 0.5f},  // 3
    {16, 32, 512, 1, 3.5f, 0.88f, 0.f},    // 4
    {32, 32, 128, 1, 3.05f, 1.95f, 0.f},   // 5
    {32, 32, 128, 2, 3.45f, 1.75f, 0.6f},  // 6
    {32, 32, 256, 1, 3.75f, 1.5f, 0.f},    // 7
    {32, 64, 128, 2, 3.6f, 2.25f, 0.95f},  // 8
    {32, 64, 256, 1, 4.05f, 2.0f, 0.f},    // 9
    {64, 64, 64, 2, 3.75f, 3.35f, 0.8f},   // 10
    {64, 128, 64, 2, 4.2f, 5.5f, 0.8f},    // 11
    {128, 128, 64, 1, 5.0f, 8.5f, 0.f},    // 12
    {128, 128, 64, 2, 5.7f, 9.1f, 0.8f},   // 13
    {256, 256, 64, 1, 10.0f, 28.0f, 0.f},  // 14
};
constexpr int kNumForms = sizeof(kForms) / sizeof(kForms[0]);

// us of a launch in form f, or a negative number where it does not fit
float form_cost(const Form& f, int64_t M, int64_t N, int64_t K, int cus, int T = 1) {
  if (N % f.bn != 0 || K % f.kmul != 0 || T > f.bm) return -1.f;
  const int rpt = f.bm / T * T;
  const int64_t tiles = (M + rpt - 1) / rpt * (N / f.bn);
  const int64_t per = (tiles + cus - 1) / cus, rounds = (per + f.occ - 1) / f.occ;
  const float c = f.s * (float)K / 1024.f;
  return f.a + (float)(rounds - 1) * (f.a - 2.f) + (float)rounds * c + f.m * c * (float)(per - rounds);
}

int best_form(int64_t M, int64_t N, int64_t K, int cus) {
  int best = -1;
  float cost = 0.f;
  for (int i = 0; i < kNumForms; ++i) {
    const float c = form_cost(kForms[i], M, N, K, cus);
    if (c >= 0.f && (best < 0 || c < cost)) {
      best = i;
      cost = c;
    }
  }
  return best;
}

template <typename ST, int EPI>
int launch_form(const LinK<ST>& k, int form, hipStream_t s) {
  switch (form) {
    case 0: return launch_tile<ST, 16, 16, 1, 1, 4, 128, 4, EPI>(k, s);
    case 1: return launch_tile<ST, 16, 16, 1, 1, 8, 512, 4, EPI>(k, s);
    case 2: return launch_tile<ST, 16, 16, 1, 1, 4, 256, 4, EPI>(k, s);
    case 3: return launch_tile<ST, 16, 32, 1, 1, 4, 128, 4, EPI>(k, s);
    case 4: return launch_tile<ST, 16, 32, 1, 1, 8, 512, 3, EPI>(k, s);
    case 5: return launch_tile<ST, 32, 32, 2, 2, 2, 128, 6, EPI>(k, s);
    case 6: return launch_tile<ST, 32, 32, 1, 1, 4, 128, 4, EPI>(k, s);
    case 7: return launch_tile<ST, 32, 32, 1, 1, 8, 256, 4, EPI>(k, s);
    case 8: return launch_tile<ST, 32, 64, 1, 2, 4, 128, 3, EPI>(k, s);
    case 9: return launch_tile<ST, 32, 64, 1, 2, 4, 256, 3, EPI>(k, s);
    case 10: return launch_tile<ST, 64, 64, 2, 2, 2, 64, 4, EPI>(k, s);
    case 11: return launch_tile<ST, 64, 128, 2, 4, 1, 64, 3, EPI>(k, s);
    case 12: return launch_tile<ST, 128, 128, 2, 4, 1, 64, 4, EPI>(k, s);
    case 13: return launch_tile<ST, 128, 128, 2, 2, 1, 64, 2, EPI>(k, s);
    default: return launch_tile<ST, 256, 256, 2, 4, 1, 64, 2, EPI>(k, s);
  }
}

template <typename ST, int KV, int BN, int WN, int WK, int BK, int S, int PRO, int EPI>
int launch_norm(LinK<ST> k, hipStream_t s) {
  const dim3 grid = tile_grid(k, 16, BN);
  hipLaunchKernelGGL((lin_norm_kernel<ST, KV, 16, BN, WN, WK, BK, S, PRO, EPI>), grid, dim3(64 * WN * WK), 0, s, k);
  return check_launch("pk_linear");
}

// Outputs a workgroup of the norm form: the fewest that give no CU a second
// tile (each tile normalises its rows again), 0 if none does.  In a graph, residual
// update + norm + 512 -> 2048 with SiLU against pk_residual_norm and pk_linear: 16
// rows (16 outputs) 4.1 us against 6.1, 64 rows (32) 4.5 against 6.7, 128 rows (64)
// 5.1 against 7.0, 256 rows (128) 5.9 against 7.8; 1024 -> 4096: 16 rows (16) 6.2
// against 7.8, 64 rows (64) 7.3 against 8.6, 120 rows (128) 8.4 against 9.7, 256
// rows 12.7 against 11.2.  T: frames a stream of the convolution's tiles, 0 for none.
int norm_form(int64_t M, int64_t N, int64_t K, int cus, int T) {
  if ((K != 512 && K != 1024) || T > 16) return 0;
  const int rpt = T > 0 ? 16 / T * T : 16;
  for (int bn = T > 0 ? 32 : 16; bn <= 128; bn *= 2)
    if (N % bn == 0 && (M + rpt - 1) / rpt * (N / bn) <= cus) return bn;
  return 0;
}

template <typename ST, int KV, int PRO, int EPI>
int launch_norm_form(const LinK<ST>& k, int bn, hipStream_t s) {
  if constexpr (EPI != kEpiConv) {
    if (bn == 16) return launch_norm<ST, KV, 16, 1, 8, 512, 2, PRO, EPI>(k, s);
  }
  if (bn == 32) return launch_norm<ST, KV, 32, 1, 8, 512, 2, PRO, EPI>(k, s);
  if (bn == 64) return launch_norm<ST, KV, 64, 2, 4, 128, 3, PRO, EPI>(k, s);
  return launch_norm<ST, KV, 128, 4, 2, 128, 3, PRO, EPI>(k, s);
}

template <typename ST, int PRO, int EPI>
int launch_norm_k(const LinK<ST>& k, int bn, hipStream_t s) {
  if (k.K == 512) return launch_norm_form<ST, 1, PRO, EPI>(k, bn, s);
  return launch_norm_form<ST, 2, PRO, EPI>(k, bn, s);
}

// kEpiConv without a prologue: the tile forms whose waves hold values and gates
template <typename ST>
int launch_conv_form(const LinK<ST>& k, int cus, hipStream_t s) {
  constexpr int forms[] = {8, 10, 11, 13};
  int best = -1;
  float cost = 0.f;
  for (int f : forms) {
    const float c = form_cost(kForms[f], k.M, k.N, k.K, cus, k.T);
    if (c >= 0.f && (best < 0 || c < cost)) {
      best = f;
      cost = c;
    }
  }
  switch (best) {
    case 8: return launch_tile<ST, 32, 64, 1, 2, 4, 128, 3, kEpiConv>(k, s);
    case 10: return launch_tile<ST, 64, 64, 2, 2, 2, 64, 4, kEpiConv>(k, s);
    case 11: return launch_tile<ST, 64, 128, 2, 4, 1, 64, 3, kEpiConv>(k, s);
    case 13: return launch_tile<ST, 128, 128, 2, 2, 1, 64, 2, kEpiConv>(k, s);
    default: return fail(PK_ERR_UNSUPPORTED, "pk_linear: no form for %d -> %d with the convolution", k.K, k.N);
  }
}

bool row_ok(int64_t rows, int64_t stride, int64_t width) {
  return stride >= 0 && stride % 8 == 0 && (rows <= 1 || stride >= width) &&
         (rows - 1) * stride + width < (int64_t{1} << 31);
}

template <typename ST>
int linear_typed(const pk_linear_args* a, hipStream_t s) {
  const char* what = "pk_linear";
  if (a->rows < 0) return fail(PK_ERR_INVALID, "%s: rows %d < 0", what, a->rows);
  if (a->n <= 0 || a->n % 64 != 0 || a->k <= 0 || a->k % 256 != 0)
    return fail(PK_ERR_UNSUPPORTED, "%s: n %d must be a multiple of 64 and k %d of 256", what, a->n, a->k);
  if (a->activation < PK_ACT_NONE || a->activation > PK_ACT_GLU_CONV)
    return fail(PK_ERR_INVALID, "%s: unknown activation %d", what, a->activation);
  const bool glu = a->activation == PK_ACT_GLU_CONV;
  const pk_conv_args* cv = a->conv;
  if (glu) {
    if (!cv) return fail(PK_ERR_INVALID, "%s: PK_ACT_GLU_CONV needs conv", what);
    if (cv->kernel != kTaps || cv->chunk < 1 || cv->chunk > 16)
      return fail(PK_ERR_UNSUPPORTED, "%s: convolution of %d taps over %d frames (built: %d taps, up to 16 frames)", what,
                  cv->kernel, cv->chunk, kTaps);
    if (a->n != 2 * (int64_t)cv->d_model || cv->batch < 0 || a->rows != (int64_t)cv->batch * cv->chunk)
      return fail(PK_ERR_INVALID, "%s: rows %d x n %d are not conv's %d streams x %d frames x 2 x %d", what, a->rows, a->n,
                  cv->batch, cv->chunk, cv->d_model);
    if (cv->num_slots <= 0 || cv->num_layers <= 0 || cv->layer < 0 || cv->layer >= cv->num_layers ||
        (!cv->slots && cv->batch > cv->num_slots))
      return fail(PK_ERR_INVALID, "%s: layer %d / layers %d / slots %d / batch %d out of range", what, cv->layer,
                  cv->num_layers, cv->num_slots, cv->batch);
  }
  if (a->rows == 0) return PK_OK;
  const void* ptrs[4] = {a->x, a->weight, a->out, a->bias ? a->bias : a->weight};
  for (const void* q : ptrs) {
    if (!q) return fail(PK_ERR_INVALID, "%s: a tensor pointer is NULL", what);
    if (!aligned16(q)) return fail(PK_ERR_INVALID, "%s: tensors must be 16-byte aligned", what);
  }
  if (glu) {
    const void* need[3] = {cv->cache, cv->dw_weight, cv->dw_bias ? cv->dw_bias : cv->dw_weight};
    for (const void* q : need) {
      if (!q) return fail(PK_ERR_INVALID, "%s: a tensor pointer is NULL", what);
      if (!aligned16(q)) return fail(PK_ERR_INVALID, "%s: tensors must be 16-byte aligned", what);
    }
  }
  if (!row_ok(a->rows, a->x_stride, a->k) || !row_ok(a->n, a->weight_stride, a->k) ||
      !row_ok(a->rows, a->out_stride, glu ? a->n / 2 : a->n))
    return fail(PK_ERR_INVALID, "%s: row strides must be multiples of 8 elements, at least the row, and a tensor below "
                "2^31 elements", what);
  LinK<ST> k{};
  k.x = static_cast<const ST*>(a->x);
  k.x_s = a->x_stride;
  k.w = static_cast<const ST*>(a->weight);
  k.w_s = a->weight_stride;
  k.bias = static_cast<const ST*>(a->bias);
  k.out = static_cast<ST*>(a->out);
  k.out_s = a->out_stride;
  k.M = a->rows;
  k.N = a->n;
  k.K = a->k;
  if (glu) {
    k.y = static_cast<float*>(a->out);
    k.y_s = a->out_stride;
    k.cache = static_cast<ST*>(cv->cache);
    k.slots = cv->slots;
    k.pad = cv->pad_mask;
    k.lengths = cv->lengths;
    k.len_scalar = cv->length_scalar;
    k.dw = static_cast<const ST*>(cv->dw_weight);
    k.dwb = static_cast<const ST*>(cv->dw_bias);
    k.num_slots = cv->num_slots;
    k.num_layers = cv->num_layers;
    k.layer = cv->layer;
    k.T = cv->chunk;
    k.batch = cv->batch;
  }
  if (a->prologue != PK_PRO_NONE) {
    if (a->prologue < PK_PRO_NONE || a->prologue > PK_PRO_NORM_SILU)
      return fail(PK_ERR_INVALID, "%s: unknown prologue %d", what, a->prologue);
    const bool res = a->prologue == PK_PRO_RESIDUAL_NORM || a->prologue == PK_PRO_RESIDUAL_NORM2, two = a->prologue == PK_PRO_RESIDUAL_NORM2;
    const void* need[7] = {a->ln_weight, a->ln_bias, a->x, res ? a->branch : a->x, res ? a->residual_out : a->x,
                           two ? a->ln0_weight : a->x, two ? a->ln0_bias : a->x};
    for (const void* q : need) {
      if (!q) return fail(PK_ERR_INVALID, "%s: a tensor pointer is NULL", what);
      if (!aligned16(q)) return fail(PK_ERR_INVALID, "%s: tensors must be 16-byte aligned", what);
    }
    if (res && (!row_ok(a->rows, a->branch_stride, a->k) || !row_ok(a->rows, a->residual_out_stride, a->k)))
      return fail(PK_ERR_INVALID, "%s: row strides must be multiples of 8 elements, at least the row", what);
    // every workgroup of a row tile reads x and branch while one writes the residual
    if (res && (a->residual_out == a->x || a->residual_out == a->branch))
      return fail(PK_ERR_INVALID, "%s: residual_out must not be x or branch", what);
    if (!(a->ln_eps >= 0.f) || !(a->ln0_eps >= 0.f) || !(a->alpha - a->alpha == 0.f))
      return fail(PK_ERR_INVALID, "%s: eps must be >= 0 and alpha finite", what);
    k.br = static_cast<const ST*>(a->branch);
    k.br_s = a->branch_stride;
    k.lnw = static_cast<const ST*>(a->ln_weight);
    k.lnb = static_cast<const ST*>(a->ln_bias);
    k.lnw0 = static_cast<const ST*>(a->ln0_weight);
    k.lnb0 = static_cast<const ST*>(a->ln0_bias);
    k.rout = static_cast<ST*>(a->residual_out);
    k.rout_s = a->residual_out_stride;
    k.alpha = a->alpha;
    k.eps = a->ln_eps;
    k.eps0 = a->ln0_eps;
  }
  DeviceGuard dg(a->device);
  if (!dg.ok) return fail(PK_ERR_HIP, "%s: cannot select device %d", what, a->device);
  const int cus = cu_count();
  if (a->prologue != PK_PRO_NONE) {
    const int bn = norm_form(k.M, k.N, k.K, cus, k.T);
    const bool silu = a->activation == PK_ACT_SILU, none = a->activation == PK_ACT_NONE;
    if (a->prologue == PK_PRO_NORM_SILU) {
      if (!none || (k.K != 512 && k.K != 1024)) return fail(PK_ERR_UNSUPPORTED, "%s: PK_PRO_NORM_SILU is built for k 512 and 1024 without activation", what);
      k.xf = static_cast<const float*>(a->x);
      if (bn) return launch_norm_k<ST, kProNormSilu, kEpiNone>(k, bn, s);
      if (!a->residual_out || !aligned16(a->residual_out) || !row_ok(k.M, a->residual_out_stride, k.K))
        return fail(PK_ERR_INVALID, "%s: PK_PRO_NORM_SILU on this many rows needs residual_out", what);
      ST* const h = static_cast<ST*>(a->residual_out);
      const dim3 grid((unsigned)((k.M + 3) / 4));
      if (k.K == 512)
        hipLaunchKernelGGL((norm_silu_kernel<ST, 1>), grid, dim3(256), 0, s, k.xf, k.x_s, k.lnw, k.lnb, k.eps, h, a->residual_out_stride, k.M);
      else
        hipLaunchKernelGGL((norm_silu_kernel<ST, 2>), grid, dim3(256), 0, s, k.xf, k.x_s, k.lnw, k.lnb, k.eps, h, a->residual_out_stride, k.M);
      const int rc = check_launch(what);
      if (rc != PK_OK) return rc;
      k.x = h;
      k.x_s = a->residual_out_stride;
      return launch_form<ST, kEpiNone>(k, best_form(k.M, k.N, k.K, cus), s);
    }
    if (!bn) return fail(PK_ERR_UNSUPPORTED, "%s: %d rows of %d -> %d are past the norm form (pk_linear_takes_norm)", what, k.M, k.K, k.N);
    switch (a->prologue) {
      case PK_PRO_NORM:
        if (!silu) return fail(PK_ERR_UNSUPPORTED, "%s: PK_PRO_NORM is built with SiLU", what);
        return launch_norm_k<ST, kProNorm, kEpiSilu>(k, bn, s);
      case PK_PRO_RESIDUAL_NORM:
        if (glu) return launch_norm_k<ST, kProResNorm, kEpiConv>(k, bn, s);
        return silu ? launch_norm_k<ST, kProResNorm, kEpiSilu>(k, bn, s) : launch_norm_k<ST, kProResNorm, kEpiNone>(k, bn, s);
      default:
        if (!silu) return fail(PK_ERR_UNSUPPORTED, "%s: PK_PRO_RESIDUAL_NORM2 is built with SiLU", what);
        return launch_norm_k<ST, kProResNorm2, kEpiSilu>(k, bn, s);
    }
  }
  if (glu) return launch_conv_form(k, cus, s);
  const int form = best_form(k.M, k.N, k.K, cus);
  if (a->activation == PK_ACT_SILU) return launch_form<ST, kEpiSilu>(k, form, s);
  return launch_form<ST, kEpiNone>(k, form, s);
}

int linear_any(const pk_linear_args* a, hipStream_t s) {
  switch (a->dtype) {
    case PK_DTYPE_F16: return linear_typed<_Float16>(a, s);
    case PK_DTYPE_BF16: return linear_typed<bf16_t>(a, s);
    case PK_DTYPE_F32: return fail(PK_ERR_UNSUPPORTED, "pk_linear: fp16 and bf16 only");
    default: return fail(PK_ERR_INVALID, "pk_linear: unknown dtype %d", a->dtype);
  }
}

}  // namespace
}  // namespace pk

extern "C" int pk_linear_takes_norm(int32_t rows, int32_t n, int32_t k, int32_t chunk) {
  return rows > 0 && n > 0 && chunk >= 0 && pk::norm_form(rows, n, k, pk::cu_count(), chunk) > 0 ? 1 : 0;
}

extern "C" int pk_linear(const pk_linear_args* args, int32_t count, void* stream) {
  pk::clear_error();
  if (!args) return pk::fail(PK_ERR_INVALID, "pk_linear: args is NULL");
  if (count < 0) return pk::fail(PK_ERR_INVALID, "pk_linear: count %d < 0", count);
  for (int32_t i = 0; i < count; ++i) {
    const int rc = pk::linear_any(args + i, static_cast<hipStream_t>(stream));
    if (rc != PK_OK) return rc;
  }
  return PK_OK;
}
