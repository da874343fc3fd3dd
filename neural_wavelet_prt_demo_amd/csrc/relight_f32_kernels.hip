// Plain FP32 form of the per-(pixel, wavelet) network for gfx950: FP32
// operands, products and accumulation on the FP32 matrix instructions (same
// reference path as relight_kernels.hip: Renderer/tinycudann/tcnn.cu:111-152,
// utils_kernels.h:51-115).
//
// Layout (v_mfma_f32_16x16x4_f32; lane l, g = l / 16, n = l % 16): A holds
// row n, contraction slot g; B column n, slot g; D rows 4g .. 4g + 3 of column
// n.  Weights are A (rows = output features), pixels the columns.  A layer's
// D block b, element i, is feature 16 b + 4 g + i of pixel n: exactly the B
// operand of the contraction step (b, i) whose slot g carries that feature.
// So the ReLU's result is the next layer's operand as it stands, and the A
// operand of steps (b, 0..3) is W[row][16 b + 4 g .. + 3], one 16-byte LDS
// read for four steps.
//
// The output layer (3 rows) would waste 13 of 16 rows there.  It runs on
// v_mfma_f32_4x4x1_16b_f32 instead: 16 blocks of 4 lanes, each block's 4
// columns four pixels at one g and its 4 rows the three channels and a zero
// row.  Each lane ends with its own g's share of its pixel's outputs, and two
// cross-lane adds complete them.
//
// What bounds it: the FP32 matrix rate (64 FLOP per cycle and SIMD, 157 TFLOP/s
// nominal; a large FP32 matrix product measures 152).  The weights stay in
// LDS (40 KB, shared by four waves; 40 16-byte reads per wavelet against 5 K
// matrix cycles per 16 pixels; the output layer's stay in 16 registers), so
// the other registers hold activations.  960 x 540, K = 64 (33 M pairs, 692
// GFLOP): 5.30 ms, 131 TFLOP/s, the matrix cores busy for 85 % of the cycles;
// with one lane per pixel on the vector ALU and one LDS read per four products
// it was 21.0 ms.
#include <hip/hip_runtime.h>

#include "device_common.hpp"
#include "kernels.hpp"
#include "relight_device.hpp"

namespace nwprt {
namespace {

using dev::f32x4;

constexpr int kBlock = 256;  // 4 waves
constexpr int kW1 = 64 * 32, kW2 = 64 * 64, kW3 = 64 * 64;
// LDS weights as 16-byte A operands [tile][lane]: W1 tiles (row block rb,
// input block b) rb * 2 + b, then W2 and W3 tiles rb * 4 + b.
constexpr int kTiles1 = 8, kTiles2 = 16, kTiles = kTiles1 + 2 * kTiles2;

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ f32x4 relu4(f32x4 v) {
  return f32x4{fmaxf(v[0], 0.f), fmaxf(v[1], 0.f), fmaxf(v[2], 0.f), fmaxf(v[3], 0.f)};
}

// One 64-output layer of the wave's NG pixel groups: NB input blocks of 16
// features, weights at `w` (A operands [4 row blocks][NB][64 lanes]).
template <int NG, int NB>
__device__ __forceinline__ void layer(const f32x4 *w, int lane, const f32x4 (&x)[NG][NB],
                                      f32x4 (&y)[NG][4]) {
#pragma unroll
  for (int rb = 0; rb < 4; ++rb) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const f32x4 a = w[(rb * NB + b) * 64 + lane];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < NG; ++j) y[j][rb] = mfma4(a[i], x[j][b][i], y[j][rb]);
    }
#pragma unroll
    for (int j = 0; j < NG; ++j) y[j][rb] = relu4(y[j][rb]);
  }
}

// Grid: one wave per 16 NG pixels (KS = 1).  After the output layer lane
// (g, n) holds pixel base + 16 (g % NG) + n; lanes g < NG write.
// KS = 4: the workgroup's four waves share 16 NG pixels, wave w taking
// wavelets 4 r + w of round r.  Each round's outputs meet in LDS (two buffers,
// one barrier a round) and every wave adds the round's terms in wavelet order,
// so the sum is the one KS = 1 forms, bit for bit.
template <int NG, int KS, bool DUMP, bool AUX>
__global__ __launch_bounds__(kBlock) void relight_f32_kernel(RelightArgs a) {
  __shared__ f32x4 wl[kTiles * 64];
  __shared__ float ts[KS > 1 ? 2 * KS * 3 * 16 * NG : 1];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int g = lane >> 4, n = lane & 15;
  for (int t = wave; t < kTiles; t += kBlock / 64) {
    const int u = t - kTiles1;
    const float *src;
    if (t < kTiles1)
      src = a.w_f32 + (16 * (t >> 1) + n) * 32 + 16 * (t & 1);
    else
      src = a.w_f32 + kW1 + (u >> 4) * kW2 + (16 * ((u & 15) >> 2) + n) * 64 + 16 * (u & 3);
    wl[t * 64 + lane] = *(const f32x4 *)(src + 4 * g);
  }
  __syncthreads();
  const int base = KS > 1 ? (int)blockIdx.x * 16 * NG
                          : (int)(blockIdx.x * (kBlock / 64) + wave) * 16 * NG;
  const int P = a.n_pixels;
  if (base >= P) return;  // KS > 1: the whole workgroup, whose waves share `base`
  const int my_px = base + 16 * (g % NG) + n;
  const bool mine = my_px < P;
  const bool hit = mine && (a.env_flag == nullptr || a.env_flag[my_px] != 0);
  float sum[3] = {0.f, 0.f, 0.f}, comp[3] = {0.f, 0.f, 0.f}, pend[3] = {0.f, 0.f, 0.f};
  if (__ballot(hit) != 0) {
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    f32x4 h[NG][2], b2[NG][4];
#pragma unroll
    for (int j = 0; j < NG; ++j) {
      const int p = base + 16 * j + n;
#pragma unroll
      for (int b = 0; b < 2; ++b)
        h[j][b] = p < P ? *(const f32x4 *)((const float *)a.features + (size_t)p * 32 + 16 * b + 4 * g)
                        : zero;
#pragma unroll
      for (int rb = 0; rb < 4; ++rb) b2[j][rb] = zero;
      // Aux inputs enter the second layer as a per-pixel constant term: the
      // accumulators start from Waux aux instead of zero.
      if (AUX) {
        const f32x4 ax = p < P ? *(const f32x4 *)((const float *)a.aux + (size_t)p * 16 + 4 * g) : zero;
#pragma unroll
        for (int rb = 0; rb < 4; ++rb) {
          const f32x4 wa = *(const f32x4 *)(a.waux_f32 + (16 * rb + n) * 16 + 4 * g);
#pragma unroll
          for (int i = 0; i < 4; ++i) b2[j][rb] = mfma4(wa[i], ax[i], b2[j][rb]);
        }
      }
    }
    // Output layer A operands: lane's row is l % 4 (row 3 zero), its slot the
    // lane's own g: W4[row][16 b + 4 g + i].
    f32x4 w4[4];
#pragma unroll
    for (int b = 0; b < 4; ++b)
      w4[b] = (n & 3) < 3
                  ? *(const f32x4 *)(a.w_f32 + kW1 + kW2 + kW3 + (n & 3) * 64 + 16 * b + 4 * g)
                  : zero;
    // Light terms in wavelet order: the clamped terms of k and k + 1 are added
    // and the pair sum enters the compensated running sum (the fused kernel's
    // order).
    auto add_term = [&](int k, int ch, float t) {
      const float term = dev::relu_f32(dev::load_invariant(a.light + 3 * k + ch) * t);
      if (k & 1) dev::neumaier_add(sum[ch], comp[ch], pend[ch] + term);
      else pend[ch] = term;
    };
    const int my_k = KS > 1 ? wave : 0;
    for (int k0 = 0; k0 < a.k; k0 += KS) {
      const int k = k0 + my_k;
      float tr[3] = {0.f, 0.f, 0.f};
      if (k < a.k) {
        // The weight reads are loop-invariant; an opaque zero offset keeps the
        // compiler from hoisting all of them out of the K loop.
        int wo = 0;
        asm volatile("" : "+s"(wo));
        const f32x4 *w = wl + wo;
        f32x4 z[NG][2];
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          const f32x4 ws = *(const f32x4 *)(a.wsel + (size_t)k * 32 + 16 * b + 4 * g);
#pragma unroll
          for (int j = 0; j < NG; ++j) z[j][b] = h[j][b] * ws;
        }
        f32x4 x[NG][4], y[NG][4];
#pragma unroll
        for (int j = 0; j < NG; ++j)
#pragma unroll
          for (int rb = 0; rb < 4; ++rb) x[j][rb] = zero;
        layer<NG, 2>(w, lane, z, x);
#pragma unroll
        for (int j = 0; j < NG; ++j)
#pragma unroll
          for (int rb = 0; rb < 4; ++rb) y[j][rb] = b2[j][rb];
        layer<NG, 4>(w + kTiles1 * 64, lane, x, y);
#pragma unroll
        for (int j = 0; j < NG; ++j)
#pragma unroll
          for (int rb = 0; rb < 4; ++rb) x[j][rb] = zero;
        layer<NG, 4>(w + (kTiles1 + kTiles2) * 64, lane, y, x);
        f32x4 o[NG];
#pragma unroll
        for (int j = 0; j < NG; ++j) o[j] = zero;
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < NG; ++j)
              o[j] = __builtin_amdgcn_mfma_f32_4x4x1f32(w4[b][i], x[j][b][i], o[j], 0, 0, 0);
#pragma unroll
        for (int ch = 0; ch < 3; ++ch) {
          // Each group's four g shares meet in two butterfly adds; the lane
          // keeps its own group's (the other groups' sums are discarded).
          float acc = 0.f;
#pragma unroll
          for (int j = 0; j < NG; ++j) {
            float v = o[j][ch];
            v += __shfl_xor(v, 16);
            v += __shfl_xor(v, 32);
            acc = g % NG == j ? v : acc;
          }
          tr[ch] = a.softplus ? dev::softplus(acc) : acc;
          if (DUMP) {
            const int q = my_px - a.dump_begin;
            if (hit && g < NG && q >= 0 && q < a.dump_count)  // background rows stay
              a.dump[((size_t)q * a.k + k) * 3 + ch] = tr[ch];
          }
        }
      }
      if constexpr (KS == 1) {
#pragma unroll
        for (int ch = 0; ch < 3; ++ch) add_term(k, ch, tr[ch]);
      } else {
        float *buf = ts + (k0 / KS & 1) * KS * 3 * 16 * NG;
        const int col = 16 * (g % NG) + n;
        if (g < NG)
#pragma unroll
          for (int ch = 0; ch < 3; ++ch) buf[(wave * 3 + ch) * 16 * NG + col] = tr[ch];
        __syncthreads();
#pragma unroll
        for (int q = 0; q < KS; ++q)
          if (k0 + q < a.k)
#pragma unroll
            for (int ch = 0; ch < 3; ++ch)
              add_term(k0 + q, ch, buf[(q * 3 + ch) * 16 * NG + col]);
      }
    }
    if (a.k & 1)
      for (int ch = 0; ch < 3; ++ch) dev::neumaier_add(sum[ch], comp[ch], pend[ch]);
  }
  if (mine && g < NG && (KS == 1 || wave == 0))
    dev::write_outputs(a, my_px, hit ? sum[0] + comp[0] : 0.f, hit ? sum[1] + comp[1] : 0.f,
                       hit ? sum[2] + comp[2] : 0.f);
}

template <int NG, int KS>
void launch_shape(const RelightArgs &a, hipStream_t s) {
  constexpr int per = kBlock / 64 / KS * 16 * NG;
  const dim3 grid((a.n_pixels + per - 1) / per), block(kBlock);
  if (a.aux) {
    if (a.dump) hipLaunchKernelGGL((relight_f32_kernel<NG, KS, true, true>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((relight_f32_kernel<NG, KS, false, true>), grid, block, 0, s, a);
  } else {
    if (a.dump) hipLaunchKernelGGL((relight_f32_kernel<NG, KS, true, false>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((relight_f32_kernel<NG, KS, false, false>), grid, block, 0, s, a);
  }
}

}  // namespace

void launch_relight_plain(const RelightArgs &a, hipStream_t s) {
  require(a.n_pixels >= 1 && a.k >= 1 && a.k <= NWPRT_MAX_K, NWPRT_ERR_INVALID_ARGUMENT,
          "relight: bad pixel count or K");
  require(a.features && a.wsel && a.light && a.w_f32 && a.direct && (!a.aux || a.waux_f32),
          NWPRT_ERR_INVALID_ARGUMENT, "relight: missing operand");
  // Shape by how many 16-pixel groups there are for the chip's 1024 SIMDs
  // (K = 64, the three forms' whole relights at the crossings): up to one a
  // SIMD the workgroup's waves split the wavelets (33 x 19: 126 us against 278
  // with one wave per 16 pixels and 468 per 32; 128 x 128: 281 / 308 / 488;
  // 181 x 181: 473 / 465 / 511); up to four a SIMD one wave takes 16 pixels
  // (256 x 256: 807 / 815 per 32); beyond, 32 pixels a wave halve the LDS
  // reads per pixel (362 x 362: 1503 against 1525; 960 x 540: 5624 / 5735).
  // The forms sum in the same order and give the same bits.
  const int groups = (a.n_pixels + 15) / 16;
  if (groups <= 1024) launch_shape<1, 4>(a, s);
  else if (groups <= 4096) launch_shape<1, 1>(a, s);
  else launch_shape<2, 1>(a, s);
  hip_check(hipGetLastError(), "relight_f32_kernel launch");
}

}  // namespace nwprt
