// Per-(pixel, wavelet) network and per-pixel reduction for gfx950.
//
// Reference path being replaced (Renderer/tinycudann/tcnn.cu:111-152): a host
// loop over image rows runs, per row, the hash grid, the per-pair Hadamard
// product with the wavelet feature (utils_kernels.h:97-115), the out_prd and
// cmp_net networks and a cast, materialising 16 + 3 floats per pair; then
// computeResponse (utils_kernels.h:51-90) sums max(light_i * T_i, 0) over K.
//
// Here one launch does all pairs of a frame and nothing per pair touches
// HBM: each wave owns 64 pixels and walks the K selected wavelets; the four
// linear layers run as chained 16x16x32 MFMAs whose results stay in VGPRs,
// and the clamped sum is carried per lane with Kahan compensation.
//
// The wave-level code (MFMA layout, layers, fused encode, per-wave relight)
// is in relight_mma16_device.hpp.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <type_traits>

#include "device_common.hpp"
#include "hashgrid_device.hpp"
#include "kernels.hpp"
#include "relight_device.hpp"
#include "relight_mma16_device.hpp"

namespace nwprt {
namespace {

using dev::f32x4;
using dev::u32x4;

constexpr int kRelightBlock = 256;  // 4 waves x 64 pixels

using namespace mma16;

// Tile-shape variants of the fused kernel (chosen per shape by the
// autotuner): GP pixel groups carried through the layers together (GP
// independent MFMA chains hide each other's result latency), the output
// layer's A tiles in VGPRs or in LDS (LDS frees 32 VGPRs for a third wave per
// SIMD), and the minimum waves per SIMD the register budget must allow.
struct MfmaVariant {
  int gp;
  bool w4_lds;
  int min_waves;
  const char *name;
};
constexpr MfmaVariant kMfmaVariants[] = {
    {2, false, 2, "gp2.w4reg.occ2"}, {4, false, 2, "gp4.w4reg.occ2"},
    {2, true, 3, "gp2.w4lds.occ3"},  {4, true, 2, "gp4.w4lds.occ2"},
    {1, true, 3, "gp1.w4lds.occ3"},  {0, false, 2, "pipe.w4reg.occ2"},
    {0, true, 2, "pipe.w4lds.occ2"},
};
constexpr int kNumMfmaVariants = sizeof(kMfmaVariants) / sizeof(kMfmaVariants[0]);

// Workgroups that take 256 pixels (64 a wave) before the ones that take 64
// together (relight_group).  The chip holds 512 workgroups of these kernels
// (256 CUs, two waves a SIMD).  Whole rounds of 512 go 64 pixels a wave; the
// rest of the frame, at most one round, is split finer where that is shorter.
// Unsplit it takes one time up to 256 workgroups (one a CU) and another up to
// 512; split, a time that grows with its pixels and, as the four waves load
// the weights and encode for a quarter of the wavelets each, has less to give
// at small K.  Behind whole rounds it gains less, because the waves that finish
// them early overlap with an unsplit rest too.  So each step of the rest has a
// least K, between where the split is the shorter one along a surface (real
// frames) and at scattered positions (every gather a line of its own); there
// it is not above the two-group step without a split by more than 1.5 %.  BF16,
// whole calls in us, unsplit / split (rounds + workgroups of the rest):
//                     scattered   surface                   scattered   surface
//   0 + 128, K =  8    48 /  40   37 / 26   1 + 192, K = 16  129 / 133   92 /  87
//   0 + 192, K = 16    57 /  58   45 / 38   1 + 320, K =  8  149 / 150   92 /  83
//   0 + 256, K = 32    74 /  83   61 / 57   1 + 384, K = 24  182 / 190  142 / 129
//   0 + 320, K =  8    76 /  84   51 / 46   2 +  64, K = 48  303 / 274  255 / 228
//   0 + 384, K = 24   100 / 108   76 / 67   4 + 192, K = 48  534 / 537  452 / 450
//   1 + 128, K = 16   126 / 120   91 / 80   4 + 320, K = 24  414 / 417  335 / 317
//   1 + 256, K = 64   241 / 256  209 / 214  4 + 384, K = 48  586 / 592  496 / 488
// Features read from memory (p1 / p2, aux) leave only the weights' loads to
// share, so those relights take the first lines behind any number of rounds
// (aux: 0 + 128, K = 1 38.3 / 38.8, 4 0.94 of the time unsplit; 0 + 256, K = 24
// 71.0 / 68.5; 3 + 320, K = 8 328 / 329, 64 0.95).
constexpr int kRoundWgs = 512;
int full_workgroups(int n_pixels, int k, bool fused) {
  const int wgs = (n_pixels + kRelightBlock - 1) / kRelightBlock;
  const int rest = wgs % kRoundWgs, rounds = wgs / kRoundWgs;
  const bool behind = fused && rounds >= 2;
  int least_k = INT_MAX;
  if (rest <= 128) least_k = fused ? 1 : 4;
  else if (rest <= 192) least_k = behind ? 40 : 16;
  else if (rest <= 256) least_k = rounds >= 1 ? INT_MAX : fused ? 32 : 16;
  else if (rest <= 320) least_k = behind ? 24 : 8;
  else if (rest <= 384) least_k = behind ? 40 : 24;
  return k >= least_k ? wgs - rest : wgs;
}

// Grid: `full` workgroups of 4 waves x 64 pixels -- wave w of the one with
// tile t = xcd_tile(b) owns pixels [64 (4 t + w), +64), so each XCD relights
// (and with the fused encode, gathers hash entries for) one contiguous band --
// then, in the instances with SPLIT, workgroups whose waves share 64 pixels.
template <typename E, bool SOFTPLUS, bool DUMP, bool AUX, int GP, bool W4LDS, int MINW, bool SPLIT>
__global__ __launch_bounds__(kRelightBlock, MINW) void relight_mfma_kernel(RelightArgs a,
                                                                           int full) {
  __shared__ u32x4 w4s[W4LDS ? 4 * 2 * 64 : 1];
  // Fused encode: [wave][pixel][16]; a sharing workgroup's features and terms.
  __shared__ uint32_t feat_lds[AUX ? (SPLIT ? kGroupLdsWords : 1) : 4 * 64 * 16];
  static_assert(kGroupLdsWords <= 4 * 64 * 16, "a sharing workgroup's LDS fits the waves' rows");
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (SPLIT && (int)blockIdx.x >= full) {
    const int tail = (int)gridDim.x - full;
    const int base = full * kRelightBlock + dev::xcd_tile((int)blockIdx.x - full, tail) * 64;
    if constexpr (AUX) {
      relight_group<E, SOFTPLUS, AUX, !AUX>(a, base, wave, lane, feat_lds);
    } else {
      // The arguments through a pointer of their own: relight_group takes
      // levels by a run-time number, and seen as the same object that makes the
      // compiler read the level parameters of the other workgroups' encode a
      // dword at a time too (BF16, 12 rounds and 64 workgroups, scattered
      // positions, whole calls: K = 32 1179 us, so 1116).
      using Args = const RelightArgs __attribute__((address_space(4)));
      Args *args = (Args *)__builtin_amdgcn_kernarg_segment_ptr();  // `a` is the first argument
      asm volatile("" : "+s"(args));
      relight_group<E, SOFTPLUS, AUX, !AUX>(*(const RelightArgs *)args, base, wave, lane, feat_lds);
    }
    return;
  }
  if (W4LDS) {
    const u32x4 *wt = (const u32x4 *)a.w_tiles;
    for (int i = threadIdx.x; i < 4 * 2 * 64; i += kRelightBlock) w4s[i] = wt[2 * 8 * 64 + i];
    __syncthreads();
  }
  const int base = (dev::xcd_tile(blockIdx.x, full) * 4 + wave) * 64;
  if (base >= a.n_pixels) return;
  relight_wave<E, SOFTPLUS, DUMP, AUX, GP, W4LDS, !AUX>(a, base, lane, w4s,
                                                       feat_lds + (AUX ? 0 : wave * 64 * 16));
}

// Frames of less than a round that are split whole: sharing workgroups only.
template <typename E, bool SOFTPLUS, bool AUX>
__global__ __launch_bounds__(kRelightBlock, 2) void relight_group_kernel(RelightArgs a) {
  __shared__ uint32_t lds[kGroupLdsWords];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  relight_group<E, SOFTPLUS, AUX, !AUX>(a, dev::xcd_tile(blockIdx.x, gridDim.x) * 64, wave, lane,
                                        lds);
}

// Persistent batch form: a machine-sized grid whose waves take work items
// (job, first pixel of a 64-pixel group) from a shared counter until the
// list is exhausted.  Jobs are whole relights with their own frame,
// scene weights, selection and K; items are listed by decreasing K so the
// tail of the launch is short items.  Output-layer tiles stay in VGPRs, so
// there is no workgroup barrier and no scene switch cost beyond reloading;
// jobs with the fused encode use their wave's own 4 KB of LDS.  HAS_AUX
// compiles in the path of jobs with aux inputs (features and aux inputs from
// the standalone encode).
template <typename E, bool SOFTPLUS, bool HAS_AUX, int GP, int MINW>
__global__ __launch_bounds__(kRelightBlock, MINW) void relight_batch_kernel(
    const RelightArgs *__restrict__ jobs, const BatchItem *__restrict__ items,
    const int *__restrict__ n_items_p, unsigned int *__restrict__ counter) {
  __shared__ uint32_t feat_lds[4 * 64 * 16];  // fused encode: [wave][pixel][16]
  const int lane = threadIdx.x & 63;
  uint32_t *my_lds = feat_lds + (threadIdx.x >> 6) * 64 * 16;
  const int n_items = *n_items_p;
  // The next item's index is fetched while the current one runs, so the
  // counter's round trip is off the critical path.
  auto fetch = [&]() {
    int it = 0;
    if (lane == 0) it = (int)atomicAdd(counter, 1u);
    return __builtin_amdgcn_readfirstlane(__shfl(it, 0));
  };
  int next = fetch();
  for (;;) {
    const int it = next;
    if (it >= n_items) break;
    next = fetch();
    const BatchItem item = items[it];
    const RelightArgs a = jobs[item.job];
    // One 64-pixel group per item: a loop over several would let the
    // compiler hoist the group's loads and spill.  Jobs with aux inputs take
    // the tile shape their single relights use (two groups at a time).
    if (HAS_AUX && a.aux)
      relight_wave<E, SOFTPLUS, false, true, 2, false, false>(a, item.base, lane, nullptr, my_lds);
    else
      relight_wave<E, SOFTPLUS, false, false, GP, false, true>(a, item.base, lane, nullptr,
                                                               my_lds);
  }
}

__global__ void reset_counter_kernel(unsigned int *counter) { *counter = 0u; }

constexpr int kW1 = 64 * 32, kW2 = 64 * 64, kW3 = 64 * 64;

// Activation calibration for the FP8 form: the BF16 network over a pixel
// subsample (a.features, a.n_pixels) and the wavelets [k0, k0 + k_chunk) of
// blockIdx.y, recording the maximum pre-activation output of layers 1..3
// (the ReLU outputs share it when positive).  A wave whose maximum of a layer
// is above the one in memory raises it by an atomicMax on the float bits, which
// order like the values for non-negative floats; the maxima start at 0.
// Bound: vector ALU (maxima and packing), 78 % of the cycles against 32 % for
// the matrix cores (16,384 pixels, K = 300: 213 us before the grid was one
// round and the atomics rare, 130 now).
template <bool AUX>
__global__ __launch_bounds__(kRelightBlock) void calib_amax_kernel(RelightArgs a, int k_chunk) {
  using E = __bf16;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int g = lane >> 4, n = lane & 15;
  const int base = (blockIdx.x * 4 + wave) * 64;
  const int k0 = blockIdx.y * k_chunk, k1 = min(a.k, k0 + k_chunk);
  const int P = a.n_pixels;
  if (base >= P || k0 >= k1) return;
  u32x4 hb[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int p = base + 16 * j + n;
    hb[j] = p < P ? dev::load_features8(a, P, p, 8 * g) : u32x4{0u, 0u, 0u, 0u};
  }
  u32x2 auxb[4], waux[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int p = base + 16 * j + n;
    auxb[j] = AUX && p < P ? *(const u32x2 *)((const uint16_t *)a.aux + (size_t)p * 16 + 4 * g)
                           : u32x2{0u, 0u};
    waux[j] = AUX ? ((const u32x2 *)a.waux_tiles)[j * 64 + lane] : u32x2{0u, 0u};
  }
  const u32x4 *wt = (const u32x4 *)a.w_tiles;
  u32x4 w2[4][2], w3[4][2];
#pragma unroll
  for (int b = 0; b < 4; ++b)
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      w2[b][kb] = wt[(0 * 8 + b * 2 + kb) * 64 + lane];
      w3[b][kb] = wt[(1 * 8 + b * 2 + kb) * 64 + lane];
    }
  const u32x4 *mk = (const u32x4 *)a.mk;
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  u32x4 next[4];
#pragma unroll
  for (int b = 0; b < 4; ++b) next[b] = mk[((size_t)k0 * 4 + b) * 64 + lane];
  float m[3] = {0.f, 0.f, 0.f};
  auto upd = [](float &mm, f32x4 c) { mm = fmaxf(mm, fmaxf(fmaxf(c[0], c[1]), fmaxf(c[2], c[3]))); };
  for (int k = k0; k < k1; ++k) {
    u32x4 a1[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) a1[b] = next[b];
    if (k + 1 < k1) {
#pragma unroll
      for (int b = 0; b < 4; ++b) next[b] = mk[((size_t)(k + 1) * 4 + b) * 64 + lane];
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      f32x4 c[4];
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        c[b] = Mfma<E>::run(a1[b], hb[j], zero);
        upd(m[0], c[b]);
      }
      u32x4 x0 = relu_pack<E>(c[0], c[1]), x1 = relu_pack<E>(c[2], c[3]);
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        c[b] = Mfma<E>::run(w2[b][1], x1, Mfma<E>::run(w2[b][0], x0, zero));
        if (AUX) c[b] = Mfma16<E>::run(waux[b], auxb[j], c[b]);
        upd(m[1], c[b]);
      }
      x0 = relu_pack<E>(c[0], c[1]);
      x1 = relu_pack<E>(c[2], c[3]);
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        c[b] = Mfma<E>::run(w3[b][1], x1, Mfma<E>::run(w3[b][0], x0, zero));
        upd(m[2], c[b]);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    float v = m[i];
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v = fmaxf(v, __shfl_xor(v, off));
    // The maxima only grow: a wave whose own is not above the one it reads
    // has nothing to add (thousands of atomics on three words took most of
    // this kernel's time).
    unsigned int *at = (unsigned int *)a.amax + i;
    if (lane == 0 && __float_as_uint(v) > __hip_atomic_load(at, __ATOMIC_RELAXED,
                                                            __HIP_MEMORY_SCOPE_AGENT))
      atomicMax(at, __float_as_uint(v));
  }
}

// Calibration subsample: calibration pixel q is frame pixel q * stride, its
// features copied in the frame's layout (zeros for a background pixel, as
// the encode pass writes them) and, with aux inputs, its 16 aux values
// (zeros for a background pixel, whose activations the relight discards);
// block 0 also clears the four maxima.  Row layout: thread i copies 16 B
// part i % 4 of pixel i / 4 (and 8 B part i % 4 of its aux row); planar:
// 8 B of plane i % 8 of pixel i / 8.
__global__ __launch_bounds__(256) void calib_gather_kernel(const uint16_t *__restrict__ feat,
                                                           const uint16_t *__restrict__ aux,
                                                           const uint8_t *__restrict__ flag,
                                                           int n_pixels, int stride,
                                                           uint16_t *__restrict__ calib,
                                                           uint16_t *__restrict__ calib_aux,
                                                           int n_cal, float *__restrict__ amax,
                                                           int planar) {
  if (blockIdx.x == 0 && threadIdx.x < 4) amax[threadIdx.x] = 0.f;
  const int i = blockIdx.x * 256 + threadIdx.x;
  const int shift = planar ? 3 : 2;
  const int q = i >> shift, part = i & ((1 << shift) - 1);
  if (q >= n_cal) return;
  const long long p = (long long)q * stride;
  const bool hit = p < n_pixels && (flag == nullptr || flag[p] != 0);
  if (planar) {
    const uint2 *src = (const uint2 *)feat;
    ((uint2 *)calib)[(size_t)part * n_cal + q] =
        hit ? src[(size_t)part * n_pixels + p] : make_uint2(0u, 0u);
  } else {
    const u32x4 v = hit ? *(const u32x4 *)(feat + p * 32 + 8 * part) : u32x4{0u, 0u, 0u, 0u};
    *(u32x4 *)(calib + (size_t)q * 32 + 8 * part) = v;
    if (aux)
      *(uint2 *)(calib_aux + (size_t)q * 16 + 4 * part) =
          hit ? *(const uint2 *)(aux + p * 16 + 4 * part) : make_uint2(0u, 0u);
  }
}

// The calibration subsample encoded from positions: thread q of plane r =
// blockIdx.y computes levels r and 15 - r of frame pixel q * stride with the standalone planar encode's
// arithmetic (plane r = levels r and 15 - r, each accumulated from zero) and
// writes the planar layout [8][n_cal][4] in BF16; background pixels get
// zeros.  Block 0 clears the four maxima.
template <bool HF16>
__global__ __launch_bounds__(256) void calib_encode_kernel(RelightArgs a, int stride,
                                                           uint16_t *__restrict__ calib,
                                                           int n_cal, float *__restrict__ amax) {
  if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x < 4) amax[threadIdx.x] = 0.f;
  const int q = blockIdx.x * 256 + threadIdx.x, r = blockIdx.y;
  if (q >= n_cal) return;
  const long long p = (long long)q * stride;
  const bool hit = p < a.n_pixels && (a.env_flag == nullptr || a.env_flag[p] != 0);
  float x[3] = {0.f, 0.f, 0.f};
  if (hit) {
    const float4 x4 = *(const float4 *)(a.position + 4 * (size_t)p);
    x[0] = x4.x;
    x[1] = x4.y;
    x[2] = x4.z;
  }
  uint2 *dst = (uint2 *)calib;
  float v[4] = {0.f, 0.f, 0.f, 0.f};
  if (hit) {
    dev::accumulate_level<2, HF16>(a.lv, a.hash, r, x, v, nullptr);
    dev::accumulate_level<2, HF16>(a.lv, a.hash, 15 - r, x, v + 2, nullptr);
  }
  dst[(size_t)r * n_cal + q] = make_uint2(dev::pack_bf16(v[0], v[1]), dev::pack_bf16(v[2], v[3]));
}

__global__ __launch_bounds__(256) void tonemap_kernel(const float *__restrict__ src,
                                                      uint32_t *__restrict__ dst, int n) {
  const int p = blockIdx.x * 256 + threadIdx.x;
  if (p >= n) return;
  const float4 v = *(const float4 *)(src + 4 * (size_t)p);
  dst[p] = dev::tonemap_rgba8(v.x, v.y, v.z);
}

// MAY_SPLIT: the rest of the frame may go to sharing workgroups.  A frame of
// which nothing is split takes the instance without them, whose registers are
// its own.
template <typename E, bool SP, bool DUMP, bool AUX, int GP, bool W4LDS, int MINW, bool MAY_SPLIT>
void launch_shape(const RelightArgs &a, hipStream_t s) {
  const int wgs = (a.n_pixels + kRelightBlock - 1) / kRelightBlock;
  if constexpr (MAY_SPLIT) {
    const int full = full_workgroups(a.n_pixels, a.k, a.fused_encode != 0);
    if (full == 0) {
      hipLaunchKernelGGL((relight_group_kernel<E, SP, AUX>), dim3((a.n_pixels + 63) / 64),
                         dim3(kRelightBlock), 0, s, a);
      return;
    }
    if (full < wgs) {
      const int rest = a.n_pixels - full * kRelightBlock;
      hipLaunchKernelGGL((relight_mfma_kernel<E, SP, DUMP, AUX, GP, W4LDS, MINW, true>),
                         dim3(full + (rest + 63) / 64), dim3(kRelightBlock), 0, s, a, full);
      return;
    }
  }
  hipLaunchKernelGGL((relight_mfma_kernel<E, SP, DUMP, AUX, GP, W4LDS, MINW, false>), dim3(wgs),
                     dim3(kRelightBlock), 0, s, a, wgs);
}

template <typename E, bool SP, int V>
void launch_v(const RelightArgs &a, hipStream_t s) {
  constexpr MfmaVariant v = kMfmaVariants[V];
  if (a.aux) {
    // Aux scenes are built for one tile shape (and variant 0's for the tap).
    if (a.dump) launch_shape<E, SP, true, true, 2, false, 2, false>(a, s);
    else launch_shape<E, SP, false, true, 2, false, 2, true>(a, s);
  } else if (a.dump && V == 0) {
    launch_shape<E, SP, true, false, v.gp, v.w4_lds, v.min_waves, false>(a, s);
  } else {
    launch_shape<E, SP, false, false, v.gp, v.w4_lds, v.min_waves,
                 V == kDefaultMfmaVariant || V == kFewWaveletsVariant>(a, s);
  }
}

template <typename E, bool SP>
void launch_sp(const RelightArgs &a, int variant, hipStream_t s) {
  if (a.dump) variant = 0;  // the transport tap is built for variant 0 only
  switch (variant) {
    case 0: launch_v<E, SP, 0>(a, s); break;
    case 1: launch_v<E, SP, 1>(a, s); break;
    case 2: launch_v<E, SP, 2>(a, s); break;
    case 3: launch_v<E, SP, 3>(a, s); break;
    case 4: launch_v<E, SP, 4>(a, s); break;
    case 5: launch_v<E, SP, 5>(a, s); break;
    case 6: launch_v<E, SP, 6>(a, s); break;
    default: fail(NWPRT_ERR_INVALID_ARGUMENT, "relight: unknown kernel variant");
  }
}

template <typename E, bool SP, int V>
void launch_batch_v(const RelightArgs *jobs, const BatchItem *items, const int *n_items,
                    unsigned int *counter, bool has_aux, int n_cu, hipStream_t s) {
  constexpr MfmaVariant v = kMfmaVariants[V];
  static_assert(!v.w4_lds, "the batch form keeps the output layer in VGPRs");
  if (has_aux)
    hipLaunchKernelGGL((relight_batch_kernel<E, SP, true, v.gp, v.min_waves>),
                       dim3(n_cu * v.min_waves), dim3(kRelightBlock), 0, s, jobs, items, n_items,
                       counter);
  else
    hipLaunchKernelGGL((relight_batch_kernel<E, SP, false, v.gp, v.min_waves>),
                       dim3(n_cu * v.min_waves), dim3(kRelightBlock), 0, s, jobs, items, n_items,
                       counter);
}

template <typename E, bool SP>
void launch_batch_e(const RelightArgs *jobs, const BatchItem *items, const int *n_items,
                    unsigned int *counter, bool has_aux, int variant, int n_cu, hipStream_t s) {
  switch (variant) {
    case 0: launch_batch_v<E, SP, 0>(jobs, items, n_items, counter, has_aux, n_cu, s); break;
    case 1: launch_batch_v<E, SP, 1>(jobs, items, n_items, counter, has_aux, n_cu, s); break;
    case 5: launch_batch_v<E, SP, 5>(jobs, items, n_items, counter, has_aux, n_cu, s); break;
    default: fail(NWPRT_ERR_INVALID_ARGUMENT, "batch: variant has no persistent form");
  }
}

template <typename E>
void launch_mfma_variant(const RelightArgs &a, int variant, hipStream_t s) {
  if (a.softplus) launch_sp<E, true>(a, variant, s);
  else launch_sp<E, false>(a, variant, s);
}

}  // namespace

// A-operand tiles of layers 2, 3 (64 x 64) and the output layer (3 x 64) for
// the chained MFMA layout above.  Tile [b][kb][lane][s] holds
// W[16 b + lane%16][f(kb, lane/16, s)] with the contraction permutation
// f(kb, g, s) = 32 kb + (s < 4 ? 4 g + s : 16 + 4 g + s - 4).  The output
// layer is stored as four variants j (in place of b): rows 4j..4j+2 hold W4,
// the other rows are zero.
void build_weight_tiles(const float *w, Elem elem, std::vector<uint16_t> &out) {
  const float *W2 = w + kW1, *W3 = W2 + kW2, *W4 = W3 + kW3;
  out.assign(3 * 4 * 2 * 64 * 8, 0);
  auto cvt = [&](float v) {
    return elem == Elem::BF16 ? f32_to_bf16_bits(v) : f32_to_f16_bits(v);
  };
  auto feat = [](int kb, int g, int s) { return 32 * kb + (s < 4 ? 4 * g + s : 16 + 4 * g + s - 4); };
  for (int layer = 0; layer < 3; ++layer)
    for (int b = 0; b < 4; ++b)
      for (int kb = 0; kb < 2; ++kb)
        for (int lane = 0; lane < 64; ++lane)
          for (int s = 0; s < 8; ++s) {
            const int row = lane & 15, g = lane >> 4, f = feat(kb, g, s);
            float v = 0.f;
            if (layer == 0) v = W2[(16 * b + row) * 64 + f];
            else if (layer == 1) v = W3[(16 * b + row) * 64 + f];
            else if (row >= 4 * b && row < 4 * b + 3) v = W4[(row - 4 * b) * 64 + f];
            out[((((size_t)layer * 4 + b) * 2 + kb) * 64 + lane) * 8 + s] = cvt(v);
          }
}

int relight_mfma_variant_count() { return kNumMfmaVariants; }

// The pipelined step is the faster one, except where the encode is fused and 8
// to 27 wavelets follow it on frames of more than two rounds: each wave's
// encode is then as long as its network, and the two-group step leaves the
// encoding waves more room (BF16, 2432 workgroups, two-group / pipelined:
// K = 8 333 / 354 us, 16 359 / 397, 24 407 / 416, 32 473 / 458, 64 748 / 718;
// along a surface 222 / 218, 257 / 280, 315 / 336, 382 / 373; 896 workgroups:
// 16 162 / 165, 24 183 / 182; p2 alone, 2496: 16 170 / 162).
int relight_mfma_default_variant(int k, int n_pixels, bool fused) {
  return fused && k >= 8 && k < 28 && n_pixels > 2 * kRoundWgs * kRelightBlock
             ? kFewWaveletsVariant
             : kDefaultMfmaVariant;
}
const char *relight_mfma_variant_name(int v) {
  return v >= 0 && v < kNumMfmaVariants ? kMfmaVariants[v].name : nullptr;
}

// A tiles of the second layer's 16 aux columns for v_mfma_f32_16x16x16:
// tile [b][lane][s] = Waux[16 b + lane%16][4 (lane/16) + s].
void build_aux_tiles(const float *waux, Elem elem, std::vector<uint16_t> &out) {
  out.assign(4 * 64 * 4, 0);
  for (int b = 0; b < 4; ++b)
    for (int lane = 0; lane < 64; ++lane)
      for (int s = 0; s < 4; ++s) {
        const float v = waux[(16 * b + (lane & 15)) * 16 + 4 * (lane >> 4) + s];
        out[((size_t)b * 64 + lane) * 4 + s] =
            elem == Elem::BF16 ? f32_to_bf16_bits(v) : f32_to_f16_bits(v);
      }
}

void launch_relight_mfma(const RelightArgs &a, Elem elem, int variant, hipStream_t s) {
  require(a.n_pixels >= 1 && a.k >= 1 && a.k <= NWPRT_MAX_K, NWPRT_ERR_INVALID_ARGUMENT,
          "relight: bad pixel count or K");
  require((a.fused_encode ? a.position && a.hash : a.features != nullptr) && a.mk && a.light &&
              a.w_tiles && a.direct,
          NWPRT_ERR_INVALID_ARGUMENT, "relight: missing operand");
  require(!a.aux || a.waux_tiles, NWPRT_ERR_INVALID_ARGUMENT, "relight: missing aux weights");
  require(!a.fused_encode || (!a.aux && a.lv.n_levels == 16), NWPRT_ERR_INVALID_ARGUMENT,
          "relight: the fused encode needs 16 x 2 grids without aux inputs");
  if (elem == Elem::BF16) {
    launch_mfma_variant<__bf16>(a, variant, s);
  } else if (elem == Elem::F16) {
    launch_mfma_variant<_Float16>(a, variant, s);
  } else {
    fail(NWPRT_ERR_INVALID_ARGUMENT, "relight: MFMA element must be BF16 or FP16");
  }
  hip_check(hipGetLastError(), "relight_mfma_kernel launch");
}

bool relight_batch_variant_ok(int v) {
  return v >= 0 && v < kNumMfmaVariants && !kMfmaVariants[v].w4_lds;
}

void launch_relight_batch(const RelightArgs *jobs, const BatchItem *items, const int *n_items,
                          unsigned int *counter, Elem elem, bool softplus, bool has_aux,
                          int variant, int n_cu, hipStream_t s) {
  require(jobs && items && n_items && counter && n_cu >= 1, NWPRT_ERR_INVALID_ARGUMENT,
          "batch: missing operand");
  if (elem == Elem::BF16) {
    if (softplus)
      launch_batch_e<__bf16, true>(jobs, items, n_items, counter, has_aux, variant, n_cu, s);
    else
      launch_batch_e<__bf16, false>(jobs, items, n_items, counter, has_aux, variant, n_cu, s);
  } else if (elem == Elem::F16) {
    if (softplus)
      launch_batch_e<_Float16, true>(jobs, items, n_items, counter, has_aux, variant, n_cu, s);
    else
      launch_batch_e<_Float16, false>(jobs, items, n_items, counter, has_aux, variant, n_cu, s);
  } else {
    fail(NWPRT_ERR_INVALID_ARGUMENT, "batch: MFMA element must be BF16 or FP16");
  }
  hip_check(hipGetLastError(), "relight_batch_kernel launch");
}

void launch_reset_counter(unsigned int *counter, hipStream_t s) {
  hipLaunchKernelGGL(reset_counter_kernel, dim3(1), dim3(1), 0, s, counter);
  hip_check(hipGetLastError(), "reset_counter_kernel launch");
}

void launch_calib_gather(const uint16_t *features, const uint16_t *aux, const uint8_t *env_flag,
                         int n_pixels, int stride, uint16_t *calib, uint16_t *calib_aux,
                         int n_cal, float *amax, bool planar, hipStream_t s) {
  require(features && calib && amax && n_pixels >= 1 && stride >= 1 && n_cal >= 1 &&
              (long long)(n_cal - 1) * stride < n_pixels && (!aux || (calib_aux && !planar)),
          NWPRT_ERR_INVALID_ARGUMENT, "calibration gather: bad subsample");
  const int threads = (planar ? 8 : 4) * n_cal;
  hipLaunchKernelGGL(calib_gather_kernel, dim3((threads + 255) / 256), dim3(256), 0, s, features,
                     aux, env_flag, n_pixels, stride, calib, calib_aux, n_cal, amax, (int)planar);
  hip_check(hipGetLastError(), "calib_gather_kernel launch");
}

void launch_calib_encode(const RelightArgs &enc, int stride, uint16_t *calib, int n_cal,
                         float *amax, hipStream_t s) {
  require(enc.position && enc.hash && calib && amax && enc.n_pixels >= 1 && stride >= 1 &&
              n_cal >= 1 && (long long)(n_cal - 1) * stride < enc.n_pixels &&
              enc.lv.n_levels == 16,
          NWPRT_ERR_INVALID_ARGUMENT, "calibration encode: bad subsample");
  const dim3 grid((n_cal + 255) / 256, 8);
  if (enc.hash_f16)
    hipLaunchKernelGGL(calib_encode_kernel<true>, grid, dim3(256), 0, s, enc, stride, calib, n_cal,
                       amax);
  else
    hipLaunchKernelGGL(calib_encode_kernel<false>, grid, dim3(256), 0, s, enc, stride, calib,
                       n_cal, amax);
  hip_check(hipGetLastError(), "calib_encode_kernel launch");
}

void launch_calibrate_amax(const RelightArgs &a, hipStream_t s) {
  require(a.n_pixels >= 1 && a.k >= 1 && a.k <= NWPRT_MAX_K && a.features && a.mk &&
              a.w_tiles && a.amax && (!a.aux || a.waux_tiles),
          NWPRT_ERR_INVALID_ARGUMENT, "calibration: missing operand");
  // As many chunks of wavelets as make one round of the chip (256 CUs, three
  // workgroups each): 16,384 pixels, K = 300: chunks of 16 (1.6 rounds, each
  // step waiting for its tiles, each wave its atomics) 213 us, so 130.
  constexpr int kRound = 768;
  const int px = (a.n_pixels + kRelightBlock - 1) / kRelightBlock;
  const int splits = std::min(a.k, std::max(1, kRound / px)), kChunk = (a.k + splits - 1) / splits;
  const dim3 grid(px, (a.k + kChunk - 1) / kChunk);
  if (a.aux)
    hipLaunchKernelGGL(calib_amax_kernel<true>, grid, dim3(kRelightBlock), 0, s, a, kChunk);
  else
    hipLaunchKernelGGL(calib_amax_kernel<false>, grid, dim3(kRelightBlock), 0, s, a, kChunk);
  hip_check(hipGetLastError(), "calib_amax_kernel launch");
}

void launch_tonemap(const float *src, uint32_t *dst, int n_pixels, hipStream_t s) {
  require(n_pixels >= 1, NWPRT_ERR_INVALID_ARGUMENT, "tonemap: no pixels");
  hipLaunchKernelGGL(tonemap_kernel, dim3((n_pixels + 255) / 256), dim3(256), 0, s, src, dst,
                     n_pixels);
  hip_check(hipGetLastError(), "tonemap_kernel launch");
}

}  // namespace nwprt
