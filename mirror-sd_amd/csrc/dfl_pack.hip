// Weight preparation kernels: the W8A16 quantiser and the HBM block packers.
//
// Weight layout in HBM (written once at load by the pack kernels): blocks of 32 rows x
// KBK k-values (KBK = 32 for int8, 16 for fp16), 1 KiB each, ordered [row-block][k-block];
// inside a block lane l's 16 bytes are
//   int8: W[rb*32 + l%32][kb*32 + 16*(l/32) + 0..15], each stored as q ^ 0x80 (= q + 128)
//   fp16: W[rb*32 + l%32][kb*16 +  8*(l/32) + 0..7]
// so one wave-wide 128-bit load reads 1 KiB contiguous and hands every lane its
// v_mfma_f32_32x32x16_f16 A-fragment directly (int8: two MFMAs per load, after the exact
// int8 -> fp16 conversion).  Per-row fp16 scales are kept apart and applied in the GEMM
// epilogue: y = s * sum x*q is exact reassociation (each fp16*int8 product is exact in fp32).
#include "dfl_common.h"
#include "dfl_kernels.h"

namespace dfl {

// Symmetric per-output-channel int8 quantisation (ane_model.py:265-279):
//   max = max_k |w[n][k]| (0 -> 1),  scale = max / 127 (fp32, correctly rounded),
//   q = clamp(rint(w / scale), -127, 127),  stored scale = fp16(scale).
// Same fp32 values as the numpy reference, so results are bit-identical.
DFL_DEV float quant_row_scale(float mx, float* smax) {
  mx = wave_max(mx);
  if ((threadIdx.x & 63) == 0) smax[threadIdx.x >> 6] = mx;
  __syncthreads();
  mx = fmaxf(fmaxf(smax[0], smax[1]), fmaxf(smax[2], smax[3]));
  if (mx == 0.f) mx = 1.0f;
  return __fdiv_rn(mx, 127.0f);
}
DFL_DEV int quant_value(float r) { return (int)fminf(fmaxf(r, -127.f), 127.f); }

// rint(w / scale).  |w / scale| <= 127 (1 + 2^-23), so w * inv (two roundings) and the
// correctly rounded quotient both lie within 2.5e-5 of the exact one: they round to the same
// integer unless w * inv comes within 1e-4 of a half, where the division is done.  A scale
// below 2^-100 has an inexact or infinite reciprocal (inv = 0 asks for the division).
DFL_DEV float quant_rint(float w, float scale, float inv) {
  const float p = w * inv;
  float r = rintf(p);
  if (inv == 0.f || fabsf(p - r) > 0.4999f) r = rintf(__fdiv_rn(w, scale));
  return r;
}

// Rows of up to 1024 * NV values (ic % 4 == 0, w 16-byte and q 4-byte aligned): the row is
// held in registers between the maximum and the rounding, so w is read once, 16 bytes a lane.
// HBM-bound (5 bytes a weight): 5120 x 17408 in 72 us, 6.15 TB/s.  The two-pass kernel below
// took 207 us: scalar loads, the second pass again from HBM, a division per weight.
template <int NV>
__global__ __launch_bounds__(256) void quantize_w8_row_kernel(const float* __restrict__ w,
                                                              int64_t ic, int8_t* __restrict__ q,
                                                              half_t* __restrict__ s) {
  __shared__ float smax[4];
  const int64_t rowi = blockIdx.x;
  const int n4 = (int)(ic >> 2);
  const floatx4* wr = reinterpret_cast<const floatx4*>(w + rowi * ic);
  floatx4 v[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int k = threadIdx.x + 256 * i;
    v[i] = (floatx4){0.f, 0.f, 0.f, 0.f};
    if (k < n4) v[i] = __builtin_nontemporal_load(wr + k);
  }
  float mx = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) mx = fmaxf(mx, fabsf(v[i][j]));
  const float scale = quant_row_scale(mx, smax);
  const float inv = scale >= 0x1p-100f ? __fdiv_rn(1.0f, scale) : 0.f;
  uint32_t* qr = reinterpret_cast<uint32_t*>(q + rowi * ic);
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int k = threadIdx.x + 256 * i;
    if (k >= n4) break;
    uint32_t o = 0u;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      o |= ((uint32_t)quant_value(quant_rint(v[i][j], scale, inv)) & 0xFFu) << (8 * j);
    qr[k] = o;
  }
  if (threadIdx.x == 0) s[rowi] = f2h(scale);
}

// Any row length and alignment: the row is read twice.
__global__ __launch_bounds__(256) void quantize_w8_kernel(const float* __restrict__ w, int64_t ic,
                                                          int8_t* __restrict__ q,
                                                          half_t* __restrict__ s) {
  __shared__ float smax[4];
  const int64_t rowi = blockIdx.x;
  const float* wr = w + rowi * ic;
  float mx = 0.f;
  for (int64_t k = threadIdx.x; k < ic; k += blockDim.x) mx = fmaxf(mx, fabsf(wr[k]));
  const float scale = quant_row_scale(mx, smax);
  int8_t* qr = q + rowi * ic;
  for (int64_t k = threadIdx.x; k < ic; k += blockDim.x)
    qr[k] = (int8_t)quant_value(rintf(__fdiv_rn(wr[k], scale)));
  if (threadIdx.x == 0) s[rowi] = f2h(scale);
}

void launch_quantize_w8(const float* w, int64_t oc, int64_t ic, int8_t* q, half_t* s,
                        hipStream_t st) {
  // one instantiation per register budget: the lanes' share of the row in 4, 8, 12 or 20
  // 16-byte loads
  const bool vec = ic % 4 == 0 && !(reinterpret_cast<uintptr_t>(w) & 15) &&
                   !(reinterpret_cast<uintptr_t>(q) & 3);
  auto* kernel = quantize_w8_kernel;
  if (vec && ic <= 4096) kernel = quantize_w8_row_kernel<4>;
  else if (vec && ic <= 8192) kernel = quantize_w8_row_kernel<8>;
  else if (vec && ic <= 12288) kernel = quantize_w8_row_kernel<12>;
  else if (vec && ic <= 20480) kernel = quantize_w8_row_kernel<20>;
  hipLaunchKernelGGL(kernel, dim3((unsigned)oc), dim3(256), 0, st, w, ic, q, s);
}

__global__ __launch_bounds__(64) void pack_i8_kernel(const int8_t* __restrict__ q,
                                                     const half_t* __restrict__ s, int K,
                                                     uint4* __restrict__ dst,
                                                     half_t* __restrict__ dscale, int rb0,
                                                     int rb_step) {
  const int kb = blockIdx.x, rb = blockIdx.y, l = threadIdx.x;
  const int KB = K / 32;
  const int drb = rb0 + rb * rb_step;
  const int8_t* src = q + (size_t)(rb * 32 + (l & 31)) * K + (size_t)kb * 32 + 16 * (l >> 5);
  uint4 v = *reinterpret_cast<const uint4*>(src);
  v.x ^= 0x80808080u;   // biased bytes q + 128 (dequant_i8x16)
  v.y ^= 0x80808080u;
  v.z ^= 0x80808080u;
  v.w ^= 0x80808080u;
  dst[((size_t)drb * KB + kb) * 64 + l] = v;
  if (kb == 0 && l < 32) dscale[(size_t)drb * 32 + l] = s[(size_t)rb * 32 + l];
}

void launch_pack_i8(const int8_t* q, const half_t* s, int rows, int K, uint4* dst,
                    half_t* dst_scale, int rb0, int rb_step, hipStream_t st) {
  hipLaunchKernelGGL(pack_i8_kernel, dim3(K / 32, rows / 32), dim3(64), 0, st, q, s, K, dst,
                     dst_scale, rb0, rb_step);
}

__global__ __launch_bounds__(64) void pack_f16_kernel(const half_t* __restrict__ w, int K,
                                                      uint4* __restrict__ dst) {
  const int kb = blockIdx.x, rb = blockIdx.y, l = threadIdx.x;
  const int KB = K / 16;
  const half_t* src = w + (size_t)(rb * 32 + (l & 31)) * K + (size_t)kb * 16 + 8 * (l >> 5);
  dst[((size_t)rb * KB + kb) * 64 + l] = *reinterpret_cast<const uint4*>(src);
}

void launch_pack_f16(const half_t* w, int rows, int K, uint4* dst, hipStream_t st) {
  hipLaunchKernelGGL(pack_f16_kernel, dim3(K / 16, rows / 32), dim3(64), 0, st, w, K, dst);
}

}  // namespace dfl
