// Residual add + LayerNorm of the OPT decoder layer for gfx950, one launch per (add, norm) pair.
//
// A decode step of OPT-13B runs two LayerNorms and two residual adds per layer on a handful of rows: as four
// element-wise launches of a tensor library they cost more in launch and memory round trips than in work.  Here
// one workgroup owns one row: it adds the residual in fp32, rounds the sum once to the 16-bit activation type
// (that rounded sum is the next residual), and normalises the rounded values — mean and variance in two passes
// over registers, fp32 — so the results are those of "add, then LayerNorm" on 16-bit tensors.
#include "aps_common.h"
#include "mfma_common.h"

namespace aps {
namespace {

constexpr int kLnThreads = 256, kLnVecs = 8;  // a row of up to 256 * 8 * 8 = 16384 elements lives in registers

struct AddLnArgs {
  char* normed; char* sum;                       // sum nullable
  const char* x; const char* residual;           // residual nullable
  const char* gamma; const char* beta;           // beta nullable
  int64_t x_stride_b, res_stride_b, normed_stride_b, sum_stride_b;
  int width;
  float eps;
  // PARTS: x is a product in K parts, fp32 planes [rows][width] that are added in order, plus its bias (nullable), rounded once
  const float* partial; const char* lin_bias;
  int64_t plane;
  int parts;
};

__device__ __forceinline__ float block_sum(float v, float* red) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
  __syncthreads();  // red may still be read from the previous reduction
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  return (red[0] + red[1]) + (red[2] + red[3]);
}

template <bool BF16>
__device__ __forceinline__ float from16(uint32_t bits) {
  if constexpr (BF16) return __uint_as_float(bits << 16);
  else return (float)__builtin_bit_cast(_Float16, (uint16_t)bits);
}
template <bool BF16>
__device__ __forceinline__ uint32_t to16(float v) {
  return BF16 ? f32_to_bf16_bits(v) : f32_to_f16_bits(v);
}

// The thread's vectors of a row of the product, rounded: parts in order, those of all vectors in flight together (a vector at a
// time 7.2 us for 5 rows of 4 parts, 10.8 for 361; so 4.9 and 9.7), then the bias.  Past the row's end: its last vector.
template <bool BF16, int VECS>
__device__ __forceinline__ void product_vecs(const AddLnArgs& g, int64_t row, int nvec, u32x4 (&a)[VECS]) {
  constexpr int ZC = VECS <= 3 ? 3 : 1;
  const float* p[VECS];
  float4v s[VECS][2];
  u32x4 c[VECS];
#pragma unroll
  for (int j = 0; j < VECS; ++j) {
    const int i = min((int)threadIdx.x + j * kLnThreads, nvec - 1);
    p[j] = g.partial + row * g.width + (int64_t)i * 8;
    s[j][0] = *(const float4v*)p[j]; s[j][1] = *(const float4v*)(p[j] + 4);
    c[j] = g.lin_bias ? *(const u32x4*)(g.lin_bias + (int64_t)i * 16) : u32x4{0u, 0u, 0u, 0u};
  }
  for (int z0 = 1; z0 < g.parts; z0 += ZC) {
    float4v t[ZC][VECS][2];
#pragma unroll
    for (int z = 0; z < ZC; ++z)
#pragma unroll
      for (int j = 0; j < VECS; ++j) {
        const float* q = p[j] + (int64_t)min(z0 + z, g.parts - 1) * g.plane;
        t[z][j][0] = *(const float4v*)q; t[z][j][1] = *(const float4v*)(q + 4);
      }
#pragma unroll
    for (int z = 0; z < ZC; ++z)
      if (z0 + z < g.parts) {
#pragma unroll
        for (int j = 0; j < VECS; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e) { s[j][0][e] += t[z][j][0][e]; s[j][1][e] += t[z][j][1][e]; }
      }
  }
#pragma unroll
  for (int j = 0; j < VECS; ++j)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float lo = s[j][e >> 1][2 * (e & 1)], hi = s[j][e >> 1][2 * (e & 1) + 1];
      if (g.lin_bias) { lo += from16<BF16>(c[j][e] & 0xffffu); hi += from16<BF16>(c[j][e] >> 16); }
      a[j][e] = to16<BF16>(lo) | (to16<BF16>(hi) << 16);
    }
}

// PARTS: the sum over a product's K parts is taken here instead of in a launch of its own that writes the product for this
// one to read (361 rows of 5120 in 4 parts: 9.7 us for 7.0 + 6.5 and the gap between them; 5 rows 4.9, and the product in front
// of it, which no longer adds its parts by itself, 35.3 instead of 39.1).
template <bool BF16, int VECS, bool PARTS>
__global__ __launch_bounds__(kLnThreads) void add_layer_norm_kernel(const AddLnArgs g) {
  __shared__ float red[4];
  const int64_t row = blockIdx.x;
  const int nvec = g.width >> 3;  // 8 elements (16 bytes) per vector
  const char* x = g.x + row * g.x_stride_b;
  const char* r = g.residual ? g.residual + row * g.res_stride_b : nullptr;
  float v[VECS][8];
  float total = 0.f;
  // scale and shift of the norm are requested with the row itself: on a handful of rows the launch lasts as long
  // as its chain of memory round trips, and these two would otherwise form a third one after the statistics
  u32x4 gw[VECS], gb[VECS];
#pragma unroll
  for (int j = 0; j < VECS; ++j) {
    const int i = min((int)threadIdx.x + j * kLnThreads, nvec - 1);
    gw[j] = *(const u32x4*)(g.gamma + (int64_t)i * 16);
    gb[j] = g.beta ? *(const u32x4*)(g.beta + (int64_t)i * 16) : u32x4{0u, 0u, 0u, 0u};
  }
  // (past the row's end: its last vector, loaded and not used, so that no load stands behind a branch; a lone vector waits for
  // none, and there a branch spares the loads)
  u32x4 pa[VECS], pb[VECS];
#pragma unroll
  for (int j = 0; j < VECS; ++j) {
    const int i = min((int)threadIdx.x + j * kLnThreads, nvec - 1);
    if (VECS > 1 || (int)threadIdx.x < nvec) {
      if constexpr (!PARTS) pa[j] = *(const u32x4*)(x + (int64_t)i * 16);
      pb[j] = r ? *(const u32x4*)(r + (int64_t)i * 16) : u32x4{0u, 0u, 0u, 0u};
    }
  }
  if constexpr (PARTS) product_vecs<BF16, VECS>(g, row, nvec, pa);
#pragma unroll
  for (int j = 0; j < VECS; ++j) {
    const int i = threadIdx.x + j * kLnThreads;
    if (i < nvec) {
      const u32x4 a = pa[j], b = pb[j];
      u32x4 s16;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float lo = from16<BF16>(a[e] & 0xffffu), hi = from16<BF16>(a[e] >> 16);
        if (r) {  // the sum is rounded once to the activation type; the norm sees the rounded sum
          lo = from16<BF16>(to16<BF16>(lo + from16<BF16>(b[e] & 0xffffu)));
          hi = from16<BF16>(to16<BF16>(hi + from16<BF16>(b[e] >> 16)));
        }
        v[j][2 * e] = lo;
        v[j][2 * e + 1] = hi;
        s16[e] = to16<BF16>(lo) | (to16<BF16>(hi) << 16);
        total += lo + hi;
      }
      if (g.sum) *(u32x4*)(g.sum + row * g.sum_stride_b + (int64_t)i * 16) = s16;
    }
  }
  const float mean = block_sum(total, red) / (float)g.width;
  float sq = 0.f;
#pragma unroll
  for (int j = 0; j < VECS; ++j) {
    if (threadIdx.x + j * kLnThreads < nvec) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float d = v[j][e] - mean;
        sq += d * d;
      }
    }
  }
  const float rstd = rsqrtf(block_sum(sq, red) / (float)g.width + g.eps);
#pragma unroll
  for (int j = 0; j < VECS; ++j) {
    const int i = threadIdx.x + j * kLnThreads;
    if (i < nvec) {
      const u32x4 w = gw[j], bb = gb[j];
      u32x4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float lo = (v[j][2 * e] - mean) * rstd * from16<BF16>(w[e] & 0xffffu) + from16<BF16>(bb[e] & 0xffffu);
        const float hi = (v[j][2 * e + 1] - mean) * rstd * from16<BF16>(w[e] >> 16) + from16<BF16>(bb[e] >> 16);
        o[e] = to16<BF16>(lo) | (to16<BF16>(hi) << 16);
      }
      *(u32x4*)(g.normed + row * g.normed_stride_b + (int64_t)i * 16) = o;
    }
  }
}

}  // namespace
}  // namespace aps

using namespace aps;

namespace {
template <bool PARTS>
int launch_add_layer_norm(const AddLnArgs& g, int64_t rows, int dtype, aps_stream_t stream) {
  const dim3 grid((unsigned)rows);
  // As many vectors per thread as the row takes, since all of them are loaded, those past the row's end too (us with the residual
  // add, f16; a load behind a branch each, always three or eight vectors, and so: 8192 rows of 768 15.6, 18.0, 12.7; 361 of
  // 2560 4.57, 4.71, 4.57; 361 of 7168 7.1, 7.3, 6.5; 8192 of 7168 112, 87.8, 87.2; 1 of 16384 6.4, 5.5, 5.5).
  const int vecs = (g.width + kLnThreads * 8 - 1) / (kLnThreads * 8);
  hipStream_t s = (hipStream_t)stream;
#define APS_LAUNCH_LN(B, V) APS_LAUNCH((add_layer_norm_kernel<B, V, PARTS>), grid, dim3(kLnThreads), 0, s, g)
#define APS_LAUNCH_LN_V(B)                \
  switch (vecs) {                         \
    case 1: APS_LAUNCH_LN(B, 1); break;   \
    case 2: APS_LAUNCH_LN(B, 2); break;   \
    case 3: APS_LAUNCH_LN(B, 3); break;   \
    case 4: APS_LAUNCH_LN(B, 4); break;   \
    default: APS_LAUNCH_LN(B, kLnVecs);   \
  }
  if (dtype == APS_BF16) { APS_LAUNCH_LN_V(true) } else { APS_LAUNCH_LN_V(false) }
#undef APS_LAUNCH_LN_V
#undef APS_LAUNCH_LN
  return launch_status();
}
}  // namespace

extern "C" int aps_add_layer_norm(void* normed, void* sum, const void* x, const void* residual, const void* gamma,
                                  const void* beta, int64_t rows, int64_t width, int64_t x_stride,
                                  int64_t residual_stride, int64_t normed_stride, int64_t sum_stride, float eps,
                                  int dtype, aps_stream_t stream) {
  if (rows < 0 || width <= 0 || !(eps >= 0.f)) return APS_ERR_INVALID_ARG;
  if (rows == 0) return APS_OK;
  if (!normed || !x || !gamma) return APS_ERR_INVALID_ARG;
  if (dtype != APS_F16 && dtype != APS_BF16) return APS_ERR_UNSUPPORTED;
  if (width % 8 != 0 || width > kLnThreads * kLnVecs * 8 || rows > 0x7fffffff) return APS_ERR_UNSUPPORTED;
  if (x_stride < width || normed_stride < width || (residual && residual_stride < width) ||
      (sum && sum_stride < width))
    return APS_ERR_INVALID_ARG;
  if (common_vec_bytes({addr(normed), addr(sum), addr(x), addr(residual), addr(gamma), addr(beta),
                        (uint64_t)x_stride * 2, (uint64_t)residual_stride * 2, (uint64_t)normed_stride * 2,
                        (uint64_t)sum_stride * 2}) != 16)
    return APS_ERR_UNSUPPORTED;
  AddLnArgs g{(char*)normed, (char*)sum, (const char*)x, (const char*)residual, (const char*)gamma,
              (const char*)beta, x_stride * 2, residual_stride * 2, normed_stride * 2, sum_stride * 2, (int)width, eps,
              nullptr, nullptr, 0, 1};
  return launch_add_layer_norm<false>(g, rows, dtype, stream);
}

// The same of a product's parts (see PARTS); pointers and width as aps_add_layer_norm wants them, rows `width` apart.
__attribute__((visibility("hidden"))) int aps_internal_parts_add_layer_norm(
    void* normed, void* sum, const float* partial, int parts, const void* lin_bias, const void* residual, const void* gamma,
    const void* beta, int64_t rows, int64_t width, int64_t residual_stride, float eps, int dtype, aps_stream_t stream) {
  AddLnArgs g{(char*)normed, (char*)sum, nullptr, (const char*)residual, (const char*)gamma, (const char*)beta, 0,
              residual_stride * 2, width * 2, width * 2, (int)width, eps, partial, (const char*)lin_bias, rows * width, parts};
  return launch_add_layer_norm<true>(g, rows, dtype, stream);
}
