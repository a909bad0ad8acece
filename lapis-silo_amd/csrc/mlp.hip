// HIP kernels of the planner's cardinality estimator: a multilayer perceptron with BF16 weights
// and FP32 accumulation, trained on the device.
//
//   forward   Z_l = A_{l-1} W_l^T + b_l,  A_l = relu(Z_l) (hidden layers), output Z_L (one unit)
//   loss      mean over the batch of (Z_L - y)^2
//   backward  dZ_L = 2 (Z_L - y) / N;  dW_l = dZ_l^T A_{l-1};  db_l = column sums of dZ_l;
//             dA_{l-1} = dZ_l W_l;  dZ_{l-1} = dA_{l-1} * [Z_{l-1} > 0]
//   update    Adam on FP32 master parameters, then the BF16 copy the products read
//
// Networks of up to 128 inputs and hidden units (the planner's is 32 -> 3 x 128 -> 1) run fused: one
// kernel takes a tile of rows through every layer and back, with FP32 matrix instructions
// (mlpFusedKernel), and one kernel sums the tiles' gradients and applies Adam (mlpUpdateKernel).
// Wider networks use one generic LDS-tiled product kernel per layer: 64 x 64 output tiles, 16-deep
// slices of both operands staged in LDS, 4 x 4 outputs per thread.
#include <hip/hip_bf16.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "mlp_kernels.h"

namespace rdb {

namespace {

constexpr int kTile = 64;
constexpr int kDepth = 16;

__device__ inline float loadB(const float* p, size_t i) { return p[i]; }
__device__ inline float loadB(const __hip_bfloat16* p, size_t i) { return __bfloat162float(p[i]); }

// C[m, n] (+)= sum_k A(m, k) * B(k, n) with A(m, k) = a[m * sam + k * sak] and
// B(k, n) = b[k * sbk + n * sbn]; then + bias[n] and relu when asked.
template <typename TB>
__global__ __launch_bounds__(256) void gemmKernel(int M, int N, int K, const float* __restrict__ a, long sam, long sak,
                                                  const TB* __restrict__ b, long sbk, long sbn, float* __restrict__ c,
                                                  long ldc, const float* __restrict__ bias, int relu, int accumulate) {
   __shared__ float as[kDepth][kTile + 1];
   __shared__ float bs[kDepth][kTile + 1];
   const int tx = threadIdx.x & 15;  // 16 x 16 threads, 4 x 4 outputs each
   const int ty = threadIdx.x >> 4;
   const int m0 = blockIdx.y * kTile;
   const int n0 = blockIdx.x * kTile;
   float acc[4][4] = {};
   for (int k0 = 0; k0 < K; k0 += kDepth) {
      for (int i = threadIdx.x; i < kDepth * kTile; i += 256) {
         const int kk = i / kTile, mm = i % kTile;
         const int m = m0 + mm, k = k0 + kk;
         as[kk][mm] = (m < M && k < K) ? a[static_cast<long>(m) * sam + static_cast<long>(k) * sak] : 0.0f;
         const int n = n0 + mm;
         bs[kk][mm] = (n < N && k < K) ? loadB(b, static_cast<size_t>(static_cast<long>(k) * sbk + static_cast<long>(n) * sbn))
                                       : 0.0f;
      }
      __syncthreads();
#pragma unroll
      for (int kk = 0; kk < kDepth; ++kk) {
         float av[4], bv[4];
#pragma unroll
         for (int r = 0; r < 4; ++r) av[r] = as[kk][ty * 4 + r];
#pragma unroll
         for (int r = 0; r < 4; ++r) bv[r] = bs[kk][tx * 4 + r];
#pragma unroll
         for (int i = 0; i < 4; ++i) {
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[i][j] += av[i] * bv[j];
         }
      }
      __syncthreads();
   }
#pragma unroll
   for (int i = 0; i < 4; ++i) {
      const int m = m0 + ty * 4 + i;
      if (m >= M) continue;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
         const int n = n0 + tx * 4 + j;
         if (n >= N) continue;
         float v = acc[i][j];
         if (bias) v += bias[n];
         if (relu) v = v > 0.0f ? v : 0.0f;
         float* out = c + static_cast<long>(m) * ldc + n;
         *out = accumulate ? *out + v : v;
      }
   }
}

// dZ = 2 (z - y) / n for the output unit, and the summed squared error.
__global__ void outputGradKernel(int n, const float* __restrict__ z, const float* __restrict__ y, float* __restrict__ dz,
                                 float* __restrict__ loss) {
   __shared__ float part[4];
   const int i = blockIdx.x * blockDim.x + threadIdx.x;
   float e2 = 0.0f;
   if (i < n) {
      const float e = z[i] - y[i];
      dz[i] = 2.0f * e / static_cast<float>(n);
      e2 = e * e;
   }
   for (int off = 32; off > 0; off >>= 1) e2 += __shfl_xor(e2, off, 64);
   if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = e2;
   __syncthreads();
   if (threadIdx.x == 0) atomicAdd(loss, part[0] + part[1] + part[2] + part[3]);
}

// dZ *= [Z > 0] (relu derivative), in place.
__global__ void reluGradKernel(long count, const float* __restrict__ z, float* __restrict__ dz) {
   const long i = blockIdx.x * static_cast<long>(blockDim.x) + threadIdx.x;
   if (i < count && !(z[i] > 0.0f)) dz[i] = 0.0f;
}

// db[o] = sum over rows of dz[r, o]; one work-group per output unit.
__global__ void columnSumKernel(int rows, int cols, const float* __restrict__ dz, float* __restrict__ db) {
   __shared__ float part[4];
   const int o = blockIdx.x;
   float s = 0.0f;
   for (int r = threadIdx.x; r < rows; r += blockDim.x) s += dz[static_cast<long>(r) * cols + o];
   for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
   if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = s;
   __syncthreads();
   if (threadIdx.x == 0) db[o] = part[0] + part[1] + part[2] + part[3];
}

__global__ void adamKernel(long n, float* __restrict__ master, __hip_bfloat16* __restrict__ w, const float* __restrict__ g,
                           float* __restrict__ m1, float* __restrict__ m2, float lr, float b1, float b2, float eps,
                           float c1, float c2) {
   const long i = blockIdx.x * static_cast<long>(blockDim.x) + threadIdx.x;
   if (i >= n) return;
   const float gi = g[i];
   const float a = b1 * m1[i] + (1.0f - b1) * gi;
   const float b = b2 * m2[i] + (1.0f - b2) * gi * gi;
   m1[i] = a;
   m2[i] = b;
   const float p = master[i] - lr * (a / c1) / (sqrtf(b / c2) + eps);
   master[i] = p;
   w[i] = __float2bfloat16(p);
}

__global__ void toBf16Kernel(long n, const float* __restrict__ src, __hip_bfloat16* __restrict__ dst) {
   const long i = blockIdx.x * static_cast<long>(blockDim.x) + threadIdx.x;
   if (i < n) dst[i] = __float2bfloat16(src[i]);
}

__global__ void fromBf16Kernel(long n, const __hip_bfloat16* __restrict__ src, float* __restrict__ dst) {
   const long i = blockIdx.x * static_cast<long>(blockDim.x) + threadIdx.x;
   if (i < n) dst[i] = __bfloat162float(src[i]);
}

// ---- fused passes of small networks ---------------------------------------------------------------
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__device__ inline float bf16Lo(uint32_t x) { return __uint_as_float(x << 16); }
__device__ inline float bf16Hi(uint32_t x) { return __uint_as_float(x & 0xFFFF0000u); }

// C += A B^T over K (a multiple of 16): `a` an LDS row of this lane's A row (32 rows), `b` this
// lane's row of a packed BF16 matrix in global memory (32 rows).  The two halves of the wavefront
// take eight consecutive k each, so that a lane's operands of eight 32x32x2 products are two 16-byte
// LDS reads and one 16-byte load; all loads of a 128-deep row are issued before the first product.
template <uint32_t kMaxK>
__device__ inline f32x16 rowsTimesPacked(const float* a, const uint16_t* b, uint32_t K, uint32_t half, f32x16 c) {
   u32x4 w[kMaxK / 16];
#pragma unroll
   for (uint32_t s = 0; s < kMaxK / 16; ++s) {
      if (16 * s < K) w[s] = *reinterpret_cast<const u32x4*>(b + 16 * s + 8 * half);
   }
#pragma unroll
   for (uint32_t s = 0; s < kMaxK / 16; ++s) {
      if (16 * s < K) {
         const f32x4 x0 = *reinterpret_cast<const f32x4*>(a + 16 * s + 8 * half);
         const f32x4 x1 = *reinterpret_cast<const f32x4*>(a + 16 * s + 8 * half + 4);
#pragma unroll
         for (uint32_t j = 0; j < 4; ++j) {
            const uint32_t p = w[s][j];
            const float xe = j < 2 ? x0[2 * (j & 1)] : x1[2 * (j & 1)];
            const float xo = j < 2 ? x0[2 * (j & 1) + 1] : x1[2 * (j & 1) + 1];
            c = __builtin_amdgcn_mfma_f32_32x32x2f32(xe, bf16Lo(p), c, 0, 0, 0);
            c = __builtin_amdgcn_mfma_f32_32x32x2f32(xo, bf16Hi(p), c, 0, 0, 0);
         }
      }
   }
   return c;
}

// One work-group (four wavefronts) takes 32 rows at a time through every layer, and with kTrain back:
// activations stay in LDS (a hidden layer's gradients overwrite its activations), wavefront w owns
// hidden units 32 w .. 32 w + 31, and weights are read once per tile from their packed BF16 copies
// (74 KB for the planner's network: L2).  The layer-by-layer form wrote and re-read every activation,
// and its weight gradients (128 x 128 outputs over thousands of rows) ran in four work-groups.
// Bound by the chain of dependent layers: a launch of one training tile per work-group takes 56 us, in which
// the matrix instructions keep a SIMD busy for 11 (26.6 k cycles, SQ_VALU_MFMA_BUSY_CYCLES); its one wavefront
// waits for half of its cycles (SQ_WAIT_ANY), for weights, LDS and the barriers between layers.  32 rows
// keep one tile per work-group at the training batch of 4,096 (128 work-groups); 16 would fill all
// CUs but double the partial gradients written.
// C layout of the 32x32 products: register i of lane l is row 8 (i / 4) + 4 (l / 32) + i % 4, column
// l % 32.
constexpr uint32_t kFusedRows = 32;
constexpr uint32_t kFusedPad = 4;  // floats after each LDS row: 16-byte reads of 16 rows hit all banks

template <bool kTrain>
__global__ __launch_bounds__(256) void mlpFusedKernel(MlpFused p) {
   extern __shared__ __align__(16) float lds[];
   const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
   const uint32_t col = lane & 31, half = lane >> 5;
   const uint32_t nh = p.n_hidden, ni = p.n_in, H = p.n_hidden_layers;
   const uint32_t hp = p.hidden_pad, ip = p.in_pad;
   const uint32_t sx = ip + kFusedPad, sh = hp + kFusedPad;
   float* xin = lds;
   float* act = lds + kFusedRows * sx;  // hidden layer l at act + l * 32 * sh
   float* dzo = act + H * kFusedRows * sh;
   const uint32_t unit = 32 * wave + col;  // this lane's hidden unit
   const size_t first = static_cast<size_t>(ni) * nh + nh, next = static_cast<size_t>(nh) * nh + nh;
   auto weights = [&](uint32_t l) -> size_t { return l == 0 ? 0 : first + (l - 1) * next; };  // of layer l's W
   auto rowOf = [&](uint32_t i) -> uint32_t { return 8 * (i >> 2) + 4 * half + (i & 3); };
   float* part = kTrain ? p.partial + static_cast<size_t>(blockIdx.x) * p.n_params : nullptr;
   float sq = 0.0f;
   bool begun = false;  // this work-group's partial gradients hold an earlier tile's
   for (size_t r0 = static_cast<size_t>(blockIdx.x) * kFusedRows; r0 < p.n; r0 += static_cast<size_t>(gridDim.x) * kFusedRows) {
      __syncthreads();  // the previous tile's readers are done
      for (uint32_t i = tid; i < kFusedRows * ip; i += 256) {
         const uint32_t r = i / ip, k = i - r * ip;
         xin[r * sx + k] = r0 + r < p.n && k < ni ? p.x[(r0 + r) * ni + k] : 0.0f;
      }
      __syncthreads();
      for (uint32_t l = 0; l < H; ++l) {
         float* out = act + l * kFusedRows * sh;
         if (32 * wave < hp) {
            f32x16 c = {};
            if (l == 0) {
               c = rowsTimesPacked<128>(xin + col * sx, p.packed + unit * ip, ip, half, c);
            } else {
               c = rowsTimesPacked<128>(out - kFusedRows * sh + col * sh,
                                        p.packed + hp * ip + (static_cast<size_t>(l - 1) * hp + unit) * hp, hp, half, c);
            }
            const float bias = unit < nh ? p.eff[weights(l) + static_cast<size_t>(l == 0 ? ni : nh) * nh + unit] : 0.0f;
#pragma unroll
            for (uint32_t i = 0; i < 16; ++i) {
               const float v = c[i] + bias;
               out[rowOf(i) * sh + unit] = v > 0.0f ? v : 0.0f;
            }
         }
         __syncthreads();
      }
      // the output unit: eight lanes per row
      const float* top = act + (H - 1) * kFusedRows * sh;
      const float* w_out = p.eff + weights(H);
      {
         const uint32_t r = tid >> 3, k0 = tid & 7;
         float z = 0.0f;
         for (uint32_t k = k0; k < nh; k += 8) z += top[r * sh + k] * w_out[k];
         for (int off = 4; off > 0; off >>= 1) z += __shfl_xor(z, off, 64);
         z += w_out[nh];
         if (!kTrain) {
            if (k0 == 0 && r0 + r < p.n) p.out[r0 + r] = z;
         } else if (k0 == 0) {
            const bool have = r0 + r < p.n;
            const float e = have ? z - p.y[r0 + r] : 0.0f;
            dzo[r] = have ? 2.0f * e / static_cast<float>(p.n) : 0.0f;
            sq += e * e;
         }
      }
      if constexpr (kTrain) {
         __syncthreads();
         auto put = [&](size_t at, float v) { part[at] = begun ? part[at] + v : v; };
         // output layer's gradients, then the top hidden layer's in place of its activations
         if (tid <= nh) {
            float g = 0.0f;
            for (uint32_t r = 0; r < kFusedRows; ++r) g += tid < nh ? dzo[r] * top[r * sh + tid] : dzo[r];
            put(weights(H) + tid, g);
         }
         __syncthreads();
         for (uint32_t i = tid; i < kFusedRows * hp; i += 256) {
            const uint32_t r = i / hp, k = i - r * hp;
            float* a = act + (H - 1) * kFusedRows * sh + r * sh + k;
            *a = *a > 0.0f ? dzo[r] * w_out[k] : 0.0f;  // (k >= nh: the activation is zero)
         }
         __syncthreads();
         for (uint32_t l = H; l-- > 0;) {
            const float* dz = act + l * kFusedRows * sh;
            const float* in = l == 0 ? xin : dz - kFusedRows * sh;
            const uint32_t si = l == 0 ? sx : sh, din = l == 0 ? ni : nh;
            const size_t at = weights(l);
            if (32 * wave < hp) {
               // dW = dZ^T in: 32 units x all inputs, four 32 x 32 tiles over the tile's 32 rows
               f32x16 g[4] = {};
               for (uint32_t s = 0; s < kFusedRows / 2; ++s) {
                  const float d = dz[(2 * s + half) * sh + unit];
#pragma unroll
                  for (uint32_t t = 0; t < 4; ++t) {
                     if (32 * t < din) {
                        // (columns past the padded input read the next row's or the activations'
                        // floats; their products are not stored)
                        const float a = in[(2 * s + half) * si + 32 * t + col];
                        g[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(d, a, g[t], 0, 0, 0);
                     }
                  }
               }
#pragma unroll
               for (uint32_t t = 0; t < 4; ++t) {
#pragma unroll
                  for (uint32_t i = 0; i < 16; ++i) {
                     const uint32_t u = 32 * wave + rowOf(i), k = 32 * t + col;
                     if (u < nh && k < din) put(at + static_cast<size_t>(u) * din + k, g[t][i]);
                  }
               }
               // db: the halves of the wavefront sum 16 rows each
               float b = 0.0f;
               for (uint32_t r = 0; r < kFusedRows / 2; ++r) b += dz[(16 * half + r) * sh + unit];
               b += __shfl_xor(b, 32, 64);
               if (half == 0 && unit < nh) put(at + static_cast<size_t>(din) * nh + unit, b);
            }
            if (l == 0) break;
            f32x16 c = {};
            if (32 * wave < hp) {  // dA = dZ W, through the packed transposed weights
               c = rowsTimesPacked<128>(dz + col * sh, p.packed_t + (static_cast<size_t>(l - 1) * hp + unit) * hp, hp, half, c);
            }
            __syncthreads();  // every wavefront has read the layer below's activations
            if (32 * wave < hp) {
               float* below = act + (l - 1) * kFusedRows * sh;
#pragma unroll
               for (uint32_t i = 0; i < 16; ++i) {
                  float* a = below + rowOf(i) * sh + unit;
                  *a = *a > 0.0f ? c[i] : 0.0f;
               }
            }
            __syncthreads();
         }
         begun = true;
      }
   }
   if constexpr (kTrain) {
      __shared__ float sums[4];
      for (int off = 32; off > 0; off >>= 1) sq += __shfl_xor(sq, off, 64);
      if (lane == 0) sums[wave] = sq;
      __syncthreads();
      if (tid == 0) p.loss_partial[blockIdx.x] = sums[0] + sums[1] + sums[2] + sums[3];
   }
}

// Sums the work-groups' partial gradients (64 parameters per work-group, a quarter of the partials
// per wavefront, four sums in flight per lane) into grad; with kAdam also the update and every copy
// of the new value.  The partials (19 MB at 128 work-groups) come from L2 and the memory-side cache.
template <bool kAdam>
__global__ __launch_bounds__(256) void mlpUpdateKernel(MlpUpdate u) {
   __shared__ float sums[4][64];
   const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
   const uint32_t i = blockIdx.x * 64 + lane;
   float s[4] = {};
   if (i < u.n_params) {
      uint32_t g = wave;
      for (; g + 12 < u.n_partials; g += 16) {
#pragma unroll
         for (uint32_t k = 0; k < 4; ++k) s[k] += u.partial[static_cast<size_t>(g + 4 * k) * u.n_params + i];
      }
      for (; g < u.n_partials; g += 4) s[0] += u.partial[static_cast<size_t>(g) * u.n_params + i];
   }
   sums[wave][lane] = (s[0] + s[1]) + (s[2] + s[3]);
   __syncthreads();
   if (wave == 1 && blockIdx.x == 0) {
      float q = 0.0f;
      for (uint32_t g = lane; g < u.n_partials; g += 64) q += u.loss_partial[g];
      for (int off = 32; off > 0; off >>= 1) q += __shfl_xor(q, off, 64);
      if (lane == 0) *u.loss = q;
   }
   if (wave != 0 || i >= u.n_params) return;
   const float gi = (sums[0][lane] + sums[1][lane]) + (sums[2][lane] + sums[3][lane]);
   if constexpr (!kAdam) {
      u.grad[i] = gi;
   } else {
      const float a = u.b1 * u.m1[i] + (1.0f - u.b1) * gi;
      const float b = u.b2 * u.m2[i] + (1.0f - u.b2) * gi * gi;
      u.m1[i] = a;
      u.m2[i] = b;
      const float v = u.master[i] - u.lr * (a / u.c1) / (sqrtf(b / u.c2) + u.eps);
      u.master[i] = v;
      const __hip_bfloat16 w = __float2bfloat16(v);
      reinterpret_cast<__hip_bfloat16*>(u.w)[i] = w;
      u.eff[i] = __bfloat162float(w);
      const uint32_t at = u.packed_at[i], at_t = u.packed_t_at[i];
      if (at != kNotPacked) reinterpret_cast<__hip_bfloat16*>(u.packed)[at] = w;
      if (at_t != kNotPacked) reinterpret_cast<__hip_bfloat16*>(u.packed_t)[at_t] = w;
   }
}

__global__ void mlpPackKernel(uint32_t n, const __hip_bfloat16* __restrict__ w, const uint32_t* __restrict__ packed_at,
                              const uint32_t* __restrict__ packed_t_at, __hip_bfloat16* __restrict__ packed,
                              __hip_bfloat16* __restrict__ packed_t) {
   const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
   if (i >= n) return;
   if (packed_at[i] != kNotPacked) packed[packed_at[i]] = w[i];
   if (packed_t_at[i] != kNotPacked) packed_t[packed_t_at[i]] = w[i];
}

unsigned blocksFor(long n) { return static_cast<unsigned>((n + 255) / 256); }

}  // namespace

hipError_t mlpGemm(int M, int N, int K, const float* a, long sam, long sak, const float* b, long sbk, long sbn, float* c,
                   long ldc, const float* bias, bool relu, bool accumulate, hipStream_t s) {
   if (M <= 0 || N <= 0) return hipSuccess;
   const dim3 grid((N + kTile - 1) / kTile, (M + kTile - 1) / kTile);
   hipLaunchKernelGGL(gemmKernel<float>, grid, dim3(256), 0, s, M, N, K, a, sam, sak, b, sbk, sbn, c, ldc, bias,
                      relu ? 1 : 0, accumulate ? 1 : 0);
   return hipGetLastError();
}

hipError_t mlpGemmBf16(int M, int N, int K, const float* a, long sam, long sak, const void* b, long sbk, long sbn,
                       float* c, long ldc, const float* bias, bool relu, bool accumulate, hipStream_t s) {
   if (M <= 0 || N <= 0) return hipSuccess;
   const dim3 grid((N + kTile - 1) / kTile, (M + kTile - 1) / kTile);
   hipLaunchKernelGGL(gemmKernel<__hip_bfloat16>, grid, dim3(256), 0, s, M, N, K, a, sam, sak,
                      static_cast<const __hip_bfloat16*>(b), sbk, sbn, c, ldc, bias, relu ? 1 : 0, accumulate ? 1 : 0);
   return hipGetLastError();
}

hipError_t mlpOutputGrad(int n, const float* z, const float* y, float* dz, float* loss, hipStream_t s) {
   if (n <= 0) return hipSuccess;
   hipLaunchKernelGGL(outputGradKernel, dim3(blocksFor(n)), dim3(256), 0, s, n, z, y, dz, loss);
   return hipGetLastError();
}

hipError_t mlpReluGrad(long count, const float* z, float* dz, hipStream_t s) {
   if (count <= 0) return hipSuccess;
   hipLaunchKernelGGL(reluGradKernel, dim3(blocksFor(count)), dim3(256), 0, s, count, z, dz);
   return hipGetLastError();
}

hipError_t mlpColumnSum(int rows, int cols, const float* dz, float* db, hipStream_t s) {
   if (cols <= 0) return hipSuccess;
   hipLaunchKernelGGL(columnSumKernel, dim3(cols), dim3(256), 0, s, rows, cols, dz, db);
   return hipGetLastError();
}

hipError_t mlpAdam(long n, float* master, void* w, const float* g, float* m1, float* m2, float lr, float b1, float b2,
                   float eps, float c1, float c2, hipStream_t s) {
   if (n <= 0) return hipSuccess;
   hipLaunchKernelGGL(adamKernel, dim3(blocksFor(n)), dim3(256), 0, s, n, master, static_cast<__hip_bfloat16*>(w), g, m1,
                      m2, lr, b1, b2, eps, c1, c2);
   return hipGetLastError();
}

hipError_t mlpToBf16(long n, const float* src, void* dst, hipStream_t s) {
   if (n <= 0) return hipSuccess;
   hipLaunchKernelGGL(toBf16Kernel, dim3(blocksFor(n)), dim3(256), 0, s, n, src, static_cast<__hip_bfloat16*>(dst));
   return hipGetLastError();
}

hipError_t mlpFromBf16(long n, const void* src, float* dst, hipStream_t s) {
   if (n <= 0) return hipSuccess;
   hipLaunchKernelGGL(fromBf16Kernel, dim3(blocksFor(n)), dim3(256), 0, s, n, static_cast<const __hip_bfloat16*>(src), dst);
   return hipGetLastError();
}

size_t mlpFusedLdsBytes(uint32_t in_pad, uint32_t hidden_pad, uint32_t n_hidden_layers) {
   return 4ULL * kFusedRows * (in_pad + kFusedPad + static_cast<size_t>(n_hidden_layers) * (hidden_pad + kFusedPad) + 1);
}

uint32_t mlpFusedGroups(uint32_t n, uint32_t max_groups) {
   return std::min(n / kFusedRows + (n % kFusedRows != 0), max_groups);
}

hipError_t mlpFusedConfigure(size_t lds_bytes) {
   const hipError_t err = hipFuncSetAttribute(reinterpret_cast<const void*>(&mlpFusedKernel<false>),
                                              hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds_bytes));
   if (err != hipSuccess) return err;
   return hipFuncSetAttribute(reinterpret_cast<const void*>(&mlpFusedKernel<true>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds_bytes));
}

hipError_t mlpFusedPass(const MlpFused& p, bool train, uint32_t groups, hipStream_t s) {
   if (p.n == 0 || groups == 0) return hipSuccess;
   const size_t lds = mlpFusedLdsBytes(p.in_pad, p.hidden_pad, p.n_hidden_layers);
   if (train) {
      hipLaunchKernelGGL(mlpFusedKernel<true>, dim3(groups), dim3(256), lds, s, p);
   } else {
      hipLaunchKernelGGL(mlpFusedKernel<false>, dim3(groups), dim3(256), lds, s, p);
   }
   return hipGetLastError();
}

hipError_t mlpUpdate(const MlpUpdate& u, bool adam, hipStream_t s) {
   if (u.n_params == 0) return hipSuccess;
   const dim3 grid((u.n_params + 63) / 64);
   if (adam) {
      hipLaunchKernelGGL(mlpUpdateKernel<true>, grid, dim3(256), 0, s, u);
   } else {
      hipLaunchKernelGGL(mlpUpdateKernel<false>, grid, dim3(256), 0, s, u);
   }
   return hipGetLastError();
}

hipError_t mlpPack(uint32_t n, const void* w, const uint32_t* packed_at, const uint32_t* packed_t_at, void* packed,
                   void* packed_t, hipStream_t s) {
   if (n == 0) return hipSuccess;
   hipLaunchKernelGGL(mlpPackKernel, dim3(blocksFor(n)), dim3(256), 0, s, n, static_cast<const __hip_bfloat16*>(w),
                      packed_at, packed_t_at, static_cast<__hip_bfloat16*>(packed), static_cast<__hip_bfloat16*>(packed_t));
   return hipGetLastError();
}

}  // namespace rdb
