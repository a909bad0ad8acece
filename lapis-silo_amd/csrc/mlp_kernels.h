// Launch wrappers of the estimator's kernels (mlp.hip).  Row-major float matrices; `b` operands of
// the *Bf16 variant are BF16 parameter matrices.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

namespace rdb {

// ---- fused passes (networks of at most kFusedMaxWidth inputs and hidden units) ------------------------
constexpr uint32_t kFusedMaxWidth = 128;
constexpr uint32_t kFusedMaxGroups = 256;  // work-groups of a pass (partial gradients): one per CU
constexpr uint32_t kNotPacked = 0xFFFFFFFFu;

// Parameters flat as the estimator holds them (per layer W out x in, then b).  Packed weights: BF16,
// zero-padded: layer 0 as hidden_pad x in_pad, hidden layers l >= 1 as hidden_pad x hidden_pad each;
// packed_t the hidden layers l >= 1 transposed.  in_pad is a multiple of 16, hidden_pad of 32.
struct MlpFused {
   const float* x = nullptr;       // n x n_in
   const float* y = nullptr;       // targets (training)
   uint32_t n = 0, n_in = 0, n_hidden = 0, n_hidden_layers = 0;
   uint32_t in_pad = 0, hidden_pad = 0;
   uint32_t n_params = 0;
   const uint16_t* packed = nullptr;
   const uint16_t* packed_t = nullptr;
   const float* eff = nullptr;     // the BF16 parameters as float (biases and the output layer)
   float* out = nullptr;           // estimates (forward only)
   float* partial = nullptr;       // per work-group n_params gradients (training)
   float* loss_partial = nullptr;  // per work-group sum of squared errors (training)
};

struct MlpUpdate {
   uint32_t n_params = 0, n_partials = 0;
   const float* partial = nullptr;
   const float* loss_partial = nullptr;
   float* loss = nullptr;  // receives the sum of squared errors
   float* grad = nullptr;  // without Adam: the summed gradients
   // with Adam
   float* master = nullptr;
   float* m1 = nullptr;
   float* m2 = nullptr;
   float* eff = nullptr;
   uint16_t* w = nullptr;         // BF16
   uint16_t* packed = nullptr;    // BF16
   uint16_t* packed_t = nullptr;  // BF16
   const uint32_t* packed_at = nullptr;    // parameter -> its place in packed / packed_t, or kNotPacked
   const uint32_t* packed_t_at = nullptr;
   float lr = 0, b1 = 0, b2 = 0, eps = 0, c1 = 1, c2 = 1;
};

size_t mlpFusedLdsBytes(uint32_t in_pad, uint32_t hidden_pad, uint32_t n_hidden_layers);
hipError_t mlpFusedConfigure(size_t lds_bytes);
uint32_t mlpFusedGroups(uint32_t n, uint32_t max_groups);
hipError_t mlpFusedPass(const MlpFused& p, bool train, uint32_t groups, hipStream_t s);
hipError_t mlpUpdate(const MlpUpdate& u, bool adam, hipStream_t s);
hipError_t mlpPack(uint32_t n, const void* w, const uint32_t* packed_at, const uint32_t* packed_t_at, void* packed,
                   void* packed_t, hipStream_t s);

// ---- generic passes -------------------------------------------------------------------------------------

// C[m, n] (+)= sum_k A(m, k) B(k, n) (+ bias[n]) (relu); A(m, k) = a[m * sam + k * sak],
// B(k, n) = b[k * sbk + n * sbn].
hipError_t mlpGemm(int M, int N, int K, const float* a, long sam, long sak, const float* b, long sbk, long sbn, float* c,
                   long ldc, const float* bias, bool relu, bool accumulate, hipStream_t s);
hipError_t mlpGemmBf16(int M, int N, int K, const float* a, long sam, long sak, const void* b, long sbk, long sbn,
                       float* c, long ldc, const float* bias, bool relu, bool accumulate, hipStream_t s);
// dz = 2 (z - y) / n; *loss += sum (z - y)^2
hipError_t mlpOutputGrad(int n, const float* z, const float* y, float* dz, float* loss, hipStream_t s);
hipError_t mlpReluGrad(long count, const float* z, float* dz, hipStream_t s);
hipError_t mlpColumnSum(int rows, int cols, const float* dz, float* db, hipStream_t s);
hipError_t mlpAdam(long n, float* master, void* w, const float* g, float* m1, float* m2, float lr, float b1, float b2,
                   float eps, float c1, float c2, hipStream_t s);
hipError_t mlpToBf16(long n, const float* src, void* dst, hipStream_t s);
hipError_t mlpFromBf16(long n, const void* src, float* dst, hipStream_t s);

}  // namespace rdb
