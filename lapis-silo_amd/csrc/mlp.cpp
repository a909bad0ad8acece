// Host side of the planner's estimator (see mlp.h).
#include "mlp.h"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <numeric>
#include <random>

#include "mlp_kernels.h"

namespace rdb {

namespace {
constexpr float kAdamB1 = 0.9f, kAdamB2 = 0.999f, kAdamEps = 1e-8f;
}

Mlp::Mlp(Context* c, uint32_t n_in, uint32_t n_hidden, uint32_t n_hidden_layers, uint64_t seed) : ctx(c) {
   if (n_in == 0 || n_hidden == 0 || n_hidden_layers == 0 || n_in > 4096 || n_hidden > 4096 || n_hidden_layers > 16) {
      fail(RDB_EINVAL, "estimator shape out of range");
   }
   dims.push_back(n_in);
   for (uint32_t l = 0; l < n_hidden_layers; ++l) dims.push_back(n_hidden);
   dims.push_back(1);
   for (size_t l = 0; l + 1 < dims.size(); ++l) {
      w_off.push_back(n_params);
      n_params += static_cast<size_t>(dims[l]) * dims[l + 1];
      b_off.push_back(n_params);
      n_params += dims[l + 1];
   }
   // He-uniform weights, zero biases
   std::vector<float> p(n_params, 0.0f);
   std::mt19937_64 rng(seed);
   for (size_t l = 0; l + 1 < dims.size(); ++l) {
      const float a = std::sqrt(6.0f / static_cast<float>(dims[l]));
      std::uniform_real_distribution<float> u(-a, a);
      for (size_t k = 0; k < static_cast<size_t>(dims[l]) * dims[l + 1]; ++k) p[w_off[l] + k] = u(rng);
   }
   master = DeviceBuffer(n_params * 4);
   bf16 = DeviceBuffer(n_params * 2);
   eff = DeviceBuffer(n_params * 4);
   grad = DeviceBuffer(n_params * 4);
   m1 = DeviceBuffer(n_params * 4);
   m2 = DeviceBuffer(n_params * 4);
   loss = DeviceBuffer(16);
   setupFused();
   setParameters(p.data());
}

// The fused passes hold a tile of rows in LDS through every layer: networks of up to 128 inputs and
// hidden units whose layers fit the LDS of a work-group.  Wider ones take the generic passes.
void Mlp::setupFused() {
   const uint32_t n_in = dims[0], nh = dims[1], H = static_cast<uint32_t>(dims.size()) - 2;
   if (n_in > kFusedMaxWidth || nh > kFusedMaxWidth) return;
   const uint32_t ip = (n_in + 15) / 16 * 16, hp = (nh + 31) / 32 * 32;
   const size_t lds = mlpFusedLdsBytes(ip, hp, H);
   if (lds > ctx->max_lds_bytes) return;
   if (lds > 64 * 1024 && mlpFusedConfigure(ctx->max_lds_bytes) != hipSuccess) {
      (void)hipGetLastError();
      return;
   }
   const size_t n_packed = static_cast<size_t>(hp) * ip + static_cast<size_t>(H - 1) * hp * hp;
   const size_t n_packed_t = static_cast<size_t>(H - 1) * hp * hp;
   std::vector<uint32_t> at(n_params, kNotPacked), at_t(n_params, kNotPacked);
   for (uint32_t l = 0; l < H; ++l) {
      const uint32_t din = dims[l];
      for (uint32_t o = 0; o < nh; ++o) {
         for (uint32_t k = 0; k < din; ++k) {
            const size_t i = w_off[l] + static_cast<size_t>(o) * din + k;
            if (l == 0) {
               at[i] = o * ip + k;
            } else {
               at[i] = hp * ip + ((l - 1) * hp + o) * hp + k;
               at_t[i] = ((l - 1) * hp + k) * hp + o;
            }
         }
      }
   }
   packed = DeviceBuffer(n_packed * 2);
   packed_t = DeviceBuffer(std::max<size_t>(n_packed_t * 2, 16));
   packed_at = DeviceBuffer(at.data(), at.size() * 4);
   packed_t_at = DeviceBuffer(at_t.data(), at_t.size() * 4);
   // the padding stays zero
   hipCheck(hipMemsetAsync(packed.as<void>(), 0, packed.bytes(), ctx->stream), "clear packed weights");
   hipCheck(hipMemsetAsync(packed_t.as<void>(), 0, packed_t.bytes(), ctx->stream), "clear packed weights");
   in_pad = ip;
   hidden_pad = hp;
   forward_groups = static_cast<uint32_t>(ctx->cu_count) *
                    std::max<uint32_t>(1, static_cast<uint32_t>(std::min<size_t>(4, ctx->max_lds_bytes / lds)));
}

void Mlp::refreshCopies() {
   hipCheck(mlpToBf16(static_cast<long>(n_params), master.as<float>(), bf16.as<void>(), ctx->stream), "estimator bf16");
   hipCheck(mlpFromBf16(static_cast<long>(n_params), bf16.as<void>(), eff.as<float>(), ctx->stream), "estimator f32");
   if (fused()) {
      hipCheck(mlpPack(static_cast<uint32_t>(n_params), bf16.as<void>(), packed_at.as<uint32_t>(),
                       packed_t_at.as<uint32_t>(), packed.as<void>(), packed_t.as<void>(), ctx->stream),
               "estimator packed weights");
   }
}

void Mlp::setParameters(const float* p) {
   hipCheck(hipMemcpyAsync(master.as<void>(), p, n_params * 4, hipMemcpyHostToDevice, ctx->stream), "upload parameters");
   hipCheck(hipMemsetAsync(m1.as<void>(), 0, n_params * 4, ctx->stream), "clear moments");
   hipCheck(hipMemsetAsync(m2.as<void>(), 0, n_params * 4, ctx->stream), "clear moments");
   adam_step = 0;
   refreshCopies();
   hipCheck(hipStreamSynchronize(ctx->stream), "synchronize");
}

std::vector<float> Mlp::parameters() const {
   std::vector<float> p(n_params);
   hipCheck(hipMemcpyAsync(p.data(), eff.as<void>(), n_params * 4, hipMemcpyDeviceToHost, ctx->stream), "copy parameters");
   hipCheck(hipStreamSynchronize(ctx->stream), "synchronize");
   return p;
}

void Mlp::reserve(size_t n) {
   if (n <= rows_capacity) return;
   const size_t cap = std::max<size_t>(n, 1024);
   size_t width = 0;
   for (size_t l = 1; l < dims.size(); ++l) width += dims[l];
   const uint32_t widest = *std::max_element(dims.begin(), dims.end());
   x = DeviceBuffer(cap * dims[0] * 4);
   y = DeviceBuffer(cap * 4);
   rows_capacity = cap;
   if (fused()) {
      acts = DeviceBuffer(cap * 4);  // the estimates
      return;
   }
   acts = DeviceBuffer(cap * width * 4);
   dz0 = DeviceBuffer(cap * widest * 4);
   dz1 = DeviceBuffer(cap * widest * 4);
}

float* Mlp::estimates() const { return fused() ? acts.as<float>() : act(dims.size() - 2); }

float* Mlp::act(size_t layer) const {
   size_t off = 0;
   for (size_t l = 0; l < layer; ++l) off += dims[l + 1];
   return acts.as<float>() + off * rows_capacity;
}

MlpFused Mlp::fusedPass(const float* x_dev, size_t n) const {
   MlpFused p;
   p.x = x_dev;
   p.n = static_cast<uint32_t>(n);
   p.n_in = dims[0];
   p.n_hidden = dims[1];
   p.n_hidden_layers = static_cast<uint32_t>(dims.size()) - 2;
   p.in_pad = in_pad;
   p.hidden_pad = hidden_pad;
   p.n_params = static_cast<uint32_t>(n_params);
   p.packed = packed.as<uint16_t>();
   p.packed_t = packed_t.as<uint16_t>();
   p.eff = eff.as<float>();
   return p;
}

void Mlp::fusedTrainPass(const float* x_dev, const float* y_dev, size_t n, float* loss_dev, const float* adam_lr) {
   const uint32_t groups = mlpFusedGroups(static_cast<uint32_t>(n), kFusedMaxGroups);
   const size_t need = groups * (n_params + 1) * 4;
   if (partial.bytes() < need) {
      hipCheck(hipStreamSynchronize(ctx->stream), "synchronize");
      partial = DeviceBuffer(need);
   }
   MlpFused p = fusedPass(x_dev, n);
   p.y = y_dev;
   p.partial = partial.as<float>();
   p.loss_partial = partial.as<float>() + groups * n_params;
   hipCheck(mlpFusedPass(p, true, groups, ctx->stream), "estimator training pass");
   MlpUpdate u;
   u.n_params = p.n_params;
   u.n_partials = groups;
   u.partial = p.partial;
   u.loss_partial = p.loss_partial;
   u.loss = loss_dev;
   u.grad = grad.as<float>();
   if (adam_lr != nullptr) {
      ++adam_step;
      u.master = master.as<float>();
      u.m1 = m1.as<float>();
      u.m2 = m2.as<float>();
      u.eff = eff.as<float>();
      u.w = bf16.as<uint16_t>();
      u.packed = packed.as<uint16_t>();
      u.packed_t = packed_t.as<uint16_t>();
      u.packed_at = packed_at.as<uint32_t>();
      u.packed_t_at = packed_t_at.as<uint32_t>();
      u.lr = *adam_lr;
      u.b1 = kAdamB1;
      u.b2 = kAdamB2;
      u.eps = kAdamEps;
      u.c1 = 1.0f - std::pow(kAdamB1, static_cast<float>(adam_step));
      u.c2 = 1.0f - std::pow(kAdamB2, static_cast<float>(adam_step));
   }
   hipCheck(mlpUpdate(u, adam_lr != nullptr, ctx->stream), "estimator update");
}

void Mlp::forwardDevice(const float* x_dev, size_t n) {
   if (fused()) {
      MlpFused p = fusedPass(x_dev, n);
      p.out = estimates();
      hipCheck(mlpFusedPass(p, false, mlpFusedGroups(p.n, forward_groups), ctx->stream), "estimator forward");
      return;
   }
   const size_t L = dims.size() - 1;
   const float* in = x_dev;
   for (size_t l = 0; l < L; ++l) {
      const long din = dims[l], dout = dims[l + 1];
      hipCheck(mlpGemmBf16(static_cast<int>(n), static_cast<int>(dout), static_cast<int>(din), in, din, 1,
                           bf16.as<uint16_t>() + w_off[l], 1, din, act(l), dout, eff.as<float>() + b_off[l], l + 1 < L,
                           false, ctx->stream),
               "estimator forward");
      in = act(l);
   }
}

float Mlp::backwardDevice(const float* x_dev, const float* y_dev, size_t n) {
   const size_t L = dims.size() - 1;
   hipCheck(hipMemsetAsync(loss.as<void>(), 0, 4, ctx->stream), "clear loss");
   float* dz = dz0.as<float>();
   float* dz_prev = dz1.as<float>();
   hipCheck(mlpOutputGrad(static_cast<int>(n), act(L - 1), y_dev, dz, loss.as<float>(), ctx->stream), "output gradient");
   for (size_t l = L; l-- > 0;) {
      const long din = dims[l], dout = dims[l + 1];
      const float* in = l == 0 ? x_dev : act(l - 1);
      // dW = dZ^T in
      hipCheck(mlpGemm(static_cast<int>(dout), static_cast<int>(din), static_cast<int>(n), dz, 1, dout, in, din, 1,
                       grad.as<float>() + w_off[l], din, nullptr, false, false, ctx->stream),
               "weight gradient");
      hipCheck(mlpColumnSum(static_cast<int>(n), static_cast<int>(dout), dz, grad.as<float>() + b_off[l], ctx->stream),
               "bias gradient");
      if (l == 0) break;
      // dA = dZ W, then the relu derivative of the layer below
      hipCheck(mlpGemmBf16(static_cast<int>(n), static_cast<int>(din), static_cast<int>(dout), dz, dout, 1,
                           bf16.as<uint16_t>() + w_off[l], din, 1, dz_prev, din, nullptr, false, false, ctx->stream),
               "activation gradient");
      hipCheck(mlpReluGrad(static_cast<long>(n) * din, act(l - 1), dz_prev, ctx->stream), "relu gradient");
      std::swap(dz, dz_prev);
   }
   float sq = 0.0f;
   hipCheck(hipMemcpyAsync(&sq, loss.as<void>(), 4, hipMemcpyDeviceToHost, ctx->stream), "copy loss");
   hipCheck(hipStreamSynchronize(ctx->stream), "synchronize");
   return sq;
}

void Mlp::predict(const float* x_host, size_t n, float* y_host) {
   if (n == 0) return;
   reserve(n);
   hipCheck(hipMemcpyAsync(x.as<void>(), x_host, n * dims[0] * 4, hipMemcpyHostToDevice, ctx->stream), "upload features");
   forwardDevice(x.as<float>(), n);
   hipCheck(hipMemcpyAsync(y_host, estimates(), n * 4, hipMemcpyDeviceToHost, ctx->stream), "copy estimates");
   hipCheck(hipStreamSynchronize(ctx->stream), "synchronize");
}

float Mlp::gradients(const float* x_host, const float* y_host, size_t n, float* grads_host) {
   if (n == 0) fail(RDB_EINVAL, "no rows");
   reserve(n);
   hipCheck(hipMemcpyAsync(x.as<void>(), x_host, n * dims[0] * 4, hipMemcpyHostToDevice, ctx->stream), "upload features");
   hipCheck(hipMemcpyAsync(y.as<void>(), y_host, n * 4, hipMemcpyHostToDevice, ctx->stream), "upload targets");
   float sq = 0.0f;
   if (fused()) {
      fusedTrainPass(x.as<float>(), y.as<float>(), n, loss.as<float>(), nullptr);
      hipCheck(hipMemcpyAsync(&sq, loss.as<void>(), 4, hipMemcpyDeviceToHost, ctx->stream), "copy loss");
   } else {
      forwardDevice(x.as<float>(), n);
      sq = backwardDevice(x.as<float>(), y.as<float>(), n);
   }
   hipCheck(hipMemcpyAsync(grads_host, grad.as<void>(), n_params * 4, hipMemcpyDeviceToHost, ctx->stream), "copy gradients");
   hipCheck(hipStreamSynchronize(ctx->stream), "synchronize");
   return sq / static_cast<float>(n);
}

float Mlp::train(const float* x_host, const float* y_host, size_t n, uint32_t epochs, uint32_t batch, float lr,
                 uint64_t seed) {
   if (n == 0 || batch == 0) fail(RDB_EINVAL, "no rows");
   const size_t d = dims[0];
   // the whole (shuffled) set is resident; minibatches are slices of it
   if (train_x.bytes() < n * d * 4) train_x = DeviceBuffer(n * d * 4);
   if (train_y.bytes() < n * 4) train_y = DeviceBuffer(n * 4);
   const DeviceBuffer &xs = train_x, &ys = train_y;
   const size_t n_batches = (n + batch - 1) / batch;
   if (fused() && losses.bytes() < n_batches * 4) losses = DeviceBuffer(n_batches * 4);
   std::vector<float> batch_loss(n_batches);
   std::vector<size_t> perm(n);
   std::iota(perm.begin(), perm.end(), size_t{0});
   std::mt19937_64 rng(seed);
   std::vector<float> xb(n * d), yb(n);
   reserve(std::min<size_t>(batch, n));
   constexpr float b1 = kAdamB1, b2 = kAdamB2, eps = kAdamEps;
   float last = 0.0f;
   for (uint32_t e = 0; e < epochs; ++e) {
      std::shuffle(perm.begin(), perm.end(), rng);
      for (size_t i = 0; i < n; ++i) {
         std::memcpy(xb.data() + i * d, x_host + perm[i] * d, d * 4);
         yb[i] = y_host[perm[i]];
      }
      hipCheck(hipMemcpyAsync(xs.as<void>(), xb.data(), n * d * 4, hipMemcpyHostToDevice, ctx->stream), "upload features");
      hipCheck(hipMemcpyAsync(ys.as<void>(), yb.data(), n * 4, hipMemcpyHostToDevice, ctx->stream), "upload targets");
      double sum = 0.0;
      if (fused()) {
         // the minibatches' losses stay on the device until the epoch's end: no wait between updates
         for (size_t b = 0; b < n_batches; ++b) {
            const size_t s = b * batch;
            fusedTrainPass(xs.as<float>() + s * d, ys.as<float>() + s, std::min<size_t>(batch, n - s),
                           losses.as<float>() + b, &lr);
         }
         hipCheck(hipMemcpyAsync(batch_loss.data(), losses.as<void>(), n_batches * 4, hipMemcpyDeviceToHost, ctx->stream),
                  "copy losses");
         hipCheck(hipStreamSynchronize(ctx->stream), "synchronize");
         for (float l : batch_loss) sum += l;
         last = static_cast<float>(sum / static_cast<double>(n));
         continue;
      }
      for (size_t s = 0; s < n; s += batch) {
         const size_t m = std::min<size_t>(batch, n - s);
         forwardDevice(xs.as<float>() + s * d, m);
         sum += backwardDevice(xs.as<float>() + s * d, ys.as<float>() + s, m);
         ++adam_step;
         const float c1 = 1.0f - std::pow(b1, static_cast<float>(adam_step));
         const float c2 = 1.0f - std::pow(b2, static_cast<float>(adam_step));
         hipCheck(mlpAdam(static_cast<long>(n_params), master.as<float>(), bf16.as<void>(), grad.as<float>(), m1.as<float>(),
                          m2.as<float>(), lr, b1, b2, eps, c1, c2, ctx->stream),
                  "adam");
         hipCheck(mlpFromBf16(static_cast<long>(n_params), bf16.as<void>(), eff.as<float>(), ctx->stream), "estimator f32");
      }
      last = static_cast<float>(sum / static_cast<double>(n));
   }
   hipCheck(hipStreamSynchronize(ctx->stream), "synchronize");
   return last;
}

}  // namespace rdb
