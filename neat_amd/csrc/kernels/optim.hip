// Adam step for the grid and decoder parameters: the update of torch::optim::Adam as the reference runs it
// (geometry.h:66-88 OptimizerStep; param groups geometry_ex_ex.cpp:40-49 and geometry.cpp:90-97), in one pass over
// param / grad / exp_avg / exp_avg_sq. Purely HBM-bound: 16 B read + 12 B written per parameter (20 B more read and
// nothing more written with weight decay off).
//   exp_avg    = beta1 exp_avg + (1 - beta1) grad
//   exp_avg_sq = beta2 exp_avg_sq + (1 - beta2) grad^2
//   param     -= lr / (1 - beta1^step) * exp_avg / (sqrt(exp_avg_sq) / sqrt(1 - beta2^step) + eps)
#include <cmath>

#include "common.hpp"

namespace neat
{
namespace
{

struct AdamArgs
{
    float lr_bc1;     // lr / (1 - beta1^step)
    float bc2_sqrt;   // sqrt(1 - beta2^step)
    float beta1, one_minus_beta1;
    float beta2, one_minus_beta2;
    float eps, weight_decay;
};

__device__ __forceinline__ void adam_one(float& p, float g, float& m, float& v, const AdamArgs& a)
{
    if (a.weight_decay != 0.f) g = g + p * a.weight_decay;
    m = m * a.beta1 + g * a.one_minus_beta1;
    v = v * a.beta2 + (g * g) * a.one_minus_beta2;
    const float denom = sqrtf(v) / a.bc2_sqrt + a.eps;
    p = p - a.lr_bc1 * (m / denom);
}

typedef float f32x4 __attribute__((ext_vector_type(4)));

template <bool kStream>
__device__ __forceinline__ f32x4 load4(const float* p)
{
    const f32x4* q = reinterpret_cast<const f32x4*>(p);
    return kStream ? __builtin_nontemporal_load(q) : *q;
}

template <bool kStream>
__device__ __forceinline__ void store4(float* p, f32x4 v)
{
    f32x4* q = reinterpret_cast<f32x4*>(p);
    if (kStream)
        __builtin_nontemporal_store(v, q);
    else
        *q = v;
}

// Four parameters per thread, one visit each (every block's loads are independent of the others': a fixed number of
// blocks striding over the arrays kept fewer of them in flight). kStream: the arrays are larger than the caches, so
// nothing is kept there. Bound by HBM; 161 M parameters (28 B each): 0.96 to 1.06 ms with 8192 striding blocks, 0.83 ms
// with one visit per thread, 0.76 ms (5.9 TB/s) streaming as well.
template <bool kStream>
__global__ void __launch_bounds__(256) k_adam(float* __restrict__ p, const float* __restrict__ g, float* __restrict__ m,
                                              float* __restrict__ v, int64_t n, AdamArgs a)
{
    const int64_t i = 4 * ((int64_t)blockIdx.x * blockDim.x + threadIdx.x);
    if (i + 4 <= n)
    {
        f32x4 pp = load4<kStream>(p + i), gg = load4<kStream>(g + i);
        f32x4 mm = load4<kStream>(m + i), vv = load4<kStream>(v + i);
#pragma unroll
        for (int k = 0; k < 4; ++k)
        {
            float pk = pp[k], mk = mm[k], vk = vv[k];
            adam_one(pk, gg[k], mk, vk, a);
            pp[k] = pk;
            mm[k] = mk;
            vv[k] = vk;
        }
        store4<kStream>(p + i, pp);
        store4<kStream>(m + i, mm);
        store4<kStream>(v + i, vv);
        return;
    }
    for (int64_t j = i; j < n; ++j) adam_one(p[j], g[j], m[j], v[j], a);
}

// the last-level cache of the card
constexpr int64_t kCacheBytes = (int64_t)256 << 20;
constexpr int64_t kAdamLaunch = (int64_t)1 << 33;  // parameters of a launch, at most

}  // namespace
}  // namespace neat

using namespace neat;

extern "C" int neat_adam_step(neat_stream_t stream, float* param, const float* grad, float* exp_avg,
                              float* exp_avg_sq, int64_t n, double lr, double beta1, double beta2, double eps,
                              double weight_decay, int64_t step)
{
    NEAT_REQUIRE(n >= 0 && step >= 1, "neat_adam_step: bad sizes (n %lld, step %lld)", (long long)n, (long long)step);
    if (n == 0) return NEAT_OK;
    NEAT_REQUIRE(param && grad && exp_avg && exp_avg_sq, "neat_adam_step: null pointer");
    const uintptr_t mis = reinterpret_cast<uintptr_t>(param) | reinterpret_cast<uintptr_t>(grad) |
                          reinterpret_cast<uintptr_t>(exp_avg) | reinterpret_cast<uintptr_t>(exp_avg_sq);
    NEAT_REQUIRE((mis & 15) == 0, "neat_adam_step: buffers must be 16-byte aligned");
    NEAT_REQUIRE(beta1 >= 0 && beta1 < 1 && beta2 >= 0 && beta2 < 1 && eps >= 0 && lr >= 0,
                 "neat_adam_step: bad hyper-parameters");
    AdamArgs a;
    const double bc1 = 1.0 - std::pow(beta1, (double)step);
    const double bc2 = 1.0 - std::pow(beta2, (double)step);
    a.lr_bc1          = (float)(lr / bc1);
    a.bc2_sqrt        = (float)std::sqrt(bc2);
    a.beta1           = (float)beta1;
    a.one_minus_beta1 = (float)(1.0 - beta1);
    a.beta2           = (float)beta2;
    a.one_minus_beta2 = (float)(1.0 - beta2);
    a.eps             = (float)eps;
    a.weight_decay    = (float)weight_decay;
    // a launch holds fewer than 2^32 threads, i.e. 2^34 parameters
    for (int64_t i = 0; i < n; i += kAdamLaunch)
    {
        const int64_t m       = std::min(n - i, kAdamLaunch);
        const unsigned blocks = grid_for((m + 3) / 4, 256);
        if (16 * n > kCacheBytes)
            k_adam<true><<<blocks, 256, 0, as_stream(stream)>>>(param + i, grad + i, exp_avg + i, exp_avg_sq + i, m, a);
        else
            k_adam<false><<<blocks, 256, 0, as_stream(stream)>>>(param + i, grad + i, exp_avg + i, exp_avg_sq + i, m, a);
        NEAT_LAUNCHED();
    }
    return NEAT_OK;
}
