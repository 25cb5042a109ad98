// FP32 decoder backward (8 -> H -> H -> 1, relu) with the gradient products on the BF16 matrix cores, for tiles of 32
// samples per wave.
//
// An FP32 value is the sum of three BF16 values (8 significant bits each), v = p0 + p1 + p2, and a product of two such
// sums has nine exact partial products; v_mfma_f32_32x32x16_bf16 adds them in FP32 at 16 times the rate of
// v_mfma_f32_32x32x2_f32. The backward of a relu decoder needs far fewer than nine:
//   - D2 = dL/dZ2 = (w3 dz) [Z2 > 0] enters as its 0/1 mask, which is one plane: w3 is folded into the transposed
//     hidden-layer weights (and into the rows of the hidden-weight gradient at the end), dz into the other factor.
//   - planes ride in spare rows and columns: dL/dx has 8 of 32 result rows, so the three planes of W0 are rows 0..7,
//     8..15, 16..23 of one operand; the first-layer gradient has 8 of 32 result columns, so the three planes of x are
//     column groups of one operand, the ones that give the bias gradient a column beside them, and the planes of dz
//     three more columns (the hidden bias gradient).
// All nine partial products are taken everywhere, so the only roundings are those of FP32 accumulation.
//
// The pre-activations, forward and recomputed, take the six partial products down to 2^-18 and leave out less than 2^-26
// of each product. The hidden layer's bias is added behind the products, as the plain evaluation does: in front of them
// every one of the sums would be rounded at the bias's size. Error of the output against 64 bits, H = 64, FP32 matrix
// cores / bias in front / behind: random decoder 2.0e-7 / 1.7e-7 / 1.7e-7 (relu), 2.6e-7 / 2.1e-7 / 2.0e-7 (silu);
// biases that cancel the sums to a tenth of their terms 3.0e-6 / 3.2e-6 / 1.6e-6 and 1.2e-6 / 1.7e-6 / 0.8e-6. It costs
// 1 of 57 us for 10^6 rows.
//
// The relu masks of the backward are those of the plain FP32 evaluation (tile_forward_exact: 32x32x2 products and
// their order of additions), up to a margin of 8 roundings. A pre-activation in split form differs from that one by a few
// roundings, so a tile with a unit that close to zero (3 and 9% of the tiles of random decoders with H = 32 and 64) is
// evaluated again in plain FP32: flipping the units within rounding of zero would by itself move the gradient by 3e-4.
// The margin is a measured one, not a bound: over 10^9 units of random decoders the two differed by at most 2.9
// roundings of the largest sum that |x|, |h1| and the weights allow, with biases that cancel the sums to a hundredth by
// 4.8.
//
// In a tile with infinities, NaN or values beyond the planes' range the pre-activations and masks are the plain ones and
// x is split without leaving FP32's range; the gradient products are still taken in planes, which hold what fits FP32
// as w3 W1, h1 dz and dL/dh1 dz: where these overflow, or below 2^-110 (of whose planes the last is lost in BF16's
// denormals), plain FP32 products could do better.
#pragma once

#include "mfma_mlp.hpp"

namespace neat
{

// v = p[0] + p[1] + p[2], each the BF16 rounding of what the ones before it leave
__device__ __forceinline__ void split3(float v, __bf16 (&p)[3])
{
    p[0]          = (__bf16)v;
    const float r = v - (float)p[0];
    p[1]          = (__bf16)r;
    p[2]          = (__bf16)(r - (float)p[1]);
}

// The same for any v: the first plane cut off instead of rounded, so that no finite value becomes an infinite one, and an
// infinity or NaN in it alone.
__device__ __forceinline__ void split3_any(float v, __bf16 (&p)[3])
{
    const bool nan   = v != v, finite = fabsf(v) < INFINITY;
    const uint32_t u = (__float_as_uint(v) & 0xFFFF0000u) | (nan ? 0x400000u : 0u);
    p[0]             = __builtin_bit_cast(__bf16, (unsigned short)(u >> 16));
    const float r    = finite ? v - __uint_as_float(u) : 0.f;
    p[1]             = (__bf16)r;
    p[2]             = (__bf16)(r - (float)p[1]);
}

// the three planes of 8 values as fragments, converted two at a time
__device__ __forceinline__ void split3_frag(const float (&v)[8], bf16x8 (&p)[3])
{
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    u32x4 o[3];
#pragma unroll
    for (int q = 0; q < 4; ++q)
    {
        f32x2 r = {v[2 * q], v[2 * q + 1]};
#pragma unroll
        for (int k = 0; k < 3; ++k)
        {
            const uint32_t u = __builtin_bit_cast(uint32_t, __builtin_convertvector(r, bf16x2));
            o[k][q]          = u;
            if (k < 2)
            {
                r[0] = r[0] - __uint_as_float(u << 16);
                r[1] = r[1] - __uint_as_float(u & 0xFFFF0000u);
            }
        }
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) p[k] = __builtin_bit_cast(bf16x8, o[k]);
}

// Weights of the forward in LDS, as BF16 planes:
//   w1[3][MT][64]          first layer: dst row 32mt + l%32, slots 0..3 and 4..7 the channels 4g..4g+3 (g = l/32) of
//                          planes (0, 0), (1, 1), (0, 2): against x in planes (0, 1), (0, 1), (2, 0) these are the
//                          six partial products down to 2^-18
//   w2[3][MT][MT][2][64]   hidden layer: dst row 32mt + l%32, src row 32ms + crow(8st + j, l/32)
//   vec                    b0, b1, w3 (FP32), b2 at vec[3][0]
//   norm                   largest row sum of |W0|, largest |b0|, the same of W1 and b1 (float bits)
template <int H>
struct WeightLDSSplitFwd
{
    static constexpr int MT = H / 32;
    bf16x8 w1[3][MT][64];
    bf16x8 w2[3][MT][MT][2][64];
    float vec[4][64];
    uint32_t norm[4];
};

// Packed parameter layout as load_weights (C = 8). Ends in a barrier. kRelu (relu decoders only): a unit without any
// weight or bias gets the bias -1, which leaves it as inactive as its pre-activation of exactly zero would; at zero it
// would send every tile of the backward to the plain evaluation. On the trained bench field, most of whose units are
// such: FP32 step of 53.7 M samples 19.0 ms with the zeros, 13.7 ms like this.
template <int H, bool kRelu = false>
__device__ void load_weights_split_fwd(const float* params, WeightLDSSplitFwd<H>& w)
{
    constexpr int MT = H / 32, C = 8;
    const float* W0 = params;
    const float* b0 = W0 + H * C;
    const float* W1 = b0 + H;
    const float* b1 = W1 + H * H;
    const float* W2 = b1 + H;
    const float* b2 = W2 + H;
    if (threadIdx.x < 4) w.norm[threadIdx.x] = 0u;
    __syncthreads();
    // row sums, 8 lanes to a row (blockDim.x is a multiple of 64, so a row's lanes stay together)
    for (int t = threadIdx.x; t < H * 8; t += blockDim.x)
    {
        const int r = t >> 3, q = t & 7;
        float a0 = fabsf(W0[r * C + q]), a1 = 0.f;
#pragma unroll
        for (int k = 0; k < H / 8; ++k) a1 += fabsf(W1[r * H + q * (H / 8) + k]);
#pragma unroll
        for (int off = 4; off >= 1; off >>= 1)
        {
            a0 += __shfl_xor(a0, off);
            a1 += __shfl_xor(a1, off);
        }
        if (q == 0)
        {
            // non-negative floats (and NaN above them) order like their bit patterns
            atomicMax(&w.norm[0], __float_as_uint(a0));
            atomicMax(&w.norm[1], __float_as_uint(fabsf(b0[r])));
            atomicMax(&w.norm[2], __float_as_uint(a1));
            atomicMax(&w.norm[3], __float_as_uint(fabsf(b1[r])));
            w.vec[0][r] = kRelu && a0 == 0.f && b0[r] == 0.f ? -1.f : b0[r];
            w.vec[1][r] = kRelu && a1 == 0.f && b1[r] == 0.f ? -1.f : b1[r];
        }
    }
    for (int t = threadIdx.x; t < MT * 64; t += blockDim.x)
    {
        const int mt = t / 64, l = t % 64, g = l >> 5, r = 32 * mt + (l & 31);
        bf16x8 f[3];
#pragma unroll
        for (int j = 0; j < 4; ++j)
        {
            __bf16 p[3];
            split3(W0[r * C + 4 * g + j], p);
            f[0][j] = f[0][j + 4] = f[2][j] = p[0];
            f[1][j] = f[1][j + 4] = p[1];
            f[2][j + 4]           = p[2];
        }
#pragma unroll
        for (int k = 0; k < 3; ++k) w.w1[k][mt][l] = f[k];
    }
    for (int t = threadIdx.x; t < MT * MT * 2 * 64; t += blockDim.x)
    {
        const int l = t % 64, st = (t / 64) % 2, ms = (t / 128) % MT, mt = t / (128 * MT);
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = W1[(32 * mt + (l & 31)) * H + 32 * ms + crow(st * 8 + j, l >> 5)];
        bf16x8 p[3];
        split3_frag(v, p);
#pragma unroll
        for (int k = 0; k < 3; ++k) w.w2[k][mt][ms][st][l] = p[k];
    }
    for (int t = threadIdx.x; t < 64; t += blockDim.x)
    {
        if (t >= H) w.vec[0][t] = w.vec[1][t] = 0.f;
        w.vec[2][t] = t < H ? W2[t] : 0.f;
        w.vec[3][t] = t == 0 ? b2[0] : 0.f;
    }
    __syncthreads();
}

__device__ __forceinline__ f32x16 mma_bf16(const bf16x8& a, const bf16x8& b, const f32x16& c)
{
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// 16 floats of a per-row vector in accumulator order (rows 32mt + crow(i, g))
__device__ __forceinline__ f32x16 row_vec(const float* v, int mt, int g)
{
    f32x16 r;
#pragma unroll
    for (int q = 0; q < 4; ++q)
    {
        const float4 f = *reinterpret_cast<const float4*>(v + 32 * mt + 8 * q + 4 * g);
        r[4 * q] = f.x; r[4 * q + 1] = f.y; r[4 * q + 2] = f.z; r[4 * q + 3] = f.w;
    }
    return r;
}

// The pre-activations of both hidden layers in the steps of tile_forward_mfma<PrecF32, H>, plain FP32 matrix products, the
// weights read from global memory (row crow(4q, g).. of a fragment are 4 consecutive floats).
template <int H, int ACT>
__device__ __forceinline__ void tile_forward_exact(const float* __restrict__ params, const WeightLDSSplitFwd<H>& w,
                                                   const float (&x4)[4], float beta, f32x16 (&z1)[H / 32],
                                                   f32x16 (&z2)[H / 32])
{
    constexpr int MT = H / 32, C = 8;
    const int l = threadIdx.x & 63, n = l & 31, g = l >> 5;
    const float* W0 = params;
    const float* W1 = params + H * C + H;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
    {
        f32x16 a = {};
#pragma unroll
        for (int s = 0; s < 4; ++s) a = PrecF32::mma1(W0[(32 * mt + n) * C + 4 * g + s], x4[s], a);
        __builtin_amdgcn_sched_barrier(0);
        const f32x16 b = row_vec(w.vec[0], mt, g);
#pragma unroll
        for (int i = 0; i < 16; ++i) a[i] += b[i];
        z1[mt] = a;
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
    {
        f32x16 a = {};
#pragma unroll
        for (int ms = 0; ms < MT; ++ms)
#pragma unroll
            for (int q = 0; q < 4; ++q)
            {
                // rows crow(4q.., g): 4 consecutive floats. One group at a time: hoisted, the loads would spill
                float wv[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) wv[j] = W1[(32 * mt + n) * H + 32 * ms + 8 * q + 4 * g + j];
#pragma unroll
                for (int j = 0; j < 4; ++j) a = PrecF32::mma(wv[j], act_f(ACT, z1[ms][4 * q + j], beta), a);
                __builtin_amdgcn_sched_barrier(0);
            }
        const f32x16 b = row_vec(w.vec[1], mt, g);
#pragma unroll
        for (int i = 0; i < 16; ++i) a[i] += b[i];
        z2[mt] = a;
    }
}

// x in three planes, and the first layer's operands: slots 0..3, 4..7 = planes 0, 1 (xa) and 2, 0 (xb)
struct SplitX
{
    bf16x8 p[3], a, b;
    __device__ explicit SplitX(const float (&x4)[4])
    {
        const float v[8] = {x4[0], x4[1], x4[2], x4[3], 0.f, 0.f, 0.f, 0.f};
        split3_frag(v, p);
#pragma unroll
        for (int j = 0; j < 4; ++j)
        {
            a[j]     = p[0][j];
            a[j + 4] = p[1][j];
            b[j]     = p[2][j];
            b[j + 4] = p[0][j];
        }
    }
    // p for values of any size
    __device__ void split_any(const float (&x4)[4])
    {
#pragma unroll
        for (int j = 0; j < 4; ++j)
        {
            __bf16 q[3];
            split3_any(x4[j], q);
#pragma unroll
            for (int k = 0; k < 3; ++k) p[k][j] = q[k];
        }
    }
};

// first-layer pre-activations of units 32mt + ..
template <int H>
__device__ __forceinline__ f32x16 split_layer1(const WeightLDSSplitFwd<H>& w, const SplitX& x, int mt)
{
    const int l = threadIdx.x & 63;
    f32x16 z    = mma_bf16(w.w1[2][mt][l], x.b, row_vec(w.vec[0], mt, l >> 5));
    z           = mma_bf16(w.w1[1][mt][l], x.a, z);
    return mma_bf16(w.w1[0][mt][l], x.a, z);
}

// the largest |x| of the lane's sample
__device__ __forceinline__ float max_abs_x(const float (&x4)[4])
{
    const float m = fmaxf(fmaxf(fabsf(x4[0]), fabsf(x4[1])), fmaxf(fabsf(x4[2]), fabsf(x4[3])));
    return fmaxf(m, __shfl_xor(m, 32));
}

// Output pre-activation of the lane's sample (x4: its 4 channels), a tile of 32 samples per wave: the products in split
// form, six partial products each, the output layer in FP32. A tile whose inputs or sums could leave the range that
// splits into finite planes (infinities and NaN among them) is evaluated in plain FP32.
template <int H, int ACT>
__device__ __forceinline__ float tile_forward_split(const float* __restrict__ params, const WeightLDSSplitFwd<H>& w,
                                                    const float (&x4)[4], float beta)
{
    constexpr int MT = H / 32;
    const int l = threadIdx.x & 63, g = l >> 5;
    asm volatile("" ::: "memory");  // keeps the weight fragments in LDS: hoisted out of the tile loop they spill
    float part = 0.f;
    {
        const float s1 = fmaf(__uint_as_float(w.norm[0]), max_abs_x(x4), __uint_as_float(w.norm[1]));
        const float s2 = fmaf(__uint_as_float(w.norm[2]), s1, __uint_as_float(w.norm[3]));
        // (fmaxf passes over a NaN in x; the sum does not)
        const bool fine = s1 < 1e30f && s2 < 1e30f && fabsf((x4[0] + x4[1]) + (x4[2] + x4[3])) < 1e30f;
        if (__any(!fine))
        {
            f32x16 z1[MT], z2[MT];
            tile_forward_exact<H, ACT>(params, w, x4, beta, z1, z2);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
            {
                const f32x16 w3 = row_vec(w.vec[2], mt, g);
#pragma unroll
                for (int i = 0; i < 16; ++i) part = fmaf(w3[i], act_f(ACT, z2[mt][i], beta), part);
            }
            return part + __shfl_xor(part, 32) + w.vec[3][0];
        }
    }
    bf16x8 h[MT][2][3];
    {
        const SplitX x(x4);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
        {
            const f32x16 a = split_layer1<H>(w, x, mt);
#pragma unroll
            for (int st = 0; st < 2; ++st)
            {
                float u[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) u[j] = act_f(ACT, a[8 * st + j], beta);
                split3_frag(u, h[mt][st]);
            }
        }
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
    {
        f32x16 a = {};
        // weight plane k against the planes 0..2-k of h, the smallest products first
#pragma unroll
        for (int k = 2; k >= 0; --k)
#pragma unroll
            for (int ms = 0; ms < MT; ++ms)
#pragma unroll
                for (int st = 0; st < 2; ++st)
                {
                    const bf16x8 f = w.w2[k][mt][ms][st][l];
#pragma unroll
                    for (int q = 2 - k; q >= 0; --q) a = mma_bf16(f, h[ms][st][q], a);
                }
        const f32x16 b = row_vec(w.vec[1], mt, g), w3 = row_vec(w.vec[2], mt, g);
#pragma unroll
        for (int i = 0; i < 16; ++i) part = fmaf(w3[i], act_f(ACT, a[i] + b[i], beta), part);
    }
    return part + __shfl_xor(part, 32) + w.vec[3][0];
}

// What the backward adds:
//   w2t[3][MT][MT][2][64]  transposed hidden layer times the output weights: dst = first-layer unit 32mt + l%32,
//                          src = hidden unit 32ms + crow(8st + j, l/32)
//   w1t[MT][2][64]         transposed first layer: row l%32 = 8 plane + channel (rows 24..31 zero), src as above
template <int H>
struct WeightLDSSplit : WeightLDSSplitFwd<H>
{
    static constexpr int MT = H / 32;
    bf16x8 w2t[3][MT][MT][2][64];
    bf16x8 w1t[MT][2][64];
};

// `copy` (LDS, the parameters' size) takes the parameters first, in one pass over global memory: the layouts below read
// them in scattered order, several passes. Ends in a barrier.
template <int H>
__device__ void load_weights_split(const float* __restrict__ params, float* copy, WeightLDSSplit<H>& w)
{
    constexpr int MT = H / 32, C = 8;
    for (int t = threadIdx.x; t < H * C + H + H * H + H + H + 1; t += blockDim.x) copy[t] = params[t];
    __syncthreads();
    const float* W0 = copy;
    const float* W1 = W0 + H * C + H;
    const float* W2 = W1 + H * H + H;
    load_weights_split_fwd<H, true>(copy, w);
    for (int t = threadIdx.x; t < MT * MT * 2 * 64; t += blockDim.x)
    {
        const int l = t % 64, st = (t / 64) % 2, ms = (t / 128) % MT, mt = t / (128 * MT);
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j)
        {
            const int src = 32 * ms + crow(st * 8 + j, l >> 5);
            v[j]          = W1[src * H + 32 * mt + (l & 31)] * W2[src];
        }
        bf16x8 p[3];
        split3_frag(v, p);
#pragma unroll
        for (int k = 0; k < 3; ++k) w.w2t[k][mt][ms][st][l] = p[k];
    }
    for (int t = threadIdx.x; t < MT * 2 * 64; t += blockDim.x)
    {
        const int l = t % 64, st = (t / 64) % 2, ms = t / 128, m = l & 31;
        bf16x8 f = {};
        if (m < 24)
        {
#pragma unroll
            for (int j = 0; j < 8; ++j)
            {
                __bf16 p[3];
                split3(W0[(32 * ms + crow(st * 8 + j, l >> 5)) * C + (m & 7)], p);
                f[j] = m < 8 ? p[0] : (m < 16 ? p[1] : p[2]);
            }
        }
        w.w1t[ms][st][l] = f;
    }
    __syncthreads();
}

// One wave's transpose tiles in LDS: three planes of a 32-row tile. Plane 0 holds, first, the tile T of the columns
// that the first-layer and bias gradients contract with: 0..7, 8..15, 16..23 the planes of x, kTOnes ones, kTDz.. the
// planes of dz.
constexpr int kTOnes = 24, kTDz = 25;
struct SplitStage
{
    unsigned short plane[3][32 * kTrRow];
};

// A wave's running parameter-gradient products, of every other wave with the opposite sign (so that the accumulation's
// rounding down cancels between them): G = [Z2 > 0] (dz h1)^T (the hidden-weight gradient without its row
// factor w3), E (columns as T), and the output layer's: the bias's on every lane of the lower half, the weights' h2 dz
// summed over the tile, one row per lane (transpose_sum).
//
// The output weights' gradient also follows from G, as sum_c W1[r][c] G[r][c] + b1[r] (sum_n [z2[r] > 0] dz), but keeps
// G's roundings at the size of its terms: with biases that cancel the sums over c to a tenth / a hundredth and output
// gradients of one sign (H = 64, 10^6 rows) 1.4e-7 / 8.0e-7 from 64 bits, where the FP32 matrix cores gave 0.7e-7 /
// 0.8e-7 and these sums give 0.6e-7 / 1.2e-7. They take 11 of 191 us there, and 0.45 of 15.0 ms of the projector's FP32
// step of 53.3 M samples.
template <int MT>
struct SplitAcc
{
    f32x16 G[MT][MT];
    f32x16 E[MT];
    float b3, w3, sign;
    __device__ SplitAcc() : b3(0.f), w3(0.f), sign((blockIdx.x + (threadIdx.x >> 6)) & 1 ? -1.f : 1.f)
    {
#pragma unroll
        for (int a = 0; a < MT; ++a)
        {
            E[a] = f32x16{};
#pragma unroll
            for (int b = 0; b < MT; ++b) G[a][b] = f32x16{};
        }
    }
};

// s fragments (st = 0, 1) of the planes whose h fragments are hf
template <int NP>
__device__ __forceinline__ void transpose_planes(SplitStage& sg, const bf16x8 (&hf)[2][NP], bf16x8 (&sf)[2][NP])
{
    wave_lds_fence();  // the previous reads of the tiles are issued before these stores
#pragma unroll
    for (int st = 0; st < 2; ++st)
#pragma unroll
        for (int k = 0; k < NP; ++k) tr_store(sg.plane[k], hf[st][k], st);
    wave_lds_fence();
#pragma unroll
    for (int st = 0; st < 2; ++st)
#pragma unroll
        for (int k = 0; k < NP; ++k) sf[st][k] = tr_load(sg.plane[k], st);
}

// the smallest |a[i]|, NaN-ignoring (a NaN shows in the bound it is compared with)
__device__ __forceinline__ float min_abs(const f32x16& a)
{
    float m = fabsf(a[0]);
#pragma unroll
    for (int i = 1; i < 16; ++i) m = fminf(m, fabsf(a[i]));
    return m;
}

// x of lane l ^ B of the same 16-lane row (B = 4: of lane l ^ 7)
template <int B>
__device__ __forceinline__ float lane_xor(float x)
{
    constexpr int kCtl = B == 1 ? 0xB1 : (B == 2 ? 0x4E : (B == 4 ? 0x141 : 0x128));  // quad_perm, half mirror, ror:8
    return __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(x), kCtl, 0xF, 0xF, true));
}

// One step of transpose_sum: the lane keeps the lower or the upper half of the first 2 N values, by bit B of its number, and
// adds its partner's.
template <int B, int N>
__device__ __forceinline__ void transpose_step(float* v)
{
    const bool up = threadIdx.x & B;
#pragma unroll
    for (int i = 0; i < N; ++i)
    {
        const float keep = up ? v[i + N] : v[i], give = up ? v[i] : v[i + N];
        v[i]             = keep + lane_xor<B>(give);
    }
}

// The sum of value j = n / (32 / N) over the 32 lanes of each half wave, on lane n of the half, of N = 16 or 32 values per
// lane: halving the values in every step takes about 3 N instructions, the N sums one by one 5 N. The steps are taken to
// the end for every tile, so that a lane keeps one running sum: with 4, 8 or 16 of them and the last steps once at the end
// the projector's FP32 step takes 15.5, 17.0 and 19.3 ms instead of 15.0 (registers).
template <int N>
__device__ __forceinline__ float transpose_sum(float (&v)[N])
{
#pragma unroll
    for (int i = 0; i < N / 2; ++i)
    {
        const auto s = __builtin_amdgcn_permlane16_swap(__float_as_uint(v[i]), __float_as_uint(v[i + N / 2]), false,
                                                        false);
        v[i] = __uint_as_float(s[0]) + __uint_as_float(s[1]);
    }
    transpose_step<8, N / 4>(v);
    transpose_step<4, N / 8>(v);
    transpose_step<2, N / 16>(v);
    if constexpr (N == 32)
        transpose_step<1, 1>(v);
    else
        v[0] += lane_xor<1>(v[0]);
    return v[0];
}

// Backward of one tile of 32 samples on a wave (arguments as tile_backward_mfma): adds the tile's parameter-gradient
// products to acc and returns dL/dx in dx (channels 4g..4g+3 of the lane's sample, g = lane / 32).
template <int H>
__device__ __forceinline__ void tile_backward_split(const float* __restrict__ params, const WeightLDSSplit<H>& w,
                                                    const float (&x4)[4], float gy, bool valid, int last_act,
                                                    float beta, SplitStage& sg, SplitAcc<H / 32>& acc, float (&dx)[4])
{
    constexpr int MT = H / 32;
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    const int l = threadIdx.x & 63, n = l & 31, hg = l >> 5;
    asm volatile("" ::: "memory");  // as in tile_forward_split
    SplitX x(x4);
    f32x16 z1[MT], z2[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) z1[mt] = split_layer1<H>(w, x, mt);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) z2[mt] = f32x16{};
    float hmax = 0.f;
    bf16x8 h0[MT][2];
    // all the smaller partial products first, then those of the first planes, then the bias (as tile_forward_split)
#pragma unroll
    for (int ms = 0; ms < MT; ++ms)
    {
#pragma unroll
        for (int st = 0; st < 2; ++st)
        {
            float u[8];
            bf16x8 h[3];
#pragma unroll
            for (int j = 0; j < 8; ++j)
            {
                u[j] = act_f(NEAT_ACT_RELU, z1[ms][8 * st + j], beta);
                hmax = fmaxf(hmax, u[j]);
            }
            split3_frag(u, h);
            h0[ms][st] = h[0];
#pragma unroll
            for (int k = 2; k >= 0; --k)
#pragma unroll
                for (int q = 2 - k; q >= (k == 0 ? 1 : 0); --q)
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt) z2[mt] = mma_bf16(w.w2[k][mt][ms][st][l], h[q], z2[mt]);
        }
    }
    __builtin_amdgcn_sched_barrier(0);  // mixed with the pass above this one would spill
#pragma unroll
    for (int ms = 0; ms < MT; ++ms)
#pragma unroll
        for (int st = 0; st < 2; ++st)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) z2[mt] = mma_bf16(w.w2[0][mt][ms][st][l], h0[ms][st], z2[mt]);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
    {
        const f32x16 b = row_vec(w.vec[1], mt, hg);
#pragma unroll
        for (int i = 0; i < 16; ++i) z2[mt][i] += b[i];
    }
    {
        // 8 roundings of the largest sums that |x|, |h1| and the weights allow (the margin of the note on top)
        constexpr float u8 = 8.f / 16777216.f;
        float m1 = min_abs(z1[0]), m2 = min_abs(z2[0]);
        if constexpr (MT == 2)
        {
            m1 = fminf(m1, min_abs(z1[1]));
            m2 = fminf(m2, min_abs(z2[1]));
        }
        hmax = fmaxf(hmax, __shfl_xor(hmax, 32));
        const float a0 = __uint_as_float(w.norm[0]), c0 = __uint_as_float(w.norm[1]);
        const float a1 = __uint_as_float(w.norm[2]), c1 = __uint_as_float(w.norm[3]);
        const float t1 = u8 * fmaf(a0, max_abs_x(x4), c0);
        const float t2 = fmaf(a1, t1, u8 * fmaf(a1, hmax, c1));
        // a NaN or infinity anywhere takes the plain evaluation too
        const bool fine = fabsf((x4[0] + x4[1]) + (x4[2] + x4[3])) < 1e30f && t2 < 1e30f;
        if (__any(!(fine && m1 > t1 && m2 > t2))) tile_forward_exact<H, NEAT_ACT_RELU>(params, w, x4, beta, z1, z2);
        if (__any(!fine)) x.split_any(x4);
    }
    float z = 0.f;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
    {
        const f32x16 w3 = row_vec(w.vec[2], mt, hg);
#pragma unroll
        for (int i = 0; i < 16; ++i) z = fmaf(w3[i], act_f(NEAT_ACT_RELU, z2[mt][i], beta), z);
    }
    z = z + __shfl_xor(z, 32) + w.vec[3][0];
    const float dz = valid ? acc.sign * (gy * act_d(last_act, z, beta)) : 0.f;
    if (hg == 0) acc.b3 += dz;
    {
        float v[16 * MT];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int i = 0; i < 16; ++i) v[16 * mt + i] = act_f(NEAT_ACT_RELU, z2[mt][i], beta) * dz;
        acc.w3 += transpose_sum(v);
    }
    // T
    unsigned short* T = sg.plane[0];
    {
        __bf16 dp[3];
        split3(dz, dp);
        wave_lds_fence();
#pragma unroll
        for (int k = 0; k < 3; ++k)
        {
            const u32x4 u = __builtin_bit_cast(u32x4, x.p[k]);
            *reinterpret_cast<uint2*>(&T[n * kTrRow + 8 * k + 4 * hg]) = make_uint2(u[0], u[1]);
            if (hg == 0) T[n * kTrRow + kTDz + k] = __builtin_bit_cast(unsigned short, dp[k]);
        }
        if (hg == 0) T[n * kTrRow + kTOnes] = 0x3F80;
    }
    // the hidden layer's mask
    bf16x8 mh[MT][2][1];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
    {
#pragma unroll
        for (int st = 0; st < 2; ++st)
        {
            u32x4 u;
#pragma unroll
            for (int q = 0; q < 4; ++q)
                u[q] = (z2[mt][8 * st + 2 * q] > 0.f ? 0x3F80u : 0u) |
                       (z2[mt][8 * st + 2 * q + 1] > 0.f ? 0x3F800000u : 0u);
            mh[mt][st][0] = __builtin_bit_cast(bf16x8, u);
        }
    }
    wave_lds_fence();
    // the columns of T as B fragments: those of the first layer, those of dz
    bf16x8 bx[2], bz[2];
#pragma unroll
    for (int st = 0; st < 2; ++st)
    {
        const bf16x8 t = tr_load(T, st);
        bx[st]         = n <= kTOnes ? t : bf16x8{};
        bz[st]         = (n >= kTDz && n < kTDz + 3) ? t : bf16x8{};
    }
    // dL/dZ1 per 32-unit tile, dL/dx, and the first layer's gradients
    f32x16 xa = {};
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
    {
        f32x16 a = {};
#pragma unroll
        for (int k = 2; k >= 0; --k)
#pragma unroll
            for (int ms = 0; ms < MT; ++ms)
#pragma unroll
                for (int st = 0; st < 2; ++st) a = mma_bf16(w.w2t[k][mt][ms][st][l], mh[ms][st][0], a);
        bf16x8 dh[2][3], ds[2][3];
#pragma unroll
        for (int st = 0; st < 2; ++st)
        {
            float v[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = z1[mt][8 * st + j] > 0.f ? a[8 * st + j] * dz : 0.f;
            split3_frag(v, dh[st]);
#pragma unroll
            for (int k = 0; k < 3; ++k) xa = mma_bf16(w.w1t[mt][st][l], dh[st][k], xa);
        }
        transpose_planes<3>(sg, dh, ds);
#pragma unroll
        for (int st = 0; st < 2; ++st)
#pragma unroll
            for (int k = 0; k < 3; ++k) acc.E[mt] = mma_bf16(ds[st][k], bx[st], acc.E[mt]);
    }
    // the three row groups of W0's planes
#pragma unroll
    for (int j = 0; j < 4; ++j) dx[j] = acc.sign * (xa[j] + (xa[j + 4] + xa[j + 8]));
    // the hidden layer's gradients
    bf16x8 ms_[MT][2][1];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
    {
        transpose_planes<1>(sg, mh[mt], ms_[mt]);
#pragma unroll
        for (int st = 0; st < 2; ++st) acc.E[mt] = mma_bf16(ms_[mt][st][0], bz[st], acc.E[mt]);
    }
#pragma unroll
    for (int m1 = 0; m1 < MT; ++m1)
    {
        bf16x8 hh[2][3], hs[2][3];
#pragma unroll
        for (int st = 0; st < 2; ++st)
        {
            float v[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = act_f(NEAT_ACT_RELU, z1[m1][8 * st + j], beta) * dz;
            split3_frag(v, hh[st]);
        }
        transpose_planes<3>(sg, hh, hs);
#pragma unroll
        for (int m2 = 0; m2 < MT; ++m2)
#pragma unroll
            for (int st = 0; st < 2; ++st)
#pragma unroll
                for (int k = 2; k >= 0; --k) acc.G[m2][m1] = mma_bf16(ms_[m2][st][0], hs[st][k], acc.G[m2][m1]);
    }
}

// Floats of a wave's sums as put_split_sums lays them out: G [H][H], E [H][32], w3 [H], b3.
template <int H>
constexpr int split_sums()
{
    return H * H + 33 * H + 1;
}

// A wave's sums, with their sign put right, written to `red` (add: added to it).
template <int H>
__device__ __forceinline__ void put_split_sums(SplitAcc<H / 32>& acc, float* red, bool add)
{
    constexpr int MT = H / 32;
    const int l = threadIdx.x & 63, n = l & 31, hg = l >> 5;
    auto put = [&](int i, float v) {
        v *= acc.sign;
        red[i] = add ? red[i] + v : v;
    };
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
    {
#pragma unroll
        for (int i = 0; i < 16; ++i)
        {
            const int r = 32 * mt + crow(i, hg);
#pragma unroll
            for (int m1 = 0; m1 < MT; ++m1) put(r * H + 32 * m1 + n, acc.G[mt][m1][i]);
            put(H * H + r * 32 + n, acc.E[mt][i]);
        }
    }
    float b3 = acc.b3;
#pragma unroll
    for (int off = 16; off >= 1; off >>= 1) b3 += __shfl_xor(b3, off);
    if (l == 0) put(H * H + 33 * H, b3);
    const int j = n / (2 / MT);  // transpose_sum's value on this lane
    if (n % (2 / MT) == 0) put(H * H + 32 * H + 32 * (j / 16) + crow(j % 16, hg), acc.w3);
}

// The workgroup's parameter-gradient slice, in the packed layout: its waves' sums added in a fixed order in LDS (in the
// transpose tiles, which are done with; as many waves at a time as have room there), the hidden layer's rows times
// w3, then stored. NW waves; called by every thread.
template <int H, int NW>
__device__ __forceinline__ void write_split_partials(const WeightLDSSplit<H>& w, SplitAcc<H / 32>& acc,
                                                     SplitStage (&stage)[NW], float* part)
{
    constexpr int C = 8, ob0 = H * C, oW1 = ob0 + H, ob1 = oW1 + H * H, oW2 = ob1 + H, ob2 = oW2 + H;
    constexpr int Q = split_sums<H>(), kFit = (int)(sizeof(stage) / (Q * sizeof(float))), NS = kFit < NW ? kFit : NW;
    static_assert(NS >= 1, "a wave's sums fit the transpose tiles");
    float* red = reinterpret_cast<float*>(&stage[0]);
    const int wave = threadIdx.x >> 6;
    __syncthreads();
    for (int k = 0; k < NW; k += NS)
    {
        if (wave >= k && wave < k + NS) put_split_sums<H>(acc, red + (wave - k) * Q, k > 0);
        __syncthreads();
    }
    for (int t = threadIdx.x; t < Q; t += blockDim.x)
    {
        float v = red[t];
#pragma unroll
        for (int k = 1; k < NS; ++k) v += red[k * Q + t];
        red[t] = v;
    }
    __syncthreads();
    const float* E = red + H * H;
    for (int t = threadIdx.x; t < H * C; t += blockDim.x)
    {
        const float* e = E + (t / C) * 32 + t % C;
        part[t]        = e[0] + (e[8] + e[16]);
    }
    for (int t = threadIdx.x; t < H * H; t += blockDim.x) part[oW1 + t] = red[t] * w.vec[2][t / H];
    for (int r = threadIdx.x; r < H; r += blockDim.x)
    {
        const float* e = E + r * 32 + kTDz;
        part[ob0 + r]  = E[r * 32 + kTOnes];
        part[ob1 + r]  = (e[0] + (e[1] + e[2])) * w.vec[2][r];
        part[oW2 + r]  = E[32 * H + r];
    }
    if (threadIdx.x == 0) part[ob2] = E[33 * H];
}

}  // namespace neat
