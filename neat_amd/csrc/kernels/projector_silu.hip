// Forward and backward of the fused projector for BF16 decoders with silu hidden layers.
#include "projector_dev.hpp"

namespace neat
{

constexpr int kBf16Threads = 512;  // 8 waves, two per SIMD

// columns of the tile T that the first-layer and bias gradients contract with (as BwdAcc's): 0..7 x, then ones, dz, ones
__device__ __forceinline__ bf16x8 column_if(bool keep, const bf16x8& t) { return keep ? t : bf16x8{}; }

// BF16 h fragment of slots 8st..8st+7, rounded to nearest even, one conversion per pair
__device__ __forceinline__ bf16x8 h_frag(const f32x16& z, int st)
{
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    u32x4 r;
#pragma unroll
    for (int q = 0; q < 4; ++q)
    {
        const f32x2 v = {z[8 * st + 2 * q], z[8 * st + 2 * q + 1]};
        r[q]          = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
    }
    return __builtin_bit_cast(bf16x8, r);
}

// s fragments (st = 0, 1) of the tile whose h fragments are hf, through this wave's transpose tile
__device__ __forceinline__ void transpose_frags(unsigned short* tile, const bf16x8 (&hf)[2], bf16x8 (&sf)[2])
{
    wave_lds_fence();  // the previous reads of the tile are issued before these stores
    tr_store(tile, hf[0], 0);
    tr_store(tile, hf[1], 1);
    wave_lds_fence();
    sf[0] = tr_load(tile, 0);
    sf[1] = tr_load(tile, 1);
}

// Backward of one tile of 32 samples: the steps of tile_backward_mfma in BF16 (every operand of a product rounded once,
// the products in the same order up to dL/dx), with each activation and its derivative taken once, right behind the
// pre-activation, and the operands of the weight gradients (which contract over the samples) taken from LDS transposes
// of the fragments the other products use. Returns dL/dx in registers 0..3. stash: this wave's 64 H / 8 float4 in LDS.
template <int H>
__device__ __forceinline__ f32x16 tile_backward_bf16(const WeightLDS<PrecBF16, H>& w, const float (&x4)[4], float gy,
                                                     bool valid, float beta, unsigned short* tile, float4* stash,
                                                     BwdAcc<H / 32>& acc)
{
    typedef PrecBF16 P;
    constexpr int MT = H / 32;
    const int l = threadIdx.x & 63, n = l & 31, hg = l >> 5;
    asm volatile("" ::: "memory");  // keeps the weight fragments in LDS: hoisted out of the tile loop they spill
    const s16x4 xf = x_step<P>(x4, 0);
    bf16x8 h1[MT][2];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
    {
        f32x16 z = P::mma1(w.w1[mt][0][l], xf, f32x16{});
#pragma unroll
        for (int i = 0; i < 16; ++i) z[i] += w.vec[0][32 * mt + crow(i, hg)];
        f32x16 a, d;
#pragma unroll
        for (int i = 0; i < 16; ++i)
        {
            a[i] = act_f(NEAT_ACT_SILU, z[i], beta);
            d[i] = act_d(NEAT_ACT_SILU, z[i], beta);
        }
        // act'(z1) waits in LDS for dL/dZ1: held in registers it would spill
#pragma unroll
        for (int q = 0; q < 4; ++q)
            stash[(4 * mt + q) * 64 + l] = make_float4(d[4 * q], d[4 * q + 1], d[4 * q + 2], d[4 * q + 3]);
#pragma unroll
        for (int st = 0; st < 2; ++st) h1[mt][st] = h_frag(a, st);
    }
    f32x16 d2[MT];  // act'(z2), then dL/dZ2
    bf16x8 h2[MT][2];
    float part = 0.f;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
    {
        f32x16 z = {};
#pragma unroll
        for (int ms = 0; ms < MT; ++ms)
#pragma unroll
            for (int st = 0; st < 2; ++st) z = P::mma(w.w2[mt][ms][st][l], h1[ms][st], z);
#pragma unroll
        for (int i = 0; i < 16; ++i) z[i] += w.vec[1][32 * mt + crow(i, hg)];
        f32x16 a;
#pragma unroll
        for (int i = 0; i < 16; ++i)
        {
            a[i]      = act_f(NEAT_ACT_SILU, z[i], beta);
            d2[mt][i] = act_d(NEAT_ACT_SILU, z[i], beta);
            part      = fmaf(w.vec[2][32 * mt + crow(i, hg)], a[i], part);
        }
#pragma unroll
        for (int st = 0; st < 2; ++st) h2[mt][st] = h_frag(a, st);
    }
    const float z  = part + __shfl_xor(part, 32) + w.vec[3][0];
    const float dz = valid ? gy * act_d(NEAT_ACT_SOFTPLUS, z, beta) : 0.f;
    if (hg == 0) acc.b3 += dz;
    // T: x, 1, dz, 1
    wave_lds_fence();
    *reinterpret_cast<s16x4*>(&tile[n * kTrRow + 4 * hg]) = xf;
    if (hg == 0)
    {
        tile[n * kTrRow + kXOnes1] = 0x3F80;
        tile[n * kTrRow + kXDz]    = (unsigned short)bf16_bits(dz);
        tile[n * kTrRow + kXOnes2] = 0x3F80;
    }
    bf16x8 d2h[MT][2];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
    {
#pragma unroll
        for (int i = 0; i < 16; ++i) d2[mt][i] = w.vec[2][32 * mt + crow(i, hg)] * dz * d2[mt][i];
#pragma unroll
        for (int st = 0; st < 2; ++st) d2h[mt][st] = h_frag(d2[mt], st);
    }
    wave_lds_fence();
    bf16x8 t[2];
#pragma unroll
    for (int st = 0; st < 2; ++st) t[st] = tr_load(tile, st);
    bf16x8 h1s[MT][2];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) transpose_frags(tile, h1[mt], h1s[mt]);
#pragma unroll
    for (int m2 = 0; m2 < MT; ++m2)
    {
        bf16x8 s[2];
        transpose_frags(tile, h2[m2], s);
#pragma unroll
        for (int st = 0; st < 2; ++st) acc.E[m2] = P::mma(s[st], column_if(n == kXDz, t[st]), acc.E[m2]);
        transpose_frags(tile, d2h[m2], s);
#pragma unroll
        for (int st = 0; st < 2; ++st)
        {
            acc.E[m2] = P::mma(s[st], column_if(n == kXOnes2, t[st]), acc.E[m2]);
#pragma unroll
            for (int m1 = 0; m1 < MT; ++m1) acc.dW2[m2][m1] = P::mma(s[st], h1s[m1][st], acc.dW2[m2][m1]);
        }
    }
    f32x16 dx = {};
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
    {
        f32x16 a = {};
#pragma unroll
        for (int ms = 0; ms < MT; ++ms)
#pragma unroll
            for (int st = 0; st < 2; ++st) a = P::mma(w.w2t[mt][ms][st][l], d2h[ms][st], a);
#pragma unroll
        for (int q = 0; q < 4; ++q)
        {
            const float4 d = stash[(4 * mt + q) * 64 + l];
            a[4 * q] *= d.x;
            a[4 * q + 1] *= d.y;
            a[4 * q + 2] *= d.z;
            a[4 * q + 3] *= d.w;
        }
        bf16x8 dh[2], s[2];
#pragma unroll
        for (int st = 0; st < 2; ++st)
        {
            dh[st] = h_frag(a, st);
            dx     = P::mma(w.w1t[mt][st][l], dh[st], dx);
        }
        transpose_frags(tile, dh, s);
#pragma unroll
        for (int st = 0; st < 2; ++st) acc.E[mt] = P::mma(s[st], column_if(n <= kXOnes1, t[st]), acc.E[mt]);
    }
    return dx;
}

// Persistent workgroups over the chunks, one tile per wave at a time; writes dL/dfeature ([S][8] BF16), the packed cell
// coordinates, each slot's largest |dL/dfeature| and one parameter-gradient slice per wave.
//
// Bound by vector work: two activations with their derivatives per unit are a third of the 1,500 vector instructions of a
// tile. 10.1 M samples, H = 64: 3.34 ms in the form it replaces (one wave per SIMD, activations taken up to four times
// per unit with the general division, operands staged value by value), 1.68 ms like this.
template <int H>
__global__ void __launch_bounds__(kBf16Threads, 2) k_bf16_bwd(ProjGeom g, Plan p, const float* __restrict__ params,
                                                              const void* grid_lowp, const float* grad_proj,
                                                              float* dfeat, float4* sgc, unsigned int* dmax,
                                                              float* partials, int32_t P_total)
{
    typedef PrecBF16 P;
    __shared__ WeightLDS<P, H> w;
    __shared__ ChunkCtx cx;
    __shared__ __align__(16) unsigned short s_tr[kBf16Threads / 64][32 * kTrRow];
    __shared__ float4 s_stash[kBf16Threads / 64][H / 8 * 64];
    load_weights<P, H, 8>(params, w);
    const int l = threadIdx.x & 63, wave = threadIdx.x >> 6, hg = l >> 5;
    BwdAcc<H / 32> acc;
    float amax            = 0.f;  // largest |dL/dfeature| this lane wrote
    const int32_t nchunks = (int32_t)p.chunk_off1[g.N];
    for (int32_t c = blockIdx.x; c < nchunks; c += (int32_t)gridDim.x)
    {
        const int32_t slot = p.chunk1_slot[c];
        const int32_t q0 = p.chunk1_q0[c], q1 = p.chunk1_q1[c], nseg = q1 - q0;
        if (nseg == 0) continue;
        const int64_t base = p.nm_soff[q0];
        __syncthreads();  // the previous chunk's readers of cx are done (and the weights are in place)
        load_chunk_ctx(g, p, q0, q1, base, grad_proj, cx);
        NodeBox nb;
        node_bounds(g, g.seg_node[p.perm[q0]], nb);
        const void* ngrid = node_grid_ptr(g, grid_lowp, true, slot);
        __syncthreads();
        const int32_t nsamp = cx.beg[nseg];
        float cmax          = 0.f;  // this chunk's
        for (int32_t w0 = 0; w0 < nsamp; w0 += kFwdChunk)
        {
            const int32_t wn = min(kFwdChunk, nsamp - w0);
            expand_window(cx, nseg, w0, wn);
            __syncthreads();
            for (int32_t p0 = wave * 64; p0 < wn; p0 += kBf16Threads)
            {
                PairIn cur;
                fetch_pair<true, true>(g, cx, p0, w0, wn, base, nb, ngrid, sgc, cur);
                // one copy of the tile code for both halves of the pair
#pragma unroll 1
                for (int h = 0; h < 2; ++h)
                {
                    if (h == 1 && p0 + 32 >= wn) break;
                    float xs[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) xs[j] = h ? cur.xb[j] : cur.xa[j];
                    const int32_t i  = p0 + 32 * h + (l & 31);
                    const bool valid = i < wn;
                    const f32x16 dx =
                        tile_backward_bf16<H>(w, xs, h ? cur.vb : cur.va, valid, g.beta, s_tr[wave], s_stash[wave],
                                                   acc);
                    if (valid)
                    {
                        // this lane's 4 channels
                        *reinterpret_cast<uint2*>(reinterpret_cast<unsigned short*>(dfeat) + (base + w0 + i) * 8 +
                                                  4 * hg) = bf16x4_bits(dx[0], dx[1], dx[2], dx[3]);
                        cmax = fmaxf(cmax, fmaxf(fmaxf(fabsf(dx[0]), fabsf(dx[1])), fmaxf(fabsf(dx[2]), fabsf(dx[3]))));
                    }
                }
            }
            __syncthreads();
        }
        amax = fmaxf(amax, cmax);
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) cmax = fmaxf(cmax, __shfl_xor(cmax, off));
        if (l == 0) atomicMax(dmax + 1 + slot, __float_as_uint(cmax));
    }
    write_param_partials<H, 8>(acc, partials + ((int64_t)blockIdx.x * (kBf16Threads / 64) + wave) * P_total);
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) amax = fmaxf(amax, __shfl_xor(amax, off));
    if (l == 0) atomicMax(dmax, __float_as_uint(amax));  // non-negative floats order like their bit patterns
}

// Forward: persistent workgroups over the chunks, a pair of 32-sample tiles per wave at a time; per-segment sums
// sequential in j, as in the other forms. Three waves per SIMD: 0.98 ms on the samples above, against 1.10 with two and
// 0.97 with four.
constexpr int kBf16FwdThreads = 768;

template <int H>
__global__ void __launch_bounds__(kBf16FwdThreads, 3) k_bf16_fwd(ProjGeom g, Plan p, const float* __restrict__ params,
                                                                 const void* grid_lowp, float* seg_partial,
                                                                 float* sample_out)
{
    __shared__ WeightLDS<PrecBF16, H> w;
    __shared__ ChunkCtx cx;
    __shared__ float s_contrib[kFwdChunk];
    __shared__ float s_seg[kSegCap];
    load_weights<PrecBF16, H, 8>(params, w);
    const int l = threadIdx.x & 63, wave = threadIdx.x >> 6, hg = l >> 5;
    const int32_t nchunks = (int32_t)p.chunk_off1[g.N];
    for (int32_t c = blockIdx.x; c < nchunks; c += (int32_t)gridDim.x)
    {
        const int32_t slot = p.chunk1_slot[c];
        const int32_t q0 = p.chunk1_q0[c], q1 = p.chunk1_q1[c], nseg = q1 - q0;
        if (nseg == 0) continue;
        const int64_t base = p.nm_soff[q0];
        __syncthreads();  // the previous chunk's readers of cx / s_seg are done (and the weights are in place)
        load_chunk_ctx(g, p, q0, q1, base, nullptr, cx);
        for (int32_t t = threadIdx.x; t < nseg; t += blockDim.x) s_seg[t] = 0.f;
        NodeBox nb;
        node_bounds(g, g.seg_node[p.perm[q0]], nb);
        const void* ngrid = node_grid_ptr(g, grid_lowp, true, slot);
        __syncthreads();
        const int32_t nsamp = cx.beg[nseg];
        for (int32_t w0 = 0; w0 < nsamp; w0 += kFwdChunk)
        {
            const int32_t wn = min(kFwdChunk, nsamp - w0);
            expand_window(cx, nseg, w0, wn);
            __syncthreads();
            for (int32_t p0 = wave * 64; p0 < wn; p0 += kBf16FwdThreads)
            {
                PairIn cur;
                fetch_pair<true, false>(g, cx, p0, w0, wn, base, nb, ngrid, nullptr, cur);
                float z[2] = {0.f, 0.f};
                // one copy of the tile code for both halves of the pair
#pragma unroll 1
                for (int h = 0; h < 2; ++h)
                {
                    if (h == 1 && p0 + 32 >= wn) break;
                    asm volatile("" ::: "memory");  // keeps the weight fragments in LDS (tile_backward_bf16)
                    float x[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) x[j] = h ? cur.xb[j] : cur.xa[j];
                    Fwd<H / 32> f;
                    tile_forward_mfma<PrecBF16, H>(w, x, g.beta, f);
                    z[0] = h ? z[0] : f.z;
                    z[1] = h ? f.z : z[1];
                }
                // lane l takes sample p0 + l: tile A on the lower lanes, B on the upper ones
                const int32_t i = p0 + l;
                if (i < wn)
                {
                    const float y = act_f(NEAT_ACT_SOFTPLUS, hg ? z[1] : z[0], g.beta);
                    s_contrib[i]  = y * (hg ? cur.vb : cur.va);
                    if (sample_out) sample_out[base + w0 + i] = y;
                }
            }
            __syncthreads();
            for (int32_t t = threadIdx.x; t < nseg; t += blockDim.x)
            {
                const int32_t a = max(cx.beg[t], w0), b = min(cx.beg[t + 1], w0 + wn);
                if (a >= b) continue;
                float acc = 0.f;
                for (int32_t i = a; i < b; ++i) acc += s_contrib[i - w0];
                s_seg[t] += acc;
            }
            __syncthreads();
        }
        for (int32_t t = threadIdx.x; t < nseg; t += blockDim.x) seg_partial[cx.k[t]] = s_seg[t];
    }
}

int launch_bf16_fwd(hipStream_t s, int H, int workgroups, const ProjGeom& g, const Plan& p, const float* params,
                    const void* grid_bf16, float* seg_partial, float* sample_out)
{
    if (H == 64)
        k_bf16_fwd<64><<<workgroups, kBf16FwdThreads, 0, s>>>(g, p, params, grid_bf16, seg_partial, sample_out);
    else
        k_bf16_fwd<32><<<workgroups, kBf16FwdThreads, 0, s>>>(g, p, params, grid_bf16, seg_partial, sample_out);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int bf16_bwd_slices(int workgroups) { return workgroups * (kBf16Threads / 64); }

int launch_bf16_bwd(hipStream_t s, int H, int workgroups, const ProjGeom& g, const Plan& p, const float* params,
                    const void* grid_bf16, const float* grad_proj, float* dfeat, float4* sgc, unsigned int* dmax,
                    float* partials, int32_t P_total)
{
    if (H == 64)
        k_bf16_bwd<64><<<workgroups, kBf16Threads, 0, s>>>(g, p, params, grid_bf16, grad_proj, dfeat, sgc, dmax,
                                                           partials, P_total);
    else
        k_bf16_bwd<32><<<workgroups, kBf16Threads, 0, s>>>(g, p, params, grid_bf16, grad_proj, dfeat, sgc, dmax,
                                                           partials, P_total);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace neat
