// FP32 forward of the fused projector, and its backward for relu hidden layers, with the decoder's products on the BF16
// matrix cores in split form (split_mlp.hpp).
//
// On the FP32 matrix cores a tile of 32 samples with H = 64 took 4,608 cycles of products forward and 21,000 backward
// (a 32x32x2 product is 64 cycles); in split form it is 1,730 and 4,160, beside about 2,200 and 5,900 cycles of vector
// work. Measured on 53.3 M samples (2^18 rays, 4096 grids of 17^3 x 8): forward 7.37 -> 3.6 ms, backward 28.3 -> 9.2 ms
// (0.5 ms are the tiles whose pre-activations are recomputed on the FP32 matrix cores, all of them would cost 2.5 ms
// more; 0.9 ms the order of the sums and the output weights' own, see split_mlp.hpp). The gather of the node grid takes
// about 1.3 ms of the backward; two waves per SIMD leave the matrix cores idle two thirds of the time, the rest being
// vector work and exposed LDS latency.
#include "projector_dev.hpp"
#include "split_mlp.hpp"

namespace neat
{

// Backward: persistent workgroups over the chunks, one tile of 32 samples per wave at a time; writes dL/dfeature and the
// grid coordinate of every sample (for the scatter), and one slice of the parameter gradient per workgroup.
constexpr int kSplitThreads = 512;  // 8 waves, two per SIMD (one workgroup's LDS fills a CU)

template <int H>
__global__ void __launch_bounds__(kSplitThreads, 2) k_split_bwd(ProjGeom g, Plan p, const float* __restrict__ params,
                                                                const float* grad_proj, float* dfeat, float4* sgc,
                                                                unsigned int* dmax, float* partials, int32_t P_total)
{
    __shared__ WeightLDSSplit<H> w;
    __shared__ ChunkCtx cx;
    __shared__ __align__(16) SplitStage stage[kSplitThreads / 64];
    load_weights_split<H>(params, reinterpret_cast<float*>(&stage[0]), w);
    const int l = threadIdx.x & 63, wave = threadIdx.x >> 6, hg = l >> 5;
    SplitStage& sg = stage[wave];
    SplitAcc<H / 32> acc;
    float amax = 0.f;  // largest |dL/dfeature| this lane wrote
    const int32_t nchunks = (int32_t)p.chunk_off1[g.N];
    for (int32_t c = blockIdx.x; c < nchunks; c += (int32_t)gridDim.x)
    {
        const int32_t slot = p.chunk1_slot[c];
        const int32_t q0 = p.chunk1_q0[c], q1 = p.chunk1_q1[c], nseg = q1 - q0;
        if (nseg == 0) continue;
        const int64_t base = p.nm_soff[q0];
        __syncthreads();
        load_chunk_ctx(g, p, q0, q1, base, grad_proj, cx);
        NodeBox nb;
        node_bounds(g, g.seg_node[p.perm[q0]], nb);
        const void* ngrid = node_grid_ptr(g, nullptr, false, slot);
        __syncthreads();
        const int32_t nsamp = cx.beg[nseg];
        for (int32_t w0 = 0; w0 < nsamp; w0 += kFwdChunk)
        {
            const int32_t wn = min(kFwdChunk, nsamp - w0);
            expand_window(cx, nseg, w0, wn);
            __syncthreads();
            for (int32_t p0 = wave * 64; p0 < wn; p0 += kSplitThreads)
            {
                PairIn cur;
                fetch_pair<false, true>(g, cx, p0, w0, wn, base, nb, ngrid, sgc, cur);
                // one copy of the tile code for both halves of the pair
#pragma unroll 1
                for (int h = 0; h < 2; ++h)
                {
                    if (h == 1 && p0 + 32 >= wn) break;
                    float xs[4], dx[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) xs[j] = h ? cur.xb[j] : cur.xa[j];
                    const int32_t i  = p0 + 32 * h + (l & 31);
                    const bool valid = i < wn;
                    tile_backward_split<H>(params, w, xs, h ? cur.vb : cur.va, valid, NEAT_ACT_SOFTPLUS, g.beta, sg, acc, dx);
                    if (valid)
                    {
                        // [2][S][4]: channel halves
                        *reinterpret_cast<float4*>(dfeat + ((int64_t)hg * g.S + base + w0 + i) * 4) =
                            make_float4(dx[0], dx[1], dx[2], dx[3]);
                        amax = fmaxf(amax, fmaxf(fmaxf(fabsf(dx[0]), fabsf(dx[1])), fmaxf(fabsf(dx[2]), fabsf(dx[3]))));
                    }
                }
            }
            __syncthreads();
        }
    }
    write_split_partials<H>(w, acc, stage, partials + (int64_t)blockIdx.x * P_total);
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) amax = fmaxf(amax, __shfl_xor(amax, off));
    if (l == 0) atomicMax(dmax, __float_as_uint(amax));  // non-negative floats order like their bit patterns
}

// Forward: persistent workgroups over the chunks, a pair of 32-sample tiles per wave at a time; per-segment sums
// sequential in j, as in the other forms. Three waves per SIMD: 3.43 ms at the size above, against 3.59 with two (512
// threads) and 3.63 with four (1024 threads, which spills).
constexpr int kSplitFwdThreads = 768;

template <int H, int ACT>
__global__ void __launch_bounds__(kSplitFwdThreads, 3) k_split_fwd(ProjGeom g, Plan p, const float* __restrict__ params,
                                                                   float* seg_partial, float* sample_out)
{
    __shared__ WeightLDSSplitFwd<H> w;
    __shared__ ChunkCtx cx;
    __shared__ float s_contrib[kFwdChunk];
    __shared__ float s_seg[kSegCap];
    load_weights_split_fwd<H>(params, w);
    const int l = threadIdx.x & 63, wave = threadIdx.x >> 6, n = l & 31, hg = l >> 5;
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
        const void* ngrid = node_grid_ptr(g, nullptr, false, slot);
        __syncthreads();
        const int32_t nsamp = cx.beg[nseg];
        for (int32_t w0 = 0; w0 < nsamp; w0 += kFwdChunk)
        {
            const int32_t wn = min(kFwdChunk, nsamp - w0);
            expand_window(cx, nseg, w0, wn);
            __syncthreads();
            for (int32_t p0 = wave * 64; p0 < wn; p0 += kSplitFwdThreads)
            {
                PairIn cur;
                fetch_pair<false, false>(g, cx, p0, w0, wn, base, nb, ngrid, nullptr, cur);
                float z[2] = {0.f, 0.f};
                // one copy of the tile code for both halves of the pair
#pragma unroll 1
                for (int h = 0; h < 2; ++h)
                {
                    if (h == 1 && p0 + 32 >= wn) break;
                    float x[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) x[j] = h ? cur.xb[j] : cur.xa[j];
                    const float zh = tile_forward_split<H, ACT>(params, w, x, g.beta);
                    z[0]           = h ? z[0] : zh;
                    z[1]           = h ? zh : z[1];
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

int launch_split_fwd(hipStream_t s, int H, int act, int workgroups, const ProjGeom& g, const Plan& p,
                     const float* params, float* seg_partial, float* sample_out)
{
    if (H == 64 && act == NEAT_ACT_RELU)
        k_split_fwd<64, NEAT_ACT_RELU><<<workgroups, kSplitFwdThreads, 0, s>>>(g, p, params, seg_partial, sample_out);
    else if (H == 64)
        k_split_fwd<64, NEAT_ACT_SILU><<<workgroups, kSplitFwdThreads, 0, s>>>(g, p, params, seg_partial, sample_out);
    else if (act == NEAT_ACT_RELU)
        k_split_fwd<32, NEAT_ACT_RELU><<<workgroups, kSplitFwdThreads, 0, s>>>(g, p, params, seg_partial, sample_out);
    else
        k_split_fwd<32, NEAT_ACT_SILU><<<workgroups, kSplitFwdThreads, 0, s>>>(g, p, params, seg_partial, sample_out);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int launch_split_bwd(hipStream_t s, int H, int workgroups, const ProjGeom& g, const Plan& p, const float* params,
                     const float* grad_proj, float* dfeat, float4* sgc, unsigned int* dmax, float* partials,
                     int32_t P_total)
{
    if (H == 64)
        k_split_bwd<64><<<workgroups, kSplitThreads, 0, s>>>(g, p, params, grad_proj, dfeat, sgc, dmax, partials,
                                                             P_total);
    else
        k_split_bwd<32><<<workgroups, kSplitThreads, 0, s>>>(g, p, params, grad_proj, dfeat, sgc, dmax, partials,
                                                             P_total);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace neat
