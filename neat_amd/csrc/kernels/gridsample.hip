// Indirect trilinear grid sample, forward and backward (IndirectGridSample3D.cu:432-572 and :584-791).
//
// One thread per sample. The grid is addressed through element strides (N, C, Z, Y, X); when the channel stride is
// 1 (channels-last-3d, the layout the module layer stores its grid in) each corner's C channels are one contiguous
// run and are read with 16-byte vector loads. The arithmetic (corner weights from the unclamped neighbours, indices
// clamped to the border, per-channel sum in the corner order tnw tne tsw tse bnw bne bsw bse) follows the reference
// and is compiled without contraction, so the forward is bit-identical to the oracle.
#include "gridsample_dev.hpp"

namespace neat
{

// kChannelsLast: a corner's channels are one contiguous run, read with 16-byte loads. kLanes lanes share a sample, each
// taking every kLanes-th channel quad: bound by the cache lines an instruction touches, of which 8 channels then cost one
// per corner instead of one per corner and quad. 13.0 M samples, 4096 grids of 17^3 x 8: 523 us with one lane a sample,
// 345 us with two. Per channel the arithmetic is the same, so are the bits.
template <bool kChannelsLast, int kLanes = 1>
__global__ void __launch_bounds__(256) k_gs3d_fwd(GridArgs g, const int64_t* index, const float* uv, int64_t S,
                                                  float* out)
{
    const int64_t l = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t i = l / kLanes;
    if (i >= S) return;
    const int64_t n = index[i];
    if constexpr (kChannelsLast)
    {
        const int32_t c0 = 4 * (int32_t)(l % kLanes);
        if (n < 0 || n >= g.N)
        {
            // a slot outside the grid (e.g. -1 for an inactive node) samples zeros instead of reading out of bounds
            for (int c = c0; c < g.C; c += 4 * kLanes)
                *reinterpret_cast<float4*>(out + i * g.C + c) = make_float4(0.f, 0.f, 0.f, 0.f);
            return;
        }
        const Tri t = trilinear(g, n, uv[3 * i], uv[3 * i + 1], uv[3 * i + 2]);
        for (int c = c0; c < g.C; c += 4 * kLanes)
        {
            float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
            for (int k = 0; k < 8; ++k)
            {
                float4 v = *reinterpret_cast<const float4*>(g.grid + t.off[k] + c);
                acc.x += v.x * t.w[k];
                acc.y += v.y * t.w[k];
                acc.z += v.z * t.w[k];
                acc.w += v.w * t.w[k];
            }
            *reinterpret_cast<float4*>(out + i * g.C + c) = acc;
        }
    }
    else
    {
        if (n < 0 || n >= g.N)
        {
            for (int c = 0; c < g.C; ++c) out[i * g.C + c] = 0.f;
            return;
        }
        const Tri t = trilinear(g, n, uv[3 * i], uv[3 * i + 1], uv[3 * i + 2]);
        for (int c = 0; c < g.C; ++c)
        {
            float acc = 0.f;
#pragma unroll
            for (int k = 0; k < 8; ++k) acc += g.grid[t.off[k] + c * g.s1] * t.w[k];
            out[i * g.C + c] = acc;
        }
    }
}

// Backward for any strides: one thread per sample, the grid gradient with one float atomic per corner and channel (as
// the reference, IndirectGridSample3D.cu:691-698) and the uv gradient with the reference's product order (:752-790).
// Channels-last gradients take k_gs3d_bwd_cl below, whose atomics coalesce.
__global__ void __launch_bounds__(256) k_gs3d_bwd(GridArgs g, const int64_t* index, const float* uv, int64_t S,
                                                  const float* grad_out, float* grad_grid, float* grad_uv)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= S) return;
    const int64_t n = index[i];
    if (n < 0 || n >= g.N)
    {
        if (grad_uv) grad_uv[3 * i] = grad_uv[3 * i + 1] = grad_uv[3 * i + 2] = 0.f;
        return;
    }
    Tri t    = trilinear(g, n, uv[3 * i], uv[3 * i + 1], uv[3 * i + 2]);
    float ix = t.ix, iy = t.iy, iz = t.iz;
    float x0 = (float)t.x0, y0 = (float)t.y0, z0 = (float)t.z0;
    float x1 = x0 + 1, y1 = y0 + 1, z1 = z0 + 1;
    float gix = 0.f, giy = 0.f, giz = 0.f;
    for (int c = 0; c < g.C; ++c)
    {
        float go = grad_out[i * g.C + c];
        float val[8];
#pragma unroll
        for (int k = 0; k < 8; ++k)
        {
            int64_t o = t.off[k] + c * g.s1;
            if (grad_grid) atomicAdd(grad_grid + o, t.w[k] * go);
            val[k] = g.grid[o];
        }
        if (grad_uv)
        {
            float m1 = -1;
            gix += m1 * val[0] * (y1 - iy) * (z1 - iz) * go;
            gix += val[1] * (y1 - iy) * (z1 - iz) * go;
            gix += m1 * val[2] * (iy - y0) * (z1 - iz) * go;
            gix += val[3] * (iy - y0) * (z1 - iz) * go;
            gix += m1 * val[4] * (y1 - iy) * (iz - z0) * go;
            gix += val[5] * (y1 - iy) * (iz - z0) * go;
            gix += m1 * val[6] * (iy - y0) * (iz - z0) * go;
            gix += val[7] * (iy - y0) * (iz - z0) * go;

            giy += m1 * val[0] * (x1 - ix) * (z1 - iz) * go;
            giy += m1 * val[1] * (ix - x0) * (z1 - iz) * go;
            giy += val[2] * (x1 - ix) * (z1 - iz) * go;
            giy += val[3] * (ix - x0) * (z1 - iz) * go;
            giy += m1 * val[4] * (x1 - ix) * (iz - z0) * go;
            giy += m1 * val[5] * (ix - x0) * (iz - z0) * go;
            giy += val[6] * (x1 - ix) * (iz - z0) * go;
            giy += val[7] * (ix - x0) * (iz - z0) * go;

            giz += m1 * val[0] * (x1 - ix) * (y1 - iy) * go;
            giz += m1 * val[1] * (ix - x0) * (y1 - iy) * go;
            giz += m1 * val[2] * (x1 - ix) * (iy - y0) * go;
            giz += m1 * val[3] * (ix - x0) * (iy - y0) * go;
            giz += val[4] * (x1 - ix) * (y1 - iy) * go;
            giz += val[5] * (ix - x0) * (y1 - iy) * go;
            giz += val[6] * (x1 - ix) * (iy - y0) * go;
            giz += val[7] * (ix - x0) * (iy - y0) * go;
        }
    }
    if (grad_uv)
    {
        grad_uv[3 * i + 0] = gix * (float)(g.X - 1) / 2;
        grad_uv[3 * i + 1] = giy * (float)(g.Y - 1) / 2;
        grad_uv[3 * i + 2] = giz * (float)(g.Z - 1) / 2;
    }
}

// Backward for a channels-last grid and gradient (channel stride 1, C a multiple of CL).
//
// What bounds the scatter is the number of atomic requests, not their bytes: one thread per sample issues C * 8
// atomics whose 64 lanes all hit different lines. Here 2 CL lanes hold the CL consecutive channels of the two corners
// of an x edge, which are neighbours in memory, so an atomic instruction makes 32 / CL requests of 8 CL contiguous
// bytes; and a lane group walks a run of `run` consecutive samples, keeping the current trilinear cell's corner sums
// in registers and adding them to memory only when the run leaves the cell (samples of a ray stay in a cell for about
// 4 steps; samples in any other order only merge less). The uv gradient runs first, one thread per sample: the 8
// corners' channel products are summed into one value per corner, of which the three derivatives are 12 terms each;
// the coordinates stay in LDS for the walk.
//
// Measured on 13.0 M samples of cone-beam rays through 4096 grids of 17^3 x 8, with the uv gradient: 37.0 ms with one
// thread per sample, 2.7 ms with groups of 8 lanes for one corner, 2.03 ms like this (the bytes alone, 1.3 GB, would
// take about 0.25 ms; the atomic requests are what is left). Runs of at most 16 / 32 / 64 samples: 2.06 / 2.03 / 2.04.
constexpr int kGsThreads = 256;
constexpr int kGsRun     = 32;   // samples of a lane group, at most
constexpr int kGsTile    = kGsThreads / 8 * kGsRun;  // samples of a block, at most (groups of 8 lanes: CL = 4)

template <int CL>
__global__ void __launch_bounds__(kGsThreads) k_gs3d_bwd_cl(GridArgs g, const int64_t* __restrict__ index,
                                                            const float* __restrict__ uv, int64_t S, int32_t run,
                                                            bool vec4, const float* __restrict__ grad_out,
                                                            float* __restrict__ grad_grid, float* __restrict__ grad_uv)
{
    __shared__ float s_x[3][kGsTile];  // grid coordinates
    __shared__ int32_t s_n[kGsTile];   // slot, -1: outside the grid
    const int32_t tile = kGsThreads / (2 * CL) * run;
    const int64_t i0   = (int64_t)blockIdx.x * tile;
    const int32_t ns = (int32_t)min<int64_t>(tile, S - i0);
    for (int32_t j = threadIdx.x; j < ns; j += kGsThreads)
    {
        const int64_t i = i0 + j;
        const int64_t n = index[i];
        const bool in   = n >= 0 && n < g.N;
        s_n[j]          = in ? (int32_t)n : -1;
        if (!in)
        {
            if (grad_uv) grad_uv[3 * i] = grad_uv[3 * i + 1] = grad_uv[3 * i + 2] = 0.f;
            continue;
        }
        const Tri t = trilinear(g, n, uv[3 * i], uv[3 * i + 1], uv[3 * i + 2]);
        s_x[0][j]   = t.ix;
        s_x[1][j]   = t.iy;
        s_x[2][j]   = t.iz;
        if (!grad_uv) continue;
        float d[8] = {};
        for (int c = 0; c < g.C; c += 4)
        {
            float go[4];
            if (vec4)
            {
                const float4 v = *reinterpret_cast<const float4*>(grad_out + i * g.C + c);
                go[0] = v.x; go[1] = v.y; go[2] = v.z; go[3] = v.w;
            }
            else
            {
#pragma unroll
                for (int q = 0; q < 4; ++q) go[q] = grad_out[i * g.C + c + q];
            }
#pragma unroll
            for (int k = 0; k < 8; ++k)
            {
                float v[4];
                if (vec4)
                {
                    const float4 f = *reinterpret_cast<const float4*>(g.grid + t.off[k] + c);
                    v[0] = f.x; v[1] = f.y; v[2] = f.z; v[3] = f.w;
                }
                else
                {
#pragma unroll
                    for (int q = 0; q < 4; ++q) v[q] = g.grid[t.off[k] + c + q];
                }
#pragma unroll
                for (int q = 0; q < 4; ++q) d[k] = fmaf(v[q], go[q], d[k]);
            }
        }
        const float fx1 = t.ix - (float)t.x0, fx0 = (float)(t.x0 + 1) - t.ix;
        const float fy1 = t.iy - (float)t.y0, fy0 = (float)(t.y0 + 1) - t.iy;
        const float fz1 = t.iz - (float)t.z0, fz0 = (float)(t.z0 + 1) - t.iz;
        // corner k takes the upper neighbour on x / y / z iff bit 0 / 1 / 2 of k is set
        const float gx = ((d[1] - d[0]) * fy0 + (d[3] - d[2]) * fy1) * fz0 +
                         ((d[5] - d[4]) * fy0 + (d[7] - d[6]) * fy1) * fz1;
        const float gy = ((d[2] - d[0]) * fx0 + (d[3] - d[1]) * fx1) * fz0 +
                         ((d[6] - d[4]) * fx0 + (d[7] - d[5]) * fx1) * fz1;
        const float gz = ((d[4] - d[0]) * fx0 + (d[5] - d[1]) * fx1) * fy0 +
                         ((d[6] - d[2]) * fx0 + (d[7] - d[3]) * fx1) * fy1;
        grad_uv[3 * i + 0] = gx * (float)(g.X - 1) / 2;
        grad_uv[3 * i + 1] = gy * (float)(g.Y - 1) / 2;
        grad_uv[3 * i + 2] = gz * (float)(g.Z - 1) / 2;
    }
    if (!grad_grid) return;
    __syncthreads();
    const int32_t ch = threadIdx.x % CL, xb = (threadIdx.x / CL) & 1;
    const int32_t j0 = (int32_t)(threadIdx.x / (2 * CL)) * run, j1 = min(ns, j0 + run);
    for (int32_t c = ch; c < g.C; c += CL)
    {
        float acc[4];  // corners (y0, z0), (y1, z0), (y0, z1), (y1, z1) of this lane's x and channel
        int32_t cn = -1, cx = 0, cy = 0, cz = 0;  // the cell whose sums acc holds (cn < 0: none)
        auto flush = [&]() {
            float* base = grad_grid + cn * g.s0 + clip_i(cx + xb, g.X) * g.s4 + c;
            const int64_t oy[2] = {clip_i(cy, g.Y) * g.s3, clip_i(cy + 1, g.Y) * g.s3};
            const int64_t oz[2] = {clip_i(cz, g.Z) * g.s2, clip_i(cz + 1, g.Z) * g.s2};
#pragma unroll
            for (int k = 0; k < 4; ++k) atomicAdd(base + oz[k >> 1] + oy[k & 1], acc[k]);
        };
        for (int32_t j = j0; j < j1; ++j)
        {
            const int32_t n = s_n[j];
            if (n < 0) continue;
            const float ix = s_x[0][j], iy = s_x[1][j], iz = s_x[2][j];
            const float go = grad_out[(i0 + j) * g.C + c];
            const int32_t x0 = (int)floorf(ix), y0 = (int)floorf(iy), z0 = (int)floorf(iz);
            if (n != cn || x0 != cx || y0 != cy || z0 != cz)
            {
                if (cn >= 0) flush();
                cn = n;
                cx = x0;
                cy = y0;
                cz = z0;
#pragma unroll
                for (int k = 0; k < 4; ++k) acc[k] = 0.f;
            }
            const float fx    = xb ? ix - (float)x0 : (float)(x0 + 1) - ix;
            const float fy[2] = {(float)(y0 + 1) - iy, iy - (float)y0};
            const float fz[2] = {(float)(z0 + 1) - iz, iz - (float)z0};
#pragma unroll
            for (int k = 0; k < 4; ++k) acc[k] += fx * fy[k & 1] * fz[k >> 1] * go;
        }
        if (cn >= 0) flush();
    }
}

}  // namespace neat

using namespace neat;

static int make_grid_args(GridArgs& g, const float* grid, int64_t N, int32_t C, int32_t Z, int32_t Y, int32_t X,
                          const int64_t* strides)
{
    NEAT_REQUIRE(grid && strides, "grid and strides must not be null");
    NEAT_REQUIRE(N > 0 && C > 0 && Z > 0 && Y > 0 && X > 0, "grid dims must be positive");
    g = GridArgs{grid, strides[0], strides[1], strides[2], strides[3], strides[4], N, C, Z, Y, X};
    return NEAT_OK;
}

static bool channels_last(const GridArgs& g)
{
    return g.s1 == 1 && g.C % 4 == 0 && g.s4 % 4 == 0 && g.s3 % 4 == 0 && g.s2 % 4 == 0 && g.s0 % 4 == 0 &&
           (reinterpret_cast<uintptr_t>(g.grid) % 16) == 0;
}

extern "C"
{
    int neat_gs3d_fwd(neat_stream_t stream, const float* grid, int64_t N, int32_t C, int32_t Z, int32_t Y, int32_t X,
                      const int64_t* strides, const int64_t* index, const float* uv, int64_t S, float* out)
    {
        GridArgs g;
        int st = make_grid_args(g, grid, N, C, Z, Y, X, strides);
        if (st) return st;
        NEAT_REQUIRE(S >= 0, "num_samples < 0");
        if (S == 0) return NEAT_OK;
        NEAT_REQUIRE(index && uv && out, "neat_gs3d_fwd: null pointer");
        hipStream_t s = as_stream(stream);
        const bool cl = channels_last(g) && (reinterpret_cast<uintptr_t>(out) % 16) == 0;
        if (cl && C % 8 == 0 && S < INT32_MAX - 256)  // a launch holds fewer than 2^32 threads
            k_gs3d_fwd<true, 2><<<grid_for(2 * S, 256), 256, 0, s>>>(g, index, uv, S, out);
        else if (cl)
            k_gs3d_fwd<true><<<grid_for(S, 256), 256, 0, s>>>(g, index, uv, S, out);
        else
            k_gs3d_fwd<false><<<grid_for(S, 256), 256, 0, s>>>(g, index, uv, S, out);
        NEAT_LAUNCHED();
        return NEAT_OK;
    }

    int neat_gs3d_bwd(neat_stream_t stream, const float* grid, int64_t N, int32_t C, int32_t Z, int32_t Y, int32_t X,
                      const int64_t* strides, const int64_t* index, const float* uv, int64_t S, const float* grad_out,
                      float* grad_grid, float* grad_uv)
    {
        GridArgs g;
        int st = make_grid_args(g, grid, N, C, Z, Y, X, strides);
        if (st) return st;
        NEAT_REQUIRE(S >= 0, "num_samples < 0");
        if (S == 0) return NEAT_OK;
        NEAT_REQUIRE(index && uv && grad_out, "neat_gs3d_bwd: null pointer");
        hipStream_t s = as_stream(stream);
        if (g.s1 == 1 && C % 4 == 0 && N < INT32_MAX)
        {
            // lane groups for 8 (or 4) consecutive channels; runs of up to 32 samples while 2048 blocks remain
            const int32_t CL = C % 8 == 0 ? 8 : 4, groups = kGsThreads / (2 * CL);
            int32_t run      = 4;
            while (run < kGsRun && S >= (int64_t)2048 * groups * run * 2) run *= 2;
            const unsigned nb   = (unsigned)((S + (int64_t)groups * run - 1) / ((int64_t)groups * run));
            const bool vec4     = channels_last(g) && (reinterpret_cast<uintptr_t>(grad_out) % 16) == 0;
            if (CL == 8)
                k_gs3d_bwd_cl<8><<<nb, kGsThreads, 0, s>>>(g, index, uv, S, run, vec4, grad_out, grad_grid, grad_uv);
            else
                k_gs3d_bwd_cl<4><<<nb, kGsThreads, 0, s>>>(g, index, uv, S, run, vec4, grad_out, grad_grid, grad_uv);
        }
        else
        {
            k_gs3d_bwd<<<grid_for(S, 256), 256, 0, s>>>(g, index, uv, S, grad_out, grad_grid, grad_uv);
        }
        NEAT_LAUNCHED();
        return NEAT_OK;
    }
}
