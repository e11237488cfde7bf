// Exact residual ||X - Xhat||^2 and ||X||^2 over row-sorted views and dense
// tile pools, plus the factor unpermutation of the export path.
//
// The model value of an element follows common.cu:303-334: sums over the even
// and the odd ranks, each term (a*b*c)*lambda_r, pred = p0 + p1.
// Per-workgroup partials are summed in a fixed order (deterministic).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "../host/hip_util.hpp"

namespace {

constexpr int THREADS = 256;

// A lane group of LPE lanes takes an element, lane q of it the rank pairs q, q
// + LPE, ...: with a lane an element every load touches 64 lines.  p0 and p1
// are the even and the odd ranks' sums.  The whole call, a lane an element
// with one thread adding the partials -> this: 15.1 M nonzeros in dense tiles
// R = 8 339 -> 176 us, 16 529 -> 296, 25 567 -> 510, 32 841 -> 505, 100 1654 ->
// 1390; a view of 2 M power-law nonzeros R = 8 131 -> 51, 32 230 -> 98, 64 354
// -> 158; 3 M flatter ones R = 32 512 -> 160.
template <int LPE>
__device__ double model_value(const double* __restrict__ pa, const double* __restrict__ pb,
                              const double* __restrict__ pc, const double* __restrict__ lam, int R,
                              int q)
{
    double p0 = 0.0, p1 = 0.0;
    int r = 2 * q;
    // whole pairs only: a condition on the second rank keeps the compiler from
    // joining a row's two loads
    for (; r + 1 < R; r += 2 * LPE)
    {
        double x0 = pa[r] * pb[r] * pc[r];
        double x1 = pa[r + 1] * pb[r + 1] * pc[r + 1];
        if (lam)
        {
            x0 *= lam[r];
            x1 *= lam[r + 1];
        }
        p0 += x0;
        p1 += x1;
    }
    if (r < R)   // the last rank of an odd R
    {
        double x = pa[r] * pb[r] * pc[r];
        if (lam) x *= lam[r];
        p0 += x;
    }
    double p = p0 + p1;
#pragma unroll
    for (int o = 1; o < LPE; o <<= 1) p += __shfl_xor(p, o, 64);
    return p;
}

__device__ void block_sum2(double a, double b, double* __restrict__ out2)
{
    __shared__ double ra[THREADS], rb[THREADS];
    ra[threadIdx.x] = a;
    rb[threadIdx.x] = b;
    __syncthreads();
    for (int off = THREADS / 2; off > 0; off >>= 1)
    {
        if (int(threadIdx.x) < off)
        {
            ra[threadIdx.x] += ra[threadIdx.x + off];
            rb[threadIdx.x] += rb[threadIdx.x + off];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0)
    {
        out2[0] = ra[0];
        out2[1] = rb[0];
    }
}

template <int LPE>
__global__ __launch_bounds__(THREADS) void residual_view_kernel(
    const uint64_t* __restrict__ coords, const double* __restrict__ vals, size_t nnz,
    const double* __restrict__ A, const double* __restrict__ B, const double* __restrict__ C,
    const double* __restrict__ lam, int R, double* __restrict__ part)
{
    constexpr int EPB = THREADS / LPE;
    double res = 0.0, xx = 0.0;
    const int q = int(threadIdx.x) % LPE;
    for (size_t e = size_t(blockIdx.x) * EPB + threadIdx.x / LPE; e < nnz;
         e += size_t(gridDim.x) * EPB)
    {
        const uint64_t pc = coords[e];
        const double v = vals[e];
        const uint32_t i = uint32_t(pc >> 30) & 0x7FFFu, j = uint32_t(pc >> 15) & 0x7FFFu,
                       k = uint32_t(pc) & 0x7FFFu;
        const double d = v - model_value<LPE>(A + size_t(i) * R, B + size_t(j) * R,
                                              C + size_t(k) * R, lam, R, q);
        if (q == 0)
        {
            res += d * d;
            xx += v * v;
        }
    }
    block_sum2(res, xx, part + 2 * size_t(blockIdx.x));
}

template <int LPE>
__global__ __launch_bounds__(THREADS) void residual_tiles_kernel(
    const int32_t* __restrict__ tiles4, const uint64_t* __restrict__ off,
    const int32_t* __restrict__ lid, const double* __restrict__ pval, size_t ntiles,
    const double* __restrict__ A, const double* __restrict__ B, const double* __restrict__ C,
    const double* __restrict__ lam, int R, double* __restrict__ part)
{
    constexpr int EPB = THREADS / LPE;
    double res = 0.0, xx = 0.0;
    const int q = int(threadIdx.x) % LPE;
    for (size_t t = blockIdx.x; t < ntiles; t += gridDim.x)
    {
        const int b0 = tiles4[4 * t] * 16, b1 = tiles4[4 * t + 1] * 16, b2 = tiles4[4 * t + 2] * 16;
        for (uint64_t e = off[t] + threadIdx.x / LPE; e < off[t + 1]; e += EPB)
        {
            const int l = lid[e];
            const double v = pval[e];
            const size_t i = size_t(b0 + (l >> 8)), j = size_t(b1 + ((l >> 4) & 15)),
                         k = size_t(b2 + (l & 15));
            const double d = v - model_value<LPE>(A + i * R, B + j * R, C + k * R, lam, R, q);
            if (q == 0)
            {
                res += d * d;
                xx += v * v;
            }
        }
    }
    block_sum2(res, xx, part + 2 * size_t(blockIdx.x));
}

// out2 += the P partials' sums, in a fixed order.  One thread adding them in
// turn took 95 us for 2048 partials (a load's latency each).
__global__ __launch_bounds__(THREADS) void finalize_add_kernel(const double* __restrict__ part,
                                                               int P, double* __restrict__ out2)
{
    __shared__ double t[2];
    double a = 0.0, b = 0.0;
    for (int p = threadIdx.x; p < P; p += THREADS)
    {
        a += part[2 * p];
        b += part[2 * p + 1];
    }
    block_sum2(a, b, t);
    if (threadIdx.x != 0) return;
    out2[0] += t[0];
    out2[1] += t[1];
}

__global__ void unpermute_kernel(const double* __restrict__ src, double* __restrict__ dst,
                                 const int32_t* __restrict__ perm, size_t dim, int R)
{
    const size_t total = dim * size_t(R);
    const size_t stride = size_t(gridDim.x) * blockDim.x;
    for (size_t x = size_t(blockIdx.x) * blockDim.x + threadIdx.x; x < total; x += stride)
    {
        const size_t old = x / size_t(R);
        const int r = int(x % size_t(R));
        dst[x] = src[size_t(perm[old]) * R + r];
    }
}

// lanes an element.  The whole call at 1 / 2 / 4 lanes: 15.1 M nonzeros in
// dense tiles (rows from L1) R = 4 100 / 114 / 189 us, 8 178 / 176 / 193, 12
// 225 / 230 / 290, 16 373 / 319 / 296, 32 685 / 585 / 505; 3 M flat power-law
// nonzeros in a view R = 4 71 / 57 / 66, 8 115 / 80 / 68, 12 160 / 104 / 102,
// 16 211 / 128 / 97, 32 390 / 234 / 160 (more lanes, fewer lines a load, but
// fewer elements in flight and more shuffles)
template <class Run>
void residual_lanes(int R, Run run)
{
    if (R <= 12) run(std::integral_constant<int, 2>{});
    else run(std::integral_constant<int, 4>{});
}

}  // namespace

extern "C" int cptc_residual3_view(const uint64_t* d_coords, const double* d_vals, size_t nnz,
                                   const double* d_A, const double* d_B, const double* d_C,
                                   const double* d_lambda, int R, double* d_out2, void* stream)
{
    CPTC_REQUIRE(R >= 1 && d_A && d_B && d_C && d_out2, CPTC_ERR_ARG,
                 "cptc_residual3_view: bad arguments");
    if (nnz == 0) return CPTC_OK;
    CPTC_REQUIRE(d_coords && d_vals, CPTC_ERR_ARG, "cptc_residual3_view: null view");
    hipStream_t s = cptc::as_stream(stream);
    const int P = int(cptc::grid_for(nnz, THREADS, 2048));
    void* buf = nullptr;
    CPTC_TRY(cptc::scratch_get(cptc::SCR_REDUCE, size_t(P) * 2 * sizeof(double), &buf));
    double* part = static_cast<double*>(buf);
    residual_lanes(R, [&](auto L) {
        hipLaunchKernelGGL(residual_view_kernel<decltype(L)::value>, dim3(P), dim3(THREADS), 0, s,
                           d_coords, d_vals, nnz, d_A, d_B, d_C, d_lambda, R, part);
    });
    CPTC_LAUNCHED();
    hipLaunchKernelGGL(finalize_add_kernel, dim3(1), dim3(THREADS), 0, s, part, P, d_out2);
    CPTC_LAUNCHED();
    return CPTC_OK;
}

extern "C" int cptc_residual3_tiles(const int32_t* d_tiles, const uint64_t* d_pool_off,
                                    const int32_t* d_pool_lid, const double* d_pool_val,
                                    size_t ntiles, const double* d_A, const double* d_B,
                                    const double* d_C, const double* d_lambda, int R,
                                    double* d_out2, void* stream)
{
    CPTC_REQUIRE(R >= 1 && d_A && d_B && d_C && d_out2, CPTC_ERR_ARG,
                 "cptc_residual3_tiles: bad arguments");
    if (ntiles == 0) return CPTC_OK;
    CPTC_REQUIRE(d_tiles && d_pool_off && d_pool_lid && d_pool_val, CPTC_ERR_ARG,
                 "cptc_residual3_tiles: null pool");
    hipStream_t s = cptc::as_stream(stream);
    const int P = int(ntiles < 2048 ? ntiles : 2048);
    void* buf = nullptr;
    CPTC_TRY(cptc::scratch_get(cptc::SCR_REDUCE, size_t(P) * 2 * sizeof(double), &buf));
    double* part = static_cast<double*>(buf);
    residual_lanes(R, [&](auto L) {
        hipLaunchKernelGGL(residual_tiles_kernel<decltype(L)::value>, dim3(P), dim3(THREADS), 0, s,
                           d_tiles, d_pool_off, d_pool_lid, d_pool_val, ntiles, d_A, d_B, d_C,
                           d_lambda, R, part);
    });
    CPTC_LAUNCHED();
    hipLaunchKernelGGL(finalize_add_kernel, dim3(1), dim3(THREADS), 0, s, part, P, d_out2);
    CPTC_LAUNCHED();
    return CPTC_OK;
}

extern "C" int cptc_unpermute_factor(const double* d_perm_factor, double* d_orig,
                                     const int32_t* d_perm, size_t dim, int R, void* stream)
{
    CPTC_REQUIRE(R >= 1 && d_perm_factor && d_orig && d_perm, CPTC_ERR_ARG,
                 "cptc_unpermute_factor: bad arguments");
    if (dim == 0) return CPTC_OK;
    hipLaunchKernelGGL(unpermute_kernel, dim3(cptc::grid_for(dim * size_t(R), 256, 4096)),
                       dim3(256), 0, cptc::as_stream(stream), d_perm_factor, d_orig, d_perm, dim,
                       R);
    CPTC_LAUNCHED();
    return CPTC_OK;
}
