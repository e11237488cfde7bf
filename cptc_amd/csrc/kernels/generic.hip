// Kernels of the generic N-order CP-ALS path for CDNA4 (wave64): the FP64
// segment MTTKRP, dense-unit packing and outer weights, the Gram Hadamard,
// the ridge Cholesky solve, column normalisation and the exact residual.
// The dense-unit MFMA contraction shares dense_tiles.hip with order 3.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "../host/hip_util.hpp"
#include "block_sweep.hpp"

namespace {

constexpr int WAVE = 64;
constexpr int MAXM = CPTC_MAX_MODES;

struct Factors
{
    const double* p[MAXM];
};

template <int VEC>
struct Row;
template <>
struct Row<2>
{
    double x[2];
    __device__ void load(const double* __restrict__ q)
    {
        const double2 v = *reinterpret_cast<const double2*>(q);
        x[0] = v.x;
        x[1] = v.y;
    }
};
template <>
struct Row<1>
{
    double x[1];
    __device__ void load(const double* __restrict__ q) { x[0] = *q; }
};

// ------------------------------------------------------ segment MTTKRP --
//
// One workgroup (4 waves) per row segment.  A lane owns VEC consecutive
// ranks; LPE = RT / VEC lanes cover one element, so a wave carries
// EPW = 64 / LPE element slots (R = 32 -> 4, 16 -> 8, 8 -> 16).  Each slot
// walks a contiguous chunk of the segment.
//
// The segment's other coordinates come in NO = N - 1 levels (the view's row
// order, G[q] = factor of level q).  The slot evaluates the sum as a tree
// over equal coordinate prefixes (the CSF form of the MTTKRP):
//   acc = sum_{o0} G0[o0] * sum_{o1} G1[o1] * ... * sum_{o_last} v * G_last[o_last]
// t[k] holds the open partial sum under the current prefix o0..ok; when
// o_k changes, levels deeper than k-1 are closed (t[k] * G_k[cur_k] is
// added one level up).  Each factor row is therefore gathered once per run
// of its prefix; in a view without runs this is one gather per level per
// element, the plain product.  Skipped (dense) elements touch nothing.
template <int N, int RT, int VEC, int UNROLL>
__global__ __launch_bounds__(256) void seg_nd_kernel(
    Factors F, const uint32_t* __restrict__ sc, uint64_t nnz,
    const double* __restrict__ vals, const uint8_t* __restrict__ skip,
    const uint32_t* __restrict__ seg_row, const uint32_t* __restrict__ seg_start,
    const uint32_t* __restrict__ seg_cnt, const uint8_t* __restrict__ single,
    double* __restrict__ FtV, int R)
{
    constexpr int NO = N - 1;                // levels
    constexpr int NL = (NO > 1) ? NO - 1 : 1; // run levels (0 .. NO-2)
    constexpr int LPE = RT / VEC;
    constexpr int EPW = WAVE / LPE;
    constexpr int WAVES = 4;
    constexpr int SLOTS = EPW * WAVES;

    const uint32_t seg = blockIdx.x;
    const uint32_t row = seg_row[seg];
    const uint32_t start = seg_start[seg];
    const uint32_t cnt = seg_cnt[seg];

    const int tid = threadIdx.x;
    const int lane = tid & (WAVE - 1);
    const int wave = tid / WAVE;
    const int slot = lane / LPE;
    const int r0 = (lane % LPE) * VEC;
    const bool rank_ok = r0 < R;
    const int rr = rank_ok ? r0 : 0;

    const uint32_t g = uint32_t(wave * EPW + slot);
    const uint32_t chunk = (cnt + SLOTS - 1) / SLOTS;
    uint32_t lo = start + g * chunk;
    const uint32_t hi = (g * chunk + chunk < cnt) ? lo + chunk : start + cnt;
    if (lo > hi) lo = hi;

    double acc[VEC];
    double t[NL][VEC];
    uint32_t cur[NL];
#pragma unroll
    for (int k = 0; k < VEC; ++k) acc[k] = 0.0;
#pragma unroll
    for (int l = 0; l < NL; ++l)
    {
        cur[l] = 0;
#pragma unroll
        for (int k = 0; k < VEC; ++k) t[l][k] = 0.0;
    }
    bool open = false;

    // close run levels from NO-2 down to `to` (all of them when to == 0)
    auto close_levels = [&](int to) {
#pragma unroll
        for (int l = NL - 1; l >= 0; --l)
        {
            if (l < to) break;
            Row<VEC> f;
            f.load(F.p[l] + size_t(cur[l]) * R + rr);
#pragma unroll
            for (int k = 0; k < VEC; ++k)
            {
                const double x = t[l][k] * f.x[k];
                if (l == 0)
                    acc[k] += x;
                else
                    t[l - 1][k] += x;
                t[l][k] = 0.0;
            }
        }
    };

    // one live element: coordinates o[0..NO-1], value-weighted last-level row p
    auto consume = [&](const uint32_t* o, const double* p) {
        if constexpr (NO == 1)
        {
#pragma unroll
            for (int k = 0; k < VEC; ++k) acc[k] += p[k];
        }
        else
        {
            int L = NL;
            if (!open)
            {
                L = 0;
                open = true;
            }
            else
            {
#pragma unroll
                for (int l = NL - 1; l >= 0; --l)
                    if (o[l] != cur[l]) L = l;
                if (L < NL) close_levels(L);
            }
#pragma unroll
            for (int l = 0; l < NL; ++l)
                if (l >= L) cur[l] = o[l];
#pragma unroll
            for (int k = 0; k < VEC; ++k) t[NL - 1][k] += p[k];
        }
    };

    uint32_t e = lo;
    for (; e + UNROLL <= hi; e += UNROLL)
    {
        uint32_t c[UNROLL][NO];
        double v[UNROLL];
        bool live[UNROLL];
#pragma unroll
        for (int u = 0; u < UNROLL; ++u)
        {
            v[u] = __builtin_nontemporal_load(vals + e + u);
            live[u] = skip ? (__builtin_nontemporal_load(skip + e + u) == 0) : true;
#pragma unroll
            for (int q = 0; q < NO; ++q) c[u][q] = __builtin_nontemporal_load(sc + q * nnz + e + u);
        }
        double p[UNROLL][VEC];
#pragma unroll
        for (int u = 0; u < UNROLL; ++u)
        {
            Row<VEC> f;
            if (live[u])
                f.load(F.p[NO - 1] + size_t(c[u][NO - 1]) * R + rr);
#pragma unroll
            for (int k = 0; k < VEC; ++k) p[u][k] = live[u] ? v[u] * f.x[k] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < UNROLL; ++u)
            if (live[u]) consume(c[u], p[u]);
    }
    for (; e < hi; ++e)
    {
        if (skip && __builtin_nontemporal_load(skip + e) != 0) continue;
        uint32_t c[NO];
#pragma unroll
        for (int q = 0; q < NO; ++q) c[q] = __builtin_nontemporal_load(sc + q * nnz + e);
        const double v = __builtin_nontemporal_load(vals + e);
        Row<VEC> f;
        f.load(F.p[NO - 1] + size_t(c[NO - 1]) * R + rr);
        double p[VEC];
#pragma unroll
        for (int k = 0; k < VEC; ++k) p[k] = v * f.x[k];
        consume(c, p);
    }
    if constexpr (NO > 1)
        if (open) close_levels(0);
    if (!rank_ok)
#pragma unroll
        for (int k = 0; k < VEC; ++k) acc[k] = 0.0;

#pragma unroll
    for (int off = LPE; off < WAVE; off <<= 1)
#pragma unroll
        for (int k = 0; k < VEC; ++k) acc[k] += __shfl_xor(acc[k], off, WAVE);

    __shared__ double red[WAVES][RT];
    if (slot == 0)
#pragma unroll
        for (int k = 0; k < VEC; ++k) red[wave][r0 + k] = acc[k];
    __syncthreads();
    const bool store = single && single[seg] != 0;
    for (int x = tid; x < R; x += WAVE * WAVES)
    {
        double tot = 0.0;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) tot += red[w][x];
        double* out = FtV + size_t(row) * R + x;
        if (store)
            *out = tot;
        else if (tot != 0.0)
            atomicAdd(out, tot);
    }
}

template <int N, int RT, int VEC>
void launch_seg(const Factors& F, int mode, const uint32_t* sc, uint64_t nnz, const double* vals,
                const uint8_t* skip, const uint32_t* row, const uint32_t* st, const uint32_t* cn,
                const uint8_t* single, uint64_t nseg, double* FtV, int R, hipStream_t s)
{
    (void)mode;
    constexpr int UNROLL = (N <= 4) ? 4 : 2;
    hipLaunchKernelGGL((seg_nd_kernel<N, RT, VEC, UNROLL>), dim3(unsigned(nseg)), dim3(256), 0, s,
                       F, sc, nnz, vals, skip, row, st, cn, single, FtV, R);
}

template <int N, int VEC>
void launch_seg_r(const Factors& F, int mode, const uint32_t* sc, uint64_t nnz,
                  const double* vals, const uint8_t* skip, const uint32_t* row, const uint32_t* st,
                  const uint32_t* cn, const uint8_t* single, uint64_t nseg, double* FtV, int R,
                  hipStream_t s)
{
    if (R <= 8)
        launch_seg<N, 8, VEC>(F, mode, sc, nnz, vals, skip, row, st, cn, single, nseg, FtV, R, s);
    else if (R <= 16)
        launch_seg<N, 16, VEC>(F, mode, sc, nnz, vals, skip, row, st, cn, single, nseg, FtV, R, s);
    else
        launch_seg<N, 32, VEC>(F, mode, sc, nnz, vals, skip, row, st, cn, single, nseg, FtV, R, s);
}

template <int VEC>
void launch_seg_n(int N, const Factors& F, int mode, const uint32_t* sc, uint64_t nnz,
                  const double* vals, const uint8_t* skip, const uint32_t* row,
                  const uint32_t* st, const uint32_t* cn, const uint8_t* single, uint64_t nseg,
                  double* FtV, int R, hipStream_t s)
{
    switch (N)
    {
    case 2: launch_seg_r<2, VEC>(F, mode, sc, nnz, vals, skip, row, st, cn, single, nseg, FtV, R, s); break;
    case 3: launch_seg_r<3, VEC>(F, mode, sc, nnz, vals, skip, row, st, cn, single, nseg, FtV, R, s); break;
    case 4: launch_seg_r<4, VEC>(F, mode, sc, nnz, vals, skip, row, st, cn, single, nseg, FtV, R, s); break;
    case 5: launch_seg_r<5, VEC>(F, mode, sc, nnz, vals, skip, row, st, cn, single, nseg, FtV, R, s); break;
    case 6: launch_seg_r<6, VEC>(F, mode, sc, nnz, vals, skip, row, st, cn, single, nseg, FtV, R, s); break;
    case 7: launch_seg_r<7, VEC>(F, mode, sc, nnz, vals, skip, row, st, cn, single, nseg, FtV, R, s); break;
    default: launch_seg_r<8, VEC>(F, mode, sc, nnz, vals, skip, row, st, cn, single, nseg, FtV, R, s); break;
    }
}

// ------------------------------------------------------------ dense units --

// One workgroup per unit: FP64 accumulation in LDS (duplicates summed), one
// rounding to FP32 per cell.
__global__ __launch_bounds__(256) void units_pack_kernel(const uint32_t* __restrict__ unit6,
                                                         const uint32_t* __restrict__ lid,
                                                         const double* __restrict__ val,
                                                         float* __restrict__ tiles)
{
    __shared__ double T[4096];
    const size_t u = blockIdx.x;
    for (int c = threadIdx.x; c < 4096; c += 256) T[c] = 0.0;
    __syncthreads();
    const uint32_t n = unit6[6 * u + 3], st = unit6[6 * u + 4];
    for (uint32_t e = threadIdx.x; e < n; e += 256) atomicAdd(&T[lid[st + e] & 4095u], val[st + e]);
    __syncthreads();
    float4* out = reinterpret_cast<float4*>(tiles + u * 4096);
    for (int c = threadIdx.x; c < 1024; c += 256)
        out[c] = make_float4(float(T[4 * c]), float(T[4 * c + 1]), float(T[4 * c + 2]),
                             float(T[4 * c + 3]));
}

// The same cells in FP64 (the per-unit sums' operand): one workgroup per
// unit, FP64 accumulation in LDS (duplicates summed), written as doubles.
__global__ __launch_bounds__(256) void units_pack_f64_kernel(const uint32_t* __restrict__ unit6,
                                                             const uint32_t* __restrict__ lid,
                                                             const double* __restrict__ val,
                                                             double* __restrict__ img)
{
    __shared__ double T[4096];
    const size_t u = blockIdx.x;
    for (int c = threadIdx.x; c < 4096; c += 256) T[c] = 0.0;
    __syncthreads();
    const uint32_t n = unit6[6 * u + 3], st = unit6[6 * u + 4];
    for (uint32_t e = threadIdx.x; e < n; e += 256) atomicAdd(&T[lid[st + e] & 4095u], val[st + e]);
    __syncthreads();
    double2* out = reinterpret_cast<double2*>(img + u * 4096);
    for (int c = threadIdx.x; c < 2048; c += 256) out[c] = make_double2(T[2 * c], T[2 * c + 1]);
}

__global__ void units_weights_kernel(const uint32_t* __restrict__ unit6, uint64_t nunits,
                                     const uint32_t* __restrict__ oc, int nouter, Factors Fo,
                                     int R, double* __restrict__ W)
{
    const uint64_t total = nunits * uint64_t(R);
    const uint64_t stride = uint64_t(gridDim.x) * blockDim.x;
    for (uint64_t x = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; x < total; x += stride)
    {
        const uint64_t u = x / R;
        const int r = int(x % R);
        const uint32_t off = unit6[6 * u + 5];
        double w = 1.0;
#pragma unroll
        for (int k = 0; k < MAXM; ++k)
            if (k < nouter) w *= Fo.p[k][size_t(oc[off + k]) * R + r];
        W[x] = w;
    }
}

// ------------------------------------------------------------- small R x R --

__global__ void gram_hadamard_kernel(const double* __restrict__ G, int ngram, int skip, int RR,
                                     double* __restrict__ out)
{
    for (int x = blockIdx.x * blockDim.x + threadIdx.x; x < RR; x += gridDim.x * blockDim.x)
    {
        double v = 1.0;
        for (int g = 0; g < ngram; ++g)
            if (g != skip) v *= G[size_t(g) * RR + x];
        out[x] = v;
    }
}

// Ridge solve F (FtF + eps I) = FtV (generic.cu:746-819), R <= 32, eps =
// 1e-12 tr / R + 1e-300: a Cholesky factor L and two triangular solves a row.
//
// What bounds it is the chain of R pivots in one wave: there is little to
// compute (R^3 / 3 + 2 R^2 a row) and a launch has few workgroups.  Row by
// row substitutions would add 2 R more steps of that kind, so the solves are
// products instead: with X_i the inverse of diagonal block i of L (16 x 16),
// which comes out of the elimination beside L (the same row operations on the
// identity),
//   Y_1 = B_1 X_1^T,  Y_2 = (B_2 - Y_1 L_21^T) X_2^T,
//   Z_2 = Y_2 X_2,    Z_1 = (Y_1 - Z_2 L_21) X_1,
// six 16 x 16 x 16 products a 16-row tile on the FP64 matrix cores (two for R
// <= 16), computed transposed: an accumulator is then the next product's B
// operand as it stands.  The forward error bound is that of substitution (eps
// |X| |L| a solve); measured against extended precision, a row a lane -> this:
// Hadamard Grams at R = 16 3.6e-16 -> 3.3e-16, at 32 5.0e-16 -> 4.8e-16,
// condition 1e8 the same.
// Wave 0 factors; all four waves solve a tile each.
//
// Measured, launches back to back, 1000 rows (a row a lane, straight-line
// steps with two LDS round trips, a root and a division each -> this): R = 9
// 8.2 -> 4.4 us, 16 10.3 -> 5.7, 17 18.8 -> 7.1, 32 22.7 -> 10.3; 1 M rows at
// R = 32 307 -> 145.
constexpr int CHOL_RM = 32;
constexpr int CHOL_T = 256;
constexpr int CHOL_ROWS = 64;   // right-hand sides a workgroup and pass
constexpr int CHOL_LD = cptc::bsweep::LD;

using cptc::bsweep::d4;

template <int NB>
struct RidgeLds
{
    double X[NB][16 * CHOL_LD];   // inverses of L's diagonal blocks
    double L21[16 * CHOL_LD];     // NB == 2 only
};

// x plus its copy N lanes round the row of 16 (DPP row_ror)
template <int N>
__device__ __forceinline__ double chol_ror_add(double x)
{
    const uint64_t u = __builtin_bit_cast(uint64_t, x);
    const uint32_t lo =
        uint32_t(__builtin_amdgcn_mov_dpp(int(uint32_t(u)), 0x120 + N, 0xf, 0xf, true));
    const uint32_t hi =
        uint32_t(__builtin_amdgcn_mov_dpp(int(uint32_t(u >> 32)), 0x120 + N, 0xf, 0xf, true));
    return x + __builtin_bit_cast(double, (uint64_t(hi) << 32) | lo);
}

// A pivot's quotients v / d from r = 1 / d rounded, corrected once by the
// exact residual: within an ulp, at half the latency of the division.  They
// depend on v and d alone, so a factor read back gives the same X_i as the
// elimination that made it.
__device__ __forceinline__ double chol_quot(double v, double d, double r)
{
    const double q = v * r;
    return fma(r, fma(-q, d, v), q);
}

// d for which they are used; other d take the division
__device__ __forceinline__ bool chol_mid(double d) { return d >= 0x1p-450 && d <= 0x1p500; }

// d = sqrt(p) by one reciprocal root and its exact residual, and r from that
// root by two more steps: the first leaves it within an ulp of 1 / d, the
// second rounds it (for a d of 52 one-bits either neighbour, as in recip_rn).
// For p in about [2^-900, 2^1000]; WIDE takes the general root.
template <bool WIDE>
struct Root
{
    double d, r;
    __device__ __forceinline__ explicit Root(double p)
    {
        if constexpr (WIDE)
        {
            d = sqrt(p);
            r = cptc::bsweep::recip_rn(d);
        }
        else
        {
            r = __builtin_amdgcn_rsq(p);
            r = fma(0.5 * r, fma(-(p * r), r, 1.0), r);
            r = fma(0.5 * r, fma(-(p * r), r, 1.0), r);
            d = p * r;
            d = fma(0.5 * r, fma(-d, d, p), d);
            r = fma(r, fma(-d, r, 1.0), r);
            r = fma(r, fma(-d, r, 1.0), r);
        }
    }
    __device__ __forceinline__ double over(double v) const
    {
        if constexpr (WIDE)
            if (!chol_mid(d)) return v / d;
        return chol_quot(v, d, r);
    }
};

// Columns K .. nv - 1 of a 16 x 16 block (accumulator layout: element v of
// lane l is entry (l / 16 + 4 v, l % 16)) to those of L, and x, the identity
// at K = 0, to L^-1; with BELOW, b, the block right of it, to L^-1 b, by the
// same row operations (as X b its error grew with the condition of the block:
// R = 32, kappa 1e8, 7.5e-10 in the solution against 2.3e-10).  A pivot s <= 0
// (or NaN) counts as eps.
template <int K, bool WIDE, bool BELOW>
__device__ __forceinline__ void chol16_from(double (&a)[4], double (&x)[4], double (&b)[4],
                                            int lr, int lk, double eps, int nv)
{
    using namespace cptc::bsweep;
    constexpr int VK = K / 4, QK = K % 4;
    const double s = readlane_d(a[VK], 16 * QK + K);
    const double ck = bperm_d(a[VK], 16 * QK + lr);   // entry (K, lr)
    const double xk = bperm_d(x[VK], 16 * QK + lr);
    const double bk = BELOW ? bperm_d(b[VK], 16 * QK + lr) : 0.0;
    const Root<WIDE> root((s > 0.0) ? s : eps);
    const double c = lr > K ? root.over(ck) : 0.0, xs = root.over(xk);
    const double bs = BELOW ? root.over(bk) : 0.0;
#pragma unroll
    for (int v = VK; v < 4; ++v)
    {
        // L_iK in the rows below K, 0 above
        const double f = root.over(v == VK ? row_bcast_d<K, (0xf << (QK + 1)) & 0xf>(a[v])
                                           : row_bcast_d<K, 0xf>(a[v]));
        a[v] = fma(-f, c, a[v]);
        x[v] = fma(-f, xs, x[v]);
        a[v] = (lr == K) ? ((v == VK && lk == QK) ? root.d : f) : a[v];
        if (v == VK) x[v] = (lk == QK) ? xs : x[v];
        if constexpr (BELOW)
        {
            b[v] = fma(-f, bs, b[v]);
            if (v == VK) b[v] = (lk == QK) ? bs : b[v];
        }
    }
    if constexpr (K + 1 < 16)
        if (K + 1 < nv) chol16_from<K + 1, WIDE, BELOW>(a, x, b, lr, lk, eps, nv);
}

// x = L^-1 for a given block of L, the same operations
template <int K>
__device__ __forceinline__ void inv16_from(const double (&a)[4], double (&x)[4], int lr, int lk,
                                           int nv)
{
    using namespace cptc::bsweep;
    constexpr int VK = K / 4, QK = K % 4;
    const double xk = bperm_d(x[VK], 16 * QK + lr), d = readlane_d(a[VK], 16 * QK + K);
    const double xs = chol_mid(d) ? chol_quot(xk, d, recip_rn(d)) : xk / d;
#pragma unroll
    for (int v = VK; v < 4; ++v)
    {
        const double f = v == VK ? row_bcast_d<K, (0xf << (QK + 1)) & 0xf>(a[v])
                                 : row_bcast_d<K, 0xf>(a[v]);
        x[v] = fma(-f, xs, x[v]);
        if (v == VK) x[v] = (lk == QK) ? xs : x[v];
    }
    if constexpr (K + 1 < 16)
        if (K + 1 < nv) inv16_from<K + 1>(a, x, lr, lk, nv);
}

__device__ __forceinline__ void chol_identity(double (&x)[4], int lr, int lk)
{
#pragma unroll
    for (int v = 0; v < 4; ++v) x[v] = (lk + 4 * v == lr) ? 1.0 : 0.0;
}

__device__ __forceinline__ void chol_put(double* m, const double (&x)[4], int lr, int lk)
{
#pragma unroll
    for (int v = 0; v < 4; ++v) m[(lk + 4 * v) * CHOL_LD + lr] = x[v];
}

// acc + M1^T M2 of blocks in the accumulator layout
__device__ __forceinline__ d4 chol_mul(const double (&m1)[4], const double (&m2)[4], d4 acc)
{
#pragma unroll
    for (int v = 0; v < 4; ++v)
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(m1[v], m2[v], acc, 0, 0, 0);
    return acc;
}

// Wave 0: FtF + eps I = L L^T.  To w: X, L21; with OUT, L to global.
template <int NB, bool WIDE, bool OUT>
__device__ __forceinline__ void chol_factor(const double* __restrict__ FtF, int R, double eps,
                                            int lr, int lk, double (&a)[NB][4], RidgeLds<NB>& w,
                                            double* __restrict__ Lout)
{
    double x[4], p[4];   // p: A_12, then L21^T
#pragma unroll
    for (int v = 0; v < 4; ++v)
        p[v] = (NB == 2 && 16 + lr < R) ? FtF[size_t(16 + lr) * R + lk + 4 * v] : 0.0;
    chol_identity(x, lr, lk);
    chol16_from<0, WIDE, NB == 2>(a[0], x, p, lr, lk, eps, min(R, 16));
    chol_put(w.X[0], x, lr, lk);
    if constexpr (NB == 2)
    {
        double n[4];
#pragma unroll
        for (int v = 0; v < 4; ++v)
        {
            n[v] = -p[v];
            w.L21[lr * CHOL_LD + lk + 4 * v] = p[v];
        }
        const d4 u = chol_mul(n, p, d4{a[1][0], a[1][1], a[1][2], a[1][3]});
#pragma unroll
        for (int v = 0; v < 4; ++v) a[1][v] = u[v];
        chol_identity(x, lr, lk);
        double none[4];
        chol16_from<0, WIDE, false>(a[1], x, none, lr, lk, eps, R - 16);
        chol_put(w.X[1], x, lr, lk);
        if constexpr (OUT)
#pragma unroll
            for (int v = 0; v < 4; ++v)
                if (16 + lr < R)
                {
                    Lout[size_t(lk + 4 * v) * R + 16 + lr] = 0.0;
                    Lout[size_t(16 + lr) * R + lk + 4 * v] = p[v];
                }
    }
    if constexpr (OUT)
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
            for (int v = 0; v < 4; ++v)
            {
                const int r = lk + 4 * v, row = 16 * i + r, col = 16 * i + lr;
                if (row < R && col < R) Lout[size_t(row) * R + col] = r >= lr ? a[i][v] : 0.0;
            }
}

// Workgroup-wide factorisation of the matrix given by FtF's lower triangle,
// ends with a barrier.
template <int NB, bool OUT>
__device__ __forceinline__ void chol_factor_all(const double* __restrict__ FtF, int R,
                                                RidgeLds<NB>& w, double* __restrict__ Lout)
{
    if (threadIdx.x < 64)
    {
        const int lane = threadIdx.x, lr = lane & 15, lk = lane >> 4;
        double a[NB][4];
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
            for (int v = 0; v < 4; ++v)
            {
                const int row = 16 * i + lk + 4 * v, col = 16 * i + lr;
                a[i][v] = (row < R && col < R)
                              ? FtF[size_t(max(row, col)) * R + min(row, col)]
                              : 0.0;
            }
        const double dg = lane < R ? FtF[size_t(lane) * R + lane] : 0.0;
        const double t =
            chol_ror_add<1>(chol_ror_add<2>(chol_ror_add<4>(chol_ror_add<8>(dg))));
        const double tr = cptc::bsweep::readlane_d(t, 0) + cptc::bsweep::readlane_d(t, 16);
        const double eps = 1e-12 * ((tr > 0.0) ? tr / double(R) : 1.0) + 1e-300;
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
            for (int v = 0; v < 4; ++v) a[i][v] += (lk + 4 * v == lr) ? eps : 0.0;
        // eps <= every pivot's scale, and cancellation leaves no less than
        // 2^-106 of it
        const bool fits = tr >= 0x1p-700 && __all(fabs(dg) <= 0x1p900);
        if (fits)
            chol_factor<NB, false, OUT>(FtF, R, eps, lr, lk, a, w, Lout);
        else
            chol_factor<NB, true, OUT>(FtF, R, eps, lr, lk, a, w, Lout);
    }
    __syncthreads();
}

// A 16-row tile's right-hand sides, transposed: element v of lane l is entry
// 16 i + l / 16 + 4 v of row `row` = first row + l % 16
template <int NB>
__device__ __forceinline__ void chol_load_rhs(const double* __restrict__ FtV, size_t dim, int R,
                                              size_t row, int lk, double (&y)[NB][4])
{
    const double* b = FtV + row * R;
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int v = 0; v < 4; ++v)
            y[i][v] = (row < dim && 16 * i + lk + 4 * v < R) ? b[16 * i + lk + 4 * v] : 0.0;
}

// All passes of a wave over its tiles; y holds the first.
template <int NB>
__device__ __forceinline__ void chol_solve_rows(const RidgeLds<NB>& w,
                                                const double* __restrict__ FtV,
                                                double* __restrict__ F, size_t dim, int R,
                                                size_t row, int lr, int lk, double (&y)[NB][4])
{
    double x[NB][4], xt[NB][4], l[4], lt[4];
#pragma unroll
    for (int v = 0; v < 4; ++v)
    {
#pragma unroll
        for (int i = 0; i < NB; ++i)
        {
            x[i][v] = w.X[i][(lk + 4 * v) * CHOL_LD + lr];
            xt[i][v] = w.X[i][lr * CHOL_LD + lk + 4 * v];
        }
        if (NB == 2)
        {
            l[v] = -w.L21[(lk + 4 * v) * CHOL_LD + lr];
            lt[v] = -w.L21[lr * CHOL_LD + lk + 4 * v];
        }
    }
    const size_t stride = size_t(gridDim.x) * CHOL_ROWS;
    const d4 zero = {0.0, 0.0, 0.0, 0.0};
    auto set = [](double (&o)[4], d4 v) {
#pragma unroll
        for (int q = 0; q < 4; ++q) o[q] = v[q];
    };
    for (; row - lr < dim; row += stride)   // wave-uniform
    {
        double nx[NB][4];
        chol_load_rhs<NB>(FtV, dim, R, row + stride, lk, nx);
        set(y[0], chol_mul(xt[0], y[0], zero));
        if constexpr (NB == 2)
        {
            set(y[1], chol_mul(lt, y[0], d4{y[1][0], y[1][1], y[1][2], y[1][3]}));
            set(y[1], chol_mul(xt[1], y[1], zero));
            set(y[1], chol_mul(x[1], y[1], zero));
            set(y[0], chol_mul(l, y[1], d4{y[0][0], y[0][1], y[0][2], y[0][3]}));
        }
        set(y[0], chol_mul(x[0], y[0], zero));
        if (row < dim)
        {
            double* out = F + row * R;
#pragma unroll
            for (int i = 0; i < NB; ++i)
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    if (16 * i + lk + 4 * v < R) out[16 * i + lk + 4 * v] = y[i][v];
        }
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
            for (int v = 0; v < 4; ++v) y[i][v] = nx[i][v];
    }
}

template <int NB>
__global__ __launch_bounds__(64) void chol_factor_kernel(const double* __restrict__ FtF, int R,
                                                         double* __restrict__ Lout)
{
    __shared__ RidgeLds<NB> w;
    chol_factor_all<NB, true>(FtF, R, w, Lout);
}

template <int NB>
__global__ __launch_bounds__(CHOL_T) void chol_apply_kernel(const double* __restrict__ Lg,
                                                            const double* __restrict__ FtV,
                                                            double* __restrict__ F, size_t dim,
                                                            int R)
{
    __shared__ RidgeLds<NB> w;
    const int lane = threadIdx.x & 63, wave = threadIdx.x / 64, lr = lane & 15, lk = lane >> 4;
    const size_t row = size_t(blockIdx.x) * CHOL_ROWS + size_t(wave) * 16 + size_t(lr);
    double y[NB][4];
    chol_load_rhs<NB>(FtV, dim, R, row, lk, y);
    if (wave < NB)   // a diagonal block each
    {
        double a[4], x[4];
#pragma unroll
        for (int v = 0; v < 4; ++v)
        {
            const int i = 16 * wave + lk + 4 * v, k = 16 * wave + lr;
            a[v] = (i < R && k < R) ? Lg[size_t(i) * R + k] : 0.0;
        }
        chol_identity(x, lr, lk);
        inv16_from<0>(a, x, lr, lk, min(R - 16 * wave, 16));
        chol_put(w.X[wave], x, lr, lk);
    }
    else if (NB == 2 && wave == 2)
    {
        double a[4];
#pragma unroll
        for (int v = 0; v < 4; ++v)
        {
            const int i = 16 + lk + 4 * v;
            a[v] = i < R ? Lg[size_t(i) * R + lr] : 0.0;
        }
        chol_put(w.L21, a, lr, lk);
    }
    __syncthreads();
    chol_solve_rows<NB>(w, FtV, F, dim, R, row, lr, lk, y);
}

// Both in one launch, every workgroup factoring for itself: the same bits
// (chol_quot).
template <int NB>
__global__ __launch_bounds__(CHOL_T) void chol_solve_kernel(const double* __restrict__ FtF,
                                                            const double* __restrict__ FtV,
                                                            double* __restrict__ F, size_t dim,
                                                            int R)
{
    __shared__ RidgeLds<NB> w;
    const int lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4;
    const size_t row =
        size_t(blockIdx.x) * CHOL_ROWS + size_t(threadIdx.x / 64) * 16 + size_t(lr);
    double y[NB][4];
    chol_load_rhs<NB>(FtV, dim, R, row, lk, y);   // in flight beside the factorisation
    chol_factor_all<NB, false>(FtF, R, w, nullptr);
    chol_solve_rows<NB>(w, FtV, F, dim, R, row, lr, lk, y);
}

// Column sums of squares: P partials of R each (deterministic).
__global__ __launch_bounds__(256) void colsq_partial_kernel(const double* __restrict__ F,
                                                            size_t rows, int R,
                                                            double* __restrict__ part)
{
    // 256 threads = (256 / R) row lanes x R ranks (R <= 32 -> >= 8 row lanes)
    __shared__ double red[256];
    const int r = threadIdx.x % R;
    const int rl = threadIdx.x / R;
    const int nrl = 256 / R;
    double acc = 0.0;
    if (rl < nrl)
        for (size_t i = size_t(blockIdx.x) * nrl + rl; i < rows; i += size_t(gridDim.x) * nrl)
        {
            const double v = F[i * R + r];
            acc += v * v;
        }
    red[threadIdx.x] = acc;
    __syncthreads();
    if (threadIdx.x < R)
    {
        double t = 0.0;
        for (int q = 0; q < nrl; ++q) t += red[q * R + threadIdx.x];
        part[size_t(blockIdx.x) * R + threadIdx.x] = t;
    }
}

// Every block re-reduces the partials (P x R, small), divides its rows, and
// block 0 writes lambda.
__global__ __launch_bounds__(256) void normalize_nd_kernel(double* __restrict__ F, size_t rows,
                                                           int R, const double* __restrict__ part,
                                                           int P, double* __restrict__ lambda)
{
    __shared__ double nrm[32];
    if (threadIdx.x < R)
    {
        double s = 0.0;
        for (int p = 0; p < P; ++p) s += part[size_t(p) * R + threadIdx.x];
        double n = sqrt(s);
        if (!isfinite(n) || n < 1e-14) n = 1.0;
        nrm[threadIdx.x] = n;
        if (blockIdx.x == 0) lambda[threadIdx.x] = n;
    }
    __syncthreads();
    const size_t total = rows * size_t(R);
    const size_t stride = size_t(gridDim.x) * blockDim.x;
    for (size_t x = size_t(blockIdx.x) * blockDim.x + threadIdx.x; x < total; x += stride)
        F[x] /= nrm[x % R];
}

// A small factor's update tail in one workgroup (rows x R <= SMALL_UPDATE_MAX,
// R <= 32): the normalisation of normalize_nd_kernel (lambda_r = the column's
// 2-norm, 1 when it is not finite or below 1e-14; F /= lambda), the Gram
// G_mode = F^T F of the normalised factor and, when next >= 0, the next
// mode's FtF = prod_{g != next} G_g in mode order (gram_hadamard_kernel) and
// its first nzero FtV entries zeroed: one launch instead of six.  Rows are
// staged in LDS 64 at a time; each Gram entry sums its rows in order.
constexpr int SMALL_UPDATE_MAX = 1 << 16;

__global__ __launch_bounds__(1024) void small_update_kernel(
    double* __restrict__ F, int rows, int R, double* __restrict__ lambda, double* __restrict__ grams,
    int ngram, int mode, int next, double* __restrict__ FtF, double* __restrict__ FtV, int nzero)
{
    __shared__ double red[1024];
    __shared__ double nrm[32];
    __shared__ double tile[64 * 32];
    const int tid = threadIdx.x;
    const int RR = R * R;
    const int r = tid % R, rl = tid / R, nrl = 1024 / R;
    double acc = 0.0;
    if (rl < nrl)
        for (int i = rl; i < rows; i += nrl)
        {
            const double v = F[size_t(i) * R + r];
            acc += v * v;
        }
    red[tid] = acc;
    __syncthreads();
    if (tid < R)
    {
        double sq = 0.0;
        for (int q = 0; q < nrl; ++q) sq += red[q * R + tid];
        double n = sqrt(sq);
        if (!isfinite(n) || n < 1e-14) n = 1.0;
        nrm[tid] = n;
        lambda[tid] = n;
    }
    __syncthreads();
    // Gram entry e = tid % RR, row group q = tid / RR of NQ: group q sums the
    // rows i = q mod NQ, then the groups' sums are added in group order
    const int NQ = 1024 / RR;
    const int e = tid % RR, q = tid / RR;
    const int a = e / R, b = e % R;
    double g = 0.0;
    for (int i0 = 0; i0 < rows; i0 += 64)
    {
        const int nr = min(64, rows - i0);
        for (int x = tid; x < nr * R; x += 1024)
        {
            const double v = F[size_t(i0) * R + x] / nrm[x % R];
            F[size_t(i0) * R + x] = v;
            tile[x] = v;
        }
        __syncthreads();
        if (q < NQ)
            for (int i = q; i < nr; i += NQ) g += tile[i * R + a] * tile[i * R + b];
        __syncthreads();
    }
    red[tid] = g;
    __syncthreads();
    if (tid < RR)
    {
        g = 0.0;
        for (int p = 0; p < NQ; ++p) g += red[p * RR + tid];
        grams[size_t(mode) * RR + tid] = g;
    }
    if (next >= 0)
    {
        if (tid < RR)
        {
            double v = 1.0;
            for (int gm = 0; gm < ngram; ++gm)
                if (gm != next) v *= (gm == mode) ? g : grams[size_t(gm) * RR + tid];
            FtF[tid] = v;
        }
        for (int x = tid; x < nzero; x += 1024) FtV[x] = 0.0;
    }
}

// --------------------------------------------------------- exact residual --

__global__ __launch_bounds__(256) void residual_nd_kernel(int nmodes,
                                                          const uint32_t* __restrict__ coords,
                                                          const double* __restrict__ vals,
                                                          uint64_t nnz, Factors F,
                                                          const double* __restrict__ lambda,
                                                          int R, double* __restrict__ part)
{
    __shared__ double red[2][256];
    double res = 0.0, sq = 0.0;
    const uint64_t stride = uint64_t(gridDim.x) * blockDim.x;
    for (uint64_t e = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; e < nnz; e += stride)
    {
        const double* rowp[MAXM];
#pragma unroll
        for (int m = 0; m < MAXM; ++m)
            rowp[m] = (m < nmodes) ? F.p[m] + size_t(coords[uint64_t(m) * nnz + e]) * R : nullptr;
        double xhat = 0.0;
        for (int r = 0; r < R; ++r)
        {
            double p = lambda ? lambda[r] : 1.0;
#pragma unroll
            for (int m = 0; m < MAXM; ++m)
                if (m < nmodes) p *= rowp[m][r];
            xhat += p;
        }
        const double v = vals[e];
        const double d = v - xhat;
        res += d * d;
        sq += v * v;
    }
    red[0][threadIdx.x] = res;
    red[1][threadIdx.x] = sq;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1)
    {
        if (int(threadIdx.x) < h)
        {
            red[0][threadIdx.x] += red[0][threadIdx.x + h];
            red[1][threadIdx.x] += red[1][threadIdx.x + h];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0)
    {
        part[2 * size_t(blockIdx.x)] = red[0][0];
        part[2 * size_t(blockIdx.x) + 1] = red[1][0];
    }
}

// out2 += the P partials' sums, in a fixed order
__global__ __launch_bounds__(256) void finalize_add2_kernel(const double* __restrict__ part, int P,
                                                            double* __restrict__ out2)
{
    __shared__ double red[256];
    // thread t: sum t % 2, partials t / 2, t / 2 + 128, ...
    double t = 0.0;
    for (int p = int(threadIdx.x) / 2; p < P; p += 128) t += part[2 * size_t(p) + threadIdx.x % 2];
    red[threadIdx.x] = t;
    __syncthreads();
    for (int h = 128; h >= 2; h >>= 1)
    {
        if (int(threadIdx.x) < h) red[threadIdx.x] += red[threadIdx.x + h];
        __syncthreads();
    }
    if (threadIdx.x < 2) out2[threadIdx.x] += red[threadIdx.x];
}

// diagonal blocks of 16
template <class Run>
void chol_blocks(int R, Run run)
{
    if (R <= 16) run(std::integral_constant<int, 1>{});
    else run(std::integral_constant<int, 2>{});
}

// 1024 workgroups, four to a CU, take further rows in passes
dim3 chol_grid(size_t dim)
{
    return dim3(unsigned(std::min<size_t>((dim + CHOL_ROWS - 1) / CHOL_ROWS, 1024)));
}

bool factors_ok(int n, const double* const* h_F)
{
    if (!h_F) return false;
    for (int m = 0; m < n; ++m)
        if (!h_F[m]) return false;
    return true;
}

}  // namespace

extern "C" uint64_t cptc_gen_hash(uint64_t x)
{
    x += 0x9E3779B97F4A7C15ull;
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
    x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
    return x ^ (x >> 31);
}

extern "C" int cptc_mttkrp_seg_nd(int nmodes, int mode, const uint32_t* d_scoords,
                                  const int* level_modes, const double* d_vals,
                                  const uint8_t* d_skip, uint64_t nnz, const uint32_t* d_seg_row,
                                  const uint32_t* d_seg_start, const uint32_t* d_seg_cnt,
                                  const uint8_t* d_single, uint64_t nseg,
                                  const double* const* h_F, double* d_FtV, int R, void* stream)
{
    CPTC_REQUIRE(nmodes >= 2 && nmodes <= MAXM && mode >= 0 && mode < nmodes, CPTC_ERR_ARG,
                 "cptc_mttkrp_seg_nd: nmodes %d mode %d", nmodes, mode);
    CPTC_REQUIRE(R >= 1 && R <= 32, CPTC_ERR_ARG, "cptc_mttkrp_seg_nd: R %d (1..32)", R);
    if (nseg == 0) return CPTC_OK;
    CPTC_REQUIRE(nseg < (uint64_t(1) << 31) && nnz <= 0x7FFFFFFFull, CPTC_ERR_ARG,
                 "cptc_mttkrp_seg_nd: %llu segments / %llu nnz", (unsigned long long)nseg,
                 (unsigned long long)nnz);
    CPTC_REQUIRE(d_scoords && d_vals && d_seg_row && d_seg_start && d_seg_cnt && d_FtV &&
                     factors_ok(nmodes, h_F),
                 CPTC_ERR_ARG, "cptc_mttkrp_seg_nd: null pointer");
    // factors in level order (the d_scoords rows)
    Factors F{};
    bool aligned = (R % 2 == 0);
    unsigned seen = 1u << mode;
    for (int q = 0; q < nmodes - 1; ++q)
    {
        const int m = level_modes ? level_modes[q] : (q < mode ? q : q + 1);
        CPTC_REQUIRE(m >= 0 && m < nmodes && !(seen & (1u << m)), CPTC_ERR_ARG,
                     "cptc_mttkrp_seg_nd: level_modes is not a permutation of the other modes");
        seen |= 1u << m;
        F.p[q] = h_F[m];
        if (reinterpret_cast<uintptr_t>(h_F[m]) & 15) aligned = false;
    }
    hipStream_t s = cptc::as_stream(stream);
    if (aligned)
        launch_seg_n<2>(nmodes, F, mode, d_scoords, nnz, d_vals, d_skip, d_seg_row, d_seg_start,
                        d_seg_cnt, d_single, nseg, d_FtV, R, s);
    else
        launch_seg_n<1>(nmodes, F, mode, d_scoords, nnz, d_vals, d_skip, d_seg_row, d_seg_start,
                        d_seg_cnt, d_single, nseg, d_FtV, R, s);
    CPTC_LAUNCHED();
    return CPTC_OK;
}

extern "C" int cptc_units_pack_nd(const uint32_t* d_unit6, uint64_t nunits, const uint32_t* d_lid,
                                  const double* d_val, float* d_tiles, void* stream)
{
    if (nunits == 0) return CPTC_OK;
    CPTC_REQUIRE(d_unit6 && d_lid && d_val && d_tiles, CPTC_ERR_ARG,
                 "cptc_units_pack_nd: null pointer");
    CPTC_REQUIRE(nunits < (uint64_t(1) << 31), CPTC_ERR_ARG, "cptc_units_pack_nd: too many units");
    hipLaunchKernelGGL(units_pack_kernel, dim3(unsigned(nunits)), dim3(256), 0,
                       cptc::as_stream(stream), d_unit6, d_lid, d_val, d_tiles);
    CPTC_LAUNCHED();
    return CPTC_OK;
}

extern "C" int cptc_units_pack_nd_f64(const uint32_t* d_unit6, uint64_t nunits,
                                      const uint32_t* d_lid, const double* d_val, double* d_img,
                                      void* stream)
{
    if (nunits == 0) return CPTC_OK;
    CPTC_REQUIRE(d_unit6 && d_lid && d_val && d_img, CPTC_ERR_ARG,
                 "cptc_units_pack_nd_f64: null pointer");
    CPTC_REQUIRE((reinterpret_cast<uintptr_t>(d_img) & 15) == 0, CPTC_ERR_ARG,
                 "cptc_units_pack_nd_f64: the image must be 16-byte aligned");
    CPTC_REQUIRE(nunits < (uint64_t(1) << 31), CPTC_ERR_ARG,
                 "cptc_units_pack_nd_f64: too many units");
    hipLaunchKernelGGL(units_pack_f64_kernel, dim3(unsigned(nunits)), dim3(256), 0,
                       cptc::as_stream(stream), d_unit6, d_lid, d_val, d_img);
    CPTC_LAUNCHED();
    return CPTC_OK;
}

extern "C" int cptc_units_weights_nd(const uint32_t* d_unit6, uint64_t nunits,
                                     const uint32_t* d_outer_coords, int nouter,
                                     const int* outer_modes, const double* const* h_F, int R,
                                     double* d_W, void* stream)
{
    CPTC_REQUIRE(R >= 1 && nouter >= 0 && nouter <= MAXM - 3, CPTC_ERR_ARG,
                 "cptc_units_weights_nd: R %d nouter %d", R, nouter);
    if (nunits == 0) return CPTC_OK;
    CPTC_REQUIRE(d_unit6 && d_W && (nouter == 0 || (d_outer_coords && outer_modes && h_F)),
                 CPTC_ERR_ARG, "cptc_units_weights_nd: null pointer");
    Factors Fo{};
    for (int k = 0; k < nouter; ++k)
    {
        CPTC_REQUIRE(outer_modes[k] >= 0 && outer_modes[k] < MAXM && h_F[outer_modes[k]],
                     CPTC_ERR_ARG, "cptc_units_weights_nd: outer mode %d", outer_modes[k]);
        Fo.p[k] = h_F[outer_modes[k]];
    }
    const uint64_t total = nunits * uint64_t(R);
    hipLaunchKernelGGL(units_weights_kernel, dim3(cptc::grid_for(total, 256, 65536)), dim3(256), 0,
                       cptc::as_stream(stream), d_unit6, nunits, d_outer_coords, nouter, Fo, R,
                       d_W);
    CPTC_LAUNCHED();
    return CPTC_OK;
}

extern "C" int cptc_gram_hadamard(const double* d_grams, int ngram, int skip, int R,
                                  double* d_out, void* stream)
{
    CPTC_REQUIRE(R >= 1 && ngram >= 0 && d_out && (ngram == 0 || d_grams), CPTC_ERR_ARG,
                 "cptc_gram_hadamard: bad arguments");
    const int RR = R * R;
    hipLaunchKernelGGL(gram_hadamard_kernel, dim3(cptc::grid_for(size_t(RR), 256, 256)),
                       dim3(256), 0, cptc::as_stream(stream), d_grams, ngram, skip, RR, d_out);
    CPTC_LAUNCHED();
    return CPTC_OK;
}

extern "C" int cptc_chol_ridge_factor(const double* d_FtF, double* d_L, int R, void* stream)
{
    CPTC_REQUIRE(R >= 1 && R <= CHOL_RM, CPTC_ERR_ARG, "cptc_chol_ridge_factor: R %d (1..32)", R);
    CPTC_REQUIRE(d_FtF && d_L, CPTC_ERR_ARG, "cptc_chol_ridge_factor: null pointer");
    hipStream_t s = cptc::as_stream(stream);
    auto run = [&](auto NB) {
        hipLaunchKernelGGL(chol_factor_kernel<decltype(NB)::value>, dim3(1), dim3(64), 0, s,
                           d_FtF, R, d_L);
    };
    chol_blocks(R, run);
    CPTC_LAUNCHED();
    return CPTC_OK;
}

extern "C" int cptc_chol_ridge_apply(const double* d_L, const double* d_FtV, double* d_F,
                                     size_t dim, int R, void* stream)
{
    CPTC_REQUIRE(R >= 1 && R <= CHOL_RM, CPTC_ERR_ARG, "cptc_chol_ridge_apply: R %d (1..32)", R);
    if (dim == 0) return CPTC_OK;
    CPTC_REQUIRE(d_L && d_FtV && d_F, CPTC_ERR_ARG, "cptc_chol_ridge_apply: null pointer");
    CPTC_REQUIRE(dim / 64 < (size_t(1) << 31), CPTC_ERR_ARG, "cptc_chol_ridge_apply: %zu rows",
                 dim);
    hipStream_t s = cptc::as_stream(stream);
    auto run = [&](auto NB) {
        hipLaunchKernelGGL(chol_apply_kernel<decltype(NB)::value>, chol_grid(dim), dim3(CHOL_T), 0,
                           s, d_L, d_FtV, d_F, dim, R);
    };
    chol_blocks(R, run);
    CPTC_LAUNCHED();
    return CPTC_OK;
}

extern "C" int cptc_chol_ridge_solve(const double* d_FtF, const double* d_FtV, double* d_F,
                                     size_t dim, int R, void* stream)
{
    CPTC_REQUIRE(R >= 1 && R <= CHOL_RM, CPTC_ERR_ARG, "cptc_chol_ridge_solve: R %d (1..32)", R);
    if (dim == 0) return CPTC_OK;
    CPTC_REQUIRE(d_FtF && d_FtV && d_F, CPTC_ERR_ARG, "cptc_chol_ridge_solve: null pointer");
    CPTC_REQUIRE(dim / 64 < (size_t(1) << 31), CPTC_ERR_ARG, "cptc_chol_ridge_solve: %zu rows",
                 dim);
    hipStream_t s = cptc::as_stream(stream);
    auto run = [&](auto NB) {
        hipLaunchKernelGGL(chol_solve_kernel<decltype(NB)::value>, chol_grid(dim), dim3(CHOL_T), 0,
                           s, d_FtF, d_FtV, d_F, dim, R);
    };
    chol_blocks(R, run);
    CPTC_LAUNCHED();
    return CPTC_OK;
}

extern "C" int cptc_gen_normalize(double* d_F, size_t rows, int R, double* d_lambda, void* stream)
{
    CPTC_REQUIRE(R >= 1 && R <= 32 && d_F && d_lambda, CPTC_ERR_ARG,
                 "cptc_gen_normalize: R %d (1..32) or null pointer", R);
    const int nrl = 256 / R;
    const int P = int(cptc::grid_for(rows, unsigned(nrl) * 8, 256));
    void* buf = nullptr;
    CPTC_TRY(cptc::scratch_get(cptc::SCR_REDUCE, size_t(P) * R * sizeof(double), &buf));
    double* part = static_cast<double*>(buf);
    hipStream_t s = cptc::as_stream(stream);
    hipLaunchKernelGGL(colsq_partial_kernel, dim3(P), dim3(256), 0, s, d_F, rows, R, part);
    CPTC_LAUNCHED();
    hipLaunchKernelGGL(normalize_nd_kernel, dim3(cptc::grid_for(rows * size_t(R), 256, 1024)),
                       dim3(256), 0, s, d_F, rows, R, part, P, d_lambda);
    CPTC_LAUNCHED();
    return CPTC_OK;
}

extern "C" int cptc_gen_normalize_gram(double* d_F, size_t rows, int R, double* d_lambda,
                                       double* d_grams, int ngram, int mode, int next,
                                       double* d_FtF, double* d_FtV, size_t nzero, void* stream)
{
    CPTC_REQUIRE(R >= 1 && R <= 32 && rows >= 1 && rows * size_t(R) <= size_t(SMALL_UPDATE_MAX),
                 CPTC_ERR_ARG, "cptc_gen_normalize_gram: rows %zu x R %d (R <= 32, <= %d values)",
                 rows, R, SMALL_UPDATE_MAX);
    CPTC_REQUIRE(ngram >= 1 && mode >= 0 && mode < ngram && next >= -1 && next < ngram &&
                     nzero <= (size_t(1) << 24),
                 CPTC_ERR_ARG, "cptc_gen_normalize_gram: ngram %d mode %d next %d nzero %zu",
                 ngram, mode, next, nzero);
    CPTC_REQUIRE(d_F && d_lambda && d_grams && (next < 0 || d_FtF) && (nzero == 0 || d_FtV),
                 CPTC_ERR_ARG, "cptc_gen_normalize_gram: null pointer");
    hipLaunchKernelGGL(small_update_kernel, dim3(1), dim3(1024), 0, cptc::as_stream(stream), d_F,
                       int(rows), R, d_lambda, d_grams, ngram, mode, next, d_FtF, d_FtV,
                       next >= 0 ? int(nzero) : 0);
    CPTC_LAUNCHED();
    return CPTC_OK;
}

extern "C" int cptc_residual_nd(int nmodes, const uint32_t* d_coords, const double* d_vals,
                                uint64_t nnz, const double* const* h_F, const double* d_lambda,
                                int R, double* d_out2, void* stream)
{
    CPTC_REQUIRE(nmodes >= 1 && nmodes <= MAXM && R >= 1 && d_out2, CPTC_ERR_ARG,
                 "cptc_residual_nd: nmodes %d R %d", nmodes, R);
    if (nnz == 0) return CPTC_OK;
    CPTC_REQUIRE(d_coords && d_vals && factors_ok(nmodes, h_F), CPTC_ERR_ARG,
                 "cptc_residual_nd: null pointer");
    Factors F{};
    for (int m = 0; m < nmodes; ++m) F.p[m] = h_F[m];
    const int P = int(cptc::grid_for(nnz, 256 * 8, 2048));
    void* buf = nullptr;
    CPTC_TRY(cptc::scratch_get(cptc::SCR_REDUCE, size_t(P) * 2 * sizeof(double), &buf));
    double* part = static_cast<double*>(buf);
    hipStream_t s = cptc::as_stream(stream);
    hipLaunchKernelGGL(residual_nd_kernel, dim3(P), dim3(256), 0, s, nmodes, d_coords, d_vals, nnz,
                       F, d_lambda, R, part);
    CPTC_LAUNCHED();
    hipLaunchKernelGGL(finalize_add2_kernel, dim3(1), dim3(256), 0, s, part, P, d_out2);
    CPTC_LAUNCHED();
    return CPTC_OK;
}
