// Inverse of a small symmetric positive definite matrix in the registers of
// one workgroup (or one wave) by the symmetric sweep (Gauss-Jordan without
// pivoting in its symmetric form); included by small_la.hip.  SweepWave (R <=
// 32) and SweepQuad (R <= 64) take one pivot at a time; Blocks (R <= 128)
// takes 16 at a time on the FP64 matrix cores:
//
// The matrix, R <= 16 NB, padded with the identity, is held as the 16 x 16
// blocks of its lower block triangle.  A block sits in the accumulator
// layout of v_mfma_f64_16x16x4f64: element v of lane l is entry (l / 16 +
// 4 v, l % 16), which is also the instruction's B operand for K step v, and
// the A operand of the transposed block.  Sweeping block pivot K with P =
// A_KK = L D L^T, X = L^-1, all inside one wave:
//   U_i  = A_iK X^T,  F_i = U_i D^-1          (the LDL^T factor's columns)
//   A_ij -= F_i U_j^T                         (i, j != K)
//   A_iK = F_i X (= A_iK P^-1),  A_KK = -X^T D^-1 X (= -P^-1)
// and after every block pivot the matrix is -A^-1.  The updates are those of
// a blocked LDL^T factorization, so the error stays that of the column by
// column algorithm; with the explicit P^-1 in their place (one product less
// per block) it grew with the condition of P (kappa 1e8, R = 128: 2e-9
// against 4e-10).  The scalar pivots are the LDL^T pivots, so the acceptance
// test of the caller is the Cholesky one.
//
// Why blocks: an unblocked sweep or a column Cholesky pays a workgroup
// barrier and an LDS round trip per column (R of them, ~800 clocks each); here
// a column costs a reciprocal and one rank-1 update inside a wave, the rest
// of the matrix is touched R / 16 times with 16 x 16 x 16 products, and the
// pivot block of step K + 1 is factored in the shadow of the other waves'
// updates of step K, ahead of its wave's own other blocks.
//
// Measured, a solve's launches back to back, before (column Cholesky above R
// = 64, a workgroup sweep with two barriers a pivot below) and now: R = 16
// 6.8 -> 4.7 us, 32 11.6 -> 9.7, 64 27.1 -> 22.5, 65 146 -> 20, 100 319 -> 30,
// 128 623 -> 38.5 (768 threads; 512: 41, 1024 spill: 81).
#pragma once

#include <hip/hip_runtime.h>

namespace cptc {
namespace bsweep {

typedef double d4 __attribute__((ext_vector_type(4)));

// LDS row stride of a staged block: an operand read takes lane l to entry
// (l % 16, 4 s + l / 16), and 18 doubles a row put a half-wave's 32 entries
// on distinct bank pairs
constexpr int LD = 18;
constexpr int BLK = 16 * LD;

// doubles of LDS that Blocks<NB, *>::sweep works in: D^-1 and X of two pivot
// blocks and the panels U and F
constexpr int lds_doubles(int nb) { return 32 + (2 * nb + 2) * BLK; }

__device__ __forceinline__ double readlane_d(double x, int lane)
{
    const long long b = __double_as_longlong(x);
    const unsigned lo = unsigned(__builtin_amdgcn_readlane(int(b), lane));
    const unsigned hi = unsigned(__builtin_amdgcn_readlane(int(b >> 32), lane));
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// lane N of each row of 16 lanes to the whole row (DPP row_newbcast); rows of
// lanes outside ROWS get 0
template <int N, int ROWS>
__device__ __forceinline__ double row_bcast_d(double x)
{
    const long long b = __double_as_longlong(x);
    unsigned lo, hi;
    if constexpr (ROWS == 0xf)
    {
        lo = unsigned(__builtin_amdgcn_mov_dpp(int(b), 0x150 + N, ROWS, 0xf, true));
        hi = unsigned(__builtin_amdgcn_mov_dpp(int(b >> 32), 0x150 + N, ROWS, 0xf, true));
    }
    else
    {
        lo = unsigned(__builtin_amdgcn_update_dpp(0, int(b), 0x150 + N, ROWS, 0xf, false));
        hi = unsigned(__builtin_amdgcn_update_dpp(0, int(b >> 32), 0x150 + N, ROWS, 0xf, false));
    }
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

__device__ __forceinline__ double bperm_d(double x, int lane)
{
    const long long b = __double_as_longlong(x);
    const unsigned lo = unsigned(__builtin_amdgcn_ds_bpermute(4 * lane, int(b)));
    const unsigned hi = unsigned(__builtin_amdgcn_ds_bpermute(4 * lane, int(b >> 32)));
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// 1 / p from the hardware estimate and two Newton steps (within an ulp), at a
// third of the division's latency.  For p outside about [2^-1000, 2^1000]
// the result is of no use; matrices with such pivots are declined anyway
// (fast_inverse_ok: the squares in ||A||_F over- or underflow).
__device__ __forceinline__ double recip(double p)
{
    double r = __builtin_amdgcn_rcp(p);
    r = fma(fma(-p, r, 1.0), r, r);
    return fma(fma(-p, r, 1.0), r, r);
}

// 1 / p as the division gives it (one more step: from within an ulp, the
// rounded quotient), for the same p
__device__ __forceinline__ double recip_rn(double p)
{
    const double r = recip(p);
    return fma(fma(-p, r, 1.0), r, r);
}

// Columns K .. 15 of a block's LDL^T (a: becomes D L^T on and above the
// diagonal, x: L^-1, from the identity).  Column K reaches the lane's rows by
// row_newbcast (a row of 16 lanes holds one matrix row), rows K of a and x
// reach the lane's column by permutes that run beside the reciprocal (in
// registers, by lane-row exchanges, they took three times the instructions:
// 350 against 215 clocks a column).  nv: rows of the block inside the matrix
// (the padding needs no elimination).
template <int K>
__device__ __forceinline__ void ldl16_from(double (&a)[4], double (&x)[4], int lr, double tau,
                                           int nv, int& ok)
{
    constexpr int VK = K / 4, QK = K % 4;
    const double p = readlane_d(a[VK], 16 * QK + K);
    if (!(p > tau)) ok = 0;
    if constexpr (K < 15)
    {
        const double rk = bperm_d(a[VK], 16 * QK + lr);
        const double xk = bperm_d(x[VK], 16 * QK + lr);
        const double ip = recip(p);
#pragma unroll
        for (int v = QK == 3 ? VK + 1 : VK; v < 4; ++v)
        {
            // a_ik / a_kk in the rows below K, 0 above
            const double f = (v == VK ? row_bcast_d<K, (0xf << (QK + 1)) & 0xf>(a[v])
                                      : row_bcast_d<K, 0xf>(a[v])) * ip;
            a[v] = fma(-f, rk, a[v]);
            x[v] = fma(-f, xk, x[v]);
        }
        if (K + 1 < nv) ldl16_from<K + 1>(a, x, lr, tau, nv, ok);
    }
}

// order of a wave's own LDS accesses across lanes
__device__ __forceinline__ void sync_wave()
{
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// The symmetric sweep one scalar pivot at a time (Beaton's SWEEP operator),
// on the full matrix, for R <= 64, where 16-column blocks have little left to
// save and the interleaved updates round about half as much on matrices of
// kappa >= 1e8 (R = 32, kappa 1e8: 3e-10 against 8e-10 with 16 x 16 pivots):
//   a_kk -> -1 / a_kk,  a_ik -> a_ik / a_kk,  a_kj -> a_kj / a_kk,
//   a_ij -> a_ij - (a_ik / a_kk) a_kj;
// after every pivot the matrix is -A^-1.  M x M blocks of 16 x 16 a wave, in
// the layout above.
//
// SweepWave: the whole matrix in one wave, no barriers.  a_kj is taken from
// column k (a_jk) and the pivot's reciprocal is the rounded one, so every
// entry goes through the roundings of the plain column sweep and the inverse
// has its bits (an over-ranked model on the split-bf16 tiles turns a last bit
// here into 4e-4 of a factor in five iterations).  Column k reaches the lane's
// rows by row_newbcast; a lane then holds rows 16 i + l / 16 + 4 v of it for
// every v, keeps v = (l % 16) / 4, and one permute (lane 16 (l % 4) + l % 16)
// brings it row 16 i + l % 16, its columns' entries.  With row k by permutes
// and the two-step reciprocal R = 16 took 4.4 us a launch and 32 8.9.
template <int M>
struct SweepWave
{
    double a[M][M][4];

    template <int K>
    __device__ __forceinline__ void from(int R, int lr, int lk, double tau, int& ok)
    {
        constexpr int KB = K / 16, KL = K % 16, VK = KL / 4, QK = KL % 4;
        const double p = readlane_d(a[KB][KB][VK], 16 * QK + KL);
        double c[M][4], r[M];   // a_ik, a_jk
#pragma unroll
        for (int i = 0; i < M; ++i)
#pragma unroll
            for (int v = 0; v < 4; ++v) c[i][v] = row_bcast_d<KL, 0xf>(a[i][KB][v]);
#pragma unroll
        for (int j = 0; j < M; ++j)
        {
            const double lo = lr < 4 ? c[j][0] : c[j][1], hi = lr < 12 ? c[j][2] : c[j][3];
            r[j] = bperm_d(lr < 8 ? lo : hi, 16 * (lr % 4) + lr);
        }
        if (!(p > tau)) ok = 0;
        const double ip = recip_rn(p);
        const bool jk = lr == KL, ik = lk == QK;
#pragma unroll
        for (int i = 0; i < M; ++i)
#pragma unroll
            for (int v = 0; v < 4; ++v)
            {
                const double f = c[i][v] * ip;
#pragma unroll
                for (int j = 0; j < M; ++j)
                {
                    double x = fma(-f, r[j], a[i][j][v]);
                    if (j == KB) x = jk ? f : x;
                    if (i == KB && v == VK)
                    {
                        double y = a[i][j][v] * ip;
                        if (j == KB) y = jk ? -ip : y;
                        x = ik ? y : x;
                    }
                    a[i][j][v] = x;
                }
            }
        if constexpr (K % 4 == 3)
            if (!ok) return;   // declined: the Jacobi path follows
        if constexpr (K + 1 < 16 * M)
            if (K + 1 < R) from<K + 1>(R, lr, lk, tau, ok);
    }
};

// SweepQuad: R <= 64 over four waves, wave (wi, wj) the 32 x 32 quarter at
// (32 wi, 32 wj), padded with the identity to an even R.  Pivots go in pairs:
// the two columns and rows pass through LDS (two buffers) with one barrier a
// pair, and every wave brings the second ones up to date itself (one pivot a
// barrier: R = 64 26.3 us a launch against 22.5).
constexpr int QUAD_LD = 18;
constexpr int QUAD_BUF = 2 * (4 * QUAD_LD + 64);   // columns k, k + 1, rows k, k + 1
constexpr int QUAD_LDS = 2 * QUAD_BUF;             // doubles of LDS

struct SweepQuad
{
    double a[2][2][4];

    // pivot k = 32 h + K of the pair held in c (this wave's rows), r (its
    // columns): a after the sweep of that pivot, ip = 1 / a_kk.  On return f =
    // c ip
    template <int K>
    __device__ __forceinline__ void apply(const double (&c)[2][4], const double (&r)[2], double ip,
                                          int h, int wi, int wj, int lr, int lk, double (&f)[2][4])
    {
        constexpr int KB = K / 16, KL = K % 16, VK = KL / 4, QK = KL % 4;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int v = 0; v < 4; ++v)
            {
                f[i][v] = c[i][v] * ip;
#pragma unroll
                for (int j = 0; j < 2; ++j) a[i][j][v] = fma(-f[i][v], r[j], a[i][j][v]);
            }
        if (wj == h)   // wave-uniform
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int v = 0; v < 4; ++v) a[i][KB][v] = lr == KL ? f[i][v] : a[i][KB][v];
        if (wi == h)
#pragma unroll
            for (int j = 0; j < 2; ++j)
            {
                double y = r[j] * ip;
                if (j == KB && wj == h) y = lr == KL ? -ip : y;
                a[KB][j][VK] = lk == QK ? y : a[KB][j][VK];
            }
    }

    template <int K>   // pivots 32 h + K and + 1, K even
    __device__ __forceinline__ void from(int R, int h, int wi, int wj, int lr, int lk, double tau,
                                         double* lds, int& ok)
    {
        constexpr int KB = K / 16, KL = K % 16, VK = KL / 4, QK = KL % 4;
        // entry (row 32 w + 16 i + lk + 4 v) of a column at [lk][8 w + 4 i + v]
        double* col = lds + ((K / 2) & 1) * QUAD_BUF;
        double* row = col + 2 * 4 * QUAD_LD;
        if (wj == h && (lr == KL || lr == KL + 1))
        {
            double* o = col + (lr - KL) * 4 * QUAD_LD + lk * QUAD_LD + 8 * wi;
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int v = 0; v < 4; ++v) o[4 * i + v] = a[i][KB][v];
        }
        if (wi == h && (lk == QK || lk == QK + 1))
#pragma unroll
            for (int j = 0; j < 2; ++j) row[(lk - QK) * 64 + 32 * wj + 16 * j + lr] = a[KB][j][VK];
        __syncthreads();
        const double* pc = col + 8 * h + 4 * KB + VK;   // entries (k, .), (k + 1, .)
        const double p00 = pc[QK * QUAD_LD], p10 = pc[(QK + 1) * QUAD_LD];
        const double p01 = pc[(4 + QK) * QUAD_LD], p11 = pc[(4 + QK + 1) * QUAD_LD];
        double c0[2][4], c1[2][4], r0[2], r1[2], f[2][4];
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int v = 0; v < 4; ++v)
            {
                c0[i][v] = col[lk * QUAD_LD + 8 * wi + 4 * i + v];
                c1[i][v] = col[(4 + lk) * QUAD_LD + 8 * wi + 4 * i + v];
            }
#pragma unroll
        for (int j = 0; j < 2; ++j)
        {
            r0[j] = row[32 * wj + 16 * j + lr];
            r1[j] = row[64 + 32 * wj + 16 * j + lr];
        }
        if (!(p00 > tau)) ok = 0;
        const double ip0 = recip(p00);
        const double f10 = p10 * ip0;
        const double q11 = fma(-f10, p01, p11);
        if (32 * h + K + 1 < R && !(q11 > tau)) ok = 0;
        const double ip1 = recip(q11);
        apply<K>(c0, r0, ip0, h, wi, wj, lr, lk, f);
        // column and row k + 1 after that pivot
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int v = 0; v < 4; ++v)
            {
                c1[i][v] = fma(-f[i][v], p01, c1[i][v]);
                if (i == KB && v == VK) c1[i][v] = (wi == h && lk == QK) ? p01 * ip0 : c1[i][v];
            }
#pragma unroll
        for (int j = 0; j < 2; ++j)
        {
            r1[j] = fma(-f10, r0[j], r1[j]);
            if (j == KB) r1[j] = (wj == h && lr == KL) ? f10 : r1[j];
        }
        apply<K + 1>(c1, r1, ip1, h, wi, wj, lr, lk, f);
        if constexpr (K + 2 < 32)
            if (32 * h + K + 2 < R) from<K + 2>(R, h, wi, wj, lr, lk, tau, lds, ok);
    }
};

// The blocks of the lower block triangle over WAVES waves: diagonal block i
// is slot i / WAVES of wave i % WAVES, the off-diagonal blocks (slots DS ..)
// go round the waves from wave NB on, so that a wave with a diagonal block,
// which may be the next pivot, has the fewest others.
template <int NB, int WAVES>
struct Blocks
{
    static constexpr int NOFF = NB * (NB - 1) / 2;
    static constexpr int DS = (NB + WAVES - 1) / WAVES;
    static constexpr int S = DS + (NOFF + WAVES - 1) / WAVES;
    double a[S][4];
    int bi[S], bj[S];   // wave-uniform; -1: no such block at this R

    __device__ __forceinline__ void place(int wave, int nb)
    {
        wave = __builtin_amdgcn_readfirstlane(wave);
#pragma unroll
        for (int s = 0; s < DS; ++s)
        {
            const int i = s * WAVES + wave;
            bi[s] = bj[s] = i < nb ? i : -1;
        }
#pragma unroll
        for (int s = DS; s < S; ++s)
        {
            int u = (s - DS) * WAVES + (wave + WAVES * NB - NB) % WAVES, i = 1;
            while (u >= i) u -= i++;   // u = i (i - 1) / 2 + j, j < i
            bi[s] = i < nb ? i : -1;
            bj[s] = i < nb ? u : -1;
        }
    }

    // entry (r, c) of the padded matrix from get(r, c), r, c < R; the loads
    // are unconditional (a select around a load becomes a branch with a wait)
    template <class Get>
    __device__ __forceinline__ void load(int R, Get get)
    {
        const int l = int(threadIdx.x) % 64, lr = l % 16, lk = l / 16;
#pragma unroll
        for (int s = 0; s < S; ++s)
#pragma unroll
            for (int v = 0; v < 4; ++v)
                a[s][v] = get(min(max(16 * bi[s], 0) + lk + 4 * v, R - 1),
                              min(max(16 * bj[s], 0) + lr, R - 1));
#pragma unroll
        for (int s = 0; s < S; ++s)
#pragma unroll
            for (int v = 0; v < 4; ++v)
            {
                const int r = 16 * bi[s] + lk + 4 * v, c = 16 * bj[s] + lr;
                if (bi[s] < 0 || r >= R || c >= R) a[s][v] = r == c ? 1.0 : 0.0;
            }
    }

    // put(r, c, x) for every entry of the full R x R matrix held here
    template <class Put>
    __device__ __forceinline__ void store(int R, Put put) const
    {
        const int l = int(threadIdx.x) % 64, lr = l % 16, lk = l / 16;
#pragma unroll
        for (int s = 0; s < S; ++s)
        {
            if (bi[s] < 0) continue;
#pragma unroll
            for (int v = 0; v < 4; ++v)
            {
                const int r = 16 * bi[s] + lk + 4 * v, c = 16 * bj[s] + lr;
                if (r >= R || c >= R) continue;
                put(r, c, a[s][v]);
                if (s >= DS) put(c, r, a[s][v]);
            }
        }
    }

    // this lane's share of ||A||_F^2 (off-diagonal blocks stand for two) and
    // of the largest diagonal entry
    __device__ __forceinline__ void norms(int R, double& fro2, double& md) const
    {
        const int l = int(threadIdx.x) % 64, lr = l % 16, lk = l / 16;
        fro2 = 0.0;
        md = 0.0;
#pragma unroll
        for (int s = 0; s < S; ++s)
#pragma unroll
            for (int v = 0; v < 4; ++v)
            {
                const int r = 16 * bi[s] + lk + 4 * v, c = 16 * bj[s] + lr;
                const bool in = bi[s] >= 0 && r < R && c < R;
                const double x = in ? a[s][v] : 0.0;
                fro2 += (s < DS ? 1.0 : 2.0) * x * x;
                if (s < DS && in && r == c) md = fmax(md, x);
            }
    }

    // Sweeps every block pivot.  Returns 0 in a wave that met a pivot <= tau
    // (or not finite) -- the values are then of no use -- else 1.  All WAVES
    // waves call it; lds holds lds_doubles(NB) doubles.
    __device__ __forceinline__ int sweep(int R, int nb, double tau, double* lds)
    {
        const int l = int(threadIdx.x) % 64, lr = l % 16, lk = l / 16;
        double* const Dp = lds;                 // [2] 1 / D of a pivot block
        double* const Xp = lds + 32;            // [2] X of a pivot block
        double* const Up = Xp + 2 * BLK;        // [NB] panel U_i
        double* const Fp = Up + NB * BLK;       // [NB] panel -F_i
        const int own = lk * LD + lr;           // entry (lk + 4 v, lr): + 4 v LD
        const int tr = lr * LD + lk;            // entry (lr, lk + 4 v): + 4 v
        int ok = 1;
        // A_ij -= F_i U_j^T
        auto update = [&](int s) {
            const double* f = Fp + bi[s] * BLK + tr;
            const double* u = Up + bj[s] * BLK + tr;
            d4 acc = {a[s][0], a[s][1], a[s][2], a[s][3]};
#pragma unroll
            for (int q = 0; q < 4; ++q)
                acc = __builtin_amdgcn_mfma_f64_16x16x4f64(f[4 * q], u[4 * q], acc, 0, 0, 0);
#pragma unroll
            for (int v = 0; v < 4; ++v) a[s][v] = acc[v];
        };
#pragma unroll 1
        for (int K = -1; K < nb; ++K)
        {
            const double* X = Xp + (K & 1) * BLK;
            const double* D = Dp + (K & 1) * 16;
            if (K >= 0)
            {
                __syncthreads();   // X and D^-1 of pivot K; the last panels are read
#pragma unroll
                for (int s = DS; s < S; ++s)
                {
                    if (bi[s] < 0) continue;
                    if (bj[s] == K)   // A_iK: U_i = A_iK X^T (A operand: A_iK transposed, by LDS)
                    {
                        double* u = Up + bi[s] * BLK;
                        double* f = Fp + bi[s] * BLK;
                        const double ic = D[lr];
#pragma unroll
                        for (int v = 0; v < 4; ++v) u[own + 4 * v * LD] = a[s][v];
                        sync_wave();
                        double c[4];
#pragma unroll
                        for (int q = 0; q < 4; ++q) c[q] = u[tr + 4 * q];
                        sync_wave();
                        d4 ua = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
                        for (int q = 0; q < 4; ++q)
                            ua = __builtin_amdgcn_mfma_f64_16x16x4f64(c[q], X[tr + 4 * q], ua, 0, 0, 0);
#pragma unroll
                        for (int v = 0; v < 4; ++v)
                        {
                            u[own + 4 * v * LD] = ua[v];
                            f[own + 4 * v * LD] = -ua[v] * ic;
                        }
                    }
                    else if (bi[s] == K)   // A_Kj = A_jK^T: U_j^T = X A_Kj
                    {
                        double* u = Up + bj[s] * BLK;
                        double* f = Fp + bj[s] * BLK;
                        d4 ua = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
                        for (int q = 0; q < 4; ++q)
                            ua = __builtin_amdgcn_mfma_f64_16x16x4f64(X[tr + 4 * q], a[s][q], ua, 0, 0, 0);
#pragma unroll
                        for (int v = 0; v < 4; ++v)
                        {
                            u[tr + 4 * v] = ua[v];
                            f[tr + 4 * v] = -ua[v] * D[lk + 4 * v];
                        }
                    }
                }
                __syncthreads();   // the panels of pivot K
            }
            // the next pivot block first
#pragma unroll
            for (int s = 0; s < DS; ++s)
            {
                if (bi[s] != K + 1) continue;   // K + 1 == nb: none
                if (K >= 0) update(s);
                double d[4], x[4];
#pragma unroll
                for (int v = 0; v < 4; ++v)
                {
                    d[v] = a[s][v];
                    x[v] = (lk + 4 * v == lr) ? 1.0 : 0.0;
                }
                ldl16_from<0>(d, x, lr, tau, R - 16 * (K + 1), ok);
                // 1 / D: pivot c is left in lane 16 (c % 4) + c, element c / 4
                const int vc = lr / 4;
                const double dv = vc == 0 ? d[0] : vc == 1 ? d[1] : vc == 2 ? d[2] : d[3];
                const double dc = recip(bperm_d(dv, 16 * (lr % 4) + lr));
                double* Xn = Xp + ((K + 1) & 1) * BLK;
#pragma unroll
                for (int v = 0; v < 4; ++v) Xn[own + 4 * v * LD] = x[v];
                if (lk == 0) Dp[((K + 1) & 1) * 16 + lr] = dc;
                d4 acc = {0.0, 0.0, 0.0, 0.0};   // -X^T D^-1 X
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    acc = __builtin_amdgcn_mfma_f64_16x16x4f64(
                        x[q], -bperm_d(dc, lk + 4 * q) * x[q], acc, 0, 0, 0);
#pragma unroll
                for (int v = 0; v < 4; ++v) a[s][v] = acc[v];
            }
            if (K < 0) continue;
#pragma unroll
            for (int s = 0; s < S; ++s)
            {
                if (bi[s] < 0) continue;
                if (s < DS)
                {
                    if (bi[s] != K && bi[s] != K + 1) update(s);
                }
                else if (bj[s] == K)   // A_iK = F_i X
                {
                    const double* f = Fp + bi[s] * BLK + tr;
                    d4 w = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        w = __builtin_amdgcn_mfma_f64_16x16x4f64(f[4 * q], X[own + 4 * q * LD], w, 0, 0, 0);
#pragma unroll
                    for (int v = 0; v < 4; ++v) a[s][v] = -w[v];
                }
                else if (bi[s] == K)   // A_Kj = X^T F_j^T
                {
                    const double* f = Fp + bj[s] * BLK + tr;
                    d4 w = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        w = __builtin_amdgcn_mfma_f64_16x16x4f64(X[own + 4 * q * LD], f[4 * q], w, 0, 0, 0);
#pragma unroll
                    for (int v = 0; v < 4; ++v) a[s][v] = -w[v];
                }
                else
                    update(s);
            }
        }
        return ok;
    }
};

}  // namespace bsweep
}  // namespace cptc
