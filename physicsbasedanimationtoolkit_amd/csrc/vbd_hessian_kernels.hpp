// Device kernels of the adjoint's assembled step Hessian and of its fused
// conjugate-gradient iteration.
//
// The step Hessian H = M / h^2 + sum_e w_e d2Psi_e/dx2 is fixed during one
// linear solve (it is evaluated at the step's minimiser), so it is assembled
// once per solve into 3x3 blocks over the updated vertices (block-sparse rows,
// columns ascending) and every product of the solve is a block-sparse
// matrix-vector product: 40 bytes per block (36 B of values + the column)
// instead of re-evaluating the Stable Neo-Hookean Hessian of every incident tet
// per product. RowAssemble forms each tet's blocks once per row vertex and
// sums every block's terms in a fixed order. For tet e with shape-function gradient rows
// g_a, g_b of two of its vertices, F its deformation gradient and J = det F, the
// block is
//   w mu (g_a . g_b) I + w lambda (cof F g_a)(cof F g_b)^T
//     - w lambda (J - alpha) [F (g_a x g_b)]_x
// (d2Psi/dF2 = mu I + lambda cof F (x) cof F + lambda (J - alpha) d2J/dF2
// contracted with g_a and g_b; d2J/dF2 contracts to the cross-product matrix).
// The terms are formed in FP64 and kept in FP32; each block sums them in FP64
// in a fixed order (ascending tet) and is stored in FP32.
#pragma once

#include "vbd_adjoint_kernels.hpp"

#include <type_traits>

namespace pbat_vbd::device {

// Values of the block-sparse step Hessian, structure of arrays per block:
// a = (h00, h01, h02, h10), b = (h11, h12, h20, h21), c = h22.
struct BsrValues
{
    float4* __restrict__ a;
    float4* __restrict__ b;
    float* __restrict__ c;
};

// Sparsity pattern and assembly sources: block k sits in row blockRow[k] at
// column col[k]; its sources src[srcPtr[k] .. srcPtr[k+1]) are 16 e + 4 la + lb
// (tet e, local vertex la of the row vertex, lb of the column vertex),
// ascending in e.
struct BsrPattern
{
    int const* __restrict__ rowPtr; // nRows + 1
    int const* __restrict__ col;
    int const* __restrict__ blockRow;
    int const* __restrict__ srcPtr;
    int const* __restrict__ src;
    int nRows;
    int nBlocks;
};

// General assembly (rows longer than RowAssemble takes): one thread per block,
// each source's tet recomputed. Diagonal blocks also receive m_i / h^2 I and
// write the FP64-inverted block to dinv[2 i], dinv[2 i + 1] as
// (00, 01, 02, 11), (12, 22).
__global__ __launch_bounds__(256) void BsrAssemble(float4 const* __restrict__ xs, int4 const* __restrict__ tetv,
                                                   float4 const* __restrict__ tgp, BsrPattern p, double invDt2,
                                                   BsrValues v, float4* __restrict__ dinv,
                                                   int const* __restrict__ rowVertex)
{
    int const k = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x);
    if (k >= p.nBlocks)
        return;
    int const i = p.blockRow[k], j = p.col[k];
    double H[3][3] = {{0., 0., 0.}, {0., 0., 0.}, {0., 0., 0.}};
    for (int s = p.srcPtr[k]; s < p.srcPtr[k + 1]; ++s)
    {
        int const code = p.src[s];
        int const e = code >> 4, la = (code >> 2) & 3, lb = code & 3;
        int4 const t = tetv[e];
        float4 const q0 = tgp[3 * e], q1 = tgp[3 * e + 1], q2 = tgp[3 * e + 2];
        float4 const x0 = xs[t.x], x1 = xs[t.y], x2 = xs[t.z], x3 = xs[t.w];
        double g[4][3] = {{0., 0., 0.}, {q0.x, q0.y, q0.z}, {q0.w, q1.x, q1.y}, {q1.z, q1.w, q2.x}};
        for (int c = 0; c < 3; ++c)
            g[0][c] = -(g[1][c] + g[2][c] + g[3][c]);
        double const d[3][3] = {{double(x1.x) - x0.x, double(x1.y) - x0.y, double(x1.z) - x0.z},
                                {double(x2.x) - x0.x, double(x2.y) - x0.y, double(x2.z) - x0.z},
                                {double(x3.x) - x0.x, double(x3.y) - x0.y, double(x3.z) - x0.z}};
        double F[3][3]; // F[row][col] = sum_k d[k][row] g[k + 1][col]
        for (int r = 0; r < 3; ++r)
            for (int c = 0; c < 3; ++c)
                F[r][c] = d[0][r] * g[1][c] + d[1][r] * g[2][c] + d[2][r] * g[3][c];
        double cof[3][3]; // column c = f_{c+1} x f_{c+2}
        for (int c = 0; c < 3; ++c)
        {
            int const c1 = (c + 1) % 3, c2 = (c + 2) % 3;
            cof[0][c] = F[1][c1] * F[2][c2] - F[2][c1] * F[1][c2];
            cof[1][c] = F[2][c1] * F[0][c2] - F[0][c1] * F[2][c2];
            cof[2][c] = F[0][c1] * F[1][c2] - F[1][c1] * F[0][c2];
        }
        double const J = F[0][0] * cof[0][0] + F[1][0] * cof[1][0] + F[2][0] * cof[2][0];
        double const* ga = g[la];
        double const* gb = g[lb];
        double ca[3], cb[3], w[3];
        double const gx[3] = {ga[1] * gb[2] - ga[2] * gb[1], ga[2] * gb[0] - ga[0] * gb[2],
                              ga[0] * gb[1] - ga[1] * gb[0]};
        for (int r = 0; r < 3; ++r)
        {
            ca[r] = cof[r][0] * ga[0] + cof[r][1] * ga[1] + cof[r][2] * ga[2];
            cb[r] = cof[r][0] * gb[0] + cof[r][1] * gb[1] + cof[r][2] * gb[2];
            w[r] = F[r][0] * gx[0] + F[r][1] * gx[1] + F[r][2] * gx[2];
        }
        double const wmu = q2.y, wlam = q2.z, sk = double(q2.z) * (J - double(q2.w));
        double const dg = wmu * (ga[0] * gb[0] + ga[1] * gb[1] + ga[2] * gb[2]);
        // - sk [w]_x with [w]_x = [[0, -w2, w1], [w2, 0, -w0], [-w1, w0, 0]]
        double const S[3][3] = {{0., sk * w[2], -sk * w[1]}, {-sk * w[2], 0., sk * w[0]}, {sk * w[1], -sk * w[0], 0.}};
        for (int r = 0; r < 3; ++r)
            for (int c = 0; c < 3; ++c)
                H[r][c] += (r == c ? dg : 0.) + wlam * ca[r] * cb[c] + S[r][c];
    }
    if (i == j)
    {
        double const m = double(xs[rowVertex[i]].w) * invDt2;
        H[0][0] += m, H[1][1] += m, H[2][2] += m;
        Inverse3 const C(H[0][0], 0.5 * (H[0][1] + H[1][0]), 0.5 * (H[0][2] + H[2][0]), H[1][1],
                         0.5 * (H[1][2] + H[2][1]), H[2][2]);
        dinv[2 * i] = make_float4(static_cast<float>(C.c00 * C.inv), static_cast<float>(C.c01 * C.inv),
                                  static_cast<float>(C.c02 * C.inv), static_cast<float>(C.c11 * C.inv));
        dinv[2 * i + 1] = make_float4(static_cast<float>(C.c12 * C.inv), static_cast<float>(C.c22 * C.inv), 0.f, 0.f);
    }
    v.a[k] = make_float4(static_cast<float>(H[0][0]), static_cast<float>(H[0][1]), static_cast<float>(H[0][2]),
                         static_cast<float>(H[1][0]));
    v.b[k] = make_float4(static_cast<float>(H[1][1]), static_cast<float>(H[1][2]), static_cast<float>(H[2][0]),
                         static_cast<float>(H[2][1]));
    v.c[k] = static_cast<float>(H[2][2]);
}

// The FP32 state's tet (F, cof F, J in FP64) and the Stable Neo-Hookean
// constants, for the blocks
//   H(a, b) = w mu (g_a . g_b) I + w lambda (cof F g_a)(cof F g_b)^T
//             - w lambda (J - alpha) [F (g_a x g_b)]_x.
struct TetHessian
{
    double g[4][3];  // shape-function gradient rows
    double F[3][3];  // F[row][col]
    double cg[4][3]; // cof F g_l
    double wmu, wlam, sk;
    __device__ __forceinline__ TetHessian(float4 const* __restrict__ xs, int4 const& t, float4 const& q0,
                                          float4 const& q1, float4 const& q2)
    {
        float4 const x0 = xs[t.x], x1 = xs[t.y], x2 = xs[t.z], x3 = xs[t.w];
        double const G[3][3] = {{q0.x, q0.y, q0.z}, {q0.w, q1.x, q1.y}, {q1.z, q1.w, q2.x}};
#pragma unroll
        for (int c = 0; c < 3; ++c)
        {
            g[1][c] = G[0][c], g[2][c] = G[1][c], g[3][c] = G[2][c];
            g[0][c] = -(G[0][c] + G[1][c] + G[2][c]);
        }
        double const d[3][3] = {{double(x1.x) - x0.x, double(x1.y) - x0.y, double(x1.z) - x0.z},
                                {double(x2.x) - x0.x, double(x2.y) - x0.y, double(x2.z) - x0.z},
                                {double(x3.x) - x0.x, double(x3.y) - x0.y, double(x3.z) - x0.z}};
#pragma unroll
        for (int r = 0; r < 3; ++r)
#pragma unroll
            for (int c = 0; c < 3; ++c)
                F[r][c] = d[0][r] * G[0][c] + d[1][r] * G[1][c] + d[2][r] * G[2][c];
        double cof[3][3]; // column c = f_{c+1} x f_{c+2}
#pragma unroll
        for (int c = 0; c < 3; ++c)
        {
            int const c1 = (c + 1) % 3, c2 = (c + 2) % 3;
            cof[0][c] = F[1][c1] * F[2][c2] - F[2][c1] * F[1][c2];
            cof[1][c] = F[2][c1] * F[0][c2] - F[0][c1] * F[2][c2];
            cof[2][c] = F[0][c1] * F[1][c2] - F[1][c1] * F[0][c2];
        }
        double const J = F[0][0] * cof[0][0] + F[1][0] * cof[1][0] + F[2][0] * cof[2][0];
        wmu = q2.y, wlam = q2.z, sk = double(q2.z) * (J - double(q2.w));
#pragma unroll
        for (int l = 0; l < 4; ++l)
#pragma unroll
            for (int r = 0; r < 3; ++r)
                cg[l][r] = cof[r][0] * g[l][0] + cof[r][1] * g[l][1] + cof[r][2] * g[l][2];
    }
    // H(a, b) for the row's gradient row ga and cof F ga, column lb
    template <int lb>
    __device__ __forceinline__ void Block(double const (&ga)[3], double const (&ca)[3], double (&H)[9]) const
    {
        double const* gb = g[lb];
        double const gx[3] = {ga[1] * gb[2] - ga[2] * gb[1], ga[2] * gb[0] - ga[0] * gb[2],
                              ga[0] * gb[1] - ga[1] * gb[0]};
        double w[3];
#pragma unroll
        for (int r = 0; r < 3; ++r)
            w[r] = sk * (F[r][0] * gx[0] + F[r][1] * gx[1] + F[r][2] * gx[2]);
        double const dg = wmu * (ga[0] * gb[0] + ga[1] * gb[1] + ga[2] * gb[2]);
        // - sk [F (g_a x g_b)]_x with [w]_x = [[0, -w2, w1], [w2, 0, -w0], [-w1, w0, 0]]
        double const S[9] = {0., w[2], -w[1], -w[2], 0., w[0], w[1], -w[0], 0.};
#pragma unroll
        for (int r = 0; r < 3; ++r)
#pragma unroll
            for (int c = 0; c < 3; ++c)
                H[3 * r + c] = (r == c ? dg : 0.) + wlam * ca[r] * cg[lb][c] + S[3 * r + c];
    }
};

template <int kCtrl>
__device__ __forceinline__ double DppRead(double x)
{
    int const lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), kCtrl, 0xF, 0xF, false);
    int const hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), kCtrl, 0xF, 0xF, false);
    return __hiloint2double(hi, lo);
}

template <int L>
__device__ __forceinline__ double GroupSum(double x)
{
    if constexpr (L >= 2)
        x += DppRead<0xB1>(x);
    if constexpr (L >= 4)
        x += DppRead<0x4E>(x);
    if constexpr (L >= 8)
        x += DppRead<0x141>(x);
    if constexpr (L >= 16)
        x += DppRead<0x140>(x);
    if constexpr (L >= 32)
        x += __shfl_xor(x, 16);
    if constexpr (L >= 64)
        x += __shfl_xor(x, 32);
    return x;
}

// Row-major assembly: incidences of row i (tet e, local vertex la of the row
// vertex) in incCode[incPtr[i] .. incPtr[i + 1]) as 4 e + la, ascending e;
// incSlot holds, per incidence, the position in the row of the tet's local
// vertices 0..3 (-1: not updated).
struct RowAssembleArgs
{
    float4 const* __restrict__ xs;
    int4 const* __restrict__ tetv;
    float4 const* __restrict__ tgp;
    int const* __restrict__ incPtr;
    int const* __restrict__ incCode;
    int4 const* __restrict__ incSlot;
    uint2 const* __restrict__ sources; // RowAssembleShort
    int const* __restrict__ rowPtr;
    int const* __restrict__ col;
    int nRows;
    double invDt2;
    BsrValues v;
    float4* __restrict__ dinv;
    int const* __restrict__ rowVertex; // vertex of each row
};

// 32 lanes per row, two rows per wave, one wave per workgroup. The row's
// incidences are taken 32 at a time, one per lane: the lane forms its tet's
// F, cof F and J in FP64 and the four blocks (la, lb), lb = 0..3. The diagonal
// block (la, la) of every incidence is summed over the row's lanes by a
// fixed-order butterfly in FP64; the three others are staged in LDS as FP32,
// and lane l then adds, for each off-diagonal block it owns (l, l + 32, ..., NB
// of them, below the row length), the staged blocks that fall on it in
// incidence order (ascending tet), in FP64, visiting only the incidences its
// block appears in (a bit mask from the staged row positions). Diagonal blocks
// also receive m_i / h^2 I and write the FP64-inverted block to dinv[2 i],
// dinv[2 i + 1] as (00, 01, 02, 11), (12, 22).
template <int NB>
__global__ __launch_bounds__(64) void RowAssemble(RowAssembleArgs a)
{
    constexpr int L = 32;
    __shared__ float stage[2][L][4][9];
    __shared__ int4 slotS[2][L];
    int const lane = static_cast<int>(threadIdx.x) & (L - 1), half = static_cast<int>(threadIdx.x) >> 5;
    int const i = static_cast<int>(blockIdx.x) * 2 + half;
    int kb = 0, ke = 0, rb = 0, nb = 0;
    if (i < a.nRows)
        kb = a.incPtr[i], ke = a.incPtr[i + 1], rb = a.rowPtr[i], nb = a.rowPtr[i + 1] - rb;
    int const mine = (ke - kb + L - 1) / L;
    int const batches = max(mine, __shfl_xor(mine, 32)); // uniform over the wave
    double acc[NB][9];
#pragma unroll
    for (int o = 0; o < NB; ++o)
#pragma unroll
        for (int c = 0; c < 9; ++c)
            acc[o][c] = 0.;
    double diag[9] = {0., 0., 0., 0., 0., 0., 0., 0., 0.};
    int diagSlot = -1; // the row vertex's position in its row (from its first incidence)
    for (int bt = 0; bt < batches; ++bt)
    {
        int const k = kb + bt * L + lane;
        double Hd[9] = {0., 0., 0., 0., 0., 0., 0., 0., 0.};
        if (k < ke)
        {
            int const code = a.incCode[k];
            int const e = code >> 2, la = code & 3;
            int4 const sl = a.incSlot[k];
            TetHessian const T(a.xs, a.tetv[e], a.tgp[3 * e], a.tgp[3 * e + 1], a.tgp[3 * e + 2]);
            double ga[3], ca[3];
#pragma unroll
            for (int c = 0; c < 3; ++c)
            {
                ga[c] = la == 0 ? T.g[0][c] : la == 1 ? T.g[1][c] : la == 2 ? T.g[2][c] : T.g[3][c];
                ca[c] = la == 0 ? T.cg[0][c] : la == 1 ? T.cg[1][c] : la == 2 ? T.cg[2][c] : T.cg[3][c];
            }
            double H[9];
            auto keep = [&](int lb) {
                if (lb == la)
                {
#pragma unroll
                    for (int c = 0; c < 9; ++c)
                        Hd[c] = H[c];
                }
                else
                {
#pragma unroll
                    for (int c = 0; c < 9; ++c)
                        stage[half][lane][lb][c] = static_cast<float>(H[c]);
                }
            };
            T.Block<0>(ga, ca, H);
            keep(0);
            T.Block<1>(ga, ca, H);
            keep(1);
            T.Block<2>(ga, ca, H);
            keep(2);
            T.Block<3>(ga, ca, H);
            keep(3);
            slotS[half][lane] = sl;
        }
        // diagonal terms: butterfly over the row's 32 lanes (idle lanes add 0)
#pragma unroll
        for (int c = 0; c < 9; ++c)
        {
            double v = Hd[c];
#pragma unroll
            for (int off = 1; off < L; off <<= 1)
                v += __shfl_xor(v, off, L);
            diag[c] += v;
        }
        __syncthreads();
        if (bt == 0)
        {
            // every row has an incidence; lane 0 of the row holds its first
            int const code0 = kb < ke ? a.incCode[kb] : 0;
            int4 const s0 = slotS[half][0];
            int const la0 = code0 & 3;
            diagSlot = kb < ke ? (la0 == 0 ? s0.x : la0 == 1 ? s0.y : la0 == 2 ? s0.z : s0.w) : -1;
        }
        int const cnt = min(L, max(0, ke - kb - bt * L));
#pragma unroll
        for (int o = 0; o < NB; ++o)
        {
            int const b = lane + o * L;
            if (b >= nb || b == diagSlot)
                continue;
            unsigned mask = 0u;
            for (int j = 0; j < cnt; ++j)
            {
                int4 const sl = slotS[half][j];
                if (sl.x == b || sl.y == b || sl.z == b || sl.w == b)
                    mask |= 1u << j;
            }
            while (mask)
            {
                int const j = __builtin_ctz(mask);
                mask &= mask - 1u;
                int4 const sl = slotS[half][j];
                int const s = sl.x == b ? 0 : sl.y == b ? 1 : sl.z == b ? 2 : 3;
#pragma unroll
                for (int c = 0; c < 9; ++c)
                    acc[o][c] += stage[half][j][s][c];
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int o = 0; o < NB; ++o)
    {
        int const b = lane + o * L;
        if (b >= nb)
            continue;
        int const kBlock = rb + b;
        double* H = acc[o];
        if (b == diagSlot)
        {
            double const m = double(a.xs[a.rowVertex[i]].w) * a.invDt2;
#pragma unroll
            for (int c = 0; c < 9; ++c)
                H[c] = diag[c];
            H[0] += m, H[4] += m, H[8] += m;
            Inverse3 const C(H[0], 0.5 * (H[1] + H[3]), 0.5 * (H[2] + H[6]), H[4], 0.5 * (H[5] + H[7]), H[8]);
            a.dinv[2 * i] = make_float4(static_cast<float>(C.c00 * C.inv), static_cast<float>(C.c01 * C.inv),
                                        static_cast<float>(C.c02 * C.inv), static_cast<float>(C.c11 * C.inv));
            a.dinv[2 * i + 1] =
                make_float4(static_cast<float>(C.c12 * C.inv), static_cast<float>(C.c22 * C.inv), 0.f, 0.f);
        }
        a.v.a[kBlock] = make_float4(static_cast<float>(H[0]), static_cast<float>(H[1]), static_cast<float>(H[2]),
                                    static_cast<float>(H[3]));
        a.v.b[kBlock] = make_float4(static_cast<float>(H[4]), static_cast<float>(H[5]), static_cast<float>(H[6]),
                                    static_cast<float>(H[7]));
        a.v.c[kBlock] = static_cast<float>(H[8]);
    }
}

// The same for patterns whose rows have at most 32 blocks and 32 incidences and whose
// off-diagonal blocks have at most 8 sources: the sources of a block are listed (bytes
// 4 incidence + local vertex, ascending, 255 behind the last), so no lane looks for
// them, the staged values lie value-major (lanes on different banks), and the
// symmetric diagonal is summed as 6 values across DPP rows. 224,000 rows 346 -> 189 us,
// 36,000 rows 63 -> 34; what is left is the FP64 arithmetic of a tet per lane.
[[maybe_unused]] static __global__ __launch_bounds__(64) void RowAssembleShort(RowAssembleArgs a)
{
    constexpr int L = 32;
    __shared__ float stage[2][36][L + 1];
    int const lane = static_cast<int>(threadIdx.x) & (L - 1), half = static_cast<int>(threadIdx.x) >> 5;
    int const i = static_cast<int>(blockIdx.x) * 2 + half;
    int kb = 0, ke = 0, rb = 0, nb = 0;
    if (i < a.nRows)
        kb = a.incPtr[i], ke = a.incPtr[i + 1], rb = a.rowPtr[i], nb = a.rowPtr[i + 1] - rb;
    uint2 const list = lane < nb ? a.sources[rb + lane] : make_uint2(~0u, ~0u);
    bool const isDiag = lane < nb && a.col[rb + lane] == i;
    double d6[6] = {0., 0., 0., 0., 0., 0.};
    if (kb + lane < ke)
    {
        int const code = a.incCode[kb + lane];
        int const e = code >> 2, la = code & 3;
        TetHessian const T(a.xs, a.tetv[e], a.tgp[3 * e], a.tgp[3 * e + 1], a.tgp[3 * e + 2]);
        double ga[3], ca[3];
#pragma unroll
        for (int c = 0; c < 3; ++c)
        {
            ga[c] = la == 0 ? T.g[0][c] : la == 1 ? T.g[1][c] : la == 2 ? T.g[2][c] : T.g[3][c];
            ca[c] = la == 0 ? T.cg[0][c] : la == 1 ? T.cg[1][c] : la == 2 ? T.cg[2][c] : T.cg[3][c];
        }
        // the block (la, la), whose skew part vanishes
        double const dg = T.wmu * (ga[0] * ga[0] + ga[1] * ga[1] + ga[2] * ga[2]);
        d6[0] = dg + T.wlam * ca[0] * ca[0], d6[1] = T.wlam * ca[0] * ca[1], d6[2] = T.wlam * ca[0] * ca[2];
        d6[3] = dg + T.wlam * ca[1] * ca[1], d6[4] = T.wlam * ca[1] * ca[2], d6[5] = dg + T.wlam * ca[2] * ca[2];
        auto put = [&](int lb, double const (&H)[9]) {
#pragma unroll
            for (int c = 0; c < 9; ++c)
                stage[half][9 * lb + c][lane] = static_cast<float>(H[c]);
        };
        double H[9];
        T.Block<0>(ga, ca, H), put(0, H);
        T.Block<1>(ga, ca, H), put(1, H);
        T.Block<2>(ga, ca, H), put(2, H);
        T.Block<3>(ga, ca, H), put(3, H);
    }
#pragma unroll
    for (int c = 0; c < 6; ++c)
        d6[c] = GroupSum<L>(d6[c]);
    __syncthreads();
    if (lane >= nb)
        return;
    double H[9];
    if (isDiag)
    {
        double const m = double(a.xs[a.rowVertex[i]].w) * a.invDt2;
        H[0] = d6[0] + m, H[4] = d6[3] + m, H[8] = d6[5] + m;
        H[1] = H[3] = d6[1], H[2] = H[6] = d6[2], H[5] = H[7] = d6[4];
        Inverse3 const C(H[0], H[1], H[2], H[4], H[5], H[8]);
        a.dinv[2 * i] = make_float4(static_cast<float>(C.c00 * C.inv), static_cast<float>(C.c01 * C.inv),
                                    static_cast<float>(C.c02 * C.inv), static_cast<float>(C.c11 * C.inv));
        a.dinv[2 * i + 1] =
            make_float4(static_cast<float>(C.c12 * C.inv), static_cast<float>(C.c22 * C.inv), 0.f, 0.f);
    }
    else
    {
#pragma unroll
        for (int c = 0; c < 9; ++c)
            H[c] = 0.;
#pragma unroll
        for (int k = 0; k < 8; ++k)
        {
            unsigned int const b = ((k < 4 ? list.x : list.y) >> (8 * (k & 3))) & 255u;
            if (b == 255u)
                break;
            float const* const from = &stage[half][9 * (b & 3u)][b >> 2];
#pragma unroll
            for (int c = 0; c < 9; ++c)
                H[c] += from[c * (L + 1)];
        }
    }
    int const k = rb + lane;
    a.v.a[k] = make_float4(static_cast<float>(H[0]), static_cast<float>(H[1]), static_cast<float>(H[2]),
                           static_cast<float>(H[3]));
    a.v.b[k] = make_float4(static_cast<float>(H[4]), static_cast<float>(H[5]), static_cast<float>(H[6]),
                           static_cast<float>(H[7]));
    a.v.c[k] = static_cast<float>(H[8]);
}

enum class BsrMode : int
{
    kProduct = 0,        // out = H y
    kProductDot = 1,     // out = H y, acc[mesh] += y . H y
    kGaussSeidel = 2,    // rows of one colour: y_i += D_i^-1 (b_i - (H y)_i)
    kGaussSeidelDot = 3  // same, then acc[mesh] += b_i . y_i
};

struct BsrArgs
{
    int const* __restrict__ rowPtr;
    int const* __restrict__ col;
    float4 const* __restrict__ va;
    float4 const* __restrict__ vb;
    float const* __restrict__ vc;
    float4* __restrict__ y;          // vector multiplied (Gauss-Seidel: updated in place)
    float4 const* __restrict__ b;    // right-hand side (Gauss-Seidel)
    float4* __restrict__ out;        // product
    float4 const* __restrict__ dinv; // inverse diagonal blocks (Gauss-Seidel)
    int const* __restrict__ meshOf;
    CgState cg;
    double* __restrict__ acc; // accumulators (dot modes), array accArray
    int accArray;
    int vbeg, vend;
    int xcdChunk;
};

// (H v)_row over blocks [kb, ke) of one row: lane l of the row's L lanes takes
// blocks l, l + L, ..., the first K of them loaded together before
// accumulating; the group sum leaves the product in every lane of the group.
template <int L, int K>
__device__ __forceinline__ float3 RowProduct(BsrArgs const& a, int kb, int ke, int lane)
{
    float hx = 0.f, hy = 0.f, hz = 0.f;
    int cj[K];
    float4 A[K], B[K];
    float C[K];
#pragma unroll
    for (int u = 0; u < K; ++u)
    {
        int const k = kb + lane + u * L;
        cj[u] = -1;
        if (k < ke)
        {
            cj[u] = a.col[k];
            A[u] = a.va[k];
            B[u] = a.vb[k];
            C[u] = a.vc[k];
        }
    }
    float4 P[K];
#pragma unroll
    for (int u = 0; u < K; ++u)
        if (cj[u] >= 0)
            P[u] = a.y[cj[u]];
#pragma unroll
    for (int u = 0; u < K; ++u)
        if (cj[u] >= 0)
        {
            hx += A[u].x * P[u].x + A[u].y * P[u].y + A[u].z * P[u].z;
            hy += A[u].w * P[u].x + B[u].x * P[u].y + B[u].y * P[u].z;
            hz += B[u].z * P[u].x + B[u].w * P[u].y + C[u] * P[u].z;
        }
    for (int k = kb + lane + K * L; k < ke; k += L)
    {
        float4 const Ak = a.va[k], Bk = a.vb[k];
        float const Ck = a.vc[k];
        float4 const Pk = a.y[a.col[k]];
        hx += Ak.x * Pk.x + Ak.y * Pk.y + Ak.z * Pk.z;
        hy += Ak.w * Pk.x + Bk.x * Pk.y + Bk.y * Pk.z;
        hz += Bk.z * Pk.x + Bk.w * Pk.y + Ck * Pk.z;
    }
    return make_float3(GroupSum<L>(hx), GroupSum<L>(hy), GroupSum<L>(hz));
}

// L lanes per row of [vbeg, vend): products and Gauss-Seidel passes.
template <int L, int K, BsrMode M>
__global__ __launch_bounds__(256) void BsrKernel(BsrArgs a)
{
    constexpr bool kGS = M == BsrMode::kGaussSeidel || M == BsrMode::kGaussSeidelDot;
    constexpr bool kDot = M == BsrMode::kGaussSeidelDot || M == BsrMode::kProductDot;
    int block = static_cast<int>(blockIdx.x);
    if (a.xcdChunk > 0)
        block = (block & 7) * a.xcdChunk + (block >> 3);
    int const tid = block * static_cast<int>(blockDim.x) + static_cast<int>(threadIdx.x);
    int const lane = tid & (L - 1);
    int const row = a.vbeg + tid / L;
    bool const active = row < a.vend;
    int kb = 0, ke = 0;
    if (active)
    {
        kb = a.rowPtr[row];
        ke = a.rowPtr[row + 1];
    }
    float3 const h = RowProduct<L, K>(a, kb, ke, lane);
    bool const leader = active && lane == 0;
    double dot = 0.;
    if (leader)
    {
        if constexpr (kGS)
        {
            float4 const bo = a.b[row], yo = a.y[row];
            float const rx = bo.x - h.x, ry = bo.y - h.y, rz = bo.z - h.z;
            float4 const D0 = a.dinv[2 * row], D1 = a.dinv[2 * row + 1];
            float4 const r = make_float4(yo.x + D0.x * rx + D0.y * ry + D0.z * rz,
                                         yo.y + D0.y * rx + D0.w * ry + D1.x * rz,
                                         yo.z + D0.z * rx + D1.x * ry + D1.y * rz, 0.f);
            a.y[row] = r;
            dot = double(bo.x) * r.x + double(bo.y) * r.y + double(bo.z) * r.z;
        }
        else
        {
            a.out[row] = make_float4(h.x, h.y, h.z, 0.f);
            if constexpr (M == BsrMode::kProductDot)
            {
                float4 const yr = a.y[row];
                dot = double(yr.x) * h.x + double(yr.y) * h.y + double(yr.z) * h.z;
            }
        }
    }
    if constexpr (kDot)
        BlockAccumulate(dot, leader ? a.meshOf[row] : -1, a.acc, a.accArray, a.cg.nM);
}

// ---- fused conjugate gradients -----------------------------------------------
// Preconditioned CG in the one-reduction form of Chronopoulos and Gear: with
// z = M^-1 r and w = H z, delta = z . w and gamma = r . z give
//   beta = gamma / gamma_old,  alpha = gamma / (delta - beta gamma / alpha_old),
//   p = z + beta p,  s = w + beta s (= H p),  y += alpha p,  r -= alpha s,
// so the product needs no direction and an iteration has one point where every
// sum of the mesh is needed (CgUpdate1), at the head of a launch that has to wait
// for the product anyway. The product reads one vector per block instead of two
// (z and p_old), and no launch of its own takes the scalars (32^3: 4.6 us of 27).
//
// Two-level: M^-1 = q(D^-1 H) D^-1 + Z (Z^T H Z)^-1 Z^T, q the degree-2 Chebyshev
// polynomial for the spectrum [kChebyMax / kChebyRatio, kChebyMax] of D^-1 H (the
// smoother of the modes the coarse space leaves). kChebyMax = 4 bounds the
// spectrum when the tets' Hessians are positive semi-definite (each couples 4
// vertices); above it q lambda = 1 - T_3 stays positive (T_3 is odd), so M^-1 stays
// positive definite where indefinite tets push the spectrum past it. It halves the
// iterations for two more products each (24^3: 241 -> 120 iterations from zero),
// and one of them shares its launch with the coarse product.
// Per iteration: CgUpdate1 (y, r, z1 = D^-1 r / theta, rc = Z^T r); CoarsePoly
// (coarse product, z2); BsrPoly<kPolyLast> (z3 + Z zc, r . z); BsrPoly<kPolyProduct>
// (w, z . w).
//
// Row chunks: each run of rows of one mesh (and one colour) is cut into chunks of
// at most kChunkThreads / L rows, numbered mesh-major, so the chunks of a mesh are
// consecutive and every chunk holds rows of one mesh. A chunk's sums depend only
// on its own rows, every sum is taken in a fixed order and no atomics are used, so
// a solve gives the same bits on every run and a mesh gives the same bits alone or
// in a batch.
constexpr int kChunkThreads = 512;
constexpr double kChebyMax = 4., kChebyRatio = 45.;

struct ChebyConstants
{
    float invTheta; // z1 = invTheta D^-1 r
    float a2, b2;   // z2 = z1 + a2 z1 + b2 D^-1 (r - H z1)
    float a3, b3;   // z3 = z2 + a3 (z2 - z1) + b3 D^-1 (r - H z2)
};

inline ChebyConstants MakeCheby()
{
    double const lo = kChebyMax / kChebyRatio, theta = 0.5 * (kChebyMax + lo), half = 0.5 * (kChebyMax - lo);
    double const sigma = theta / half, r1 = 1. / sigma, r2 = 1. / (2. * sigma - r1), r3 = 1. / (2. * sigma - r2);
    return ChebyConstants{static_cast<float>(1. / theta), static_cast<float>(r2 * r1),
                          static_cast<float>(2. * r2 / half), static_cast<float>(r3 * r2),
                          static_cast<float>(2. * r3 / half)};
}

// Sum over the wave in a fixed order, in every lane: 16-lane rows by DPP, then
// the four row sums in order.
__device__ __forceinline__ double ReadLane(double x, int lane)
{
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(x), lane),
                            __builtin_amdgcn_readlane(__double2loint(x), lane));
}

__device__ __forceinline__ double WaveSum(double x)
{
    x += DppRead<0xB1>(x);
    x += DppRead<0x4E>(x);
    x += DppRead<0x141>(x);
    x += DppRead<0x140>(x);
    return ((ReadLane(x, 0) + ReadLane(x, 16)) + ReadLane(x, 32)) + ReadLane(x, 48);
}

// Thread t of a group of N threads sums v[b + t], v[b + t + N], ... in that
// order, issuing the loads U at a time (the order, and so the bits, do not
// depend on U). Out-of-range entries load the last one and add an exact 0:
// written as a guarded load the compiler branches around each and waits after it.
template <int N, int U = 8>
__device__ __forceinline__ double StridedSum(double const* __restrict__ v, int b, int e, int t)
{
    double s = 0.;
    for (int k0 = b + t; k0 < e; k0 += U * N)
    {
        double x[U];
#pragma unroll
        for (int u = 0; u < U; ++u)
            x[u] = v[min(k0 + u * N, e - 1)];
#pragma unroll
        for (int u = 0; u < U; ++u)
            s += k0 + u * N < e ? x[u] : 0.;
    }
    return s;
}

// Sums of V values over the 128 threads of a workgroup in a fixed order (each
// wave's sum, then wave 0 + wave 1); every thread calls it and gets the sums in v.
template <int V>
__device__ __forceinline__ void Sum128(double (&v)[V], double (*lds)[V])
{
#pragma unroll
    for (int i = 0; i < V; ++i)
        v[i] = WaveSum(v[i]);
    __syncthreads();
    if ((threadIdx.x & 63) == 0)
#pragma unroll
        for (int i = 0; i < V; ++i)
            lds[threadIdx.x >> 6][i] = v[i];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < V; ++i)
        v[i] = lds[0][i] + lds[1][i];
}

// The recurrence's vectors y, r, p and s are kept in FP64: the one-reduction form
// never forms H p, so an FP32 s drifts from it and an FP32 p from what s and y
// have seen (errors of 3e-6 against 1.9e-6 of the classical form at the same
// tolerance); w = H z is summed and kept in FP64 too. z and the preconditioner stay
// FP32.
struct Vec3d
{
    double x, y, z;
};

// Device arrays of the fused solvers, rows aggregate-major.
struct FusedArgs
{
    // Hessian blocks
    int const* __restrict__ rowPtr;
    int const* __restrict__ col;
    float4 const* __restrict__ va;
    float4 const* __restrict__ vb;
    float const* __restrict__ vc;
    float4 const* __restrict__ dinv;
    // vectors
    Vec3d* y;
    Vec3d* r;
    Vec3d* p;
    Vec3d* s;
    float4* z;  // z1 of the polynomial, then z
    float4* z2;
    Vec3d* w; // H z
    float4 const* y0; // initial guess
    float4 const* b;
    // per chunk: (first row, end row, mesh, 0); its r . z and z . w
    int4 const* __restrict__ chunks;
    double* gammaPart;
    double* deltaPart;
    int nChunks;
    // per aggregate: (mesh, first row, end row, whether it is its mesh's first), its r . r (and r . z for block Jacobi) of the even and odd iterations, b . b
    int4 const* __restrict__ aggInfo;
    double* rrPart[2];
    double* rzPart[2];
    double* bbPart;
    int* aggDone; // its mesh's done flag
    int nAgg;
    // coarse space (two-level): restriction, correction (2 float4 per aggregate:
    // translation, rotation), offsets d and aggregate of each row
    double* rc;
    float4* zc;
    float4 const* __restrict__ coarseD;
    int const* __restrict__ aggOfRow;
    float const* __restrict__ coarseF;
    int4 const* __restrict__ coarseInfo;           // per aggregate: (b0, n, ., .)
    long long const* __restrict__ coarseRowOffset; // per aggregate: its first row in coarseF
    int xcdChunk; // > 0: row workgroups per XCD
    int coarseBlocks; // CoarsePoly: workgroups of the coarse product (a multiple of 8)
    ChebyConstants q;
    CgState cg;
    int* doneOut; // host-mapped copy of the done flags
};

__device__ __forceinline__ float4 ApplyInverse(float4 const& D0, float4 const& D1, float x, float y, float z)
{
    return make_float4(D0.x * x + D0.y * y + D0.z * z, D0.y * x + D0.w * y + D1.x * z, D0.z * x + D1.x * y + D1.y * z,
                       0.f);
}

// Blocks of the row that thread t works on, of the rows [first, end).
template <int L>
__device__ __forceinline__ int2 RowExtent(FusedArgs const& a, int first, int end)
{
    int const row = first + static_cast<int>(threadIdx.x) / L;
    return row < end ? make_int2(a.rowPtr[row], a.rowPtr[row + 1]) : make_int2(0, 0);
}

// H v of threads / L consecutive rows (the thread's extent given), L lanes per row:
// lane l takes blocks l, l + L, ... The products land in LDS; after the barrier
// thread t < R finishes row first + t, its loads issued before the product (one
// thread per row reads whole lines; a leader per row would read a quarter of each).
// Sums in T.
template <int L, class T>
__device__ __forceinline__ void RowProducts(FusedArgs const& a, float4 const* v, int2 extent, T (*h)[3])
{
    int const t = static_cast<int>(threadIdx.x), lane = t & (L - 1);
    T hx = 0, hy = 0, hz = 0;
    for (int k = extent.x + lane; k < extent.y; k += L)
    {
        int const j = a.col[k];
        float4 const A = a.va[k], B = a.vb[k];
        float const C = a.vc[k];
        float4 const P = v[j];
        T const px = P.x, py = P.y, pz = P.z;
        hx += A.x * px + A.y * py + A.z * pz;
        hy += A.w * px + B.x * py + B.y * pz;
        hz += B.z * px + B.w * py + C * pz;
    }
    hx = GroupSum<L>(hx), hy = GroupSum<L>(hy), hz = GroupSum<L>(hz);
    if (lane == 0)
        h[t / L][0] = hx, h[t / L][1] = hy, h[t / L][2] = hz;
}

// zc = (Z^T H Z)^-1 rc for aggregate g's kCoarseDofs rows, by the kCoarseWaves
// waves of the workgroup: wave w takes the 64-column chunks w, w + kCoarseWaves,
// ... of its mesh's n columns, loads rc and the rows' entries of kU of them at
// once, then accumulates in FP64 (kU chosen for the largest mesh; the order of
// the terms does not depend on it, and on n only); the waves' sums are added in
// order. Out-of-range lanes load column n - 1 and drop it, so that every load of
// a pass is in flight together.
constexpr int kCoarseWaves = 4;

template <int kU>
__device__ __forceinline__ void CoarseRows(FusedArgs const& a, int g)
{
    constexpr int kR = kCoarseDofs, kW = kCoarseWaves;
    __shared__ double part[kW][kR];
    int const t = static_cast<int>(threadIdx.x), wave = t >> 6, lane = t & 63;
    int4 const inf = a.coarseInfo[g];
    long long const off = a.coarseRowOffset[g];
    if (a.aggDone[g] != 0)
        return; // the mesh has converged (uniform over the workgroup)
    int const b0 = inf.x, n = inf.y;
    float const* A = a.coarseF + off;
    double s[kR];
#pragma unroll
    for (int i = 0; i < kR; ++i)
        s[i] = 0.;
    for (int c0 = wave; c0 * 64 < n; c0 += kW * kU)
    {
        double x[kU];
        float v[kR][kU];
#pragma unroll
        for (int u = 0; u < kU; ++u)
        {
            int const j = min((c0 + kW * u) * 64 + lane, n - 1);
            x[u] = a.rc[b0 + j];
#pragma unroll
            for (int i = 0; i < kR; ++i)
                v[i][u] = A[static_cast<size_t>(i) * n + j];
        }
#pragma unroll
        for (int u = 0; u < kU; ++u)
            if ((c0 + kW * u) * 64 + lane >= n)
                x[u] = 0.;
#pragma unroll
        for (int i = 0; i < kR; ++i)
#pragma unroll
            for (int u = 0; u < kU; ++u)
                s[i] += double(v[i][u]) * x[u];
    }
#pragma unroll
    for (int i = 0; i < kR; ++i)
        s[i] = WaveSum(s[i]);
    if (lane == 0)
#pragma unroll
        for (int i = 0; i < kR; ++i)
            part[wave][i] = s[i];
    __syncthreads();
    if (t < kR)
    {
        double tot = part[0][t];
        for (int w = 1; w < kW; ++w)
            tot += part[w][t];
        reinterpret_cast<float*>(a.zc)[8 * static_cast<size_t>(g) + (t < 3 ? t : t + 1)] = static_cast<float>(tot);
    }
}

// The coarse product (workgroups below coarseBlocks, one per aggregate) next to
// the polynomial's first product (half a chunk each): both read what CgUpdate1
// wrote and neither needs the other.
template <int L, int kU>
__global__ __launch_bounds__(256) void CoarsePoly(FusedArgs a)
{
    int w = static_cast<int>(blockIdx.x);
    if (w < a.coarseBlocks)
    {
        if (w < a.nAgg)
            CoarseRows<kU>(a, w);
        return;
    }
    w -= a.coarseBlocks;
    if (a.xcdChunk > 0)
        w = (w & 7) * a.xcdChunk + (w >> 3);
    if (w >= 2 * a.nChunks)
        return; // padding of the XCD order
    constexpr int R = 256 / L;
    __shared__ float h[R][3];
    int4 const ch = a.chunks[w >> 1];
    int const t = static_cast<int>(threadIdx.x), first = ch.x + (w & 1) * R, i = first + t;
    bool const mine = t < R && i < ch.y;
    int2 const extent = RowExtent<L>(a, first, ch.y); // in flight with the done flag
    if (a.cg.F[kDone * a.cg.nM + ch.z] != 0)
        return;
    Vec3d r{0., 0., 0.};
    float4 z1 = make_float4(0.f, 0.f, 0.f, 0.f), D0 = z1, D1 = z1;
    if (mine)
        r = a.r[i], z1 = a.z[i], D0 = a.dinv[2 * i], D1 = a.dinv[2 * i + 1];
    RowProducts<L>(a, a.z, extent, h);
    __syncthreads();
    if (!mine)
        return;
    // z2 = (1 + a2) z1 + b2 D^-1 (r - H z1)
    float4 const q = ApplyInverse(D0, D1, static_cast<float>(r.x) - h[t][0], static_cast<float>(r.y) - h[t][1],
                                  static_cast<float>(r.z) - h[t][2]);
    a.z2[i] = make_float4(z1.x + (a.q.a2 * z1.x + a.q.b2 * q.x), z1.y + (a.q.a2 * z1.y + a.q.b2 * q.y),
                          z1.z + (a.q.a2 * z1.z + a.q.b2 * q.z), 0.f);
}

enum class PolyMode : int
{
    kPolyLast,    // z = z3 + Z zc, r . z per chunk
    kPolyProduct, // w = H z, z . w per chunk
    kResidual     // r = b - H y0
};

// One workgroup of kChunkThreads per row chunk (XCD-aware order when xcdChunk > 0).
template <int L, PolyMode M>
__global__ __launch_bounds__(kChunkThreads) void BsrPoly(FusedArgs a)
{
    constexpr int R = kChunkThreads / L;
    using T = std::conditional_t<M == PolyMode::kPolyLast, float, double>;
    __shared__ T h[R][3];
    __shared__ double part[kChunkThreads / 64];
    int w = static_cast<int>(blockIdx.x);
    if (a.xcdChunk > 0)
        w = (w & 7) * a.xcdChunk + (w >> 3);
    if (w >= a.nChunks)
        return;
    int4 const ch = a.chunks[w];
    int const t = static_cast<int>(threadIdx.x), i = ch.x + t;
    bool const mine = t < R && i < ch.y;
    int2 const extent = RowExtent<L>(a, ch.x, ch.y); // in flight with the done flag
    if (M != PolyMode::kResidual && a.cg.F[kDone * a.cg.nM + ch.z] != 0)
        return; // the chunk's mesh has converged: its vectors no longer change
    float4 const zero = make_float4(0.f, 0.f, 0.f, 0.f);
    Vec3d r{0., 0., 0.};
    float4 z1 = zero, z2 = zero, D0 = zero, D1 = zero, d = zero, ct = zero, cr = zero;
    if (mine)
    {
        z1 = M == PolyMode::kResidual ? a.b[i] : a.z[i];
        if constexpr (M == PolyMode::kPolyLast)
        {
            int const g = a.aggOfRow[i];
            r = a.r[i], z2 = a.z2[i], D0 = a.dinv[2 * i], D1 = a.dinv[2 * i + 1];
            d = a.coarseD[i], ct = a.zc[2 * g], cr = a.zc[2 * g + 1];
        }
    }
    RowProducts<L>(a, M == PolyMode::kPolyLast ? a.z2 : M == PolyMode::kResidual ? a.y0 : a.z, extent, h);
    __syncthreads();
    double dot = 0.;
    if (mine)
    {
        if constexpr (M == PolyMode::kPolyLast)
        {
            float4 const q =
                ApplyInverse(D0, D1, static_cast<float>(r.x) - h[t][0], static_cast<float>(r.y) - h[t][1],
                             static_cast<float>(r.z) - h[t][2]);
            float4 const z = make_float4(
                z2.x + (a.q.a3 * (z2.x - z1.x) + a.q.b3 * q.x) + (ct.x + (cr.y * d.z - cr.z * d.y)),
                z2.y + (a.q.a3 * (z2.y - z1.y) + a.q.b3 * q.y) + (ct.y + (cr.z * d.x - cr.x * d.z)),
                z2.z + (a.q.a3 * (z2.z - z1.z) + a.q.b3 * q.z) + (ct.z + (cr.x * d.y - cr.y * d.x)), 0.f);
            a.z[i] = z; // nobody else reads z in this launch
            dot = r.x * z.x + r.y * z.y + r.z * z.z;
        }
        else if constexpr (M == PolyMode::kPolyProduct)
        {
            a.w[i] = Vec3d{h[t][0], h[t][1], h[t][2]};
            dot = z1.x * h[t][0] + z1.y * h[t][1] + z1.z * h[t][2];
        }
        else
            a.r[i] = Vec3d{z1.x - h[t][0], z1.y - h[t][1], z1.z - h[t][2]};
    }
    if constexpr (M == PolyMode::kResidual)
        return;
    // the chunk's rows in a fixed order: each wave's, then the waves in order
    double* const out = M == PolyMode::kPolyLast ? a.gammaPart : a.deltaPart;
    if constexpr (R <= 64)
    {
        if (t < 64)
        {
            dot = WaveSum(dot);
            if (t == 0)
                out[w] = dot;
        }
    }
    else
    {
        dot = WaveSum(dot);
        if ((t & 63) == 0)
            part[t >> 6] = dot;
        __syncthreads();
        if (t == 0)
        {
            for (int k = 1; k < kChunkThreads / 64; ++k)
                dot += part[k];
            out[w] = dot;
        }
    }
}

// z1 (two-level) or z = D^-1 r of one row, and its share of an aggregate's sums
// (r . r, r . z, sum r_i, sum d_i x r_i).
template <bool kTwoLevel>
__device__ __forceinline__ void RowResidual(float4* zOut, float invTheta, int i, Vec3d const& r, float4 const& D0,
                                            float4 const& D1, float4 const& d, double (&s)[8])
{
    float4 z = ApplyInverse(D0, D1, static_cast<float>(r.x), static_cast<float>(r.y), static_cast<float>(r.z));
    if constexpr (kTwoLevel)
        z.x *= invTheta, z.y *= invTheta, z.z *= invTheta;
    zOut[i] = z;
    s[0] += r.x * r.x + r.y * r.y + r.z * r.z;
    s[1] += r.x * z.x + r.y * z.y + r.z * z.z;
    if constexpr (kTwoLevel)
    {
        s[2] += r.x, s[3] += r.y, s[4] += r.z;
        s[5] += d.y * r.z - d.z * r.y, s[6] += d.z * r.x - d.x * r.z, s[7] += d.x * r.y - d.y * r.x;
    }
}

template <bool kTwoLevel>
__device__ __forceinline__ void StoreAggregate(double* rr, double* rz, double* rc, int g, double const (&s)[8])
{
    rr[g] = s[0];
    rz[g] = s[1];
    if constexpr (kTwoLevel)
        for (int c = 0; c < kCoarseDofs; ++c)
            rc[kCoarseDofs * g + c] = s[2 + c];
}

// Start of a solve, one workgroup of 128 per aggregate (r = b - H y0 formed before):
// y = y0, p = s = 0, z and the aggregate's sums, b . b among them.
template <bool kTwoLevel>
__global__ __launch_bounds__(128) void CgStartRows(FusedArgs a)
{
    __shared__ double lds[2][8], ldsB[2][1];
    int const g = static_cast<int>(blockIdx.x), t = static_cast<int>(threadIdx.x);
    int4 const inf = a.aggInfo[g];
    double s[8] = {0., 0., 0., 0., 0., 0., 0., 0.}, bb[1] = {0.};
    for (int i = inf.y + t; i < inf.z; i += 128)
    {
        float4 const b = a.b[i], y = a.y0[i];
        a.y[i] = Vec3d{y.x, y.y, y.z};
        a.p[i] = a.s[i] = Vec3d{0., 0., 0.};
        bb[0] += Dot3(b, b);
        RowResidual<kTwoLevel>(a.z, a.q.invTheta, i, a.r[i], a.dinv[2 * i], a.dinv[2 * i + 1],
                               kTwoLevel ? a.coarseD[i] : make_float4(0.f, 0.f, 0.f, 0.f), s);
    }
    Sum128<8>(s, lds);
    Sum128<1>(bb, ldsB);
    if (t == 0)
    {
        StoreAggregate<kTwoLevel>(a.rrPart[0], a.rzPart[0], a.rc, g, s);
        a.bbPart[g] = bb[0];
        a.aggDone[g] = 0;
    }
}

// End of a solve: y into the rows' FP32 vector and into the vertices' order.
__global__ __launch_bounds__(256) void CgSolution(Vec3d const* __restrict__ y, float4* __restrict__ rows,
                                                  float4* __restrict__ out, int const* __restrict__ rowVertex, int n)
{
    int const i = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x);
    if (i >= n)
        return;
    Vec3d const v = y[i];
    float4 const f = make_float4(static_cast<float>(v.x), static_cast<float>(v.y), static_cast<float>(v.z), 0.f);
    rows[i] = f;
    out[rowVertex[i]] = f;
}

// Start and end of a solve, one workgroup of 64 per mesh: b . b and r . r from the
// aggregates' sums of iteration parity `parity`. The start clears the recurrence's
// scalars; the end records the residual of a mesh that ran out of iterations.
__global__ __launch_bounds__(64) void CgMesh(FusedArgs a, int const* __restrict__ meshAggBegin, int start, int parity)
{
    int const m = static_cast<int>(blockIdx.x), nM = a.cg.nM, t = static_cast<int>(threadIdx.x);
    int const done = a.cg.F[kDone * nM + m];
    if (!start && done != 0)
        return;
    int const a0 = meshAggBegin[m], a1 = meshAggBegin[m + 1];
    double const rr = WaveSum(StridedSum<64>(a.rrPart[parity], a0, a1, t));
    double const bb = start ? WaveSum(StridedSum<64>(a.bbPart, a0, a1, t)) : a.cg.P[kBb * nM + m];
    if (t != 0)
        return;
    int const d = !(bb > 0.) || rr <= a.cg.tol2 * bb ? 1 : 0;
    if (start)
    {
        a.cg.P[kBb * nM + m] = bb;
        a.cg.P[kGamma * nM + m] = 0., a.cg.P[kAlpha * nM + m] = 1.;
        a.cg.F[kIters * nM + m] = 0;
    }
    a.cg.P[kRrLast * nM + m] = rr;
    a.cg.F[kDone * nM + m] = d;
    a.doneOut[m] = d;
}

// Head of an iteration, one workgroup of 128 threads per aggregate: the mesh's
// gamma, delta and r . r from the partial sums (in a fixed order, by every
// workgroup of the mesh), the stopping test |r| <= tol |b|, alpha and beta, then
// over the aggregate's rows p, s, y, r, z (z1) and the aggregate's sums. Scalars
// and r . r are kept per iteration parity (the old and new arrays of the
// arguments): a workgroup may run before another of its mesh has read the old
// ones. The mesh's first aggregate records them and the done flag; every workgroup
// comes to the same test and sets its aggregate's own flag.
// Bound by latency: the arguments, the descriptor, the sums with the scalars and
// rows, and the stores are one memory trip each. So the arguments are a struct of
// their own read at once, nothing but the descriptor and the flag decides whether
// to go on, and rows and sums are loaded branch-free (out-of-range threads read
// the last entry and drop it): guarded and looped loads waited for each other, 8.6
// us a launch on 32^3 against 6.3 (5.5 at 10,000 rows).
struct CgUpdateArgs
{
    int4 const* __restrict__ aggInfo;
    int4 const* __restrict__ aggRange;
    int* aggDone;
    double const* gammaOld; // per mesh
    double const* alphaOld;
    double const* bb;
    double const* gammaPart; // per chunk (two-level) or per aggregate
    double const* deltaPart;
    double const* rrOld;
    Vec3d const* __restrict__ w;
    float4* z;
    Vec3d* p;
    Vec3d* s;
    Vec3d* y;
    Vec3d* r;
    float4 const* __restrict__ dinv;
    float4 const* __restrict__ coarseD;
    double tol2;
    double* gammaNew;
    double* alphaNew;
    double* rrNew;
    double* rzNew;
    double* rc;
    double* rrLast; // per mesh
    int* done;
    int* iters;
    int* doneOut;
    float invTheta;
};

// Entries b + t, b + t + 128, ... of v, the first U loaded at once.
template <int U>
struct PartialSum
{
    double x[U];
    __device__ __forceinline__ void Load(double const* __restrict__ v, int b, int e, int t)
    {
#pragma unroll
        for (int u = 0; u < U; ++u)
            x[u] = v[min(b + t + 128 * u, e - 1)];
    }
    __device__ __forceinline__ double Sum(double const* __restrict__ v, int b, int e, int t) const
    {
        double s = 0.;
#pragma unroll
        for (int u = 0; u < U; ++u)
            s += b + t + 128 * u < e ? x[u] : 0.;
        if (e - b > 128 * U)
            s += StridedSum<128>(v, b + 128 * U, e, t);
        return s;
    }
};

template <bool kTwoLevel>
__global__ __launch_bounds__(128) void CgUpdate1(CgUpdateArgs a)
{
    __shared__ double lds3[2][3], lds8[2][8];
    int const g = static_cast<int>(blockIdx.x), t = static_cast<int>(threadIdx.x);
    int4 const inf = a.aggInfo[g], rg = a.aggRange[g];
    int const done = a.aggDone[g];
    // keep the descriptor's loads together with the flag's
    asm volatile("" ::"s"(inf.x), "s"(inf.y), "s"(rg.x), "s"(rg.z), "s"(done));
    if (done != 0)
        return;
    int const m = inf.x, i0 = min(inf.y + t, inf.z - 1);
    bool const mine = inf.y + t < inf.z;
    int const gb = kTwoLevel ? rg.x : rg.z, ge = kTwoLevel ? rg.y : rg.w;
    PartialSum<9> pg, pd;
    PartialSum<4> pr;
    pg.Load(a.gammaPart, gb, ge, t);
    pd.Load(a.deltaPart, rg.x, rg.y, t);
    pr.Load(a.rrOld, rg.z, rg.w, t);
    double const gammaOld = a.gammaOld[m], alphaOld = a.alphaOld[m], bb = a.bb[m];
    Vec3d const w0 = a.w[i0], p0 = a.p[i0], s0 = a.s[i0], y0 = a.y[i0], r0 = a.r[i0];
    float4 const z0 = a.z[i0], D0 = a.dinv[2 * i0], D1 = a.dinv[2 * i0 + 1];
    float4 d0 = make_float4(0.f, 0.f, 0.f, 0.f);
    if constexpr (kTwoLevel)
        d0 = a.coarseD[i0];
    double v[3] = {pg.Sum(a.gammaPart, gb, ge, t), pd.Sum(a.deltaPart, rg.x, rg.y, t),
                   pr.Sum(a.rrOld, rg.z, rg.w, t)};
    Sum128<3>(v, lds3);
    double const gamma = v[0], rr = v[2];
    // beta = gamma / gammaOld, alpha = gamma / (delta - beta gamma / alphaOld)
    double const beta = gammaOld != 0. ? gamma / gammaOld : 0.;
    double const den = v[1] - beta * gamma / alphaOld;
    double const alpha = den != 0. ? gamma / den : 0.;
    bool const stop = rr <= a.tol2 * bb;
    if (inf.w != 0 && t == 0)
    {
        a.rrLast[m] = rr;
        if (stop)
        {
            a.done[m] = 1;
            a.doneOut[m] = 1;
        }
        else
        {
            a.iters[m] += 1;
            a.gammaNew[m] = gamma;
            // alpha = 0 only after a breakdown (gamma = 0 or den = 0)
            a.alphaNew[m] = alpha != 0. ? alpha : 1.;
        }
    }
    if (stop)
    {
        if (t == 0)
            a.aggDone[g] = 1;
        return;
    }
    double sum[8] = {0., 0., 0., 0., 0., 0., 0., 0.};
    auto update = [&](int i, Vec3d const& w, float4 const& z, Vec3d p, Vec3d s, Vec3d y, Vec3d r, float4 const& E0,
                      float4 const& E1, float4 const& d) {
        p.x = z.x + beta * p.x, p.y = z.y + beta * p.y, p.z = z.z + beta * p.z;
        s.x = w.x + beta * s.x, s.y = w.y + beta * s.y, s.z = w.z + beta * s.z;
        y.x += alpha * p.x, y.y += alpha * p.y, y.z += alpha * p.z;
        r.x -= alpha * s.x, r.y -= alpha * s.y, r.z -= alpha * s.z;
        a.p[i] = p, a.s[i] = s, a.y[i] = y, a.r[i] = r;
        RowResidual<kTwoLevel>(a.z, a.invTheta, i, r, E0, E1, d, sum);
    };
    if (mine)
        update(i0, w0, z0, p0, s0, y0, r0, D0, D1, d0);
    for (int i = inf.y + t + 128; i < inf.z; i += 128)
        update(i, a.w[i], a.z[i], a.p[i], a.s[i], a.y[i], a.r[i], a.dinv[2 * i], a.dinv[2 * i + 1],
               kTwoLevel ? a.coarseD[i] : make_float4(0.f, 0.f, 0.f, 0.f));
    Sum128<8>(sum, lds8);
    if (t == 0)
        StoreAggregate<kTwoLevel>(a.rrNew, a.rzNew, a.rc, g, sum);
}

// ---- small meshes: a whole CG solve in one workgroup --------------------------
// CG preconditioned by symmetric coloured block Gauss-Seidel on meshes of at most
// kCgLocalRows updated vertices, one workgroup per mesh. As launches an iteration is
// 2 colours + 4 of them, 3 us each however few rows they have; here the passes are
// workgroup barriers apart, z lies in LDS, and the one-reduction recurrence of the
// fused solvers (FP64 vectors and products) takes its sums without a launch. The
// forward pass from z = 0 reads the blocks left of the diagonal only and the reverse
// pass, z_i -= D_i^-1 sum_(j > i) H_ij z_j, those right of it, whose FP64 sums it leaves
// for the product: an iteration reads one and a half matrices instead of three.
// One CU issues all of it: a pass takes 1 us for its chain of instructions alone, and
// 10 ns a row. Blocks and rows by place, loaded a pass ahead, took 57 us per iteration
// at 1,872 rows with 8 lanes a row (two rounds a colour) and 47 with 4; the blocks
// packed by halves 48; chunks of 16 rows padded to one length, 1 KB a load, 56.
constexpr int kCgLocalThreads = 1024, kCgLocalLanes = 4;

struct CgLocalArgs
{
    int4 const* __restrict__ rows; // first block, end of the lower ones, first upper one, end
    int const* __restrict__ place; // of each block's column in its mesh
    float4 const* __restrict__ va;
    float4 const* __restrict__ vb;
    float const* __restrict__ vc;
    LocalRange const* __restrict__ ranges; // per mesh nColors + 1
    int2 const* __restrict__ meshes;       // per mesh: (first entry of verts, vertices)
    int const* __restrict__ verts;         // row of each place
    float4 const* __restrict__ dinvRows;
    float4 const* __restrict__ b;
    float4* out; // y0, then the solution; like b and dinvRows by row, the rest by place
    float4* dinv;
    Vec3d* y;
    Vec3d* r;
    Vec3d* p;
    Vec3d* s;
    Vec3d* w;
    float4* z;
    CgState cg;
    int nColors, maxRows;
};

// Block extents of each place's row, and the places of its columns (ascending).
[[maybe_unused]] static __global__ __launch_bounds__(256) void CgLocalRowTable(
    int const* __restrict__ rowPtr, int const* __restrict__ col, int const* __restrict__ verts,
    int const* __restrict__ placeOf, int4* __restrict__ rows, int* __restrict__ place, int nRows, int nV)
{
    int const e = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x);
    int const i = e < nV ? verts[e] : nRows;
    if (i >= nRows) // fixed vertices have no row
        return;
    int const kb = rowPtr[i], ke = rowPtr[i + 1];
    int lower = kb, upper = kb;
    for (int k = kb; k < ke; ++k)
    {
        int const j = col[k];
        place[k] = placeOf[j];
        lower += j < i, upper += j <= i;
    }
    rows[e] = make_int4(kb, lower, upper, ke);
}

// Blocks [lo, hi) of one row times z by the row's kCgLocalLanes lanes: up to kSlots of
// a lane loaded ahead (Load), as many as the longest row of the wave takes (a load
// costs its cycles for every lane, used or not), then summed (Sum), longer rows in a
// loop. Slots past the end hold a block of the same row, summed with a zero vector:
// another mesh's block could be non-finite. first is the row's first block.
struct LocalRow
{
    static constexpr int kSlots = 4;
    float4 A[kSlots], B[kSlots];
    float C[kSlots];
    int j[kSlots];
    int lo, hi, slots;
    template <class V>
    __device__ __forceinline__ static V At(V const* p, unsigned int bytes)
    {
        return *reinterpret_cast<V const*>(reinterpret_cast<char const*>(p) + bytes);
    }
    __device__ __forceinline__ void Load(CgLocalArgs const& a, int first, int lo_, int hi_, int lane)
    {
        lo = lo_ + lane, hi = hi_;
        slots = 0;
#pragma unroll
        for (int u = 0; u < kSlots; ++u)
            if (__any(lo + u * kCgLocalLanes < hi))
            {
                slots = u + 1;
                int const k = max(min(lo + u * kCgLocalLanes, hi - 1), first);
                unsigned int const o = static_cast<unsigned int>(k) * 4u; // 32-bit offsets from scalar bases
                A[u] = At(a.va, o * 4u), B[u] = At(a.vb, o * 4u), C[u] = At(a.vc, o), j[u] = At(a.place, o);
            }
    }
    template <class T>
    __device__ __forceinline__ static void Add(T (&h)[3], float4 const& A, float4 const& B, float C, float4 const& z)
    {
        T const x = z.x, y = z.y, w = z.z;
        h[0] += A.x * x + A.y * y + A.z * w;
        h[1] += A.w * x + B.x * y + B.y * w;
        h[2] += B.z * x + B.w * y + C * w;
    }
    template <class T>
    __device__ __forceinline__ void Sum(CgLocalArgs const& a, float4 const* z, T (&h)[3]) const
    {
        h[0] = h[1] = h[2] = T(0);
#pragma unroll
        for (int u = 0; u < kSlots; ++u)
            if (u < slots)
            {
                float4 q = z[j[u]];
                bool const used = lo + u * kCgLocalLanes < hi;
                q = make_float4(used ? q.x : 0.f, used ? q.y : 0.f, used ? q.z : 0.f, 0.f);
                Add(h, A[u], B[u], C[u], q);
            }
        if (slots == kSlots)
            for (int k = lo + kSlots * kCgLocalLanes; k < hi; k += kCgLocalLanes)
                Add(h, a.va[k], a.vb[k], a.vc[k], z[a.place[k]]);
#pragma unroll
        for (int c = 0; c < 3; ++c)
            h[c] = GroupSum<kCgLocalLanes>(h[c]);
    }
};

// first: from y0 (out); else the iterations go on from the vectors and scalars that an
// earlier launch left. At most `iterations` of them, so a launch always ends soon.
[[maybe_unused]] static __global__ __launch_bounds__(kCgLocalThreads) void CgLocal(CgLocalArgs a, int first,
                                                                                  int iterations)
{
    constexpr int L = kCgLocalLanes, G = kCgLocalThreads / L;
    extern __shared__ float4 cgLds[];
    float4* const zL = cgLds;
    LocalRange* const ranges = reinterpret_cast<LocalRange*>(cgLds + a.maxRows);
    __shared__ double red[kCgLocalThreads / 64][3];
    int const m = static_cast<int>(blockIdx.x), nM = a.cg.nM, t = static_cast<int>(threadIdx.x);
    int const lane = t & (L - 1), g = t / L, nC = a.nColors;
    double* const P = a.cg.P + m;
    if (!first && a.cg.F[kDone * nM + m] != 0)
        return;
    int const base = a.meshes[m].x;
    int const* const verts = a.verts + base;
    a.rows += base, a.dinv += 2 * base, a.z += base;
    a.y += base, a.r += base, a.p += base, a.s += base, a.w += base;
    for (int c = t; c <= nC; c += kCgLocalThreads)
        ranges[c] = a.ranges[static_cast<size_t>(m) * (nC + 1) + c];
    __syncthreads();
    int const nR = ranges[nC].lbeg; // the fixed vertices follow
    if (nR == 0) // every vertex of the mesh is fixed: no row to read
    {
        if (t == 0)
            P[kBb * nM] = P[kRrLast * nM] = 0., a.cg.F[kDone * nM + m] = 1;
        return;
    }
    int const colour0 = ranges[0].count, lastColour = ranges[nC - 1].lbeg;
    auto sum3 = [&](double u, double v, double w, double (&out)[3]) {
        double const x[3] = {WaveSum(u), WaveSum(v), WaveSum(w)};
        if ((t & 63) == 0)
            red[t >> 6][0] = x[0], red[t >> 6][1] = x[1], red[t >> 6][2] = x[2];
        __syncthreads();
        out[0] = out[1] = out[2] = 0.;
#pragma unroll
        for (int k = 0; k < kCgLocalThreads / 64; ++k)
            out[0] += red[k][0], out[1] += red[k][1], out[2] += red[k][2];
    };
    // Passes of the preconditioner: forward over colours 1 .. nC - 1, reverse over
    // nC - 2 .. 0. A pass's first G rows are loaded during the pass before (their
    // extents one pass earlier), so that they arrive behind its reductions and barrier.
    int const nPasses = 2 * (nC - 1);
    auto colourOf = [&](int k) { return k < nC - 1 ? k + 1 : 2 * nC - 3 - k; };
    auto clamped = [&](LocalRange const& rg, int r) {
        return max(rg.lbeg + min(r, rg.count - 1), 0); // a colour without rows: its neighbour's, unused
    };
    int4 e;
    LocalRow q;
    float4 D0, D1;
    Vec3d rq;
    auto extents = [&](int k, int r) { e = a.rows[clamped(ranges[colourOf(k)], r)]; };
    auto blocks = [&](int k, int r) {
        int const i = clamped(ranges[colourOf(k)], r);
        bool const forward = k < nC - 1;
        q.Load(a, e.x, forward ? e.x : e.z, forward ? e.y : e.w, lane);
        D0 = a.dinv[2 * i], D1 = a.dinv[2 * i + 1];
    };
    // z = M^-1 r: the first colour's rows have z = D^-1 r already
    auto precondition = [&] {
        if (nPasses > 0)
        {
            extents(0, g);
            blocks(0, g);
            extents(min(1, nPasses - 1), g);
        }
        __syncthreads();
        for (int k = 0; k < nPasses; ++k)
        {
            LocalRange const rg = ranges[colourOf(k)];
            bool const forward = k < nC - 1;
            // whole waves leave the loop together: Load asks every lane
            for (int r0 = t / 64 * (64 / L); r0 < rg.count; r0 += G)
            {
                int const r = r0 + (t & 63) / L, i = clamped(rg, r);
                if (r >= G)
                {
                    extents(k, r);
                    blocks(k, r);
                }
                if (forward)
                    rq = a.r[i];
                bool const mine = lane == 0 && r < rg.count;
                if (forward)
                {
                    float h[3];
                    q.Sum(a, zL, h);
                    if (mine)
                        zL[i] = ApplyInverse(D0, D1, static_cast<float>(rq.x) - h[0],
                                             static_cast<float>(rq.y) - h[1], static_cast<float>(rq.z) - h[2]);
                }
                else
                {
                    // the columns right of the diagonal are final: their share of H z
                    double h[3];
                    q.Sum(a, zL, h);
                    if (mine)
                    {
                        float4 const d = ApplyInverse(D0, D1, static_cast<float>(h[0]), static_cast<float>(h[1]),
                                                      static_cast<float>(h[2])),
                                     z = zL[i];
                        zL[i] = make_float4(z.x - d.x, z.y - d.y, z.z - d.z, 0.f);
                        a.w[i] = Vec3d{h[0], h[1], h[2]};
                    }
                }
            }
            if (k + 1 < nPasses)
            {
                if (rg.count > G)
                    extents(k + 1, g);
                blocks(k + 1, g);
                extents(min(k + 2, nPasses - 1), g);
            }
            __syncthreads();
        }
    };
    // every row's product, body(place, r, sums): whole or without the blocks right of
    // the diagonal
    auto product = [&](bool whole, auto&& body) {
        int r = g;
        int4 x = a.rows[min(r, nR - 1)];
        for (int w0 = t / 64 * (64 / L); w0 < nR; w0 += G, r += G)
        {
            q.Load(a, x.x, x.x, whole ? x.w : x.z, lane);
            rq = a.r[min(r, nR - 1)];
            x = a.rows[min(r + G, nR - 1)];
            double h[3];
            q.Sum(a, zL, h);
            if (lane == 0 && r < nR)
                body(r, rq, h);
        }
    };
    // w = H z, gamma = r . z, delta = z . w, with the sum of rr
    double gamma = 0., delta = 0., rr = 0., sums[3];
    auto productAndSums = [&] {
        gamma = delta = 0.;
        product(false, [&](int i, Vec3d const& r, double const (&h)[3]) {
            float4 const z = zL[i];
            Vec3d w = i < lastColour ? a.w[i] : Vec3d{0., 0., 0.};
            w.x += h[0], w.y += h[1], w.z += h[2];
            a.w[i] = w;
            gamma += r.x * z.x + r.y * z.y + r.z * z.z;
            delta += z.x * w.x + z.y * w.y + z.z * w.z;
        });
        sum3(gamma, delta, rr, sums);
        gamma = sums[0], delta = sums[1], rr = sums[2];
    };
    auto startRow = [&](int i, Vec3d const& r, float4 const& E0, float4 const& E1) {
        if (i < colour0)
            zL[i] = ApplyInverse(E0, E1, static_cast<float>(r.x), static_cast<float>(r.y), static_cast<float>(r.z));
    };
    double gammaOld = 0., alphaOld = 1., bb;
    if (first)
    {
        for (int i = t; i < nR; i += kCgLocalThreads)
            zL[i] = a.out[verts[i]];
        __syncthreads();
        bb = 0.;
        product(true, [&](int i, Vec3d const&, double const (&h)[3]) {
            float4 const b = a.b[verts[i]];
            Vec3d const r{b.x - h[0], b.y - h[1], b.z - h[2]};
            a.r[i] = r;
            bb += Dot3(b, b);
            rr += r.x * r.x + r.y * r.y + r.z * r.z;
        });
        sum3(bb, rr, 0., sums);
        bb = sums[0], rr = sums[1];
        bool const done = !(bb > 0.) || rr <= a.cg.tol2 * bb;
        if (t == 0)
        {
            P[kBb * nM] = bb, P[kRrLast * nM] = rr;
            a.cg.F[kDone * nM + m] = done ? 1 : 0;
        }
        if (done)
            return;
        __syncthreads(); // every thread has its sums
        for (int i = t; i < nR; i += kCgLocalThreads)
        {
            int const row = verts[i];
            float4 const y = zL[i], E0 = a.dinvRows[2 * row], E1 = a.dinvRows[2 * row + 1];
            a.y[i] = Vec3d{y.x, y.y, y.z};
            a.p[i] = a.s[i] = Vec3d{0., 0., 0.};
            a.dinv[2 * i] = E0, a.dinv[2 * i + 1] = E1;
            startRow(i, a.r[i], E0, E1);
        }
        __syncthreads(); // dinv, before the passes load it ahead
        precondition();
        productAndSums();
    }
    else
    {
        bb = P[kBb * nM], gamma = P[kGamma * nM], gammaOld = P[kGamma1 * nM], delta = P[kAlpha1 * nM];
        alphaOld = P[kAlpha * nM];
        for (int i = t; i < nR; i += kCgLocalThreads)
            zL[i] = a.z[i];
    }
    int it = 0;
    bool done = false;
    while (it < iterations && !done)
    {
        double const beta = gammaOld != 0. ? gamma / gammaOld : 0.;
        double const den = delta - beta * gamma / alphaOld;
        double const alpha = den != 0. ? gamma / den : 0.;
        gammaOld = gamma;
        alphaOld = alpha != 0. ? alpha : 1.; // 0 only after a breakdown
        rr = 0.;
#pragma unroll 1
        for (int i = t; i < nR; i += kCgLocalThreads)
        {
            float4 const z = zL[i], E0 = a.dinv[2 * i], E1 = a.dinv[2 * i + 1];
            Vec3d const w = a.w[i];
            Vec3d p = a.p[i], s = a.s[i], y = a.y[i], r = a.r[i];
            p.x = z.x + beta * p.x, p.y = z.y + beta * p.y, p.z = z.z + beta * p.z;
            s.x = w.x + beta * s.x, s.y = w.y + beta * s.y, s.z = w.z + beta * s.z;
            y.x += alpha * p.x, y.y += alpha * p.y, y.z += alpha * p.z;
            r.x -= alpha * s.x, r.y -= alpha * s.y, r.z -= alpha * s.z;
            a.p[i] = p, a.s[i] = s, a.y[i] = y, a.r[i] = r;
            rr += r.x * r.x + r.y * r.y + r.z * r.z;
            startRow(i, r, E0, E1);
        }
        precondition();
        productAndSums();
        ++it;
        done = rr <= a.cg.tol2 * bb;
    }
    for (int i = t; i < nR; i += kCgLocalThreads)
    {
        Vec3d const y = a.y[i];
        a.out[verts[i]] =
            make_float4(static_cast<float>(y.x), static_cast<float>(y.y), static_cast<float>(y.z), 0.f);
        a.z[i] = zL[i];
    }
    if (t == 0)
    {
        P[kGamma * nM] = gamma, P[kGamma1 * nM] = gammaOld, P[kAlpha1 * nM] = delta, P[kAlpha * nM] = alphaOld;
        P[kRrLast * nM] = rr;
        a.cg.F[kDone * nM + m] = done ? 1 : 0;
        a.cg.F[kIters * nM + m] += it;
    }
}

// A solve's statistics without a host round trip: out = (largest per-mesh
// iteration count, largest per-mesh |r| / |b| at its last iteration).
__global__ __launch_bounds__(64) void SolveStats(CgState cg, double* __restrict__ out)
{
    int const nM = cg.nM, lane = static_cast<int>(threadIdx.x);
    int it = 0;
    double rel = 0.;
    for (int m = lane; m < nM; m += 64)
    {
        it = max(it, cg.F[kIters * nM + m]);
        double const bb = cg.P[kBb * nM + m];
        if (bb > 0.)
            rel = fmax(rel, sqrt(cg.P[kRrLast * nM + m] / bb));
    }
    for (int off = 32; off > 0; off >>= 1)
    {
        it = max(it, __shfl_xor(it, off));
        rel = fmax(rel, __shfl_xor(rel, off));
    }
    if (lane == 0)
    {
        out[0] = it;
        out[1] = rel;
    }
}

// A vector from the vertices' order into the solver's row order.
__global__ __launch_bounds__(256) void GatherRows(float4* __restrict__ out, float4 const* __restrict__ in,
                                                  int const* __restrict__ rowVertex, int n)
{
    int const s = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x);
    if (s < n)
        out[s] = in[rowVertex[s]];
}

// ---- initial guess of a backward solve from the previous solutions ----
// With s_1, ..., s_k the previous solves' solutions (newest first), the basis
// b_j = the j-th backward difference at s_1 (b_0 = s_1, b_1 = s_1 - s_2,
// b_2 = s_1 - 2 s_2 + s_3, ...: the same span, far better conditioned than the
// nearly parallel solutions themselves) and y0 = sum_j c_j b_j with, per mesh,
// (B^T H B) c = B^T b: the element of the span closest to the solution in the
// H-norm, which is the norm CG minimises. Polynomial extrapolation of the
// solutions is one element of that span.
constexpr int kProjMax = 8;
constexpr int kProjPairs = kProjMax * (kProjMax + 1) / 2;
constexpr int kProjTerms = kProjPairs + kProjMax; // b_p . H b_q (p <= q), b_p . b

struct ProjArgs
{
    float4 const* hist[kProjMax]; // previous solutions, newest first
    float4* basis[kProjMax];
    float4* hb[kProjMax];         // H b_j
    float4 const* __restrict__ rhs;
    float4* __restrict__ y;
    int const* __restrict__ aggPtr;
    int const* __restrict__ aggVerts;
    int const* __restrict__ meshAggBegin;
    int const* __restrict__ meshOf;
    double* __restrict__ part; // kProjTerms x nAgg, term-major
    double* __restrict__ coef; // kProjMax x nM
    int k, n, nM, nAgg;
};

// H b_j for the k basis vectors at once, 16 lanes per row: every block of the
// row is read once and applied to the k vectors (one pass over the Hessian
// instead of k); lane sums in block order, then the 16-lane butterfly.
__global__ __launch_bounds__(256) void ProjProducts(ProjArgs a, int const* __restrict__ rowPtr,
                                                    int const* __restrict__ col, float4 const* __restrict__ va,
                                                    float4 const* __restrict__ vb, float const* __restrict__ vc)
{
    constexpr int L = 16;
    int const tid = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x);
    int const row = tid / L, lane = tid & (L - 1);
    int kb = 0, ke = 0;
    if (row < a.n)
        kb = rowPtr[row], ke = rowPtr[row + 1];
    float hx[kProjMax], hy[kProjMax], hz[kProjMax];
#pragma unroll
    for (int v = 0; v < kProjMax; ++v)
        hx[v] = hy[v] = hz[v] = 0.f;
    for (int k = kb + lane; k < ke; k += L)
    {
        float4 const A = va[k], B = vb[k];
        float const C = vc[k];
        int const j = col[k];
#pragma unroll
        for (int v = 0; v < kProjMax; ++v)
        {
            if (v >= a.k)
                break;
            float4 const P = a.basis[v][j];
            hx[v] += A.x * P.x + A.y * P.y + A.z * P.z;
            hy[v] += A.w * P.x + B.x * P.y + B.y * P.z;
            hz[v] += B.z * P.x + B.w * P.y + C * P.z;
        }
    }
#pragma unroll
    for (int v = 0; v < kProjMax; ++v)
    {
        if (v >= a.k)
            break;
        float const x = GroupSum<L>(hx[v]), y = GroupSum<L>(hy[v]), z = GroupSum<L>(hz[v]);
        if (lane == 0 && row < a.n)
            a.hb[v][row] = make_float4(x, y, z, 0.f);
    }
}

__global__ __launch_bounds__(256) void ProjBasis(ProjArgs a)
{
    int const i = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x);
    if (i >= a.n)
        return;
    float4 s[kProjMax];
#pragma unroll
    for (int j = 0; j < kProjMax; ++j)
        s[j] = j < a.k ? a.hist[j][i] : make_float4(0.f, 0.f, 0.f, 0.f);
    a.basis[0][i] = s[0];
    // d holds the differences of the current order, b their first entry
#pragma unroll
    for (int o = 1; o < kProjMax; ++o)
    {
        if (o >= a.k)
            break;
#pragma unroll
        for (int j = 0; j + o < kProjMax; ++j)
            s[j] = make_float4(s[j].x - s[j + 1].x, s[j].y - s[j + 1].y, s[j].z - s[j + 1].z, 0.f);
        a.basis[o][i] = s[0];
    }
}

// One 128-thread workgroup per aggregate: its vertices' b_p . H b_q and
// b_p . b in FP64, summed in a fixed order.
__global__ __launch_bounds__(128) void ProjGram(ProjArgs a)
{
    __shared__ double lds[2][kProjTerms];
    int const g = static_cast<int>(blockIdx.x), t = static_cast<int>(threadIdx.x);
    double acc[kProjTerms];
#pragma unroll
    for (int u = 0; u < kProjTerms; ++u)
        acc[u] = 0.;
    for (int kk = a.aggPtr[g] + t; kk < a.aggPtr[g + 1]; kk += 128)
    {
        int const i = a.aggVerts[kk];
        float4 b[kProjMax], hb[kProjMax];
#pragma unroll
        for (int j = 0; j < kProjMax; ++j)
        {
            b[j] = j < a.k ? a.basis[j][i] : make_float4(0.f, 0.f, 0.f, 0.f);
            hb[j] = j < a.k ? a.hb[j][i] : make_float4(0.f, 0.f, 0.f, 0.f);
        }
        float4 const r = a.rhs[i];
        int u = 0;
#pragma unroll
        for (int p = 0; p < kProjMax; ++p)
#pragma unroll
            for (int q = p; q < kProjMax; ++q, ++u)
                if (q < a.k)
                    acc[u] += Dot3(b[p], hb[q]);
#pragma unroll
        for (int p = 0; p < kProjMax; ++p)
            if (p < a.k)
                acc[kProjPairs + p] += Dot3(b[p], r);
    }
    Sum128<kProjTerms>(acc, lds);
    if (t < kProjTerms)
    {
        double v = 0.;
#pragma unroll
        for (int u = 0; u < kProjTerms; ++u)
            v = u == t ? acc[u] : v;
        a.part[static_cast<size_t>(t) * a.nAgg + g] = v;
    }
}

// Sum of v[b .. e) over one wave in a fixed order; every lane gets it.
__device__ __forceinline__ double MeshSum(double const* __restrict__ v, int b, int e, int lane)
{
    double s = StridedSum<64>(v, b, e, lane);
    for (int off = 32; off > 0; off >>= 1)
        s += __shfl_xor(s, off);
    return s;
}

// One workgroup per mesh: the mesh's sums over its aggregates in a fixed order
// (each by one wave), then (B^T H B) c = B^T b scaled to a unit diagonal and
// solved by LDL^T, dropping a basis vector whose pivot falls below 1e-6
// (numerically in the span of the others) or whose diagonal is not positive.
__global__ __launch_bounds__(256) void ProjSolve(ProjArgs a)
{
    __shared__ double sums[kProjTerms];
    int const m = static_cast<int>(blockIdx.x);
    int const wave = static_cast<int>(threadIdx.x >> 6), lane = static_cast<int>(threadIdx.x & 63);
    int const a0 = a.meshAggBegin[m], a1 = a.meshAggBegin[m + 1];
    // term u (in use: both basis indices below k) summed by wave u mod 4
    {
        int u = 0;
#pragma unroll
        for (int p = 0; p < kProjMax; ++p)
#pragma unroll
            for (int q = p; q < kProjMax; ++q, ++u)
                if ((u & 3) == wave)
                {
                    double const v = q < a.k ? MeshSum(a.part + static_cast<size_t>(u) * a.nAgg, a0, a1, lane) : 0.;
                    if (lane == 0)
                        sums[u] = v;
                }
#pragma unroll
        for (int p = 0; p < kProjMax; ++p, ++u)
            if ((u & 3) == wave)
            {
                double const v = p < a.k ? MeshSum(a.part + static_cast<size_t>(u) * a.nAgg, a0, a1, lane) : 0.;
                if (lane == 0)
                    sums[u] = v;
            }
    }
    __syncthreads();
    if (threadIdx.x != 0)
        return;
    double sum[kProjTerms];
#pragma unroll
    for (int u = 0; u < kProjTerms; ++u)
        sum[u] = sums[u];

    int const k = a.k;
    double G[kProjMax][kProjMax], f[kProjMax], sc[kProjMax], L[kProjMax][kProjMax], d[kProjMax], c[kProjMax];
    bool use[kProjMax];
    {
        int u = 0;
        for (int p = 0; p < kProjMax; ++p)
            for (int q = p; q < kProjMax; ++q, ++u)
                G[p][q] = G[q][p] = sum[u];
        for (int p = 0; p < kProjMax; ++p)
            f[p] = sum[kProjPairs + p];
    }
    for (int p = 0; p < kProjMax; ++p)
    {
        use[p] = p < k && G[p][p] > 0.;
        sc[p] = use[p] ? 1. / sqrt(G[p][p]) : 0.;
    }
    for (int p = 0; p < kProjMax; ++p)
    {
        d[p] = 0.;
        for (int q = 0; q < kProjMax; ++q)
            L[p][q] = 0.;
    }
    for (int p = 0; p < kProjMax; ++p)
    {
        if (!use[p])
            continue;
        double dp = G[p][p] * sc[p] * sc[p];
        for (int q = 0; q < p; ++q)
            if (use[q])
                dp -= L[p][q] * L[p][q] * d[q];
        if (!(dp > 1e-6))
        {
            use[p] = false;
            continue;
        }
        d[p] = dp;
        for (int r = p + 1; r < kProjMax; ++r)
        {
            if (!use[r])
                continue;
            double v = G[r][p] * sc[r] * sc[p];
            for (int q = 0; q < p; ++q)
                if (use[q])
                    v -= L[r][q] * L[p][q] * d[q];
            L[r][p] = v / dp;
        }
    }
    // L D L^T c~ = f~ over the kept vectors
    for (int p = 0; p < kProjMax; ++p)
    {
        double v = use[p] ? f[p] * sc[p] : 0.;
        for (int q = 0; q < p; ++q)
            v -= L[p][q] * c[q];
        c[p] = use[p] ? v : 0.;
    }
    for (int p = 0; p < kProjMax; ++p)
        c[p] = use[p] ? c[p] / d[p] : 0.;
    for (int p = kProjMax - 1; p >= 0; --p)
    {
        double v = c[p];
        for (int q = p + 1; q < kProjMax; ++q)
            v -= L[q][p] * c[q];
        c[p] = use[p] ? v : 0.;
    }
    for (int p = 0; p < kProjMax; ++p)
        a.coef[static_cast<size_t>(m) * kProjMax + p] = c[p] * sc[p];
}

__global__ __launch_bounds__(256) void ProjCombine(ProjArgs a)
{
    int const i = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x);
    if (i >= a.n)
        return;
    double const* c = a.coef + static_cast<size_t>(a.meshOf[i]) * kProjMax;
    double x = 0., y = 0., z = 0.;
#pragma unroll
    for (int j = 0; j < kProjMax; ++j)
    {
        if (j >= a.k)
            break;
        float4 const b = a.basis[j][i];
        x += c[j] * b.x, y += c[j] * b.y, z += c[j] * b.z;
    }
    a.y[i] = make_float4(static_cast<float>(x), static_cast<float>(y), static_cast<float>(z), 0.f);
}

// In-place inversion of every mesh's symmetric positive definite block by block
// sweeps: with the pivot block P = A[K, K] of the rows and columns K = [k, k + b)
// (b = min(kPivot, n - k)), a step is
//   A[K, K] <- -P^-1,   A[i, K] <- A[i, K] P^-1,   A[K, j] <- P^-1 A[K, j],
//   A[i, j] <- A[i, j] - A[i, K] P^-1 A[K, j]     (i, j outside K),
// which keeps A symmetric, so only the 64 x 64 tiles (I, J), I >= J, are stored and
// updated; after ceil(n / kPivot) steps they hold -A^-1. A step is one launch
// (CoarseSweep): it reads the pivot's columns from a panel of their own and
// P^-1 from a buffer of its own, both left by the launch before it, which wrote
// them from the tiles it updated; the tile that holds the next pivot block comes
// first and inverts it while the others update. The panel and P^-1 alternate
// between two buffers, so a launch reads none of what it writes.
// Bound by latency: the tile's trip to memory and back (12 us a step on 752 rows)
// and, on the tile of the next pivot, the 32 elimination steps (8.6 us). The 2,058 x
// 2,058 block of a 32^3 mesh: 24.6 us a step (65 steps), 752 rows 20.5. As two
// launches over all tiles, the pivot block inverted entry-parallel in LDS, a step
// took 66 and 45 us.
constexpr int kPivot = 32;
// LDS row strides (doubles) for which the MFMA operand reads hit distinct banks
constexpr int kPivotStride = 48, kPanelStride = 80, kWStride = 34;

typedef double v4d __attribute__((ext_vector_type(4)));

struct CoarseSweepArgs
{
    double* A;
    double* panel[2]; // nM x kPivot x stride: panel[q][i] = A[i][k + q]
    double* inv[2];   // nM x kPivot x kPivot
    int stride;
    CoarseArgs c;
};

// 1 / x to FP64 accuracy without the range handling of a division (pivots of an
// SPD matrix).
__device__ __forceinline__ double Reciprocal(double x)
{
    double r = __builtin_amdgcn_rcp(x);
    r = fma(r, fma(-x, r, 1.), r);
    return fma(r, fma(-x, r, 1.), r);
}

// Inverse of the kPivot x kPivot SPD matrix S (LDS) into out, by a workgroup of 256
// (Gauss-Jordan, no pivoting): thread (wave w, half h, lane j < 32) keeps column j of
// rows 8 w + 4 h .. + 3 in registers. Per step the pivot row goes through LDS (one
// barrier, two buffers) and the rows' entries of the pivot column come from the
// wave's own lanes (8.6 us in all).
__device__ __forceinline__ void InvertPivot(double (*S)[kPivotStride], double* __restrict__ out)
{
    static_assert(kPivot == 32, "a half-wave per row");
    __shared__ double pivotRow[2][kPivot];
    int const t = static_cast<int>(threadIdx.x), w = t >> 6, half = (t >> 5) & 1, j = t & 31;
    int const i0 = 8 * w + 4 * half;
    double a[4];
#pragma unroll
    for (int u = 0; u < 4; ++u)
        a[u] = S[i0 + u][j];
#pragma unroll 1
    for (int q4 = 0; q4 < kPivot; q4 += 4)
#pragma unroll
        for (int v = 0; v < 4; ++v)
        {
            int const q = q4 + v;
            if (i0 == q4)
                pivotRow[v & 1][j] = a[v];
            double f[4]; // the rows' entries of column q
#pragma unroll
            for (int u = 0; u < 4; ++u)
            {
                double const lo = ReadLane(a[u], q), hi = ReadLane(a[u], 32 + q);
                f[u] = half ? hi : lo;
            }
            __syncthreads();
            double const inv = Reciprocal(pivotRow[v & 1][q]);
            bool const own = j == q;
            double const row = own ? inv : pivotRow[v & 1][j] * inv;
#pragma unroll
            for (int u = 0; u < 4; ++u)
                a[u] = i0 + u == q ? row : (own ? 0. : a[u]) - f[u] * row;
        }
#pragma unroll
    for (int u = 0; u < 4; ++u)
        out[(i0 + u) * kPivot + j] = a[u];
}

// What step k needs of the matrix before the first step: its panel and, by the
// first workgroup of each mesh, its pivot block's inverse (grid.x = 64-row tiles).
__global__ __launch_bounds__(256) void CoarseSweepFirst(CoarseSweepArgs a)
{
    __shared__ double S[kPivot][kPivotStride];
    int const m = static_cast<int>(blockIdx.y), t = static_cast<int>(threadIdx.x);
    int const n = kCoarseDofs * (a.c.meshAggBegin[m + 1] - a.c.meshAggBegin[m]);
    int const i0 = static_cast<int>(blockIdx.x) * 64;
    if (i0 >= n)
        return;
    int const b = min(kPivot, n);
    double const* A = a.A + a.c.meshOffset[m];
    double* V = a.panel[0] + static_cast<size_t>(m) * kPivot * a.stride;
    for (int e = t; e < 64 * kPivot; e += 256)
    {
        int const i = i0 + e / kPivot, q = e % kPivot;
        if (i < n)
            V[static_cast<size_t>(q) * a.stride + i] = q < b ? A[static_cast<size_t>(i) * n + q] : 0.;
    }
    if (i0 != 0)
        return;
    for (int e = t; e < kPivot * kPivot; e += 256)
    {
        int const r = e / kPivot, q = e % kPivot;
        S[r][q] = (r < b && q < b) ? A[static_cast<size_t>(r) * n + q] : r == q ? 1. : 0.;
    }
    __syncthreads();
    InvertPivot(S, a.inv[0] + static_cast<size_t>(m) * kPivot * kPivot);
}

// One step on the tiles (I, J), I >= J, numbered I (I + 1) / 2 + J over the tiles
// of the largest mesh (grid.y = mesh): W = A[I, K] P^-1 formed in LDS, then A[I, J] -=
// W A[K, J], both by FP64 MFMA (16 x 16 x 4; operands: lane l holds row or column l
// mod 16 and k = l / 16; results: column l mod 16 and rows l / 16 + 4 r). On the
// vector units the products waited on their LDS operands (4 times the reads).
__global__ __launch_bounds__(256) void CoarseSweep(CoarseSweepArgs a, int k, int parity)
{
    __shared__ double Vi[kPivot][kPanelStride], Vj[kPivot][kPanelStride], W[64][kWStride], P[kPivot][kPivotStride];
    int const m = static_cast<int>(blockIdx.y), t = static_cast<int>(threadIdx.x);
    int const n = kCoarseDofs * (a.c.meshAggBegin[m + 1] - a.c.meshAggBegin[m]);
    if (k >= n)
        return;
    int const kn = k + kPivot, tn = kn / 64; // the next pivot and its tile
    // the tile of the next pivot block trades places with the first
    int idx = static_cast<int>(blockIdx.x);
    int const diag = kn < n ? tn * (tn + 1) / 2 + tn : 0;
    idx = idx == 0 ? diag : idx == diag ? 0 : idx;
    int I = static_cast<int>((sqrtf(8.f * static_cast<float>(idx) + 1.f) - 1.f) * 0.5f);
    while (I * (I + 1) / 2 > idx)
        --I;
    while ((I + 1) * (I + 2) / 2 <= idx)
        ++I;
    int const J = idx - I * (I + 1) / 2, i0 = 64 * I, j0 = 64 * J;
    if (i0 >= n)
        return;
    int const b = min(kPivot, n - k), bn = kn < n ? min(kPivot, n - kn) : 0;
    double* const A = a.A + a.c.meshOffset[m];
    size_t const at = static_cast<size_t>(m) * kPivot * a.stride;
    double const* V = a.panel[parity] + at;
    double* const Vn = a.panel[parity ^ 1] + at;
    double const* inv = a.inv[parity] + static_cast<size_t>(m) * kPivot * kPivot;
    int const lane = t & 63, wave = t >> 6, l16 = lane & 15, l4 = lane >> 4;
    // the wave's 32 x 32 quadrant as 2 x 2 MFMA tiles; entry (x, y, r) of a thread:
    auto rowOf = [&](int x, int r) { return 32 * (wave >> 1) + 16 * x + l4 + 4 * r; };
    auto colOf = [&](int y) { return 32 * (wave & 1) + 16 * y + l16; };
    // in flight while the panels are staged
    v4d acc[2][2];
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                acc[x][y][r] = A[static_cast<size_t>(min(i0 + rowOf(x, r), n - 1)) * n + min(j0 + colOf(y), n - 1)];
#pragma unroll
    for (int u = 0; u < kPivot * 64 / 256; ++u)
    {
        int const e = t + 256 * u, q = e / 64, cc = e % 64;
        Vi[q][cc] = i0 + cc < n ? V[static_cast<size_t>(q) * a.stride + min(i0 + cc, n - 1)] : 0.;
        Vj[q][cc] = j0 + cc < n ? V[static_cast<size_t>(q) * a.stride + min(j0 + cc, n - 1)] : 0.;
    }
#pragma unroll
    for (int u = 0; u < kPivot * kPivot / 256; ++u)
    {
        int const e = t + 256 * u;
        P[e / kPivot][e % kPivot] = inv[e];
    }
    __syncthreads();
    // X^T P^-1 for rows 16 wave .. + 15 (columns 16 y + l16 of the result)
    auto form = [&](double (*X)[kPanelStride], v4d (&w)[2]) {
        w[0] = w[1] = v4d{0., 0., 0., 0.};
#pragma unroll
        for (int q = 0; q < kPivot; q += 4)
        {
            double const x = X[q + l4][16 * wave + l16];
            w[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(x, P[q + l4][l16], w[0], 0, 0, 0);
            w[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(x, P[q + l4][16 + l16], w[1], 0, 0, 0);
        }
    };
    v4d w[2];
    form(Vi, w);
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
        for (int r = 0; r < 4; ++r)
            W[16 * wave + l4 + 4 * r][16 * y + l16] = -w[y][r];
    __syncthreads();
    // rows in K take P^-1 A[K, j] = (A[j, K] P^-1)^T: formed in Vi's place
    bool const rowsInK = k >= i0 && k < i0 + 64, colsInK = k >= j0 && k < j0 + 64;
    if (rowsInK)
    {
        form(Vj, w);
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                Vi[16 * y + l16][16 * wave + l4 + 4 * r] = w[y][r];
        __syncthreads();
    }
#pragma unroll
    for (int q = 0; q < kPivot; q += 4)
    {
        double x[2], y[2];
#pragma unroll
        for (int u = 0; u < 2; ++u)
        {
            x[u] = W[32 * (wave >> 1) + 16 * u + l16][q + l4];
            y[u] = Vj[q + l4][32 * (wave & 1) + 16 * u + l16];
        }
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int v = 0; v < 2; ++v)
                acc[u][v] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[u], y[v], acc[u][v], 0, 0, 0);
    }
    // f(local row, local column, entry) over the thread's entries
    auto each = [&](auto&& f) {
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int y = 0; y < 2; ++y)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                {
                    double e = acc[x][y][r];
                    f(rowOf(x, r), colOf(y), e);
                    acc[x][y][r] = e;
                }
    };
    if (rowsInK || colsInK)
        each([&](int r, int c, double& e) {
            int const iq = i0 + r - k, jq = j0 + c - k;
            bool const iK = iq >= 0 && iq < b, jK = jq >= 0 && jq < b;
            if (iK && jK)
                e = -P[iq][jq];
            else if (iK)
                e = Vi[iq][c];
            else if (jK)
                e = -W[r][jq];
        });
    each([&](int r, int c, double& e) {
        if (i0 + r < n && j0 + c < n)
            A[static_cast<size_t>(i0 + r) * n + j0 + c] = e;
    });
    if (bn == 0 || (I != tn && J != tn))
        return;
    // the next panel: columns of tiles (I, tn), rows of tiles (tn, J) to its left
    int const kk = kn - 64 * tn;
    each([&](int r, int c, double& e) {
        int const q = (J == tn ? c : r) - kk, i = J == tn ? i0 + r : j0 + c;
        if (q >= 0 && q < bn && i < n && (J != tn || j0 + c < n))
            Vn[static_cast<size_t>(q) * a.stride + i] = e;
    });
    // rows of the panel past the matrix are zero
    if (bn < kPivot)
    {
        int const x0 = J == tn ? i0 : j0;
        for (int e = t; e < 64 * (kPivot - bn); e += 256)
            if (x0 + e % 64 < n)
                Vn[static_cast<size_t>(bn + e / 64) * a.stride + x0 + e % 64] = 0.;
    }
    if (I != J)
        return;
    // the next pivot block's inverse
    __syncthreads();
    each([&](int r, int c, double& e) {
        int const rq = r - kk, cq = c - kk;
        if (rq >= 0 && rq < kPivot && cq >= 0 && cq < kPivot)
            P[rq][cq] = (rq < bn && cq < bn) ? e : rq == cq ? 1. : 0.;
    });
    __syncthreads();
    InvertPivot(P, a.inv[parity ^ 1] + static_cast<size_t>(m) * kPivot * kPivot);
}

// Guard after inversion: a mesh block whose inverse has a non-positive or
// non-finite diagonal entry (an indefinite coarse operator) is zeroed, which
// leaves that mesh with the block-Jacobi preconditioner. One workgroup per mesh;
// A holds minus the inverse.
__global__ __launch_bounds__(256) void CoarseGuard(double* __restrict__ buf, CoarseArgs c)
{
    __shared__ int bad;
    int const m = static_cast<int>(blockIdx.x);
    int const n = kCoarseDofs * (c.meshAggBegin[m + 1] - c.meshAggBegin[m]);
    double* A = buf + c.meshOffset[m];
    if (threadIdx.x == 0)
        bad = 0;
    __syncthreads();
    for (int i = static_cast<int>(threadIdx.x); i < n; i += static_cast<int>(blockDim.x))
    {
        double const d = -A[static_cast<size_t>(i) * n + i];
        if (!(d > 0.) || !isfinite(d))
            bad = 1;
    }
    __syncthreads();
    if (!bad)
        return;
    for (int64_t k = threadIdx.x; k < static_cast<int64_t>(n) * n; k += blockDim.x)
        A[k] = 0.;
}

// The guarded inverse from its lower triangle, rounded to FP32 for the CG's coarse
// products (grid.y = mesh): it halves the bytes every iteration reads.
__global__ __launch_bounds__(256) void CoarseToFloat(double const* __restrict__ buf, CoarseArgs c,
                                                     float* __restrict__ out)
{
    int const m = static_cast<int>(blockIdx.y);
    int const n = kCoarseDofs * (c.meshAggBegin[m + 1] - c.meshAggBegin[m]);
    int64_t const idx = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (idx >= static_cast<int64_t>(n) * n)
        return;
    int64_t const i = idx / n, j = idx % n;
    double const* A = buf + c.meshOffset[m];
    out[c.meshOffset[m] + idx] = -static_cast<float>(i >= j ? A[i * n + j] : A[j * n + i]);
}

// Rotation offsets of the coarse space, one workgroup of 128 per aggregate g
// (rows aggRows[aggPtr[g] .. aggPtr[g + 1]), positions xs of their vertices):
// c the centroid, s the RMS radius, coarseD[row] = ((x - c) / s, 1), or 0 when
// the aggregate has no extent or its vertices are nearly collinear (the sum of
// the 2x2 principal minors of sum (x - c)(x - c)^T below 1e-3 of its trace
// squared). All sums in a fixed order.
__global__ __launch_bounds__(128) void CoarseBasis(int const* __restrict__ aggPtr, int const* __restrict__ aggRows,
                                                   int const* __restrict__ rowVertex,
                                                   float4 const* __restrict__ xs, float4* __restrict__ coarseD)
{
    __shared__ double lds3[2][3];
    __shared__ double lds6[2][6];
    int const g = static_cast<int>(blockIdx.x), t = static_cast<int>(threadIdx.x);
    int const kb = aggPtr[g], ke = aggPtr[g + 1];
    double c[3] = {0., 0., 0.};
    for (int k = kb + t; k < ke; k += 128)
    {
        float4 const x = xs[rowVertex[aggRows[k]]];
        c[0] += x.x, c[1] += x.y, c[2] += x.z;
    }
    Sum128<3>(c, lds3);
    double const n = static_cast<double>(ke - kb);
    for (double& v : c)
        v /= n;
    double S[6] = {0., 0., 0., 0., 0., 0.}; // xx, yy, zz, xy, xz, yz
    for (int k = kb + t; k < ke; k += 128)
    {
        float4 const x = xs[rowVertex[aggRows[k]]];
        double const dx = x.x - c[0], dy = x.y - c[1], dz = x.z - c[2];
        S[0] += dx * dx, S[1] += dy * dy, S[2] += dz * dz;
        S[3] += dx * dy, S[4] += dx * dz, S[5] += dy * dz;
    }
    Sum128<6>(S, lds6);
    double const tr = S[0] + S[1] + S[2];
    double const minors = S[0] * S[1] - S[3] * S[3] + S[0] * S[2] - S[4] * S[4] + S[1] * S[2] - S[5] * S[5];
    bool const use = tr > 0. && minors >= 1e-3 * tr * tr;
    double const inv = use ? 1. / sqrt(tr / n) : 0.;
    for (int k = kb + t; k < ke; k += 128)
    {
        int const row = aggRows[k];
        float4 const x = xs[rowVertex[row]];
        coarseD[row] = use ? make_float4(static_cast<float>((x.x - c[0]) * inv), static_cast<float>((x.y - c[1]) * inv),
                                         static_cast<float>((x.z - c[2]) * inv), 1.f)
                           : make_float4(0.f, 0.f, 0.f, 0.f);
    }
}

// Galerkin coarse operator Z^T H Z from the assembled blocks: coarse block k
// (aggregates cbA[k], cbB[k] of one mesh) is the sum over the fine blocks H_ij
// with i in cbA[k] and j in cbB[k] of Z_i^T H_ij Z_j, with D = [d]_x:
//   [ H        -H D_j      ]
//   [ D_i H    -D_i H D_j  ]
// One wave per coarse block: lane l takes the group's fine blocks l, l + 64, ...
// in ascending order, then a fixed butterfly; the wave writes the 6x6 entries
// into the mesh's dense row-major matrix (zeroed beforehand), so the operator
// is the same on every run. An aggregate without rotations (d = 0) gets an
// identity rotation diagonal, decoupled from everything else.
struct CoarseFromBsrArgs
{
    int const* __restrict__ cbA;
    int const* __restrict__ cbB;
    int const* __restrict__ cbSrcPtr;
    int const* __restrict__ cbSrc;
    int nCoarseBlocks;
    float4 const* __restrict__ va;
    float4 const* __restrict__ vb;
    float const* __restrict__ vc;
    int const* __restrict__ blockRow;
    int const* __restrict__ col;
    float4 const* __restrict__ coarseD;
    CoarseArgs c;
    double* __restrict__ Ac;
};

__device__ __forceinline__ void Skew(float4 const& d, double (&D)[3][3])
{
    D[0][0] = 0., D[0][1] = -d.z, D[0][2] = d.y;
    D[1][0] = d.z, D[1][1] = 0., D[1][2] = -d.x;
    D[2][0] = -d.y, D[2][1] = d.x, D[2][2] = 0.;
}

__global__ __launch_bounds__(256) void CoarseFromBsr(CoarseFromBsrArgs a)
{
    constexpr int kN = kCoarseDofs;
    int const wave = static_cast<int>(threadIdx.x >> 6), lane = static_cast<int>(threadIdx.x & 63);
    int const k = static_cast<int>(blockIdx.x) * 4 + wave;
    if (k >= a.nCoarseBlocks)
        return;
    double s[kN * kN];
#pragma unroll
    for (int e = 0; e < kN * kN; ++e)
        s[e] = 0.;
    int const q0 = a.cbSrcPtr[k], q1 = a.cbSrcPtr[k + 1];
    for (int q = q0 + lane; q < q1; q += 64)
    {
        int const f = a.cbSrc[q];
        float4 const A = a.va[f], B = a.vb[f];
        float const C = a.vc[f];
        float4 const di = a.coarseD[a.blockRow[f]], dj = a.coarseD[a.col[f]];
        double const H[3][3] = {{A.x, A.y, A.z}, {A.w, B.x, B.y}, {B.z, B.w, C}};
        double Di[3][3], Dj[3][3], HD[3][3], DH[3][3];
        Skew(di, Di);
        Skew(dj, Dj);
#pragma unroll
        for (int r = 0; r < 3; ++r)
#pragma unroll
            for (int cc = 0; cc < 3; ++cc)
            {
                HD[r][cc] = H[r][0] * Dj[0][cc] + H[r][1] * Dj[1][cc] + H[r][2] * Dj[2][cc];
                DH[r][cc] = Di[r][0] * H[0][cc] + Di[r][1] * H[1][cc] + Di[r][2] * H[2][cc];
            }
#pragma unroll
        for (int r = 0; r < 3; ++r)
#pragma unroll
            for (int cc = 0; cc < 3; ++cc)
            {
                s[r * kN + cc] += H[r][cc];
                s[r * kN + 3 + cc] -= HD[r][cc];
                s[(3 + r) * kN + cc] += DH[r][cc];
                s[(3 + r) * kN + 3 + cc] -= Di[r][0] * HD[0][cc] + Di[r][1] * HD[1][cc] + Di[r][2] * HD[2][cc];
            }
    }
#pragma unroll
    for (int e = 0; e < kN * kN; ++e)
        for (int off = 32; off > 0; off >>= 1)
            s[e] += __shfl_xor(s[e], off);
    if (lane != 0)
        return;
    int const ga = a.cbA[k], gb = a.cbB[k];
    if (ga == gb && a.coarseD[a.blockRow[a.cbSrc[q0]]].w == 0.f)
#pragma unroll
        for (int r = 3; r < kN; ++r)
#pragma unroll
            for (int cc = 3; cc < kN; ++cc)
                s[r * kN + cc] = r == cc ? 1. : 0.;
    int const m = a.c.aggMesh[ga];
    int const a0 = a.c.meshAggBegin[m];
    int const n = kN * (a.c.meshAggBegin[m + 1] - a0);
    double* const Am = a.Ac + a.c.meshOffset[m];
    int const ra = kN * (ga - a0), cb = kN * (gb - a0);
    for (int r = 0; r < kN; ++r)
        for (int cc = 0; cc < kN; ++cc)
            Am[static_cast<size_t>(ra + r) * n + cb + cc] = s[r * kN + cc];
}

} // namespace pbat_vbd::device
