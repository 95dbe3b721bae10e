// Device kernels of the MI355X VBD integrator (gfx950, wave64).
//
// Data layout in HBM (internal vertex numbering = colour-major, see
// vbd_integrator.hip):
//   xm[v]    float4 (x, y, z, m)      position and lumped mass
//   xtil[v]  float4 (x~, 0)           inertial target
//   xt[v]    float4 (x_t, 0)          positions at the start of the substep
//   vel[v], vprev[v], aext[v]  float4 velocities and external acceleration
//   star records (per updated vertex, in sweep order): its neighbours (8 B each)
//            and its incident tets (12 B each) with constants of their GP rows
//            and materials (see SweepArgs)
//   tgp[3e..3e+2]  float4 x3 (48 B) per tet: rows 1..3 of the shape function
//            gradients GP (row 0 = -(row1+row2+row3)), w*mu, w*lambda, alpha
//   tetv[e]  int4 vertex ids of tet e
//   (tgp and tetv serve the energy reduction and traces, not the sweep)
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "vbd_contact_kernels.hpp"

namespace pbat_vbd::device {

// ---- cross-lane sums over groups of L consecutive lanes (L | 64) ----------
template <int kCtrl>
__device__ __forceinline__ float DppRead(float x)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), kCtrl, 0xF, 0xF, false));
}

// Butterfly over L lanes: every lane of the group ends with the group sum.
//   quad_perm[1,0,3,2] (0xB1), quad_perm[2,3,0,1] (0x4E) -> quad sums,
//   row_half_mirror (0x141) pairs the two quads of 8 lanes,
//   row_mirror (0x140) pairs the two halves of a 16-lane row,
//   then ds_swizzle / bpermute for 32 and 64.
template <int L>
__device__ __forceinline__ float GroupSum(float x)
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

// 3x3 symmetric block and gradient of one vertex.
struct Block
{
    float h00, h01, h02, h11, h12, h22;
    float g0, g1, g2;
};

template <int L>
__device__ __forceinline__ void GroupSum(Block& B)
{
    B.h00 = GroupSum<L>(B.h00);
    B.h01 = GroupSum<L>(B.h01);
    B.h02 = GroupSum<L>(B.h02);
    B.h11 = GroupSum<L>(B.h11);
    B.h12 = GroupSum<L>(B.h12);
    B.h22 = GroupSum<L>(B.h22);
    B.g0 = GroupSum<L>(B.g0);
    B.g1 = GroupSum<L>(B.g1);
    B.g2 = GroupSum<L>(B.g2);
}

// Elastic contribution of one incident tet to vertex i's block (Stable
// Neo-Hookean, physics/StableNeoHookeanEnergy.h), with c = cof(F) g:
//   grad_i += w mu F g + w lambda (J - alpha) c
//   Hess_i += w mu |g|^2 I + w lambda c c^T
// (the d2J/dF2 term of the SNH Hessian contracts to zero for one vertex:
// det(F0 + x_i g^T) is affine in x_i). alpha = 1 + mu/lambda, so
// w lambda (J - alpha) = w lambda (J - 1) - w mu.
// With a, b, c the tet's other vertices, d_k = x_k - x, G the matrix of their
// shape-function gradient rows g_a, g_b, g_c, g = -(g_a + g_b + g_c) the own
// row and kappa = det G, F = D G with D = [d_a d_b d_c], so
//   F g = sum_k gamma_k d_k (gamma_k = g_k . g),   J = kappa (d_a . n),
//   c = cof(D) cof(G) g = -kappa n,   |g|^2 = -sum_k gamma_k,
// where n = (d_b - d_a) x (d_c - d_a) (the column sum of cof D) and G^-T g =
// -(1, 1, 1). The gamma terms are linear in the d_k, so over the whole star
// they fold into one constant per neighbour j,
//   Gamma_j = sum over the tets holding j of w mu gamma_k
// (summed in FP64 on the host), and a tet is left with A = w lambda kappa^2 and
// B = kappa (w lambda + w mu):
//   grad_i = sum_j Gamma_j d_j - sum_e (A (d_a . n) - B) n
//   Hess_i = -(sum_j Gamma_j) I + sum_e A n n^T.
__device__ __forceinline__ void AccumulateTet(float A, float Bk, float4 const& da, float4 const& db,
                                              float4 const& dc, Block& B)
{
    float const ex = db.x - da.x, ey = db.y - da.y, ez = db.z - da.z;
    float const fx = dc.x - da.x, fy = dc.y - da.y, fz = dc.z - da.z;
    float const nx = ey * fz - ez * fy, ny = ez * fx - ex * fz, nz = ex * fy - ey * fx;
    float const coef = A * (da.x * nx + da.y * ny + da.z * nz) - Bk;
    B.g0 -= coef * nx;
    B.g1 -= coef * ny;
    B.g2 -= coef * nz;
    float const anx = A * nx, any = A * ny, anz = A * nz;
    B.h00 += anx * nx;
    B.h11 += any * ny;
    B.h22 += anz * nz;
    B.h01 += anx * ny;
    B.h02 += anx * nz;
    B.h12 += any * nz;
}

struct StepConstants
{
    float dt;       // substep h
    float dt2;      // h^2
    float kD;       // Rayleigh damping coefficient
    float detHZero; // skip threshold on |det H|
    unsigned int* fp64Solves; // counts 3x3 solves taken by the FP64 path (nullable)
};

// Rayleigh damping of the elastic block (sim/vbd/Kernels.h:173-191).
__device__ __forceinline__ void Damp(Block& B, float4 const& xv, float4 const& xtv, StepConstants const& c)
{
    if (c.kD != 0.f)
    {
        float const D = c.kD / c.dt;
        float const ux = xv.x - xtv.x, uy = xv.y - xtv.y, uz = xv.z - xtv.z;
        B.g0 += D * (B.h00 * ux + B.h01 * uy + B.h02 * uz);
        B.g1 += D * (B.h01 * ux + B.h11 * uy + B.h12 * uz);
        B.g2 += D * (B.h02 * ux + B.h12 * uy + B.h22 * uz);
        float const s = 1.f + D;
        B.h00 *= s, B.h01 *= s, B.h02 *= s, B.h11 *= s, B.h12 *= s, B.h22 *= s;
    }
}

__device__ __forceinline__ float3 InertiaNewtonStep(Block B, float4 const& xv, float4 const& xl,
                                                    StepConstants const& c);

// Damping, inertia and the 3x3 Newton step of one vertex
// (sim/vbd/Kernels.h:173-191, 304-339). Returns the displacement to subtract.
__device__ __forceinline__ float3 NewtonStep(Block B, float4 const& xv, float4 const& xl, float4 const& xtv,
                                             StepConstants const& c)
{
    Damp(B, xv, xtv, c);
    return InertiaNewtonStep(B, xv, xl, c);
}

// Inertia and the 3x3 Newton step (sim/vbd/Kernels.h:304-339).
__device__ __forceinline__ float3 InertiaNewtonStep(Block B, float4 const& xv, float4 const& xl,
                                                    StepConstants const& c)
{
    float const K = xv.w / c.dt2;
    B.h00 += K, B.h11 += K, B.h22 += K;
    B.g0 += K * (xv.x - xl.x);
    B.g1 += K * (xv.y - xl.y);
    B.g2 += K * (xv.z - xl.z);
    // adjugate of the symmetric block
    float const a00 = B.h11 * B.h22 - B.h12 * B.h12;
    float const a01 = B.h02 * B.h12 - B.h01 * B.h22;
    float const a02 = B.h01 * B.h12 - B.h02 * B.h11;
    float const det = B.h00 * a00 + B.h01 * a01 + B.h02 * a02;
    if (!(fabsf(det) > c.detHZero))
        return make_float3(0.f, 0.f, 0.f);
    float const dscale = fabsf(B.h00 * B.h11 * B.h22);
    if (fabsf(det) < 1e-4f * dscale)
    {
        // ill-conditioned block: solve in FP64 from the FP32 entries
        if (c.fp64Solves)
            atomicAdd(c.fp64Solves, 1u);
        double const h00 = B.h00, h01 = B.h01, h02 = B.h02, h11 = B.h11, h12 = B.h12, h22 = B.h22;
        double const b00 = h11 * h22 - h12 * h12, b01 = h02 * h12 - h01 * h22, b02 = h01 * h12 - h02 * h11;
        double const b11 = h00 * h22 - h02 * h02, b12 = h01 * h02 - h00 * h12, b22 = h00 * h11 - h01 * h01;
        double const dd = h00 * b00 + h01 * b01 + h02 * b02;
        double const gx = B.g0, gy = B.g1, gz = B.g2;
        return make_float3(static_cast<float>((b00 * gx + b01 * gy + b02 * gz) / dd),
                           static_cast<float>((b01 * gx + b11 * gy + b12 * gz) / dd),
                           static_cast<float>((b02 * gx + b12 * gy + b22 * gz) / dd));
    }
    float const a11 = B.h00 * B.h22 - B.h02 * B.h02;
    float const a12 = B.h01 * B.h02 - B.h00 * B.h12;
    float const a22 = B.h00 * B.h11 - B.h01 * B.h01;
    float const inv = 1.f / det;
    return make_float3((a00 * B.g0 + a01 * B.g1 + a02 * B.g2) * inv, (a01 * B.g0 + a11 * B.g1 + a12 * B.g2) * inv,
                       (a02 * B.g0 + a12 * B.g1 + a22 * B.g2) * inv);
}

// Star records of the updated vertices, in sweep order, so a colour pass streams
// them. Row v holds the vertex's distinct neighbours and its incident tets
// (CSR rows through rowPtr = (first neighbour, first tet), or fixed-stride rows
// of nbrStride and incStride entries, padded with (v, 0) and zero tets):
//   nbr[k] int2      (neighbour j, Gamma_j as bits)
//   inc[k] StarInc   positions a | b << 8 | c << 16 of the tet's other vertices
//                    in the vertex's neighbour row, then A and B
// 12 B per tet and 8 B per neighbour (AccumulateTet).
struct StarInc
{
    unsigned int pk;
    float A, B;
};

// Neighbours a star row may hold: its positions are 8 bits wide.
constexpr int kMaxStarNeighbours = 256;

struct SweepArgs
{
    int2 const* __restrict__ rowPtr;
    int2 const* __restrict__ nbr;
    StarInc const* __restrict__ inc;
    float4* __restrict__ xm;
    float4 const* __restrict__ xtil;
    float4 const* __restrict__ xt;
    int vbeg;
    int vend;
    int xcdChunk;  // > 0: blocks per XCD for the XCD-aware block order
    int ntStream;  // != 0: read the star records with non-temporal loads
    int nbrStride; // > 0: fixed-stride rows
    int incStride;
    int ldsStride; // neighbour offsets a vertex keeps in LDS
    StepConstants c;
    ContactSweep contact; // contact sweeps only
    // meshes with a vertex of more than kMaxStarNeighbours neighbours
    // (VbdSweepWide): per tet the other vertices with A as bits, and
    // (w mu gamma_a, w mu gamma_b, w mu gamma_c, B)
    int4 const* __restrict__ wideIds;
    float4 const* __restrict__ wideGeo;
};

typedef int v2i __attribute__((ext_vector_type(2)));

// Loads of the star records and of the adjoint's incidence records, optionally
// with the non-temporal hint.
__device__ __forceinline__ int2 LoadNbr(int2 const* p, bool nt)
{
    if (nt)
    {
        v2i const r = __builtin_nontemporal_load(reinterpret_cast<v2i const*>(p));
        return make_int2(r.x, r.y);
    }
    return *p;
}

__device__ __forceinline__ StarInc LoadInc(StarInc const* p, bool nt)
{
    if (nt)
        return StarInc{__builtin_nontemporal_load(&p->pk), __builtin_nontemporal_load(&p->A),
                       __builtin_nontemporal_load(&p->B)};
    return *p;
}

// Inertia, Newton step and write of one vertex, with the contact block of a
// contact sweep (added after damping and before inertia); the group's first lane.
template <bool C>
__device__ __forceinline__ void FinishVertex(SweepArgs const& a, int v, Block& B, Block const& Cb, float4 const& own,
                                             float4 const& xl, float4 const& xto)
{
    if constexpr (C)
    {
        Damp(B, own, xto, a.c);
        B.h00 += Cb.h00, B.h01 += Cb.h01, B.h02 += Cb.h02, B.h11 += Cb.h11, B.h12 += Cb.h12, B.h22 += Cb.h22;
        B.g0 += Cb.g0, B.g1 += Cb.g1, B.g2 += Cb.g2;
        float3 const dx = InertiaNewtonStep(B, own, xl, a.c);
        a.contact.xb[v] = make_float4(own.x - dx.x, own.y - dx.y, own.z - dx.z, own.w);
    }
    else
    {
        // the start position only matters with damping: loaded here rather than
        // held in registers through the incidence loop
        float3 const dx = NewtonStep(B, own, xl, (a.c.kD != 0.f) ? a.xt[v] : own, a.c);
        a.xm[v] = make_float4(own.x - dx.x, own.y - dx.y, own.z - dx.z, own.w);
    }
}

// Position of vertex j as a sweep reads it.
template <bool C>
__device__ __forceinline__ float4 SweepPosition(SweepArgs const& a, int j)
{
    if constexpr (C)
        return ContactPosition(a.contact, a.xm, j);
    else
        return a.xm[j];
}

// The contact part of a contact sweep: the lane's contact records (slots lane,
// lane + L, ...), issued early, and the copy back of the previous colour's new
// positions.
template <int L>
struct ContactSlots
{
    static constexpr int kSlots = (kMaxContacts + L - 1) / L;
    int4 rec[kSlots];
    float4 xto;
    __device__ __forceinline__ void Load(SweepArgs const& a, int v, bool active, int lane, int tid, float4 const& own)
    {
        xto = own;
#pragma unroll
        for (int j = 0; j < kSlots; ++j)
        {
            int const k = lane + j * L;
            rec[j] = (active && k < kMaxContacts) ? a.contact.rec[static_cast<size_t>(v) * kMaxContacts + k]
                                                  : make_int4(-1, -1, -1, 0);
        }
        if (active)
            xto = a.xt[v];
        int const pend = a.contact.pendBeg + tid;
        if (pend < a.contact.pendEnd)
            a.xm[pend] = a.contact.xb[pend];
    }
    __device__ __forceinline__ void Accumulate(SweepArgs const& a, float4 const& own, Block& Cb) const
    {
        float3 const xo = make_float3(own.x, own.y, own.z), xt3 = make_float3(xto.x, xto.y, xto.z);
#pragma unroll
        for (int j = 0; j < kSlots; ++j)
            if (rec[j].x >= 0)
                AccumulateContact(xt3, xo, a.contact, a.xm, a.xt, rec[j], a.c.dt, __int_as_float(rec[j].w),
                                  a.contact.muF, a.contact.epsv, Cb);
    }
};

// One colour of one VBD sweep (sim/vbd/Integrator.cpp:73-136,
// gpu/impl/vbd/Kernels.cuh:148-233). L lanes of a wave cooperate on each vertex:
// lane l takes neighbours and tets l, l + L, ... of the vertex's rows, the loads
// of its first N neighbours and K tets issued together. A neighbour's position
// is gathered once per vertex; its offset d_j goes to LDS (the group's own slots,
// exchanged within the wave: no barrier), from which the tets read their three.
// The group reduces its 9 partial sums with DPP and its first lane applies the
// Newton update in place: vertices of one colour share no tet, so none reads
// what another vertex of the colour writes.
// What bounds it: on 256 meshes (107,000 vertices a colour, 373 MB of records,
// beyond the last-level cache) the stream of records, 4.1 TB/s of the 4.9 that the
// counters see with positions and targets; on 64^3 that
// stream (15 MB a launch) and the VALU next to a fixed ~3 us of launch ramp and
// dependent loads; on small meshes the latter alone. Per launch, best shape: 64^3
// 6.33 us, 80^3 8.5, 256 meshes 11.5. With 32 B and three 16-byte position gathers
// per tet (72 gathers a vertex instead of 14) the L1's gather rate and the record
// stream took 9.06, 16.2 and 22.0.
// With C (scenes in contact), the vertex's contact terms join its block after
// damping and before inertia (gpu/impl/vbd/Kernels.cuh:200-230), and the new
// positions go to contact.xb, so contact terms of the colour read positions from
// before its pass (the reference's write buffer, gpu/impl/vbd/Integrator.cu:303-326).
// The previous colour's positions are read from xb and copied back to xm by
// this launch; the last colour of an iteration is copied back by the host.
// Dynamic LDS: blockDim / L x ldsStride float4.
template <int L, int K, bool C = false>
__global__ __launch_bounds__(256) void VbdSweep(SweepArgs a)
{
    constexpr int N = (K + 1) / 2; // about 0.6 neighbours per tet
    extern __shared__ float4 starLds[];
    int block = static_cast<int>(blockIdx.x);
    if (a.xcdChunk > 0)
    {
        // Blocks are dealt to the 8 XCDs round-robin; give each XCD a
        // contiguous range of vertices so neighbouring vertices share its L2.
        // The host pads the grid to 8 * xcdChunk blocks, which makes this a
        // permutation of [0, gridDim.x).
        block = (block & 7) * a.xcdChunk + (block >> 3);
    }
    int const tid = block * static_cast<int>(blockDim.x) + static_cast<int>(threadIdx.x);
    int const lane = tid & (L - 1);
    int const v = a.vbeg + tid / L;
    bool const active = v < a.vend;
    float4* const d = starLds + (static_cast<int>(threadIdx.x) / L) * a.ldsStride;
    int nb = 0, ne = 0, kb = 0, ke = 0;
    float4 own = make_float4(0.f, 0.f, 0.f, 0.f);
    float4 xl = own;
    if (active)
    {
        if (a.incStride > 0)
        {
            // fixed stride: the rows' addresses need no prefix load
            nb = v * a.nbrStride, ne = nb + a.nbrStride;
            kb = v * a.incStride, ke = kb + a.incStride;
        }
        else
        {
            int2 const p0 = a.rowPtr[v], p1 = a.rowPtr[v + 1];
            nb = p0.x, ne = p1.x, kb = p0.y, ke = p1.y;
        }
        own = a.xm[v];
        if (lane == 0)
            xl = a.xtil[v]; // issued now, used after the reduction
    }
    bool const nt = a.ntStream != 0;
    ContactSlots<L> contact;
    if constexpr (C)
        contact.Load(a, v, active, lane, tid, own);
    int2 J[N];
#pragma unroll
    for (int j = 0; j < N; ++j)
    {
        int const k = nb + lane + j * L;
        J[j] = make_int2(-1, 0);
        if (k < ne)
            J[j] = LoadNbr(a.nbr + k, nt);
    }
    StarInc I[K];
#pragma unroll
    for (int j = 0; j < K; ++j)
    {
        int const k = kb + lane + j * L;
        if (k < ke)
            I[j] = LoadInc(a.inc + k, nt);
    }
    float4 p[N];
#pragma unroll
    for (int j = 0; j < N; ++j)
        if (J[j].x >= 0)
            p[j] = SweepPosition<C>(a, J[j].x);
    // contact terms: summed apart from the elastic block, which is damped alone;
    // here their dependent loads overlap the neighbours'
    Block Cb{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if constexpr (C)
        contact.Accumulate(a, own, Cb);
    Block B{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    float gsum = 0.f;
    auto neighbour = [&](int slot, float G, float4 const& pj) {
        float4 const dj = make_float4(pj.x - own.x, pj.y - own.y, pj.z - own.z, 0.f);
        B.g0 += G * dj.x, B.g1 += G * dj.y, B.g2 += G * dj.z;
        gsum += G;
        d[slot] = dj;
    };
#pragma unroll
    for (int j = 0; j < N; ++j)
        if (J[j].x >= 0)
            neighbour(lane + j * L, __int_as_float(J[j].y), p[j]);
    // neighbours beyond N per lane (vertices of unusually many neighbours)
    for (int k = nb + lane + N * L; k < ne; k += L)
    {
        int2 const q = LoadNbr(a.nbr + k, nt);
        neighbour(k - nb, __int_as_float(q.y), SweepPosition<C>(a, q.x));
    }
    B.h00 -= gsum, B.h11 -= gsum, B.h22 -= gsum;
    // the offsets are exchanged within the wave, whose LDS accesses stay in order
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int j = 0; j < K; ++j)
        if (kb + lane + j * L < ke)
            AccumulateTet(I[j].A, I[j].B, d[I[j].pk & 255u], d[(I[j].pk >> 8) & 255u], d[(I[j].pk >> 16) & 255u], B);
    // tets beyond K per lane
    for (int k = kb + lane + K * L; k < ke; k += L)
    {
        StarInc const q = LoadInc(a.inc + k, nt);
        AccumulateTet(q.A, q.B, d[q.pk & 255u], d[(q.pk >> 8) & 255u], d[(q.pk >> 16) & 255u], B);
    }
    GroupSum<L>(B);
    if constexpr (C)
        GroupSum<L>(Cb);
    if (!active || lane != 0)
        return;
    FinishVertex<C>(a, v, B, Cb, own, xl, contact.xto);
}

// The sweep of a mesh that has a vertex of more than kMaxStarNeighbours
// neighbours: one wave per vertex, every tet with its own three gathers and
// gradient constants (CSR rows).
template <bool C>
__global__ __launch_bounds__(256) void VbdSweepWide(SweepArgs a)
{
    constexpr int L = 64;
    int const tid = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x);
    int const lane = tid & (L - 1);
    int const v = a.vbeg + tid / L;
    bool const active = v < a.vend;
    int kb = 0, ke = 0;
    float4 own = make_float4(0.f, 0.f, 0.f, 0.f);
    float4 xl = own;
    if (active)
    {
        kb = a.rowPtr[v].y, ke = a.rowPtr[v + 1].y;
        own = a.xm[v];
        if (lane == 0)
            xl = a.xtil[v];
    }
    ContactSlots<L> contact;
    if constexpr (C)
        contact.Load(a, v, active, lane, tid, own);
    Block B{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int k = kb + lane; k < ke; k += L)
    {
        int4 const id = a.wideIds[k];
        float4 const geo = a.wideGeo[k];
        float4 const pa = SweepPosition<C>(a, id.x), pb = SweepPosition<C>(a, id.y), pc = SweepPosition<C>(a, id.z);
        float4 const da = make_float4(pa.x - own.x, pa.y - own.y, pa.z - own.z, 0.f);
        float4 const db = make_float4(pb.x - own.x, pb.y - own.y, pb.z - own.z, 0.f);
        float4 const dc = make_float4(pc.x - own.x, pc.y - own.y, pc.z - own.z, 0.f);
        B.g0 += geo.x * da.x + geo.y * db.x + geo.z * dc.x;
        B.g1 += geo.x * da.y + geo.y * db.y + geo.z * dc.y;
        B.g2 += geo.x * da.z + geo.y * db.z + geo.z * dc.z;
        float const dg = geo.x + geo.y + geo.z;
        B.h00 -= dg, B.h11 -= dg, B.h22 -= dg;
        AccumulateTet(__int_as_float(id.w), geo.w, da, db, dc, B);
    }
    GroupSum<L>(B);
    Block Cb{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if constexpr (C)
    {
        contact.Accumulate(a, own, Cb);
        GroupSum<L>(Cb);
    }
    if (!active || lane != 0)
        return;
    FinishVertex<C>(a, v, B, Cb, own, xl, contact.xto);
}

// Star records in fixed-stride rows from the CSR rows, one thread per
// (vertex, entry) of the longer row; unused entries are (v, 0) and zero tets.
[[maybe_unused]] static __global__ __launch_bounds__(256) void StarFixedStride(
    int2 const* __restrict__ rowPtr, int2 const* __restrict__ nbr, StarInc const* __restrict__ inc,
    int2* __restrict__ nbrE, StarInc* __restrict__ incE, int nRows, int nbrStride, int incStride)
{
    int const W = max(nbrStride, incStride);
    long long const t = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
    int const v = static_cast<int>(t / W), k = static_cast<int>(t % W);
    if (v >= nRows)
        return;
    int2 const p0 = rowPtr[v], p1 = rowPtr[v + 1];
    if (k < nbrStride)
        nbrE[static_cast<size_t>(v) * nbrStride + k] = p0.x + k < p1.x ? nbr[p0.x + k] : make_int2(v, 0);
    if (k < incStride)
        incE[static_cast<size_t>(v) * incStride + k] = p0.y + k < p1.y ? inc[p0.y + k] : StarInc{0u, 0.f, 0.f};
}

// Initial iterate of a substep (gpu/impl/vbd/Integrator.cu:190-248; sim/vbd/Kernels.h:24-94)
// from x_t, v, v_{t-1} (AdaptiveVbd) and the external acceleration.
__device__ __forceinline__ float3 InitialIterate(float4 const& p, float4 const& u, float4 const& w, float4 const& g,
                                                 float dt, float dt2, int strategy)
{
    if (strategy == 0) // Position
        return make_float3(p.x, p.y, p.z);
    if (strategy == 1) // Inertia
        return make_float3(p.x + dt * u.x, p.y + dt * u.y, p.z + dt * u.z);
    if (strategy == 2) // KineticEnergyMinimum
        return make_float3(p.x + dt * u.x + dt2 * g.x, p.y + dt * u.y + dt2 * g.y, p.z + dt * u.z + dt2 * g.z);
    float const an2 = g.x * g.x + g.y * g.y + g.z * g.z;
    float at = 0.f;
    if (an2 != 0.f)
    {
        if (strategy == 3) // AdaptiveVbd
        {
            float const dot = ((u.x - w.x) / dt) * g.x + ((u.y - w.y) / dt) * g.y + ((u.z - w.z) / dt) * g.z;
            at = fminf(fmaxf(dot / an2, 0.f), 1.f);
        }
        else // AdaptivePbat
        {
            float const vn = sqrtf(u.x * u.x + u.y * u.y + u.z * u.z) + 1.17549435e-38f;
            float const dot = (u.x / vn) * g.x + (u.y / vn) * g.y + (u.z / vn) * g.z;
            at = fminf(fabsf(dot / an2), 1.f);
        }
    }
    float const s = dt2 * at;
    return make_float3(p.x + dt * u.x + s * g.x, p.y + dt * u.y + s * g.y, p.z + dt * u.z + s * g.z);
}

__device__ __forceinline__ float4 InertialTarget(float4 const& p, float4 const& u, float4 const& g, float dt, float dt2)
{
    return make_float4(p.x + dt * u.x + dt2 * g.x, p.y + dt * u.y + dt2 * g.y, p.z + dt * u.z + dt2 * g.z, 0.f);
}

// Substep begin: inertial target x~ = xt + h v + h^2 a and the initial iterate.
[[maybe_unused]] static __global__ __launch_bounds__(256) void SubstepBegin(float4* __restrict__ xm, float4* __restrict__ xtil,
                                                    float4 const* __restrict__ xt, float4 const* __restrict__ vel,
                                                    float4 const* __restrict__ vprev, float4 const* __restrict__ aext,
                                                    int n, float dt, float dt2, int strategy)
{
    int const i = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x);
    if (i >= n)
        return;
    float4 const p = xt[i];
    float4 const u = vel[i];
    float4 const g = aext[i];
    xtil[i] = InertialTarget(p, u, g, dt, dt2);
    float3 const x0 = InitialIterate(p, u, strategy == 3 ? vprev[i] : u, g, dt, dt2, strategy);
    float const mass = xm[i].w;
    xm[i] = make_float4(x0.x, x0.y, x0.z, mass);
}

// Substep end (gpu/impl/vbd/Integrator.cu:329-347): vprev <- v, v = (x - xt)/h, xt <- x.
// Every vertex passes here once per substep, so this is where a non-finite
// position or velocity (a diverged solve, a NaN set by the caller) is flagged:
// *nonfinite = 1 (nullable; written only then).
[[maybe_unused]] static __global__ __launch_bounds__(256) void SubstepEnd(float4 const* __restrict__ xm, float4* __restrict__ xt,
                                                  float4* __restrict__ vel, float4* __restrict__ vprev, int n,
                                                  float dt, int* __restrict__ nonfinite)
{
    int const i = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x);
    if (i >= n)
        return;
    float4 const x = xm[i];
    float4 const p = xt[i];
    vprev[i] = vel[i];
    float4 const u = make_float4((x.x - p.x) / dt, (x.y - p.y) / dt, (x.z - p.z) / dt, 0.f);
    vel[i] = u;
    xt[i] = make_float4(x.x, x.y, x.z, 0.f);
    if (nonfinite && !(isfinite(x.x) && isfinite(x.y) && isfinite(x.z) && isfinite(u.x) && isfinite(u.y) &&
                       isfinite(u.z)))
        *nonfinite = 1;
}

// ---- vertex data between the host's order and the device's --------------------
// Vertices [first, first + count) of a packed host matrix (3 values per vertex, the
// host's order, in pinned memory that src / out maps) into or out of the device's order,
// 256 per workgroup, packed through LDS so that the link sees whole 16-byte accesses.
// As a host loop over the vertices with a pageable copy, get took 482 us at 64^3
// (274,625 vertices) and 58 at 32^3, now 182 and 31; set of a C-ordered matrix, the
// caller's transposition included, 1,430 and 184, now 328 and 61 (vertex-major: 826 and
// 107, now 150 and 37).
template <class T>
struct alignas(16) Quad16
{
    T v[16 / sizeof(T)];
};

[[maybe_unused]] static __global__ __launch_bounds__(256) void UploadVertices(
    float const* __restrict__ src, int const* __restrict__ iperm, float const* __restrict__ mass, int first, int count,
    float4* __restrict__ dst, float4* __restrict__ second)
{
    __shared__ Quad16<float> s[192];
    int const t = static_cast<int>(threadIdx.x), v0 = static_cast<int>(blockIdx.x) * 256;
    int const values = 3 * min(256, count - v0);
    float* const f = s[0].v;
    if (4 * t + 4 <= values)
        s[t] = reinterpret_cast<Quad16<float> const*>(src + 3 * static_cast<size_t>(v0))[t];
    else
        for (int k = 4 * t; k < min(values, 4 * t + 4); ++k)
            f[k] = src[3 * static_cast<size_t>(v0) + k];
    __syncthreads();
    if (3 * t >= values)
        return;
    int const o = first + v0 + t, v = iperm[o];
    float4 const x = make_float4(f[3 * t], f[3 * t + 1], f[3 * t + 2], 0.f);
    dst[v] = make_float4(x.x, x.y, x.z, mass ? mass[o] : 0.f);
    if (second)
        second[v] = x;
}

// S: float4 entries, or 3 packed T
template <class T, class S>
__global__ __launch_bounds__(256) void DownloadVertices(S const* __restrict__ src, int const* __restrict__ iperm,
                                                        int first, int count, T* __restrict__ out)
{
    constexpr int Q = 16 / sizeof(T);
    __shared__ Quad16<T> s[768 / Q];
    int const t = static_cast<int>(threadIdx.x), v0 = static_cast<int>(blockIdx.x) * 256;
    int const values = 3 * min(256, count - v0);
    T* const f = s[0].v;
    if (3 * t < values)
    {
        size_t const v = static_cast<size_t>(iperm[first + v0 + t]);
        if constexpr (sizeof(S) == sizeof(float4))
        {
            float4 const x = src[v];
            f[3 * t] = x.x, f[3 * t + 1] = x.y, f[3 * t + 2] = x.z;
        }
        else
            f[3 * t] = src[3 * v], f[3 * t + 1] = src[3 * v + 1], f[3 * t + 2] = src[3 * v + 2];
    }
    __syncthreads();
    T* const o = out + 3 * static_cast<size_t>(v0);
    for (int k = t; k * Q < values; k += 256)
        if ((k + 1) * Q <= values)
            reinterpret_cast<Quad16<T>*>(o)[k] = s[k];
        else
            for (int j = k * Q; j < values; ++j)
                o[j] = f[j];
}

[[maybe_unused]] static __global__ __launch_bounds__(256) void ToFloats(double const* __restrict__ src,
                                                                       float* __restrict__ out, int n)
{
    int const k = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x);
    if (k < n)
        out[k] = static_cast<float>(src[k]);
}

// ---- small meshes: a whole step in one launch --------------------------------
// Star records of a vertex in fixed-size rows whose entries name places in LDS (a
// mesh's positions, 16 bytes each) by their byte offset: kLocalNbr neighbours
// (offset, Gamma as bits) and kLocalInc tets (the other vertices' offsets a | b << 16
// and c, A, B); unused entries hold the vertex itself and zeros, so no entry needs a
// test.
struct LocalInc
{
    unsigned int ab, c;
    float A, B;
};
constexpr int kLocalNbr = 16, kLocalInc = 24;

// Vertices of one mesh and colour (the last entry of a mesh: its fixed vertices):
// internal range [vbeg, vbeg + count), places in the mesh from lbeg.
struct LocalRange
{
    int vbeg, count, lbeg;
};

struct LocalStepArgs
{
    int2 const* __restrict__ nbr;
    LocalInc const* __restrict__ inc;
    LocalRange const* __restrict__ ranges; // per mesh nColors + 1
    int2 const* __restrict__ meshes;       // per mesh: (first entry of verts, vertices)
    int const* __restrict__ verts;         // internal vertex of each place
    float4* xm;
    float4* xtil;
    float4* xt;
    float4* vel;
    float4* vprev;
    float4 const* __restrict__ aext;
    float4* xkm1; // Chebyshev: the previous two iterates (else null)
    float4* xkm2;
    float rho2;
    int nColors, iterations, substeps, strategy, maxVerts;
    StepConstants c;
    int* nonfinite;
};

// A mesh's largest colour up to which its vertices get 8 lanes each (the shortest
// chain), else 2 (the least work per vertex), and up to which meshes are stepped in one
// workgroup each. A workgroup of kLocalThreads has lanes for every vertex of a colour
// at once. Cubes, us per colour against a launch's 3.0: 7^3 (56 vertices a colour)
// 1.45, 8^3 (81) 2.5, 9^3 (113) 2.7, 10^3 (151) 3.1, 11^3 (198) 3.9. 4 lanes are not
// built; a trial took 2.0, 2.3, 2.7 and 3.3, at the same precision (velocities after four
// steps of 8^3, mean distance from FP64 over 12 meshes: 0.88e-4 of their norm with 2
// lanes, 0.91e-4 with 4, 0.90e-4 at 16 x 2, 0.82..0.99e-4 by mesh).
// Batches, us a step of 20 iterations here / as launches in their best shape: 512 of 5^3
// 195 / 591, 1,024 of 7^3 921 / 1,079, of 8^3 1,018 / 1,440, of 9^3 1,334 / 2,086.
constexpr int kLocalThreads = 512;
constexpr int kLocalFewVertices = kLocalThreads / 8;
constexpr int kLocalManyLanes = 2;
constexpr int kLocalMaxColour = 128;

// Most updated vertices of a mesh whose Gauss-Seidel-preconditioned solves run in one
// workgroup (CgLocal). us per iteration there / as launches: 18 rows 7.6 / 48, 100 14.5 /
// 55, 294 19 / 59, 648 24 / 61, 1,872 47 / 63, 2,730 66 / 65, 3,150 75 / 61. Batches, us a
// solve: 512 meshes of 180 rows 1,178 / 3,728, of 648 rows 3,272 / 9,545, of 1,210 rows
// 6,620 / 19,344; 256 of 2,028 rows 6,558 / 14,414.
constexpr int kCgLocalRows = 2400;

// omega of the Chebyshev update after iteration k (sim/vbd/Kernels.h:97-102 in FP32
// as gpu/impl/vbd/ChebyshevIntegrator.cu:28-33 evaluates it, operator precedence
// included: for k >= 2, 4/4 - rho2 * omega).
__host__ __device__ inline float ChebyshevOmega(int k, float rho2, float omega)
{
    return (k == 0) ? 1.f : (k == 1) ? 2.f / (2.f - rho2) : 4.f / 4.f - rho2 * omega;
}

// The iterations of one substep on one mesh by a workgroup, positions and inertial
// targets in LDS, L lanes per vertex: the arithmetic of VbdSweep<L, .> in its order.
// Every thread works on one vertex of a colour (threads past its end on the last
// one, without writing). Its records are loaded into registers a colour ahead, as
// soon as the current ones are used, so the loads pass behind the reduction, the
// Newton step and the barrier; a pass is LDS reads, arithmetic and a barrier.
template <int L>
__device__ __forceinline__ void LocalIterations(LocalStepArgs const& a, float4* pos, float4 const* til,
                                                LocalRange const* ranges, int2 mesh)
{
    constexpr int NK = kLocalNbr / L, NT = kLocalInc / L;
    int const t = static_cast<int>(threadIdx.x), lane = t & (L - 1), r = t / L, nC = a.nColors;
    int2 J[NK];
    LocalInc I[NT];
    auto load = [&](int v) {
        int2 const* const n = a.nbr + v * kLocalNbr + lane;
        LocalInc const* const e = a.inc + v * kLocalInc + lane;
#pragma unroll
        for (int j = 0; j < NK; ++j)
            J[j] = n[j * L];
#pragma unroll
        for (int j = 0; j < NT; ++j)
            I[j] = e[j * L];
    };
    auto at = [&](unsigned int offset) {
        return *reinterpret_cast<float4 const*>(reinterpret_cast<char const*>(pos) + offset);
    };
    LocalRange rg = ranges[0];
    int last = max(rg.count - 1, 0);
    load(rg.vbeg + min(r, last));
    float omega = 0.f;
    for (int k = 0; k < a.iterations; ++k)
    {
        for (int c = 0; c < nC; ++c)
        {
            int const mine = min(r, last), v = rg.vbeg + mine, place = rg.lbeg + mine;
            bool const write = lane == 0 && r < rg.count;
            float4 const own = pos[place], xl = til[place];
            rg = ranges[c + 1 == nC ? 0 : c + 1];
            last = max(rg.count - 1, 0);
            auto offset = [&](unsigned int j) {
                float4 const q = at(j);
                return make_float4(q.x - own.x, q.y - own.y, q.z - own.z, 0.f);
            };
            Block B{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            float gsum = 0.f;
#pragma unroll
            for (int j = 0; j < NK; ++j)
            {
                float const G = __int_as_float(J[j].y);
                float4 const dj = offset(static_cast<unsigned int>(J[j].x));
                B.g0 += G * dj.x, B.g1 += G * dj.y, B.g2 += G * dj.z;
                gsum += G;
            }
            B.h00 -= gsum, B.h11 -= gsum, B.h22 -= gsum;
#pragma unroll
            for (int j = 0; j < NT; ++j)
                AccumulateTet(I[j].A, I[j].B, offset(I[j].ab & 65535u), offset(I[j].ab >> 16), offset(I[j].c), B);
            load(rg.vbeg + min(r, last));
            GroupSum<L>(B);
            if (write)
            {
                float3 const dx = NewtonStep(B, own, xl, (a.c.kD != 0.f) ? a.xt[v] : own, a.c);
                pos[place] = make_float4(own.x - dx.x, own.y - dx.y, own.z - dx.z, own.w);
            }
            __syncthreads();
        }
        if (a.xkm1)
        {
            // Chebyshev (ChebyshevUpdate); the arrays follow the internal order
            omega = ChebyshevOmega(k, a.rho2, omega);
            for (int i = t; i < mesh.y; i += static_cast<int>(blockDim.x))
            {
                int const v = a.verts[mesh.x + i];
                float4 x = pos[i];
                if (k > 1)
                {
                    float4 const b = a.xkm2[v];
                    x.x = omega * (x.x - b.x) + b.x;
                    x.y = omega * (x.y - b.y) + b.y;
                    x.z = omega * (x.z - b.z) + b.z;
                    pos[i] = x;
                }
                a.xkm2[v] = a.xkm1[v];
                a.xkm1[v] = x;
            }
            __syncthreads();
        }
    }
}

// A whole step of one small mesh per workgroup: the substeps' begin, every colour of
// every iteration with a workgroup barrier between them, and the end. A launch per
// colour takes 3 us however few vertices it has; a pass here, bound by the chain of
// LDS reads, reduction, Newton step and barrier, takes 0.9 us on 5 vertices a colour
// and 1.45 us on 56 (20 iterations: 3^3 280 -> 113 us, 7^3 452 -> 232; 48 meshes of
// 2^3..6^3 465 -> 186). With the records loaded at the pass instead of a colour ahead a
// pass took 2.0 us, with CSR rows, whose tail needs a loop, 1.3..1.5. Dynamic LDS: 2
// maxVerts float4, then the mesh's ranges.
[[maybe_unused]] static __global__ __launch_bounds__(kLocalThreads) void VbdStepLocal(LocalStepArgs a)
{
    extern __shared__ float4 localLds[];
    float4* const pos = localLds;
    float4* const til = localLds + a.maxVerts;
    LocalRange* const ranges = reinterpret_cast<LocalRange*>(localLds + 2 * a.maxVerts);
    int const m = static_cast<int>(blockIdx.x), t = static_cast<int>(threadIdx.x), nt = static_cast<int>(blockDim.x);
    int2 const mesh = a.meshes[m];
    for (int c = t; c <= a.nColors; c += nt)
        ranges[c] = a.ranges[static_cast<size_t>(m) * (a.nColors + 1) + c];
    __syncthreads();
    int largest = 0;
    for (int c = 0; c < a.nColors; ++c)
        largest = max(largest, ranges[c].count);
    float const dt = a.c.dt, dt2 = a.c.dt2;
    bool bad = false;
    for (int s = 0; s < a.substeps; ++s)
    {
        for (int i = t; i < mesh.y; i += nt)
        {
            int const v = a.verts[mesh.x + i];
            float4 const p = a.xt[v], u = a.vel[v], g = a.aext[v];
            float4 const l = InertialTarget(p, u, g, dt, dt2);
            float3 const x0 = InitialIterate(p, u, a.strategy == 3 ? a.vprev[v] : u, g, dt, dt2, a.strategy);
            a.xtil[v] = til[i] = l;
            pos[i] = make_float4(x0.x, x0.y, x0.z, a.xm[v].w);
        }
        __syncthreads();
        if (largest == 0) // every vertex of the mesh is fixed
            ;
        else if (largest <= kLocalFewVertices)
            LocalIterations<8>(a, pos, til, ranges, mesh);
        else
            LocalIterations<kLocalManyLanes>(a, pos, til, ranges, mesh);
        for (int i = t; i < mesh.y; i += nt)
        {
            int const v = a.verts[mesh.x + i];
            float4 const x = pos[i], p = a.xt[v];
            a.vprev[v] = a.vel[v];
            float4 const u = make_float4((x.x - p.x) / dt, (x.y - p.y) / dt, (x.z - p.z) / dt, 0.f);
            a.vel[v] = u;
            a.xt[v] = make_float4(x.x, x.y, x.z, 0.f);
            a.xm[v] = x;
            bad = bad || !(isfinite(x.x) && isfinite(x.y) && isfinite(x.z) && isfinite(u.x) && isfinite(u.y) &&
                           isfinite(u.z));
        }
        __syncthreads(); // the next substep's threads read xt of other vertices
    }
    if (bad && a.nonfinite)
        *a.nonfinite = 1;
}

// Star constants of changed moduli in every layout of the rows: a tet entry's A = w
// lambda kappa^2 and B = kappa (w lambda + w mu), a neighbour's Gamma_j = sum of w mu
// gamma_k over the row's tets holding it, in FP64 and in row order as the host builds
// them. shape[k] = (gamma_a, gamma_b, gamma_c, kappa) and tet[k] the tet of CSR entry k;
// tgp holds (., w mu, w lambda, .) in its third float4 per tet. In wide rows (wideGeo
// given) the tets carry their own gradient constants instead.
// kMaterialLanes lanes per row: each stages its tets' w mu gamma_k in LDS (read by the
// lanes of its own wave: no barrier) and sums those of its neighbours. Bound by three
// dependent loads and the walk over the row. Setting the moduli, us: 4^3 cells 20, 64^3
// 1,190; 5,000 random points (rows of up to 69 tets) 69, 60,000 413. With a thread per
// entry that walked the whole row in global memory, and the copies filled by launches of
// their own, 32, 1,880, 116 and 720.
constexpr int kMaterialLanes = 32;

struct StarMaterialArgs
{
    int2 const* __restrict__ rowPtr;
    int2* __restrict__ nbr;
    StarInc* __restrict__ inc;
    float4 const* __restrict__ shape;
    int const* __restrict__ tet;
    float4 const* __restrict__ tgp;
    int4* __restrict__ wideIds;
    float4* __restrict__ wideGeo;
    int2* __restrict__ nbrE; // copies, null where there are none
    StarInc* __restrict__ incE;
    int2* __restrict__ nbrL;
    LocalInc* __restrict__ incL;
    int nRows, nbrStride, incStride;
};

[[maybe_unused]] static __global__ __launch_bounds__(256) void StarMaterial(StarMaterialArgs a)
{
    constexpr int L = kMaterialLanes, R = 256 / L, U = 8;
    __shared__ double wS[R][L][3];
    __shared__ unsigned int pkS[R][L];
    int const lane = static_cast<int>(threadIdx.x) & (L - 1), g = static_cast<int>(threadIdx.x) / L;
    auto exchange = [] {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    for (long long v = static_cast<long long>(blockIdx.x) * R + g; v < a.nRows;
         v += static_cast<long long>(gridDim.x) * R)
    {
        int2 const p0 = a.rowPtr[v], p1 = a.rowPtr[v + 1];
        int const nI = p1.y - p0.y, nN = a.wideGeo ? 0 : p1.x - p0.x;
        for (int n0 = 0; n0 == 0 || n0 < nN; n0 += L)
        {
            int const k = n0 + lane;
            unsigned int const me = static_cast<unsigned int>(k);
            double G = 0.;
            for (int e0 = 0; e0 < nI; e0 += L)
            {
                int const j = e0 + lane, e = p0.y + j;
                if (j < nI)
                {
                    float4 const m = a.tgp[3 * static_cast<size_t>(a.tet[e]) + 2], s = a.shape[e];
                    double const wmu = m.y, wlam = m.z, kappa = s.w;
                    if (n0 == 0)
                    {
                        float const A = static_cast<float>(wlam * kappa * kappa);
                        float const B = static_cast<float>(kappa * (wlam + wmu));
                        if (a.wideGeo)
                        {
                            a.wideIds[e].w = __float_as_int(A);
                            a.wideGeo[e] = make_float4(static_cast<float>(wmu * s.x), static_cast<float>(wmu * s.y),
                                                       static_cast<float>(wmu * s.z), B);
                        }
                        else
                            a.inc[e].A = A, a.inc[e].B = B;
                        if (a.incE)
                            a.incE[v * a.incStride + j].A = A, a.incE[v * a.incStride + j].B = B;
                        if (a.incL)
                            a.incL[v * kLocalInc + j].A = A, a.incL[v * kLocalInc + j].B = B;
                    }
                    pkS[g][lane] = a.inc[e].pk;
                    wS[g][lane][0] = wmu * s.x, wS[g][lane][1] = wmu * s.y, wS[g][lane][2] = wmu * s.z;
                }
                else
                    pkS[g][lane] = 0u, wS[g][lane][0] = wS[g][lane][1] = wS[g][lane][2] = 0.;
                exchange();
                // whole batches of staged tets, branch-free; those past the row add zeros
                for (int q0 = 0; q0 < min(L, nI - e0) && nN > 0; q0 += U)
                {
                    double w[U];
#pragma unroll
                    for (int u = 0; u < U; ++u)
                    {
                        unsigned int const pk = pkS[g][q0 + u];
                        double const* const x = wS[g][q0 + u];
                        w[u] = (pk & 255u) == me ? x[0] : 0.;
                        w[u] += ((pk >> 8) & 255u) == me ? x[1] : 0.;
                        w[u] += ((pk >> 16) & 255u) == me ? x[2] : 0.;
                    }
#pragma unroll
                    for (int u = 0; u < U; ++u)
                        G += w[u];
                }
                exchange();
            }
            if (k < nN)
            {
                int const bits = __float_as_int(static_cast<float>(G));
                a.nbr[p0.x + k].y = bits;
                if (a.nbrE)
                    a.nbrE[v * a.nbrStride + k].y = bits;
                if (a.nbrL)
                    a.nbrL[v * kLocalNbr + k].y = bits;
            }
        }
    }
}

// Local records of the current star records, one thread per (vertex, entry);
// place[v] is vertex v's place in its mesh.
[[maybe_unused]] static __global__ __launch_bounds__(256) void LocalRecords(
    int2 const* __restrict__ rowPtr, int2 const* __restrict__ nbr, StarInc const* __restrict__ inc,
    int const* __restrict__ place, int2* __restrict__ nbrL, LocalInc* __restrict__ incL, int nRows)
{
    static_assert(kLocalNbr <= kLocalInc, "one thread per tet entry");
    int const t = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x);
    int const v = t / kLocalInc, k = t % kLocalInc;
    if (v >= nRows)
        return;
    int2 const p0 = rowPtr[v], p1 = rowPtr[v + 1];
    unsigned int const own = 16u * static_cast<unsigned int>(place[v]);
    if (k < kLocalNbr)
    {
        bool const used = p0.x + k < p1.x;
        int2 const q = used ? nbr[p0.x + k] : make_int2(v, 0);
        nbrL[v * kLocalNbr + k] = make_int2(16 * place[q.x], q.y);
    }
    LocalInc out{own | own << 16, own, 0.f, 0.f};
    if (p0.y + k < p1.y)
    {
        StarInc const q = inc[p0.y + k];
        auto at = [&](unsigned int j) {
            return 16u * static_cast<unsigned int>(place[nbr[p0.x + static_cast<int>(j)].x]);
        };
        out = LocalInc{at(q.pk & 255u) | at((q.pk >> 8) & 255u) << 16, at((q.pk >> 16) & 255u), q.A, q.B};
    }
    incL[v * kLocalInc + k] = out;
}

// Chebyshev semi-iterative update after iteration k (sim/vbd/Kernels.h:104-118,
// gpu/impl/vbd/ChebyshevIntegrator.cu:38-59): x = omega (x - x_{k-2}) + x_{k-2}
// for k > 1, then x_{k-2} = x_{k-1}, x_{k-1} = x.
[[maybe_unused]] static __global__ __launch_bounds__(256) void ChebyshevUpdate(float4* __restrict__ xm,
                                                                               float4* __restrict__ xkm1,
                                                                               float4* __restrict__ xkm2, int n,
                                                                               int k, float omega)
{
    int const i = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x);
    if (i >= n)
        return;
    float4 x = xm[i];
    if (k > 1)
    {
        float4 const a = xkm2[i];
        x.x = omega * (x.x - a.x) + a.x;
        x.y = omega * (x.y - a.y) + a.y;
        x.z = omega * (x.z - a.z) + a.z;
        xm[i] = x;
    }
    xkm2[i] = xkm1[i];
    xkm1[i] = x;
}

// ---- Anderson acceleration (gpu/impl/vbd/AndersonIntegrator.cu:36-105) ------
// After VBD iteration k >= 1 of a substep, with G = x, F = G - x_{k-1} and the
// window of the last min(k, m) differences DG, DF (column (k-1) mod m is the
// newest): alpha = argmin |DF alpha - F| and x = G - DG alpha. The least
// squares is solved from the FP64 Gram matrix DF^T DF and DF^T F; only the
// newest column's row of the Gram matrix is recomputed each iteration.

constexpr int kMaxAndersonWindow = 16;
constexpr int kAndersonSpread = 16; // atomic targets per accumulated value
constexpr int kAndersonStride = 16; // doubles between targets (128 B)

// Accumulated values of one iteration: 2 kMaxAndersonWindow values
// (DF_j . DF_new, then DF_j . F), each over kAndersonSpread targets.
__host__ __device__ constexpr int AndersonAccDoubles()
{
    return 2 * kMaxAndersonWindow * kAndersonSpread * kAndersonStride;
}

// Before iteration 0 of a substep: x_{k-1} = x; clear both accumulator sets.
[[maybe_unused]] static __global__ __launch_bounds__(256) void AndersonStart(float4 const* __restrict__ xm,
                                                                             float4* __restrict__ xkm1, int n,
                                                                             double* __restrict__ acc)
{
    int const i = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x);
    if (i < n)
        xkm1[i] = xm[i];
    if (blockIdx.x == 0)
        for (int j = static_cast<int>(threadIdx.x); j < 2 * AndersonAccDoubles(); j += static_cast<int>(blockDim.x))
            acc[j] = 0.;
}

// After iteration 0: G_{k-1} = x, F_{k-1} = x - x_{k-1}, then x_{k-1} = x.
[[maybe_unused]] static __global__ __launch_bounds__(256) void AndersonFirst(float4 const* __restrict__ xm,
                                                                             float4* __restrict__ xkm1,
                                                                             float4* __restrict__ gkm1,
                                                                             float4* __restrict__ fkm1, int n)
{
    int const i = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x);
    if (i >= n)
        return;
    float4 const g = xm[i], p = xkm1[i];
    gkm1[i] = make_float4(g.x, g.y, g.z, 0.f);
    fkm1[i] = make_float4(g.x - p.x, g.y - p.y, g.z - p.z, 0.f);
    xkm1[i] = make_float4(g.x, g.y, g.z, 0.f);
}

__device__ __forceinline__ double Dot3d(float4 const& u, float4 const& w)
{
    return double(u.x) * w.x + double(u.y) * w.y + double(u.z) * w.z;
}

// After iteration k >= 1: update the window (column col) and accumulate
// DF_j . DF_col and DF_j . F for j < mk into acc. blockDim = 256.
template <int M>
__global__ __launch_bounds__(256) void AndersonWindow(float4 const* __restrict__ xm, float4 const* __restrict__ xkm1,
                                                      float4* __restrict__ gkm1, float4* __restrict__ fkm1,
                                                      float4* __restrict__ dgk, float4* __restrict__ dfk, int n,
                                                      int col, int mk, double* __restrict__ acc)
{
    __shared__ double red[4][2 * M];
    int const i = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x);
    double vals[2 * M];
#pragma unroll
    for (int j = 0; j < 2 * M; ++j)
        vals[j] = 0.;
    if (i < n)
    {
        float4 const g = xm[i], p = xkm1[i], g1 = gkm1[i], f1 = fkm1[i];
        float4 const f = make_float4(g.x - p.x, g.y - p.y, g.z - p.z, 0.f);
        float4 const dg = make_float4(g.x - g1.x, g.y - g1.y, g.z - g1.z, 0.f);
        float4 const df = make_float4(f.x - f1.x, f.y - f1.y, f.z - f1.z, 0.f);
        dgk[static_cast<size_t>(col) * n + i] = dg;
        dfk[static_cast<size_t>(col) * n + i] = df;
        gkm1[i] = make_float4(g.x, g.y, g.z, 0.f);
        fkm1[i] = f;
#pragma unroll
        for (int j = 0; j < M; ++j)
            if (j < mk)
            {
                float4 const dj = (j == col) ? df : dfk[static_cast<size_t>(j) * n + i];
                vals[j] = Dot3d(dj, df);
                vals[M + j] = Dot3d(dj, f);
            }
    }
    int const lane = static_cast<int>(threadIdx.x & 63), wave = static_cast<int>(threadIdx.x >> 6);
#pragma unroll
    for (int j = 0; j < 2 * M; ++j)
    {
        if ((j < M ? j : j - M) >= mk)
            continue; // a window column not filled yet (uniform over the launch)
        double v = vals[j];
        for (int off = 32; off > 0; off >>= 1)
            v += __shfl_xor(v, off);
        if (lane == 0)
            red[wave][j] = v;
    }
    __syncthreads();
    int const nw = static_cast<int>((blockDim.x + 63) / 64);
    int const t = static_cast<int>(threadIdx.x);
    if (t < 2 * M && ((t < M) ? t : t - M) < mk)
    {
        double sum = 0.;
        for (int w = 0; w < nw; ++w)
            sum += red[w][t];
        int const slot = static_cast<int>(blockIdx.x) & (kAndersonSpread - 1);
        int const idx = (t < M) ? t : kMaxAndersonWindow + (t - M);
        atomicAdd(acc + (static_cast<size_t>(idx) * kAndersonSpread + slot) * kAndersonStride, sum);
    }
}

// After AndersonWindow: every workgroup forms the mk x mk Gram matrix (the
// previous one, gramOld, with row and column col replaced) and solves for
// alpha by an FP64 Cholesky factorisation that drops columns whose pivot is
// below 1e-13 of the largest diagonal (a zero or dependent difference); the
// first workgroup stores the Gram matrix (gramNew) and clears accNext. Then
// x = G - DG alpha and x_{k-1} = x.
[[maybe_unused]] static __global__ __launch_bounds__(256) void AndersonApply(float4* __restrict__ xm, float4* __restrict__ xkm1,
                                                     float4 const* __restrict__ gkm1,
                                                     float4 const* __restrict__ dgk, int n, int m, int col, int mk,
                                                     double const* __restrict__ acc, double* __restrict__ accNext,
                                                     double const* __restrict__ gramOld, double* __restrict__ gramNew)
{
    constexpr int W = kMaxAndersonWindow;
    __shared__ double sG[W * W], sL[W * W];
    __shared__ double sb[W], sy[W], sa[W];
    __shared__ int sKeep[W];
    __shared__ float sAlpha[W];
    int const t = static_cast<int>(threadIdx.x);
    auto sum = [&](int idx) {
        double s = 0.;
        for (int k = 0; k < kAndersonSpread; ++k)
            s += acc[(static_cast<size_t>(idx) * kAndersonSpread + k) * kAndersonStride];
        return s;
    };
    if (t < mk * mk)
    {
        int const r = t / mk, c = t % mk;
        double g;
        if (r == col)
            g = sum(c);
        else if (c == col)
            g = sum(r);
        else
            g = gramOld[r * m + c];
        sG[r * W + c] = g;
        if (blockIdx.x == 0)
            gramNew[r * m + c] = g;
    }
    if (t < mk)
        sb[t] = sum(kMaxAndersonWindow + t);
    __syncthreads();
    if (t == 0)
    {
        // Cholesky factor L (column j of L in sL[. * W + j]) with dropped columns
        double dmax = 0.;
        for (int j = 0; j < mk; ++j)
            dmax = fmax(dmax, sG[j * W + j]);
        for (int j = 0; j < mk; ++j)
        {
            double d = sG[j * W + j];
            for (int p = 0; p < j; ++p)
                d -= sL[j * W + p] * sL[j * W + p];
            int const keep = (d > 1e-13 * dmax && d > 0.) ? 1 : 0;
            sKeep[j] = keep;
            double const ljj = keep ? sqrt(d) : 0.;
            sL[j * W + j] = ljj;
            for (int r = j + 1; r < mk; ++r)
            {
                double v = sG[r * W + j];
                for (int p = 0; p < j; ++p)
                    v -= sL[r * W + p] * sL[j * W + p];
                sL[r * W + j] = keep ? v / ljj : 0.;
            }
        }
        for (int j = 0; j < mk; ++j)
        {
            double v = sb[j];
            for (int p = 0; p < j; ++p)
                v -= sL[j * W + p] * sy[p];
            sy[j] = sKeep[j] ? v / sL[j * W + j] : 0.;
        }
        for (int j = mk - 1; j >= 0; --j)
        {
            double v = sy[j];
            for (int p = j + 1; p < mk; ++p)
                v -= sL[p * W + j] * sa[p];
            sa[j] = sKeep[j] ? v / sL[j * W + j] : 0.;
        }
        for (int j = 0; j < mk; ++j)
            sAlpha[j] = static_cast<float>(sa[j]);
    }
    if (blockIdx.x == 0)
        for (int j = t; j < AndersonAccDoubles(); j += static_cast<int>(blockDim.x))
            accNext[j] = 0.;
    __syncthreads();
    int const i = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x);
    if (i >= n)
        return;
    float4 const g = gkm1[i];
    float x0 = g.x, x1 = g.y, x2 = g.z;
    for (int j = 0; j < mk; ++j)
    {
        float4 const d = dgk[static_cast<size_t>(j) * n + i];
        float const aj = sAlpha[j];
        x0 -= aj * d.x, x1 -= aj * d.y, x2 -= aj * d.z;
    }
    float const mass = xm[i].w;
    xm[i] = make_float4(x0, x1, x2, mass);
    xkm1[i] = make_float4(x0, x1, x2, 0.f);
}

// w Psi(F) of tet e in FP64: Stable Neo-Hookean (physics/StableNeoHookeanEnergy.h:737-755)
// with the quadrature weight folded into the tgp record's (w mu, w lambda).
__device__ inline double TetElasticEnergy(int4 const* __restrict__ tetv, float4 const* __restrict__ tgp,
                                          float4 const* __restrict__ xm, int e)
{
    int4 const t = tetv[e];
    float4 const q0 = tgp[3 * e], q1 = tgp[3 * e + 1], q2 = tgp[3 * e + 2];
    float4 const p0 = xm[t.x], p1 = xm[t.y], p2 = xm[t.z], p3 = xm[t.w];
    double const r[3][3] = {{q0.x, q0.y, q0.z}, {q0.w, q1.x, q1.y}, {q1.z, q1.w, q2.x}};
    double const d[3][3] = {{double(p1.x) - p0.x, double(p1.y) - p0.y, double(p1.z) - p0.z},
                            {double(p2.x) - p0.x, double(p2.y) - p0.y, double(p2.z) - p0.z},
                            {double(p3.x) - p0.x, double(p3.y) - p0.y, double(p3.z) - p0.z}};
    double F[3][3]; // F[row][col] = sum_k d[k][row] r[k][col]
    double I2 = 0.;
    for (int rr = 0; rr < 3; ++rr)
        for (int c = 0; c < 3; ++c)
        {
            F[rr][c] = d[0][rr] * r[0][c] + d[1][rr] * r[1][c] + d[2][rr] * r[2][c];
            I2 += F[rr][c] * F[rr][c];
        }
    double const J = F[0][0] * (F[1][1] * F[2][2] - F[2][1] * F[1][2]) -
                     F[0][1] * (F[1][0] * F[2][2] - F[2][0] * F[1][2]) +
                     F[0][2] * (F[1][0] * F[2][1] - F[2][0] * F[1][1]);
    double const q = J - double(q2.w);
    return 0.5 * double(q2.y) * (I2 - 3.) + 0.5 * double(q2.z) * q * q;
}

// Sum three doubles over a 256-thread workgroup; the result is valid in thread 0.
__device__ inline void BlockSum3(double& a, double& b, double& c)
{
    __shared__ double red[3][4];
    for (int off = 32; off > 0; off >>= 1)
    {
        a += __shfl_xor(a, off);
        b += __shfl_xor(b, off);
        c += __shfl_xor(c, off);
    }
    int const w = static_cast<int>(threadIdx.x) / 64;
    if ((threadIdx.x & 63) == 0)
    {
        red[0][w] = a;
        red[1][w] = b;
        red[2][w] = c;
    }
    __syncthreads();
    if (threadIdx.x == 0)
    {
        a = red[0][0] + red[0][1] + red[0][2] + red[0][3];
        b = red[1][0] + red[1][1] + red[1][2] + red[1][3];
        c = red[2][0] + red[2][1] + red[2][2] + red[2][3];
    }
}

// FP64 energy reduction: out[0] += 1/2 m |v|^2, out[2] += -m a.x over vertices,
// out[1] += w Psi(F) over tets. One atomic per block and term. blockDim = 256.
[[maybe_unused]] static __global__ __launch_bounds__(256) void EnergyTerms(float4 const* __restrict__ xm, float4 const* __restrict__ vel,
                                                   float4 const* __restrict__ aext, int4 const* __restrict__ tetv,
                                                   float4 const* __restrict__ tgp, int nV, int nT,
                                                   double* __restrict__ out)
{
    double K = 0., U = 0., P = 0.;
    int const stride = static_cast<int>(gridDim.x * blockDim.x);
    for (int i = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x); i < nV; i += stride)
    {
        float4 const x = xm[i], u = vel[i], g = aext[i];
        double const m = x.w;
        K += 0.5 * m * (double(u.x) * u.x + double(u.y) * u.y + double(u.z) * u.z);
        P -= m * (double(g.x) * x.x + double(g.y) * x.y + double(g.z) * x.z);
    }
    for (int e = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x); e < nT; e += stride)
        U += TetElasticEnergy(tetv, tgp, xm, e);
    BlockSum3(K, U, P);
    if (threadIdx.x == 0)
    {
        atomicAdd(out + 0, K);
        atomicAdd(out + 1, U);
        atomicAdd(out + 2, P);
    }
}

// Trust-region reductions (gpu/impl/vbd/TrustRegionIntegrator.cu:265-364 objective
// terms without contact, :471-489 squared step): per workgroup partial sums of
// m |x - x~|^2, w Psi(F) and, when xprev is given, |x - xprev|^2, written to
// part[3 * blockIdx.x + j]. No atomics, so SumPartials3 gives the same bits on
// every run. blockDim = 256.
[[maybe_unused]] static __global__ __launch_bounds__(256) void ObjectiveTerms(
    float4 const* __restrict__ xm, float4 const* __restrict__ xtil, float4 const* __restrict__ xprev,
    int4 const* __restrict__ tetv, float4 const* __restrict__ tgp, int nV, int nT, double* __restrict__ part,
    double const* __restrict__ gate)
{
    if (gate && *gate == 0.)
        return; // not needed this time: the partials keep their last values
    double K = 0., U = 0., D = 0.;
    int const stride = static_cast<int>(gridDim.x * blockDim.x);
    for (int i = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x); i < nV; i += stride)
    {
        float4 const x = xm[i], y = xtil[i];
        double const dx = double(x.x) - y.x, dy = double(x.y) - y.y, dz = double(x.z) - y.z;
        K += double(x.w) * (dx * dx + dy * dy + dz * dz);
        if (xprev)
        {
            float4 const p = xprev[i];
            double const ex = double(x.x) - p.x, ey = double(x.y) - p.y, ez = double(x.z) - p.z;
            D += ex * ex + ey * ey + ez * ez;
        }
    }
    for (int e = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x); e < nT; e += stride)
        U += TetElasticEnergy(tetv, tgp, xm, e);
    BlockSum3(K, U, D);
    if (threadIdx.x == 0)
    {
        part[3 * blockIdx.x + 0] = K;
        part[3 * blockIdx.x + 1] = U;
        part[3 * blockIdx.x + 2] = D;
    }
}

// Gradient of the incremental potential f = 1/2 |x - x~|_M^2 + h^2 sum_e w_e Psi_e
// (sim::vbd::Integrator::ObjectiveFunctionGradient, sim/vbd/Integrator.cpp:168-200) in
// FP64 from the FP32 state, kGradientLanes lanes per vertex v of [0, nV):
//   g_v = m_v (x_v - x~_v) + h^2 sum_{(e, l) incident to v} (w_e P(F_e)) gp_{e,l}
// with P(F) = mu F + lambda (J - alpha) cof F the Stable Neo-Hookean stress
// (physics/StableNeoHookeanEnergy.h:766-795) and gp_{e,l} row l of the tet's shape
// function gradients. inc lists 4 e + l per vertex (CSR vtp), ascending e, so each
// vertex's sum has a fixed order (no atomics). grad: 3 doubles per vertex (internal
// order). part[3 b] receives workgroup b's sum of |g_v|^2 over v < nUpd (the
// non-Dirichlet vertices), part[3 b + 1..2] = 0. blockDim = 256.
// One lane per vertex walked its 24 tets alone, a load chain each, on half a wave per
// SIMD at 32^3: 34.7 us; 8 lanes: 20.6 (objective and gradient 234 -> 218 with the copies).
constexpr int kGradientLanes = 8;
[[maybe_unused]] static __global__ __launch_bounds__(256) void ObjectiveGradient(
    float4 const* __restrict__ xm, float4 const* __restrict__ xtil, int const* __restrict__ vtp,
    int const* __restrict__ inc, int4 const* __restrict__ tetv, float4 const* __restrict__ tgp, int nV, int nUpd,
    double dt2, double* __restrict__ grad, double* __restrict__ part)
{
    constexpr int L = kGradientLanes;
    int const lane = static_cast<int>(threadIdx.x) & (L - 1);
    int const v = static_cast<int>(blockIdx.x) * (256 / L) + static_cast<int>(threadIdx.x) / L;
    double r2 = 0.;
    double gx = 0., gy = 0., gz = 0.;
    if (v < nV)
    {
        for (int k = vtp[v] + lane; k < vtp[v + 1]; k += L)
        {
            int const e = inc[k] >> 2, l = inc[k] & 3;
            int4 const t = tetv[e];
            float4 const q0 = tgp[3 * e], q1 = tgp[3 * e + 1], q2 = tgp[3 * e + 2];
            float4 const p0 = xm[t.x], p1 = xm[t.y], p2 = xm[t.z], p3 = xm[t.w];
            double const r[3][3] = {{q0.x, q0.y, q0.z}, {q0.w, q1.x, q1.y}, {q1.z, q1.w, q2.x}};
            double const d[3][3] = {{double(p1.x) - p0.x, double(p1.y) - p0.y, double(p1.z) - p0.z},
                                    {double(p2.x) - p0.x, double(p2.y) - p0.y, double(p2.z) - p0.z},
                                    {double(p3.x) - p0.x, double(p3.y) - p0.y, double(p3.z) - p0.z}};
            double F[3][3]; // F[row][col] = sum_k d[k][row] r[k][col]
            for (int rr = 0; rr < 3; ++rr)
                for (int c = 0; c < 3; ++c)
                    F[rr][c] = d[0][rr] * r[0][c] + d[1][rr] * r[1][c] + d[2][rr] * r[2][c];
            double cof[3][3]; // column c = f_{c+1} x f_{c+2}
            for (int c = 0; c < 3; ++c)
            {
                int const c1 = (c + 1) % 3, c2 = (c + 2) % 3;
                cof[0][c] = F[1][c1] * F[2][c2] - F[2][c1] * F[1][c2];
                cof[1][c] = F[2][c1] * F[0][c2] - F[0][c1] * F[2][c2];
                cof[2][c] = F[0][c1] * F[1][c2] - F[1][c1] * F[0][c2];
            }
            double const J = F[0][0] * cof[0][0] + F[1][0] * cof[1][0] + F[2][0] * cof[2][0];
            double const wmu = q2.y, s = double(q2.z) * (J - double(q2.w));
            double gp[3];
            for (int c = 0; c < 3; ++c)
                gp[c] = (l == 0) ? -(r[0][c] + r[1][c] + r[2][c]) : r[l - 1][c];
            double out[3];
            for (int rr = 0; rr < 3; ++rr)
                out[rr] = (wmu * F[rr][0] + s * cof[rr][0]) * gp[0] + (wmu * F[rr][1] + s * cof[rr][1]) * gp[1] +
                          (wmu * F[rr][2] + s * cof[rr][2]) * gp[2];
            gx += out[0], gy += out[1], gz += out[2];
        }
    }
#pragma unroll
    for (int o = 1; o < L; o <<= 1)
        gx += __shfl_xor(gx, o), gy += __shfl_xor(gy, o), gz += __shfl_xor(gz, o);
    if (v < nV && lane == 0)
    {
        float4 const x = xm[v], y = xtil[v];
        double const m = x.w;
        gx = m * (double(x.x) - y.x) + dt2 * gx;
        gy = m * (double(x.y) - y.y) + dt2 * gy;
        gz = m * (double(x.z) - y.z) + dt2 * gz;
        grad[3 * v] = gx, grad[3 * v + 1] = gy, grad[3 * v + 2] = gz;
        if (v < nUpd)
            r2 = gx * gx + gy * gy + gz * gz;
    }
    double z0 = 0., z1 = 0.;
    BlockSum3(r2, z0, z1);
    if (threadIdx.x == 0)
    {
        part[3 * blockIdx.x] = r2;
        part[3 * blockIdx.x + 1] = 0.;
        part[3 * blockIdx.x + 2] = 0.;
    }
}

// ---- linear trust-region path (gpu/impl/vbd/TrustRegionIntegrator.cu:36-263) ----
// The model's FP64 scalars live in device memory; TrModel and the epilogue of
// the objective's last reduction (SumPartials3) update them between the sweeps,
// so a step reads nothing back to the host and can be replayed from a graph.
enum TrSlot
{
    kTrF = 0,   // f_k
    kTrT,       // t_k
    kTrFm1,     // f_{k-1}
    kTrFm2,     // f_{k-2}
    kTrTm1,     // t_{k-1}
    kTrTm2,     // t_{k-2}
    kTrR2,      // squared trust radius
    kTrQa,      // model m(t) = qa t^2 + qb t + qc
    kTrQb,
    kTrQc,
    kTrFVbd,    // f at the VBD iterate
    kTrStep,    // step length t tried this iteration
    kTrUpper,   // upper bound of t
    kTrAttempt, // 1 when t is tried (t != 1)
    kTrRevert,  // 1 when the tried step is rolled back
    kTrSlots
};

struct TrConstants
{
    double dt2, tau2, eta, small, fltMin, fltMax;
};

// f = 1/2 sum m |x - x~|^2 + h^2 sum w Psi from the reduced sums (K, U, .)
__device__ inline double TrObjective(double const* sums, double dt2) { return 0.5 * sums[0] + dt2 * sums[1]; }

// Start of a substep: f_0 at the initial iterate, empty history, R = 0.
__device__ inline void TrBegin(double* __restrict__ s, double const* __restrict__ sums, TrConstants const& c)
{
    s[kTrF] = TrObjective(sums, c.dt2);
    s[kTrT] = -1.;
    s[kTrFm1] = s[kTrFm2] = s[kTrTm1] = s[kTrTm2] = s[kTrR2] = 0.;
}

// After a plain iteration k < 2: the history shifts, then f_k, t_k = k.
__device__ inline void TrPlain(double* __restrict__ s, double const* __restrict__ sums, TrConstants const& c, int k)
{
    s[kTrFm2] = s[kTrFm1], s[kTrFm1] = s[kTrF];
    s[kTrTm2] = s[kTrTm1], s[kTrTm1] = s[kTrT];
    s[kTrF] = TrObjective(sums, c.dt2);
    s[kTrT] = static_cast<double>(k);
}

// Before the sweep of iteration k >= 2 (ConstructModel and UpdateIterates): times
// shifted so that t_k = 0, the quadratic through the last three (t, f) by
// Cramer's rule, then the history shifts.
[[maybe_unused]] static __global__ void TrModel(double* __restrict__ s)
{
    if (threadIdx.x != 0)
        return;
    double const tk = s[kTrT];
    double const tkm2 = s[kTrTm2] - tk, tkm1 = s[kTrTm1] - tk;
    double const fk = s[kTrF], fkm1 = s[kTrFm1], fkm2 = s[kTrFm2];
    double const det = tkm2 * tkm2 * tkm1 - tkm1 * tkm1 * tkm2;
    double const r2 = fkm2 - fk, r1 = fkm1 - fk;
    s[kTrQa] = (r2 * tkm1 - r1 * tkm2) / det;
    s[kTrQb] = (tkm2 * tkm2 * r1 - tkm1 * tkm1 * r2) / det;
    s[kTrQc] = fk;
    s[kTrFm2] = fkm1, s[kTrFm1] = fk;
    s[kTrTm2] = tkm1, s[kTrTm1] = 0.;
    s[kTrT] = 0.;
}

// After the sweep (sums at the VBD iterate, sums[2] = |dx|^2): the radius, the
// model's optimal step clamped to [1, R/|dx|] (ModelOptimalStep), and whether
// it is tried.
__device__ inline void TrDecide(double* __restrict__ s, double const* __restrict__ sums, TrConstants const& c)
{
    double const fVbd = TrObjective(sums, c.dt2), dx2 = sums[2];
    double R2 = s[kTrR2];
    if (R2 < dx2 + c.small)
        R2 = c.tau2 * dx2;
    double const lower = 1., upper = sqrt(R2 / dx2);
    double const qa = s[kTrQa], qb = s[kTrQb];
    double tstar = 0.;
    if (fabs(qa) > c.fltMin)
        tstar = qa > c.fltMin ? -qb / (2. * qa) : c.fltMax;
    else if (fabs(qb) > c.fltMin)
        tstar = qb > 0. ? -c.fltMax : c.fltMax;
    double const t = tstar < lower ? lower : (upper < tstar ? upper : tstar);
    s[kTrR2] = R2, s[kTrFVbd] = fVbd, s[kTrUpper] = upper, s[kTrStep] = t;
    s[kTrAttempt] = (fabs(t - lower) < c.small) ? 0. : 1.;
}

// After the tried step (sums at x(t), read only when a step was tried): keep it
// when the actual over the predicted decrease exceeds eta, growing R at the
// bound; otherwise shrink R and roll back (or keep the VBD iterate when nothing
// was tried). Logs (t, accepted) at slot.
__device__ inline void TrAccept(double* __restrict__ s, double const* __restrict__ sums, TrConstants const& c,
                                double* __restrict__ logT, int* __restrict__ logAccepted, int slot)
{
    bool const attempt = s[kTrAttempt] != 0.;
    double const t = s[kTrStep];
    bool accepted = false;
    if (attempt)
    {
        double const fk = TrObjective(sums, c.dt2);
        s[kTrF] = fk;
        double const mNext = s[kTrQa] * t * t + s[kTrQb] * t + s[kTrQc];
        double const fkm1 = s[kTrFm1];
        accepted = (fkm1 - fk) / (fkm1 - mNext) > c.eta;
    }
    if (accepted)
    {
        if ((s[kTrUpper] - t) < c.small)
            s[kTrR2] *= c.tau2;
        s[kTrT] = t;
        s[kTrRevert] = 0.;
    }
    else
    {
        s[kTrR2] /= c.tau2;
        s[kTrRevert] = attempt ? 1. : 0.;
        if (!attempt)
            s[kTrF] = s[kTrFVbd];
        s[kTrT] = s[kTrTm1] + 1.;
    }
    logT[slot] = t;
    logAccepted[slot] = accepted ? 1 : 0;
}

// After a rollback: f_k at the restored VBD iterate.
__device__ inline void TrRevert(double* __restrict__ s, double const* __restrict__ sums, TrConstants const& c)
{
    if (s[kTrRevert] != 0.)
        s[kTrF] = TrObjective(sums, c.dt2);
}

// Trust-region update that runs after a reduction, on its sums (SumPartials3).
enum TrOp : int
{
    kTrOpNone = 0,
    kTrOpBegin,
    kTrOpPlain,
    kTrOpDecide,
    kTrOpAccept,
    kTrOpRevert
};

struct TrEpilogue
{
    int op;          // TrOp
    double* s;       // trust-region state
    TrConstants c;
    double* logT;    // kTrOpAccept: decision log
    int* logAccepted;
    int slot;        // kTrOpAccept: log slot
    int k;           // kTrOpPlain: iteration
};

// out[j] = sum over b < nb of part[3 b + j], in a fixed order. One workgroup of 256.
// The sums are skipped when gate points at 0; the epilogue's trust-region update
// runs either way (it reads the sums only when they were formed).
[[maybe_unused]] static __global__ __launch_bounds__(256) void SumPartials3(double const* __restrict__ part, int nb,
                                                                           double* __restrict__ out,
                                                                           double const* __restrict__ gate,
                                                                           TrEpilogue e)
{
    if (!(gate && *gate == 0.))
    {
        double a = 0., b = 0., c = 0.;
        for (int k = static_cast<int>(threadIdx.x); k < nb; k += static_cast<int>(blockDim.x))
        {
            a += part[3 * k];
            b += part[3 * k + 1];
            c += part[3 * k + 2];
        }
        BlockSum3(a, b, c);
        if (threadIdx.x == 0)
        {
            out[0] = a;
            out[1] = b;
            out[2] = c;
        }
    }
    if (threadIdx.x != 0)
        return;
    switch (e.op)
    {
    case kTrOpBegin:
        TrBegin(e.s, out, e.c);
        break;
    case kTrOpPlain:
        TrPlain(e.s, out, e.c, e.k);
        break;
    case kTrOpDecide:
        TrDecide(e.s, out, e.c);
        break;
    case kTrOpAccept:
        TrAccept(e.s, out, e.c, e.logT, e.logAccepted, e.slot);
        break;
    case kTrOpRevert:
        TrRevert(e.s, out, e.c);
        break;
    default:
        break;
    }
}

// Trust-region step along the line through x_k (xkm1) and the VBD iterate
// (gpu/impl/vbd/TrustRegionIntegrator.cu:491-522): x = x_k + t (x - x_k), or, with
// rollback, x = x_k + (x - x_k) / t, t from the device state; nothing happens
// unless the state says the step is tried (rolled back). Masses in xm.w are kept.
[[maybe_unused]] static __global__ void LinearPathStep(float4* __restrict__ xm, float4 const* __restrict__ xkm1, int n,
                                                       double const* __restrict__ s, int rollback)
{
    int const i = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x);
    if (i >= n || s[rollback ? kTrRevert : kTrAttempt] == 0.)
        return;
    float const t = static_cast<float>(s[kTrStep]);
    float4 const x = xm[i], p = xkm1[i];
    float4 r;
    if (rollback)
        r = make_float4(p.x + (x.x - p.x) / t, p.y + (x.y - p.y) / t, p.z + (x.z - p.z) / t, x.w);
    else
        r = make_float4(p.x + t * (x.x - p.x), p.y + t * (x.y - p.y), p.z + t * (x.z - p.z), x.w);
    xm[i] = r;
}

[[maybe_unused]] static __global__ void ZeroDoubles(double* p, int n)
{
    int const i = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x);
    if (i < n)
        p[i] = 0.;
}

} // namespace pbat_vbd::device
