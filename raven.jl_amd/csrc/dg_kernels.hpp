// The laws, fluxes and face indexing shared by the stage kernels, and the
// fused 1-D DGSEM stage kernel for gfx950 (CDNA4, wave64).
//
// One fused launch computes, for every cell, Raven's weak-form volume term
// (dgsem.jl:257-348), its surface term with the Rusanov/central flux
// (dgsem.jl:733-784, numericalfluxes.jl:27-50) and the low-storage RK update
// (odesolvers.jl:55-57):
//     dq = a*dq + L(q_in);   q_out = q_in + b_dt*dq
//
// Neighbour states are read through per-face records (neighbour cell, face,
// orientation), so a face costs 8 bytes of index traffic instead of
// Nq^(dim-1) 8-byte node indices.  Owner-computes: each cell evaluates the
// numerical flux of all of its faces; no atomics, deterministic results.
#pragma once

#include <hip/hip_runtime.h>

#include "common.hpp"

namespace rv {

template <int B, int E>
struct IPow {
    static constexpr int v = B * IPow<B, E - 1>::v;
};
template <int B>
struct IPow<B, 0> {
    static constexpr int v = 1;
};

// Blocks are dealt to the 8 XCDs round-robin; renumber them so that each XCD
// walks a contiguous range of cells (neighbours then share that XCD's L2).
__device__ inline int64_t xcd_remap(int64_t b, int64_t nb)
{
    constexpr int64_t NX = 8;
    const int64_t q = nb / NX, r = nb % NX;
    const int64_t x = b % NX, idx = b / NX;
    return x * q + (x < r ? x : r) + idx;
}

// Each wave works in its own LDS slab and a wavefront's LDS operations
// complete in issue order, so ordering the compiler's memory operations is all
// the synchronisation a slab needs (no s_barrier tying a block's waves).
__device__ inline void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// A value every lane of the wave holds, moved to scalar registers.
__device__ inline int64_t wave_uniform(int64_t v)
{
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)(uint64_t)v);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)((uint64_t)v >> 32));
    return (int64_t)(((uint64_t)hi << 32) | lo);
}

// Lane l's value of v, broadcast to the whole wave (two v_readlane_b32).
__device__ inline double readlane_f64(double v, int l)
{
    const uint64_t b = (uint64_t)__double_as_longlong(v);
    const uint32_t lo = __builtin_amdgcn_readlane((int)(uint32_t)b, l);
    const uint32_t hi = __builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), l);
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

// Volume index of node m of face f (faces ordered -x,+x,-y,+y,-z,+z; face
// nodes over the remaining directions, first fastest: lobattocells.jl:2020-2050).
template <int DIM, int NQ>
__device__ __host__ inline int face_node(int f, int m)
{
    const int d = f >> 1;
    const int fixed = (f & 1) ? NQ - 1 : 0;
    if constexpr (DIM == 1) {
        return fixed;
    } else if constexpr (DIM == 2) {
        return d == 0 ? fixed + NQ * m : m + NQ * fixed;
    } else {
        const int a = m % NQ, b = m / NQ;
        if (d == 0)
            return fixed + NQ * a + NQ * NQ * b;
        if (d == 1)
            return a + NQ * fixed + NQ * NQ * b;
        return a + NQ * b + NQ * NQ * fixed;
    }
}

// Face-node permutation of a conforming neighbour: bit 2 swaps the two face
// directions, then bit 0 / bit 1 reverse the first / second one.
template <int DIM, int NQ>
__device__ __host__ inline int orient_node(int o, int m)
{
    if constexpr (DIM == 1) {
        return 0;
    } else if constexpr (DIM == 2) {
        return (o & 1) ? NQ - 1 - m : m;
    } else {
        int a = m % NQ, b = m / NQ;
        if (o & 4) {
            const int t = a;
            a = b;
            b = t;
        }
        if (o & 1)
            a = NQ - 1 - a;
        if (o & 2)
            b = NQ - 1 - b;
        return a + NQ * b;
    }
}

// --------------------------------------------------------------------------
// Balance laws (euler.jl:29-68, advection.jl:18-19).
// --------------------------------------------------------------------------
template <int DIM, int LAW>
struct LawInfo {
    static constexpr int NS = LAW == LAW_ADVECTION ? 1 : DIM + 2;
};

// Primitive helpers of the Euler law: velocity and pressure.
template <int DIM, typename R>
__device__ inline void euler_prim(const R *q, R gm1, R *u, R &p, R &rinv)
{
    rinv = R(1) / q[0];
#pragma unroll
    for (int d = 0; d < DIM; ++d)
        u[d] = q[1 + d] * rinv;
    R dot = q[1] * q[1];
#pragma unroll
    for (int d = 1; d < DIM; ++d)
        dot = dot + q[1 + d] * q[1 + d];
    p = gm1 * (q[DIM + 1] - dot * (R(0.5) * rinv));
}

// Row c of Raven's Euler flux matrix F (dim x Ns): F[c, s] for all s.
template <int DIM, typename R>
__device__ inline void euler_flux_row(int c, const R *q, const R *u, R p, R *f)
{
    f[0] = q[1 + c];
#pragma unroll
    for (int b = 0; b < DIM; ++b) {
        R v = q[1 + c] * u[b];
        if (b == c)
            v = v + p;
        f[1 + b] = v;
    }
    f[DIM + 1] = u[c] * (q[DIM + 1] + p);
}

template <int DIM, int LAW, typename R>
struct Law {
    static constexpr int NS = LawInfo<DIM, LAW>::NS;
    R gm1, gamma, u[3];

    __device__ inline Law(const StageParams &P)
    {
        gamma = R(P.gamma);
        gm1 = R(P.gamma - 1.0);
        u[0] = R(P.u[0]);
        u[1] = R(P.u[1]);
        u[2] = R(P.u[2]);
    }

    // flux row c of state q
    __device__ inline void flux_row(int c, const R *q, R *f) const
    {
        if constexpr (LAW == LAW_ADVECTION) {
            f[0] = u[c] * q[0];
        } else {
            R uu[DIM], p, rinv;
            euler_prim<DIM, R>(q, gm1, uu, p, rinv);
            euler_flux_row<DIM, R>(c, q, uu, p, f);
        }
    }

    // all flux rows F[c][s]
    __device__ inline void flux_all(const R *q, R (*F)[NS]) const
    {
        if constexpr (LAW == LAW_ADVECTION) {
#pragma unroll
            for (int c = 0; c < DIM; ++c)
                F[c][0] = u[c] * q[0];
        } else {
            R uu[DIM], p, rinv;
            euler_prim<DIM, R>(q, gm1, uu, p, rinv);
#pragma unroll
            for (int c = 0; c < DIM; ++c)
                euler_flux_row<DIM, R>(c, q, uu, p, F[c]);
        }
    }

    // wavespeed along unit normal n (|n.u| + c for Euler, |n.u| for advection)
    __device__ inline R wavespeed(const R *n, const R *q) const
    {
        if constexpr (LAW == LAW_ADVECTION) {
            R s = n[0] * u[0];
#pragma unroll
            for (int d = 1; d < DIM; ++d)
                s = s + n[d] * u[d];
            return fabs(s);
        } else {
            R uu[DIM], p, rinv;
            euler_prim<DIM, R>(q, gm1, uu, p, rinv);
            R nu = n[0] * uu[0];
#pragma unroll
            for (int d = 1; d < DIM; ++d)
                nu = nu + n[d] * uu[d];
            return fabs(nu) + sqrt(gamma * p * rinv);
        }
    }

    // wavespeed along +-e_c: |u_c| + c
    __device__ inline R wavespeed_axis(int c, const R *q) const
    {
        if constexpr (LAW == LAW_ADVECTION) {
            return fabs(u[c]);
        } else {
            R uu[DIM], p, rinv;
            euler_prim<DIM, R>(q, gm1, uu, p, rinv);
            return fabs(uu[c]) + sqrt(gamma * p * rinv);
        }
    }
};

// --------------------------------------------------------------------------
// Numerical fluxes, and the 1-D kernel.
// --------------------------------------------------------------------------

// Loads and stores of a cell's own dq and q_out: plain (ST = 0), or streaming
// (ST = 1: non-temporal, no reuse expected in L2).  The choice is a kernel
// variant picked by the launcher from StageParams::streaming: behind a
// run-time branch the compiler merges the two accesses and drops the hint.
template <int ST, typename T>
__device__ __attribute__((always_inline)) inline T load_dq(const T *p)
{
    if constexpr (ST)
        return __builtin_nontemporal_load(p);
    else
        return *p;
}

template <int ST, typename T>
__device__ __attribute__((always_inline)) inline void store_out(T v, T *p)
{
    if constexpr (ST)
        __builtin_nontemporal_store(v, p);
    else
        *p = v;
}
template <int DIM, int NQ, int LAW, typename R, int GEO, int FLUX>
struct Stage {
    static constexpr int NS = LawInfo<DIM, LAW>::NS;
    static constexpr int NP = IPow<NQ, DIM>::v;
    static constexpr int NP2 = NP / NQ;   // pencils per cell = face nodes per face
    static constexpr int EPW = 64 / NP2;  // cells per wave
    static constexpr int NF = 2 * DIM;
    static_assert(EPW >= 1, "Nq^(dim-1) must not exceed the wave size");

    // Neighbour state of face f at face node pen.
    __device__ static inline void neighbour_state(const StageParams &P, const R *qbase,
                                                  int64_t e, int f, int pen, const R *qm,
                                                  R *qp)
    {
        const FaceRec rec = P.faces[e * NF + f];
        if (rec.x >= 0) {
            const int fn = rec.y & 7, o = (rec.y >> 3) & 7;
            const int node = face_node<DIM, NQ>(fn, orient_node<DIM, NQ>(o, pen));
            const R *qn = qbase + (int64_t)rec.x * (NS * NP) + node;
#pragma unroll
            for (int s = 0; s < NS; ++s)
                qp[s] = qn[s * NP];
        } else if (rec.x == FACE_SELF) {
#pragma unroll
            for (int s = 0; s < NS; ++s)
                qp[s] = qm[s];
        } else {
            const int64_t off = P.explicit_idx[(int64_t)rec.y + pen];
#pragma unroll
            for (int s = 0; s < NS; ++s)
                qp[s] = qbase[off + s * NP];
        }
    }

    // Numerical flux for an axis-aligned unit normal sgn*e_c.
    __device__ static inline void nflux_axis(const Law<DIM, LAW, R> &law, int c, R sgn,
                                             const R *fm, const R *qm, const R *qp, R *nf)
    {
        R fp[NS];
        law.flux_row(c, qp, fp);
        if constexpr (FLUX == FLUX_RUSANOV) {
            const R wm = law.wavespeed_axis(c, qm), wp = law.wavespeed_axis(c, qp);
            const R lam = wm > wp ? wm : wp;
#pragma unroll
            for (int s = 0; s < NS; ++s)
                nf[s] = ((fm[s] + fp[s]) * R(0.5)) * sgn - (lam * (qp[s] - qm[s])) * R(0.5);
        } else {
#pragma unroll
            for (int s = 0; s < NS; ++s)
                nf[s] = ((fm[s] + fp[s]) * R(0.5)) * sgn;
        }
    }

    // Numerical flux for a general unit normal n.
    __device__ static inline void nflux_general(const Law<DIM, LAW, R> &law, const R *n,
                                                const R *qm, const R *qp, R *nf)
    {
        R Fm[DIM][NS], Fp[DIM][NS];
        law.flux_all(qm, Fm);
        law.flux_all(qp, Fp);
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            R fc = ((Fm[0][s] + Fp[0][s]) * R(0.5)) * n[0];
#pragma unroll
            for (int c = 1; c < DIM; ++c)
                fc = fc + ((Fm[c][s] + Fp[c][s]) * R(0.5)) * n[c];
            nf[s] = fc;
        }
        if constexpr (FLUX == FLUX_RUSANOV) {
            const R wm = law.wavespeed(n, qm), wp = law.wavespeed(n, qp);
            const R lam = wm > wp ? wm : wp;
#pragma unroll
            for (int s = 0; s < NS; ++s)
                nf[s] = nf[s] - (lam * (qp[s] - qm[s])) * R(0.5);
        }
    }
};

// Have the arguments that a stage needs read with the first ones.  Left alone the
// compiler reads them where they are first used, and each of these groups is
// another trip to memory on the path of a launch that is one wave's latency
// (Nq = 4 FP64 on 16^2 cells, us per LSRK stage, with the launch's shape read
// from the arguments as well: Euler 3.52 -> 3.32, advection 2.85 -> 2.44).
template <int GEO, int LAW, typename R>
__device__ __attribute__((always_inline)) inline void read_args(const StageParams &P)
{
    asm volatile("" ::"s"(P.faces), "s"(P.explicit_idx));
    if constexpr (GEO == GEO_AFFINE)
        asm volatile("" ::"s"(P.affine), "s"(P.Dw), "s"(P.winv));
    else if constexpr (sizeof(R) == 4)
        asm volatile("" ::"s"(P.vgeo32), "s"(P.mji32), "s"(P.sgeo32), "s"(P.Dt));
    else
        asm volatile("" ::"s"(P.vgeo), "s"(P.mji), "s"(P.sgeo), "s"(P.Dt));
    if constexpr (LAW == LAW_EULER)
        asm volatile("" ::"s"(P.gamma));
    else
        asm volatile("" ::"s"(P.u[0]), "s"(P.u[1]));
}

// The 1-D cells [cell0, cell0 + 64 / Nq) of a wave, a lane per node: states
// with lane-contiguous addresses, the fluxes of a cell exchanged through the
// wave's LDS row, the numerical flux of a face on the cell's end lanes.  A 1-D
// stage is a few waves: it waits for one wave's chain of loads and the launch.
template <int NQ, int LAW, typename R, int GEO, int FLUX, int ST>
__device__ __attribute__((always_inline)) inline void stage_wave_1d(const StageParams &P,
                                                                    int64_t cell0, R *wlds)
{
    using S = Stage<1, NQ, LAW, R, GEO, FLUX>;
    constexpr int NS = S::NS, C = 64 / NQ;
    constexpr bool GEN = GEO == GEO_GENERAL;
    const int lane = threadIdx.x & 63;
    const int c = lane / NQ, i = lane - c * NQ;
    const int64_t e = cell0 + c;
    const Law<1, LAW, R> law(P);
    if (c < C && e < P.K) {
        const bool on = P.dir_mask & 1;
        const int side = i == NQ - 1;
        const bool face = on && (i == 0 || side);
        const int64_t off = e * (NS * NQ) + i;
        const R *qin = static_cast<const R *>(P.q_in);
        R *dq = static_cast<R *>(P.dq) + off;
        R *qo = static_cast<R *>(P.q_out) + off;
        R q[NS], qp[NS], dqo[NS], m[NQ], g = R(1), mji = R(1), nv[1] = {side ? R(1) : R(-1)}, lift;
#pragma unroll
        for (int s = 0; s < NS; ++s)
            q[s] = qin[off + s * NQ];
        if (P.read_dq) {
#pragma unroll
            for (int s = 0; s < NS; ++s)
                dqo[s] = load_dq<ST>(dq + s * NQ);
        }
        const double *M = GEN ? P.Dt : P.Dw;
#pragma unroll
        for (int n = 0; n < NQ; ++n)
            m[n] = R(M[i * NQ + n]);
        if constexpr (GEN) {
            g = R(P.vgeo[e * NQ + i]);
            mji = R(P.mji[e * NQ + i]);
        } else {
            mji = R(P.affine[e]);
        }
        if (face) {
            S::neighbour_state(P, qin, e, side, 0, q, qp);
            if constexpr (GEN) {
                nv[0] = R(P.sgeo[(e * 2 + side) * 2]);
                lift = R(P.sgeo[(e * 2 + side) * 2 + 1]);
            } else {
                lift = R(P.winv[i]);
            }
        }
        R f[NS];
        law.flux_row(0, q, f);
#pragma unroll
        for (int s = 0; s < NS; ++s)
            wlds[s * 64 + lane] = g * f[s];
        R nf[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s)
            nf[s] = R(0);
        if (face) {
            if constexpr (GEN)
                S::nflux_general(law, nv, q, qp, nf);
            else
                S::nflux_axis(law, 0, nv[0], f, q, qp, nf);
#pragma unroll
            for (int s = 0; s < NS; ++s)
                nf[s] = lift * nf[s];
        }
        wave_lds_sync();
        const R a = R(P.a), bdt = R(P.b_dt);
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            R v = R(0);
            if (on) {
                const R *row = wlds + s * 64 + lane - i;
                v = m[0] * row[0];
#pragma unroll
                for (int n = 1; n < NQ; ++n)
                    v = v + m[n] * row[n];
                v = mji * (v - nf[s]);
            }
            if (P.read_dq)
                v = a * dqo[s] + v;
            store_out<ST>(v, dq + s * NQ);
            if (P.write_q)
                store_out<ST>(R(q[s] + bdt * v), qo + s * NQ);
        }
    }
}

// P.wpb waves per block; each has its own LDS rows.
template <int NQ, int LAW, typename R, int GEO, int FLUX, int ST>
__global__ void __launch_bounds__(256) dg_stage_kernel_1d(const StageParams P)
{
    __shared__ R lds[4][LawInfo<1, LAW>::NS * 64];
    const int wave = threadIdx.x >> 6;
    read_args<GEO, LAW, double>(P);
    const int64_t blk = xcd_remap(blockIdx.x, P.blocks);
    stage_wave_1d<NQ, LAW, R, GEO, FLUX, ST>(P, (blk * P.wpb + wave) * (64 / NQ), lds[wave]);
}

// The right-hand side alone of FP32 advection on large 1-D grids: a lane per
// cell.  A node is four bytes, and with no q_out written what a wave does besides
// counts most: here the operator is uniform (scalar loads) and a cell's fluxes
// stay in its lane.  us per right-hand side, a lane per node / per cell: 600000
// cells of Nq = 5 15.0 / 9.3, 375000 of Nq = 8 17.9 / 12.0, 62500 4.5 / 4.2, below
// the same; FP64, whose strided lanes fetch twice the lines, 375000 of Nq = 8 20.1
// / 21.8, 500000 of Nq = 6 15.3 / 19.0.
constexpr int64_t CELL_NODES_1D = 400000;
template <int NQ, int LAW, typename R, int GEO, int FLUX>
__global__ void __launch_bounds__(64) dg_rhs_cell_kernel_1d(const StageParams P)
{
    using S = Stage<1, NQ, LAW, R, GEO, FLUX>;
    static_assert(S::NS == 1, "advection");
    constexpr bool GEN = GEO == GEO_GENERAL;
    const int64_t e = xcd_remap(blockIdx.x, P.blocks) * 64 + threadIdx.x;
    if (e >= P.K)
        return;
    const Law<1, LAW, R> law(P);
    const R *qin = static_cast<const R *>(P.q_in);
    R *dq = static_cast<R *>(P.dq) + e * NQ;
    R q[NQ], f[NQ], qp[2], nf[2];
#pragma unroll
    for (int n = 0; n < NQ; ++n)
        q[n] = qin[e * NQ + n];
#pragma unroll
    for (int side = 0; side < 2; ++side)
        S::neighbour_state(P, qin, e, side, 0, q + (side ? NQ - 1 : 0), qp + side);
#pragma unroll
    for (int n = 0; n < NQ; ++n)
        law.flux_row(0, q + n, f + n);
#pragma unroll
    for (int side = 0; side < 2; ++side) {
        const int end = side ? NQ - 1 : 0;
        if constexpr (GEN) {
            const R nv[1] = {R(P.sgeo[(e * 2 + side) * 2])};
            S::nflux_general(law, nv, q + end, qp + side, nf + side);
            nf[side] = R(P.sgeo[(e * 2 + side) * 2 + 1]) * nf[side];
        } else {
            S::nflux_axis(law, 0, side ? R(1) : R(-1), f + end, q + end, qp + side, nf + side);
            nf[side] = R(P.winv[end]) * nf[side];
        }
    }
    if constexpr (GEN) {
#pragma unroll
        for (int n = 0; n < NQ; ++n)
            f[n] = R(P.vgeo[e * NQ + n]) * f[n];
    }
    const double RV_GLOBAL *M = GEN ? P.Dt : P.Dw;
    const bool on = P.dir_mask & 1;
    const R a = R(P.a);
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
        R x = R(M[i * NQ]) * f[0];
#pragma unroll
        for (int n = 1; n < NQ; ++n)
            x = x + R(M[i * NQ + n]) * f[n];
        if (i == 0 || i == NQ - 1)
            x = x - nf[i != 0];
        x = on ? R(GEN ? P.mji[e * NQ + i] : P.affine[e]) * x : R(0);
        dq[i] = P.read_dq ? a * dq[i] + x : x;
    }
}

// Launch a stage kernel of wpb waves per workgroup; 0, or -1 with HIP's error
// left for the caller.  A small stage takes less than its launch, so the launch
// is one runtime call: the <<<>>> syntax makes two (it puts the shape aside and
// fetches it back) and then the last error was asked for, 2.71 against 2.55 us
// on the host.
inline int launch_stage(void (*kernel)(StageParams), int64_t blocks, int wpb, size_t lds,
                        void *stream, const StageParams &P0)
{
    StageParams P = P0;
    P.blocks = (uint32_t)blocks;
    P.wpb = wpb;
    void *argv[] = {&P};
    return hipLaunchKernel(reinterpret_cast<const void *>(kernel), dim3(P.blocks), dim3(64 * wpb),
                           argv, lds, static_cast<hipStream_t>(stream)) == hipSuccess
               ? 0
               : -1;
}

template <int NQ, int LAW, typename R, int GEO, int FLUX>
int launch_stage_1d(const StageParams &P, void *stream, int wpb)
{
    if (P.K <= 0)
        return 0;
    if (wpb != 1 && wpb != 2 && wpb != 4)
        wpb = 1;
    if constexpr (LAW == LAW_ADVECTION && sizeof(R) == 4) {
        if (!P.write_q && P.K * NQ > CELL_NODES_1D) {
            return launch_stage(&dg_rhs_cell_kernel_1d<NQ, LAW, R, GEO, FLUX>, (P.K + 63) / 64, 1,
                                0, stream, P);
        }
    }
    const int64_t cells = (int64_t)wpb * (64 / NQ);
    const int64_t blocks = (P.K + cells - 1) / cells;
    if constexpr (form_streams(1, NQ, LAW, sizeof(R), GEO, 0)) {
        if (P.streaming) {
            return launch_stage(&dg_stage_kernel_1d<NQ, LAW, R, GEO, FLUX, 1>, blocks, wpb, 0,
                                stream, P);
        }
    }
    return launch_stage(&dg_stage_kernel_1d<NQ, LAW, R, GEO, FLUX, 0>, blocks, wpb, 0, stream, P);
}

}  // namespace rv
