// FluxDifferencingForm stage kernel (dgsem.jl:1-17, 163-255, 514-608):
// the volume term from a symmetric two-point flux instead of the weak form,
//   dq(ijk) += sum_dir sum_n [ -MJI D[id,n] l_g(ijk) . f#(q_ijk, q_n)
//                              + f#(q_ijk, q_n) . l_g(n) MJI D[n,id] ],
// l_g = MJ dRdX[dir, :], n running over the line through ijk along dir, with
// f# = CentralFlux (numericalfluxes.jl:39-42) or, for Euler,
// EntropyConservativeFlux (euler.jl:150-184, logavg numericalfluxes.jl:9-22),
// fused with the surface term (dgsem.jl:733-784) and the LSRK update
// dq = a dq + L(q), q_out = q + b dt dq (odesolvers.jl:55-57).  The surface
// flux is Rusanov or the volume form's own two-point flux f#(q-, q+)' n
// (surfaceflux, numericalfluxes.jl:27-37), the pairing of Raven's
// entropy-conservation tests.
//
// Two kernels, chosen by fd_by_line (common.hpp):
//
// The line kernel (fd_stage; Euler with the entropy-conservative flux, grids
// that fill the device): a lane owns a LINE (Nq nodes along one direction) of
// a cell, and a workgroup the dim Nq^(dim-1) lines of each of its C cells.
//  * phase 0: the workgroup reads its cells' states and leaves each node's
//    primitives in LDS;
//  * phase 1: each lane walks the Nq (Nq - 1) / 2 symmetric pairs of its line,
//    every two-point flux evaluated once and added to both ends in registers,
//    then adds the numerical fluxes of the two faces its line ends on (the
//    line's index is the face node's);
//  * phase 2: the directions' sums meet in LDS, in the primitives' place, one
//    direction after another (fixed order, deterministic);
//  * phase 3: the update, with lane-contiguous accesses; q comes from the
//    caches a second time.
// Affine cells read the velocities with the line's direction first (LDS holds
// u, v, w, u, v), so that one code serves every direction and only row 0 of
// the flux is formed; curved cells form the flux along the pair's metric
// vector D[n,i] l_n - D[i,n] l_i.
//
// It is bound by FP64 (or unpacked FP32) vector issue and HBM together: 52 or
// 60 instructions a pair (short or long series), 10.5 pairs a node at Nq = 8.
// On 32^3 cells of Nq = 8 a FP64 stage takes 0.86 ms (a thread per node with the
// pairs' terms exchanged through an LDS buffer took 2.00 ms): 2.94 GB moved (3.4
// TB/s), vector units busy 66 % of the cycles.
//
// The node kernel (fd_stage_node; everything else): a lane per node, each pair
// evaluated from both ends.  The fluxes of the central forms cost little, and
// small grids wait for the chain of one wave.  Pairs that need logarithms cost
// most: with log_factor in place of the library's logarithm, 375000 1-D cells of
// Nq = 8 with such states take 157 us a FP64 stage (216 us without it), 56^2 of
// Nq = 8 32 (43); its registers make stages of smooth states on grids near the
// switch up to 10 % longer (7^3 of Nq = 8 25.9 -> 28.5).
//
// A relaxation stage (RX, the RLSRK step of odesolvers.jl:117-151) keeps
// k = L(q) apart from a dq, forms dq = a dq + k at the end and leaves each
// workgroup's sum of MJ v(q) . k (the stage's entropy production) in
// P.eprod[workgroup].
//
// Compiled once per (dim, precision) with -DFD_DIM and -DFD_REAL; api.hip asks
// every unit for a launcher.
#include <type_traits>

#include <hip/hip_runtime.h>

#include "common.hpp"
#include "dg_kernels.hpp"
#include "entropy.hpp"

#ifndef FD_DIM
#error "FD_DIM must be defined"
#endif

namespace rv {

namespace {

// F = atanh(f) / f = log(zeta) / 2f as a series in u = f^2, and 1 / 2F, the
// factors of the logarithmic mean (a + b) / 2F (logavg, numericalfluxes.jl:
// 9-22, zeta = a / b, f = (a - b) / (a + b)).  Two lengths: for u < LIMIT[k]
// the TERMS[k] terms leave a remainder below the type's rounding (FP64:
// u^8 / 17 < 6e-18 below 1e-2, u^4 / 9 < 1.2e-17 below 1e-4; FP32: u^4 / 9
// and u^2 / 5 < 2e-9).
template <typename R>
struct LogSeries {
    static constexpr int TERMS[2] = {sizeof(R) == 8 ? 8 : 4, sizeof(R) == 8 ? 4 : 2};
    static constexpr double LIMIT[2] = {1e-2, 1e-4};
    static constexpr double FLIMIT[2] = {1e-1, 1e-2};  // the same for f
    static constexpr int MOST = 11;
    double f[MOST], g[MOST];
    constexpr LogSeries() : f{}, g{}
    {
        for (int k = 0; k < MOST; ++k)
            f[k] = 1.0 / (2 * k + 1);
        // the reciprocal series: sum_{j <= k} f_j g_{k-j} = 0 for k > 0
        for (int k = 0; k < MOST; ++k) {
            double v = k == 0 ? 0.5 : 0.0;
            for (int j = 1; j <= k; ++j)
                v -= f[j] * g[k - j];
            g[k] = v;
        }
    }
};

template <typename R, int TERMS>
__device__ __forceinline__ R atanh_series(R u)
{
    constexpr LogSeries<R> c;
    R v = R(c.f[TERMS - 1]);
#pragma unroll
    for (int k = TERMS - 2; k >= 0; --k)
        v = v * u + R(c.f[k]);
    return v;
}
template <typename R, int SHORT>
__device__ __forceinline__ R series_f(R u)
{
    return atanh_series<R, LogSeries<R>::TERMS[SHORT]>(u);
}
template <typename R, int SHORT>
__device__ __forceinline__ R series_g(R u)
{
    constexpr LogSeries<R> c;
    R v = R(c.g[c.TERMS[SHORT] - 1]);
#pragma unroll
    for (int k = c.TERMS[SHORT] - 2; k >= 0; --k)
        v = v * u + R(c.g[k]);
    return v;
}

// 1 / x from the hardware estimate by Newton's method (x and 1 / x normal; NaN
// for zero and infinity): two steps from v_rcp_f64's about 2^-24, one from
// v_rcp_f32's 1 ulp
__device__ __forceinline__ double recip(double x)
{
    double r = __builtin_amdgcn_rcp(x);
    r = __builtin_fma(__builtin_fma(-x, r, 1.0), r, r);
    return __builtin_fma(__builtin_fma(-x, r, 1.0), r, r);
}
__device__ __forceinline__ float recip(float x)
{
    const float r = __builtin_amdgcn_rcpf(x);
    return __builtin_fmaf(__builtin_fmaf(-x, r, 1.0f), r, r);
}

// r = recip(x) with a division's values for zero, infinity and NaN
__device__ __forceinline__ double recip_any(double x, double r)
{
    return __builtin_amdgcn_div_fixup(r, x, 1.0);
}
__device__ __forceinline__ float recip_any(float x, float r)
{
    return __builtin_amdgcn_div_fixupf(r, x, 1.0f);
}

// F = log(a / b) / 2f beyond the series, or (INV) 1 / 2F; s = a + b, d = a - b,
// is = 1 / s.  In FP64
//   log(a / b) = k log 2 + 2 atanh((a' - b') / (a' + b')),
// a' and b' the mantissas, one of them halved where their ratio leaves
// [1/sqrt 2, sqrt 2]: (a' - b') / (a' + b') is then at most 0.172, and 11 terms
// leave a remainder below the rounding (u^11 / 23 < 1e-18).  About half the
// operations of a division, the library's logarithm and another division;
// against the exact value on 2 M random pairs at most 2.9 eps and 0.57 eps rms,
// those 3.4 and 0.89.  FP32's logarithm is an instruction and stays.
template <bool INV>
__device__ __forceinline__ float log_factor(float a, float b, float, float d, float is)
{
    const float l = log(a / b), f = d * is;
    return INV ? f / l : l / (2.0f * f);
}
template <bool INV>
__device__ __forceinline__ double log_factor(double a, double b, double s, double d, double is)
{
    double f = d * is;
    // (positive normal numbers)
    if (!(__builtin_amdgcn_class(a, 0x100) && __builtin_amdgcn_class(b, 0x100)))
        return INV ? f / log(a / b) : log(a / b) / (2.0 * f);
    double ma = __builtin_amdgcn_frexp_mant(a), mb = __builtin_amdgcn_frexp_mant(b);
    const bool up = ma > 1.4142135623730951 * mb, down = mb > 1.4142135623730951 * ma;
    ma = up ? 0.5 * ma : ma;
    mb = down ? 0.5 * mb : mb;
    const double k = __builtin_amdgcn_frexp_exp(a) - __builtin_amdgcn_frexp_exp(b) +
                     (up ? 1 : 0) - (down ? 1 : 0);
    const double t = (ma - mb) * recip(ma + mb);
    const double l = k * 0.34657359027997264 + t * atanh_series<double, 11>(t * t);
    // l / f (INV: f / 2l), f and the quotient corrected by their remainders
    f = (d - f * s) * is + f;
    const double x = INV ? 0.5 * f : l, y = INV ? l : f;
    const double r = recip(y), q = x * r;
    return (x - q * y) * r + q;
}

// A node of a line, what the two-point flux takes from it, and the flux of a
// pair along a metric vector m (GEN) or along component 0 of the (permuted)
// velocity.  LDS holds the NV values of a node that values() forms.
template <int DIM, int LAW, int VF, typename R, bool GEN>
struct TwoPoint {
    static constexpr int NS = LawInfo<DIM, LAW>::NS;
    static constexpr bool ADV = LAW == LAW_ADVECTION;
    static constexpr bool EC = VF == FLUX_EC && !ADV;
    static constexpr int NV = ADV ? 1 : 2 + DIM;

    // EC: rho, b = rho / p (twice Raven's b) and half the velocity; central
    // Euler: rho, p, the velocity and (v) E + p; advection: q in rho
    struct Node {
        R rho, b, u[DIM], v;
    };

    // the values of a node: rho, b (EC) or p, u / 2 (EC) or u
    __device__ static __forceinline__ void values(const Law<DIM, LAW, R> &law, const R *q, R *x)
    {
        x[0] = q[0];
        if constexpr (!ADV) {
            const R rinv = R(1) / q[0];
            R dot = q[1] * q[1];
#pragma unroll
            for (int d = 1; d < DIM; ++d)
                dot = dot + q[1 + d] * q[1 + d];
            const R p = law.gm1 * (q[DIM + 1] - dot * (R(0.5) * rinv));
            x[1] = EC ? q[0] / p : p;
#pragma unroll
            for (int d = 0; d < DIM; ++d)
                x[2 + d] = EC ? R(0.5) * (q[1 + d] * rinv) : q[1 + d] * rinv;
        }
    }

    __device__ static __forceinline__ Node node(const Law<DIM, LAW, R> &law, const R *x)
    {
        Node a;
        a.rho = x[0];
        a.b = a.v = R(0);
        if constexpr (!ADV) {
            a.b = x[1];
            R uu = R(0);
#pragma unroll
            for (int d = 0; d < DIM; ++d) {
                a.u[d] = x[2 + d];
                uu = d == 0 ? x[2] * x[2] : uu + x[2 + d] * x[2 + d];
            }
            if constexpr (!EC)
                a.v = a.b * (law.gamma / law.gm1) + R(0.5) * a.rho * uu;
        }
        return a;
    }

    // f#(a, b) along m (GEN), else component 0.  SERIES: which of the log
    // series (the caller has made sure that every u = f^2 is below its limit,
    // and that rho and b are far from the ends of the type's range), or for any
    // pair of states -1, or -2 with log_factor in place of the library's
    // logarithm (not in the line kernel: 10 to 30 more registers there spill).
    template <int SERIES>
    __device__ static __forceinline__ void flux(const Law<DIM, LAW, R> &law, const Node &a,
                                                const Node &b, const R *m, R *F)
    {
        if constexpr (ADV) {
            R un = law.u[0];
            if constexpr (GEN) {
                un = law.u[0] * m[0];
#pragma unroll
                for (int d = 1; d < DIM; ++d)
                    un = un + law.u[d] * m[d];
            }
            F[0] = R(0.5) * un * (a.rho + b.rho);
        } else if constexpr (!EC) {
            R una = a.u[0], unb = b.u[0];
            if constexpr (GEN) {
                una = a.u[0] * m[0], unb = b.u[0] * m[0];
#pragma unroll
                for (int d = 1; d < DIM; ++d) {
                    una = una + a.u[d] * m[d];
                    unb = unb + b.u[d] * m[d];
                }
            }
            una = R(0.5) * una, unb = R(0.5) * unb;
            const R fa = a.rho * una, fb = b.rho * unb;
            const R p = R(0.5) * (a.b + b.b);
            F[0] = fa + fb;
#pragma unroll
            for (int d = 0; d < DIM; ++d) {
                const R v = fa * a.u[d] + fb * b.u[d];
                F[1 + d] = GEN ? v + p * m[d] : d == 0 ? v + p : v;
            }
            F[DIM + 1] = una * a.v + unb * b.v;
        } else {
            // EntropyConservativeFlux (euler.jl:150-184).  With s = a + b and
            // f = (a - b) / (a + b): rho's logarithmic mean is s_rho / 2F, the
            // pressure average s_rho / s_b, and the energy flux
            //   f_rho (1 / (2 gm1 blog) - (u2)avg / 2 + |uavg|^2) + p uavg
            // = f_rho (2 F_b / (gm1 s_b) + u_a . u_b / 2) + p uavg
            // with s_b of twice Raven's b.  In FP64 one reciprocal of s_rho s_b
            // serves both quotients where the caller knows the product's range
            // (SERIES >= 0); FP32's range is too small for the product.
            const R sr = a.rho + b.rho, dr = a.rho - b.rho;
            const R sb = a.b + b.b, db = a.b - b.b;
            R isr, isb;
            if constexpr (sizeof(R) == 8 && SERIES >= 0) {
                const R i = recip(sr * sb);
                isr = i * sb;
                isb = i * sr;
            } else {
                isr = recip(sr);
                isb = recip(sb);
            }
            const R fr = dr * isr, fb = db * isb;
            const R ur = fr * fr, ub = fb * fb;
            R G, Fb;  // 1 / 2F of rho, F of b
            if constexpr (SERIES >= 0) {
                G = series_g<R, SERIES>(ur);
                Fb = series_f<R, SERIES>(ub);
            } else {
                // the logarithm beyond the series; there a sum that is zero or
                // infinite (its f is NaN) divides as a division would
                if (ur < R(LogSeries<R>::LIMIT[0])) {
                    G = series_g<R, 0>(ur);
                } else {
                    isr = recip_any(sr, isr);
                    G = SERIES == -2 ? log_factor<true>(a.rho, b.rho, sr, dr, isr)
                                     : dr * isr / log(a.rho / b.rho);
                }
                if (ub < R(LogSeries<R>::LIMIT[0])) {
                    Fb = series_f<R, 0>(ub);
                } else {
                    isb = recip_any(sb, isb);
                    Fb = SERIES == -2 ? log_factor<false>(a.b, b.b, sb, db, isb)
                                      : log(a.b / b.b) / (R(2) * (db * isb));
                }
            }
            R ua[DIM];
#pragma unroll
            for (int d = 0; d < DIM; ++d)
                ua[d] = a.u[d] + b.u[d];
            R un = ua[0];
            if constexpr (GEN) {
                un = ua[0] * m[0];
#pragma unroll
                for (int d = 1; d < DIM; ++d)
                    un = un + ua[d] * m[d];
            }
            const R f0 = un * (sr * G);
            const R p = sr * isb;
            R e = (R(2) * a.u[0]) * b.u[0];  // (2 a.u is common to a node's pairs)
#pragma unroll
            for (int d = 1; d < DIM; ++d)
                e = e + (R(2) * a.u[d]) * b.u[d];
            e = (Fb * isb) * (R(2) / law.gm1) + e;
            F[0] = f0;
#pragma unroll
            for (int d = 0; d < DIM; ++d)
                F[1 + d] = GEN ? f0 * ua[d] + p * m[d] : d == 0 ? f0 * ua[0] + p : f0 * ua[d];
            e = f0 * e + p * un;
            F[DIM + 1] = e;
        }
    }
};

template <int DIM, int NQ, int LAW, typename R, int GEO, int VF, int SF>
struct FD {
    static constexpr int NS = LawInfo<DIM, LAW>::NS;
    static constexpr int NP = IPow<NQ, DIM>::v;
    static constexpr int NL = NP / NQ;  // lines per direction, face nodes per face
    static constexpr int NF = 2 * DIM;
    static constexpr bool GEN = GEO == GEO_GENERAL;
    using TP = TwoPoint<DIM, LAW, VF, R, GEN>;
    static constexpr int C = fd_cells_per_workgroup(DIM, NQ);
    static constexpr int TASKS = C * DIM * NL;
    static constexpr int THREADS = (TASKS + 63) / 64 * 64;
    static constexpr int ITER = (C * NP + THREADS - 1) / THREADS;  // nodes per thread
    // rows of Nq nodes are padded to an odd length in LDS, so that the lanes
    // walking x-lines fall in different banks
    static constexpr int PR = NQ | 1;
    static constexpr int CS = NL * PR;
    static constexpr int CMP = C * CS;  // one component of the workgroup's cells
    // components: rho, b, then u, v, w and (affine) u, v again
    static constexpr int NC = TP::NV + (GEN ? 0 : DIM - 1);
    static constexpr int POOL = CMP * (NC > NS ? NC : NS);
    // FP64: the line's sums take 2 Nq Ns registers; partners are read from LDS
    // at every pair instead of being held, so that three waves share a SIMD
    static constexpr bool REREAD = sizeof(R) == 8 && NQ >= 5;
    // the faces' states are requested before the pairs where they fit the
    // registers next to the line's sums (32-bit words)
    static constexpr bool EARLY = NS * (NQ + 4) * (int)(sizeof(R) / 4) <= 80;
    // the node kernel's workgroup
    static constexpr int NODE_C = fd_node_cells(DIM, NQ);
    static constexpr int NODE_THREADS = (NODE_C * NP + 63) / 64 * 64;
    using S = Stage<DIM, NQ, LAW, R, GEO, FLUX_RUSANOV>;
};

// P.eprod[workgroup] = the sum of its threads' products (a relaxation stage),
// compensated, in a fixed order: a butterfly of (sum, compensation) pairs
// inside each wave (both lanes of a pair form the same sum), then the wave
// sums in wave order
template <int THREADS>
__device__ __forceinline__ void store_product(const StageParams &P, double prod, double pc)
{
    __shared__ double red[2 * (THREADS / 64)];
    const int t = threadIdx.x;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const double os = __shfl_xor(prod, off), oc = __shfl_xor(pc, off);
        comp_add(prod, pc, os, oc);
    }
    if ((t & 63) == 0) {
        red[2 * (t >> 6)] = prod;
        red[2 * (t >> 6) + 1] = pc;
    }
    __syncthreads();
    if (t == 0) {
        double sum = red[0], comp = red[1];
        for (int w = 1; w < THREADS / 64; ++w)
            comp_add(sum, comp, red[2 * w], red[2 * w + 1]);
        P.eprod[blockIdx.x] = sum + comp;
    }
}

template <int DIM, int NQ, int LAW, typename R, int GEO, int VF, int SF, bool RX, int ST>
__device__ __forceinline__ void fd_stage(const StageParams &P)
{
    using T = FD<DIM, NQ, LAW, R, GEO, VF, SF>;
    using S = typename T::S;
    using TP = typename T::TP;
    using Node = typename TP::Node;
    constexpr int NS = T::NS, NP = T::NP, NL = T::NL, NF = T::NF, PR = T::PR, CMP = T::CMP;
    constexpr bool GEN = T::GEN;
    static_assert(TP::EC && DIM > 1, "the line kernel's forms (fd_has_line_kernel)");
    __shared__ __align__(16) R lds[T::POOL];
    const int t = threadIdx.x;
    const int64_t cell0 = xcd_remap(blockIdx.x, P.blocks) * T::C;
    const Law<DIM, LAW, R> law(P);
    const R *qin = static_cast<const R *>(P.q_in);
    // cells past the last one repeat its work and store nothing
    auto cell = [&](int c) {
        const int64_t e = cell0 + c;
        return e < P.K ? e : P.K - 1;
    };

    // ---- phase 0: primitives
    {
        R q[T::ITER][NS];
#pragma unroll
        for (int it = 0; it < T::ITER; ++it) {
            const int v = t + it * T::THREADS;
            if (v < T::C * NP) {
                const int c = v / NP, node = v - c * NP;
                const R *qe = qin + cell(c) * (NS * NP) + node;
#pragma unroll
                for (int s = 0; s < NS; ++s)
                    q[it][s] = qe[s * NP];
            }
        }
#pragma unroll
        for (int it = 0; it < T::ITER; ++it) {
            const int v = t + it * T::THREADS;
            if (v < T::C * NP) {
                const int c = v / NP, node = v - c * NP;
                R *x = lds + c * T::CS + node + (PR - NQ) * (node / NQ);
                R val[TP::NV];
                TP::values(law, q[it], val);
#pragma unroll
                for (int k = 0; k < TP::NV; ++k)
                    x[k * CMP] = val[k];
                if constexpr (!GEN) {
#pragma unroll
                    for (int d = 0; d + 1 < DIM; ++d)
                        x[(TP::NV + d) * CMP] = val[2 + d];
                }
            }
        }
    }
    __syncthreads();

    // ---- phase 1: a line per lane
    int dir = t / (T::C * NL);
    if constexpr (T::C * NL % 64 == 0)
        dir = __builtin_amdgcn_readfirstlane(dir);  // a wave has one direction
    const bool line_on = t < T::TASKS && ((P.dir_mask >> dir) & 1);
    // the line's cell and index, its first node and stride: unpadded, and in
    // the LDS layout
    const int nstr = dir == 0 ? 1 : dir == 1 ? NQ : NQ * NQ;
    const int lstr = dir == 0 ? 1 : dir == 1 ? PR : PR * NQ;
    struct Line {
        int c, l, nbase, lbase;
    };
    auto line_of = [&](int tt) {
        Line r;
        r.c = T::C == 1 ? 0 : (tt - dir * (T::C * NL)) / NL;
        r.l = tt - dir * (T::C * NL) - r.c * NL;
        r.nbase = dir == 0 ? r.l * NQ : dir == 1 ? r.l % NQ + (r.l / NQ) * (NQ * NQ) : r.l;
        r.lbase = r.c * T::CS + (dir == 0   ? r.l * PR
                                 : dir == 1 ? r.l % NQ + (r.l / NQ) * (PR * NQ)
                                            : r.l % NQ + (r.l / NQ) * PR);
        return r;
    };
    // (an opaque copy of the thread's index: what is derived from it again
    // after the pairs need not be held in registers through them)
    auto fresh = [](int tt) {
        asm volatile("" : "+v"(tt));
        return tt;
    };
    const int uoff = GEN ? 0 : dir * CMP;
    R acc[NQ][NS];
    R scale = R(0);  // dRdX of the line's cell and direction (curved cells: 1)
    if (line_on) {
        const Line line = line_of(t);
        int lbase = line.lbase;
        const int64_t e = cell(line.c);
        auto load = [&](int n) {
            const R *x = lds + lbase + n * lstr;
            R val[TP::NV];
            val[0] = x[0];
            val[1] = x[CMP];
#pragma unroll
            for (int d = 0; d < DIM; ++d)
                val[2 + d] = x[uoff + (2 + d) * CMP];
            return TP::node(law, val);
        };
        // FP32 state reads the FP32 copies of the geometry (every use
        // rounds to the state's type)
        constexpr bool G32 = GEN && sizeof(R) == 4;
        using GT = typename std::conditional<G32, float, double>::type;
        const GT RV_GLOBAL *vgeo, *sgeo;
        if constexpr (G32)
            vgeo = P.vgeo32, sgeo = P.sgeo32;
        else
            vgeo = P.vgeo, sgeo = P.sgeo;
        const int64_t gbase = (e * DIM + dir) * DIM * NP + line.nbase;
        auto metric = [&](int n, R *lg) {
#pragma unroll
            for (int d = 0; d < DIM; ++d)
                lg[d] = R(vgeo[gbase + n * nstr + d * NP]);
        };
        FaceRec rec[2];
#pragma unroll
        for (int side = 0; side < 2; ++side)
            rec[side] = P.faces[e * NF + 2 * dir + side];
        // uniform tables through the scalar cache: S[i][n] = D[n,i] w_n / w_i -
        // D[i,n] (affine) and D[i,n] (curved)
        using Tab = const R __attribute__((address_space(4)));
        Tab *S_in = (Tab *)(static_cast<const R RV_GLOBAL *>(P.fdtab));
        Tab *Dtab = S_in + NQ * NQ;

        // the faces the line ends on (surfaceterm!): both ends' states from
        // memory (the caches hold the cell's own), momentum with the line's
        // direction first on affine cells
        R qm[2][NS], qp[2][NS];
        int l;
        auto face_states = [&](int tt) {
            const Line ln = line_of(tt);
            l = ln.l;
            lbase = ln.lbase;
            int comp[NS];
#pragma unroll
            for (int s = 0; s < NS; ++s)
                comp[s] = s;
            if constexpr (!GEN) {
#pragma unroll
                for (int d = 0; d < DIM; ++d) {
                    const int k = dir + d;
                    comp[1 + d] = 1 + (k >= DIM ? k - DIM : k);
                }
            }
#pragma unroll
            for (int side = 0; side < 2; ++side) {
                const R *qe = qin + e * (NS * NP) + ln.nbase + (side ? (NQ - 1) * nstr : 0);
#pragma unroll
                for (int s = 0; s < NS; ++s)
                    qm[side][s] = qe[comp[s] * NP];
                const FaceRec rc = rec[side];
                if (rc.x != FACE_SELF) {
                    int64_t off;
                    if (rc.x >= 0) {
                        const int fn = rc.y & 7, o = (rc.y >> 3) & 7;
                        off = (int64_t)rc.x * (NS * NP) +
                              face_node<DIM, NQ>(fn, orient_node<DIM, NQ>(o, l));
                    } else {
                        off = P.explicit_idx[(int64_t)rc.y + l];
                    }
#pragma unroll
                    for (int s = 0; s < NS; ++s)
                        qp[side][s] = qin[off + comp[s] * NP];
                } else {
#pragma unroll
                    for (int s = 0; s < NS; ++s)
                        qp[side][s] = qm[side][s];
                }
            }
        };
        if constexpr (T::EARLY)
            face_states(t);

        // Which log series serves every pair of the wave's lines: a pair's f is
        // at most that of the line's extremes.  The extremes are taken on the
        // leading 32 bits (positive values order as their bits do; a negative
        // or NaN value fails the test), the largest rounded up.  They are
        // compared without squares, which would leave the type's range, and
        // each is kept where the flux's reciprocals are normal numbers (FP64
        // takes one of the product of the sums of rho and of b).
        constexpr int W = sizeof(R) / 4;  // 32-bit words per value
        constexpr R LEAST = W == 2 ? R(1e-140) : R(1e-37), MOST = W == 2 ? R(1e140) : R(1e37);
        const uint32_t *w = reinterpret_cast<const uint32_t *>(lds) + W * lbase + (W - 1);
        bool ok[2] = {true, true};
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            uint32_t lo = w[W * k * CMP], hi = lo;
#pragma unroll
            for (int n = 1; n < NQ; ++n) {
                const uint32_t v = w[W * (n * lstr + k * CMP)];
                lo = v < lo ? v : lo;
                hi = v > hi ? v : hi;
            }
            R x0, x1;
            if constexpr (W == 2) {
                x0 = __longlong_as_double((long long)((uint64_t)lo << 32));
                x1 = __longlong_as_double((long long)((uint64_t)hi << 32 | 0xffffffffu));
            } else {
                x0 = __uint_as_float(lo);
                x1 = __uint_as_float(hi);
            }
            const R d = fabs(x1 - x0), s = x1 + x0;
            ok[0] = ok[0] && x0 > LEAST && x1 < MOST;
#pragma unroll
            for (int j = 0; j < 2; ++j)
                ok[j] = ok[j] && d < R(LogSeries<R>::FLIMIT[j]) * s;
        }
        ok[1] = ok[1] && ok[0];
        // 0: short series, 1: long series, 2: logarithms
        const int rough = __all(ok[1]) ? 0 : __all(ok[0]) ? 1 : 2;
        auto pairs = [&](auto series) {
            constexpr int SERIES = decltype(series)::value;
#pragma unroll
            for (int i = 0; i + 1 < NQ; ++i) {
                if constexpr (T::REREAD) {
                    // (an opaque copy of the addresses: partners are read
                    // again for each i and not kept)
                    asm volatile("" : "+v"(lbase));
                }
                // (an opaque condition ends the basic block: the scheduler
                // would otherwise hoist later nodes' reads and spill)
                int go = 1;
                asm volatile("" : "+s"(go));
                if (go == 0)
                    continue;
                const Node a = load(i);
                R la[DIM];
                if constexpr (GEN)
                    metric(i, la);
#pragma unroll
                for (int n = i + 1; n < NQ; ++n) {
                    const Node b = load(n);
                    R F[NS], wi = R(1), wn = R(-1);
                    if constexpr (GEN) {
                        R lb[DIM], m[DIM];
                        metric(n, lb);
                        const R Dni = Dtab[n * NQ + i], Din = Dtab[i * NQ + n];
#pragma unroll
                        for (int d = 0; d < DIM; ++d)
                            m[d] = Dni * lb[d] - Din * la[d];
                        TP::template flux<SERIES>(law, a, b, m, F);
                    } else {
                        TP::template flux<SERIES>(law, a, b, nullptr, F);
                        wi = S_in[i * NQ + n], wn = S_in[n * NQ + i];
                    }
#pragma unroll
                    for (int s = 0; s < NS; ++s) {
                        acc[i][s] = i == 0 && n == 1 ? wi * F[s] : acc[i][s] + wi * F[s];
                        acc[n][s] = i == 0 ? wn * F[s] : acc[n][s] + wn * F[s];
                    }
                }
            }
        };
        if (rough == 0) {
            pairs(std::integral_constant<int, 1>{});
        } else if (rough == 1) {
            pairs(std::integral_constant<int, 0>{});
        } else {
            // a rolled loop (its indexes are the same on every lane): the
            // accumulators are addressed by weights that are zero elsewhere,
            // by the partner's only where registers allow the outer loop to
            // be unrolled (2-D, Nq = 7, 12321 curved cells, FP64: 75.7 ->
            // 74.1 us a stage; 3-D cells then spill: Nq = 8, 18^3, 136 ->
            // 155 us without a logarithm)
            constexpr int UNROLL = DIM == 2 && NQ >= 6 ? NQ : 1;
#pragma unroll
            for (int n = 0; n < NQ; ++n)
#pragma unroll
                for (int s = 0; s < NS; ++s)
                    acc[n][s] = R(0);
#pragma unroll(UNROLL)
            for (int i = 0; i + 1 < NQ; ++i) {
                const Node a = load(i);
                R la[DIM];
                if constexpr (GEN)
                    metric(i, la);
#pragma unroll 1
                for (int n = i + 1; n < NQ; ++n) {
                    const Node b = load(n);
                    R F[NS], wi, wn;
                    if constexpr (GEN) {
                        R lb[DIM], m[DIM];
                        metric(n, lb);
                        const R Dni = Dtab[n * NQ + i], Din = Dtab[i * NQ + n];
#pragma unroll
                        for (int d = 0; d < DIM; ++d)
                            m[d] = Dni * lb[d] - Din * la[d];
                        TP::template flux<-1>(law, a, b, m, F);
                        wi = R(1), wn = R(-1);
                    } else {
                        TP::template flux<-1>(law, a, b, nullptr, F);
                        wi = S_in[i * NQ + n], wn = S_in[n * NQ + i];
                    }
#pragma unroll
                    for (int k = 0; k < NQ; ++k) {
                        if (UNROLL > 1 && k < i)
                            continue;
                        const R w = k == i ? wi : k == n ? wn : R(0);
#pragma unroll
                        for (int s = 0; s < NS; ++s)
                            acc[k][s] = acc[k][s] + w * F[s];
                    }
                }
            }
        }

        if constexpr (!T::EARLY)
            face_states(fresh(t));
#pragma unroll
        for (int side = 0; side < 2; ++side) {
            constexpr int LAST = NQ - 1;
            const int end = side ? LAST : 0;
            R nf[NS], lift;
            R nv[DIM];
            if constexpr (GEN) {
                const GT RV_GLOBAL *sg = sgeo + ((e * NF + 2 * dir + side) * (DIM + 1)) * NL + l;
#pragma unroll
                for (int d = 0; d < DIM; ++d)
                    nv[d] = R(sg[d * NL]);
                lift = R(sg[DIM * NL]);
            } else {
                lift = R(P.winv[end]);
            }
            if constexpr (SF != FLUX_RUSANOV) {
                // twopointflux(q-, q+)' n; on an affine face n = +-e_dir
                static_assert(SF == VF, "the surface flux is Rusanov or the volume form's own");
                R val[TP::NV], F[NS];
                TP::values(law, qp[side], val);
                TP::template flux<-1>(law, load(end), TP::node(law, val), nv, F);
#pragma unroll
                for (int s = 0; s < NS; ++s)
                    nf[s] = GEN || side ? F[s] : -F[s];
            } else if constexpr (GEN) {
                S::nflux_general(law, nv, qm[side], qp[side], nf);
            } else {
                R fm[NS];
                law.flux_row(0, qm[side], fm);
                S::nflux_axis(law, 0, side ? R(1) : R(-1), fm, qm[side], qp[side], nf);
            }
#pragma unroll
            for (int s = 0; s < NS; ++s)
                acc[end][s] = acc[end][s] - lift * nf[s];
        }
        scale = GEN ? R(1) : R(P.affine[e * DIM + dir]);
    } else {
#pragma unroll
        for (int n = 0; n < NQ; ++n)
#pragma unroll
            for (int s = 0; s < NS; ++s)
                acc[n][s] = R(0);
    }

    // ---- the update's loads, in flight through phase 2
    const R a = R(P.a), bdt = R(P.b_dt);
    R *dq = static_cast<R *>(P.dq);
    R *qo = static_cast<R *>(P.q_out);
    double prod = 0.0, pc = 0.0;
    R q[T::ITER][NS], dqo[T::ITER][NS], mji[T::ITER];
    double mj[T::ITER];
#pragma unroll
    for (int it = 0; it < T::ITER; ++it) {
        const int v = t + it * T::THREADS;
        const int cc = v / NP, node = v - cc * NP;
        const int64_t e = cell0 + cc;
        if (v < T::C * NP && e < P.K) {
            const int64_t off = e * (NS * NP) + node;
#pragma unroll
            for (int s = 0; s < NS; ++s)
                q[it][s] = qin[off + s * NP];
            if (P.read_dq) {
#pragma unroll
                for (int s = 0; s < NS; ++s)
                    dqo[it][s] = load_dq<ST>(dq + off + s * NP);
            }
            mji[it] = GEN && sizeof(R) == 4 ? R(P.mji32[e * NP + node])
                      : GEN                 ? R(P.mji[e * NP + node])
                                            : R(1);
            mj[it] = RX ? P.mj[e * NP + node] : 0.0;
        }
    }

    // ---- phase 2: x, then y, then z
    const int lbase = line_of(fresh(t)).lbase;
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
        __syncthreads();
        if (t < T::TASKS && dir == d) {
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                int k = s;
                if constexpr (!GEN) {
                    if (s > 0 && s <= DIM)
                        k = 1 + (s - 1 + d) % DIM;
                }
                R *x = lds + k * CMP + lbase;
#pragma unroll
                for (int n = 0; n < NQ; ++n) {
                    const R v = GEN ? acc[n][s] : scale * acc[n][s];
                    x[n * lstr] = d == 0 ? v : x[n * lstr] + v;
                }
            }
        }
    }
    __syncthreads();

    // ---- phase 3: update
#pragma unroll
    for (int it = 0; it < T::ITER; ++it) {
        const int v = t + it * T::THREADS;
        const int cc = v / NP, node = v - cc * NP;
        const int64_t e = cell0 + cc;
        if (v < T::C * NP && e < P.K) {
            const int64_t off = e * (NS * NP) + node;
            const R *x = lds + cc * T::CS + node + (PR - NQ) * (node / NQ);
            R k[NS];
#pragma unroll
            for (int s = 0; s < NS; ++s)
                k[s] = GEN ? mji[it] * x[s * CMP] : x[s * CMP];
            if constexpr (RX) {
                // the dEta term v(q) . k (odesolvers.jl:130-134)
                double xd[NS], kd[NS];
#pragma unroll
                for (int s = 0; s < NS; ++s) {
                    xd[s] = (double)q[it][s];
                    kd[s] = (double)k[s];
                }
                double w;
                if constexpr (DIM == 3)
                    w = law_entropy_dot_3d<LAW>(xd, kd, P.gamma);
                else
                    w = law_entropy_dot<LAW, DIM>(xd, kd, P.gamma);
                comp_add(prod, pc, mj[it] * w, 0.0);
            }
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                const R val = P.read_dq ? a * dqo[it][s] + k[s] : k[s];
                store_out<ST>(val, dq + off + s * NP);
                if (P.write_q)
                    store_out<ST>(R(q[it][s] + bdt * val), qo + off + s * NP);
            }
        }
    }
    if constexpr (RX)
        store_product<T::THREADS>(P, prod, pc);
}

// A lane per node, which evaluates the fluxes with its dim (Nq - 1) line
// partners itself: each pair twice, but in short code, with no sums to move
// between directions and one barrier.
template <int DIM, int NQ, int LAW, typename R, int GEO, int VF, int SF, bool RX, int ST>
__device__ __forceinline__ void fd_stage_node(const StageParams &P)
{
    using T = FD<DIM, NQ, LAW, R, GEO, VF, SF>;
    using S = typename T::S;
    using TP = typename T::TP;
    constexpr int NS = T::NS, NP = T::NP, NL = T::NL, NF = T::NF, NV = TP::NV;
    constexpr bool GEN = T::GEN;
    // advection on curved cells: a node's u . l_d, so that a pair reads its
    // partner's from LDS and not the partner's metric terms from memory (curved
    // 24^3 cells of Nq = 6, FP64: 213 -> 141 us a stage)
    constexpr bool UL = GEN && TP::ADV;
    __shared__ R lds[NV + (UL ? DIM : 0)][T::NODE_THREADS];
    const int t = threadIdx.x;
    const int c = t / NP, node = t - c * NP;
    const int64_t e = xcd_remap(blockIdx.x, P.blocks) * T::NODE_C + c;
    const bool active = c < T::NODE_C && e < P.K;
    const Law<DIM, LAW, R> law(P);
    const R *qin = static_cast<const R *>(P.q_in);
    R *dq = static_cast<R *>(P.dq);
    R *qo = static_cast<R *>(P.q_out);
    const int64_t off = e * (NS * NP) + node;
    const int ijk[3] = {node % NQ, DIM > 1 ? (node / NQ) % NQ : 0, DIM > 2 ? node / (NQ * NQ) : 0};
    constexpr bool G32 = GEN && DIM > 1 && sizeof(R) == 4;
    using GT = typename std::conditional<G32, float, double>::type;
    const GT RV_GLOBAL *vgeo, *sgeo;
    if constexpr (G32)
        vgeo = P.vgeo32, sgeo = P.sgeo32;
    else
        vgeo = P.vgeo, sgeo = P.sgeo;

    // the node's own loads, and the neighbour states of the faces it lies on
    // (one per direction: Nq > 1)
    R q[NS], x[NV], qp[DIM][NS], dqo[NS], mji = R(1), ul[DIM];
    double mj = 0.0;
    bool on_face[DIM];
    int side[DIM], m[DIM];
    if (active) {
        FaceRec rec[DIM];
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
            side[d] = ijk[d] == NQ - 1;
            on_face[d] = ((P.dir_mask >> d) & 1) && (side[d] || ijk[d] == 0);
            m[d] = DIM == 1   ? 0
                   : DIM == 2 ? ijk[1 - d]
                   : d == 0   ? ijk[1] + NQ * ijk[2]
                   : d == 1   ? ijk[0] + NQ * ijk[2]
                              : ijk[0] + NQ * ijk[1];
            if (on_face[d])
                rec[d] = P.faces[e * NF + 2 * d + side[d]];
        }
#pragma unroll
        for (int s = 0; s < NS; ++s)
            q[s] = qin[off + s * NP];
        if (P.read_dq) {
#pragma unroll
            for (int s = 0; s < NS; ++s)
                dqo[s] = load_dq<ST>(dq + off + s * NP);
        }
        if constexpr (GEN)
            mji = G32 ? R(P.mji32[e * NP + node]) : R(P.mji[e * NP + node]);
        if constexpr (RX)
            mj = P.mj[e * NP + node];
        TP::values(law, q, x);
#pragma unroll
        for (int k = 0; k < NV; ++k)
            lds[k][t] = x[k];
        if constexpr (UL) {
#pragma unroll
            for (int d = 0; d < DIM; ++d) {
                const int64_t g = ((e * DIM + d) * DIM) * NP + node;
                ul[d] = law.u[0] * R(vgeo[g]);
#pragma unroll
                for (int j = 1; j < DIM; ++j)
                    ul[d] = ul[d] + law.u[j] * R(vgeo[g + j * NP]);
                lds[NV + d][t] = ul[d];
            }
        }
#pragma unroll
        for (int d = 0; d < DIM; ++d)
            if (on_face[d]) {
                int64_t o = off;  // a self-mapped face: q+ = q-
                if (rec[d].x >= 0)
                    o = (int64_t)rec[d].x * (NS * NP) +
                        face_node<DIM, NQ>(rec[d].y & 7,
                                           orient_node<DIM, NQ>((rec[d].y >> 3) & 7, m[d]));
                else if (rec[d].x == FACE_EXPLICIT)
                    o = P.explicit_idx[(int64_t)rec[d].y + m[d]];
#pragma unroll
                for (int s = 0; s < NS; ++s)
                    qp[d][s] = qin[o + s * NP];
            }
    }
    __syncthreads();
    double prod = 0.0, pc = 0.0;
    if (active) {
        const typename TP::Node a = TP::node(law, x);
        const R *tab = static_cast<const R *>(P.fdtab);
        R k[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s)
            k[s] = R(0);
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
            if (!((P.dir_mask >> d) & 1))
                continue;
            // the line's direction first (affine cells form component 0)
            auto turned = [&](const typename TP::Node &b) {
                typename TP::Node r = b;
                if constexpr (!GEN) {
#pragma unroll
                    for (int j = 0; j < DIM; ++j)
                        r.u[j] = b.u[(d + j) % DIM];
                }
                return r;
            };
            Law<DIM, LAW, R> lawd = law;
            if constexpr (!GEN) {
#pragma unroll
                for (int j = 0; j < DIM; ++j)
                    lawd.u[j] = law.u[(d + j) % DIM];
            }
            const typename TP::Node ad = turned(a);
            const int i = ijk[d];
            const int stride = d == 0 ? 1 : d == 1 ? NQ : NQ * NQ;
            const int64_t g = ((e * DIM + d) * DIM) * NP + node;
            R la[DIM], kd[NS];
            if constexpr (GEN && !UL) {
#pragma unroll
                for (int j = 0; j < DIM; ++j)
                    la[j] = R(vgeo[g + j * NP]);
            }
#pragma unroll
            for (int s = 0; s < NS; ++s)
                kd[s] = R(0);
            // (two partners in flight: a wave's chain is what small grids wait for)
#pragma unroll 2
            for (int it = 0; it < NQ - 1; ++it) {
                R y[NV], F[NS], mv[DIM], w = R(1);
                const int n = it + (it >= i);
                const int to = (n - i) * stride;
#pragma unroll
                for (int j = 0; j < NV; ++j)
                    y[j] = lds[j][t + to];
                if constexpr (GEN) {
                    const R *D = tab + NQ * NQ;
                    const R Dni = D[n * NQ + i], Din = D[i * NQ + n];
                    if constexpr (UL) {
                        F[0] = R(0.5) * (Dni * lds[NV + d][t + to] - Din * ul[d]) * (ad.rho + y[0]);
                    } else {
#pragma unroll
                        for (int j = 0; j < DIM; ++j)
                            mv[j] = Dni * R(vgeo[g + to + j * NP]) - Din * la[j];
                    }
                } else {
                    w = tab[i * NQ + n];
                }
                if constexpr (!UL)
                    TP::template flux<-2>(lawd, ad, turned(TP::node(law, y)), mv, F);
#pragma unroll
                for (int s = 0; s < NS; ++s)
                    kd[s] = kd[s] + w * F[s];
            }
            if (on_face[d]) {
                R nf[NS], nv[DIM], lift;
                if constexpr (GEN) {
                    const GT RV_GLOBAL *sg =
                        sgeo + ((e * NF + 2 * d + side[d]) * (DIM + 1)) * NL + m[d];
#pragma unroll
                    for (int j = 0; j < DIM; ++j)
                        nv[j] = R(sg[j * NL]);
                    lift = R(sg[DIM * NL]);
                } else {
                    lift = R(P.winv[i]);
                }
                // the states with the direction's momentum first (affine cells)
                R qm[NS], qq[NS];
#pragma unroll
                for (int s = 0; s < NS; ++s) {
                    const int o = GEN || TP::ADV || s == 0 || s > DIM ? s : 1 + (d + s - 1) % DIM;
                    qm[s] = q[o];
                    qq[s] = qp[d][o];
                }
                if constexpr (SF != FLUX_RUSANOV) {
                    R y[NV], F[NS];
                    TP::values(lawd, qq, y);
                    TP::template flux<-2>(lawd, ad, TP::node(lawd, y), nv, F);
#pragma unroll
                    for (int s = 0; s < NS; ++s)
                        nf[s] = GEN || side[d] ? F[s] : -F[s];
                } else if constexpr (GEN) {
                    S::nflux_general(lawd, nv, qm, qq, nf);
                } else {
                    R fm[NS];
                    lawd.flux_row(0, qm, fm);
                    S::nflux_axis(lawd, 0, side[d] ? R(1) : R(-1), fm, qm, qq, nf);
                }
#pragma unroll
                for (int s = 0; s < NS; ++s)
                    kd[s] = kd[s] - lift * nf[s];
            }
            const R scale = GEN ? R(1) : R(P.affine[e * DIM + d]);
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                const int o = GEN || TP::ADV || s == 0 || s > DIM ? s : 1 + (d + s - 1) % DIM;
                k[o] = k[o] + scale * kd[s];
            }
        }
        const R ca = R(P.a), bdt = R(P.b_dt);
        if constexpr (GEN) {
#pragma unroll
            for (int s = 0; s < NS; ++s)
                k[s] = mji * k[s];
        }
        if constexpr (RX) {
            // the dEta term v(q) . k (odesolvers.jl:130-134)
            double xd[NS], kd[NS];
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                xd[s] = (double)q[s];
                kd[s] = (double)k[s];
            }
            if constexpr (DIM == 3)
                prod = mj * law_entropy_dot_3d<LAW>(xd, kd, P.gamma);
            else
                prod = mj * law_entropy_dot<LAW, DIM>(xd, kd, P.gamma);
        }
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const R val = P.read_dq ? ca * dqo[s] + k[s] : k[s];
            store_out<ST>(val, dq + off + s * NP);
            if (P.write_q)
                store_out<ST>(R(q[s] + bdt * val), qo + off + s * NP);
        }
    }
    if constexpr (RX)
        store_product<T::NODE_THREADS>(P, prod, pc);
}

template <int DIM, int NQ, int LAW, typename R, int GEO, int VF, int SF>
constexpr int fd_waves_per_simd()
{
    return sizeof(R) == 8 ? (GEO == GEO_GENERAL && NQ >= 6 ? 2 : 3) : 4;
}

// (RX: the relaxation stage)
template <int DIM, int NQ, int LAW, typename R, int GEO, int VF, int SF, bool RX, int ST>
__global__ void __launch_bounds__((FD<DIM, NQ, LAW, R, GEO, VF, SF>::THREADS))
    __attribute__((amdgpu_waves_per_eu(fd_waves_per_simd<DIM, NQ, LAW, R, GEO, VF, SF>())))
        dg_fd_line_kernel(const StageParams P)
{
    fd_stage<DIM, NQ, LAW, R, GEO, VF, SF, RX, ST>(P);
}

template <int DIM, int NQ, int LAW, typename R, int GEO, int VF, int SF, bool RX, int ST>
__global__ void __launch_bounds__((FD<DIM, NQ, LAW, R, GEO, VF, SF>::NODE_THREADS))
    dg_fd_node_kernel(const StageParams P)
{
    fd_stage_node<DIM, NQ, LAW, R, GEO, VF, SF, RX, ST>(P);
}

template <int DIM, int NQ, int LAW, typename R, int GEO, int VF, int SF, bool RX, int ST>
int launch_fd_st(const StageParams &P, void *stream)
{
    using T = FD<DIM, NQ, LAW, R, GEO, VF, SF>;
    if constexpr (fd_has_line_kernel(DIM, NQ, LAW, (int)sizeof(R), VF)) {
        if (fd_by_line(DIM, NQ, LAW, (int)sizeof(R), VF, P.K)) {
            return launch_stage(&dg_fd_line_kernel<DIM, NQ, LAW, R, GEO, VF, SF, RX, ST>,
                                (P.K + T::C - 1) / T::C, T::THREADS / 64, 0, stream, P);
        }
    }
    return launch_stage(&dg_fd_node_kernel<DIM, NQ, LAW, R, GEO, VF, SF, RX, ST>,
                        (P.K + T::NODE_C - 1) / T::NODE_C, T::NODE_THREADS / 64, 0, stream, P);
}

template <int DIM, int NQ, int LAW, typename R, int GEO, int VF, int SF, bool RX>
int launch_fd(const StageParams &P, void *stream, int)
{
    if (P.K <= 0)
        return 0;
    if constexpr (form_streams(DIM, NQ, LAW, sizeof(R), GEO, VF)) {
        if (P.streaming)
            return launch_fd_st<DIM, NQ, LAW, R, GEO, VF, SF, RX, 1>(P, stream);
    }
    return launch_fd_st<DIM, NQ, LAW, R, GEO, VF, SF, RX, 0>(P, stream);
}

template <int NQ, int LAW, int VF, int SF, bool RX>
StageLauncher pick_geo(const KernelKey &k)
{
    using R = FD_REAL;
    return k.geo == GEO_GENERAL ? &launch_fd<FD_DIM, NQ, LAW, R, GEO_GENERAL, VF, SF, RX>
                                : &launch_fd<FD_DIM, NQ, LAW, R, GEO_AFFINE, VF, SF, RX>;
}

// surface flux: Rusanov, or the volume form's own two-point flux; the fused
// relaxation stage is built for the latter (the entropy-conservative pairing)
template <int NQ, int LAW, int VF>
StageLauncher pick_surface(const KernelKey &k)
{
    if (k.flux == FLUX_RUSANOV)
        return k.relax ? nullptr : pick_geo<NQ, LAW, VF, FLUX_RUSANOV, false>(k);
    if (k.flux == VF)
        return k.relax ? pick_geo<NQ, LAW, VF, VF, true>(k) : pick_geo<NQ, LAW, VF, VF, false>(k);
    return nullptr;
}

template <int NQ>
StageLauncher pick_fd(const KernelKey &k)
{
    if constexpr (IPow<NQ, FD_DIM>::v > 512) {
        return nullptr;
    } else {
        if (k.law == LAW_ADVECTION)
            return k.vflux == FLUX_CENTRAL ? pick_surface<NQ, LAW_ADVECTION, FLUX_CENTRAL>(k)
                                           : nullptr;
        if (k.vflux == FLUX_CENTRAL)
            return pick_surface<NQ, LAW_EULER, FLUX_CENTRAL>(k);
        if (k.vflux == FLUX_EC)
            return pick_surface<NQ, LAW_EULER, FLUX_EC>(k);
        return nullptr;
    }
}

}  // namespace

StageLauncher FD_FN(const KernelKey &k)
{
    if (k.dim != FD_DIM || k.real_bytes != (int)sizeof(FD_REAL))
        return nullptr;
    switch (k.nq) {
    case 2: return pick_fd<2>(k);
    case 3: return pick_fd<3>(k);
    case 4: return pick_fd<4>(k);
    case 5: return pick_fd<5>(k);
    case 6: return pick_fd<6>(k);
    case 7: return pick_fd<7>(k);
    case 8: return pick_fd<8>(k);
    default: return nullptr;
    }
}

}  // namespace rv
