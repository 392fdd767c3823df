// Internal definitions shared by the host API and the kernel instantiation units.
#pragma once

#include <cstdint>
#include <string>

namespace rv {

enum LawId : int { LAW_ADVECTION = 1, LAW_EULER = 2 };
enum GeoId : int { GEO_AFFINE = 1, GEO_GENERAL = 2 };
enum FluxId : int { FLUX_RUSANOV = 1, FLUX_CENTRAL = 2, FLUX_EC = 3 };

// Per-face neighbour record, one per (face, cell):
//   x >= 0 : neighbour cell; y = neighbour face | orientation << 3
//   x == -1: q+ = q- (boundary code != 0 with the identity boundary state,
//            or a self-mapped face: Raven's non-conforming / ghost faces)
//   x == -2: explicit per-node offsets; y = index of the face's first entry
//            in the explicit table (cell offsets e*Ns*Np + node, int64)
constexpr int FACE_SELF = -1;
constexpr int FACE_EXPLICIT = -2;

struct FaceRec {
    int32_t x;
    int32_t y;
};

// Device code reads the arrays below through global-memory (address space
// 1) pointers, also when a StageParams comes out of a device table (batches):
// a pointer loaded from memory is otherwise a generic one, compiled to flat
// loads that also count against the LDS wait counter.  The host pass sees
// plain pointers; the layout is the same.
#if defined(__HIP_DEVICE_COMPILE__)
#define RV_GLOBAL __attribute__((address_space(1)))
#else
#define RV_GLOBAL
#endif

// A host-side device pointer as the parameter structs hold it.
template <typename T>
inline T RV_GLOBAL *as_global(T *p)
{
    return (T RV_GLOBAL *)p;
}

// Arguments of one fused DG stage launch.  Pointers are device pointers.  What the
// affine weak form reads comes first, in two 64-byte lines of the (cold) scalar
// cache.
struct StageParams {
    int64_t K;            // cells
    const void RV_GLOBAL *q_in;  // state read (R)
    void RV_GLOBAL *q_out;       // state written (R), nullptr in RHS mode
    void RV_GLOBAL *dq;          // register (R)
    double a;             // dq = a*dq + L
    double b_dt;          // q_out = q_in + b_dt*dq
    // (fields of one word: batches read them through a table, where the scalar unit
    // loads words and the vector unit anything shorter, for branches to wait for)
    uint32_t read_dq : 1;    // load dq (a != 0 or increment)
    uint32_t write_q : 1;    // stage mode
    uint32_t streaming : 1;  // dq and q_out through L2 as streaming (non-temporal) accesses
    uint32_t dir_mask : 8;   // active directions (bit d)
    uint32_t unused : 21;
    // the launch's own shape (launch_stage): workgroups and waves in each.  The
    // kernels read it here, with the rest, and not through blockDim and gridDim,
    // which the runtime puts behind the arguments: two more lines to fetch
    uint32_t blocks;
    int32_t wpb, pad;
    const FaceRec RV_GLOBAL *faces;        // (2dim, K)
    const int64_t RV_GLOBAL *explicit_idx; // explicit face-node offsets
    // affine geometry: per cell, per direction: dRdX[d,d] (FP64)
    const double RV_GLOBAL *affine;        // (K, dim)
    // operators (FP64, device)
    const double RV_GLOBAL *Dw;    // [i*Nq + n] = D[n,i] w_n / w_i  (affine)
    const double RV_GLOBAL *winv;  // [i] = 1/w_i
    double gamma;
    double u[3];
    const double RV_GLOBAL *Dt;    // [i*Nq + n] = D[n,i]            (general)
    // general geometry (FP64): wJ*dRdX rows, MJI, face normals and wsJ
    const double RV_GLOBAL *vgeo;  // (K, dim, dim, Np): [e][d][c][node] = wJ*dRdX[d,c]
    const double RV_GLOBAL *mji;   // (K, Np)
    const double RV_GLOBAL *mj;    // (K, Np) = wJ
    const double RV_GLOBAL *sgeo;  // (K, 2dim, dim+1, Nfp): n_c ..., wsJ
    // FP32 handles, 2-D and 3-D general cells: vgeo, mji, sgeo and (for the 3-D column
    // kernel) mj rounded to FP32 once (the stage kernels round every use of them to the state type,
    // so reading these gives the same results with half the geometry bytes)
    const float RV_GLOBAL *vgeo32;
    const float RV_GLOBAL *mji32;
    const float RV_GLOBAL *sgeo32;
    const float RV_GLOBAL *mj32;
    // flux differencing, in the state's type: [i*Nq + n] = D[n,i] w_n / w_i - D[i,n]
    // (affine), then [i*Nq + n] = D[i,n] (general)
    const void RV_GLOBAL *fdtab;
    // relaxation stage (the flux-differencing kernels built for it): dq = a dq + k
    // with k = L(q_in) accumulated alone, and each workgroup stores
    // sum MJ v(q_in) . k over its nodes at eprod[workgroup]
    double RV_GLOBAL *eprod;
    // mortar updates the 3-D column kernel adds after its stores (nullptr:
    // none): per cell its slot in mdelta or -1, per (cell, face) the face
    // kind, and the per-(slot, face) updates of mortar_face_kernel
    const int32_t RV_GLOBAL *mslot;
    const int32_t RV_GLOBAL *mkind;
    const void RV_GLOBAL *mdelta;
};

// Whether a stage larger than the caches streams dq and q_out past them
// (StageParams::streaming).  A launch writes a cell's states in pieces: the
// weak form Nq^2 values (2-D a cell, 3-D a plane), flux differencing a cell.
// Streamed pieces that end inside a 128-byte line reach HBM as partial writes,
// where the caches would have joined them; one state per cell (advection)
// leaves no gaps between the cells.  us per Euler stage, streamed / not: 3-D Nq = 8
// FP64 28^3 348 / 389, Nq = 4 FP64 46^3 196 / 242, but Nq = 5 FP64 44^3 594 /
// 448, FP32 412 / 272, Nq = 7 FP32 32^3 316 / 256; 2-D Nq = 8 FP64 390^2 274 /
// 286, Nq = 4 FP32 760^2 198 / 167, Nq = 5 FP64 620^2 356 / 318; entropy-
// conservative form, 2-D Nq = 5 FP64 620^2 385 / 351, curved 3-D Nq = 5 FP32
// 40^3 380 / 367.  On 3-D affine cells whole 32-byte sectors are enough up to
// about 30^3 cells of Nq = 6 and cost little beyond (FP64 30^3 227 / 241, 38^3 474 /
// 462; not curved ones: 394 / 377, 794 / 729), and for flux differencing any cell
// (Nq = 5 FP64 40^3 376 / 402).
constexpr bool stage_streams(int dim, int nq, int law, int real_bytes, int geo, int vflux)
{
    if (law == LAW_ADVECTION)
        return true;
    const bool brick3 = dim == 3 && geo == GEO_AFFINE;
    const int piece = (dim == 1 ? nq : dim == 3 && vflux ? nq * nq * nq : nq * nq) * real_bytes;
    return piece % (brick3 && vflux ? 1 : brick3 ? 32 : 128) == 0;
}

// The Infinity Cache.  A stage touches three states; beyond this in all nothing
// of dq and q_out survives to the next one.
constexpr int64_t CACHE_BYTES = (int64_t)256 << 20;

// ... and weak-form brick launches that stream although their pieces end inside
// lines.  While one state fits the cache, streaming the others leaves q there:
// that is worth the partial writes where pieces are long, and to a right-hand
// side alone, which writes only dq.  us, streamed / not, state in MB: right-hand
// sides 2-D Nq = 6 FP64 122 73.1 / 75.4, 244 135 / 170, Nq = 7 FP64 244 148 / 183,
// Nq = 6 FP32 100 70.3 / 67.5, 122 86 / 96, Nq = 4 FP32 122 83 / 97, 200 134 / 166,
// but 244 215 / 202, Nq = 5 FP64 244 172 / 184, 488 368 / 361, Nq = 3 FP64 100 77.5 /
// 71.3, 155 118 / 135, 244 236 / 212; 3-D Nq = 5 FP64 156 110 / 121, 305 228 / 230,
// 596 458 / 435, Nq = 7 FP64 159 161 / 153; stages 2-D Nq = 6 FP64 122 126 / 132, 244
// 247 / 255, 489 520 / 504, Nq = 5 FP64 244 298 / 281.
constexpr bool resident_streams(int dim, int nq, int law, int geo, int real_bytes, int vflux,
                                bool write_q, int64_t state)
{
    if (law == LAW_ADVECTION || geo != GEO_AFFINE || vflux || dim == 1)
        return false;
    const int piece = nq * nq * real_bytes;
    if (write_q)
        return dim == 2 && piece >= 288 && state <= CACHE_BYTES;
    // (below, q and dq fit the cache together)
    if (20 * state <= 9 * CACHE_BYTES)
        return false;
    if (dim == 2)
        return piece >= 64 && state <= (piece >= 128 ? CACHE_BYTES : CACHE_BYTES / 6 * 5);
    return piece >= 128 && nq <= 6 && (state <= CACHE_BYTES || piece % 16 == 0);
}

// Whether a launch streams, and whether any launch of a form does (its streaming
// variant is then built).
inline bool launch_streams(int dim, int nq, int law, int real_bytes, int geo, int vflux,
                           bool write_q, int64_t state)
{
    return 3 * state > CACHE_BYTES &&
           (stage_streams(dim, nq, law, real_bytes, geo, vflux) ||
            resident_streams(dim, nq, law, geo, real_bytes, vflux, write_q, state));
}
constexpr bool form_streams(int dim, int nq, int law, int real_bytes, int geo, int vflux)
{
    return stage_streams(dim, nq, law, real_bytes, geo, vflux) ||
           resident_streams(dim, nq, law, geo, real_bytes, vflux, false, CACHE_BYTES / 2) ||
           resident_streams(dim, nq, law, geo, real_bytes, vflux, true, 0);
}

// Waves of a workgroup of the 3-D column kernel that packs its cells across
// lanes (dg_plane3.hpp), 1: nothing to gain.
constexpr int plane3_pack_waves(int nq) { return nq == 5 ? 2 : nq == 6 || nq == 7 ? 4 : 1; }

// Whether a launch over K cells packs them.  Packing fills lanes but ties the
// waves of a workgroup together: with one wave per cell and at most 1024 cells
// of Nq = 6 or 2048 of Nq = 7 every cell is resident at once (one or two waves
// per SIMD) and packing only lengthens each wave's chain; beyond the caches, where the waits
// are longest, FP32 and curved cells gain from independent waves too, and
// Nq = 7, whose cells leave few lanes idle, in every form but affine FP64 in
// the caches.  us per Euler stage, packed / one wave per cell: 8^3 cells of
// Nq = 6 FP64 16.4 / 13.0, 12^3 21.3 / 22.5, 20^3 72.1 / 78.8, 38^3 470 / 528, FP32 274 / 258, curved
// FP32 404 / 393, FP64 729 / 789; 7^3 of Nq = 7 FP64 25.0 / 16.8, 12^3 43.7 / 37.8, 17^3 84.6 / 87.5,
// FP32 42.7 / 39.9, curved FP64 146 / 140, 32^3 FP64 549 / 520, curved 921 / 802, FP32
// 256 / 235; Nq = 5 10^3 FP64 12.1 / 14.1, 44^3 FP64 448 / 445, FP32 272 / 260, curved
// FP32 408 / 385, FP64 717 / 698.
inline bool plane3_packed(int nq, int law, int real_bytes, int geo, int64_t K, bool write_q)
{
    if (plane3_pack_waves(nq) == 1)
        return false;
    const int ns = law == LAW_ADVECTION ? 1 : 5;
    const bool large = 3 * K * nq * nq * nq * ns * real_bytes > CACHE_BYTES;
    const bool curved = geo != GEO_AFFINE;
    if (nq == 5)
        return !(large && ((real_bytes == 4 && write_q) || curved));
    if (K <= (nq == 6 ? 1024 : 2048))
        return false;
    // (a right-hand side alone writes less and waits less: FP32 29^3 75.6 / 89.4
    // us, 36^3 137 / 172, 49^3 399 / 445)
    if (nq == 6)
        return !(large && real_bytes == 4 && (write_q || curved));
    return real_bytes == 8 && !curved && !large;
}

// Product slots (StageParams::eprod) the 3-D column kernel's relaxation stage
// writes, one per wave launched: a packed launch has 64 G / Nq^2 cells to a
// workgroup of G waves, the others 64 / Nq^2 cells to a wave and wpb waves to a
// workgroup.
inline int64_t plane3_relax_slots(int nq, int law, int real_bytes, int geo, int64_t K, int wpb)
{
    const int nq2 = nq * nq;
    if (plane3_packed(nq, law, real_bytes, geo, K, true)) {
        const int g = plane3_pack_waves(nq), cpg = 64 * g / nq2;
        return (K + cpg - 1) / cpg * g;
    }
    if (wpb != 1 && wpb != 2 && wpb != 4)
        wpb = 1;
    const int epw = 64 / nq2;
    const int64_t waves = (K + epw - 1) / epw;
    return (waves + wpb - 1) / wpb * wpb;
}

// Default waves per workgroup of a launch over K cells (rv_set_waves_per_block).
// Measured on MI355X for the 3-D column kernel on 32^3 cells of Nq = 8: a fused
// stage is fastest with four for FP64 (0.50 ms against 0.52 ms with one or two)
// and two for FP32 (one, two and four within 2 %); a right-hand side alone with
// one for FP64 (0.36 ms against 0.37 and 0.40 ms) and two for FP32.  Grids of at
// most 1024 waves spread over the CUs (a workgroup of four waves each would leave
// half of them idle): 216 cells of Nq = 8 FP64 15.7 us per stage against 18.4, 343
// of Nq = 7 16.8 against 21.4.
inline int default_waves(int dim, int nq, int real_bytes, int64_t K, bool write_q)
{
    const int epw = nq > 8 ? 1 : 64 / (nq * nq);
    if (dim != 3 || K <= (int64_t)1024 * epw)
        return 1;
    return real_bytes == 4 ? 2 : write_q ? 4 : 1;
}
// ... and of a batch's launch of one kind, whose members have `cells` cells in all:
// what the first member was given (chosen, 0: nothing), else one for FP64 Euler and
// two for the others (the first member's own default would make the launch depend
// on the members' order).  us per step, one / two / four waves: six members of 14^3
// and one of 3^3 cells of Nq = 8 FP64 Euler 1473 / 1494 / 1548, Nq = 7 1205 / 1248 /
// 1445, 4 of 32^3 of Nq = 7 8715 / 8993 / 10993; FP32 Euler 16 of 8^3 of Nq = 6 213 /
// 204 / 203, advection 8 of 20^3 of Nq = 5 275 / 259 / 258; few cells: 3 of 8^3 of
// Nq = 5 FP32 Euler 59 / 67 / 60.
inline int kind_waves(int dim, int nq, int law, int real_bytes, int64_t cells, int chosen)
{
    if (chosen)
        return chosen;
    return law == LAW_EULER && real_bytes == 8 ? 1 : default_waves(dim, nq, 4, cells, true);
}

// Launch the fused stage for one kernel configuration; returns false when no
// kernel is instantiated for it.
using StageLauncher = int (*)(const StageParams &, void *stream, int waves_per_block);

struct KernelKey {
    int dim, nq, law, real_bytes, geo, flux;
    int vflux = 0;  // 0: weak form; else the flux-differencing form's two-point flux
    int relax = 0;  // the fused relaxation stage (StageParams::eprod) of a flux-differencing kernel
};

// Mortar coupling of hanging faces (mortar.hip), launched after a stage.
// One non-conforming face of a mortar cell: its cell e (and slot li in the
// list of mortar cells), face f and partners (hanging: coarse cell, sub-face;
// covered: the 2^(dim-1) fine cells; covered faces come first)
struct MortarPair {
    int64_t e, li;
    int64_t part[4];
    int64_t f;
};

struct MortarParams {
    StageParams stage;       // the stage just launched (states, law, mji)
    int64_t ncells;          // cells with non-conforming faces
    const int64_t RV_GLOBAL *cells;
    // their non-conforming (cell, face) pairs: covered (coarse) sides first,
    // which take longer, then hanging (fine) sides
    int64_t npairs, ncovered;
    const MortarPair RV_GLOBAL *pairs;
    const int32_t RV_GLOBAL *kind;     // (K, 2dim): 0 conforming, 1 hanging, 2 covered
    const int64_t RV_GLOBAL *partner;  // (K, 2dim, 4), see forest_mortars
    const double RV_GLOBAL *sgeo;      // surface geometry with the lift weights kept
    const double RV_GLOBAL *halves;    // tohalves_1d, (2, Nq, Nq) row-major
    void RV_GLOBAL *delta;             // (ncells, 2dim, Ns, Nfp) per-face updates (R)
};
// phase 0: the per-face updates (before the stage kernel); phase 1: adding
// them to dq and q_out (after a stage kernel that does not add them itself)
using MortarLauncher = int (*)(const MortarParams &, void *stream, int phase);
MortarLauncher find_mortar_launcher(int dim, int nq, int law, int real_bytes, int flux);

// Flux-differencing kernels (fluxdiff.hip): whole cells per workgroup.  The
// line kernel (2-D and 3-D): a lane per line of a cell (dim Nq^(dim-1) lines
// each); 2-D fills one wave, 3-D takes few cells that leave few idle lanes in
// 2 to 4 waves (Nq = 2 to 8: 192/192, 189/192, 192/192, 225/256, 108/128,
// 147/192, 192/192 lanes; at Nq = 5, 5 cells in 6 waves leave 9 lanes idle
// but took 110 us against 83 us per FP64 stage of 24^3 cells: two such
// workgroups fit a CU and wait together).
constexpr int fd_cells_per_workgroup(int dim, int nq)
{
    return dim == 2 ? 32 / nq : nq == 2 ? 16 : nq == 3 ? 7 : nq == 4 ? 4 : nq == 5 ? 3 : 1;
}
// The node kernel: a lane per node, in 1-D one wave, else up to 256 lanes or
// one cell.
constexpr int fd_node_cells(int dim, int nq)
{
    int np = 1;
    for (int d = 0; d < dim; ++d)
        np *= nq;
    const int most = dim == 1 ? 64 : 256;
    return np >= most ? 1 : most / np;
}
// The line kernel's forms.  Not 2-D Nq = 2 in FP32: two lines of one pair each
// are less work than the sums that move between directions, and twice as many
// lanes hide the faces' reads (us per stage, line / node: 387^2 cells Rusanov
// 26.2 / 16.1, own flux 18.5 / 16.3, curved 33.0 / 18.0 and 24.8 / 17.4; 1414^2 291
// / 192; in FP64 224^2 own flux 8.4 / 9.3, 612^2 Rusanov 52.5 / 47.3).
constexpr bool fd_has_line_kernel(int dim, int nq, int law, int real_bytes, int vflux)
{
    return dim > 1 && law == LAW_EULER && vflux == FLUX_EC &&
           !(dim == 2 && nq == 2 && real_bytes == 4);
}
// Whether a launch over K cells takes the line kernel: from about one wave per
// SIMD of the device on (FP64; FP32, whose chains are shorter, from 1.75).
// Below, the chain of one wave and the fetch of its code are all that counts
// (the line kernel's unrolled pairs are about 15 KB a wave); above, the line
// kernel's half as many fluxes do.  Measured, us per Euler stage, line / node
// (waves of the line kernel): 2-D Nq = 8 FP64, 40^2 cells (400) 20.5 / 12.5,
// 100^2 (2500) 25.1 / 41.5; 3-D Nq = 6 FP64, 8^3 (1024) 24.6 / 21.3, 10^3
// (2000) 26.5 / 33.1; 3-D Nq = 8, 8^3 (1536) FP64 39.0 / 48.9, FP32 23.0 /
// 20.7; 24^3 FP64 315 / 658, FP32 185 / 260.
inline bool fd_by_line(int dim, int nq, int law, int real_bytes, int vflux, int64_t K)
{
    if (!fd_has_line_kernel(dim, nq, law, real_bytes, vflux))
        return false;
    const int c = fd_cells_per_workgroup(dim, nq);
    const int waves = (c * dim * (dim == 2 ? nq : nq * nq) + 63) / 64;
    return (K + c - 1) / c * waves >= (real_bytes == 8 ? 1152 : 1792);
}
inline int64_t fd_workgroups(int dim, int nq, int law, int real_bytes, int vflux, int64_t K)
{
    const int c = fd_by_line(dim, nq, law, real_bytes, vflux, K) ? fd_cells_per_workgroup(dim, nq)
                                                                 : fd_node_cells(dim, nq);
    return (K + c - 1) / c;
}

// Entropy passes of the relaxation LSRK step (entropy.hip).  Each pass runs
// RELAX_BLOCKS workgroups over contiguous node ranges and leaves per workgroup
// two Neumaier sums (value, compensation) in partial[4*block ..]: the entropy
// integral sum MJ eta(x) at +0 and the entropy product sum MJ v(x).k at +2.
enum RelaxMode : int {
    RELAX_ETA = 0,      // x = q; eta sum; q0 = q when q0 is given (the step's copy)
    RELAX_PRODUCT = 1,  // x = q (p of entropyproduct); product sum with k
    RELAX_STAGE = 2,    // x = q; product with k; dq = a dq + k; q += b dt dq
    RELAX_NEWTON = 3,   // (first: k = qf - q0); q = x = q0 + gamma k; both sums
    RELAX_AXPY = 4      // q = q0 + gamma k; no sums
};
constexpr int RELAX_BLOCKS = 2048;  // 8 workgroups of 4 waves per CU
constexpr int RELAX_THREADS = 256;
struct RelaxParams {
    int mode, law, dim, real_bytes;
    int64_t Np, K;
    double gas_gamma;     // the Euler law's ratio of specific heats
    const double *MJ;     // (K, Np)
    void *q, *k, *dq;     // (K, Ns, Np) states of the handle's precision
    void *q0;             // read by RELAX_NEWTON / RELAX_AXPY, written by RELAX_ETA
    double a, b_dt;       // RELAX_STAGE
    int read_dq;          // RELAX_STAGE: a != 0
    int first;            // RELAX_NEWTON: form k = qf - q0 first
    const void *qf;       // RELAX_NEWTON first: the state after the stages (may be q or k)
    double relax;         // RELAX_NEWTON / RELAX_AXPY: gamma
    double *partial;      // 4 * RELAX_BLOCKS doubles
};
int launch_relax(const RelaxParams &P, void *stream);

// Compensated sums of per-workgroup partials on the device, in a fixed order
// (deterministic): for slot a in [0, nslots) and b in [0, nwhich),
//   out[a * nwhich + b] = sum over i in [0, n) of
//       src[a * slot_stride + b * which_stride + (i / group) * group_stride + i % group].
int launch_slot_sums(const double *src, int64_t n, int nslots, int nwhich, int64_t slot_stride,
                     int64_t which_stride, int group, int64_t group_stride, double *out,
                     void *stream);

// Batched stages (batch.hip): one work-list item per wave's worth of cells of
// one member; `kind` selects the member's (Nq, law, precision) routine.
struct BatchItem {
    int32_t member;
    int32_t kind;
    int64_t cell0;
};
// kind id, and cells and LDS bytes per item of a batch member: [0] in the
// work-list kernel (a wave per item), [1] when its kind launches on its own
// (2-D Nq = 5, 6, 7: a packed workgroup per item); false when the batch
// kernels do not cover (dim, nq, law, precision)
bool batch_kind(int dim, int nq, int law, int real_bytes, int *kind, int cells_per_item[2],
                int slab_bytes[2]);
// waves of the batch kernel resident on the whole device at once
int batch_resident_waves(int dim, int wpb, int slab_bytes, int64_t *waves);
// one persistent launch over the work list (members: device table)
int launch_batch(int dim, const StageParams *members, const BatchItem *items, int64_t nitems,
                 int64_t nwaves, int slab_bytes, int wpb, void *stream);
// one launch for the items [first, first + count) of a single kind
int launch_batch_kind(int dim, int kind, const StageParams *members, const BatchItem *items,
                      int64_t first, int64_t count, int slab_bytes, int wpb, void *stream);

// Host-side grid generation (host_grid.cpp): Raven's brick GridManager +
// generate restated for uniform bricks, and the LobattoCell 1-D operators.
struct BrickSpec {
    int dim, nq, level;
    int n[3], periodic[3];
    double lo[3], hi[3];
};
int64_t brick_numcells(const BrickSpec &b);
// tree and quadrant coordinates (K x dim), p4est brick order
void brick_quadrants(const BrickSpec &b, int32_t *tree, int32_t *quad);
// vertex coordinates of the coarse brick along d (n[d]+1 values, correctly
// rounded lattice lo + (hi-lo)*i/n like Julia's range(lo, stop=hi, length=n+1))
void brick_vertices(const BrickSpec &b, int d, double *v);
void lobatto_operators(int nq, double *x, double *w, double *D);
// tohalves_1d (lobattocells.jl:15-16): interpolation from the GLL points to
// the GLL points of the lower / upper half, row-major [a][b] = l_b(y_a)
void lobatto_halves(int nq, double *lower, double *upper);
// full Raven-layout arrays (any pointer may be null)
void brick_arrays(const BrickSpec &b, double *points, double *metrics, double *surf,
                  int64_t *vmapM, int64_t *vmapP, int64_t *bc);
int64_t brick_dtoc(const BrickSpec &b, int64_t *dtoc);
// per-cell diagonal of dRdX (K x dim) and neighbour cell per face (K x 2dim,
// -1 on non-periodic boundaries) without per-node arrays
void brick_affine(const BrickSpec &b, double *drdx, double *J);
void brick_neighbours(const BrickSpec &b, int64_t *nbr);

// Adaptive brick forest (forest.cpp): leaves after adapt! with 2:1 balance.
struct Forest;
Forest *forest_new(const BrickSpec &b);
void forest_free(Forest *f);
Forest *forest_clone(const Forest *f);
// per (cell, face), e * 2dim + f: the conforming neighbour (-1 when none),
// the face kind (0 conforming or boundary, 1 hanging, 2 covered) and the
// boundary code; any pointer may be null
void forest_faces(const Forest *f, int64_t *nbr, int32_t *kind, int64_t *bc);
BrickSpec forest_spec(const Forest *f);
int64_t forest_size(const Forest *f);
// adapt! with Raven's flags (0x00 coarsen, 0x10 refine, anything else keeps),
// flags overwritten with the outcome; -1 when a refined leaf would pass the
// finest level
int forest_adapt(Forest *f, uint8_t *flags);
// tree lattice coordinates (K x dim), levels (K), coordinates inside the tree
// at each leaf's level (K x dim); any pointer may be null
void forest_cells(const Forest *f, int32_t *tree, int32_t *level, int32_t *quad);
// points (Np, dim, K), vmapM / vmapP (2dim*Nfp, K) 1-based, boundary codes
// (2dim, K) and face kinds (2dim, K: 0 conforming or boundary, 1 hanging on a
// coarser neighbour, 2 covered by finer neighbours); any pointer may be null
void forest_arrays(const Forest *f, int nq, double *points, int64_t *vmapM, int64_t *vmapP,
                   int64_t *bc, int32_t *kind);
// partners of the non-conforming faces, (K, 2dim, 4): a hanging face holds
// (coarse cell, sub-face index s1 + 2*s2, -1, -1); a covered face holds the
// 2^(dim-1) finer cells in sub-face order; conforming faces hold -1
void forest_mortars(const Forest *f, int64_t *partner);
// Raven's non-conforming face tables per face group g < dim: the number of
// distinct non-conforming interfaces and of non-conforming (cell, face) pairs
void forest_nc_counts(const Forest *f, int64_t *nunique, int64_t *nfaces);
// vmapNC[g] (Nfp, 1 + 2^(dim-1), nunique[g]) 1-based, nctoface[g] (2,
// nunique[g]), nctypes[g] and ncids[g] (nfaces[g], ncids 1-based); any
// group's pointers may be null
void forest_nctables(const Forest *f, int nq, int64_t *const *vmapNC, int8_t *const *nctoface,
                     int8_t *const *nctypes, int64_t *const *ncids);
// face kinds and partners (as forest_arrays / forest_mortars give them) from
// Raven's vmapNC / nctoface; 0, -1 (an index out of range) or -2 (a table that
// is not an aligned face pairing)
int mortars_from_nctables(int dim, int nq, int64_t K, const int64_t *nunique,
                          const int64_t *const *vmapNC, const int8_t *const *nctoface,
                          int32_t *kind, int64_t *partner);
// continuous numbering of the forest's nodes, hanging nodes included, as
// Raven's dtoc (1-based, first appearance); returns the number of continuous
// nodes
int64_t forest_dtoc(const Forest *f, int nq, int64_t *dtoc);

}  // namespace rv
