// kernels.hip -- CDNA4 (gfx950) kernels of one low-storage RK3 stage of the DG-SEM wave solver.
//
// Data layout in HBM (structure of arrays, element-major, elements in Hilbert-curve order):
//   q      [K][3][(N+1)^2]   state (p, u, v), reference node order i*(N+1)+j
//   g      [K][3][(N+1)^2]   RK register, alive within a step only; the stage kernel's own order
//                            within each workgroup tile (see stage_kernel)
//   wave   [K][4][N+1]       outgoing characteristics at the side points of the current state (two
//                            buffers, ping-pong)
//   trace  [K][4][3][N+1]    element traces of the current state (two buffers), of the sides that
//                            need all three (see stage_kernel)
//   verts  [K][4][2]         element vertices (metrics are recomputed from them per node)
//   side_nb[K][4]            neighbour element*4+side, or -(1+index) into the BcSide records
//
// One fused stage kernel replaces the reference's per-phase kernels of one stage
// (include/solvers/Solver2D_t.tcu:45-52): a workgroup stages the (N+1)^2 tiles of EPB elements in
// LDS, computes the upwind flux on its 4 sides from its own and the neighbours' outgoing
// characteristics, applies volume + lift, the RK update, and writes the characteristics of the
// updated state for the next stage. Per element and stage HBM traffic is the state and RK register
// (read + write), and the characteristics of its sides (one value a point, read and written).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <climits>
#include <cmath>
#include <type_traits>

#include "device.hpp"
#include "internal.hpp"

namespace ndg {

template <int N>
struct Shape {
    static constexpr int NF = N + 1;
    static constexpr int NE = NF * NF;
    static constexpr int EPB = NE >= 256 ? 1 : 256 / NE;  // elements per workgroup
    static constexpr int THREADS = ((EPB * NE + 63) / 64) * 64;
};

// The stage's time, which the inflow ghost reads: the step's start time in device memory (so that a
// captured step replays with the time advancing) plus the stage's part of the step; the step's last
// stage leaves the next step's start time. One workgroup of one order group is given `next`.
struct StageClock {
    const double *start;
    double part;   // b_s dt (include/solvers/Solver2D_t.tpp:16, :45-63), rounded on the host
    double *next;  // null but in the step's last stage
    double dt;
    __device__ __forceinline__ double time() const { return *start + part; }
    __device__ __forceinline__ void advance() const {
        if (next && blockIdx.x == 0 && threadIdx.x == 0) *next = *start + dt;
    }
};

// The reference plane wave g(x, t) (include/functions/analytical_solution.tpp:5-11).
__device__ __forceinline__ void plane_wave(double x, double y, double t, double cw, double &p, double &u,
                                           double &v) {
    const double kx = 0.707106781186548, ky = 0.707106781186548, x0 = -0.2, y0 = -0.2;
    const double d = 0.120112240878645;
    const double a = kx * (x - x0) + ky * (y - y0) - cw * t;
    p = exp(-a * a / (d * d));
    u = p * kx;  // the reference's p k / c at c = 1 (and the plane wave of the speed-c system)
    v = p * ky;
}

// The outward normal that the characteristic of side s of element e is formed with: its record's,
// where it has one.
__device__ __forceinline__ void side_normal(const double *verts, const int32_t *side_nb, const BcSide *bc, int64_t e,
                                            int s, double &nx, double &ny) {
    side_geometry(verts + e * 8, s, nx, ny);
    const int32_t cd = side_nb[e * 4 + s];
    if (cd < 0) {
        nx = bc[-1 - cd].nx;
        ny = bc[-1 - cd].ny;
    }
}

// Trace k of side s of one element tile (src/entities/Element2D_t.cpp:86-125): sides 2 and 3
// run counter-clockwise, i.e. reversed with respect to the xi / eta index.
template <int N>
__device__ __forceinline__ double side_trace(const double *tile, const double *lm, const double *lp,
                                             int s, int k) {
    constexpr int NF = N + 1;
    double acc = 0.0;
    if (s == 0) {
#pragma unroll
        for (int j = 0; j < NF; ++j) acc += lm[j] * tile[k * NF + j];
    } else if (s == 1) {
#pragma unroll
        for (int j = 0; j < NF; ++j) acc += lp[j] * tile[j * NF + k];
    } else if (s == 2) {
#pragma unroll
        for (int j = 0; j < NF; ++j) acc += lp[j] * tile[(N - k) * NF + j];
    } else {
#pragma unroll
        for (int j = 0; j < NF; ++j) acc += lm[j] * tile[j * NF + (N - k)];
    }
    return acc;
}

// ---------------------------------------------------------------------------------------------
// Traces and outgoing characteristics (see stage_kernel) of the current state, used after the state
// is set; the stage kernel writes them afterwards.
template <int N>
__global__ void __launch_bounds__(Shape<N>::THREADS)
traces_kernel(const double *__restrict__ verts, const int32_t *__restrict__ side_nb, const BcSide *__restrict__ bc,
              const double *__restrict__ tab, const double *__restrict__ q, double *__restrict__ tr,
              double *__restrict__ w, int64_t K) {
    using S = Shape<N>;
    constexpr int NF = S::NF, NE = S::NE, EPB = S::EPB, T = S::THREADS;
    __shared__ double s_lm[NF], s_lp[NF];
    __shared__ double s_q[EPB * 3 * NE];
    __shared__ double s_n[EPB * 8];  // outward normal per side
    const int tid = threadIdx.x;
    const int64_t e0 = (int64_t)blockIdx.x * EPB;
    const int nel = (int)min<int64_t>(EPB, K - e0);
    for (int r = tid; r < NF; r += T) {  // l(-1) is the reverse of l(+1), as in the stage kernel
        s_lm[r] = tab[NF * NF + NF + N - r];
        s_lp[r] = tab[NF * NF + NF + r];
    }
    const double *qg = q + e0 * 3 * NE;
    for (int r = tid; r < nel * 3 * NE; r += T) s_q[r] = qg[r];
    for (int r = tid; r < nel * 4; r += T) side_normal(verts, side_nb, bc, e0 + r / 4, r % 4, s_n[2 * r], s_n[2 * r + 1]);
    __syncthreads();
    for (int r = tid; r < nel * 4 * NF; r += T) {
        const int el = r / (4 * NF), s = (r / NF) % 4, k = r % NF;
        const double *qe = s_q + el * 3 * NE;
        const double p = side_trace<N>(qe, s_lm, s_lp, s, k), u = side_trace<N>(qe + NE, s_lm, s_lp, s, k),
                     v = side_trace<N>(qe + 2 * NE, s_lm, s_lp, s, k);
        double *to = tr + (e0 + el) * 12 * NF + s * 3 * NF + k;
        to[0] = p;
        to[NF] = u;
        to[2 * NF] = v;
        w[e0 * 4 * NF + r] = p + kWaveSpeed * (u * s_n[8 * el + 2 * s] + v * s_n[8 * el + 2 * s + 1]);
    }
}

// ---------------------------------------------------------------------------------------------
// One fused RK stage. A workgroup is three waves, one per field (p, u, v); lane (element e, line l)
// of the wave for field f handles one (N+1)-point line of that field for EPB = floor(64/(N+1))
// elements. Every field-dependent branch is therefore wave-uniform (a scalar branch, no masked
// lanes), the D^ contractions run in registers, and LDS carries the element tiles:
//   P0  every HBM read of the tile is issued before any is waited on: state tile -> LDS, the
//       thread's RK-register line, and for each side point the outgoing characteristics of the
//       element and of its neighbour -> registers
//   P1  D^ (y_eta f - x_eta g) along the thread's xi line (Solver2D_t.cpp:71-100) and
//       D^ (-y_xi f + x_xi g) along its eta line (:104-133), both from the state tile; then the upwind
//       flux of the side points (boundary_conditions / project_to_faces / calculate_wave_fluxes /
//       project_to_elements, Mesh2D_t.cpp:3731-3935, Solver2D_t.cpp:48-63) and, by wave 2, the side
//       normals and edge Jacobians
//   P2  the lifts; d_xi to LDS
//   P3  eta lines: G = (-d_xi - d_eta)/J, RK update (Solver2D_t.cpp:138-172), the new state to LDS,
//       its traces on sides 0 and 2 from the line in registers
//   P4  coalesced store of q, traces on sides 1 and 3 from the new tile's columns
//   P5  the new outgoing characteristic of every side point, for the next stage.
//
// The upwind flux of a side point needs from the other element only the characteristic that leaves
// it, w = p + u.n with its own outward normal n: on a side shared by two elements the normals are
// opposite, so this is p - u.n in the receiver's normal. One value a point is exchanged instead of
// the three traces: 4 (N+1) values an element are written once and read twice (the element's own
// from the same tile) instead of 12 (N+1) written and read, 7,200 instead of 8,290 bytes an element
// and stage at N = 8. Sides where that is not enough carry a record (code < 0): boundary ghosts are
// built from the element's own traces, read back as the last stage wrote them; a mortar side's flux comes from
// the mortar kernel; a periodic side whose partner does not run parallel to it reads the partner's
// three traces. Elements write the three traces of the sides with a record (and with kTraceAll of
// every side) for these.
//
// What bounds it: HBM at large sizes, the phases' latency at small ones. 512 x 512, N = 8: 316 to 323 us a
// launch over runs, 5.84 to 5.97 TB/s of the 1.89 GB it moves (a plain in-place copy of two streams reaches
// 5.3 to 5.8 here); 421 us and 2.18 GB with the traces exchanged. 512 x 512, N = 4: 116 us (164 us before). 128 x
// 128, N = 8 (in the last-level cache): 24.3 us, 33.2 us before; 16 x 16, N = 6 (29 workgroups): 5.7
// us from launch to launch, 7.0 us before. What made the difference, at N = 8:
//  - the state and the RK register are streamed past the caches (non-temporal, in 16-byte words on
//    whole 128-byte lines) where they are larger than these (stage_flags): 401 -> 324 us at 512 x 512;
//  - D^ out of the scalar loads (LaneTable) and by even and odd parts (contract): 25 us instead of
//    28 us at 128 x 128;
//  - the entries of D^ as DPP operands (rows): 256 x 256, N = 12 in 184 us instead of 189 us, 48 x 48,
//    N = 16 in 19.2 us instead of 20.4 us (and 35 registers fewer), 512 x 512 in 321 us instead of 325 us;
//  - the own traces of a side with a record loaded with the tile, not formed again from its lines:
//    23 x 23, N = 4 with walls, inflow and outflow 5.8 us instead of 6.7 us, 48 x 48, N = 16: 16.6 us
//    instead of 19.2 us;
//  - what the geometry reads after the contractions (side codes, the line's coordinate) loaded with the
//    tile: 256 x 256, N = 12 in 182 us instead of 188 us, 512 x 512 in 317 us instead of 320 us;
//  - no branch inside the line loops and no wait among the loads (a condition on the field in a loop
//    kept each LDS read from overlapping the next: 3,700 cycles for the update of a line, 1,700 now);
//  - five barriers instead of six, LDS for five workgroups a CU instead of four.
//
// RHS_ONLY writes G (the compute_dg_wave_derivative output) and leaves the state alone. MORTAR: the mesh may
// have mortar sides, whose own flux components P2 takes. Meshes without have a kernel without: 128 x 128,
// N = 8 in 24.3 us instead of 25.3 us, 256 x 256, N = 7 in 68.8 us instead of 69.3 us. flags:
// kRkFirst, the step's first stage (a = 0: the RK register is not read); kRkLast, the step's last
// stage, whose RK register no one reads (the next step's first stage overwrites it), so it is not
// stored.
// The new state goes to q_out, which is q for the in-place step (q and q_out are therefore not
// restrict; every value of q a workgroup reads precedes, through barriers, its writes).
// A workgroup takes epb <= EPB consecutive elements (fewer gives more workgroups for a small
// order group); remap != 0 applies the XCD-contiguous block order.
//
// LDS at N = 8 is 31,920 bytes, which the 1,280-byte allocation steps still let fit five times into
// a CU's 160 KB.

// Values per (field, line index) of a workgroup tile in the RK register: whole 128-byte lines for
// the full tiles, whole 16-byte words for the tuner's smaller ones.
template <int N>
__host__ __device__ constexpr int rk_run(int epb) {
    return epb == LineShape<N>::EPB ? (LineShape<N>::EPB * (N + 1) + 15) / 16 * 16 : (epb * (N + 1) + 1) / 2 * 2;
}

// The state tile in LDS: [element][f][i][j] with the row stride padded to an odd number of values,
// so that lanes on consecutive rows fall on different banks (at even N + 1 the unpadded rows of a
// column of lanes share a few banks).
template <int N>
struct StageTile {
    using S = LineShape<N>;
    static constexpr int NFP = S::NF | 1;                       // padded row stride
    static constexpr int NEP = S::NF * NFP;                     // one field of one element
    static constexpr int kFlux = S::EPB * 8 * S::NF;            // (w_L - w_R)/2 and (w_L + w_R)/2 per side point
    static constexpr int QPT = (S::EPB * 3 * S::NE + 15 + 2 * S::T - 1) / (2 * S::T);  // pairs per thread
    // LDS index of value r of a tile in the state's order
    __device__ static __forceinline__ int at(int r) { return NFP == S::NF ? r : r + (int)((unsigned)r / S::NF); }
};

// n values from p with the hardware's bounds check: a load outside [0, n) gives 0, a store outside it
// is dropped, so a tile's loads and stores need no branch for its remainder.
struct Buffer {
    static constexpr int kNonTemporal = 2;  // the instruction's nt bit
    __amdgpu_buffer_rsrc_t rsrc;
    __device__ __forceinline__ Buffer(const double *p, int n)
        : rsrc(__builtin_amdgcn_make_buffer_rsrc((void *)p, 0, n * 8, 0x00027000)) {}
    __device__ __forceinline__ double load(int i) const {
        return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(rsrc, i * 8, 0, 0));
    }
    // values i and i + 1, p + i on a 16-byte boundary; past the caches with kNonTemporal
    template <int kHow>
    __device__ __forceinline__ double2 load2(int i) const {
        return __builtin_bit_cast(double2, __builtin_amdgcn_raw_buffer_load_b128(rsrc, i * 8, 0, kHow));
    }
    __device__ __forceinline__ void store(int i, double v) const {
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(Words2, v), rsrc, i * 8, 0, 0);
    }
    template <int kHow>
    __device__ __forceinline__ void store2(int i, double2 v) const {
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(Words4, v), rsrc, i * 8, 0, kHow);
    }
    typedef unsigned int Words2 __attribute__((ext_vector_type(2)));
    typedef unsigned int Words4 __attribute__((ext_vector_type(4)));
};

// tid, opaque to the compiler, so that indices formed from it are formed again rather than kept in
// registers since an earlier phase.
__device__ __forceinline__ int fresh(int tid) {
    asm volatile("" : "+v"(tid));
    return tid;
}

// Values from a tile's first value down to the 128-byte line it starts in: the tile's loads and
// stores start there (the values before the tile masked), so that each wave instruction covers
// whole lines.
__device__ __forceinline__ int line_lead(const double *p) { return (int)(((uintptr_t)p >> 3) & 15); }

// What the flux of a side point with a record needs of it (an inflow ghost reads its nodes too).
struct SideRecord {
    double nx, ny, tx, ty, sf;
    int64_t slot;
    int32_t kind, n_faces;
    __device__ __forceinline__ void load(const BcSide *r) {
        nx = r->nx;
        ny = r->ny;
        tx = r->tx;
        ty = r->ty;
        sf = r->sf;
        slot = r->slot;
        kind = r->kind;
        n_faces = r->n_faces;
    }
};

// (w_L - w_R)/2 and (w_L + w_R)/2 of point k of side s with a record: a boundary ghost (Mesh2D_t.cpp:
// 4298-4730), a periodic side of another direction, or a mortar side, which has the three components of
// its projected flux instead, already times the edge Jacobian: its faces may lie off the side's line by
// what the topology allows. The normal is the record's, tr the side's own traces.
template <int N, bool MORTAR>
__device__ __forceinline__ void record_flux(const SideRecord &rec, const BcSide *bc, const double (&tr)[3],
                                            const double *x, const double *tr_in, const double *side_flux, int k,
                                            const StageClock &clock, double cw, double &fa, double &fb,
                                            double &fc) {
    constexpr int NF = N + 1;
    constexpr double c = kWaveSpeed;
    if (MORTAR && rec.kind == kKindMortar) {  // projected by the mortar kernel (already x sf)
        const double *sfl = side_flux + rec.slot + k;
        double f0 = sfl[0], f1 = sfl[NF], f2 = sfl[2 * NF];
        for (int m = 1; m < rec.n_faces; ++m) {  // a side covered by several faces
            const double *s2 = sfl + m * 3 * NF;
            f0 += s2[0];
            f1 += s2[NF];
            f2 += s2[2 * NF];
        }
        fa = f0;
        fb = f1;
        fc = f2;
        return;
    }
    const double pL = tr[0], uL = tr[1], vL = tr[2];
    double pR = 0.0, uR = 0.0, vR = 0.0;
    if (rec.kind == NDG_BC_WALL || rec.kind == NDG_BC_SYMMETRY) {
        // ghost = sf * own trace, normal velocity reversed (Mesh2D_t.cpp:4377-4433)
        pR = pL * rec.sf;
        const double ux = uL * rec.sf, uy = vL * rec.sf;
        const double l0 = -(ux * rec.nx + uy * rec.ny);
        const double l1 = ux * rec.tx + uy * rec.ty;
        uR = rec.nx * l0 + rec.tx * l1;
        vR = rec.ny * l0 + rec.ty * l1;
    } else if (rec.kind == NDG_BC_OUTFLOW) {
        pR = pL * rec.sf;
        uR = uL * rec.sf;
        vR = vL * rec.sf;
    } else if (rec.kind == NDG_BC_INFLOW) {
        // ghost trace = g(x, t) at the ghost's nodes, seen reversed (Mesh2D_t.cpp:4575-4599)
        const double interp = (x[N - k] + 1) / 2;
        const double X = bc->bx * interp + bc->ax * (1 - interp);
        const double Y = bc->by * interp + bc->ay * (1 - interp);
        plane_wave(X, Y, clock.time(), cw, pR, uR, vR);
    } else if (rec.kind == kKindTrace) {
        const double *nb = tr_in + rec.slot + (N - k);
        pR = nb[0];
        uR = nb[NF];
        vR = nb[2 * NF];
    }
    const double wL = pL + c * (uL * rec.nx + vL * rec.ny);
    const double wR = pR - c * (uR * rec.nx + vR * rec.ny);
    fa = c * (wL - wR) / 2;
    fb = (wL + wR) / 2;
}

// The mortar sides' third flux component has a place of its own in LDS, but at N = 7, 8, where it would leave
// room for four workgroups a CU instead of five: there it lies in the d_xi tile, at the price of a barrier
// (160 x 160 of orders 4 to 12: 50.3 us a stage, 51.1 us with the barrier at every order).
template <int N>
constexpr bool kOwnFluxPlace = N != 7 && N != 8;
template <int N>
constexpr int flux_place() { return kOwnFluxPlace<N> ? LineShape<N>::EPB * 4 * (N + 1) : 0; }

template <int N>
constexpr int stage_lds() {
    return LineShape<N>::EPB * 6 * StageTile<N>::NEP + StageTile<N>::kFlux + LineShape<N>::EPB * 12 + flux_place<N>();
}

template <int N, bool RHS_ONLY, bool MORTAR>
__device__ __forceinline__ void
stage_tile(const double *__restrict__ verts, const int32_t *__restrict__ side_nb,
           const BcSide *__restrict__ bc, const double *__restrict__ tab,
           const double *q, double *q_out, double *__restrict__ g, const double *__restrict__ w_in,
           double *__restrict__ w_out, const double *__restrict__ tr_in, double *__restrict__ tr_out,
           double *__restrict__ rhs, const double *__restrict__ side_flux, int64_t K, int flags, double a,
           double gdt, const StageClock &clock, int epb, double cw, int64_t blk,
           double *__restrict__ s_q,     // the state tile
           double *__restrict__ s_d,     // vertices, then d_xi, then the new traces on sides 1 and 3
           double *__restrict__ s_f,     // fluxes, then the new traces on sides 0 and 2
           double *__restrict__ s_side,  // outward normal and edge Jacobian (negative: a mortar side) per side
           double *__restrict__ s_place) // flux_place values
{
    const bool first = flags & kRkFirst, store_g = !(flags & kRkLast), once = flags & kStream;
    using S = LineShape<N>;
    using L = StageTile<N>;
    constexpr int NF = S::NF, NE = S::NE, EPB = S::EPB, T = S::T, FPT = S::FPT, NFP = L::NFP, NEP = L::NEP;
    constexpr double c = kWaveSpeed;
    double *const s_v = s_d, *const s_fc = kOwnFluxPlace<N> ? s_place : s_d + EPB * 8;
    static_assert(EPB * (kOwnFluxPlace<N> ? 8 : 8 + 4 * NF) <= EPB * 3 * NEP, "what shares the tile fits it");
    const double *lm = tab + NF * NF;
    const double *lp = lm + NF;
    const double *x = lp + 2 * NF;
    const double *lpw = tab + table_stage_offset(N);  // l(+1) / w; that of l(-1) is its reverse

    const int tid = threadIdx.x;
    const int f = __builtin_amdgcn_readfirstlane(tid >> 6);  // field of this wave
    const int lane = tid & 63;
    const int64_t e0 = blk * epb;
    const int nel = (int)min<int64_t>(epb, K - e0);
    const int n_val = nel * 3 * NE, n_pt = nel * 4 * NF;
    const bool active = lane < nel * NF;
    // lanes past the tile's lines work on line 0 of its first element, so that every lane takes part
    // in the D^ broadcasts, and store nothing
    const int el = active ? lane / NF : 0, l = active ? lane % NF : 0;

    clock.advance();

    __builtin_amdgcn_s_setprio(3);  // issue this workgroup's loads ahead of other waves' math
    // P0
    int32_t code[FPT];
#pragma unroll
    for (int it = 0; it < FPT; ++it) {
        const int item = tid + it * T;
        code[it] = item < n_pt ? side_nb[e0 * 4 + item / NF] : INT32_MIN;
    }
    const int32_t side_code = side_nb[(e0 + el) * 4 + min(l, 3)];  // of the side this thread forms in wave 2
    const double x_l = x[l];
    // The RK register lives only within a step (the first stage writes it without reading it), so
    // its layout is the kernel's own: within the workgroup's tile it is stored as [f][j / 2][el][i][j % 2]
    // (an odd last j by itself), so that the row owners of all the tile's elements read and write two
    // line indices j with consecutive lanes on consecutive 16-byte words, each such run starting on a
    // 128-byte line.
    const int run = rk_run<N>(epb);
    const Buffer g_buf(RHS_ONLY ? nullptr : g + (blk * 3 + f) * NF * run, RHS_ONLY ? 0 : NF * run);
    const double *qg = q + e0 * 3 * NE;
    const int lead = line_lead(qg), q_last = lead + n_val - 1;
    const Buffer q_buf(qg - lead, lead + n_val), v_buf(verts + e0 * 8, nel * 8), w_buf(w_in + e0 * 4 * NF, n_pt);
    double2 qreg[L::QPT], g_old[NF / 2];
    double vreg[S::VPT], own[FPT], g_odd = 0.0;
    LaneTable<even_odd_len(NF)> Dh;
    auto load_tile = [&](auto how) {
        constexpr int kHow = decltype(how)::value;
#pragma unroll
        for (int it = 0; it < L::QPT; ++it) {
            const int i = 2 * (tid + it * T);
            qreg[it] = q_buf.load2<kHow>(i == q_last ? i - 1 : i);  // the last value as the second of a pair
        }
#pragma unroll
        for (int it = 0; it < S::VPT; ++it) vreg[it] = v_buf.load(tid + it * T);
        Dh.load(lpw + NF);
#pragma unroll
        for (int it = 0; it < FPT; ++it) own[it] = w_buf.load(tid + it * T);
        if (!RHS_ONLY && !first) {
#pragma unroll
            for (int j = 0; j < NF / 2; ++j) g_old[j] = g_buf.load2<kHow>(2 * j * run + 2 * lane);
            if (NF % 2) g_odd = g_buf.load(NF / 2 * 2 * run + lane);
        }
    };
    if (once) load_tile(std::integral_constant<int, Buffer::kNonTemporal>());
    else load_tile(std::integral_constant<int, 0>());
    SideRecord rec[FPT];
    double tr[FPT][3];  // the own traces of a side with a record
    uint64_t with_record[FPT];
#pragma unroll
    for (int it = 0; it < FPT; ++it) with_record[it] = __ballot(code[it] < 0 && code[it] != INT32_MIN);
#pragma unroll
    for (int it = 0; it < FPT; ++it)
        if (code[it] < 0 && code[it] != INT32_MIN) {
            const int item = tid + it * T;
            const double *from = tr_in + (e0 * 4 + item / NF) * 3 * NF + item % NF;
            for (int m = 0; m < 3; ++m) tr[it][m] = from[m * NF];
            rec[it].load(bc + (-1 - code[it]));
        }
    double ext[FPT];
#pragma unroll
    for (int it = 0; it < FPT; ++it) {
        const int32_t cd = max(code[it], 0);  // side 0 of the group for sides with a record
        const int k = (tid + it * T) % NF;
        ext[it] = w_in[(int64_t)cd * NF + (N - k)];
    }
    __builtin_amdgcn_s_setprio(0);
    // in the order of the loads; the whole of the LDS tiles is written, with zeros past the last
    // element; the own characteristics wait in the flux array
#pragma unroll
    for (int it = 0; it < L::QPT; ++it) {
        const int r = 2 * (tid + it * T) - lead;
        const bool inside = 2 * (it + 1) * T <= EPB * 3 * NE;
        if (r + lead == q_last) qreg[it] = make_double2(qreg[it].y, 0.0);
        if ((it > 0 || r >= 0) && (inside || r < EPB * 3 * NE)) s_q[L::at(r)] = qreg[it].x;
        if ((it > 0 || r >= -1) && (inside || r + 1 < EPB * 3 * NE)) s_q[L::at(r + 1)] = qreg[it].y;
    }
#pragma unroll
    for (int it = 0; it < S::VPT; ++it) {
        const int r = tid + it * T;
        if ((it + 1) * T <= EPB * 8 || r < EPB * 8) s_v[r] = vreg[it];
    }
#pragma unroll
    for (int it = 0; it < FPT; ++it) {
        const int item = tid + it * T;
        if ((it + 1) * T <= EPB * 4 * NF || item < EPB * 4 * NF) s_f[item] = own[it];
    }
    __syncthreads();

    // the points of sides with a record (before the contractions, whose sums would be live beside them)
#pragma unroll
    for (int it = 0; it < FPT; ++it)
        if (with_record[it]) {  // skipped by a wave without
            const int item = tid + it * T;
            if (code[it] >= 0 || code[it] == INT32_MIN) continue;
            record_flux<N, MORTAR>(rec[it], bc + (-1 - code[it]), tr[it], x, tr_in, side_flux, item % NF, clock, cw, s_f[item],
                           s_f[EPB * 4 * NF + item], s_fc[item]);
        }

    // P1. Metric lines from the vertices (include/functions/quad_metrics.tpp:3-8): x_eta, y_eta
    // are linear in xi, x_xi, y_xi in eta.
    const double *tq = s_q + el * 3 * NEP;
    const double *P = s_v + el * 8;
    double vx[NF], ve[NF];
    {
        double F[NF];
        // a line's value at coordinate t is m + d t, from its values P_a -> P_b at t = -1 and at t = +1
        auto mean = [&](int a0, int a1, int b0, int b1) { return ((P[b1] - P[b0]) + (P[a1] - P[a0])) / 4; };
        auto slope = [&](int a0, int a1, int b0, int b1) { return ((P[b1] - P[b0]) - (P[a1] - P[a0])) / 4; };
        const double *col = tq + l, *row = tq + l * NFP;  // node (k, l) at col[k * NFP], (l, k) at row[k]
        if (f == 0) {
            const double xe_m = mean(0, 6, 2, 4), xe_d = slope(0, 6, 2, 4), ye_m = mean(1, 7, 3, 5), ye_d = slope(1, 7, 3, 5);
#pragma unroll
            for (int k = 0; k < NF; ++k)
                F[k] = (ye_m + ye_d * x[k]) * col[NEP + k * NFP] - (xe_m + xe_d * x[k]) * col[2 * NEP + k * NFP];
        } else {  // y_eta p, -x_eta p
            const int o = f == 1 ? 1 : 0;
            const double m = mean(o, 6 + o, 2 + o, 4 + o), d = slope(o, 6 + o, 2 + o, 4 + o), sign = f == 1 ? 1.0 : -1.0;
#pragma unroll
            for (int k = 0; k < NF; ++k) F[k] = (sign * m + sign * d * x[k]) * col[k * NFP];
        }
        contract<NF>(Dh, F, vx);
        __builtin_amdgcn_sched_barrier(0);  // one line's operands in registers at a time
        if (f == 0) {
            const double xx_m = mean(0, 2, 6, 4), xx_d = slope(0, 2, 6, 4), yx_m = mean(1, 3, 7, 5), yx_d = slope(1, 3, 7, 5);
#pragma unroll
            for (int k = 0; k < NF; ++k)
                F[k] = (xx_m + xx_d * x[k]) * row[2 * NEP + k] - (yx_m + yx_d * x[k]) * row[NEP + k];
        } else {  // -y_xi p, x_xi p
            const int o = f == 1 ? 1 : 0;
            const double m = mean(o, 2 + o, 6 + o, 4 + o), d = slope(o, 2 + o, 6 + o, 4 + o), sign = f == 1 ? -1.0 : 1.0;
#pragma unroll
            for (int k = 0; k < NF; ++k) F[k] = (sign * m + sign * d * x[k]) * row[k];
        }
        contract<NF>(Dh, F, ve);
    }
    // the Jacobian of a bilinear element is linear in eta along the thread's eta line: jac_m + jac_d eta
    double jac_m, jac_d;
    {
        const double xeta = ((P[6] - P[0]) + (P[4] - P[2]) + ((P[4] - P[2]) - (P[6] - P[0])) * x_l) / 4;
        const double yeta = ((P[7] - P[1]) + (P[5] - P[3]) + ((P[5] - P[3]) - (P[7] - P[1])) * x_l) / 4;
        jac_m = (((P[4] - P[6]) + (P[2] - P[0])) * yeta - xeta * ((P[5] - P[7]) + (P[3] - P[1]))) / 4;
        jac_d = (((P[4] - P[6]) - (P[2] - P[0])) * yeta - xeta * ((P[5] - P[7]) - (P[3] - P[1]))) / 4;
    }
    // fluxes of the side points, side geometry (sides l, l + N + 1, ... of the wave's elements)
    const int t1 = fresh(tid);
#pragma unroll
    for (int it = 0; it < FPT; ++it) {
        const int item = t1 + it * T;
        if (item < n_pt && !__builtin_amdgcn_inverse_ballot_w64(with_record[it])) {
            const double w = s_f[item];
            s_f[item] = c * (w - ext[it]) / 2;
            s_f[EPB * 4 * NF + item] = (w + ext[it]) / 2;
        }
    }
    if (f == 2 && active)
        for (int s = l; s < 4; s += NF) {
            double *sd = s_side + (el * 4 + s) * 3;
            sd[2] = side_geometry(P, s, sd[0], sd[1]);
            if (const int32_t cd = s == l ? side_code : side_nb[(e0 + el) * 4 + s]; cd < 0) {
                const BcSide &rec = bc[-1 - cd];
                sd[0] = rec.nx;
                sd[1] = rec.ny;
                if (MORTAR && rec.kind == kKindMortar) sd[2] = -1.0;
            }
        }
    __syncthreads();

    // P2. Lifts: the thread's column j = l of d_xi and row i = l of d_eta. The flux of field f at a
    // side point is (w_L - w_R)/2 (p) or the normal's component times (w_L + w_R)/2 (u, v), times
    // the edge Jacobian, and the field's own component on a mortar side.
    {
        const double *side = s_side + el * 12;
        const double *fl = s_f + (f == 0 ? 0 : EPB * 4 * NF) + el * 4 * NF;
        const double v1 = fl[NF + l], v3 = fl[3 * NF + N - l], v2 = fl[2 * NF + N - l], v0 = fl[l];
        const double *n = side + (f == 2 ? 1 : 0);
        const double n0 = f ? n[0] : 1.0, n1 = f ? n[3] : 1.0, n2 = f ? n[6] : 1.0, n3 = f ? n[9] : 1.0;
        double Fr = (n1 * v1) * side[5], Fl = (n3 * v3) * side[11], Ft = (n2 * v2) * side[8], Fb = (n0 * v0) * side[2];
        if (MORTAR) {
            const double *own = f == 2 ? s_fc + el * 4 * NF : fl;
            if (kOwnFluxPlace<N>) {
                const double o1 = own[NF + l], o3 = own[3 * NF + N - l], o2 = own[2 * NF + N - l], o0 = own[l];
                Fr = side[5] < 0.0 ? o1 : Fr;
                Fl = side[11] < 0.0 ? o3 : Fl;
                Ft = side[8] < 0.0 ? o2 : Ft;
                Fb = side[2] < 0.0 ? o0 : Fb;
            } else {  // (these reads all at once would spill)
                if (side[5] < 0.0) Fr = own[NF + l];
                if (side[11] < 0.0) Fl = own[3 * NF + N - l];
                if (side[8] < 0.0) Ft = own[2 * NF + N - l];
                if (side[2] < 0.0) Fb = own[l];
                __syncthreads();  // d_xi replaces the third components
            }
        }
        double *d = s_d + el * 3 * NEP + f * NEP + l;
#pragma unroll
        for (int i = 0; i < NF; ++i) {
            vx[i] += Fr * lpw[i] + Fl * lpw[N - i];
            ve[i] += Ft * lpw[i] + Fb * lpw[N - i];
        }
        if (active)
#pragma unroll
            for (int i = 0; i < NF; ++i) d[i * NFP] = vx[i];
    }
    __syncthreads();

    // P3. The thread's eta line i = l of field f: the right-hand side replaces ve, then the new RK
    // register line, which goes straight to HBM, and the new state line, which replaces the old
    // one in the tile (no one else reads it until the barrier). One loop an operation, so that the
    // nodes' chains overlap.
    double *qrow = s_q + el * 3 * NEP + f * NEP + l * NFP;
    {
        double *d = s_d + el * 3 * NEP + f * NEP + l * NFP;
#pragma unroll
        for (int j = 0; j < NF; ++j) ve[j] = (d[j] + ve[j]) * (-cw * recip(jac_m + jac_d * x[j]));
        if (RHS_ONLY) {
            if (active)
#pragma unroll
                for (int j = 0; j < NF; ++j) d[j] = ve[j];
        } else if (!first) {
#pragma unroll
            for (int j = 0; j < NF / 2; ++j) {
                ve[2 * j] = a * g_old[j].x + ve[2 * j];
                ve[2 * j + 1] = a * g_old[j].y + ve[2 * j + 1];
            }
            if (NF % 2) ve[NF - 1] = a * g_odd + ve[NF - 1];
        }
    }
    if (!RHS_ONLY && active) {
        if (store_g) {
            auto store_lines = [&](auto how) {
#pragma unroll
                for (int j = 0; j < NF / 2; ++j)
                    g_buf.store2<decltype(how)::value>(2 * j * run + 2 * lane, make_double2(ve[2 * j], ve[2 * j + 1]));
            };
            if (once) store_lines(std::integral_constant<int, Buffer::kNonTemporal>());
            else store_lines(std::integral_constant<int, 0>());
            if (NF % 2) g_buf.store(NF / 2 * 2 * run + lane, ve[NF - 1]);
        }
        double t0 = 0.0, t2 = 0.0;
#pragma unroll
        for (int j = 0; j < NF; ++j) ve[j] = qrow[j] + gdt * ve[j];
#pragma unroll
        for (int j = 0; j < NF; ++j) {
            qrow[j] = ve[j];
            t0 += lp[N - j] * ve[j];
            t2 += lp[j] * ve[j];
        }
        double *tr = s_f + (el * 3 + f) * 2 * NF;
        tr[l] = t0;
        tr[NF + (N - l)] = t2;
    }
    __syncthreads();

    // P4
    if (RHS_ONLY) {
        double *rg = rhs + e0 * 3 * NE;
        for (int r = tid; r < n_val; r += T) rg[r] = s_d[L::at(r)];
        return;
    }
    if (active) {
        const double *col = s_q + el * 3 * NEP + f * NEP + l;
        double t1 = 0.0, t3 = 0.0;
#pragma unroll
        for (int j = 0; j < NF; ++j) {
            const double v = col[j * NFP];
            t1 += lp[j] * v;
            t3 += lp[N - j] * v;
        }
        double *tr = s_d + (el * 3 + f) * 2 * NF;
        tr[l] = t1;
        tr[NF + (N - l)] = t3;
    }
    {
        // pairs wholly inside the tile; its first and last value alone where a pair straddles an end
        double *qw = q_out + e0 * 3 * NE;
        const int t4 = fresh(tid);
        const int lead_out = line_lead(qw), end = lead_out + n_val;
        const Buffer out_buf(qw - lead_out, end & ~1);
        auto value = [&](int r) { return s_q[min(max(L::at(r), 0), EPB * 3 * NEP - 1)]; };
        auto store_tile = [&](auto how) {
#pragma unroll
            for (int it = 0; it < L::QPT; ++it) {
                const int i = 2 * (t4 + it * T), r = i - lead_out;
                const double2 v = make_double2(value(r), value(r + 1));
                if (it > 0 || r >= 0) out_buf.store2<decltype(how)::value>(i, v);
            }
        };
        if (once) store_tile(std::integral_constant<int, Buffer::kNonTemporal>());
        else store_tile(std::integral_constant<int, 0>());
        if ((lead_out & 1) && tid == 0) qw[0] = s_q[0];
        if ((end & 1) && tid == 64) qw[n_val - 1] = s_q[L::at(n_val - 1)];
    }
    __syncthreads();

    // P5
    const int t5 = fresh(tid);
#pragma unroll
    for (int it = 0; it < FPT; ++it) {
        const int item = t5 + it * T;
        if (item >= n_pt) continue;
        const int fe = item / (4 * NF), s = (item / NF) % 4, k = item % NF;
        const double *tr = ((s & 1) ? s_d : s_f) + fe * 6 * NF + (s >> 1) * NF + k;
        const double *sd = s_side + (fe * 4 + s) * 3;
        const double p = tr[0], u = tr[2 * NF], v = tr[4 * NF];
        w_out[e0 * 4 * NF + item] = p + c * (u * sd[0] + v * sd[1]);
        if (__builtin_amdgcn_inverse_ballot_w64(with_record[it]) || (flags & kTraceAll)) {
            double *to = tr_out + (e0 + fe) * 12 * NF + s * 3 * NF + k;
            to[0] = p;
            to[NF] = u;
            to[2 * NF] = v;
        }
    }
}

template <int N, bool RHS_ONLY>
__global__ void __launch_bounds__(192) __attribute__((amdgpu_waves_per_eu(N <= 8 ? 4 : N <= 12 ? 3 : 2)))
stage_kernel(const double *__restrict__ verts, const int32_t *__restrict__ side_nb,
             const BcSide *__restrict__ bc, const double *__restrict__ tab,
             const double *q, double *q_out, double *__restrict__ g, const double *__restrict__ w_in,
             double *__restrict__ w_out, const double *__restrict__ tr_in, double *__restrict__ tr_out,
             double *__restrict__ rhs, const double *__restrict__ side_flux, int64_t K, int flags, double a,
             double gdt, StageClock clock, int epb, int remap, double cw) {
    using L = StageTile<N>;
    constexpr int EPB = LineShape<N>::EPB, place = RHS_ONLY ? flux_place<N>() : 0;
    __shared__ double s_q[EPB * 3 * L::NEP], s_d[EPB * 3 * L::NEP], s_f[L::kFlux], s_side[EPB * 12], s_place[place ? place : 1];
    stage_tile<N, RHS_ONLY, RHS_ONLY>(verts, side_nb, bc, tab, q, q_out, g, w_in, w_out, tr_in, tr_out, rhs, side_flux, K,
                                      flags, a, gdt, clock, epb, cw,
                                      remap ? xcd_block(blockIdx.x, gridDim.x) : (int64_t)blockIdx.x, s_q, s_d, s_f, s_side,
                                      s_place);
}

// The stage of a mesh with mortar faces.
template <int N>
__global__ void __launch_bounds__(192) __attribute__((amdgpu_waves_per_eu(N <= 8 ? 4 : N <= 12 ? 3 : 2)))
stage_mortar_kernel(const double *__restrict__ verts, const int32_t *__restrict__ side_nb,
                    const BcSide *__restrict__ bc, const double *__restrict__ tab,
                    const double *q, double *q_out, double *__restrict__ g, const double *__restrict__ w_in,
                    double *__restrict__ w_out, const double *__restrict__ tr_in, double *__restrict__ tr_out,
                    double *__restrict__ rhs, const double *__restrict__ side_flux, int64_t K, int flags, double a,
                    double gdt, StageClock clock, int epb, int remap, double cw) {
    using L = StageTile<N>;
    constexpr int EPB = LineShape<N>::EPB, place = flux_place<N>();
    __shared__ double s_q[EPB * 3 * L::NEP], s_d[EPB * 3 * L::NEP], s_f[L::kFlux], s_side[EPB * 12], s_place[place ? place : 1];
    stage_tile<N, false, true>(verts, side_nb, bc, tab, q, q_out, g, w_in, w_out, tr_in, tr_out, rhs, side_flux, K, flags, a,
                               gdt, clock, epb, cw, remap ? xcd_block(blockIdx.x, gridDim.x) : (int64_t)blockIdx.x, s_q, s_d,
                               s_f, s_side, s_place);
}

// The stages of several order groups in one launch: the workgroups of group i are [first[i], first[i + 1]). Small
// groups are bound by their launches, each as long as the latency of one workgroup: 96 x 96 elements of
// orders 1, 3, 5, 7, 9 take 17.4 us a stage instead of 38.8 us with a launch a group (stage_groups_fit has the line).
struct StageGroups {
    int n;
    int first[kMaxOrder + 2];
    struct Part {
        int N, epb, remap;
        int64_t K, e_begin, q_off, tr_off, g_off;
        const double *tab;
        const float *tab32;
    } part[kMaxOrder];
};

// Calls run(order, part, tile) for the workgroup's group.
template <int Top, class Run>
__device__ __forceinline__ void run_group(const StageGroups &groups, Run &&run) {
    int i = 0;
    while (i + 1 < groups.n && (int)blockIdx.x >= groups.first[i + 1]) ++i;
    const StageGroups::Part &G = groups.part[i];
    const int b = (int)blockIdx.x - groups.first[i], n_blocks = groups.first[i + 1] - groups.first[i];
    const int64_t blk = G.remap ? xcd_block(b, n_blocks) : b;
    switch (G.N) {
#define NDG_RUN(n) \
    case n:        \
        if constexpr (n <= Top) run(std::integral_constant<int, n>(), G, blk); \
        break;
        NDG_RUN(1) NDG_RUN(2) NDG_RUN(3) NDG_RUN(4) NDG_RUN(5) NDG_RUN(6) NDG_RUN(7) NDG_RUN(8)
        NDG_RUN(9) NDG_RUN(10) NDG_RUN(11) NDG_RUN(12) NDG_RUN(13) NDG_RUN(14) NDG_RUN(15) NDG_RUN(16)
#undef NDG_RUN
    }
}

constexpr int max_stage_lds(int a, int b) { return a > b ? a : b; }
template <int N>
constexpr int most_stage_lds() {
    if constexpr (N == 1) return stage_lds<1>();
    else return max_stage_lds(stage_lds<N>(), most_stage_lds<N - 1>());
}

template <int Top>  // the largest order among the groups
__global__ void __launch_bounds__(192) __attribute__((amdgpu_waves_per_eu(Top <= 8 ? 4 : Top <= 12 ? 3 : 2)))
stage_groups_kernel(StageGroups groups, const double *__restrict__ verts, const int32_t *__restrict__ side_nb,
                    const BcSide *__restrict__ bc, const double *q, double *q_out, double *__restrict__ g,
                    const double *__restrict__ w_in, double *__restrict__ w_out, const double *__restrict__ tr_in,
                    double *__restrict__ tr_out, const double *__restrict__ side_flux, int flags, double a, double gdt,
                    StageClock clock, double cw) {
    __shared__ double mem[most_stage_lds<Top>()];
    run_group<Top>(groups, [&](auto order, const StageGroups::Part &G, int64_t blk) {
        constexpr int N = decltype(order)::value;
        constexpr int EPB = LineShape<N>::EPB, tile = EPB * 3 * StageTile<N>::NEP;
        stage_tile<N, false, true>(verts + G.e_begin * 8, side_nb + G.e_begin * 4, bc, G.tab, q + G.q_off, q_out + G.q_off,
                             g + G.g_off, w_in + G.tr_off / 3, w_out + G.tr_off / 3, tr_in + G.tr_off,
                             tr_out + G.tr_off, nullptr, side_flux, G.K, flags, a, gdt, clock, G.epb, cw, blk, mem,
                             mem + tile, mem + 2 * tile, mem + 2 * tile + StageTile<N>::kFlux,
                             mem + 2 * tile + StageTile<N>::kFlux + EPB * 12);
    });
}

// ---------------------------------------------------------------------------------------------
// FP32 form with a compensated state. The right-hand side (traces, flux, volume, lift) and the RK
// register are FP32; the state is the unevaluated sum qh + ql of two floats, updated with an
// error-free two-sum so that the accumulation over many steps keeps ~48 bits. Geometry (metric
// lines, normals, edge Jacobians) is evaluated in FP64 from the FP64 vertices and rounded once.
// Same thread layout and phases as stage_kernel.

// qh + ql += d exactly up to the final rounding of ql (Knuth two-sum, then fast two-sum
// renormalisation); contraction is off so that the error terms are exact.
__device__ __forceinline__ void two_sum_add(float &hi, float &lo, float d) {
#pragma clang fp contract(off)
    const float s = hi + d;
    const float bb = s - hi;
    const float err = (hi - (s - bb)) + (d - bb);
    const float l = lo + err;
    const float h = s + l;
    lo = l - (h - s);
    hi = h;
}

// Position in the FP32 form's gl32 (the RK register's order in tiles of epb elements and runs of `run`
// values, see stage_kernel) of value (element e, field f, node (i, j)); nf = N + 1.
__device__ __forceinline__ int64_t c32_tile_index(int64_t e, int f, int i, int j, int nf, int epb, int run) {
    const int64_t blk = e / epb, base = (blk * 3 + f) * nf * run;
    const int at = (int)(e - blk * epb) * nf + i;
    return j < nf / 2 * 2 ? base + (j & ~1) * run + 2 * at + (j & 1) : base + j * run + at;
}

// q and qh are in reference node order; gl32 (RK register in x, low state word in y) is in the
// FP32 stage kernel's tile order. Thread r writes one float2. The register's word starts at zero: it
// carries no value from one step to the next, and a step's first stage does not use what it loads there.
__global__ void to_c32_kernel(const double *__restrict__ q, float *__restrict__ qh, float2 *__restrict__ gl32,
                              int64_t n, int nf, int epb, int run) {
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= n) return;
    const int ne = nf * nf, node = (int)(r % ne), i = node / nf, j = node % nf;
    const int64_t e = r / (3 * ne);
    const int f = (int)((r / ne) % 3);
    const double v = q[r];
    const float h = (float)v;
    qh[r] = h;
    gl32[c32_tile_index(e, f, i, j, nf, epb, run)] = make_float2(0.f, (float)(v - (double)h));
}

__global__ void from_c32_kernel(const float *__restrict__ qh, const float2 *__restrict__ gl32,
                                double *__restrict__ q, int64_t n, int nf, int epb, int run) {
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= n) return;
    const int ne = nf * nf, node = (int)(r % ne), i = node / nf, j = node % nf;
    const int64_t e = r / (3 * ne);
    const int f = (int)((r / ne) % 3);
    const float2 w = gl32[c32_tile_index(e, f, i, j, nf, epb, run)];
    q[r] = (double)qh[r] + (double)w.y;
}

// p + u.n with one fused product, as every place must round it (left to the compiler, a pair of products
// becomes a vector of two here and there and loses it).
__device__ __forceinline__ float characteristic32(float p, float u, float v, float nx, float ny) {
    return p + fmaf(v, ny, u * nx);
}

template <int N>
__global__ void __launch_bounds__(192)
traces_c32_kernel(const double *__restrict__ verts, const int32_t *__restrict__ side_nb, const BcSide *__restrict__ bc,
                  const float *__restrict__ tab, const float *__restrict__ qh, float *__restrict__ tr,
                  float *__restrict__ w, int64_t K) {
    using S = LineShape<N>;
    constexpr int NF = S::NF, NE = S::NE, EPB = S::EPB, T = S::T;
    __shared__ float s_q[EPB * 3 * NE], s_tr[EPB * 12 * NF];
    const float *lm = tab + NF * NF;
    const float *lp = lm + NF;
    const int tid = threadIdx.x;
    const int f = tid >> 6, lane = tid & 63, el = lane / NF, l = lane % NF;
    const int64_t e0 = (int64_t)blockIdx.x * EPB;
    const int nel = (int)min<int64_t>(EPB, K - e0);
    for (int r = tid; r < nel * 3 * NE; r += T) s_q[r] = qh[e0 * 3 * NE + r];
    __syncthreads();
    if (el < nel) {
        const float *tq = s_q + el * 3 * NE + f * NE;
        float t0 = 0.f, t1 = 0.f, t2 = 0.f, t3 = 0.f;
        for (int j = 0; j < NF; ++j) {
            const float row = tq[l * NF + j], col = tq[j * NF + l];
            t0 += lm[j] * row;
            t2 += lp[j] * row;
            t1 += lp[j] * col;
            t3 += lm[j] * col;
        }
        float *to = s_tr + el * 12 * NF + f * NF;
        to[l] = t0;
        to[6 * NF + (N - l)] = t2;
        to[3 * NF + l] = t1;
        to[9 * NF + (N - l)] = t3;
    }
    __syncthreads();
    for (int r = tid; r < nel * 12 * NF; r += T) tr[e0 * 12 * NF + r] = s_tr[r];
    for (int r = tid; r < nel * 4 * NF; r += T) {
        const int fe = r / (4 * NF), s = (r / NF) % 4, k = r % NF;
        double nx, ny;
        side_normal(verts, side_nb, bc, e0 + fe, s, nx, ny);
        const float *t = s_tr + fe * 12 * NF + s * 3 * NF + k;
        w[e0 * 4 * NF + r] = characteristic32(t[0], t[NF], t[2 * NF], (float)nx, (float)ny);
    }
}

// n floats from p, in 16-byte words, bounds-checked as Buffer's values are.
struct Buffer32 {
    __amdgpu_buffer_rsrc_t rsrc;
    __device__ __forceinline__ Buffer32(const float *p, int n)
        : rsrc(__builtin_amdgcn_make_buffer_rsrc((void *)p, 0, n * 4, 0x00027000)) {}
    __device__ __forceinline__ float load(int i) const {
        return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, i * 4, 0, 0));
    }
    template <int kHow>
    __device__ __forceinline__ float2 load2(int i) const {
        return __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(rsrc, i * 4, 0, kHow));
    }
    template <int kHow>
    __device__ __forceinline__ float4 load4(int i) const {
        return __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, i * 4, 0, kHow));
    }
    __device__ __forceinline__ void store(int i, float v) const {
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), rsrc, i * 4, 0, 0);
    }
    template <int kHow>
    __device__ __forceinline__ void store2(int i, float2 v) const {
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(Buffer::Words2, v), rsrc, i * 4, 0, kHow);
    }
    template <int kHow>
    __device__ __forceinline__ void store4(int i, float4 v) const {
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(Buffer::Words4, v), rsrc, i * 4, 0, kHow);
    }
};

// LaneTable of floats.
template <int L>
struct LaneTable32 {
    float v[(L + 15) / 16];
    __device__ __forceinline__ void load(const float *t) {
        const int m = threadIdx.x & 15;
#pragma unroll
        for (int p = 0; p < (L + 15) / 16; ++p) v[p] = t[min(p * 16 + m, L - 1)];
    }
};

// a[i S] (+)= D(entry E + i Step) F for the R rows i, a column of D^ at a time: the entry is a DPP operand of the
// multiply-add (the compiler moves it to a register first, with a wait: three issues instead of
// one). A block first waits out the two cycles that a register written just before it takes to reach
// a DPP instruction, and within one every row is another register.
template <bool kSet, int E, int Step, int R, int L>
__device__ __forceinline__ void rows32(const LaneTable32<L> &D, float F, float *a) {
#define NDG_MAC32(o, d, f, e) "v_fmac_f32_dpp %" #o ", %" #d ", %" #f " row_newbcast:%" #e " row_mask:0xf bank_mask:0xf\n\t"
#define NDG_MUL32(o, d, f, e) "v_mul_f32_dpp %" #o ", %" #d ", %" #f " row_newbcast:%" #e " row_mask:0xf bank_mask:0xf\n\t"
#define NDG_ENTRY32(i) D.v[(E + (i) * Step) / 16]
#define NDG_LANE32(i) (E + (i) * Step) % 16
    if constexpr (R > 4) {
        rows32<kSet, E, Step, 4>(D, F, a);
        rows32<kSet, E + 4 * Step, Step, R - 4>(D, F, a + 4);
    } else if constexpr (R == 4 && kSet) {
        asm volatile("s_nop 1\n\t" NDG_MUL32(0, 4, 8, 9) NDG_MUL32(1, 5, 8, 10) NDG_MUL32(2, 6, 8, 11)
                         NDG_MUL32(3, 7, 8, 12)
                     : "=&v"(a[0]), "=&v"(a[1]), "=&v"(a[2]), "=&v"(a[3])
                     : "v"(NDG_ENTRY32(0)), "v"(NDG_ENTRY32(1)), "v"(NDG_ENTRY32(2)), "v"(NDG_ENTRY32(3)), "v"(F),
                       "n"(NDG_LANE32(0)), "n"(NDG_LANE32(1)), "n"(NDG_LANE32(2)), "n"(NDG_LANE32(3)));
    } else if constexpr (R == 4) {
        asm volatile("s_nop 1\n\t" NDG_MAC32(0, 4, 8, 9) NDG_MAC32(1, 5, 8, 10) NDG_MAC32(2, 6, 8, 11)
                         NDG_MAC32(3, 7, 8, 12)
                     : "+&v"(a[0]), "+&v"(a[1]), "+&v"(a[2]), "+&v"(a[3])
                     : "v"(NDG_ENTRY32(0)), "v"(NDG_ENTRY32(1)), "v"(NDG_ENTRY32(2)), "v"(NDG_ENTRY32(3)), "v"(F),
                       "n"(NDG_LANE32(0)), "n"(NDG_LANE32(1)), "n"(NDG_LANE32(2)), "n"(NDG_LANE32(3)));
    } else if constexpr (R > 0) {
        if constexpr (kSet)
            asm volatile("s_nop 1\n\t" NDG_MUL32(0, 1, 2, 3)
                         : "=&v"(a[0])
                         : "v"(NDG_ENTRY32(0)), "v"(F), "n"(NDG_LANE32(0)));
        else
            asm volatile("s_nop 1\n\t" NDG_MAC32(0, 1, 2, 3)
                         : "+&v"(a[0])
                         : "v"(NDG_ENTRY32(0)), "v"(F), "n"(NDG_LANE32(0)));
        rows32<kSet, E + Step, Step, R - 1>(D, F, a + 1);
    }
#undef NDG_MAC32
#undef NDG_MUL32
#undef NDG_ENTRY32
#undef NDG_LANE32
}

// a = D^ F, each row summed in the order of the line's nodes.
template <int NF, int k = 0>
__device__ __forceinline__ void contract32(const LaneTable32<NF * NF> &D, const float *F, float *a) {
    rows32<k == 0, k, NF, NF>(D, F[k], a);
    if constexpr (k + 1 < NF) contract32<NF, k + 1>(D, F, a);
}

// record_flux in FP32: (w_L - w_R)/2, (w_L + w_R)/2 and, for a mortar side, the three flux components.
template <int N, bool MORTAR>
__device__ __forceinline__ void record_flux32(const SideRecord &rec, const BcSide *bc, const float (&tr)[3],
                                              const double *x64, const float *tr_in, const float *side_flux, int k,
                                              const StageClock &clock, double cw, float &fa, float &fb, float &fc) {
    constexpr int NF = N + 1;
    const int kind = rec.kind;
    if (MORTAR && kind == kKindMortar) {
        const float *sfl = side_flux + bc->slot + k;
        float f0 = sfl[0], f1 = sfl[NF], f2 = sfl[2 * NF];
        const int n_faces = bc->n_faces;
        for (int m = 1; m < n_faces; ++m) {
            const float *s2 = sfl + m * 3 * NF;
            f0 += s2[0];
            f1 += s2[NF];
            f2 += s2[2 * NF];
        }
        fa = f0;
        fb = f1;
        fc = f2;
        return;
    }
    const float pL = tr[0], uL = tr[1], vL = tr[2];
    const float nx = (float)rec.nx, ny = (float)rec.ny, gs = (float)rec.sf;
    float pR = 0.f, uR = 0.f, vR = 0.f;
    if (kind == NDG_BC_WALL || kind == NDG_BC_SYMMETRY) {
        const float tx = (float)bc->tx, ty = (float)bc->ty;
        pR = pL * gs;
        const float ux = uL * gs, uy = vL * gs;
        const float l0 = -fmaf(uy, ny, ux * nx);
        const float l1 = fmaf(uy, ty, ux * tx);
        uR = fmaf(tx, l1, nx * l0);
        vR = fmaf(ty, l1, ny * l0);
    } else if (kind == NDG_BC_OUTFLOW) {
        pR = pL * gs;
        uR = uL * gs;
        vR = vL * gs;
    } else if (kind == NDG_BC_INFLOW) {
        const double interp = (x64[N - k] + 1) / 2;
        const double X = bc->bx * interp + bc->ax * (1 - interp);
        const double Y = bc->by * interp + bc->ay * (1 - interp);
        double p64, u64, v64;
        plane_wave(X, Y, clock.time(), cw, p64, u64, v64);
        pR = (float)p64;
        uR = (float)u64;
        vR = (float)v64;
    } else if (kind == kKindTrace) {
        const float *nb = tr_in + bc->slot + (N - k);
        pR = nb[0];
        uR = nb[NF];
        vR = nb[2 * NF];
    }
    const float wL = characteristic32(pL, uL, vL, nx, ny);
    const float wR = characteristic32(pR, -uR, -vR, nx, ny);
    fa = (wL - wR) * 0.5f;
    fb = (wL + wR) * 0.5f;
}

// The FP32 stage: stage_kernel's phases, exchange and streaming; every sum in the order and every
// product with the rounding of the form without them, so the results are the same bit for bit (the
// D^ entries are therefore not folded into even and odd parts, and a mortar side keeps its three flux
// components). gl holds the RK register and the low state word of each value, interleaved, in the
// RK register's tile order of the shape's full tiles (the launch always uses them, so the low words
// keep their places from one step to the next). A side with a record reads its own traces back, loaded
// with the tile; formed again from the tile's lines they cost a wall mesh of 96 x 96, N = 8 0.4 us.
// Bound by memory at large sizes: 384 x 384, N = 7 in 126 us a launch, 157 us with three traces
// exchanged a point, 4-byte cached accesses and D^ in scalar registers; 512 x 512, N = 8: 293 and
// 350 us; 256 x 256, N = 12: 170 and 186 us; 48 x 48, N = 16: 16.1 and 18.1 us. Where one round of
// workgroups fills the chip the wait for the tile decides: 128 x 128, N = 8: 22.7 and 24.2 us, 96 x 96:
// 13.6 and 13.7 us. There the vertices in 16-byte words and no code for mortar sides on meshes without
// (MORTAR) count: 14.3 us with eight loads of a coordinate and one kernel for all meshes.
template <int N, bool MORTAR>
__device__ __forceinline__ void
stage_c32_tile(const double *__restrict__ verts, const int32_t *__restrict__ side_nb,
               const BcSide *__restrict__ bc, const double *__restrict__ tab64,
               const float *__restrict__ tab, float *__restrict__ qh, float2 *__restrict__ gl,
               const float *__restrict__ w_in, float *__restrict__ w_out, const float *__restrict__ tr_in,
               float *__restrict__ tr_out, const float *__restrict__ side_flux, int64_t K, int flags, float a, float gdt,
               const StageClock &clock, double cw, int64_t blk,
               float *__restrict__ s_q,     // the state tile
               float *__restrict__ s_d,     // d_xi, then the new traces on sides 1 and 3
               float *__restrict__ s_f,     // fluxes, then the new traces on sides 0 and 2
               float *__restrict__ s_met,   // metric lines
               float *__restrict__ s_side)  // outward normal and edge Jacobian (negative: a mortar side)
{
    const bool first = flags & kRkFirst, once = flags & kStream;
    using S = LineShape<N>;
    constexpr int NF = S::NF, NE = S::NE, EPB = S::EPB, T = S::T, FPT = S::FPT, NFP = NF | 1, NEP = NF * NFP;
    constexpr int QP4 = (EPB * 3 * NE + 31 + 4 * T - 1) / (4 * T);  // 16-byte words of the tile per thread
    constexpr int run = rk_run<N>(EPB);
    const float *lm = tab + NF * NF;
    const float *lp = lm + NF;
    const float *winv = lp + 3 * NF;
    const double *x64 = tab64 + NF * NF + 3 * NF;

    const int tid = threadIdx.x;
    const int f = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63;
    const int64_t e0 = blk * EPB;
    const int nel = (int)min<int64_t>(EPB, K - e0);
    const int n_val = nel * 3 * NE, n_pt = nel * 4 * NF;
    const bool active = lane < nel * NF;
    const int el = active ? lane / NF : 0, l = active ? lane % NF : 0;

    clock.advance();

    __builtin_amdgcn_s_setprio(3);  // issue this workgroup's loads ahead of other waves' math
    // P0
    int32_t code[FPT];
#pragma unroll
    for (int it = 0; it < FPT; ++it) {
        const int item = tid + it * T;
        code[it] = item < n_pt ? side_nb[e0 * 4 + item / NF] : INT32_MIN;
    }
    double P[8];  // the element's vertices; in the wave that forms the sides, from side l's first one on
    const int side = min(l, 3);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const double2 v = ((const double2 *)verts)[(e0 + el) * 4 + (f == 2 ? (side + k) & 3 : k)];
        P[2 * k] = v.x;
        P[2 * k + 1] = v.y;
    }
    const int32_t side_code = side_nb[(e0 + el) * 4 + side];
    const float *qg = qh + e0 * 3 * NE;
    const int lead = (int)(((uintptr_t)qg >> 2) & 31), end = lead + n_val;
    // words wholly inside the tile by the bounds check; the values of a last partial word one by one
    const Buffer32 q_buf(qg - lead, end & ~3), q_all(qg - lead, end), w_buf(w_in + e0 * 4 * NF, n_pt);
    const Buffer32 gl_buf((const float *)(gl + (blk * 3 + f) * NF * run), 2 * NF * run);
    float4 qreg[QP4], gl_old[NF / 2];
    float own[FPT], q_rest = 0.f;
    float2 gl_odd = make_float2(0.f, 0.f);
    LaneTable32<NF * NF> Dh;
    auto load_tile = [&](auto how) {
        constexpr int kHow = decltype(how)::value;
#pragma unroll
        for (int it = 0; it < QP4; ++it) qreg[it] = q_buf.load4<kHow>(4 * (tid + it * T));
        q_rest = q_all.load((end & ~3) + (tid & 3));
        Dh.load(tab);
#pragma unroll
        for (int it = 0; it < FPT; ++it) own[it] = w_buf.load(tid + it * T);
#pragma unroll
        for (int j = 0; j < NF / 2; ++j) gl_old[j] = gl_buf.load4<kHow>(4 * (j * run + lane));
        if (NF % 2) gl_odd = gl_buf.load2<kHow>(2 * (NF / 2 * 2 * run + lane));
    };
    if (once) load_tile(std::integral_constant<int, Buffer::kNonTemporal>());
    else load_tile(std::integral_constant<int, 0>());
    SideRecord rec[FPT];
    float tr[FPT][3];  // the own traces of a side with a record
    uint64_t with_record[FPT];
#pragma unroll
    for (int it = 0; it < FPT; ++it) with_record[it] = __ballot(code[it] < 0 && code[it] != INT32_MIN);
#pragma unroll
    for (int it = 0; it < FPT; ++it)
        if (code[it] < 0 && code[it] != INT32_MIN) {
            const int item = tid + it * T;
            const float *from = tr_in + (e0 * 4 + item / NF) * 3 * NF + item % NF;
            for (int m = 0; m < 3; ++m) tr[it][m] = from[m * NF];
            rec[it].load(bc + (-1 - code[it]));
        }
    float ext[FPT];
#pragma unroll
    for (int it = 0; it < FPT; ++it) {
        const int32_t cd = max(code[it], 0);  // side 0 of the group for sides with a record
        const int k = (tid + it * T) % NF;
        ext[it] = w_in[(int64_t)cd * NF + (N - k)];
    }
    __builtin_amdgcn_s_setprio(0);
    auto at = [](int r) { return NFP == NF ? r : r + (int)((unsigned)r / NF); };
    auto put_q = [&](int r, float v) {
        if (r >= 0 && r < EPB * 3 * NE) s_q[at(r)] = v;
    };
#pragma unroll
    for (int it = 0; it < QP4; ++it) {
        const int i = 4 * (tid + it * T), r = i - lead;
        if (i < (end & ~3)) {
            put_q(r, qreg[it].x);
            put_q(r + 1, qreg[it].y);
            put_q(r + 2, qreg[it].z);
            put_q(r + 3, qreg[it].w);
        }
    }
    if (tid < (end & 3)) put_q((end & ~3) + tid - lead, q_rest);
#pragma unroll
    for (int it = 0; it < FPT; ++it) {
        const int item = tid + it * T;
        if ((it + 1) * T <= EPB * 4 * NF || item < EPB * 4 * NF) s_f[item] = own[it];
    }
    if (active && f < 2) {  // metric lines (in FP64, rounded once)
        const double t = x64[l];
        float *met = s_met + el * 4 * NF + 2 * f * NF;
        // x_eta, y_eta along xi; x_xi, y_xi along eta
        const double ax = f == 0 ? P[6] : P[2], ay = f == 0 ? P[7] : P[3], bx = f == 0 ? P[2] : P[6],
                     by = f == 0 ? P[3] : P[7];
        met[l] = (float)(((1 - t) * (ax - P[0]) + (1 + t) * (P[4] - bx)) / 4);
        met[NF + l] = (float)(((1 - t) * (ay - P[1]) + (1 + t) * (P[5] - by)) / 4);
    }
    if (active && f == 2)  // sides l, l + N + 1, ... (N + 1 lanes cover the four)
        for (int s = l; s < 4; s += NF) {
            double nx, ny;
            float sf = (float)(s == l ? side_geometry(P, 0, nx, ny) : side_geometry(verts + (e0 + el) * 8, s, nx, ny));
            if (const int32_t cd = s == l ? side_code : side_nb[(e0 + el) * 4 + s]; cd < 0) {
                const BcSide &r = bc[-1 - cd];
                nx = r.nx;
                ny = r.ny;
                if (MORTAR && r.kind == kKindMortar) sf = -1.f;
            }
            float *sd = s_side + (el * 4 + s) * 3;
            sd[0] = (float)nx;
            sd[1] = (float)ny;
            sd[2] = sf;
        }
    __syncthreads();

#pragma unroll
    for (int it = 0; it < FPT; ++it)
        if (with_record[it]) {  // skipped by a wave without
            const int item = tid + it * T;
            if (code[it] >= 0 || code[it] == INT32_MIN) continue;
            record_flux32<N, MORTAR>(rec[it], bc + (-1 - code[it]), tr[it], x64, tr_in, side_flux, item % NF, clock, cw,
                             s_f[item], s_f[EPB * 4 * NF + item], s_f[EPB * 8 * NF + item]);
        }

    // P1
    const float *tq = s_q + el * 3 * NEP;
    const float *met = s_met + el * 4 * NF;
    float vx[NF], ve[NF];
    {
        float F[NF];
        const float *col = tq + l, *row = tq + l * NFP;  // node (k, l) at col[k * NFP], (l, k) at row[k]
        if (f == 0) {
#pragma unroll
            for (int k = 0; k < NF; ++k) {
                const float xeta = met[k], yeta = met[NF + k];
                F[k] = yeta * col[NEP + k * NFP] - xeta * col[2 * NEP + k * NFP];
            }
        } else if (f == 1) {
#pragma unroll
            for (int k = 0; k < NF; ++k) F[k] = met[NF + k] * col[k * NFP];
        } else {
#pragma unroll
            for (int k = 0; k < NF; ++k) F[k] = -(met[k] * col[k * NFP]);
        }
        contract32<NF>(Dh, F, vx);
        if (f == 0) {
#pragma unroll
            for (int k = 0; k < NF; ++k) {
                const float xxi = met[2 * NF + k], yxi = met[3 * NF + k];
                F[k] = -yxi * row[NEP + k] + xxi * row[2 * NEP + k];
            }
        } else if (f == 1) {
#pragma unroll
            for (int k = 0; k < NF; ++k) F[k] = -met[3 * NF + k] * row[k];
        } else {
#pragma unroll
            for (int k = 0; k < NF; ++k) F[k] = met[2 * NF + k] * row[k];
        }
        contract32<NF>(Dh, F, ve);
    }
    const int t1 = fresh(tid);
#pragma unroll
    for (int it = 0; it < FPT; ++it) {
        const int item = t1 + it * T;
        if (item < n_pt && !__builtin_amdgcn_inverse_ballot_w64(with_record[it])) {
            const float w = s_f[item];
            s_f[item] = (w - ext[it]) * 0.5f;
            s_f[EPB * 4 * NF + item] = (w + ext[it]) * 0.5f;
        }
    }
    __syncthreads();

    // P2
    {
        const float *side = s_side + el * 12;
        const float *fl = s_f + el * 4 * NF;
        auto flux = [&](int s, int k) {
            const float sf = side[3 * s + 2];
            const float va = fl[(f == 0 ? 0 : EPB * 4 * NF) + s * NF + k];
            if (MORTAR && sf < 0.f) return fl[f * EPB * 4 * NF + s * NF + k];  // the mortar side's own component
            return f == 0 ? va * sf : (side[3 * s + (f == 2 ? 1 : 0)] * va) * sf;
        };
        const float Fr = flux(1, l), Fl = flux(3, N - l), Ft = flux(2, N - l), Fb = flux(0, l);
        float *d = s_d + el * 3 * NEP + f * NEP + l;
#pragma unroll
        for (int i = 0; i < NF; ++i) {
            vx[i] += (Fr * lp[i] + Fl * lm[i]) * winv[i];
            ve[i] += (Ft * lp[i] + Fb * lm[i]) * winv[i];
        }
        if (active)
#pragma unroll
            for (int i = 0; i < NF; ++i) d[i * NFP] = vx[i];
    }
    __syncthreads();

    // P3
    {
        float *d = s_d + el * 3 * NEP + f * NEP + l * NFP;
        float *qrow = s_q + el * 3 * NEP + f * NEP + l * NFP;
        const float xeta_i = met[l], yeta_i = met[NF + l];
#pragma unroll
        for (int j = 0; j < NF; ++j) {
            const float jac = met[2 * NF + j] * yeta_i - xeta_i * met[3 * NF + j];
            ve[j] = (float)cw * ((-d[j] - ve[j]) / jac);
        }
        float h[NF], lo[NF];
#pragma unroll
        for (int j = 0; j < NF; ++j) {
            const float2 w = j / 2 < NF / 2 ? (j % 2 ? make_float2(gl_old[j / 2].z, gl_old[j / 2].w)
                                                     : make_float2(gl_old[j / 2].x, gl_old[j / 2].y))
                                            : gl_odd;
            ve[j] = first ? ve[j] : a * w.x + ve[j];
            h[j] = qrow[j];
            lo[j] = w.y;
            two_sum_add(h[j], lo[j], gdt * ve[j]);
        }
        if (active) {
            auto store_lines = [&](auto how) {
#pragma unroll
                for (int j = 0; j < NF / 2; ++j)
                    gl_buf.store4<decltype(how)::value>(4 * (j * run + lane),
                                                        make_float4(ve[2 * j], lo[2 * j], ve[2 * j + 1], lo[2 * j + 1]));
                if (NF % 2) gl_buf.store2<decltype(how)::value>(2 * (NF / 2 * 2 * run + lane),
                                                                make_float2(ve[NF - 1], lo[NF - 1]));
            };
            if (once) store_lines(std::integral_constant<int, Buffer::kNonTemporal>());
            else store_lines(std::integral_constant<int, 0>());
            float t0 = 0.f, t2 = 0.f;
#pragma unroll
            for (int j = 0; j < NF; ++j) {
                qrow[j] = h[j];
                t0 += lm[j] * h[j];
                t2 += lp[j] * h[j];
            }
            float *tr = s_f + (el * 3 + f) * 2 * NF;
            tr[l] = t0;
            tr[NF + (N - l)] = t2;
        }
    }
    __syncthreads();

    // P4
    if (active) {
        const float *col = s_q + el * 3 * NEP + f * NEP + l;
        float t1 = 0.f, t3 = 0.f;
#pragma unroll
        for (int j = 0; j < NF; ++j) {
            const float v = col[j * NFP];
            t1 += lp[j] * v;
            t3 += lm[j] * v;
        }
        float *tr = s_d + (el * 3 + f) * 2 * NF;
        tr[l] = t1;
        tr[NF + (N - l)] = t3;
    }
    {
        // words wholly inside the tile; the values of a word that straddles an end one by one
        const int t4 = fresh(tid);
        auto value = [&](int r) { return s_q[min(max(at(r), 0), EPB * 3 * NEP - 1)]; };
        auto store_tile = [&](auto how) {
#pragma unroll
            for (int it = 0; it < QP4; ++it) {
                const int i = 4 * (t4 + it * T), r = i - lead;
                const float4 v = make_float4(value(r), value(r + 1), value(r + 2), value(r + 3));
                if (it > 0 || r >= 0) q_buf.store4<decltype(how)::value>(i, v);
            }
        };
        if (once) store_tile(std::integral_constant<int, Buffer::kNonTemporal>());
        else store_tile(std::integral_constant<int, 0>());
        const int head = min((4 - (lead & 3)) & 3, n_val), tail = lead + head <= (end & ~3) ? end & 3 : 0;
        if (tid < head) q_all.store(lead + tid, s_q[at(tid)]);
        if (tid >= 64 && tid < 64 + tail) q_all.store((end & ~3) + tid - 64, s_q[at((end & ~3) + tid - 64 - lead)]);
    }
    __syncthreads();

    // P5
    const int t5 = fresh(tid);
#pragma unroll
    for (int it = 0; it < FPT; ++it) {
        const int item = t5 + it * T;
        if (item >= n_pt) continue;
        const int fe = item / (4 * NF), s = (item / NF) % 4, k = item % NF;
        const float *tr = ((s & 1) ? s_d : s_f) + fe * 6 * NF + (s >> 1) * NF + k;
        const float *sd = s_side + (fe * 4 + s) * 3;
        const float p = tr[0], u = tr[2 * NF], v = tr[4 * NF];
        w_out[e0 * 4 * NF + item] = characteristic32(p, u, v, sd[0], sd[1]);
        if (__builtin_amdgcn_inverse_ballot_w64(with_record[it]) || (flags & kTraceAll)) {
            float *to = tr_out + (e0 + fe) * 12 * NF + s * 3 * NF + k;
            to[0] = p;
            to[NF] = u;
            to[2 * NF] = v;
        }
    }
}

template <int N>
struct StageTile32 {
    static constexpr int EPB = LineShape<N>::EPB, NF = N + 1, tile = EPB * 3 * NF * (NF | 1), flux = EPB * 12 * NF,
                         met = EPB * 4 * NF, side = EPB * 12, lds = 2 * tile + flux + met + side;
};

template <int N>
__global__ void __launch_bounds__(192) __attribute__((amdgpu_waves_per_eu(N <= 9 ? 5 : 4)))
stage_c32_kernel(const double *__restrict__ verts, const int32_t *__restrict__ side_nb,
                 const BcSide *__restrict__ bc, const double *__restrict__ tab64,
                 const float *__restrict__ tab, float *__restrict__ qh, float2 *__restrict__ gl,
                 const float *__restrict__ w_in, float *__restrict__ w_out, const float *__restrict__ tr_in,
                 float *__restrict__ tr_out, const float *__restrict__ side_flux, int64_t K, int flags, float a, float gdt,
                 StageClock clock, int remap, double cw) {
    using L = StageTile32<N>;
    __shared__ float s_q[L::tile], s_d[L::tile], s_f[L::flux], s_met[L::met], s_side[L::side];
    stage_c32_tile<N, false>(verts, side_nb, bc, tab64, tab, qh, gl, w_in, w_out, tr_in, tr_out, side_flux, K, flags, a, gdt, clock,
                      cw, remap ? xcd_block(blockIdx.x, gridDim.x) : (int64_t)blockIdx.x, s_q, s_d, s_f, s_met, s_side);
}

// The stage of a mesh with mortar faces.
template <int N>
__global__ void __launch_bounds__(192) __attribute__((amdgpu_waves_per_eu(N <= 9 ? 5 : 4)))
stage_c32_mortar_kernel(const double *__restrict__ verts, const int32_t *__restrict__ side_nb,
                        const BcSide *__restrict__ bc, const double *__restrict__ tab64,
                        const float *__restrict__ tab, float *__restrict__ qh, float2 *__restrict__ gl,
                        const float *__restrict__ w_in, float *__restrict__ w_out, const float *__restrict__ tr_in,
                        float *__restrict__ tr_out, const float *__restrict__ side_flux, int64_t K, int flags, float a, float gdt,
                        StageClock clock, int remap, double cw) {
    using L = StageTile32<N>;
    __shared__ float s_q[L::tile], s_d[L::tile], s_f[L::flux], s_met[L::met], s_side[L::side];
    stage_c32_tile<N, true>(verts, side_nb, bc, tab64, tab, qh, gl, w_in, w_out, tr_in, tr_out, side_flux, K, flags, a, gdt, clock,
                      cw, remap ? xcd_block(blockIdx.x, gridDim.x) : (int64_t)blockIdx.x, s_q, s_d, s_f, s_met, s_side);
}

template <int N>
constexpr int most_stage_lds32() {
    if constexpr (N == 1) return StageTile32<1>::lds;
    else return max_stage_lds(StageTile32<N>::lds, most_stage_lds32<N - 1>());
}

// stage_groups_kernel for the FP32 form.
template <int Top>
__global__ void __launch_bounds__(192) __attribute__((amdgpu_waves_per_eu(Top <= 8 ? 5 : Top <= 12 ? 4 : 3)))
stage_c32_groups_kernel(StageGroups groups, const double *__restrict__ verts, const int32_t *__restrict__ side_nb,
                        const BcSide *__restrict__ bc, float *__restrict__ qh, float2 *__restrict__ gl,
                        const float *__restrict__ w_in, float *__restrict__ w_out, const float *__restrict__ tr_in,
                        float *__restrict__ tr_out, const float *__restrict__ side_flux, int flags, float a, float gdt,
                        StageClock clock, double cw) {
    __shared__ float mem[most_stage_lds32<Top>()];
    run_group<Top>(groups, [&](auto order, const StageGroups::Part &G, int64_t blk) {
        constexpr int N = decltype(order)::value;
        using L = StageTile32<N>;
        float *s_f = mem + 2 * L::tile, *s_met = s_f + L::flux;
        stage_c32_tile<N, true>(verts + G.e_begin * 8, side_nb + G.e_begin * 4, bc, G.tab, G.tab32, qh + G.q_off, gl + G.g_off,
                          w_in + G.tr_off / 3, w_out + G.tr_off / 3, tr_in + G.tr_off, tr_out + G.tr_off, side_flux,
                          G.K, flags, a, gdt, clock, cw, blk, mem, mem + L::tile, s_f, s_met, s_met + L::met);
    });
}

// ---------------------------------------------------------------------------------------------
// Initial conditions (src/meshes/Mesh2D_t.cpp:1192-1216; pulses have no reference counterpart).
template <int N>
__global__ void ic_kernel(const double *__restrict__ verts, const double *__restrict__ tab,
                          double *__restrict__ q, int64_t K, int kind, int n_pulses,
                          const double *__restrict__ pulses, double Lx, double Ly) {
    constexpr int NF = N + 1, NE = NF * NF;
    const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= K * NE) return;
    const int64_t e = gid / NE;
    const int node = (int)(gid % NE), i = node / NF, j = node % NF;
    const double *x = tab + NF * NF + 3 * NF;
    const double *P = verts + e * 8;
    const double xi = x[i], eta = x[j];
    const double X = (P[0] * (1 - xi) * (1 - eta) + P[2] * (xi + 1) * (1 - eta) +
                      P[4] * (xi + 1) * (eta + 1) + P[6] * (1 - xi) * (eta + 1)) / 4;
    const double Y = (P[1] * (1 - xi) * (1 - eta) + P[3] * (xi + 1) * (1 - eta) +
                      P[5] * (xi + 1) * (eta + 1) + P[7] * (1 - xi) * (eta + 1)) / 4;
    double p = 0.0, u = 0.0, v = 0.0;
    if (kind == NDG_IC_PLANE_WAVE) {
        plane_wave(X, Y, 0.0, 1.0, p, u, v);
    } else if (kind == NDG_IC_PERIODIC_PULSES) {
        // the 3 x 3 periodic images of each pulse, (mx, my) in {-1, 0, 1}^2
        for (int k = 0; k < n_pulses; ++k) {
            const double w = pulses[4 * k + 2];
            for (int mx = -1; mx <= 1; ++mx)
                for (int my = -1; my <= 1; ++my) {
                    const double dx = X - (pulses[4 * k] + mx * Lx), dy = Y - (pulses[4 * k + 1] + my * Ly);
                    p += pulses[4 * k + 3] * exp(-M_LN2 * (dx * dx + dy * dy) / (w * w));
                }
        }
    } else {
        for (int k = 0; k < n_pulses; ++k) {
            const double dx = X - pulses[4 * k], dy = Y - pulses[4 * k + 1], w = pulses[4 * k + 2];
            p += pulses[4 * k + 3] * exp(-M_LN2 * (dx * dx + dy * dy) / (w * w));
        }
    }
    double *qe = q + e * 3 * NE + node;
    qe[0] = p;
    qe[NE] = u;
    qe[2 * NE] = v;
}

// ---------------------------------------------------------------------------------------------
// CFL time step: min over elements of CFL * delta_min / (N^2 c) (src/solvers/Solver2D_t.cpp:19-29,
// Element2D_t.cpp:772-775), reduced in two passes on the device; no host round trip per block.
__device__ __forceinline__ double edge_len(const double *P, int a, int b) {
#pragma clang fp contract(off)
    const double dx = P[2 * a] - P[2 * b], dy = P[2 * a + 1] - P[2 * b + 1];
    return sqrt(dx * dx + dy * dy);
}

__device__ __forceinline__ double wave_min(double v) {
    for (int off = 32; off > 0; off >>= 1) v = fmin(v, __shfl_down(v, off, 64));
    return v;
}

__global__ void __launch_bounds__(256)
dt_partial_kernel(const double *__restrict__ verts, int64_t K, int N, double cfl, double cw,
                  double *__restrict__ partial) {
#pragma clang fp contract(off)
    __shared__ double s_min[4];
    double v = INFINITY;
    for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < K; e += (int64_t)gridDim.x * 256) {
        const double *P = verts + e * 8;
        const double d = fmin(fmin(fmin(edge_len(P, 1, 0), edge_len(P, 2, 3)),
                                   fmin(edge_len(P, 1, 2), edge_len(P, 0, 3))),
                              fmin(edge_len(P, 1, 3), edge_len(P, 2, 0)));
        v = fmin(cfl * d / (N * N * cw), v);
    }
    v = wave_min(v);
    if ((threadIdx.x & 63) == 0) s_min[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) partial[blockIdx.x] = fmin(fmin(s_min[0], s_min[1]), fmin(s_min[2], s_min[3]));
}

__global__ void __launch_bounds__(256)
dt_final_kernel(const double *__restrict__ partial, int n, double *__restrict__ out) {
    __shared__ double s_min[4];
    double v = INFINITY;
    for (int k = threadIdx.x; k < n; k += 256) v = fmin(v, partial[k]);
    v = wave_min(v);
    if ((threadIdx.x & 63) == 0) s_min[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) out[0] = fmin(fmin(s_min[0], s_min[1]), fmin(s_min[2], s_min[3]));
}

// ---------------------------------------------------------------------------------------------
// Pressure estimator (src/entities/Element2D_t.cpp:274-343): spectrum of the last
// min(N+1, 4) modal indices, least-squares fit of its log-decay, error and flags. FP64 throughout.
// out[e] = {error, sigma, refine, coarsen}.
//
// A thread forms the coefficient pair (i, pm), (pm, i) of one element, or its (pm, pm), from the element's nodes in
// LDS and the two modes' rows in registers; the sums of each spectrum entry and the fit follow in the
// order of the loops they restate (the fit is ill-conditioned, so the order is kept to the bit). Bound
// by FP64 arithmetic. With one thread an element, each walking its own lines of memory, 256 x 256, N = 8
// took 188 us and 400 elements of order 12 some 150 us; now 41 and 8 us.
template <int N>
struct EstimateShape {
    static constexpr int NF = N + 1, n = NF < 4 ? NF : 4, low = N + 1 - n;  // the first modal index
    __host__ __device__ static constexpr int first(int ni) { return ni * (low + 1) + ni * (ni - 1) / 2; }
    static constexpr int tasks = first(n);  // pm + 1 for each pm of [low, N]
    static constexpr int T = 256, EPB = T / tasks;
};

template <int N>
__global__ void __launch_bounds__(256)
estimate_kernel(const double *__restrict__ tab, const double *__restrict__ q, int64_t K,
                double tol_min, double tol_max, double *__restrict__ out) {
    using S = EstimateShape<N>;
    constexpr int NF = N + 1, NE = NF * NF, n = S::n, tasks = S::tasks, T = S::T, EPB = S::EPB;
    __shared__ double s_m[NE], s_p[EPB * NE], s_v[EPB * tasks], s_spec[EPB * n], s_log[EPB * n];
    const int tid = threadIdx.x;
    const int64_t e0 = (int64_t)blockIdx.x * EPB;
    const int nel = (int)min<int64_t>(EPB, K - e0);
    for (int r = tid; r < NE; r += T) s_m[r] = tab[NF * NF + 5 * NF + r];
    for (int r = tid; r < nel * NE; r += T) s_p[r] = q[(e0 + r / NE) * 3 * NE + r % NE];
    __syncthreads();
    if (tid < nel * tasks) {
        const int t = tid % tasks;
        int ni = 0;
#pragma unroll
        for (int k = 1; k < n; ++k) ni += t >= S::first(k);
        const int i = t - S::first(ni), pm = S::low + ni;
        const double *p = s_p + tid / tasks * NE, *Mi = s_m + i * NF, *Mp = s_m + pm * NF;
        double mi[NF], mp[NF];
#pragma unroll
        for (int l = 0; l < NF; ++l) {
            mi[l] = Mi[l];
            mp[l] = Mp[l];
        }
        double lx = 0.0, ly = 0.0;
        for (int k = 0; k < NF; ++k) {
            const double mik = Mi[k], mpk = Mp[k];
#pragma unroll
            for (int l = 0; l < NF; ++l) {
                const double v = p[k * NF + l];
                lx = fma(v * mik, mp[l], lx);
                ly = fma(v * mpk, mi[l], ly);
            }
        }
        s_v[tid] = i == pm ? fabs(lx) : fabs(lx) + fabs(ly);
    }
    __syncthreads();
    if (tid < nel * n) {
        const int ni = tid % n;
        const double *v = s_v + tid / n * tasks + S::first(ni);
        double spec = 0.0;
        for (int i = 0; i <= S::low + ni; ++i) spec += v[i];
        s_spec[tid] = spec;
        s_log[tid] = log(spec);
    }
    __syncthreads();
    if (tid >= nel) return;
    const double *ls = s_log + tid * n;
    double xa = 0.0, ya = 0.0;
    for (int i = 0; i < n; ++i) {
        xa += S::low + i;
        ya += ls[i];
    }
    xa /= n;
    ya /= n;
    double num = 0.0, den = 0.0;
    for (int i = 0; i < n; ++i) {
        const int pp = S::low + i;
        num += (pp - xa) * (ls[i] - ya);
        den += (pp - xa) * (pp - xa);
    }
    const double sig = num / den;
    const double C = exp(ya - sig * xa);
    const double sigma = fabs(sig);
    const double last = s_spec[tid * n + n - 1];
    const double err = sqrt(fma(last, last, C * C * 0.5 / sigma * exp(-2 * sigma * (N + 1))));
    double *o = out + 4 * (e0 + tid);
    o[0] = err;
    o[1] = sigma;
    o[2] = err > tol_min ? 1.0 : 0.0;
    o[3] = err < tol_max ? 1.0 : 0.0;
}

// ---------------------------------------------------------------------------------------------
// Sets a value of the device clock (DeviceMesh::clock).
__global__ void clock_set_kernel(double *clock, double t) {
    if (threadIdx.x == 0) *clock = t;
}

// ---------------------------------------------------------------------------------------------
// Non-conforming (mortar) faces, FP64 arithmetic (the traces and the output are of type T: double,
// or float in the FP32 form). Restates, for one face:
//   project_to_faces (src/meshes/Mesh2D_t.cpp:3803-3893): each side's trace is copied when the
//     element order equals the face order, else interpolated barycentrically at
//     xi = (x_face + 1) scale + 2 offset - 1 with the exact-node shortcut (right side reversed);
//   calculate_wave_fluxes (src/solvers/Solver2D_t.cpp:48-63);
//   project_to_elements (src/meshes/Mesh2D_t.cpp:3895-4003): conforming copy (left forward, right
//     backward and negated) or the Gauss-quadrature L2 projection, times the edge Jacobian and the
//     face scale, accumulated over face nodes in order.

__device__ __forceinline__ bool ulp2_equal(double a, double b) {
    return fabs(a - b) <= DBL_EPSILON * fabs(a + b) * 2 || fabs(a - b) < DBL_MIN;
}

// Loads n <= 32 * kMaxItems values src[0..n) into dst through registers, every load in flight
// before the first LDS write (lane i of a 32-lane half takes items i, i + 32, ...).
template <typename T, int kMaxItems>
__device__ __forceinline__ void stage_to_lds(const T *__restrict__ src, double *dst, int n, int i) {
    double v[kMaxItems];
#pragma unroll
    for (int it = 0; it < kMaxItems; ++it) {
        const int idx = i + 32 * it;
        v[it] = idx < n ? (double)src[idx] : 0.0;
    }
#pragma unroll
    for (int it = 0; it < kMaxItems; ++it) {
        const int idx = i + 32 * it;
        if (idx < n) dst[idx] = v[it];
    }
}

// One wave per face: lanes 0..31 handle the left side, lanes 32..63 the right side. Each half first
// stages its element trace and its interpolation and projection matrices (built on the host with
// the reference's exact-node shortcuts, see MortarFace) into LDS with all loads in flight, then
// lane i computes face node i (interpolation) and element node i (projection); face states and
// flux go through LDS. M bounds N + 1 of every face and side (checked on the host when the kernel
// is chosen): a smaller M gives a smaller LDS footprint and more faces resident per CU.
template <typename T, int M>
__global__ void __launch_bounds__(64)
mortar_kernel(const MortarFace *__restrict__ faces, const double *__restrict__ mats,
              const T *__restrict__ tr, T *__restrict__ side_flux) {
    constexpr int kMat = M * M, kMatItems = (kMat + 31) / 32, kTrItems = (3 * M + 31) / 32;
    __shared__ double s_tr[2][3 * M];   // element traces, left and right
    __shared__ double s_mi[2][kMat];    // interpolation matrices [face node][element node]
    __shared__ double s_mp[2][kMat];    // projection matrices [element node][face node]
    __shared__ double s_st[2][3][M];    // face states, left and right
    __shared__ double s_f[3][M];        // face flux
    const MortarFace fc = faces[blockIdx.x];
    const int lane = threadIdx.x;
    const int side = lane >> 5, i = lane & 31;
    const int Nf = fc.Nf;
    const int Ne = side ? fc.NR : fc.NL;
    // selects, not fc.mat[side]: a lane-dependent index would put the whole record in scratch
    const int64_t mi = side ? fc.mat[1] : fc.mat[0], mp = side ? fc.mat[3] : fc.mat[2];
    stage_to_lds<T, kTrItems>(tr + (side ? fc.trR : fc.trL), s_tr[side], 3 * (Ne + 1), i);
    if (mi >= 0) stage_to_lds<double, kMatItems>(mats + mi, s_mi[side], (Nf + 1) * (Ne + 1), i);
    if (mp >= 0) stage_to_lds<double, kMatItems>(mats + mp, s_mp[side], (Ne + 1) * (Nf + 1), i);
    __syncthreads();
    // project_to_faces (src/meshes/Mesh2D_t.cpp:3803-3893)
    if (i <= Nf) {
        const double *te = s_tr[side];
        double v0 = 0.0, v1 = 0.0, v2 = 0.0;
        if (mi < 0) {
            const int k = side ? Nf - i : i;
            v0 = te[k];
            v1 = te[(Ne + 1) + k];
            v2 = te[2 * (Ne + 1) + k];
        } else {
            // unrolled to M with every LDS read issued unconditionally (all in bounds: i <= Nf < M,
            // j < M), only the terms j <= Ne accumulated, in the same order
            const double *row = s_mi[side] + i * (Ne + 1);
#pragma unroll
            for (int j = 0; j < M; ++j) {
                const double w = row[j], a0 = te[j], a1 = te[(Ne + 1) + j], a2 = te[2 * (Ne + 1) + j];
                if (j <= Ne) {
                    v0 += w * a0;
                    v1 += w * a1;
                    v2 += w * a2;
                }
            }
        }
        s_st[side][0][i] = v0;
        s_st[side][1][i] = v1;
        s_st[side][2][i] = v2;
    }
    __syncthreads();
    // calculate_wave_fluxes (src/solvers/Solver2D_t.cpp:48-63)
    if (lane <= Nf) {
        const double c = kWaveSpeed;
        const double wl = s_st[0][0][lane] + c * (s_st[0][1][lane] * fc.nx + s_st[0][2][lane] * fc.ny);
        const double wr = s_st[1][0][lane] - c * (s_st[1][1][lane] * fc.nx + s_st[1][2][lane] * fc.ny);
        s_f[0][lane] = c * (wl - wr) / 2;
        s_f[1][lane] = fc.nx * (wl + wr) / 2;
        s_f[2][lane] = fc.ny * (wl + wr) / 2;
    }
    __syncthreads();
    // project_to_elements (src/meshes/Mesh2D_t.cpp:3895-4006), times the edge Jacobian
    const int64_t slot = side ? fc.slotR : fc.slotL;
    if (slot < 0 || i > Ne) return;
    const double sf = side ? fc.sfR : fc.sfL;
    T *out = side_flux + slot;
    if (mp < 0) {
        for (int f = 0; f < 3; ++f)
            out[f * (Ne + 1) + i] = side ? (T)(-s_f[f][Nf - i] * sf) : (T)(s_f[f][i] * sf);
        return;
    }
    const double *row = s_mp[side] + i * (Nf + 1);
    double a0 = 0.0, a1 = 0.0, a2 = 0.0;
#pragma unroll
    for (int j = 0; j < M; ++j) {  // as the interpolation: i <= Ne < M, j < M
        const double w = row[j], f0 = s_f[0][j], f1 = s_f[1][j], f2 = s_f[2][j];
        if (j <= Nf) {
            a0 += w * f0;
            a1 += w * f1;
            a2 += w * f2;
        }
    }
    out[i] = (T)(a0 * sf);
    out[(Ne + 1) + i] = (T)(a1 * sf);
    out[2 * (Ne + 1) + i] = (T)(a2 * sf);
}

// ---------------------------------------------------------------------------------------------
// Launchers: dispatch on the (uniform) order N.
// ---------------------------------------------------------------------------------------------
// Solution transfer after adaptation, one workgroup per new element: a copy when neither order nor
// geometry changes, else Element2D_t::interpolate_from (src/entities/Element2D_t.cpp:345-579) at
// the new nodes (same geometry) or at the given reference coordinates in the old element (a child):
// the old element's node when both coordinates match a node (almost_equal, the last matching
// index wins), a 1D barycentric interpolation along the other coordinate when one matches, else
// the tensor barycentric interpolation.
__global__ void __launch_bounds__(256)
transfer_kernel(const double *__restrict__ q_old, double *__restrict__ q_new,
                const TransferRec *__restrict__ recs, const double *__restrict__ coords,
                const double *__restrict__ tab1d) {
    const TransferRec R = recs[blockIdx.x];
    const int No = R.N_old, Nn = R.N_new, nfo = No + 1, nf = Nn + 1, neo = nfo * nfo, ne = nf * nf;
    const double *src = q_old + R.old_off;
    double *dst = q_new + R.new_off;
    if (No == Nn && R.coord_off < 0) {
        for (int r = threadIdx.x; r < 3 * ne; r += 256) dst[r] = src[r];
        return;
    }
    const double *xo = tab1d + (3 * No + 0) * kTab1dStride, *lo = tab1d + (3 * No + 2) * kTab1dStride;
    const double *xn = tab1d + (3 * Nn + 0) * kTab1dStride;
    for (int r = threadIdx.x; r < 3 * ne; r += 256) {
        const int f = r / ne, node = r % ne, i = node / nf, j = node % nf;
        const double X = R.coord_off >= 0 ? coords[R.coord_off + 2 * node] : xn[i];
        const double Y = R.coord_off >= 0 ? coords[R.coord_off + 2 * node + 1] : xn[j];
        dst[r] = interpolate_at(src + f * neo, No, X, Y, xo, lo);
    }
}

hipError_t launch_transfer(const double *q_old, double *q_new, const TransferRec *recs, const double *coords,
                           int64_t K, const double *tab1d, hipStream_t s) {
    if (K <= 0) return hipSuccess;
    hipLaunchKernelGGL(transfer_kernel, dim3((unsigned)K), dim3(256), 0, s, q_old, q_new, recs, coords, tab1d);
    return hipGetLastError();
}

// Mesh2D_t::get_solution (src/meshes/Mesh2D_t.cpp:4237-4249) with
// Element2D_t::interpolate_solution (src/entities/Element2D_t.cpp:581-604): for each element (one
// workgroup, caller's order) and output point (i, j) of the n x n uniform grid, x and y by the
// bilinear map at ((i / (n - 1)) * 2 - 1, (j / (n - 1)) * 2 - 1), and each field as
// sum_m sum_k q[m][k] I[i][m] I[j][k] with the order's uniform-grid interpolation matrix I.
// With rhs given, also Mesh2D_t::get_complete_solution (src/meshes/Mesh2D_t.cu:5096-5155,
// src/entities/Element2D_t.cu:623-665): the right-hand side (laid out as q) and
// |g(x_mk, time) - q[m][k]| of the plane wave at the solution nodes, interpolated
// with the same weights. The element's state, right-hand side and node errors are staged in LDS.
// Output layout [x, y, p, u, v (, dp, du, dv, |dp|, |du|, |dv|)][element][i * n + j].
constexpr int kOutMaxNe = (kMaxOrder + 1) * (kMaxOrder + 1);

__global__ __launch_bounds__(64) void output_kernel(const double *__restrict__ q, const double *__restrict__ rhs,
                                                    const double *__restrict__ verts,
                                                    const OutputRec *__restrict__ recs,
                                                    const double *__restrict__ interp,
                                                    const double *__restrict__ tab1d, int n, int64_t K,
                                                    double time, double cw, double *__restrict__ out) {
    __shared__ double s_q[3 * kOutMaxNe], s_r[3 * kOutMaxNe], s_a[3 * kOutMaxNe];
    const int64_t e = blockIdx.x;
    const OutputRec R = recs[e];
    const int nf = R.N + 1, ne = nf * nf, nn = n * n;
    const double *I = interp + R.i_off;
    const double *P = verts + 8 * R.dev;
    const double *src = q + R.q_off;
    const bool complete = rhs != nullptr;
    const double *nodes = tab1d + 3 * R.N * kTab1dStride;
    for (int r = threadIdx.x; r < 3 * ne; r += 64) {
        const double v = src[r];
        s_q[r] = v;
        if (complete) {
            const int c = r / ne, mk = r - c * ne, m = mk / nf, k = mk - m * nf;
            s_r[r] = rhs[R.q_off + r];
            const double xi = nodes[m], eta = nodes[k];
            const double w0 = (1 - xi) * (1 - eta), w1 = (xi + 1) * (1 - eta), w2 = (xi + 1) * (eta + 1),
                         w3 = (1 - xi) * (eta + 1);
            const double X = (P[0] * w0 + P[2] * w1 + P[4] * w2 + P[6] * w3) / 4;
            const double Y = (P[1] * w0 + P[3] * w1 + P[5] * w2 + P[7] * w3) / 4;
            double g[3];
            plane_wave(X, Y, time, cw, g[0], g[1], g[2]);
            s_a[r] = fabs(g[c] - v);
        }
    }
    __syncthreads();
    const int64_t plane = K * nn;
    for (int r = threadIdx.x; r < nn; r += 64) {
        const int i = r / n, j = r % n;
        const double xi = (double)i / (double)(n - 1) * 2 - 1, eta = (double)j / (double)(n - 1) * 2 - 1;
        const double w0 = (1 - xi) * (1 - eta), w1 = (xi + 1) * (1 - eta), w2 = (xi + 1) * (eta + 1),
                     w3 = (1 - xi) * (eta + 1);
        const double x = (P[0] * w0 + P[2] * w1 + P[4] * w2 + P[6] * w3) / 4;
        const double y = (P[1] * w0 + P[3] * w1 + P[5] * w2 + P[7] * w3) / 4;
        double f[9] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
        for (int m = 0; m < nf; ++m) {
            const double a = I[i * nf + m];
            for (int k = 0; k < nf; ++k) {
                const double b = I[j * nf + k];
                const int mk = m * nf + k;
                for (int c = 0; c < 3; ++c) f[c] += s_q[c * ne + mk] * a * b;
                if (complete)
                    for (int c = 0; c < 3; ++c) {
                        f[3 + c] += s_r[c * ne + mk] * a * b;
                        f[6 + c] += s_a[c * ne + mk] * a * b;
                    }
            }
        }
        const int64_t at = e * nn + r;
        out[at] = x;
        out[plane + at] = y;
        const int nfield = complete ? 9 : 3;
        for (int c = 0; c < nfield; ++c) out[(2 + c) * plane + at] = f[c];
    }
}

hipError_t launch_output(const double *q, const double *rhs, const double *verts, const OutputRec *recs,
                         const double *interp, const double *tab1d, int n, int64_t K, double time, double cw,
                         double *out, hipStream_t s) {
    if (K <= 0) return hipSuccess;
    hipLaunchKernelGGL(output_kernel, dim3((unsigned)K), dim3(64), 0, s, q, rhs, verts, recs, interp, tab1d, n, K,
                       time, cw, out);
    return hipGetLastError();
}

#define NDG_FOR_ORDERS(X) X(1) X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(11) X(12) X(13) X(14) X(15) X(16)
bool order_supported(int N) { return N >= 1 && N <= kMaxOrder; }

#define CASES_1(F, ...) \
    case 1: return F<1>(__VA_ARGS__); case 2: return F<2>(__VA_ARGS__); case 3: return F<3>(__VA_ARGS__); \
    case 4: return F<4>(__VA_ARGS__); case 5: return F<5>(__VA_ARGS__); case 6: return F<6>(__VA_ARGS__); \
    case 7: return F<7>(__VA_ARGS__); case 8: return F<8>(__VA_ARGS__); case 9: return F<9>(__VA_ARGS__); \
    case 10: return F<10>(__VA_ARGS__); case 11: return F<11>(__VA_ARGS__); case 12: return F<12>(__VA_ARGS__); \
    case 13: return F<13>(__VA_ARGS__); case 14: return F<14>(__VA_ARGS__); case 15: return F<15>(__VA_ARGS__); \
    case 16: return F<16>(__VA_ARGS__);

// Launchers: every per-element kernel runs once per order group, on the group's slices of the
// device buffers.

template <int N>
static hipError_t traces_n(const DeviceMesh &m, const Group &G, hipStream_t s) {
    using S = Shape<N>;
    const int64_t blocks = (G.K + S::EPB - 1) / S::EPB;
    hipLaunchKernelGGL(traces_kernel<N>, dim3((unsigned)blocks), dim3(S::THREADS), 0, s, m.verts + G.e_begin * 8,
                       m.side_nb + G.e_begin * 4, m.bc, G.tab, m.q + G.q_off, m.trace[m.cur] + G.tr_off,
                       m.wave[m.cur] + G.tr_off / 3, G.K);
    return hipGetLastError();
}

// Elements per workgroup actually used for group G (a tuning choice, at most the shape's EPB).
template <int N>
static int group_epb(const Group &G, int precision) {
    const int e = G.tune[precision].epb;
    return e >= 1 && e <= LineShape<N>::EPB ? e : LineShape<N>::EPB;
}

template <int N>
static int stage_epb_n(const Group &G) {
    return group_epb<N>(G, NDG_PRECISION_FP64);
}

int stage_tile_epb(const Group &G) {
    switch (G.N) { CASES_1(stage_epb_n, G) }
    return 1;
}

template <int N>
static int stage_run_n(int epb) { return rk_run<N>(epb); }

int stage_run(int N, int epb) {
    switch (N) { CASES_1(stage_run_n, epb) }
    return 0;
}

int stage_tile_run(const Group &G) { return stage_run(G.N, stage_tile_epb(G)); }

// Enough for every tile size a launch may take: a last tile with few elements is as long as a full one,
// so that for few elements neither the largest size nor the smallest needs the most.
template <int N>
static int64_t rk_values_n(int64_t K) {
    int64_t most = 0;
    for (int epb = 1; epb <= LineShape<N>::EPB; ++epb) most = std::max(most, (K + epb - 1) / epb * rk_run<N>(epb));
    return 3 * (N + 1) * most;
}

int64_t stage_rk_values(int N, int64_t K) {
    switch (N) { CASES_1(rk_values_n, K) }
    return 0;
}

// The state and the RK register go past the caches when a stage's bytes (these, both buffers of
// characteristics, vertices and codes) no longer fit the last-level cache of 256 MB from one stage to the
// next, so that they leave room for what is read again. Measured, us a stage past and through the caches,
// FP64: N = 8: 200 x 200 (182 MB) 55.4 and 48.8, 216 x 216 (212 MB) 60.9 and 55.4, 232 x 232 (245 MB) 71.6
// and 64.3, 248 x 248 (279 MB) 79.5 and 78.2, 264 x 264 (317 MB) 92.0 and 92.7, 512 x 512 (1.2 GB) 324 and
// 401; N = 12: 160 x 160 (231 MB) 76.1 and 67.9; N = 4: 360 x 360 (207 MB) 60.4 and 55.7, 384 x 384 (236 MB)
// 67.6 and 74.4, 400 x 400 (256 MB) 74.1 and 80.5; N = 2: 580 x 580 (237 MB) 73.0 and 66.8; N = 6: 288 x 288
// (239 MB) 68.1 and 71.0. The FP32 form: N = 8: 224 x 224 (165 MB) 58.1 and 52.5, 256 x 256 (215 MB) 80.4 and
// 65.7, 264 x 264 (229 MB) 87.5 and 70.7, 272 x 272 (243 MB) 89.1 and 91.7, 288 x 288 (272 MB) 99.7 and 108,
// 512 x 512 (861 MB) 271 and 287; N = 12: 184 x 184 (223 MB) 84.8 and 76.9, 192 x 192 (243 MB) 96.8 and 95.4;
// N = 4: 460 x 460 (241 MB) 84.7 and 72.9, 480 x 480 (263 MB) 89.6 and 98.4.
static int stage_flags(const DeviceMesh &m, int precision) {
    const bool c32 = precision == NDG_PRECISION_FP32_COMPENSATED;
    const int64_t bytes = (c32 ? 12 : 16) * m.n_q + (c32 ? 8 : 16) * (m.n_tr / 3) + 80 * m.K;
    return (m.trace_all ? kTraceAll : 0) | (bytes > kStreamBytes[precision] ? kStream : 0);
}

// The clock has a start time for each trace buffer that a step can begin with: three stages flip it
// three times, so the next step begins with the other one.
static StageClock stage_clock(const DeviceMesh &m, const Group &G, int stage, double dt) {
    constexpr double kB[3] = {0.0, 1.0 / 3.0, 0.75};
    const int begin = m.cur ^ (stage & 1);
    double *next = stage == 2 && m.has_inflow && &G == &m.groups[0] ? m.clock + (1 - begin) : nullptr;
    return StageClock{m.clock + begin, kB[stage] * dt, next, dt};
}

static int stage_rk_flags(const DeviceMesh &m, int stage) {
    return (stage == 0 ? kRkFirst : 0) | (stage == 2 && !m.keep_last_rk ? kRkLast : 0) | stage_flags(m, NDG_PRECISION_FP64);
}

template <int N>
static hipError_t stage_n(DeviceMesh &m, const Group &G, int stage, double a, double gdt, double dt, hipStream_t s) {
    using S = LineShape<N>;
    const int epb = group_epb<N>(G, NDG_PRECISION_FP64);
    const int64_t blocks = (G.K + epb - 1) / epb;
    auto *const kernel = m.n_faces ? stage_mortar_kernel<N> : stage_kernel<N, false>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(S::T), 0, s, m.verts + G.e_begin * 8,
                       m.side_nb + G.e_begin * 4, m.bc, G.tab, m.q + G.q_off, (m.q_out ? m.q_out : m.q) + G.q_off,
                       m.g + G.g_off, m.wave[m.cur] + G.tr_off / 3, m.wave[1 - m.cur] + G.tr_off / 3,
                       m.trace[m.cur] + G.tr_off,
                       m.trace[1 - m.cur] + G.tr_off, nullptr, m.side_flux, G.K,
                       stage_rk_flags(m, stage), a, gdt,
                       stage_clock(m, G, stage, dt), epb, G.tune[NDG_PRECISION_FP64].remap, m.wave_speed);
    return hipGetLastError();
}

template <int N>
static hipError_t rhs_n(DeviceMesh &m, const Group &G, hipStream_t s) {
    using S = LineShape<N>;
    const int64_t blocks = (G.K + S::EPB - 1) / S::EPB;
    hipLaunchKernelGGL((stage_kernel<N, true>), dim3((unsigned)blocks), dim3(S::T), 0, s, m.verts + G.e_begin * 8,
                       m.side_nb + G.e_begin * 4, m.bc, G.tab, m.q + G.q_off, m.q + G.q_off, nullptr,
                       m.wave[m.cur] + G.tr_off / 3, nullptr, m.trace[m.cur] + G.tr_off, nullptr, m.rhs + G.q_off, m.side_flux,
                       G.K, stage_flags(m, NDG_PRECISION_FP64), 0.0, 0.0,
                       StageClock{m.clock + kRhsClock, 0.0, nullptr, 0.0}, S::EPB, 1, m.wave_speed);
    return hipGetLastError();
}

template <int N>
static hipError_t ic_n(const DeviceMesh &m, const Group &G, int kind, int n_pulses, const double *pulses,
                       double Lx, double Ly, hipStream_t s) {
    const int64_t total = G.K * (N + 1) * (N + 1);
    hipLaunchKernelGGL(ic_kernel<N>, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, m.verts + G.e_begin * 8,
                       G.tab, m.q + G.q_off, G.K, kind, n_pulses, pulses, Lx, Ly);
    return hipGetLastError();
}

template <int N>
static hipError_t estimate_n(const DeviceMesh &m, const Group &G, double tol_min, double tol_max, double *out,
                             hipStream_t s) {
    using S = EstimateShape<N>;
    hipLaunchKernelGGL(estimate_kernel<N>, dim3((unsigned)((G.K + S::EPB - 1) / S::EPB)), dim3(S::T), 0, s, G.tab,
                       m.q + G.q_off, G.K, tol_min, tol_max, out + 4 * G.e_begin);
    return hipGetLastError();
}

template <int N>
static hipError_t traces_c32_n(const DeviceMesh &m, const Group &G, hipStream_t s) {
    using S = LineShape<N>;
    const int64_t blocks = (G.K + S::EPB - 1) / S::EPB;
    hipLaunchKernelGGL(traces_c32_kernel<N>, dim3((unsigned)blocks), dim3(S::T), 0, s, m.verts + G.e_begin * 8,
                       m.side_nb + G.e_begin * 4, m.bc, G.tab32, m.qh + G.q_off, m.trace32[m.cur] + G.tr_off,
                       m.wave32[m.cur] + G.tr_off / 3, G.K);
    return hipGetLastError();
}

static int stage_c32_flags(const DeviceMesh &m, int stage) {
    return (stage == 0 ? kRkFirst : 0) | stage_flags(m, NDG_PRECISION_FP32_COMPENSATED);
}

template <int N>
static hipError_t stage_c32_n(DeviceMesh &m, const Group &G, int stage, double a, double gdt, double dt,
                              hipStream_t s) {
    using S = LineShape<N>;
    const int64_t blocks = (G.K + S::EPB - 1) / S::EPB;
    auto *const kernel = m.n_faces ? stage_c32_mortar_kernel<N> : stage_c32_kernel<N>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(S::T), 0, s, m.verts + G.e_begin * 8,
                       m.side_nb + G.e_begin * 4, m.bc, G.tab, G.tab32, m.qh + G.q_off, m.gl32 + G.g_off,
                       m.wave32[m.cur] + G.tr_off / 3, m.wave32[1 - m.cur] + G.tr_off / 3, m.trace32[m.cur] + G.tr_off,
                       m.trace32[1 - m.cur] + G.tr_off, m.side_flux32, G.K, stage_c32_flags(m, stage), (float)a, (float)gdt,
                       stage_clock(m, G, stage, dt), G.tune[NDG_PRECISION_FP32_COMPENSATED].remap, m.wave_speed);
    return hipGetLastError();
}

template <int N>
static int max_epb_n() { return LineShape<N>::EPB; }

int stage_max_epb(int N) {
    switch (N) { CASES_1(max_epb_n) }
    return 0;
}

hipError_t launch_group_stage(DeviceMesh &m, int group, int stage, double a, double gdt, double dt, hipStream_t s) {
    const Group &G = m.groups[group];
    if (m.precision == NDG_PRECISION_FP32_COMPENSATED) {
        switch (G.N) { CASES_1(stage_c32_n, m, G, stage, a, gdt, dt, s) }
    } else {
        switch (G.N) { CASES_1(stage_n, m, G, stage, a, gdt, dt, s) }
    }
    return hipErrorInvalidValue;
}

// Autotuning probe: stage 0 form with a = 0 and gdt = 0, so that the state and the current traces
// are left as they are.
hipError_t launch_group_probe(DeviceMesh &m, int group, hipStream_t s) {
    return launch_group_stage(m, group, 0, 0.0, 0.0, 0.0, s);
}



template <typename Fn>
static hipError_t for_groups(const DeviceMesh &m, Fn &&fn) {
    for (const Group &G : m.groups) {
        const hipError_t e = fn(G);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t launch_traces(const DeviceMesh &m, hipStream_t s) {
    return for_groups(m, [&](const Group &G) -> hipError_t {
        switch (G.N) { CASES_1(traces_n, m, G, s) }
        return hipErrorInvalidValue;
    });
}

template <int M>
static hipError_t mortar_m(DeviceMesh &m, hipStream_t s) {
    const unsigned blocks = (unsigned)m.n_faces;
    if (m.precision == NDG_PRECISION_FP32_COMPENSATED)
        hipLaunchKernelGGL((mortar_kernel<float, M>), dim3(blocks), dim3(64), 0, s, m.faces, m.mortar_mats,
                           m.trace32[m.cur], m.side_flux32);
    else
        hipLaunchKernelGGL((mortar_kernel<double, M>), dim3(blocks), dim3(64), 0, s, m.faces, m.mortar_mats,
                           m.trace[m.cur], m.side_flux);
    return hipGetLastError();
}

hipError_t launch_mortar(DeviceMesh &m, hipStream_t s) {
    if (m.n_faces == 0) return hipSuccess;
    static_assert(kMaxOrder + 1 <= 32, "a mortar side is handled by one 32-lane half wave");
    if (m.mortar_nodes < 1 || m.mortar_nodes > kMaxOrder + 1) return hipErrorInvalidValue;
    if (m.mortar_nodes <= 9) return mortar_m<9>(m, s);
    if (m.mortar_nodes <= 13) return mortar_m<13>(m, s);
    return mortar_m<kMaxOrder + 1>(m, s);
}

// Workgroups per group beyond the first up to which one launch takes the stages of all groups: each
// launch that it saves is worth some 6 us, and each workgroup costs a little more there, because its
// registers and LDS are those of the largest order compiled into the kernel (4 workgroups a CU up to order
// 8, 3 to order 12, 2 above). Measured, us a stage with one launch and with one a group, in parallel
// graph branches where these are the faster: orders 4, 6, 8: 4,184 workgroups 46.3 and 50.5, 7,438 69.4
// and 68.8; orders 10, 12: 944 workgroups 23.9 and 27.8, 3,774 58.5 and 55.0; orders 4 to 12 (5 groups):
// 549 workgroups 18.1 and 39.6, 3,421 50.1 and 58.1, 8,759 115 and 105; orders 14, 16: 693 workgroups
// 25.9 and 28.8, 2,770 64.9 and 61.7; orders 8 to 16 (5 groups): 1,900 workgroups 48.4 and 60.0, 3,377
// 69.9 and 67.4. The FP32 form, whose kernels lose less occupancy there, takes the same line: orders 4 to 12:
// 549 workgroups 18.1 and 39.3, 3,421 43.1 and 57.0; orders 10, 12: 944 workgroups 20.2 and 28.2.
static int64_t groups_blocks(int top) { return top <= 8 ? 2048 : top <= 12 ? 1152 : 640; }

static int stage_epb(const DeviceMesh &m, const Group &G) {
    return m.precision == NDG_PRECISION_FP32_COMPENSATED ? stage_max_epb(G.N) : stage_tile_epb(G);
}

template <int Top>
static hipError_t stage_groups_top(DeviceMesh &m, const StageGroups &P, int stage, double a, double gdt, double dt,
                                   hipStream_t s) {
    if (m.precision == NDG_PRECISION_FP32_COMPENSATED)
        hipLaunchKernelGGL(stage_c32_groups_kernel<Top>, dim3((unsigned)P.first[P.n]), dim3(192), 0, s, P, m.verts,
                           m.side_nb, m.bc, m.qh, m.gl32, m.wave32[m.cur], m.wave32[1 - m.cur], m.trace32[m.cur],
                           m.trace32[1 - m.cur], m.side_flux32, stage_c32_flags(m, stage), (float)a, (float)gdt,
                           stage_clock(m, m.groups[0], stage, dt), m.wave_speed);
    else
        hipLaunchKernelGGL(stage_groups_kernel<Top>, dim3((unsigned)P.first[P.n]), dim3(192), 0, s, P, m.verts, m.side_nb,
                           m.bc, m.q, m.q_out ? m.q_out : m.q, m.g, m.wave[m.cur], m.wave[1 - m.cur], m.trace[m.cur],
                           m.trace[1 - m.cur], m.side_flux, stage_rk_flags(m, stage), a, gdt,
                           stage_clock(m, m.groups[0], stage, dt), m.wave_speed);
    return hipGetLastError();
}

bool stage_groups_fit(const DeviceMesh &m) {
    if (m.groups.size() < 2) return false;
    int64_t blocks = 0;
    int top = 0;
    for (const Group &G : m.groups) {
        const int epb = stage_epb(m, G);
        blocks += (G.K + epb - 1) / epb;
        top = std::max(top, G.N);
    }
    return blocks <= groups_blocks(top) * (int64_t)(m.groups.size() - 1);
}

hipError_t launch_groups(DeviceMesh &m, int stage, double a, double gdt, double dt, hipStream_t s) {
    if (!stage_groups_fit(m)) {
        for (int g = 0; g < (int)m.groups.size(); ++g)
            if (const hipError_t e = launch_group_stage(m, g, stage, a, gdt, dt, s); e != hipSuccess) return e;
        return hipSuccess;
    }
    StageGroups P;
    P.n = (int)m.groups.size();
    P.first[0] = 0;
    int top = 0;
    for (int i = 0; i < P.n; ++i) {
        const Group &G = m.groups[i];
        const int epb = stage_epb(m, G);
        P.part[i] = {G.N, epb, G.tune[m.precision].remap, G.K, G.e_begin, G.q_off, G.tr_off, G.g_off, G.tab, G.tab32};
        P.first[i + 1] = P.first[i] + (int)((G.K + epb - 1) / epb);
        top = std::max(top, G.N);
    }
    if (top <= 8) return stage_groups_top<8>(m, P, stage, a, gdt, dt, s);
    if (top <= 12) return stage_groups_top<12>(m, P, stage, a, gdt, dt, s);
    return stage_groups_top<kMaxOrder>(m, P, stage, a, gdt, dt, s);
}

hipError_t launch_stage(DeviceMesh &m, int stage, double a, double gdt, double dt, hipStream_t s) {
    hipError_t e = launch_mortar(m, s);
    if (e != hipSuccess || (e = launch_groups(m, stage, a, gdt, dt, s)) != hipSuccess) return e;
    m.cur = 1 - m.cur;
    return hipSuccess;
}

hipError_t launch_rhs(DeviceMesh &m, double t, hipStream_t s) {
    if (m.has_inflow) hipLaunchKernelGGL(clock_set_kernel, dim3(1), dim3(64), 0, s, m.clock + kRhsClock, t);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if ((e = launch_mortar(m, s)) != hipSuccess) return e;
    return for_groups(m, [&](const Group &G) -> hipError_t {
        switch (G.N) { CASES_1(rhs_n, m, G, s) }
        return hipErrorInvalidValue;
    });
}

hipError_t launch_ic(const DeviceMesh &m, int kind, int n_pulses, const double *pulses, double Lx, double Ly,
                     hipStream_t s) {
    return for_groups(m, [&](const Group &G) -> hipError_t {
        switch (G.N) { CASES_1(ic_n, m, G, kind, n_pulses, pulses, Lx, Ly, s) }
        return hipErrorInvalidValue;
    });
}

hipError_t launch_estimate(const DeviceMesh &m, double tol_min, double tol_max, double *out, hipStream_t s) {
    return for_groups(m, [&](const Group &G) -> hipError_t {
        switch (G.N) { CASES_1(estimate_n, m, G, tol_min, tol_max, out, s) }
        return hipErrorInvalidValue;
    });
}

hipError_t launch_traces_c32(const DeviceMesh &m, hipStream_t s) {
    return for_groups(m, [&](const Group &G) -> hipError_t {
        switch (G.N) { CASES_1(traces_c32_n, m, G, s) }
        return hipErrorInvalidValue;
    });
}


template <int N>
static int c32_run_n() { return rk_run<N>(LineShape<N>::EPB); }

static int c32_run(int N) {
    switch (N) { CASES_1(c32_run_n) }
    return 0;
}

// q and qh are in reference node order; gl32 in the FP32 stage's tile order (tiles of the
// shape's EPB elements). Run per group (the order depends on N).
hipError_t launch_to_c32(DeviceMesh &m, hipStream_t s) {
    return for_groups(m, [&](const Group &G) -> hipError_t {
        const int64_t n = G.K * 3 * (int64_t)(G.N + 1) * (G.N + 1);
        hipLaunchKernelGGL(to_c32_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, m.q + G.q_off,
                           m.qh + G.q_off, m.gl32 + G.g_off, n, G.N + 1, stage_max_epb(G.N), c32_run(G.N));
        return hipGetLastError();
    });
}

hipError_t launch_from_c32(DeviceMesh &m, hipStream_t s) {
    return for_groups(m, [&](const Group &G) -> hipError_t {
        const int64_t n = G.K * 3 * (int64_t)(G.N + 1) * (G.N + 1);
        hipLaunchKernelGGL(from_c32_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, m.qh + G.q_off,
                           m.gl32 + G.g_off, m.q + G.q_off, n, G.N + 1, stage_max_epb(G.N), c32_run(G.N));
        return hipGetLastError();
    });
}

// One partial minimum per workgroup of every group (at most 1024 in total), then one final pass.
hipError_t launch_delta_t(const DeviceMesh &m, double cfl, double *dt_dev, hipStream_t s) {
    int used = 0;
    for (const Group &G : m.groups) {
        const int blocks = (int)std::max<int64_t>(1, std::min<int64_t>((G.K + 255) / 256,
                                                                      1024 / (int64_t)m.groups.size()));
        if (used + blocks > m.scratch_len) return hipErrorInvalidValue;
        hipLaunchKernelGGL(dt_partial_kernel, dim3(blocks), dim3(256), 0, s, m.verts + G.e_begin * 8, G.K, G.N, cfl,
                           m.wave_speed, m.scratch + used);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        used += blocks;
    }
    hipLaunchKernelGGL(dt_final_kernel, dim3(1), dim3(256), 0, s, m.scratch, used, dt_dev);
    return hipGetLastError();
}

hipError_t launch_clock_set(DeviceMesh &m, double t, hipStream_t s) {
    if (!m.has_inflow) return hipSuccess;  // nothing reads the stage time
    hipLaunchKernelGGL(clock_set_kernel, dim3(1), dim3(64), 0, s, m.clock + m.cur, t);
    return hipGetLastError();
}

}  // namespace ndg
