// gfx950 device kernels for the MG-CFD hot path.
//
// Data layout in HBM (set up by runtime.hip):
//   dats         the reference's own AoS layout x[i * dim + v] (double or
//                int), in the runtime's internal element order; one gathered
//                node is one ~40-byte record, i.e. one or two cache lines
//   edge map     int2 per edge (internal ids)
//   weights      packed double4 {w0, w1, w2, |w|} per edge or per
//                incidence, rebuilt whenever the weight dat changes (|w| is
//                the reference's ewt, flux.h:48-50)
//   inverse map  CSR per target node: the incidences that INC into it, in
//                the reference's element order (OP2 sequential order)
//
// Kernels marked "exact" disable FMA contraction and keep the reference's
// operation order and true divisions, so they are bitwise equal to the
// sequential CPU evaluation.  "fast" kernels use one reciprocal of the
// density, refined hardware reciprocal and square-root estimates, and FMA
// contraction.
#pragma once

#include <hip/hip_runtime.h>
#include <cfloat>
#include <cmath>
#include <cstdint>
#include <type_traits>

namespace mgcfd {

constexpr double kGamma = 1.4;
constexpr int kBlock = 256;
constexpr int kWave = 64;
constexpr int kPart = 256;       // nodes per flux workgroup (one mesh part)

struct Consts {
    double sc;          // smoothing_coefficient
    double ffv[5];      // ff_variable
    double ffmx[3], ffmy[3], ffmz[3], ffde[3];
};

// Flux-tensor and thermodynamic state of one node (inlined_funcs.h:70-129).
struct Th {
    double rho, mx, my, mz, E;
    double ux, uy, uz;
    double speed, c, p;
    double fxx, fxy, fxz, fyy, fyz, fzz;   // momentum flux (symmetric)
    double fdx, fdy, fdz;                  // energy flux
};

// Flux tensor from velocity, momentum and pressure (inlined_funcs.h:70-96).
__device__ __forceinline__ void flux_tensor_exact(Th& t)
{
#pragma clang fp contract(off)
    t.fxx = t.ux * t.mx + t.p;
    t.fxy = t.ux * t.my;
    t.fxz = t.ux * t.mz;
    t.fyy = t.uy * t.my + t.p;
    t.fyz = t.uy * t.mz;
    t.fzz = t.uz * t.mz + t.p;
    const double de_p = t.E + t.p;
    t.fdx = t.ux * de_p;
    t.fdy = t.uy * de_p;
    t.fdz = t.uz * de_p;
}

// The fast form writes its multiply-adds out and contracts nothing else, so
// that every instantiation of a kernel rounds alike: the gather's shapes
// follow a level's number of blocks, and a mesh's result must not depend on
// the meshes it shares a level with.
__device__ __forceinline__ void flux_tensor_fast(Th& t)
{
#pragma clang fp contract(off)
    t.fxx = fma(t.ux, t.mx, t.p);
    t.fxy = t.ux * t.my;
    t.fxz = t.ux * t.mz;
    t.fyy = fma(t.uy, t.my, t.p);
    t.fyz = t.uy * t.mz;
    t.fzz = fma(t.uz, t.mz, t.p);
    const double de_p = t.E + t.p;
    t.fdx = t.ux * de_p;
    t.fdy = t.uy * de_p;
    t.fdz = t.uz * de_p;
}

template <bool EXACT>
__device__ __forceinline__ void flux_tensor(Th& t)
{
    if constexpr (EXACT) flux_tensor_exact(t);
    else flux_tensor_fast(t);
}

// Reciprocal and square root of the fast kernels (not the correctly rounded
// library expansions).  FP64: the hardware estimates (v_rcp_f64, v_rsq_f64:
// relative error about 2^-24, measured over 2^20 inputs spanning 2^+-20)
// refined by one Newton-Raphson step each -- 1/x: r += r (1 - x r); sqrt z
// from y = 1/sqrt z: g = z y, g += (z - g g) y / 2 -- which leaves about
// 2^-47 relative (the tests hold the fluxes to 1e-12).  The square root is
// taken of z = x + 2^-1000, which changes no x above 2^-947 and keeps x = 0
// finite (2^-500).  FP32: the hardware instructions (1 ulp).
__device__ __forceinline__ double part_rcp(double x)
{
#pragma clang fp contract(off)
    const double r = __builtin_amdgcn_rcp(x);
    return fma(r, fma(-x, r, 1.0), r);
}
__device__ __forceinline__ double part_sqrt(double x)
{
#pragma clang fp contract(off)
    const double z = x + 0x1p-1000;
    const double y = __builtin_amdgcn_rsq(z);
    const double g = z * y;
    return fma(fma(-g, g, z), 0.5 * y, g);
}
__device__ __forceinline__ float part_rcp(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ float part_sqrt(float x) { return __builtin_amdgcn_sqrtf(x); }
// sqrt(a b + c), the guard against 0 folded into the sum.
__device__ __forceinline__ double part_sqrt(double a, double b, double c)
{
#pragma clang fp contract(off)
    const double z = fma(a, b, c + 0x1p-1000);
    const double y = __builtin_amdgcn_rsq(z);
    const double g = z * y;
    return fma(fma(-g, g, z), 0.5 * y, g);
}

// Reference order: u = m / rho, |u|^2, p, c = sqrt(gamma p / rho).
__device__ __forceinline__ void thermo_exact(const double* U, Th& t)
{
#pragma clang fp contract(off)
    t.rho = U[0]; t.mx = U[1]; t.my = U[2]; t.mz = U[3]; t.E = U[4];
    t.ux = t.mx / t.rho;
    t.uy = t.my / t.rho;
    t.uz = t.mz / t.rho;
    const double ssq = t.ux * t.ux + t.uy * t.uy + t.uz * t.uz;
    t.speed = sqrt(ssq);
    t.p = (kGamma - 1.0) * (t.E - 0.5 * t.rho * ssq);
    t.c = sqrt(kGamma * t.p / t.rho);
    flux_tensor_exact(t);
}

// Pressure of a node from its velocity.
__device__ __forceinline__ double pressure_exact(const Th& t)
{
#pragma clang fp contract(off)
    const double ssq = t.ux * t.ux + t.uy * t.uy + t.uz * t.uz;
    return (kGamma - 1.0) * (t.E - 0.5 * t.rho * ssq);
}
__device__ __forceinline__ double pressure_fast(const Th& t)
{
#pragma clang fp contract(off)
    const double ssq = fma(t.uz, t.uz, fma(t.uy, t.uy, t.ux * t.ux));
    return (kGamma - 1.0) * fma(-0.5 * t.rho, ssq, t.E);
}

__device__ __forceinline__ void thermo_fast(const double* U, Th& t)
{
#pragma clang fp contract(off)
    t.rho = U[0]; t.mx = U[1]; t.my = U[2]; t.mz = U[3]; t.E = U[4];
    const double inv = part_rcp(t.rho);
    t.ux = t.mx * inv;
    t.uy = t.my * inv;
    t.uz = t.mz * inv;
    t.speed = part_sqrt(fma(t.uz, t.uz, fma(t.uy, t.uy, t.ux * t.ux)));
    t.p = pressure_fast(t);
    t.c = part_sqrt(kGamma * t.p * inv);
    flux_tensor_fast(t);
}

template <bool EXACT>
__device__ __forceinline__ void thermo(const double* U, Th& t)
{
    if constexpr (EXACT) thermo_exact(U, t);
    else thermo_fast(U, t);
}

__device__ __forceinline__ void load5(const double* __restrict__ x, int i, double U[5])
{
    const double* p = x + (size_t)i * 5;
#pragma unroll
    for (int v = 0; v < 5; v++) U[v] = p[v];
}

__device__ __forceinline__ void store5(double* __restrict__ x, int i, const double U[5])
{
    double* p = x + (size_t)i * 5;
#pragma unroll
    for (int v = 0; v < 5; v++) p[v] = U[v];
}

// Increment that edge (own, oth) adds to node 'own' (flux.h:139-207).  The
// reference computes factor_a and factor_b with the same operand order taken
// from the endpoint's own side; with fx = -0.5 w (or +0.5 w on the b side,
// whose terms the reference subtracts) one formula serves both roles exactly.
__device__ __forceinline__ void edge_increment_exact(const Th& o, const Th& t, double ewt, double sc,
                                                     double fx, double fy, double fz, double inc[5])
{
#pragma clang fp contract(off)
    const double factor = -ewt * sc * 0.5 * (o.speed + t.speed + o.c + t.c);
    inc[0] = factor * (o.rho - t.rho) + fx * (o.mx + t.mx) + fy * (o.my + t.my) + fz * (o.mz + t.mz);
    inc[4] = factor * (o.E - t.E) + fx * (o.fdx + t.fdx) + fy * (o.fdy + t.fdy) + fz * (o.fdz + t.fdz);
    inc[1] = factor * (o.mx - t.mx) + fx * (o.fxx + t.fxx) + fy * (o.fxy + t.fxy) + fz * (o.fxz + t.fxz);
    inc[2] = factor * (o.my - t.my) + fx * (o.fxy + t.fxy) + fy * (o.fyy + t.fyy) + fz * (o.fyz + t.fyz);
    inc[3] = factor * (o.mz - t.mz) + fx * (o.fxz + t.fxz) + fy * (o.fyz + t.fyz) + fz * (o.fzz + t.fzz);
}

// factor d + fx sx + fy sy + fz sz.
__device__ __forceinline__ double fast_term(double factor, double d, double fx, double sx, double fy, double sy,
                                            double fz, double sz)
{
#pragma clang fp contract(off)
    return fma(fz, sz, fma(fy, sy, fma(fx, sx, factor * d)));
}

// The other end's products are added to the own node's tensors as they are
// formed (formed apart, the 300K-node cycle takes 387 us, so 382).
__device__ __forceinline__ void edge_increment_fast(const Th& o, const Th& t, double ewt, double sc,
                                                    double fx, double fy, double fz, double inc[5])
{
#pragma clang fp contract(off)
    const double factor = -ewt * sc * 0.5 * (o.speed + t.speed + o.c + t.c);
    const double de = t.E + t.p;
    const double sxx = o.fxx + fma(t.ux, t.mx, t.p), sxy = fma(t.ux, t.my, o.fxy), sxz = fma(t.ux, t.mz, o.fxz);
    const double syy = o.fyy + fma(t.uy, t.my, t.p), syz = fma(t.uy, t.mz, o.fyz);
    const double szz = o.fzz + fma(t.uz, t.mz, t.p);
    const double sdx = fma(t.ux, de, o.fdx), sdy = fma(t.uy, de, o.fdy), sdz = fma(t.uz, de, o.fdz);
    inc[0] = fast_term(factor, o.rho - t.rho, fx, o.mx + t.mx, fy, o.my + t.my, fz, o.mz + t.mz);
    inc[4] = fast_term(factor, o.E - t.E, fx, sdx, fy, sdy, fz, sdz);
    inc[1] = fast_term(factor, o.mx - t.mx, fx, sxx, fy, sxy, fz, sxz);
    inc[2] = fast_term(factor, o.my - t.my, fx, sxy, fy, syy, fz, syz);
    inc[3] = fast_term(factor, o.mz - t.mz, fx, sxz, fy, syz, fz, szz);
}

template <bool EXACT>
__device__ __forceinline__ void edge_increment(const Th& o, const Th& t, double ewt, double sc, double fx,
                                               double fy, double fz, double inc[5])
{
    if constexpr (EXACT) edge_increment_exact(o, t, ewt, sc, fx, fy, fz, inc);
    else edge_increment_fast(o, t, ewt, sc, fx, fy, fz, inc);
}

__device__ __forceinline__ double add_exact(double a, double b)
{
#pragma clang fp contract(off)
    return a + b;
}

// Workgroup index remapped so that each of the 8 XCDs (which receive
// workgroups round-robin) walks one contiguous slice of the iteration space
// and keeps its neighbours in its own L2.
__device__ __forceinline__ int xcd_block()
{
    const int nb = gridDim.x, b = blockIdx.x;
    const int per = nb / 8, rem = nb % 8;
    const int x = b % 8, k = b / 8;
    // XCD x's slice starts at x * per + min(x, rem) (the first rem slices
    // hold one more); no branch, so the kernel's first loads issue together
    return x * per + min(x, rem) + k;
}

__device__ __forceinline__ bool halted(const int* status) { return status && *status != 0; }

// base[i], or 0 when base is null, read by one load with no branch around it
// (a null base reads a zero word).  Kernels that test their context's status
// late (before their first global write, not at entry) read it this way with
// their first loads, so its round trip overlaps theirs instead of preceding
// them.
__device__ int kZeroWord = 0;     // never written
__device__ __forceinline__ int word_or_zero(const int* base, int i) { return *(base ? base + i : &kZeroWord); }
__device__ __forceinline__ int status_of(const int* status) { return word_or_zero(status, 0); }

// ------------------------------------------------------------------------
// Edge flux, blocked gather (default).  A workgroup owns the nodes
// [n0, n0 + cnt) of one compact mesh part; inside a part the nodes are ordered
// by decreasing degree.
//  1. Stage: the owned nodes' states arrive as one run of 5 * cnt doubles
//     (consecutive lanes, consecutive doubles), the halo (neighbours owned by
//     other parts) node by node, up to NH per thread.  Each staged node's
//     velocity, speed and speed of sound are formed once and kept with its
//     conserved variables as kGRec doubles in LDS.  The pressure is formed
//     again per incidence: 9 operations, against 8 bytes of every record,
//     which at 80 bytes keep three workgroups of a 300K-node level on a CU.
//  2. Walk: thread t adds, in the reference's edge order, the increment of
//     each of its node's edges, reading the other endpoint from LDS.  The
//     k-th incidences of all threads of a block are stored contiguously
//     (jagged-diagonal order: j0 + jpref[k] + t), so the per-incidence
//     loads {LDS slot | b-role << 31} and the weight components w0 | w1 | w2
//     (SoA) are coalesced.  They are double-buffered in registers: chunks
//     of CH incidences, the first in flight with the staging loads, chunk
//     c+1 loading while chunk c is evaluated.  |w| is recomputed with the
//     reference's expression (flux.h:48-50).
// Every node sums its edges in OP2's sequential order; with EXACT (no FMA
// contraction, true divisions) the result is bitwise the reference's.
// Deterministic, no atomics, one launch.  Bound by the incidences' bytes on
// large levels (28 per incidence, two incidences per edge) and by each
// thread's serial walk on small ones.  930K-edge flux 35.0 us with 96-byte
// records and at most 256 halo nodes per block, 27.5 us now; cycle of a
// 300K-node solve 837 -> 572 us, 1M nodes 2259 -> 1341 us.
// ------------------------------------------------------------------------
constexpr int kGRec = 10;        // doubles per record {rho, mx, my, mz, E, ux, uy, uz, |u|, c}

struct BlkInfo {
    int n0, cnt;    // owned nodes [n0, n0 + cnt)
    int h0, nh;     // halo ids halo[h0 .. h0 + nh)
    int j0, p0;     // first jagged entry; start of the diagonal offsets in jpref
    int g0, pad;    // first partial sum of the block's nodes (one per 64)
};

// The derived half of a record from its conserved variables r[0..4].
template <bool EXACT>
__device__ __forceinline__ void derive_record(double* r)
{
    double U[5];
#pragma unroll
    for (int v = 0; v < 5; v++) U[v] = r[v];
    Th th;
    thermo<EXACT>(U, th);
    r[5] = th.ux; r[6] = th.uy; r[7] = th.uz; r[8] = th.speed; r[9] = th.c;
}

template <bool EXACT>
__device__ __forceinline__ void load_record(const double* rec, Th& t)
{
    const double2* r = reinterpret_cast<const double2*>(rec);
    const double2 a = r[0], b = r[1], c = r[2], d = r[3], e = r[4];
    t.rho = a.x; t.mx = a.y; t.my = b.x; t.mz = b.y; t.E = c.x;
    t.ux = c.y; t.uy = d.x; t.uz = d.y; t.speed = e.x; t.c = e.y;
    t.p = EXACT ? pressure_exact(t) : pressure_fast(t);
    flux_tensor<EXACT>(t);
}

// CH incidences of one thread: {slot | role} codes and weight components.
template <int CH>
struct IncChunk {
    unsigned r[CH];
    double x0[CH], x1[CH], x2[CH];
};

// LPN lanes share a node: lane l takes its incidences l, l + LPN, ...; q0
// counts a lane's own.
template <int CH, int LPN>
__device__ __forceinline__ void load_chunk(IncChunk<CH>& c, int q0, int l, int deg, int jb,
                                           const int* __restrict__ jp, const unsigned* __restrict__ jslot,
                                           const double* __restrict__ jw, int nent)
{
#pragma unroll
    for (int i = 0; i < CH; i++) {
        const int q = (q0 + i) * LPN + l;
        c.r[i] = 0;
        c.x0[i] = c.x1[i] = c.x2[i] = 0.0;
        if (q < deg) {
            const int at = jb + jp[q];
            c.r[i] = jslot[at];
            c.x0[i] = jw[at];
            c.x1[i] = jw[nent + at];
            c.x2[i] = jw[2 * nent + at];
        }
    }
}

// x of lane K of this lane's group of LPN lanes (LPN 2 or 4).
template <int LPN, int K>
__device__ __forceinline__ double group_lane(double x)
{
    constexpr int ctrl = LPN == 4 ? K * 0x55 : K ? 0xf5 : 0xa0;      // quad_perm
    const int lo = __double2loint(x), hi = __double2hiint(x);
    return __hiloint2double(__builtin_amdgcn_update_dpp(hi, hi, ctrl, 0xf, 0xf, true),
                            __builtin_amdgcn_update_dpp(lo, lo, ctrl, 0xf, 0xf, true));
}

template <bool EXACT, int LPN, int K = 0>
__device__ __forceinline__ void add_group(const double d[5], double acc[5])
{
    if constexpr (K < LPN) {
#pragma unroll
        for (int v = 0; v < 5; v++) acc[v] = add_exact(acc[v], group_lane<LPN, K>(d[v]));
        add_group<EXACT, LPN, K + 1>(d, acc);
    }
}

template <bool EXACT>
__device__ __forceinline__ void incidence(unsigned r, double x0, double x1, double x2, const double* sm, const Th& o,
                                          double sc, double d[5])
{
    Th th;
    load_record<EXACT>(sm + (int)(r & 0x7fffffffu) * kGRec, th);
    double ewt;
    {
#pragma clang fp contract(off)
        ewt = sqrt(x0 * x0 + x1 * x1 + x2 * x2);
    }
    double fx = -0.5 * x0, fy = -0.5 * x1, fz = -0.5 * x2;
    if (r & 0x80000000u) { fx = -fx; fy = -fy; fz = -fz; }   // node is endpoint b
    edge_increment<EXACT>(o, th, ewt, sc, fx, fy, fz, d);
}

// The increments of a chunk added in incidence order.  With several lanes per
// node each lane evaluates its own, and all of them add the group's in lane
// order (-0.0 where a lane has none, which leaves every sum as it is), so
// every lane holds the node's sum.  The lanes of a group agree on the loop
// bounds, so the exchange reads active lanes only.
template <bool EXACT, int CH, int LPN>
__device__ __forceinline__ void walk_chunk(const IncChunk<CH>& c, int q0, int l, int deg, const double* sm,
                                           const Th& o, double sc, double acc[5])
{
#pragma unroll
    for (int i = 0; i < CH; i++) {
        if ((q0 + i) * LPN < deg) {
            double d[5] = {-0.0, -0.0, -0.0, -0.0, -0.0};
            if (LPN == 1 || (q0 + i) * LPN + l < deg)
                incidence<EXACT>(c.r[i], c.x0[i], c.x1[i], c.x2[i], sm, o, sc, d);
            if constexpr (LPN > 1) {
                add_group<EXACT, LPN>(d, acc);
            } else {
#pragma unroll
                for (int v = 0; v < 5; v++) acc[v] = add_exact(acc[v], d[v]);
            }
        }
    }
}

// The jagged plan of one map, as the gather kernels take it.
struct GatherPlan {
    const BlkInfo* blk;
    const int* halo;
    const int* jpref;
    const int* nptr;            // CSR over every node: its degree
    const unsigned* jslot;
    const double* jw;           // w0 | w1 | w2, nent entries each
    int nent;
};

// Steps 1 and 2 for one block of at most PN nodes, LPN lanes to a node (PN *
// LPN threads): acc holds the start value of the thread's node (t / LPN) and
// receives its edge flux, in each of its lanes; o: the node's own state.
// LDS: one record per staged node.  Ends without a barrier.
template <bool EXACT, int CH, int NH, int PN, int LPN>
__device__ __forceinline__ void gather_block(const GatherPlan& G, const BlkInfo& B, const double* __restrict__ vin,
                                             double sc, double* sm, double acc[5], Th& o)
{
    constexpr int T = PN * LPN, FL = (5 * PN + T - 1) / T;
    const int t = threadIdx.x, n = t / LPN, l = t % LPN;
    const bool own = n < B.cnt;
    const int last = 5 * B.cnt - 1, hmax = max(B.nh - 1, 0);
    const size_t base = (size_t)B.n0 * 5;
    int hn[NH];
    double x[FL], U[NH][5];
#pragma unroll
    for (int k = 0; k < NH; k++) hn[k] = (G.halo + B.h0)[min((unsigned)t + k * T, (unsigned)hmax)];
    // uniform bases and small per-lane indexes: no 64-bit address arithmetic per
    // lane (cycle of a 300K-node solve 450 -> 424 us)
    const double* xin = vin + base;
#pragma unroll
    for (int i = 0; i < FL; i++) x[i] = xin[min((unsigned)t + i * T, (unsigned)last)];
    const int* np = G.nptr + B.n0;
    const unsigned nd = min((unsigned)n, (unsigned)B.cnt - 1u);
    const int deg = own ? np[nd + 1] - np[nd] : 0;
    const int jb = B.j0 + n;
    const int* jp = G.jpref + B.p0;
    IncChunk<CH> A, C;
    load_chunk<CH, LPN>(A, 0, l, deg, jb, jp, G.jslot, G.jw, G.nent);
#pragma unroll
    for (int k = 0; k < NH; k++)
#pragma unroll
        for (int v = 0; v < 5; v++) U[k][v] = vin[(size_t)hn[k] * 5 + v];
#pragma unroll
    for (int i = 0; i < FL; i++) {
        const int j = t + i * T;
        if (j <= last) sm[j + (j / 5) * (kGRec - 5)] = x[i];
    }
#pragma unroll
    for (int k = 0; k < NH; k++)
        if (t + k * T < B.nh) {
            double* r = sm + (B.cnt + t + k * T) * kGRec;
#pragma unroll
            for (int v = 0; v < 5; v++) r[v] = U[k][v];
            derive_record<EXACT>(r);
        }
    __syncthreads();
    if (t < B.cnt) derive_record<EXACT>(sm + t * kGRec);
    __syncthreads();
    if (!own) return;
    load_record<EXACT>(sm + n * kGRec, o);
    for (int q0 = 0; q0 * LPN < deg; q0 += 2 * CH) {
        load_chunk<CH, LPN>(C, q0 + CH, l, deg, jb, jp, G.jslot, G.jw, G.nent);
        walk_chunk<EXACT, CH, LPN>(A, q0, l, deg, sm, o, sc, acc);
        if ((q0 + CH) * LPN >= deg) break;
        load_chunk<CH, LPN>(A, q0 + 2 * CH, l, deg, jb, jp, G.jslot, G.jw, G.nent);
        walk_chunk<EXACT, CH, LPN>(C, q0 + CH, l, deg, sm, o, sc, acc);
    }
}

template <bool EXACT, int CH, int NH, int PN, int LPN>
__global__ __launch_bounds__(PN * LPN) void k_flux_blocked_pf(GatherPlan G, const double* __restrict__ var,
                                                              double* __restrict__ flux, Consts k,
                                                              const int* __restrict__ status, int fresh)
{
    extern __shared__ double sm[];
    if (halted(status)) return;
    const BlkInfo B = G.blk[xcd_block()];
    const int n = threadIdx.x / LPN;
    double acc[5];
    if (fresh) {
#pragma unroll
        for (int v = 0; v < 5; v++) acc[v] = 0.0;
    } else {
        load5(flux, B.n0 + min(n, B.cnt - 1), acc);
    }
    Th o;
    gather_block<EXACT, CH, NH, PN, LPN>(G, B, var, k.sc, sm, acc, o);
    if (n < B.cnt && threadIdx.x % LPN == 0) store5(flux, B.n0 + n, acc);
}

// Per-incidence weight components (SoA) of k_flux_blocked_pf.
__global__ void k_pack_incidence_weights3(int n, const int* __restrict__ eid, const double* __restrict__ w,
                                          double* __restrict__ out)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const int e = eid[k];
    double a = 0.0, b = 0.0, c = 0.0;
    if (e >= 0) { a = w[3 * (size_t)e]; b = w[3 * (size_t)e + 1]; c = w[3 * (size_t)e + 2]; }
    out[k] = a;
    out[n + k] = b;
    out[2 * (size_t)n + k] = c;
}

// ------------------------------------------------------------------------
// Edge flux, edge-parallel over mesh parts with node state and increments
// in LDS.  Workgroup b owns the nodes [n0, n0 + cnt) of one compact part and
// every edge with at least one endpoint among them ("local edges": interior
// edges once, cut edges once on each side).
//  1. Load (all loads issued before the barrier, flat and coalesced): owned
//     variables and halo variables as raw {rho, m, E} records in LDS, the
//     old flux of owned nodes into the LDS accumulators, and this thread's
//     local edges {slot a, slot b, owner flags, colour} with their weights.
//  2. Each thread evaluates its edges once: both endpoint states from their
//     LDS records (one density reciprocal each, fast form), then inc =
//     factor (U_a - U_b) + sum_k f_k (F_a + F_b)_k with f = -w/2; node a
//     gains +inc and node b gains -inc (flux.h:139-207 with factor_b ==
//     factor_a up to rounding).  Raw records keep the LDS footprint at
//     48 B per staged node, so more workgroups share a CU.
//  3. Accumulation into the LDS accumulators: COLOURED walks the edge
//     colours of the part (no two edges of one colour share an owned node),
//     one barrier per colour, so the summation order is fixed by the plan and
//     results are deterministic; otherwise LDS FP64 atomics (ds_add_f64) in
//     arrival order.
//  4. The accumulators are stored as one coalesced block.
// Not bitwise the sequential order (ulp-level drift, as the fast gather).
// ------------------------------------------------------------------------
constexpr int kPRec = 6;    // doubles per LDS node record of k_flux_part {rho, mx, my, mz, E, -}

struct PartInfo {
    int n0, cnt;    // owned nodes [n0, n0 + cnt)
    int h0, nh;     // halo ids halo[h0 .. h0 + nh)
    int e0, ne;     // local edges [e0, e0 + ne)
    int ncol, g0;   // edge colours (COLOURED); first partial sum of the part's nodes (one per 64)
};

// One endpoint of an edge as the increment needs it.
template <typename R>
struct PState;
template <>
struct PState<double> {
    double rho, mx, my, mz, E, inv, p, s;   // inv = 1 / rho, s = |u| + c
};
template <>
struct PState<float> {
    float rho, mx, my, mz, E, ux, uy, uz, e, p, s;   // e: internal energy (p = 0.4 e)
};

// The multiply-adds of the part kernels' arithmetic are written out, and
// nothing else is contracted, so that every instantiation of a kernel (threads
// per part, edges per thread) rounds alike: a deterministic variant's result
// is the same bit for bit whichever one a level's size selects.
__device__ __forceinline__ double part_fma(double a, double b, double c) { return fma(a, b, c); }
__device__ __forceinline__ double part_dot(double a0, double a1, double a2, double b0, double b1, double b2)
{
#pragma clang fp contract(off)
    return part_fma(a2, b2, part_fma(a1, b1, a0 * b0));
}

// The derived part of an FP64 endpoint from its conserved variables: 1 / rho,
// the pressure and (SPEED) the wave speed |u| + c.  The kinetic energy is u . m,
// which is as large as the state itself: |m|^2 / rho would take two operations
// less per endpoint (0.2-0.5% of a cycle) and overflow or vanish for states
// beyond about 1e+-154.
template <bool SPEED>
__device__ __forceinline__ void part_derive(PState<double>& t)
{
#pragma clang fp contract(off)
    t.inv = part_rcp(t.rho);
    const double k = part_dot(t.mx * t.inv, t.my * t.inv, t.mz * t.inv, t.mx, t.my, t.mz);     // rho |u|^2
    t.p = (kGamma - 1.0) * part_fma(-0.5, k, t.E);
    if constexpr (SPEED) t.s = part_sqrt(k, t.inv, 0.0) + part_sqrt(kGamma * t.p, t.inv, 0.0);
}

// The same of an FP32 endpoint, with its velocity (the FP32 increment goes
// through both flux tensors).
template <bool SPEED>
__device__ __forceinline__ void part_derive(PState<float>& t)
{
#pragma clang fp contract(off)
    const float inv = part_rcp(t.rho);
    t.ux = t.mx * inv; t.uy = t.my * inv; t.uz = t.mz * inv;
    const float ssq = fmaf(t.uz, t.uz, fmaf(t.ux, t.ux, t.uy * t.uy));
    t.e = fmaf(-(0.5f * t.rho), ssq, t.E);
    t.p = (float)(kGamma - 1.0) * t.e;
    if constexpr (SPEED) t.s = part_sqrt(ssq) + part_sqrt((float)kGamma * t.p * inv);
}

// Wave speed |u| + c of a node state, computed once per staged node and kept
// in its record (R arithmetic: FP64, or FP32 for mixed precision).
template <typename R>
__device__ __forceinline__ R part_speed(R rho, R mx, R my, R mz, R E)
{
    PState<R> t;
    t.rho = rho; t.mx = mx; t.my = my; t.mz = mz; t.E = E;
    part_derive<true>(t);
    return t.s;
}

// Increment of node a for edge (a, b); node b gains -inc.  (f0, f1, f2) =
// -w / 2, the packed weights, so |w| / 2 is |f| and the dissipation factor
// -|w| sc (s_a + s_b) / 2 is -|f| sc (s_a + s_b).  FP64: the convective part is
// taken along the face: with v = (m . f) / rho of each endpoint, F f =
// {m . f, m v + p f, (E + p) v}, which needs no flux tensor.  The edge phase is
// bound by FP64 issue once a part's data is staged: 98 FP64 instructions per
// edge with the wave speeds formed here (40-byte records), against 136 with
// the tensors of both endpoints.  Tensors -> along the face, three alternating
// runs: 930K-edge flux over five rotating meshes 18.8 -> 18.3 us, cycle of a
// 300K-node solve 345 -> 341 us, of a 1M-node solve 768 -> 746 us.
__device__ __forceinline__ void part_increment(const PState<double>& a, const PState<double>& b, double f0, double f1,
                                               double f2, double sc, double inc[5])
{
#pragma clang fp contract(off)
    const double factor = -sc * part_sqrt(f2, f2, part_fma(f1, f1, f0 * f0)) * (a.s + b.s);
    const double fa = part_dot(f0, f1, f2, a.mx, a.my, a.mz), fb = part_dot(f0, f1, f2, b.mx, b.my, b.mz);
    const double va = fa * a.inv, vb = fb * b.inv, ps = a.p + b.p;
    inc[0] = part_fma(factor, a.rho - b.rho, fa + fb);
    inc[1] = part_fma(factor, a.mx - b.mx, part_fma(va, a.mx, part_fma(vb, b.mx, f0 * ps)));
    inc[2] = part_fma(factor, a.my - b.my, part_fma(va, a.my, part_fma(vb, b.my, f1 * ps)));
    inc[3] = part_fma(factor, a.mz - b.mz, part_fma(va, a.mz, part_fma(vb, b.mz, f2 * ps)));
    inc[4] = part_fma(factor, a.E - b.E, part_fma(va, a.E + a.p, vb * (b.E + b.p)));
}

// FP32: through the flux tensors F_a + F_b (symmetric) and the energy flux.
// FP32 issue does not bound the mixed-precision kernels (the form above gains
// them 1%), and the tensors' rounding errors are the smaller for a uniform
// state (8.8e-8 of the flux against 1.0e-7).
__device__ __forceinline__ void part_increment(const PState<float>& a, const PState<float>& b, float f0, float f1,
                                               float f2, float sc, float inc[5])
{
#pragma clang fp contract(off)
    constexpr float g = (float)(kGamma - 1.0);
    const float factor = -part_sqrt(fmaf(f2, f2, fmaf(f0, f0, f1 * f1))) * sc * (a.s + b.s);
    const float dea = fmaf(g, a.e, a.E), deb = fmaf(g, b.e, b.E);       // E + p
    const float sxx = fmaf(g, b.e, fmaf(b.ux, b.mx, fmaf(a.ux, a.mx, a.p)));
    const float syy = fmaf(g, b.e, fmaf(b.uy, b.my, fmaf(a.uy, a.my, a.p)));
    const float szz = fmaf(g, b.e, fmaf(b.uz, b.mz, fmaf(a.uz, a.mz, a.p)));
    const float sxy = fmaf(a.ux, a.my, b.ux * b.my), sxz = fmaf(a.ux, a.mz, b.ux * b.mz);
    const float syz = fmaf(a.uy, a.mz, b.uy * b.mz);
    const float sdx = fmaf(a.ux, dea, b.ux * deb), sdy = fmaf(a.uy, dea, b.uy * deb);
    const float sdz = fmaf(a.uz, dea, b.uz * deb);
    inc[0] = fmaf(f2, a.mz + b.mz, fmaf(f1, a.my + b.my, fmaf(f0, a.mx + b.mx, factor * (a.rho - b.rho))));
    inc[1] = fmaf(f2, sxz, fmaf(f1, sxy, fmaf(factor, a.mx - b.mx, f0 * sxx)));
    inc[2] = fmaf(f2, syz, fmaf(f1, syy, fmaf(f0, sxy, factor * (a.my - b.my))));
    inc[3] = fmaf(f2, szz, fmaf(f1, syz, fmaf(f0, sxz, factor * (a.mz - b.mz))));
    inc[4] = fmaf(f2, sdz, fmaf(f1, sdy, fmaf(factor, a.E - b.E, f0 * sdx)));
}

// Adds inc to owned endpoint a and -inc to owned endpoint b (FP64 adds; an
// FP32 increment is converted first).
template <typename O>
__device__ __forceinline__ void part_apply(double* acc, unsigned code, const O inc[5])
{
    const int sa = code & 1023u, sb = (code >> 10) & 1023u;
    if (code & (1u << 20)) {
#pragma unroll
        for (int v = 0; v < 5; v++) atomicAdd(acc + sa * 5 + v, (double)inc[v]);
    }
    if (code & (1u << 21)) {
#pragma unroll
        for (int v = 0; v < 5; v++) atomicAdd(acc + sb * 5 + v, -(double)inc[v]);
    }
}

// LDS node records of the part kernels: the raw state {rho, m, E} and, with
// six values, the wave speed |u| + c, which staging forms once per node; the
// rest of each endpoint is derived per edge -- the small record lets more
// workgroups share a CU, which pays more than deriving each state once.
// FP32 records have six values; FP64 ones six, or five (40 bytes) when
// 48-byte records would leave fewer than four workgroups per CU and in the
// kernel with the fused stage.
constexpr int kPRec32 = 6;     // values an FP32 record takes up (24 bytes: 8-byte aligned), with or without speed

template <typename R, int RS>
__host__ __device__ constexpr int part_stride()
{
    static_assert(RS == 5 || RS == 6, "record size");
    return sizeof(R) == sizeof(double) ? RS : kPRec32;
}

// Doubles that 'n' records take up.
template <typename R, int RS>
__host__ __device__ constexpr size_t part_rec_doubles(int n)
{
    return ((size_t)n * part_stride<R, RS>() * sizeof(R) + sizeof(double) - 1) / sizeof(double);
}

template <typename R, int RS>
__device__ __forceinline__ PState<R> part_rec_state(const R* r)
{
    PState<R> t;
    if constexpr (part_stride<R, RS>() == 6) {
        using R2 = typename std::conditional<sizeof(R) == 8, double2, float2>::type;
        const R2* q = reinterpret_cast<const R2*>(r);
        const R2 a = q[0], b = q[1], c = q[2];
        t.rho = a.x; t.mx = a.y; t.my = b.x; t.mz = b.y; t.E = c.x; t.s = c.y;
    } else {
        t.rho = r[0]; t.mx = r[1]; t.my = r[2]; t.mz = r[3]; t.E = r[4];
    }
    part_derive<RS == 5>(t);
    return t;
}

// Marks a loaded register as needed here: the compiler waits for its load at
// this point and cannot sink the load into a later divergent branch (where it
// would be issued alone under its own wait).
template <typename V>
__device__ __forceinline__ void part_ready(const V& v)
{
    asm volatile("" ::"v"(v));
}

// Local-edge codes and weights of one part, EPT per thread (code 0: none).
template <typename R, int T, int EPT>
__device__ __forceinline__ void part_load_edges(const PartInfo& P, const unsigned* __restrict__ ecode,
                                                const R* __restrict__ ew, long long nloc, int t, unsigned code[EPT],
                                                R w0[EPT], R w1[EPT], R w2[EPT])
{
#pragma unroll
    for (int i = 0; i < EPT; i++) {
        const int j = t + i * T;
        code[i] = 0;
        w0[i] = w1[i] = w2[i] = R(0);
        if (j < P.ne) {
            const long long e = P.e0 + j;
            code[i] = ecode[e];
            w0[i] = ew[e];
            w1[i] = ew[nloc + e];
            w2[i] = ew[2 * nloc + e];
        }
    }
}

// The part's local edges, each increment added to its owned endpoints with
// LDS atomics.
template <typename R, int EPT, int RS>
__device__ __forceinline__ void part_edges_atomic(const R* rec, double* acc, const unsigned code[EPT],
                                                  const R w0[EPT], const R w1[EPT], const R w2[EPT], R sc)
{
#pragma unroll
    for (int i = 0; i < EPT; i++) {
        if (!code[i]) continue;
        const PState<R> a = part_rec_state<R, RS>(rec + (code[i] & 1023u) * part_stride<R, RS>());
        const PState<R> b = part_rec_state<R, RS>(rec + ((code[i] >> 10) & 1023u) * part_stride<R, RS>());
        R inc[5];
        part_increment(a, b, w0[i], w1[i], w2[i], sc, inc);
        part_apply(acc, code[i], inc);
    }
}

// Accumulates the part's local edges (codes and weights in registers) into
// the LDS accumulators; ends with a barrier.  Coloured: all increments are
// formed first, then one short phase per colour adds them, so that the colour
// walk is a chain of LDS additions and not of whole edge increments.  LAZY:
// each increment is formed in its colour's phase, which holds none across the
// phases.  (One stage with fused update, formed in the phases -> up front:
// 30K nodes 10.0 -> 7.8 us, 645 parts 25.9 -> 20.8, 3907 parts 77.5 -> 70.6;
// FP32 with six or more edges per thread, whose workgroups the registers
// limit to fewer per CU, 3907 parts 60.8 -> 64.0: it alone stays LAZY.)
template <typename R, int EPT, bool COLOURED, int RS, bool LAZY>
__device__ __forceinline__ void part_edges(const PartInfo& P, const R* rec, double* acc, const unsigned code[EPT],
                                           const R w0[EPT], const R w1[EPT], const R w2[EPT], R sc)
{
    constexpr int ST = part_stride<R, RS>();
    if constexpr (COLOURED && LAZY) {
        for (int c = 0; c < P.ncol; c++) {
#pragma unroll
            for (int i = 0; i < EPT; i++)
                if (code[i] && (int)(code[i] >> 22) == c) {
                    const PState<R> a = part_rec_state<R, RS>(rec + (code[i] & 1023u) * ST);
                    const PState<R> b = part_rec_state<R, RS>(rec + ((code[i] >> 10) & 1023u) * ST);
                    R inc[5];
                    part_increment(a, b, w0[i], w1[i], w2[i], sc, inc);
                    part_apply(acc, code[i], inc);
                }
            __syncthreads();
        }
    } else if constexpr (COLOURED) {
        R inc[EPT][5];      // held in the arithmetic's precision until the colour walk
#pragma unroll
        for (int i = 0; i < EPT; i++)
            if (code[i]) {
                const PState<R> a = part_rec_state<R, RS>(rec + (code[i] & 1023u) * ST);
                const PState<R> b = part_rec_state<R, RS>(rec + ((code[i] >> 10) & 1023u) * ST);
                part_increment(a, b, w0[i], w1[i], w2[i], sc, inc[i]);
            }
        for (int c = 0; c < P.ncol; c++) {
#pragma unroll
            for (int i = 0; i < EPT; i++)
                if (code[i] && (int)(code[i] >> 22) == c) part_apply(acc, code[i], inc[i]);
            __syncthreads();
        }
    } else {
        part_edges_atomic<R, EPT, RS>(rec, acc, code, w0, w1, w2, sc);
        __syncthreads();
    }
}

// Staging of one part, shared by the part kernels.  The owned nodes' state
// arrives as one run of 5 * cnt doubles (x, FL per thread), the halo node by
// node (NPT per thread); all loads are clamped into the part (the plan pads
// the halo list by one entry), so that they issue without branches and under
// few waits.  part_records writes the records (RS 6: without the owned nodes'
// wave speeds).
template <int T, int NPT>
__device__ __forceinline__ void part_load_halo(const PartInfo& P, const int* __restrict__ halo, int t, int nd[NPT])
{
    const int hmax = max(P.nh - 1, 0);
#pragma unroll
    for (int k = 0; k < NPT; k++) nd[k] = halo[P.h0 + min(t + k * T, hmax)];
}

template <typename R, int T, int NPT, int FL, int RS>
__device__ __forceinline__ void part_records(const PartInfo& P, int t, const double x[FL], const double U[NPT][5],
                                             R* rec)
{
    constexpr int ST = part_stride<R, RS>();
    const int last = 5 * P.cnt - 1;
#pragma unroll
    for (int i = 0; i < FL; i++) {
        const int j = t + i * T;
        if (j <= last) rec[ST == 5 ? j : j + j / 5] = (R)x[i];
    }
#pragma unroll
    for (int k = 0; k < NPT; k++)
        if (t + k * T < P.nh) {
            R* r = rec + (P.cnt + t + k * T) * ST;
#pragma unroll
            for (int v = 0; v < 5; v++) r[v] = (R)U[k][v];
            if constexpr (RS == 6) r[5] = part_speed<R>(r[0], r[1], r[2], r[3], r[4]);
        }
}

// Staging of the edge-flux kernel with six-value records: owned and halo nodes
// alike node by node (slot t + k T, NPT * T >= rec_cap), so that each thread
// forms its nodes' wave speeds from registers and one barrier suffices.  (As
// runs, with the owned wave speeds formed behind a second barrier, mixed
// precision takes 14.8 us on 930K edges against 14.0, FP64 18.4 against 18.0.)
template <int T, int NPT>
__device__ __forceinline__ void part_slot_entries(const PartInfo& P, const int* __restrict__ halo, int t, int nd[NPT])
{
    const int hmax = max(P.nh - 1, 0);
#pragma unroll
    for (int k = 0; k < NPT; k++) nd[k] = halo[P.h0 + min(max(t + k * T - P.cnt, 0), hmax)];
}

template <typename R, int T, int NPT>
__device__ __forceinline__ void part_slot_records(const PartInfo& P, int t, const double U[NPT][5], R* rec)
{
    const int nrec = P.cnt + P.nh;
#pragma unroll
    for (int k = 0; k < NPT; k++)
        if (t + k * T < nrec) {
            R* r = rec + (t + k * T) * part_stride<R, 6>();
            const R x0 = (R)U[k][0], x1 = (R)U[k][1], x2 = (R)U[k][2], x3 = (R)U[k][3], x4 = (R)U[k][4];
            r[0] = x0; r[1] = x1; r[2] = x2; r[3] = x3; r[4] = x4;
            r[5] = part_speed<R>(x0, x1, x2, x3, x4);
        }
}

// LDS: R records [rec_cap * 6] (rounded up to doubles), then FP64
// accumulators [cnt * 5].  R = double: the FP64 kernel; R = float: mixed
// precision (records, weights and increment arithmetic in FP32, each
// increment converted to FP64 and accumulated in FP64 from the FP64 flux).
// One workgroup per part; RS values per record; NPT: halo nodes per thread
// (RS 5) or staged nodes per thread (RS 6).
template <typename R, int T, int EPT, int NPT, bool COLOURED, int RS>
__global__ __launch_bounds__(T) void k_flux_part(
    const PartInfo* __restrict__ parts, const int* __restrict__ halo, const unsigned* __restrict__ ecode,
    const R* __restrict__ ew, long long nloc, int rec_cap, const double* __restrict__ var,
    double* __restrict__ flux, Consts k, const int* __restrict__ status, int fresh)
{
    constexpr int FL = (5 * kPart + T - 1) / T;
    extern __shared__ double sm[];
    const int halt = status_of(status);     // tested before the store
    const PartInfo P = parts[xcd_block()];
    const int t = threadIdx.x;
    R* rec = reinterpret_cast<R*>(sm);
    double* acc = sm + part_rec_doubles<R, RS>(rec_cap);
    const int last = 5 * P.cnt - 1;
    const size_t base = (size_t)P.n0 * 5;
    // 1. loads: halo entries, owned states, edge codes and weights, then halo
    // states and the owned flux; records and accumulators into LDS
    int nd[NPT];
    unsigned code[EPT];
    R w0[EPT], w1[EPT], w2[EPT];
    double x[FL], fl[FL], U[NPT][5];
    if constexpr (RS == 6) {
        part_slot_entries<T, NPT>(P, halo, t, nd);
    } else {
        part_load_halo<T, NPT>(P, halo, t, nd);
#pragma unroll
        for (int i = 0; i < FL; i++) x[i] = var[base + min(t + i * T, last)];
    }
    part_load_edges<R, T, EPT>(P, ecode, ew, nloc, t, code, w0, w1, w2);
#pragma unroll
    for (int q = 0; q < NPT; q++) {
        part_ready(nd[q]);
        if (RS == 6) nd[q] = t + q * T < P.cnt ? P.n0 + t + q * T : nd[q];
    }
#pragma unroll
    for (int q = 0; q < NPT; q++)
#pragma unroll
        for (int v = 0; v < 5; v++) U[q][v] = var[(size_t)nd[q] * 5 + v];
#pragma unroll
    for (int i = 0; i < FL; i++) fl[i] = fresh ? 0.0 : flux[base + min(t + i * T, last)];
    if constexpr (RS == 6) part_slot_records<R, T, NPT>(P, t, U, rec);
    else part_records<R, T, NPT, FL, RS>(P, t, x, U, rec);
#pragma unroll
    for (int i = 0; i < FL; i++)
        if (t + i * T <= last) acc[t + i * T] = fl[i];
    __syncthreads();
    // 2./3. edges
    part_edges<R, EPT, COLOURED, RS, false>(P, rec, acc, code, w0, w1, w2, (R)k.sc);
    if (halt) return;
    // 4. store
    double* fw = flux + base;
    for (int j = t; j <= last; j += T) fw[j] = acc[j];
}

// Local-edge weights of the part kernels (Real: FP64, or FP32 for mixed
// precision): -w / 2 of each local edge's weights, gathered from the weight
// dat into three component arrays.  The halving is exact.
template <typename Real>
__global__ void k_pack_part_weights(long long n, const int* __restrict__ eid, const double* __restrict__ w,
                                    Real* __restrict__ out)
{
    const long long k = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const size_t e = (size_t)eid[k];
    out[k] = (Real)(-0.5 * w[3 * e]);
    out[n + k] = (Real)(-0.5 * w[3 * e + 1]);
    out[2 * n + k] = (Real)(-0.5 * w[3 * e + 2]);
}

// ------------------------------------------------------------------------
// Edge flux, node-centric gather without LDS: one thread per node, every
// incidence re-evaluates the neighbour's state from global memory.
// ------------------------------------------------------------------------
template <bool EXACT>
__global__ __launch_bounds__(kBlock) void k_flux_gather(
    int n_targets, const int* __restrict__ targets, const int* __restrict__ ptr,
    const int2* __restrict__ inc, const double4* __restrict__ wpk,
    const double* __restrict__ var, double* __restrict__ flux, Consts k,
    const int* __restrict__ status, int fresh)
{
    if (halted(status)) return;
    const int tid = xcd_block() * kBlock + threadIdx.x;
    if (tid >= n_targets) return;
    const int n = targets ? targets[tid] : tid;
    double U[5], acc[5];
    load5(var, n, U);
    if (fresh) {
#pragma unroll
        for (int v = 0; v < 5; v++) acc[v] = 0.0;
    } else {
        load5(flux, n, acc);
    }
    Th o;
    thermo<EXACT>(U, o);
    const int beg = ptr[tid], end = ptr[tid + 1];
    for (int q = beg; q < end; q++) {
        const int2 r = inc[q];
        const double4 w = wpk[r.y & 0x7fffffff];
        double X[5];
        load5(var, r.x, X);
        Th t;
        thermo<EXACT>(X, t);
        double fx = -0.5 * w.x, fy = -0.5 * w.y, fz = -0.5 * w.z;
        if (r.y < 0) { fx = -fx; fy = -fy; fz = -fz; }   // node is endpoint b
        double d[5];
        edge_increment<EXACT>(o, t, w.w, k.sc, fx, fy, fz, d);
#pragma unroll
        for (int v = 0; v < 5; v++) acc[v] = add_exact(acc[v], d[v]);
    }
    store5(flux, n, acc);
}

// Edge flux, edge-parallel with FP64 hardware atomics (global_atomic_add_f64).
__global__ __launch_bounds__(kBlock) void k_flux_atomic(
    int n_edges, const int2* __restrict__ e2n, const double4* __restrict__ wpk,
    const double* __restrict__ var, double* __restrict__ flux, Consts k, const int* __restrict__ status)
{
    if (halted(status)) return;
    const int e = xcd_block() * kBlock + threadIdx.x;
    if (e >= n_edges) return;
    const int2 ab = e2n[e];
    const double4 w = wpk[e];
    double Ua[5], Ub[5];
    load5(var, ab.x, Ua);
    load5(var, ab.y, Ub);
    Th a, b;
    thermo_fast(Ua, a);
    thermo_fast(Ub, b);
    const double fx = -0.5 * w.x, fy = -0.5 * w.y, fz = -0.5 * w.z;
    double da[5], db[5];
    edge_increment_fast(a, b, w.w, k.sc, fx, fy, fz, da);
    edge_increment_fast(b, a, w.w, k.sc, -fx, -fy, -fz, db);
#pragma unroll
    for (int v = 0; v < 5; v++) {
        unsafeAtomicAdd(&flux[5 * (size_t)ab.x + v], da[v]);
        unsafeAtomicAdd(&flux[5 * (size_t)ab.y + v], db[v]);
    }
}

// unstructured_stream.h:7-57 as a gather: same data movement as the flux
// kernel with (almost) no arithmetic.
__global__ __launch_bounds__(kBlock) void k_stream_gather(
    int n_targets, const int* __restrict__ targets, const int* __restrict__ ptr,
    const int2* __restrict__ inc, const double4* __restrict__ wpk,
    const double* __restrict__ var, double* __restrict__ flux)
{
#pragma clang fp contract(off)
    const int tid = xcd_block() * kBlock + threadIdx.x;
    if (tid >= n_targets) return;
    const int n = targets ? targets[tid] : tid;
    double acc[5];
    load5(flux, n, acc);
    for (int q = ptr[tid]; q < ptr[tid + 1]; q++) {
        const int2 r = inc[q];
        double u[5];
        load5(var, r.x, u);
        if (r.y >= 0) {     // node is a: fluxes_a += b-values (+ weights)
            const double4 w = wpk[r.y];
            acc[0] += u[0] + w.x;
            acc[1] += u[1] + w.z;
            acc[2] += u[2];
            acc[3] += u[3];
            acc[4] += u[4] + w.y;
        } else {            // node is b: fluxes_b += a-values
#pragma unroll
            for (int v = 0; v < 5; v++) acc[v] += u[v];
        }
    }
    store5(flux, n, acc);
}

// Plain device-to-device copy (16-byte elements, grid-stride): the
// calibration kernel for bandwidth and for the HBM traffic counters.
__global__ __launch_bounds__(kBlock) void k_stream_copy(size_t n, const double2* __restrict__ a,
                                                        double2* __restrict__ b)
{
    for (size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (size_t)gridDim.x * kBlock) b[i] = a[i];
}

// Rows [r0, r0 + rows) of a dat in the caller's element order, written to
// pinned host memory: row r is the device's row idx[r] (idx null: row r).
// Bound by the host link: consecutive lanes write consecutive elements.
template <typename E>
__global__ __launch_bounds__(kBlock) void k_fetch_rows(int r0, int rows, int dim, const int* __restrict__ idx,
                                                       const E* __restrict__ src, E* __restrict__ out)
{
    const int n = rows * dim;
    for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
        const int r = i / dim, v = i - r * dim;
        out[i] = src[(size_t)(idx ? idx[r0 + r] : r0 + r) * dim + v];
    }
}

// Packed edge weights {w0, w1, w2, |w|} (flux.h:48-50).
__global__ void k_pack_weights(int n, const double* __restrict__ w, double4* __restrict__ out)
{
#pragma clang fp contract(off)
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n) return;
    const double a = w[3 * (size_t)e], b = w[3 * (size_t)e + 1], c = w[3 * (size_t)e + 2];
    out[e] = make_double4(a, b, c, sqrt(a * a + b * b + c * c));
}

// ------------------------------------------------------------------------
// Boundary / far-field flux (flux.h:14-39): one thread per boundary node,
// entries in boundary-element order.
// ------------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void k_bnd_flux(
    int n_targets, const int* __restrict__ targets, const int* __restrict__ ptr,
    const int* __restrict__ ent, const int* __restrict__ group, const double* __restrict__ bw,
    const double* __restrict__ var, double* __restrict__ flux, Consts k, const int* __restrict__ status)
{
#pragma clang fp contract(off)
    if (halted(status)) return;
    const int tid = blockIdx.x * blockDim.x + threadIdx.x;
    if (tid >= n_targets) return;
    const int n = targets[tid];
    double U[5], acc[5];
    load5(var, n, U);
    load5(flux, n, acc);
    Th b;
    thermo_exact(U, b);
    for (int q = ptr[tid]; q < ptr[tid + 1]; q++) {
        const int e = ent[q];
        const int g = group[e];
        const double w0 = bw[3 * (size_t)e], w1 = bw[3 * (size_t)e + 1], w2 = bw[3 * (size_t)e + 2];
        if (g <= 2) {
            // flux_boundary.elem_func:50-54
            acc[0] = acc[0] + 0.0;
            acc[1] = acc[1] + w0 * b.p;
            acc[2] = acc[2] + w1 * b.p;
            acc[3] = acc[3] + w2 * b.p;
            acc[4] = acc[4] + 0.0;
        } else if (g <= 7) {
            // flux_wall.elem_func:103-130
            const double fx = 0.5 * w0, fy = 0.5 * w1, fz = 0.5 * w2;
            acc[0] += fx * (k.ffv[1] + b.mx) + fy * (k.ffv[2] + b.my) + fz * (k.ffv[3] + b.mz);
            acc[4] += fx * (k.ffde[0] + b.fdx) + fy * (k.ffde[1] + b.fdy) + fz * (k.ffde[2] + b.fdz);
            acc[1] += fx * (k.ffmx[0] + b.fxx) + fy * (k.ffmx[1] + b.fxy) + fz * (k.ffmx[2] + b.fxz);
            acc[2] += fx * (k.ffmy[0] + b.fxy) + fy * (k.ffmy[1] + b.fyy) + fz * (k.ffmy[2] + b.fyz);
            acc[3] += fx * (k.ffmz[0] + b.fxz) + fy * (k.ffmz[1] + b.fyz) + fz * (k.ffmz[2] + b.fzz);
        }
    }
    store5(flux, n, acc);
}

// ------------------------------------------------------------------------
// Element-wise kernels
// ------------------------------------------------------------------------
__global__ void k_fill5(int n, double* __restrict__ x, Consts k, int use_ff)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
#pragma unroll
    for (int v = 0; v < 5; v++) x[5 * (size_t)i + v] = use_ff ? k.ffv[v] : 0.0;
}

__global__ void k_fill(size_t n, double* __restrict__ x, double val)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) x[i] = val;
}

__global__ void k_fill_u64(size_t n, unsigned long long* __restrict__ x, unsigned long long val)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) x[i] = val;
}

__global__ void k_fill_i(size_t n, int* __restrict__ x, int val)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) x[i] = val;
}

__global__ void k_scale(size_t n, double* __restrict__ w, double s)
{
#pragma clang fp contract(off)
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) w[i] *= s;
}

__global__ void k_copy(size_t n, const double* __restrict__ src, double* __restrict__ dst,
                       const int* __restrict__ status)
{
    if (halted(status)) return;
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[i] = src[i];
}

// Block-wide reductions over a 256-thread workgroup (4 waves of 64).
template <int NT = kBlock>
__device__ __forceinline__ double block_min(double x)
{
    __shared__ double sm[NT / kWave];
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) {
        const double y = __shfl_down(x, o, kWave);
        x = (y < x) ? y : x;
    }
    const int lane = threadIdx.x % kWave, w = threadIdx.x / kWave;
    if (lane == 0) sm[w] = x;
    __syncthreads();
    if (threadIdx.x == 0) {
        x = sm[0];
        for (int i = 1; i < NT / kWave; i++) x = (sm[i] < x) ? sm[i] : x;
    }
    return x;
}

// block_min with the result in every thread.
template <int NT = kBlock>
__device__ __forceinline__ double block_min_all(double x)
{
    __shared__ double bc;
    x = block_min<NT>(x);
    if (threadIdx.x == 0) bc = x;
    __syncthreads();
    return bc;
}

template <int NT = kBlock>
__device__ __forceinline__ double block_sum(double x)
{
#pragma clang fp contract(off)
    __shared__ double sm[NT / kWave];
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) x += __shfl_down(x, o, kWave);
    const int lane = threadIdx.x % kWave, w = threadIdx.x / kWave;
    if (lane == 0) sm[w] = x;
    __syncthreads();
    if (threadIdx.x == 0) {
        x = sm[0];
        for (int i = 1; i < NT / kWave; i++) x += sm[i];
    }
    return x;
}

template <int NT = kBlock>
__device__ __forceinline__ int block_sum_i(int x)
{
    __shared__ int smi[NT / kWave];
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) x += __shfl_down(x, o, kWave);
    const int lane = threadIdx.x % kWave, w = threadIdx.x / kWave;
    if (lane == 0) smi[w] = x;
    __syncthreads();
    if (threadIdx.x == 0) {
        x = smi[0];
        for (int i = 1; i < NT / kWave; i++) x += smi[i];
    }
    return x;
}

// Publication of a level's minimum dt by the kernels that compute dt
// (get_min_dt_kernel, time_stepping_kernels.h:34-41, fused into them): every
// workgroup folds its minimum into one of kMinSlots slots of its mesh with a
// 64-bit atomic min on an order-preserving integer image of the double, so
// the first Runge-Kutta stage reduces kMinSlots values instead of one per
// workgroup of the level.  The atomics need no fence (the stage is the next
// kernel on the stream), and spreading the workgroups over slots keeps them
// off one address.  The second stage resets the slots to the empty value
// for the next smoothing step.  min is exact: the order of the atomics does
// not change the result.
constexpr int kMinSlots = 64;
constexpr unsigned long long kMinEmpty = 0xFFEFFFFFFFFFFFFFull;    // min_key(DBL_MAX)

// Order-preserving image of a double (not NaN): unsigned order of the images
// is the order of the values; -0.0 and +0.0 share the image of +0.0.
__device__ __forceinline__ unsigned long long min_key(double d)
{
    const unsigned long long b = (unsigned long long)__double_as_longlong(d == 0.0 ? 0.0 : d);
    return (b >> 63) ? ~b : (b | 0x8000000000000000ull);
}

__device__ __forceinline__ double min_unkey(unsigned long long k)
{
    return __longlong_as_double((long long)((k >> 63) ? (k & 0x7FFFFFFFFFFFFFFFull) : ~k));
}

struct MinPub {
    const int* sblk;            // first block of each segment (null: one segment of gridDim.x blocks)
    unsigned long long* slots;  // kMinSlots per segment
};

// m: the minimum of block b of the level (valid in thread 0).
__device__ __forceinline__ void min_publish(const MinPub& p, int seg, int b, double m)
{
    if (threadIdx.x == 0 && p.slots) {
        const int lo = p.sblk ? p.sblk[seg] : 0;
        atomicMin(p.slots + (size_t)seg * kMinSlots + (b - lo) % kMinSlots, min_key(m));
    }
}

// Candidates for get_min_dt_kernel: like the reference's 'dt < min_dt' test
// starting from DBL_MAX, NaN and values >= DBL_MAX never win.
__device__ __forceinline__ double min_candidate(double d) { return (d < DBL_MAX) ? d : DBL_MAX; }

// calculate_dt_kernel (time_stepping_kernels.h:13-32).  With 'old' non-null
// it also performs copy_double_kernel (copy_double_kernel.h:6-13) and with
// 'part' non-null it emits the per-workgroup min for get_min_dt_kernel.
// dt of node i with state U (time_stepping_kernels.h:13-32).
__device__ __forceinline__ double calc_dt_state(int i, const double U[5], const double* __restrict__ vol,
                                                double* __restrict__ dt)
{
#pragma clang fp contract(off)
    const double rho = U[0], E = U[4];
    const double ux = U[1] / rho, uy = U[2] / rho, uz = U[3] / rho;
    const double ssq = ux * ux + uy * uy + uz * uz;
    const double p = (kGamma - 1.0) * (E - 0.5 * rho * ssq);
    const double c = sqrt(kGamma * p / rho);
    const double v = 0.5 * (cbrt(vol[i]) / (sqrt(ssq) + c));
    dt[i] = v;
    return v;
}

// dt of node i (time_stepping_kernels.h:13-32), optionally saving old = var.
__device__ __forceinline__ double calc_dt_node(int i, const double* __restrict__ var,
                                               const double* __restrict__ vol, double* __restrict__ dt,
                                               double* __restrict__ old)
{
    double U[5];
    load5(var, i, U);
    if (old) store5(old, i, U);
    return calc_dt_state(i, U, vol, dt);
}

// The next smoothing step's calculate_dt + copy (time_stepping_kernels.h:13-32,
// copy_double_kernel.h:6-13) on the level a restriction or prolongation has
// just produced, done by that kernel's thread for its node: dt, old = var and
// the per-workgroup minimum, over plain blocks or a segment block table
// ({segment, first, end} per workgroup, batched solves).
struct DtArgs {
    const int4* blk;
    const double* vol;
    double* dt;
    double* old;
    MinPub pub;
};

__global__ __launch_bounds__(kBlock) void k_calc_dt(
    int n, const double* __restrict__ var, const double* __restrict__ vol,
    double* __restrict__ dt, double* __restrict__ old, const int* __restrict__ status, MinPub pub)
{
#pragma clang fp contract(off)
    if (halted(status)) return;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    double d = DBL_MAX;
    if (i < n) d = min_candidate(calc_dt_node(i, var, vol, dt, old));
    if (pub.slots) min_publish(pub, 0, blockIdx.x, block_min(d));
}

// The standalone reduction loops (get_min_dt, calc_rms, the counts): every
// workgroup of a grid of bounded size reduces a strided share and leaves one
// partial result -- in pinned host memory, where the host combines them after
// the one synchronisation the loop needs anyway (no second kernel, no copy).
constexpr int kRedBlocks = 1024;

// get_min_dt_kernel: per-workgroup min of dt.
__global__ __launch_bounds__(kBlock) void k_min_part(int n, const double* __restrict__ x,
                                                      double* __restrict__ part)
{
    double d = DBL_MAX;
    for (long long i = (long long)blockIdx.x * kBlock + threadIdx.x; i < n; i += (long long)gridDim.x * kBlock) {
        const double y = min_candidate(x[i]);
        d = (y < d) ? y : d;
    }
    const double m = block_min(d);
    if (threadIdx.x == 0) part[blockIdx.x] = m;
}

// Final min over device partials; *out = min(init, partials).
__global__ __launch_bounds__(kBlock) void k_min_final(int np, const double* __restrict__ part, double init,
                                                       double* __restrict__ out)
{
    double m = DBL_MAX;
    for (int i = threadIdx.x; i < np; i += kBlock) m = (part[i] < m) ? part[i] : m;
    m = block_min(m);
    if (threadIdx.x == 0) *out = (m < init) ? m : init;
}

// compute_step_factor_kernel (time_stepping_kernels.h:43-64): sf = min_dt / V.
__global__ void k_step_factor(int n, const double* __restrict__ vol, const double* __restrict__ dmin,
                              double hmin, double* __restrict__ sf, const int* __restrict__ status)
{
    if (halted(status)) return;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double m = dmin ? *dmin : hmin;
    sf[i] = m / vol[i];
}

// time_step_kernel (time_stepping_kernels.h:66-86), one thread per double of
// the [n][5] arrays.
__global__ __launch_bounds__(kBlock) void k_time_step(long long n5, int rk, const double* __restrict__ sf,
                                                      double* __restrict__ flux, const double* __restrict__ old,
                                                      double* __restrict__ var)
{
#pragma clang fp contract(off)
    const long long j = (long long)blockIdx.x * kBlock + threadIdx.x;
    if (j >= n5) return;
    const double factor = sf[j / 5] / (double)(3 + 1 - rk);
    var[j] = old[j] + factor * flux[j];
    flux[j] = 0.0;
}

// One Runge-Kutta stage of a multigrid smoothing step after its edge flux,
// fused into one pass over the nodes: the node's boundary and far-field
// increments (flux.h:14-39, k_bnd_flux's arithmetic in boundary-element
// order), on the first stage the minimum dt (each workgroup reduces the
// per-workgroup minima of k_calc_dt over its mesh, as k_min_final does,
// euler3d.cpp:480-484) and the step factor (time_stepping_kernels.h:43-64),
// the stage update (time_stepping_kernels.h:66-86) and on the last stage the
// residual with its per-workgroup sum of squares and NaN/Inf count
// (validation.h:27-44, 102-115).  Each node sees the same operations in the
// same order as with the separate loops.
struct StageArgs {
    int n, rk;
    const int4* blk;           // batched solves: {segment, first, end} per workgroup; null: plain blocks over n
    const int* sblk;           // batched solves: first workgroup of each segment
    unsigned long long* mslots;   // minimum-dt slots (kMinSlots per segment): read by the first stage,
    int nmslots;                  // reset by the second
    int* mstatus;              // abort code 1 on a negative minimum: one status, or per segment
    int* abort_level;          // ... and the level it arose on
    int level;
    int* zero;                 // first stage: a counter the last stage accumulates into, cleared
    const double* vol;
    double* sf;
    double* flux;
    const double* old;
    double* var;
    const int* bptr;           // boundary elements of node i: bnw[bptr[i] .. bptr[i + 1]) (null: none)
    const double4* bnw;        // per boundary element in that order: {w0, w1, w2, group}
    const Consts* kseg;        // batched solves: far-field constants per segment
    double* res;               // last stage: residual, or null
    double* part;              // last stage, finest level: per-workgroup sum of squares
    int* bad;                  // ... NaN/Inf count: one counter (atomic) ...
    int* badpart;              // ... or per workgroup
    int zero_flux;             // reset the flux to zero (else the next edge flux starts fresh)
    const int* status;
};

// Minimum over the 64 lanes of a wave, in every lane: row shifts leave each
// row's minimum in its last lane, two broadcasts carry it to lane 63.
template <int CTRL, int ROWS>
__device__ __forceinline__ double wave_min_step(double x)
{
    const int lo = __double2loint(x), hi = __double2hiint(x);
    const double y = __hiloint2double(__builtin_amdgcn_update_dpp(hi, hi, CTRL, ROWS, 0xf, false),
                                      __builtin_amdgcn_update_dpp(lo, lo, CTRL, ROWS, 0xf, false));
    return y < x ? y : x;
}
__device__ __forceinline__ double wave_min(double x)
{
    x = wave_min_step<0x111, 0xf>(x);      // row_shr 1, 2, 4, 8
    x = wave_min_step<0x112, 0xf>(x);
    x = wave_min_step<0x114, 0xf>(x);
    x = wave_min_step<0x118, 0xf>(x);
    x = wave_min_step<0x142, 0xa>(x);      // row_bcast 15
    x = wave_min_step<0x143, 0xc>(x);      // row_bcast 31
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(x), 63),
                            __builtin_amdgcn_readlane(__double2loint(x), 63));
}

// First stage: the minimum dt of the workgroup's mesh, reduced by each wave
// from the mesh's slots that the kernel computing dt filled (min_publish;
// 'slot' is this lane's, loaded early); the mesh's first workgroup raises
// abort code 1 on a negative value (euler3d.cpp:476-484).  Second stage: the
// slots are reset for the next smoothing step.
static_assert(kMinSlots == kWave, "one slot per lane");
__device__ __forceinline__ double stage_min_dt(const StageArgs& a, int seg, unsigned long long slot, bool first)
{
    const double mdt = wave_min(min_candidate(min_unkey(slot)));
    if (first && threadIdx.x == 0) {
        if (mdt < 0.0 && a.mstatus[seg] == 0) {
            a.mstatus[seg] = 1;
            *a.abort_level = a.level;
        }
        if (a.zero) *a.zero = 0;
    }
    return mdt;
}

template <int NT>
__device__ __forceinline__ void stage_reset_min(const StageArgs& a)
{
    if (a.rk == 1 && blockIdx.x == 0)
        for (int i = threadIdx.x; i < a.nmslots; i += NT) a.mslots[i] = kMinEmpty;
}

// A node's boundary and far-field increments (flux.h:14-39) added to its flux
// f in boundary-element order; U: its state, [q0, q1): its elements.
__device__ __forceinline__ void stage_bnd(const StageArgs& a, const Consts& k, const double U[5], int q0, int q1,
                                          double f[5])
{
#pragma clang fp contract(off)
    Th b;
    thermo_exact(U, b);
    for (int q = q0; q < q1; q++) {
        const double4 bq = a.bnw[q];
        const int g = (int)bq.w;
        const double w0 = bq.x, w1 = bq.y, w2 = bq.z;
        if (g <= 2) {
            f[0] = f[0] + 0.0;
            f[1] = f[1] + w0 * b.p;
            f[2] = f[2] + w1 * b.p;
            f[3] = f[3] + w2 * b.p;
            f[4] = f[4] + 0.0;
        } else if (g <= 7) {
            const double fx = 0.5 * w0, fy = 0.5 * w1, fz = 0.5 * w2;
            f[0] += fx * (k.ffv[1] + b.mx) + fy * (k.ffv[2] + b.my) + fz * (k.ffv[3] + b.mz);
            f[4] += fx * (k.ffde[0] + b.fdx) + fy * (k.ffde[1] + b.fdy) + fz * (k.ffde[2] + b.fdz);
            f[1] += fx * (k.ffmx[0] + b.fxx) + fy * (k.ffmx[1] + b.fxy) + fz * (k.ffmx[2] + b.fxz);
            f[2] += fx * (k.ffmy[0] + b.fxy) + fy * (k.ffmy[1] + b.fyy) + fz * (k.ffmy[2] + b.fyz);
            f[3] += fx * (k.ffmz[0] + b.fxz) + fy * (k.ffmz[1] + b.fyz) + fz * (k.ffmz[2] + b.fzz);
        }
    }
}

// One node of a Runge-Kutta stage, in the reference's order: f holds node
// i's edge flux; the node's boundary and far-field increments are added
// (stage_bnd, its state read from vin), the step factor is formed on the
// first stage (time_stepping_kernels.h:43-64), the update written to a.var
// (:66-86), the flux reset when asked, and on the last stage the residual
// with its square sum and NaN/Inf count (validation.h:27-44,102-115).
// o: node i's old state; vs: its volume on the first stage, else its step
// factor; [q0, q1): its boundary elements (all loaded by the caller, which
// may issue the loads early).
__device__ __forceinline__ void stage_node(const StageArgs& a, const Consts& k0, int seg, int i,
                                           const double* __restrict__ vin, double f[5], double mdt,
                                           const double o[5], double vs, int q0, int q1, double& s, int& nb)
{
#pragma clang fp contract(off)
    double u[5];
    if (q0 < q1) {
        double U[5];
        load5(vin, i, U);
        stage_bnd(a, a.kseg ? a.kseg[seg] : k0, U, q0, q1, f);
    }
    double sfi;
    if (a.rk == 0) {
        sfi = mdt / vs;
        a.sf[i] = sfi;
    } else {
        sfi = vs;
    }
    const double factor = sfi / (double)(3 + 1 - a.rk);
#pragma unroll
    for (int v = 0; v < 5; v++) u[v] = o[v] + factor * f[v];
    store5(a.var, i, u);
    if (a.zero_flux) {
        const double z[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
        store5(a.flux, i, z);
    }
    if (a.res) {
        double r[5];
#pragma unroll
        for (int v = 0; v < 5; v++) {
            r[v] = u[v] - o[v];
            s += r[v] * r[v];
            nb += (isnan(u[v]) || isinf(u[v])) ? 1 : 0;
        }
        store5(a.res, i, r);
    }
}

// The last stage's per-workgroup square sum and NaN/Inf count (slot w).
template <int NT>
__device__ __forceinline__ void stage_sums(const StageArgs& a, int w, double s, int nb)
{
    if (a.part) {
        const double t = block_sum<NT>(s);
        if (threadIdx.x == 0) a.part[w] = t;
    }
    if (a.bad || a.badpart) {
        const int t = block_sum_i<NT>(nb);
        if (threadIdx.x == 0) {
            if (a.badpart) a.badpart[w] = t;
            else if (t) atomicAdd(a.bad, t);
        }
    }
}

// The same of the kernels with a fused stage: one square sum per 64 nodes
// (thread t: node t of the workgroup's), slots g0 and up.  A level's sums
// are the same whatever parts and threads its size selects, since parts
// start at multiples of 64 nodes of their 256-node patch (patches at their
// mesh's first node).
template <int T>
__device__ __forceinline__ void stage_group_sums(const StageArgs& a, int g0, int cnt, double s, int nb)
{
#pragma clang fp contract(off)
    const int t = threadIdx.x;
    if (a.part) {
#pragma unroll
        for (int o = kWave / 2; o > 0; o >>= 1) s += __shfl_down(s, o, kWave);
        if (t % kWave == 0 && t < cnt) a.part[g0 + t / kWave] = s;
    }
    if (a.bad || a.badpart) {
        nb = block_sum_i<T>(nb);
        if (t == 0) {
            if (a.badpart)
                for (int k = 0; k * kWave < cnt; k++) a.badpart[g0 + k] = k ? 0 : nb;
            else if (nb) atomicAdd(a.bad, nb);
        }
    }
}

// The stage's boundary table: the weights and group of each boundary
// element, in the node -> boundary-element CSR order of 'bent', so a node
// reads its elements as one contiguous run.
__global__ void k_pack_bnd(int nq, const int* __restrict__ bent, const double* __restrict__ bw,
                           const int* __restrict__ bgroup, double4* __restrict__ out)
{
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= nq) return;
    const size_t e = (size_t)bent[q];
    out[q] = make_double4(bw[3 * e], bw[3 * e + 1], bw[3 * e + 2], (double)bgroup[e]);
}

__global__ __launch_bounds__(kBlock) void k_stage(StageArgs a, Consts k0)
{
    if (halted(a.status)) return;
    stage_reset_min<kBlock>(a);
    int i, lim, seg = 0;
    bool first;                // first workgroup of its mesh
    if (a.blk) {
        const int4 B = a.blk[blockIdx.x];
        seg = B.x;
        i = B.y + threadIdx.x;
        lim = B.z;
        first = (int)blockIdx.x == a.sblk[seg];
    } else {
        i = blockIdx.x * blockDim.x + threadIdx.x;
        lim = a.n;
        first = blockIdx.x == 0;
    }
    double mdt = 0.0;
    if (a.rk == 0) {
        mdt = stage_min_dt(a, seg, a.mslots[(size_t)seg * kMinSlots + threadIdx.x % kMinSlots], first);
        if (mdt < 0.0 && a.status) return;   // a halting context aborts before any update
    }
    double s = 0.0;
    int nb = 0;
    if (i < lim) {
        double f[5], o[5];
        load5(a.flux, i, f);
        load5(a.old, i, o);
        const int q0 = a.bptr ? a.bptr[i] : 0, q1 = a.bptr ? a.bptr[i + 1] : 0;
        stage_node(a, k0, seg, i, a.var, f, mdt, o, a.rk == 0 ? a.vol[i] : a.sf[i], q0, q1, s, nb);
    }
    stage_sums<kBlock>(a, blockIdx.x, s, nb);
}

// Node i's factor of the stage update; the step factor itself
// (time_stepping_kernels.h:43-64) is formed on the first stage.  vs: the
// node's volume on the first stage, else its step factor.
__device__ __forceinline__ double stage_factor(const StageArgs& a, int i, double mdt, double vs)
{
    double sfi = vs;
    if (a.rk == 0) {
        sfi = mdt / vs;
        a.sf[i] = sfi;
    }
    return sfi / (double)(3 + 1 - a.rk);
}

// The stage update of a workgroup's owned nodes as one run of doubles
// [base, base + last] of every [n][5] array: u = o + factor f
// (time_stepping_kernels.h:66-86), the flux reset when asked, on the last
// stage the residual with its square sum and NaN/Inf count.  fac, acc: the
// nodes' factors and fluxes in LDS; o: the old state, T apart.  The square
// sum is formed node by node (thread t: node t), so that the reduction does
// not depend on the number of threads.
template <int T, int FL>
__device__ __forceinline__ void stage_run(const StageArgs& a, size_t base, int last, const double o[FL],
                                          const double* fac, double* acc, double& s, int& nb)
{
#pragma clang fp contract(off)
#pragma unroll
    for (int i = 0; i < FL; i++) {
        const int j = threadIdx.x + i * T;
        if (j <= last) {
            const double u = o[i] + fac[j / 5] * acc[j];
            a.var[base + j] = u;
            if (a.zero_flux) a.flux[base + j] = 0.0;
            if (a.res) {
                const double r = u - o[i];
                nb += (isnan(u) || isinf(u)) ? 1 : 0;
                a.res[base + j] = r;
                if (a.part) acc[j] = r;      // this thread alone has read it
            }
        }
    }
    if (a.part) {
        __syncthreads();
        const int j = threadIdx.x * 5;
        if (j <= last)
            for (int v = 0; v < 5; v++) s += acc[j + v] * acc[j + v];
    }
}

// The blocked gather fused with its Runge-Kutta stage, as the part kernels
// below: the thread that has summed its node's edges adds the boundary
// increments, then the update runs over the block's run of doubles.  The
// stages read one state buffer and write another (vin, a.var).  Against the
// flux kernel and a stage kernel of its own this saves a launch (about 4 us
// each on a small level) and the flux's way through memory per stage: cycle of
// a 300K-node solve 572 -> 468 us, 1M nodes 1341 -> 1187 us, 10K 280 -> 234 us.
template <bool EXACT, int CH, int NH, int PN, int LPN>
__global__ __launch_bounds__(PN * LPN) void k_gather_stage(GatherPlan G, const int* __restrict__ pseg,
                                                           const int* __restrict__ pfirst,
                                                           const double* __restrict__ vin, int fresh, StageArgs a,
                                                           Consts k0)
{
    constexpr int T = PN * LPN, FL = (5 * PN + T - 1) / T;
    extern __shared__ double sm[];
    const int halt = status_of(a.status);      // tested before the first global write
    const int p = xcd_block(), t = threadIdx.x, n = t / LPN;
    const BlkInfo B = G.blk[p];
    const int seg = word_or_zero(pseg, p);
    const int last = 5 * B.cnt - 1, own = B.n0 + min(n, B.cnt - 1);
    const bool head = n < B.cnt && t % LPN == 0;       // one lane per owned node
    const size_t base = (size_t)B.n0 * 5;
    const double vs = a.rk == 0 ? a.vol[own] : a.sf[own];
    const int q0 = a.bptr ? a.bptr[own] : 0, q1 = a.bptr ? a.bptr[own + 1] : 0;
    const unsigned long long slot = a.rk == 0 ? a.mslots[(size_t)seg * kMinSlots + t % kMinSlots] : kMinEmpty;
    double acc[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    if (!fresh) load5(a.flux, own, acc);
    Th o;
    gather_block<EXACT, CH, NH, PN, LPN>(G, B, vin, k0.sc, sm, acc, o);
    if (halt) return;
    double mdt = 0.0;
    if (a.rk == 0) {
        mdt = stage_min_dt(a, seg, slot, pseg ? p == pfirst[seg] : p == 0);
        if (mdt < 0.0 && a.status) return;
    }
    double old[FL];
#pragma unroll
    for (int i = 0; i < FL; i++) old[i] = (a.old + base)[min((unsigned)t + i * T, (unsigned)last)];
    double f = 0.0;
    if (head) {
        if (q0 < q1) {
            const double U[5] = {o.rho, o.mx, o.my, o.mz, o.E};
            stage_bnd(a, a.kseg ? a.kseg[seg] : k0, U, q0, q1, acc);
        }
        f = stage_factor(a, own, mdt, vs);
    }
    __syncthreads();            // every record has been read: the space takes the fluxes and factors
    double* fl = sm;
    double* fac = sm + 5 * PN;
    if (head) {
#pragma unroll
        for (int v = 0; v < 5; v++) fl[n * 5 + v] = acc[v];
        fac[n] = f;
    }
    __syncthreads();
    double s = 0.0;
    int nb = 0;
    stage_run<T, FL>(a, base, last, old, fac, fl, s, nb);
    stage_group_sums<T>(a, B.g0, B.cnt, s, nb);
    stage_reset_min<T>(a);
}

// The FP64 / mixed part kernel fused with its Runge-Kutta stage (device
// multigrid driver): a part's accumulators hold the complete edge flux of its
// owned nodes, so the stage update of those nodes runs in the same
// workgroup.  Other parts read the stage's input state as their halo while
// this one writes its update, so the input (vin) and the update (a.var) are
// different buffers.  The edge flux starts from the flux dat where that may
// hold something (fresh == 0), else from zero; it is not written back.
// pseg / pfirst: segment of each part and first part of each segment
// (batched solves), null for one mesh.  Returns false when the context has
// halted or aborts (negative minimum dt).
//
// Bound by memory traffic on levels that fill the chip, by one workgroup's
// latency on smaller ones.  A part's owned nodes are one run of 5 * cnt
// doubles in every [n][5] array, and the stage update is the same for each
// double, so the owned state, the old state, the old flux and all results
// move as that run, consecutive doubles by consecutive lanes (per-node
// accesses at a 40-byte stride touch three times as many lines); only the
// halo is gathered node by node.  Cycle of a 1M-node solve 908 -> 863 us,
// 300K nodes 397 -> 384 us, 10K 213 -> 196 us (the minimum-dt slots, one per
// lane, are loaded early too).  NPT: halo nodes per thread; PN: most owned
// nodes.
template <typename R, int T, int EPT, int NPT, bool COLOURED, int RS, int PN>
__device__ __forceinline__ bool part_stage_one(
    int p, const PartInfo* __restrict__ parts, const int* __restrict__ halo, const unsigned* __restrict__ ecode,
    const R* __restrict__ ew, long long nloc, int rec_cap, const double* __restrict__ vin, int fresh,
    const StageArgs& a, const Consts& k0, const int* __restrict__ pseg, const int* __restrict__ pfirst, double* sm)
{
    constexpr int ST = part_stride<R, RS>();
    constexpr int FL = (5 * PN + T - 1) / T;
    static_assert(T >= PN, "one owned node per thread");
    // a halted context writes nothing: the status is tested after the edge
    // phase (which writes only LDS), so its load overlaps the staging loads
    const int halt = status_of(a.status);
    const PartInfo P = parts[p];
    const int seg = word_or_zero(pseg, p);
    const int t = threadIdx.x;
    R* rec = reinterpret_cast<R*>(sm);
    double* acc = sm + part_rec_doubles<R, RS>(rec_cap);
    double* fac = acc + 5 * PN;
    // 1. loads, all clamped into the part so that they issue without branches
    const int last = 5 * P.cnt - 1;
    const size_t base = (size_t)P.n0 * 5;
    int nd[NPT];
    unsigned code[EPT];
    R w0[EPT], w1[EPT], w2[EPT];
    double x[FL], o[FL], U[NPT][5];
    part_load_halo<T, NPT>(P, halo, t, nd);
#pragma unroll
    for (int i = 0; i < FL; i++) x[i] = vin[base + min(t + i * T, last)];
    part_load_edges<R, T, EPT>(P, ecode, ew, nloc, t, code, w0, w1, w2);
    const int own = P.n0 + min(t, max(P.cnt - 1, 0));
    const double vs = a.rk == 0 ? a.vol[own] : a.sf[own];
    const int q0 = a.bptr ? a.bptr[own] : 0, q1 = a.bptr ? a.bptr[own + 1] : 0;
    const unsigned long long slot = a.rk == 0 ? a.mslots[(size_t)seg * kMinSlots + t % kMinSlots] : kMinEmpty;
#pragma unroll
    for (int k = 0; k < NPT; k++) {
        part_ready(nd[k]);
#pragma unroll
        for (int v = 0; v < 5; v++) U[k][v] = vin[(size_t)nd[k] * 5 + v];
    }
#pragma unroll
    for (int i = 0; i < FL; i++) o[i] = a.rk == 0 ? x[i] : a.old[base + min(t + i * T, last)];
    // 2. records and accumulators into LDS
#pragma unroll
    for (int i = 0; i < FL; i++) {
        const int j = t + i * T;
        if (j <= last) acc[j] = fresh ? 0.0 : a.flux[base + j];
    }
    part_records<R, T, NPT, FL, RS>(P, t, x, U, rec);
    __syncthreads();
    if constexpr (RS == 6) {
        if (t < P.cnt) {
            R* r = rec + t * ST;
            r[5] = part_speed<R>(r[0], r[1], r[2], r[3], r[4]);
        }
        __syncthreads();
    }
    // 3. edges
    part_edges<R, EPT, COLOURED, RS, (sizeof(R) == 4 && EPT > 4)>(P, rec, acc, code, w0, w1, w2, (R)k0.sc);
    if (halt) return false;
    // 4. the owned nodes' boundary increments and step factors
    double mdt = 0.0;
    if (a.rk == 0) {
        mdt = stage_min_dt(a, seg, slot, pseg ? p == pfirst[seg] : p == 0);
        if (mdt < 0.0 && a.status) return false;
    }
    if (t < P.cnt) {
        if (q0 < q1) {
            double f[5], u[5];
#pragma unroll
            for (int v = 0; v < 5; v++) {
                f[v] = acc[t * 5 + v];
                u[v] = sizeof(R) == sizeof(double) ? (double)rec[t * ST + v] : vin[base + t * 5 + v];
            }
            stage_bnd(a, a.kseg ? a.kseg[seg] : k0, u, q0, q1, f);
#pragma unroll
            for (int v = 0; v < 5; v++) acc[t * 5 + v] = f[v];
        }
        fac[t] = stage_factor(a, own, mdt, vs);
    }
    __syncthreads();
    // 5. update over the run
    double s = 0.0;
    int nb = 0;
    stage_run<T, FL>(a, base, last, o, fac, acc, s, nb);
    stage_group_sums<T>(a, P.g0, P.cnt, s, nb);
    return true;
}

// One workgroup per part.
template <typename R, int T, int EPT, int NPT, bool COLOURED, int RS, int PN>
__global__ __launch_bounds__(T) void k_flux_part_stage(
    const PartInfo* __restrict__ parts, const int* __restrict__ pseg, const int* __restrict__ pfirst,
    const int* __restrict__ halo, const unsigned* __restrict__ ecode, const R* __restrict__ ew, long long nloc,
    int rec_cap, const double* __restrict__ vin, int fresh, StageArgs a, Consts k0)
{
    extern __shared__ double sm[];
    if (part_stage_one<R, T, EPT, NPT, COLOURED, RS, PN>(xcd_block(), parts, halo, ecode, ew, nloc, rec_cap, vin, fresh,
                                                     a, k0, pseg, pfirst, sm))
        stage_reset_min<T>(a);
}

// Persistent workgroups (a grid of a multiple of 8, below nparts): the
// workgroups of each XCD walk that XCD's contiguous slice of the parts with
// a stride, so the slice's halo stays in the XCD's L2 as it does with one
// workgroup per part.  A kernel of its own: the loop costs the one-part
// kernel ~30 VGPRs, a wave per SIMD.
template <typename R, int T, int EPT, int NPT, bool COLOURED, int RS>
__global__ __launch_bounds__(T) void k_flux_part_stage_persistent(
    const PartInfo* __restrict__ parts, const int* __restrict__ halo, const unsigned* __restrict__ ecode,
    const R* __restrict__ ew, long long nloc, int rec_cap, const double* __restrict__ vin, int fresh,
    StageArgs a, Consts k0, const int* __restrict__ pseg, const int* __restrict__ pfirst, int nparts)
{
    extern __shared__ double sm[];
    if (halted(a.status)) return;
    stage_reset_min<T>(a);
    const int x = blockIdx.x % 8, k = blockIdx.x / 8, g = gridDim.x / 8;
    const int per = nparts / 8, rem = nparts % 8;
    const int lo = (x < rem) ? x * (per + 1) : rem * (per + 1) + (x - rem) * per;
    const int hi = lo + per + (x < rem ? 1 : 0);
    for (int p = lo + k; p < hi; p += g) {
        if (!part_stage_one<R, T, EPT, NPT, COLOURED, RS, kPart>(p, parts, halo, ecode, ew, nloc, rec_cap, vin, fresh, a,
                                                          k0, pseg, pfirst, sm))
            return;
        __syncthreads();        // the next part reuses the LDS
    }
}

// residual_kernel (validation.h:27-35), one thread per double.
__global__ __launch_bounds__(kBlock) void k_residual(long long n5, const double* __restrict__ old,
                                                     const double* __restrict__ var, double* __restrict__ res)
{
    const long long j = (long long)blockIdx.x * kBlock + threadIdx.x;
    if (j < n5) res[j] = var[j] - old[j];
}

// calc_rms_kernel as a standalone loop: sum of squares of n doubles per
// workgroup.
__global__ __launch_bounds__(kBlock) void k_sumsq_part(long long n, const double* __restrict__ r,
                                                        double* __restrict__ part)
{
#pragma clang fp contract(off)
    double s = 0.0;
    for (long long i = (long long)blockIdx.x * kBlock + threadIdx.x; i < n; i += (long long)gridDim.x * kBlock)
        s += r[i] * r[i];
    const double t = block_sum(s);
    if (threadIdx.x == 0) part[blockIdx.x] = t;
}

// Sum of the partials [lo, hi) by one workgroup.  Each thread keeps four
// partial sums over entries NT apart, so four loads are in flight per thread
// instead of one (a level-0 sum of an 8M-node mesh has 125K partials); the
// order is fixed, so the sum is deterministic.
template <int NT>
__device__ __forceinline__ double strided_sum(const double* __restrict__ x, const int* __restrict__ cnt, int lo,
                                              int hi, int& nb)
{
#pragma clang fp contract(off)
    double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
    int c = 0;
    int i = lo + (int)threadIdx.x;
    for (; i + 3 * NT < hi; i += 4 * NT) {
        s0 += x[i];
        s1 += x[i + NT];
        s2 += x[i + 2 * NT];
        s3 += x[i + 3 * NT];
        if (cnt) c += cnt[i] + cnt[i + NT] + cnt[i + 2 * NT] + cnt[i + 3 * NT];
    }
    for (; i < hi; i += NT) {
        s0 += x[i];
        if (cnt) c += cnt[i];
    }
    nb = c;
    return (s0 + s1) + (s2 + s3);
}

// The device driver's level-0 RMS sqrt(sum / n) of every mesh, stored at
// hist[mesh][*cycle] (euler3d.cpp:532-537), and abort code 2 on a non-zero
// bad-value count (euler3d.cpp:539-548).  One workgroup per mesh; in a cycle
// with a restriction it is one of that kernel's workgroups (mg_sum), which
// takes the reduction's own launch and latency off the cycle.
struct SumArgs {
    int n;                  // meshes
    int np;                 // partial sums of a single mesh ...
    const int* sblk;        // ... or each mesh's first one (n + 1)
    const double* part;
    const int* badpart;     // NaN/Inf counts per partial sum, or
    const int* bad;         // one count (halting contexts)
    int nodes;
    const int* seg_nodes;   // nodes of each mesh (null: 'nodes')
    double* hist;
    int cap;                // history entries of a mesh
    const int* cycle;
    int* sstatus;           // per mesh
};

__device__ __forceinline__ void mg_sum(const SumArgs& a, int m)
{
#pragma clang fp contract(off)
    const int lo = a.sblk ? a.sblk[m] : 0, hi = a.sblk ? a.sblk[m + 1] : a.np;
    const int c = *a.cycle;
    const int bad = a.bad ? *a.bad : 0;
    int nb = 0;
    const double s = block_sum(strided_sum<kBlock>(a.part, a.badpart, lo, hi, nb));
    if (a.badpart) nb = block_sum_i(nb);
    if (threadIdx.x == 0) {
        if (c < a.cap) a.hist[(size_t)m * a.cap + c] = sqrt(s / (double)(a.seg_nodes ? a.seg_nodes[m] : a.nodes));
        if (nb + bad > 0 && a.sstatus[m] == 0) a.sstatus[m] = 2;
    }
}

__global__ __launch_bounds__(kBlock) void k_mg_sum(SumArgs a, const int* __restrict__ status)
{
    if (halted(status)) return;
    mg_sum(a, blockIdx.x);
}

// count_bad_vals (validation.h:102-115) and count_non_zeros
// (validation.h:91-100) over n doubles: per-workgroup counts.
template <bool BAD>
__global__ __launch_bounds__(kBlock) void k_count(long long n, const double* __restrict__ x, int* __restrict__ part)
{
    int c = 0;
    for (long long i = (long long)blockIdx.x * kBlock + threadIdx.x; i < n; i += (long long)gridDim.x * kBlock) {
        const double u = x[i];
        c += (BAD ? isnan(u) || isinf(u) : u > 0.0) ? 1 : 0;
    }
    c = block_sum_i(c);
    if (threadIdx.x == 0) part[blockIdx.x] = c;
}

// identify_differences (validation.h:46-89) fused with count_non_zeros
// (validation.h:91-100) when 'count' is set.
__global__ __launch_bounds__(kBlock) void k_identify_differences(
    int n, const double* __restrict__ test, const double* __restrict__ master,
    double* __restrict__ diff, int* __restrict__ count)
{
#pragma clang fp contract(off)
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    int c = 0;
    if (i < n) {
        double tv[5], mv[5], r[5];
        load5(test, i, tv);
        load5(master, i, mv);
#pragma unroll
        for (int v = 0; v < 5; v++) {
            double acc = mv[v] * 10.0e-8;
            if (acc < 0.0) acc *= -1.0;
            if (acc < 3.0e-19) acc = 3.0e-19;
            double d = tv[v] - mv[v];
            if (d < 0.0) d *= -1.0;
            r[v] = (d > acc) ? d : 0.0;
            c += (r[v] > 0.0) ? 1 : 0;
        }
        if (diff) store5(diff, i, r);
    }
    if (count) {
        c = block_sum_i(c);
        if (threadIdx.x == 0 && c) atomicAdd(count, c);
    }
}

// ------------------------------------------------------------------------
// Multigrid transfer (mg.h:29-88)
// ------------------------------------------------------------------------

// up_pre_kernel: zero the coarse targets of every fine node (writes of the
// same value from several children are benign).
__global__ void k_up_pre(int nf, const int* __restrict__ f2c, double* __restrict__ vc,
                         int* __restrict__ scratch, const int* __restrict__ status)
{
    if (halted(status)) return;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nf) return;
    const int c = f2c[i];
    const double z[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    store5(vc, c, z);
    scratch[c] = 0;
}

// up_kernel as a gather over the children of each coarse node, children in
// fine-node order; with 'fused' the up_pre zeroing and the up_post mean are
// folded in (one pass, same arithmetic).
__global__ __launch_bounds__(kBlock) void k_up_gather(
    int n_targets, const int* __restrict__ targets, const int* __restrict__ ptr,
    const int* __restrict__ child, const double* __restrict__ vf, double* __restrict__ vc,
    int* __restrict__ scratch, int fused, const int* __restrict__ status)
{
#pragma clang fp contract(off)
    if (halted(status)) return;
    const int tid = blockIdx.x * blockDim.x + threadIdx.x;
    if (tid >= n_targets) return;
    const int c = targets ? targets[tid] : tid;
    const int beg = ptr[tid], end = ptr[tid + 1];
    double acc[5];
    int cnt;
    if (fused) {
        if (beg == end) return;           // no children: stale value kept (mg.h:58)
#pragma unroll
        for (int v = 0; v < 5; v++) acc[v] = 0.0;
        cnt = 0;
    } else {
        load5(vc, c, acc);
        cnt = scratch[c];
    }
    for (int q = beg; q < end; q++) {
        double x[5];
        load5(vf, child[q], x);
#pragma unroll
        for (int v = 0; v < 5; v++) acc[v] += x[v];
        cnt += 1;
    }
    if (fused) {
        const double avg = cnt == 0 ? 1.0 : 1.0 / (double)cnt;
#pragma unroll
        for (int v = 0; v < 5; v++) acc[v] *= avg;
    }
    store5(vc, c, acc);
    scratch[c] = cnt;
}

// up_post_kernel: mean over children (count 0 keeps the value), one thread per
// double.
__global__ __launch_bounds__(kBlock) void k_up_post(long long n5, double* __restrict__ vc,
                                                    const int* __restrict__ scratch)
{
#pragma clang fp contract(off)
    const long long j = (long long)blockIdx.x * kBlock + threadIdx.x;
    if (j >= n5) return;
    const int s = scratch[j / 5];
    vc[j] *= s == 0 ? 1.0 : 1.0 / (double)s;
}

// The nodes [lo, lo + cnt) of one transfer workgroup, and its segment.
struct NodeBlock {
    int lo, cnt, seg;
};
__device__ __forceinline__ NodeBlock node_block(const int4* blk, int b, int n)
{
    if (blk) {
        const int4 B = blk[b];
        return {B.y, B.z - B.y, B.x};
    }
    return {b * kBlock, min(kBlock, n - b * kBlock), 0};
}

// A workgroup's states in LDS (five doubles per node) written to [n][5]
// arrays as one run, consecutive doubles by consecutive lanes.
__device__ __forceinline__ void store_run(const NodeBlock& B, const double* lds, double* __restrict__ a,
                                          double* __restrict__ b)
{
    const size_t base = (size_t)B.lo * 5;
    for (int j = threadIdx.x; j < 5 * B.cnt; j += kBlock) {
        const double x = lds[j];
        if (a) a[base + j] = x;
        b[base + j] = x;
    }
}

// up_pre + up + up_post (mg.h:29-64) as one gather per coarse node of a
// restriction whose every coarse node is a target (dense plan), followed by
// the coarse level's calculate_dt.  The first sum.n workgroups reduce the
// level-0 RMS instead (a restriction from level 0): they run beside the
// restriction, which reads the bad-value count itself and stops as the
// status they set would stop it.  vc null: the state is needed only as the
// old state (the fused stages read that and write the variables).  Bound by
// the children's gather; with the results stored per node instead of as runs
// the 1M-node solve's restrictions took 32, 21 and 16 us, now 22, 15 and 12.
__global__ __launch_bounds__(kBlock) void k_up_gather_dt(
    int nc, const int* __restrict__ ptr, const int* __restrict__ child, const double* __restrict__ vf,
    const double* __restrict__ vc0, double* __restrict__ vc, int* __restrict__ scratch,
    const int* __restrict__ status, DtArgs d, SumArgs sum)
{
#pragma clang fp contract(off)
    __shared__ double run[5 * kBlock];
    if (halted(status)) return;
    if ((int)blockIdx.x < sum.n) {
        mg_sum(sum, blockIdx.x);
        return;
    }
    if (sum.bad && *sum.bad > 0) return;
    const int b = blockIdx.x - sum.n;
    const NodeBlock B = node_block(d.blk, b, nc);
    const int t = threadIdx.x;
    double m = DBL_MAX;
    if (t < B.cnt) {
        const int c = B.lo + t;
        const int beg = ptr[c], end = ptr[c + 1];
        double acc[5];
        if (beg == end) {
            load5(vc0, c, acc);            // no children: stale value kept (mg.h:58)
        } else {
#pragma unroll
            for (int v = 0; v < 5; v++) acc[v] = 0.0;
            int cnt = 0;
            for (int q = beg; q < end; q++) {
                double x[5];
                load5(vf, child[q], x);
#pragma unroll
                for (int v = 0; v < 5; v++) acc[v] += x[v];
                cnt += 1;
            }
            const double avg = 1.0 / (double)cnt;
#pragma unroll
            for (int v = 0; v < 5; v++) acc[v] *= avg;
            scratch[c] = cnt;
        }
#pragma unroll
        for (int v = 0; v < 5; v++) run[t * 5 + v] = acc[v];
        m = min_candidate(calc_dt_state(c, acc, d.vol, d.dt));
    }
    m = block_min(m);                      // its barrier also completes the run
    store_run(B, run, vc, d.old);
    min_publish(d.pub, B.seg, b, m);
}

// Inverse distance 1 / |p - q| as mg.h:134,147,170,183 form it (exact:
// no contraction, IEEE square root and division).
__device__ __forceinline__ double down_v2_idist(const double* __restrict__ p, const double* __restrict__ q)
{
#pragma clang fp contract(off)
    const double dx = p[0] - q[0], dy = p[1] - q[1], dz = p[2] - q[2];
    return 1.0 / sqrt(dx * dx + dy * dy + dz * dz);
}

// down_v2_kernel (mg.h:101-191) as a gather: one thread per fine node walks
// its incidences of the edge map in element order (the OP2 sequential order)
// and applies, for its own side of each edge, what the reference applies
// through its OP_INC pointers:
//   - the node coincides with its coarse parent: the sums are set to the
//     parent's residual and 1 (mg.h:124-132, 160-167), on every such edge;
//   - side a: + w(a, parent a) r(parent a) + w(parent b, a) r(parent b);
//   - side b: + w(b, parent b) r(parent b) + w(parent a, b) r(parent b) --
//     the reference's b side takes b's parent residual in both terms.
// The sums start from the dats' values (OP_INC), so the result is bitwise
// the sequential one.  e2mg is the edge-->mg_nodes map, internal ids.
__global__ __launch_bounds__(kBlock) void k_down_v2(
    int n_targets, const int* __restrict__ targets, const int* __restrict__ ptr, const int2* __restrict__ inc,
    const int* __restrict__ e2mg, const double* __restrict__ xf, const double* __restrict__ xc,
    const double* __restrict__ rc, double* __restrict__ rp, double* __restrict__ wsum)
{
#pragma clang fp contract(off)
    const int tid = blockIdx.x * blockDim.x + threadIdx.x;
    if (tid >= n_targets) return;
    const int n = targets ? targets[tid] : tid;
    const double x2[3] = {xf[3 * (size_t)n], xf[3 * (size_t)n + 1], xf[3 * (size_t)n + 2]};
    double acc[5], w = wsum[n];
    load5(rp, n, acc);
    for (int q = ptr[tid]; q < ptr[tid + 1]; q++) {
        const unsigned code = (unsigned)inc[q].y;
        const size_t e = code & 0x7fffffffu;
        const int side = (int)(code >> 31);
        const int own = e2mg[2 * e + side], oth = e2mg[2 * e + (1 - side)];
        const double* x1 = xc + 3 * (size_t)own;
        double r1[5];
        load5(rc, own, r1);
        if (x2[0] - x1[0] == 0.0 && x2[1] - x1[1] == 0.0 && x2[2] - x1[2] == 0.0) {
#pragma unroll
            for (int v = 0; v < 5; v++) acc[v] = r1[v];
            w = 1.0;
            continue;
        }
        double d = down_v2_idist(x2, x1);
#pragma unroll
        for (int v = 0; v < 5; v++) acc[v] += d * r1[v];
        w += d;
        d = down_v2_idist(xc + 3 * (size_t)oth, x2);
        if (side == 0) load5(rc, oth, r1);
#pragma unroll
        for (int v = 0; v < 5; v++) acc[v] += d * r1[v];
        w += d;
    }
    store5(rp, n, acc);
    wsum[n] = w;
}

// down_v2_kernel_post (mg.h:193-204): var += res - rp / wsum.
__global__ void k_down_v2_post(int n, const double* __restrict__ rp, const double* __restrict__ wsum,
                               const double* __restrict__ rf, double* __restrict__ vf)
{
#pragma clang fp contract(off)
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double u[5], r[5], p[5];
    load5(vf, i, u);
    load5(rf, i, r);
    load5(rp, i, p);
    const double w = wsum[i];
#pragma unroll
    for (int v = 0; v < 5; v++) u[v] += r[v] - (p[v] / w);
    store5(vf, i, u);
}

// down_kernel (mg.h:66-88).  DT: followed by the fine
// level's calculate_dt.  END: the cycle's last kernel, which also moves the
// cycle counter on.  The fine states and residuals come and go as runs of
// doubles (consecutive lanes, consecutive doubles); each thread gathers its
// node's coarse residual and distances into LDS, where the run's doubles
// find them.  vf_out null: the state is needed only as the old state.  Bound by
// memory traffic on large levels (550K nodes 33 -> 24 us, 370K 24 -> 19 us
// against per-node loads and stores), by its latency below 50K nodes (5 us).
template <bool DT, bool END>
__global__ __launch_bounds__(kBlock) void k_down_mg(
    int nf, const int* __restrict__ f2c, const double* vf, double* vf_out, const double* __restrict__ rf,
    const double* __restrict__ xf, const double* __restrict__ rc, const double* __restrict__ xc,
    const int* __restrict__ status, int* __restrict__ cycle, DtArgs d)
{
#pragma clang fp contract(off)
    __shared__ double step[5 * kBlock], dist[4 * kBlock];
    if (halted(status)) return;
    const int b = blockIdx.x, t = threadIdx.x;
    if (END && b == 0 && t == 0) *cycle += 1;
    const NodeBlock B = node_block(d.blk, b, nf);
    const size_t base = (size_t)B.lo * 5;
    const int last = 5 * B.cnt - 1;
    const int i = B.lo + min(t, B.cnt - 1);
    const int c = f2c[i];
    double u[5], r[5];
#pragma unroll
    for (int k = 0; k < 5; k++) {
        const size_t j = base + min(t + k * kBlock, last);
        u[k] = vf[j];
        r[k] = rf[j];
    }
    const double dx = fabs(xf[3 * (size_t)i] - xc[3 * (size_t)c]);
    const double dy = fabs(xf[3 * (size_t)i + 1] - xc[3 * (size_t)c + 1]);
    const double dz = fabs(xf[3 * (size_t)i + 2] - xc[3 * (size_t)c + 2]);
    double ra[5];
    load5(rc, c, ra);
#pragma unroll
    for (int v = 0; v < 5; v++) step[t * 5 + v] = ra[v];
    dist[t * 4] = sqrt(dx * dx + dy * dy + dz * dz);
    dist[t * 4 + 1] = dx;
    dist[t * 4 + 2] = dy;
    dist[t * 4 + 3] = dz;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 5; k++) {
        const int j = t + k * kBlock;
        if (j <= last) {
            const int n = j / 5, v = j % 5;
            u[k] -= dist[n * 4 + (v & 3)] * (step[j] - r[k]);
            if (vf_out) vf_out[base + j] = u[k];
            if constexpr (DT) {
                d.old[base + j] = u[k];
                step[j] = u[k];              // this thread alone reads entry j
            }
        }
    }
    if constexpr (DT) {
        __syncthreads();
        double m = DBL_MAX;
        if (t < B.cnt) m = min_candidate(calc_dt_state(i, step + t * 5, d.vol, d.dt));
        min_publish(d.pub, B.seg, b, block_min(m));
    }
}

// ------------------------------------------------------------------------
// Setup (misc.h:40-84)
// ------------------------------------------------------------------------

// calculate_cell_volumes, edge part: tetra volume per edge and the weight
// rewrite w <- (d/|d|)|w| / |d|.
__global__ void k_cell_volumes_edge(int ne, const int2* __restrict__ e2n, const double* __restrict__ x,
                                    double* __restrict__ w, double* __restrict__ tv)
{
#pragma clang fp contract(off)
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= ne) return;
    const int2 ab = e2n[e];
    double d[3];
    double dist = 0.0;
#pragma unroll
    for (int i = 0; i < 3; i++) {
        d[i] = x[3 * (size_t)ab.y + i] - x[3 * (size_t)ab.x + i];
        dist += d[i] * d[i];
    }
    dist = sqrt(dist);
    double* we = w + 3 * (size_t)e;
    double area = 0.0;
#pragma unroll
    for (int i = 0; i < 3; i++) area += we[i] * we[i];
    area = sqrt(area);
    tv[e] = (1.0 / 3.0) * 0.5 * dist * area;
#pragma unroll
    for (int i = 0; i < 3; i++) {
        double r = (d[i] / dist) * area;
        r /= dist;
        we[i] = r;
    }
}

// calculate_cell_volumes, node part: volumes INC in edge order.
__global__ void k_cell_volumes_node(int n_targets, const int* __restrict__ targets,
                                    const int* __restrict__ ptr, const int2* __restrict__ inc,
                                    const double* __restrict__ tv, double* __restrict__ vol)
{
#pragma clang fp contract(off)
    const int tid = blockIdx.x * blockDim.x + threadIdx.x;
    if (tid >= n_targets) return;
    const int n = targets ? targets[tid] : tid;
    double acc = vol[n];
    for (int q = ptr[tid]; q < ptr[tid + 1]; q++) acc += tv[inc[q].y & 0x7fffffff];
    vol[n] = acc;
}

// ------------------------------------------------------------------------
// Batched solves: per-node work over a segment block table {segment, lo, hi}
// whose blocks never straddle two meshes.
// ------------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void k_calc_dt_seg(const int4* __restrict__ blk, const double* __restrict__ var,
                                                        const double* __restrict__ vol, double* __restrict__ dt,
                                                        double* __restrict__ old, const int* __restrict__ halt,
                                                        MinPub pub)
{
    if (halted(halt)) return;
    const int4 B = blk[blockIdx.x];
    const int i = B.y + threadIdx.x;
    double d = DBL_MAX;
    if (i < B.z) d = min_candidate(calc_dt_node(i, var, vol, dt, old));
    min_publish(pub, B.x, blockIdx.x, block_min(d));
}

// Cycle counter of one-level contexts: counts cycles that ran (a halted
// context stops counting).
__global__ void k_bump(int* c, const int* __restrict__ status)
{
    if (threadIdx.x == 0 && !halted(status)) *c += 1;
}

// Convergence stop of served solves, run after the cycle counter moved on:
// segment s whose L0 RMS of the cycle that just ran has dropped to 'drop'
// times its first cycle's gets status 3, which halts every later kernel of a
// one-segment context (the state stays that of the converged cycle).  In a
// context of several segments nothing halts: the segment's cycle count goes
// to segcyc[s], k_snap_converged copies its state this cycle, and the next
// call marks it copied (snapflag).
__global__ void k_converge(int nseg, int* __restrict__ sstatus, const double* __restrict__ rms, int cap,
                           const int* __restrict__ cycle, double drop, int* __restrict__ snapflag,
                           int* __restrict__ segcyc)
{
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= nseg) return;
    if (sstatus[s] == 3) {
        if (snapflag) snapflag[s] = 1;
        return;
    }
    if (sstatus[s] != 0) return;
    const int c = *cycle - 1;       // the cycle that just ran
    if (c >= 1 && c < cap && rms[(size_t)s * cap + c] <= drop * rms[(size_t)s * cap]) {
        sstatus[s] = 3;
        if (segcyc) segcyc[s] = c + 1;
    }
}

// Level-0 state of the segments that converged in the cycle that just ran
// (status 3, not yet copied), one workgroup per segment block {segment, lo,
// hi}: the result of a served request that keeps running with the other
// members of its group.
__global__ __launch_bounds__(kBlock) void k_snap_converged(int nblocks, const int4* __restrict__ blk,
                                                           const int* __restrict__ sstatus,
                                                           const int* __restrict__ snapflag,
                                                           const double* __restrict__ var, double* __restrict__ snap)
{
    const int b = blockIdx.x;
    if (b >= nblocks) return;
    const int4 q = blk[b];
    if (sstatus[q.x] != 3 || snapflag[q.x]) return;
    for (int i = 5 * q.y + threadIdx.x; i < 5 * q.z; i += kBlock) snap[i] = var[i];
}

}  // namespace mgcfd
