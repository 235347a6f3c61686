// galhip_p3d.hip -- kernels of the 3-D polar grid (p3d): cylindrical rings
// x spokes x z-planes, linear (trilinear) interpolation (jmass = 2).
//
// Mesh cell (ring, plane, spoke) is ((ring)*ngz + plane)*na + spoke, 0-based
// (SRC/lib15/weight.f:232).  The field is held interleaved as one 4-vector
// per cell, (F_x, F_y, F_z, potential), so that an interpolation corner is
// one 16-byte (FP32) load.
//
// Particle kernels:
//   p3_massgn_kernel  massgn of every on-grid particle (massgn.f:140-172)
//   p3_push_kernel    getacc (grdacc.f:189-211, getacc.f:106-151) + stpgrp
//                     + offgrd (|z| > zm or R > rgrid, offgrd.f:69-72) +
//                     addoff + rezgrp with spherical zone radii
//                     (zoneno.f:40-41) + massgn at the new position
//   p3_tmcent_kernel  tmcent's half-step velocity shift
//   p3_gather_kernel  weight / grdacc for given positions (parity checks)
// Solve (p3fndf.f:37-104), FP32 or FP64:
//   p3_analyse_kernel wavefront per (planes, ring): zoncmb + scaled, then the
//                     azimuthal components of the active harmonics
//                     (p3manl.f:60-89) as direct sums
//   p3_zfwd_kernel    block per (columns, ring): the doubled vertical transform of each
//                     component column, zero-padded to 2 ngz (p3manl.f:90-101)
//   p3_conv_kernel    block per (type, k_z, m): the radial contraction with
//                     that Green's matrix (p3conv.f:139-226); table streamed
//                     once, field ring per thread
//   p3_zinv_kernel    block per (columns, type, ring): inverse vertical transform,
//                     first ngz planes (p3fsyn.f:59-91)
//   p3_synth_kernel   block per (planes, ring): inverse azimuthal transform,
//                     1/(2 ngz na) (p3fsyn.f:92-129) and polcat
// p3_green_kernel: p3grnm's tables in FP64 (p3grnm.f:93-263), p3gwrt's
//   per-(k_z, m) matrices with the field ring fastest (p3gwrt.f:46-64).
#include "galhip_p3d.h"

#include <algorithm>
#include <climits>

namespace gh {

constexpr int P3_BLOCK = 256;    // solve kernels
constexpr int P3_PBLOCK = 512;   // particle kernels without a deposit (those: P3Shape)

// (u, t) of particle i: the second half of its record's second R4
template <typename R>
__device__ __forceinline__ void p3_set_ut(const P3Args<R> &a, long long i, R u, R t) {
    reinterpret_cast<typename Vec2<R>::T *>(a.rec + 2 * i + 1)[1] = mk2(u, t);
}
constexpr int P3_MAX_NA = 2048;
constexpr int P3_MAX_NM = 128;   // compact components (2 ng)
constexpr int P3_MAX_NR = 1024;

template <typename R> __device__ __forceinline__ R p3_wave_sum(R v) { return wave_sum_dpp(v); }

// (u, t) of a position as weight() forms them (weight.f:210-218): the FP32
// logarithm and angle of the p2d grid, t = 0 on the axis.
template <typename R>
__device__ __forceinline__ void ut3(R x, R y, const P3Args<R> &a, R &u, R &t) {
    const R rr = sqrt(x * x + y * y);
    ut_of(x, y, rr, a.k, u, t);
    if (!(rr > (R)0)) t = (R)0;
}

// A position's grid coordinates (weight.f:210-230): u, t (folded into the
// sector for mass assignment) and zz = (z + zm) / dzg.
template <typename R> struct P3Pos {
    R u, t, zz;
};
template <typename R>
__device__ __forceinline__ P3Pos<R> pos3(R u, R t, R z, const P3Args<R> &a, bool fold) {
    P3Pos<R> p;
    p.u = u;
    p.t = fold ? (R)fmod(t, a.thmax) : t;
    p.zz = div_rn(z + a.zm, a.dzg);
    return p;
}

// Hides a position's origin from the optimiser (no instruction is issued).
__device__ __forceinline__ void opaque3(P3Pos<float> &p) {
    asm volatile("" : "+v"(p.u), "+v"(p.t), "+v"(p.zz));
}
__device__ __forceinline__ void opaque3(P3Pos<double> &p) {
    asm volatile("" : "+v"(p.u), "+v"(p.t), "+v"(p.zz));
}

// ut3 in the push (ut_push); rr the position's cylindrical radius
template <typename R>
__device__ __forceinline__ void ut3_push(R x, R y, R rr, const P3Args<R> &a, R &u, R &t,
                                         const double *tab) {
    ut_push(x, y, rr, a.k, u, t, tab);
    if (!(rr > (R)0)) t = (R)0;
}

// The cell of a position: ring and plane of the low corner (jmass 2,
// weight.f:219-231) or the nearest node (jmass 3, ring >= 1, t rounding to
// na folded to spoke 0; weight.f:281-292).  For jmass 2 the spoke is na when t
// has rounded to na.
template <typename R, int J>
__device__ __forceinline__ void loc3(const P3Pos<R> &p, const P3Args<R> &a, int &ring, int &plane,
                                     int &spoke) {
    const R h = J == 3 ? (R)0.5 : (R)0;
    ring = J == 3 ? (int)(p.u + h) : (int)p.u;
    plane = J == 3 ? (int)(p.zz + h) : (int)p.zz;
    spoke = J == 3 ? (int)(p.t + h) : (int)p.t;
    if (ring > a.nr - 2) ring = a.nr - 2;
    if (J == 3 && ring < 1) ring = 1;
    if (plane < 0) plane = 0;
    if (plane > a.ngz - 2) plane = a.ngz - 2;
    if (J == 3 && spoke == a.na) spoke = 0;
}
template <typename R>
__device__ __forceinline__ int cell_index(const P3Args<R> &a, int ring, int plane, int spoke) {
    return (ring * a.ngz + plane) * a.na + spoke;
}

// The weights of a position in cell (ring, plane): 8 in the reference's order
// (bit 0 = dt, bit 1 = dz, bit 2 = du; weight.f:232-248), or 27, spoke
// offset -1, 0, +1 fastest, then plane, then ring (weight.f:281-300).
template <typename R>
__device__ __forceinline__ void weights3(const P3Pos<R> &p, int ring, int plane, R (&w)[8]) {
    const R du = p.u - (R)ring, dt = p.t - (R)(int)p.t, dz = p.zz - (R)plane;
    const R one = (R)1;
    w[0] = (one - dt) * (one - dz) * (one - du);
    w[1] = dt * (one - dz) * (one - du);
    w[2] = (one - dt) * dz * (one - du);
    w[3] = dt * dz * (one - du);
    w[4] = (one - dt) * (one - dz) * du;
    w[5] = dt * (one - dz) * du;
    w[6] = (one - dt) * dz * du;
    w[7] = dt * dz * du;
}
template <typename R>
__device__ __forceinline__ void weights3(const P3Pos<R> &p, int ring, int plane, R (&w)[27]) {
    const R h = (R)0.5;
    R dp[3][3];
#pragma unroll
    for (int i = 0; i < 3; i++) {
        const R dd = i == 0 ? p.t + h - (R)(int)(p.t + h) : i == 1 ? p.zz + h - (R)plane
                                                                    : p.u + h - (R)ring;
        dp[0][i] = (R)1 - (R)2 * dd + dd * dd;
        dp[1][i] = (R)1 + (R)2 * dd - (R)2 * (dd * dd);
        dp[2][i] = dd * dd;
    }
#pragma unroll
    for (int k = 0; k < 3; k++)
#pragma unroll
        for (int j = 0; j < 3; j++)
#pragma unroll
            for (int i = 0; i < 3; i++)
                w[9 * k + 3 * j + i] = (R)0.125 * dp[i][0] * dp[j][1] * dp[k][2];
}

// weights per particle of interpolation scheme J (jmass 2 or 3)
template <int J> struct P3NW { static constexpr int v = J == 3 ? 27 : 8; };

// cell index, its parts and the weights of a position given its (u, t)
template <typename R, int J>
__device__ __forceinline__ int cellJ(R u, R t, R z, const P3Args<R> &a, bool fold,
                                     R (&w)[P3NW<J>::v], int &ring, int &plane, int &spoke) {
    const P3Pos<R> p = pos3(u, t, z, a, fold);
    loc3<R, J>(p, a, ring, plane, spoke);
    weights3(p, ring, plane, w);
    return cell_index(a, ring, plane, spoke);
}

// grdacc's corners (grdacc.f:193-203): c, c+1 (wrapped when c+1 is a
// multiple of na), the next plane (+na), and the same one ring out.
__device__ __forceinline__ void corners3(int c, int spoke, int na, int ngz, int ic[8]) {
    const bool wrap = spoke + 1 == na;   // (c + 1) mod na == 0
    ic[0] = c;
    ic[1] = wrap ? c + 1 - na : c + 1;
    ic[2] = c + na;
    ic[3] = ic[1] + na;
    ic[4] = c + ngz * na;
    ic[5] = wrap ? ic[4] + 1 - na : ic[4] + 1;
    ic[6] = ic[4] + na;
    ic[7] = ic[5] + na;
}

// the 27 cells about a central cell c (grdacc.f:262-275, massgn.f:182-195):
// spoke -1, 0, +1 (with the azimuthal wrap) fastest, then plane -1, 0, +1
// (-+ na), then ring -1, 0, +1 (-+ ngz na), as flat indices
__device__ __forceinline__ void corners27(int c, int spoke, int na, int ngz, int ic[27]) {
    int m[3];
    m[1] = c;
    m[0] = spoke == 0 ? c - 1 + na : c - 1;          // c mod na == 0
    m[2] = spoke + 1 == na ? c + 1 - na : c + 1;     // (c + 1) mod na == 0
#pragma unroll
    for (int k = 0; k < 3; k++)
#pragma unroll
        for (int j = 0; j < 3; j++)
#pragma unroll
            for (int i = 0; i < 3; i++) ic[9 * k + 3 * j + i] = m[i] + (j - 1) * na + (k - 1) * ngz * na;
}

// spoke: the central cell's spoke as cellJ gives it (c mod na, or na for a
// linear cell at t == na)
template <int J> __device__ __forceinline__ void cornersJ(int c, int spoke, int na, int ngz,
                                                          int *ic) {
    if constexpr (J == 3) corners27(c, spoke, na, ngz, ic);
    else corners3(c, spoke, na, ngz, ic);
}

template <typename R>
__device__ __forceinline__ R tsfac3(const P3Args<R> &a, int iz) {
    return (R)step_ratio(a.nstep, a.nz, iz);
}

// zoneno with spherical boundaries (zoneno.f:40-55, setrun.f:810)
template <typename R>
__device__ __forceinline__ int zoneno3(const P3Args<R> &a, R x, R y, R z) {
    const R rad = sqrt(x * x + y * y + z * z);
    int k = 1;
    if (a.nz > 1)
        for (int i = 1; i <= a.nz; i++)
            if (rad >= a.zbr[i - 1]) k = i;
    return k;
}

// chstep, RVLF branch (chstep.f:22-31), one component
template <typename R>
__device__ __forceinline__ void chstep1(R tfac, R ox, R &ov, R &acc, R &nx, R &nv) {
    const R h = (R)0.5;
    ov = tfac * (ov + h * acc * ((R)1 - tfac));
    acc = acc * tfac * tfac;
    nv = ov + acc;
    nx = ox + nv;
}

// getacc of one particle of list z0: the three Cartesian components
// interpolated at its position (component sums in corner order), the fixed
// force of the spherical radius, the zone rescaling.
template <typename R, int J>
__device__ __forceinline__ void getacc3(const P3Args<R> &a, R ox, R oy, R oz, R u, R t,
                                        int z0, R acc[3]) {
    typedef typename Vec4<R>::T R4;
    constexpr int NW = P3NW<J>::v;
    acc[0] = acc[1] = acc[2] = (R)0;
    if (z0 != a.nz + 1) {
        R w[NW];
        int ic[NW];
        int rg, pl, sp;
        const int c = cellJ<R, J>(u, t, oz, a, false, w, rg, pl, sp);
        cornersJ<J>(c, sp, a.na, a.ngz, ic);
        R sx = (R)0, sy = (R)0, sz = (R)0;
        // a corner outside the field array (the last ring with t == na; for
        // jmass 3 also the first ring's bottom plane) reads 0: cell 0 is read
        // instead and its weight is 0.  Only a wavefront with such a lane
        // tests its corners.
        const int reach = (a.ngz + 1) * a.na + 1;   // largest corner offset
        if (any_lane(c + reach >= a.mesh || (J == 3 && c < reach))) {
#pragma unroll
            for (int q = 0; q < NW; q++)
                if (ic[q] < 0 || ic[q] >= a.mesh) {
                    ic[q] = 0;
                    w[q] = (R)0;
                }
        }
#pragma unroll
        for (int q = 0; q < NW; q++) {
            const R4 f = a.fld[ic[q]];
            sx = sx + f.x * w[q];
            sy = sy + f.y * w[q];
            sz = sz + f.z * w[q];
        }
        if (a.fixforce) {
            R r2 = (R)0;
            r2 = r2 + ox * ox;
            r2 = r2 + oy * oy;
            r2 = r2 + oz * oz;
            const R rr = sqrt_rn(r2);
            R fr = (R)fixforce((double)rr, a.nfr, a.fr_inv_dr, a.fr_c);
            if (fr != (R)0) {
                fr = div_rn(fr, rr);
                sx = sx + fr * ox;
                sy = sy + fr * oy;
                sz = sz + fr * oz;
            }
        }
        acc[0] = sx;
        acc[1] = sy;
        acc[2] = sz;
    }
    if (a.nz > 1 && z0 > 1) {
        R t = tsfac3(a, z0);
        t = t * t;
        acc[0] = t * acc[0];
        acc[1] = t * acc[1];
        acc[2] = t * acc[2];
    }
}

// Launch shapes of the push and the mass assignment by particles per thread;
// push averaged over an eight-step sort cycle, us.
// Linear FP32, two particles per thread: they share the window's reductions,
// clearing and flush, and 20 KB of LDS leave seven wavefronts per SIMD (2e7
// particles on 200 x 256 x 125: one particle per thread in blocks of 512 with 4096
// cells 681; two in blocks of 256 with 4096, 3072, 2560, 2048 cells 708, 640, 623,
// 736; four 697; two in blocks of 512 689-706).  Fewer particles wait for a
// block's own latency, which grows with the particles per thread, and a sparse
// grid's blocks for the passes that a smaller window takes: two and one per thread
//   n                1e5        1e6        3e6        8e6
//   61 x  90 x  45   38   26    49   40    77   79    159  184
//  140 x 200 x  81   49   40    73   68   125  121    238  256
//  200 x 256 x 125   53   45   129  116   212  197    344  351
// Quadratic: 256 threads with 4096 cells (140 x 200 x 81, 2e6, FP64: 512 threads
// 306, 256 with 2560, 3328 cells 293, 287, with 4096 275; FP32 224 and 194).  Its
// FP64 push spills 14 registers (36 bytes) in the gather of the 27 corners at four
// wavefronts per SIMD; three without spills are slower (512 threads, same case:
// 408 us against 318).
template <typename R, int J, int PPT> struct P3Shape {
    static constexpr int block = PPT == 2 || J == 3 ? 256 : 512;
    static constexpr int tile = PPT == 2 ? 2560 : 4096;
    static constexpr int waves = PPT == 2 ? 7 : 4;
};
constexpr long long P3_TWO = 5000000;   // linear FP32: two per thread above
constexpr int P3_PASSES = 8;   // window passes before the direct fallback

// LDS of a block's deposit.
template <int TILE> struct Deposit3Lds {
    long long tile[TILE];
    int jr[GH_MAXZ], kr[GH_MAXZ];    // central ring ranges by zone
    int box[12];                     // two (min, max) x (ring, plane, spoke) boxes
    unsigned long long ref[2];       // two reference keys
};
template <int TB, int TILE>
__device__ __forceinline__ void deposit3_init(Deposit3Lds<TILE> &s) {
    const int tid = threadIdx.x;
#pragma unroll
    for (int j = 0; j < TILE; j += TB) s.tile[j + tid] = 0;
    if (tid < GH_MAXZ) {
        s.jr[tid] = INT_MAX;
        s.kr[tid] = -1;
    }
    if (tid < 12) s.box[tid] = (tid & 1) ? -1 : INT_MAX;
    if (tid < 2) s.ref[tid] = ~0ull;
}

struct P3Ref {
    int zone, ring, plane, spoke;
};

// Block-level fixed-point deposit.  The block's particles (sorted by cell,
// so a block covers a few neighbouring cells) are accumulated into an LDS
// window spanning the (ring, plane, spoke) box of their corners, then the
// window's non-zero cells are added to the zone array with one global atomic
// each (consecutive cells of a row, so the atomics of a wave coalesce) and
// cleared.  The corners of a central cell are the next ring, plane and spoke
// (jmass 2) or the cells one either side (jmass 3); spokes wrap around the
// ring, so the window's spoke axis runs past na (or below 0) and the flush
// folds it back.  A box larger than TILE cells is clipped to at most 8 rings
// and 8 planes, then as many spokes as fit, placed about a reference cell.
// The particles it leaves out (outliers that have moved away from the
// block's cells, the far rows of a block in a sparse region, other zones)
// get the next pass's window, up to P3_PASSES passes: the first pass takes
// the zone and cell of the block's middle particle, a later one those of the
// first pending particle in particle order from there, which is always
// inside its own window.
// Particles whose corners leave the row structure (the plane next to the
// last or, for jmass 3, the first; a linear cell at t == na) and those still
// left after the last pass add their corners to the zone array directly.
// Integer sums: the result does not depend on the grouping.  Every thread of
// the block must call it; dz[k]: the deposit's zone (0: none).
template <typename R, int J, int PPT, int TB, int TILE>
__device__ __forceinline__ void deposit3_block(const P3Args<R> &a, Deposit3Lds<TILE> &s,
                                               P3Pos<R> (&pos)[PPT], unsigned dzone, P3Ref ref) {
    constexpr int NW = P3NW<J>::v;
    constexpr int LO = J == 3 ? 1 : 0;   // corner cells below the central one
    const int tid = threadIdx.x, lane = tid & 63;
    unsigned pend = 0;
#pragma unroll
    for (int k = 0; k < PPT; k++) {
        int ring, plane, spoke;
        loc3<R, J>(pos[k], a, ring, plane, spoke);
        if ((dzone >> (4 * k) & 15u) && plane - LO >= 0 && plane + 1 < a.ngz && spoke < a.na &&
            ring - LO >= 0)
            pend |= 1u << k;
    }
    unsigned direct = 0;
#pragma unroll
    for (int k = 0; k < PPT; k++)
        if ((dzone >> (4 * k) & 15u) && !(pend >> k & 1u)) direct |= 1u << k;
    auto in_zone = [&](int k, int z) {
        return (pend >> k & 1u) && (int)(dzone >> (4 * k) & 15u) == z;
    };
    // the quadratic scheme's 27 fixed-point weights are formed once: again in
    // every pass, as the linear one's eight, they cost 3 to 9 % (140 x 200 x 81, 3e5,
    // FP64: 104 us, so 96)
    constexpr bool KEEP = J == 3 && PPT == 1;
    long long v0[NW];
    if constexpr (KEEP) {
        int ring, plane, spoke;
        loc3<R, J>(pos[0], a, ring, plane, spoke);
        R w[NW];
        weights3(pos[0], ring, plane, w);
        quant_n<R, NW>(w, a.qbits, dzone != 0, v0);
    }
#pragma unroll 1
    for (int pass = 0;; pass++) {
        int *const sb = s.box + 6 * (pass & 1);
        // cells and weights are formed again from the grid coordinates
        if (!KEEP)
#pragma unroll
            for (int k = 0; k < PPT; k++) opaque3(pos[k]);
        {
            int r0 = INT_MAX, r1 = -1, p0 = INT_MAX, p1 = -1, q0 = INT_MAX, q1 = -1;
#pragma unroll
            for (int k = 0; k < PPT; k++) {
                int ring, plane, spoke;
                loc3<R, J>(pos[k], a, ring, plane, spoke);
                if (in_zone(k, ref.zone)) {
                    r0 = min(r0, ring);
                    r1 = max(r1, ring);
                    p0 = min(p0, plane);
                    p1 = max(p1, plane);
                    q0 = min(q0, spoke);
                    q1 = max(q1, spoke);
                }
            }
            r0 = wave_min_i32(r0);
            r1 = wave_max_i32(r1);
            p0 = wave_min_i32(p0);
            p1 = wave_max_i32(p1);
            q0 = wave_min_i32(q0);
            q1 = wave_max_i32(q1);
            if (lane == 0 && r1 >= 0) {
                atomicMin(&sb[0], r0);
                atomicMax(&sb[1], r1);
                atomicMin(&sb[2], p0);
                atomicMax(&sb[3], p1);
                atomicMin(&sb[4], q0);
                atomicMax(&sb[5], q1);
            }
        }
        __syncthreads();
        // the box of the pending corners, clipped about the reference cell
        int r0 = sb[0] - LO, p0 = sb[2] - LO, q0 = sb[4] - LO;
        int NR = sb[1] - sb[0] + 2 + LO, NP = sb[3] - sb[2] + 2 + LO;
        int NQ = sb[5] - sb[4] + 2 + LO;
        const bool some = sb[1] >= 0;
        if (tid == 0) {
            if (some) {
                atomicMin(&s.jr[ref.zone - 1], sb[0]);
                atomicMax(&s.kr[ref.zone - 1], sb[1]);
            }
            // the other box and key were last read before this barrier
            int *const nb = s.box + 6 * ((pass + 1) & 1);
#pragma unroll
            for (int k = 0; k < 6; k++) nb[k] = (k & 1) ? -1 : INT_MAX;
            s.ref[(pass + 1) & 1] = ~0ull;
        }
        if (some && (long long)NR * NP * NQ > TILE) {
            if (NR > 8) {
                r0 = min(max(ref.ring - LO - 3, r0), r0 + NR - 8);
                NR = 8;
            }
            if (NP > 8) {
                p0 = min(max(ref.plane - LO - 3, p0), p0 + NP - 8);
                NP = 8;
            }
            const int mq = TILE / (NR * NP);
            if (NQ > mq) {
                q0 = min(max(ref.spoke - LO - (mq - 2 - LO) / 2, q0), q0 + NQ - mq);
                NQ = mq;
            }
        }
        const int ncell = some ? NR * NP * NQ : 0;
#pragma unroll
        for (int k = 0; k < PPT; k++) {
            int ring, plane, spoke;
            loc3<R, J>(pos[k], a, ring, plane, spoke);
            const bool inside = in_zone(k, ref.zone) && ring - LO >= r0 && ring - r0 + 1 < NR &&
                                plane - LO >= p0 && plane - p0 + 1 < NP && spoke - LO >= q0 &&
                                spoke - q0 + 1 < NQ;
            if (inside) {
                long long v[NW];
                if constexpr (KEEP) {
#pragma unroll
                    for (int q = 0; q < NW; q++) v[q] = v0[q];
                } else {
                    R w[NW];
                    weights3(pos[k], ring, plane, w);
                    quant_n<R, NW>(w, a.qbits, true, v);
                }
                const int b = ((ring - r0) * NP + (plane - p0)) * NQ + (spoke - q0);
#pragma unroll
                for (int q = 0; q < NW; q++) {
                    int o;
                    if constexpr (J == 3)
                        o = b + (q % 3 - 1) + ((q / 3) % 3 - 1) * NQ + (q / 9 - 1) * NP * NQ;
                    else
                        o = b + ((q & 1) ? 1 : 0) + ((q & 2) ? NQ : 0) + ((q & 4) ? NP * NQ : 0);
                    atomicAdd((unsigned long long *)&s.tile[o], (unsigned long long)v[q]);
                }
                pend &= ~(1u << k);
            }
        }
        // the next reference: the lowest particle index, counted from the
        // block's middle, among the pending deposits
        if (any_lane(pend != 0)) {
            int myrot = INT_MAX;
            unsigned lo = 0, hi = 0;
#pragma unroll
            for (int k = 0; k < PPT; k++) {
                const int rot = (k * TB + tid - TB * PPT / 2) & (TB * PPT - 1);
                int ring, plane, spoke;
                loc3<R, J>(pos[k], a, ring, plane, spoke);
                if ((pend >> k & 1u) && rot < myrot) {
                    myrot = rot;
                    lo = ((unsigned)plane << 13) | (unsigned)spoke;
                    hi = ((unsigned)rot << 16) | ((dzone >> (4 * k) & 15u) << 11) | (unsigned)ring;
                }
            }
            const int wmin = wave_min_i32(myrot);
            const int fl = __ffsll((long long)__ballot(myrot == wmin)) - 1;
            const unsigned wl = __builtin_amdgcn_readlane(lo, fl);
            const unsigned wh = __builtin_amdgcn_readlane(hi, fl);
            if (lane == 0) atomicMin(&s.ref[pass & 1], ((unsigned long long)wh << 32) | wl);
        }
        __syncthreads();
        // flush: the window's cells over all threads in storage order, one
        // global atomic per non-zero cell; the (ring, plane, spoke) offsets of
        // cell e advanced by the block size with carries instead of divided
        // out per cell; window spokes q0 + dq lie in [-1, na]
        if (tid < ncell) {
            const int t1 = div_small(TB, NQ), sq = TB - t1 * NQ;
            const int sr = div_small(t1, NP), spl = t1 - sr * NP;
            const int u1 = div_small(tid, NQ);
            int dq = tid - u1 * NQ, dr = div_small(u1, NP);
            int dp = u1 - dr * NP;
            for (int e = tid; e < ncell; e += TB) {
                const long long tv = s.tile[e];
                if (tv != 0) {
                    s.tile[e] = 0;
                    int sp = q0 + dq;
                    sp = sp >= a.na ? sp - a.na : sp < 0 ? sp + a.na : sp;
                    atomicAdd((unsigned long long *)&a.mfx[ref.zone - 1][((r0 + dr) * a.ngz + (p0 + dp)) * a.na + sp],
                              (unsigned long long)tv);
                }
                dq += sq;
                const int c1 = dq >= NQ ? 1 : 0;
                dq -= c1 * NQ;
                dp += spl + c1;
                const int c2 = dp >= NP ? 1 : 0;
                dp -= c2 * NP;
                dr += sr + c2;
            }
        }
        const unsigned long long kref = s.ref[pass & 1];
        if (kref == ~0ull || pass + 1 >= P3_PASSES) break;   // uniform
        const unsigned rh = (unsigned)(kref >> 32), rl = (unsigned)kref;
        ref.zone = (int)((rh >> 11) & 0xF);
        ref.ring = (int)(rh & 0x7FF);
        ref.plane = (int)(rl >> 13);
        ref.spoke = (int)(rl & 0x1FFF);
    }
    direct |= pend;
    if (any_lane(direct != 0)) {
#pragma unroll
        for (int k = 0; k < PPT; k++) {
            if (!(direct >> k & 1u)) continue;
            const int z = (int)(dzone >> (4 * k) & 15u);
            int ring, plane, spoke;
            loc3<R, J>(pos[k], a, ring, plane, spoke);
            R w[NW];
            weights3(pos[k], ring, plane, w);
            long long v[NW];
            quant_n<R, NW>(w, a.qbits, true, v);
            atomicMin(&s.jr[z - 1], ring);
            atomicMax(&s.kr[z - 1], ring);
            int ic[NW];
            cornersJ<J>(cell_index(a, ring, plane, spoke), spoke, a.na, a.ngz, ic);
#pragma unroll
            for (int q = 0; q < NW; q++)
                if (v[q] != 0) deposit_global(a.mfx, a.nz, a.mesh, z, ic[q], v[q]);
        }
    }
}

// jrad/krad from the block's central rings: 1-based rings j+1..j+2 about a
// central ring j (massgn.f:146-149), j..j+2 for jmass 3 (massgn.f:176-179)
template <int TILE>
__device__ __forceinline__ void deposit3_ranges(const Deposit3Lds<TILE> &s, int nz, int nr, int lo,
                                                int *jrad, int *krad, int rstride) {
    const int tid = threadIdx.x;
    if (tid < nz && s.kr[tid] >= 0) {
        const int k = s.kr[tid] + 2;
        widen_range(jrad, krad, rstride, blockIdx.x, tid + 1, s.jr[tid] + 1 - lo, k < nr ? k : nr);
    }
}

template <typename R, int J, int PPT>
__global__ __launch_bounds__((P3Shape<R, J, PPT>::block), (P3Shape<R, J, PPT>::waves)) void p3_massgn_kernel(P3Args<R> a) {
    constexpr int TB = P3Shape<R, J, PPT>::block, TILE = P3Shape<R, J, PPT>::tile;
    __shared__ Deposit3Lds<TILE> s_dep;
    __shared__ P3Ref s_ref0;
    const int tid = threadIdx.x;
    const long long base = (long long)blockIdx.x * (TB * PPT);
    const int nblk = (int)min((long long)(TB * PPT), a.n - base);
    P3Pos<R> pos[PPT];
    unsigned dzone = 0;
#pragma unroll
    for (int k = 0; k < PPT; k++) {
        const int j = k * TB + tid;
        pos[k].u = pos[k].t = pos[k].zz = (R)0;
        if (j < nblk) {
            const int z = a.zone[base + j];
            const typename Vec4<R>::T p = a.rec[2 * (base + j)];
            R u, t;
            ut3(p.x, p.y, a, u, t);
            p3_set_ut(a, base + j, u, t);
            if (z >= 1 && z <= a.nz) {
                pos[k] = pos3(u, t, p.z, a, a.nsect > 1);
                dzone |= (unsigned)z << (4 * k);
            }
        }
        if (j == nblk >> 1) {
            s_ref0.zone = max(1, (int)(dzone >> (4 * k) & 15u));
            loc3<R, J>(pos[k], a, s_ref0.ring, s_ref0.plane, s_ref0.spoke);
        }
    }
    deposit3_init<TB>(s_dep);
    __syncthreads();
    const P3Ref ref = s_ref0;
    deposit3_block<R, J, PPT, TB>(a, s_dep, pos, dzone, ref);
    __syncthreads();
    deposit3_ranges(s_dep, a.nz, a.nr, J == 3 ? 1 : 0, a.jrad, a.krad, a.rstride);
}

template <typename R, int J, int PPT>
__global__ __launch_bounds__((P3Shape<R, J, PPT>::block), (P3Shape<R, J, PPT>::waves)) void p3_push_kernel(P3Args<R> a) {
    typedef typename Vec4<R>::T R4;
    constexpr int TB = P3Shape<R, J, PPT>::block, TILE = P3Shape<R, J, PPT>::tile;
    __shared__ Deposit3Lds<TILE> s_dep;
    __shared__ int s_dn, s_np;
    __shared__ double s_tab[UtTab<R>::n];
    const int tid = threadIdx.x, nz = a.nz, nlists = nz + 1;
    const long long base = (long long)blockIdx.x * (TB * PPT);
    const int nblk = (int)min((long long)(TB * PPT), a.n - base);
    R4 *const rec = a.rec + 2 * base;
    uint8_t *const zb = a.zone + base;
    // on a full step every list moves: no wait for the zones before the load
    const bool full = a.mzone == nz;
    int zin[PPT];
    R4 st[PPT], sv[PPT];   // (x, y, z, vx), (vy, vz, u, t)
#pragma unroll
    for (int k = 0; k < PPT; k++) zin[k] = zb[min(k * TB + tid, nblk - 1)];
    const int zmid = zb[nblk >> 1];
    const R4 m0 = rec[2 * (nblk >> 1)], m1 = rec[2 * (nblk >> 1) + 1];
    auto load_state = [&]() {
#pragma unroll
        for (int k = 0; k < PPT; k++) {
            const int j = min(k * TB + tid, nblk - 1);
            st[k] = rec[2 * j];
            sv[k] = rec[2 * j + 1];
        }
    };
    if (full) load_state();
    for (int j = tid; j < UtTab<R>::n; j += TB) s_tab[j] = ut_tab_entry<R>(j);
    deposit3_init<TB>(s_dep);
    if (tid == 0) s_dn = s_np = 0;
    unsigned mv = 0;   // bit k: particle k moves
    if (!full)
#pragma unroll
        for (int k = 0; k < PPT; k++)
            if (k * TB + tid < nblk && zin[k] <= a.mzone) mv |= 1u << k;
    if (!__syncthreads_or(full ? 1 : (int)mv)) return;
    if (full) {
#pragma unroll
        for (int k = 0; k < PPT; k++)
            if (k * TB + tid < nblk && (zin[k] != nlists || a.offanal)) mv |= 1u << k;
    } else {
        load_state();
    }
    P3Ref ref;
    ref.zone = min(max(zmid, 1), nz);
    loc3<R, J>(pos3(m1.z, m1.w, m0.z, a, a.nsect > 1), a, ref.ring, ref.plane, ref.spoke);
    ref.ring = max(ref.ring, 0);
    ref.spoke = min(max(ref.spoke, 0), a.na);
    // the new states take the old ones' registers and are stored after every
    // load has been used
    P3Pos<R> pos[PPT];
    unsigned dzone = 0, zch = 0;
    int np = 0, nplus = 0, nminus = 0;
#pragma unroll
    for (int k = 0; k < PPT; k++) {
        bool plus = false, minus = false;
        const bool move = mv >> k & 1u;
        np += __popcll(__ballot(move));
        pos[k].u = pos[k].t = pos[k].zz = (R)0;
        if (move) {
            const int z0 = zin[k];
            const bool offlist = z0 == nlists;
            R o[3] = {st[k].x, st[k].y, st[k].z};
            R ov[3] = {st[k].w, sv[k].x, sv[k].y};
            R acc[3], nv[3], nx[3];
            getacc3<R, J>(a, o[0], o[1], o[2], sv[k].z, sv[k].w, z0, acc);
            // stpgrp
#pragma unroll
            for (int d = 0; d < 3; d++) {
                nv[d] = ov[d] + acc[d];
                nx[d] = o[d] + nv[d];
            }
            int znew = z0;
            R rnew = sqrt_rn(nx[0] * nx[0] + nx[1] * nx[1]);
            const R az = nx[2] < (R)0 ? -nx[2] : nx[2];
            const bool off = (az > a.zm) || (rnew > a.rgrid);
            if (!offlist) {
                if (off) {
                    znew = nlists;
                    plus = true;
                    if (a.offanal && z0 < nz) {
                        const R tfac = tsfac3(a, nz) / tsfac3(a, z0);
#pragma unroll
                        for (int d = 0; d < 3; d++) chstep1(tfac, o[d], ov[d], acc[d], nx[d], nv[d]);
                        rnew = sqrt(nx[0] * nx[0] + nx[1] * nx[1]);
                    }
                }
            } else if (!off) {
                minus = true;
                znew = nz;
            }
            // rezgrp
            if (a.mzone > 1 && !offlist && znew <= a.mzone) {
                int kz = zoneno3(a, nx[0], nx[1], nx[2]);
                if (kz > a.mzone) kz = a.mzone;
                if (kz > znew) kz = zoneno3(a, o[0], o[1], o[2]);
                if (kz != znew) {
                    const R tfac = tsfac3(a, kz) / tsfac3(a, znew);
#pragma unroll
                    for (int d = 0; d < 3; d++) chstep1(tfac, o[d], ov[d], acc[d], nx[d], nv[d]);
                    rnew = sqrt(nx[0] * nx[0] + nx[1] * nx[1]);
                    znew = kz;
                }
            }
            R un, tn;
            ut3_push(nx[0], nx[1], rnew, a, un, tn, s_tab);
            st[k] = mk4(nx[0], nx[1], nx[2], nv[0]);
            sv[k] = mk4(nv[1], nv[2], un, tn);
            if (znew != z0) zch |= 1u << k;
            zin[k] = znew;
            if (znew >= 1 && znew <= nz) {
                pos[k] = pos3(un, tn, nx[2], a, a.nsect > 1);
                dzone |= (unsigned)znew << (4 * k);
            }
        }
        nplus += __popcll(__ballot(plus));
        nminus += __popcll(__ballot(minus));
    }
#pragma unroll
    for (int k = 0; k < PPT; k++) {
        const int j = k * TB + tid;
        if (mv >> k & 1u) {
            rec[2 * j] = st[k];
            rec[2 * j + 1] = sv[k];
            if (zch >> k & 1u) zb[j] = (uint8_t)zin[k];
        }
    }
    // block sums of the off-grid change and the pushes
    if ((tid & 63) == 0) {
        if (nplus != nminus) atomicAdd(&s_dn, nplus - nminus);
        if (np) atomicAdd(&s_np, np);
    }
    deposit3_block<R, J, PPT, TB>(a, s_dep, pos, dzone, ref);
    __syncthreads();
    deposit3_ranges(s_dep, nz, a.nr, J == 3 ? 1 : 0, a.jrad, a.krad, a.rstride);
    if (tid == 0) {
        if (s_dn) atomicAdd((unsigned long long *)&a.counters[0], (unsigned long long)(long long)s_dn);
        count_pushes(a.pushes, blockIdx.x, s_np);
    }
}

// (u, t) of every particle's position (after a load)
template <typename R>
__global__ __launch_bounds__(P3_PBLOCK) void p3_ut_kernel(P3Args<R> a) {
    const long long i = (long long)blockIdx.x * P3_PBLOCK + threadIdx.x;
    if (i >= a.n) return;
    const typename Vec4<R>::T p = a.rec[2 * i];
    R u, t;
    ut3(p.x, p.y, a, u, t);
    p3_set_ut(a, i, u, t);
}

template <typename R, int J>
__global__ __launch_bounds__(P3_PBLOCK) void p3_tmcent_kernel(P3Args<R> a) {
    const long long i = (long long)blockIdx.x * P3_PBLOCK + threadIdx.x;
    if (i >= a.n) return;
    typename Vec4<R>::T p = a.rec[2 * i];
    typename Vec4<R>::T q = a.rec[2 * i + 1];   // (vy, vz, u, t)
    R acc[3];
    getacc3<R, J>(a, p.x, p.y, p.z, q.z, q.w, a.zone[i], acc);
    p.w = p.w - a.fac * acc[0];
    q.x = q.x - a.fac * acc[1];
    q.y = q.y - a.fac * acc[2];
    a.rec[2 * i] = p;
    a.rec[2 * i + 1] = q;
}

template <typename R, int J>
__global__ __launch_bounds__(P3_PBLOCK) void p3_gather_kernel(P3GatherArgs<R> b) {
    typedef typename Vec4<R>::T R4;
    constexpr int NW = P3NW<J>::v;
    const long long i = (long long)blockIdx.x * P3_PBLOCK + threadIdx.x;
    if (i >= b.n) return;
    R w[NW];
    R u, t;
    ut3(b.x[i], b.y[i], b.g, u, t);
    int rg, pl, sp;
    const int c = cellJ<R, J>(u, t, b.z[i], b.g, b.fold != 0, w, rg, pl, sp);
    if (b.cell) b.cell[i] = c;
    if (b.wt)
        for (int q = 0; q < NW; q++) b.wt[NW * i + q] = w[q];
    if (b.acc) {
        int ic[NW];
        cornersJ<J>(c, sp, b.g.na, b.g.ngz, ic);
        R s[3] = {(R)0, (R)0, (R)0};
        for (int q = 0; q < NW; q++) {
            R4 f = (ic[q] >= 0 && ic[q] < b.g.mesh) ? b.fld[ic[q]] : mk4((R)0, (R)0, (R)0, (R)0);
            s[0] = s[0] + f.x * w[q];
            s[1] = s[1] + f.y * w[q];
            s[2] = s[2] + f.z * w[q];
        }
        for (int d = 0; d < 3; d++) b.acc[3 * i + d] = s[d];
    }
}

// icheck's global integrals for the 3-D grid (SRC/lib15/icheck.f:24-70):
// per-block FP64 sums of 11 quantities in a fixed order (int_split's
// particles per thread, as on the p2d grid), then a block per quantity adds the block
// sums in a fixed order.  [0] count, [1..3] position, [4..6] velocity per
// zone-1 step ((v + a/2)/tfac when centred), [7] v^2, [8] Lz, [9] the grid
// potential interpolated with the particle's own weights (grid particles),
// [10] the fixed potential of the spherical radius.
constexpr int NINT3 = 11;

template <typename R, int J>
__global__ __launch_bounds__(P3_INT_BLOCK) void p3_integrals_kernel(P3Args<R> a, int per, int with_pot,
                                                                 const double4 *fp_c, int nfp,
                                                                 double fp_dr, int centred,
                                                                 double *part) {
    typedef typename Vec4<R>::T R4;
    __shared__ double red[P3_INT_BLOCK / 64][NINT3];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    double v[NINT3];
#pragma unroll
    for (int q = 0; q < NINT3; q++) v[q] = 0.0;
    for (int k = 0; k < per; k++) {
        const long long i = ((long long)blockIdx.x * per + k) * P3_INT_BLOCK + tid;
        if (i >= a.n) break;
        const int z = a.zone[i];
        if (z >= 1) {
            const R4 p = a.rec[2 * i];
            const R4 q4 = a.rec[2 * i + 1];
            const typename Vec2<R>::T q2 = mk2(q4.x, q4.y);
            const typename Vec2<R>::T ut = mk2(q4.z, q4.w);
            R vx = p.w, vy = q2.x, vz = q2.y;
            if (centred) {
                R acc[3];
                getacc3<R, J>(a, p.x, p.y, p.z, ut.x, ut.y, z, acc);
                vx = vx + (R)0.5 * acc[0];
                vy = vy + (R)0.5 * acc[1];
                vz = vz + (R)0.5 * acc[2];
            }
            const int zs = z <= a.nz ? z : a.nz;
            const double sf = 1.0 / (double)a.nstep[zs - 1];
            const double x = p.x, y = p.y, zz = p.z;
            const double ux = vx * sf, uy = vy * sf, uz = vz * sf;
            v[0] += 1.0;
            v[1] += x;
            v[2] += y;
            v[3] += zz;
            v[4] += ux;
            v[5] += uy;
            v[6] += uz;
            v[7] += ux * ux + uy * uy + uz * uz;
            v[8] += x * uy - y * ux;
            if (with_pot && z <= a.nz) {
                constexpr int NW = P3NW<J>::v;
                R w[NW];
                int ic[NW];
                int rg, pl, sp;
                const int c = cellJ<R, J>(ut.x, ut.y, p.z, a, false, w, rg, pl, sp);
                cornersJ<J>(c, sp, a.na, a.ngz, ic);
                double ph = 0.0;
                for (int k = 0; k < NW; k++)
                    if (ic[k] >= 0 && ic[k] < a.mesh) ph += (double)w[k] * (double)a.fld[ic[k]].w;
                v[9] += ph;
            }
            if (nfp > 0)
                v[10] += fixforce(sqrt(x * x + y * y + zz * zz), nfp, 1.0 / fp_dr, fp_c);
        }
    }
#pragma unroll
    for (int q = 0; q < NINT3; q++) {
        const double t = wave_sum_dpp(v[q]);
        if (lane == 0) red[wave][q] = t;
    }
    __syncthreads();
    if (tid < NINT3) {
        double t = 0.0;
        for (int w = 0; w < P3_INT_BLOCK / 64; w++) t += red[w][tid];
        part[(long long)tid * gridDim.x + blockIdx.x] = t;
    }
}

__global__ __launch_bounds__(P3_INT_BLOCK) void p3_integrals_sum_kernel(const double *part, int nb,
                                                                     double *out) {
    __shared__ double red[P3_INT_BLOCK / 64];
    const int tid = threadIdx.x, q = blockIdx.x;
    double t = 0.0;
    for (int b = tid; b < nb; b += P3_INT_BLOCK) t += part[(long long)q * nb + b];
    t = wave_sum_dpp(t);
    if ((tid & 63) == 0) red[tid >> 6] = t;
    __syncthreads();
    if (tid == 0) {
        double s = 0.0;
        for (int w = 0; w < P3_INT_BLOCK / 64; w++) s += red[w];
        out[q] = s;
    }
}

// Sort keys: the particle's cell shifted right by kshift (kmax for the
// off-grid list, which sorts last), with the identity permutation.
template <typename R, int J>
__global__ __launch_bounds__(P3_PBLOCK) void p3_key_kernel(P3Args<R> a, int kshift,
                                                          unsigned kmax, unsigned *key,
                                                          unsigned *perm) {
    const long long i = (long long)blockIdx.x * P3_PBLOCK + threadIdx.x;
    if (i >= a.n) return;
    const int z = a.zone[i];
    unsigned k = kmax;
    if (z >= 1 && z <= a.nz) {
        const typename Vec4<R>::T p = a.rec[2 * i];
        const typename Vec4<R>::T q = a.rec[2 * i + 1];
        const typename Vec2<R>::T ut = mk2(q.z, q.w);
        int ring, plane, spoke;
        loc3<R, J>(pos3(ut.x, ut.y, p.z, a, false), a, ring, plane, spoke);
        k = (unsigned)(cell_index(a, ring, plane, spoke) >> kshift);
    }
    key[i] = k;
    perm[i] = (unsigned)i;
}

template <typename R>
__global__ __launch_bounds__(P3_PBLOCK) void p3_permute_kernel(P3PermArgs<R> p) {
    // (all loads before the first store: a load waits for the stores before it.
    // Store by store 2e7 particles took 797 us, so 614.)
    typedef typename Vec4<R>::T R4;
    const long long i = (long long)blockIdx.x * P3_PBLOCK + threadIdx.x;
    if (i >= p.n) return;
    const long long j = p.perm[i];
    const R4 r0 = p.rec_in[2 * j], r1 = p.rec_in[2 * j + 1];
    const uint8_t z = p.zin[j];
    const unsigned id = p.iin[j];
    p.rec_out[2 * i] = r0;
    p.rec_out[2 * i + 1] = r1;
    p.zout[i] = z;
    p.iout[i] = id;
}

// load: planar host arrays staged on the device (x, y, z, vx in s4 and vy, vz
// in s2, n values each, one after another) -> particle records ((u, t) set
// by p3_ut_kernel afterwards); ids = load order
template <typename R>
__global__ __launch_bounds__(P3_PBLOCK) void p3_interleave_kernel(const R *__restrict__ s4,
                                                                  const R *__restrict__ s2,
                                                                  typename Vec4<R>::T *__restrict__ rec,
                                                                  unsigned *__restrict__ id,
                                                                  long long n) {
    const long long i = (long long)blockIdx.x * P3_PBLOCK + threadIdx.x;
    if (i >= n) return;
    typename Vec4<R>::T a;
    a.x = s4[i];
    a.y = s4[n + i];
    a.z = s4[2 * n + i];
    a.w = s4[3 * n + i];
    rec[2 * i] = a;
    rec[2 * i + 1] = mk4(s2[i], s2[n + i], (R)0, (R)0);
    id[i] = (unsigned)i;
}

// Unload: interleaved storage -> planar arrays in load order, zones widened,
// from the records' places as on the p2d grid: 2e7 particles 3930 us when
// each wrote its seven values where they belong, 790 (and 280 for the places) so;
// 2e4 5.0 us and 2.6 + 2.5.
template <typename R, bool GATHER>
__global__ __launch_bounds__(P3_PBLOCK) void p3_deinterleave_kernel(
    const typename Vec4<R>::T *__restrict__ rec, const uint8_t *__restrict__ zone,
    const unsigned *__restrict__ ord, R *__restrict__ d4, R *__restrict__ d2,
    int *__restrict__ iz, long long n) {
    const long long t = (long long)blockIdx.x * P3_PBLOCK + threadIdx.x;
    if (t >= n) return;
    const long long o = ord[t], i = GATHER ? o : t, p = GATHER ? t : o;
    const typename Vec4<R>::T a = rec[2 * i];
    const typename Vec4<R>::T b = rec[2 * i + 1];
    const int z = zone[i];
    d4[p] = a.x;
    d4[n + p] = a.y;
    d4[2 * n + p] = a.z;
    d4[3 * n + p] = a.w;
    d2[p] = b.x;
    d2[n + p] = b.y;
    iz[p] = z;
}

// ---- field solve ------------------------------------------------------------------

// Solve shapes.  All transforms are direct sums in the order of one sum per
// output (j, p or k ascending), whatever the shape, so that results do not
// depend on it; what the shapes share is the twiddle, read from LDS once for
// several planes or columns.  200 rings x 125 planes x 256 spokes, 9 harmonics:
//   analysis  `planes` planes a wavefront, cosine and sine sums of a harmonic
//             together (sums once per component before, each formed twice):
//             100 -> 50 us; 4 planes 56 (registers: 4 wavefronts a SIMD instead
//             of 7), 1 plane 65.  Floor: 77 MB, 15 us; conversions and the
//             wavefront sums are what is left.
//   synthesis `splanes` planes a block: 101 -> 48 us; 2 planes 48, 8 planes 52.
//             It stores the three force components only (57 us when it reads
//             the potential to store whole vectors): 77 MB.
template <typename R> struct P3Solve {
    static constexpr int planes = sizeof(R) == 4 ? 2 : 1;
    static constexpr int splanes = sizeof(R) == 4 ? 4 : 2;
};

// combined, scaled mass of a cell (zoncmb + scaled)
template <typename R>
__device__ __forceinline__ R p3_cell_mass(const P3SolveArgs<R> &a, size_t idx) {
    double acc = (double)a.mfx[0][idx] * a.q;
    for (int z = 2; z <= a.nz; z++) {
        if (a.use_new[z - 1]) acc = acc + a.fnew[z - 1] * ((double)a.mfx[z - 1][idx] * a.q);
        if (a.use_old[z - 1]) acc = acc + a.fold[z - 1] * ((double)a.moz[z - 1][idx] * a.q);
    }
    return (R)(acc * a.pmass);
}

// grid (planes / (4 wavefronts x PL), nr, 1): a wavefront takes PL planes of a
// ring and, HB at a time, all harmonics.  SPLIT: gridDim.z passes of HB harmonics,
// a wavefront takes one of them, and one more wavefront a block looks the ranges up
// while the others load their first masses (24 x 64 x 16: 5.1 -> 4.6 us,
// 45 x 90 x 31: 5.5 -> 5.1)
template <typename R, int PL, int HB, bool SPLIT>
__global__ __launch_bounds__(P3_BLOCK + 64) void p3_analyse_kernel(P3SolveArgs<R> a) {
    constexpr int WAVES = P3_BLOCK / 64, LOOK = SPLIT ? WAVES : 0;   // the look-up's wavefront
    typedef typename Vec2<R>::T R2;
    extern __shared__ unsigned char p3_lds[];
    R2 *tws = (R2 *)p3_lds;                   // [na]
    __shared__ int s_rng[4], s_ok, s_jr[GH_MAXZ], s_kr[GH_MAXZ];
    const int tid = threadIdx.x, na = a.na, nm = a.nm, lane = tid & 63;
    const int ir = blockIdx.y + 1;
    const int wave = tid >> 6, plane0 = wave < WAVES ? (blockIdx.x * WAVES + wave) * PL : a.ngz;
    size_t row[PL];
#pragma unroll
    for (int p = 0; p < PL; p++)
        row[p] = ((size_t)(ir - 1) * a.ngz + min(plane0 + p, a.ngz - 1)) * na;
    R ahead[PL];
    if (SPLIT && plane0 < a.ngz && lane < na)
#pragma unroll
        for (int p = 0; p < PL; p++) ahead[p] = p3_cell_mass(a, row[p] + lane);
    if (wave == LOOK) combine_ranges(a.jrad, a.krad, a.rstride, a.nz, s_jr, s_kr);
    if (tid == 64 * LOOK) {
        int kr[GH_MAXZ], rg[4] = {0, 0, 0, 0};
        const bool ok = solve_ranges(s_jr, s_kr, a.nz, a.nr, a.mzone, a.lpot,
                                     a.explicit_zones, a.jzone, a.kzone, kr, rg);
        s_ok = ok;
        for (int q = 0; q < 4; q++) s_rng[q] = rg[q];
        if (blockIdx.x == 0 && ir == 1 && blockIdx.z == 0) {
            for (int q = 0; q < 4; q++) a.ranges[q] = ok ? rg[q] : -1;
            if (ok)
                for (int z = 1; z < a.nz; z++) a.krad[z] = kr[z];
        }
    }
    if (wave < WAVES)
        for (int j = tid; j < na; j += P3_BLOCK) tws[j] = mk2(a.tw[2 * j], a.tw[2 * j + 1]);
    __syncthreads();
    if (plane0 >= a.ngz) return;
    const bool active = s_ok && ir >= s_rng[0] && ir <= s_rng[1];
    // the slot of the i-th harmonic: two slots each, one for m = 0 (and the last
    // one for m = na / 2)
    const int zero = nm > 0 && a.slot_m[0] == 0;
    auto slot = [&](int i) { return zero && i ? 2 * i - 1 : 2 * i; };
    int i0 = (int)blockIdx.z * HB;
    bool first = true;
    do {
        // the harmonics i0 .. i0 + HB - 1
        int k[HB], step[HB];
#pragma unroll
        for (int h = 0; h < HB; h++) {
            const int s = slot(i0 + h), m = s < nm ? a.slot_m[s] : 0;
            // (m < P3_MAX_NA: 32 bits hold the products)
            k[h] = (m * lane) % na;
            step[h] = (m * 64) % na;
        }
        R sa[HB][PL], sb[HB][PL];
#pragma unroll
        for (int h = 0; h < HB; h++)
#pragma unroll
            for (int p = 0; p < PL; p++) sa[h][p] = sb[h][p] = (R)0;
        for (int j = lane; j < na; j += 64) {
            R rv[PL];
#pragma unroll
            for (int p = 0; p < PL; p++)
                rv[p] = SPLIT && j == lane ? ahead[p]
                        : first            ? p3_cell_mass(a, row[p] + j)
                                           : a.rho[row[p] + j];
            if (first && blockIdx.z == 0)
#pragma unroll
                for (int p = 0; p < PL; p++)
                    if (plane0 + p < a.ngz) a.rho[row[p] + j] = rv[p];
            if (!active) continue;
#pragma unroll
            for (int h = 0; h < HB; h++) {
                const R2 w = tws[k[h]];
#pragma unroll
                for (int p = 0; p < PL; p++) {
                    sa[h][p] += rv[p] * w.x;
                    sb[h][p] += rv[p] * w.y;
                }
                k[h] += step[h];
                if (k[h] >= na) k[h] -= na;
            }
        }
        if (!active) return;
#pragma unroll
        for (int h = 0; h < HB; h++) {
            const int s = slot(i0 + h);
            const bool pair = s + 1 < nm && a.slot_p[s + 1];
            R va = 0, vb = 0;
#pragma unroll
            for (int p = 0; p < PL; p++) {
                const R ta = p3_wave_sum(sa[h][p]), tb = p3_wave_sum(sb[h][p]);
                if (lane == p) {
                    va = ta;
                    vb = -tb;
                }
            }
            R *out = a.A + ((size_t)(ir - 1) * nm + s) * a.ngz + plane0 + lane;
            if (s < nm && lane < PL && plane0 + lane < a.ngz) {
                out[0] = va;
                if (pair) out[a.ngz] = vb;
            }
        }
        first = false;
        i0 += HB;
    } while (!SPLIT && slot(i0) < nm);
}

// The vertical twiddles (cos, sin of 2 pi k / P) in LDS with one pad entry
// after every 256 bytes: the transforms read them at index p k mod P across
// consecutive k (or q), a stride that puts many lanes on one bank when it is
// a multiple of a large power of two; the pad spreads those over the banks.
template <typename R> constexpr int tz_shift() { return sizeof(R) == 4 ? 5 : 4; }
template <typename R> __host__ __device__ constexpr size_t tz_words(size_t P) {
    return 2 * (P + (P >> tz_shift<R>()) + 1);
}
template <typename R> __device__ __forceinline__ int tz_at(int idx) {
    return idx + (idx >> tz_shift<R>());
}
template <typename R>
__device__ __forceinline__ void tz_stage(const R *twz, int P, typename Vec2<R>::T *tz) {
    for (int e = threadIdx.x; e < P; e += blockDim.x) tz[tz_at<R>(e)] = mk2(twz[2 * e], twz[2 * e + 1]);
}

// The ring of a vertical transform's block: consecutive blocks go to the eight
// XCDs in turn, and neighbouring rings, which share the lines of the
// [column][k][ring] arrays, to one of them.
__device__ __forceinline__ int p3_ring(int nr) {
    const int b = blockIdx.x, x = b & 7, q = nr >> 3, r = nr & 7;
    return x * q + min(x, r) + (b >> 3);
}

// grid (nr, columns / CB): the doubled vertical transform of some component
// columns of one ring
template <typename R, int CB>
__global__ __launch_bounds__(P3_BLOCK) void p3_zfwd_kernel(P3SolveArgs<R> a) {
    extern __shared__ unsigned char p3_lds[];
    const int ngz = a.ngz, P = 2 * ngz, nm = a.nm;
    const int s0 = blockIdx.y * CB, ncol = min(CB, nm - s0);
    typedef typename Vec2<R>::T R2;
    R2 *tz = (R2 *)p3_lds;                    // [P]
    R *col = (R *)p3_lds + tz_words<R>(P);             // [ngz][CB]
    const int ir = p3_ring(a.nr) + 1, tid = threadIdx.x;
    const int jrs = a.ranges[0], krs = a.ranges[1];
    if (jrs < 1 || ir < jrs || ir > krs) return;
    const R *src = a.A + ((size_t)(ir - 1) * nm + s0) * ngz;
    for (int e = tid; e < CB * ngz; e += blockDim.x) {
        const int c = e / ngz, p = e - c * ngz;
        col[p * CB + c] = c < ncol ? src[e] : (R)0;
    }
    tz_stage<R>(a.twz, P, tz);
    __syncthreads();
    // [column][k][ring]: the contraction reads and writes rings
    R *dst = a.M + (size_t)s0 * P * a.nr + (ir - 1);
    const size_t nr = a.nr;
    for (int k = tid; k <= ngz; k += blockDim.x) {
        R sa[CB], sb[CB];
#pragma unroll
        for (int c = 0; c < CB; c++) sa[c] = sb[c] = (R)0;
        int idx = 0;
#pragma unroll 4
        for (int p = 0; p < ngz; p++) {
            const R2 w = tz[tz_at<R>(idx)];
#pragma unroll
            for (int c = 0; c < CB; c++) {
                const R v = col[p * CB + c];
                sa[c] += v * w.x;
                sb[c] += v * w.y;
            }
            idx += k;
            if (idx >= P) idx -= P;
        }
#pragma unroll
        for (int c = 0; c < CB; c++) {
            if (c >= ncol) break;
            R *h = dst + (size_t)c * P * nr;
            if (k == 0) h[0] = sa[c];
            else if (k == ngz) h[(P - 1) * nr] = sa[c];
            else {
                h[(2 * k - 1) * nr] = sa[c];
                h[2 * k * nr] = -sb[c];
            }
        }
    }
}

// grid (ng, ngz + 1, ntypes): block (m, k_z, type) applies one Green's matrix.
// Reading the tables bounds it: three types of 9 x 126 matrices of 200 x 200,
// 544 MB, in 128 us (4.2 TB/s; a copy reaches 5.3).  With M and W by ring
// first the 4-byte accesses of the source rings and results, a line each, made
// it 154.
template <typename R>
__global__ __launch_bounds__(P3_BLOCK) void p3_conv_kernel(P3SolveArgs<R> a) {
    typedef typename Vec4<R>::T R4;
    __shared__ R4 rhs[P3_MAX_NR];
    const int im = blockIdx.x + 1, iz = blockIdx.y + 1, type = blockIdx.z;
    const int ng = a.ng, ngz = a.ngz, mmax = a.mmax, nm = a.nm, nr = a.nr;
    if (type == 1 && (im < 2 || im > min(ng, mmax - 1))) return;
    if (type == 2 && (iz < 2 || iz > ngz)) return;
    if (a.lg[im - 1]) return;
    const int jrs = a.ranges[0], krs = a.ranges[1], jrf = a.ranges[2], krf = a.ranges[3];
    if (jrs < 1) return;
    const int P = 2 * ngz;
    const bool nvskip = iz > 1 && iz <= ngz;
    const bool naskip = im > 1 && im < mmax;
    const int p = max(1, 2 * (iz - 1)) - 1;
    const int sc = a.slot_of[im - 1], ss = sc + 1;
    int src[4], dst[4];
    R sgn[4];
    bool val[4];
    dst[0] = sc * P + p; dst[1] = sc * P + p + 1; dst[2] = ss * P + p; dst[3] = ss * P + p + 1;
    if (type == 0 || type == 3) {
        for (int q = 0; q < 4; q++) { src[q] = dst[q]; sgn[q] = (R)1; }
        val[0] = true; val[1] = nvskip; val[2] = naskip; val[3] = naskip && nvskip;
    } else if (type == 1) {
        src[0] = ss * P + p; src[1] = ss * P + p + 1; src[2] = sc * P + p; src[3] = sc * P + p + 1;
        sgn[0] = sgn[1] = (R)1; sgn[2] = sgn[3] = (R)-1;
        val[0] = val[2] = true; val[1] = val[3] = nvskip;
    } else {
        src[0] = sc * P + p + 1; src[1] = sc * P + p; src[2] = ss * P + p + 1; src[3] = ss * P + p;
        sgn[0] = sgn[2] = (R)1; sgn[1] = sgn[3] = (R)-1;
        val[0] = val[1] = true; val[2] = val[3] = naskip;
    }
    const int nrs = krs - jrs + 1;
    for (int e = threadIdx.x; e < 4 * nrs; e += P3_BLOCK) {
        const int q = e / nrs, is = jrs + (e - q * nrs);
        reinterpret_cast<R *>(rhs)[4 * (is - 1) + q] = val[q] ? sgn[q] * a.M[(size_t)src[q] * nr + (is - 1)] : (R)0;
    }
    __syncthreads();
    const R *Gm = a.G + ((((size_t)type * (ngz + 1) + (iz - 1)) * ng + (im - 1)) * nr) * nr;
    for (int ir = jrf + threadIdx.x; ir <= krf; ir += P3_BLOCK) {
        R s0 = 0, s1 = 0, s2 = 0, s3 = 0;
        const R *g = Gm + (ir - 1);
#pragma unroll 8
        for (int is = jrs; is <= krs; is++) {
            const R gv = g[(size_t)(is - 1) * nr];
            const R4 r = rhs[is - 1];
            s0 += gv * r.x;
            s1 += gv * r.y;
            s2 += gv * r.z;
            s3 += gv * r.w;
        }
        R *w = a.W + (size_t)type * nm * P * nr + (ir - 1);
        if (val[0]) w[(size_t)dst[0] * nr] = s0;
        if (val[1]) w[(size_t)dst[1] * nr] = s1;
        if (val[2]) w[(size_t)dst[2] * nr] = s2;
        if (val[3]) w[(size_t)dst[3] * nr] = s3;
    }
}

// grid (nr, ntypes, columns / CB): inverse vertical transform of
// some columns of one ring
template <typename R, int CB>
__global__ __launch_bounds__(P3_BLOCK) void p3_zinv_kernel(P3SolveArgs<R> a) {
    extern __shared__ unsigned char p3_lds[];
    const int ngz = a.ngz, P = 2 * ngz, nm = a.nm;
    const int s0 = blockIdx.z * CB, ncol = min(CB, nm - s0);
    typedef typename Vec2<R>::T R2;
    R2 *tz = (R2 *)p3_lds;                    // [P]
    R *h = (R *)p3_lds + tz_words<R>(P);               // [P][CB]
    const int ir = p3_ring(a.nr) + 1, type = blockIdx.y, tid = threadIdx.x;
    const int jrs = a.ranges[0], jrf = a.ranges[2], krf = a.ranges[3];
    if (jrs < 1 || ir < jrf || ir > krf) return;
    const R *src = a.W + ((size_t)type * nm + s0) * P * a.nr + (ir - 1);
    for (int e = tid; e < CB * P; e += blockDim.x) {
        const int c = e / P, k = e - c * P;
        h[k * CB + c] = c < ncol ? src[(size_t)e * a.nr] : (R)0;
    }
    tz_stage<R>(a.twz, P, tz);
    __syncthreads();
    R *dst = a.Z + ((size_t)type * a.nr + (ir - 1)) * ngz * nm + s0;
    for (int q = tid; q < ngz; q += blockDim.x) {
        R v[CB];
#pragma unroll
        for (int c = 0; c < CB; c++) {
            const R e = h[(P - 1) * CB + c];
            v[c] = h[c] + ((q & 1) ? -e : e);
        }
        int idx = q;
#pragma unroll 4
        for (int k = 1; k < ngz; k++) {
            const R2 w = tz[tz_at<R>(idx)];
            const R *hk = h + (2 * k - 1) * CB;
            // (v + 2 x rounds as the fused product does: 2 x is exact)
#pragma unroll
            for (int c = 0; c < CB; c++)
                v[c] = fma((R)2, hk[c] * w.x - hk[CB + c] * w.y, v[c]);
            idx += q;
            if (idx >= P) idx -= P;
        }
#pragma unroll
        for (int c = 0; c < CB; c++)
            if (c < ncol) dst[(size_t)q * nm + c] = v[c];
    }
}

// grid (planes / P3Solve::planes, nr): inverse azimuthal transform of the
// active components of some planes of a ring, scale, polcat; interleaved
// field store
template <typename R, bool LPOT, int PL>
__global__ __launch_bounds__(P3_BLOCK) void p3_synth_kernel(P3SolveArgs<R> a) {
    typedef typename Vec4<R>::T R4;
    typedef typename Vec2<R>::T R2;
    constexpr int NT = LPOT ? 4 : 3;
    extern __shared__ unsigned char p3_lds[];
    R4 *zc = (R4 *)p3_lds;                    // [nm][PL]
    R2 *tws = (R2 *)(zc + a.nm * PL);         // [na]
    const int plane0 = blockIdx.x * PL, ir = blockIdx.y + 1, tid = threadIdx.x;
    const int na = a.na, nm = a.nm, ngz = a.ngz, mmax = a.mmax;
    const int jrs = a.ranges[0], jrf = a.ranges[2], krf = a.ranges[3];
    if (jrs < 1 || ir < jrf || ir > krf) return;
    for (int e = tid; e < 4 * PL * nm; e += blockDim.x) {
        const int t = e / (PL * nm), r = e - t * (PL * nm), p = r / nm, s = r - p * nm;
        R v = (R)0;
        if (t < NT && !(t == 1 && a.ng == 1) && plane0 + p < ngz)
            v = a.Z[(((size_t)t * a.nr + (ir - 1)) * ngz + plane0 + p) * nm + s];
        reinterpret_cast<R *>(zc)[4 * (s * PL + p) + t] = v;
    }
    for (int j = tid; j < na; j += blockDim.x) tws[j] = mk2(a.tw[2 * j], a.tw[2 * j + 1]);
    __syncthreads();
    const R scale = (R)1 / (R)(2 * ngz * na);
    const size_t row = ((size_t)(ir - 1) * ngz + plane0) * na;
    for (int j = tid; j < na; j += blockDim.x) {
        R F[PL][NT];
#pragma unroll
        for (int p = 0; p < PL; p++)
#pragma unroll
            for (int t = 0; t < NT; t++) F[p][t] = (R)0;
        // k = (m j) mod na, advanced with m (the slots come in ascending m)
        int mcur = 0, k = 0;
        for (int s = 0; s < nm; s++) {
            const int m = a.slot_m[s], part = a.slot_p[s];
            for (; mcur < m; mcur++) {
                k += j;
                if (k >= na) k -= na;
            }
            const R2 w = tws[k];
            R b = part ? (R)-2 * w.y : (R)2 * w.x;
            if (m == 0) b = (R)1;
            if (m == mmax - 1) b = (j & 1) ? (R)-1 : (R)1;
#pragma unroll
            for (int p = 0; p < PL; p++) {
                const R4 z = zc[s * PL + p];
                F[p][0] += z.x * b;
                F[p][1] += z.y * b;
                F[p][2] += z.z * b;
                if (LPOT) F[p][NT - 1] += z.w * b;
            }
        }
        const R cp = tws[j].x, sn = tws[j].y;
#pragma unroll
        for (int p = 0; p < PL; p++) {
            if (plane0 + p >= ngz) break;
            const R F0 = F[p][0] * scale, F1 = F[p][1] * scale;
            R *f = reinterpret_cast<R *>(a.fld + row + (size_t)p * na + j);
            const R x = F0 * cp - F1 * sn, y = F0 * sn + F1 * cp, z = F[p][2] * scale;
            if (LPOT) {
                *reinterpret_cast<R4 *>(f) = mk4(x, y, z, F[p][NT - 1] * scale);
            } else {
                // the potential of the last solve that formed it stays
                f[0] = x;
                f[1] = y;
                f[2] = z;
            }
        }
    }
}

// ---- Green's tables (FP64) --------------------------------------------------------

__device__ double p3_softm(double ds) {
    if (ds <= 0.0) return 0.0;
    if (ds < 1.0)
        return 4.0 * ds * ds * ds * (1.0 / 3.0 - 0.3 * ds * ds + 0.125 * ds * ds * ds);
    if (ds < 2.0)
        return -1.0 / 15.0 + ds * ds * ds *
               (8.0 / 3.0 - 3.0 * ds + 1.2 * ds * ds - ds * ds * ds / 6.0);
    return 1.0;
}

// radfor / azifor / vrtfor / grnfun with the field point at height zf
// (radfor.f:25-38, azifor.f:25-40, vrtfor.f:25-40, sftpot.f:20-40)
__device__ double p3_kernel(int type, double rs, double rf, double cth, double sth,
                            double zf, double eps, int tsoft) {
    const double d2 = rs * rs + rf * rf - 2.0 * rs * rf * cth + zf * zf;
    if (type == 3) {
        if (tsoft == 1) return -1.0 / sqrt(d2 + eps * eps);
        const double x = sqrt(d2) / eps;
        if (x <= 0.0) return -1.4 / eps;
        if (x < 1.0) return (-1.4 + x * x * (2.0 / 3.0 - 0.3 * x * x + 0.1 * x * x * x)) / eps;
        if (x < 2.0)
            return (-1.6 + 1.0 / (15.0 * x) +
                    x * x * (4.0 / 3.0 - x + 0.3 * x * x - x * x * x / 30.0)) / eps;
        return -1.0 / sqrt(d2);
    }
    const double num = type == 0 ? rs * cth - rf : type == 1 ? -rs * sth : -zf;
    if (tsoft == 1) {
        const double e = d2 + eps * eps;
        return num / (e * sqrt(e));
    }
    if (type == 2 ? zf != 0.0 : d2 > 0.0)
        return num * p3_softm(sqrt(d2) / eps) / (d2 * sqrt(d2));
    return 0.0;
}

constexpr int GREEN3_BLOCK = 128;
constexpr int GREEN3_CHUNK = 16;

// grid (nr, nr, 4): block (is, ir, type).  Phase 1: thread per height iz,
// the angular DCT-I / DST-I of the kernel samples for the kept harmonics
// (GREEN3_CHUNK at a time), filtered; phase 2: the vertical DCT-I (DST-I
// for F_z) of each harmonic's column.  twd: cos, sin of 2 pi k / na;
// twzd: cos, sin of 2 pi k / (2 ngz).
__global__ __launch_bounds__(GREEN3_BLOCK) void p3_green_kernel(
    double *__restrict__ G, const double *__restrict__ twd,
    const double *__restrict__ twzd, const int *__restrict__ lg, int nr, int na,
    int ngz, int ng, double alpha, double dzg, double eps, int tsoft) {
    extern __shared__ unsigned char p3_lds[];
    double *T = (double *)p3_lds;   // [nzp][nmq]
    const int is = blockIdx.x + 1, ir = blockIdx.y + 1, type = blockIdx.z;
    const int mmax = na / 2 + 1, P = 2 * ngz;
    const bool azim = type == 1, vert = type == 2;
    if (azim && ng == 1) return;
    const int it1 = azim ? 2 : 1, it2 = azim ? mmax - 1 : mmax;
    const int npt = it2 - it1 + 1;
    const int iz1 = vert ? 2 : 1, iz2 = vert ? ngz : ngz + 1;
    const int nzp = iz2 - iz1 + 1;
    const int nmq = azim ? min(ng, mmax - 1) - 1 : min(ng, mmax);
    if (nmq <= 0) return;
    const double rs = exp(alpha * (double)(is - 1)) - 1.0;
    const double rf = exp(alpha * (double)(ir - 1)) - 1.0;
    for (int iz = iz1 + threadIdx.x; iz <= iz2; iz += GREEN3_BLOCK) {
        const double zf = dzg * (double)(iz - 1);
        for (int m0 = 0; m0 < nmq; m0 += GREEN3_CHUNK) {
            double acc[GREEN3_CHUNK];
            int idx[GREEN3_CHUNK], inc[GREEN3_CHUNK];
#pragma unroll
            for (int u = 0; u < GREEN3_CHUNK; u++) {
                acc[u] = 0.0;
                // output index mo = m0 + u: harmonic mo (DCT) or mo + 1 (DST);
                // sample q has angle index it - 1 = q (DCT) or q + 1 (DST)
                const int h = azim ? m0 + u + 1 : m0 + u;
                inc[u] = h % na;
                idx[u] = azim ? inc[u] : 0;
            }
            for (int q = 0; q < npt; q++) {
                const int k = it1 - 1 + q;
                const double f = p3_kernel(type, rs, rf, twd[2 * k], twd[2 * k + 1], zf, eps, tsoft);
                const double wq = azim ? 2.0 : ((q == 0 || q == npt - 1) ? 1.0 : 2.0);
                const double fw = wq * f;
#pragma unroll
                for (int u = 0; u < GREEN3_CHUNK; u++) {
                    acc[u] += fw * (azim ? twd[2 * idx[u] + 1] : twd[2 * idx[u]]);
                    idx[u] += inc[u];
                    if (idx[u] >= na) idx[u] -= na;
                }
            }
#pragma unroll
            for (int u = 0; u < GREEN3_CHUNK; u++) {
                const int mo = m0 + u;
                if (mo >= nmq) break;
                const int h = azim ? mo + 1 : mo;
                T[(size_t)(iz - iz1) * nmq + mo] = (h >= ng || lg[h]) ? 0.0 : acc[u];
            }
        }
    }
    __syncthreads();
    const size_t nn = (size_t)nr * nr;
    for (int o = threadIdx.x; o < nzp * nmq; o += GREEN3_BLOCK) {
        const int p = o / nmq, mo = o - p * nmq;
        double v = 0.0;
        if (!vert) {
            // DCT-I over nzp = ngz + 1 points
            v = T[mo] + ((p & 1) ? -T[(size_t)(nzp - 1) * nmq + mo] : T[(size_t)(nzp - 1) * nmq + mo]);
            int id = p;
            for (int k = 1; k < nzp - 1; k++) {
                v += 2.0 * T[(size_t)k * nmq + mo] * twzd[2 * id];
                id += p;
                if (id >= P) id -= P;
            }
        } else {
            // DST-I over nzp = ngz - 1 points: output i = p + 1
            const int i = p + 1;
            int id = i;
            for (int k = 1; k <= nzp; k++) {
                v += 2.0 * T[(size_t)(k - 1) * nmq + mo] * twzd[2 * id + 1];
                id += i;
                if (id >= P) id -= P;
            }
        }
        const int kz = vert ? p + 1 : p;
        const int m = azim ? mo + 1 : mo;
        G[((((size_t)type * (ngz + 1) + kz) * ng + m) * nn) + (size_t)(is - 1) * nr + (ir - 1)] = v;
    }
}

// ---- launchers ------------------------------------------------------------------------

static unsigned p3_blocks(long long n) { return (unsigned)((n + P3_PBLOCK - 1) / P3_PBLOCK); }
template <typename R, int J, int PPT> static void p3_massgn(const P3Args<R> &a, hipStream_t s) {
    constexpr int TB = P3Shape<R, J, PPT>::block, per = TB * PPT;
    hipLaunchKernelGGL(HIP_KERNEL_NAME(p3_massgn_kernel<R, J, PPT>),
                       dim3((unsigned)((a.n + per - 1) / per)), dim3(TB), 0, s, a);
}
template <typename R, int J, int PPT> static void p3_push(const P3Args<R> &a, hipStream_t s) {
    constexpr int TB = P3Shape<R, J, PPT>::block, per = TB * PPT;
    hipLaunchKernelGGL(HIP_KERNEL_NAME(p3_push_kernel<R, J, PPT>),
                       dim3((unsigned)((a.n + per - 1) / per)), dim3(TB), 0, s, a);
}

template <typename R> hipError_t launch_p3_massgn(const P3Args<R> &a, hipStream_t s) {
    if (a.n <= 0) return hipSuccess;
    if (a.jmass == 3) p3_massgn<R, 3, 1>(a, s);
    else if (sizeof(R) == 8 || a.n <= P3_TWO) p3_massgn<R, 2, 1>(a, s);
    else if constexpr (sizeof(R) == 4) p3_massgn<R, 2, 2>(a, s);
    return hipGetLastError();
}

template <typename R> hipError_t launch_p3_push(const P3Args<R> &a, hipStream_t s) {
    if (a.n <= 0) return hipSuccess;
    if (a.jmass == 3) p3_push<R, 3, 1>(a, s);
    else if (sizeof(R) == 8 || a.n <= P3_TWO) p3_push<R, 2, 1>(a, s);
    else if constexpr (sizeof(R) == 4) p3_push<R, 2, 2>(a, s);
    return hipGetLastError();
}

template <typename R> hipError_t launch_p3_ut(const P3Args<R> &a, hipStream_t s) {
    if (a.n <= 0) return hipSuccess;
    hipLaunchKernelGGL(p3_ut_kernel<R>, dim3(p3_blocks(a.n)), dim3(P3_PBLOCK), 0, s, a);
    return hipGetLastError();
}

template <typename R> hipError_t launch_p3_tmcent(const P3Args<R> &a, hipStream_t s) {
    if (a.n <= 0) return hipSuccess;
    if (a.jmass == 3)
        hipLaunchKernelGGL(HIP_KERNEL_NAME(p3_tmcent_kernel<R, 3>), dim3(p3_blocks(a.n)), dim3(P3_PBLOCK), 0, s, a);
    else
        hipLaunchKernelGGL(HIP_KERNEL_NAME(p3_tmcent_kernel<R, 2>), dim3(p3_blocks(a.n)), dim3(P3_PBLOCK), 0, s, a);
    return hipGetLastError();
}

template <typename R> hipError_t launch_p3_gather(const P3GatherArgs<R> &b, hipStream_t s) {
    if (b.n <= 0) return hipSuccess;
    if (b.g.jmass == 3)
        hipLaunchKernelGGL(HIP_KERNEL_NAME(p3_gather_kernel<R, 3>), dim3(p3_blocks(b.n)), dim3(P3_PBLOCK), 0, s, b);
    else
        hipLaunchKernelGGL(HIP_KERNEL_NAME(p3_gather_kernel<R, 2>), dim3(p3_blocks(b.n)), dim3(P3_PBLOCK), 0, s, b);
    return hipGetLastError();
}

template <typename R>
hipError_t launch_p3_key(const P3Args<R> &a, int kshift, unsigned kmax, unsigned *key,
                         unsigned *perm, hipStream_t s) {
    if (a.n <= 0) return hipSuccess;
    if (a.jmass == 3)
        hipLaunchKernelGGL(HIP_KERNEL_NAME(p3_key_kernel<R, 3>), dim3(p3_blocks(a.n)), dim3(P3_PBLOCK), 0, s, a,
                           kshift, kmax, key, perm);
    else
        hipLaunchKernelGGL(HIP_KERNEL_NAME(p3_key_kernel<R, 2>), dim3(p3_blocks(a.n)), dim3(P3_PBLOCK), 0, s, a,
                           kshift, kmax, key, perm);
    return hipGetLastError();
}

template <typename R>
hipError_t launch_p3_interleave(const R *s4, const R *s2, typename Vec4<R>::T *rec,
                                unsigned *id, long long n, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(p3_interleave_kernel<R>, dim3(p3_blocks(n)), dim3(P3_PBLOCK), 0, s, s4,
                       s2, rec, id, n);
    return hipGetLastError();
}

template <typename R>
hipError_t launch_p3_deinterleave(const typename Vec4<R>::T *rec, const uint8_t *zone,
                                  const unsigned *id, unsigned *inv, R *d4, R *d2, int *iz,
                                  long long n, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    const dim3 grid(p3_blocks(n)), block(P3_PBLOCK);
    if (n < UNLOAD_GATHER) {
        hipLaunchKernelGGL(HIP_KERNEL_NAME(p3_deinterleave_kernel<R, false>), grid, block, 0, s,
                           rec, zone, id, d4, d2, iz, n);
        return hipGetLastError();
    }
    hipError_t e = launch_inverse_order(id, inv, n, s);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(HIP_KERNEL_NAME(p3_deinterleave_kernel<R, true>), grid, block, 0, s, rec,
                       zone, (const unsigned *)inv, d4, d2, iz, n);
    return hipGetLastError();
}

template <typename R> hipError_t launch_p3_permute(const P3PermArgs<R> &p, hipStream_t s) {
    if (p.n <= 0) return hipSuccess;
    hipLaunchKernelGGL(p3_permute_kernel<R>, dim3(p3_blocks(p.n)), dim3(P3_PBLOCK), 0, s, p);
    return hipGetLastError();
}

template <typename R>
hipError_t launch_p3_integrals(const P3Args<R> &a, int with_pot, const double4 *fp_c,
                               int nfp, double fp_dr, int centred,
                               double *part, double *out, hipStream_t s) {
    const IntSplit sp = int_split(a.n, P3_INT_BLOCK);
    const unsigned nb = (unsigned)sp.nb;
    if (nb && a.jmass == 3)
        hipLaunchKernelGGL(HIP_KERNEL_NAME(p3_integrals_kernel<R, 3>), dim3(nb),
                           dim3(P3_INT_BLOCK), 0, s, a, sp.per, with_pot, fp_c, nfp, fp_dr, centred, part);
    else if (nb)
        hipLaunchKernelGGL(HIP_KERNEL_NAME(p3_integrals_kernel<R, 2>), dim3(nb),
                           dim3(P3_INT_BLOCK), 0, s, a, sp.per, with_pot, fp_c, nfp, fp_dr, centred, part);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(p3_integrals_sum_kernel, dim3(NINT3), dim3(P3_INT_BLOCK), 0, s, part, (int)nb,
                       out);
    return hipGetLastError();
}

// Limits the launches below rely on (checked again by the context set-up).
// (the limits of whole-ring transforms; contexts beyond them are refused)
template <typename R> bool p3_solve_fits(const P3SolveArgs<R> &a) {
    const size_t P = 2 * (size_t)a.ngz;
    return a.na <= P3_MAX_NA && a.nm <= P3_MAX_NM && a.nr <= P3_MAX_NR &&
           ((size_t)a.nm * a.ngz + tz_words<R>(P)) * sizeof(R) <= 48 * 1024 &&
           ((size_t)a.nm * P + tz_words<R>(P)) * sizeof(R) <= 48 * 1024;
}

// block of whole wavefronts for n lanes
static dim3 p3_lanes(int n) { return dim3(std::min(P3_BLOCK, (n + 63) / 64 * 64)); }

// The vertical transforms by CB columns a block.  The forward transform takes
// three, the inverse nine or three.  Below 1500 columns of all rings (2000, of all
// types, in the inverse) one: more blocks for a chip that is not full (61 rings, 45 planes, 5
// columns: forward 6.5 us by threes, 4.6 by one, inverse 7.7 and 6.6; 140 rings, 17
// columns: forward 10.0 and 11.8).  The inverse reads a column twice as often as it multiplies it, from
// LDS: nine columns share a twiddle (three types of 200 rings, 17 columns:
// 46 us, three at a time 60) if that leaves four blocks a CU, else three, for
// more blocks (three types of 61 rings, 9 columns, FP64: 22 us and 9.8 us).
// With fewer columns in the context, no more of them than it has stand in LDS.
template <typename R, int CB>
static hipError_t p3_vertical(const P3SolveArgs<R> &a, bool inverse, hipStream_t s) {
    const size_t P = 2 * (size_t)a.ngz;
    const unsigned nc = (a.nm + CB - 1) / CB;
    if (inverse)
        hipLaunchKernelGGL(HIP_KERNEL_NAME(p3_zinv_kernel<R, CB>), dim3(a.nr, a.ntypes, nc),
                           p3_lanes(a.ngz), (CB * P + tz_words<R>(P)) * sizeof(R), s, a);
    else
        hipLaunchKernelGGL(HIP_KERNEL_NAME(p3_zfwd_kernel<R, CB>), dim3(a.nr, nc),
                           p3_lanes(a.ngz + 1), (CB * a.ngz + tz_words<R>(P)) * sizeof(R), s, a);
    return hipGetLastError();
}
template <typename R>
static hipError_t p3_vertical(const P3SolveArgs<R> &a, bool inverse, hipStream_t s) {
    if (a.nm == 0) return hipSuccess;
    if (a.nm < 3 || a.nr * a.nm * (inverse ? a.ntypes : 1) < (inverse ? 2000 : 1500))
        return p3_vertical<R, 1>(a, inverse, s);
    if (inverse && a.nm >= 9 && (long long)a.nr * a.ntypes * ((a.nm + 8) / 9) >= 1024)
        return p3_vertical<R, 9>(a, inverse, s);
    return p3_vertical<R, 3>(a, inverse, s);
}

template <typename R, int PL, int HB, bool SPLIT = false>
static void p3_analysis(const P3SolveArgs<R> &a, hipStream_t s) {
    constexpr unsigned per = P3_BLOCK / 64 * PL;
    const unsigned passes = SPLIT ? std::max(1, (a.nharm + HB - 1) / HB) : 1;
    hipLaunchKernelGGL(HIP_KERNEL_NAME(p3_analyse_kernel<R, PL, HB, SPLIT>),
                       dim3((a.ngz + per - 1) / per, a.nr, passes),
                       dim3(P3_BLOCK + (SPLIT ? 64 : 0)), 2 * a.na * sizeof(R), s, a);
}
template <typename R, int PL> static void p3_analysis(const P3SolveArgs<R> &a, hipStream_t s) {
    switch (harm_per_pass(a.nharm)) {
    case 3: return p3_analysis<R, PL, 3>(a, s);
    case 5: return p3_analysis<R, PL, 5>(a, s);
    case 7: return p3_analysis<R, PL, 7>(a, s);
    default: return p3_analysis<R, PL, 9>(a, s);
    }
}

template <typename R, bool LPOT, int PL>
static void p3_synthesis(const P3SolveArgs<R> &a, hipStream_t s) {
    hipLaunchKernelGGL(HIP_KERNEL_NAME(p3_synth_kernel<R, LPOT, PL>),
                       dim3((a.ngz + PL - 1) / PL, a.nr), p3_lanes(a.na),
                       (4 * (size_t)a.nm * PL + 2 * a.na) * sizeof(R), s, a);
}
template <typename R, int PL> static void p3_synthesis(const P3SolveArgs<R> &a, hipStream_t s) {
    if (a.lpot) p3_synthesis<R, true, PL>(a, s);
    else p3_synthesis<R, false, PL>(a, s);
}

// A wavefront per plane of a ring leaves a small grid's chip idle and takes its
// harmonics one pass after the other: below P3_SPLIT planes of all rings each pass
// of three harmonics gets wavefronts of its own, and the synthesis one plane a
// block (24 rings x 16 planes, 9 harmonics: analysis 10.0 -> 4.9 us, synthesis 7.6
// -> 5.6; 61 x 45: 9.8 and 10.1, 8.2 and 9.0); below P3_PAIR a wavefront takes one
// plane (61 x 45 10.5 -> 9.8; 100 x 61 12.5 and 15.0).
constexpr int P3_SPLIT = 2000, P3_PAIR = 3000;

template <typename R> hipError_t launch_p3_solve(const P3SolveArgs<R> &a, hipStream_t s) {
    if (!p3_solve_fits(a)) return hipErrorInvalidValue;
    const int cells = a.nr * a.ngz;   // rings of all planes
    if (cells < P3_SPLIT) p3_analysis<R, 1, 3, true>(a, s);
    else if (cells < P3_PAIR) p3_analysis<R, 1>(a, s);
    else p3_analysis<R, P3Solve<R>::planes>(a, s);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if ((e = p3_vertical(a, false, s)) != hipSuccess) return e;
    hipLaunchKernelGGL(p3_conv_kernel<R>, dim3(a.ng, a.ngz + 1, a.ntypes), dim3(P3_BLOCK),
                       0, s, a);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if ((e = p3_vertical(a, true, s)) != hipSuccess) return e;
    if (cells < P3_SPLIT) p3_synthesis<R, 1>(a, s);
    else p3_synthesis<R, P3Solve<R>::splanes>(a, s);
    return hipGetLastError();
}

hipError_t launch_p3_green(double *G, const double *twd, const double *twzd, const int *lg,
                           int nr, int na, int ngz, int ng, double alpha, double dzg,
                           double eps, int tsoft, hipStream_t s) {
    const int mmax = na / 2 + 1;
    const size_t lds = sizeof(double) * (size_t)(ngz + 1) * (ng < mmax ? ng : mmax);
    if (lds > 48 * 1024) return hipErrorInvalidValue;
    hipLaunchKernelGGL(p3_green_kernel, dim3(nr, nr, 4), dim3(GREEN3_BLOCK), lds, s, G, twd,
                       twzd, lg, nr, na, ngz, ng, alpha, dzg, eps, tsoft);
    return hipGetLastError();
}

#define P3_INST(R)                                                                     \
    template hipError_t launch_p3_massgn<R>(const P3Args<R> &, hipStream_t);          \
    template hipError_t launch_p3_push<R>(const P3Args<R> &, hipStream_t);            \
    template hipError_t launch_p3_tmcent<R>(const P3Args<R> &, hipStream_t);          \
    template hipError_t launch_p3_ut<R>(const P3Args<R> &, hipStream_t);              \
    template hipError_t launch_p3_integrals<R>(const P3Args<R> &, int, const double4 *, \
                                               int, double, int,                       \
                                               double *, double *, hipStream_t);       \
    template hipError_t launch_p3_gather<R>(const P3GatherArgs<R> &, hipStream_t);    \
    template hipError_t launch_p3_solve<R>(const P3SolveArgs<R> &, hipStream_t);      \
    template bool p3_solve_fits<R>(const P3SolveArgs<R> &);                            \
    template hipError_t launch_p3_key<R>(const P3Args<R> &, int, unsigned, unsigned *,  \
                                         unsigned *, hipStream_t);                     \
    template hipError_t launch_p3_permute<R>(const P3PermArgs<R> &, hipStream_t);          \
    template hipError_t launch_p3_interleave<R>(const R *, const R *, typename Vec4<R>::T *,  \
                                                unsigned *, long long, hipStream_t);          \
    template hipError_t launch_p3_deinterleave<R>(const typename Vec4<R>::T *, const uint8_t *, \
                                                  const unsigned *, unsigned *, R *, R *, int *, \
                                                  long long, hipStream_t);
P3_INST(float)
P3_INST(double)

}  // namespace gh
