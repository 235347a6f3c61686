// galhip_push.hip -- the fused particle kernel of the p2d step, the mass
// assignment of masset, the group-level gather kernel and the sort helpers.
//
// push_kernel does, for each particle of the zones due at this step, what
// the reference's per-group pipeline does (SRC/lib15/step.f:186-234):
//   getacc/grdacc  CIC weights at the old position, 4-corner interpolation
//                  of the Cartesian field, fixed radial force, zone scaling
//                  (getacc.f:35-163, grdacc.f:40-66)
//   stpgrp/offgrd  RVLF leap-frog and the off-grid test (stpgrp.f:27-56,
//                  offgrd.f:55-59, addoff.f:30-70)
//   rezgrp/chstep  zone changes (rezgrp.f:30-50, zoneno.f, chstep.f:22-31)
//   massgn         weights at the new position, scatter into the zone's
//                  mass array (massgn.f:68-89)
// in one pass over the particle arrays.
//
// The old position's weights are not recomputed: every particle carries the
// (u, t) grid coordinates that its last mass assignment formed from the
// same position with the same formulas (weight.f forms them twice per step,
// once for the forces and once for the masses), so the transcendental part
// runs once per push.
//
// Mass sums are 64-bit fixed point (weight x 2^qbits): integer adds
// commute, so the sums are bit-identical for any processing order and need
// no float atomics.  Each block deposits into an LDS tile that covers the
// rings x spokes window of its particles (particles are kept ordered by
// cell, so the window is small) and flushes every non-zero tile cell with
// one 64-bit global atomic.  Global 64-bit atomics are the scarce resource
// on MI355X (about 24 G/s device-wide), LDS atomics far less so.
#include "galhip_kern.h"
#include <climits>

namespace gh {

constexpr int PB = GH_PUSH_BLOCK;      // threads per block

// Launch shapes by particles per thread, measured (push time, us; FP32, 128
// spokes | 512 spokes where two figures are given):
//   particles       1 per thread     2            4
//   5e4             13.1 | 26.4      16.0 | 34.1  22.0 | 45.4
//   8e5             24.3 | 27.9      24.3 | 31.9  26.3 | 42.7
//   2e6             45.6 | 47.9      43.7 | 44.7  44.3 | 45.7
//   1e7, 3 zones    124              104          102
// FP64, 3e6 in 3 zones: 55.8, 56.2, 60.6; 1e7: 169, -, 170; never sorted again, a
// block's particles lie all over the disc, and more of them share the flush of a
// window (93 x 128, step us): 3e6 91.7, 81.0, 79.1; 1e7 281, 248, 241.  A block's own latency is what a
// small count waits for, and it grows with the particles per thread; a large
// one pays for the window work of every block.  The tile: 3072 cells in one
// copy against 1024 in two copies (lanes of one cell spread over them) takes
// the ensemble's push from 171 to 143 us, 1e7 particles in 3 zones from 101.8
// to 101.1 us (fewer second passes, the same LDS).  Wavefronts per SIMD: as
// many as the registers allow without spills.
template <typename R, bool COMP, int PPT> struct PushShape {
    static constexpr int tile = PPT == 1 ? 2048 : 3072;
    static constexpr int waves = PPT == 1 ? 8 : (COMP ? 5 : 6);
};
constexpr int PUSH_PASSES = 8;         // deposit window passes before global atomics
constexpr int CLIP_RINGS = 16;          // rings of a window that had to be clipped

template <typename R>
__device__ __forceinline__ R tsfac(const PushArgs<R> &a, int iz) {
    return (R)step_ratio(a.nstep, a.nz, iz);
}

// zoneno for a position of known radius (zoneno.f:40-55)
template <typename R>
__device__ __forceinline__ int zone_of(const PushArgs<R> &a, R rad) {
    // the first two boundaries in uniform branches with the radii read at
    // fixed offsets; only more than three zones take the loop
    int z = 1;
    if (a.nz >= 2) {
        if (rad >= a.zbr[1]) z = 2;
        if (a.nz >= 3) {
            if (rad >= a.zbr[2]) z = 3;
            for (int i = 4; i <= a.nz; i++)
                if (rad >= a.zbr[i - 1]) z = i;
        }
    }
    return z;
}

template <typename R>
__device__ __forceinline__ void chstep(R tfac, R ox, R oy, R &ovx, R &ovy,
                                       R &ax, R &ay, R &nx, R &ny, R &nvx,
                                       R &nvy) {
    const R h = (R)0.5;
    ovx = tfac * (ovx + h * ax * ((R)1 - tfac));
    ax = ax * tfac * tfac;
    nvx = ovx + ax;
    nx = ox + nvx;
    ovy = tfac * (ovy + h * ay * ((R)1 - tfac));
    ay = ay * tfac * tfac;
    nvy = ovy + ay;
    ny = oy + nvy;
}

// Compensated position update: the position is hi + lo, and the new
// (hi, lo) = TwoSum(hi, v + lo) (Knuth's two-sum, exact without fused
// operations), so each update's rounding error is carried, not dropped.
template <typename R>
__device__ __forceinline__ R comp_add(R x, R v, R lo, R &lo_out) {
    const R y = v + lo;
    const R s = x + y;
    const R bp = s - x;
    lo_out = (x - (s - bp)) + (y - bp);
    return s;
}

__device__ __forceinline__ int wave_min(int v) { return wave_min_i32(v); }
__device__ __forceinline__ int wave_max(int v) { return wave_max_i32(v); }

// Hides a value's origin from the optimiser (no instruction is issued).
__device__ __forceinline__ void opaque(float2 &v) { asm volatile("" : "+v"(v.x), "+v"(v.y)); }
__device__ __forceinline__ void opaque(double2 &v) { asm volatile("" : "+v"(v.x), "+v"(v.y)); }

// LDS of a block's deposit.
template <int TILE> struct DepositLds {
    long long tile[TILE];
    int jr[GH_MAXZ], kr[GH_MAXZ];    // ring ranges by zone
    int box[8];                      // two (ring min, max, offset min, max) boxes
    unsigned long long ref[2];       // two reference keys
};

// Set up before the block's first barrier.
template <int TILE> __device__ __forceinline__ void deposit_init(DepositLds<TILE> &s) {
    const int tid = threadIdx.x;
#pragma unroll
    for (int j = 0; j < TILE; j += PB) s.tile[j + tid] = 0;
    if (tid < GH_MAXZ) {
        s.jr[tid] = INT_MAX;
        s.kr[tid] = -1;
    }
    if (tid == 0) {
        s.box[0] = s.box[4] = INT_MAX;
        s.box[1] = s.box[5] = -1;
        s.box[2] = s.box[6] = INT_MAX;
        s.box[3] = s.box[7] = INT_MIN;
        s.ref[0] = s.ref[1] = ~0ull;
    }
}

// The reference of the first deposit window: the block's middle particle.
struct PushRef {
    int zone, ring, spoke;
};
template <typename R2> __device__ __forceinline__ PushRef push_ref(R2 ut, int zone, int nz, int nr, int na) {
    PushRef r;
    r.zone = min(max(zone, 1), nz);
    r.ring = min(max((int)ut.x, 0), nr - 2);
    r.spoke = min(max((int)ut.y, 0), na - 1);
    return r;
}

// The block's deposits (massgn.f:68-89).  A pass takes a zone, a reference cell and the box of
// the zone's pending deposits (rings x spoke offsets from the reference
// spoke, which wrap around the ring); a box over TILE cells is
// clipped about the reference.  The deposits inside go to the LDS tile,
// which is then flushed with one global atomic per touched cell and
// cleared.  What the clip or a second zone leaves pending gets the next
// pass.  The first pass's reference is the block's middle particle, a
// later one's the pending deposit first in particle order from there
// (always inside its own window); after PUSH_PASSES passes (and for a
// cell on the last ring) the corners go to global atomics directly.
// cu: (u, t) of the thread's particles, t folded into the sector; dzone: their
// zones, four bits each (0: no deposit).  Every thread of the block calls it.
template <typename R, int PPT, int TILE>
__device__ __forceinline__ void deposit_block(const PushArgs<R> &a, DepositLds<TILE> &s,
                                              typename Vec2<R>::T (&cu)[PPT], unsigned dzone,
                                              PushRef ref, int qbits, long long mo) {
    const int tid = threadIdx.x, lane = tid & 63;
    const int na = a.na, nr = a.nr, nz = a.nz, half = na >> 1;
    auto cell_of = [&](int k, int &ring, int &spoke) {
        ring = min((int)cu[k].x, nr - 2);
        spoke = (int)cu[k].y;
        if (spoke >= na) {
            ring++;
            spoke -= na;
        }
    };
    unsigned pend = 0;
#pragma unroll
    for (int k = 0; k < PPT; k++) {
        int ring, spoke;
        cell_of(k, ring, spoke);
        if ((dzone >> (4 * k) & 15u) && ring + 1 < nr) pend |= 1u << k;
    }
    // pending deposits of zone z
    auto in_zone = [&](int k, int z) {
        return (pend >> k & 1u) && (int)(dzone >> (4 * k) & 15u) == z;
    };
#pragma unroll 1
    for (int pass = 0;; pass++) {
        int *const bx = s.box + 4 * (pass & 1);
        // cells and weights are formed again from (u, t) in every pass: kept
        // across the passes they would not fit the registers
#pragma unroll
        for (int k = 0; k < PPT; k++) opaque(cu[k]);
        // ring and spoke-offset box of the zone's pending deposits
        {
            int rmin = INT_MAX, rmax = -1, dmin = INT_MAX, dmax = INT_MIN;
#pragma unroll
            for (int k = 0; k < PPT; k++) {
                int ring, d;
                cell_of(k, ring, d);
                d -= ref.spoke;
                if (d < -half) d += na;
                else if (d >= half) d -= na;
                if (in_zone(k, ref.zone)) {
                    rmin = min(rmin, ring);
                    rmax = max(rmax, ring);
                    dmin = min(dmin, d);
                    dmax = max(dmax, d);
                }
            }
            rmin = wave_min(rmin);
            rmax = wave_max(rmax);
            dmin = wave_min(dmin);
            dmax = wave_max(dmax);
            if (lane == 0 && rmax >= 0) {
                atomicMin(&bx[0], rmin);
                atomicMax(&bx[1], rmax);
                atomicMin(&bx[2], dmin);
                atomicMax(&bx[3], dmax);
            }
        }
        __syncthreads();
        // tile: rings [r0, r0 + th) x spoke offsets [d0, d0 + tw)
        int r0 = bx[0], th = bx[1] - bx[0] + 2, d0 = bx[2], tw = bx[3] - bx[2] + 2;
        const bool some = bx[1] >= 0;
        if (tid == 0) {
            if (some) {
                atomicMin(&s.jr[ref.zone - 1], bx[0]);
                atomicMax(&s.kr[ref.zone - 1], bx[1]);
            }
            // the other box and key were last read before this barrier
            int *const nb = s.box + 4 * ((pass + 1) & 1);
            nb[0] = INT_MAX;
            nb[1] = -1;
            nb[2] = INT_MAX;
            nb[3] = INT_MIN;
            s.ref[(pass + 1) & 1] = ~0ull;
        }
        if (some && th * tw > TILE) {
            if (th > CLIP_RINGS) {
                r0 = min(max(ref.ring - (CLIP_RINGS / 2 - 1), r0), r0 + th - CLIP_RINGS);
                th = CLIP_RINGS;
            }
            const int mw = TILE / th;
            if (tw > mw) {
                d0 = min(max(-((mw - 2) >> 1), d0), d0 + tw - mw);
                tw = mw;
            }
        }
        const int tlen = some ? th * tw : 0;
#pragma unroll
        for (int k = 0; k < PPT; k++) {
            R w[4];
            int ring, d;
            cic(cu[k].x, cu[k].y, nr, na, ring, d, w);
            d -= ref.spoke;
            if (d < -half) d += na;
            else if (d >= half) d -= na;
            if (!in_zone(k, ref.zone) || ring < r0 || ring - r0 + 1 >= th || d < d0 ||
                d - d0 + 1 >= tw)
                continue;
            long long qv[4];
            quant_n<R, 4>(w, qbits, true, qv);
            const int b = (ring - r0) * tw + (d - d0);
            const int ti[4] = {b, b + 1, b + tw, b + tw + 1};
#pragma unroll
            for (int q = 0; q < 4; q++)
                atomicAdd((unsigned long long *)&s.tile[ti[q]], (unsigned long long)qv[q]);
            pend &= ~(1u << k);
        }
        // the next pass's reference: the lowest particle index, counted from
        // the block's middle, among the pending deposits
        if (any_lane(pend != 0)) {
            int myrot = INT_MAX, mypack = 0;
#pragma unroll
            for (int k = 0; k < PPT; k++) {
                const int rot = (k * PB + tid - PB * PPT / 2) & (PB * PPT - 1);
                int ring, spoke;
                cell_of(k, ring, spoke);
                if ((pend >> k & 1u) && rot < myrot) {
                    myrot = rot;
                    mypack = (int)((dzone >> (4 * k) << 28) | ((unsigned)ring << 16) |
                                   (unsigned)spoke);
                }
            }
            const int wmin = wave_min(myrot);
            const int fl = __ffsll((long long)__ballot(myrot == wmin)) - 1;
            const int pk = __builtin_amdgcn_readlane(mypack, fl);
            if (lane == 0)
                atomicMin(&s.ref[pass & 1], ((unsigned long long)(unsigned)wmin << 32) | (unsigned)pk);
        }
        __syncthreads();
        // flush: one global atomic per touched cell, the tile's cells over
        // all threads in storage order (a row's cells are consecutive
        // spokes, so a wave's atomics coalesce); (row, col) advanced by the
        // block size with a carry
        if (tid < tlen) {
            const int drow = div_small(PB, tw), dcol = PB - drow * tw;
            int row = div_small(tid, tw), col = tid - row * tw;
            for (int j = tid; j < tlen; j += PB) {
                const long long v = s.tile[j];
                if (v != 0) {
                    s.tile[j] = 0;
                    int spoke = ref.spoke + d0 + col;
                    if (spoke < 0) spoke += na;
                    else if (spoke >= na) spoke -= na;
                    if (spoke >= na) spoke -= na;
                    atomicAdd((unsigned long long *)&a.mfx[ref.zone - 1][mo + (r0 + row) * na + spoke],
                              (unsigned long long)v);
                }
                row += drow;
                col += dcol;
                if (col >= tw) {
                    col -= tw;
                    row++;
                }
            }
        }
        const unsigned long long kref = s.ref[pass & 1];
        if (kref == ~0ull || pass + 1 >= PUSH_PASSES) break;   // uniform
        ref.zone = (int)((kref >> 28) & 0xF);
        ref.ring = (int)((kref >> 16) & 0xFFF);
        ref.spoke = (int)(kref & 0xFFFF);
    }
    // what no pass took (and cells on the last ring): global atomics
#pragma unroll
    for (int k = 0; k < PPT; k++) {
        const int z = (int)(dzone >> (4 * k) & 15u);
        R w[4];
        int ring, spoke;
        cic(cu[k].x, cu[k].y, nr, na, ring, spoke, w);
        if (z == 0 || (ring + 1 < nr && !(pend >> k & 1u))) continue;
        long long qv[4];
        quant_n<R, 4>(w, qbits, true, qv);
        atomicMin(&s.jr[z - 1], ring);
        atomicMax(&s.kr[z - 1], ring);
        int ic[4];
        corners_rs(ring, spoke, na, ic);
#pragma unroll
        for (int q = 0; q < 4; q++)
            if (qv[q] != 0) deposit_global(a.mfx, nz, a.mesh, z, ic[q], qv[q], mo);
    }
}

// The block's ring ranges join the grid's (after a barrier).
template <int TILE>
__device__ __forceinline__ void deposit_ranges(const DepositLds<TILE> &s, int nz, int nr, int *jrad,
                                               int *krad, int rstride) {
    const int tid = threadIdx.x;
    if (tid < nz && s.kr[tid] >= 0) {
        const int k = s.kr[tid] + 2;
        widen_range(jrad, krad, rstride, blockIdx.x, tid + 1, s.jr[tid] + 1, k < nr ? k : nr);
    }
}

// ENS: an ensemble launch, the block's particles and member from a.blk.
// COMP: compensated positions (a.xlo holds the low words).
// PPT: particles per thread (see push_ppt).
template <typename R, bool ENS, bool COMP, int PPT>
__global__ __launch_bounds__(PB, (PushShape<R, COMP, PPT>::waves)) void push_kernel(PushArgs<R> a) {
    typedef typename Vec2<R>::T R2;
    typedef typename Vec4<R>::T R4;
    __shared__ DepositLds<PushShape<R, COMP, PPT>::tile> s_dep;
    __shared__ int s_dnoff, s_pushes;
    // the logarithm and arc-tangent tables, read per particle by ut_push
    __shared__ double s_tab[UtTab<R>::n];

    const int tid = threadIdx.x, lane = tid & 63;
    // the block's particles and its grid (ensembles: member eb.x)
    const int4 eb = ENS ? a.blk[blockIdx.x] : make_int4(0, 0, 0, 0);
    const long long base = ENS ? (long long)eb.y : (long long)blockIdx.x * (PB * PPT);
    const long long mo = ENS ? (long long)eb.x * a.mesh : 0;
    const R2 *const fld = a.fld + mo;
    int *const jrad = a.jrad + (ENS ? eb.x * GH_MAXZ : 0);
    int *const krad = a.krad + (ENS ? eb.x * GH_MAXZ : 0);
    long long *const counters = a.counters + (ENS ? eb.x * 4 : 0);
    const int qbits = ENS ? a.qbits_m[eb.x] : a.qbits;
    const int nz = a.nz, nlists = a.nz + 1, na = a.na, nr = a.nr;
    // the block's particles through block-based pointers and 32-bit
    // offsets (uniform base, per-lane offset: no 64-bit address arithmetic)
    R4 *const xvb = a.xv + base;
    R2 *const utb = a.ut + base;
    R2 *const lob = COMP ? a.xlo + base : nullptr;
    uint8_t *const zb = a.zone + base;
    const int nblk = ENS ? eb.z : (int)min((long long)(PB * PPT), a.n - base);
    // On a full step every list moves: the particles are loaded without
    // waiting for their zones, one memory latency instead of two.  Other
    // steps look at the zones first, since many blocks have nothing to move.
    const bool full = a.mzone == nz;
    int zin[PPT];
    R4 st[PPT];
    R2 cu[PPT], lo_[COMP ? PPT : 1];
#pragma unroll
    for (int k = 0; k < PPT; k++) zin[k] = zb[min(k * PB + tid, nblk - 1)];
    const int zmid = zb[nblk >> 1];
    const R2 umid = utb[nblk >> 1];
    auto load_state = [&]() {
#pragma unroll
        for (int k = 0; k < PPT; k++) {
            const int j = min(k * PB + tid, nblk - 1);
            cu[k] = utb[j];
            st[k] = xvb[j];
            if (COMP) lo_[k] = lob[j];
        }
    };
    if (full) load_state();
    // LDS set-up while the loads are in flight
    for (int j = tid; j < UtTab<R>::n; j += PB) s_tab[j] = ut_tab_entry<R>(j);
    deposit_init(s_dep);
    if (tid == 0) s_dnoff = s_pushes = 0;
    unsigned mv = 0;   // bit k: particle k moves
    if (!full)
#pragma unroll
        for (int k = 0; k < PPT; k++)
            if (k * PB + tid < nblk && zin[k] <= a.mzone) mv |= 1u << k;
    // every thread reaches this barrier; a block with nothing to move exits
    if (!__syncthreads_or(full ? 1 : (int)mv)) return;
    if (full) {
#pragma unroll
        for (int k = 0; k < PPT; k++)
            if (k * PB + tid < nblk && (zin[k] != nlists || a.offanal)) mv |= 1u << k;
    } else {
        load_state();
    }
    const PushRef ref = push_ref(umid, zmid, nz, nr, na);

    // grdacc's reads for particle k: the four field corners of its old cell
    // (weights of the old position from its (u, t)) and its interval of the
    // fixed-force table, straight from the L2 (particles are ordered by cell,
    // so a wavefront touches a few lines).  Staging the block's field window
    // in LDS cost two more barriers and a wavefront reduction for its box,
    // and held the registers and the LDS of a sixth wavefront per SIMD.
    R2 f[4];
    double4 fc;
    auto gather = [&](int k) {
        R w[4];
        int ring, spoke, ic[4];
        const bool grid = (mv >> k & 1u) && zin[k] != nlists;
        cic(grid ? cu[k].x : (R)0, grid ? cu[k].y : (R)0, nr, na, ring, spoke, w);
        corners_rs(ring, spoke, na, ic);
#pragma unroll
        for (int q = 0; q < 4; q++) f[q] = fld[ic[q] < a.mesh ? ic[q] : 0];
        if (a.fixforce) {
            const R rr = sqrt_rn(st[k].x * st[k].x + st[k].y * st[k].y);
            fc = a.fr_c[fixforce_index((double)rr, a.nfr, a.fr_inv_dr)];
        }
    };
    // zones of the deposits, four bits per particle (0: none); the new
    // state takes the registers of the old one, stored once every load has
    // been used: a load waits for the stores issued before it
    unsigned dzone = 0, zch = 0;
    int npush = 0, nplus = 0, nminus = 0;   // lane counts by ballot (uniform)
#pragma unroll
    for (int k = 0; k < PPT; k++) {
        gather(k);
        bool plus = false, minus = false;   // leaving the grid, returning
        const bool move = mv >> k & 1u;
        npush += __popcll(__ballot(move));
        if (move) {
            opaque(cu[k]);
            const int z0 = zin[k];
            const bool offlist = z0 == nlists;
            R ox = st[k].x, oy = st[k].y, ovx = st[k].z, ovy = st[k].w;
            const R rr = sqrt_rn(ox * ox + oy * oy);
            R ax_ = 0, ay_ = 0;
            if (!offlist) {
                R w[4];
                int ring, spoke, ic[4];
                cic(cu[k].x, cu[k].y, nr, na, ring, spoke, w);
                corners_rs(ring, spoke, na, ic);
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    // the last ring with t == na points past the field: 0
                    const R wq = ic[q] < a.mesh ? w[q] : (R)0;
                    ax_ = ax_ + f[q].x * wq;
                    ay_ = ay_ + f[q].y * wq;
                }
                if (a.fixforce) {
                    const int kf = fixforce_index((double)rr, a.nfr, a.fr_inv_dr);
                    const R fr = (R)fixforce_at((double)rr, kf, a.nfr, a.fr_inv_dr, &fc, kf);
                    if (fr != (R)0) {
                        const R fo = div_rn(fr, rr);
                        ax_ = ax_ + fo * ox;
                        ay_ = ay_ + fo * oy;
                    }
                }
            }
            if (nz > 1 && z0 > 1) {
                R t = tsfac(a, z0);
                t = t * t;
                ax_ = t * ax_;
                ay_ = t * ay_;
            }
            R nvx = ovx + ax_, nvy = ovy + ay_;
            R nx = ox + nvx, ny = oy + nvy;
            R2 lo = zero2<R>(), elo = zero2<R>();
            if (COMP) {
                lo = lo_[k];
                nx = comp_add(ox, nvx, lo.x, elo.x);
                ny = comp_add(oy, nvy, lo.y, elo.y);
            }
            int znew = z0;
            R rnew = sqrt_rn(nx * nx + ny * ny);
            bool off = rnew > a.rgrid;
            if (!offlist) {
                if (off) {
                    znew = nlists;
                    plus = true;
                    if (a.offanal && z0 < nz) {
                        R tfac = tsfac(a, nz) / tsfac(a, z0);
                        chstep(tfac, ox, oy, ovx, ovy, ax_, ay_, nx, ny, nvx, nvy);
                        if (COMP) {
                            nx = comp_add(ox, nvx, lo.x, elo.x);
                            ny = comp_add(oy, nvy, lo.y, elo.y);
                        }
                        rnew = sqrt(nx * nx + ny * ny);
                    }
                }
            } else if (!off) {
                minus = true;
                znew = nz;
            }
            if (a.mzone > 1 && !offlist && znew <= a.mzone) {
                int kz = zone_of(a, rnew);
                if (kz > a.mzone) kz = a.mzone;
                if (kz > znew) kz = zone_of(a, rr);
                if (kz != znew) {
                    R tfac = tsfac(a, kz) / tsfac(a, znew);
                    chstep(tfac, ox, oy, ovx, ovy, ax_, ay_, nx, ny, nvx, nvy);
                    if (COMP) {
                        nx = comp_add(ox, nvx, lo.x, elo.x);
                        ny = comp_add(oy, nvy, lo.y, elo.y);
                    }
                    rnew = sqrt(nx * nx + ny * ny);
                    znew = kz;
                }
            }
            st[k] = mk4(nx, ny, nvx, nvy);
            if (COMP) lo_[k] = elo;
            if (znew != z0) zch |= 1u << k;
            zin[k] = znew;
            if (znew >= 1 && znew <= nz) {
                R u, t;
                ut_push(nx, ny, rnew, a.k, u, t, s_tab);
                cu[k] = mk2(u, t);
                dzone |= (unsigned)znew << (4 * k);
            }
        }
        nplus += __popcll(__ballot(plus));
        nminus += __popcll(__ballot(minus));
    }
#pragma unroll
    for (int k = 0; k < PPT; k++) {
        const int j = k * PB + tid;
        if (mv >> k & 1u) {
            xvb[j] = st[k];
            if (COMP) lob[j] = lo_[k];
            if (zch >> k & 1u) zb[j] = (uint8_t)zin[k];
            if (dzone >> (4 * k) & 15u) utb[j] = cu[k];
        }
        // the deposit's angle is folded into the sector
        if (a.nsect > 1) cu[k].y = (R)fmod(cu[k].y, a.thmax);
    }
    // the wave's pushes and off-grid change, added to the block's counters by
    // one lane
    if (lane == 0) {
        if (npush) atomicAdd(&s_pushes, npush);
        if (nplus != nminus) atomicAdd(&s_dnoff, nplus - nminus);
    }
    deposit_block<R, PPT>(a, s_dep, cu, dzone, ref, qbits, mo);
    __syncthreads();
    deposit_ranges(s_dep, nz, nr, jrad, krad, a.rstride);
    if (tid == 0) {
        if (s_dnoff) atomicAdd((unsigned long long *)&counters[0],
                               (unsigned long long)(long long)s_dnoff);
        count_pushes(a.pushes, blockIdx.x, s_pushes);
    }
}

// masset / massgn for every on-grid particle without a push: also fills the
// particles' (u, t) so the next push finds them.  ENS: the members' blocks
// of a.blk.  The push's deposit and its particles per thread (with a reduction
// over the wavefront per cell and global atomics it took 530 us for 1e7
// particles, 108 us now).
template <typename R, bool ENS, int PPT>
__global__ __launch_bounds__(PB, (PushShape<R, false, PPT>::waves)) void massgn_kernel(PushArgs<R> a) {
    typedef typename Vec2<R>::T R2;
    __shared__ DepositLds<PushShape<R, false, PPT>::tile> s_dep;
    __shared__ R2 s_mid;
    __shared__ int s_zmid;
    const int tid = threadIdx.x;
    const int4 eb = ENS ? a.blk[blockIdx.x] : make_int4(0, 0, 0, 0);
    const long long base = ENS ? (long long)eb.y : (long long)blockIdx.x * (PB * PPT);
    const int nblk = ENS ? eb.z : (int)min((long long)(PB * PPT), a.n - base);
    R2 cu[PPT];
    unsigned dzone = 0;
#pragma unroll
    for (int k = 0; k < PPT; k++) {
        const int j = k * PB + tid;
        cu[k] = zero2<R>();
        const int z = j < nblk ? a.zone[base + j] : 0;
        if (z >= 1 && z <= a.nz) {
            const typename Vec4<R>::T st = a.xv[base + j];
            R u, t;
            ut_of(st.x, st.y, sqrt(st.x * st.x + st.y * st.y), a.k, u, t);
            a.ut[base + j] = mk2(u, t);
            cu[k] = mk2(u, a.nsect > 1 ? (R)fmod(t, a.thmax) : t);
            dzone |= (unsigned)z << (4 * k);
        }
    }
    // the middle particle's cell from the thread that has formed it
#pragma unroll
    for (int k = 0; k < PPT; k++)
        if (k * PB + tid == nblk >> 1) {
            s_mid = cu[k];
            s_zmid = (int)(dzone >> (4 * k) & 15u);
        }
    deposit_init(s_dep);
    __syncthreads();
    const PushRef ref = push_ref(s_mid, s_zmid, a.nz, a.nr, a.na);
    deposit_block<R, PPT>(a, s_dep, cu, dzone, ref, ENS ? a.qbits_m[eb.x] : a.qbits,
                          ENS ? (long long)eb.x * a.mesh : 0);
    __syncthreads();
    deposit_ranges(s_dep, a.nz, a.nr, a.jrad + (ENS ? eb.x * GH_MAXZ : 0),
                   a.krad + (ENS ? eb.x * GH_MAXZ : 0), a.rstride);
}

// (u, t) of every particle's position (after a load)
template <typename R>
__global__ __launch_bounds__(GH_BLOCK) void ut_kernel(PushArgs<R> a) {
    typedef typename Vec4<R>::T R4;
    long long i = (long long)blockIdx.x * GH_BLOCK + threadIdx.x;
    if (i >= a.n) return;
    const R4 st = a.xv[i];
    R x = st.x, y = st.y;
    R rr = sqrt(x * x + y * y), u, t;
    ut_of(x, y, rr, a.k, u, t);
    a.ut[i] = mk2(u, t);
}

// weight(jst, old) and grdacc(jst) for arbitrary positions.
template <typename R>
__global__ __launch_bounds__(GH_BLOCK) void gather_kernel(GatherArgs<R> a) {
    typedef typename Vec2<R>::T R2;
    long long i = (long long)blockIdx.x * GH_BLOCK + threadIdx.x;
    if (i >= a.n) return;
    R w[4], rr, u, t;
    int c = weight1<R>(a.x[i], a.y[i], a.nr, a.k, a.fold != 0, a.thmax, w, rr,
                       u, t);
    if (a.cell) a.cell[i] = c;
    if (a.wt)
        for (int q = 0; q < 4; q++) a.wt[4 * i + q] = w[q];
    if (a.acc) {
        int ic[4];
        corners_rs(c / a.k.na, c % a.k.na, a.k.na, ic);
        int mesh = a.nr * a.k.na;
        R ax = 0, ay = 0;
        for (int q = 0; q < 4; q++) {
            R2 f = ic[q] < mesh ? a.fld[ic[q]] : zero2<R>();
            ax = ax + f.x * w[q];
            ay = ay + f.y * w[q];
        }
        a.acc[2 * i] = ax;
        a.acc[2 * i + 1] = ay;
    }
}

// getacc for one particle of list z0 (getacc.f:35-163): grid acceleration
// interpolated with the CIC weights of its cached (u, t) (grdacc.f:40-66),
// fixed radial force, zone rescaling; none off the grid.  The push's
// operation order.
template <typename R>
__device__ __forceinline__ void getacc1(const PushArgs<R> &a, const typename Vec4<R>::T &st,
                                        const typename Vec2<R>::T &cu, int z0, R &ax,
                                        R &ay) {
    typedef typename Vec2<R>::T R2;
    ax = 0;
    ay = 0;
    if (z0 != a.nz + 1) {
        R w[4];
        int ring, spoke, ic[4];
        cic(cu.x, cu.y, a.nr, a.na, ring, spoke, w);
        corners_rs(ring, spoke, a.na, ic);
        for (int q = 0; q < 4; q++) {
            R2 f = ic[q] < a.mesh ? a.fld[ic[q]] : zero2<R>();
            ax = ax + f.x * w[q];
            ay = ay + f.y * w[q];
        }
        if (a.fixforce) {
            const R rr = sqrt(st.x * st.x + st.y * st.y);
            R fr = (R)fixforce((double)rr, a.nfr, a.fr_inv_dr, a.fr_c);
            if (fr != (R)0) {
                fr = fr / rr;
                ax = ax + fr * st.x;
                ay = ay + fr * st.y;
            }
        }
    }
    if (a.nz > 1 && z0 > 1) {
        R t = tsfac(a, z0);
        t = t * t;
        ax = t * ax;
        ay = t * ay;
    }
}

// tmcent / tmcgrp for the retarded-velocity leap-frog (tmcent.f,
// tmcgrp.f:26-36): every particle's velocity minus fac times its getacc
// acceleration.
template <typename R>
__global__ __launch_bounds__(GH_BLOCK) void tmcent_kernel(PushArgs<R> a, R fac) {
    const long long i = (long long)blockIdx.x * GH_BLOCK + threadIdx.x;
    if (i >= a.n) return;
    typename Vec4<R>::T st = a.xv[i];
    R ax, ay;
    getacc1(a, st, a.ut[i], (int)a.zone[i], ax, ay);
    st.z = st.z - fac * ax;
    st.w = st.w - fac * ay;
    a.xv[i] = st;
}

// ---- group-level routines (parity use) --------------------------------------
//
// The lib15 routines that act on one group of particles -- getacc(jst),
// stpgrp(jst) with offgrd/addoff and rezgrp(jst) -- on a caller's group (device
// copies of its arrays), in the push kernel's operation order: the push fuses
// the same steps, and massgn, for every particle of a step.

// getacc(jst) (getacc.f:35-163) at the group's positions, their (u, t) formed
// as the push's cache holds them
template <typename R>
__global__ __launch_bounds__(GH_BLOCK) void getacc_group_kernel(PushArgs<R> a,
                                                                 typename Vec2<R>::T *acc) {
    const long long i = (long long)blockIdx.x * GH_BLOCK + threadIdx.x;
    if (i >= a.n) return;
    const typename Vec4<R>::T st = a.xv[i];
    const R rr = sqrt(st.x * st.x + st.y * st.y);
    R u, t, ax, ay;
    ut_of(st.x, st.y, rr, a.k, u, t);
    getacc1(a, st, mk2(u, t), (int)a.zone[i], ax, ay);
    acc[i] = mk2(ax, ay);
}

// stpgrp(jst) (stpgrp.f:27-56) with the given accelerations, the off-grid
// test and list change (offgrd.f:55-59, addoff.f:30-70, with chstep to the
// top zone's step when offanal), and rezgrp(jst) at the current mzone
// (rezgrp.f:30-50, zoneno.f:40-55, chstep.f:22-31); zones updated in place.
template <typename R>
__global__ __launch_bounds__(GH_BLOCK) void stpgrp_group_kernel(PushArgs<R> a,
                                                                 const typename Vec2<R>::T *acc) {
    const long long i = (long long)blockIdx.x * GH_BLOCK + threadIdx.x;
    if (i >= a.n) return;
    const typename Vec4<R>::T st = a.xv[i];
    const int nz = a.nz, nlists = nz + 1, z0 = a.zone[i];
    const bool offlist = z0 == nlists;
    R ox = st.x, oy = st.y, ovx = st.z, ovy = st.w;
    R ax_ = acc[i].x, ay_ = acc[i].y;
    R nvx = ovx + ax_, nvy = ovy + ay_;
    R nx = ox + nvx, ny = oy + nvy;
    int znew = z0;
    R rnew = sqrt(nx * nx + ny * ny);
    const bool off = rnew > a.rgrid;
    if (!offlist) {
        if (off) {
            znew = nlists;
            if (a.offanal && z0 < nz) {
                const R tfac = tsfac(a, nz) / tsfac(a, z0);
                chstep(tfac, ox, oy, ovx, ovy, ax_, ay_, nx, ny, nvx, nvy);
                rnew = sqrt(nx * nx + ny * ny);
            }
        }
    } else if (!off) {
        znew = nz;
    }
    if (a.mzone > 1 && !offlist && znew <= a.mzone) {
        int kz = zone_of(a, rnew);
        if (kz > a.mzone) kz = a.mzone;
        if (kz > znew) kz = zone_of(a, sqrt(ox * ox + oy * oy));
        if (kz != znew) {
            const R tfac = tsfac(a, kz) / tsfac(a, znew);
            chstep(tfac, ox, oy, ovx, ovy, ax_, ay_, nx, ny, nvx, nvy);
            znew = kz;
        }
    }
    a.xv[i] = mk4(nx, ny, nvx, nvy);
    a.zone[i] = (uint8_t)znew;
}

// ---- global integrals (icheck, SRC/lib15/icheck.f:24-70) ------------------
//
// Per particle, in FP64: 1, x, y, vx, vy, v^2, x vy - y vx, the grid
// potential interpolated with the CIC weights of its cached (u, t) (zones
// 1..nz, when a potential is given), the fixed potential (Hermite table,
// when given).  Velocities are per zone-1 step: the stored ones carry the
// step factor of their zone (the off-grid list that of the top zone).
// centred: the velocities time-centred as icheck takes them, v + a/2 in
// the working precision (anlgrp's (v + a/2)/tfac) before the division.  A
// thread adds several particles (int_split) before its block reduces: the wavefront
// reductions of the nine FP64 sums cost as much as a particle's terms.  Each
// block writes its sums; a second pass, a block per sum, adds them in a
// fixed order, so the result does not depend on scheduling.  1e7 particles:
// kernel 207 -> 131 us, sum of the blocks 190 -> 7 us.
constexpr int NINT = 9;
constexpr int INT_SUM_BLOCK = 512;

template <typename R>
__global__ __launch_bounds__(GH_BLOCK) void integrals_kernel(PushArgs<R> a, int per, const R *pot,
                                                             const double4 *fp_c, int nfp,
                                                             double fp_dr, int centred,
                                                             double *part) {
    __shared__ double red[GH_BLOCK / 64][NINT];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    double v[NINT];
#pragma unroll
    for (int q = 0; q < NINT; q++) v[q] = 0.0;
    for (int k = 0; k < per; k++) {
        const long long i = ((long long)blockIdx.x * per + k) * GH_BLOCK + tid;
        if (i >= a.n) break;
        const int z = a.zone[i];
        if (z >= 1) {
            typename Vec4<R>::T st = a.xv[i];
            if (centred) {
                R ax, ay;
                getacc1(a, st, a.ut[i], z, ax, ay);
                st.z = st.z + (R)0.5 * ax;
                st.w = st.w + (R)0.5 * ay;
            }
            const int zs = z <= a.nz ? z : a.nz;
            const double sf = 1.0 / (double)a.nstep[zs - 1];
            const double x = st.x, y = st.y, vx = st.z * sf, vy = st.w * sf;
            v[0] += 1.0;
            v[1] += x;
            v[2] += y;
            v[3] += vx;
            v[4] += vy;
            v[5] += vx * vx + vy * vy;
            v[6] += x * vy - y * vx;
            if (pot && z <= a.nz) {
                R w[4];
                int ring, spoke, ic[4];
                const typename Vec2<R>::T cu = a.ut[i];
                cic(cu.x, cu.y, a.nr, a.na, ring, spoke, w);
                corners_rs(ring, spoke, a.na, ic);
                double ph = 0.0;
                for (int q = 0; q < 4; q++)
                    if (ic[q] < a.mesh) ph += (double)w[q] * (double)pot[ic[q]];
                v[7] += ph;
            }
            if (nfp > 0)
                v[8] += fixforce(sqrt(x * x + y * y), nfp, 1.0 / fp_dr, fp_c);
        }
    }
#pragma unroll
    for (int q = 0; q < NINT; q++) {
        const double t = wave_sum_dpp(v[q]);
        if (lane == 0) red[wave][q] = t;
    }
    __syncthreads();
    if (tid < NINT) {
        double t = 0.0;
        for (int w = 0; w < GH_BLOCK / 64; w++) t += red[w][tid];
        part[(long long)tid * gridDim.x + blockIdx.x] = t;
    }
}

// block q: out[q] = sum over blocks of part[q][b], in a fixed order
__global__ __launch_bounds__(INT_SUM_BLOCK) void integrals_sum_kernel(const double *part, int nb,
                                                                      double *out) {
    __shared__ double red[INT_SUM_BLOCK / 64];
    const int tid = threadIdx.x, q = blockIdx.x;
    double t = 0.0;
    for (int b = tid; b < nb; b += INT_SUM_BLOCK) t += part[(long long)q * nb + b];
    t = wave_sum_dpp(t);
    if ((tid & 63) == 0) red[tid >> 6] = t;
    __syncthreads();
    if (tid == 0) {
        double s = 0.0;
        for (int w = 0; w < INT_SUM_BLOCK / 64; w++) s += red[w];
        out[q] = s;
    }
}

// sort key: the cell of the particle's (u, t) shifted right by kshift so
// that keys fit 16 bits (two radix passes); off-grid particles last.
template <typename R>
__global__ __launch_bounds__(GH_BLOCK) void key_kernel(
    const typename Vec2<R>::T *__restrict__ ut,
    const uint8_t *__restrict__ zone, long long n, int nr, int na, int nz,
    int kshift, unsigned kmax, unsigned short *__restrict__ key) {
    long long i = (long long)blockIdx.x * GH_BLOCK + threadIdx.x;
    if (i >= n) return;
    unsigned k = kmax;
    int z = zone[i];
    if (z >= 1 && z <= nz) {
        R w[4];
        int ring, spoke;
        typename Vec2<R>::T c = ut[i];
        cic(c.x, c.y, nr, na, ring, spoke, w);
        k = (unsigned)(ring * na + spoke) >> kshift;
        if (k >= kmax) k = kmax - 1;
    }
    key[i] = (unsigned short)k;
}

// Ensemble sort key: (member << kbits) | the member's cell key (off-grid
// particles last within their member), so that one stable sort groups the
// members in order and cells within each.  One block per entry of the push
// block table, which never straddles two members.
template <typename R>
__global__ __launch_bounds__(GH_BLOCK) void key_ens_kernel(
    const typename Vec2<R>::T *__restrict__ ut, const uint8_t *__restrict__ zone,
    int nr, int na, int nz, int kbits, unsigned kmax, const int4 *__restrict__ blk,
    unsigned *__restrict__ key, unsigned *__restrict__ idx) {
    // block b: the push block table's (member, first particle, count)
    const int4 b = blk[blockIdx.x];
    for (int j = threadIdx.x; j < b.z; j += GH_BLOCK) {
        const long long i = (long long)b.y + j;
        unsigned k = kmax;
        const int z = zone[i];
        if (z >= 1 && z <= nz) {
            R w[4];
            int ring, spoke;
            const typename Vec2<R>::T c = ut[i];
            cic(c.x, c.y, nr, na, ring, spoke, w);
            k = (unsigned)(ring * na + spoke);
            if (k >= kmax) k = kmax - 1;
        }
        key[i] = ((unsigned)b.x << kbits) | k;
        idx[i] = (unsigned)i;
    }
}

// one pass moving every particle array to sorted order
template <typename R> struct PermArgs {
    const typename Vec4<R>::T *xv_in;
    typename Vec4<R>::T *xv_out;
    const typename Vec2<R>::T *ut_in;
    typename Vec2<R>::T *ut_out;
    const uint8_t *zin;
    uint8_t *zout;
    const unsigned *iin;
    unsigned *iout;
    const unsigned *perm;
    long long n;
    const typename Vec2<R>::T *lo_in;   // compensated positions' low words, or NULL
    typename Vec2<R>::T *lo_out;
};

template <typename R>
__global__ __launch_bounds__(GH_BLOCK) void permute_all_kernel(PermArgs<R> p) {
    typedef typename Vec2<R>::T R2;
    const long long i = (long long)blockIdx.x * GH_BLOCK + threadIdx.x;
    if (i >= p.n) return;
    const unsigned s = p.perm[i];
    const typename Vec4<R>::T xv = p.xv_in[s];
    const R2 ut = p.ut_in[s];
    const uint8_t z = p.zin[s];
    const unsigned id = p.iin[s];
    R2 lo = mk2((R)0, (R)0);
    if (p.lo_in) lo = p.lo_in[s];
    p.xv_out[i] = xv;
    p.ut_out[i] = ut;
    p.zout[i] = z;
    p.iout[i] = id;
    if (p.lo_in) p.lo_out[i] = lo;
}

// load: planar host arrays (x, y, vx, vy, es*n bytes each, staged one after
// another in s) -> interleaved storage; ids = load order
template <typename R>
__global__ __launch_bounds__(GH_BLOCK) void interleave_kernel(const R *__restrict__ s,
                                                              typename Vec4<R>::T *__restrict__ xv,
                                                              unsigned *__restrict__ id,
                                                              long long n) {
    const long long i = (long long)blockIdx.x * GH_BLOCK + threadIdx.x;
    if (i >= n) return;
    typename Vec4<R>::T v;
    v.x = s[i];
    v.y = s[n + i];
    v.z = s[2 * n + i];
    v.w = s[3 * n + i];
    xv[i] = v;
    id[i] = (unsigned)i;
}

// Unload: interleaved storage -> planar arrays in load order, zones widened to
// int32.  Written where each particle belongs, its five values touch five lines
// each used for four bytes (1e7: 630 us); so only its place is written (inv),
// and the records, a line each, are read in load order: 137 + 362 us.  A small
// set stays in the L2, and the second launch costs more than it saves: below
// UNLOAD_GATHER particles each value is written where it belongs (2e4: 3.7 us
// against 2.0 + 2.3 and the gap between the launches; 1e5: 7.0 against 2.7 + 2.9
// and the gap).
__global__ __launch_bounds__(GH_BLOCK) void inverse_order_kernel(const unsigned *__restrict__ id,
                                                                 unsigned *__restrict__ inv,
                                                                 long long n) {
    const long long i = (long long)blockIdx.x * GH_BLOCK + threadIdx.x;
    if (i < n) inv[id[i]] = (unsigned)i;
}

// ord: GATHER the places inv, else the load-order ids
template <typename R, bool GATHER>
__global__ __launch_bounds__(GH_BLOCK) void deinterleave_kernel(const typename Vec4<R>::T *__restrict__ xv,
                                                                const uint8_t *__restrict__ zone,
                                                                const unsigned *__restrict__ ord,
                                                                R *__restrict__ d,
                                                                int *__restrict__ iz, long long n) {
    const long long t = (long long)blockIdx.x * GH_BLOCK + threadIdx.x;
    if (t >= n) return;
    const long long o = ord[t], i = GATHER ? o : t, p = GATHER ? t : o;
    const typename Vec4<R>::T v = xv[i];
    const int z = zone[i];
    d[p] = v.x;
    d[n + p] = v.y;
    d[2 * n + p] = v.z;
    d[3 * n + p] = v.w;
    iz[p] = z;
}

// ---- host launchers ---------------------------------------------------------

static inline unsigned nblocks(long long n, long long per) {
    return (unsigned)((n + per - 1) / per);
}

template <typename R, bool COMP, int PPT>
static void launch_push_c(const PushArgs<R> &a, hipStream_t s) {
    if (a.blk)
        hipLaunchKernelGGL(HIP_KERNEL_NAME(push_kernel<R, true, COMP, PPT>), dim3(a.nblocks),
                           dim3(PB), 0, s, a);
    else
        hipLaunchKernelGGL(HIP_KERNEL_NAME(push_kernel<R, false, COMP, PPT>),
                           dim3(nblocks(a.n, PB * PPT)), dim3(PB), 0, s, a);
}

// a.ppt: push_ppt's choice (an ensemble's block table is made for it)
template <typename R>
hipError_t launch_push(const PushArgs<R> &a, hipStream_t s) {
    if (a.n <= 0) return hipSuccess;
    if constexpr (sizeof(R) == 4) {
        if (a.ppt == 1) {
            if (a.xlo) launch_push_c<R, true, 1>(a, s);
            else launch_push_c<R, false, 1>(a, s);
        } else {
            if (a.xlo) launch_push_c<R, true, 4>(a, s);
            else launch_push_c<R, false, 4>(a, s);
        }
    } else {
        if (a.xlo) return hipErrorInvalidValue;   // compensated positions are FP32 only
        if (a.ppt == 1) launch_push_c<R, false, 1>(a, s);
        else if (a.ppt == 2 && !a.blk)
            hipLaunchKernelGGL(HIP_KERNEL_NAME(push_kernel<R, false, false, 2>),
                               dim3(nblocks(a.n, PB * 2)), dim3(PB), 0, s, a);
        else return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <typename R, int PPT>
static void launch_massgn_p(const PushArgs<R> &a, hipStream_t s) {
    if (a.blk)
        hipLaunchKernelGGL(HIP_KERNEL_NAME(massgn_kernel<R, true, PPT>), dim3(a.nblocks), dim3(PB),
                           0, s, a);
    else
        hipLaunchKernelGGL(HIP_KERNEL_NAME(massgn_kernel<R, false, PPT>),
                           dim3(nblocks(a.n, PB * PPT)), dim3(PB), 0, s, a);
}

template <typename R>
hipError_t launch_massgn(const PushArgs<R> &a, hipStream_t s) {
    if (a.n <= 0) return hipSuccess;
    if (a.ppt == 1) launch_massgn_p<R, 1>(a, s);
    else if constexpr (sizeof(R) == 4) launch_massgn_p<R, 4>(a, s);
    else if (a.ppt == 2 && !a.blk)
        hipLaunchKernelGGL(HIP_KERNEL_NAME(massgn_kernel<R, false, 2>), dim3(nblocks(a.n, PB * 2)),
                           dim3(PB), 0, s, a);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

template <typename R>
hipError_t launch_getacc_group(const PushArgs<R> &a, typename Vec2<R>::T *acc, hipStream_t s) {
    if (a.n <= 0) return hipSuccess;
    hipLaunchKernelGGL(getacc_group_kernel<R>, dim3(nblocks(a.n, GH_BLOCK)), dim3(GH_BLOCK), 0,
                       s, a, acc);
    return hipGetLastError();
}

template <typename R>
hipError_t launch_stpgrp_group(const PushArgs<R> &a, const typename Vec2<R>::T *acc,
                               hipStream_t s) {
    if (a.n <= 0) return hipSuccess;
    hipLaunchKernelGGL(stpgrp_group_kernel<R>, dim3(nblocks(a.n, GH_BLOCK)), dim3(GH_BLOCK), 0,
                       s, a, acc);
    return hipGetLastError();
}

template <typename R>
hipError_t launch_ut(const PushArgs<R> &a, hipStream_t s) {
    if (a.n <= 0) return hipSuccess;
    hipLaunchKernelGGL(ut_kernel<R>, dim3(nblocks(a.n, GH_BLOCK)),
                       dim3(GH_BLOCK), 0, s, a);
    return hipGetLastError();
}

template <typename R>
hipError_t launch_gather(const GatherArgs<R> &a, hipStream_t s) {
    if (a.n <= 0) return hipSuccess;
    hipLaunchKernelGGL(gather_kernel<R>, dim3(nblocks(a.n, GH_BLOCK)),
                       dim3(GH_BLOCK), 0, s, a);
    return hipGetLastError();
}

template <typename R>
hipError_t launch_integrals(const PushArgs<R> &a, const R *pot, const double4 *fp_c,
                            int nfp, double fp_dr, int centred,
                            double *part, double *out, hipStream_t s) {
    const IntSplit sp = int_split(a.n, GH_BLOCK);
    const unsigned nb = (unsigned)sp.nb;
    if (nb)
        hipLaunchKernelGGL(integrals_kernel<R>, dim3(nb), dim3(GH_BLOCK), 0, s, a, sp.per, pot,
                           fp_c, nfp, fp_dr, centred, part);
    hipLaunchKernelGGL(integrals_sum_kernel, dim3(NINT), dim3(INT_SUM_BLOCK), 0, s,
                       (const double *)part, (int)nb, out);
    return hipGetLastError();
}

template <typename R>
hipError_t launch_tmcent(const PushArgs<R> &a, R fac, hipStream_t s) {
    if (a.n <= 0) return hipSuccess;
    hipLaunchKernelGGL(tmcent_kernel<R>, dim3(nblocks(a.n, GH_BLOCK)),
                       dim3(GH_BLOCK), 0, s, a, fac);
    return hipGetLastError();
}

template <typename R>
hipError_t launch_key(const typename Vec2<R>::T *ut, const uint8_t *zone,
                      long long n, int nr, int na, int nz, int kshift,
                      unsigned kmax, unsigned short *key, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(key_kernel<R>, dim3(nblocks(n, GH_BLOCK)), dim3(GH_BLOCK),
                       0, s, ut, zone, n, nr, na, nz, kshift, kmax, key);
    return hipGetLastError();
}

template <typename R>
hipError_t launch_key_ens(const typename Vec2<R>::T *ut, const uint8_t *zone, int nblk,
                          int nr, int na, int nz, int kbits, unsigned kmax, const int4 *blk,
                          unsigned *key, unsigned *idx, hipStream_t s) {
    if (nblk <= 0) return hipSuccess;
    hipLaunchKernelGGL(key_ens_kernel<R>, dim3(nblk), dim3(GH_BLOCK), 0, s, ut, zone, nr, na,
                       nz, kbits, kmax, blk, key, idx);
    return hipGetLastError();
}

template <typename R>
hipError_t launch_interleave(const R *stage, typename Vec4<R>::T *xv, unsigned *id, long long n,
                             hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(interleave_kernel<R>, dim3(nblocks(n, GH_BLOCK)), dim3(GH_BLOCK), 0, s,
                       stage, xv, id, n);
    return hipGetLastError();
}

hipError_t launch_inverse_order(const unsigned *id, unsigned *inv, long long n, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(inverse_order_kernel, dim3(nblocks(n, GH_BLOCK)), dim3(GH_BLOCK), 0, s, id,
                       inv, n);
    return hipGetLastError();
}

// inv: scratch of n words
template <typename R>
hipError_t launch_deinterleave(const typename Vec4<R>::T *xv, const uint8_t *zone,
                               const unsigned *id, unsigned *inv, R *stage, int *iz, long long n,
                               hipStream_t s) {
    if (n <= 0) return hipSuccess;
    const dim3 grid(nblocks(n, GH_BLOCK)), block(GH_BLOCK);
    if (n < UNLOAD_GATHER) {
        hipLaunchKernelGGL(HIP_KERNEL_NAME(deinterleave_kernel<R, false>), grid, block, 0, s, xv,
                           zone, id, stage, iz, n);
        return hipGetLastError();
    }
    hipError_t e = launch_inverse_order(id, inv, n, s);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(HIP_KERNEL_NAME(deinterleave_kernel<R, true>), grid, block, 0, s, xv, zone,
                       (const unsigned *)inv, stage, iz, n);
    return hipGetLastError();
}

template <typename R>
hipError_t launch_permute_all(const PermArgs<R> &p, hipStream_t s) {
    if (p.n <= 0) return hipSuccess;
    hipLaunchKernelGGL(permute_all_kernel<R>, dim3(nblocks(p.n, GH_BLOCK)),
                       dim3(GH_BLOCK), 0, s, p);
    return hipGetLastError();
}

#define GH_INST(R)                                                            \
    template hipError_t launch_push<R>(const PushArgs<R> &, hipStream_t);     \
    template hipError_t launch_massgn<R>(const PushArgs<R> &, hipStream_t);   \
    template hipError_t launch_ut<R>(const PushArgs<R> &, hipStream_t);       \
    template hipError_t launch_getacc_group<R>(const PushArgs<R> &,           \
                                               typename Vec2<R>::T *, hipStream_t); \
    template hipError_t launch_stpgrp_group<R>(const PushArgs<R> &,           \
                                               const typename Vec2<R>::T *,   \
                                               hipStream_t);                  \
    template hipError_t launch_gather<R>(const GatherArgs<R> &, hipStream_t); \
    template hipError_t launch_tmcent<R>(const PushArgs<R> &, R, hipStream_t); \
    template hipError_t launch_integrals<R>(const PushArgs<R> &, const R *,     \
                                            const double4 *, int, double, int,   \
                                            double *, double *, hipStream_t);    \
    template hipError_t launch_key<R>(const typename Vec2<R>::T *,           \
                                      const uint8_t *, long long, int, int,   \
                                      int, int, unsigned, unsigned short *,   \
                                      hipStream_t);                           \
    template hipError_t launch_key_ens<R>(const typename Vec2<R>::T *, const uint8_t *, \
                                          int, int, int, int, int, unsigned,          \
                                          const int4 *, unsigned *, unsigned *,       \
                                          hipStream_t);                               \
    template hipError_t launch_permute_all<R>(const PermArgs<R> &, hipStream_t); \
    template hipError_t launch_interleave<R>(const R *, typename Vec4<R>::T *, unsigned *, \
                                             long long, hipStream_t);                      \
    template hipError_t launch_deinterleave<R>(const typename Vec4<R>::T *, const uint8_t *, \
                                               const unsigned *, unsigned *, R *, int *,     \
                                               long long, hipStream_t);
GH_INST(float)
GH_INST(double)

}  // namespace gh
