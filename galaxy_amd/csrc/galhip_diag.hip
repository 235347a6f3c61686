// galhip_diag.hip -- analysis-step diagnostics of the particles: the
// log-spiral coefficients of lgspia (SRC/lib15/lgspia.f:44-110), normalised
// by the population as phyprp does (SRC/lib15/phyprp.f:182-197).
//
// For harmonic index im = 1..nm and pitch index j = 1..np,
//   A[j][im] = sum over particles of exp(i im (nsect theta + k_j a)) / count,
//   a = nsect ln(R / lscale) / 4,
// over the particles on the grid (and off it when offanal), equal masses.
// Each particle forms e^{i nsect theta} from (x + i y) / R and e^{i a}, then
// the powers and pitch factors by complex products in FP64, as the
// reference's recurrences do: index j = jc + k (jc = np/2 + 1, k >= 0)
// takes e^{i k im a}, its mirror np + 1 - j the conjugate (for even np
// index np/2 is left at 0, as in the reference).
//
// The sums take 8 FP64 operations per coefficient pair and particle and read
// 9 bytes (FP32) per particle.  The latency of dependent FP64 products bounds
// them: VALU issue is busy half of the time, with six wavefronts on a CU (1150
// instructions per particle at 25 pitches x 6 harmonics).  A wavefront owns one
// harmonic and a run of pitches for the whole pass, so its sums stay in
// registers (four products per pitch and its mirror) and are reduced over
// the lanes once at the end; the particles' e^{i nsect theta} and e^{i a}
// are formed once per block, a tile at a time, and handed to the wavefronts
// through LDS.  25 pitches x 6 harmonics of 1e7 particles: 0.64 ms against
// 6.36 ms with each coefficient reduced over the wavefront per particle.
//
// Sums are deterministic: the order depends only on n, np and nm.
#include "galhip_ctx.h"

#include <algorithm>

namespace gh {

constexpr int LG_MAXQ = 512;     // np * nm coefficients at most
constexpr int LG_MAXW = 8;       // wavefronts per block at most
constexpr int LG_HARM = 16;      // harmonics per wavefront at most without pitches
constexpr int LG_SUM_BLOCK = 256;

// How the coefficients are dealt out: a unit is harmonic im with len pitch
// offsets (unit u: im = u / nch + 1, offsets (u % nch) len + 1 ..); without
// pitches (np <= 2) a unit is len harmonics from u len + 1 on.  A block has one
// wavefront per unit of its group.
struct LgPlan {
    int kmax;      // largest pitch offset
    int nch, len;  // runs per harmonic (of the harmonics) and their length
    int units;
    int groups;    // gridDim.y
    int waves;     // wavefronts per block
    int nb;        // gridDim.x
};

// Runs of at most 12 offsets: 48 FP64 sums (96 VGPRs) per lane, three
// wavefronts per SIMD; 8 of the 168 registers go to scratch (36 bytes) all the same.
// Runs of 8 and 4 offsets do not spill, but form the tile again for more groups: 1e7
// particles, 25 pitches x 6 harmonics 0.64 ms, 1.17 and 1.35.  Without pitches a harmonic of its own per wavefront spends
// its time on forming z^im and, beyond eight harmonics, the tile again for every
// group: runs of LG_HARM harmonics, each the product of the last one and z (4e6
// particles, 512 harmonics: 27.0 ms one by one, 2.14 so; 64: 2.35 and 0.25;
// before the wavefronts had units 11.1 and 2.08).
static LgPlan lg_plan(long long n, int np, int nm) {
    LgPlan p;
    p.kmax = np - (np / 2 + 1);
    const int all = p.kmax ? p.kmax : nm, most_len = p.kmax ? 12 : LG_HARM;
    p.nch = (all + most_len - 1) / most_len;
    p.len = (all + p.nch - 1) / p.nch;
    p.units = p.kmax ? nm * p.nch : (nm + p.len - 1) / p.len;
    p.groups = (p.units + LG_MAXW - 1) / LG_MAXW;
    p.waves = (p.units + p.groups - 1) / p.groups;
    // twelve wavefronts per CU (three per SIMD) over 256 CUs
    const long long tiles = (n + 64 * p.waves - 1) / (64 * p.waves);
    const long long most = std::max(1, 256 * 12 / (p.waves * p.groups));
    p.nb = (int)std::max<long long>(1, std::min(tiles, most));
    return p;
}

// z^e for e >= 1 by squaring
__device__ __forceinline__ void cpow(double zr, double zi, int e, double &pr, double &pi) {
    while (!(e & 1)) {
        const double t = fma(zr, zr, -(zi * zi));
        zi = 2.0 * (zr * zi);
        zr = t;
        e >>= 1;
    }
    pr = zr;
    pi = zi;
    while (e >>= 1) {
        double t = fma(zr, zr, -(zi * zi));
        zi = 2.0 * (zr * zi);
        zr = t;
        if (e & 1) {
            t = fma(pr, zr, -(pi * zi));
            pi = fma(pi, zr, pr * zi);
            pr = t;
        }
    }
}

// A particle's e^{i nsect theta} and, if PITCH, e^{i a}; false if it is not among
// those summed (its factors are left as they were).
template <typename R, bool PITCH>
__device__ __forceinline__ bool lg_factors(const typename Vec4<R>::T *__restrict__ xv, int ps,
                                           const uint8_t *__restrict__ zone, long long i, int nz,
                                           int offanal, int nsect, double inv_lscale, double &c1,
                                           double &s1, double &ca, double &sa) {
    const int z = zone[i];
    const bool inc = z >= 1 && (z <= nz || (offanal && z == nz + 1));
    // x, y lead the particle's data
    const typename Vec2<R>::T p = *reinterpret_cast<const typename Vec2<R>::T *>(xv + i * ps);
    const double x = (double)p.x, y = (double)p.y;
    const double rc = sqrt(x * x + y * y);
    if (!(inc && rc > 0.0)) return false;
    const double cx = x / rc, sy = y / rc;
    c1 = cx;
    s1 = sy;
    for (int m = 2; m <= nsect; m++) {
        const double t = c1 * cx - s1 * sy;
        s1 = s1 * cx + c1 * sy;
        c1 = t;
    }
    if (PITCH) sincos(0.25 * (double)nsect * log(rc * inv_lscale), &sa, &ca);
    return true;
}

// The block's particle count, by the blocks of the first group.
__device__ __forceinline__ void lg_count(double cnt, double *s_cnt, double *out) {
    const int tid = threadIdx.x;
    cnt = wave_sum_dpp(cnt);
    if ((tid & 63) == 0) s_cnt[tid >> 6] = cnt;
    __syncthreads();
    if (tid == 0) {
        double v = 0.0;
        for (int k = 0; k < (int)blockDim.x / 64; k++) v += s_cnt[k];
        *out = v;
    }
}

// No pitches (np 1 or 2): a wavefront's harmonics in turn.
template <typename R>
__global__ __launch_bounds__(64 * LG_MAXW, 3) void lgsp_harm_kernel(
    const typename Vec4<R>::T *__restrict__ xv, int ps, const uint8_t *__restrict__ zone,
    long long n, int nz, int offanal, int nsect, int np, int nm, LgPlan pl,
    double *__restrict__ part) {
    __shared__ double2 s_z[64 * LG_MAXW];
    __shared__ double s_cnt[LG_MAXW];
    const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, T = blockDim.x;
    const int unit = blockIdx.y * pl.waves + w;
    const bool work = unit < pl.units;         // uniform over the wavefront
    const int im0 = work ? unit * pl.len + 1 : 1;
    double sr[LG_HARM], si[LG_HARM], cnt = 0.0;
#pragma unroll
    for (int h = 0; h < LG_HARM; h++) sr[h] = si[h] = 0.0;
    const long long stride = (long long)gridDim.x * T;
    for (long long base = (long long)blockIdx.x * T; base < n; base += stride) {
        const long long i = base + tid;
        double c1 = 0.0, s1 = 0.0, ca, sa;
        if (i < n && lg_factors<R, false>(xv, ps, zone, i, nz, offanal, nsect, 1.0, c1, s1, ca, sa))
            cnt += 1.0;
        __syncthreads();   // the last tile has been read
        s_z[tid] = make_double2(c1, s1);
        __syncthreads();
        if (work)
            for (int e = lane; e < T; e += 64) {
                const double2 z = s_z[e];
                double zr, zi;
                cpow(z.x, z.y, im0, zr, zi);
#pragma unroll
                for (int h = 0; h < LG_HARM; h++) {
                    if (h >= pl.len) break;    // uniform
                    sr[h] += zr;
                    si[h] += zi;
                    const double t = fma(zr, z.x, -(zi * z.y));
                    zi = fma(zi, z.x, zr * z.y);
                    zr = t;
                }
            }
    }
    const size_t nb = gridDim.x, b = blockIdx.x;
    const int nq = np * nm;
#pragma unroll
    for (int h = 0; h < LG_HARM; h++) {
        if (!work || h >= pl.len || im0 + h > nm) break;
        const double vr = wave_sum_dpp(sr[h]), vi = wave_sum_dpp(si[h]);
        if (lane) continue;
        // the last pitch index; the first of two holds none
        const int q = (np - 1) * nm + im0 + h - 1;
        part[(size_t)q * nb + b] = vr;
        part[(size_t)(nq + q) * nb + b] = vi;
        if (np == 2) {
            part[(size_t)(q - nm) * nb + b] = 0.0;
            part[(size_t)(nq + q - nm) * nb + b] = 0.0;
        }
    }
    if (blockIdx.y == 0) lg_count(cnt, s_cnt, part + 2 * (size_t)nq * nb + b);
}

// part[q][block]: q = [cos parts][sin parts][count].  KC: pitch offsets of
// a run at most.
template <typename R, int KC>
__global__ __launch_bounds__(64 * LG_MAXW, 3) void lgsp_part_kernel(
    const typename Vec4<R>::T *__restrict__ xv, int ps, const uint8_t *__restrict__ zone,
    long long n, int nz, int offanal, int nsect, int np, int nm, double inv_lscale, LgPlan pl,
    double *__restrict__ part) {
    __shared__ double2 s_z[64 * LG_MAXW], s_w[64 * LG_MAXW];
    __shared__ double s_cnt[LG_MAXW];
    const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, T = blockDim.x;
    const int nq = np * nm, jc = np / 2 + 1;   // 1-based centre (offset 0)
    const int unit = blockIdx.y * pl.waves + w;
    const bool work = unit < pl.units;         // uniform over the wavefront
    const int im = work ? unit / pl.nch + 1 : 1;
    const int k0 = work ? (unit - (im - 1) * pl.nch) * pl.len + 1 : 1;
    // gr zr, gi zi, gi zr, gr zi summed for offsets k0 ..; z itself
    double p1[KC], p2[KC], p3[KC], p4[KC], zsr = 0.0, zsi = 0.0, cnt = 0.0;
#pragma unroll
    for (int k = 0; k < KC; k++) p1[k] = p2[k] = p3[k] = p4[k] = 0.0;
    const long long stride = (long long)gridDim.x * T;
    for (long long base = (long long)blockIdx.x * T; base < n; base += stride) {
        const long long i = base + tid;
        double c1 = 0.0, s1 = 0.0, ca = 1.0, sa = 0.0;
        if (i < n && lg_factors<R, true>(xv, ps, zone, i, nz, offanal, nsect, inv_lscale, c1, s1, ca, sa))
            cnt += 1.0;
        __syncthreads();   // the last tile has been read
        s_z[tid] = make_double2(c1, s1);
        s_w[tid] = make_double2(ca, sa);
        __syncthreads();
        if (work)
            for (int e = lane; e < T; e += 64) {
                double zr, zi, wr, wi, gr = 1.0, gi = 0.0;
                cpow(s_z[e].x, s_z[e].y, im, zr, zi);
                cpow(s_w[e].x, s_w[e].y, im, wr, wi);
                if (k0 > 1) cpow(wr, wi, k0 - 1, gr, gi);
                zsr += zr;
                zsi += zi;
#pragma unroll
                for (int k = 0; k < KC; k++) {
                    const double t = fma(gr, wr, -(gi * wi));
                    gi = fma(gi, wr, gr * wi);
                    gr = t;
                    p1[k] = fma(gr, zr, p1[k]);
                    p2[k] = fma(gi, zi, p2[k]);
                    p3[k] = fma(gi, zr, p3[k]);
                    p4[k] = fma(gr, zi, p4[k]);
                }
            }
    }
    const size_t nb = gridDim.x, b = blockIdx.x;
    if (work) {
        // q = (j - 1) nm + im - 1 for pitch index j
        const double r0 = wave_sum_dpp(zsr), i0 = wave_sum_dpp(zsi);
        if (lane == 0 && k0 == 1) {
            const int q = (jc - 1) * nm + im - 1;
            part[(size_t)q * nb + b] = r0;
            part[(size_t)(nq + q) * nb + b] = i0;
        }
        if (lane == 0 && k0 == 1 && np % 2 == 0) {   // index np / 2 holds no pitch
            const int q = (np / 2 - 1) * nm + im - 1;
            part[(size_t)q * nb + b] = 0.0;
            part[(size_t)(nq + q) * nb + b] = 0.0;
        }
#pragma unroll
        for (int k = 0; k < KC; k++) {
            if (k >= pl.len || k0 + k > pl.kmax) break;
            const double a1 = wave_sum_dpp(p1[k]), a2 = wave_sum_dpp(p2[k]);
            const double a3 = wave_sum_dpp(p3[k]), a4 = wave_sum_dpp(p4[k]);
            if (lane == 0) {
                // offset k0 + k: g z; its mirror: conj(g) z
                const int qp = (jc + k0 + k - 1) * nm + im - 1;
                const int qm = (np - jc - k0 - k) * nm + im - 1;
                part[(size_t)qp * nb + b] = a1 - a2;
                part[(size_t)(nq + qp) * nb + b] = a3 + a4;
                part[(size_t)qm * nb + b] = a1 + a2;
                part[(size_t)(nq + qm) * nb + b] = a4 - a3;
            }
        }
    }
    if (blockIdx.y == 0) lg_count(cnt, s_cnt, part + 2 * (size_t)nq * nb + b);
}

// Fixed-order sum of row[0 .. nb) over the block.
__device__ __forceinline__ double lg_row_sum(const double *__restrict__ row, int nb,
                                             double *red) {
    const int tid = threadIdx.x;
    double v = 0.0;
    for (int b = tid; b < nb; b += LG_SUM_BLOCK) v += row[b];
    v = wave_sum_dpp(v);
    __syncthreads();
    if ((tid & 63) == 0) red[tid >> 6] = v;
    __syncthreads();
    v = red[0];
    for (int k = 1; k < LG_SUM_BLOCK / 64; k++) v += red[k];
    return v;
}

// block q: out[q] = (sum of the blocks' partials of q) / count
__global__ __launch_bounds__(LG_SUM_BLOCK) void lgsp_sum_kernel(const double *__restrict__ part,
                                                                 int nb, int nq,
                                                                 double *__restrict__ out) {
    __shared__ double red[LG_SUM_BLOCK / 64];
    const double v = lg_row_sum(part + (size_t)blockIdx.x * nb, nb, red);
    const double cnt = lg_row_sum(part + 2 * (size_t)nq * nb, nb, red);
    if (threadIdx.x == 0) out[blockIdx.x] = cnt > 0.0 ? v * (1.0 / cnt) : 0.0;
}

template <typename R, int KC>
static void launch_lgsp_part(const void *xv, int ps, const uint8_t *zone, long long n, int nz,
                             int offanal, int nsect, int np, int nm, double lscale,
                             const LgPlan &pl, double *part, hipStream_t s) {
    hipLaunchKernelGGL(HIP_KERNEL_NAME(lgsp_part_kernel<R, KC>), dim3(pl.nb, pl.groups),
                       dim3(64 * pl.waves), 0, s, (const typename Vec4<R>::T *)xv, ps, zone, n,
                       nz, offanal, nsect, np, nm, 1.0 / lscale, pl, part);
}

template <typename R>
hipError_t launch_lgspia(const void *xv, int ps, const uint8_t *zone, long long n, int nz,
                         int offanal, int nsect, int np, int nm, double lscale, double *part,
                         double *out, hipStream_t s) {
    if (np * nm > LG_MAXQ) return hipErrorInvalidValue;
    const LgPlan pl = lg_plan(n, np, nm);
    if (pl.kmax == 0)
        hipLaunchKernelGGL(lgsp_harm_kernel<R>, dim3(pl.nb, pl.groups), dim3(64 * pl.waves), 0, s,
                           (const typename Vec4<R>::T *)xv, ps, zone, n, nz, offanal, nsect, np, nm,
                           pl, part);
    else if (pl.len <= 4)
        launch_lgsp_part<R, 4>(xv, ps, zone, n, nz, offanal, nsect, np, nm, lscale, pl, part, s);
    else if (pl.len <= 8)
        launch_lgsp_part<R, 8>(xv, ps, zone, n, nz, offanal, nsect, np, nm, lscale, pl, part, s);
    else
        launch_lgsp_part<R, 12>(xv, ps, zone, n, nz, offanal, nsect, np, nm, lscale, pl, part, s);
    hipLaunchKernelGGL(lgsp_sum_kernel, dim3(2 * np * nm), dim3(LG_SUM_BLOCK), 0, s,
                       (const double *)part, pl.nb, np * nm, out);
    return hipGetLastError();
}

}  // namespace gh

using namespace gh;

extern "C" int galhip_lgspia(galhip_ctx *c, int32_t np, int32_t nm, double lscale,
                             double *out) {
    if (!c || !out) return gh_fail(GALHIP_EINVAL, "null argument");
    if (np < 1 || nm < 1 || (long long)np * nm > LG_MAXQ)
        return gh_fail(GALHIP_EINVAL, "LGSPIA: np x nm = %d x %d out of range (at most %d)", np,
                       nm, LG_MAXQ);
    if (!(lscale > 0.0)) return gh_fail(GALHIP_EINVAL, "LGSPIA: lscale must be positive");
    const int nq = np * nm;
    double *part = nullptr, *dout = nullptr;
    int nbmax = 1;
    for (int m = 0; m < c->nmem; m++) {
        const long long nm_ = c->ens ? c->m_off[m + 1] - c->m_off[m] : c->n;
        nbmax = std::max(nbmax, lg_plan(nm_, np, nm).nb);
    }
    int rc = dalloc(&part, sizeof(double) * (size_t)nbmax * (2 * nq + 1)) |
             dalloc(&dout, sizeof(double) * (size_t)c->nmem * 2 * nq);
    if (!rc) {
        hipError_t e = hipSuccess;
        const size_t esz = c->prec == GALHIP_FP32 ? sizeof(float4) : sizeof(double4);
        // 4-vectors per particle: (x, y, vx, vy) on p2d, a two-vector record on p3d
        const int ps = c->p3d ? 2 : 1;
        for (int m = 0; m < c->nmem && e == hipSuccess; m++) {
            const long long off = c->ens ? c->m_off[m] : 0;
            const long long cnt = c->ens ? c->m_off[m + 1] - off : c->n;
            const void *xv = (const char *)c->xv + (size_t)off * ps * esz;
            const uint8_t *zn = c->zone + off;
            e = c->prec == GALHIP_FP32
                    ? launch_lgspia<float>(xv, ps, zn, cnt, c->nz, c->offanal, c->nsect, np,
                                           nm, lscale, part,
                                           dout + 2 * nq * m, c->s)
                    : launch_lgspia<double>(xv, ps, zn, cnt, c->nz, c->offanal, c->nsect, np,
                                            nm, lscale, part,
                                            dout + 2 * nq * m, c->s);
        }
        if (e == hipSuccess)
            e = hipMemcpyAsync(out, dout, sizeof(double) * (size_t)c->nmem * 2 * nq,
                               hipMemcpyDeviceToHost, c->s);
        if (e == hipSuccess) e = hipStreamSynchronize(c->s);
        if (e != hipSuccess) rc = gh_fail(GALHIP_EHIP, "lgspia: %s", hipGetErrorString(e));
    }
    dfree(part);
    dfree(dout);
    return rc;
}
