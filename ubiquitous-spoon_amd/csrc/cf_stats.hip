/*
 * cf_stats.hip -- plane statistics of a run's fields on the device: the
 * x-y means, correlations and central moments of get.c:100-174 and
 * get_xy_avg (get.c:281-307), and the one-dimensional cross-spectra of
 * get_xy_spec (get.c:5-97), at every interior level.
 *
 * Fields are in the device layout [nz][ny][nx]: a level is one contiguous
 * plane.  Plane sums are two-stage and in a fixed order (per workgroup a
 * strided thread sum and a tree, then a tree over the workgroups'
 * partials), so a statistic is bitwise repeatable.
 */
#include "cf_kernels.h"

#include <hip/hip_runtime.h>

/* a level's sum from its nbl <= 64 partials, in every lane of the wave */
static __device__ __forceinline__ double level_sum(const double *part, int k, int nbl)
{
    const int lane = threadIdx.x & 63;
    return wave_sum(lane < nbl ? part[(size_t) k * nbl + lane] : 0.0);
}

/* Plane statistics take two passes, since a central sum needs the means:
 * k_stat_sum leaves each workgroup's partial sum, k_stat_central's
 * workgroups sum those themselves, k_stat_finish scales the last ones.  The
 * launches bound them (the passes read what the caches hold), so a
 * correlation is three of them with both means in the first: 4.4 + 4.3 + 2.8
 * us at 128 x 97 x 128, in place of 6.6 x 3 + 7.7 x 3 with a finish after
 * each sum and 64 workgroups a level.
 * Partials of (field blockIdx.z, level, workgroup). */
template <typename T>
__global__ void __launch_bounds__(256) k_stat_sum(const T *a, const T *b, int P, int nbl, double *part)
{
    const int k = blockIdx.y, bl = blockIdx.x, nz = gridDim.y;
    const T *ak = (blockIdx.z ? b : a) + (size_t) k * P;
    const int per = (P + nbl - 1) / nbl;
    const int lo = bl * per, hi = lo + per < P ? lo + per : P;
    double s = 0.0;
#pragma unroll 4
    for (int t = lo + (int) threadIdx.x; t < hi; t += 256) s += (double) ak[t];
    __shared__ double red[4];
    s = block_sum<4>(s, red);
    if (threadIdx.x == 0) part[((size_t) blockIdx.z * nz + k) * nbl + bl] = s;
}

/* MODE 1: sum of (a - ma)(b - mb), 2: sum of (a - ma)^en, the means being
 * scale times the sums of pa and pb */
template <typename T, int MODE>
__global__ void __launch_bounds__(256) k_stat_central(const T *a, const T *b, const double *pa, const double *pb,
                                                      double scale, double en, int P, int nbl, double *part)
{
    const int k = blockIdx.y, bl = blockIdx.x;
    const T *ak = a + (size_t) k * P;
    const T *bk = MODE == 1 ? b + (size_t) k * P : nullptr;
    const double mak = scale * level_sum(pa, k, nbl);
    const double mbk = MODE == 1 ? scale * level_sum(pb, k, nbl) : 0.0;
    const int per = (P + nbl - 1) / nbl;
    const int lo = bl * per, hi = lo + per < P ? lo + per : P;
    constexpr int U = MODE == 1 ? 4 : 1;      /* pow fills the registers */
    double s = 0.0;
#pragma unroll U
    for (int t = lo + (int) threadIdx.x; t < hi; t += 256) {
        const double x = (double) ak[t];
        if (MODE == 1) s += (x - mak) * ((double) bk[t] - mbk);
        else s += pow(x - mak, en);
    }
    __shared__ double red[4];
    s = block_sum<4>(s, red);
    if (threadIdx.x == 0) part[(size_t) k * nbl + bl] = s;
}

/* out[k] = scale * (the level's sum), plus off[k] when given (a field
 * stored relative to a per-level profile); a wave per level */
__global__ void __launch_bounds__(256) k_stat_finish(const double *part, int nbl, int nz, double scale, double *out,
                                                     const double *off)
{
    const int k = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (k >= nz) return;
    const double s = level_sum(part, k, nbl);
    if ((threadIdx.x & 63) == 0) out[k] = off ? s * scale + off[k] : s * scale;
}

/* One-dimensional cross-spectra of FFT3D spectra A, B [nz][nkx][ny]:
 * specx[ix][k] sums the conjugate products over ky without the (0, 0) mode;
 * specy[t][k], t <= ny/2, sums over kx the mode ky = t and the mirror of
 * ky = ny - t (imaginary part negated) in the columns where get.c:46-84
 * takes them.
 *
 * One pass over A and B, which bounds it: a wave holds CF_SPEC_ROWS rows kx
 * of a level and marches along ky, so a row's sum stays in the wave and a
 * column's leaves one partial a wave -- of every row, and of the rows that
 * have a mirror.  128 x 97 x 128: 7.5 us, with 9.4 for the launch that sums
 * the partials into host memory; a workgroup per level with a barrier tree
 * per row took 111 us. */
__global__ void __launch_bounds__(256) k_stat_spec(const double2 *A, const double2 *B, int nx, int ny, int nkx,
                                                   int nz, double2 *specx, double2 *part)
{
    const int lane = threadIdx.x & 63, ng = (nkx + CF_SPEC_ROWS - 1) / CF_SPEC_ROWS;
    const int wv = blockIdx.x * 4 + ((int) threadIdx.x >> 6);
    if (wv >= ng * nz) return;
    const int k = wv / ng, g = wv - k * ng, ix0 = g * CF_SPEC_ROWS;
    const size_t base = ((size_t) k * nkx + ix0) * ny;
    double2 *pk = part + ((size_t) g * nz + k) * ny * 2;
    double sr[CF_SPEC_ROWS], si[CF_SPEC_ROWS];
#pragma unroll
    for (int q = 0; q < CF_SPEC_ROWS; q++) sr[q] = si[q] = 0.0;
    for (int iy = lane; iy < ny; iy += 64) {
        double2 u[CF_SPEC_ROWS], v[CF_SPEC_ROWS];
#pragma unroll
        for (int q = 0; q < CF_SPEC_ROWS; q++) {
            const size_t e = base + (size_t) (ix0 + q < nkx ? q : 0) * ny + iy;
            u[q] = A[e];
            v[q] = B[e];
        }
        double2 all = make_double2(0.0, 0.0), mir = make_double2(0.0, 0.0);
#pragma unroll
        for (int q = 0; q < CF_SPEC_ROWS; q++) {
            const int ix = ix0 + q;
            if (ix < nkx && (ix != 0 || iy != 0)) {
                const double pr = u[q].x * v[q].x + u[q].y * v[q].y, pi = u[q].y * v[q].x - u[q].x * v[q].y;
                sr[q] += pr;
                si[q] += pi;
                all.x += pr;
                all.y += pi;
                if (ix != 0 && 2 * ix != nx) { mir.x += pr; mir.y += pi; }
            }
        }
        pk[2 * iy] = all;
        pk[2 * iy + 1] = mir;
    }
#pragma unroll
    for (int q = 0; q < CF_SPEC_ROWS; q++) {
        const double r = wave_sum(sr[q]), i = wave_sum(si[q]);
        if (lane == 0 && ix0 + q < nkx) specx[(size_t) (ix0 + q) * nz + k] = make_double2(r, i);
    }
}

/* out: the nkx rows of specx, then specy from k_stat_spec's partials in
 * the order of kx; a thread per value, k fastest */
__global__ void __launch_bounds__(256) k_stat_spec_finish(const double2 *specx, const double2 *part, int ny, int nkx,
                                                          int nz, double2 *out)
{
    const int e = blockIdx.x * 256 + threadIdx.x, nsx = nkx * nz;
    if (e >= nsx + (ny / 2 + 1) * nz) return;
    if (e < nsx) { out[e] = specx[e]; return; }
    const int t = (e - nsx) / nz, k = (e - nsx) - t * nz;
    const int iyc = t > 0 ? ny - t : 0;         /* the ky whose mirror is t */
    const int ng = (nkx + CF_SPEC_ROWS - 1) / CF_SPEC_ROWS;
    double2 s = make_double2(0.0, 0.0);
#pragma unroll 4
    for (int g = 0; g < ng; g++) {
        const double2 *pk = part + ((size_t) g * nz + k) * ny * 2;
        const double2 a = pk[2 * t], m = pk[2 * iyc + 1];
        s.x += a.x + m.x;
        s.y += a.y - m.y;
    }
    out[e] = s;
}

/* FP32 storage to FP64 for the spectra */
template <typename T>
__global__ void k_stat_widen(const T *in, double *out, size_t n)
{
    const size_t i = (size_t) blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = (double) in[i];
}

#define INST_(T)                                                                                                     \
    template __global__ void k_stat_sum<T>(const T *, const T *, int, int, double *);                                \
    template __global__ void k_stat_central<T, 1>(const T *, const T *, const double *, const double *, double,      \
                                                  double, int, int, double *);                                       \
    template __global__ void k_stat_central<T, 2>(const T *, const T *, const double *, const double *, double,      \
                                                  double, int, int, double *);
INST_(double)
INST_(float)
#undef INST_
template __global__ void k_stat_widen<float>(const float *, double *, size_t);
