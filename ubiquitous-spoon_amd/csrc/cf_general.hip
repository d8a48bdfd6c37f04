/*
 * cf_general.hip -- the general substep path: order 2 or 4 (fourth.c
 * stencils), with or without the passive scalar.  Same device layout as
 * the order-2 fast path (z-slowest, no ghost cells): periodic neighbours
 * by index wrap, wall ghosts from the host-built closures (cf_tables.h).
 *
 * One substep (chanfast.c:395-656 / :1319-1580):
 *   k_grhs            explicit tendency f (advection, x-y diffusion,
 *                     buoyancy) and the implicit right-hand side
 *                     h = H(q) + gam dt f + zet dt (g + forcing) - lift
 *                     of u, v, w and c
 *   k_spike / k_spike4   the wall-reduced z solves (order 2 / 4), with the
 *                     mass-flux / scalar-mean forcing beside them (Book)
 *   k_div_fftx<.., ORD>, k_ffty, k_poisson2|4, k_ffty, k_fftx_inv  pressure
 *   k_gproject           projection + forcing correction into the state
 * Each stencil kernel reads its neighbours straight from global memory
 * (the caches catch the reuse); one thread per output point.
 */
#include "cf_kernels.h"

static constexpr double A1d = 1.125 / 1.0;      /* fourth.c:3-6 */
static constexpr double A2d = -0.125 / 3.0;
static constexpr double B1d = 1.125 / 2.0;
static constexpr double B2d = -0.125 / 2.0;

/* ------------------------------------------------------------ points */

static __device__ __forceinline__ size_t rowof(int k, int j, int nx, size_t P) { return (size_t) k * P + (size_t) j * nx; }

/* One thread's point (i, j, k) of a 256-thread workgroup that takes 256
 * consecutive cells of a level (a row's end does not idle its lanes: 90 of
 * 128 lanes worked in 64-wide row blocks at nx = 90).  The level is
 * uniform, so a value's address is a scalar base and a 32-bit byte offset
 * in the plane. */
template <typename T> struct Pt {
    int nx, ny, nz, i, j, k;
    size_t P;
    bool act;
    __device__ __forceinline__ Pt(const RunDev &R, const Blk &b)
    {
        nx = R.g.nx; ny = R.g.ny; nz = R.g.nz; k = b.z;
        P = (size_t) nx * ny;
        const int e = (int) b.x * 256 + (int) threadIdx.x;
        act = e < (int) P;
        const int ec = act ? e : (int) P - 1;
        j = qdiv(ec, nx, R.rnx);
        i = ec - j * nx;
    }
    /* byte offset in the plane of the point shifted by (d, e), periodic */
    __device__ __forceinline__ unsigned off(int d, int e) const
    {
        return (unsigned) (wrapm(j + e, ny) * nx + wrapm(i + d, nx)) * (unsigned) sizeof(T);
    }
    __device__ __forceinline__ T at(gp<const T> f, int kk, unsigned o) const
    {
        return *(gp<const T>) ((gp<const char>) (f + (size_t) kk * P) + o);
    }
    __device__ __forceinline__ void put(gp<T> f, T v) const { *(gp<T>) ((gp<char>) (f + (size_t) k * P) + off(0, 0)) = v; }
};

/* a cell field's values at levels k-3..k+3 of the point's column (those
 * within RCH of k), ghosts from the closure (ghost m of a wall = G[m] .
 * (x0, x1, x2) + B[m] bc; order 2 has the one next to the wall) */
template <int ORD, int RCH, typename T>
static __device__ __forceinline__ void cell_col7(const Pt<T> &p, gp<const T> q, const Clos1 *C, double bcb, double bct, T o[7])
{
    const unsigned cc = p.off(0, 0);
    const int k = p.k, nz = p.nz;
#pragma unroll
    for (int t = 0; t < 7; t++) {
        const int kk = k - 3 + t;
        const bool reach = t - 3 <= RCH && 3 - t <= RCH;
        o[t] = (reach && kk >= 0 && kk < nz) ? p.at(q, kk, cc) : (T) 0;
    }
    if (k < 3) {
        const Clos1 &B = C[0];
        const T x0 = p.at(q, 0, cc);
        const T x1 = ORD == 4 ? p.at(q, 1, cc) : (T) 0, x2 = ORD == 4 ? p.at(q, 2, cc) : (T) 0;
#pragma unroll
        for (int m = 0; m < (ORD == 4 ? 3 : 1); m++) {
            const int t = -1 - m - k + 3;
            if (t >= 0) o[t] = (T) B.G[m][0] * x0 + (T) B.G[m][1] * x1 + (T) B.G[m][2] * x2 + (T) (B.B[m] * bcb);
        }
    }
    if (k > nz - 4) {
        const Clos1 &Tp = C[1];
        const T x0 = p.at(q, nz - 1, cc);
        const T x1 = ORD == 4 ? p.at(q, nz - 2, cc) : (T) 0, x2 = ORD == 4 ? p.at(q, nz - 3, cc) : (T) 0;
#pragma unroll
        for (int m = 0; m < (ORD == 4 ? 3 : 1); m++) {
            const int t = nz + m - k + 3;
            if (t <= 6) o[t] = (T) Tp.G[m][0] * x0 + (T) Tp.G[m][1] * x1 + (T) Tp.G[m][2] * x2 + (T) (Tp.B[m] * bct);
        }
    }
}

/* w at face level kk as the advection terms see it: the wall faces -1 and
 * nz-1 are 0 and the ghost faces mirror oddly about them (apply_bc_w and
 * the in-place ghost rewrite of massflux*4, advect.c:100-131) */
template <typename T>
static __device__ __forceinline__ T wadv(const Pt<T> &p, gp<const T> w, unsigned o, int kk)
{
    if (kk >= 0 && kk <= p.nz - 2) return p.at(w, kk, o);
    if (kk == -1 || kk == p.nz - 1) return (T) 0;
    if (kk < -1) return -p.at(w, -2 - kk, o);
    return -p.at(w, 2 * (p.nz - 1) - kk, o);
}

/* w at levels k-3..k+3 for the implicit operator: closure ghosts
 * (apply_bc_w2/4 is re-applied before helmholtz1d_operator_w) */
template <int ORD, typename T>
static __device__ __forceinline__ void face_col7(const Pt<T> &p, gp<const T> w, const Clos1 *C, T o[7])
{
    const unsigned cc = p.off(0, 0);
    const int k = p.k, nz = p.nz;
#pragma unroll
    for (int t = 0; t < 7; t++) {
        const int kk = k - 3 + t;
        const bool reach = ORD == 4 || (t >= 2 && t <= 4);
        o[t] = (reach && kk >= 0 && kk <= nz - 2) ? p.at(w, kk, cc) : (T) 0;
    }
    if (k < 3) {
        const Clos1 &B = C[0];
        const T x0 = p.at(w, 0, cc);
        const T x1 = ORD == 4 ? p.at(w, 1, cc) : (T) 0, x2 = ORD == 4 ? p.at(w, 2, cc) : (T) 0;
#pragma unroll
        for (int m = 0; m < (ORD == 4 ? 3 : 1); m++) {
            const int t = -1 - m - k + 3;
            if (t >= 0) o[t] = (T) B.G[m][0] * x0 + (T) B.G[m][1] * x1 + (T) B.G[m][2] * x2;
        }
    }
    if (k > nz - 5) {
        const Clos1 &Tp = C[1];
        const T x0 = p.at(w, nz - 2, cc);
        const T x1 = ORD == 4 ? p.at(w, nz - 3, cc) : (T) 0, x2 = ORD == 4 ? p.at(w, nz - 4, cc) : (T) 0;
#pragma unroll
        for (int m = 0; m < (ORD == 4 ? 3 : 1); m++) {
            const int t = nz - 1 + m - k + 3;
            if (t <= 6) o[t] = (T) Tp.G[m][0] * x0 + (T) Tp.G[m][1] * x1 + (T) Tp.G[m][2] * x2;
        }
    }
}

/* The stencils below divide by cell sizes through their host-computed
 * reciprocals, with the sizes that a flux and its cell volume share
 * cancelled: an FP64 division is a dozen instructions, and the per-field
 * kernels were bound by their arithmetic (10 and more divisions a point;
 * four fields at 90x73x75 in 24 us, 44 before). */

/* the second difference of a line at unit spacing, twice staggered */
template <int ORD, typename T>
static __device__ __forceinline__ T d2(const T *X)
{
    if (ORD == 2) return (X[4] - X[3]) - (X[3] - X[2]);
    const T A1 = (T) A1d, A2 = (T) A2d;
    const T p3h = A1 * (X[5] - X[4]) + A2 * (X[6] - X[3]);
    const T p1h = A1 * (X[4] - X[3]) + A2 * (X[5] - X[2]);
    const T m1h = A1 * (X[3] - X[2]) + A2 * (X[4] - X[1]);
    const T m3h = A1 * (X[2] - X[1]) + A2 * (X[3] - X[0]);
    return A1 * (p1h - m1h) + A2 * (p3h - m3h);
}

/* cell/face 1-D Helmholtz operators (diffuseu.c:107-170, diffusew.c:107-172)
 * Q + nudt d2Q/dz2: in are the reciprocal spacings between the levels (four
 * of them about Q[3]: -3/2, -1/2, +1/2, +3/2), out the reciprocal height */
template <int ORD, typename T>
static __device__ __forceinline__ T helm(const T *Q, T rm3, T rm1, T rp1, T rp3, T rout, T nudt)
{
    if (ORD == 2) return Q[3] + nudt * (((Q[4] - Q[3]) * rp1 - (Q[3] - Q[2]) * rm1) * rout);
    const T A1 = (T) A1d, A2 = (T) A2d;
    const T p3h = A1 * (Q[5] - Q[4]) + A2 * (Q[6] - Q[3]);
    const T p1h = A1 * (Q[4] - Q[3]) + A2 * (Q[5] - Q[2]);
    const T m1h = A1 * (Q[3] - Q[2]) + A2 * (Q[4] - Q[1]);
    const T m3h = A1 * (Q[2] - Q[1]) + A2 * (Q[3] - Q[0]);
    return Q[3] + nudt * ((A1 * (p1h * rp1 - m1h * rm1) + A2 * (p3h * rp3 - m3h * rm3)) * rout);
}

/* a quantity at the middle of points 1 and 2 of four */
template <int ORD, typename T>
static __device__ __forceinline__ T mid(T m, T a, T b, T p)
{
    return ORD == 2 ? (T) 0.5 * (a + b) : (T) B1d * (a + b) + (T) B2d * (m + p);
}

/* the flux difference of one direction from the fluxes at +1/2, -1/2 and,
 * order 4, +3/2, -3/2 */
template <int ORD, typename T>
static __device__ __forceinline__ T dif(T p1, T m1, T p3, T m3)
{
    return ORD == 2 ? p1 - m1 : (T) A1d * (p1 - m1) + (T) A2d * (p3 - m3);
}

/* wall values of u/v the advection of u/v uses on the wall faces
 * (advect.c:336-341, :539-554); Qb = levels -2..1, Qt = nz-2..nz+1 */
template <int ORD, typename T>
static __device__ __forceinline__ T wall_interp(T gm2, T gm1, T x0, T x1)
{
    if (ORD == 2) return (T) 0.5 * (gm1 + x0);
    return (T) (0.5 * A2d) * (gm2 + x1) + (T) (0.5 * (A1d + 2.0 * A2d)) * (gm1 + x0);
}

/* the reductions of a workgroup at one level: the sum of r (one value per
 * thread) times the level's weight of each statistic of the substep (mwq
 * [nz][4]) into mpart (n slots a statistic) and, where cflpart is set, the
 * maximum of cfl (>= 0) */
static __device__ __forceinline__ void block_store(double r, const double *__restrict__ mwq, int k, int s,
                                                   double *__restrict__ mpart, double cfl,
                                                   double *__restrict__ cflpart, unsigned bidx, unsigned n)
{
    __shared__ double red[8];
    const int t = threadIdx.x;
    const double w = wave_sum(r), c = cflpart ? wave_max_nonneg(cfl) : 0.0;
    if ((t & 63) == 0) { red[t >> 6] = w; red[4 + (t >> 6)] = c; }
    __syncthreads();
    if (t < book_stats(s)) mpart[(size_t) t * n + bidx] = mwq[4 * k + t] * (((red[0] + red[1]) + red[2]) + red[3]);
    if (cflpart && t == 0) cflpart[bidx] = fmax(fmax(red[4], red[5]), fmax(red[6], red[7]));
}

/* ------------------------------------------------------------ u and v */

/* advectu2/4 or advectv2/4 + laplacexy + buoyancy, then the right-hand side
 * of solve_helmholtz1d_u (chanfast.c:465-477) of u (AX = 0) or v (AX = 1):
 * a is the advected field, the other horizontal velocity o; "along" is the
 * direction of a.  CFL partials of u at s == 0. */
template <int ORD, bool SC, int AX, typename T>
static __device__ __forceinline__ void rhsuv_body(const RunDev &R, const int s, const GFields<T> &F,
    const double *__restrict__ scal, double *__restrict__ cflpart, double cfldt, double *__restrict__ mpart, const Blk b)
{
    const Pt<T> p(R, b);
    const int k = p.k, nz = p.nz;
    const gp<const T> a = (gp<const T>) (AX == 0 ? F.u : F.v), o = (gp<const T>) (AX == 0 ? F.v : F.u);
    const gp<const T> w = (gp<const T>) F.w, c = (gp<const T>) F.c, g = (gp<const T>) F.g[AX];
    const cp<double> rdz = (cp<double>) R.rdz + CF_NGT, rdzh = (cp<double>) R.rdzh + CF_NGT, dz = (cp<double>) R.dzt + CF_NGT;
    double cflv = 0.0, rsum = 0.0;
    if (p.act) {
        constexpr int LO = ORD == 2 ? 2 : 0, HI = ORD == 2 ? 4 : 6;
        auto al = [&](int d) { return AX == 0 ? p.off(d, 0) : p.off(0, d); };      /* d along a's direction */
        auto cr = [&](int d) { return AX == 0 ? p.off(0, d) : p.off(d, 0); };      /* d across it */
        auto ac = [&](int d, int e) { return AX == 0 ? p.off(d, e) : p.off(e, d); };
        const double bc = AX == 0 ? R.ubc : R.vbc;
        T Z[7], A[7], C[7];
        cell_col7<ORD, ORD == 2 ? 1 : 3>(p, a, R.cl.cell, bc, bc, Z);
#pragma unroll
        for (int t = 0; t < 7; t++) {
            A[t] = t < LO || t > HI ? (T) 0 : (t == 3 ? Z[3] : p.at(a, k, al(t - 3)));
            C[t] = t < LO || t > HI ? (T) 0 : (t == 3 ? Z[3] : p.at(a, k, cr(t - 3)));
        }
        const T Q0 = Z[3];
        /* massfluxx / massfluxy (advect.c:6-200): velocities interpolated to
         * a's point along its direction */
        auto VA = [&](int d) -> T { return mid<ORD, T>(d >= -2 ? A[2 + d] : (T) 0, A[3 + d], A[4 + d], d <= 1 ? A[5 + d] : (T) 0); };
        auto VC = [&](int e) -> T {
            return mid<ORD, T>(ORD == 4 ? p.at(o, k, ac(-1, e)) : (T) 0, p.at(o, k, ac(0, e)), p.at(o, k, ac(1, e)),
                               ORD == 4 ? p.at(o, k, ac(2, e)) : (T) 0);
        };
        auto VZ = [&](int e) -> T {
            const int kk = k + e;
            return mid<ORD, T>(ORD == 4 ? wadv(p, w, al(-1), kk) : (T) 0, wadv(p, w, al(0), kk), wadv(p, w, al(1), kk),
                               ORD == 4 ? wadv(p, w, al(2), kk) : (T) 0);
        };
        const T fa = dif<ORD, T>(VA(0) * (Q0 + A[4]), VA(-1) * (Q0 + A[2]), ORD == 4 ? VA(1) * (Q0 + A[6]) : (T) 0,
                                 ORD == 4 ? VA(-2) * (Q0 + A[0]) : (T) 0);
        const T fc = dif<ORD, T>(VC(0) * (Q0 + C[4]), VC(-1) * (Q0 + C[2]), ORD == 4 ? VC(1) * (Q0 + C[6]) : (T) 0,
                                 ORD == 4 ? VC(-2) * (Q0 + C[0]) : (T) 0);
        /* Z[t] is level k - 3 + t; wall values from levels -2..1 / nz-2..nz+1 */
        const T w0 = VZ(0), wm = VZ(-1), wp = ORD == 4 ? VZ(1) : (T) 0, wm2 = ORD == 4 ? VZ(-2) : (T) 0;
        T zp = w0 * (Q0 + Z[4]), zm = wm * (Q0 + Z[2]), zp3 = wp * (Q0 + Z[6]), zm3 = wm2 * (Q0 + Z[0]);
        const T two = (T) 2;
        if (k == nz - 1) {
            const T bct = wall_interp<ORD>(Z[5], Z[4], Z[3], Z[2]);
            zp = w0 * (two * bct);
            zp3 = -wm * (Z[1] + Z[4]) + two * w0 * (two * bct);
        }
        if (ORD == 4 && k == nz - 2) zp3 = wp * (two * wall_interp<ORD>(Z[6], Z[5], Z[4], Z[3]));
        if (k == 0) {
            const T bcb = wall_interp<ORD>(Z[1], Z[2], Z[3], Z[4]);
            zm = wm * (two * bcb);
            zm3 = -w0 * (Z[5] + Z[2]) + two * wm * (two * bcb);
        }
        if (ORD == 4 && k == 1) zm3 = wm2 * (two * wall_interp<ORD>(Z[0], Z[1], Z[2], Z[3]));
        const T rx = (T) R.rdx, ry = (T) R.rdy, ra = AX == 0 ? rx : ry, rc = AX == 0 ? ry : rx;
        T f = (T) -0.5 * (fa * ra + fc * rc + dif<ORD, T>(zp, zm, zp3, zm3) * (T) rdz[k]);
        /* the x-y diffusion: explicit in f (chanfast, diffuseu.c:286-359), or
         * in the 3-D Helmholtz operator of h when every diffusion term is
         * implicit (channel, helmholtz_operator_u, diffuseu.c:362-457) */
        const T lxy = d2<ORD>(A) * (ra * ra) + d2<ORD>(C) * (rc * rc);
        if (!R.implicit) f += (T) R.nu * lxy;
        if (SC && R.betg[AX] != 0.0)        /* add_buoyancy2/4, scalar.c:6-76 */
            f += mid<ORD, T>(ORD == 4 ? p.at(c, k, al(-1)) : (T) 0, p.at(c, k, al(0)), p.at(c, k, al(1)),
                             ORD == 4 ? p.at(c, k, al(2)) : (T) 0) * (T) R.betg[AX];
        const SubCoef &S = R.sc[s];
        T h = helm<ORD>(Z, ORD == 4 ? (T) rdzh[k - 2] : (T) 0, (T) rdzh[k - 1], (T) rdzh[k], ORD == 4 ? (T) rdzh[k + 1] : (T) 0,
                        (T) rdz[k], (T) S.nuadt);
        if (R.implicit) h += (T) S.nuadt * lxy;
        /* the explicit part rounds h once, here and in w and c: adding its two
         * terms one after the other, FP32 runs with the scalar err 1 to 4%
         * more in v and w (32x129x32, nu dt 2e-5, 40 steps: 5.71e-6 and
         * 6.56e-6 against 5.51e-6 and 6.30e-6) */
        if (s > 0)
            h += (T) S.gamdt * f
               + (T) S.zetdt * (p.at(g, k, p.off(0, 0)) + (AX == 0 ? (T) ((cp<double>) scal)[R.m_prev_slot[s]] : (T) 0));
        else h += (T) S.gamdt * f;
        h -= (T) ((cp<double>) R.liftg)[((size_t) s * 4 + AX) * nz + k];
        if (s < 2) p.put((gp<T>) F.f[AX], f);     /* the last substep's tendency is never read */
        /* the z solve's right-hand side is h dvol (diffuseu.c:202); the
         * spectral solve takes h and applies dvol itself */
        const T rr = h * (T) dz[k];
        p.put((gp<T>) F.r[AX], R.implicit ? h : rr);
        rsum = (double) rr;
        if (AX == 0 && cflpart)             /* get_cfl, get.c:390-417 */
            cflv = fmax(fmax(fabs((double) Q0) * cfldt * R.rdx, fabs((double) p.at(o, k, p.off(0, 0))) * cfldt * R.rdy),
                        fabs((double) p.at(w, k, p.off(0, 0))) * cfldt * rdzh[k]);
    }
    if (AX == 0)
        block_store(rsum, R.mwq + (size_t) (s * 2) * 4 * nz, k, s, mpart, cflv, cflpart, b.z * b.nx + b.x, b.nx * b.nz);
}

/* ------------------------------------------------------------ w */

template <int ORD, bool SC, typename T>
static __device__ __forceinline__ void rhsw_body(const RunDev &R, const int s, const GFields<T> &F, const Blk b)
{
    const Pt<T> p(R, b);
    const int k = p.k, nz = p.nz;
    if (!p.act) return;
    const gp<T> fo = (gp<T>) F.f[2], ro = (gp<T>) F.r[2];
    if (k == nz - 1) {                    /* top wall face: f = 0 (advect.c:301), no unknown */
        if (s < 2) p.put(fo, (T) 0);
        p.put(ro, (T) 0);
        return;
    }
    const gp<const T> u = (gp<const T>) F.u, v = (gp<const T>) F.v, w = (gp<const T>) F.w, c = (gp<const T>) F.c;
    const cp<double> rdz = (cp<double>) R.rdz + CF_NGT, rdzh = (cp<double>) R.rdzh + CF_NGT, dz = (cp<double>) R.dzt + CF_NGT;
    constexpr int LO = ORD == 2 ? 2 : 0, HI = ORD == 2 ? 4 : 6;
    const unsigned cc = p.off(0, 0);
    T WA[7], WH[7], WX[7], WY[7];
#pragma unroll
    for (int t = 0; t < 7; t++) WA[t] = t < LO || t > HI ? (T) 0 : wadv(p, w, cc, k - 3 + t);
    face_col7<ORD>(p, w, R.cl.face, WH);
#pragma unroll
    for (int t = 0; t < 7; t++) {
        WX[t] = t < LO || t > HI ? (T) 0 : (t == 3 ? WA[3] : p.at(w, k, p.off(t - 3, 0)));
        WY[t] = t < LO || t > HI ? (T) 0 : (t == 3 ? WA[3] : p.at(w, k, p.off(0, t - 3)));
    }
    const T Q0 = WA[3];
    /* a cell field at level kk with closure ghosts, for the z-interpolated
     * fluxes and the buoyancy */
    auto cell = [&](gp<const T> fld, unsigned o, int kk, double bcb, double bct) -> T {
        if (kk >= 0 && kk < nz) return p.at(fld, kk, o);
        const bool lo = kk < 0;
        const Clos1 &Cl = R.cl.cell[lo ? 0 : 1];
        const int m = lo ? -1 - kk : kk - nz;
        const T x0 = p.at(fld, lo ? 0 : nz - 1, o);
        const T x1 = ORD == 4 ? p.at(fld, lo ? 1 : nz - 2, o) : (T) 0;
        const T x2 = ORD == 4 ? p.at(fld, lo ? 2 : nz - 3, o) : (T) 0;
        return (T) Cl.G[m][0] * x0 + (T) Cl.G[m][1] * x1 + (T) Cl.G[m][2] * x2 + (T) (Cl.B[m] * (lo ? bcb : bct));
    };
    /* massfluxz (advect.c:201-283): volume fluxes interpolated to the w-point in z */
    const T dm = ORD == 4 ? (T) dz[k - 1] : (T) 0, d0 = (T) dz[k], d1 = (T) dz[k + 1], d2_ = ORD == 4 ? (T) dz[k + 2] : (T) 0;
    auto VZ = [&](gp<const T> fld, unsigned o, double bc) -> T {
        return mid<ORD, T>(ORD == 4 ? dm * cell(fld, o, k - 1, bc, bc) : (T) 0, d0 * cell(fld, o, k, bc, bc),
                           d1 * cell(fld, o, k + 1, bc, bc), ORD == 4 ? d2_ * cell(fld, o, k + 2, bc, bc) : (T) 0);
    };
    auto UZ = [&](int d) -> T { return VZ(u, p.off(d, 0), R.ubc); };
    auto YZ = [&](int e) -> T { return VZ(v, p.off(0, e), R.vbc); };
    auto WZ = [&](int e) -> T {     /* at face k + e from WA[2+e..5+e] */
        return mid<ORD, T>(e >= -2 ? WA[2 + e] : (T) 0, WA[3 + e], WA[4 + e], e <= 1 ? WA[5 + e] : (T) 0);
    };
    const T fx = dif<ORD, T>(UZ(0) * (Q0 + WX[4]), UZ(-1) * (Q0 + WX[2]), ORD == 4 ? UZ(1) * (Q0 + WX[6]) : (T) 0,
                             ORD == 4 ? UZ(-2) * (Q0 + WX[0]) : (T) 0);
    const T fy = dif<ORD, T>(YZ(0) * (Q0 + WY[4]), YZ(-1) * (Q0 + WY[2]), ORD == 4 ? YZ(1) * (Q0 + WY[6]) : (T) 0,
                             ORD == 4 ? YZ(-2) * (Q0 + WY[0]) : (T) 0);
    const T fz = dif<ORD, T>(WZ(0) * (Q0 + WA[4]), WZ(-1) * (Q0 + WA[2]), ORD == 4 ? WZ(1) * (Q0 + WA[6]) : (T) 0,
                             ORD == 4 ? WZ(-2) * (Q0 + WA[0]) : (T) 0);
    const T rx = (T) R.rdx, ry = (T) R.rdy, rh = (T) rdzh[k];
    T f = (T) -0.5 * ((fx * rx + fy * ry + fz) * rh);
    const T lxy = d2<ORD>(WX) * (rx * rx) + d2<ORD>(WY) * (ry * ry);
    if (!R.implicit) f += (T) R.nu * lxy;
    if (SC && R.betg[2] != 0.0)
        f += mid<ORD, T>(ORD == 4 ? cell(c, cc, k - 1, R.cbot, R.ctop) : (T) 0, cell(c, cc, k, R.cbot, R.ctop),
                         cell(c, cc, k + 1, R.cbot, R.ctop), ORD == 4 ? cell(c, cc, k + 2, R.cbot, R.ctop) : (T) 0)
             * (T) R.betg[2];
    const SubCoef &S = R.sc[s];
    T h = helm<ORD>(WH, ORD == 4 ? (T) rdz[k - 1] : (T) 0, (T) rdz[k], (T) rdz[k + 1], ORD == 4 ? (T) rdz[k + 2] : (T) 0, rh,
                    (T) S.nuadt);
    if (R.implicit) h += (T) S.nuadt * lxy;
    if (s > 0) h += (T) S.gamdt * f + (T) S.zetdt * p.at((gp<const T>) F.g[2], k, cc);
    else h += (T) S.gamdt * f;
    h -= (T) ((cp<double>) R.liftg)[((size_t) s * 4 + 2) * nz + k];
    if (s < 2) p.put(fo, f);                  /* the last substep's tendency is never read */
    p.put(ro, R.implicit ? h : h * ((T) 0.5 * (d1 + d0)));    /* times the face volume (diffusew.c:205) */
}

/* ------------------------------------------------------------ c */

template <int ORD, typename T>
static __device__ __forceinline__ void rhsc_body(const RunDev &R, const int s, const GFields<T> &F,
    const double *__restrict__ scal, double *__restrict__ mpart, const Blk b)
{
    const Pt<T> p(R, b);
    const int k = p.k, nz = p.nz;
    const gp<const T> u = (gp<const T>) F.u, v = (gp<const T>) F.v, w = (gp<const T>) F.w, c = (gp<const T>) F.c;
    const cp<double> rdz = (cp<double>) R.rdz + CF_NGT, rdzh = (cp<double>) R.rdzh + CF_NGT, dz = (cp<double>) R.dzt + CF_NGT;
    double rsum = 0.0;
    if (p.act) {
        constexpr int LO = ORD == 2 ? 1 : 0, HI = ORD == 2 ? 5 : 6;   /* QUICK reaches two cells */
        const unsigned cc = p.off(0, 0);
        T Cz[7], CX[7], CY[7];
        cell_col7<ORD, ORD == 2 ? 2 : 3>(p, c, R.cl.cell, R.cbot, R.ctop, Cz);
#pragma unroll
        for (int t = 0; t < 7; t++) {
            CX[t] = t < LO || t > HI ? (T) 0 : (t == 3 ? Cz[3] : p.at(c, k, p.off(t - 3, 0)));
            CY[t] = t < LO || t > HI ? (T) 0 : (t == 3 ? Cz[3] : p.at(c, k, p.off(0, t - 3)));
        }
        const T qk = (T) -0.125;
        /* QUICK face value upwinded by the sign of the face velocity */
        auto quick = [&](T fl, T cm, T c0, T c1, T c2) -> T {
            T cf = (T) 0.5 * (c0 + c1);
            cf += fl > (T) 0 ? qk * (c1 - (T) 2.0 * c0 + cm) : qk * (c2 - (T) 2.0 * c1 + c0);
            return fl * cf;
        };
        const T u0 = p.at(u, k, cc), um = p.at(u, k, p.off(-1, 0)), v0 = p.at(v, k, cc), vm = p.at(v, k, p.off(0, -1));
        const T w0 = wadv(p, w, cc, k), wm = wadv(p, w, cc, k - 1);
        const T fx = quick(u0, CX[2], CX[3], CX[4], CX[5]) - quick(um, CX[1], CX[2], CX[3], CX[4]);
        const T fy = quick(v0, CY[2], CY[3], CY[4], CY[5]) - quick(vm, CY[1], CY[2], CY[3], CY[4]);
        const T fz = quick(w0, Cz[2], Cz[3], Cz[4], Cz[5]) - quick(wm, Cz[1], Cz[2], Cz[3], Cz[4]);
        const T rx = (T) R.rdx, ry = (T) R.rdy;
        T f = -(fx * rx + fy * ry + fz * (T) rdz[k]);
        const T lxy = d2<ORD>(CX) * (rx * rx) + d2<ORD>(CY) * (ry * ry);
        if (!R.implicit) f += (T) R.kap * lxy;
        const SubCoef &S = R.sc[s];
        T h = helm<ORD>(Cz, ORD == 4 ? (T) rdzh[k - 2] : (T) 0, (T) rdzh[k - 1], (T) rdzh[k], ORD == 4 ? (T) rdzh[k + 1] : (T) 0,
                        (T) rdz[k], (T) S.kadt);
        if (R.implicit) h += (T) S.kadt * lxy;
        if (s > 0)
            h += (T) S.gamdt * f + (T) S.zetdt * (p.at((gp<const T>) F.g[3], k, cc) + (T) ((cp<double>) scal)[SC_MC0 + (s + 2) % 3]);
        else h += (T) S.gamdt * f;
        h -= (T) ((cp<double>) R.liftg)[((size_t) s * 4 + 3) * nz + k];
        if (s < 2) p.put((gp<T>) F.f[3], f);      /* the last substep's tendency is never read */
        const T rr = h * (T) dz[k];
        p.put((gp<T>) F.r[3], R.implicit ? h : rr);
        rsum = (double) rr;
    }
    block_store(rsum, R.mwq + (size_t) (s * 2 + 1) * 4 * nz, k, s, mpart, 0.0, nullptr, b.z * b.nx + b.x, b.nx * b.nz);
}

/* ------------------------------------------------------------ all fields */

/* One launch for every field of a substep: the z index of the grid counts
 * (level, field), field fastest, so that the workgroups reading the same
 * level of u, v, w and c run together.  A launch per field cost a small
 * grid 4 us each and left most CUs idle (four of 13 us at 90x73x75). */
template <int ORD, bool SC, typename T>
static __device__ __forceinline__ void grhs_body(const RunDev &R, const int s, const GFields<T> &F,
    const double *__restrict__ scal, double *__restrict__ cflpart, double cfldt, double *__restrict__ mpart, Blk b)
{
    constexpr unsigned nf = SC ? 4 : 3;
    const unsigned fld = b.z % nf;
    b.z /= nf;
    b.nz /= nf;
    if (fld == 0) rhsuv_body<ORD, SC, 0>(R, s, F, scal, cflpart, cfldt, mpart, b);
    else if (fld == 1) rhsuv_body<ORD, SC, 1>(R, s, F, scal, nullptr, cfldt, nullptr, b);
    else if (fld == 2) rhsw_body<ORD, SC>(R, s, F, b);
    else if constexpr (SC) rhsc_body<ORD>(R, s, F, scal, mpart + (size_t) 4 * b.nx * b.nz, b);
}

template <int ORD, bool SC, typename T>
__global__ __launch_bounds__(256) void k_grhs(const RunDev R, const int s, const GFields<T> F,
    const double *__restrict__ scal, double *__restrict__ cflpart, double cfldt, double *__restrict__ mpart)
{
    grhs_body<ORD, SC, T>(kernarg_run(), s, F, scal, cflpart, cfldt, mpart, blk_native());
}

/* ------------------------------------------------------------ solve */

/* order-4 wall-reduced z solves (solve_helmholtz1d_u4 / _w4 with
 * heptdag.c:5-61), constant coefficients from the host, one thread per
 * (column, field), in place.  Fields 0 u, 1 v, 2 w (nz-1 unknowns, top
 * wall := 0), 3 c. */
template <typename T>
static __device__ __forceinline__ void solve4_body(const RunDev &R, const int s,
    T *__restrict__ ru, T *__restrict__ rv, T *__restrict__ rw, T *__restrict__ rc, const Blk b)
{
    const int nx = R.g.nx, ny = R.g.ny, nz = R.g.nz;
    const size_t P = (size_t) nx * ny;
    const size_t col = (size_t) b.x * blockDim.x + threadIdx.x;
    const int f = b.y;
    if (col >= P || f > 3) return;
    T *x = f == 0 ? ru : (f == 1 ? rv : (f == 2 ? rw : rc));
    const int type = f == 2 ? 2 : (f == 3 ? 1 : 0);
    const HeptTab HT = R.hp[s][type];
    const int n = HT.n;
    const double *A = HT.t, *AL = A + n, *BE = AL + n, *ID = BE + n, *Pp = ID + n, *Qq = Pp + n, *Rr = Qq + n;
    T *xc = x + col;
    T s1 = 0, s2 = 0, s3 = 0;
    constexpr int BT = 8;
    for (int i0 = 0; i0 < n; i0 += BT) {
        T hb[BT];
#pragma unroll
        for (int t = 0; t < BT; t++) hb[t] = i0 + t < n ? xc[(size_t) (i0 + t) * P] : (T) 0;
#pragma unroll
        for (int t = 0; t < BT; t++) {
            const int i = i0 + t;
            if (i < n) {
                const T si = (hb[t] - (T) A[i] * s3 - (T) AL[i] * s2 - (T) BE[i] * s1) * (T) ID[i];
                xc[(size_t) i * P] = si;
                s3 = s2; s2 = s1; s1 = si;
            }
        }
    }
    T x1 = 0, x2 = 0, x3 = 0;
    for (int i0 = n - 1; i0 >= 0; i0 -= BT) {
        T sb[BT];
#pragma unroll
        for (int t = 0; t < BT; t++) sb[t] = i0 - t >= 0 ? xc[(size_t) (i0 - t) * P] : (T) 0;
#pragma unroll
        for (int t = 0; t < BT; t++) {
            const int i = i0 - t;
            if (i >= 0) {
                const T xi = sb[t] - (T) Pp[i] * x1 - (T) Qq[i] * x2 - (T) Rr[i] * x3;
                xc[(size_t) i * P] = xi;
                x3 = x2; x2 = x1; x1 = xi;
            }
        }
    }
    if (f == 2) xc[(size_t) (nz - 1) * P] = (T) 0;
}

template <typename T>
__global__ __launch_bounds__(256) void k_gsolve4(const RunDev R, const int s, const int nbx,
    T *__restrict__ ru, T *__restrict__ rv, T *__restrict__ rw, T *__restrict__ rc, const Book B)
{
    if (blockIdx.x == 0) book_body(R, B);
    else solve4_body<T>(R, s, ru, rv, rw, rc, blk_solve(blockIdx.x - 1, nbx));
}

template __global__ void k_gsolve4<double>(const RunDev, const int, const int, double *, double *, double *, double *, const Book);
template __global__ void k_gsolve4<float>(const RunDev, const int, const int, float *, float *, float *, float *, const Book);

/* ------------------------------------------------------------ Poisson, order 4 */

/* pressure_poisson4 (pressure.c:357-444): per (kx, ky) the wall-reduced
 * heptadiagonal system with the 4th-order modified wavenumbers on the
 * diagonal, factored in the recurrence of heptdag.c:5-61; the U factors
 * go to S (3 per level), the forward sweep in place in Y.  Real and
 * imaginary parts share the factors. */
template <typename Ar, typename C>
static __device__ __forceinline__ void pois4_mode(const Pois4Tab &T, C *__restrict__ y, double *__restrict__ S,
                                                  size_t M, int nz, double lxd, double lyd, int variant)
{
    /* the rows go through registers in blocks of BT: every load of a block
     * is in flight before the first row's recurrence needs it (one wave per
     * 64 modes leaves no other waves to hide a per-row load latency) */
    constexpr int BT = 8;
    const Ar lx = (Ar) lxd, ly = (Ar) lyd;
    const double *bd = T.band[variant];
    double *Sp = S, *Sq = S + (size_t) nz * M, *Sr = S + (size_t) 2 * nz * M;
    Ar p1 = 0, p2 = 0, p3 = 0, q1 = 0, q2 = 0, q3 = 0, r1 = 0, r2 = 0, r3 = 0;
    Ar s1x = 0, s2x = 0, s3x = 0, s1y = 0, s2y = 0, s3y = 0;
    for (int i0 = 0; i0 < nz; i0 += BT) {
        C rb[BT];
#pragma unroll
        for (int t = 0; t < BT; t++) rb[t] = y[(size_t) min(i0 + t, nz - 1) * M];
#pragma unroll
        for (int t = 0; t < BT; t++) {
            const int i = i0 + t;
            if (i < nz) {
                const Ar a = (Ar) bd[i], b = (Ar) bd[nz + i], c = (Ar) bd[2 * nz + i];
                const Ar d = (Ar) bd[3 * nz + i] - lx * (Ar) T.ex[i] - ly * (Ar) T.ey[i];
                const Ar e = (Ar) bd[4 * nz + i], f = (Ar) bd[5 * nz + i], g = (Ar) bd[6 * nz + i];
                const Ar alp = b - a * p3;
                const Ar bet = c - a * q3 - alp * p2;
                const Ar den = d - a * r3 - alp * q2 - bet * p1;
                const Ar iden = (Ar) 1 / den;
                const Ar pi = (e - alp * r2 - bet * q1) * iden;
                const Ar qi = (f - bet * r1) * iden;
                const Ar ri = g * iden;
                const C rh = rb[t];
                const Ar dv = (Ar) T.dvol[i];
                const Ar six = ((Ar) rh.x * dv - a * s3x - alp * s2x - bet * s1x) * iden;
                const Ar siy = ((Ar) rh.y * dv - a * s3y - alp * s2y - bet * s1y) * iden;
                C o;
                o.x = six; o.y = siy;
                y[(size_t) i * M] = o;
                Sp[(size_t) i * M] = pi; Sq[(size_t) i * M] = qi; Sr[(size_t) i * M] = ri;
                p3 = p2; p2 = p1; p1 = pi;
                q3 = q2; q2 = q1; q1 = qi;
                r3 = r2; r2 = r1; r1 = ri;
                s3x = s2x; s2x = s1x; s1x = six;
                s3y = s2y; s2y = s1y; s1y = siy;
            }
        }
    }
    Ar x1x = 0, x2x = 0, x3x = 0, x1y = 0, x2y = 0, x3y = 0;
    for (int i0 = nz - 1; i0 >= 0; i0 -= BT) {
        C sb[BT];
        double pb[BT], qb[BT], rbv[BT];
#pragma unroll
        for (int t = 0; t < BT; t++) {
            const size_t o = (size_t) max(i0 - t, 0) * M;
            sb[t] = y[o]; pb[t] = Sp[o]; qb[t] = Sq[o]; rbv[t] = Sr[o];
        }
#pragma unroll
        for (int t = 0; t < BT; t++) {
            const int i = i0 - t;
            if (i >= 0) {
                const Ar xix = (Ar) sb[t].x - (Ar) pb[t] * x1x - (Ar) qb[t] * x2x - (Ar) rbv[t] * x3x;
                const Ar xiy = (Ar) sb[t].y - (Ar) pb[t] * x1y - (Ar) qb[t] * x2y - (Ar) rbv[t] * x3y;
                C o;
                o.x = xix; o.y = xiy;
                y[(size_t) i * M] = o;
                x3x = x2x; x2x = x1x; x1x = xix;
                x3y = x2y; x2y = x1y; x1y = xiy;
            }
        }
    }
}

template <typename T>
static __device__ __forceinline__ void pois4_body(const RunDev &R, const Pois4Tab T_,
                                                  typename Cplx<T>::type *__restrict__ Y, double *__restrict__ S, const Blk b)
{
    const int ny = R.g.ny, nz = R.g.nz, nkx = R.g.nkx;
    const size_t M = (size_t) ny * nkx;
    const size_t qm = (size_t) b.x * blockDim.x + threadIdx.x;
    if (qm >= M) return;
    const int kx = (int) (qm / ny), ky = (int) (qm % ny);
    const int variant = (kx == 0 && ky == 0) ? 1 : 0;
    const bool low = kx <= CF_F64_KLOW && (ky <= CF_F64_KLOW || ny - ky <= CF_F64_KLOW);
    if (sizeof(T) == sizeof(double) || low)
        pois4_mode<double>(T_, Y + qm, S + qm, M, nz, R.lamx[kx], R.lamy[ky], variant);
    else
        pois4_mode<T>(T_, Y + qm, S + qm, M, nz, R.lamx[kx], R.lamy[ky], variant);
}

template <typename T>
__global__ __launch_bounds__(256) void k_poisson4(const RunDev R, const Pois4Tab T_,
                                                  typename Cplx<T>::type *__restrict__ Y, double *__restrict__ S)
{
    pois4_body<T>(R, T_, Y, S, blk_native());
}

template __global__ void k_poisson4<double>(const RunDev, const Pois4Tab, double2 *, double *);
template __global__ void k_poisson4<float>(const RunDev, const Pois4Tab, float2 *, double *);

/* The same solve split at the middle row m = nz / 2 ("twisted"), for
 * nz >= 6: wave 0 of a 128-thread workgroup eliminates rows 0..m-1 of 64
 * modes from the top (the recurrence above), wave 1 rows nz-1..m from the
 * bottom (the same recurrence on the mirrored bands), so each dependent
 * chain is half as long and twice as many waves run.  Each side's last
 * three relations,
 *   top:    x_R + p x_{R+1} + q x_{R+2} + r x_{R+3} = s   (R = m-3..m-1)
 *   bottom: x_R + p x_{R-1} + q x_{R-2} + r x_{R-3} = s   (R = m..m+2),
 * couple the six unknowns x_{m-3..m+2}; both waves solve that 6x6 system
 * (unit diagonal, no pivoting) and back-substitute their own half.  Every
 * row is still eliminated once, from the rows on its side only, as in the
 * sequential elimination; results differ from it by round-off. */
template <typename Ar, typename C>
static __device__ __forceinline__ void p4t_sweep(const Pois4Tab &T, C *__restrict__ y, double *__restrict__ S,
                                                 size_t M, int nz, double lxd, double lyd, int variant, int side,
                                                 double *__restrict__ xme)
{
    constexpr int BT = 8;
    const int m = nz / 2, cnt = side == 0 ? m : nz - m;
    const Ar lx = (Ar) lxd, ly = (Ar) lyd;
    const double *bd = T.band[variant];
    /* band offsets -3..+3 as seen from this side (mirrored for the bottom) */
    const double *ba = bd + (side == 0 ? 0 : 6) * nz, *bb = bd + (side == 0 ? 1 : 5) * nz, *bc = bd + (side == 0 ? 2 : 4) * nz;
    const double *be = bd + (side == 0 ? 4 : 2) * nz, *bf = bd + (side == 0 ? 5 : 1) * nz, *bg = bd + (side == 0 ? 6 : 0) * nz;
    const double *bdd = bd + 3 * nz;
    double *Sp = S, *Sq = S + (size_t) nz * M, *Sr = S + (size_t) 2 * nz * M;
    Ar p1 = 0, p2 = 0, p3 = 0, q1 = 0, q2 = 0, q3 = 0, r1 = 0, r2 = 0, r3 = 0;
    Ar s1x = 0, s2x = 0, s3x = 0, s1y = 0, s2y = 0, s3y = 0;
    for (int j0 = 0; j0 < cnt; j0 += BT) {
        C rb[BT];
#pragma unroll
        for (int t = 0; t < BT; t++) {
            const int j = min(j0 + t, cnt - 1);
            rb[t] = y[(size_t) (side == 0 ? j : nz - 1 - j) * M];
        }
#pragma unroll
        for (int t = 0; t < BT; t++) {
            const int j = j0 + t;
            if (j < cnt) {
                const int i = side == 0 ? j : nz - 1 - j;
                const Ar a = (Ar) ba[i], b = (Ar) bb[i], c = (Ar) bc[i];
                const Ar d = (Ar) bdd[i] - lx * (Ar) T.ex[i] - ly * (Ar) T.ey[i];
                const Ar e = (Ar) be[i], f = (Ar) bf[i], g = (Ar) bg[i];
                const Ar alp = b - a * p3;
                const Ar bet = c - a * q3 - alp * p2;
                const Ar den = d - a * r3 - alp * q2 - bet * p1;
                const Ar iden = (Ar) 1 / den;
                const Ar pi = (e - alp * r2 - bet * q1) * iden;
                const Ar qi = (f - bet * r1) * iden;
                const Ar ri = g * iden;
                const Ar dv = (Ar) T.dvol[i];
                const Ar six = ((Ar) rb[t].x * dv - a * s3x - alp * s2x - bet * s1x) * iden;
                const Ar siy = ((Ar) rb[t].y * dv - a * s3y - alp * s2y - bet * s1y) * iden;
                C o;
                o.x = six; o.y = siy;
                y[(size_t) i * M] = o;
                Sp[(size_t) i * M] = pi; Sq[(size_t) i * M] = qi; Sr[(size_t) i * M] = ri;
                p3 = p2; p2 = p1; p1 = pi;
                q3 = q2; q2 = q1; q1 = qi;
                r3 = r2; r2 = r1; r1 = ri;
                s3x = s2x; s2x = s1x; s1x = six;
                s3y = s2y; s2y = s1y; s1y = siy;
            }
        }
    }
    /* the relations of local rows cnt-1, cnt-2, cnt-3 (five values each) */
    xme[0 * 64] = (double) p1; xme[1 * 64] = (double) q1; xme[2 * 64] = (double) r1;
    xme[3 * 64] = (double) s1x; xme[4 * 64] = (double) s1y;
    xme[5 * 64] = (double) p2; xme[6 * 64] = (double) q2; xme[7 * 64] = (double) r2;
    xme[8 * 64] = (double) s2x; xme[9 * 64] = (double) s2y;
    xme[10 * 64] = (double) p3; xme[11 * 64] = (double) q3; xme[12 * 64] = (double) r3;
    xme[13 * 64] = (double) s3x; xme[14 * 64] = (double) s3y;
}

template <typename Ar, typename C>
static __device__ __forceinline__ void p4t_finish(C *__restrict__ y, const double *__restrict__ S, size_t M, int nz,
                                                  int side, const double *__restrict__ xt, const double *__restrict__ xb)
{
    constexpr int BT = 8;
    const int m = nz / 2, cnt = side == 0 ? m : nz - m;
    /* the 6x6 system over z_u = x_{m-3+u}: rows 0..2 the top relations of
     * R = m-3, m-2, m-1 (exported as local rows cnt-3, cnt-2, cnt-1 of the
     * top), rows 3..5 the bottom relations of R = m, m+1, m+2 */
    Ar A[6][6], bx[6], by[6];
#pragma unroll
    for (int r = 0; r < 6; r++) {
#pragma unroll
        for (int c = 0; c < 6; c++) A[r][c] = (Ar) 0;
    }
#pragma unroll
    for (int k = 0; k < 3; k++) {
        /* top: relation of R = m-1-k is the export slot k (local row cnt-1-k) */
        const int r = 2 - k;                      /* matrix row and unknown index of R */
        A[r][r] = (Ar) 1;
        A[r][r + 1] = (Ar) xt[(5 * k + 0) * 64];
        A[r][r + 2] = (Ar) xt[(5 * k + 1) * 64];
        A[r][r + 3] = (Ar) xt[(5 * k + 2) * 64];
        bx[r] = (Ar) xt[(5 * k + 3) * 64];
        by[r] = (Ar) xt[(5 * k + 4) * 64];
        /* bottom: relation of R = m+k is the export slot k (local row cnt_b-1-k) */
        const int rb = 3 + k;
        A[rb][rb] = (Ar) 1;
        A[rb][rb - 1] = (Ar) xb[(5 * k + 0) * 64];
        A[rb][rb - 2] = (Ar) xb[(5 * k + 1) * 64];
        A[rb][rb - 3] = (Ar) xb[(5 * k + 2) * 64];
        bx[rb] = (Ar) xb[(5 * k + 3) * 64];
        by[rb] = (Ar) xb[(5 * k + 4) * 64];
    }
#pragma unroll
    for (int c = 0; c < 6; c++) {
        const Ar ip = (Ar) 1 / A[c][c];
#pragma unroll
        for (int r = c + 1; r < 6; r++) {
            const Ar f = A[r][c] * ip;
#pragma unroll
            for (int k = c + 1; k < 6; k++) A[r][k] -= f * A[c][k];
            bx[r] -= f * bx[c];
            by[r] -= f * by[c];
        }
    }
    Ar zx[6], zy[6];
#pragma unroll
    for (int r = 5; r >= 0; r--) {
        Ar vx = bx[r], vy = by[r];
#pragma unroll
        for (int k = r + 1; k < 6; k++) { vx -= A[r][k] * zx[k]; vy -= A[r][k] * zy[k]; }
        const Ar ip = (Ar) 1 / A[r][r];
        zx[r] = vx * ip;
        zy[r] = vy * ip;
    }
    const double *Sp = S, *Sq = S + (size_t) nz * M, *Sr = S + (size_t) 2 * nz * M;
    /* own three unknowns of the six, then back-substitution of the rest of
     * this side, moving away from the middle */
    Ar x1x, x2x, x3x, x1y, x2y, x3y;
    if (side == 0) {
#pragma unroll
        for (int u = 0; u < 3; u++) {
            C o; o.x = zx[u]; o.y = zy[u];
            y[(size_t) (m - 3 + u) * M] = o;
        }
        x1x = zx[0]; x2x = zx[1]; x3x = zx[2]; x1y = zy[0]; x2y = zy[1]; x3y = zy[2];
    } else {
#pragma unroll
        for (int u = 3; u < 6; u++) {
            C o; o.x = zx[u]; o.y = zy[u];
            y[(size_t) (m - 3 + u) * M] = o;
        }
        x1x = zx[5]; x2x = zx[4]; x3x = zx[3]; x1y = zy[5]; x2y = zy[4]; x3y = zy[3];
    }
    for (int j0 = cnt - 4; j0 >= 0; j0 -= BT) {
        C sb[BT];
        double pb[BT], qb[BT], rbv[BT];
#pragma unroll
        for (int t = 0; t < BT; t++) {
            const int j = max(j0 - t, 0);
            const size_t o = (size_t) (side == 0 ? j : nz - 1 - j) * M;
            sb[t] = y[o]; pb[t] = Sp[o]; qb[t] = Sq[o]; rbv[t] = Sr[o];
        }
#pragma unroll
        for (int t = 0; t < BT; t++) {
            const int j = j0 - t;
            if (j >= 0) {
                const Ar xix = (Ar) sb[t].x - (Ar) pb[t] * x1x - (Ar) qb[t] * x2x - (Ar) rbv[t] * x3x;
                const Ar xiy = (Ar) sb[t].y - (Ar) pb[t] * x1y - (Ar) qb[t] * x2y - (Ar) rbv[t] * x3y;
                C o;
                o.x = xix; o.y = xiy;
                y[(size_t) (side == 0 ? j : nz - 1 - j) * M] = o;
                x3x = x2x; x2x = x1x; x1x = xix;
                x3y = x2y; x2y = x1y; x1y = xiy;
            }
        }
    }
}

template <typename T>
__global__ __launch_bounds__(128) void k_poisson4t(const RunDev R, const Pois4Tab T_,
                                                   typename Cplx<T>::type *__restrict__ Y, double *__restrict__ S)
{
    typedef typename Cplx<T>::type C;
    __shared__ double xch[2][15 * 64];
    const int ny = R.g.ny, nz = R.g.nz, nkx = R.g.nkx;
    const size_t M = (size_t) ny * nkx;
    const int lane = threadIdx.x & 63;
    const int side = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   /* 0 top, 1 bottom */
    const size_t q0 = (size_t) blockIdx.x * 64 + lane;
    const bool act = q0 < M;
    const size_t qm = act ? q0 : M - 1;           /* idle lanes repeat the last mode, and never write */
    const int kx = (int) (qm / ny), ky = (int) (qm % ny);
    const int variant = (kx == 0 && ky == 0) ? 1 : 0;
    const bool low = kx <= CF_F64_KLOW && (ky <= CF_F64_KLOW || ny - ky <= CF_F64_KLOW);
    const bool wide = sizeof(T) == sizeof(double) || low;
    /* lanes past the last mode take part in the barrier only */
    double *xme = &xch[side][lane];
    if (act) {
        if (wide) p4t_sweep<double, C>(T_, Y + qm, S + qm, M, nz, R.lamx[kx], R.lamy[ky], variant, side, xme);
        else p4t_sweep<T, C>(T_, Y + qm, S + qm, M, nz, R.lamx[kx], R.lamy[ky], variant, side, xme);
    }
    __syncthreads();
    if (!act) return;
    const double *xt = &xch[0][lane], *xb = &xch[1][lane];
    if (wide) p4t_finish<double, C>(Y + qm, S + qm, M, nz, side, xt, xb);
    else p4t_finish<T, C>(Y + qm, S + qm, M, nz, side, xt, xb);
}

template __global__ void k_poisson4t<double>(const RunDev, const Pois4Tab, double2 *, double *);
template __global__ void k_poisson4t<float>(const RunDev, const Pois4Tab, float2 *, double *);

/* ------------------------------------------------------------ projection */

/* project2/4 (pressure.c:120-195) of the mass-flux corrected solve
 * output into the state: u = (u* + h1 m) - dt dp/dx, v, w likewise (the
 * top-wall face := 0), c = c* + h1c mc.  For order 4 the first pressure
 * ghost equals the adjacent interior value (the copy row of the closure,
 * pressure.c:534-632), which w at the first and last interior face uses. */
/* (us, u), (vs, v), (ws, w) may be the same arrays (in-place projection):
 * each thread reads and writes only its own point of them */
template <int ORD, typename T>
static __device__ __forceinline__ void proj_body(const RunDev &R, const T *us,
    const T *vs, const T *ws, const T *cs,
    const double *__restrict__ h1u, const double *__restrict__ mu, const double *__restrict__ h1c,
    const double *__restrict__ mc, const T *__restrict__ p, double dtp,
    T *u, T *v, T *w, T *c, const Blk b)
{
    const T A1 = (T) A1d, A2 = (T) A2d;
    const int nx = R.g.nx, ny = R.g.ny, nz = R.g.nz, k = b.z;
    int i, j;
    if (!proj_cell(R, b, i, j)) return;
    const size_t P = (size_t) nx * ny;
    const size_t row = rowof(k, j, nx, P), q = row + i;
    const double *rdzh = R.rdzh + CF_NGT;
    const T m = mu ? (T) *mu : (T) 0;
    const T p0 = p[q];
    const int ip = wrapm(i + 1, nx), jp = wrapm(j + 1, ny);
    T gx, gy;
    if (ORD == 2) {
        gx = p[row + ip] - p0;
        gy = p[rowof(k, jp, nx, P) + i] - p0;
    } else {
        const int im = wrapm(i - 1, nx), ip2 = wrapm(i + 2, nx), jm = wrapm(j - 1, ny), jp2 = wrapm(j + 2, ny);
        gx = A1 * (p[row + ip] - p0) + A2 * (p[row + ip2] - p[row + im]);
        gy = A1 * (p[rowof(k, jp, nx, P) + i] - p0) + A2 * (p[rowof(k, jp2, nx, P) + i] - p[rowof(k, jm, nx, P) + i]);
    }
    u[q] = (us[q] + (h1u ? (T) h1u[k + 1] * m : (T) 0)) - gx * (T) (dtp * R.rdx);
    v[q] = vs[q] - gy * (T) (dtp * R.rdy);
    if (k < nz - 1) {
        const T p1 = p[q + P];
        T gz;
        if (ORD == 2) gz = p1 - p0;
        else {
            const T pm = k > 0 ? p[q - P] : p0;
            const T p2 = k + 2 < nz ? p[q + 2 * P] : p1;
            gz = A1 * (p1 - p0) + A2 * (p2 - pm);
        }
        w[q] = ws[q] - gz * (T) (dtp * rdzh[k]);
    } else {
        w[q] = (T) 0;
    }
    if (c) c[q] = cs[q] + (h1c ? (T) h1c[k + 1] * (mc ? (T) *mc : (T) 0) : (T) 0);
}

template <int ORD, typename T>
__global__ __launch_bounds__(256) void k_gproject(const RunDev R, const T *us,
    const T *vs, const T *ws, const T *cs,
    const double *__restrict__ h1u, const double *__restrict__ mu, const double *__restrict__ h1c,
    const double *__restrict__ mc, const T *__restrict__ p, double dtp,
    T *u, T *v, T *w, T *c)
{
    proj_body<ORD, T>(R, us, vs, ws, cs, h1u, mu, h1c, mc, p, dtp, u, v, w, c, blk_native());
}

template <typename T> struct GPick {
    template <int ORD, bool SC> static void fill(GSel<T> &S)
    {
        S.rhs = k_grhs<ORD, SC, T>;
        S.proj = k_gproject<ORD, T>;
    }
};

template <typename T>
GSel<T> pick_general(int order, int scalar)
{
    GSel<T> S;
    if (order == 4) {
        if (scalar) GPick<T>::template fill<4, true>(S);
        else GPick<T>::template fill<4, false>(S);
    } else {
        if (scalar) GPick<T>::template fill<2, true>(S);
        else GPick<T>::template fill<2, false>(S);
    }
    return S;
}

template GSel<double> pick_general<double>(int, int);
template GSel<float> pick_general<float>(int, int);

/* ------------------------------------------------------------ batched launches
 * Runs of one (order, scalar, precision) with any grid sizes and
 * coefficients go out together: each launch below is persistent over the
 * virtual blocks of all runs (batch_loop), each run reading its own
 * parameter block and buffers from the GArgs table.  Substep index s in
 * 0..2; s == 3 is a stand-alone projection of the state (dt = dt_adhoc). */

template <int ORD, bool SC, typename T>
__global__ __launch_bounds__(256) void kb_rhs(const GArgs<T> *__restrict__ A, const unsigned *__restrict__ vs,
                                              int nrun, int s)
{
    batch_loop(vs, nrun, [&](int r, unsigned lb) {
        const GArgs<T> &a = A[r];
        T *const *fnew = (s % 2 == 0) ? a.fa : a.fb;
        T *const *gold = (s % 2 == 0) ? a.fb : a.fa;
        GFields<T> F;
        F.u = a.u; F.v = a.v; F.w = a.w; F.c = a.c;
        for (int t = 0; t < 4; t++) { F.g[t] = gold[t]; F.f[t] = fnew[t]; }
        F.r[0] = a.ru; F.r[1] = a.rv; F.r[2] = a.rw; F.r[3] = a.rc;
        grhs_body<ORD, SC, T>(a.R, s, F, a.scal, s == 0 ? a.cflpart : (double *) nullptr, a.dt, a.part,
                              blk_of(a, ST_RHSG, lb));
    });
}

template <int ORD, typename T>
__global__ __launch_bounds__(256) void kb_proj(const GArgs<T> *__restrict__ A, const unsigned *__restrict__ vs,
                                               int nrun, int s)
{
    batch_loop(vs, nrun, [&](int r, unsigned lb) {
        const GArgs<T> &a = A[r];
        const Blk b = blk_of(a, ST_PROJ, lb);
        if (s < 3) {
            const int nz = a.R.g.nz;
            const double *h1u = a.R.h1 + (size_t) (s * 2 + 0) * (nz + 2);
            const double *h1c = a.R.h1 + (size_t) (s * 2 + 1) * (nz + 2);
            const bool sc = a.R.scalar != 0;
            proj_body<ORD, T>(a.R, a.ru, a.rv, a.rw, a.rc, h1u, a.scal + SC_M0 + s, sc ? h1c : nullptr,
                              a.scal + SC_MC0 + s, a.p, a.R.sc[s].abdt, a.u, a.v, a.w, sc ? a.c : nullptr, b);
        } else {
            proj_body<ORD, T>(a.R, a.u, a.v, a.w, nullptr, nullptr, nullptr, nullptr, nullptr, a.p, a.dt_adhoc,
                              a.u, a.v, a.w, nullptr, b);
        }
    });
}

template <typename T>
__global__ __launch_bounds__(256) void kb_solve4(const GArgs<T> *__restrict__ a_, const unsigned *__restrict__ vs, int nrun, int s)
{
    batch_loop(vs, nrun, [&](int r, unsigned lb) {
        const GArgs<T> &a = a_[r];
        solve4_body<T>(a.R, s, a.ru, a.rv, a.rw, a.rc, blk_of(a, ST_SOLVE, lb));
    });
}

template <typename T>
__global__ __launch_bounds__(256) void kb_mass(const GArgs<T> *__restrict__ a_, const unsigned *__restrict__ vs, int nrun, int s)
{
    batch_loop(vs, nrun, [&](int r, unsigned lb) {
        (void) lb;
        const GArgs<T> &a = a_[r];
        Book B;
        B.s = s;
        B.n = a.gblocks;
        B.part = a.part;
        B.cflpart = s == 0 ? a.cflpart : nullptr;
        B.scal = a.scal; B.logbuf = a.logbuf;
        B.dt = a.dt;
        book_body(a.R, B);
    });
}

template <typename T>
__global__ __launch_bounds__(256) void kb_poisson4(const GArgs<T> *__restrict__ a_, const unsigned *__restrict__ vs, int nrun, int s)
{
    batch_loop(vs, nrun, [&](int r, unsigned lb) {
        const GArgs<T> &a = a_[r];
        pois4_body<T>(a.R, a.pt4[s], a.X, a.S4, blk_of(a, ST_MODE, lb));
    });
}

#define CF_INST_B(T)                                                                                              \
    template __global__ void kb_solve4<T>(const GArgs<T> *, const unsigned *, int, int);                          \
    template __global__ void kb_mass<T>(const GArgs<T> *, const unsigned *, int, int);                            \
    template __global__ void kb_poisson4<T>(const GArgs<T> *, const unsigned *, int, int);
CF_INST_B(double)
CF_INST_B(float)
#undef CF_INST_B

template <typename T> struct BPick {
    template <int ORD, bool SC> static void fill(BSel<T> &S)
    {
        S.rhs = kb_rhs<ORD, SC, T>;
        S.proj = kb_proj<ORD, T>;
    }
};

template <typename T>
BSel<T> pick_batched(int order, int scalar)
{
    BSel<T> S;
    if (order == 4) {
        if (scalar) BPick<T>::template fill<4, true>(S);
        else BPick<T>::template fill<4, false>(S);
    } else {
        if (scalar) BPick<T>::template fill<2, true>(S);
        else BPick<T>::template fill<2, false>(S);
    }
    return S;
}

template BSel<double> pick_batched<double>(int, int);
template BSel<float> pick_batched<float>(int, int);
