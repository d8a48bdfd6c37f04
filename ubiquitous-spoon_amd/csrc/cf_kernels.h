/*
 * cf_kernels.h -- kernel parameter blocks and kernel prototypes shared
 * by cf_kernels.hip (definitions) and cf_run.hip (launches).
 */
#ifndef CF_KERNELS_H
#define CF_KERNELS_H

#include "cf_dev.h"
#include "cf_tables.h"

/* slots of the per-run device scalar block */
enum {
    SC_M0 = 0,      /* mass-flux forcing of substeps 0..2 */
    SC_MC0 = 3,     /* scalar-mean forcing of substeps 0..2 */
    SC_STEP = 6,    /* completed steps */
    SC_CFL = 7,     /* cfl at the start of the current step */
    SC_ZERO = 8,    /* always 0 */
    SC_CFL0 = 9,    /* cflmode 1: cfl of the state at the start of a step, with the previous dt */
    SC_TICKET = 10, /* kb_level_mass: workgroups done, a 32-bit counter (0 between launches) */
    SC_N = 16
};

#define CF_MAX_RAD 16
#ifndef CF_RHS_WAVES
#define CF_RHS_WAVES 3          /* occupancy target (waves per SIMD) of k_rhs2t */
#endif
/* xy tile of the fast-path RHS (one thread per column, 256 threads; 32 x 8 measured faster
 * than 64 x 4 and 16 x 16 at 256x193x256) */
#define CF_RT_X 32
#define CF_RT_Y 8
#ifndef CF_RHS_KC
#define CF_RHS_KC 16             /* target levels per z-chunk of k_rhs2t (16: 264 us, 24: 270 us, 32: 266 us at 256x193x256) */
#endif
#ifndef CF_RHS_KC_BATCH
#define CF_RHS_KC_BATCH 24       /* ... of kb_rhs2t, whose launches cover many runs */
#endif
/* xy tile of the fused order-4 RHS (k_rhs4t); nx and ny must be multiples */
#define CF_R4_X 32
#define CF_R4_Y 8
#ifndef CF_R4_KC
#define CF_R4_KC 8               /* target levels per z-chunk of the order-4 RHS (8: 153 us, 16: 164 us, 32: 198 us per launch at 192x129x192) */
#endif
#ifndef CF_R4_WAVES
#define CF_R4_WAVES 2            /* occupancy target (waves per SIMD) of the order-4 RHS */
#endif
#define CF_SPIKE_LMAX 32        /* rows per chunk held in registers */
#define CF_SPIKE_SMAX 8         /* chunks (waves) per workgroup */
#define CF_F64_KLOW 4           /* FP32 runs solve Poisson modes |kx|, |ky| <= this in FP64 */

/* Partitioned (spike) solve of one constant-coefficient tridiagonal
 * system split into S chunks of L rows: per-chunk Thomas factors, the
 * left/right spike vectors and the inverse of the 2S x 2S interface
 * system, all column-independent (host-built). */
struct SpikeTab {
    int n, S, L;
    const double *a, *ib, *gam, *vl, *wr, *minv;
};

/* order-4 partitioned z solve of one system over n unknowns, S chunks of L
 * rows (cf_spike4.hip): f = 7 S L chunk-local heptdag factors
 * (a | al | be | iden | p | q | r), vw = 6 S L spikes (three left, three
 * right), minv = the inverse interface system, 6 CF_SPIKE4_SMAX square */
struct Spike4Tab {
    int n, S, L;
    const double *f, *vw, *minv;
};

/* ghost closures of cell (Dirichlet) and face fields at both walls */
struct Clos {
    Clos1 cell[2], face[2];     /* [0] bottom, [1] top */
};

/* factors of one wall-reduced order-4 z system over n unknowns:
 * t[0..7n) = a | al | be | iden | p | q | r (cf_tables.h, hept_factor) */
struct HeptTab {
    int n;
    const double *t;
};

/* order-4 Poisson z-tables for one dt: the wall-reduced bands at zero
 * horizontal wavenumber for the Neumann bottom (band[0]) and the
 * Dirichlet-mean bottom of the (0,0) mode (band[1]), 7 nz each (column
 * offsets -3..+3, level fastest), the diagonal shifts per unit modified
 * wavenumber and the volumes (pressure.c:357-444) */
struct Pois4Tab {
    const double *band[2];
    const double *ex, *ey, *dvol;
};

/* Everything a substep kernel needs that is fixed for the run: passed by
 * value (a few hundred bytes of kernel arguments). */
struct RunDev {
    Grid g;
    const double *dzt;          /* nz + 6: dzt[k + 3] = dz of level k (mirrored ghosts) */
    SubCoef sc[3];
    double nu, prandtl;
    double ubc, vbc, cbot, ctop;
    double lift[3][4];          /* boundary lift of u (bot, top) and v (bot, top), per substep */
    int m_prev_slot[3];         /* scalar slot holding the previous substep's forcing */
    const double *th;           /* Thomas factors [s][type 0..3][a, ibet, gam][nz] */
    SpikeTab sp[3][3];          /* [s][type 0 cell-nu, 1 cell-kappa, 2 face-nu] */
    const double *rdz;          /* 1 / dz, level-indexed like dzt (offset CF_NGT) */
    const double *rdzh;         /* 1 / (0.5 (dz_k + dz_k+1)), offset CF_NGT */
    double rdx, rdy, rdxdy;
    double rnx;                 /* 1 / nx, for qdiv */
    const double *stat1;        /* [s][kind][vol1, bot1, top1, cl1] */
    const double *h1;           /* [s][kind][nz + 2] unit-forcing profile, level k at k + 1 */
    /* the constraint's statistics of the solved field (bulk value, bottom and
     * top wall gradient, centreline) as weighted sums: over the plane means A
     * of the solution, l . A + mcf with l = mlf [kind][4][nz]; over the means
     * of the solve's right-hand side, with mwq = (solve)^-T l [s][kind][nz][4] */
    const double *mwq, *mlf;
    double mcf[2][4];
    int cmode[2];
    double ctarget[2], cfixed[2];
    int logcap;
    double cfl_log;             /* > 0: the cfl.dat value of the step (cflmode 1 logs want_cfl) */
    /* FFT plans */
    int radx[CF_MAX_RAD], nradx, rady[CF_MAX_RAD], nrady;
    const double2 *twx, *twy;
    const float2 *twx32, *twy32;  /* the same twiddles rounded to FP32 */
    const double *lamx, *lamy;  /* modified wavenumbers 2 - 2 cos(2 pi k / n) */
    /* complex x lines per block: the inverse x FFT, the divergence + x FFT,
     * the forward x FFT on its own */
    int fx_pairs, dx_pairs, px_pairs;
    int fy_cols;                /* kx columns per y-FFT block */
    /* general path (order 4 and/or the scalar) */
    Clos cl;
    int scalar;
    double betg[3];
    double kap;                 /* scalar diffusivity nu / Pr */
    const double *liftg;        /* [s][field u, v, w, c][nz] boundary-lift profiles */
    HeptTab hp[3][3];           /* order-4 implicit z factors [s][type 0 cell-nu, 1 cell-kappa, 2 face-nu] */
    Spike4Tab s4[3][3];         /* ... as partitioned-solve tables (n = 0: none) */
    int implicit;               /* 1: every diffusion term implicit (channel2/4): x-y diffusion in h, not f */
    /* FP32 storage on the fused path: u is stored as u - U(z), U a per-level
     * FP64 profile, so storage rounding scales with the deviation from U
     * instead of with u.  Layout: [nz + 2] U with the wall ghosts at 0 and
     * nz + 1, then [3][nz] U's share of each substep's implicit right-hand
     * side.  Null: no offset (FP64, or the general path). */
    const double *uoff;
};

/* A workgroup's coordinates in one run's launch grid: blockIdx / gridDim
 * of a single-run launch, or decoded from a batched launch's virtual block. */
struct Blk {
    unsigned x, y, z, nx, ny, nz;
};
static __device__ __forceinline__ Blk blk_native()
{
    Blk b;
    b.x = blockIdx.x; b.y = blockIdx.y; b.z = blockIdx.z;
    b.nx = gridDim.x; b.ny = gridDim.y; b.nz = gridDim.z;
    return b;
}

/* The cells that a projection's 256-thread workgroup takes.  Rows that start
 * where a cache line does and leave at most one lane in five idle go in tiles
 * of 64 x 4: p's rows above and below serve four rows (order 2 at 256x65x256
 * 37.6 us, 256 consecutive cells of a level 41.0, at 160x97x150 26.2 and 28.1;
 * order 4 with the scalar at 192x65x192 30.6 and 32.7, at 120x65x125 16.1 and
 * 19.7).  Other rows go as consecutive cells (90x129x90 12.0 us, in tiles
 * 17.1; 300x65x300 57 and 61, in FP32 30 and 39; order 4 with the scalar at
 * 250x65x250 alone 72 and 68). */
static inline __host__ __device__ bool proj_tiles(int nx)
{
    const int full = (nx + 63) & ~63;
    return (nx & 7) == 0 && 5 * (full - nx) <= full;
}
struct ProjGrid { unsigned x, y; };
static inline ProjGrid proj_blocks(int nx, int ny)
{
    ProjGrid g;
    if (proj_tiles(nx)) { g.x = (unsigned) (nx + 63) / 64; g.y = (unsigned) (ny + 3) / 4; }
    else { g.x = ((unsigned) nx * (unsigned) ny + 255) / 256; g.y = 1; }
    return g;
}
/* cell (i, j) of this thread in workgroup b; false: none */
static __device__ __forceinline__ bool proj_cell(const RunDev &R, const Blk &b, int &i, int &j)
{
    const int nx = R.g.nx, t = threadIdx.x;
    if (proj_tiles(nx)) {
        i = (int) b.x * 64 + (t & 63);
        j = (int) b.y * 4 + (t >> 6);
        return i < nx && j < R.g.ny;
    }
    const int e = (int) b.x * 256 + t;
    if (e >= nx * R.g.ny) return false;
    j = qdiv(e, nx, R.rnx);
    i = e - j * nx;
    return true;
}

/* the column block of workgroup b (nbx of them a field) of a z solve */
static __device__ __forceinline__ Blk blk_solve(unsigned b, unsigned nbx)
{
    Blk r;
    r.y = 0;
    while (b >= nbx) { b -= nbx; r.y++; }   /* at most three times */
    r.x = b;
    r.z = 0;
    r.nx = nbx; r.ny = 4; r.nz = 1;
    return r;
}

/* launch stages of a batched step; each run's grid per stage is dims[stage] */
enum { ST_PROJ = 0, ST_RHSG, ST_SOLVE, ST_ONE, ST_DIVX, ST_FFTX, ST_FFTY, ST_MODE, ST_RHS2, ST_LEVEL, CF_NST };
#define CF_BATCH_MAX 256        /* runs per batched launch */

/* Where a substep's projected velocity comes from: the previous
 * substep's solve output, its pressure, mass-flux profile and forcing
 * (h1, m may be null: no correction) and its projection dt. */
template <typename T> struct ProjSrcT {
    const T *us, *vs, *ws, *p;               /* state of storage type T */
    const double *h1, *m;
    double dtp;
};
typedef ProjSrcT<double> ProjSrc;

/* z-tables of the Poisson operator for one dt (pressure.c:318-339) */
struct PoisTab {
    const double *a, *c, *bz, *ex, *ey, *dvol;
    double db_neu, db_dir, db_top;
};

/* z-solve chunk lengths compiled for the spike kernels: a run's tables
 * hold L rows per chunk, L the smallest of these with CF_SPIKE_SMAX L >= nz
 * (0: nz beyond CF_SPIKE_SMAX CF_SPIKE_LMAX, Thomas instead) */
#define CF_SPIKE_LSET(X) X(4) X(6) X(8) X(10) X(12) X(14) X(16) X(20) X(24) X(28) X(32)
static inline int spike_L(int nz)
{
    static const int set[] = { 4, 6, 8, 10, 12, 14, 16, 20, 24, 28, 32 };
    /* six chunks where a compiled length gives exactly six (measured faster
     * than seven at nz = 65 and 129; nz = 97 would round to five, slower) */
    const int need6 = (nz + 5) / 6;
    for (int l : set)
        if (l >= need6) {
            if ((nz + l - 1) / l == 6) return l;
            break;
        }
    const int need = (nz + CF_SPIKE_SMAX - 1) / CF_SPIKE_SMAX;
    for (int l : set)
        if (l >= need) return l;
    return 0;
}

/* order-4 spike solve: at most CF_SPIKE4_SMAX chunks of L rows, L a
 * compiled length; one L serves the cell (nz) and face (nz - 1) systems,
 * and every chunk but a system's last has L >= 6 rows, the last >= 3, so
 * a chunk's three-row couplings reach only its neighbours (0: none fits,
 * the sequential sweep instead) */
#define CF_SPIKE4_SMAX 8
#define CF_SPIKE4_LSET(X) X(6) X(8) X(10) X(12) X(14) X(16) X(18) X(20) X(24) X(28) X(32)
static inline int spike4_L(int nz)
{
    static const int set[] = { 6, 8, 10, 12, 14, 16, 18, 20, 24, 28, 32 };
    auto fits = [](int n, int l) {
        const int S = (n + l - 1) / l;
        return S <= CF_SPIKE4_SMAX && (S == 1 || n - (S - 1) * l >= 3);
    };
    for (int l : set)
        if (fits(nz, l) && fits(nz - 1, l)) return l;
    return 0;
}

/* LDS of the FFT kernels: lines of n elements at stride fft_ld(n), then
 * the n twiddles of the passes, staged once per workgroup */
#ifndef CF_FFT_PAD
#define CF_FFT_PAD 1
#endif
static inline __host__ __device__ int fft_ld(int n) { return n + CF_FFT_PAD; }
/* FFT lengths done in two register passes, n = P1 P2 (P1 = fft2_p1(n),
 * 0 for the Stockham passes): the y FFT (CF_FY2), the inverse x FFT and
 * the order-2 divergence + x FFT (CF_FX2) where they measured faster than
 * the Stockham passes -- the inverse x FFT in FP32 and for lengths up to
 * 128 in FP64, the divergence in FP32 at 256 (esz: bytes per stored real) */
#ifndef CF_FY2
#define CF_FY2 1
#endif
#ifndef CF_FX2
#define CF_FX2 1
#endif
static constexpr __host__ __device__ int fft2_p1(int n) { return n == 256 ? 16 : (n == 128 || n == 64 ? 8 : 0); }
static constexpr __host__ __device__ int fy2_p1(int n) { return CF_FY2 ? fft2_p1(n) : 0; }
static constexpr __host__ __device__ int fx2_p1(int n) { return CF_FX2 ? fft2_p1(n) : 0; }
static constexpr __host__ __device__ bool fxi2_on(int n, int esz) { return fx2_p1(n) > 0 && (esz == 4 || n <= 128); }
static constexpr __host__ __device__ bool divx2_on(int n, int esz) { return fx2_p1(n) > 0 && esz == 4 && n == 256; }
/* y lines sit in LDS as P1 rows of P2 + 1 */
static inline __host__ __device__ int fy_ld(int n) { return fy2_p1(n) ? n + fy2_p1(n) : fft_ld(n); }
/* x line pairs: P1 rows of P2 + 1 and 2 more, so the unpacking writes of
 * neighbouring pairs (lanes along the pair) fall on distinct bank groups */
static constexpr __host__ __device__ int fx_ld(int n, int esz)
{
    return fxi2_on(n, esz) ? n + fx2_p1(n) + 2 : n + CF_FFT_PAD;
}
/* line pairs per x-FFT workgroup: CF_FX_ELEMS complex elements (at least
 * one pair); 2048 where the two-pass forms run, so that a pass has 128 or
 * 256 (pair, column) tasks.  The Stockham kernels take the pair count
 * from the run (RunDev::fx_pairs); the two-pass ones compile it in, and
 * for their lengths it does not depend on the element size, except at 256,
 * whose two-pass forms are FP32 only (FP32 runs launch FP64 x FFTs only
 * through the Stockham kernels there). */
#ifndef CF_FX_ELEMS
#define CF_FX_ELEMS 1024
#endif
static constexpr __host__ __device__ int fx_pairs_of(int nx, int esz)
{
    return fxi2_on(nx, esz) ? 2048 / nx : (CF_FX_ELEMS / nx > 0 ? CF_FX_ELEMS / nx : 1);
}
/* ... per workgroup of the divergence + x FFT: as many elements as its 256
 * threads gather in one round of loads (two each, three in FP32), so that a
 * workgroup waits for memory once (64 x 65 x 64 in FP64: 8 pairs 7.3 us, 32
 * pairs 15.3); at 256 the pair counts its register passes are built for */
static constexpr __host__ __device__ int dx_pairs_of(int nx, int esz)
{
    if (divx2_on(nx, esz) || nx == 256) return fx_pairs_of(nx, esz);
    const int e = esz == 4 ? 768 : 512;
    return e / nx > 0 ? e / nx : 1;
}

/* lengths whose divergence + x FFT is compiled for batches of an order and
 * element size: those without register spills */
static inline bool bdivx_compiled(int order, int n, int esz)
{
    return order == 2 && (n == 32 || n == 48 || n == 64 || n == 96 || n == 128 || (n == 192 && esz == 8));
}
/* FFT lengths with their plan compiled in (single runs) */
#define CF_FFT_SIZES(X) X(16) X(20) X(24) X(30) X(32) X(40) X(48) X(60) X(64) X(80) X(96) \
    X(120) X(128) X(160) X(192) X(240) X(256) X(320) X(384) X(480) X(512)
static inline bool fft_compiled(int n)
{
    switch (n) {
#define X_(N) case N:
    CF_FFT_SIZES(X_)
#undef X_
        return true;
    default: return false;
    }
}

/* ... per workgroup of a single run's divergence + x FFT (paired: at
 * order 2, whose compiled lengths have a second instance for it) and of its
 * forward x FFT.  Few pairs are few consecutive lines, so a mode's
 * half-spectrum values go out in short runs (one pair: 32 bytes in FP64); a
 * grid of many lines is bound by those stores and takes full workgroups,
 * once there are two of them for each CU.  With fewer the one round of loads
 * counts for more (400 x 33 x 32: 14.8 us, full 16.9).  One round -> full
 * (us): run-time plans 300 x 65 x 150 FP64 53 -> 37, 400 x 129 x 400 FP64
 * 375 -> 298, FP32 260 -> 210; compiled lengths, which lose less to short
 * runs and more to a second round, two pairs instead of one at order 2 (384
 * x 129 x 384 203 -> 171, FP32 512 x 129 x 512 240 -> 189) and none at order
 * 4 (one pair 512 x 65 x 256 80, two 89); the order-4 implicit solves,
 * forward x FFT included, 384 x 129 x 384 1,547 -> 1,357 a substep */
static inline int run_dx_pairs(int nx, int esz, bool paired, long npairs)
{
    const int one = dx_pairs_of(nx, esz), most = 1024 / nx;
    const int full = fft_compiled(nx) ? (paired && one == 1 && most >= 2 ? 2 : one) : (one < 4 && most > one ? most : one);
    return npairs / full >= 512 ? full : one;
}

#ifndef CF_P2S_NC
#define CF_P2S_NC 16
#endif
#ifndef CF_P2S_MW
#define CF_P2S_MW 16
#endif
#ifndef CF_P2S_XCD
#define CF_P2S_XCD 1
#endif
/* order-2 Poisson: the partitioned solve (at most 16 z-chunks of L rows
 * per mode, 16 modes per 256-thread workgroup), L a compiled chunk length
 * >= nz / 16, covers nz <= 512; beyond that one thread per mode (256
 * modes per workgroup). */
#define CF_P2S_LSET(X) X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(11) X(12) X(13) X(14) X(15) X(16) \
                       X(20) X(24) X(28) X(32)
static inline int pois2_L_of(int need)
{
    static const int set[] = { 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15, 16, 20, 24, 28, 32 };
    for (int l : set)
        if (l >= need) return l;
    return 0;
}
/* chunk length for nz (0: one thread per mode) */
static inline int pois2_L(int nz) { return pois2_L_of((nz + CF_P2S_NC - 1) / CF_P2S_NC); }
/* dynamic LDS of the partitioned solve: its six z tables in FP64 (an all-FP32
 * launch uses half of it) */
static inline size_t pois2_lds(int L, int nz) { return L > 0 ? 6 * sizeof(double) * (size_t) nz : 0; }
/* workgroup shape: CF_P2S_NC z-chunks x CF_P2S_MW modes; a z-level of the
 * group is CF_P2S_MW contiguous complex values (256 B in FP64) */
#define CF_P2S_THREADS (CF_P2S_NC * CF_P2S_MW)
/* modes per workgroup: CF_P2S_MW partitioned, or one per thread (L = 0) */
static inline size_t pois2_modes_per_block(int L) { return L > 0 ? CF_P2S_MW : CF_P2S_THREADS; }
static inline unsigned pois2_blocks(int L, size_t M)
{
    const size_t per = pois2_modes_per_block(L);
    return (unsigned) ((M + per - 1) / per);
}
/* FP32 storage: the leading workgroups of the order-2 Poisson grid that
 * can hold an FP64 island mode (kx <= CF_F64_KLOW: modes below
 * (CF_F64_KLOW + 1) ny in the kx-major order) */
static inline unsigned pois2_island_blocks(int L, int ny, size_t M)
{
    const size_t per = pois2_modes_per_block(L);
    const size_t n = ((size_t) (CF_F64_KLOW + 1) * (size_t) ny + per - 1) / per;
    const unsigned all = pois2_blocks(L, M);
    return n < all ? (unsigned) n : all;
}

/* One run of a batched launch: its parameter block, buffers (storage
 * precision T), Poisson tables and per-stage grid shapes.  An array of
 * these lives in device memory; batched kernels read the entry of the run
 * a virtual block belongs to. */
template <typename T> struct GArgs {
    RunDev R;
    T *u, *v, *w, *c, *ru, *rv, *rw, *rc, *fa[4], *fb[4], *p;
    typename Cplx<T>::type *X;
    double *G, *S4, *scal, *logbuf, *part, *cflpart, *lsum;
    double dt;                  /* step */
    double dt_adhoc;            /* dt of a stand-alone projection (substep index 3) */
    int gblocks;                /* CFL partials of the run's RHS launch */
    int rhs_kc;                 /* levels per z-chunk of the fast-path RHS */
    PoisTab pt[4];              /* substeps 0..2, stand-alone projection */
    Pois4Tab pt4[4];
    unsigned dims[CF_NST][3];
};

/* Persistent loop of a batched launch: vstart[0..nrun] is the prefix of the
 * runs' virtual block counts for this stage; each workgroup walks virtual
 * blocks vb = blockIdx.x, + gridDim.x, ..., finds the run by binary search
 * and calls fn(run, local block).  A barrier separates iterations (bodies
 * reuse their LDS). */
template <typename F>
static __device__ __forceinline__ void batch_loop(const unsigned *__restrict__ vstart, int nrun, F &&fn)
{
    __shared__ unsigned lvs[CF_BATCH_MAX + 1];
    const int tid = threadIdx.x + threadIdx.y * blockDim.x;
    const int nt = blockDim.x * blockDim.y;
    for (int t = tid; t <= nrun; t += nt) lvs[t] = vstart[t];
    __syncthreads();
    /* every thread searches for the same virtual block, so the run and the
     * local block are workgroup-uniform: readfirstlane keeps them (and the
     * argument-table loads they index) in scalar registers */
    const unsigned total = (unsigned) __builtin_amdgcn_readfirstlane((int) lvs[nrun]);
    for (unsigned vb = blockIdx.x; vb < total; vb += gridDim.x) {
        int lo = 0, hi = nrun - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            const unsigned v = (unsigned) __builtin_amdgcn_readfirstlane((int) lvs[mid]);
            if (v <= vb) lo = mid; else hi = mid - 1;
        }
        const unsigned lb = vb - (unsigned) __builtin_amdgcn_readfirstlane((int) lvs[lo]);
        fn(lo, lb);
        __syncthreads();
    }
}

/* local block index -> Blk in a run's grid of the given stage */
template <typename T>
static __device__ __forceinline__ Blk blk_of(const GArgs<T> &a, int stage, unsigned lb)
{
    Blk b;
    b.nx = a.dims[stage][0]; b.ny = a.dims[stage][1]; b.nz = a.dims[stage][2];
    b.x = lb % b.nx;
    const unsigned r = lb / b.nx;
    b.y = r % b.ny;
    b.z = r / b.ny;
    return b;
}

/* The RunDev that is a kernel's first argument, where it lies in the
 * argument segment.  A kernel that reaches the parameter block through
 * selected addresses (the wall closures of several fields) otherwise copies
 * the whole of it to scratch memory first: 2.2 KB a lane. */
static __device__ __forceinline__ const RunDev &kernarg_run()
{
    return *(const RunDev *) (cp<RunDev>) __builtin_amdgcn_kernarg_segment_ptr();
}

/* Values that the workgroups of one launch hand to the last of them: stored
 * and read at device scope, so they pass the caches that the XCDs do not
 * share, and no cache has to be written back or invalidated (a release
 * fence per workgroup wrote the dirty L2 lines of the whole XCD back:
 * 200 us over the 4644 workgroups of one plane sum). */
static __device__ __forceinline__ void dev_store(double *p, double v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
static __device__ __forceinline__ double dev_load(const double *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

/* True in the last of n workgroups to call it, counted with a device-scope
 * ticket.  Thread 0 waits for its own dev_stores to complete before it
 * counts, so the last workgroup's dev_loads see those of every other.  Only
 * which workgroup is last is a race.  The last one ends with ticket_reset;
 * the next launch starts from 0.  (1-D workgroups.) */
static __device__ __forceinline__ bool last_block(double *__restrict__ scal, unsigned n)
{
    __shared__ int last;
    if (threadIdx.x == 0) {
        __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
        last = __hip_atomic_fetch_add((unsigned *) (scal + SC_TICKET), 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
               == n - 1;
    }
    __syncthreads();
    return last != 0;
}
static __device__ __forceinline__ void ticket_reset(double *__restrict__ scal)
{
    __hip_atomic_store((unsigned *) (scal + SC_TICKET), 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

/* The cfl.dat record of a step that starts with CFL number mx (one thread) */
static __device__ __forceinline__ void cfl_record(const RunDev &R, double mx, double dt, double *__restrict__ scal,
                                                  double *__restrict__ logbuf)
{
    long idx = (long) scal[SC_STEP] % R.logcap;
    double *lg = logbuf + (size_t) idx * 13;
    for (int t = 0; t < 13; t++) lg[t] = 0.0;
    lg[0] = scal[SC_STEP] + 1.0;
    lg[1] = dt;
    lg[2] = R.cfl_log > 0.0 ? R.cfl_log : mx;
    scal[SC_CFL] = lg[2];
}

/* The forcing of kind 0 (u, chanfast.c:485-530) or 1 (c, :572-617) of
 * substep s from the statistics v of the solved field (bulk value, bottom
 * and top wall gradient, centreline; the last three in the last substep
 * only) and the unit forcing's (stat1), and in the last substep the
 * pstat / cstat record (one thread) */
static __device__ __forceinline__ void force_record(const RunDev &R, int s, int kind, const double v[4],
                                                    double *__restrict__ scal, double *__restrict__ logbuf)
{
    const double *s1 = R.stat1 + (size_t) (s * 2 + kind) * 4;   /* vol1, bot1, top1, cl1 */
    const double m = R.cmode[kind] == 1 ? (R.ctarget[kind] - v[0]) / s1[0] : R.cfixed[kind];
    scal[(kind == 0 ? SC_M0 : SC_MC0) + s] = m;
    if (s == 2) {
        long idx = (long) scal[SC_STEP] % R.logcap;
        double *lg = logbuf + (size_t) idx * 13 + (kind == 0 ? 3 : 8);
        lg[0] = m; lg[1] = v[1] + s1[1] * m; lg[2] = v[2] + s1[2] * m; lg[3] = v[0] + s1[0] * m; lg[4] = v[3] + s1[3] * m;
    }
}

/* Bookkeeping of a substep by one workgroup, from the RHS launch's partial
 * sums, beside the z solve (whose result it does not need): the plane
 * averages of the solved field that the constraint takes (get_xy_avg,
 * get.c:281-307; get_z_avg, :490-502) are linear in the right-hand side,
 * and the solve is the same for every column, so
 *   l . mean(S^-1 r) = (S^-T l) . mean(r),
 * a weighted sum that the RHS kernels form on the way.  Reading the solved
 * field again, in one or two launches between the solve and the
 * divergence, took 5 us of every substep of a small grid, 12 at
 * 256x193x256 and 20 at 192x129x192 with the scalar.
 * n workgroups of the RHS launch each left a partial sum per statistic:
 * part [kind][4][n]. */
struct Book {
    int s, n;
    const double *part, *cflpart;           /* cflpart: the first substep's n CFL maxima, else null */
    double *scal, *logbuf;
    double dt;
};
static __device__ __forceinline__ constexpr int book_stats(int s) { return s == 2 ? 4 : 1; }

/* one thread's share: v[0..7] the statistics of u and c, v[8] the CFL
 * maximum; NF statistics, KINDS fields at compile time, so that the loads of
 * four rounds of every array are in flight together */
template <int NF, int KINDS, bool CFL>
static __device__ __forceinline__ void book_share(const Book &B, double v[9])
{
    const gp<const double> p = (gp<const double>) B.part, cf = (gp<const double>) B.cflpart;
    const int nt = blockDim.x;
    for (int e0 = threadIdx.x; e0 < B.n; e0 += 4 * nt) {
        double x[4][NF * KINDS], c[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int e = e0 + u * nt, ec = e < B.n ? e : B.n - 1;
#pragma unroll
            for (int q = 0; q < NF * KINDS; q++) {
                const double t = p[(size_t) (q / NF * 4 + q % NF) * B.n + ec];
                x[u][q] = e < B.n ? t : 0.0;
            }
            c[u] = CFL ? cf[ec] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
#pragma unroll
            for (int q = 0; q < NF * KINDS; q++) v[q / NF * 4 + q % NF] += x[u][q];
            if (CFL) v[8] = fmax(v[8], c[u]);
        }
    }
}

static __device__ __forceinline__ void book_body(const RunDev &R, const Book &B)
{
    __shared__ double sh[9][8];             /* up to eight waves */
    const int nt = blockDim.x, nw = nt >> 6, tid = threadIdx.x, nz = R.g.nz, s = B.s;
    const int kinds = R.scalar ? 2 : 1, nf = book_stats(s);
    const double scale = 1.0 / ((double) R.g.nx * (double) R.g.ny);
    double v[9];
#pragma unroll
    for (int q = 0; q < 9; q++) v[q] = 0.0;
    if (s == 2) {
        if (kinds == 2) book_share<4, 2, false>(B, v);
        else book_share<4, 1, false>(B, v);
    } else if (B.cflpart) {
        if (kinds == 2) book_share<1, 2, true>(B, v);
        else book_share<1, 1, true>(B, v);
    } else {
        if (kinds == 2) book_share<1, 2, false>(B, v);
        else book_share<1, 1, false>(B, v);
    }
#pragma unroll
    for (int q = 0; q < 8; q++) v[q] *= scale;
    if (R.uoff) {                           /* stored u is u - U(z): the profile's share */
        const cp<double> U = (cp<double>) R.uoff + 1, l = (cp<double>) R.mlf;
        for (int k = tid; k < nz; k += nt) {
#pragma unroll
            for (int f = 0; f < 4; f++)
                if (f < nf) v[f] += l[f * nz + k] * U[k];
        }
    }
#pragma unroll
    for (int q = 0; q < 9; q++) {
        const double w = q == 8 ? wave_max_nonneg(v[q]) : wave_sum(v[q]);
        if ((tid & 63) == 0) sh[q][tid >> 6] = w;
    }
    __syncthreads();
    if (tid != 0) return;
    for (int q = 0; q < 9; q++) {
        double t = sh[q][0];
        for (int w = 1; w < nw; w++) t = q == 8 ? fmax(t, sh[q][w]) : t + sh[q][w];
        v[q] = t;
    }
    if (B.cflpart) cfl_record(R, v[8], B.dt, B.scal, B.logbuf);
    for (int kind = 0; kind < kinds; kind++) {
        double a[4];
        for (int f = 0; f < 4; f++) a[f] = v[4 * kind + f] + R.mcf[kind][f];
        force_record(R, s, kind, a, B.scal, B.logbuf);
    }
    if (s == 2) B.scal[SC_STEP] += 1.0;
}

/* The statistics' partial sums (SUMS) and the CFL maximum (CFL) of one
 * 256-thread workgroup of a marching RHS kernel, substep s: a[f] the thread's
 * weighted sums, cfl its maximum; sh: 20 doubles of LDS. */
template <int s, bool SUMS, bool CFL>
static __device__ __forceinline__ void book_store(double *part_, unsigned n, unsigned blk, int tid, const double a[4],
                                                  double *sh, double *cflpart_, double cfl)
{
    const gp<double> part = (gp<double>) part_, cflpart = (gp<double>) cflpart_;
    const int wave = tid >> 6;
    const bool lane0 = (tid & 63) == 0;
#pragma unroll
    for (int f = 0; f < (SUMS ? book_stats(s) : 0); f++) {
        const double w = wave_sum(a[f]);
        if (lane0) sh[4 * f + wave] = w;
    }
    if constexpr (CFL) {
        const double w = wave_max_nonneg(cfl);
        if (lane0) sh[16 + wave] = w;
    }
    __syncthreads();
    if (SUMS && tid < book_stats(s))
        part[(size_t) tid * n + blk] = ((sh[4 * tid] + sh[4 * tid + 1]) + sh[4 * tid + 2]) + sh[4 * tid + 3];
    if (CFL && tid == 0) cflpart[blk] = fmax(fmax(sh[16], sh[17]), fmax(sh[18], sh[19]));
}

/* off (may be null): a per-level profile subtracted on the way in and
 * added on the way out */
template <typename T> __global__ void k_io_to_dev(const double *io, T *dev, int nx, int ny, int nz, const double *off);
template <typename T> __global__ void k_dev_to_io(const T *dev, double *io, int nx, int ny, int nz, const double *off);
/* The z solves of a single run: workgroup 0 does the substep's bookkeeping,
 * the others solve nbx column blocks of each field in turn. */
template <typename T> using k_zsolve_t = void (*)(const RunDev, const int, const int, T *, T *, T *, T *, const Book);
template <typename T>
__global__ void k_thomas(const RunDev R, const int s, const int nbx, T *ru, T *rv, T *rw, T *rc, const Book B);
template <typename T> using k_spike_t = k_zsolve_t<T>;
__global__ void k_book(const RunDev R, const Book B);
template <typename T> k_spike_t<T> pick_spike(int L);
template <typename T> k_spike_t<T> pick_spike4(int L);
template <typename T>
__global__ void k_cfl_plain(const RunDev R, const T *u, const T *v, const T *w, double dt, double *part);
__global__ void k_cfl_reduce(const double *part, int nb, double *scal);
/* kernel pointer types of the FFT passes for storage precision T */
template <typename T> struct KSel {
    typedef typename Cplx<T>::type C;
    typedef void (*div_t)(const RunDev, const T *, const T *, const T *, const double *, const double *, C *);
    typedef void (*ffty_t)(const RunDev, C *, int);
    typedef void (*fftxi_t)(const RunDev, const C *, T *);
    typedef void (*pois2_t)(const RunDev, const PoisTab, C *, double *);
    typedef void (*rhs2_t)(const RunDev, const ProjSrcT<T>, const T *, const T *, const T *, const double *, T *, T *, T *,
                           T *, T *, T *, double *, double, int, double *);
};
typedef void (*k_fftx_plain_t)(const RunDev, const double *, double2 *);
template <typename T> typename KSel<T>::rhs2_t pick_rhs2(int s);
template <typename T> typename KSel<T>::div_t pick_div_fftx(int nx, int order, int pairs);
k_fftx_plain_t pick_fftx_plain(int nx);
template <typename T> typename KSel<T>::ffty_t pick_ffty(int ny);
template <typename T> typename KSel<T>::fftxi_t pick_fftx_inv(int nx);
template <typename T> typename KSel<T>::pois2_t pick_poisson2(int lmax);
KSel<float>::pois2_t pick_poisson2_islands(int lmax);
/* levels of a field's part of G: the one-thread-per-mode solve's checkpoints */
#define CF_P2_GLEV(nz) ((nz) > 3 * (((nz) + 15) / 16) ? (size_t) (nz) : (size_t) 3 * (((nz) + 15) / 16))
typedef void (*k_hsolve2_t)(const RunDev, const PoisTab, const PoisTab, const PoisTab, int, double2 *, double *, const Book);
k_hsolve2_t pick_hsolve2(int lmax);
/* ALL: no output is null */
template <typename T, bool ALL>
__global__ void k_project2(const RunDev R, const T *us, const T *vs, const T *ws, const double *h1, const double *mptr,
                           const T *p, double dtp, T *u, T *v, T *w);
template <typename T>
__global__ void k_maxdiv_part(const RunDev R, const T *u, const T *v, const T *w, double *part, int nb);

/* general path (cf_general.hip), storage and arithmetic precision T */
/* the fields of one substep: state, previous tendencies, new tendencies,
 * right-hand sides (u, v, w, c) */
template <typename T> struct GFields {
    const T *u, *v, *w, *c;
    const T *g[4];
    T *f[4], *r[4];
};
template <typename T> struct GSel {
    typedef void (*rhs_t)(const RunDev, const int, const GFields<T>, const double *, double *, double, double *);
    typedef void (*proj_t)(const RunDev, const T *, const T *, const T *, const T *, const double *,
                           const double *, const double *, const double *, const T *, double, T *, T *, T *, T *);
    rhs_t rhs;
    proj_t proj;
};
template <typename T> GSel<T> pick_general(int order, int scalar);

/* the order-4 explicit stage (cf_rhs4.hip): u and v in one launch, w and c
 * in another; grid (nx / CF_R4_X) * (ny / CF_R4_Y) * nch blocks of 256,
 * nch z-chunks */
template <typename T> struct R4Sel {
    typedef void (*uv_t)(const RunDev, const T *u, const T *v, const T *w, const T *c, const T *gu, const T *gv,
                         const double *scal, T *fu, T *fv, T *ru, T *rv, double *cflpart, double cfldt, int nch,
                         double *mpart);
    typedef void (*wc_t)(const RunDev, const T *u, const T *v, const T *w, const T *c, const T *gw, const T *gc,
                         const double *scal, T *fw, T *fc, T *rw, T *rc, int nch, double *mpart);
};
template <typename T> typename R4Sel<T>::uv_t pick_rhs4_uv(bool sc, int s);
template <typename T> typename R4Sel<T>::wc_t pick_rhs4_wc(bool sc, int s);

/* batched launches (cf_general.hip, cf_kernels.hip): a = device array of
 * nrun GArgs, vs = that stage's virtual-block prefix (nrun + 1) */
template <typename T> struct BSel {
    typedef void (*divx_t_)(const GArgs<T> *, const unsigned *, int, int);
    typedef void (*rhs_t)(const GArgs<T> *, const unsigned *, int, int);
    rhs_t rhs;
    rhs_t proj;
    typedef void (*kb_t)(const GArgs<T> *, const unsigned *, int, int);
};
template <typename T> BSel<T> pick_batched(int order, int scalar);
template <typename T> typename BSel<T>::divx_t_ pick_batched_divx(int order);
template <typename T> __global__ void kb_poisson4(const GArgs<T> *a, const unsigned *vs, int nrun, int s);
template <typename T> __global__ void kb_solve4(const GArgs<T> *a, const unsigned *vs, int nrun, int s);
template <typename T> typename BSel<T>::kb_t pick_batched_spike(int L);
template <typename T> __global__ void kb_thomas(const GArgs<T> *a, const unsigned *vs, int nrun, int s);
template <typename T> __global__ void kb_mass(const GArgs<T> *a, const unsigned *vs, int nrun, int s);
/* batched order-2 fast path (FP64 or FP32 storage) */
template <typename T> typename BSel<T>::kb_t pick_batched_rhs2(int s);
template <typename T> typename BSel<T>::kb_t pick_batched_spike_sums(int L);
template <typename T> __global__ void kb_level_mass(const GArgs<T> *a, const unsigned *vs, int nrun, int s);
/* batched FFT passes: one launch per group of runs of one length; lengths
 * in CF_BFFT_SIZES have their plan compiled in, the others share a launch
 * with the runtime plan (key 0) */
#define CF_BFFT_SIZES(X) X(32) X(48) X(64) X(96) X(128) X(192) X(256)
static inline int bfft_key(int n)
{
    switch (n) {
#define X_(N) case N: return N;
    CF_BFFT_SIZES(X_)
#undef X_
    default: return 0;
    }
}
template <typename T> typename BSel<T>::kb_t pick_batched_divx_n(int order, int n);
template <typename T> typename BSel<T>::kb_t pick_batched_ffty(int n);
template <typename T> typename BSel<T>::kb_t pick_batched_fftxi(int n);
template <typename T> typename BSel<T>::kb_t pick_batched_poisson(int L);
BSel<float>::kb_t pick_batched_poisson_islands(int L);
template <typename T>
__global__ void k_gsolve4(const RunDev R, const int s, const int nbx, T *ru, T *rv, T *rw, T *rc, const Book B);
template <typename T>
__global__ void k_poisson4(const RunDev R, const Pois4Tab T_, typename Cplx<T>::type *Y, double *S);
/* the twisted form (nz >= 6): grid ceil(M / 64) blocks of 128 */
template <typename T>
__global__ void k_poisson4t(const RunDev R, const Pois4Tab T_, typename Cplx<T>::type *Y, double *S);

/* plane statistics (cf_stats.hip) */
template <typename T> __global__ void k_stat_sum(const T *a, const T *b, int P, int nbl, double *part);
template <typename T, int MODE>
__global__ void k_stat_central(const T *a, const T *b, const double *pa, const double *pb, double scale, double en,
                               int P, int nbl, double *part);
__global__ void k_stat_finish(const double *part, int nbl, int nz, double scale, double *out, const double *off);
#define CF_SPEC_ROWS 8          /* rows kx per wave of k_stat_spec */
__global__ void k_stat_spec(const double2 *A, const double2 *B, int nx, int ny, int nkx, int nz, double2 *specx,
                            double2 *part);
__global__ void k_stat_spec_finish(const double2 *specx, const double2 *part, int ny, int nkx, int nz, double2 *out);
template <typename T> __global__ void k_stat_widen(const T *in, double *out, size_t n);
/* workgroups (partials) per level of a plane statistic: 8 cells a thread, up
 * to the 64 partials that one wave sums */
#define CF_STAT_NBL 64
static inline int stat_nbl(size_t P) { return (int) (P / 2048 < 1 ? 1 : P / 2048 > CF_STAT_NBL ? CF_STAT_NBL : P / 2048); }

#endif
