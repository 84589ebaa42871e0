// ac4_pairs.hip -- pair observables of a device frame store:
//
//  ac4_frames_overlap_cage  Analysis/overlap_cage_rel.c:4-269 (paths relative
//      to the reference checkout): the overlap of each particle's
//      displacement relative to the mean displacement of its neighbours
//      within 1.3 sigma at the origin (its cage), relaxMPICR1_a_<a>.dat.
//  ac4_frames_guu           Analysis/guu.c:3-300: the displacement-
//      displacement correlation g_uu(r) of the active particles at the lag
//      nearest tau, guuTauAlphaAct.dat.
//
// Cage overlap, per origin: particles are binned on the cell grid of
// GetList (cells of edge 1/(int)(L/cell_cut) in box units); k_cg_list
// gives every particle its neighbours in the order GetList's traversal
// appends them (for particle i: the j < i whose own scan finds i, ascending;
// then i's own scan, own cell then the 13 half-stencil cells, each ascending;
// then the j > i whose scan finds i, ascending), so the cage sums are formed
// in the reference's order; the per-lag count is exact.  Needs at least 3
// cells per edge, where the 27 cells around a cell are distinct (the
// reference's small-box double counting is not reproduced).
//
// g_uu, a batch of origins per launch: displacements of the active particles
// and their MSD and mean-displacement sums (k_gu_disp), then all active pairs
// i < j on triangles of 256 x 256 tiles (k_gu_hist, a persistent grid) with
// the histogram of a bin range in LDS, and the workgroups' histograms summed
// (k_gu_reduce).  Bin indices are those of correctly rounded sqrt and
// division (gu_bin), so the pair counts are exact; the two weighted
// histograms are FP64 sums whose order follows the LDS atomics (agreement
// with the reference to rounding).
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>
#include <string.h>
#include <vector>
#include "ac4_internal.h"

#define PR_THREADS 256
#define CG_CAP 64            // neighbours per particle within 1.3 sigma (about 13 at rho = 1.2)
#define GU_TILE 256
#define GU_REC 8             // doubles of a particle: wrapped origin position, displacement, its components, padding
#define GU_SPLIT 4           // threads that share a row of a tile
#define GU_T (GU_SPLIT * GU_TILE)
#define GU_LDS_BINS 6144     // bins per pass: 6144 * 20 B = 120 KB of LDS
#define GU_BATCH (64u << 20) // bytes of displacements of one launch's origins
#define PR_TIME_STEP 0.005   // Analysis/global.h:19
#define PR_DIVIDE_TO 2.0     // Analysis/global.h:21
#define PR_PI 3.14159265358979
#define PR_RHO 1.2

__device__ __forceinline__ double pr_wrap(double v) {  // the while loops of read_all_data.c LoadOrigin
    return (v >= 1.0 || v < 0.0) ? v - floor(v) : v;
}
__device__ __forceinline__ double pr_mi(double d) {  // overlap_cage_rel.c:85-96, guu.c:157-168
    if (d >= 0.5)
        d -= 1.0;
    else if (d < -0.5)
        d += 1.0;
    return d;
}

// ------------------------------------------------------------ cage overlap

// wrapped origin positions and their GetList cell (1-based, :210-216)
__global__ void __launch_bounds__(PR_THREADS) k_cg_bin(const double *__restrict__ x0, const double *__restrict__ y0,
                                                       const double *__restrict__ z0, int n, int nc, double cs,
                                                       double *wx, double *wy, double *wz, int *cell,
                                                       unsigned int *cnt) {
    const int i = blockIdx.x * PR_THREADS + threadIdx.x;
    if (i >= n) return;
    const double x = pr_wrap(x0[i]), y = pr_wrap(y0[i]), z = pr_wrap(z0[i]);
    wx[i] = x;
    wy[i] = y;
    wz[i] = z;
    int c = (int)(1 + floor(x / cs) + floor(y / cs) * nc + floor(z / cs) * nc * nc);
    const int ncell = nc * nc * nc;
    c = c < 1 ? 1 : (c > ncell ? ncell : c);
    cell[i] = c;
    atomicAdd(&cnt[c], 1u);
}

// exclusive scan of cnt[0..m) into start[0..m], one block
__global__ void __launch_bounds__(1024) k_pr_scan(const unsigned int *__restrict__ cnt, int m, int *start) {
    __shared__ int s_part[1024];
    const int t = threadIdx.x, per = (m + 1023) / 1024;
    const int b0 = t * per, b1 = min(m, b0 + per);
    int sum = 0;
    for (int b = b0; b < b1; b++) sum += (int)cnt[b];
    s_part[t] = sum;
    __syncthreads();
    for (int d = 1; d < 1024; d <<= 1) {
        const int v = t >= d ? s_part[t - d] : 0;
        __syncthreads();
        s_part[t] += v;
        __syncthreads();
    }
    int run = s_part[t] - sum;
    for (int b = b0; b < b1; b++) {
        start[b] = run;
        run += (int)cnt[b];
    }
    if (t == 1023) start[m] = s_part[1023];
}

__global__ void __launch_bounds__(PR_THREADS) k_cg_scatter(const int *__restrict__ cell, int n,
                                                           const int *__restrict__ start, unsigned int *fill,
                                                           int *mem) {
    const int i = blockIdx.x * PR_THREADS + threadIdx.x;
    if (i >= n) return;
    const int c = cell[i];
    mem[start[c] + (int)atomicAdd(&fill[c], 1u)] = i;
}

// len_check of overlap_cage_rel.c:253-269
__device__ __forceinline__ bool cg_near(double ax, double ay, double az, double bx, double by, double bz, double L) {
    double dx = ax - bx, dy = ay - by, dz = az - bz;
    if (dx < -0.5) dx += 1.0;
    if (dx > 0.5) dx -= 1.0;
    if (dy < -0.5) dy += 1.0;
    if (dy > 0.5) dy -= 1.0;
    if (dz < -0.5) dz += 1.0;
    if (dz > 0.5) dz -= 1.0;
    const double dr2 = (dx * dx + dy * dy + dz * dz) * L * L;
    return dr2 < 1.3 * 1.3;
}

// the 13 half-stencil offsets of maps() (overlap_cage_rel.c:297-309)
__constant__ int c_hs[13][3] = {{1, 0, 0},  {1, 1, 0},  {0, 1, 0},  {-1, 1, 0}, {1, 0, -1}, {1, 1, -1}, {0, 1, -1},
                                {-1, 1, -1}, {1, 0, 1}, {1, 1, 1},  {0, 1, 1},  {-1, 1, 1}, {0, 0, 1}};

__device__ __forceinline__ int cg_cell_at(int c, int dx, int dy, int dz, int nc) {  // getcell_I (:273-277)
    const int q = c - 1;
    const int ix = q % nc, iy = (q / nc) % nc, iz = q / (nc * nc);
    return 1 + (ix + dx + nc) % nc + ((iy + dy + nc) % nc) * nc + ((iz + dz + nc) % nc) * nc * nc;
}

// Neighbour list of particle i in GetList's append order.  keys: group 0 =
// found by j < i, 1 = i's own scan (sub = stencil slot + 1, own cell 0),
// 2 = found by j > i; sorted by (group, sub, index).
__global__ void __launch_bounds__(PR_THREADS) k_cg_list(const double *__restrict__ wx, const double *__restrict__ wy,
                                                        const double *__restrict__ wz, const int *__restrict__ cell,
                                                        int n, int nc, double L, const int *__restrict__ start,
                                                        const int *__restrict__ mem, int *nn, int *nb,
                                                        unsigned long long *key, int *overflow) {
    const int i = blockIdx.x * PR_THREADS + threadIdx.x;
    if (i >= n) return;
    const double xi = wx[i], yi = wy[i], zi = wz[i];
    const int c = cell[i];
    int k = 0;
    int *lst = nb + (size_t)i * CG_CAP;
    unsigned long long *ky = key + (size_t)i * CG_CAP;
    auto put = [&](unsigned long long kk, int j) {
        if (k < CG_CAP) {
            ky[k] = kk;
            lst[k] = j;
        }
        k++;
    };
    for (int q = start[c]; q < start[c + 1]; q++) {  // own cell (:221-233)
        const int j = mem[q];
        if (j == i || !cg_near(xi, yi, zi, wx[j], wy[j], wz[j], L)) continue;
        put(j < i ? (unsigned long long)j : (1ull << 60) | (unsigned long long)j, j);
    }
    for (int s = 0; s < 13; s++) {
        const int c2 = cg_cell_at(c, c_hs[s][0], c_hs[s][1], c_hs[s][2], nc);  // i's scan (:235-248)
        for (int q = start[c2]; q < start[c2 + 1]; q++) {
            const int j = mem[q];
            if (cg_near(xi, yi, zi, wx[j], wy[j], wz[j], L))
                put((1ull << 60) | ((unsigned long long)(s + 1) << 32) | (unsigned long long)j, j);
        }
        const int c3 = cg_cell_at(c, -c_hs[s][0], -c_hs[s][1], -c_hs[s][2], nc);  // scans that reach i
        for (int q = start[c3]; q < start[c3 + 1]; q++) {
            const int j = mem[q];
            if (cg_near(wx[j], wy[j], wz[j], xi, yi, zi, L))
                put(j < i ? (unsigned long long)j : (2ull << 60) | (unsigned long long)j, j);
        }
    }
    if (k > CG_CAP) {
        atomicMax(overflow, k);
        k = CG_CAP;
    }
    for (int a = 1; a < k; a++) {  // insertion sort by key
        const unsigned long long kk = ky[a];
        const int jj = lst[a];
        int b = a - 1;
        while (b >= 0 && ky[b] > kk) {
            ky[b + 1] = ky[b];
            lst[b + 1] = lst[b];
            b--;
        }
        ky[b + 1] = kk;
        lst[b + 1] = jj;
    }
    nn[i] = k;
}

// DX = L * (one-correction minimum image of x_t - x0), unwrapped (:80-100);
// grid (particle blocks, lags of the origin)
__global__ void __launch_bounds__(PR_THREADS) k_cg_disp(const double *__restrict__ X, const double *__restrict__ Y,
                                                        const double *__restrict__ Z, int n, size_t f0,
                                                        const int *__restrict__ lagf, double L, double *DX,
                                                        double *DY, double *DZ) {
    const int i = blockIdx.x * PR_THREADS + threadIdx.x;
    if (i >= n) return;
    const size_t ft = (size_t)lagf[blockIdx.y] * n, o = (size_t)blockIdx.y * n + i;
    DX[o] = L * pr_mi(X[ft + i] - X[f0 + i]);
    DY[o] = L * pr_mi(Y[ft + i] - Y[f0 + i]);
    DZ[o] = L * pr_mi(Z[ft + i] - Z[f0 + i]);
}

// cage-relative overlap count of one lag (:109-131); grid (particle blocks, lags)
__global__ void __launch_bounds__(PR_THREADS) k_cg_count(const double *__restrict__ DX, const double *__restrict__ DY,
                                                         const double *__restrict__ DZ, int n,
                                                         const int *__restrict__ nn, const int *__restrict__ nb,
                                                         double param, unsigned int *count) {
    const int i = blockIdx.x * PR_THREADS + threadIdx.x;
    const size_t o = (size_t)blockIdx.y * n;
    int hit = 0;
    if (i < n) {
        const int m = nn[i];
        const int *lst = nb + (size_t)i * CG_CAP;
        double dx = 0.0, dy = 0.0, dz = 0.0;
        for (int k = 0; k < m; k++) {
            const size_t p = o + lst[k];
            dx += DX[p];
            dy += DY[p];
            dz += DZ[p];
        }
        dx = dx / (double)m;
        dy = dy / (double)m;
        dz = dz / (double)m;
        const double Xi = DX[o + i], Yi = DY[o + i], Zi = DZ[o + i];
        double r2 = (Xi * Xi + Yi * Yi + Zi * Zi);
        r2 += (dx * dx + dy * dy + dz * dz);
        r2 -= 2.00 * (Xi * dx + Yi * dy + Zi * dz);
        hit = r2 < param ? 1 : 0;
    }
    const unsigned long long b = __ballot(hit);
    __shared__ unsigned int s_c;
    if (threadIdx.x == 0) s_c = 0;
    __syncthreads();
    if ((threadIdx.x & 63) == 0) atomicAdd(&s_c, (unsigned int)__popcll(b));
    __syncthreads();
    if (threadIdx.x == 0) atomicAdd(&count[blockIdx.y], s_c);
}

// ------------------------------------------------------------------- g_uu

// active particles m (ascending index act[m]) of each origin of a batch
// (grid: particle blocks x origins, frame offsets fo[o] = {origin, lag}):
// displacement to the lag frame (guu.c:151-180) and wrapped origin position
// (LoadOrigin) to the record g[o][m]; the block's sums of L*L*r2 and r (the terms of
// MSDtPP and MDtPP, guu.c:172-173) to acc[(o*gridDim.x + block)*2], added up
// by the host in origin and block order.  (One thread adding them in
// particle order took 301 us per origin at 5000 active particles, more than
// twice the pair histogram.)
__global__ void __launch_bounds__(PR_THREADS) k_gu_disp(const double *__restrict__ X, const double *__restrict__ Y,
                                                        const double *__restrict__ Z, int n,
                                                        const int2 *__restrict__ fo, const int *__restrict__ act,
                                                        int na, double L, double *gall, double *acc) {
    const int m = blockIdx.x * PR_THREADS + threadIdx.x;
    const size_t f0 = (size_t)fo[blockIdx.y].x * n, ft = (size_t)fo[blockIdx.y].y * n;
    double *g = gall + ((size_t)blockIdx.y * na + m) * GU_REC;
    double msd = 0.0, md = 0.0;
    if (m < na) {
        const int i = act[m];
        const double dx = pr_mi(X[ft + i] - X[f0 + i]), dy = pr_mi(Y[ft + i] - Y[f0 + i]),
                     dz = pr_mi(Z[ft + i] - Z[f0 + i]);
        const double r2 = (dx * dx + dy * dy + dz * dz);
        md = L * sqrt(r2);  // drt
        msd = L * L * r2;
        g[0] = pr_wrap(X[f0 + i]);
        g[1] = pr_wrap(Y[f0 + i]);
        g[2] = pr_wrap(Z[f0 + i]);
        g[3] = md;
        g[4] = L * dx;
        g[5] = L * dy;
        g[6] = L * dz;
    }
    __shared__ double s_w[2][PR_THREADS / 64];
    msd = ac4_wave_sum(msd);
    md = ac4_wave_sum(md);
    if ((threadIdx.x & 63) == 0) {
        s_w[0][threadIdx.x >> 6] = msd;
        s_w[1][threadIdx.x >> 6] = md;
    }
    __syncthreads();
    if (threadIdx.x < 2) {
        double t = 0.0;
        for (int w = 0; w < PR_THREADS / 64; w++) t += s_w[threadIdx.x][w];
        acc[((size_t)blockIdx.y * gridDim.x + blockIdx.x) * 2 + threadIdx.x] = t;
    }
}

// (int)(sqrt(r2) / bin), the bin of guu.c:205-206 with its correctly rounded
// sqrt and division.  An estimate decides wherever it is further from a whole
// number than its error: r2 times v_rsq_f64 (5.3e-8 relative measured over
// 2.7e8 values) is the square root to 5e-15 after one Newton step, and the
// products after it round to 2e-16; 1e-11 is taken, relative.  r2 = 0 gives
// NaN and the exact form.  (A 32-bit estimate, taken as 1e-6, left every fifth
// wave of 64 pairs to the exact form: 622 against 500 us for 20 origins of
// 5000 active particles.)
__device__ __forceinline__ int gu_bin(double r2, double bin, double rbin) {
    const double y = __builtin_amdgcn_rsq(r2), t = r2 * y;
    const double e = fma(t * 0.5, fma(-t, y, 1.0), t) * rbin;
    const double f = floor(e), m = 1e-11 * e;
    if (e - f > m && f + 1.0 - e > m) return (int)f;
    return (int)(sqrt(r2) / bin);
}

// Pairs (row m1 < column m2) of the tiles of the upper triangle of every
// origin of the batch, bins [b0, b0+nbins), item i = origin i / ntri, tile
// i % ntri; workgroup w takes items w, w + gridDim.x, ... and keeps one
// histogram in LDS over all of them, written to its own rows of pc/p1/p2 at
// the end (k_gu_reduce adds the workgroups in order).  Bound by the issue of
// the FP64 pair arithmetic (46 instructions) beside three LDS atomics per
// pair.  GU_SPLIT threads share a row (a part of the tile's columns each), so
// that two workgroups of 16 waves fit a CU; a column is the same for a whole
// wave and its record comes by scalar loads, which leaves the LDS to the
// histogram.  One launch per origin, a workgroup per tile, each flushed by
// global atomics: 135 us per origin on 210 workgroups at 5000 active particles;
// a persistent grid over 20 origins with the columns in LDS 60, with 16 waves
// per workgroup 42, with scalar loads 31, with the 64-bit bin estimate 25.
__global__ void __launch_bounds__(GU_T) k_gu_hist(const double *__restrict__ gall, int na, double L, double bin,
                                                         double rbin, int b0, int nbins, int ntile,
                                                         int ntri, int nitem, unsigned int *__restrict__ pc,
                                                         double *__restrict__ p1, double *__restrict__ p2) {
    extern __shared__ unsigned char s_raw[];
    unsigned int *s_c = (unsigned int *)s_raw;
    double *s_1 = (double *)(s_raw + ((sizeof(unsigned int) * nbins + 15) & ~(size_t)15));
    double *s_2 = s_1 + nbins;
    const int t = threadIdx.x, row = t & (GU_TILE - 1), part = __builtin_amdgcn_readfirstlane(t / GU_TILE);
    for (int b = t; b < nbins; b += GU_T) {
        s_c[b] = 0;
        s_1[b] = 0.0;
        s_2[b] = 0.0;
    }
    __syncthreads();
    for (int it = blockIdx.x; it < nitem; it += gridDim.x) {
        const int o = it / ntri;
        const double *g = gall + (size_t)o * GU_REC * na;
        // tile (tr, tc), tr <= tc, of the triangle
        int q = it - o * ntri, tr = 0;
        while (q >= ntile - tr) {
            q -= ntile - tr;
            tr++;
        }
        const int mi = tr * GU_TILE + row, j0 = (tr + q) * GU_TILE + part * (GU_TILE / GU_SPLIT);
        const int j1 = min(j0 + GU_TILE / GU_SPLIT, na);
        if (mi >= na) continue;
        const double *gi = g + (size_t)mi * GU_REC;
        const double xi = gi[0], yi = gi[1], zi = gi[2], ri = gi[3], ui = gi[4], vi = gi[5], wi = gi[6];
        for (int j = j0; j < j1; j++) {
            if (j <= mi) continue;
            const double *c = g + (size_t)j * GU_REC;  // the same for the whole wave: scalar loads
            // guu.c:198-213: x0_j - x0_i, one correction (pr_mi; rint differs
            // from it in the sign of a difference of exactly a half alone)
            double dx = c[0] - xi, dy = c[1] - yi, dz = c[2] - zi;
            dx -= rint(dx);
            dy -= rint(dy);
            dz -= rint(dz);
            const double r2 = L * L * (dx * dx + dy * dy + dz * dz);
            const int b = gu_bin(r2, bin, rbin) - b0;
            if ((unsigned)b < (unsigned)nbins) {  // b0 + nbins <= the number of bins
                atomicAdd(&s_c[b], 1u);
                atomicAdd(&s_1[b], 2.0 * (ri * c[3]));
                atomicAdd(&s_2[b], 2.0 * (ui * c[4] + vi * c[5] + wi * c[6]));
            }
        }
    }
    __syncthreads();
    const size_t w0 = (size_t)blockIdx.x * nbins;
    for (int b = t; b < nbins; b += GU_T) {
        pc[w0 + b] = s_c[b];
        p1[w0 + b] = s_1[b];
        p2[w0 + b] = s_2[b];
    }
}

// the workgroups' histograms added to the totals in a fixed order: 64 bins per
// workgroup, its wave q every GU_RW-th histogram, then the waves in order
#define GU_RW 16
__global__ void __launch_bounds__(64 * GU_RW) k_gu_reduce(const unsigned int *__restrict__ pc,
                                                          const double *__restrict__ p1, const double *__restrict__ p2,
                                                          int nw, int nbins, int b0, unsigned long long *hc, double *h1,
                                                          double *h2) {
    __shared__ unsigned long long s_c[GU_RW][64];
    __shared__ double s_1[GU_RW][64], s_2[GU_RW][64];
    const int l = threadIdx.x & 63, q = threadIdx.x >> 6, b = blockIdx.x * 64 + l;
    unsigned long long c = 0;
    double a1 = 0.0, a2 = 0.0;
    if (b < nbins)
#pragma unroll 4
        for (int w = q; w < nw; w += GU_RW) {
            const size_t k = (size_t)w * nbins + b;
            c += pc[k];
            a1 += p1[k];
            a2 += p2[k];
        }
    s_c[q][l] = c;
    s_1[q][l] = a1;
    s_2[q][l] = a2;
    __syncthreads();
    if (q == 0 && b < nbins) {
        for (int w = 1; w < GU_RW; w++) {
            c += s_c[w][l];
            a1 += s_1[w][l];
            a2 += s_2[w][l];
        }
        hc[b0 + b] += c;
        h1[b0 + b] += a1;
        h2[b0 + b] += a2;
    }
}

#define PTRY(e) do { int rc_ = (e); if (rc_ != AC4_OK) return rc_; } while (0)

extern "C" int ac4_frames_overlap_cage(ac4_frames *f, int gap, double factor, double a, double cell_cut,
                                       const char *path, int *pair_counts, int cap_pairs, int *npairs) {
    ac4_frames_view v;
    PTRY(ac4_frames_view_get(f, &v));
    AC4_REQUIRE(gap > 0 && factor > 1.0 && a > 0.0 && cell_cut > 0.0 && v.count >= 2, AC4_EARG,
                "ac4_frames_overlap_cage: bad arguments");
    const int n = v.n, nf = v.count;
    const double L = v.L;
    std::vector<int> fidx;
    PTRY(ac4_frames_steps(v, fidx));
    const int nc = (int)(L / cell_cut);  // maps(), :283
    AC4_REQUIRE(nc >= 3, AC4_EARG,
                "ac4_frames_overlap_cage: %d cells per edge (L/cell_cut); at least 3 are needed", nc);
    const int ncell = nc * nc * nc;
    const double cs = 1.0 / (double)nc;
    ac4_walk_t w;
    memset(&w, 0, sizeof w);
    PTRY(ac4_walk(fidx.data(), nf, gap, factor, 1, &w));  // origins counted on k*gap+1 (:23-30)
    const int maxint = w.maximal_interval;
    std::vector<int> cur(w.cur, w.cur + w.np), oth(w.oth, w.oth + w.np), slot(w.slot, w.slot + w.np);
    ac4_walk_free(&w);
    AC4_REQUIRE(maxint > 0, AC4_EARG, "ac4_frames_overlap_cage: no lag");
    const int noi = 10 + (int)(log((double)maxint) / log(factor));
    const int np = (int)cur.size();
    int maxlag = 0;
    for (int p = 0, q; p < np; p = q) {
        for (q = p; q < np && cur[q] == cur[p]; q++) {}
        maxlag = std::max(maxlag, q - p);
    }
    AcDevBuf B;
    double *d_w, *d_D;
    int *d_cell, *d_start, *d_mem, *d_nn, *d_nb, *d_lag, *d_over;
    unsigned int *d_cnt, *d_count;
    unsigned long long *d_key;
    PTRY(B.get(&d_w, (size_t)3 * n));
    PTRY(B.get(&d_D, (size_t)3 * n * std::max(maxlag, 1)));
    PTRY(B.get(&d_cell, n));
    PTRY(B.get(&d_cnt, (size_t)2 * (ncell + 1)));
    PTRY(B.get(&d_start, ncell + 2));
    PTRY(B.get(&d_mem, n));
    PTRY(B.get(&d_nn, n));
    PTRY(B.get(&d_nb, (size_t)n * CG_CAP));
    PTRY(B.get(&d_key, (size_t)n * CG_CAP));
    PTRY(B.get(&d_lag, std::max(maxlag, 1)));
    PTRY(B.get(&d_over, 1));
    PTRY(B.get(&d_count, std::max(np, 1)));
    hipStream_t s = v.s;
    AC4_HIP(hipMemsetAsync(d_count, 0, sizeof(unsigned int) * std::max(np, 1), s));
    AC4_HIP(hipMemsetAsync(d_over, 0, sizeof(int), s));
    const unsigned gb = (unsigned)((n + PR_THREADS - 1) / PR_THREADS);
    // origins visited by the do-while of :59-154; a pair's origin is its cur
    for (int p = 0, q; p < np; p = q) {
        for (q = p; q < np && cur[q] == cur[p]; q++) {}
        const size_t f0 = (size_t)cur[p] * n;
        AC4_HIP(hipMemsetAsync(d_cnt, 0, sizeof(unsigned int) * 2 * (ncell + 1), s));
        hipLaunchKernelGGL(k_cg_bin, dim3(gb), dim3(PR_THREADS), 0, s, v.x + f0, v.y + f0, v.z + f0, n, nc, cs, d_w,
                           d_w + n, d_w + 2 * (size_t)n, d_cell, d_cnt);
        hipLaunchKernelGGL(k_pr_scan, dim3(1), dim3(1024), 0, s, d_cnt, ncell + 1, d_start);
        hipLaunchKernelGGL(k_cg_scatter, dim3(gb), dim3(PR_THREADS), 0, s, d_cell, n, d_start, d_cnt + ncell + 1,
                           d_mem);
        hipLaunchKernelGGL(k_cg_list, dim3(gb), dim3(PR_THREADS), 0, s, d_w, d_w + n, d_w + 2 * (size_t)n, d_cell, n,
                           nc, L, d_start, d_mem, d_nn, d_nb, d_key, d_over);
        std::vector<int> lags(oth.begin() + p, oth.begin() + q);
        AC4_HIP(hipMemcpyAsync(d_lag, lags.data(), sizeof(int) * lags.size(), hipMemcpyHostToDevice, s));
        const size_t nl = lags.size();
        hipLaunchKernelGGL(k_cg_disp, dim3(gb, (unsigned)nl), dim3(PR_THREADS), 0, s, v.x, v.y, v.z, n, f0, d_lag, L,
                           d_D, d_D + nl * n, d_D + 2 * nl * n);
        hipLaunchKernelGGL(k_cg_count, dim3(gb, (unsigned)nl), dim3(PR_THREADS), 0, s, d_D, d_D + nl * n,
                           d_D + 2 * nl * n, n, d_nn, d_nb, a * a, d_count + p);
        AC4_HIP(hipGetLastError());
        AC4_HIP(hipStreamSynchronize(s));  // lags and scratch are reused by the next origin
    }
    std::vector<unsigned int> cnt(std::max(np, 1));
    int over = 0;
    AC4_HIP(hipMemcpyAsync(cnt.data(), d_count, sizeof(unsigned int) * std::max(np, 1), hipMemcpyDeviceToHost, s));
    AC4_HIP(hipMemcpyAsync(&over, d_over, sizeof(int), hipMemcpyDeviceToHost, s));
    AC4_HIP(hipStreamSynchronize(s));
    AC4_REQUIRE(over == 0, AC4_ECAP, "ac4_frames_overlap_cage: %d neighbours within 1.3 (at most %d)", over, CG_CAP);
    // :132-167: SUM = count/N per pair, accumulated per slot in walk order
    std::vector<double> c(noi, 0.0), x4(noi, 0.0), dt(noi, 0.0);
    std::vector<int> counters(noi, 0);
    for (int p = 0; p < np; p++) {
        const int t = slot[p];
        AC4_REQUIRE(t < noi, AC4_EARG, "ac4_frames_overlap_cage: slot %d beyond %d", t, noi);
        const double SUM = (double)cnt[p] / (double)n;
        c[t] += SUM;
        x4[t] += SUM * SUM;
        counters[t]++;
        dt[t] = PR_TIME_STEP * (double)(fidx[oth[p]] - fidx[cur[p]]);
        if (pair_counts && p < cap_pairs) pair_counts[p] = (int)cnt[p];
    }
    if (npairs) *npairs = np;
    if (path) {
        FILE *fo = fopen(path, "wb");
        AC4_REQUIRE(fo, AC4_EIO, "ac4_frames_overlap_cage: cannot write %s", path);
        fprintf(fo, "0.0\t1.0\t0.0\n");
        for (int k = 1; k < noi; k++)
            if (counters[k])
                fprintf(fo, "%.14lf\t%.14lf\t%.14lf\n", dt[k], c[k] / (double)counters[k],
                        x4[k] / (double)counters[k] - c[k] * c[k] / ((double)(counters[k] * counters[k])));
        AC4_REQUIRE(fclose(fo) == 0, AC4_EIO, "ac4_frames_overlap_cage: write error on %s", path);
    }
    return AC4_OK;
}

extern "C" int ac4_frames_guu(ac4_frames *f, const int *act_tag, int gap, double factor, double tau,
                              const char *path, double *hist3, int *maxbin_out, int *frame_num_out,
                              int *n_origins_out) {
    ac4_frames_view v;
    PTRY(ac4_frames_view_get(f, &v));
    AC4_REQUIRE(act_tag && gap > 0 && factor > 1.0 && v.count >= 2, AC4_EARG, "ac4_frames_guu: bad arguments");
    const int n = v.n, nf = v.count;
    const double L = v.L;
    std::vector<int> fidx;
    PTRY(ac4_frames_steps(v, fidx));
    const double bin = 0.005;
    const double MaxBin = (int)(0.5 * L / bin);  // guu.c:17
    const int maxbin = (int)MaxBin;
    const int maxint = 200 * gap / PR_DIVIDE_TO;  // guu.c:30-31
    // guu.c:67-115: lag ladder of the first frame, FrameNum nearest tau
    int frame_num = 0;
    {
        std::vector<double> dt(1, 0.0);
        const int cf = fidx[0];
        int other = 0, offset = 1;
        while (other < nf && offset < maxint) {
            const int of = cf + offset;
            while (other < nf && fidx[other] != of) other++;
            if (other < nf) {
                dt.push_back(PR_TIME_STEP * (double)(of - cf));
                if ((int)(offset * factor) == offset)
                    offset++;
                else
                    offset = (int)(((double)offset) * factor);
            }
        }
        double inter = 1000.0;
        for (size_t i = 1; i < dt.size(); i++)
            if (fabs(dt[i] - tau) < inter) {
                frame_num = (int)(dt[i] * 200.0);
                inter = fabs(dt[i] - tau);
            }
    }
    std::vector<int> act;
    for (int i = 0; i < n; i++)
        if (act_tag[i] == 1) act.push_back(i);
    const int na = (int)act.size();
    // guu.c:138-231: the origins and their lag frames
    std::vector<int2> fo;
    int current = 0, on = 0;
    do {
        const int cf = fidx[current];
        int other = current;
        while (other < nf && fidx[other] != cf + frame_num) other++;
        if (other >= nf) break;
        fo.push_back(make_int2(current, other));
        on++;
        while (current < nf && fidx[current] != on * gap) current++;
    } while (current < nf);
    const int ntile = (na + GU_TILE - 1) / GU_TILE;
    AC4_REQUIRE((long long)ntile * (ntile + 1) / 2 < 2147483647LL, AC4_EARG, "ac4_frames_guu: %d active particles", na);
    const int ntri = ntile * (ntile + 1) / 2;
    const int pass_bins = std::min(maxbin, GU_LDS_BINS);
    const size_t lds = ((sizeof(unsigned int) * pass_bins + 15) & ~(size_t)15) + sizeof(double) * 2 * pass_bins;
    // origins of one launch: as many as GU_BATCH bytes of displacements hold
    const size_t per = sizeof(double) * GU_REC * (size_t)std::max(na, 1);
    const int batch = (int)std::max<size_t>(1, std::min<size_t>(std::max(on, 1), std::min<size_t>(GU_BATCH / per, 65535)));
    // the persistent grid: the workgroups that are resident together
    // (160 KB of LDS per CU, at most two of sixteen waves), no more than a
    // batch has tiles; a box of less than
    // two bins' length has no bins and no LDS
    int dev = 0, ncu = 256;
    (void)hipGetDevice(&dev);
    if (hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) ncu = 256;
    const long long items = std::max<long long>(1, std::min<long long>((long long)ntri * batch, 2147483647LL));
    const int grid = (int)std::min<long long>(
        items, ncu * (long long)std::max<size_t>(1, std::min<size_t>(2, 163840 / std::max<size_t>(lds, 1))));
    const int dblk = (na + PR_THREADS - 1) / PR_THREADS;
    // one allocation: act and fo (one copy in), the totals and k_gu_disp's
    // sums (one copy out), then the batch's records and the partial histograms
    const size_t mb = std::max(maxbin, 1), pb = (size_t)grid * std::max(pass_bins, 1);
    const size_t in_b = sizeof(int2) * std::max(on, 1) + ((sizeof(int) * std::max(na, 1) + 7) & ~(size_t)7);
    const size_t out_n = 3 * mb + (size_t)2 * std::max(on, 1) * std::max(dblk, 1);  // 64-bit words
    AcDevBuf B;
    char *d_all;
    PTRY(B.get(&d_all, in_b + 8 * out_n + sizeof(double) * ((size_t)batch * GU_REC * std::max(na, 1) + 2 * pb) +
                           sizeof(unsigned int) * pb));
    int2 *const d_fo = (int2 *)d_all;
    int *const d_act = (int *)(d_fo + std::max(on, 1));
    unsigned long long *const d_hc = (unsigned long long *)(d_all + in_b);
    double *const d_h1 = (double *)(d_hc + mb), *const d_h2 = d_h1 + mb, *const d_acc = d_h2 + mb,
           *const d_g = (double *)d_hc + out_n, *const d_p1 = d_g + (size_t)batch * GU_REC * std::max(na, 1),
           *const d_p2 = d_p1 + pb;
    unsigned int *const d_pc = (unsigned int *)(d_p2 + pb);
    hipStream_t s = v.s;
    std::vector<char> in(in_b, 0);
    if (on) memcpy(in.data(), fo.data(), sizeof(int2) * on);
    if (na) memcpy(in.data() + sizeof(int2) * std::max(on, 1), act.data(), sizeof(int) * na);
    AC4_HIP(hipMemcpyAsync(d_all, in.data(), in_b, hipMemcpyHostToDevice, s));
    AC4_HIP(hipMemsetAsync(d_hc, 0, 8 * 3 * mb, s));
    AC4_HIP(hipFuncSetAttribute((const void *)k_gu_hist, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    for (int o0 = 0; na && o0 < on; o0 += batch) {
        const int no = std::min(batch, on - o0);
        hipLaunchKernelGGL(k_gu_disp, dim3(dblk, no), dim3(PR_THREADS), 0, s, v.x, v.y, v.z, n, d_fo + o0, d_act, na, L,
                           d_g, d_acc + (size_t)2 * o0 * dblk);
        const long long all = (long long)ntri * no;
        AC4_REQUIRE(all < 2147483647LL - grid, AC4_EARG, "ac4_frames_guu: %d active particles", na);
        const int nitem = (int)all, gw = std::min(grid, nitem);
        for (int b0 = 0; b0 < maxbin; b0 += pass_bins) {
            const int nbins = std::min(pass_bins, maxbin - b0);
            hipLaunchKernelGGL(k_gu_hist, dim3(gw), dim3(GU_T), lds, s, d_g, na, L, bin, 1.0 / bin,
                               b0, nbins, ntile, ntri, nitem, d_pc, d_p1, d_p2);
            hipLaunchKernelGGL(k_gu_reduce, dim3((nbins + 63) / 64), dim3(64 * GU_RW), 0, s, d_pc, d_p1, d_p2, gw, nbins, b0,
                               d_hc, d_h1, d_h2);
        }
        AC4_HIP(hipGetLastError());
    }
    std::vector<unsigned long long> res(out_n, 0);
    AC4_HIP(hipMemcpyAsync(res.data(), d_hc, 8 * out_n, hipMemcpyDeviceToHost, s));
    AC4_HIP(hipStreamSynchronize(s));
    const unsigned long long *const hc = res.data();
    const double *const h1 = (const double *)(hc + mb), *const h2 = h1 + mb, *const part = h2 + mb;
    double acc[2] = {0.0, 0.0};
    for (size_t k = 0; k < (size_t)2 * on * dblk; k++) acc[k & 1] += part[k];
    // guu.c:250-276
    const double MSDt = acc[0] / ((double)n * (double)on);
    const double MDt = acc[1] / ((double)n * (double)on);
    const double norm = (4.0 * PR_PI * (PR_RHO)*bin * (double)n * (double)on);
    const double norm1 = (4.0 * PR_PI * PR_RHO * bin * (double)n * (double)on * (double)(MDt * MDt));
    const double norm2 = (4.0 * PR_PI * PR_RHO * bin * (double)n * (double)on * (double)(MSDt));
    if (hist3)
        for (int i = 0; i < maxbin; i++) {
            hist3[i] = 2.0 * (double)hc[i];
            hist3[maxbin + i] = h1[i];
            hist3[2 * (size_t)maxbin + i] = h2[i];
        }
    if (maxbin_out) *maxbin_out = maxbin;
    if (frame_num_out) *frame_num_out = frame_num;
    if (n_origins_out) *n_origins_out = on;
    if (path) {
        FILE *fo = fopen(path, "wb");
        AC4_REQUIRE(fo, AC4_EIO, "ac4_frames_guu: cannot write %s", path);
        for (int i = 1; i < MaxBin; i++) {
            const double r = (double)(i + 1) * bin;
            const double hist = 2.0 * (double)hc[i];
            fprintf(fo, "%0.10g\t%.10g\t%.10g\t%.10g\t%.10g\n", r, (hist / (norm * r * r)), (h1[i] / (norm1 * r * r)),
                    h2[i] / (norm1 * r * r), h2[i] / (norm2 * r * r));
        }
        AC4_REQUIRE(fclose(fo) == 0, AC4_EIO, "ac4_frames_guu: write error on %s", path);
    }
    return AC4_OK;
}
