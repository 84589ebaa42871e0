// ac4_analysis.hip -- streaming dynamic-heterogeneity analysis on MI355X.
//
// Replaces Analysis/msd_pos.c, overlap.c, S4Qt.c and Fsqt.c (paths relative
// to the reference checkout).  The reference loads every frame into host RAM
// and walks (origin, lag) pairs with one MPI_Reduce per pair; here frames are
// pushed once in file order, origin frames stay resident in HBM, and each
// pushed frame is compared with all origins whose walk it completes in one
// launch (k_frame: MSD sums, overlap counts and S4 masks of every pair, and
// the copy of an origin frame to its resident place), with a second one for
// Fs (k_fs).  The walk is known when the handle is made, so the pairs of every
// frame and the origins' places are laid out on the device then.  S4's phase
// sums are formed once per origin over all of its lags on the FP64 matrix
// cores.  Per-pair results are reduced in a fixed order and accumulated into
// lag slots in the reference's origin order on the device, so integer
// observables (overlap counts) reproduce the reference's output bit for
// bit.
#include <hip/hip_runtime.h>
#include <math.h>
#include <string.h>
#include <algorithm>
#include <chrono>
#include <vector>
#include <map>
#include "ac4_internal.h"

#define ABLK 256
#define A_PI 3.14159265358979 // Analysis/global.h:14

__constant__ int c_dg[AC4_NQ];  // permutations of each GetQ vector

struct Job {       // one (origin, lag) pair evaluated against the pushed frame
    int org;       // the origin's place among the resident frames
    int p0, p1;    // pair of the MSD walk and of the overlap/S4/Fs walk, -1 where it is none (or not asked for)
    int slot;      // lag slot, the number of wraps S4 and Fs apply to the origin
};
// resident origin frames: x, y, z of place k at f + (3*k + {0,1,2})*n
struct Origins {
    double *f;
    size_t n;
    __host__ __device__ double *at(int k, int c) const { return f + ((size_t)3 * k + c) * n; }
};

__device__ __forceinline__ double minimg_ana(double d) {  // overlap.c:67-78
    if (d >= 0.5)
        d -= 1.0;
    else if (d < -0.5)
        d += 1.0;
    return d;
}
__device__ __forceinline__ double wrap1(double v) {  // S4Qt.c:102-113
    if (v >= 1.0) v -= 1.0;
    if (v < 0.0) v += 1.0;
    return v;
}
// x0 after the per-lag single-if wrap has run `times` times (S4Qt.c:101-114
// wraps the resident origin coordinates again at every lag).
__device__ __forceinline__ double wrapn(double v, int times) {
    for (int k = 0; k < times; k++) {
        double w = wrap1(v);
        if (w == v) break;
        v = w;
    }
    return v;
}

template <int NV, int T = ABLK>
__device__ __forceinline__ void block_sum_store(double (&v)[NV], double *out) {
    __shared__ double s_red[NV][T / 64];
    for (int k = 0; k < NV; k++) {
        double w = ac4_wave_sum(v[k]);
        if ((threadIdx.x & 63) == 0) s_red[k][threadIdx.x >> 6] = w;
    }
    __syncthreads();
    if (threadIdx.x < NV) {
        double s = 0.0;
        for (int w = 0; w < T / 64; w++) s += s_red[threadIdx.x][w];
        out[threadIdx.x] = s;
    }
}

// The pushed frame: its arrays (device), n particles, the types the caller may
// leave out (flag), and what tells the host that it has been read.
struct Frame {
    const double *x, *y, *z;
    const int *ty;
    int n, flag;
    double L, param;
    int obs;
    Origins org;
    int keep;             // place the frame is copied to, or -1
    // read(): every workgroup says when it has read its part of the frame; the
    // last one stores seq to the host's word, so the caller may have its
    // arrays back (null: nobody waits).  Groups of READ_GRP workgroups, then
    // the groups: atomics on one line are done one after the other (about 8
    // ns each), so the counts lie a line apart.
    unsigned *count, *word, seq;
};
#define READ_GRP 64
#define READ_PAD 32
__device__ __forceinline__ void frame_read(const Frame &F, int b, int nb) {  // one thread of workgroup b of nb
    if (!F.word) return;
    const auto last = [](unsigned *c, int of) {
        if (__hip_atomic_fetch_add(c, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1u != (unsigned)of) return false;
        __hip_atomic_store(c, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // for the next frame
        return true;
    };
    const int g = b / READ_GRP, ng = (nb + READ_GRP - 1) / READ_GRP;
    if (!last(F.count + (1 + g) * READ_PAD, min(READ_GRP, nb - g * READ_GRP))) return;
    if (ng > 1 && !last(F.count, ng)) return;
    __hip_atomic_store(F.word, F.seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// What k_frame and k_frame_fs leave per pair and block of particles:
// MSD sums (msd_pos.c:64-76) in msdp[(p0*nb + b)*3 + v];
// overlap count (overlap.c:61-84) in ovp[p1*nb + b];
// S4's overlap mask (S4Qt.c:125-133), bit i of mask[p1*nwords + i/32], count
// in s4p[p1*nb + b].
struct FrameOut {
    int ppb, nb;  // particles per block (a multiple of the block's threads), blocks
    double *msdp;
    int *ovp, *s4p, nwords;
    unsigned *mask;
};

// One pushed frame against the origins of its jobs: block b of row `row` on T
// threads (a row per job, then one that copies the frame to its place as an
// origin); workgroup wg of nwg.  S4's coordinates take the reference's
// per-lag single-if wraps (wrapn) exactly as it applies them.
template <int T>
__device__ __forceinline__ void frame_block(const Job *__restrict__ jobs, int nj, int row, int b, const Frame &F,
                                            const FrameOut &O, int wg, int nwg) {
    const double *__restrict__ x = F.x, *__restrict__ y = F.y, *__restrict__ z = F.z;
    const int *__restrict__ ty = F.ty;
    const int obs = F.obs, n = F.n, flag = F.flag;
    const double L = F.L, param = F.param;
    const int i0 = b * O.ppb, i1 = min(n, i0 + O.ppb), lane = threadIdx.x & 63;
    if (row >= nj) {  // the frame is an origin: keep it
        double *ox = F.org.at(F.keep, 0), *oy = F.org.at(F.keep, 1), *oz = F.org.at(F.keep, 2);
        for (int i = i0 + threadIdx.x; i < i1; i += T) {
            ox[i] = x[i];
            oy[i] = y[i];
            oz[i] = z[i];
        }
        __syncthreads();
        if (threadIdx.x == 0) frame_read(F, wg, nwg);
        return;
    }
    const Job J = jobs[row];
    const double *ox = F.org.at(J.org, 0), *oy = F.org.at(J.org, 1), *oz = F.org.at(J.org, 2);
    double v[3] = {0.0, 0.0, 0.0};
    int nov = 0, ns4 = 0;
    for (int t = i0; t < i1; t += T) {
        const int i = t + threadIdx.x;
        bool ov = false, s4 = false;
        if (i < i1) {
            const double xa = x[i], ya = y[i], za = z[i], xb = ox[i], yb = oy[i], zb = oz[i];
            const bool use = ty[i] != 1 || flag == 0;
            double dx = xa - xb, dy = ya - yb, dz = za - zb;
            if (J.p0 >= 0 && use) {
                double r2 = L * L * (dx * dx + dy * dy + dz * dz);
                double r3 = r2 * r2;
                double r4 = L * L * L * L * (dx * dx * dx * dx + dy * dy * dy * dy + dz * dz * dz * dz);
                v[0] += r2;  // sum
                v[1] += r4;  // sumSq
                v[2] += r3;  // sumCube
            }
            if (J.p1 >= 0 && (obs & AC4_OBS_OVERLAP)) {
                dz = minimg_ana(dz);
                dy = minimg_ana(dy);
                dx = minimg_ana(dx);
                ov = use && L * L * (dx * dx + dy * dy + dz * dz) < param;
            }
            if (J.p1 >= 0 && (obs & AC4_OBS_S4)) {
                const double x0 = wrapn(xb, J.slot), y0 = wrapn(yb, J.slot), z0 = wrapn(zb, J.slot);
                double ex = wrap1(xa) - x0, ey = wrap1(ya) - y0, ez = wrap1(za) - z0;
                ez = minimg_ana(ez);
                ey = minimg_ana(ey);
                ex = minimg_ana(ex);
                s4 = L * L * (ex * ex + ey * ey + ez * ez) < param;  // S4Qt.c:131-132
            }
        }
        nov += __popcll(__ballot(ov));
        if (J.p1 >= 0 && (obs & AC4_OBS_S4)) {
            const unsigned long long m = __ballot(s4);
            const int w = (t + (threadIdx.x & ~63)) >> 5;  // first of the wave's two words
            unsigned *row = O.mask + (size_t)J.p1 * O.nwords;
            if (lane == 0 && w < O.nwords) row[w] = (unsigned)m;
            if (lane == 1 && w + 1 < O.nwords) row[w + 1] = (unsigned)(m >> 32);
            ns4 += __popcll(m);
        }
    }
    __shared__ int s_c[2][T / 64];
    if (lane == 0) { s_c[0][threadIdx.x >> 6] = nov; s_c[1][threadIdx.x >> 6] = ns4; }
    __syncthreads();
    if (threadIdx.x == 0) frame_read(F, wg, nwg);
    if (J.p0 >= 0) block_sum_store<3, T>(v, O.msdp + ((size_t)J.p0 * O.nb + b) * 3);
    if (J.p1 >= 0 && threadIdx.x < 2 && (obs & (threadIdx.x == 0 ? AC4_OBS_OVERLAP : AC4_OBS_S4))) {
        int c = 0;
        for (int w = 0; w < T / 64; w++) c += s_c[threadIdx.x][w];
        (threadIdx.x == 0 ? O.ovp : O.s4p)[(size_t)J.p1 * O.nb + b] = c;
    }
}

// The frame without Fs: grid (blocks, rows).  k_msd_pairs and k_counts add the
// blocks up, for all pairs at once.  A frame has about one job, so a push is
// latencies whatever it does: three kernels, each with a reduction kernel of
// its own, the jobs copied from the host and a synchronisation per walk took
// 83 us per frame of 50000 particles (MSD, overlap, S4); one launch and one synchronisation 21.4,
// one launch whose workgroups say that they have read the frame 15.9 (the
// host's word arrives 4 us before the stream's end is seen: 7.7 against 11.8
// us for an empty kernel).
__global__ void __launch_bounds__(ABLK) k_frame(const Job *__restrict__ jobs, int nj, Frame F, FrameOut O) {
    frame_block<ABLK>(jobs, nj, blockIdx.y, blockIdx.x, F, O, blockIdx.y * gridDim.x + blockIdx.x,
                      gridDim.x * gridDim.y);
}

// out[p*3 + v] = the MSD sums of pair p over its nb blocks, in a fixed order;
// one workgroup per pair
__global__ void __launch_bounds__(ABLK) k_msd_pairs(const double *__restrict__ msdp, int nb, double *out) {
    double v[3] = {0.0, 0.0, 0.0};
    for (int b = threadIdx.x; b < nb; b += ABLK)
        for (int k = 0; k < 3; k++) v[k] += msdp[((size_t)blockIdx.x * nb + b) * 3 + k];
    block_sum_store<3>(v, out + (size_t)blockIdx.x * 3);
}

// out[p] = count of pair p over its nb blocks; one wave per pair
__global__ void __launch_bounds__(64) k_counts(const int *__restrict__ c, int nb, double *out) {
    int v = 0;
    for (int b = threadIdx.x; b < nb; b += 64) v += c[(size_t)blockIdx.x * nb + b];
    v = ac4_wave_sum_i(v);
    if (threadIdx.x == 0) out[blockIdx.x] = (double)v;
}

// Permutation s of a degeneracy-d vector in the order of S4Qt.c:133-214.
__host__ __device__ __forceinline__ void perm_q(int d, int s, int a, int b, int c, int &o0, int &o1, int &o2) {
    if (d == 1 || s == 0) { o0 = a; o1 = b; o2 = c; return; }
    if (d == 3) {
        if (s == 1) { o0 = b; o1 = c; o2 = a; } else { o0 = c; o1 = a; o2 = b; }
        return;
    }
    switch (s) {
        case 1: o0 = a; o1 = c; o2 = b; break;
        case 2: o0 = b; o1 = a; o2 = c; break;
        case 3: o0 = b; o1 = c; o2 = a; break;
        case 4: o0 = c; o1 = a; o2 = b; break;
        default: o0 = c; o1 = b; o2 = a; break;
    }
}

// The permuted GetQ vectors as columns (S4 and Fs)
#define S4_NCOL 576           // the 573 permuted vectors, padded to whole 16-column tiles
__constant__ int c_pv[3 * S4_NCOL];  // permuted vector (o0, o1, o2) per column; zero in the padding
__constant__ int c_pcol[AC4_NQ];     // first column of each GetQ vector

// ---------------------------------------------------------------- Fs
// Fsqt.c:103-222: for each (origin, lag) pair the sums over particles of
// exp(i q.p), p the particle's displacement, for the 573 permutations of the
// GetQ vectors.  q is a lattice vector (o0, o1, o2) of the box, so the phase
// factorises: exp(i q.p) = X[o0] Y[o1] Z[o2] with X[m] = exp(2 pi i m p_x).
// The sum over particles of products of two factors is a matrix product with
// the particles as the inner dimension, and every permuted vector is one
// entry of it: (i, j, j) is X[i] (YZ)[j] (and the same for the other axes:
// three products of 15 x 15), (0, k, i) with k = 1, 2 one factor of each of
// two axes (a product of 6 rows with 3 x 21 columns), (1, 0, 0) a row with a
// column of ones.  v_mfma_f64_16x16x4f64 takes 20 products of 16 x 16 per four
// particles, where forming each of the 573 phases took 573 sincos per
// particle (34 instructions each).  Per workgroup and tile of FS_P particles:
// the factors of the three axes, m = 1 ... 21, by sincos of the exactly
// reduced m p (63 per particle), the 45 products of two axes, both in LDS;
// then in each set of four waves wave w < 3 takes the product of axis w with
// the other two (real and imaginary parts, four MFMAs) and one of the eight
// tiles of the (0, k, i) group, wave 3 the other five.  The FS_SETS sets
// take every FS_SETS-th MFMA step and are added at the end in a fixed order: a
// frame has about one pair, so the launch is as long as one workgroup's tiles,
// and four waves per SIMD make them shorter.  Tiles of 16 particles: the 63
// factors of each are one round of the workgroup's threads, a set has one
// MFMA step, and a small frame's workgroups hold half as many particles.  1000
// and 20011 particles, per pair: one sincos per vector and particle 33.6 and
// 59.5 us, this 8.2 and 15.8 (tiles of 32 and the sets added one after the
// other 9.5 and 17.4; one set of waves, the displacements loaded per tile 13.3
// and 27.5).
#define FS_P 16        // particles of a tile
#define FS_M 21        // largest component of a GetQ vector
#define FS_J 15        // largest j of the (i, j, j) vectors
#define FS_RL 33       // row of a table: up to 32 values, padded against bank conflicts
#define FS_TILES 14    // accumulated 16 x 16 tiles: 3 x {cos, sin}, then the (0, k, i) group's 8
#define FS_LOAD 256    // particles whose displacements are loaded together
#define FS_NBLK 256    // workgroups per pair, at most
#define FS_WAIT 32     // jobs whose partials one reduction takes, at least (at most 21 MB)
#define FS_SETS 4      // sets of four waves per workgroup
#define FS_T (256 * FS_SETS)

typedef double ac4_d4 __attribute__((ext_vector_type(4)));

// rows of the axis table (axis a, component m = 0 ... 21, c = 0 cos, 1 sin) and of the product table (j = 1 ... 15)
__device__ __forceinline__ int fs_ax(int a, int m, int c) { return ((a * (FS_M + 1) + m) * 2 + c) * FS_RL; }
__device__ __forceinline__ int fs_pr(int a, int j, int c) {
    return (3 * (FS_M + 1) * 2 + (a * FS_J + j - 1) * 2 + c) * FS_RL;
}
#define FS_LDS ((3 * (FS_M + 1) * 2 + 3 * FS_J * 2) * FS_RL)  // doubles; the accumulated tiles reuse it

// cos and sin sums of the permuted vector (o0, o1, o2) from the accumulated tiles s_t[tile][row][column]
__device__ __forceinline__ void fs_entry(const double *s_t, int o0, int o1, int o2, double &c, double &s) {
    const int o[3] = {o0, o1, o2};
    const int nz = (o0 != 0) + (o1 != 0) + (o2 != 0);
    if (nz == 3) {
        const int a = o1 == o2 ? 0 : (o0 == o2 ? 1 : 2), j = a == 0 ? o1 : o0;  // axis of the odd component
        const int e = (o[a] - 1) * 16 + j - 1;
        c = s_t[(2 * a) * 256 + e];
        s = s_t[(2 * a + 1) * 256 + e];
        return;
    }
    // row axis: a component of 1 or 2; column axis: the other one, or the column of ones
    int ra = o0 != 0 ? 0 : (o1 != 0 ? 1 : 2), ca = o2 != 0 ? 2 : (o1 != 0 ? 1 : 0);
    if (o[ra] > 2) { const int t = ra; ra = ca; ca = t; }
    const int r = 2 * ra + o[ra] - 1, q = nz == 2 ? ca * FS_M + o[ca] - 1 : 63;
    const double *t0 = s_t + (6 + 2 * (q >> 4)) * 256 + (q & 15), *t1 = t0 + 256;
    c = t0[r * 16] - t1[(r + 6) * 16];
    s = t0[(r + 6) * 16] + t1[r * 16];
}

// Block blk (ppb particles, a multiple of FS_P) of job J; out[n] = cos sum,
// out[AC4_NQ + n] = sin sum, averaged over the vector's permutations.
__device__ __forceinline__ void fs_block(const Job &J, int blk, int ppb, const Frame &F, double *__restrict__ out, int wg,
                                         int nwg) {
    const double *__restrict__ x = F.x, *__restrict__ y = F.y, *__restrict__ z = F.z;
    const int *__restrict__ ty = F.ty;
    const int n = F.n, flag = F.flag;
    __shared__ double s_t[FS_LDS];
    __shared__ double s_p[3][FS_LOAD];
    __shared__ double s_use[FS_LOAD];
    const int t = threadIdx.x, lane = t & 63, set = t >> 8, wv = (t >> 6) & 3, i16 = lane & 15, k4 = lane >> 4;
    const double *ox = F.org.at(J.org, 0), *oy = F.org.at(J.org, 1), *oz = F.org.at(J.org, 2);
    // for the end: this thread's permuted vector, and of its output value the columns
    const int pc = min(t, S4_NCOL - 1), o0 = c_pv[3 * pc], o1 = c_pv[3 * pc + 1], o2 = c_pv[3 * pc + 2];
    const int oq = t < 2 * AC4_NQ ? t % AC4_NQ : 0, od = c_dg[oq], oc = c_pcol[oq];
    ac4_d4 acc[5];
    for (int q = 0; q < 5; q++) acc[q] = ac4_d4{0.0, 0.0, 0.0, 0.0};
    // operand rows of this lane (in the tables, without the particle): the
    // axis row i16 + 1 and product column i16 + 1 of waves 0-2; the (0, k, i)
    // group's row and its four columns
    const int oth = wv < 3 ? wv : 0;
    const int xa = fs_ax(oth, i16 + 1, 0), pb = fs_pr(oth, min(i16 + 1, FS_J), 0);
    const int kr = min(i16, 11), ka = fs_ax((kr % 6) >> 1, (kr & 1) + 1, kr / 6);
    int kb[4];
    for (int q = 0; q < 4; q++) {
        const int cq = 16 * q + i16;
        kb[q] = cq < 3 * FS_M ? fs_ax(cq / FS_M, cq % FS_M + 1, 0) : fs_ax(0, 0, 0);
    }
    const int i0 = blk * ppb, i1 = min(n, i0 + ppb);
    for (int tb = i0; tb < i1; tb += FS_P) {
        const int lb = (tb - i0) & (FS_LOAD - 1);  // the tile among the loaded particles
        if (lb == 0 && t < FS_LOAD) {
            const int i = tb + t;
            double p0 = 0.0, p1 = 0.0, p2 = 0.0, use = 0.0;
            if (i < i1) {
                const int ti = ty[i];
                const double xb = ox[i], yb = oy[i], zb = oz[i], xc = x[i], yc = y[i], zc = z[i];
                if (ti != 1 || flag == 0) {
                    // phases of the displacement (Fsqt.c:145-146)
                    p0 = minimg_ana(wrap1(xc) - wrapn(xb, J.slot));
                    p1 = minimg_ana(wrap1(yc) - wrapn(yb, J.slot));
                    p2 = minimg_ana(wrap1(zc) - wrapn(zb, J.slot));
                    use = 1.0;
                }
            }
            s_p[0][t] = p0; s_p[1][t] = p1; s_p[2][t] = p2;
            s_use[t] = use;
        }
        if (lb == 0) {
            __syncthreads();
            if (t == FS_T - 1 && tb + FS_LOAD >= i1) frame_read(F, wg, nwg);
        }
        if (t < FS_P) {
            s_t[fs_ax(0, 0, 0) + t] = s_use[lb + t];  // the column of ones
            s_t[fs_ax(0, 0, 1) + t] = 0.0;
        }
        const int pp = t & (FS_P - 1);
        const bool use = s_use[lb + pp] != 0.0;
        for (int e = t / FS_P; e < 3 * FS_M; e += FS_T / FS_P) {
            const int a = e / FS_M, m = e - a * FS_M + 1;
            // Fsqt.c:147-213 forms arg = q.L.p with q = 2*A_PI/L*(o0,o1,o2);
            // in turns the component's part is m p, its whole turns taken off
            // the unrounded product.  The reference's A_PI and its invL*L
            // differ from pi and 1 in the 15th digit: below 1e-12 in the phase.
            const double p = s_p[a][lb + pp], f = fma((double)m, p, -rint((double)m * p));
            double sn, cs;
            ac4_sincos_turns(f, &sn, &cs);
            s_t[fs_ax(a, m, 0) + pp] = use ? cs : 0.0;
            s_t[fs_ax(a, m, 1) + pp] = use ? sn : 0.0;
        }
        __syncthreads();
        for (int e = t / FS_P; e < 3 * FS_J; e += FS_T / FS_P) {
            const int a = e / FS_J, j = e - a * FS_J + 1, b = a == 0 ? 1 : 0, c = a == 2 ? 1 : 2;
            const double cb = s_t[fs_ax(b, j, 0) + pp], sb = s_t[fs_ax(b, j, 1) + pp], cc = s_t[fs_ax(c, j, 0) + pp],
                         sc = s_t[fs_ax(c, j, 1) + pp];
            s_t[fs_pr(a, j, 0) + pp] = fma(cb, cc, -(sb * sc));
            s_t[fs_pr(a, j, 1) + pp] = fma(sb, cc, cb * sc);
        }
        __syncthreads();
        if (wv < 3) {
            const int kq = kb[0] * (wv == 0 || wv == 1) + kb[1] * (wv == 2) + (wv == 1 ? FS_RL : 0);  // tiles 0, 1, 2
#pragma unroll
            for (int st = set; st < FS_P / 4; st += FS_SETS) {
                const int q = 4 * st + k4;
                const double ac = s_t[xa + q], as = s_t[xa + FS_RL + q], bc = s_t[pb + q], bs = s_t[pb + FS_RL + q];
                acc[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(ac, bc, acc[0], 0, 0, 0);
                acc[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(as, bc, acc[1], 0, 0, 0);
                acc[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(-as, bs, acc[0], 0, 0, 0);
                acc[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(ac, bs, acc[1], 0, 0, 0);
                acc[2] = __builtin_amdgcn_mfma_f64_16x16x4f64(s_t[ka + q], s_t[kq + q], acc[2], 0, 0, 0);
            }
        } else {
#pragma unroll
            for (int st = set; st < FS_P / 4; st += FS_SETS) {
                const int q = 4 * st + k4;
                const double a = s_t[ka + q];  // tiles 3 ... 7: columns 16..31 sin, 32..47 and 48..63 cos and sin
                acc[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, s_t[kb[1] + FS_RL + q], acc[0], 0, 0, 0);
                acc[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, s_t[kb[2] + q], acc[1], 0, 0, 0);
                acc[2] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, s_t[kb[2] + FS_RL + q], acc[2], 0, 0, 0);
                acc[3] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, s_t[kb[3] + q], acc[3], 0, 0, 0);
                acc[4] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, s_t[kb[3] + FS_RL + q], acc[4], 0, 0, 0);
            }
        }
        __syncthreads();
    }
    // the accumulated tiles to LDS (element e of lane l: row l/16 + 4*e, column
    // l%16): sets 0 and 1 to two areas, sets 2 and 3 added to them
    static_assert(FS_SETS == 4 && 2 * FS_TILES * 256 <= FS_LDS, "two areas of tiles in the tables' place");
    for (int w = 0; w < 2; w++) {
        if (set >> 1 == w)
#pragma unroll
            for (int q = 0; q < 5; q++) {
                if (wv < 3 && q >= 3) continue;
                const int tile = (set & 1) * FS_TILES + (wv < 3 ? (q < 2 ? 2 * wv + q : 6 + wv) : 9 + q);
                for (int e = 0; e < 4; e++) {
                    double *d = &s_t[tile * 256 + (k4 + 4 * e) * 16 + i16];
                    *d = w == 0 ? acc[q][e] : *d + acc[q][e];
                }
            }
        __syncthreads();
    }
    // the permuted vectors' sums, then each vector's average over its permutations
    double c = 0.0, sn = 0.0;
    if (t < S4_NCOL - 3) {
        double c1, s1;
        fs_entry(s_t, o0, o1, o2, c, sn);
        fs_entry(s_t + FS_TILES * 256, o0, o1, o2, c1, s1);
        c += c1;
        sn += s1;
    }
    __syncthreads();
    if (t < S4_NCOL) {
        s_t[t] = c;
        s_t[S4_NCOL + t] = sn;
    }
    __syncthreads();
    if (t < 2 * AC4_NQ) {
        const double *src = s_t + (t < AC4_NQ ? 0 : S4_NCOL) + oc;
        double v = 0.0;
        for (int k = 0; k < od; k++) v += src[k];
        out[t] = od == 1 ? v : v / (double)od;
    }
}

// The frame with Fs in one launch: workgroups [0, nj*fs_nb) Fs, a job's block
// each (partial[(job*fs_nb + blk)*2*AC4_NQ + value]), the rest `rows` rows of
// O.nb frame blocks.  As two launches, a reduction and the stream's end waited
// for: 25.6 us per frame of 1000 particles, all four observables, and 31.7 of
// 20011, Fs alone; this, the partials of FS_WAIT jobs reduced together, 11.1
// and 16.8 (with Fs tiles of 32).
__global__ void __launch_bounds__(FS_T) k_frame_fs(const Job *__restrict__ jobs, int nj, int nf, int fs_nb, int fs_ppb,
                                                   Frame F, FrameOut O, double *partial) {
    const int wg = blockIdx.x, nwg = gridDim.x;
    if (wg >= nj * fs_nb) {
        const int k = wg - nj * fs_nb;
        frame_block<FS_T>(jobs, nf, k / O.nb, k % O.nb, F, O, wg, nwg);
        return;
    }
    const int j = wg / fs_nb;
    const Job J = jobs[j];
    if (J.p1 < 0) {
        if (threadIdx.x == 0) frame_read(F, wg, nwg);
        return;
    }
    fs_block(J, wg - j * fs_nb, fs_ppb, F, partial + (size_t)wg * (AC4_NQ * 2), wg, nwg);
}

// ---------------------------------------------------------------- S4
// S4Qt.c:101-216 sums, for each (origin, lag) pair and GetQ vector q, the
// phase exp(i q.r0) of every particle that still overlaps its origin
// position at the lag (|r(t) - r0| < a), averaged over q's permutations.
// The phase depends on the origin frame alone, so it is evaluated once per
// origin and shared by all of that origin's lags:
//   k_frame(_fs) at each lag frame: the overlap mask of the pair, one bit per
//               particle (and the overlap count of the pair);
//   k_s4_origin when the origin's last lag has been masked: the mask matrix
//               M[lags][particle] times the phase matrix P[particle][573
//               permuted vectors] on FP64 matrix cores, P formed in registers
//               and never stored;
//   k_s4_reduce sums the chunk partials in a fixed order and divides by the
//               number of each vector's permutations.
//
// As in Fs a phase is a product of one factor each of two tables (the axis
// factors exp(2 pi i m x), m = 0 ... 21, and the products (j, j) of two axes),
// built per tile of particles in LDS: 63 sincos and 45 products per particle
// for 573 phases of four multiplications, where a sincos per phase (34
// instructions) took 2/5 of the time.  One workgroup takes its particles
// through all 36 column tiles (12 waves, three tiles each), so the tables are
// built once.  The lags are 16 rows per v_mfma_f64_16x16x4f64 and, for what is
// left of them, 4 per v_mfma_f64_4x4x4f64 (four blocks of 4 x 4, the four
// columns each of the same B operand; the same rate, 64 against 68 TFLOP/s
// measured): 22 lags cost 24 rows, not 32.  The bound is the issue of the FP64 matrix
// and vector instructions, which share their rate: of 78.7 us at 50000
// particles and 22 lags 52 are the products, 10 the tables; a workgroup per
// chunk and column tile with a sincos per phase took 110, its reduction of
// 576 columns per lag 13.5 (k_s4_reduce's 324 values 4.8).
#define S4_NCT (S4_NCOL / 16) // column tiles
#define S4_P 32        // particles of a tile, at most
#define S4_WAVES 12
#define S4_CPW (S4_NCT / S4_WAVES)  // column tiles of a wave
#define S4_T (64 * S4_WAVES)
#define S4_LAGS 32     // lags of one pass, at most
#define S4_CHUNKS 256  // workgroups of a pass, at most
#define S4_SMALL 3072  // particles up to which k_s4_small is the faster one
#define S4_SMALL_CHUNKS 64

// The table rows (cos; sin at + FS_RL) whose product is the permuted vector (o0, o1, o2)
__device__ __forceinline__ void s4_rows(int o0, int o1, int o2, int &u, int &v) {
    const int o[3] = {o0, o1, o2};
    if (o0 != 0 && o1 != 0 && o2 != 0) {  // (i, j, j): the odd component with the product of the equal ones
        const int a = o1 == o2 ? 0 : (o0 == o2 ? 1 : 2), j = a == 0 ? o1 : o0;
        u = fs_ax(a, o[a], 0);
        v = fs_pr(a, j, 0);
        return;
    }
    // up to two components; axis 0's m = 0 is the row of ones
    const int a = o0 != 0 ? 0 : (o1 != 0 ? 1 : 2), b = o2 != 0 ? 2 : 1;
    u = o[a] != 0 ? fs_ax(a, o[a], 0) : fs_ax(0, 0, 0);
    v = b != a && o[b] != 0 ? fs_ax(b, o[b], 0) : fs_ax(0, 0, 0);
}

// One origin, one pass of nl <= 16*NT16 + 4*NT4 of its lags: grid (chunks of
// ppb particles), tiles of tp <= S4_P particles (both multiples of 4).
// v_mfma_f64_16x16x4f64: lane l = i + 16k holds A[i][k] (mask bit of lag i,
// particle k) and B[k][j] with j = i (phase of vector j for particle k); the
// accumulator's element e of lane l is row l/16 + 4*e, column l%16.
// v_mfma_f64_4x4x4f64: the same B; lane l holds A[l%4][l/16], and the
// accumulator of lane l is row l/16, column l%16.
// part[((chunk*nl + lag)*2 + {cos,sin})*AC4_NQ + vector]: sums over the
// vector's permutations.
template <int NT16, int NT4>
__global__ void __launch_bounds__(S4_T) k_s4_origin(const double *__restrict__ x0, const double *__restrict__ y0,
                                                    const double *__restrict__ z0, int n, int nwords,
                                                    const unsigned *__restrict__ mask, const int *__restrict__ lags,
                                                    int nl, int ppb, int tp, double *__restrict__ part) {
    constexpr int NR = NT16 + NT4, ROWS = 16 * NT16 + 4 * NT4;
    constexpr int LDS = FS_LDS > ROWS * S4_NCOL ? FS_LDS : ROWS * S4_NCOL;
    __shared__ double s_t[LDS];  // the tables, then the sums of one of cos and sin
    __shared__ double s_p[3][S4_P];
    __shared__ int s_dc[AC4_NQ];  // permutations and first column of each vector, for the end
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6, i16 = lane & 15, k4 = lane >> 4, pp = t & (S4_P - 1);
    int u[S4_CPW], v[S4_CPW];
#pragma unroll
    for (int c = 0; c < S4_CPW; c++) {
        const int col = (wv * S4_CPW + c) * 16 + i16;
        s4_rows(c_pv[3 * col], c_pv[3 * col + 1], c_pv[3 * col + 2], u[c], v[c]);
    }
    const unsigned *mrow[NR];  // this lane's lag of each row tile
    bool live[NR];
#pragma unroll
    for (int r = 0; r < NR; r++) {
        const int l = r < NT16 ? 16 * r + i16 : 16 * NT16 + 4 * (r - NT16) + (lane & 3);
        live[r] = l < nl;
        mrow[r] = mask + (size_t)lags[live[r] ? l : 0] * nwords;
    }
    ac4_d4 ac[S4_CPW][NT16 > 0 ? NT16 : 1], as[S4_CPW][NT16 > 0 ? NT16 : 1];
    double bc[S4_CPW][NT4 > 0 ? NT4 : 1], bs[S4_CPW][NT4 > 0 ? NT4 : 1];
#pragma unroll
    for (int c = 0; c < S4_CPW; c++) {
        for (int r = 0; r < NT16; r++) ac[c][r] = as[c][r] = ac4_d4{0.0, 0.0, 0.0, 0.0};
        for (int r = 0; r < NT4; r++) bc[c][r] = bs[c][r] = 0.0;
    }
    const int i0 = blockIdx.x * ppb, i1 = min(n, i0 + ppb);
    // exp(i q.r0) is periodic in r0 with the box, so the stored origin
    // coordinate is used as it is, whatever single-if wraps the reference
    // applies to it at a given lag.  A particle past n has no mask bit: its
    // (clamped) phase is multiplied by zero; so has one of the next chunk.
    const double *src = t < S4_P ? x0 : (t < 2 * S4_P ? y0 : z0);
    double p = t < 3 * S4_P ? src[min(i0 + pp, n - 1)] : 0.0;
    if (t < AC4_NQ) s_dc[t] = c_pcol[t] << 3 | c_dg[t];
    if (t < S4_P) {
        s_t[fs_ax(0, 0, 0) + t] = 1.0;
        s_t[fs_ax(0, 0, 1) + t] = 0.0;
    }
    for (int tb = i0; tb < i1; tb += tp) {
        if (t < 3 * S4_P) s_p[t / S4_P][pp] = p;
        // the mask words of this tile, loaded while its tables are built
        const int w = tb >> 5, sh = tb & 31, cnt = min(tp, i1 - tb);
        unsigned mw[NR], mx[NR];
#pragma unroll
        for (int r = 0; r < NR; r++) {
            mw[r] = mrow[r][w];
            mx[r] = mrow[r][sh + cnt > 32 ? w + 1 : w];
        }
        __syncthreads();
        if (t < 3 * S4_P) p = src[min(tb + tp + pp, n - 1)];  // the next tile's
        for (int e = t / S4_P; e < 3 * FS_M; e += S4_T / S4_P) {
            const int a = e / FS_M, m = e - a * FS_M + 1;
            const double q = s_p[a][pp], f = fma((double)m, q, -rint((double)m * q));
            double sn, cs;
            ac4_sincos_turns(f, &sn, &cs);
            s_t[fs_ax(a, m, 0) + pp] = cs;
            s_t[fs_ax(a, m, 1) + pp] = sn;
        }
        __syncthreads();
        for (int e = t / S4_P; e < 3 * FS_J; e += S4_T / S4_P) {
            const int a = e / FS_J, j = e - a * FS_J + 1, b = a == 0 ? 1 : 0, c = a == 2 ? 1 : 2;
            const double cb = s_t[fs_ax(b, j, 0) + pp], sb = s_t[fs_ax(b, j, 1) + pp], cc = s_t[fs_ax(c, j, 0) + pp],
                         sc = s_t[fs_ax(c, j, 1) + pp];
            s_t[fs_pr(a, j, 0) + pp] = fma(cb, cc, -(sb * sc));
            s_t[fs_pr(a, j, 1) + pp] = fma(sb, cc, cb * sc);
        }
        __syncthreads();
        // the bits of the tile's particles, its first one lowest
#pragma unroll
        for (int r = 0; r < NR; r++) {
            const unsigned long long m = (unsigned long long)mx[r] << 32 | mw[r];
            mw[r] = live[r] ? (unsigned)(m >> sh) & (cnt < 32 ? (1u << cnt) - 1u : ~0u) : 0u;
        }
        for (int st = 0; st < tp; st += 4) {
            const int q = st + k4;
            double a[NR];
#pragma unroll
            for (int r = 0; r < NR; r++) a[r] = (mw[r] >> q) & 1u ? 1.0 : 0.0;
#pragma unroll
            for (int c = 0; c < S4_CPW; c++) {
                const double uc = s_t[u[c] + q], us = s_t[u[c] + FS_RL + q], vc = s_t[v[c] + q], vs = s_t[v[c] + FS_RL + q];
                const double pc = fma(uc, vc, -(us * vs)), ps = fma(us, vc, uc * vs);
#pragma unroll
                for (int r = 0; r < NT16; r++) {
                    ac[c][r] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[r], pc, ac[c][r], 0, 0, 0);
                    as[c][r] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[r], ps, as[c][r], 0, 0, 0);
                }
#pragma unroll
                for (int r = 0; r < NT4; r++) {
                    bc[c][r] = __builtin_amdgcn_mfma_f64_4x4x4f64(a[NT16 + r], pc, bc[c][r], 0, 0, 0);
                    bs[c][r] = __builtin_amdgcn_mfma_f64_4x4x4f64(a[NT16 + r], ps, bs[c][r], 0, 0, 0);
                }
            }
        }
        __syncthreads();
    }
    const int oq = t % AC4_NQ, od = s_dc[oq] & 7, oc = s_dc[oq] >> 3;  // this thread's vector, its columns
#pragma unroll
    for (int sn = 0; sn < 2; sn++) {
#pragma unroll
        for (int c = 0; c < S4_CPW; c++) {
            double *d = &s_t[(wv * S4_CPW + c) * 16 + i16 + k4 * S4_NCOL];
#pragma unroll
            for (int r = 0; r < NT16; r++)
#pragma unroll
                for (int e = 0; e < 4; e++) d[(16 * r + 4 * e) * S4_NCOL] = sn ? as[c][r][e] : ac[c][r][e];
#pragma unroll
            for (int r = 0; r < NT4; r++) d[(16 * NT16 + 4 * r) * S4_NCOL] = sn ? bs[c][r] : bc[c][r];
        }
        __syncthreads();
        // thread t: vector t % AC4_NQ of lags t / AC4_NQ, + S4_T / AC4_NQ, ...
        for (int l = t / AC4_NQ; l < nl && t < S4_T / AC4_NQ * AC4_NQ; l += S4_T / AC4_NQ) {
            const double *w = s_t + l * S4_NCOL + oc;
            double sum = w[0];
            if (od > 1) sum = (sum + w[1]) + w[2];
            if (od > 3) sum = ((sum + w[3]) + w[4]) + w[5];
            part[(((size_t)blockIdx.x * nl + l) * 2 + sn) * AC4_NQ + oq] = sum;
        }
        __syncthreads();
    }
}

// Per lag l of the pass and value v (v < AC4_NQ: cos sum of vector v, else
// sin sum of vector v - AC4_NQ): grid (nl, ceil(2*AC4_NQ/64)), 1024 threads.
// Wave w sums chunks w, w+16, ..., the 16 wave sums are added in order and
// divided by the number of permutations.  s4[pair*2*AC4_NQ + v].
#define S4_RW 16
__global__ void __launch_bounds__(64 * S4_RW) k_s4_reduce(const double *__restrict__ part, int nchunk, int nl,
                                                          const int *__restrict__ lags, double *__restrict__ s4) {
    const int l = blockIdx.x;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int v = blockIdx.y * 64 + lane;
    const bool ok = v < 2 * AC4_NQ;
    const double *src = part + (size_t)l * 2 * AC4_NQ + (ok ? v : 0);
    double acc = 0.0;
#pragma unroll 4
    for (int c = wv; c < nchunk; c += S4_RW) acc += src[(size_t)c * nl * 2 * AC4_NQ];
    __shared__ double s_w[S4_RW][64];
    s_w[wv][lane] = acc;
    __syncthreads();
    if (wv == 0 && ok) {
        double tot = s_w[0][lane];
        for (int w = 1; w < S4_RW; w++) tot += s_w[w][lane];
        s4[(size_t)lags[l] * 2 * AC4_NQ + v] = tot / (double)c_dg[v < AC4_NQ ? v : v - AC4_NQ];
    }
}

// The same for small systems (n <= S4_SMALL), where the launch is as long as
// one workgroup: a workgroup per chunk and column tile, each phase by a sincos
// of its own, the waves' particles split further.  us per origin with its
// reduction, 22 lags: 1000 particles 12.0 against k_s4_origin's 18.2, 4000 the
// same, 50000 124 against 83.5.
// One pass of up to RT*16 lags: grid (chunks, S4_NCT), 256 threads.  Wave w of block (c, ct) takes the mask words
// [(4c+w)*wpw, (4c+w+1)*wpw) -- 32 particles each, 4 per MFMA step -- and
// the 16 permuted vectors of column tile ct.  v_mfma_f64_16x16x4f64 operand
// layout: lane l = i + 16k holds A[i][k] (mask bit of lag i, particle k) and
// B[k][j] with j = i (phase of vector j for particle k); the accumulator's
// element e of lane l is row l/16 + 4*e, column l%16.  The four waves'
// sums are added in wave order through LDS, and the block writes
// part[((c*rows + row)*2 + {cos,sin})*S4_NCOL + column].
template <int RT>
__global__ void __launch_bounds__(256) k_s4_small(const double *__restrict__ x0, const double *__restrict__ y0,
                                                   const double *__restrict__ z0, int n, int nwords,
                                                   const unsigned *__restrict__ mask, const int *__restrict__ lags,
                                                   int nl, int wpw, double *__restrict__ part) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int ct = blockIdx.y;
    const int i16 = lane & 15, k = lane >> 4;
    const int col = ct * 16 + i16;
    const double o0 = (double)c_pv[3 * col], o1 = (double)c_pv[3 * col + 1], o2 = (double)c_pv[3 * col + 2];
    const unsigned *mrow[RT];
    bool live[RT];
    for (int r = 0; r < RT; r++) {
        const int l = 16 * r + i16;
        live[r] = l < nl;
        mrow[r] = mask + (size_t)lags[live[r] ? l : 0] * nwords;
    }
    ac4_d4 ac[RT], as[RT];
    for (int r = 0; r < RT; r++) {
        ac[r] = ac4_d4{0.0, 0.0, 0.0, 0.0};
        as[r] = ac4_d4{0.0, 0.0, 0.0, 0.0};
    }
    const int w0 = (blockIdx.x * 4 + wv) * wpw;
    const int w1 = min(w0 + wpw, nwords);
    for (int w = w0; w < w1; w++) {
        unsigned mw[RT];
        for (int r = 0; r < RT; r++) mw[r] = live[r] ? mrow[r][w] : 0u;
#pragma unroll
        for (int kk = 0; kk < 8; kk++) {
            // A particle past n has no mask bit: its (clamped) phase is
            // multiplied by zero.  exp(i q.r0) is periodic in r0 with the
            // box, so the stored origin coordinate is used as it is, whatever
            // single-if wraps the reference applies to it at a given lag.
            const int i = min(32 * w + 4 * kk + k, n - 1);
            double s, c;
            ac4_sincos_turns(fma(o2, z0[i], fma(o1, y0[i], o0 * x0[i])), &s, &c);
            const int bit = 4 * kk + k;
            for (int r = 0; r < RT; r++) {
                const double a = ((mw[r] >> bit) & 1u) ? 1.0 : 0.0;
                ac[r] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, c, ac[r], 0, 0, 0);
                as[r] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, s, as[r], 0, 0, 0);
            }
        }
    }
    __shared__ double s_acc[RT * 16 * 32];
    for (int step = 0; step < 4; step++) {
        if (wv == step)
            for (int r = 0; r < RT; r++)
                for (int e = 0; e < 4; e++) {
                    const int row = 16 * r + k + 4 * e;
                    double *pc = &s_acc[row * 32 + i16], *ps = &s_acc[row * 32 + 16 + i16];
                    if (step == 0) { *pc = ac[r][e]; *ps = as[r][e]; }
                    else { *pc += ac[r][e]; *ps += as[r][e]; }
                }
        __syncthreads();
    }
    const int rows = RT * 16;
    for (int t = threadIdx.x; t < rows * 32; t += 256) {
        const int row = t >> 5, cc = t & 31, sn = cc >> 4;
        part[((size_t)(blockIdx.x * rows + row) * 2 + sn) * S4_NCOL + ct * 16 + (cc & 15)] = s_acc[t];
    }
}

// Per lag l of the pass and value v (v < AC4_NQ: cos sum of vector v, else
// sin sum of vector v - AC4_NQ): grid (nl, ceil(2*AC4_NQ/64)), 256 threads.
// Wave w sums chunks w, w+4, ... (each over the vector's permutations in
// order); the four wave sums are added in wave order and divided by the
// number of permutations.  s4[pair*2*AC4_NQ + v].
__global__ void __launch_bounds__(256) k_s4_small_reduce(const double *__restrict__ part, int nchunk, int rows,
                                                   const int *__restrict__ lags, double *__restrict__ s4) {
    const int l = blockIdx.x;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int v = blockIdx.y * 64 + lane;
    const bool ok = v < 2 * AC4_NQ;
    const int sn = ok && v >= AC4_NQ ? 1 : 0;
    const int q = ok ? v - sn * AC4_NQ : 0;
    const int d = c_dg[q], c0 = c_pcol[q];
    double acc = 0.0;
    if (ok)
        for (int c = wv; c < nchunk; c += 4) {
            const double *src = part + ((size_t)(c * rows + l) * 2 + sn) * S4_NCOL + c0;
            double t = 0.0;
            for (int s = 0; s < d; s++) t += src[s];
            acc += t;
        }
    __shared__ double s_w[4][64];
    s_w[wv][lane] = acc;
    __syncthreads();
    if (wv == 0 && ok) {
        const double tot = ((s_w[0][lane] + s_w[1][lane]) + s_w[2][lane]) + s_w[3][lane];
        s4[(size_t)lags[l] * 2 * AC4_NQ + v] = tot / (double)d;
    }
}

// Fixed-order sum over blocks of Fs's partials: out[p1*nv + v] = sum_b partial[(job*nb+b)*nv + v].
// Grid (jobs, ceil(nv/64)), 256 threads: lane l of wave w takes value
// v = 64*blockIdx.y + l (consecutive values, coalesced loads) and the blocks
// b = w, w+4, w+8, ... with 8 loads in flight; the four wave sums are added
// in wave order.  The order depends on nb and nv only.
__global__ void __launch_bounds__(256) k_reduce_jobs(const Job *__restrict__ jobs, int nb, int nv,
                                                     const double *__restrict__ partial, double *out) {
    __shared__ double s_w[4][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, v = blockIdx.y * 64 + lane;
    if (jobs[blockIdx.x].p1 < 0) return;  // uniform over the workgroup
    double acc = 0.0;
    if (v < nv) {
        const double *p = partial + (size_t)blockIdx.x * nb * nv + v;
        int b = w;
        for (; b + 28 < nb; b += 32) {
            double t[8];
#pragma unroll
            for (int u = 0; u < 8; u++) t[u] = p[(size_t)(b + 4 * u) * nv];
#pragma unroll
            for (int u = 0; u < 8; u++) acc += t[u];
        }
        for (; b < nb; b += 4) acc += p[(size_t)b * nv];
    }
    s_w[w][lane] = acc;
    __syncthreads();
    if (w == 0 && v < nv) {
        out[(size_t)jobs[blockIdx.x].p1 * nv + v] = ((s_w[0][lane] + s_w[1][lane]) + s_w[2][lane]) + s_w[3][lane];
    }
}

// Slot accumulation in walk (origin) order, msd_pos.c:87-93 / overlap.c:89-94 /
// S4Qt.c:231-236.  mode 0: sum += val/div; mode 1: s = val/div (div>0) or val;
// sum += s; sq += s*s.
__global__ void k_slots(const double *__restrict__ vals, int nv, const int *__restrict__ ptr,
                        const int *__restrict__ pairs, int nslots, int mode, double div, double *sum, double *sq) {
    const int t = blockIdx.x;
    for (int v = threadIdx.x; v < nv; v += blockDim.x) {
        double a = 0.0, b = 0.0;
        for (int k = ptr[t]; k < ptr[t + 1]; k++) {
            double s = vals[(size_t)pairs[k] * nv + v];
            if (div > 0.0) s = s / div;
            a += s;
            if (mode == 1) b += s * s;
        }
        sum[(size_t)t * nv + v] = a;
        if (mode == 1) sq[(size_t)t * nv + v] = b;
    }
}

// ------------------------------------------------------------------ host
struct WalkInfo {
    ac4_walk_t w;
    std::vector<int> last_use;             // per origin pos: last frame pos needing it
    std::vector<int> slot_ptr, slot_pairs; // CSR of pairs per slot (walk order)
    int nslots = 0, used = 0;              // slots, those up to the last that has a pair
};

struct ac4_ana {
    int n = 0, nframes = 0, gap = 0, obs = 0, flag = 0;
    double L = 0, invL = 0, factor = 1.4, a = 0.3, param = 0.09;
    std::vector<int> fidx;
    WalkInfo W[2];
    // the plan: each frame's jobs (CSR by frame position) and their origin
    // frames, each origin's place among the resident frames (-1: no origin),
    // the origins by the frame of their last lag; which origins are resident
    std::vector<Job> jobs;
    std::vector<int> jorg, jptr, place;
    std::vector<std::vector<int>> ends;
    std::vector<char> resident;
    Origins org{nullptr, 0};    // the resident frames
    double *cur = nullptr;      // a frame pushed from the host that is no origin: x, y, z
    int *cur_t = nullptr;       // types of a frame pushed from the host
    int last_pos = -1;
    double *d_msd = nullptr, *d_ov = nullptr, *d_s4 = nullptr, *d_s4m = nullptr, *d_fs = nullptr;
    double *d_part = nullptr, *d_msdp = nullptr;
    int *d_ovp = nullptr, *d_s4p = nullptr;  // per block: overlap counts of the overlap and the S4 rule
    Job *d_jobs = nullptr;
    unsigned *d_read = nullptr, *h_read = nullptr, seq = 0;  // Frame::count, ::word (pinned, with the first device push), ::seq
    bool stale = false;         // frames came in since d_msd, d_ov and d_s4m were formed from the blocks' values
    // S4 by origin: pair ids per origin (CSR, walk order), origins whose
    // last lag is frame pos, the pairs' overlap masks and the chunk partials
    std::vector<int> s4_optr, s4_opairs;
    std::vector<std::vector<int>> s4_end;
    std::vector<char> s4_done;
    int *d_s4_opairs = nullptr;
    unsigned *d_s4mask = nullptr;
    double *d_s4part = nullptr;
    int nwords = 0, s4_ppb = 16, s4_tp = 16, s4_nchunk = 1, s4_wpw = 1;
    int fs_j0 = 0, fs_j1 = 0, fs_wait = 0;  // jobs whose Fs partials are in d_part, how many it holds
    int max_jobs = 0, ppb = ABLK, nb = 0, fs_ppb = FS_P, fs_nb = 0;
    std::vector<int> vx, vy, vz, qsq;
    std::vector<double> qval;
    char *mem = nullptr;        // all of them
    hipStream_t stream = nullptr;
    int dev = 0;                // the device the handle was made on
    bool finalized = false;
    // slot results
    std::vector<double> m0, m1, m2, c, x4, s4c, s4s, s4c2, s4s2, fsc, fss, fsc2, fss2;
    std::vector<int> cnt0, cnt1;
    std::vector<double> dt0, dt1;
    int noi_msd = 0, noi_ov = 0;
};

#define TRY(e) do { int rc_ = (e); if (rc_ != AC4_OK) return rc_; } while (0)

static void build_walk_info(ac4_ana *an, WalkInfo &W, int rule) {
    ac4_walk(an->fidx.data(), an->nframes, an->gap, an->factor, rule, &W.w);
    W.last_use.assign(an->nframes, -1);
    for (int p = 0; p < W.w.np; p++) W.last_use[W.w.cur[p]] = std::max(W.last_use[W.w.cur[p]], W.w.oth[p]);
}

// The jobs of every frame and the origins' places.  The two walks visit the
// same origins and lags up to their longest lag, so their pairs are matched:
// one job reads an origin for both.  An origin holds its place from its own
// frame to its last lag's; a place is taken over by the first origin after
// that (a frame that is both a last lag and an origin takes another place:
// both are in use in its launch).  Returns the number of places.
static int build_plan(ac4_ana *an) {
    const bool want0 = (an->obs & AC4_OBS_MSD) != 0,
               want1 = (an->obs & (AC4_OBS_OVERLAP | AC4_OBS_S4 | AC4_OBS_FS)) != 0;
    const int nf = an->nframes;
    std::vector<int> last(nf, -1);
    for (int o = 0; o < nf; o++) last[o] = std::max(an->W[0].last_use[o], an->W[1].last_use[o]);
    an->place.assign(nf, -1);
    an->resident.assign(nf, 0);
    an->ends.assign(nf, {});
    int places = 0;
    std::vector<int> avail;
    for (int f = 0; f < nf; f++) {
        if (last[f] >= 0) {
            if (avail.empty()) avail.push_back(places++);
            an->place[f] = avail.back();
            avail.pop_back();
            an->ends[last[f]].push_back(f);  // a lag frame comes after its origin
        }
        for (int o : an->ends[f]) avail.push_back(an->place[o]);
    }
    std::vector<std::vector<std::pair<int, Job>>> by(nf);  // (origin frame, job) per lag frame
    for (int w = 0; w < 2; w++) {
        if (!(w == 0 ? want0 : want1)) continue;
        const ac4_walk_t &k = an->W[w].w;
        for (int p = 0; p < k.np; p++) {
            auto &v = by[k.oth[p]];
            Job *j = nullptr;
            for (auto &e : v)
                if (e.first == k.cur[p] && e.second.slot == k.slot[p] && (w == 0 ? e.second.p0 : e.second.p1) < 0) {
                    j = &e.second;
                    break;
                }
            if (!j) {
                v.push_back({k.cur[p], Job{an->place[k.cur[p]], -1, -1, k.slot[p]}});
                j = &v.back().second;
            }
            (w == 0 ? j->p0 : j->p1) = p;
        }
    }
    an->jptr.assign(nf + 1, 0);
    for (int f = 0; f < nf; f++) {
        for (auto &e : by[f]) {
            an->jorg.push_back(e.first);
            an->jobs.push_back(e.second);
        }
        an->jptr[f + 1] = (int)an->jobs.size();
        an->max_jobs = std::max(an->max_jobs, (int)by[f].size());
    }
    return places;
}

static void build_slots(WalkInfo &W, int nslots) {
    W.nslots = nslots;
    W.used = 0;
    for (int p = 0; p < W.w.np; p++) W.used = std::max(W.used, W.w.slot[p] + 1);
    W.slot_ptr.assign(nslots + 1, 0);
    for (int p = 0; p < W.w.np; p++) W.slot_ptr[W.w.slot[p] + 1]++;
    for (int t = 0; t < nslots; t++) W.slot_ptr[t + 1] += W.slot_ptr[t];
    W.slot_pairs.assign(W.w.np, 0);
    std::vector<int> fill(W.slot_ptr.begin(), W.slot_ptr.end() - 1);
    for (int p = 0; p < W.w.np; p++) W.slot_pairs[fill[W.w.slot[p]]++] = p;  // walk order kept
}

// the permuted-vector columns of S4 and Fs, and the permutations of each vector
static int set_columns(ac4_ana *an, const std::vector<int> &dg) {
    std::vector<int> pv(3 * S4_NCOL, 0), pcol(AC4_NQ, 0);
    int col = 0;
    for (int q = 0; q < AC4_NQ; q++) {
        pcol[q] = col;
        for (int s = 0; s < dg[q]; s++, col++)
            perm_q(dg[q], s, an->vx[q], an->vy[q], an->vz[q], pv[3 * col], pv[3 * col + 1], pv[3 * col + 2]);
    }
    AC4_REQUIRE(col <= S4_NCOL, AC4_EARG, "S4: %d permuted vectors exceed %d columns", col, S4_NCOL);
    AC4_HIP(hipMemcpyToSymbol(HIP_SYMBOL(c_dg), dg.data(), sizeof(int) * AC4_NQ));
    AC4_HIP(hipMemcpyToSymbol(HIP_SYMBOL(c_pv), pv.data(), sizeof(int) * 3 * S4_NCOL));
    AC4_HIP(hipMemcpyToSymbol(HIP_SYMBOL(c_pcol), pcol.data(), sizeof(int) * AC4_NQ));
    return AC4_OK;
}

// S4 by origin: the per-origin pair lists and the sizes.  Returns the number of
// chunk partials of a pass.
static size_t s4_setup(ac4_ana *an) {
    const ac4_walk_t &w = an->W[1].w;
    an->s4_optr.assign(an->nframes + 1, 0);
    for (int p = 0; p < w.np; p++) an->s4_optr[w.cur[p] + 1]++;
    for (int o = 0; o < an->nframes; o++) an->s4_optr[o + 1] += an->s4_optr[o];
    an->s4_opairs.assign(std::max(w.np, 1), 0);
    std::vector<int> fill(an->s4_optr.begin(), an->s4_optr.end() - 1);
    for (int p = 0; p < w.np; p++) an->s4_opairs[fill[w.cur[p]]++] = p;
    an->s4_end.assign(an->nframes, {});
    for (int o = 0; o < an->nframes; o++)
        if (an->W[1].last_use[o] >= 0) an->s4_end[an->W[1].last_use[o]].push_back(o);
    an->s4_done.assign(an->nframes, 0);
    an->nwords = (an->n + 31) / 32;
    an->s4_wpw = std::max(1, (an->nwords + 4 * S4_SMALL_CHUNKS - 1) / (4 * S4_SMALL_CHUNKS));
    // chunks: at least 16 particles each, at most S4_CHUNKS of them; the tiles of a chunk as even as they go
    an->s4_ppb = std::max(16, 4 * ((an->n + 4 * S4_CHUNKS - 1) / (4 * S4_CHUNKS)));
    an->s4_nchunk = (an->n + an->s4_ppb - 1) / an->s4_ppb;
    const int nt = (an->s4_ppb + S4_P - 1) / S4_P;
    an->s4_tp = 4 * ((an->s4_ppb / 4 + nt - 1) / nt);
    size_t part = (size_t)an->s4_nchunk * S4_LAGS * 2 * AC4_NQ;
    if (an->n <= S4_SMALL) {
        an->s4_nchunk = (an->nwords + 4 * an->s4_wpw - 1) / (4 * an->s4_wpw);
        part = (size_t)an->s4_nchunk * S4_LAGS * 2 * S4_NCOL;
    }
    return part;
}

// The S4 sums of every pair of origin o, from its resident frame and the
// masks its lags left; passes of up to S4_LAGS lags.
static int s4_origin(ac4_ana *an, int o) {
    AC4_REQUIRE(an->resident[o], AC4_ESTATE, "S4: origin frame %d is not resident", o);
    const double *ox = an->org.at(an->place[o], 0), *oy = an->org.at(an->place[o], 1), *oz = an->org.at(an->place[o], 2);
    hipStream_t s = an->stream;
    const int b = an->s4_optr[o], e = an->s4_optr[o + 1];
    for (int p0 = b; p0 < e; p0 += S4_LAGS) {
        const int nl = std::min(S4_LAGS, e - p0);
        if (an->n <= S4_SMALL) {
            const int rt = (nl + 15) / 16;
            hipLaunchKernelGGL(rt == 1 ? k_s4_small<1> : k_s4_small<2>, dim3(an->s4_nchunk, S4_NCT), dim3(256), 0, s, ox, oy, oz,
                               an->n, an->nwords, an->d_s4mask, an->d_s4_opairs + p0, nl, an->s4_wpw, an->d_s4part);
            hipLaunchKernelGGL(k_s4_small_reduce, dim3(nl, (2 * AC4_NQ + 63) / 64), dim3(256), 0, s, an->d_s4part,
                               an->s4_nchunk, rt * 16, an->d_s4_opairs + p0, an->d_s4);
            AC4_HIP(hipGetLastError());
            continue;
        }
        // row tiles of 16 lags, the rest in tiles of 4; more than 12 are a tile of 16 as well
        const int nt16 = (nl + 3) / 16, nt4 = std::max(0, nl - 16 * nt16 + 3) / 4;
        const int *lags = an->d_s4_opairs + p0;
        auto *k = nt16 == 2 ? k_s4_origin<2, 0>
                  : nt16 == 1 ? (nt4 == 0 ? k_s4_origin<1, 0> : nt4 == 1 ? k_s4_origin<1, 1>
                                 : nt4 == 2 ? k_s4_origin<1, 2> : k_s4_origin<1, 3>)
                              : (nt4 == 1 ? k_s4_origin<0, 1> : nt4 == 2 ? k_s4_origin<0, 2> : k_s4_origin<0, 3>);
        hipLaunchKernelGGL(k, dim3(an->s4_nchunk), dim3(S4_T), 0, s, ox, oy, oz, an->n, an->nwords, an->d_s4mask, lags, nl,
                           an->s4_ppb, an->s4_tp, an->d_s4part);
        hipLaunchKernelGGL(k_s4_reduce, dim3(nl, (2 * AC4_NQ + 63) / 64), dim3(64 * S4_RW), 0, s, an->d_s4part,
                           an->s4_nchunk, nl, lags, an->d_s4);
        AC4_HIP(hipGetLastError());
    }
    an->s4_done[o] = 1;
    return AC4_OK;
}

extern "C" int ac4_ana_create(int n, double L, int nframes, const int *fidx, int gap, double factor, double a,
                              int obs, int type_flag, ac4_ana **out) {
    AC4_REQUIRE(n > 0 && L > 0 && nframes >= 2 && fidx && out && factor > 1.0 && a > 0, AC4_EARG,
                "ac4_ana_create: bad arguments");
    int ndev = 0;
    AC4_REQUIRE(hipGetDeviceCount(&ndev) == hipSuccess && ndev > 0, AC4_EHIP,
                "ac4_ana_create: no HIP device visible (libac4 has no CPU path)");
    for (int i = 1; i < nframes; i++)
        AC4_REQUIRE(fidx[i] > fidx[i - 1], AC4_EARG, "ac4_ana_create: frame index list not increasing at %d", i);
    ac4_ana *an = new ac4_ana();
    an->n = n; an->L = L; an->invL = 1.0 / L; an->nframes = nframes; an->factor = factor; an->a = a;
    an->param = a * a;  // overlap.c:5
    an->obs = obs; an->flag = type_flag;
    an->fidx.assign(fidx, fidx + nframes);
    an->gap = gap > 0 ? gap : ac4_origin_gap(fidx, nframes);
    if (an->gap <= 0) { delete an; return AC4_EARG; }
    build_walk_info(an, an->W[0], 0);
    build_walk_info(an, an->W[1], 1);
    // slot counts: msd_pos.c:29 / overlap.c:29 (+ bounds), S4/Fs use num_of_frames
    const double lf = log(an->factor);
    an->noi_msd = 10 + (int)(log((double)an->W[0].w.maximal_interval) / lf) + 10;
    an->noi_ov = 10 + (int)(log((double)an->W[1].w.maximal_interval) / lf);
    build_slots(an->W[0], std::max(an->noi_msd, an->W[0].w.max_slot + 1));
    build_slots(an->W[1], std::max(std::max(an->noi_ov, nframes), an->W[1].w.max_slot + 1));
    const int places = build_plan(an);
    an->vx.resize(AC4_NQ); an->vy.resize(AC4_NQ); an->vz.resize(AC4_NQ); an->qsq.resize(AC4_NQ + 8);
    ac4_getq(an->vx.data(), an->vy.data(), an->vz.data(), an->qsq.data());
    std::vector<int> dg(AC4_NQ);
    an->qval.assign(AC4_NQ, 0.0);
    for (int q = 0; q < AC4_NQ; q++) {
        dg[q] = ac4_degen(an->vx[q], an->vy[q], an->vz[q]);
        // Q[n] as left by S4Qt.c:135-208: first permutation for d<=3, last (z,y,x) for d=6
        int o0 = an->vx[q], o1 = an->vy[q], o2 = an->vz[q];
        if (dg[q] == 6) { o0 = an->vz[q]; o1 = an->vy[q]; o2 = an->vx[q]; }
        double qx = 2.0 * A_PI * an->invL * (double)o0, qy = 2.0 * A_PI * an->invL * (double)o1,
               qz = 2.0 * A_PI * an->invL * (double)o2;
        an->qval[q] = qx * qx + qy * qy + qz * qz;
    }
    int rc = AC4_OK;
    auto fail = [&](int e) { ac4_ana_destroy(an); return e; };
    if (hipGetDevice(&an->dev) != hipSuccess || hipStreamCreate(&an->stream) != hipSuccess) return fail(AC4_EHIP);
    if ((obs & (AC4_OBS_S4 | AC4_OBS_FS)) && (rc = set_columns(an, dg)) != AC4_OK) return fail(rc);
    // blocks of a frame row: one tile of the block's threads each up to 256 of them, then more tiles per block
    const int fb = obs & AC4_OBS_FS ? FS_T : ABLK;
    an->ppb = fb * ((n + 256 * fb - 1) / (256 * fb));
    an->nb = (n + an->ppb - 1) / an->ppb;
    an->fs_ppb = FS_P * ((n + FS_NBLK * FS_P - 1) / (FS_NBLK * FS_P));
    an->fs_nb = (n + an->fs_ppb - 1) / an->fs_ppb;
    an->max_jobs = std::max(an->max_jobs, 1);
    const size_t np0 = std::max(an->W[0].w.np, 1), np1 = std::max(an->W[1].w.np, 1);
    // one allocation, the zeroed arrays first: masks and sums start at zero, so
    // that a pair whose lag frame never arrives contributes nothing (1000
    // particles, all four observables, an allocation and a fill for each array:
    // 353 us to create and destroy, this 200)
    struct Array {
        void **p;
        size_t bytes;
    };
    std::vector<Array> arrays[2];  // zeroed, not zeroed
    auto get = [&](auto **p, size_t count, bool zero) {
        arrays[zero ? 0 : 1].push_back({(void **)p, (sizeof(**p) * count + 255) & ~(size_t)255});
    };
    an->org.n = (size_t)n;
    get(&an->d_jobs, std::max<size_t>(an->jobs.size(), 1), false);
    get(&an->org.f, (size_t)3 * n * std::max(places, 1), false);
    const int wgs = an->max_jobs * (an->fs_nb + an->nb) + an->nb;  // workgroups of a frame, at most
    get(&an->d_read, (size_t)(2 + wgs / READ_GRP) * READ_PAD, true);
    get(&an->cur, (size_t)3 * n, false);
    get(&an->cur_t, n, false);
    if (obs & AC4_OBS_MSD) { get(&an->d_msd, 3 * np0, true); get(&an->d_msdp, 3 * np0 * an->nb, true); }
    if (obs & AC4_OBS_OVERLAP) { get(&an->d_ov, np1, true); get(&an->d_ovp, np1 * an->nb, true); }
    if (obs & AC4_OBS_FS) {
        an->fs_wait = std::max(an->max_jobs, FS_WAIT);
        get(&an->d_fs, 2 * AC4_NQ * np1, true);
        get(&an->d_part, (size_t)an->fs_wait * an->fs_nb * AC4_NQ * 2, false);
    }
    if (obs & AC4_OBS_S4) {
        const size_t part = s4_setup(an);
        get(&an->d_s4, 2 * AC4_NQ * np1, true);
        get(&an->d_s4m, np1, true);
        get(&an->d_s4p, np1 * an->nb, true);
        get(&an->d_s4mask, np1 * an->nwords, true);
        get(&an->d_s4_opairs, np1, false);
        get(&an->d_s4part, part, false);
    }
    size_t bytes[2] = {0, 0};
    for (int k = 0; k < 2; k++)
        for (const Array &v : arrays[k]) bytes[k] += v.bytes;
    if (hipMalloc((void **)&an->mem, bytes[0] + bytes[1]) != hipSuccess) {
        ac4_set_error("ac4_ana_create: cannot allocate %zu bytes", bytes[0] + bytes[1]);
        return fail(AC4_EHIP);
    }
    char *at = an->mem;
    for (int k = 0; k < 2; k++)
        for (const Array &v : arrays[k]) {
            *v.p = at;
            at += v.bytes;
        }
    if (hipMemset(an->mem, 0, bytes[0]) != hipSuccess) return fail(AC4_EHIP);
    if (!an->jobs.empty() && hipMemcpy(an->d_jobs, an->jobs.data(), sizeof(Job) * an->jobs.size(),
                                       hipMemcpyHostToDevice) != hipSuccess) return fail(AC4_EHIP);
    if ((obs & AC4_OBS_S4) && hipMemcpy(an->d_s4_opairs, an->s4_opairs.data(), sizeof(int) * np1,
                                        hipMemcpyHostToDevice) != hipSuccess) return fail(AC4_EHIP);
    *out = an;
    return AC4_OK;
}

extern "C" int ac4_ana_destroy(ac4_ana *an) {
    if (!an) return AC4_OK;
    if (an->stream) (void)hipStreamSynchronize(an->stream);
    if (an->mem) (void)hipFree(an->mem);
    if (an->h_read) (void)hipHostFree(an->h_read);
    for (auto &W : an->W) ac4_walk_free(&W.w);
    if (an->stream) (void)hipStreamDestroy(an->stream);
    delete an;
    return AC4_OK;
}

extern "C" int ac4_ana_gap(const ac4_ana *an) { return an ? an->gap : AC4_EARG; }

static void reduce_fs(ac4_ana *an) {
    if (an->fs_j1 > an->fs_j0)
        hipLaunchKernelGGL(k_reduce_jobs, dim3(an->fs_j1 - an->fs_j0, (2 * AC4_NQ + 63) / 64), dim3(256), 0, an->stream,
                           an->d_jobs + an->fs_j0, an->fs_nb, 2 * AC4_NQ, an->d_part, an->d_fs);
    an->fs_j0 = an->fs_j1;
}

// Returns when the frame of the last launch has been read, i.e. its last
// workgroup has stored h_read; should the word not come (a failed launch), or
// take long, the stream's end, with its error, is waited for instead.
static int wait_read(ac4_ana *an) {
    const auto t0 = std::chrono::steady_clock::now();
    for (unsigned k = 1; __atomic_load_n(an->h_read, __ATOMIC_ACQUIRE) != an->seq; k++)
        if ((k & 255) == 0 && std::chrono::steady_clock::now() - t0 > std::chrono::milliseconds(2)) {
            AC4_HIP(hipStreamSynchronize(an->stream));
            break;
        }
    return AC4_OK;
}

// Runs every job of the frame whose arrays (device) are x, y, z, t; keep: the
// origin place the frame is copied to, or -1; wait: return when the arrays have
// been read.
static int process_frame(ac4_ana *an, int pos, const double *x, const double *y, const double *z, const int *t,
                         int keep, bool wait) {
    hipStream_t s = an->stream;
    const int j0 = an->jptr[pos], nj = an->jptr[pos + 1] - j0;
    const int nf = an->obs & (AC4_OBS_MSD | AC4_OBS_OVERLAP | AC4_OBS_S4) ? nj : 0;  // rows of pairs
    const int rows = nf + (keep >= 0 ? 1 : 0), nfs = an->obs & AC4_OBS_FS ? nj : 0;
    if (rows + nfs == 0) return AC4_OK;  // no pair ends here (so no origin's last lag either), nothing to keep
    const Frame F{x, y, z, t, an->n, an->flag, an->L, an->param, an->obs, an->org, keep, an->d_read,
                  wait ? an->h_read : nullptr, wait ? ++an->seq : 0u};
    const FrameOut O{an->ppb, an->nb, an->d_msdp, an->d_ovp, an->d_s4p, an->nwords, an->d_s4mask};
    if (rows > 0) an->stale = true;
    if (nfs > 0) {
        // the partials of the jobs [fs_j0, fs_j1) wait for their reduction
        if (j0 != an->fs_j1 || j0 + nj - an->fs_j0 > an->fs_wait) {
            reduce_fs(an);
            an->fs_j0 = j0;
        }
        an->fs_j1 = j0 + nj;
        hipLaunchKernelGGL(k_frame_fs, dim3(nfs * an->fs_nb + rows * an->nb), dim3(FS_T), 0, s, an->d_jobs + j0, nfs, nf,
                           an->fs_nb, an->fs_ppb, F, O,
                           an->d_part + (size_t)(j0 - an->fs_j0) * an->fs_nb * (AC4_NQ * 2));
    } else {
        hipLaunchKernelGGL(k_frame, dim3(an->nb, rows), dim3(ABLK), 0, s, an->d_jobs + j0, nf, F, O);
    }
    AC4_HIP(hipGetLastError());
    // origins whose last lag this frame was: their S4 sums, before another
    // origin takes their place
    if (an->obs & AC4_OBS_S4)
        for (int o : an->s4_end[pos]) TRY(s4_origin(an, o));
    return wait ? wait_read(an) : AC4_OK;
}

// p is memory of the device dev, which its kernels read where it is (another
// device's may not be mapped there, nor the host's): 0.06 us, so a push of
// device arrays takes 0.25 of its 12 us for asking
static bool on_device(const void *p, int dev) {
    hipPointerAttribute_t a = {};
    if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type == hipMemoryTypeDevice && a.device == dev;
    (void)hipGetLastError();
    return false;
}

// kind: hipMemcpyHostToDevice for host arrays, which are copied;
// hipMemcpyDefault for arrays the kernels read where they are, or of another
// device or the host, copied too
static int push_common(ac4_ana *an, int pos, const double *x, const double *y, const double *z, const int *t,
                       hipMemcpyKind kind) {
    AC4_REQUIRE(an && pos >= 0 && pos < an->nframes && x && y && z && t, AC4_EARG, "push_frame: bad arguments");
    AC4_REQUIRE(pos > an->last_pos, AC4_ESTATE, "push_frame: frame %d after %d (frames must increase)", pos,
                an->last_pos);
    AC4_REQUIRE(!an->finalized, AC4_ESTATE, "push_frame after finalize");
    for (int j = an->jptr[pos]; j < an->jptr[pos + 1]; j++)
        AC4_REQUIRE(an->resident[an->jorg[j]], AC4_ESTATE, "origin frame %d of pair %d was not pushed", an->jorg[j],
                    an->jobs[j].p0 >= 0 ? an->jobs[j].p0 : an->jobs[j].p1);
    hipStream_t s = an->stream;
    // origins whose last lag was left out: the S4 sums of the lags that came,
    // before this frame takes a place
    if (an->obs & AC4_OBS_S4)
        for (int f = an->last_pos + 1; f < pos; f++)
            for (int o : an->s4_end[f])
                if (an->resident[o] && !an->s4_done[o]) TRY(s4_origin(an, o));
    const size_t n = an->n, b = sizeof(double) * n;
    int keep = an->place[pos];
    const bool copy = kind != hipMemcpyDefault || !on_device(x, an->dev) || !on_device(y, an->dev) ||
                      !on_device(z, an->dev) || !on_device(t, an->dev);
    if (copy) {  // an origin frame straight to its place
        double *dx = an->cur, *dy = dx + n, *dz = dy + n;
        if (keep >= 0) { dx = an->org.at(keep, 0); dy = an->org.at(keep, 1); dz = an->org.at(keep, 2); }
        AC4_HIP(hipMemcpyAsync(dx, x, b, kind, s));
        AC4_HIP(hipMemcpyAsync(dy, y, b, kind, s));
        AC4_HIP(hipMemcpyAsync(dz, z, b, kind, s));
        AC4_HIP(hipMemcpyAsync(an->cur_t, t, sizeof(int) * n, kind, s));
        x = dx; y = dy; z = dz; t = an->cur_t;
        keep = -1;
    }
    if (!copy && !an->h_read) {  // 30 us; host pushes do without it
        AC4_HIP(hipHostMalloc((void **)&an->h_read, 64, hipHostMallocDefault));
        *an->h_read = 0;
    }
    an->resident[pos] = an->place[pos] >= 0;
    TRY(process_frame(an, pos, x, y, z, t, keep, !copy));  // the caller may reuse its arrays
    if (copy) AC4_HIP(hipStreamSynchronize(s));
    // origins no pair needs any more (their places may be taken from now on)
    for (int f = an->last_pos + 1; f <= pos; f++)
        for (int o : an->ends[f]) an->resident[o] = 0;
    an->last_pos = pos;
    return AC4_OK;
}

extern "C" int ac4_ana_push_frame(ac4_ana *an, int pos, const double *x, const double *y, const double *z,
                                  const int *type) {
    return push_common(an, pos, x, y, z, type, hipMemcpyHostToDevice);
}

extern "C" int ac4_ana_push_frame_device(ac4_ana *an, int pos, const double *x, const double *y, const double *z,
                                         const int *type) {
    return push_common(an, pos, x, y, z, type, hipMemcpyDefault);
}

extern "C" int ac4_md_device_xu(ac4_md *md, int r, const double **xu, const double **yu, const double **zu,
                                const int **type, int *n);
extern "C" int ac4_ana_push_md(ac4_ana *an, int pos, ac4_md *md, int r) {
    const double *x, *y, *z;
    const int *t;
    int n = 0;
    TRY(ac4_md_device_xu(md, r, &x, &y, &z, &t, &n));
    AC4_REQUIRE(an && n == an->n, AC4_EARG, "push_md: replica has %d particles, analysis expects %d", n,
                an ? an->n : -1);
    return push_common(an, pos, x, y, z, t, hipMemcpyDefault);
}

// The slots' sums of a walk's pair values, for the slots that have pairs
// (W.used; the trajectory's frame count is the number of slots, of which a lag
// ladder fills a few dozen): 1220 slots formed, copied and split four times
// took 3.8 ms of 1000 particles' whole 20, this 0.4.
static int slots_run(ac4_ana *an, int w, const double *dvals, int nv, int mode, double div, std::vector<double> &sum,
                     std::vector<double> *sq) {
    const WalkInfo &W = an->W[w];
    const size_t m = (size_t)W.used * nv, nt = (size_t)W.used + 1 + W.w.np, tab = (nt + 1) / 2;  // tables in doubles
    std::vector<int> t(W.slot_ptr.begin(), W.slot_ptr.begin() + W.used + 1);
    t.insert(t.end(), W.slot_pairs.begin(), W.slot_pairs.end());
    std::vector<double> out(2 * m, 0.0);
    sum.assign(m, 0.0);
    if (sq) sq->assign(m, 0.0);
    if (m == 0) return AC4_OK;
    double *d = nullptr;
    AC4_HIP(hipMalloc(&d, sizeof(double) * (tab + 2 * m)));
    const int *dt = (const int *)d;
    double *dsum = d + tab;
    hipError_t e = hipMemcpyAsync(d, t.data(), sizeof(int) * nt, hipMemcpyHostToDevice, an->stream);
    hipLaunchKernelGGL(k_slots, dim3(W.used), dim3(256), 0, an->stream, dvals, nv, dt, dt + W.used + 1, W.used, mode, div,
                       dsum, dsum + m);
    if (e == hipSuccess) e = hipGetLastError();
    if (e == hipSuccess)
        e = hipMemcpyAsync(out.data(), dsum, sizeof(double) * (sq ? 2 : 1) * m, hipMemcpyDeviceToHost, an->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(an->stream);
    (void)hipFree(d);
    AC4_HIP(e);
    sum.assign(out.begin(), out.begin() + m);
    if (sq) sq->assign(out.begin() + m, out.end());
    return AC4_OK;
}

static void split_phase(const std::vector<double> &in, int ns, std::vector<double> &c, std::vector<double> &s) {
    c.assign((size_t)ns * AC4_NQ, 0.0);
    s.assign((size_t)ns * AC4_NQ, 0.0);
    for (int t = 0; t < ns; t++)
        for (int q = 0; q < AC4_NQ; q++) {
            c[(size_t)t * AC4_NQ + q] = in[(size_t)t * 2 * AC4_NQ + q];
            s[(size_t)t * AC4_NQ + q] = in[(size_t)t * 2 * AC4_NQ + AC4_NQ + q];
        }
}

// Every pair's MSD sums and overlap counts from its blocks' values
static int sum_blocks(ac4_ana *an) {
    reduce_fs(an);
    AC4_HIP(hipGetLastError());
    if (!an->stale) return AC4_OK;
    const int np0 = an->W[0].w.np, np1 = an->W[1].w.np;
    if ((an->obs & AC4_OBS_MSD) && np0 > 0)
        hipLaunchKernelGGL(k_msd_pairs, dim3(np0), dim3(ABLK), 0, an->stream, an->d_msdp, an->nb, an->d_msd);
    if ((an->obs & AC4_OBS_OVERLAP) && np1 > 0)
        hipLaunchKernelGGL(k_counts, dim3(np1), dim3(64), 0, an->stream, an->d_ovp, an->nb, an->d_ov);
    if ((an->obs & AC4_OBS_S4) && np1 > 0)
        hipLaunchKernelGGL(k_counts, dim3(np1), dim3(64), 0, an->stream, an->d_s4p, an->nb, an->d_s4m);
    AC4_HIP(hipGetLastError());
    an->stale = false;
    return AC4_OK;
}

extern "C" int ac4_ana_finalize(ac4_ana *an) {
    AC4_REQUIRE(an, AC4_EARG, "NULL handle");
    if (an->finalized) return AC4_OK;
    if (an->obs & AC4_OBS_S4)  // origins whose last lag frame is past the last one pushed
        for (int o = 0; o < an->nframes; o++)
            if (!an->s4_done[o] && an->resident[o] && an->s4_optr[o + 1] > an->s4_optr[o]) TRY(s4_origin(an, o));
    TRY(sum_blocks(an));
    AC4_HIP(hipStreamSynchronize(an->stream));
    const double tot = an->flag == 1 ? 0.8 * an->n : (double)an->n;  // msd_pos.c:26-27
    for (int w = 0; w < 2; w++) {  // counters and delta_t (msd_pos.c:90-92)
        WalkInfo &W = an->W[w];
        std::vector<int> &cn = w == 0 ? an->cnt0 : an->cnt1;
        std::vector<double> &dt = w == 0 ? an->dt0 : an->dt1;
        cn.assign(W.nslots, 0);
        dt.assign(W.nslots, 0.0);
        for (int p = 0; p < W.w.np; p++) {
            cn[W.w.slot[p]]++;
            dt[W.w.slot[p]] = 0.005 * (double)(an->fidx[W.w.oth[p]] - an->fidx[W.w.cur[p]]);
        }
    }
    if (an->obs & AC4_OBS_MSD) {
        std::vector<double> s;
        TRY(slots_run(an, 0, an->d_msd, 3, 0, tot, s, nullptr));
        const int ns = an->W[0].nslots;
        an->m0.assign(ns, 0); an->m1.assign(ns, 0); an->m2.assign(ns, 0);
        for (int t = 0; t < an->W[0].used; t++) { an->m0[t] = s[3 * t]; an->m1[t] = s[3 * t + 1]; an->m2[t] = s[3 * t + 2]; }
    }
    const int used = an->W[1].used;  // S4 and Fs are kept for these slots, zero beyond (get_phase)
    if (an->obs & AC4_OBS_OVERLAP) {
        TRY(slots_run(an, 1, an->d_ov, 1, 1, tot, an->c, &an->x4));
        an->c.resize(an->W[1].nslots, 0.0);
        an->x4.resize(an->W[1].nslots, 0.0);
    }
    if (an->obs & AC4_OBS_S4) {
        std::vector<double> s, s2;
        TRY(slots_run(an, 1, an->d_s4, 2 * AC4_NQ, 1, 0.0, s, &s2));
        split_phase(s, used, an->s4c, an->s4s);
        split_phase(s2, used, an->s4c2, an->s4s2);
    }
    if (an->obs & AC4_OBS_FS) {
        std::vector<double> s, s2;
        TRY(slots_run(an, 1, an->d_fs, 2 * AC4_NQ, 1, 0.0, s, &s2));
        split_phase(s, used, an->fsc, an->fss);
        split_phase(s2, used, an->fsc2, an->fss2);
    }
    an->finalized = true;
    return AC4_OK;
}

extern "C" int ac4_ana_nslots(const ac4_ana *an, int obs) {
    if (!an) return AC4_EARG;
    return obs == AC4_OBS_MSD ? an->W[0].nslots : an->W[1].nslots;
}

extern "C" int ac4_ana_get_msd(ac4_ana *an, double *m0, double *m1, double *m2, int *counters, double *delta_t,
                               int *num_intervals) {
    AC4_REQUIRE(an && an->finalized && (an->obs & AC4_OBS_MSD), AC4_ESTATE, "get_msd: not finalized / not requested");
    const int ns = an->W[0].nslots;
    for (int t = 0; t < ns; t++) {
        if (m0) m0[t] = an->m0[t];
        if (m1) m1[t] = an->m1[t];
        if (m2) m2[t] = an->m2[t];
        if (counters) counters[t] = an->cnt0[t];
        if (delta_t) delta_t[t] = an->dt0[t];
    }
    if (num_intervals) *num_intervals = an->noi_msd;
    return AC4_OK;
}

extern "C" int ac4_ana_get_overlap(ac4_ana *an, double *c, double *x4, int *counters, double *delta_t,
                                   int *num_intervals) {
    AC4_REQUIRE(an && an->finalized && (an->obs & AC4_OBS_OVERLAP), AC4_ESTATE,
                "get_overlap: not finalized / not requested");
    const int ns = an->W[1].nslots;
    for (int t = 0; t < ns; t++) {
        if (c) c[t] = an->c[t];
        if (x4) x4[t] = an->x4[t];
        if (counters) counters[t] = an->cnt1[t];
        if (delta_t) delta_t[t] = an->dt1[t];
    }
    if (num_intervals) *num_intervals = an->noi_ov;
    return AC4_OK;
}

extern "C" int ac4_ana_get_phase(ac4_ana *an, int obs, double *cs, double *ss, double *cs2, double *ss2,
                                 int *counters, double *delta_t, double *qval) {
    AC4_REQUIRE(an && an->finalized && (obs == AC4_OBS_S4 || obs == AC4_OBS_FS) && (an->obs & obs), AC4_ESTATE,
                "get_phase: not finalized / not requested");
    const bool s4 = obs == AC4_OBS_S4;
    const size_t ns = an->W[1].nslots, m = (size_t)an->W[1].used * AC4_NQ;
    const std::vector<double> &C = s4 ? an->s4c : an->fsc, &S = s4 ? an->s4s : an->fss, &C2 = s4 ? an->s4c2 : an->fsc2,
                              &S2 = s4 ? an->s4s2 : an->fss2;
    const auto put = [&](double *d, const std::vector<double> &v) {
        if (!d) return;
        std::copy(v.begin(), v.end(), d);
        std::fill(d + m, d + ns * AC4_NQ, 0.0);
    };
    put(cs, C);
    put(ss, S);
    put(cs2, C2);
    put(ss2, S2);
    if (counters) memcpy(counters, an->cnt1.data(), sizeof(int) * ns);
    if (delta_t) memcpy(delta_t, an->dt1.data(), sizeof(double) * ns);
    if (qval) memcpy(qval, an->qval.data(), sizeof(double) * AC4_NQ);
    return AC4_OK;
}

extern "C" int ac4_ana_npairs(const ac4_ana *an, int obs) {
    if (!an) return AC4_EARG;
    return obs == AC4_OBS_MSD ? an->W[0].w.np : an->W[1].w.np;
}

extern "C" int ac4_ana_get_pairs(ac4_ana *an, int obs, double *vals, int *ivals) {
    AC4_REQUIRE(an && (an->obs & obs), AC4_ESTATE, "get_pairs: observable not requested");
    TRY(sum_blocks(an));
    AC4_HIP(hipStreamSynchronize(an->stream));
    const size_t np = obs == AC4_OBS_MSD ? an->W[0].w.np : an->W[1].w.np;
    if (np == 0) return AC4_OK;
    if (obs == AC4_OBS_MSD && vals) AC4_HIP(hipMemcpy(vals, an->d_msd, sizeof(double) * 3 * np, hipMemcpyDeviceToHost));
    const double *cnt = obs == AC4_OBS_OVERLAP ? an->d_ov : (obs == AC4_OBS_S4 ? an->d_s4m : nullptr);
    if (cnt && ivals) {
        std::vector<double> v(np);
        AC4_HIP(hipMemcpy(v.data(), cnt, sizeof(double) * np, hipMemcpyDeviceToHost));
        for (size_t p = 0; p < np; p++) ivals[p] = (int)v[p];
    }
    if (obs == AC4_OBS_S4 && vals)
        AC4_HIP(hipMemcpy(vals, an->d_s4, sizeof(double) * 2 * AC4_NQ * np, hipMemcpyDeviceToHost));
    if (obs == AC4_OBS_FS && vals) AC4_HIP(hipMemcpy(vals, an->d_fs, sizeof(double) * 2 * AC4_NQ * np, hipMemcpyDeviceToHost));
    return AC4_OK;
}

extern "C" int ac4_ana_write(ac4_ana *an, const char *sub_dir) {
    AC4_REQUIRE(an && sub_dir, AC4_EARG, "write: bad arguments");
    if (!an->finalized) TRY(ac4_ana_finalize(an));
    char path[2048];
    const double tot = an->flag == 1 ? 0.8 * an->n : (double)an->n;
    if (an->obs & AC4_OBS_MSD) {
        snprintf(path, sizeof path, "%s/%s", sub_dir, an->flag == 1 ? "msdA.dat" : "msd.dat");
        TRY(ac4_write_msd(path, an->noi_msd, an->m0.data(), an->m1.data(), an->m2.data(), an->cnt0.data(),
                          an->dt0.data()));
    }
    if (an->obs & AC4_OBS_OVERLAP) {
        snprintf(path, sizeof path, an->flag == 1 ? "%s/relaxAA_a_%.2lf.dat" : "%s/relax_a_%.2lf.dat", sub_dir, an->a);
        TRY(ac4_write_overlap(path, an->noi_ov, an->c.data(), an->x4.data(), an->cnt1.data(), an->dt1.data()));
    }
    // S4Qt.c/Fsqt.c loop over num_of_frames slots
    const int ns = std::min(an->W[1].nslots, an->nframes);
    if (an->obs & AC4_OBS_S4) {
        snprintf(path, sizeof path, "%s/S4qt_a_%.2lf.dat", sub_dir, an->a);
        TRY(ac4_write_phase(path, 1, an->n, tot, ns, an->vx.data(), an->vy.data(), an->vz.data(), an->s4c.data(),
                            an->s4s.data(), an->s4c2.data(), an->s4s2.data(), an->cnt1.data(), an->dt1.data(),
                            an->qval.data()));
    }
    if (an->obs & AC4_OBS_FS) {
        snprintf(path, sizeof path, an->flag == 1 ? "%s/FsqtAA_a_%.2lf.dat" : "%s/Fsqt_a_%.2lf.dat", sub_dir, an->a);
        TRY(ac4_write_phase(path, 0, an->n, tot, ns, an->vx.data(), an->vy.data(), an->vz.data(), an->fsc.data(),
                            an->fss.data(), an->fsc2.data(), an->fss2.data(), an->cnt1.data(), an->dt1.data(),
                            an->qval.data()));
    }
    return AC4_OK;
}

extern "C" int ac4_sincos_turns_host(const double *f, int n, double *s, double *c) {
    AC4_REQUIRE(f && s && c && n >= 0, AC4_EARG, "sincos_turns: bad arguments");
    for (int i = 0; i < n; i++) ac4_sincos_turns(f[i], &s[i], &c[i]);
    return AC4_OK;
}

extern "C" int ac4_device_count(void) {
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) return 0;
    return n;
}
