// ac4_frames.hip -- a device-resident trajectory of one replica and the
// four-point structure factor S4(q, t) on |q| shells with seeded random
// directions, weighted by the per-particle overlap.
//
// No reference counterpart for the store: the reference writes every frame
// to data_coor.out and rereads it (Analysis/read_all_data.c:61-91).  Here the
// frames stay in HBM (x_u of 10^6 particles is 24 MB a frame, 500 frames
// 12 GB), so an analysis can pair any origin with any lag after the run.
//
// S4 on shells generalises Analysis/S4Qt.c (which uses the 162 lattice
// vectors of GetQ): for |q_k| = q0 + k*dq, k < nshell, and unit directions
// n_d, d < ndir, drawn from a seed,
//   C_{p,k,d} = sum_i w_i cos(|q_k| L n_d.s_i),  S likewise with sin,
// over particles i, with s_i the origin position of pair p wrapped into
// [0,1) and w_i = 1 when particle i overlaps between the origin and the lag
// frame of the pair (Analysis/overlap.c:61-84 arithmetic: unwrapped
// difference, one minimum-image correction, L*L*((dx*dx+dy*dy)+dz*dz) < a*a).
// From the C and S of all pairs (origins at one lag):
//   s4_ref[k] = ndir * [Var_p(Cbar) + Var_p(Sbar)] / N, Cbar = mean_d C
//               (the structure of S4Qt.c:133-267: the directions play the
//               role of the permutations, ndir the degeneracy),
//   s4_dir[k] = mean_d [Var_p(C) + Var_p(S)] / N  (the direction average of
//               (<|W(q)|^2> - |<W(q)>|^2)/N),
// with population variances over the pairs.
//
// Kernel (k_fr_phase): a workgroup stages the overlapping particles of a tile
// in LDS; each thread owns one direction and NG runs of SHELL_RUN = 27
// consecutive shells.  A run is taken about its middle shell q_c: with
// A = exp(i q_c x) and B_m = exp(i m dq x), the products cA cB, sA sB, sA cB
// and cA sB summed over the particles give both shells q_c +- m dq, so a shell
// costs two fused multiply-adds where a walk from shell to shell takes six
// operations, and the chain of B_m is shared by the thread's runs.  All in
// FP64.  The partial sums of the workgroups are added in a fixed order, so
// results are deterministic.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>
#include <string.h>
#include <algorithm>
#include <vector>
#include "ac4_internal.h"

extern "C" int ac4_md_device_xu(ac4_md *md, int r, const double **xu, const double **yu, const double **zu,
                                const int **type, int *n);

#define TRY(e) do { int rc_ = (e); if (rc_ != AC4_OK) return rc_; } while (0)
#define FR_THREADS 256
#define FR_ROLES 256   // most (direction, run) pairs of a call
#define SHELL_RUN 27   // shells of a run: the middle one and SHELL_H on either side
#define SHELL_H 13
#define PH_THREADS 512 // threads of k_fr_phase and particles of its tile
#define FOLD_SEQ 8     // teams folded one after the other
#define FR_BLOCKS 256  // its workgroups of one launch: one per CU
#define FR_PAIRS 32    // pairs of one launch, at most

struct ac4_frames {
    int n = 0, cap = 0, count = 0;
    double L = 0.0;
    double *x = nullptr, *y = nullptr, *z = nullptr;  // [cap][n], box-scaled x_u, reference order
    std::vector<long long> step;
    hipStream_t s = nullptr;
    double *part = nullptr;  // [FR_BLOCKS][ndir][nshell][2]
    size_t part_n = 0;
    double *dirs = nullptr;
    int dirs_n = 0;
    unsigned int *cnt = nullptr;
};

// Analysis/overlap.c:67-78: one minimum-image correction of an unwrapped difference
__device__ __forceinline__ double fr_minimg(double d) {
    if (d >= 0.5)
        d -= 1.0;
    else if (d < -0.5)
        d += 1.0;
    return d;
}

__global__ void __launch_bounds__(FR_THREADS) k_fr_overlap(const double *__restrict__ x, const double *__restrict__ y,
                                                           const double *__restrict__ z, int n, size_t fo, size_t ft,
                                                           double L, double a2, unsigned int *cnt) {
    const int i = blockIdx.x * FR_THREADS + threadIdx.x;
    int hit = 0;
    if (i < n) {
        double dx = x[ft + i] - x[fo + i], dy = y[ft + i] - y[fo + i], dz = z[ft + i] - z[fo + i];
        dz = fr_minimg(dz);
        dy = fr_minimg(dy);
        dx = fr_minimg(dx);
        hit = L * L * (dx * dx + dy * dy + dz * dz) < a2;
    }
    const int w = ac4_wave_sum_i(hit);
    if ((threadIdx.x & 63) == 0 && w) atomicAdd(cnt, (unsigned int)w);
}

// frame offsets (in particles) of the pairs of one launch
struct FrPairs {
    size_t o[FR_PAIRS], l[FR_PAIRS];
};

// q p in turns, less the whole turns nearest it: the product is not rounded
// before they are taken off
__device__ __forceinline__ double fr_turns(double q, double p) { return fma(q, p, -rint(q * p)); }

// Phase sums of pair blockIdx.x / bpp over the particles of block
// blockIdx.x % bpp: part[blockIdx.x][ndir][nshell][2].  Thread t is role
// t % T of team t / T, T = ndir * ceil(ngroup / NG) roles; the S = PH_THREADS
// / T teams take every S-th particle of the tile, and their sums are added in
// team order at the end.
// L2 = L * L; f0, fd: the phases of |q| = q0 and of one shell step per unit of
// n.s, in turns.  The phase of a middle shell is formed from the two reduced
// phases, so that the step's rounding, multiplied by its number there and by
// m in B_m, cancels in the shells of small |q|, where the particles' terms
// add up coherently.
// Bound by FP64 issue: per particle and role 1 + NG sincos (34 instructions
// each), 13 products of the B chain (4 each) and 54 sums and products per run
// (4 per pair of shells).  Two runs per thread (NG = 2, 255 registers, two
// waves per SIMD) share the chain; an odd number of runs below five leaves
// half of the last pair of runs idle, which costs more than the sharing
// gives, and takes NG = 1.  300000 particles, 64 directions x 108 shells, per
// pair: walking from shell to shell with the library's sincos 1220 us, this
// 411 us.
template <int NG>
__global__ void __launch_bounds__(PH_THREADS) k_fr_phase(const double *__restrict__ x, const double *__restrict__ y,
                                                         const double *__restrict__ z, int n, FrPairs pr, int bpp,
                                                         double L2, double a2, double f0, double fd, int nshell,
                                                         int ndir, int ngroup, const double *__restrict__ dirs,
                                                         double *part) {
    __shared__ double s_x[PH_THREADS], s_y[PH_THREADS], s_z[PH_THREADS];
    __shared__ int s_n[PH_THREADS / 64 + 1];
    __shared__ double s_f[PH_THREADS * 4];  // the teams' sums, four values a round
    const int t = threadIdx.x, wv = __builtin_amdgcn_readfirstlane(t >> 6);
    const int nrole = (ngroup + NG - 1) / NG, T = ndir * nrole, S = PH_THREADS / T;
    const int team = t / T;
    const bool active = team < S;
    const int pi = blockIdx.x / bpp, pb = blockIdx.x - pi * bpp;
    const size_t fo = pr.o[pi], ft = pr.l[pi];
    // direction and first middle shell of every role, read from LDS for each
    // particle (volatile): the registers are the sums'
    __shared__ double s_role[4][FR_ROLES];
    if (team == 0) {
        const int d = t / nrole, g0 = (t - d * nrole) * NG;
        for (int q = 0; q < 3; q++) s_role[q][t] = dirs[3 * d + q];
        s_role[3][t] = (double)(g0 * SHELL_RUN + SHELL_H);
    }
    const volatile double *vr = &s_role[0][t - team * T];
    double cc[NG][SHELL_H + 1], ss[NG][SHELL_H + 1], sc[NG][SHELL_H + 1], cs[NG][SHELL_H + 1];  // [0]: A alone
#pragma unroll
    for (int u = 0; u < NG; u++)
#pragma unroll
        for (int m = 0; m <= SHELL_H; m++) cc[u][m] = ss[u][m] = sc[u][m] = cs[u][m] = 0.0;
    const int per = (n + bpp - 1) / bpp;
    const int i0 = min(n, pb * per), i1 = min(n, i0 + per);
    for (int tb = i0; tb < i1; tb += PH_THREADS) {
        const int i = tb + t;
        double ox = 0.0, oy = 0.0, oz = 0.0;
        bool hit = false;
        if (i < i1) {
            ox = x[fo + i]; oy = y[fo + i]; oz = z[fo + i];
            double dx = x[ft + i] - ox, dy = y[ft + i] - oy, dz = z[ft + i] - oz;
            dz = fr_minimg(dz);
            dy = fr_minimg(dy);
            dx = fr_minimg(dx);
            hit = L2 * (dx * dx + dy * dy + dz * dz) < a2;
        }
        // the overlapping particles of the tile, in order
        const unsigned long long hm = __ballot(hit);
        __syncthreads();  // the previous tile is done with
        s_n[wv] = __popcll(hm);  // every lane the same value
        __syncthreads();
        int k = (int)__builtin_amdgcn_mbcnt_hi((unsigned)(hm >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)hm, 0u)), m = 0;
        for (int w = 0; w < PH_THREADS / 64; w++) {
            const int c = s_n[w];
            if (w < wv) k += c;
            m += c;
        }
        if (hit) {
            s_x[k] = ox - floor(ox);
            s_y[k] = oy - floor(oy);
            s_z[k] = oz - floor(oz);
        }
        __syncthreads();
        if (!active) continue;
        for (int j = team; j < m; j += S) {
            const double p = fma(vr[2 * FR_ROLES], s_z[j], fma(vr[FR_ROLES], s_y[j], vr[0] * s_x[j]));
            double c1, s1, ca[NG], sa[NG];
            const double r0 = fr_turns(f0, p), r1 = fr_turns(fd, p);
            ac4_sincos_turns(r1, &s1, &c1);
#pragma unroll
            for (int u = 0; u < NG; u++) {
                const double f = fma(vr[3 * FR_ROLES] + (double)(u * SHELL_RUN), r1, r0);
                ac4_sincos_turns(f - rint(f), &sa[u], &ca[u]);
                cc[u][0] += ca[u];
                ss[u][0] += sa[u];
            }
            double cb = c1, sb = s1;
#pragma unroll
            for (int h = 1; h <= SHELL_H; h++) {
#pragma unroll
                for (int u = 0; u < NG; u++) {
                    cc[u][h] = fma(ca[u], cb, cc[u][h]);
                    ss[u][h] = fma(sa[u], sb, ss[u][h]);
                    sc[u][h] = fma(sa[u], cb, sc[u][h]);
                    cs[u][h] = fma(ca[u], sb, cs[u][h]);
                }
                if (h < SHELL_H) {
                    const double cn = fma(cb, c1, -(sb * s1));
                    sb = fma(sb, c1, cb * s1);
                    cb = cn;
                }
            }
        }
    }
    // the shells' sums from the products, folded over the teams: in team order
    // up to FOLD_SEQ teams, else in two rounds, the first F teams every F-th
    // one's, then team 0 theirs (one shell and direction, 512 teams: in team
    // order the fold alone took 300 us)
    double *o = part + (size_t)blockIdx.x * ndir * nshell * 2;
    int te = t;
    asm volatile("" : "+v"(te));  // the role again, not kept in registers over the loop
    const int role = te % T, d = role / nrole, g0 = (role - d * nrole) * NG, tm = te / T;
    int F = 1;
    if (S > FOLD_SEQ)
        while (F * F < S) F++;
#pragma unroll
    for (int u = 0; u < NG; u++) {
        const int kc = (g0 + u) * SHELL_RUN + SHELL_H;
#pragma unroll
        for (int h = 0; h <= SHELL_H; h++) {
            if (u * SHELL_RUN + SHELL_H - h >= nshell) continue;  // no role has either shell
            // shells kc + h and kc - h: {C+, S+, C-, S-} (h = 0: the first two)
            double v[4];
            if (h == 0) {
                v[0] = cc[u][0]; v[1] = ss[u][0]; v[2] = v[3] = 0.0;
            } else {
                v[0] = cc[u][h] - ss[u][h];
                v[1] = sc[u][h] + cs[u][h];
                v[2] = cc[u][h] + ss[u][h];
                v[3] = sc[u][h] - cs[u][h];
            }
            if (S > 1) {  // uniform over the workgroup
                __syncthreads();
#pragma unroll
                for (int q = 0; q < 4; q++) s_f[q * PH_THREADS + t] = v[q];
                __syncthreads();
                if (F > 1) {
                    if (tm < F)
                        for (int w = tm + F; w < S; w += F)
#pragma unroll
                            for (int q = 0; q < 4; q++) v[q] += s_f[q * PH_THREADS + w * T + role];
                    __syncthreads();
#pragma unroll
                    for (int q = 0; q < 4; q++) s_f[q * PH_THREADS + t] = v[q];
                    __syncthreads();
                }
                if (tm == 0)
                    for (int w = 1; w < (F > 1 ? F : S); w++)
#pragma unroll
                        for (int q = 0; q < 4; q++) v[q] += s_f[q * PH_THREADS + w * T + role];
            }
            if (tm == 0) {
                const int kp = kc + h, km = kc - h;
                if (kp < nshell) {
                    o[2 * ((size_t)d * nshell + kp)] = v[0];
                    o[2 * ((size_t)d * nshell + kp) + 1] = v[1];
                }
                if (h > 0 && km < nshell) {
                    o[2 * ((size_t)d * nshell + km)] = v[2];
                    o[2 * ((size_t)d * nshell + km) + 1] = v[3];
                }
            }
        }
    }
}

// part[p*bpp][e] = sum over the blocks b of pair p = blockIdx.y of
// part[p*bpp + b][e]: 64 values per workgroup of 256 threads, wave w the
// blocks w, w+4, ... with eight loads in flight, the waves added in order
__global__ void __launch_bounds__(256) k_fr_reduce(double *part, int bpp, int ne) {
    __shared__ double s_w[4][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, e = blockIdx.x * 64 + lane;
    double *p = part + (size_t)blockIdx.y * bpp * ne;
    double a = 0.0;
    if (e < ne) {
        int b = w;
        for (; b + 28 < bpp; b += 32) {
            double v[8];
#pragma unroll
            for (int u = 0; u < 8; u++) v[u] = p[(size_t)(b + 4 * u) * ne + e];
#pragma unroll
            for (int u = 0; u < 8; u++) a += v[u];
        }
        for (; b < bpp; b += 4) a += p[(size_t)b * ne + e];
    }
    s_w[w][lane] = a;
    __syncthreads();
    if (w == 0 && e < ne) p[e] = ((s_w[0][lane] + s_w[1][lane]) + s_w[2][lane]) + s_w[3][lane];
}

extern "C" int ac4_frames_create(int n, double L, int cap, ac4_frames **out) {
    AC4_REQUIRE(n > 0 && L > 0 && cap > 0 && out, AC4_EARG, "ac4_frames_create: bad arguments");
    int ndev = 0;
    AC4_REQUIRE(hipGetDeviceCount(&ndev) == hipSuccess && ndev > 0, AC4_EHIP,
                "ac4_frames_create: no HIP device visible (libac4 has no CPU path)");
    ac4_frames *f = new ac4_frames();
    f->n = n;
    f->L = L;
    f->cap = cap;
    const size_t bytes = sizeof(double) * (size_t)n * cap;
    if (hipMalloc(&f->x, bytes) != hipSuccess || hipMalloc(&f->y, bytes) != hipSuccess ||
        hipMalloc(&f->z, bytes) != hipSuccess || hipMalloc(&f->cnt, sizeof(unsigned int)) != hipSuccess ||
        hipStreamCreate(&f->s) != hipSuccess) {
        ac4_frames_destroy(f);
        ac4_set_error("ac4_frames_create: cannot allocate %zu bytes of frames", 3 * bytes);
        return AC4_EHIP;
    }
    *out = f;
    return AC4_OK;
}

extern "C" int ac4_frames_destroy(ac4_frames *f) {
    if (!f) return AC4_OK;
    if (f->s) (void)hipStreamSynchronize(f->s);
    void *p[] = {f->x, f->y, f->z, f->part, f->dirs, f->cnt};
    for (void *q : p)
        if (q) (void)hipFree(q);
    if (f->s) (void)hipStreamDestroy(f->s);
    delete f;
    return AC4_OK;
}

extern "C" int ac4_frames_count(const ac4_frames *f) { return f ? f->count : 0; }

int ac4_frames_steps(const ac4_frames_view &v, std::vector<int> &fidx) {
    fidx.resize(v.count);
    for (int k = 0; k < v.count; k++) {
        AC4_REQUIRE(v.step[k] >= 0 && v.step[k] < 2147483647LL, AC4_EARG,
                    "frame step %lld does not fit the reference's int frame index", v.step[k]);
        fidx[k] = (int)v.step[k];
    }
    return AC4_OK;
}

int ac4_frames_view_get(const ac4_frames *f, ac4_frames_view *v) {
    AC4_REQUIRE(f && v, AC4_EARG, "frames view: bad arguments");
    v->n = f->n;
    v->count = f->count;
    v->L = f->L;
    v->x = f->x;
    v->y = f->y;
    v->z = f->z;
    v->step = f->step.data();
    v->s = f->s;
    return AC4_OK;
}

extern "C" int ac4_frames_find(const ac4_frames *f, long long step) {
    if (!f) return -1;
    for (int k = 0; k < f->count; k++)
        if (f->step[k] == step) return k;
    return -1;
}

extern "C" int ac4_frames_push(ac4_frames *f, const double *xu, const double *yu, const double *zu, long long step) {
    AC4_REQUIRE(f && xu && yu && zu, AC4_EARG, "frames_push: bad arguments");
    AC4_REQUIRE(f->count < f->cap, AC4_ECAP, "frames_push: store full (%d frames)", f->cap);
    const size_t o = (size_t)f->count * f->n, b = sizeof(double) * f->n;
    AC4_HIP(hipMemcpyAsync(f->x + o, xu, b, hipMemcpyHostToDevice, f->s));
    AC4_HIP(hipMemcpyAsync(f->y + o, yu, b, hipMemcpyHostToDevice, f->s));
    AC4_HIP(hipMemcpyAsync(f->z + o, zu, b, hipMemcpyHostToDevice, f->s));
    AC4_HIP(hipStreamSynchronize(f->s));
    f->step.push_back(step);
    f->count++;
    return AC4_OK;
}

extern "C" int ac4_frames_push_device(ac4_frames *f, const double *xu, const double *yu, const double *zu,
                                      long long step) {
    AC4_REQUIRE(f && xu && yu && zu, AC4_EARG, "frames_push_device: bad arguments");
    AC4_REQUIRE(f->count < f->cap, AC4_ECAP, "frames_push_device: store full (%d frames)", f->cap);
    const size_t o = (size_t)f->count * f->n, b = sizeof(double) * f->n;
    AC4_HIP(hipMemcpyAsync(f->x + o, xu, b, hipMemcpyDeviceToDevice, f->s));
    AC4_HIP(hipMemcpyAsync(f->y + o, yu, b, hipMemcpyDeviceToDevice, f->s));
    AC4_HIP(hipMemcpyAsync(f->z + o, zu, b, hipMemcpyDeviceToDevice, f->s));
    AC4_HIP(hipStreamSynchronize(f->s));
    f->step.push_back(step);
    f->count++;
    return AC4_OK;
}

extern "C" int ac4_frames_push_md(ac4_frames *f, ac4_md *md, int r, long long step) {
    AC4_REQUIRE(f && md, AC4_EARG, "frames_push_md: bad arguments");
    AC4_REQUIRE(f->count < f->cap, AC4_ECAP, "frames_push_md: store full (%d frames)", f->cap);
    const double *xu, *yu, *zu;
    const int *tp;
    int n = 0;
    TRY(ac4_md_device_xu(md, r, &xu, &yu, &zu, &tp, &n));  // synchronises the MD stream
    AC4_REQUIRE(n == f->n, AC4_EARG, "frames_push_md: replica has %d particles, store %d", n, f->n);
    const size_t o = (size_t)f->count * f->n, b = sizeof(double) * f->n;
    AC4_HIP(hipMemcpyAsync(f->x + o, xu, b, hipMemcpyDeviceToDevice, f->s));
    AC4_HIP(hipMemcpyAsync(f->y + o, yu, b, hipMemcpyDeviceToDevice, f->s));
    AC4_HIP(hipMemcpyAsync(f->z + o, zu, b, hipMemcpyDeviceToDevice, f->s));
    AC4_HIP(hipStreamSynchronize(f->s));
    f->step.push_back(step);
    f->count++;
    return AC4_OK;
}

extern "C" int ac4_frames_overlap(ac4_frames *f, int i0, int i1, double a, int *count) {
    AC4_REQUIRE(f && count && a > 0 && i0 >= 0 && i1 >= 0 && i0 < f->count && i1 < f->count, AC4_EARG,
                "frames_overlap: bad arguments");
    AC4_HIP(hipMemsetAsync(f->cnt, 0, sizeof(unsigned int), f->s));
    hipLaunchKernelGGL(k_fr_overlap, dim3((f->n + FR_THREADS - 1) / FR_THREADS), dim3(FR_THREADS), 0, f->s, f->x,
                       f->y, f->z, f->n, (size_t)i0 * f->n, (size_t)i1 * f->n, f->L, a * a, f->cnt);
    AC4_HIP(hipGetLastError());
    unsigned int c = 0;
    AC4_HIP(hipMemcpyAsync(&c, f->cnt, sizeof c, hipMemcpyDeviceToHost, f->s));
    AC4_HIP(hipStreamSynchronize(f->s));
    *count = (int)c;
    return AC4_OK;
}

// Unit directions from a seed: Philox-4x32-10 with counter (d, 0x5334, 0, 0),
// z = 1 - 2u, phi = 2 pi u' (uniform on the sphere, Archimedes).
extern "C" int ac4_shell_directions(int ndir, uint64_t seed, double *n3) {
    AC4_REQUIRE(ndir > 0 && n3, AC4_EARG, "shell_directions: bad arguments");
    const uint32_t key[2] = {(uint32_t)seed, (uint32_t)(seed >> 32)};
    for (int d = 0; d < ndir; d++) {
        uint32_t c[4] = {(uint32_t)d, 0x5334u, 0u, 0u}, o[4];
        ac4_philox(c, key, o);
        const double u1 = ((double)o[0] + 0.5) * (1.0 / 4294967296.0), u2 = ((double)o[1] + 0.5) * (1.0 / 4294967296.0);
        const double zz = 1.0 - 2.0 * u1, rr = sqrt(std::max(0.0, 1.0 - zz * zz)), ph = 6.283185307179586 * u2;
        n3[3 * d] = rr * cos(ph);
        n3[3 * d + 1] = rr * sin(ph);
        n3[3 * d + 2] = zz;
    }
    return AC4_OK;
}

// Variance reductions of S4 on shells from the per-pair phase sums
// ph[p][d][k][2] (host memory), as described at the top of this file.
static void s4_reduce_host(const double *ph, int npairs, int ndir, int nshell, double N, double *s4_ref,
                           double *s4_dir) {
    const size_t ne = (size_t)ndir * nshell * 2;
    const double inv_p = 1.0 / npairs;
    for (int k = 0; k < nshell; k++) {
        double mc = 0, mc2 = 0, ms = 0, ms2 = 0, dir_sum = 0;
        for (int p = 0; p < npairs; p++) {
            double c = 0, s = 0;
            for (int d = 0; d < ndir; d++) {
                const double *e = ph + (size_t)p * ne + ((size_t)d * nshell + k) * 2;
                c += e[0];
                s += e[1];
            }
            c /= ndir;
            s /= ndir;
            mc += c; mc2 += c * c; ms += s; ms2 += s * s;
        }
        mc *= inv_p; mc2 *= inv_p; ms *= inv_p; ms2 *= inv_p;
        for (int d = 0; d < ndir; d++) {
            double c1 = 0, c2 = 0, s1 = 0, s2 = 0;
            for (int p = 0; p < npairs; p++) {
                const double *e = ph + (size_t)p * ne + ((size_t)d * nshell + k) * 2;
                c1 += e[0]; c2 += e[0] * e[0]; s1 += e[1]; s2 += e[1] * e[1];
            }
            c1 *= inv_p; c2 *= inv_p; s1 *= inv_p; s2 *= inv_p;
            dir_sum += (c2 - c1 * c1) + (s2 - s1 * s1);
        }
        if (s4_ref) s4_ref[k] = ndir * ((mc2 - mc * mc) + (ms2 - ms * ms)) / N;
        if (s4_dir) s4_dir[k] = dir_sum / ndir / N;
    }
}

static int s4_check_args(ac4_frames *f, int npairs, const int *orig, const int *lagf, double a, int nshell, int ndir,
                         double dq) {
    AC4_REQUIRE(f && npairs > 0 && orig && lagf && a > 0 && nshell > 0 && ndir > 0 && dq >= 0, AC4_EARG,
                "frames_s4_shells: bad arguments");
    const int ngroup = (nshell + SHELL_RUN - 1) / SHELL_RUN;
    AC4_REQUIRE(ndir * ngroup <= FR_ROLES, AC4_EARG,
                "frames_s4_shells: ndir * ceil(nshell/%d) must be <= %d", SHELL_RUN, FR_ROLES);
    for (int p = 0; p < npairs; p++)
        AC4_REQUIRE(orig[p] >= 0 && orig[p] < f->count && lagf[p] >= 0 && lagf[p] < f->count, AC4_EARG,
                    "frames_s4_shells: pair %d refers to a frame not in the store", p);
    return AC4_OK;
}

// The phase sums of every pair to ph[npairs][ndir][nshell][2] (host) through
// part (FR_BLOCKS * ndir * nshell * 2 doubles on the device).  The FR_BLOCKS
// workgroups of a launch are shared by as many pairs as leave each workgroup
// at least one tile of particles: one pair for boxes of 131072 particles and
// more, whose workgroups then fill the device alone.
static int s4_phases(ac4_frames *f, int npairs, const int *orig, const int *lagf, double a, double q0, double dq,
                     int nshell, int ndir, const double *dirs, double *part, double *ph) {
    const int ngroup = (nshell + SHELL_RUN - 1) / SHELL_RUN;
    const size_t ne = (size_t)ndir * nshell * 2;
    const int bpp = std::max(FR_BLOCKS / FR_PAIRS, std::min(FR_BLOCKS, (f->n + PH_THREADS - 1) / PH_THREADS));
    const int batch = std::min(FR_PAIRS, FR_BLOCKS / bpp);
    const double turn = f->L / 6.283185307179586;  // phases in turns per unit |q|
    auto kern = (ngroup % 2 == 0 || ngroup >= 5) ? k_fr_phase<2> : k_fr_phase<1>;
    for (int p0 = 0; p0 < npairs; p0 += batch) {
        const int np = std::min(batch, npairs - p0);
        FrPairs pr = {};
        for (int k = 0; k < np; k++) {
            pr.o[k] = (size_t)orig[p0 + k] * f->n;
            pr.l[k] = (size_t)lagf[p0 + k] * f->n;
        }
        hipLaunchKernelGGL(kern, dim3(np * bpp), dim3(PH_THREADS), 0, f->s, f->x, f->y, f->z, f->n, pr, bpp,
                           f->L * f->L, a * a, q0 * turn, dq * turn, nshell, ndir, ngroup, dirs, part);
        hipLaunchKernelGGL(k_fr_reduce, dim3((unsigned)((ne + 63) / 64), np), dim3(256), 0, f->s, part, bpp, (int)ne);
        AC4_HIP(hipGetLastError());
        AC4_HIP(hipMemcpy2DAsync(ph + (size_t)p0 * ne, sizeof(double) * ne, part, sizeof(double) * ne * bpp,
                                 sizeof(double) * ne, np, hipMemcpyDeviceToHost, f->s));
    }
    AC4_HIP(hipStreamSynchronize(f->s));
    return AC4_OK;
}

extern "C" int ac4_frames_s4_shells(ac4_frames *f, int npairs, const int *orig, const int *lagf, double a, double q0,
                                    double dq, int nshell, int ndir, uint64_t seed, double *s4_ref, double *s4_dir,
                                    double *phases) {
    TRY(s4_check_args(f, npairs, orig, lagf, a, nshell, ndir, dq));
    const size_t ne = (size_t)ndir * nshell * 2;
    if (f->part_n < FR_BLOCKS * ne) {
        if (f->part) (void)hipFree(f->part);
        f->part = nullptr;
        f->part_n = 0;
        AC4_HIP(hipMalloc(&f->part, sizeof(double) * FR_BLOCKS * ne));
        f->part_n = FR_BLOCKS * ne;
    }
    if (f->dirs_n < ndir) {
        if (f->dirs) (void)hipFree(f->dirs);
        f->dirs = nullptr;
        f->dirs_n = 0;
        AC4_HIP(hipMalloc(&f->dirs, sizeof(double) * 3 * ndir));
        f->dirs_n = ndir;
    }
    std::vector<double> dir(3 * (size_t)ndir), own;
    if (!phases) {
        own.resize((size_t)npairs * ne);
        phases = own.data();
    }
    TRY(ac4_shell_directions(ndir, seed, dir.data()));
    AC4_HIP(hipMemcpyAsync(f->dirs, dir.data(), sizeof(double) * dir.size(), hipMemcpyHostToDevice, f->s));
    TRY(s4_phases(f, npairs, orig, lagf, a, q0, dq, nshell, ndir, f->dirs, f->part, phases));
    s4_reduce_host(phases, npairs, ndir, nshell, (double)f->n, s4_ref, s4_dir);
    return AC4_OK;
}

// ---------------------------------------------- S4 on shells, allocating nothing
// The per-block partial sums and the directions live in one file-scope device array instead of buffers of the frame store, so a
// call makes no device or host allocation.  Each GPU holds its own copy of
// the array until the process ends; its address on the current device is
// looked up once (hipGetSymbolAddress) and kept per device.  Calls that
// overlap on one GPU share the array and race.
// ndir * ceil(nshell / SHELL_RUN) <= FR_ROLES bounds ndir * nshell by
// FR_ROLES * SHELL_RUN = 6912, so ne = 2 * ndir * nshell <= 13824.
#define S4_NOALLOC_NE_MAX (2 * FR_ROLES * SHELL_RUN)
#define S4_NOALLOC_DIR_MAX FR_ROLES
#define S4_SCRATCH_DOUBLES ((size_t)FR_BLOCKS * S4_NOALLOC_NE_MAX + 3 * S4_NOALLOC_DIR_MAX)
static __device__ __align__(256) double scratch[S4_SCRATCH_DOUBLES];  // 28.3 MB per GPU
#define S4_MAX_DEV 64
static double *g_scratch_ptr[S4_MAX_DEV];

static int scratch_ptr(double **out) {
    int dev = 0;
    AC4_HIP(hipGetDevice(&dev));
    AC4_REQUIRE(dev >= 0 && dev < S4_MAX_DEV, AC4_EARG, "s4_shells_noalloc: device %d beyond %d", dev, S4_MAX_DEV);
    if (!g_scratch_ptr[dev]) {
        void *p = nullptr;
        AC4_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        AC4_REQUIRE(p != nullptr, AC4_EHIP, "s4_shells_noalloc: no device address for the scratch array");
        g_scratch_ptr[dev] = (double *)p;
    }
    *out = g_scratch_ptr[dev];
    return AC4_OK;
}

extern "C" int ac4_frames_s4_shells_noalloc(ac4_frames *f, int npairs, const int *orig, const int *lagf, double a,
                                            double q0, double dq, int nshell, int ndir, uint64_t seed,
                                            double *s4_ref, double *s4_dir, double *phases) {
    TRY(s4_check_args(f, npairs, orig, lagf, a, nshell, ndir, dq));
    AC4_REQUIRE(phases, AC4_EARG, "s4_shells_noalloc: phases (npairs*ndir*nshell*2 doubles) is required");
    const size_t ne = (size_t)ndir * nshell * 2;
    AC4_REQUIRE(ne <= S4_NOALLOC_NE_MAX, AC4_ECAP,
                "s4_shells_noalloc: ndir * nshell = %d exceeds the scratch limit of %d", ndir * nshell,
                S4_NOALLOC_NE_MAX / 2);
    double *sp = nullptr;
    TRY(scratch_ptr(&sp));
    double *part = sp, *dirs = sp + (size_t)FR_BLOCKS * S4_NOALLOC_NE_MAX;
    double dir[3 * S4_NOALLOC_DIR_MAX];  // ndir <= FR_ROLES (checked above)
    TRY(ac4_shell_directions(ndir, seed, dir));
    AC4_HIP(hipMemcpyAsync(dirs, dir, sizeof(double) * 3 * ndir, hipMemcpyHostToDevice, f->s));
    TRY(s4_phases(f, npairs, orig, lagf, a, q0, dq, nshell, ndir, dirs, part, phases));
    s4_reduce_host(phases, npairs, ndir, nshell, (double)f->n, s4_ref, s4_dir);
    return AC4_OK;
}
