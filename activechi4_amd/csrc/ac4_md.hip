// ac4_md.hip -- active Kob-Andersen MD step for MI355X (gfx950).
//
// Replaces MDcode/cell_list+forces.c, MDcode/time_evolve.c:476-609 and
// MDcode/active.c:45-85 (paths relative to the reference checkout).  The
// whole box of every replica is resident in HBM (no domain decomposition,
// MDcode/Parallel.c); replicas are packed into every launch through a block
// table (block -> replica, first particle), so one launch sequence per step
// advances all of them.
//
// Per step (every launch covers all replicas, kernels early-exit per replica):
//   k_shuffle      ShuffleActDirec when step % tau_per == 0 (swap chain of
//                  active.c:58-75 per component, Philox uniforms); in the
//                  first workgroups of k_first_half where its LDS is small
//   k_first_half   U4 U3 U4 (chain start, computed redundantly per block),
//                  U2 kick, U1 drift + wrap + max displacement (atomicMax)
//   k_bin .. k_nlist_team   counting-sort cell build + neighbour lists,
//                  executed only for replicas whose displacement criterion
//                  fired (flag read on device, so the sequence is graphable)
//   k_force        pair forces + active force + second U2 kick; in the last
//                  workgroups the sums per replica and U4 U3 U4 (chain end)
// The momentum factor of the last U3 is kept pending (p_scale) and applied at
// the next first half, so a step needs one sum of p^2 instead of four.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>
#include <string.h>
#include <stdlib.h>
#include <vector>
#include <algorithm>
#include <type_traits>
#include "ac4_internal.h"

#define BLK 256
#define LPB 16  // particles per list-build workgroup

// MDcode/global.h:24-45 (Sigma = 1.00)
#define K_LCUTSQR (6.25 * 1.00 * 1.00)
#define K_SKIN (.35 * 1.00)
#define K_CELL_CUT ((2.5 * 1.00) + (.35 * 1.00))
#define K_CELL_CUT_SQ (K_CELL_CUT * K_CELL_CUT)
#define K_DT 0.005
#define K_HALF_DT (K_DT * 0.5)
#define K_C0 0.0162665594880
#define K_C2 -0.001949973872640

struct RepC {
    int n, off, nact, off_act;
    int nc, ncell, off_cell, tau;      // list grid: nc = floor(L/2.85) cells per axis (27-cell stencil)
    int nblk, blk_off, nc_ref, tpp;    // nc_ref: the reference's grid (Parallel.c:72-80)
    int fnblk, fblk_off, ltpp, cap_n;  // force-kernel block table (tpp = 1<<ltpp lanes per particle)
    int cap_cells, lblk_off;           // lblk: list-build blocks of LPB particles
    int lnblk, lc;                     // lc: log2 of the list chunk (below)
    double L, invL, inv_cell_ref, T, f0, dof, density;
    uint32_t key0, key1;
    double qscale;  // L / 2^32: real length of one unit of a fixed-point coordinate
    double skin;    // Verlet skin: list radii 2.5 sigma_ab + skin, rebuild criterion
    float qs2;      // qscale^2 in FP32
    int xcull;      // a cell's slots are ordered by x-half, which list teams may skip (configure_rep)
    float lcut[3];         // qscreen_cut of species pair ab
    float lr2[2];          // what a particle of species a reaches in any list, squared, with a margin of 2e-3
    float rnc, cell, fix2cell;  // 1/nc, L/nc, nc/2^32
    float rcq[3], c2i[3];  // species pair ab: cutoff^2 in fixed-point units^2, C2 / sigma^2 (FP32 path)
};

// One workgroup's particles: replica, first local particle, the replica's
// first slot and its particle count.  One 16-byte load, after which the
// particle loads can be issued beside the replica's constants instead of
// after them.
struct BlkD {
    int rep, first, off, n;
};

// Fixed-point copy of a wrapped position for the FP32 force path and the
// dynamics lists: each box fraction s in [0,1) as the 32-bit integer
// floor(s * 2^32) (quantum L/2^32, below 1e-8 sigma for L < 40), with the
// species (0 or 1) in the lowest bit of x.  The 32-bit difference of two such
// coordinates, read as a signed integer, is the minimum-image separation
// (cell_list+forces.c:92-97 up to the tie at exactly half a box), exact in y
// and z and within one quantum in x.  A neighbour costs one 12-byte load: 64
// lanes gathering 12-byte records touch fewer 128-byte lines than with
// 16-byte ones, and the gathers are what bound the force kernel.
struct QPos {
    unsigned int x, y, z;
};
__host__ __device__ __forceinline__ QPos qpos(double sx, double sy, double sz, int t) {
    QPos q;
    q.x = ((unsigned int)(unsigned long long)(sx * 4294967296.0) & ~1u) | (unsigned int)(t & 1);
    q.y = (unsigned int)(unsigned long long)(sy * 4294967296.0);
    q.z = (unsigned int)(unsigned long long)(sz * 4294967296.0);
    return q;
}
__host__ __device__ __forceinline__ int ptype(const QPos &q) { return (int)(q.x & 1u); }
__host__ __device__ __forceinline__ int ptype(const double4 &q) { return (int)q.w; }

struct ChainS {
    double eta[3], peta[3], q[3];
    double S_end, p_scale;
    double pe, vir, ke, inst_T, heff, drift;
    unsigned long long maxbits;
    long long step, shuffles;
    int rebuilds, force_rebuild, err, crit;
    unsigned int done_blocks, bin_done;  // no longer counted (kept for the checkpoint layout)
    int mode;                 // 0: Nose-Hoover chain, 1: velocity-rescale ramp, 2: NVE
    int ramp_n, ramp_k;
    double ramp0, ramp1;      // target T = T*(ramp0 + (ramp1-ramp0)*k/(n-1))
};



__device__ __forceinline__ double minimg_md(double d) {  // cell_list+forces.c:92-97
    if (d < -0.5) d += 1.0;
    if (d > 0.5) d -= 1.0;
    return d;
}

// exp(-x) and (1 - exp(-x)) / x.  The chain's x are of order 1e-3: below 1/16
// both come from one series, phi = sum (-x)^k / (k+1)!, whose remainder there
// is below 3e-19, and exp(-x) = 1 - x phi: within an ulp, where 1 - exp(-x)
// loses the digits that cancel.  The chain runs on one lane between two
// kernels of the step, so the length of its serial chain of operations is
// what it costs: 4.1 -> 3.5 us (with the sums) on one box of N=1000 with this,
// the reciprocals of q and the start-of-step half kept from k_first_half.
__host__ __device__ inline double exp_phi(double x, double *phi) {
    if (fabs(x) < 0.0625) {
        double p = fma(-x, 1.0 / 3628800.0, 1.0 / 362880.0);
        p = fma(-x, p, 1.0 / 40320.0);
        p = fma(-x, p, 1.0 / 5040.0);
        p = fma(-x, p, 1.0 / 720.0);
        p = fma(-x, p, 1.0 / 120.0);
        p = fma(-x, p, 1.0 / 24.0);
        p = fma(-x, p, 1.0 / 6.0);
        p = fma(-x, p, 0.5);
        p = fma(-x, p, 1.0);
        *phi = p;
        return fma(-x, p, 1.0);
    }
    const double e = exp(-x);
    *phi = (1.0 - e) / x;
    return e;
}

// U4 propagator (MDcode/time_evolve.c:578-609) with the p^2 sum supplied;
// iq[j] = 1/q[j].
__host__ __device__ inline void nhc_u4(double t, int jStart, int jEnd, double S, double T, double dof,
                                       const double *iq, double *peta) {
    int dj = 1;
    double gj = 0.0;
    if (jStart > jEnd) dj = -1;
    int j = jStart;
    do {
        if (j == 0) {
            gj = S;
            gj -= dof * T;
        } else {
            gj = (peta[j - 1] * peta[j - 1]) * iq[j - 1] - T;
        }
        if (j == 2) {
            peta[j] = peta[j] + t * gj;
        } else {
            double phi;
            const double e = exp_phi(t * peta[j + 1] * iq[j + 1], &phi);
            peta[j] = peta[j] * e + t * gj * phi;
        }
        j = j + dj;
    } while (j - dj != jEnd);
}

// U4(dt/4,2->0) U3(dt/2) U4(dt/4,0->2) on a copy of the chain (time_evolve.c:499-501
// and :517-519); S = sum p^2 entering; returns the U3 momentum factor.
__host__ __device__ inline double nhc_half(double S, double T, double dof, const double *q, double *eta,
                                           double *peta, double *S_out) {
    const double iq[3] = {1.0 / q[0], 1.0 / q[1], 1.0 / q[2]};
    nhc_u4(K_DT * 0.25, 2, 0, S, T, dof, iq, peta);
    double t = K_DT * 0.50, phi;
    double s = exp_phi(t * peta[0] * iq[0], &phi);                     // time_evolve.c:571
    for (int i = 0; i < 3; i++) eta[i] = eta[i] + t * peta[i] * iq[i];  // :575
    double S2 = S * s * s;
    nhc_u4(K_DT * 0.25, 0, 2, S2, T, dof, iq, peta);
    *S_out = S2;
    return s;
}

__device__ __forceinline__ bool need_rebuild(const RepC &R, const ChainS &c) {
    if (c.force_rebuild) return true;
    double maxD = __longlong_as_double((long long)c.maxbits);
    maxD *= R.L * R.L;  // time_evolve.c:553
    return (c.crit == 1 ? 3.0 : 4.0) * maxD > R.skin * R.skin;  // :508 (crit 1, skin 0.35 there)
}

// The last workgroup of a replica to finish a kernel does what follows it for
// the whole replica (k_force: sums and chain update; k_bin: scan of the cell
// counts).  What the workgroups hand over goes through agent-scope relaxed
// stores and loads, which are coherent between the XCDs' L2s by themselves:
// the giver waits for its stores to arrive (wait_stores) before it counts
// itself done, and the last one, told by the count, reads.  An agent-scope
// release or acquire fence instead writes back and invalidates the L2 of the
// workgroup's XCD (buffer_wbl2, buffer_inv) and costs every other workgroup
// its gathers' L2 hits (k_force 42.3 -> 55.6 us on the 64-replica ensemble).
// Nothing waits for another workgroup.
__device__ __forceinline__ void st_agent(double *p, double v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ double ld_agent(const double *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ int ld_agent(const int *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void wait_stores() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
// Counts that several parties reach at once lie a line (DONE_PAD ints) apart:
// atomics on one line are done one after the other across the device (about
// 8 ns each; with the groups' counts side by side k_force at N=10000 was 4 us
// longer).
#define DONE_PAD 32
// one more of the `of` parties is done; true for the last, whose count starts the next launch at zero
__device__ __forceinline__ bool last_done(unsigned *count, int of) {
    const unsigned k = __hip_atomic_fetch_add(count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (k + 1u != (unsigned)of) return false;
    __hip_atomic_store(count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("" ::: "memory");  // what the others handed over is read after this
    return true;
}

// Rebuild work of one step: the blocks of the replicas due for a rebuild,
// appended by bin_end for each such replica, so the kernels after
// k_bin run a fixed grid over this list instead of one workgroup per block of
// every replica (most of which would have nothing to do).  n[0]: particle
// blocks of BLK (global block ids); n[1]: list blocks of LPB particles
// (global ids) at item + off_l; n[2]: cell blocks (replica << 16 | block of
// BLK/64 cells) at item + off_c.  The counters are cleared by k_first_half
// (and k_cell_zero for a forced rebuild).
struct WorkList {
    int *item, *n;
    int off_l, off_c;
};

// Workgroups are dispatched round-robin over the 8 XCDs (workgroup w runs on
// XCD w % 8).  Kernels that gather neighbour positions launch 8*ceil(nb/8)
// workgroups and map workgroup w to logical block (w % 8)*ceil(nb/8) + w/8, so
// every XCD works on a contiguous range of blocks (a few whole replicas) and
// finds their positions in its own L2.  Returns -1 for the padding blocks.
#define N_XCD 8
__device__ __forceinline__ int xcd_block(int nb) {
    const int per = (nb + N_XCD - 1) / N_XCD;
    const int lb = (int)(blockIdx.x % N_XCD) * per + (int)(blockIdx.x / N_XCD);
    return lb < nb ? lb : -1;
}
static inline int xcd_grid(int nb) { return ((nb + N_XCD - 1) / N_XCD) * N_XCD; }

// ---------------------------------------------------------------- kernels
// Swap shuffle of one direction component of one replica per workgroup
// (grid: replicas x 3).  The swap partners j_i = (int)(Nact*U_i) do not depend
// on the array, so the 256 lanes draw them SHUF_CH at a time into LDS and one
// lane applies the swaps in order.  The component lives in dynamic LDS when
// it fits (kcap bytes, sized from the device's LDS per workgroup), else in
// global memory.  The shuffle counter is advanced by force_end (or
// the host for an explicit shuffle), after every component has read it.
#define SHUF_CH 4096
#define SHUF_PAR_MIN 16384  // active sets above this take the parallel path (k_shuf_part, k_shuf_apply)
#define SHUF_TRACE_MAX 1024 // active sets up to this are shuffled by tracing every position back

// Lane t traces positions t, t+256, ... (C of them, independent chains side
// by side) back through the swaps na-1 ... 0; the partners come from LDS four
// at a time, the next four loaded before the current four are applied.
template <int C>
__device__ __forceinline__ void shuffle_trace(const unsigned int *s_j, const int8_t *s_k, int8_t *kg, int na) {
    int y[C];
#pragma unroll
    for (int c = 0; c < C; c++) y[c] = threadIdx.x + 256 * c;
    int q = na - 1;
    for (; q >= 0 && ((q + 1) & 3); q--) {  // down to a multiple of four
        const int jq = (int)s_j[q];
#pragma unroll
        for (int c = 0; c < C; c++) y[c] = y[c] == q ? jq : (y[c] == jq ? q : y[c]);
    }
    if (q >= 3) {
        uint4 nx = *(const uint4 *)(s_j + q - 3);
        for (; q >= 3; q -= 4) {
            const uint4 cur = nx;
            if (q >= 7) nx = *(const uint4 *)(s_j + q - 7);
            const int j4[4] = {(int)cur.w, (int)cur.z, (int)cur.y, (int)cur.x};  // partners of q, q-1, q-2, q-3
#pragma unroll
            for (int u = 0; u < 4; u++)
#pragma unroll
                for (int c = 0; c < C; c++) y[c] = y[c] == q - u ? j4[u] : (y[c] == j4[u] ? q - u : y[c]);
        }
    }
#pragma unroll
    for (int c = 0; c < C; c++) {
        const int x = threadIdx.x + 256 * c;
        if (x < na) kg[x] = s_k[y[c]];
    }
}
// One component of one replica's shuffle by a workgroup of 256 threads (the
// branch is uniform over the workgroup); s_shuf is the dynamic LDS: SHUF_CH
// partners, then kcap bytes of directions.
__device__ __forceinline__ void shuffle_comp(const RepC &R, const ChainS &c, int comp, int8_t *kx, int8_t *ky,
                                             int8_t *kz, int force, int kcap, int skip_large, unsigned int *s_shuf) {
    unsigned int *s_j = s_shuf;
    int8_t *s_k = (int8_t *)(s_shuf + SHUF_CH);
    if (!force && (c.mode == 1 || R.tau <= 0 || (c.step % R.tau) != 0)) return;
    const uint64_t sh = (uint64_t)c.shuffles;
    const int na = R.nact;
    if (skip_large && na > SHUF_PAR_MIN) return;
    int8_t *kg = (comp == 0 ? kx : (comp == 1 ? ky : kz)) + R.off_act;
    const bool lds = na <= kcap;
    int8_t *k = lds ? s_k : kg;
    if (lds)
        for (int i = threadIdx.x; i < na; i += 256) s_k[i] = kg[i];
    if (lds && na <= SHUF_TRACE_MAX) {
        // Every position at once: the swaps s = 0..na-1 in order give the
        // value at x the one that started at the position found by tracing
        // x back through them (swap s maps s <-> j_s), so the new array is a
        // gather of the old one; exactly the serial loop's result, in about
        // na^2/64 lane operations instead of na dependent LDS round trips.
        for (int q = threadIdx.x; q < na; q += 256)
            s_j[q] = (unsigned int)(int)((double)na * ac4_shuffle_uniform(R.key0, R.key1, sh, comp, q));
        __syncthreads();
        const int nch = (na + 255) / 256;  // positions per lane, traced side by side
        if (nch == 1) shuffle_trace<1>(s_j, s_k, kg, na);
        else if (nch == 2) shuffle_trace<2>(s_j, s_k, kg, na);
        else if (nch == 3) shuffle_trace<3>(s_j, s_k, kg, na);
        else shuffle_trace<4>(s_j, s_k, kg, na);
        return;
    }
    for (int c0 = 0; c0 < na; c0 += SHUF_CH) {
        const int m = min(SHUF_CH, na - c0);
        __syncthreads();
        for (int q = threadIdx.x; q < m; q += 256)
            s_j[q] = (unsigned int)(int)((double)na * ac4_shuffle_uniform(R.key0, R.key1, sh, comp, c0 + q));
        __syncthreads();
        if (threadIdx.x == 0)  // MDcode/active.c:58-63: for i: j = (int)(Nact*U[0,1)); swap(k[i], k[j])
            for (int q = 0; q < m; q++) {
                const int i = c0 + q, jj = (int)s_j[q];
                const int8_t a = k[i], b = k[jj];
                k[i] = b;
                k[jj] = a;
            }
    }
    __syncthreads();
    if (lds)
        for (int i = threadIdx.x; i < na; i += 256) kg[i] = s_k[i];
}
__global__ void __launch_bounds__(256) k_shuffle(const RepC *__restrict__ reps, const ChainS *__restrict__ chain,
                                                 int8_t *kx, int8_t *ky, int8_t *kz, int force, int kcap, int skip_large) {
    extern __shared__ unsigned int s_shuf[];
    const int r = blockIdx.x, comp = blockIdx.y;
    const RepC R = reps[r];
    shuffle_comp(R, chain[r], comp, kx, ky, kz, force, kcap, skip_large, s_shuf);
}

// The same swap sequence in parallel for large active sets.  The swaps
// i = b*SHUF_M ... b*SHUF_M + SHUF_M - 1 of block b move values only among the
// positions they touch: the block's own SHUF_M positions and the partners j_i
// outside them.  k_shuf_part finds, for block b, where the value at each
// touched position comes from (a position of the state before the block),
// one wave per block replaying the swaps on that map (lane 0 swaps, the wave
// searches the list of outside partners); k_shuf_apply then applies the
// blocks in order, each as one gather over its touched positions.  The
// result is the serial chain's, value for value.
#define SHUF_M 256
__global__ void __launch_bounds__(64) k_shuf_part(const RepC *__restrict__ reps, const ChainS *__restrict__ chain,
                                                  int force, int bmax, int2 *__restrict__ ent, int *__restrict__ ent_n) {
    __shared__ int s_own[SHUF_M];            // source of own position b0 + q
    __shared__ int s_fp[SHUF_M], s_fs[SHUF_M];  // outside positions and their sources
    __shared__ unsigned int s_j[SHUF_M];
    __shared__ int s_nf;
    const int blk = blockIdx.x, comp = blockIdx.y, r = blockIdx.z;
    const RepC R = reps[r];
    const ChainS &c = chain[r];
    if (!force && (c.mode == 1 || R.tau <= 0 || (c.step % R.tau) != 0)) return;
    const int na = R.nact, b0 = blk * SHUF_M;
    if (na <= SHUF_PAR_MIN || b0 >= na) return;
    const int m = min(SHUF_M, na - b0), lane = threadIdx.x;
    const uint64_t sh = (uint64_t)c.shuffles;
    for (int q = lane; q < m; q += 64) {
        s_own[q] = b0 + q;
        s_j[q] = (unsigned int)(int)((double)na * ac4_shuffle_uniform(R.key0, R.key1, sh, comp, b0 + q));
    }
    if (lane == 0) s_nf = 0;
    __syncthreads();
    for (int q = 0; q < m; q++) {  // MDcode/active.c:58-63, swap(k[i], k[j]) on the source map
        const int j = (int)s_j[q];
        int f = -1;  // outside slot of j
        if (j < b0 || j >= b0 + m) {
            const int nf = s_nf;
            for (int k0 = 0; k0 < nf; k0 += 64) {
                const unsigned long long hit = __ballot(k0 + lane < nf && s_fp[k0 + lane] == j);
                if (hit) {
                    f = k0 + __ffsll((long long)hit) - 1;
                    break;
                }
            }
            if (f < 0) {  // first touch of j: its value is its own
                f = nf;
                if (lane == 0) { s_fp[nf] = j; s_fs[nf] = j; s_nf = nf + 1; }
            }
        }
        if (lane == 0) {
            const int a = s_own[q];
            if (f < 0) { s_own[q] = s_own[j - b0]; s_own[j - b0] = a; }
            else { s_own[q] = s_fs[f]; s_fs[f] = a; }
        }
        __syncthreads();
    }
    const size_t e0 = ((size_t)(r * 3 + comp) * bmax + blk) * (2 * SHUF_M);
    const int nf = s_nf;
    for (int q = lane; q < m; q += 64) ent[e0 + q] = make_int2(b0 + q, s_own[q]);
    for (int q = lane; q < nf; q += 64) ent[e0 + m + q] = make_int2(s_fp[q], s_fs[q]);
    if (lane == 0) ent_n[(size_t)(r * 3 + comp) * bmax + blk] = m + nf;
}

__global__ void __launch_bounds__(2 * SHUF_M) k_shuf_apply(const RepC *__restrict__ reps,
                                                         const ChainS *__restrict__ chain, int8_t *kx, int8_t *ky,
                                                         int8_t *kz, int force, int kcap, int bmax,
                                                         const int2 *__restrict__ ent, const int *__restrict__ ent_n) {
    extern __shared__ unsigned int s_shuf[];  // same layout as k_shuffle: directions after SHUF_CH words
    int8_t *s_k = (int8_t *)(s_shuf + SHUF_CH);
    const int r = blockIdx.x, comp = blockIdx.y;
    const RepC R = reps[r];
    const ChainS &c = chain[r];
    if (!force && (c.mode == 1 || R.tau <= 0 || (c.step % R.tau) != 0)) return;
    const int na = R.nact;
    if (na <= SHUF_PAR_MIN) return;
    int8_t *kg = (comp == 0 ? kx : (comp == 1 ? ky : kz)) + R.off_act;
    const bool lds = na <= kcap;
    int8_t *k = lds ? s_k : kg;
    if (lds)
        for (int i = threadIdx.x; i < na; i += 2 * SHUF_M) s_k[i] = kg[i];
    __syncthreads();
    const int nb = (na + SHUF_M - 1) / SHUF_M;
    for (int blk = 0; blk < nb; blk++) {  // blocks in swap order
        const size_t cb = (size_t)(r * 3 + comp) * bmax + blk;
        const int ne = ent_n[cb];
        int2 e = make_int2(0, 0);
        int8_t v = 0;
        if ((int)threadIdx.x < ne) {
            e = ent[cb * (2 * SHUF_M) + threadIdx.x];
            v = k[e.y];
        }
        __syncthreads();
        if ((int)threadIdx.x < ne) k[e.x] = v;
        __syncthreads();
    }
    if (lds)
        for (int i = threadIdx.x; i < na; i += 2 * SHUF_M) kg[i] = s_k[i];
}

// The step's shuffle as the first 3*R workgroups of k_first_half (nblk = 3*R;
// 0 when it runs as k_shuffle before it): the shuffle only has to finish
// before the force kernel reads the directions, so its workgroups run beside
// the half kick instead of as a launch of their own in the step's chain.
struct ShufArgs {
    int8_t *kx, *ky, *kz;
    int kcap, nblk;
};

__global__ void __launch_bounds__(BLK) k_first_half(const RepC *__restrict__ reps, const ChainS *chain,
                                                    const BlkD *__restrict__ blkd,
                                                    double *x, double *y, double *z, double *xu, double *yu, double *zu,
                                                    double *px, double *py, double *pz, const double *__restrict__ fx,
                                                    const double *__restrict__ fy, const double *__restrict__ fz,
                                                    const double *__restrict__ xo, const double *__restrict__ yo,
                                                    const double *__restrict__ zo, const int *__restrict__ type,
                                                    double4 *pos4, QPos *posq, int q32, ChainS *chain_w,
                                                    const int *__restrict__ blk_idx, int *cnt, int *wl_n,
                                                    double *__restrict__ mid, ShufArgs sa) {
    __shared__ double s_scale[2];
    __shared__ double s_max[BLK / 64];
    if ((int)blockIdx.x < sa.nblk) {  // the step's shuffle: replica b / 3, component b % 3
        extern __shared__ unsigned int s_shuf[];
        const int rs = blockIdx.x / 3;
        const RepC Rs = reps[rs];
        shuffle_comp(Rs, chain[rs], blockIdx.x % 3, sa.kx, sa.ky, sa.kz, 0, sa.kcap, 0, s_shuf);
        return;
    }
    const int b = blockIdx.x - sa.nblk;
    const BlkD D = blkd[b];
    const int r = D.rep, i = D.first + threadIdx.x;
    const bool valid = i < D.n;
    const int g = D.off + (valid ? i : 0);
    // the particle's loads, issued before lane 0's chain half and the
    // replica's constants are waited for
    double vx = px[g], vy = py[g], vz = pz[g];
    const double hx = fx[g], hy = fy[g], hz = fz[g];
    double sx = x[g], sy = y[g], sz = z[g], ux = xu[g], uy = yu[g], uz = zu[g];
    const double ox = xo[g], oy = yo[g], oz = zo[g];
    const int ty = type[g];
    if (b == 0 && threadIdx.x < 3) wl_n[threadIdx.x] = 0;  // rebuild work of this step
    const RepC R = reps[r];
    if (threadIdx.x == 0) {
        const ChainS &c = chain[r];
        double eta[3] = {c.eta[0], c.eta[1], c.eta[2]}, peta[3] = {c.peta[0], c.peta[1], c.peta[2]}, S2;
        s_scale[0] = c.p_scale;
        s_scale[1] = (c.mode == 0 && R.n > 0) ? nhc_half(c.S_end, R.T, R.dof, c.q, eta, peta, &S2) : 1.0;
        if (blk_idx[b] == 0)  // the chain at this point of the step, for force_end
            for (int k = 0; k < 3; k++) { mid[6 * r + k] = eta[k]; mid[6 * r + 3 + k] = peta[k]; }
    }
    __syncthreads();
    // clear this replica's cell counts for a possible rebuild later in the step
    for (int c = blk_idx[b] * BLK + threadIdx.x; c < R.ncell; c += R.nblk * BLK) cnt[R.off_cell + c] = 0;
    const double ps = s_scale[0], s1 = s_scale[1];
    double d2 = 0.0;
    if (valid) {
        vx = vx * ps; vy = vy * ps; vz = vz * ps;   // end-of-step U3 of the previous step
        vx = vx * s1; vy = vy * s1; vz = vz * s1;   // U3, time_evolve.c:571-573
        vx += hx * K_HALF_DT;                       // U2, :562-564
        vy += hy * K_HALF_DT;
        vz += hz * K_HALF_DT;
        px[g] = vx; py[g] = vy; pz[g] = vz;
        double dx = vx * K_DT, dy = vy * K_DT, dz = vz * K_DT;   // U1, :532-540
        sx += dx * R.invL; sy += dy * R.invL; sz += dz * R.invL;
        ux += dx * R.invL; uy += dy * R.invL; uz += dz * R.invL;
        // applypbc1 (:15-26) loops until the coordinate is in [0,1); a
        // coordinate that is not finite or many boxes away means the run blew
        // up: flag it instead of looping
        if (!(fabs(sx) < 8.0 && fabs(sy) < 8.0 && fabs(sz) < 8.0)) {
            atomicOr(&chain_w[r].err, 2);
            sx = 0.0; sy = 0.0; sz = 0.0;
        }
        while (sx >= 1.0) sx -= 1.0;
        while (sx < 0.0) sx += 1.0;
        while (sy >= 1.0) sy -= 1.0;
        while (sy < 0.0) sy += 1.0;
        while (sz >= 1.0) sz -= 1.0;
        while (sz < 0.0) sz += 1.0;
        x[g] = sx; y[g] = sy; z[g] = sz;
        xu[g] = ux; yu[g] = uy; zu[g] = uz;
        if (q32)
            posq[g] = qpos(sx, sy, sz, ty);
        else
            pos4[g] = make_double4(sx, sy, sz, (double)ty);
        double ex = ux - ox, ey = uy - oy, ez = uz - oz;  // :547-551
        d2 = ex * ex + ey * ey + ez * ez;
    }
    d2 = ac4_wave_max(d2);
    if ((threadIdx.x & 63) == 0) s_max[threadIdx.x >> 6] = d2;
    __syncthreads();
    if (threadIdx.x == 0) {
        double m = s_max[0];
        for (int w = 1; w < BLK / 64; w++) m = fmax(m, s_max[w]);
        // The maximum only grows during this kernel (it was cleared by the
        // previous step's force epilogue), so a block whose maximum is not
        // above the value it reads needs no atomic: same-address atomics are
        // serialised across the device, one per block of a large replica.  A
        // replica of a few blocks skips the read, whose latency would end the
        // launch.
        const unsigned long long mb = (unsigned long long)__double_as_longlong(m);
        if (R.nblk <= 64 || mb > __hip_atomic_load(&chain_w[r].maxbits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
            atomicMax(&chain_w[r].maxbits, mb);
    }
}

// ---- rebuild: counting sort into cells, canonical order, permutation of the
// particle arrays into cell order, neighbour lists from LDS-staged cells.
// Binning uses the finest grid with cells >= 2.85 (list cutoff); the
// reference's own grid (MDcode/Parallel.c:72-80) is evaluated beside it for
// the cell ids update_cell_list reports.
__global__ void __launch_bounds__(BLK) k_cell_zero(const RepC *__restrict__ reps, const ChainS *__restrict__ chain,
                                                   int *cnt, int *wl_n) {
    if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x < 3) wl_n[threadIdx.x] = 0;
    const RepC R = reps[blockIdx.x];
    const int c = blockIdx.y * BLK + threadIdx.x;
    if (c >= R.ncell || !need_rebuild(R, chain[blockIdx.x])) return;
    cnt[R.off_cell + c] = 0;
}

__device__ __forceinline__ int clampc(int c, int n) { return min(max(c, 0), n - 1); }

// Binning: the reference cell id (bit-exact, for update_cell_list) and the
// list-grid cell of every particle, with the place within its cell taken by
// an atomic on the cell's count; the particle's (slot, key) is written to
// that place of its cell's row of CELL_CAP entries (the reference's
// InCell[cell][MaxPartInCell], MDcode/global.h:20,85; a fuller cell sets the
// capacity error).  key: the octant of the cell the particle is in (x bit
// highest where the list teams cull, else z), then its id, the order
// k_cell_sort puts the cell in.  The replica's last workgroup (fuse; else
// k_bin_end) then turns the cell counts into start offsets.
// The cell counts of a replica due for a rebuild turned into start offsets
// (exclusive scan) and the replica's share of the step's rebuild work appended
// to the work list, by one workgroup of nt threads.
#define BIN_END_T 1024
template <bool AGENT>
__device__ __forceinline__ void bin_end(const RepC &R, int r, const int *cnt, int *start, WorkList wl, int nt, int *s_w,
                                        int *s_base) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int *vc = cnt + R.off_cell;
    const int per = (R.ncell + nt - 1) / nt;
    const int c0 = min((int)threadIdx.x * per, R.ncell), c1 = min(c0 + per, R.ncell);
    int own = 0;
    for (int q = c0; q < c1; q++) own += AGENT ? ld_agent(vc + q) : vc[q];
    int v = own;
    for (int o = 1; o < 64; o <<= 1) {
        const int t = __shfl_up(v, o, 64);
        if (lane >= o) v += t;
    }
    if (lane == 63) s_w[w] = v;
    __syncthreads();
    int acc = v - own;
    for (int k = 0; k < w; k++) acc += s_w[k];
    for (int q = c0; q < c1; q++) {
        start[R.off_cell + q] = acc;
        acc += AGENT ? ld_agent(vc + q) : vc[q];
    }
    // this replica's share of the step's rebuild work
    const int nb = (R.n + BLK - 1) / BLK, nl = (R.n + LPB - 1) / LPB, ncb = (R.ncell + BLK / 64 - 1) / (BLK / 64);
    if (threadIdx.x == 0) {
        s_base[0] = atomicAdd(&wl.n[0], nb);
        s_base[1] = atomicAdd(&wl.n[1], nl);
        s_base[2] = atomicAdd(&wl.n[2], ncb);
    }
    __syncthreads();
    for (int q = threadIdx.x; q < nb; q += nt) wl.item[s_base[0] + q] = R.blk_off + q;
    for (int q = threadIdx.x; q < nl; q += nt) wl.item[wl.off_l + s_base[1] + q] = R.lblk_off + q;
    for (int q = threadIdx.x; q < ncb; q += nt) wl.item[wl.off_c + s_base[2] + q] = (r << 16) | q;
}

// The same as a kernel of its own, one workgroup per replica, for handles
// with a job of more than BIN_FUSE_CELLS cells, whose scan would be long for
// a k_bin workgroup (BIN_END_T threads there).
#define BIN_FUSE_CELLS 4096
__global__ void __launch_bounds__(BIN_END_T) k_bin_end(const RepC *__restrict__ reps,
                                                       const ChainS *__restrict__ chain, const int *__restrict__ cnt,
                                                       int *start, WorkList wl) {
    __shared__ int s_w[BIN_END_T / 64], s_base[3];
    const int r = blockIdx.x;
    const RepC R = reps[r];
    if (!need_rebuild(R, chain[r])) return;  // uniform over the workgroup
    bin_end<false>(R, r, cnt, start, wl, blockDim.x, s_w, s_base);
}

#define CELL_CAP 600
__global__ void __launch_bounds__(BLK) k_bin(const RepC *__restrict__ reps, ChainS *chain,
                                             const int *__restrict__ blk_rep, const int *__restrict__ blk_first,
                                             const double *__restrict__ x, const double *__restrict__ y,
                                             const double *__restrict__ z, const int *__restrict__ id, int *cnt,
                                             int *cell_of, int2 *cell_mem, int *cell_ref, int fuse, unsigned *done,
                                             int *start, WorkList wl) {
    __shared__ int s_w[BLK / 64], s_base[3], s_last;
    const int b = blockIdx.x, r = blk_rep[b];
    const RepC R = reps[r];
    if (!need_rebuild(R, chain[r])) return;  // uniform over the replica's blocks
    const int i = blk_first[b] + threadIdx.x, lane = threadIdx.x & 63;
    const bool valid = i < R.n;
    const int g = R.off + i;
    int c = -1, key = 0;
    if (valid) {
        const double sx = x[g], sy = y[g], sz = z[g];
        // reference cell id, cell_list+forces.c:73-74 (floor in double, then sum)
        const int rx = clampc((int)floor(sx * R.inv_cell_ref), R.nc_ref),
                  ry = clampc((int)floor(sy * R.inv_cell_ref), R.nc_ref),
                  rz = clampc((int)floor(sz * R.inv_cell_ref), R.nc_ref);
        cell_ref[g] = rx + ry * R.nc_ref + rz * R.nc_ref * R.nc_ref;
        const int cx = clampc((int)floor(sx * R.nc), R.nc), cy = clampc((int)floor(sy * R.nc), R.nc),
                  cz = clampc((int)floor(sz * R.nc), R.nc);
        c = cx + cy * R.nc + cz * R.nc * R.nc;
        cell_of[g] = c;
        // octant within the cell: the parity of the cell index on the grid
        // of half-width cells, clamped as the cell index is (s * 2nc is
        // exactly twice s * nc, so the half agrees with the cell).  Where the
        // list teams cull (RepC::xcull) the x bit is highest, so each x-half
        // of a cell is one slot range (k_cell_sort); elsewhere the z bit (one
        // N=10^6 box: 2.48e9 against 2.45e9 particle-steps/s with x highest).
        // n <= 2^21, so the id fits below bit 21.
        const int ox = clampc((int)floor(sx * (2 * R.nc)), 2 * R.nc) & 1,
                  oy = clampc((int)floor(sy * (2 * R.nc)), 2 * R.nc) & 1,
                  oz = clampc((int)floor(sz * (2 * R.nc)), 2 * R.nc) & 1;
        key = ((R.xcull ? ((ox << 2) | (oy << 1) | oz) : (ox | (oy << 1) | (oz << 2))) << 21) | id[g];
    }
    // one returning atomic per particle, all in flight at once: the place
    // within the cell row depends on the order the atomics land in, which
    // k_cell_sort removes (it orders each cell by key)
    // Places within the cells: the wave's particles form runs of equal cells
    // (they are in cell order from the last rebuild, up to the few that
    // moved); the first lane of each run takes the run's places with one
    // atomic, all runs at once, and the run's lanes follow in lane order.  A
    // cell that reappears in another run of the wave gets a second atomic.
    const int cp = __shfl_up(c, 1, 64);
    const bool head = valid && (lane == 0 || cp != c);  // c == -1 on invalid lanes
    const unsigned long long heads = __ballot(head);
    const unsigned long long vmask = __ballot(valid);
    const unsigned long long upto = (lane == 63) ? ~0ull : ((2ull << lane) - 1ull);
    const unsigned long long hu = heads & upto;
    const int lead = hu ? 63 - __clzll((long long)hu) : lane;  // this lane's run head
    int my_rank = 0;
    if (head) {
        // run: from this lane to the next head or the last valid lane
        const unsigned long long after = heads & ~upto;
        const int next = after ? __ffsll((long long)after) - 1 : 64 - __clzll((long long)vmask);
        my_rank = atomicAdd(&cnt[R.off_cell + c], next - lane);
    }
    const int base = __shfl(my_rank, valid ? lead : lane, 64);
    if (valid) my_rank = base + (lane - lead);
    if (valid) {
        if (my_rank < CELL_CAP) cell_mem[(size_t)(R.off_cell + c) * CELL_CAP + my_rank] = make_int2(i, key);
        else atomicOr(&chain[r].err, 1);
    }
    if (!fuse) return;
    wait_stores();  // this wave's counts are in
    __syncthreads();
    if (threadIdx.x == 0) s_last = last_done(done + r * DONE_PAD, R.nblk);
    __syncthreads();
    if (!s_last) return;
    bin_end<true>(R, r, cnt, start, wl, BLK, s_w, s_base);
}

// Distinct neighbour-cell coordinates along one axis (cells are at least one
// list radius wide); with fewer than 3 cells per axis every cell is a
// neighbour once (an aliased stencil counts pairs twice, cf.
// cell_list+forces.c:37-49 with two cells per axis).
__device__ __forceinline__ int stencil_axis(int c, int nc, int *out) {
    if (nc >= 3) { out[0] = (c + nc - 1) % nc; out[1] = c; out[2] = (c + 1) % nc; return 3; }
    for (int d = 0; d < nc; d++) out[d] = d;
    return nc;
}

// Stencil of a cell as contiguous slot ranges: the 9 (z, y) rows of the
// 27-cell stencil, each as at most two runs of consecutive cells along x (two
// where the row wraps), in stencil order.  Cells of one x-run are adjacent in
// cell order, so their members form one slot range.  NRANGE = 18 entries per
// cell, empty ones (s == e) where the grid has fewer than 3 cells per axis.
#define NRANGE 18
__device__ __forceinline__ void xruns(int cx, int nc, int *f0, int *l0, int *f1, int *l1) {
    if (nc >= 3) {
        if (cx == 0) { *f0 = nc - 1; *l0 = nc - 1; *f1 = 0; *l1 = 1; }
        else if (cx == nc - 1) { *f0 = nc - 2; *l0 = nc - 1; *f1 = 0; *l1 = 0; }
        else { *f0 = cx - 1; *l0 = cx + 1; *f1 = 0; *l1 = -1; }
    } else {
        *f0 = 0; *l0 = nc - 1; *f1 = 0; *l1 = -1;  // every cell once (stencil_axis)
    }
}

struct PartArrays {  // particle arrays that move with a particle
    double *x, *y, *z, *xu, *yu, *zu, *px, *py, *pz;
    int *type, *act, *id, *cell_ref, *cell_of;
};

// The particle arrays as a table of 2*PART_FIELDS device pointers: P's
// x y z xu yu zu px py pz (doubles) type act id cell_ref cell_of (ints), then
// the permuted copy A's in the same order.
#define PART_FIELDS 14

// the position copies the list builders and the force read, at a new slot
struct PosCopies {
    double4 *pos4;
    QPos *posq;
    double *xo, *yo, *zo;  // x_u at this rebuild (update_cell_list, cell_list+forces.c:141-146)
};

// new slot gn <- old slot go of every array that moves with a particle, into
// dst, and the position copies at gn
__device__ __forceinline__ void gather_one(const PartArrays &src, const PartArrays &dst, const PosCopies &pc, int gn,
                                           int go) {
    const double sx = src.x[go], sy = src.y[go], sz = src.z[go], ux = src.xu[go], uy = src.yu[go], uz = src.zu[go];
    const int t = src.type[go];
    dst.x[gn] = sx; dst.y[gn] = sy; dst.z[gn] = sz;
    dst.xu[gn] = ux; dst.yu[gn] = uy; dst.zu[gn] = uz;
    dst.px[gn] = src.px[go]; dst.py[gn] = src.py[go]; dst.pz[gn] = src.pz[go];
    dst.type[gn] = t; dst.act[gn] = src.act[go]; dst.id[gn] = src.id[go];
    dst.cell_ref[gn] = src.cell_ref[go]; dst.cell_of[gn] = src.cell_of[go];
    pc.pos4[gn] = make_double4(sx, sy, sz, (double)t);
    pc.posq[gn] = qpos(sx, sy, sz, t);
    pc.xo[gn] = ux;
    pc.yo[gn] = uy;
    pc.zo[gn] = uz;
}

// Members of a cell by octant of the cell (x bit highest where the list teams
// cull, else z; k_bin), and in increasing original index within an octant
// (the binning order of cell_list+forces.c:71-80): a canonical order, so lists and force sums do not
// depend on launch timing or on which replicas share the launch.  Consecutive
// slots are then nearer in space than in plain index order, so the 64 lanes of
// a force gather touch fewer cache lines.  One wave per cell: keys staged in
// LDS, each lane ranks its entries by counting and moves each of its particles
// to its new slot (start of the cell + rank) in dst, so consecutive ranks
// write consecutive slots.  xmid: the first slot of the cell's upper x-half
// (used only where the x bit is highest).
#define SORT_CAP 256
#define XHALF (4 << 21)  // keys from here on: the upper x-half of the cell
__global__ void __launch_bounds__(BLK) k_cell_sort(const RepC *__restrict__ reps, WorkList wl,
                                                   const int *__restrict__ cnt, const int *__restrict__ start,
                                                   int2 *__restrict__ cell_mem,
                                                   int *members, int2 *ranges, int *xmid, PartArrays src,
                                                   PartArrays dst, PosCopies pc) {
    __shared__ int s_m[BLK / 64][SORT_CAP];
    __shared__ int s_k[BLK / 64][SORT_CAP];
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int nit = wl.n[2];
    for (int it = blockIdx.x; it < nit; it += gridDim.x) {
        const int item = wl.item[wl.off_c + it], r = item >> 16;
        const RepC R = reps[r];
        const int c = (item & 0xffff) * (BLK / 64) + w;  // one cell per wave
        if (c >= R.ncell) continue;
        if (lane < NRANGE) {  // the cell's stencil as slot ranges, for the list builders
            const int nc = R.nc, cx = c % nc, cy = (c / nc) % nc, cz = c / (nc * nc);
            int ay[3], az[3];
            const int ny = stencil_axis(cy, nc, ay), nz = stencil_axis(cz, nc, az);
            const int row = lane >> 1, part = lane & 1, iz = row / 3, iy = row - 3 * iz;
            int2 rg = make_int2(0, 0);
            if (iz < nz && iy < ny) {
                int f0, l0, f1, l1;
                xruns(cx, nc, &f0, &l0, &f1, &l1);
                const int f = part ? f1 : f0, l = part ? l1 : l0;
                if (l >= f) {
                    const int rb = R.off_cell + ay[iy] * nc + az[iz] * nc * nc;
                    rg = make_int2(R.off + start[rb + f], R.off + start[rb + l] + cnt[rb + l]);
                }
            }
            ranges[(size_t)(R.off_cell + c) * NRANGE + lane] = rg;
        }
        const int first = start[R.off_cell + c];
        int *m = members + R.off + first;
        // the cell's members in binning order (a cell beyond CELL_CAP has set
        // the capacity error; only its first CELL_CAP are moved)
        int2 *row = cell_mem + (size_t)(R.off_cell + c) * CELL_CAP;
        const int n = min(cnt[R.off_cell + c], CELL_CAP);
        if (n <= SORT_CAP) {
            for (int k = lane; k < n; k += 64) { const int2 v = row[k]; s_m[w][k] = v.x; s_k[w][k] = v.y; }
            __syncwarp();
            int lo = 0;
            for (int k0 = 0; k0 < n; k0 += 64) lo += __popcll(__ballot(k0 + lane < n && s_k[w][k0 + lane] < XHALF));
            if (lane == 0) xmid[R.off_cell + c] = R.off + first + lo;
            for (int k = lane; k < n; k += 64) {
                const int v = s_k[w][k];
                int rank = 0;
                for (int q = 0; q < n; q++) rank += s_k[w][q] < v;
                m[rank] = s_m[w][k];
                gather_one(src, dst, pc, R.off + first + rank, R.off + s_m[w][k]);
            }
            __syncwarp();
        } else {
            if (lane == 0) {  // crowded cell: serial insertion sort of the row on the key
                for (int a = 1; a < n; a++) {
                    const int2 v = row[a];
                    int k = a - 1;
                    while (k >= 0 && row[k].y > v.y) { row[k + 1] = row[k]; k--; }
                    row[k + 1] = v;
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");  // lane 0's order, read by every lane
            __syncwarp();
            int lo = 0;
            for (int k0 = 0; k0 < n; k0 += 64) lo += __popcll(__ballot(k0 + lane < n && row[k0 + lane].y < XHALF));
            if (lane == 0) xmid[R.off_cell + c] = R.off + first + lo;
            for (int k = lane; k < n; k += 64) {
                const int sl = row[k].x;
                m[k] = sl;
                gather_one(src, dst, pc, R.off + first + k, R.off + sl);
            }
        }
    }
}


// the permuted copy back to the primary arrays, to[g] <- from[g] (the list
// builders other than the teams, which move their own particles back)
__global__ void __launch_bounds__(BLK) k_commit(const RepC *__restrict__ reps, const int *__restrict__ blk_rep,
                                                const int *__restrict__ blk_first, WorkList wl, PartArrays to,
                                                PartArrays from) {
    const int nit = wl.n[0];
    for (int it = blockIdx.x; it < nit; it += gridDim.x) {
        const int b = wl.item[it], r = blk_rep[b];
        const RepC R = reps[r];
        const int i = blk_first[b] + threadIdx.x;
        if (i >= R.n) continue;
        const int g = R.off + i;
        to.x[g] = from.x[g]; to.y[g] = from.y[g]; to.z[g] = from.z[g];
        to.xu[g] = from.xu[g]; to.yu[g] = from.yu[g]; to.zu[g] = from.zu[g];
        to.px[g] = from.px[g]; to.py[g] = from.py[g]; to.pz[g] = from.pz[g];
        to.type[g] = from.type[g]; to.act[g] = from.act[g]; to.id[g] = from.id[g];
        to.cell_ref[g] = from.cell_ref[g]; to.cell_of[g] = from.cell_of[g];
    }
}


// List radius per species pair: its force cutoff 2.5*sigma_ab plus the skin
// (0.35 in the reference, MDcode/global.h:25-31, which applies 2.85 to every
// pair); pairs are stored when ((dx*dx+dy*dy)+dz*dz)*L*L < (2.5 sigma_ab +
// skin)^2.  The reference list (< 2.85^2 for every pair,
// cell_list+forces.c:129-130) is counted beside it.
__host__ __device__ __forceinline__ double list_cut2(int ab, double skin) {
    const double rc = (ab == 0 ? (2.5 * 1.00) : (ab == 1 ? (2.5 * 0.80) : (2.5 * 0.88))) + skin;
    return rc * rc;
}

// Each replica owns cap*n list entries from off*cap.  Neighbour k of local
// particle i lives at ((k/C)*n + i)*C + k%C in that region, C = 2^lc: with a
// team of tpp > 1 lanes per particle C = tpp, so the team reads tpp
// consecutive entries per chunk; with one lane per particle C = 8, so a lane
// reads its next 8 entries as two 16-byte loads and a wave a contiguous 2 KB.
__device__ __forceinline__ size_t nl_at(const RepC &R, int cap, int k, int i) {
    return (size_t)R.off * cap + (((size_t)(k >> R.lc) * R.n + i) << R.lc) + (k & ((1 << R.lc) - 1));
}

// The particle's position at slot j; a 32-bit byte offset for the 12-byte
// records (a handle of 2^32 / 12 slots does not fit the memory).
__device__ __forceinline__ QPos ld_pos(const QPos *p, int j) {
    const unsigned u = (unsigned)j;
    unsigned u3;  // 3u by a shift and an add; the compiler's product by 12 is a multiplication at a quarter of the rate
    asm("v_lshl_add_u32 %0, %1, 1, %1" : "=v"(u3) : "v"(u));
    return *(const QPos *)((const char *)p + (size_t)(u3 << 2));
}
__device__ __forceinline__ double4 ld_pos(const double4 *p, int j) { return p[j]; }

// Dynamics-list screen shared by every builder (so all of them keep exactly
// the same pairs): minimum image from the fixed-point positions, r^2 in FP32
// in fixed-point units (fused multiply-adds) against the list radius plus a
// margin of 1e-3 sigma^2 in those units, far above the FP32 error of r^2
// (below 1e-5 sigma^2 for the list radii), so no pair within its list radius
// is lost.  Which pairs beyond the force cutoff the margin lets in does not
// change any force: a pair contributes only inside 2.5 sigma_ab.
__device__ __forceinline__ bool qscreen(const QPos &pi, const QPos &q, float ua, float ub) {
    const float dx = (float)(int)(pi.x - q.x), dy = (float)(int)(pi.y - q.y), dz = (float)(int)(pi.z - q.z);
    return __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx)) < ((q.x & 1u) ? ub : ua);
}
// list radius^2 of species pair ab plus the screen's margin, in fixed-point units^2
__host__ __device__ __forceinline__ float qscreen_cut_of(int ab, double skin, float qs2) {
    return (float)((list_cut2(ab, skin) + 1e-3) / (double)qs2);
}
__device__ __forceinline__ float qscreen_cut(int ab, const RepC &R) {
    return ab == 0 ? R.lcut[0] : (ab == 1 ? R.lcut[1] : R.lcut[2]);
}

#define NL_UNROLL 8
// Thread per particle (slots are in cell order, so the lanes of a wave scan
// the same few cells and the position loads are shared in L1); candidate
// positions are loaded NL_UNROLL at a time to keep several loads in flight.
// Dynamics lists (EXACT=false) screen candidates in FP32 with a margin of
// 1e-3 sigma^2, far above the FP32 error of r^2 (< 1e-4 for L < 100), so no
// pair within its list radius is lost.  EXACT=true (update_cell_list) tests
// every candidate with the reference's FP64 expression and also counts the
// reference's 2.85 list.
template <bool EXACT>
__global__ void __launch_bounds__(BLK) k_nlist(const RepC *__restrict__ reps, ChainS *chain,
                                               const int *__restrict__ blk_rep, const int *__restrict__ blk_first,
                                               const double4 *__restrict__ pos4, const QPos *__restrict__ posq,
                                               const int *__restrict__ cell_of, const int *__restrict__ cnt,
                                               const int *__restrict__ start, int *nn, int *nn_ref, int *nl,
                                               int stride, int cap) {
    const int b = blockIdx.x, r = blk_rep[b];
    const RepC R = reps[r];
    if (!need_rebuild(R, chain[r])) return;
    const int i = blk_first[b] + threadIdx.x;
    if (i >= R.n) return;
    const int g = R.off + i, nc = R.nc;
    const double4 pi = pos4[g];
    const QPos pq = posq[g];
    const int ti = (int)pi.w;
    const int c = cell_of[g];
    const int cx = c % nc, cy = (c / nc) % nc, cz = c / (nc * nc);
    int ax[3], ay[3], az[3];
    const int nx = stencil_axis(cx, nc, ax), ny = stencil_axis(cy, nc, ay), nz = stencil_axis(cz, nc, az);
    const double L = R.L;
    const double cut_a = list_cut2(ti, R.skin), cut_b = list_cut2(ti + 1, R.skin);
    const float ua = qscreen_cut(ti, R), ub = qscreen_cut(ti + 1, R);
    int count = 0, cref = 0;
    for (int iz = 0; iz < nz; iz++)
        for (int iy = 0; iy < ny; iy++)
            for (int ix = 0; ix < nx; ix++) {
                const int c2 = R.off_cell + ax[ix] + ay[iy] * nc + az[iz] * nc * nc;
                const int s2 = R.off + start[c2], e2 = s2 + cnt[c2];
                for (int k = s2; k < e2; k += NL_UNROLL) {
                    if (EXACT) {
                        double4 q[NL_UNROLL];
#pragma unroll
                        for (int u = 0; u < NL_UNROLL; u++) q[u] = pos4[min(k + u, e2 - 1)];
#pragma unroll
                        for (int u = 0; u < NL_UNROLL; u++) {
                            const int j = k + u;
                            if (j >= e2 || j == g) continue;
                            // cell_list+forces.c:120-130, same operation order
                            double dx = minimg_md(pi.x - q[u].x);
                            double dy = minimg_md(pi.y - q[u].y);
                            double dz = minimg_md(pi.z - q[u].z);
                            double dr2 = (dx * dx + dy * dy + dz * dz) * L * L;
                            cref += dr2 < K_CELL_CUT_SQ;
                            if (dr2 < (q[u].w == 0.0 ? cut_a : cut_b)) {
                                if (count < cap) nl[nl_at(R, cap, count, i)] = j;
                                count++;
                            }
                        }
                    } else {
                        QPos q[NL_UNROLL];
#pragma unroll
                        for (int u = 0; u < NL_UNROLL; u++) q[u] = posq[min(k + u, e2 - 1)];
#pragma unroll
                        for (int u = 0; u < NL_UNROLL; u++) {
                            const int j = k + u;
                            if (j >= e2 || j == g) continue;
                            if (qscreen(pq, q[u], ua, ub)) {
                                if (count < cap) nl[nl_at(R, cap, count, i)] = j;
                                count++;
                            }
                        }
                    }
                }
            }
    if (count > cap) atomicOr(&chain[r].err, 1);
    nn[g] = min(count, cap);
    if (EXACT) nn_ref[g] = cref;
}

// Dynamics lists, a team of NLT lanes per particle (16, 32 or 64; LPB = 16
// particles per workgroup): the team tests NLT consecutive candidates at once
// and appends the hits in candidate order (team ballot + popcount of the
// lanes below), so the list is in the order of a serial scan (stencil cells
// z, y, x; slots within a cell) while the chain of dependent loads per
// particle is NLT times shorter.  Only the replicas due for a rebuild do work
// in a step, so wide teams are what keeps enough waves in flight.  The
// control flow is uniform within a team (one home particle per team), so
// every lane of a team is active at each ballot.  FP32 screen with the margin
// described at k_nlist.
//
// The stencil's slot ranges, trimmed to what the particle can reach, are cut
// into groups of CH_GRP candidates, listed by the team in its LDS row (ct,
// CH_CAP entries): a step of the walk takes the next NLT / CH_GRP groups, one
// round CH_PER steps, with CH_PER loads in flight per lane across range
// boundaries; the same candidates in the same order as a range-by-range walk,
// which a stencil of more than CH_CAP groups (crowded cells) takes.  (Chunks
// of one range per step left 1 lane in 4 of a step idle.)
//
// Trimming: a row of cells beside the particle's own along y or z is at least
// d away, d^2 the sum of the squared distances to the faces between; along x
// the row is needed up to sqrt(rl^2 - d^2) from the particle, rl the largest
// list radius of its species.  The cell below or above along x goes where its
// face is farther, or its far half where that is farther and the cells' slots
// are ordered by x-half (RepC::xcull, xmid), or the whole row.  What goes is
// beyond every list radius, so the lists are the same pairs in the same order.
// Of 27 cells' candidates 18 are left without the halves, 16 with (species A;
// 13.6 of B), where the halves alone left 22.5.
//
// The walk is bound by vector instructions, about 30 per step (screen, place,
// store).  With the trimming, which costs some 200 per particle pair of a wave:
// 62.4 -> 59.8 us per step on the 64-replica ensemble, 50.3 -> 48.9 at N=50000
// FP64.  TRIM = false leaves it out, for handles without a replica ordered by
// x-half: one box of 1e6 (cells of 2.852, skin 0.35) builds its lists in 840 us
// without and 926 with it (895 before the step lost its multiplication by 12
// and the ballots their detour over a register).
#define CH_CAP 128
#define CH_GRP 16
#define CH_PER 4
template <int NLT, bool TRIM>
__device__ __forceinline__ void nlist_team_one(const RepC &R, int r, int i, ChainS *chain,
                                               const QPos *__restrict__ posq, const int *__restrict__ cell_of,
                                               const int2 *__restrict__ ranges, const int *__restrict__ start,
                                               const int *__restrict__ xmid, int *nn, int *nl, int cap, int2 *ct) {
    constexpr int GPS = NLT / CH_GRP;  // groups of a step
    const int lane = threadIdx.x & 63, t = lane & (NLT - 1);
    const unsigned long long tmask = (NLT == 64 ? ~0ull : ((1ull << (NLT & 63)) - 1ull)) << (lane & ~(NLT - 1));
    const unsigned long long below = (1ull << lane) - 1ull;
    const int g = R.off + i;
    const QPos pi = posq[g];
    const int ti = ptype(pi);
    const int cg = cell_of[g];
    const int2 *rgs = ranges + (size_t)(R.off_cell + cg) * NRANGE;
    const float ua = qscreen_cut(ti, R), ub = qscreen_cut(ti + 1, R);
    int count = 0;
    // the lanes whose candidate k at q is in the list (qscreen, as a wave mask:
    // the two compares' masks and-ed, the radius picked by the species bit)
    auto inlist = [&](const QPos &q, int k) -> unsigned long long {
        const float dx = (float)(int)(pi.x - q.x), dy = (float)(int)(pi.y - q.y), dz = (float)(int)(pi.z - q.z);
        const int m = __builtin_amdgcn_sbfe((int)q.x, 0, 1);
        const float cut = __int_as_float((m & __float_as_int(ub)) | (~m & __float_as_int(ua)));
        return __builtin_amdgcn_fcmpf(__builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx)), cut, 4) &  // ordered <
               __builtin_amdgcn_uicmp((unsigned)k, (unsigned)g, 33);                                      // !=
    };
    // entry p of this particle's list at nlb[(p & ~cm) * n + (p & cm)] (nl_at
    // relative to entry 0: p >> lc chunks of n << lc entries).  Both factors
    // fit 24 bits in every layout (n <= 2^21 is checked at creation), which n
    // times the chunk length does not.
    int *const nlb = nl + nl_at(R, cap, 0, i);
    const unsigned cm = (1u << R.lc) - 1u;
    // a hit's place: the team's count so far and its hits of lower lanes
    // (mbcnt of the ballot word that holds the team)
    const unsigned mlo = NLT == 32 && lane >= 32 ? 0u : ~0u;
    auto emit = [&](unsigned long long b, int k) {
        const unsigned lo = (unsigned)b, hi = (unsigned)(b >> 32);
        unsigned pos, tot;
        if (NLT == 64) {
            pos = __builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, (unsigned)count));
            tot = __popcll(b);
        } else if (NLT == 32) {
            pos = __builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo & mlo, (unsigned)count));
            tot = __popc((lo & mlo) | (hi & ~mlo));
        } else {
            const unsigned long long m = b & tmask;
            pos = count + __popcll(m & below);
            tot = __popcll(m);
        }
        if (__builtin_amdgcn_inverse_ballot_w64(b) && pos < (unsigned)cap) nlb[__umul24(pos & ~cm, (unsigned)R.n) + (pos & cm)] = k;
        count += tot;
    };
    // the home cell's stencil as slot ranges (k_cell_sort), in stencil order:
    // lane t holds ranges t and t + NLT (when NLT < NRANGE), and the team
    // lists their chunks in range order
    int2 ra = make_int2(0, 0), rb = make_int2(0, 0);
    if (t < NRANGE) ra = rgs[t];
    if (NLT < NRANGE && t + NLT < NRANGE) rb = rgs[t + NLT];
    if (TRIM && R.nc >= 3) {
        const int nc = R.nc;
        const auto div = [&](int a, int &m) {  // a / nc and the remainder
            int q = (int)((float)a * R.rnc);
            m = a - q * nc;
            if (m < 0) { q--; m += nc; }
            if (m >= nc) { q++; m -= nc; }
            return q;
        };
        int cx, cy;
        const int cz = div(div(cg, cx), cy);
        // distances to the faces of the particle's cell (FP32 errors of 1e-5 are within lr2's margin)
        const float cell = R.cell, xl = ((float)pi.x * R.fix2cell - (float)cx) * cell,
                    yl = ((float)pi.y * R.fix2cell - (float)cy) * cell, zl = ((float)pi.z * R.fix2cell - (float)cz) * cell;
        const float xr = cell - xl, rl2 = ti ? R.lr2[1] : R.lr2[0];
        const float xlh = R.xcull ? xl + 0.5f * cell : 0.0f, xrh = R.xcull ? xr + 0.5f * cell : 0.0f;
        const bool first = cx == 0, last = cx == nc - 1;
        const auto trim = [&](int q, int2 &rg) {
            const int row = q >> 1, part = q & 1, iz = row / 3, iy = row - 3 * iz;
            const float dy = iy == 1 ? 0.0f : (iy == 0 ? yl : cell - yl), dz = iz == 1 ? 0.0f : (iz == 0 ? zl : cell - zl);
            const float reach2 = rl2 - dy * dy - dz * dz;
            if (reach2 <= 0.0f) rg.y = rg.x;
            if (rg.x >= rg.y) return;
            int yy = cy + iy - 1, zz = cz + iz - 1;
            yy = yy < 0 ? nc - 1 : (yy == nc ? 0 : yy);
            zz = zz < 0 ? nc - 1 : (zz == nc ? 0 : zz);
            const int rb = R.off_cell + __mul24(__mul24(zz, nc) + yy, nc);
            // the row's part 0 holds the cell below along x, part 1 at either end of the row the cell above (xruns)
            const bool out = xl * xl >= reach2, outr = xr * xr >= reach2;
            if (part == 0 && (out || xlh * xlh >= reach2)) {
                const int *const p = out ? start + cx : xmid + (first ? nc - 1 : cx - 1);
                const int v = p[rb] + (out ? R.off : 0);
                rg.x = out && first ? rg.y : v;
            }
            if (part == (first || last ? 1 : 0) && (outr || xrh * xrh >= reach2)) {
                const int *const p = (outr ? start : xmid) + (last ? 0 : cx + 1);
                const int v = p[rb] + (outr ? R.off : 0);
                rg.y = outr && last ? rg.x : v;
            }
        };
        trim(t, ra);
        if (NLT < NRANGE) trim(t + NLT, rb);
    }
    const int na = (ra.y - ra.x + CH_GRP - 1) / CH_GRP, nb = (rb.y - rb.x + CH_GRP - 1) / CH_GRP;
    // inclusive scans over the team: within rows of 16 lanes, then the rows
    const auto scan = [&](int v) {
        v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);  // row_shr 1, 2, 4, 8
        v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);
        v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);
        v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);
        if (NLT >= 32) v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast 15 to rows 1 and 3
        if (NLT == 64) v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast 31 to rows 2 and 3
        return v;
    };
    const int pa = scan(na), pb = NLT < NRANGE ? scan(nb) : 0;
    const int tot_a = __shfl(pa, NLT - 1, NLT), ngr = tot_a + (NLT < NRANGE ? __shfl(pb, NLT - 1, NLT) : 0);
    if (ngr <= CH_CAP) {
#pragma nounroll
        for (int j = 0; j < na; j++) ct[pa - na + j] = make_int2(ra.x + j * CH_GRP, min(CH_GRP, ra.y - ra.x - j * CH_GRP));
        if (NLT < NRANGE)
            for (int j = 0; j < nb; j++)
                ct[tot_a + pb - nb + j] = make_int2(rb.x + j * CH_GRP, min(CH_GRP, rb.y - rb.x - j * CH_GRP));
        for (int j = t; j < CH_PER * GPS; j += NLT) ct[ngr + j] = make_int2(0, 0);  // empty ones up to the next whole round
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");  // the row is read by the other lanes
        const int2 *const cl = ct + t / CH_GRP;
        const int tg = t & (CH_GRP - 1);
        for (int c0 = 0; c0 < ngr; c0 += CH_PER * GPS) {
            int2 ch[CH_PER];
            int k[CH_PER];
            QPos qv[CH_PER];
#pragma unroll
            for (int u = 0; u < CH_PER; u++) ch[u] = cl[c0 + u * GPS];
#pragma unroll
            for (int u = 0; u < CH_PER; u++) {
                k[u] = tg < ch[u].y ? ch[u].x + tg : g;  // g itself: no candidate
                qv[u] = ld_pos(posq, k[u]);
            }
#pragma unroll
            for (int u = 0; u < CH_PER; u++) emit(inlist(qv[u], k[u]), k[u]);
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");  // reads done before the row is rewritten
    } else {
        for (int q = 0; q < NRANGE; q++) {
            const int2 rg = rgs[q];
            const int s2 = rg.x, e2 = rg.y;
            // two candidates per lane, both loaded before either is used
            // (an index past the range is replaced by g, which is no candidate)
            for (int k0 = s2; k0 < e2; k0 += 2 * NLT) {
                const int ka = k0 + t < e2 ? k0 + t : g, kb = k0 + NLT + t < e2 ? k0 + NLT + t : g;
                const QPos qa = ld_pos(posq, ka), qb = ld_pos(posq, kb);
                emit(inlist(qa, ka), ka);
                emit(inlist(qb, kb), kb);
            }
        }
    }
    if (t == 0) {
        if (count > cap) atomicOr(&chain[r].err, 1);
        nn[g] = min(count, cap);
    }
}

// Fixed grid over the step's list blocks (LPB particles each, one team per
// particle); plain block order spreads the few rebuilding replicas over all
// XCDs.
template <int NLT, bool MOVE, bool TRIM>
__global__ void __launch_bounds__(NLT * LPB) k_nlist_team(const RepC *__restrict__ reps, ChainS *chain,
                                                          const int *__restrict__ lblk_rep,
                                                          const int *__restrict__ lblk_first, WorkList wl,
                                                          const QPos *__restrict__ posq,
                                                          const int *__restrict__ cell_of,
                                                          const int2 *__restrict__ ranges,
                                                          const int *__restrict__ start,
                                                          const int *__restrict__ xmid, int *nn, int *nl, int cap,
                                                          void *const *__restrict__ ftab) {
    __shared__ int2 s_ct[LPB][CH_CAP + CH_PER * NLT / CH_GRP];  // each team's groups, then empty ones
    const int nit = wl.n[1];
    for (int it = blockIdx.x; it < nit; it += gridDim.x) {
        const int b = __builtin_amdgcn_readfirstlane(wl.item[wl.off_l + it]), r = __builtin_amdgcn_readfirstlane(lblk_rep[b]);
        const RepC R = reps[r];
        // MOVE: the block's LPB particles go back from the permuted copy
        // (second half of ftab) to the primary arrays (first half) here
        // instead of in k_commit: thread t moves field t / LPB of particle
        // t % LPB, loaded here and stored after the lists, so each field's LPB
        // consecutive slots are one coalesced write.  The list build reads
        // cell_of of the copy, nothing else.  The held value costs a wave of
        // occupancy, so this pays where k_commit's launch dominates (small
        // ensembles), not for large boxes.
        const int cf = (int)threadIdx.x / LPB, cg = R.off + lblk_first[b] + (int)threadIdx.x % LPB;
        const bool cpy = MOVE && cf < PART_FIELDS && cg < R.off + R.n;
        long long cv = 0;
        if (cpy)
            cv = cf < 9 ? ((const long long *)ftab[PART_FIELDS + cf])[cg] : ((const int *)ftab[PART_FIELDS + cf])[cg];
        const int i = lblk_first[b] + (int)threadIdx.x / NLT;
        if (i < R.n)  // whole team
            nlist_team_one<NLT, TRIM>(R, r, i, chain, posq, cell_of, ranges, start, xmid, nn, nl, cap, s_ct[threadIdx.x / NLT]);
        if (cpy) {
            if (cf < 9) ((long long *)ftab[cf])[cg] = cv;
            else ((int *)ftab[cf])[cg] = (int)cv;
        }
    }
}

// Dynamics lists, one wave per cell: the particles of the 27 neighbour cells
// (contiguous slot ranges) are staged in LDS in stencil order; then for each
// home particle the 64 lanes test 64 candidates at once and the hits are
// appended in candidate order by ballot + popcount, so every list is in the
// same canonical order as a serial scan.  FP32 screen with the margin
// described at k_nlist.
#define NLC_CAP 2304
__global__ void __launch_bounds__(64) k_nlist_cell(const RepC *__restrict__ reps, ChainS *chain,
                                                   const int *__restrict__ cblk_rep, const int *__restrict__ cblk_cell,
                                                   const QPos *__restrict__ posq, const int *__restrict__ cnt,
                                                   const int *__restrict__ start, int *nn, int *nl, int cap) {
    __shared__ QPos s_c[NLC_CAP];
    __shared__ int s_pre[28], s_st[27];
    const int r = cblk_rep[blockIdx.x], c = cblk_cell[blockIdx.x];
    const RepC R = reps[r];
    if (c >= R.ncell || !need_rebuild(R, chain[r])) return;
    const int lane = threadIdx.x, nc = R.nc;
    const int cx = c % nc, cy = (c / nc) % nc, cz = c / (nc * nc);
    int ax[3], ay[3], az[3];
    const int nx = stencil_axis(cx, nc, ax), ny = stencil_axis(cy, nc, ay), nz = stencil_axis(cz, nc, az);
    const int ns = nx * ny * nz;
    // lane q < ns reads stencil cell q (stencil order: x fastest, then y, z)
    int my_n = 0, my_s = 0, is_home = 0;
    if (lane < ns) {
        const int cc = ax[lane % nx] + ay[(lane / nx) % ny] * nc + az[lane / (nx * ny)] * nc * nc;
        my_n = cnt[R.off_cell + cc];
        my_s = start[R.off_cell + cc];
        is_home = cc == c;
    }
    int pre = my_n;  // inclusive scan over the stencil cells
    for (int o = 1; o < 32; o <<= 1) {
        const int v = __shfl_up(pre, o, 64);
        if (lane >= o) pre += v;
    }
    if (lane < ns) { s_pre[lane + 1] = pre; s_st[lane] = my_s; }
    if (lane == 0) s_pre[0] = 0;
    const unsigned long long hm = __ballot(is_home);
    const int hl = __ffsll((long long)hm) - 1;  // stencil index of the home cell
    const int total = __shfl(pre, ns - 1, 64);
    const int hn = __shfl(my_n, hl, 64), hs = __shfl(my_s, hl, 64), hoff = __shfl(pre - my_n, hl, 64);
    if (total > NLC_CAP) {
        if (lane == 0) atomicOr(&chain[r].err, 1);
        return;
    }
    __syncthreads();
    for (int k = lane; k < total; k += 64) {  // independent loads
        int q = 0;
        while (s_pre[q + 1] <= k) q++;
        s_c[k] = posq[R.off + s_st[q] + (k - s_pre[q])];
    }
    __syncthreads();
    const unsigned long long below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    int mine = 0;  // list length of home particle `lane` (and lane+64, ... kept below)
    for (int h = 0; h < hn; h++) {
        const QPos pi = s_c[hoff + h];
        const int ti = ptype(pi), kh = hoff + h;
        const float ua = qscreen_cut(ti, R), ub = qscreen_cut(ti + 1, R);
        int base = 0;
        for (int k0 = 0; k0 < total; k0 += 64) {
            const int k = k0 + lane;
            bool hit = false;
            if (k < total && k != kh) hit = qscreen(pi, s_c[k], ua, ub);
            const unsigned long long mask = __ballot(hit);
            if (hit) {
                const int pos = base + __popcll(mask & below);
                if (pos < cap) {
                    int q = 0;
                    while (s_pre[q + 1] <= k) q++;
                    nl[nl_at(R, cap, pos, hs + h)] = R.off + s_st[q] + (k - s_pre[q]);
                }
            }
            base += __popcll(mask);
        }
        if ((h & 63) == lane) mine = base;
        if ((h & 63) == 63 || h == hn - 1) {  // flush 64 finished counts
            const int h0 = h & ~63;
            if (lane <= h - h0) {
                if (mine > cap) atomicOr(&chain[r].err, 1);
                nn[R.off + hs + h0 + lane] = min(mine, cap);
            }
        }
    }
}

// ---- in-situ overlap Q(t) for every replica (device-resident accumulators)
// Origins every origin_every steps are kept as snapshots of x_u in reference
// order (ring of n_origin per replica); at a sample the overlap of every
// resident origin whose lag (step - origin step) is a multiple of
// sample_every below n_lags*sample_every is counted with the arithmetic of
// Analysis/overlap.c:61-84 (unwrapped difference, one minimum-image
// correction, L*L*((dx*dx+dy*dy)+dz*dz) < a*a).  Counts are integers, so the
// per-lag sums do not depend on the order of the threads.
struct OvCfg {
    int sample_every, origin_every, n_origin, n_lags;
    double a2;
};

__device__ __forceinline__ double minimg_ov(double d) {
    if (d >= 0.5)
        d -= 1.0;
    else if (d < -0.5)
        d += 1.0;
    return d;
}

// grid (particle blocks of all replicas, n_origin)
__global__ void __launch_bounds__(BLK) k_ov_count(const RepC *__restrict__ reps, const ChainS *__restrict__ chain,
                                                  const int *__restrict__ blk_rep, const int *__restrict__ blk_first,
                                                  OvCfg cfg, const int *__restrict__ id, const double *__restrict__ xu,
                                                  const double *__restrict__ yu, const double *__restrict__ zu,
                                                  double *ox, double *oy, double *oz, const long long *ostep,
                                                  unsigned int *ocnt) {
    const int b = blockIdx.x, r = blk_rep[b], o = blockIdx.y;
    const RepC R = reps[r];
    const long long step = chain[r].step;
    const int i = blk_first[b] + threadIdx.x;
    const size_t base = ((size_t)R.off * cfg.n_origin + (size_t)o * R.cap_n);  // snapshot o of replica r
    const long long s0 = ostep[(size_t)r * cfg.n_origin + o];
    int hit = 0;
    if (i < R.n && s0 >= 0 && step > s0 && (step - s0) % cfg.sample_every == 0 &&
        (step - s0) / cfg.sample_every <= cfg.n_lags) {
        const int g = R.off + i, k = id[g];
        double dx = xu[g] - ox[base + k], dy = yu[g] - oy[base + k], dz = zu[g] - oz[base + k];
        dz = minimg_ov(dz);
        dy = minimg_ov(dy);
        dx = minimg_ov(dx);
        hit = R.L * R.L * (dx * dx + dy * dy + dz * dz) < cfg.a2;
    }
    const int w = ac4_wave_sum_i(hit);
    if ((threadIdx.x & 63) == 0 && w) atomicAdd(&ocnt[(size_t)r * cfg.n_origin + o], (unsigned int)w);
}

// one thread per (replica, origin): fold the count into the lag slot, then
// store a new origin when the step is a multiple of origin_every
__global__ void k_ov_fold(const RepC *__restrict__ reps, const ChainS *__restrict__ chain, OvCfg cfg, int nrep,
                          long long *ostep, unsigned int *ocnt, double *sq, double *sq2, int *scnt) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nrep * cfg.n_origin) return;
    const int r = t / cfg.n_origin;
    const RepC R = reps[r];
    const long long step = chain[r].step, s0 = ostep[t];
    if (R.n > 0 && s0 >= 0 && step > s0 && (step - s0) % cfg.sample_every == 0) {
        const long long lag = (step - s0) / cfg.sample_every;
        if (lag <= cfg.n_lags) {
            const double q = (double)ocnt[t] / (double)R.n;  // overlap.c:82
            const size_t k = (size_t)r * (cfg.n_lags + 1) + lag;
            sq[k] += q;        // overlap.c:89-94 (origin order: one origin per lag per step)
            sq2[k] += q * q;
            scnt[k] += 1;
        }
    }
    ocnt[t] = 0u;
}

__global__ void __launch_bounds__(BLK) k_ov_origin(const RepC *__restrict__ reps, const ChainS *__restrict__ chain,
                                                   const int *__restrict__ blk_rep, const int *__restrict__ blk_first,
                                                   OvCfg cfg, const int *__restrict__ id, const double *__restrict__ xu,
                                                   const double *__restrict__ yu, const double *__restrict__ zu,
                                                   double *ox, double *oy, double *oz, long long *ostep) {
    const int b = blockIdx.x, r = blk_rep[b];
    const RepC R = reps[r];
    const long long step = chain[r].step;
    if (R.n == 0 || step % cfg.origin_every != 0) return;
    const int o = (int)((step / cfg.origin_every) % cfg.n_origin);
    const int i = blk_first[b] + threadIdx.x;
    const size_t base = ((size_t)R.off * cfg.n_origin + (size_t)o * R.cap_n);
    if (i < R.n) {
        const int g = R.off + i, k = id[g];
        ox[base + k] = xu[g];
        oy[base + k] = yu[g];
        oz[base + k] = zu[g];
    }
    if (i == 0) ostep[(size_t)r * cfg.n_origin + o] = step;
}

// Ensemble chi4 from the per-lag accumulators, FP64 on the device: one thread
// per lag sums the listed replicas in list order (so the result does not
// depend on the launch), then Q = s/c and X4 = s2/c - s*s/(c*c) in the
// expression order of Analysis/overlap.c:114-118, chi4 = Nbar * X4 with Nbar
// the mean N of the listed replicas.  out[l] = {chi4, Q, origins}.
__global__ void k_ov_chi4(const RepC *__restrict__ reps, OvCfg cfg, const int *__restrict__ list, int nlist,
                          const double *__restrict__ sq, const double *__restrict__ sq2, const int *__restrict__ scnt,
                          double *out) {
    const int l = blockIdx.x * blockDim.x + threadIdx.x;
    if (l > cfg.n_lags) return;
    double s = 0.0, s2 = 0.0, nbar = 0.0;
    long long c = 0;
    for (int k = 0; k < nlist; k++) {
        const int r = list[k];
        const size_t a = (size_t)r * (cfg.n_lags + 1) + l;
        s += sq[a];
        s2 += sq2[a];
        c += scnt[a];
        nbar += (double)reps[r].n;
    }
    nbar /= (double)nlist;
    double q = 0.0, x4 = 0.0;
    if (c > 0) {
        const double dc = (double)c;
        q = s / dc;
        x4 = s2 / dc - s * s / (dc * dc);
    }
    out[3 * l] = nbar * x4;
    out[3 * l + 1] = q;
    out[3 * l + 2] = (double)c;
}

// Clears replica r's accumulators and origins (a slot taking a new job).
__global__ void k_ov_reset(OvCfg cfg, int r, long long *ostep, unsigned int *ocnt, double *sq, double *sq2,
                           int *scnt) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < cfg.n_origin) {
        ostep[(size_t)r * cfg.n_origin + t] = -1;
        ocnt[(size_t)r * cfg.n_origin + t] = 0u;
    }
    if (t <= cfg.n_lags) {
        const size_t a = (size_t)r * (cfg.n_lags + 1) + t;
        sq[a] = 0.0;
        sq2[a] = 0.0;
        scnt[a] = 0;
    }
}

// Reference-order export of x_u and type for in-situ analysis.
__global__ void __launch_bounds__(BLK) k_export(const RepC *__restrict__ reps, const int *__restrict__ blk_rep,
                                                const int *__restrict__ blk_first, const int *__restrict__ id,
                                                const double *__restrict__ xu, const double *__restrict__ yu,
                                                const double *__restrict__ zu, const int *__restrict__ type,
                                                double *ex, double *ey, double *ez, int *et, int r_only) {
    const int b = blockIdx.x, r = blk_rep[b];
    if (r_only >= 0 && r != r_only) return;
    const RepC R = reps[r];
    const int i = blk_first[b] + threadIdx.x;
    if (i >= R.n) return;
    const int g = R.off + i, o = R.off + id[g];
    ex[o] = xu[g]; ey[o] = yu[g]; ez[o] = zu[g]; et[o] = type[g];
}

// ---- forces
template <bool FP32>
struct PairAcc;

// a value that is the same in every lane, in scalar registers
__device__ __forceinline__ double uniform(double v) {
    return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(v)), __builtin_amdgcn_readfirstlane(__double2loint(v)));
}

// 1/a for a normal positive a: the hardware's estimate (v_rcp_f64) and two
// Newton steps, within an ulp; a fifth of the instructions of a division.
__device__ __forceinline__ double rcp_newton(double a) {
    double r = __builtin_amdgcn_rcp(a);
    r = fma(fma(-a, r, 1.0), r, r);
    return fma(fma(-a, r, 1.0), r, r);
}

template <>
struct PairAcc<false> {
    // FP64 pair terms of cell_list+forces.c:183-203.  The kernel is bound by
    // the issue of these instructions and by the gathers: the reference's
    // three divisions per pair (about 20 instructions each) are one
    // reciprocal of r^2, the constants of the two possible partner species
    // are set once per particle (a partner's are picked by one fused
    // multiply-add with its species, 0.0 or 1.0), the minimum image is d -
    // rint(d) (the same value as the reference's two tests for differences
    // of wrapped coordinates), products and sums are fused, and the force is
    // summed in box units and scaled once.  N=50000, one lane per particle:
    // 47.6 -> 29.4 us.  L*L is taken with what its rounding leaves (L2r): that
    // error is the same for all pairs and adds up where theirs cancel.  Relative
    // error of the pair energy of displaced lattices of 1000 and 50000: with L*L
    // rounded 1.8e-15 and 1.0e-15, so 3e-17 and 1.8e-16, for one instruction of
    // a pair (50000 particles 0.3 % of the step).
    double fx = 0, fy = 0, fz = 0, pe = 0, vir = 0;
    double L2, L2r;
    double rc[2], s2c[2], e4[2], e8[2], c2i[2];  // value of species 0, difference of species 1
    __device__ __forceinline__ PairAcc(int ti, const RepC &R) {
        const double l2 = R.L * R.L;  // of the workgroup's replica: in scalar registers
        L2 = uniform(l2);
        L2r = uniform(fma(R.L, R.L, -l2));
        // (ti, tj) -> ab = ti + tj: sigma {1, 0.8, 0.88}, epsilon {1, 1.5, 0.5} (cell_list+forces.c:19-20)
        const auto pick = [ti](double v0, double v1, double v2, double (&out)[2]) {
            const double a = ti ? v1 : v0;
            out[0] = a;
            out[1] = (ti ? v2 : v1) - a;
        };
        pick(K_LCUTSQR * 1.00 * 1.00, K_LCUTSQR * 0.80 * 0.80, K_LCUTSQR * 0.88 * 0.88, rc);  // (r/sigma)^2 < 6.25 (:189)
        pick(1.00 * 1.00, 0.80 * 0.80, 0.88 * 0.88, s2c);
        pick(4.0 * 1.0, 4.0 * 1.5, 4.0 * 0.5, e4);
        pick(8.0 * 1.0, 8.0 * 1.5, 8.0 * 0.5, e8);
        pick(K_C2 / (1.00 * 1.00), K_C2 / (0.80 * 0.80), K_C2 / (0.88 * 0.88), c2i);
    }
    template <int EN>
    __device__ __forceinline__ void flush() {}
    template <int EN>
    __device__ __forceinline__ void add(const double4 &pi, const double4 &pj) {
        double dx = pi.x - pj.x, dy = pi.y - pj.y, dz = pi.z - pj.z;
        dx -= rint(dx);
        dy -= rint(dy);
        dz -= rint(dz);
        const double d2 = fma(dz, dz, fma(dy, dy, dx * dx)), r2 = fma(d2, L2, d2 * L2r), tj = pj.w;
        if (r2 < fma(tj, rc[1], rc[0])) {
            const double inv = rcp_newton(r2);
            const double s2 = fma(tj, s2c[1], s2c[0]) * inv, c2 = fma(tj, c2i[1], c2i[0]);
            const double s6 = s2 * s2 * s2;
            // 4 eps [s6 (s6 - 1) + C0 + C2 (r/sigma)^2], 8 eps [6 s6 (s6 - 1/2) / r^2 - C2 / sigma^2]
            if (EN) pe = fma(fma(tj, e4[1], e4[0]), fma(s6, s6 - 1.0, fma(c2, r2, K_C0)), pe);
            const double grad = fma(tj, e8[1], e8[0]) * fma(6.0 * s6 * inv, s6 - 0.5, -c2);
            fx = fma(grad, dx, fx);
            fy = fma(grad, dy, fy);
            fz = fma(grad, dz, fz);
            if (EN) vir = fma(grad, r2, vir);
        }
    }
    __device__ __forceinline__ void result(double &ox, double &oy, double &oz, const RepC &R) const {
        ox = fx * R.L; oy = fy * R.L; oz = fz * R.L;
    }
};

template <>
struct PairAcc<true> {
    // FP32 pair forces from fixed-point positions (qpos): exact minimum
    // image in integers, separations in units of L/2^32 rounded once to FP32.
    // The cutoff test runs in those units (r^2 in units^2 against the
    // cutoff divided by the unit^2), so a candidate outside costs no scaling.
    // Each FP32 pair force term is widened to FP64 and summed there (exactly
    // the compensation a Kahan sum aims at, and on CDNA4 a widening add costs
    // two FP64 instructions against five FP32 ones); the force is scaled to
    // real units at the end.  The pair energy and virial, which only feed the
    // reported PE, pressure and Heff and never the trajectory, are summed in
    // FP32 over each group of at most 8 list entries and widened once per
    // group (flush): k_force 33.4 -> 32.1 us on the 64-replica ensemble, the
    // trajectories bit for bit the same.  The pair constants of the two possible partner
    // species are set once per particle; one hardware reciprocal of r^2
    // (v_rcp_f32, within 1 ulp) replaces the two divisions, since
    // sigma^2/r^2 = (sigma/r)^2 and 1/r^2 appears in the force factor.  The
    // pair terms are formed with fused multiply-adds (each rounds once).
    double fx = 0, fy = 0, fz = 0, pe = 0, vir = 0;
    float gpe = 0.f, gvir = 0.f;  // FP32 partials of the energy and virial of up to 8 pairs
    float sg2[2], e4[2], e8[2], rcq[2], c2i[2], qs2;
    __device__ __forceinline__ PairAcc(int ti, const RepC &R) {
        // (ti, tj) -> ab = ti + tj: sigma {1, 0.8, 0.88}, epsilon {1, 1.5, 0.5}
        // (cell_list+forces.c:19-20); what depends on the box comes from RepC
        qs2 = R.qs2;
        const auto pick = [ti](float v0, float v1, float v2, float (&out)[2]) {
            out[0] = ti ? v1 : v0;
            out[1] = ti ? v2 : v1;
        };
        pick((float)(1.00 * 1.00), (float)(0.80 * 0.80), (float)(0.88 * 0.88), sg2);
        pick(4.0f * 1.0f, 4.0f * 1.5f, 4.0f * 0.5f, e4);
        pick(8.0f * 1.0f, 8.0f * 1.5f, 8.0f * 0.5f, e8);
        pick(R.rcq[0], R.rcq[1], R.rcq[2], rcq);
        pick(R.c2i[0], R.c2i[1], R.c2i[2], c2i);
    }
    // the pair's force added up; energy(species of the partner, gradient, r^2, s^6, C2/sigma^2) within the cutoff
    template <class F>
    __device__ __forceinline__ void pair(const QPos &pi, const QPos &pj, F energy) {
        const float dx = (float)(int)(pi.x - pj.x);
        const float dy = (float)(int)(pi.y - pj.y);
        const float dz = (float)(int)(pi.z - pj.z);
        const bool b = (pj.x & 1u) != 0u;
        const float rq = __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx));  // (L/2^32)^2 units
        if (rq < (b ? rcq[1] : rcq[0])) {
            const float r2 = rq * qs2;  // real units
            const float c2 = b ? c2i[1] : c2i[0];
            const float inv = __builtin_amdgcn_rcpf(r2);
            const float s2 = (b ? sg2[1] : sg2[0]) * inv;  // (sigma/r)^2
            const float s6 = s2 * s2 * s2;
            // cell_list+forces.c:194-203: 4 eps [s6 (s6 - 1) + C0 + C2 (r/sigma)^2],
            // 8 eps [6 s6 (s6 - 1/2) / r^2 - C2 / sigma^2]
            const float grad = (b ? e8[1] : e8[0]) * __builtin_fmaf(6.0f * s6 * inv, s6 - 0.5f, -c2);
            fx += (double)(grad * dx);
            fy += (double)(grad * dy);
            fz += (double)(grad * dz);
            energy(b, grad, r2, s6, c2);
        }
    }
    __device__ __forceinline__ float pot(bool b, float r2, float s6, float c2) const {
        return (b ? e4[1] : e4[0]) * __builtin_fmaf(s6, s6 - 1.0f, __builtin_fmaf(c2, r2, (float)K_C0));
    }
    template <int EN>
    __device__ __forceinline__ void add(const QPos &pi, const QPos &pj) {
        pair(pi, pj, [&](bool b, float grad, float r2, float s6, float c2) {
            if (EN) {
                gpe += pot(b, r2, s6, c2);
                gvir = __builtin_fmaf(grad, r2, gvir);
            }
        });
    }
    // the pair's terms of the energy and the virial (a factor each of two), zero beyond the cutoff, for chain()
    __device__ __forceinline__ void add_terms(const QPos &pi, const QPos &pj, float &p, float &gr, float &rr) {
        pair(pi, pj, [&](bool b, float grad, float r2, float s6, float c2) {
            p = pot(b, r2, s6, c2);
            gr = grad;
            rr = r2;
        });
    }
    // The terms of eight entries per lane of the team, summed as the list
    // layout's team, RAT times narrower, sums them: its lane's entries of eight
    // rows in order, then widened; src[k]: the lane (times 4) that has the
    // entries of rows k, k + RAT, ...  Every lane of the team sums what its
    // layout lane does.
    template <int RAT, bool QUAD>
    __device__ __forceinline__ void chain(const float (&p)[8], const float (&gr)[8], const float (&rr)[8],
                                          const int (&src)[RAT]) {
        const auto from = [&](float v, int k) {
            const int i = __float_as_int(v);
            if (!QUAD) return __int_as_float(__builtin_amdgcn_ds_bpermute(src[k], i));
            return __int_as_float(k == 0   ? __builtin_amdgcn_update_dpp(0, i, 0x00, 0xf, 0xf, true)  // quad_perm k k k k
                                  : k == 1 ? __builtin_amdgcn_update_dpp(0, i, 0x55, 0xf, 0xf, true)
                                  : k == 2 ? __builtin_amdgcn_update_dpp(0, i, 0xaa, 0xf, 0xf, true)
                                           : __builtin_amdgcn_update_dpp(0, i, 0xff, 0xf, 0xf, true));
        };
#pragma unroll
        for (int j = 0; j < RAT; j++) {
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const int u = (8 * j + i) / RAT, k = (8 * j + i) % RAT;
                gpe += from(p[u], k);
                gvir = __builtin_fmaf(from(gr[u], k), from(rr[u], k), gvir);
            }
            flush<1>();
        }
    }
    template <int EN>
    __device__ __forceinline__ void flush() {
        if (EN) {
            pe += (double)gpe; vir += (double)gvir;
            gpe = gvir = 0.f;
        }
    }
    __device__ __forceinline__ void result(double &ox, double &oy, double &oz, const RepC &R) const {
        ox = fx * R.qscale;
        oy = fy * R.qscale;
        oz = fz * R.qscale;
    }
};

// Sum over each aligned group of 2^lw lanes (2^lw <= 16), in every lane of it:
// lane exchanges within a row of 16 (quad permutes, then mirrors of the half
// row and of the row, whose quads already agree).
template <int CTRL>
__device__ __forceinline__ double dpp_add(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, true);
    return v + __hiloint2double(hi, lo);
}
__device__ __forceinline__ double team_sum(double v, int lw) {
    if (lw > 0) v = dpp_add<0xB1>(v);   // quad_perm 1 0 3 2
    if (lw > 1) v = dpp_add<0x4E>(v);   // quad_perm 2 3 0 1
    if (lw > 2) v = dpp_add<0x141>(v);  // row_half_mirror
    if (lw > 3) v = dpp_add<0x140>(v);  // row_mirror
    return v;
}
// Sum over the wave, the same in every lane, in a fixed order: the rows of
// 16 lanes, then the four rows.
__device__ __forceinline__ double wave_sum_rows(double v) {
    v = team_sum(v, 4);
    double r[4];
#pragma unroll
    for (int k = 0; k < 4; k++)
        r[k] = __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), 16 * k),
                                __builtin_amdgcn_readlane(__double2loint(v), 16 * k));
    return (r[0] + r[1]) + (r[2] + r[3]);
}

// VEC consecutive list entries, 1 or 8.  (A nontemporal load of the list
// measured 79 against 56 us per k_force launch on the 64-replica ensemble:
// the list stream is better served by the caches.)
template <int VEC>
__device__ __forceinline__ void ld_list(const int *p, int *j) {
    if (VEC == 1) {
        j[0] = p[0];
    } else {
#pragma unroll
        for (int q = 0; q < VEC; q += 4) {
            const int4 a = *(const int4 *)(p + q);
            j[q] = a.x; j[q + 1] = a.y; j[q + 2] = a.z; j[q + 3] = a.w;
        }
    }
}

// A team's walk of particle g's list of m entries, G entries per lane and
// group: the positions of a group are gathered together while the indices of
// the next are loaded; the last, partial group has its loads issued together
// too (an entry past m is replaced by g before it is used as an index).
// VEC = 1: lane t of W takes entries t, t + W, ... (row c of the walk is
// entries c*W ... c*W + W - 1, cs list words apart); the others read chunks
// of 8 entries, cs words apart, with W = 8 / |VEC| lanes: VEC = 8 the whole
// chunk, VEC = -2 entries t, t + 4 of it, two rows per chunk.  In FP64 a group
// is six entries with VEC = -2 and four with VEC = 1: 126 and 106 vector
// registers in k_force instead of 148, four waves per SIMD instead of three (us
// per step, N=50000 50.7 -> 50.1, 80000 63.5 -> 61.4, 200000 104 -> 99.5;
// teams of 8, N=20000 29.2 -> 28.7, 30000 34.6 -> 33.6; of 16 the same).
// EN = 1: the energy's FP32 terms are summed for eight entries of the lane;
// EN = 2, 4: as the list layout's team, EN times narrower, would (2^lt lanes).
template <int VEC, int EN, class PosT, class Acc>
__device__ __forceinline__ void walk_list(const int *lp, size_t cs, int W, int lt, int t, int m, int g,
                                          const PosT *__restrict__ pos, const PosT &pi, Acc &acc) {
    constexpr int V = VEC > 1 ? VEC : 1;    // entries of a load
    constexpr int RC = VEC < 0 ? -VEC : 1;  // rows per step of cs
    constexpr bool WIDE = sizeof(PosT) == 32;                       // FP64
    constexpr int G = WIDE && VEC < 0 ? 6 : WIDE && VEC == 1 ? 4 : 8;  // entries of a group
    constexpr int NR = G / V;               // rows of a group
    const int rl = W * V, full = m / rl;    // entries of a row, whole rows
    [[maybe_unused]] int src[EN > 1 ? EN : 1];
    if constexpr (EN > 1) {
        static_assert(G == 8 && V == 1, "chain() takes eight entries of a lane");
#pragma unroll
        for (int k = 0; k < EN; k++)
            src[k] = (((int)threadIdx.x & 63 & ~(W - 1)) + (t & ((1 << lt) - 1)) + (k << lt)) * 4;
    }
    int c = 0, jn[G];
    if (NR <= full) {
#pragma unroll
        for (int r = 0; r < NR; r++) ld_list<V>(lp + (r / RC) * cs + (r % RC) * W, jn + V * r);
    }
    while (c + NR <= full) {
        PosT q[G];
#pragma unroll
        for (int u = 0; u < G; u++) q[u] = ld_pos(pos, jn[u]);
        c += NR;
        lp += (NR / RC) * cs;
        if (c + NR <= full) {
#pragma unroll
            for (int r = 0; r < NR; r++) ld_list<V>(lp + (r / RC) * cs + (r % RC) * W, jn + V * r);
        }
        if constexpr (EN > 1) {
            float p[G] = {}, gr[G] = {}, rr[G] = {};
#pragma unroll
            for (int u = 0; u < G; u++) acc.add_terms(pi, q[u], p[u], gr[u], rr[u]);
            acc.template chain<EN, (VEC < 0)>(p, gr, rr, src);
        } else {
#pragma unroll
            for (int u = 0; u < G; u++) acc.template add<EN>(pi, q[u]);
            acc.template flush<EN>();
        }
    }
    const int k0 = c * rl + t * V;  // this lane's first entry of the last group
    if (EN > 1 ? c * rl < m : k0 < m) {  // chain() takes the whole team
        int jt[G];
        PosT q[G];
#pragma unroll
        for (int r = 0; r < NR; r++) {
            int *j = jt + V * r;
            if (k0 + r * rl < m) {
                ld_list<V>(lp + (r / RC) * cs + (r % RC) * W, j);
            } else {
#pragma unroll
                for (int v = 0; v < V; v++) j[v] = g;
            }
        }
#pragma unroll
        for (int u = 0; u < G; u++) q[u] = ld_pos(pos, k0 + (u / V) * rl + u % V < m ? jt[u] : g);
        if constexpr (EN > 1) {
            float p[G] = {}, gr[G] = {}, rr[G] = {};
#pragma unroll
            for (int u = 0; u < G; u++)
                if (k0 + u * rl < m) acc.add_terms(pi, q[u], p[u], gr[u], rr[u]);
            acc.template chain<EN, (VEC < 0)>(p, gr, rr, src);
        } else {
#pragma unroll
            for (int u = 0; u < G; u++)
                if (k0 + (u / V) * rl + u % V < m) acc.template add<EN>(pi, q[u]);
            acc.template flush<EN>();
        }
    }
}

// End of the force pass for one replica, on one lane: the sums a4 = {p^2, PE,
// virial, p_x} (PE and virial with EN only) to the end-of-step chain update.
// c0: the chain as it is; eta, peta: after the start-of-step half
// (k_first_half).  EN: the pass summed the pair energy and virial (the last
// step of a call; they are only reported).  late: Heff's pair energy is added
// last, by this step or, without EN, by a pass after the call's last step
// (step, not KICK; launch_energy): the same sum either way.
template <bool KICK, bool EN>
__device__ __forceinline__ void force_end(const RepC &R, ChainS &c, const ChainS &c0, double *eta, double *peta,
                                          const double *a4, int late, int step) {
    double S = a4[0], pe = a4[1], vir = a4[2], spx = a4[3];  // pe, vir: zero without EN
    pe = 0.5 * pe;                  // every pair seen from both sides
    vir = (0.5 * vir) / (3.0e0);   // cell_list+forces.c:220
    if (EN) {
        c.pe = pe;
        c.vir = vir;
    }
    if (!KICK) {
        if (EN && step) c.heff = c.heff + pe;
        return;
    }
    const double pe0 = late ? 0.0 : pe, pe1 = late ? pe : 0.0;
    const bool rebuilt = need_rebuild(R, c0);
    if (c0.mode == 2) {
        // NVE: plain velocity Verlet (AdvanceTimeNVE, MDcode/time_evolve.c:39-171,
        // same U2-U1-F-U2 order as the thermostatted step), Heff = KE + PE
        c.p_scale = 1.0;
        c.S_end = S;
        const double ke = S * 0.5;
        c.ke = ke;
        c.inst_T = 2.0 * ke / R.dof;
        c.drift = spx;
        if (EN || late) c.heff = ke + pe0 + pe1;
        if (rebuilt) c.rebuilds = c0.rebuilds + 1;
        c.maxbits = 0ull;
        c.force_rebuild = 0;
        if (R.tau > 0 && c0.step % R.tau == 0) c.shuffles = c0.shuffles + 1;  // k_shuffle ran this step
        c.step = c0.step + 1;
        return;
    }
    if (c0.mode == 1) {
        // coldstart/breakxal of MDcode/initialise.c:166-201: momenta rescaled
        // to a ramped target temperature every step, no thermostat chain
        const double f = c0.ramp_n > 1 ? c0.ramp0 + (c0.ramp1 - c0.ramp0) * (double)c0.ramp_k / (double)(c0.ramp_n - 1)
                                       : c0.ramp1;
        const double s2 = S > 0.0 ? sqrt(R.T * f * R.dof / S) : 1.0;
        c.p_scale = s2;
        const double Se = S * s2 * s2, ke = Se * 0.5;
        c.S_end = Se;
        c.ke = ke;
        c.inst_T = 2.0 * ke / R.dof;
        c.drift = spx * s2;
        if (EN || late) c.heff = ke + pe0 + pe1;
        c.ramp_k = c0.ramp_k + 1;
        if (c0.ramp_k + 1 >= c0.ramp_n) c.mode = 0;
        if (rebuilt) c.rebuilds = c0.rebuilds + 1;
        c.maxbits = 0ull;
        c.force_rebuild = 0;
        return;
    }
    double S2;
    const double s2 = nhc_half(S, R.T, R.dof, c0.q, eta, peta, &S2);  // end of step, time_evolve.c:517-519
    for (int k = 0; k < 3; k++) { c.eta[k] = eta[k]; c.peta[k] = peta[k]; }
    const double ke = S2 * 0.5;      // time_evolve.c:520
    c.S_end = S2;
    c.p_scale = s2;
    c.ke = ke;
    c.inst_T = 2.0 * ke / R.dof;     // :524
    c.drift = spx * s2;
    if (EN || late) {
        double heff = ke + pe0 + eta[0] * R.T * R.dof;  // print.c:85-87
        for (int k = 0; k < 3; k++) heff = heff + peta[k] * peta[k] / (2.0 * c0.q[k]);
        for (int k = 1; k < 3; k++) heff = heff + R.T * eta[k];
        c.heff = heff + pe1;
    }
    if (rebuilt) c.rebuilds = c0.rebuilds + 1;
    c.maxbits = 0ull;
    c.force_rebuild = 0;
    if (R.tau > 0 && c0.step % R.tau == 0) c.shuffles = c0.shuffles + 1;  // k_shuffle ran this step
    c.step = c0.step + 1;
}

// What k_force's last workgroups need: the chains, the chain variables after
// the start-of-step half, the partial sums of groups of FORCE_GRP blocks and
// the counts of finished blocks of each group and groups of each replica.
#define FORCE_GRP 64
struct EndArgs {
    ChainS *chain;
    const double *mid;
    double *gpart;
    unsigned *gdone, *rdone;
    int late, step;  // force_end
};

// Pair forces: a team of W = 2^lw lanes per particle (fixed per handle at
// creation, so a replica's results do not depend on what else is loaded)
// walks the particle's list (walk_list); the team's partial forces are
// combined by a fixed butterfly.  Each block hands over its partial sums of
// p^2 and p_x, and with EN of PE and virial; the last block of each FORCE_GRP
// adds theirs up (lane k block k, a fixed butterfly), the replica's last group
// adds the groups' in a fixed order and updates the chain (force_end).  Two
// levels: atomics on one line are done one after the other.  As a kernel of
// their own after this one, sums and update took 3.5 us of N=1000's step, 5.1
// of N=50000's and 11.4 of N=1e6's; with them, and the scan of the cell
// counts, inside: 19.7 -> 17.3 us per graph step at N=1000 FP64, 22.9 -> 20.8
// at 10000 FP32, 65.8 -> 62.0 on the 64-replica ensemble, 359 -> 349 at 1e6.
// A block's loads form a short chain (block table, then position, list
// length, active index and momentum together, then list, then neighbour
// positions): on small boxes, a few waves per CU, the launch is as
// long as that chain.  Each loaded where it was used, with the constants
// divided out per lane and the sums shuffled through LDS: 7.2 us at N=1000
// FP64 and 11.0 at N=10000 FP32 (four lanes); this 5.9 and 7.0 (sixteen).
// EN = 0 leaves out the pair energy and virial, which every step overwrites
// and only the call's last one reports: 9 of 55 instructions of an FP32 pair.
// FP32 handles whose team is 2 or 4 times the list layout's take EN = 2 or 4,
// which sums the FP32 terms of eight entries as the layout's team does, so that
// the partial sums, whose rounding shows in the seventh to ninth digit of the
// energy, do not depend on the force team's width (walk_list): four to five
// tenths more of the pass (18.3 -> 25.1 us at 50000, 162 -> 239 at 1e6).  us of
// a call of one step, 8000, 160001 and 500000 particles: with the energy in two
// kernels of its own after it 32.6, 156 and 292, this 27.6, 140 and 254.
template <bool FP32, bool KICK, int EN, int VEC>
__global__ void __launch_bounds__(BLK) k_force(const RepC *__restrict__ reps, const BlkD *__restrict__ fblk,
                                               const double4 *__restrict__ pos4, const QPos *__restrict__ posq,
                                               const int *__restrict__ nn,
                                               const int *__restrict__ nl, int cap, int lw, int lc, int lt,
                                               const int *__restrict__ act,
                                               const int8_t *__restrict__ kx, const int8_t *__restrict__ ky,
                                               const int8_t *__restrict__ kz, double *fx, double *fy, double *fz,
                                               double *px, double *py, double *pz, double *partial, int nb,
                                               EndArgs E) {
    static_assert(BLK == 256, "four waves per block");
    __shared__ double s_red[4][BLK / 64];
    const int b = xcd_block(nb);
    if (b < 0) return;
    const BlkD D = fblk[b];
    const int W = 1 << lw, t = threadIdx.x & (W - 1);
    const int i = D.first + (threadIdx.x >> lw);
    double v_p2 = 0.0, v_pe = 0.0, v_vir = 0.0, v_px = 0.0;
    double Fx = 0.0, Fy = 0.0, Fz = 0.0;
    const bool valid = i < D.n;
    const int g = D.off + (valid ? i : 0);
    // FP64: the wrapped box fractions; FP32: their fixed-point copy
    using PosT = typename std::conditional<FP32, QPos, double4>::type;
    const PosT *__restrict__ pos = (const PosT *)(FP32 ? (const void *)posq : (const void *)pos4);
    const PosT pi = ld_pos(pos, g);
    const int m = valid ? nn[g] : 0;
    const int a = act[g];
    double vx = 0.0, vy = 0.0, vz = 0.0;
    if (KICK) { vx = px[g]; vy = py[g]; vz = pz[g]; }
    const RepC &R = reps[D.rep];
    const bool active = a >= 0;
    const int ka = R.off_act + (active ? a : 0);
    const double kfx = (double)kx[ka], kfy = (double)ky[ka], kfz = (double)kz[ka];
    PairAcc<FP32> acc(ptype(pi), R);
    // entry e of particle i's list (nl_at): VEC = 1, W >= 2^lc, rows of W
    // entries are W * n words apart; else the chunks of 8 entries, 8 * n
    const size_t e0 = (size_t)(VEC > 1 ? t * VEC : t);
    const int *lp = nl + (size_t)D.off * cap + ((((e0 >> lc) * D.n + (g - D.off)) << lc) + (e0 & ((1u << lc) - 1u)));
    walk_list<VEC, EN>(lp, (size_t)D.n * (VEC == 1 ? W : 8), W, lt, t, m, g, pos, pi, acc);
    acc.result(Fx, Fy, Fz, R);
    if (EN <= 1 || t >> lt == 0) {  // EN > 1: the layout's lanes
        v_pe = acc.pe;
        v_vir = acc.vir;
    }
    Fx = team_sum(Fx, lw);
    Fy = team_sum(Fy, lw);
    Fz = team_sum(Fz, lw);
    if (valid && t == 0) {
        if (active) {  // cell_list+forces.c:207-213
            Fx += R.f0 * kfx;
            Fy += R.f0 * kfy;
            Fz += R.f0 * kfz;
        }
        fx[g] = Fx; fy[g] = Fy; fz[g] = Fz;
        if (KICK) {  // U2 after the forces, time_evolve.c:516
            vx += Fx * K_HALF_DT; vy += Fy * K_HALF_DT; vz += Fz * K_HALF_DT;
            px[g] = vx; py[g] = vy; pz[g] = vz;
            v_p2 = vx * vx + vy * vy + vz * vz;
            v_px = vx;
        }
    }
    const double v[4] = {v_p2, v_pe, v_vir, v_px};
#pragma unroll
    for (int q = 0; q < 4; q++) {
        if (!EN && (q == 1 || q == 2)) continue;
        const double w = wave_sum_rows(v[q]);
        if ((threadIdx.x & 63) == 0) s_red[q][threadIdx.x >> 6] = w;
    }
    __syncthreads();
    if (threadIdx.x >= 64) return;
    const int lane = threadIdx.x, fb = b - R.fblk_off, gr = fb / FORCE_GRP;
    const int ngr = (R.fnblk + FORCE_GRP - 1) / FORCE_GRP, gsz = min(FORCE_GRP, R.fnblk - gr * FORCE_GRP);
    const bool mine = lane < 4 && (EN || lane == 0 || lane == 3);  // lane q: sum q
    if (mine) {
        const double *w = s_red[lane];
        st_agent(partial + 4 * (size_t)b + lane, (w[0] + w[1]) + (w[2] + w[3]));
    }
    wait_stores();
    int last = 0;
    if (lane == 0) last = last_done(E.gdone + R.fblk_off + gr * FORCE_GRP, gsz);
    if (!__builtin_amdgcn_readfirstlane(last)) return;
    double a4[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int q = 0; q < 4; q++)
        if (EN || q == 0 || q == 3)
            a4[q] = lane < gsz ? ld_agent(partial + 4 * (size_t)(R.fblk_off + gr * FORCE_GRP + lane) + q) : 0.0;
#pragma unroll
    for (int q = 0; q < 4; q++)
        if (EN || q == 0 || q == 3) a4[q] = wave_sum_rows(a4[q]);
    if (ngr > 1) {
        double *gp = E.gpart + 4 * (size_t)R.fblk_off;
        if (mine) st_agent(gp + 4 * gr + lane, lane == 0 ? a4[0] : (lane == 1 ? a4[1] : (lane == 2 ? a4[2] : a4[3])));
        wait_stores();
        last = 0;
        if (lane == 0) last = last_done(E.rdone + D.rep * DONE_PAD, ngr);
        if (!__builtin_amdgcn_readfirstlane(last)) return;
        // lane k groups k, k + 64, ..., then the butterfly: groups past the
        // particles add zeros, so the slot's capacity does not show in the sums
        for (int q = 0; q < 4; q++) a4[q] = 0.0;
        for (int k = lane; k < ngr; k += 64)
#pragma unroll
            for (int q = 0; q < 4; q++)
                if (EN || q == 0 || q == 3) a4[q] += ld_agent(gp + 4 * k + q);
#pragma unroll
        for (int q = 0; q < 4; q++)
            if (EN || q == 0 || q == 3) a4[q] = wave_sum_rows(a4[q]);
    }
    if (lane == 0) {
        ChainS c0;
        double eta[3], peta[3];
        if (KICK) {
            c0 = E.chain[D.rep];
            for (int k = 0; k < 3; k++) { eta[k] = E.mid[6 * D.rep + k]; peta[k] = E.mid[6 * D.rep + 3 + k]; }
        }
        force_end<KICK, EN != 0>(R, E.chain[D.rep], c0, eta, peta, a4, E.late, E.step);
    }
}

// ------------------------------------------------------------- host side
struct ac4_md {
    int R = 0, prec = 0, ntot = 0, nblk = 0, ncell_tot = 0, nact_tot = 0, cap = 192, stride = 0, max_ncell = 0;
    std::vector<RepC> reps_h;
    RepC *reps = nullptr;
    ChainS *chain = nullptr;
    int *blk_rep = nullptr, *blk_first = nullptr, *blk_idx = nullptr;
    BlkD *blkd = nullptr, *fblk = nullptr;  // particle blocks (k_first_half) and force blocks
    int en = 1, lt = 0;  // the energy's order (k_force's EN), log2 of the list layout's lanes per particle
    int lw = 0, lc = 3, vec = 1;  // force teams: log2 lanes, log2 list chunk, list reading (k_force's VEC)
    int *cblk_rep = nullptr, *cblk_cell = nullptr;
    int fnblk = 0, lnblk = 0, ncb = 0;
    int shuf_kmax = 0;     // room for directions in LDS (bytes), at most
    int shuf_kcap = 0;     // largest Nact whose directions the shuffle keeps in LDS
    int shuf_bmax = 0;     // swap blocks of the largest slot, 0 without the parallel shuffle path
    int2 *shuf_ent = nullptr;  // its per-block source maps
    int *shuf_ent_n = nullptr;
    size_t shuf_lds = 0;   // dynamic LDS of k_shuffle
    // by the jobs in the slots (job_rules): the shuffle runs in k_first_half's
    // first workgroups; else k_shuffle, the parallel path or both are launched;
    // the scan of the cell counts is k_bin's
    bool shuf_fused = false, shuf_serial = true, shuf_par = false, bin_fuse = false;
    int *wl_item = nullptr, *wl_n = nullptr;  // rebuild work list (WorkList)
    int2 *ranges = nullptr;                    // per cell: stencil slot ranges (NRANGE)
    int *xmid = nullptr;                       // per cell: first slot of its upper x-half
    int *lblk_rep = nullptr, *lblk_first = nullptr;  // list-build block table (LPB particles per block)
    double *partial = nullptr;
    double *gpart = nullptr;                             // EndArgs
    unsigned *gdone = nullptr, *rdone = nullptr, *bdone = nullptr;  // finished blocks and groups (EndArgs), blocks of k_bin
    double *mid = nullptr;  // per replica: the chain's eta, p_eta after the start-of-step half
    PartArrays P{}, A{};  // primary and permutation scratch
    void **ftab = nullptr;  // their pointers on the device (PART_FIELDS of P, then of A)
    double *fx = nullptr, *fy = nullptr, *fz = nullptr, *xo = nullptr, *yo = nullptr, *zo = nullptr;
    double4 *pos4 = nullptr;
    QPos *posq = nullptr;
    int2 *cell_mem = nullptr;  // per cell: CELL_CAP (slot, key) of its members in binning order
    int *nn = nullptr, *nn_ref = nullptr, *nl = nullptr, *cnt = nullptr, *start = nullptr, *members = nullptr;
    int8_t *kx = nullptr, *ky = nullptr, *kz = nullptr;
    double *ex = nullptr, *ey = nullptr, *ez = nullptr;  // reference-order export
    // in-situ overlap accumulators
    OvCfg ov{0, 0, 0, 0, 0.0};
    double *ox = nullptr, *oy = nullptr, *oz = nullptr, *ov_q = nullptr, *ov_q2 = nullptr;
    long long *ov_step = nullptr;
    std::vector<char> tables;  // refresh_tables' copy of the block tables and reps
    char *mem = nullptr;       // the arrays of each_array
    int *ov_list = nullptr;     // replica list of ac4_md_overlap_chi4
    double *ov_out = nullptr;   // its per-lag results
    // frame text (ac4_md_format_frame): a slot of 80 bytes per line in
    // reference order and its length, the bytes of each block of lines, and in
    // pinned memory two pieces of the joined text (one for a frame of one
    // piece) and the words k_fmt_* leave for the host
    char *fmt_dev = nullptr, *fmt_txt = nullptr;
    unsigned char *fmt_len_dev = nullptr;
    int *fmt_bsum = nullptr;
    long long *fmt_meta = nullptr;  // [0, 1]: bytes of a piece, [2]: a value for the host's formatter
    hipEvent_t fmt_ev[2] = {nullptr, nullptr};
    size_t fmt_cap = 0;
    unsigned int *ov_cnt = nullptr;
    int *ov_n = nullptr;
    int *et = nullptr;
    hipStream_t stream = nullptr;
    // recorded steps: [0] one step, [1] GRAPH_CHUNK steps in one graph
    hipGraphExec_t gexec[2] = {nullptr, nullptr};
    int eager = 0;  // steps ac4_md_step launched one by one since the graphs were last dropped
    hipGraph_t graph[2] = {nullptr, nullptr};
    hipGraph_t rec = nullptr;  // the graph that put() adds its launches to, or null
    hipGraphNode_t rec_end = nullptr;
    hipError_t rec_err = hipSuccess;
    bool have_forces = false;
    int nlist_mode = 0;
};

#define TRY(e) do { int rc_ = (e); if (rc_ != AC4_OK) return rc_; } while (0)

template <class T>
static int dalloc(T **p, size_t n) {
    if (n == 0) n = 1;
    AC4_HIP(hipMalloc((void **)p, n * sizeof(T)));
    AC4_HIP(hipMemset(*p, 0, n * sizeof(T)));
    return AC4_OK;
}

template <class F>
static int each_part(PartArrays &a, size_t n, F get) {
    for (double **q : {&a.x, &a.y, &a.z, &a.xu, &a.yu, &a.zu, &a.px, &a.py, &a.pz}) TRY(get(q, n));
    for (int **q : {&a.type, &a.act, &a.id, &a.cell_ref, &a.cell_of}) TRY(get(q, n));
    return AC4_OK;
}

// What slots add up to, and the device arrays a handle of that many has: the
// list creation allocates and ac4_md_slot_bytes adds up, get(&array, count).
// First what refresh_tables writes, blk_rep to reps.
struct SlotCounts {
    size_t slots, n, cells, nblk, fnblk, lnblk, ncb;  // particles, cells, blocks of each kind
    size_t shuf;                                      // swap blocks of the parallel shuffle, 0 without it
};
template <class F>
static int each_array(ac4_md *md, const SlotCounts &k, F get) {
    TRY(get(&md->blk_rep, k.nblk)); TRY(get(&md->blk_first, k.nblk)); TRY(get(&md->blk_idx, k.nblk));
    TRY(get(&md->blkd, k.nblk)); TRY(get(&md->fblk, k.fnblk));
    TRY(get(&md->lblk_rep, k.lnblk)); TRY(get(&md->lblk_first, k.lnblk));
    TRY(get(&md->reps, k.slots)); TRY(get(&md->chain, k.slots)); TRY(get(&md->mid, 6 * k.slots));
    if (k.shuf) { TRY(get(&md->shuf_ent, k.shuf * 2 * SHUF_M)); TRY(get(&md->shuf_ent_n, k.shuf)); }
    TRY(get(&md->wl_item, k.nblk + k.lnblk + k.ncb)); TRY(get(&md->wl_n, (size_t)4));
    TRY(get(&md->ranges, k.cells * NRANGE)); TRY(get(&md->xmid, k.cells));
    TRY(get(&md->cblk_rep, k.cells)); TRY(get(&md->cblk_cell, k.cells));
    TRY(get(&md->cell_mem, k.cells * CELL_CAP)); TRY(get(&md->cnt, k.cells)); TRY(get(&md->start, k.cells));
    TRY(get(&md->partial, 4 * k.fnblk)); TRY(get(&md->gpart, 4 * k.fnblk)); TRY(get(&md->gdone, k.fnblk));
    TRY(get(&md->rdone, k.slots * DONE_PAD)); TRY(get(&md->bdone, k.slots * DONE_PAD));
    for (double **q : {&md->fx, &md->fy, &md->fz, &md->xo, &md->yo, &md->zo}) TRY(get(q, k.n));
    TRY(get(&md->pos4, k.n)); TRY(get(&md->posq, k.n));
    TRY(get(&md->nn, k.n)); TRY(get(&md->nn_ref, k.n)); TRY(get(&md->nl, md->cap * k.n)); TRY(get(&md->members, k.n));
    TRY(get(&md->kx, k.n)); TRY(get(&md->ky, k.n)); TRY(get(&md->kz, k.n));  // n_act is n at most
    TRY(each_part(md->P, k.n, get)); TRY(each_part(md->A, k.n, get));
    return get(&md->ftab, (size_t)2 * PART_FIELDS);
}
// those of the reference-order export and of the overlap accumulators
template <class F>
static int each_export_array(ac4_md *md, size_t n, F get) {
    TRY(get(&md->ex, n)); TRY(get(&md->ey, n)); TRY(get(&md->ez, n));
    return get(&md->et, n);
}
template <class F>
static int each_overlap_array(ac4_md *md, size_t slots, size_t n, size_t n_origin, size_t n_lags, F get) {
    for (double **q : {&md->ox, &md->oy, &md->oz}) TRY(get(q, n * n_origin));
    TRY(get(&md->ov_q, slots * (n_lags + 1))); TRY(get(&md->ov_q2, slots * (n_lags + 1)));
    TRY(get(&md->ov_n, slots * (n_lags + 1)));
    TRY(get(&md->ov_cnt, slots * n_origin)); TRY(get(&md->ov_step, slots * n_origin));
    TRY(get(&md->ov_list, slots));
    return get(&md->ov_out, 3 * (n_lags + 1));
}
static const auto alloc_array = [](auto **p, size_t n) { return dalloc(p, n); };

// each_array's arrays in one allocation, zeroed: small ones at whole pages,
// those of 2 MiB and more at multiples of that, as allocations of their own lie.
// (An allocation and a fill for each of 65 arrays: 20 slots of 2000 particles
// 1.57 ms to create and destroy, this 0.76.)
static int alloc_arrays(ac4_md *md, const SlotCounts &k) {
    size_t total = 0;
    const auto place = [&](size_t bytes) {
        const size_t to = bytes >= (2u << 20) ? 2u << 20 : 4096;
        const size_t at = (total + to - 1) / to * to;
        total = at + std::max<size_t>(bytes, 1);
        return at;
    };
    TRY(each_array(md, k, [&](auto **p, size_t n) {
        (void)place(sizeof(**p) * n);
        return AC4_OK;
    }));
    AC4_HIP(hipMalloc((void **)&md->mem, total));
    AC4_HIP(hipMemset(md->mem, 0, total));
    total = 0;
    return each_array(md, k, [&](auto **p, size_t n) {
        *(void **)p = md->mem + place(sizeof(**p) * n);
        return AC4_OK;
    });
}

// Kernel shape of handles created afterwards.  tpp: lanes per particle in
// the force kernel and of the list's layout, 1..16, or 0 = automatic (the
// layout the widest with at most TPP_LANES lanes over the handle's total
// capacity, the force team at least force_width of it).  The team
// width fixes the order of each particle's force sum, so results are bitwise
// reproducible for a given handle shape.  nlist_mode: dynamics list builder,
// 0 = one wave per cell, 1 = one thread per particle, 2/3/4 = teams of
// 16/32/64 lanes per particle.
#define TPP_LANES 65536.0

// Lanes per particle of the force kernel where they are not pinned, by the
// handle's total capacity: enough waves to hide the gathers on small handles,
// few enough that a particle's constants and sums are not paid for by too
// many lanes.  us per graph-replayed step of one box, at 1 / 2 / 4 / 8 / 16
// lanes (each with the list layout of that width):
//   FP32  10000: 32.8 28.7 24.5 23.2 22.6    20000: 41.0 36.3 33.2 32.2 32.5
//         50000: 49.2 47.7 45.7 45.4 48.4   100000: 64.5 64.9 63.6 64.5 71.9
//        200000: 92.3 86.7 85.5 91.4  106   500000:  210  200  202  222  270
//   FP64  10000: 39.9 30.5 25.5 24.5 23.7    20000: 47.8 38.1 35.7 33.7 35.1
//         50000: 56.6 52.1 51.2 51.9 56.6   100000: 79.7 75.9 72.0 78.3 87.2
//        200000:  121  113  106  121  143   500000:  288  252  252  292  361
// Four FP32 lanes reading a chunk's entries strided (k_force, VEC = -2) take
// 177.6 at 500000, 118.7 at 300000 and 44.6 at 70000; reading two consecutive
// ones 181.6, 122.5 and 45.4; eight lanes 194.9, 127.2 and 45.4.  The lines lie
// where the automatic list layout changes (TPP_LANES), so that handles between
// which a checkpoint can move, those of one layout, have one force width and
// the restored replica goes on bit for bit (14500 and 16000 particles at 8 and
// 16 lanes: FP32 22.4 and 22.1, 22.5 and 22.9; FP64 23.5 and 24.0, 24.1 and 24.4).
static int force_width(double cap_tot) {
    if (cap_tot <= 16384.0) return 16;
    if (cap_tot <= 32768.0) return 8;
    return 4;
}
static int g_tpp = 0, g_nlist_mode = 3;
static double g_skin = K_SKIN;

// Verlet skin of handles created afterwards (0.2 ... 0.6; the reference's is
// 0.35).  A larger skin rebuilds less often and gives longer lists.
extern "C" int ac4_set_skin(double skin) {
    AC4_REQUIRE(skin >= 0.2 && skin <= 0.6, AC4_EARG, "ac4_set_skin: skin must be in [0.2, 0.6]");
    g_skin = skin;
    return AC4_OK;
}

extern "C" int ac4_set_tuning(int tpp, int nlist_mode) {
    AC4_REQUIRE((tpp == 0 || tpp == 1 || tpp == 2 || tpp == 4 || tpp == 8 || tpp == 16) &&
                    (nlist_mode >= 0 && nlist_mode <= 4),
                AC4_EARG, "ac4_set_tuning: tpp in {0,1,2,4,8,16}, nlist_mode in {0,...,4}");
    g_tpp = tpp;
    g_nlist_mode = nlist_mode;
    return AC4_OK;
}

// Launch rules that follow the jobs in the slots (the capacities while no slot
// holds one): the shuffle is k_first_half's when no job needs the parallel
// path and its LDS leaves that kernel at least 5 workgroups per CU; a launch
// that no job needs is left out (each costs 1.6 to 4.5 us a step even where it
// returns at once: N=50000, whose slot could hold 50000 active particles and
// holds 5000, took three for the shuffle and one for the scan; 1e6 one).
static void job_rules(ac4_md *md) {
    bool any = false, small = false, large = false;
    int k = 0, ncell = 0;
    for (const RepC &R : md->reps_h) any |= R.n > 0;
    for (const RepC &R : md->reps_h) {
        if (any && R.n == 0) continue;
        const int na = any ? R.nact : R.cap_n;
        k = std::max(k, na);
        ncell = std::max(ncell, any ? R.ncell : R.cap_cells);
        (md->shuf_bmax > 0 && na > SHUF_PAR_MIN ? large : small) = true;
    }
    md->shuf_kcap = std::min(md->shuf_kmax, (k + 15) & ~15);
    md->shuf_lds = SHUF_CH * sizeof(unsigned int) + (size_t)md->shuf_kcap;
    md->shuf_serial = small || !any;
    md->shuf_par = md->shuf_bmax > 0 && (large || !any);
    md->shuf_fused = !md->shuf_par && md->shuf_lds <= 32768;
    md->bin_fuse = ncell <= BIN_FUSE_CELLS;
}

// Job-dependent fields of a slot (the capacity-dependent ones are fixed at
// creation).  Returns 0 or an error message.
static const char *configure_rep(RepC &R, const ac4_replica_params &q) {
    if (q.n < 2 || !(q.density > 0) || !(q.T > 0)) return "bad n/density/T";
    if (q.n > R.cap_n) return "n exceeds the slot capacity";
    const int nact = q.n_act < 0 ? (int)((double)q.n * 0.1000) : q.n_act;
    if (nact > q.n) return "n_act larger than n";
    const double L = pow((double)q.n / q.density, 0.33333333);  // MDcode/main.c:465
    const double cell_cut = std::max(K_CELL_CUT, 2.5 + R.skin);  // a cell spans the largest list radius
    if (L <= 2.0 * cell_cut) return "box too small for the list cutoff";
    R.n = q.n;
    R.nact = nact;
    R.L = L;
    R.invL = 1.0 / R.L;  // :466
    // MDcode/Parallel.c:72-80 with one process (Lpp = L): the reference grid
    const double Lpp = R.L / (double)1;
    R.nc_ref = (int)((double)((int)Lpp) / K_CELL_CUT);
    if (R.nc_ref < 1) R.nc_ref = 1;
    R.inv_cell_ref = R.L / (Lpp / (double)R.nc_ref);
    R.nc = (int)(R.L / cell_cut);  // list grid: cells at least one list radius (and 2.85) wide
    // A particle in the upper (lower) x-half of its cell is at least one cell
    // width from the lower (upper) x-half of the cell below (above) it along
    // x, for any grid of three or more cells: beyond every list radius and the
    // screen's margin once the width exceeds the largest radius by 0.01 sigma.
    R.xcull = R.nc >= 3 && R.L / R.nc >= 2.5 + R.skin + 0.01;
    R.ncell = R.nc * R.nc * R.nc;
    if (R.ncell > R.cap_cells) return "density below the slot's cell capacity (0.5)";
    R.qscale = R.L / 4294967296.0;
    R.qs2 = (float)(R.qscale * R.qscale);
    R.rnc = 1.0f / (float)R.nc;
    R.cell = (float)(R.L / R.nc);
    R.fix2cell = (float)(R.nc / 4294967296.0);
    R.lr2[0] = (float)(list_cut2(0, R.skin) + 2e-3);
    R.lr2[1] = (float)(list_cut2(2, R.skin) + 2e-3);
    for (int ab = 0; ab < 3; ab++) {  // cutoff (r/sigma)^2 < 6.25 (cell_list+forces.c:189)
        const double sig = ab == 0 ? 1.00 : (ab == 1 ? 0.80 : 0.88);
        R.lcut[ab] = qscreen_cut_of(ab, R.skin, R.qs2);
        R.rcq[ab] = (float)(K_LCUTSQR * sig * sig / (double)R.qs2);
        R.c2i[ab] = (float)(K_C2 / (sig * sig));
    }
    R.tau = q.tau_per;
    R.T = q.T;
    R.f0 = q.f0;
    R.density = q.density;
    R.dof = 3.0 * (double)q.n - 3.0;  // global.h:35
    R.key0 = (uint32_t)q.seed;
    R.key1 = (uint32_t)(q.seed >> 32);
    return nullptr;
}

static void fresh_chain(ChainS &c, const RepC &R) {
    memset(&c, 0, sizeof(ChainS));
    const double tau = .20, T = R.T;  // time_evolve.c:477-482
    for (int k = 0; k < 3; k++) c.q[k] = T * tau * tau;
    c.q[0] = R.dof * T * tau * tau;
    c.p_scale = 1.0;
    c.force_rebuild = R.n > 0 ? 1 : 0;
}

static int refresh_tables(ac4_md *md);

// cells a slot of capacity cn can hold: those of the least dense box (rho 0.5)
static int slot_cells(int cn) { return (int)pow((int)(pow((double)cn / 0.5, 1.0 / 3.0) / K_CELL_CUT) + 1, 3); }

// cap_rule > 0: the automatic force team width is taken for that total
// capacity instead of the handle's own (a server's launch groups share one
// kernel shape, so a job's arithmetic does not depend on its group)
extern "C" int ac4_md_create_slots_rule(int nslots, const int *cap_n, int precision, double cap_rule,
                                        ac4_md **out);
extern "C" int ac4_md_create_slots(int nslots, const int *cap_n, int precision, ac4_md **out) {
    return ac4_md_create_slots_rule(nslots, cap_n, precision, 0.0, out);
}
extern "C" int ac4_md_create_slots_rule(int nslots, const int *cap_n, int precision, double cap_rule,
                                        ac4_md **out) {
    AC4_REQUIRE(nslots >= 1 && cap_n && out, AC4_EARG, "ac4_md_create_slots: bad arguments");
    AC4_REQUIRE(precision == AC4_FP64 || precision == AC4_FP32, AC4_EARG, "precision must be 0 or 1");
    int ndev = 0;
    AC4_REQUIRE(hipGetDeviceCount(&ndev) == hipSuccess && ndev > 0, AC4_EHIP,
                "ac4_md_create: no HIP device visible (libac4 has no CPU path)");
    ac4_md *md = new ac4_md();
    md->R = nslots;
    md->prec = precision;
    md->nlist_mode = g_nlist_mode;
    int off = 0, off_act = 0, off_cell = 0, blk_off = 0, fblk_off = 0, lblk_off = 0;
    std::vector<int> crep, ccell;
    int ncb = 0;
    AC4_REQUIRE(nslots < 32768, AC4_EARG, "at most 32767 slots");
    double cap_tot = 0.0;
    for (int r = 0; r < nslots; r++) cap_tot += cap_n[r] > 0 ? cap_n[r] : 0;
    int tpp = g_tpp, ltpp = 0;
    if (cap_rule > 0.0) cap_tot = cap_rule;
    if (tpp == 0) {
        tpp = 1;
        while (tpp < 16 && cap_tot * tpp * 2 <= TPP_LANES) tpp *= 2;
    }
    while ((1 << ltpp) < tpp) ltpp++;
    // lanes per particle in the force kernel: the pinned width, else by the
    // handle's total capacity
    const int W = g_tpp ? tpp : std::max(tpp > 1 ? tpp : 1, force_width(cap_tot));
    while ((1 << md->lw) < W) md->lw++;
    md->lt = ltpp;
    md->en = precision == AC4_FP32 ? W / tpp : 1;  // force_width and the layout's rule: 1, 2 or 4
    md->lc = tpp == 1 ? 3 : ltpp;
    // a chunk of 8 entries read by four lanes: every fourth entry each, so
    // that the lanes of a gather are on neighbouring entries, which are mostly
    // neighbouring slots: two consecutive entries each make the gathers of a
    // wave reach more lines (us per step, FP64 N=100000 72 against 79, FP32
    // N=1e6 343 against 352); one lane takes all 8
    md->vec = W < (1 << md->lc) ? (W > 1 ? -((1 << md->lc) / W) : 8) : 1;
    for (int r = 0; r < nslots; r++) {
        RepC R;
        memset(&R, 0, sizeof R);
        const int cn = cap_n[r];
        if (cn < 2) { delete md; ac4_set_error("slot %d: capacity %d < 2", r, cn); return AC4_EARG; }
        // the cell sort's keys hold ids below 2^21, list addressing uses 24-bit products with n
        if (cn > (1 << 21)) { delete md; ac4_set_error("slot %d: capacity %d > 2^21", r, cn); return AC4_EARG; }
        R.cap_n = cn;
        R.skin = g_skin;
        R.off = off;
        R.off_act = off_act;
        R.off_cell = off_cell;
        const int cap_cells = slot_cells(cn);
        R.cap_cells = cap_cells;
        R.tpp = tpp;
        R.ltpp = ltpp;
        R.lc = tpp == 1 ? 3 : ltpp;
        R.nblk = (cn + BLK - 1) / BLK;
        R.blk_off = blk_off;
        const int ppb = BLK / W;  // particles per force block
        R.fnblk = (cn + ppb - 1) / ppb;
        R.fblk_off = fblk_off;
        R.lblk_off = lblk_off;
        R.lnblk = (cn + LPB - 1) / LPB;
        if ((cap_cells + BLK / 64 - 1) / (BLK / 64) >= 65536) { delete md; ac4_set_error("slot %d: too many cells", r); return AC4_EARG; }
        ncb += (cap_cells + BLK / 64 - 1) / (BLK / 64);
        for (int c = 0; c < cap_cells; c++) { crep.push_back(r); ccell.push_back(c); }
        off += cn;
        off_act += cn;  // room for n_act up to n
        off_cell += cap_cells;
        blk_off += R.nblk;
        fblk_off += R.fnblk;
        lblk_off += R.lnblk;
        md->max_ncell = std::max(md->max_ncell, cap_cells);
        md->reps_h.push_back(R);  // idle: n = 0
    }
    md->ntot = off;
    md->nact_tot = off_act;
    md->ncell_tot = off_cell;
    md->nblk = blk_off;
    md->stride = off;
    md->fnblk = fblk_off;
    md->lnblk = lblk_off;
    md->ncb = ncb;
    {  // k_shuffle: the partner chunk plus one component in LDS when it fits
        int dev = 0, lds = 65536, cap_max = 0;
        (void)hipGetDevice(&dev);
        if (hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess) lds = 65536;
        for (int r = 0; r < nslots; r++) cap_max = std::max(cap_max, cap_n[r]);
        const int room = lds - (int)(SHUF_CH * sizeof(unsigned int));
        md->shuf_kmax = std::max(0, std::min(room, (cap_max + 15) & ~15));
        md->shuf_lds = SHUF_CH * sizeof(unsigned int) + (size_t)md->shuf_kmax;
        if (md->shuf_lds > 65536 &&
            (hipFuncSetAttribute((const void *)k_shuffle, hipFuncAttributeMaxDynamicSharedMemorySize,
                                 (int)md->shuf_lds) != hipSuccess ||
             hipFuncSetAttribute((const void *)k_shuf_apply, hipFuncAttributeMaxDynamicSharedMemorySize,
                                 (int)md->shuf_lds) != hipSuccess)) {
            (void)hipGetLastError();
            md->shuf_kmax = 65536 - (int)(SHUF_CH * sizeof(unsigned int));
        }
        md->shuf_bmax = cap_max > SHUF_PAR_MIN ? (cap_max + SHUF_M - 1) / SHUF_M : 0;
    }
    job_rules(md);
    int rc = AC4_OK;
    const SlotCounts counts{(size_t)nslots, (size_t)off, (size_t)off_cell, (size_t)md->nblk, (size_t)md->fnblk,
                            (size_t)md->lnblk, (size_t)md->ncb, (size_t)nslots * 3 * md->shuf_bmax};
    if ((rc = alloc_arrays(md, counts)) != AC4_OK) { ac4_md_destroy(md); return rc; }
    {
        void *tab[2 * PART_FIELDS];
        for (int k = 0; k < 2; k++) {
            const PartArrays &a = k ? md->A : md->P;
            void *f[PART_FIELDS] = {a.x, a.y, a.z, a.xu, a.yu, a.zu, a.px, a.py, a.pz,
                                    a.type, a.act, a.id, a.cell_ref, a.cell_of};
            for (int q = 0; q < PART_FIELDS; q++) tab[k * PART_FIELDS + q] = f[q];
        }
        if (hipMemcpy(md->ftab, tab, sizeof tab, hipMemcpyHostToDevice) != hipSuccess) {
            ac4_md_destroy(md);
            ac4_set_error("ac4_md_create: field table upload failed");
            return AC4_EHIP;
        }
    }
    if (hipStreamCreate(&md->stream) != hipSuccess) {
        ac4_md_destroy(md);
        ac4_set_error("hipStreamCreate failed");
        return AC4_EHIP;
    }
    AC4_HIP(hipMemcpy(md->cblk_rep, crep.data(), sizeof(int) * off_cell, hipMemcpyHostToDevice));
    AC4_HIP(hipMemcpy(md->cblk_cell, ccell.data(), sizeof(int) * off_cell, hipMemcpyHostToDevice));
    std::vector<ChainS> ch(nslots);
    for (int r = 0; r < nslots; r++) fresh_chain(ch[r], md->reps_h[r]);
    AC4_HIP(hipMemcpy(md->chain, ch.data(), sizeof(ChainS) * nslots, hipMemcpyHostToDevice));
    std::vector<int> neg(off, -1), ids(off);
    for (int r = 0; r < nslots; r++)
        for (int i = 0; i < md->reps_h[r].cap_n; i++) ids[md->reps_h[r].off + i] = i;
    AC4_HIP(hipMemcpy(md->P.act, neg.data(), sizeof(int) * off, hipMemcpyHostToDevice));
    AC4_HIP(hipMemcpy(md->P.id, ids.data(), sizeof(int) * off, hipMemcpyHostToDevice));
    md->have_forces = true;  // nothing loaded yet; set_state asks for a force evaluation
    if ((rc = refresh_tables(md)) != AC4_OK) { ac4_md_destroy(md); return rc; }
    *out = md;
    return AC4_OK;
}

template <class T>
static int h2d(T *dst, const T *src, size_t n, hipStream_t s);

static void drop_graphs(ac4_md *md) {
    for (int k = 0; k < 2; k++) {
        if (md->gexec[k]) { (void)hipGraphExecDestroy(md->gexec[k]); md->gexec[k] = nullptr; }
        md->eager = 0;
        if (md->graph[k]) { (void)hipGraphDestroy(md->graph[k]); md->graph[k] = nullptr; }
    }
}

// Block tables of the occupied slots only (all slots while none is
// occupied), in slot order: the step's launch grids skip idle slots, whose
// blocks would only exit.  A replica's blocks, and so its arithmetic (every
// per-replica sum runs over its own blocks in their order), do not change.
// The recorded step graphs are dropped: their grids change.
static int refresh_tables(ac4_md *md) {
    bool any = false;
    for (const RepC &R : md->reps_h) any |= R.n > 0;
    // the tables as they lie on the device, in one copy
    char *const first = (char *)md->blk_rep;
    md->tables.resize((size_t)((char *)(md->reps + md->R) - first));
    const auto host = [&](auto *dev) { return (decltype(dev))(md->tables.data() + ((char *)dev - first)); };
    int *const br = host(md->blk_rep), *const bf = host(md->blk_first), *const bi = host(md->blk_idx),
        *const lr = host(md->lblk_rep), *const lf = host(md->lblk_first);
    BlkD *const bd = host(md->blkd), *const fd = host(md->fblk);
    int nb = 0, nfb = 0, nlb = 0;
    for (int r = 0; r < md->R; r++) {
        RepC &R = md->reps_h[r];
        if (any && R.n == 0) continue;
        R.blk_off = nb;
        for (int k = 0; k < R.nblk; k++, nb++) {
            br[nb] = r;
            bf[nb] = k * BLK;
            bi[nb] = k;
            bd[nb] = BlkD{r, k * BLK, R.off, R.n};
        }
        R.fblk_off = nfb;
        for (int k = 0; k < R.fnblk; k++) fd[nfb++] = BlkD{r, k * (BLK >> md->lw), R.off, R.n};
        R.lblk_off = nlb;
        for (int k = 0; k < R.lnblk; k++, nlb++) {
            lr[nlb] = r;
            lf[nlb] = k * LPB;
        }
    }
    memcpy(host(md->reps), md->reps_h.data(), sizeof(RepC) * md->R);
    hipStream_t s = md->stream;
    AC4_HIP(hipStreamSynchronize(s));
    drop_graphs(md);
    job_rules(md);
    AC4_HIP(hipMemcpyAsync(first, md->tables.data(), md->tables.size(), hipMemcpyHostToDevice, s));
    AC4_HIP(hipStreamSynchronize(s));
    md->nblk = nb;
    md->fnblk = nfb;
    md->lnblk = nlb;
    return AC4_OK;
}

extern "C" int ac4_md_assign(ac4_md *md, int slot, const ac4_replica_params *p) {
    AC4_REQUIRE(md && slot >= 0 && slot < md->R && p, AC4_EARG, "ac4_md_assign: bad arguments");
    RepC R = md->reps_h[slot];
    const char *why = configure_rep(R, *p);
    AC4_REQUIRE(!why, AC4_EARG, "slot %d: %s", slot, why ? why : "");
    // the block tables hold the replica's n, the launch rules its n_act and cells
    const RepC &old = md->reps_h[slot];
    const bool same = old.n == R.n && old.nact == R.nact && old.ncell == R.ncell;
    md->reps_h[slot] = R;
    ChainS c;
    fresh_chain(c, R);
    AC4_HIP(hipMemcpyAsync(md->reps + slot, &md->reps_h[slot], sizeof(RepC), hipMemcpyHostToDevice, md->stream));
    AC4_HIP(hipMemcpyAsync(md->chain + slot, &c, sizeof(ChainS), hipMemcpyHostToDevice, md->stream));
    AC4_HIP(hipStreamSynchronize(md->stream));
    return same ? AC4_OK : refresh_tables(md);
}

extern "C" int ac4_md_release(ac4_md *md, int slot) {
    AC4_REQUIRE(md && slot >= 0 && slot < md->R, AC4_EARG, "ac4_md_release: bad arguments");
    RepC &R = md->reps_h[slot];
    R.n = 0; R.nact = 0; R.ncell = 0; R.tau = 0; R.nc = 0;
    ChainS c;
    fresh_chain(c, R);
    AC4_HIP(hipMemcpyAsync(md->reps + slot, &R, sizeof(RepC), hipMemcpyHostToDevice, md->stream));
    AC4_HIP(hipMemcpyAsync(md->chain + slot, &c, sizeof(ChainS), hipMemcpyHostToDevice, md->stream));
    AC4_HIP(hipStreamSynchronize(md->stream));
    return refresh_tables(md);
}

extern "C" int ac4_md_slot_n(const ac4_md *md, int slot) {
    if (!md || slot < 0 || slot >= md->R) return AC4_EARG;
    return md->reps_h[slot].n;
}

extern "C" int ac4_md_create(int n_rep, const ac4_replica_params *p, int precision, ac4_md **out) {
    AC4_REQUIRE(n_rep >= 1 && p && out, AC4_EARG, "ac4_md_create: bad arguments");
    std::vector<int> caps(n_rep);
    for (int r = 0; r < n_rep; r++) caps[r] = p[r].n;
    ac4_md *md = nullptr;
    TRY(ac4_md_create_slots(n_rep, caps.data(), precision, &md));
    for (int r = 0; r < n_rep; r++) {
        int rc = ac4_md_assign(md, r, &p[r]);
        if (rc != AC4_OK) { ac4_md_destroy(md); return rc; }
    }
    *out = md;
    return AC4_OK;
}

static void free_fmt(ac4_md *md) {
    for (void *q : {(void *)md->fmt_dev, (void *)md->fmt_len_dev, (void *)md->fmt_bsum})
        if (q) (void)hipFree(q);
    for (void *q : {(void *)md->fmt_txt, (void *)md->fmt_meta})
        if (q) (void)hipHostFree(q);
    for (hipEvent_t &ev : md->fmt_ev) {
        if (ev) (void)hipEventDestroy(ev);
        ev = nullptr;
    }
    md->fmt_dev = md->fmt_txt = nullptr;
    md->fmt_len_dev = nullptr;
    md->fmt_bsum = nullptr;
    md->fmt_meta = nullptr;
    md->fmt_cap = 0;
}

extern "C" int ac4_md_destroy(ac4_md *md) {
    if (!md) return AC4_OK;
    if (md->stream) (void)hipStreamSynchronize(md->stream);
    drop_graphs(md);
    void *ptrs[] = {md->mem, md->ox, md->oy, md->oz, md->ov_q, md->ov_q2, md->ov_step, md->ov_cnt, md->ov_n, md->ov_list,
                    md->ov_out, md->ex, md->ey, md->ez, md->et};
    for (void *q : ptrs)
        if (q) (void)hipFree(q);
    free_fmt(md);
    if (md->stream) (void)hipStreamDestroy(md->stream);
    delete md;
    return AC4_OK;
}

extern "C" int ac4_md_total_particles(const ac4_md *md) { return md ? md->ntot : 0; }

// Device bytes a slot of capacity cap_n adds to a handle: the arrays
// ac4_md_create_slots and ac4_md_overlap_enable allocate and the
// reference-order export's, the force blocks counted at the widest team (16
// lanes a particle) and the parallel-shuffle tables at their largest, as if
// this slot were the largest of its handle.
extern "C" long long ac4_md_slot_bytes(int cap_n, int n_origin, int n_lags) {
    if (cap_n < 2 || n_origin < 0 || n_lags < 0) return AC4_EARG;
    const size_t n = cap_n, cells = slot_cells(cap_n), fnb = (n * 16 + BLK - 1) / BLK;
    const SlotCounts k{1, n, cells, (n + BLK - 1) / BLK, fnb, (n + LPB - 1) / LPB, (cells + BLK / 64 - 1) / (BLK / 64),
                       cap_n > SHUF_PAR_MIN ? 3 * ((n + SHUF_M - 1) / SHUF_M) : 0};
    ac4_md md;  // for the arrays' types
    long long b = 0;
    const auto add = [&](auto **p, size_t count) {
        b += (long long)(sizeof(**p) * count);
        return AC4_OK;
    };
    (void)each_array(&md, k, add);
    (void)each_export_array(&md, n, add);
    if (n_origin > 0) (void)each_overlap_array(&md, 1, n, n_origin, n_lags, add);
    return b;
}


static int check_rep(const ac4_md *md, int r) {
    AC4_REQUIRE(md && r >= 0 && r < md->R, AC4_EARG, "bad handle or replica index %d", r);
    AC4_REQUIRE(md->reps_h[r].n > 0, AC4_ESTATE, "slot %d is idle (no job assigned)", r);
    return AC4_OK;
}

template <class T>
static int h2d(T *dst, const T *src, size_t n, hipStream_t s) {
    AC4_HIP(hipMemcpyAsync(dst, src, n * sizeof(T), hipMemcpyHostToDevice, s));
    return AC4_OK;
}
template <class T>
static int d2h(T *dst, const T *src, size_t n, hipStream_t s) {
    AC4_HIP(hipMemcpyAsync(dst, src, n * sizeof(T), hipMemcpyDeviceToHost, s));
    return AC4_OK;
}
static int get_chain(ac4_md *md, int r, ChainS *c) {
    TRY(d2h(c, md->chain + r, 1, md->stream));
    AC4_HIP(hipStreamSynchronize(md->stream));
    return AC4_OK;
}
static int put_chain(ac4_md *md, int r, const ChainS *c) {
    TRY(h2d(md->chain + r, c, 1, md->stream));
    AC4_HIP(hipStreamSynchronize(md->stream));
    return AC4_OK;
}
static int get_chains(ac4_md *md, std::vector<ChainS> &c) {
    c.resize(md->R);
    TRY(d2h(c.data(), md->chain, md->R, md->stream));
    AC4_HIP(hipStreamSynchronize(md->stream));
    return AC4_OK;
}
static int put_chains(ac4_md *md, const std::vector<ChainS> &c) {
    TRY(h2d(md->chain, c.data(), md->R, md->stream));
    AC4_HIP(hipStreamSynchronize(md->stream));
    return AC4_OK;
}

// Sets error bits on replica r as the kernels do when a list or cell
// overflows or a coordinate runs away, without any of those happening: the
// way tests exercise the failure handling of the callers.
extern "C" int ac4_md_raise_error(ac4_md *md, int r, int bits) {
    TRY(check_rep(md, r));
    AC4_REQUIRE(bits > 0 && bits < 4, AC4_EARG, "raise_error: bits must be 1, 2 or 3");
    ChainS c;
    TRY(get_chain(md, r, &c));
    c.err |= bits;
    return put_chain(md, r, &c);
}

// Error bits of every replica (bit 0: neighbour list or cell over capacity,
// bit 1: non-finite or runaway coordinate); err[r] for r < R.
extern "C" int ac4_md_errors(ac4_md *md, int *err) {
    AC4_REQUIRE(md && err, AC4_EARG, "errors: bad arguments");
    std::vector<ChainS> c;
    TRY(get_chains(md, c));
    for (int r = 0; r < md->R; r++) err[r] = md->reps_h[r].n > 0 ? c[r].err : 0;
    return AC4_OK;
}

// slot -> reference index map of replica r
static int get_ids(ac4_md *md, int r, std::vector<int> &id) {
    const RepC &R = md->reps_h[r];
    id.resize(R.n);
    TRY(d2h(id.data(), md->P.id + R.off, R.n, md->stream));
    AC4_HIP(hipStreamSynchronize(md->stream));
    return AC4_OK;
}
template <class T>
static int fetch_unpermuted(ac4_md *md, int r, const T *dev, T *out, const std::vector<int> &id) {
    const RepC &R = md->reps_h[r];
    std::vector<T> tmp(R.n);
    TRY(d2h(tmp.data(), dev + R.off, R.n, md->stream));
    AC4_HIP(hipStreamSynchronize(md->stream));
    for (int i = 0; i < R.n; i++) out[id[i]] = tmp[i];
    return AC4_OK;
}

static int set_state_impl(ac4_md *md, int r, const double *x, const double *y, const double *z, const double *xu,
                          const double *yu, const double *zu, const double *px, const double *py, const double *pz,
                          const int *type, const int *act_tag, const int *kx, const int *ky, const int *kz,
                          bool slot_local);

extern "C" int ac4_md_set_state(ac4_md *md, int r, const double *x, const double *y, const double *z,
                                const double *xu, const double *yu, const double *zu, const double *px,
                                const double *py, const double *pz, const int *type, const int *act_tag,
                                const int *kx, const int *ky, const int *kz) {
    return set_state_impl(md, r, x, y, z, xu, yu, zu, px, py, pz, type, act_tag, kx, ky, kz, false);
}

// Loads a job into a slot without touching the other slots: its forces start
// at zero and its list is built inside its first step (used by the server, so
// admitting a job never changes the running replicas' arithmetic).
extern "C" int ac4_md_load_slot(ac4_md *md, int r, const double *x, const double *y, const double *z,
                                const double *xu, const double *yu, const double *zu, const double *px,
                                const double *py, const double *pz, const int *type, const int *act_tag,
                                const int *kx, const int *ky, const int *kz) {
    return set_state_impl(md, r, x, y, z, xu, yu, zu, px, py, pz, type, act_tag, kx, ky, kz, true);
}

static int set_state_impl(ac4_md *md, int r, const double *x, const double *y, const double *z, const double *xu,
                          const double *yu, const double *zu, const double *px, const double *py, const double *pz,
                          const int *type, const int *act_tag, const int *kx, const int *ky, const int *kz,
                          bool slot_local) {
    TRY(check_rep(md, r));
    AC4_REQUIRE(x && y && z && xu && yu && zu && px && py && pz && type, AC4_EARG, "set_state: NULL array");
    const RepC &R = md->reps_h[r];
    const int n = R.n, g = R.off;
    std::vector<double4> p4(n);
    std::vector<QPos> q4(n);
    std::vector<int> ids(n);
    double keblk = 0.0;  // time_evolve.c:586-589 order
    for (int i = 0; i < n; i++) {
        AC4_REQUIRE(type[i] == 0 || type[i] == 1, AC4_EARG, "set_state: type[%d]=%d not in {0,1}", i, type[i]);
        AC4_REQUIRE(x[i] >= 0.0 && x[i] < 1.0 && y[i] >= 0.0 && y[i] < 1.0 && z[i] >= 0.0 && z[i] < 1.0, AC4_EARG,
                    "set_state: wrapped coordinate of particle %d outside [0,1)", i);
        p4[i] = make_double4(x[i], y[i], z[i], (double)type[i]);
        q4[i] = qpos(x[i], y[i], z[i], type[i]);
        keblk += px[i] * px[i] + py[i] * py[i] + pz[i] * pz[i];
        ids[i] = i;
    }
    hipStream_t s = md->stream;
    // a loaded state is stored in reference order (slot = index)
    TRY(h2d(md->P.x + g, x, n, s)); TRY(h2d(md->P.y + g, y, n, s)); TRY(h2d(md->P.z + g, z, n, s));
    TRY(h2d(md->P.xu + g, xu, n, s)); TRY(h2d(md->P.yu + g, yu, n, s)); TRY(h2d(md->P.zu + g, zu, n, s));
    TRY(h2d(md->xo + g, xu, n, s)); TRY(h2d(md->yo + g, yu, n, s)); TRY(h2d(md->zo + g, zu, n, s));
    TRY(h2d(md->P.px + g, px, n, s)); TRY(h2d(md->P.py + g, py, n, s)); TRY(h2d(md->P.pz + g, pz, n, s));
    TRY(h2d(md->P.type + g, type, n, s));
    TRY(h2d(md->P.id + g, ids.data(), n, s));
    TRY(h2d(md->pos4 + g, p4.data(), n, s));
    TRY(h2d(md->posq + g, q4.data(), n, s));
    std::vector<int> at;
    if (act_tag) {
        for (int i = 0; i < n; i++)
            AC4_REQUIRE(act_tag[i] >= -1 && act_tag[i] < R.nact, AC4_EARG, "set_state: actTag[%d]=%d out of range", i, act_tag[i]);
        at.assign(act_tag, act_tag + n);
    } else {  // keep the current tags, brought back to reference order
        std::vector<int> cur;
        TRY(get_ids(md, r, cur));
        at.resize(n);
        TRY(fetch_unpermuted(md, r, (const int *)md->P.act, at.data(), cur));
    }
    TRY(h2d(md->P.act + g, at.data(), n, s));
    if (kx && ky && kz && R.nact > 0) {
        std::vector<int8_t> a(R.nact), b(R.nact), c(R.nact);
        for (int i = 0; i < R.nact; i++) { a[i] = (int8_t)kx[i]; b[i] = (int8_t)ky[i]; c[i] = (int8_t)kz[i]; }
        TRY(h2d(md->kx + R.off_act, a.data(), R.nact, s));
        TRY(h2d(md->ky + R.off_act, b.data(), R.nact, s));
        TRY(h2d(md->kz + R.off_act, c.data(), R.nact, s));
        AC4_HIP(hipStreamSynchronize(s));
    }
    ChainS c;
    TRY(get_chain(md, r, &c));  // also completes the copies above
    c.S_end = keblk;
    c.p_scale = 1.0;
    c.force_rebuild = 1;
    c.maxbits = 0ull;
    c.step = 0;  // a loaded state starts a new run (MDcode/main.c:238-240: start = 0)
    c.mode = 0;
    c.err = 0;
    TRY(put_chain(md, r, &c));
    if (slot_local) {
        AC4_HIP(hipMemsetAsync(md->fx + g, 0, sizeof(double) * n, s));
        AC4_HIP(hipMemsetAsync(md->fy + g, 0, sizeof(double) * n, s));
        AC4_HIP(hipMemsetAsync(md->fz + g, 0, sizeof(double) * n, s));
        AC4_HIP(hipStreamSynchronize(s));
    } else {
        md->have_forces = false;
    }
    return AC4_OK;
}

// NVE (on != 0) or back to the Nose-Hoover chain (on == 0) for replica r; the
// chain variables are kept and resume where they were.
extern "C" int ac4_md_set_nve(ac4_md *md, int r, int on) {
    TRY(check_rep(md, r));
    ChainS c;
    TRY(get_chain(md, r, &c));
    AC4_REQUIRE(c.mode != 1, AC4_ESTATE, "set_nve: replica %d is in a relaxation ramp", r);
    c.mode = on ? 2 : 0;
    return put_chain(md, r, &c);
}

// Velocity-rescale ramp for one slot only, applied by its next nsteps steps.
extern "C" int ac4_md_relax_slot(ac4_md *md, int r, int nsteps, double f_start, double f_end) {
    TRY(check_rep(md, r));
    AC4_REQUIRE(nsteps > 0 && f_start > 0 && f_end > 0, AC4_EARG, "relax_slot: bad arguments");
    ChainS c;
    TRY(get_chain(md, r, &c));
    c.mode = 1; c.ramp_n = nsteps; c.ramp_k = 0; c.ramp0 = f_start; c.ramp1 = f_end;
    return put_chain(md, r, &c);
}

extern "C" int ac4_md_get_state(ac4_md *md, int r, double *x, double *y, double *z, double *xu, double *yu,
                                double *zu, double *px, double *py, double *pz, int *kx, int *ky, int *kz) {
    TRY(check_rep(md, r));
    const RepC &R = md->reps_h[r];
    std::vector<int> id;
    TRY(get_ids(md, r, id));
    double *outs[] = {x, y, z, xu, yu, zu, px, py, pz};
    const double *devs[] = {md->P.x, md->P.y, md->P.z, md->P.xu, md->P.yu, md->P.zu, md->P.px, md->P.py, md->P.pz};
    for (int k = 0; k < 9; k++)
        if (outs[k]) TRY(fetch_unpermuted(md, r, devs[k], outs[k], id));
    ChainS ch;
    TRY(get_chain(md, r, &ch));
    const double ps = ch.p_scale;  // pending end-of-step U3 factor
    if (ps != 1.0)
        for (int i = 0; i < R.n; i++) {
            if (px) px[i] = px[i] * ps;
            if (py) py[i] = py[i] * ps;
            if (pz) pz[i] = pz[i] * ps;
        }
    if ((kx || ky || kz) && R.nact > 0) {
        std::vector<int8_t> a(R.nact), b(R.nact), c(R.nact);
        TRY(d2h(a.data(), md->kx + R.off_act, R.nact, md->stream));
        TRY(d2h(b.data(), md->ky + R.off_act, R.nact, md->stream));
        TRY(d2h(c.data(), md->kz + R.off_act, R.nact, md->stream));
        AC4_HIP(hipStreamSynchronize(md->stream));
        for (int i = 0; i < R.nact; i++) {
            if (kx) kx[i] = a[i];
            if (ky) ky[i] = b[i];
            if (kz) kz[i] = c[i];
        }
    }
    return AC4_OK;
}

extern "C" int ac4_md_get_forces(ac4_md *md, int r, double *fx, double *fy, double *fz) {
    TRY(check_rep(md, r));
    std::vector<int> id;
    TRY(get_ids(md, r, id));
    if (fx) TRY(fetch_unpermuted(md, r, (const double *)md->fx, fx, id));
    if (fy) TRY(fetch_unpermuted(md, r, (const double *)md->fy, fy, id));
    if (fz) TRY(fetch_unpermuted(md, r, (const double *)md->fz, fz, id));
    return AC4_OK;
}

extern "C" int ac4_md_set_chain(ac4_md *md, int r, const double *c9) {
    TRY(check_rep(md, r));
    AC4_REQUIRE(c9, AC4_EARG, "set_chain: NULL");
    ChainS c;
    TRY(get_chain(md, r, &c));
    for (int k = 0; k < 3; k++) { c.eta[k] = c9[k]; c.peta[k] = c9[3 + k]; c.q[k] = c9[6 + k]; }
    return put_chain(md, r, &c);
}

// fixDrift (MDcode/initialise.c:104-138) for replica r: the momenta summed in
// reference particle order and divided by N are subtracted from every
// particle.  The pending end-of-step U3 factor is applied first (the
// reference's momenta are final after a step), and the sum of p^2 the next
// step's thermostat starts from is recomputed.  mean3 (nullable) receives
// the mean that was removed.
// ---- frame text on the device (MDcode/print.c:4-16 line format)
// One number as glibc's %.5lf: v = m*2^e exactly, q = round-half-even of
// m*10^5*2^e (the 70-bit product kept as two 64-bit words), printed as
// q/10^5 "." q%10^5 with the sign of v.  Values with |v| >= 1e12 or not
// finite set *bad (the host formats those frames).
__device__ __forceinline__ char *fmt_put_u64(char *o, unsigned long long v) {
    if (v < 10) {
        *o++ = (char)('0' + (int)v);
        return o;
    }
    char t[24];
    int k = 0;
    do {
        t[k++] = (char)('0' + v % 10ull);
        v /= 10ull;
    } while (v);
    while (k) *o++ = t[--k];
    return o;
}
__device__ __forceinline__ char *fmt5_dev(char *o, double v, int *bad) {
    const unsigned long long bits = (unsigned long long)__double_as_longlong(v);
    const int neg = (int)(bits >> 63), ex = (int)((bits >> 52) & 0x7ff);
    const unsigned long long frac = bits & ((1ull << 52) - 1);
    if (ex == 0x7ff || fabs(v) >= 1e12) {
        *bad = 1;
        return o;
    }
    const unsigned long long m = ex ? (frac | (1ull << 52)) : frac;
    const int e = ex ? ex - 1075 : -1074;  // v = m * 2^e, e < 0 for |v| < 1e12 unless v is 0
    unsigned long long q = 0;
    if (m != 0 && e < 0 && -e <= 71) {
        const unsigned long long lo = m * 100000ull, hi = __umul64hi(m, 100000ull);  // t = hi:lo < 2^70
        const int sh = -e;
        // q = t >> sh; rounding bit sh-1 and the sticky bits below it
        q = sh >= 64 ? hi >> (sh - 64) : ((lo >> sh) | (hi << (64 - sh)));
        const int rb = sh - 1;
        const unsigned long long rbit = rb >= 64 ? (hi >> (rb - 64)) & 1ull : (lo >> rb) & 1ull;
        bool sticky;
        if (rb >= 64)
            sticky = lo != 0ull || (rb > 64 && (hi & ((1ull << (rb - 64)) - 1ull)) != 0ull);
        else
            sticky = rb > 0 && (lo & ((1ull << rb) - 1ull)) != 0ull;
        if (rbit && (sticky || (q & 1ull))) q++;
    } else if (m != 0 && e >= 0) {
        *bad = 1;  // an integer of 2^52 or more: not below 1e12
        return o;
    }
    if (neg) *o++ = '-';
    unsigned fp;
    if (q < 1000ull * 100000ull) {  // up to three digits before the point: 32-bit arithmetic
        const unsigned q32 = (unsigned)q, ip = q32 / 100000u;
        fp = q32 - ip * 100000u;
        if (ip >= 100u) *o++ = (char)('0' + ip / 100u);
        if (ip >= 10u) *o++ = (char)('0' + ip / 10u % 10u);
        *o++ = (char)('0' + ip % 10u);
    } else {
        o = fmt_put_u64(o, q / 100000ull);
        fp = (unsigned)(q % 100000ull);
    }
    *o++ = '.';
#pragma unroll
    for (int d = 4; d >= 0; d--) {
        o[d] = (char)('0' + fp % 10u);
        fp /= 10u;
    }
    return o + 5;
}

// line of the particle in slot s of replica R, written to slot id[s] (its
// reference index) of out (FMT_LINE bytes each), formed in LDS and stored 16
// bytes at a time (50000 lines: 6.2 us; formed in scratch memory and stored
// byte by byte 11.7)
#define FMT_LINE 80
__global__ void __launch_bounds__(BLK) k_fmt_frame(const RepC *__restrict__ reps, int r, const double *__restrict__ xu,
                                                   const double *__restrict__ yu, const double *__restrict__ zu,
                                                   const int *__restrict__ type, const int *__restrict__ id,
                                                   char *out, unsigned char *len, long long *meta) {
    __shared__ uint4 s_line[BLK][FMT_LINE / 16];
    const RepC R = reps[r];
    const int s = blockIdx.x * BLK + threadIdx.x;
    if (s >= R.n) return;
    const int g = R.off + s, i = id[g];
    char *const line = (char *)s_line[threadIdx.x];
    int b = 0;
    char *o = fmt5_dev(line, xu[g], &b);
    *o++ = '\t';
    o = fmt5_dev(o, yu[g], &b);
    *o++ = '\t';
    o = fmt5_dev(o, zu[g], &b);
    *o++ = '\t';
    const int t = type[g];
    if (t < 0) {
        *o++ = '-';
        o = fmt_put_u64(o, (unsigned long long)(-(long long)t));
    } else {
        o = fmt_put_u64(o, (unsigned long long)t);
    }
    *o++ = '\n';
    const int k = (int)(o - line);
    uint4 *dst = (uint4 *)(out + (size_t)i * FMT_LINE);
#pragma unroll
    for (int c = 0; c < FMT_LINE / 16; c++)
        if (16 * c < k) dst[c] = s_line[threadIdx.x][c];
    len[i] = (unsigned char)k;
    if (b) meta[2] = 1;  // pinned; every writer stores the same
}

// bytes of each block of BLK lines (reference order)
__global__ void __launch_bounds__(BLK) k_fmt_bsum(int n, const unsigned char *__restrict__ len, int *__restrict__ bsum) {
    __shared__ int s_w[BLK / 64];
    const int i = blockIdx.x * BLK + threadIdx.x;
    const int w = ac4_wave_sum_i(i < n ? (int)len[i] : 0);
    if ((threadIdx.x & 63) == 0) s_w[threadIdx.x >> 6] = w;
    __syncthreads();
    if (threadIdx.x == 0) bsum[blockIdx.x] = s_w[0] + s_w[1] + s_w[2] + s_w[3];
}

// One piece of the text: lines of the blocks [b0, b0 + gridDim.x) from their
// slots to txt (pinned host memory), and the piece's bytes to *bytes.  A block
// adds up the blocks of the piece before it, joins its lines in LDS and stores
// the joined text 16 bytes at a time, so that the bus carries whole words.
#define FMT_PIECE 128  // blocks of a piece, at most
__global__ void __launch_bounds__(BLK) k_fmt_pack(int n, int b0, const char *__restrict__ slots,
                                                  const unsigned char *__restrict__ len, const int *__restrict__ bsum,
                                                  char *__restrict__ txt, long long *bytes) {
    __shared__ uint4 s_buf[BLK * FMT_LINE / 16 + 1];
    __shared__ int s_w[2][BLK / 64];
    char *const s_txt = (char *)s_buf;
    const int t = threadIdx.x, lane = t & 63, w = t >> 6, b = b0 + blockIdx.x, i = b * BLK + t;
    static_assert(FMT_PIECE <= BLK, "one block sum per thread");
    const int k = i < n ? (int)len[i] : 0;
    uint4 v[FMT_LINE / 16];
    const uint4 *src = (const uint4 *)(slots + (size_t)(i < n ? i : 0) * FMT_LINE);
#pragma unroll
    for (int c = 0; c < FMT_LINE / 16; c++)
        if (16 * c < k) v[c] = src[c];
    const int before = ac4_wave_sum_i(t < (int)blockIdx.x ? bsum[b0 + t] : 0);
    int at = k;
    for (int o = 1; o < 64; o <<= 1) {
        const int u = __shfl_up(at, o, 64);
        if (lane >= o) at += u;
    }
    if (lane == 63) s_w[0][w] = at;
    if (lane == 0) s_w[1][w] = before;  // the wave's sum is in its first lane
    __syncthreads();
    const int off = s_w[1][0] + s_w[1][1] + s_w[1][2] + s_w[1][3], h = off & 15;
    at += h - k;
    for (int q = 0; q < w; q++) at += s_w[0][q];
    const int end = h + s_w[0][0] + s_w[0][1] + s_w[0][2] + s_w[0][3];  // the block's text: s_txt[h, end)
#pragma unroll
    for (int c = 0; c < FMT_LINE / 16; c++) {
        const unsigned u[4] = {v[c].x, v[c].y, v[c].z, v[c].w};
#pragma unroll
        for (int q = 0; q < 16; q++)
            if (16 * c + q < k) s_txt[at + 16 * c + q] = (char)(u[q / 4] >> (8 * (q % 4)));
    }
    __syncthreads();
    char *const dst = txt + (off - h);
    for (int q = 16 * t; q < end; q += 16 * BLK) {
        if (q >= h && q + 16 <= end)
            *(uint4 *)(dst + q) = s_buf[q / 16];
        else  // words shared with the neighbouring blocks
            for (int c = max(q, h); c < min(q + 16, end); c++) dst[c] = s_txt[c];
    }
    if (t == 0 && blockIdx.x == gridDim.x - 1) *bytes = off - h + end;
}

// data_coor.out text of replica r's current frame (x_u, y_u, z_u, type in
// reference order), formatted and joined on the device; byte for byte the
// text of ac4_format_frame on the same values, which formats a frame holding
// a value the device formatter leaves to the host.
extern "C" long long ac4_md_format_frame(ac4_md *md, int r, char *out, long long cap) {
    TRY(check_rep(md, r));
    const RepC &R = md->reps_h[r];
    const int n = R.n;
    AC4_REQUIRE(out && cap >= 80LL * n, AC4_EARG, "format_frame: buffer needs 80 bytes a line");
    const int nb = (n + BLK - 1) / BLK, np = (nb + FMT_PIECE - 1) / FMT_PIECE;
    const auto piece_bytes = [](int blocks) { return (size_t)std::min(blocks, FMT_PIECE) * BLK * FMT_LINE; };
    if ((size_t)n > md->fmt_cap) {
        free_fmt(md);
        const size_t cn = (size_t)n;
        AC4_HIP(hipMalloc(&md->fmt_dev, FMT_LINE * cn));
        AC4_HIP(hipMalloc(&md->fmt_len_dev, cn));
        AC4_HIP(hipMalloc(&md->fmt_bsum, sizeof(int) * nb));
        AC4_HIP(hipHostMalloc((void **)&md->fmt_txt, piece_bytes(nb) * (np > 1 ? 2 : 1), hipHostMallocDefault));
        AC4_HIP(hipHostMalloc((void **)&md->fmt_meta, 3 * sizeof(long long), hipHostMallocDefault));
        for (hipEvent_t &ev : md->fmt_ev) AC4_HIP(hipEventCreateWithFlags(&ev, hipEventDisableTiming));
        md->fmt_cap = cn;
    }
    if (n == 0) return 0;
    hipStream_t s = md->stream;
    volatile long long *meta = md->fmt_meta;
    meta[2] = 0;
    hipLaunchKernelGGL(k_fmt_frame, dim3(nb), dim3(BLK), 0, s, md->reps, r, md->P.xu, md->P.yu, md->P.zu, md->P.type,
                       md->P.id, md->fmt_dev, md->fmt_len_dev, md->fmt_meta);
    hipLaunchKernelGGL(k_fmt_bsum, dim3(nb), dim3(BLK), 0, s, n, md->fmt_len_dev, md->fmt_bsum);
    AC4_HIP(hipGetLastError());
    // the pieces over the bus straight from their kernel, two under way; the
    // host copies one to the caller's buffer while the next is written.  A
    // copy from the device to the caller's pageable memory takes 90 us for the
    // 1.55 MB of 50000 lines, this way 27 over the bus and 18 by memcpy; the
    // whole call 142 -> 82 us (the two small results alone, copied to pageable
    // memory, took 20 of it).  Pages of the pinned pieces cost the host 1.6 us
    // each when it first reads them, in a handle's first frame: 100000 lines
    // 0.34 -> 0.93 ms, then 218 -> 142 us a frame (200000: 0.54 -> 1.11 ms, 376
    // -> 226 us).  Pieces of a half and a quarter of the size: 0.62 and 0.51 ms,
    // but 154 and 204 us (271 and 365).
    const auto pack = [&](int p) {
        const int b0 = p * FMT_PIECE;
        hipLaunchKernelGGL(k_fmt_pack, dim3(std::min(FMT_PIECE, nb - b0)), dim3(BLK), 0, s, n, b0, md->fmt_dev,
                           md->fmt_len_dev, md->fmt_bsum, md->fmt_txt + (p & 1) * piece_bytes(nb), md->fmt_meta + (p & 1));
        if (p + 1 < np) AC4_HIP(hipEventRecord(md->fmt_ev[p & 1], s));
        AC4_HIP(hipGetLastError());
        return AC4_OK;
    };
    for (int p = 0; p < std::min(np, 2); p++) TRY(pack(p));
    bool bad = false;
    long long total = 0;
    for (int p = 0; p < np && !bad; p++) {
        if (p + 1 < np)
            AC4_HIP(hipEventSynchronize(md->fmt_ev[p & 1]));
        else
            AC4_HIP(hipStreamSynchronize(s));
        bad = meta[2] != 0;  // known with the first piece
        const long long k = meta[p & 1];
        AC4_REQUIRE(k > 0 && k <= (long long)piece_bytes(nb) && total + k <= (long long)FMT_LINE * n, AC4_ESTATE,
                    "format_frame: piece of %lld bytes", k);
        if (!bad) memcpy(out + total, md->fmt_txt + (p & 1) * piece_bytes(nb), (size_t)k);
        total += k;
        if (!bad && p + 2 < np) TRY(pack(p + 2));
    }
    if (bad) {  // a value the device formatter does not cover: the host formats the frame
        std::vector<double> x(n), y(n), z(n);
        std::vector<int> id, ty(n);
        TRY(get_ids(md, r, id));
        TRY(fetch_unpermuted(md, r, (const double *)md->P.xu, x.data(), id));
        TRY(fetch_unpermuted(md, r, (const double *)md->P.yu, y.data(), id));
        TRY(fetch_unpermuted(md, r, (const double *)md->P.zu, z.data(), id));
        TRY(fetch_unpermuted(md, r, (const int *)md->P.type, ty.data(), id));
        return ac4_format_frame(n, x.data(), y.data(), z.data(), ty.data(), out, cap);
    }
    return total;
}

extern "C" int ac4_md_fix_drift(ac4_md *md, int r, double *mean3) {
    TRY(check_rep(md, r));
    const RepC &R = md->reps_h[r];
    const int n = R.n;
    AC4_REQUIRE(n > 0, AC4_ESTATE, "fix_drift: replica %d holds no particles", r);
    std::vector<int> id;
    TRY(get_ids(md, r, id));
    ChainS c;
    TRY(get_chain(md, r, &c));
    double *dev[3] = {md->P.px, md->P.py, md->P.pz};
    std::vector<double> p[3], tmp(n);
    for (int a = 0; a < 3; a++) {
        p[a].resize(n);
        TRY(d2h(tmp.data(), dev[a] + R.off, n, md->stream));
        AC4_HIP(hipStreamSynchronize(md->stream));
        for (int k = 0; k < n; k++) p[a][id[k]] = tmp[k] * c.p_scale;
    }
    double m[3];
    for (int a = 0; a < 3; a++) {
        double sum = 0.0;
        for (int i = 0; i < n; i++) sum += p[a][i];
        m[a] = sum / (double)n;
    }
    double keblk = 0.0;  // time_evolve.c:586-589 order
    for (int i = 0; i < n; i++) {
        p[0][i] -= m[0];
        p[1][i] -= m[1];
        p[2][i] -= m[2];
        keblk += p[0][i] * p[0][i] + p[1][i] * p[1][i] + p[2][i] * p[2][i];
    }
    for (int a = 0; a < 3; a++) {
        for (int k = 0; k < n; k++) tmp[k] = p[a][id[k]];
        TRY(h2d(dev[a] + R.off, tmp.data(), n, md->stream));
        AC4_HIP(hipStreamSynchronize(md->stream));
    }
    c.p_scale = 1.0;
    c.S_end = keblk;
    TRY(put_chain(md, r, &c));
    if (mean3)
        for (int a = 0; a < 3; a++) mean3[a] = m[a];
    return AC4_OK;
}

extern "C" int ac4_md_get_chain(ac4_md *md, int r, double *c9) {
    TRY(check_rep(md, r));
    ChainS c;
    TRY(get_chain(md, r, &c));
    for (int k = 0; k < 3; k++) { c9[k] = c.eta[k]; c9[3 + k] = c.peta[k]; c9[6 + k] = c.q[k]; }
    return AC4_OK;
}

extern "C" int ac4_md_set_rebuild_criterion(ac4_md *md, int criterion) {
    AC4_REQUIRE(md && (criterion == 0 || criterion == 1), AC4_EARG, "criterion must be 0 (safe) or 1 (reference)");
    std::vector<ChainS> c;
    TRY(get_chains(md, c));
    for (auto &e : c) e.crit = criterion;
    return put_chains(md, c);
}

// A launch of the step's chain: on the handle's stream, or, while steps are
// recorded, as the next node of the graph.  Stream capture would fail other
// threads: while any stream is being captured, their calls on the null stream
// (a plain hipMemcpy, the creation of another handle) return an error, in every
// capture mode, and can end the capture.
template <class... P>
static void put(ac4_md *md, void (*kern)(P...), dim3 grid, dim3 block, size_t lds,
                typename std::common_type<P>::type... a) {
    void *args[] = {(void *)&a...};
    if (!md->rec) {
        (void)hipLaunchKernel((const void *)kern, grid, block, args, lds, md->stream);  // the callers ask hipGetLastError
        return;
    }
    hipKernelNodeParams q{};
    q.func = (void *)kern;
    q.gridDim = grid;
    q.blockDim = block;
    q.sharedMemBytes = (unsigned)lds;
    q.kernelParams = args;
    hipGraphNode_t node = nullptr;
    const hipError_t e = hipGraphAddKernelNode(&node, md->rec, &md->rec_end, md->rec_end ? 1 : 0, &q);
    if (e == hipSuccess) md->rec_end = node;
    else if (md->rec_err == hipSuccess) md->rec_err = e;
}

// Cell counts are cleared by k_first_half inside a step; outside a step
// (update_cell_list) with_zero clears them first.
// fixed grid of the work-list kernels: enough workgroups to fill the device
#define WL_GRID 1024
#define TEAM_MOVE_N 400000
static int launch_rebuild(ac4_md *md, bool with_zero = false) {
    const int cy = (md->max_ncell + BLK - 1) / BLK;
    const WorkList wl{md->wl_item, md->wl_n, md->nblk, md->nblk + md->lnblk};
    const int gb = std::min(md->nblk, WL_GRID), gl = std::min(md->lnblk, WL_GRID), gc = std::min(md->ncb, WL_GRID);
    if (with_zero)
        put(md, k_cell_zero, dim3(md->R, cy), dim3(BLK), 0, md->reps, md->chain, md->cnt, md->wl_n);
    put(md, k_bin, dim3(md->nblk), dim3(BLK), 0, md->reps, md->chain, md->blk_rep, md->blk_first,
        md->P.x, md->P.y, md->P.z, md->P.id, md->cnt, md->P.cell_of, md->cell_mem, md->P.cell_ref,
        md->bin_fuse ? 1 : 0, md->bdone, md->start, wl);
    if (!md->bin_fuse)
        put(md, k_bin_end, dim3(md->R), dim3(BIN_END_T), 0, md->reps, md->chain, md->cnt, md->start, wl);
    put(md, k_cell_sort, dim3(gc), dim3(BLK), 0, md->reps, wl, md->cnt, md->start,
        md->cell_mem, md->members, md->ranges, md->xmid, md->P, md->A,
        PosCopies{md->pos4, md->posq, md->xo, md->yo, md->zo});
    // 16- and 32-lane list teams of handles up to TEAM_MOVE_N particles move
    // the permuted arrays back themselves (measured: 64 replicas, 1.5e5
    // particles, 134.5 -> 130.0 us per step; one box of 1e6, 686 -> 701 us)
    const bool team_moves = !with_zero && (md->nlist_mode == 2 || md->nlist_mode == 3) && md->ntot <= TEAM_MOVE_N;
    if (!team_moves)
        put(md, k_commit, dim3(gb), dim3(BLK), 0, md->reps, md->blk_rep, md->blk_first, wl, md->P,
            md->A);
    if (with_zero)  // update_cell_list: the reference's FP64 test and its 2.85 count
        put(md, k_nlist<true>, dim3(md->nblk), dim3(BLK), 0, md->reps, md->chain, md->blk_rep,
            md->blk_first, md->pos4, md->posq, md->P.cell_of, md->cnt, md->start, md->nn, md->nn_ref,
            md->nl, md->stride, md->cap);
    else if (md->nlist_mode >= 2) {
        const int w = md->nlist_mode == 2 ? 16 : (md->nlist_mode == 3 ? 32 : 64);
        bool trim = false;  // any replica whose cells are ordered by x-half
        for (int r = 0; r < md->R; r++) trim |= md->reps_h[r].n > 0 && md->reps_h[r].xcull;
        auto kern = trim ? (w == 16 ? (team_moves ? k_nlist_team<16, true, true> : k_nlist_team<16, false, true>)
                                    : (w == 32 ? (team_moves ? k_nlist_team<32, true, true> : k_nlist_team<32, false, true>)
                                               : k_nlist_team<64, false, true>))
                         : (w == 16 ? (team_moves ? k_nlist_team<16, true, false> : k_nlist_team<16, false, false>)
                                    : (w == 32 ? (team_moves ? k_nlist_team<32, true, false> : k_nlist_team<32, false, false>)
                                               : k_nlist_team<64, false, false>));
        put(md, kern, dim3(gl), dim3(w * LPB), 0, md->reps, md->chain, md->lblk_rep, md->lblk_first, wl,
            md->posq, md->A.cell_of, md->ranges, md->start, md->xmid, md->nn, md->nl, md->cap, md->ftab);
    }
    else if (md->nlist_mode == 0)
        put(md, k_nlist_cell, dim3(md->ncell_tot), dim3(64), 0, md->reps, md->chain, md->cblk_rep,
            md->cblk_cell, md->posq, md->cnt, md->start, md->nn, md->nl, md->cap);
    else
        put(md, k_nlist<false>, dim3(md->nblk), dim3(BLK), 0, md->reps, md->chain, md->blk_rep,
            md->blk_first, md->pos4, md->posq, md->P.cell_of, md->cnt, md->start, md->nn, md->nn_ref,
            md->nl, md->stride, md->cap);
    AC4_HIP(hipGetLastError());
    return AC4_OK;
}

template <bool FP32, bool KICK, int EN>
static int launch_force_kernel(ac4_md *md, bool step) {
    auto kern = k_force<FP32, KICK, EN, 1>;
    if constexpr (EN <= 1) {
        if (md->vec == 8) kern = k_force<FP32, KICK, EN, 8>;
    }
    if constexpr (FP32 ? EN == 0 || EN == 4 : true) {
        if (md->vec < 0) kern = k_force<FP32, KICK, EN, -2>;
    }
    put(md, kern, dim3(xcd_grid(md->fnblk)), dim3(BLK), 0, md->reps, md->fblk, md->pos4,
        md->posq, md->nn, md->nl, md->cap, md->lw, md->lc, md->lt, md->P.act, md->kx, md->ky, md->kz, md->fx,
        md->fy, md->fz, md->P.px, md->P.py, md->P.pz, md->partial, md->fnblk,
        EndArgs{md->chain, md->mid, md->gpart, md->gdone, md->rdone, md->en > 1 ? 1 : 0, step ? 1 : 0});
    AC4_HIP(hipGetLastError());
    return AC4_OK;
}
// energy: form the pair energy and virial in this pass (without KICK always);
// step: also complete Heff (after a step without them)
template <bool KICK>
static int launch_force(ac4_md *md, bool energy, bool step = false) {
    if constexpr (KICK) {
        if (!energy)
            return md->prec == AC4_FP32 ? launch_force_kernel<true, true, 0>(md, step) : launch_force_kernel<false, true, 0>(md, step);
    }
    if (md->prec != AC4_FP32) return launch_force_kernel<false, KICK, 1>(md, step);
    return md->en == 1   ? launch_force_kernel<true, KICK, 1>(md, step)
           : md->en == 2 ? launch_force_kernel<true, KICK, 2>(md, step)
                         : launch_force_kernel<true, KICK, 4>(md, step);
}
// The energy after a call whose last step is the end of a recorded chunk, on
// handles that form it in the layout's order (EN > 1: four to five tenths more
// of the pass, so chunks leave it out): the forces once more, with it.
static int launch_energy(ac4_md *md) { return md->en > 1 ? launch_force<false>(md, true, true) : AC4_OK; }

static void launch_shuffle(ac4_md *md, int force) {
    if (md->shuf_serial)
        put(md, k_shuffle, dim3(md->R, 3), dim3(256), md->shuf_lds, md->reps, md->chain, md->kx, md->ky,
            md->kz, force, md->shuf_kcap, md->shuf_bmax > 0 ? 1 : 0);
    if (md->shuf_par) {  // more than SHUF_PAR_MIN active particles
        put(md, k_shuf_part, dim3(md->shuf_bmax, 3, md->R), dim3(64), 0, md->reps, md->chain, force,
            md->shuf_bmax, md->shuf_ent, md->shuf_ent_n);
        put(md, k_shuf_apply, dim3(md->R, 3), dim3(2 * SHUF_M), md->shuf_lds, md->reps, md->chain,
            md->kx, md->ky, md->kz, force, md->shuf_kcap, md->shuf_bmax, md->shuf_ent,
            md->shuf_ent_n);
    }
}
// with_shuffle: the step's shuffle runs in k_first_half's first 3*R
// workgroups (handles whose shuffle LDS is small, see shuf_fused)
static void launch_first_half(ac4_md *md, bool with_shuffle) {
    const ShufArgs sa{md->kx, md->ky, md->kz, md->shuf_kcap, with_shuffle ? 3 * md->R : 0};
    put(md, k_first_half, dim3(md->nblk + sa.nblk), dim3(BLK), with_shuffle ? md->shuf_lds : 0,
        md->reps, md->chain, md->blkd, md->P.x, md->P.y, md->P.z, md->P.xu, md->P.yu,
        md->P.zu, md->P.px, md->P.py, md->P.pz, md->fx, md->fy, md->fz, md->xo, md->yo, md->zo,
        md->P.type, md->pos4, md->posq, md->prec == AC4_FP32 ? 1 : 0, md->chain, md->blk_idx, md->cnt,
        md->wl_n, md->mid, sa);
}

// One MD step, one chain of launches on the handle's stream (also when
// recorded in a graph).  The shuffle, which only the force kernel needs, once
// ran on a second graph branch beside the half kick and the rebuild: the
// fork and join cost more than the overlap gave (about 9 us per step).  It
// now runs inside k_first_half where its LDS allows, else as k_shuffle first.
// last: the call's last step, whose pair energy and virial a caller can read
// (each step overwrites them, so the steps before it do not form them).
static int launch_step(ac4_md *md, bool last) {
    if (md->shuf_fused) {
        launch_first_half(md, true);
    } else {
        launch_shuffle(md, 0);
        launch_first_half(md, false);
    }
    AC4_HIP(hipGetLastError());
    TRY(launch_rebuild(md));
    return launch_force<true>(md, last);
}

static int check_err(ac4_md *md) {
    std::vector<ChainS> c;
    TRY(get_chains(md, c));
    for (int r = 0; r < md->R; r++) {
        AC4_REQUIRE(!(c[r].err & 1), AC4_ECAP, "replica %d: neighbour list exceeded %d entries", r, md->cap);
        AC4_REQUIRE(!(c[r].err & 2), AC4_ESTATE, "replica %d: non-finite or runaway coordinate (run blew up)", r);
    }
    return AC4_OK;
}

static int force_rebuild_all(ac4_md *md) {
    std::vector<ChainS> c;
    TRY(get_chains(md, c));
    for (auto &e : c) e.force_rebuild = 1;
    TRY(put_chains(md, c));
    TRY(launch_rebuild(md, true));
    TRY(get_chains(md, c));
    for (auto &e : c) { e.force_rebuild = 0; e.maxbits = 0ull; }
    return put_chains(md, c);
}

extern "C" int ac4_md_update_cell_list(ac4_md *md, int r_out, int *cell_out, int *full_count_out) {
    AC4_REQUIRE(md, AC4_EARG, "NULL handle");
    TRY(force_rebuild_all(md));
    if (r_out >= 0 && r_out < md->R) {
        std::vector<int> id;
        TRY(get_ids(md, r_out, id));
        if (cell_out) TRY(fetch_unpermuted(md, r_out, (const int *)md->P.cell_ref, cell_out, id));
        if (full_count_out) TRY(fetch_unpermuted(md, r_out, (const int *)md->nn_ref, full_count_out, id));
    }
    return check_err(md);
}

extern "C" int ac4_md_calculate_forces(ac4_md *md, double *out2) {
    AC4_REQUIRE(md, AC4_EARG, "NULL handle");
    std::vector<ChainS> c;
    TRY(get_chains(md, c));
    bool stale = false;
    for (auto &e : c) stale |= e.force_rebuild != 0;
    if (stale) TRY(force_rebuild_all(md));
    TRY(launch_force<false>(md, true));
    TRY(get_chains(md, c));
    if (out2)
        for (int r = 0; r < md->R; r++) { out2[2 * r] = c[r].pe; out2[2 * r + 1] = c[r].vir; }
    md->have_forces = true;
    return check_err(md);
}

// Steps are replayed from recorded graphs: GRAPH_CHUNK steps per launch (one
// launch per ten steps instead of one per step: 1.53e9 -> 1.60e9
// particle-steps/s on the 64-replica ensemble in three launch groups; 25 steps
// instead of ten: 2.093e9 -> 2.101e9), and a one-step graph for the remainder.  Every step's kernels and arguments are the same (the step
// state lives on the device), so a chunk replays exactly the steps launched
// one by one.
#define GRAPH_CHUNK 25
static int record_steps(ac4_md *md, int k) {
    const int m = k ? GRAPH_CHUNK : 1;
    hipGraph_t g = nullptr;
    AC4_HIP(hipGraphCreate(&g, 0));
    md->rec = g;
    md->rec_end = nullptr;
    md->rec_err = hipSuccess;
    int rc = AC4_OK;
    for (int q = 0; q < m && rc == AC4_OK; q++) rc = launch_step(md, q == m - 1 && md->en == 1);
    md->rec = nullptr;
    hipGraphExec_t x = nullptr;
    hipError_t e = md->rec_err;
    if (rc == AC4_OK && e == hipSuccess) e = hipGraphInstantiate(&x, g, nullptr, nullptr, 0);
    if (rc != AC4_OK || e != hipSuccess) {  // nothing of a failed recording is kept
        (void)hipGraphDestroy(g);
        if (rc != AC4_OK) return rc;
        AC4_HIP(e);
    }
    md->graph[k] = g;
    md->gexec[k] = x;
    return AC4_OK;
}

static int ready_graphs(ac4_md *md) {
    if (!md->have_forces) TRY(ac4_md_calculate_forces(md, nullptr));
    for (int k = 0; k < 2; k++)
        if (!md->gexec[k]) TRY(record_steps(md, k));
    return AC4_OK;
}

// Steps launched one by one.  On a small handle the five launches of a step
// cost the host more than the step takes on the device (us per step launched
// and replayed: N=1000 FP64 23.1 and 17.3, 8000 26.3 and 20.8, N=16000 FP32
// 28.1 and 23.0), and recording GRAPH_CHUNK steps about 1.1 ms: once a
// handle of at most STEP_GRAPH_N particles has launched STEP_GRAPH_PAY steps
// that way, its further calls replay whole chunks from the graph, as
// ac4_md_step_graph does (the same kernels and arguments: the results are the
// same bit for bit), and launch the rest.  Larger handles are bound by the
// device (N=50000 FP64: 50.2 and 48.9); short runs never pay for a recording.
#define STEP_GRAPH_N 32768
#define STEP_GRAPH_PAY 300
extern "C" int ac4_md_step(ac4_md *md, int nsteps) {
    AC4_REQUIRE(md && nsteps >= 0, AC4_EARG, "bad arguments");
    if (!md->have_forces) TRY(ac4_md_calculate_forces(md, nullptr));
    int k = 0;
    if (md->ntot <= STEP_GRAPH_N && nsteps >= GRAPH_CHUNK && (md->gexec[1] || md->eager >= STEP_GRAPH_PAY)) {
        if (!md->gexec[1] && record_steps(md, 1) != AC4_OK) {
            (void)hipGetLastError();
            md->eager = 0;  // launched as before, another try later
        }
        for (; md->gexec[1] && nsteps - k >= GRAPH_CHUNK; k += GRAPH_CHUNK)
            AC4_HIP(hipGraphLaunch(md->gexec[1], md->stream));
    }
    md->eager = std::min(md->eager + nsteps - k, STEP_GRAPH_PAY);
    if (k > 0 && k == nsteps) return launch_energy(md);
    for (; k < nsteps; k++) TRY(launch_step(md, k == nsteps - 1));
    return AC4_OK;
}

// A step after the chunks: from the one-step graph, or, the call's last one
// where that graph leaves the energy out, launched.
static int launch_rest(ac4_md *md, bool last) {
    if (last && md->en > 1) return launch_step(md, true);
    AC4_HIP(hipGraphLaunch(md->gexec[0], md->stream));
    return AC4_OK;
}

extern "C" int ac4_md_step_graph(ac4_md *md, int nsteps) {
    AC4_REQUIRE(md && nsteps >= 0, AC4_EARG, "bad arguments");
    TRY(ready_graphs(md));
    for (int k = 0; k < nsteps / GRAPH_CHUNK; k++) AC4_HIP(hipGraphLaunch(md->gexec[1], md->stream));
    const int rest = nsteps % GRAPH_CHUNK;
    for (int k = 0; k < rest; k++) TRY(launch_rest(md, k == rest - 1));
    return rest == 0 && nsteps > 0 ? launch_energy(md) : AC4_OK;
}

// Several handles stepped together: each on its own stream, the graph
// replays interleaved step by step so that the handles' kernels overlap on
// the device (one handle's force kernel beside another's list rebuild).
// Every handle's arithmetic is that of ac4_md_step_graph alone.
extern "C" int ac4_md_step_graph_multi(ac4_md *const *mds, int nh, int nsteps) {
    AC4_REQUIRE(mds && nh > 0 && nsteps >= 0, AC4_EARG, "step_graph_multi: bad arguments");
    for (int h = 0; h < nh; h++) {
        AC4_REQUIRE(mds[h], AC4_EARG, "step_graph_multi: handle %d is NULL", h);
        for (int q = 0; q < h; q++)
            AC4_REQUIRE(mds[q] != mds[h], AC4_EARG, "step_graph_multi: handle %d appears twice", h);
        TRY(ready_graphs(mds[h]));  // forces and the recorded steps of every handle first
    }
    for (int k = 0; k < nsteps / GRAPH_CHUNK; k++)
        for (int h = 0; h < nh; h++) AC4_HIP(hipGraphLaunch(mds[h]->gexec[1], mds[h]->stream));
    const int rest = nsteps % GRAPH_CHUNK;
    for (int k = 0; k < rest; k++)
        for (int h = 0; h < nh; h++) TRY(launch_rest(mds[h], k == rest - 1));
    for (int h = 0; h < nh && rest == 0 && nsteps > 0; h++) TRY(launch_energy(mds[h]));
    return AC4_OK;
}

extern "C" int ac4_md_relax(ac4_md *md, int nsteps, double f_start, double f_end) {
    AC4_REQUIRE(md && nsteps > 0 && f_start > 0 && f_end > 0, AC4_EARG, "relax: bad arguments");
    if (!md->have_forces) TRY(ac4_md_calculate_forces(md, nullptr));
    std::vector<ChainS> c;
    TRY(get_chains(md, c));
    for (auto &e : c) { e.mode = 1; e.ramp_n = nsteps; e.ramp_k = 0; e.ramp0 = f_start; e.ramp1 = f_end; }
    TRY(put_chains(md, c));
    for (int k = 0; k < nsteps; k++) TRY(launch_step(md, k == nsteps - 1));
    return check_err(md);
}

// Eager steps with HIP events (on the handle's stream) around each launch
// group; ms = average ms per step of {first_half, rebuild group, force,
// shuffle, force end}: the per-replica sums and the chain update run in
// k_force's last workgroups, and the last entry is the empty interval between
// two events; where the shuffle runs inside k_first_half its time is in the first entry
// and the fourth is the empty interval between two events.
extern "C" int ac4_md_kernel_times(ac4_md *md, int nsteps, double *ms) {
    AC4_REQUIRE(md && nsteps > 0 && ms, AC4_EARG, "kernel_times: bad arguments");
    if (!md->have_forces) TRY(ac4_md_calculate_forces(md, nullptr));
    hipStream_t s = md->stream;
    hipEvent_t ev[6];
    for (auto &e : ev) AC4_HIP(hipEventCreate(&e));
    double acc[5] = {0, 0, 0, 0, 0};
    for (int k = 0; k < nsteps; k++) {
        AC4_HIP(hipEventRecord(ev[0], s));
        if (!md->shuf_fused) launch_shuffle(md, 0);
        AC4_HIP(hipEventRecord(ev[1], s));
        launch_first_half(md, md->shuf_fused);
        AC4_HIP(hipEventRecord(ev[2], s));
        TRY(launch_rebuild(md));
        AC4_HIP(hipEventRecord(ev[3], s));
        TRY(launch_force<true>(md, k == nsteps - 1));
        AC4_HIP(hipEventRecord(ev[4], s));
        AC4_HIP(hipEventRecord(ev[5], s));
        AC4_HIP(hipEventSynchronize(ev[5]));
        float t[5];
        for (int q = 0; q < 5; q++) AC4_HIP(hipEventElapsedTime(&t[q], ev[q], ev[q + 1]));
        acc[3] += t[0]; acc[0] += t[1]; acc[1] += t[2]; acc[2] += t[3]; acc[4] += t[4];
    }
    for (auto &e : ev) (void)hipEventDestroy(e);
    for (int q = 0; q < 5; q++) ms[q] = acc[q] / nsteps;
    return check_err(md);
}

extern "C" int ac4_md_shuffle(ac4_md *md) {
    AC4_REQUIRE(md, AC4_EARG, "NULL handle");
    launch_shuffle(md, 1);
    AC4_HIP(hipGetLastError());
    std::vector<ChainS> c;
    TRY(get_chains(md, c));  // synchronises
    for (auto &e : c) e.shuffles += 1;
    return put_chains(md, c);
}

extern "C" int ac4_md_shuffle_uniforms(ac4_md *md, int r, double *u) {
    TRY(check_rep(md, r));
    AC4_REQUIRE(u, AC4_EARG, "NULL output");
    ChainS c;
    TRY(get_chain(md, r, &c));
    const RepC &R = md->reps_h[r];
    for (int comp = 0; comp < 3; comp++)
        for (int i = 0; i < R.nact; i++)
            u[comp * R.nact + i] = ac4_shuffle_uniform(R.key0, R.key1, (uint64_t)c.shuffles, comp, i);
    return AC4_OK;
}

extern "C" int ac4_md_stats(ac4_md *md, int r, double *out8) {
    TRY(check_rep(md, r));
    ChainS c;
    TRY(get_chain(md, r, &c));
    const RepC &R = md->reps_h[r];
    out8[0] = c.pe;
    out8[1] = c.vir;
    out8[2] = c.ke;
    out8[3] = c.inst_T;
    out8[4] = R.density * c.inst_T + c.vir / (R.L * R.L * R.L);  // print.c:83
    out8[5] = c.drift;
    out8[6] = c.heff;
    out8[7] = (double)c.step;
    return AC4_OK;
}

extern "C" int ac4_md_rebuilds(ac4_md *md, int r) {
    TRY(check_rep(md, r));
    ChainS c;
    TRY(get_chain(md, r, &c));
    return c.rebuilds;
}

extern "C" int ac4_md_sync(ac4_md *md) {
    AC4_REQUIRE(md, AC4_EARG, "NULL handle");
    AC4_HIP(hipStreamSynchronize(md->stream));
    return check_err(md);
}

extern "C" int ac4_philox4x32(const uint32_t *ctr4, const uint32_t *key2, uint32_t *out4) {
    AC4_REQUIRE(ctr4 && key2 && out4, AC4_EARG, "NULL argument");
    ac4_philox(ctr4, key2, out4);
    return AC4_OK;
}

// Reference-order x_u of every active slot into the export buffers and one
// copy to the host (xyz[3][ntot], slot offsets as ac4_md_slot_offset).
extern "C" int ac4_md_export_all(ac4_md *md, double *xu, double *yu, double *zu) {
    AC4_REQUIRE(md && xu && yu && zu, AC4_EARG, "export_all: bad arguments");
    if (!md->ex) {
        TRY(each_export_array(md, md->ntot, alloc_array));
    }
    hipLaunchKernelGGL(k_export, dim3(md->nblk), dim3(BLK), 0, md->stream, md->reps, md->blk_rep, md->blk_first,
                       md->P.id, md->P.xu, md->P.yu, md->P.zu, md->P.type, md->ex, md->ey, md->ez, md->et, -1);
    AC4_HIP(hipGetLastError());
    TRY(d2h(xu, (const double *)md->ex, md->ntot, md->stream));
    TRY(d2h(yu, (const double *)md->ey, md->ntot, md->stream));
    TRY(d2h(zu, (const double *)md->ez, md->ntot, md->stream));
    AC4_HIP(hipStreamSynchronize(md->stream));
    return check_err(md);
}

extern "C" int ac4_md_overlap_enable(ac4_md *md, int sample_every, int origin_every, int n_origin, int n_lags,
                                     double a) {
    AC4_REQUIRE(md && sample_every > 0 && origin_every > 0 && origin_every % sample_every == 0 && n_origin > 0 &&
                    n_lags > 0 && a > 0,
                AC4_EARG, "overlap_enable: bad arguments (origin_every must be a multiple of sample_every)");
    AC4_REQUIRE(!md->ox, AC4_ESTATE, "overlap accumulators already enabled");
    md->ov = OvCfg{sample_every, origin_every, n_origin, n_lags, a * a};
    TRY(each_overlap_array(md, md->R, md->ntot, n_origin, n_lags, alloc_array));
    std::vector<long long> none((size_t)md->R * n_origin, -1);
    AC4_HIP(hipMemcpy(md->ov_step, none.data(), sizeof(long long) * none.size(), hipMemcpyHostToDevice));
    return AC4_OK;
}

// Counts overlaps for the current step (every replica) and stores a new
// origin when due.  Call when the step counters are multiples of sample_every.
extern "C" int ac4_md_overlap_sample(ac4_md *md) {
    AC4_REQUIRE(md && md->ox, AC4_ESTATE, "overlap accumulators not enabled");
    hipStream_t s = md->stream;
    hipLaunchKernelGGL(k_ov_count, dim3(md->nblk, md->ov.n_origin), dim3(BLK), 0, s, md->reps, md->chain,
                       md->blk_rep, md->blk_first, md->ov, md->P.id, md->P.xu, md->P.yu, md->P.zu, md->ox, md->oy,
                       md->oz, md->ov_step, md->ov_cnt);
    const int nt = md->R * md->ov.n_origin;
    hipLaunchKernelGGL(k_ov_fold, dim3((nt + 255) / 256), dim3(256), 0, s, md->reps, md->chain, md->ov, md->R,
                       md->ov_step, md->ov_cnt, md->ov_q, md->ov_q2, md->ov_n);
    hipLaunchKernelGGL(k_ov_origin, dim3(md->nblk), dim3(BLK), 0, s, md->reps, md->chain, md->blk_rep,
                       md->blk_first, md->ov, md->P.id, md->P.xu, md->P.yu, md->P.zu, md->ox, md->oy, md->oz,
                       md->ov_step);
    AC4_HIP(hipGetLastError());
    return AC4_OK;
}

// Per-lag sums of replica r: sq[l] = sum_o Q_o(l*sample_every), sq2 likewise
// for Q^2, cnt[l] = number of origins (l = 0..n_lags).
extern "C" int ac4_md_overlap_get(ac4_md *md, int r, double *sq, double *sq2, int *cnt) {
    AC4_REQUIRE(md && md->ox && r >= 0 && r < md->R, AC4_EARG, "overlap_get: bad arguments");
    const size_t nl = md->ov.n_lags + 1, off = (size_t)r * nl;
    if (sq) TRY(d2h(sq, (const double *)md->ov_q + off, nl, md->stream));
    if (sq2) TRY(d2h(sq2, (const double *)md->ov_q2 + off, nl, md->stream));
    if (cnt) TRY(d2h(cnt, (const int *)md->ov_n + off, nl, md->stream));
    AC4_HIP(hipStreamSynchronize(md->stream));
    return AC4_OK;
}

// chi4(l) pooled over the listed replicas and their origins (k_ov_chi4):
// out3[3*l + {0,1,2}] = {Nbar*(<Q^2>-<Q>^2), <Q>, origins}, l = 0..n_lags.
extern "C" int ac4_md_overlap_chi4(ac4_md *md, int nlist, const int *list, double *out3) {
    AC4_REQUIRE(md && md->ox && nlist > 0 && list && out3, AC4_EARG, "overlap_chi4: bad arguments");
    for (int k = 0; k < nlist; k++)
        AC4_REQUIRE(list[k] >= 0 && list[k] < md->R && md->reps_h[list[k]].n > 0, AC4_EARG,
                    "overlap_chi4: entry %d names replica %d, which is not a running replica", k, list[k]);
    const int nl = md->ov.n_lags + 1;
    AC4_HIP(hipMemcpyAsync(md->ov_list, list, sizeof(int) * nlist, hipMemcpyHostToDevice, md->stream));
    hipLaunchKernelGGL(k_ov_chi4, dim3((nl + 255) / 256), dim3(256), 0, md->stream, md->reps, md->ov, md->ov_list,
                       nlist, md->ov_q, md->ov_q2, md->ov_n, md->ov_out);
    AC4_HIP(hipGetLastError());
    TRY(d2h(out3, (const double *)md->ov_out, 3 * (size_t)nl, md->stream));
    AC4_HIP(hipStreamSynchronize(md->stream));
    return AC4_OK;
}

// Starts replica r's accumulators afresh (no origins, zero sums).
extern "C" int ac4_md_overlap_reset(ac4_md *md, int r) {
    AC4_REQUIRE(md && md->ox && r >= 0 && r < md->R, AC4_EARG, "overlap_reset: bad arguments");
    const int nt = std::max(md->ov.n_origin, md->ov.n_lags + 1);
    hipLaunchKernelGGL(k_ov_reset, dim3((nt + 255) / 256), dim3(256), 0, md->stream, md->ov, r, md->ov_step,
                       md->ov_cnt, md->ov_q, md->ov_q2, md->ov_n);
    AC4_HIP(hipGetLastError());
    return AC4_OK;
}

extern "C" int ac4_md_slot_offset(const ac4_md *md, int slot) {
    if (!md || slot < 0 || slot >= md->R) return AC4_EARG;
    return md->reps_h[slot].off;
}

// Reference-order device copies of x_u and type of replica r for in-situ
// analysis (ac4_analysis.hip); the copies are complete when this returns.
extern "C" int ac4_md_device_xu(ac4_md *md, int r, const double **xu, const double **yu, const double **zu,
                                const int **type, int *n) {
    TRY(check_rep(md, r));
    if (!md->ex) {
        TRY(each_export_array(md, md->ntot, alloc_array));
    }
    hipLaunchKernelGGL(k_export, dim3(md->nblk), dim3(BLK), 0, md->stream, md->reps, md->blk_rep, md->blk_first,
                       md->P.id, md->P.xu, md->P.yu, md->P.zu, md->P.type, md->ex, md->ey, md->ez, md->et, r);
    AC4_HIP(hipGetLastError());
    AC4_HIP(hipStreamSynchronize(md->stream));
    const RepC &R = md->reps_h[r];
    *xu = md->ex + R.off;
    *yu = md->ey + R.off;
    *zu = md->ez + R.off;
    *type = md->et + R.off;
    *n = R.n;
    return AC4_OK;
}

// ------------------------------------------------------ exact checkpoints
// A replica's complete device state in slot (cell) order: particle arrays,
// forces, the last-rebuild positions, the cell tables, the neighbour list and
// the chain.  Restoring copies it back without recomputing anything, so the
// continued run is bitwise the one that was interrupted.  Slot and cell
// indices are stored replica-local, so the target may be another slot, of a
// handle with the same shape (precision, list capacity and layout, team
// width, skin) configured with the same replica parameters.
struct CkHead {
    char magic[8];
    int32_t version, n, nact, ncell, cap, lc, tpp, prec;
    double L, skin, T, f0;
    int32_t tau, pad;
    uint64_t seed, chain_bytes, total;
    // in-situ overlap state (ac4_md_overlap_enable) when the handle has it:
    // the origin snapshots in reference order, their steps, the per-lag sums
    int32_t ov_sample, ov_origin_every, ov_n_origin, ov_n_lags;
    double ov_a2;
};
static const char k_ck_magic[8] = {'A', 'C', '4', 'C', 'K', 'P', 'T', '1'};

static size_t ck_ov_bytes(const ac4_md *md, const RepC &R) {
    if (!md->ox) return 0;
    const size_t no = md->ov.n_origin, nl = md->ov.n_lags + 1;
    return no * 3 * (size_t)R.n * sizeof(double) + no * sizeof(long long) + nl * (2 * sizeof(double) + sizeof(int));
}
static size_t ck_bytes(const ac4_md *md, const RepC &R) {
    const size_t n = R.n, nc = R.ncell;
    return sizeof(CkHead) + sizeof(ChainS) + n * (15 * sizeof(double) + sizeof(double4) + sizeof(QPos)) +
           n * 7 * sizeof(int) + 3 * (size_t)R.nact + nc * 2 * sizeof(int) + n * sizeof(int) +
           nc * NRANGE * sizeof(int2) + (size_t)md->cap * n * sizeof(int) + ck_ov_bytes(md, R);
}

extern "C" long long ac4_md_checkpoint_size(ac4_md *md, int r) {
    if (check_rep(md, r) != AC4_OK) return AC4_EARG;
    return (long long)ck_bytes(md, md->reps_h[r]);
}

template <class T>
static int ck_io(bool save, T *dev, size_t n, char *&p, hipStream_t s) {
    if (save)
        TRY(d2h((T *)p, (const T *)dev, n, s));
    else
        TRY(h2d(dev, (const T *)p, n, s));
    p += n * sizeof(T);
    return AC4_OK;
}

static int ck_arrays(ac4_md *md, int r, bool save, char *p) {
    const RepC &R = md->reps_h[r];
    hipStream_t s = md->stream;
    const size_t g = R.off, n = R.n, c0 = R.off_cell, nc = R.ncell;
    double *dv[15] = {md->P.x, md->P.y, md->P.z, md->P.xu, md->P.yu, md->P.zu, md->P.px, md->P.py, md->P.pz,
                      md->xo, md->yo, md->zo, md->fx, md->fy, md->fz};
    for (double *a : dv) TRY(ck_io(save, a + g, n, p, s));
    TRY(ck_io(save, md->pos4 + g, n, p, s));
    TRY(ck_io(save, md->posq + g, n, p, s));
    int *iv[7] = {md->P.type, md->P.act, md->P.id, md->P.cell_ref, md->P.cell_of, md->nn, md->nn_ref};
    for (int *a : iv) TRY(ck_io(save, a + g, n, p, s));
    TRY(ck_io(save, md->kx + R.off_act, (size_t)R.nact, p, s));
    TRY(ck_io(save, md->ky + R.off_act, (size_t)R.nact, p, s));
    TRY(ck_io(save, md->kz + R.off_act, (size_t)R.nact, p, s));
    TRY(ck_io(save, md->cnt + c0, nc, p, s));
    TRY(ck_io(save, md->start + c0, nc, p, s));
    TRY(ck_io(save, md->members + g, n, p, s));
    int2 *rg = (int2 *)p;
    TRY(ck_io(save, md->ranges + c0 * NRANGE, nc * NRANGE, p, s));
    int *nl = (int *)p;
    TRY(ck_io(save, md->nl + g * md->cap, (size_t)md->cap * n, p, s));
    if (md->ox) {  // origin snapshots of this replica, its origin steps, its per-lag sums
        const size_t no = md->ov.n_origin, nl1 = md->ov.n_lags + 1;
        for (size_t o = 0; o < no; o++) {
            const size_t base = g * no + o * (size_t)R.cap_n;
            TRY(ck_io(save, md->ox + base, n, p, s));
            TRY(ck_io(save, md->oy + base, n, p, s));
            TRY(ck_io(save, md->oz + base, n, p, s));
        }
        TRY(ck_io(save, md->ov_step + (size_t)r * no, no, p, s));
        TRY(ck_io(save, md->ov_q + (size_t)r * nl1, nl1, p, s));
        TRY(ck_io(save, md->ov_q2 + (size_t)r * nl1, nl1, p, s));
        TRY(ck_io(save, md->ov_n + (size_t)r * nl1, nl1, p, s));
    }
    AC4_HIP(hipStreamSynchronize(s));
    if (save) {  // replica-local slot indices
        for (size_t k = 0; k < nc * NRANGE; k++)
            if (rg[k].y > rg[k].x) { rg[k].x -= (int)g; rg[k].y -= (int)g; }
        for (size_t k = 0; k < (size_t)md->cap * n; k++) nl[k] -= (int)g;
    }
    return AC4_OK;
}

extern "C" int ac4_md_checkpoint(ac4_md *md, int r, void *buf, long long cap) {
    TRY(check_rep(md, r));
    const RepC &R = md->reps_h[r];
    AC4_REQUIRE(buf && cap >= (long long)ck_bytes(md, R), AC4_EARG, "checkpoint: buffer smaller than %zu bytes",
                ck_bytes(md, R));
    AC4_REQUIRE(R.n > 0, AC4_ESTATE, "checkpoint: slot %d is idle", r);
    AC4_HIP(hipStreamSynchronize(md->stream));
    CkHead h;
    memset(&h, 0, sizeof h);
    memcpy(h.magic, k_ck_magic, 8);
    h.version = 3; h.n = R.n; h.nact = R.nact; h.ncell = R.ncell; h.cap = md->cap; h.lc = R.lc; h.tpp = R.tpp;
    h.prec = md->prec; h.L = R.L; h.skin = R.skin; h.T = R.T; h.f0 = R.f0; h.tau = R.tau;
    h.seed = (uint64_t)R.key0 | ((uint64_t)R.key1 << 32);
    h.chain_bytes = sizeof(ChainS);
    h.total = ck_bytes(md, R);
    if (md->ox) {
        h.ov_sample = md->ov.sample_every; h.ov_origin_every = md->ov.origin_every;
        h.ov_n_origin = md->ov.n_origin; h.ov_n_lags = md->ov.n_lags; h.ov_a2 = md->ov.a2;
    }
    char *p = (char *)buf;
    memcpy(p, &h, sizeof h);
    p += sizeof h;
    ChainS c;
    TRY(get_chain(md, r, &c));
    memcpy(p, &c, sizeof c);
    p += sizeof c;
    return ck_arrays(md, r, true, p);
}

extern "C" int ac4_md_restore(ac4_md *md, int r, const void *buf, long long len) {
    TRY(check_rep(md, r));
    const RepC &R = md->reps_h[r];
    AC4_REQUIRE(buf && len >= (long long)sizeof(CkHead), AC4_EARG, "restore: no checkpoint");
    CkHead h;
    memcpy(&h, buf, sizeof h);
    AC4_REQUIRE(!memcmp(h.magic, k_ck_magic, 8) && h.version == 3 && h.chain_bytes == sizeof(ChainS), AC4_EARG,
                "restore: not a checkpoint of this library version");
    AC4_REQUIRE((long long)h.total == len && h.total == ck_bytes(md, R), AC4_EARG,
                "restore: checkpoint of %lld bytes does not fit slot %d", len, r);
    AC4_REQUIRE(h.n == R.n && h.nact == R.nact && h.ncell == R.ncell && h.cap == md->cap && h.lc == R.lc &&
                    h.tpp == R.tpp && h.prec == md->prec && h.L == R.L && h.skin == R.skin,
                AC4_EARG, "restore: the slot's replica or handle shape differs from the checkpoint's");
    const bool ov_same = md->ox ? (h.ov_sample == md->ov.sample_every && h.ov_origin_every == md->ov.origin_every &&
                                   h.ov_n_origin == md->ov.n_origin && h.ov_n_lags == md->ov.n_lags &&
                                   h.ov_a2 == md->ov.a2)
                                : h.ov_n_origin == 0;
    AC4_REQUIRE(ov_same, AC4_EARG, "restore: the overlap accumulators of the checkpoint and the handle differ");
    const uint64_t seed = (uint64_t)R.key0 | ((uint64_t)R.key1 << 32);
    AC4_REQUIRE(h.seed == seed && h.T == R.T && h.f0 == R.f0 && h.tau == R.tau, AC4_EARG,
                "restore: slot %d runs seed %llu, T %g, f0 %g, tau %d; the checkpoint seed %llu, T %g, f0 %g, tau %d",
                r, (unsigned long long)seed, R.T, R.f0, R.tau, (unsigned long long)h.seed, h.T, h.f0, h.tau);
    std::vector<char> tmp((const char *)buf, (const char *)buf + len);  // local copy: indices are rebased
    char *p = tmp.data() + sizeof h;
    ChainS c;
    memcpy(&c, p, sizeof c);
    p += sizeof c;
    const size_t g = R.off, n = R.n, nc = R.ncell;
    // rebase the replica-local indices onto this slot before copying
    char *q = p + n * (15 * sizeof(double) + sizeof(double4) + sizeof(QPos)) + n * 7 * sizeof(int) +
              3 * (size_t)R.nact + nc * 2 * sizeof(int) + n * sizeof(int);
    int2 *rg = (int2 *)q;
    for (size_t k = 0; k < nc * NRANGE; k++)
        if (rg[k].y > rg[k].x) { rg[k].x += (int)g; rg[k].y += (int)g; }
    int *nl = (int *)(q + nc * NRANGE * sizeof(int2));
    for (size_t k = 0; k < (size_t)md->cap * n; k++) nl[k] += (int)g;
    TRY(ck_arrays(md, r, false, p));
    c.done_blocks = 0u;
    c.bin_done = 0u;
    return put_chain(md, r, &c);
}
