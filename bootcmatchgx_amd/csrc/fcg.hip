// fcg.hip -- flexible CG vector kernels (flexibileConjugateGradients_v3,
// src/solver/fcg/FCG.cu:27-175) with the scalar recurrences kept on the
// device.  The reference reads every dot product back to the host
// (triple_innerproduct, src/op/triple_inner_product.cu:64-101; norm_MPI,
// src/datastruct/vector.cu:492-516); here the scalars, the convergence test
// and the iteration count live in FcgState so a whole iteration can be
// replayed from a hipGraph and the host only polls a flag.
//
// Reductions are deterministic: a fixed number of partial blocks (a function
// of n and k only), a fixed in-block tree, then one block per column (or the
// workgroup that finishes last, few partials) summing them in a fixed tree.  k vectors are interleaved (x[i*k + c]); every
// column has its own scalars and stop flag.
#include "kernels.h"

#include <algorithm>

namespace bcmgx {

// Partial-sum blocks of the streaming FCG and CG kernels: a function of n and k
// only, so the reduction order never changes.  These kernels are bound by
// memory, so what counts is bytes in flight: a block per 512 elements (two a
// thread) until the 256 CUs hold four blocks each.  Counting rows alone (one
// block per 2048 rows) left the chip idle on several columns: the update of
// 65600 x 64 took 463 us in 33 blocks and takes 49 in 1024, 720000 x 16
// 225 -> 132 us, 131150 x 5 (CG) 31 -> 7.5 us, 125000 x 1 6.2 -> 4.4 us.  Blocks
// of 256 or 1024 elements are within noise of these; 2048 blocks gain 5 % at
// 720000 x 16 and lose 8 % at 2097152 x 32 and 1-2 us in each of the two
// kernels that sum the partials.
int fcg_partial_blocks(int n, int k) {
    long long b = ((long long)n * k + 511) / 512;
    if (b < 1) b = 1;
    if (b > 1024) b = 1024;
    return (int)b;
}

// the streaming kernels' split of a block: its first R * k threads (R = WG / k)
// take R rows of k columns each, one element a thread, so a block reads
// consecutive elements and keeps its lanes busy for any k (255 of 256 at k = 5,
// 231 at k = 33), and s[][] holds the rows' sums in the same order as a split by
// a power of two when k is one
struct RowSplit {
    int R, rl, c;
    __device__ explicit RowSplit(int k) {
        R = WG / k;
        rl = threadIdx.x / k;
        c = threadIdx.x - rl * k;
    }
    __device__ bool active() const { return rl < R; }
    // s[c] <- the sum of column c over the block's R rows, in a fixed tree
    template <int NV>
    __device__ void sum(double (*s)[WG], int k) const {
        int h = 1;
        while (2 * h < R) h <<= 1;
        for (; h > 0; h >>= 1) {
            if (rl < h && rl + h < R)
#pragma unroll
                for (int m = 0; m < NV; m++) s[m][threadIdx.x] += s[m][threadIdx.x + h * k];
            __syncthreads();
        }
    }
};

// sum partials of column blockIdx.x in a fixed tree; thread 0 gets the totals
template <int NV>
__device__ void sum_partials(const double* __restrict__ partials, int nblk, int k, int c, double* out, double (*s)[WG]) {
    int tid = threadIdx.x;
    double acc[NV];
#pragma unroll
    for (int m = 0; m < NV; m++) acc[m] = 0.0;
    for (int b = tid; b < nblk; b += WG)
#pragma unroll
        for (int m = 0; m < NV; m++) acc[m] += partials[((long long)b * k + c) * 3 + m];
#pragma unroll
    for (int m = 0; m < NV; m++) s[m][tid] = acc[m];
    __syncthreads();
    for (int st = WG / 2; st > 0; st >>= 1) {
        if (tid < st)
#pragma unroll
            for (int m = 0; m < NV; m++) s[m][tid] += s[m][tid + st];
        __syncthreads();
    }
    if (tid == 0)
#pragma unroll
        for (int m = 0; m < NV; m++) out[m] = s[m][0];
}

// What follows a reduction, per column from its totals.  FIN_SCALARS: FCG's theta, delta,
// theta2; FIN_STEP: FCG's ||r||, iteration count and convergence; FIN_BETA, FIN_ALPHA,
// FIN_ALPHA0 (first iteration) and FIN_CG: the same of CG.
enum { FIN_NONE, FIN_SCALARS, FIN_STEP, FIN_BETA, FIN_ALPHA, FIN_ALPHA0, FIN_CG };
constexpr int fin_values(int fin) { return fin == FIN_SCALARS ? 3 : fin == FIN_ALPHA0 ? 2 : 1; }
struct FinArgs {
    FcgState* st;
    int* all_done;
    int* ndone;
    unsigned* tickets;  // null: a kernel of its own sums the partials
    double rtol;
    int itnlim, phase;
};

template <int FIN>
__device__ void fin_column(FcgState& S, const double* tot, const FinArgs& a, int k) {
    bool stop = false;
    if constexpr (FIN == FIN_SCALARS) {
        if (S.done) return;
        S.alpha = tot[0];
        S.beta = tot[1];
        S.gamma = tot[2];
        S.theta = S.gamma / S.delta;                        // FCG.cu:132
        S.delta = S.beta - ((S.gamma * S.gamma) / S.delta);  // FCG.cu:135
        S.theta2 = S.alpha / S.delta;                       // FCG.cu:136
        if (a.phase == 0) {  // the x step of this iteration waits for the pair's second update
            S.pend = S.theta2;
            S.pad1 = 1;
        }
    } else if constexpr (FIN == FIN_STEP) {
        // l2 = ||r||; iter++; stop when !(l2 > rtol*delta0 && iter < itnlim)  (FCG.cu:146-156)
        if (a.phase == 1) S.pad1 = 0;  // this pair's update added the waiting step
        if (S.done) return;
        S.l2 = sqrt(tot[0]);
        S.iter += 1;
        stop = !(S.l2 > a.rtol * S.delta0 && S.iter < a.itnlim);
    } else if constexpr (FIN == FIN_BETA) {
        // rho = r.u, beta = rho / rho_prev  (CG_HS.cu:89-101)
        if (S.done) return;
        S.alpha = tot[0];
        S.theta = S.alpha / S.delta;
    } else if constexpr (FIN == FIN_ALPHA || FIN == FIN_ALPHA0) {
        // (first iteration: rho = u.r) gamma = p.s, alpha = rho / gamma; rho_prev = rho  (CG_HS.cu:112-129)
        if (S.done) return;
        if constexpr (FIN == FIN_ALPHA0) S.alpha = tot[1];
        S.gamma = tot[0];
        S.theta2 = S.alpha / S.gamma;
        S.delta = S.alpha;
    } else if constexpr (FIN == FIN_CG) {
        // l2 = ||r||; converged when l2 < rtol delta0, else the iteration count
        // advances and itnlim stops the column (CG_HS.cu:134-163)
        if (S.done) return;
        S.l2 = sqrt(tot[0]);
        if (S.l2 < a.rtol * S.delta0) {
            S.pad0 = 1;
            stop = true;
        } else if (++S.iter >= a.itnlim) {
            stop = true;
        }
    }
    if (stop) {
        S.done = 1;
        if (atomicAdd(a.ndone, 1) + 1 == k) *a.all_done = 1;
    }
}

// The partials of a kernel of their own, one workgroup per column
template <int FIN>
__global__ __launch_bounds__(WG) void k_final(const double* __restrict__ partials, int nblk, int k, FinArgs a) {
    constexpr int NV = fin_values(FIN);
    if (*a.all_done) return;
    __shared__ double s[NV][WG];
    double tot[NV];
    int c = blockIdx.x;
    sum_partials<NV>(partials, nblk, k, c, tot, s);
    if (threadIdx.x == 0) fin_column<FIN>(a.st[c], tot, a, k);
}

// The end of a reducing kernel whose block's sums are in s[m][c] (m < NV, c < k): its partials
// are left for k_final, or (tickets given) the workgroup that finishes last sums everyone's,
// one wave a column, and does k_final's work: a launch of its own costs 4-5 us in a replayed
// graph for less than one of work.  A partial is exchanged into its place at device scope and
// the old value waited for, so it is visible across the XCDs before the workgroup takes its
// ticket; no L2 is written back for it.  Tickets are taken 32 workgroups to a counter and then
// 32 counters to one (1024 on one word queue up for microseconds), 64 bytes apart; the last
// taker clears each for the next kernel.
template <int FIN>
__device__ __forceinline__ void block_end(double (*s)[WG], double* partials, int k, const FinArgs& a) {
    constexpr int NV = fin_values(FIN);
    int tid = threadIdx.x, nblk = gridDim.x;
    if (!a.tickets) {
        if (tid < k) {
#pragma unroll
            for (int m = 0; m < NV; m++) partials[((long long)blockIdx.x * k + tid) * 3 + m] = s[m][tid];
        }
        return;
    }
    if (tid < k) {
        unsigned long long old[NV];
#pragma unroll
        for (int m = 0; m < NV; m++)
            old[m] = __hip_atomic_exchange((unsigned long long*)partials + ((long long)blockIdx.x * k + tid) * 3 + m,
                                           (unsigned long long)__double_as_longlong(s[m][tid]), __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int m = 0; m < NV; m++) asm volatile("" ::"v"(old[m]));  // back, so at the device's point of coherence
    }
    __shared__ int last;
    __syncthreads();
    if (tid == 0) {
        unsigned group = blockIdx.x / 32, groups = (nblk + 31) / 32;
        unsigned size = group + 1 < groups ? 32 : nblk - group * 32;
        unsigned* mine = a.tickets + 16 * (1 + group);
        last = 0;
        if (__hip_atomic_fetch_add(mine, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == size - 1) {
            __hip_atomic_store(mine, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (__hip_atomic_fetch_add(a.tickets, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == groups - 1) {
                __hip_atomic_store(a.tickets, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                last = 1;
            }
        }
    }
    __syncthreads();
    if (!last) return;
    for (int c = tid / 64; c < k; c += WG / 64) {
        double acc[NV];
#pragma unroll
        for (int m = 0; m < NV; m++) acc[m] = 0.0;
        for (int b0 = tid & 63; b0 < nblk; b0 += 4 * 64) {  // four blocks' partials in flight
            double v[4][NV];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                int b = b0 + u * 64 < nblk ? b0 + u * 64 : b0;
#pragma unroll
                for (int m = 0; m < NV; m++)
                    v[u][m] = __longlong_as_double((long long)__hip_atomic_load(
                        (const unsigned long long*)partials + ((long long)b * k + c) * 3 + m, __ATOMIC_RELAXED,
                        __HIP_MEMORY_SCOPE_AGENT));
            }
#pragma unroll
            for (int u = 0; u < 4; u++)
#pragma unroll
                for (int m = 0; m < NV; m++) acc[m] += b0 + u * 64 < nblk ? v[u][m] : 0.0;
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1)
#pragma unroll
            for (int m = 0; m < NV; m++) acc[m] += __shfl_xor(acc[m], o, 64);
        if ((tid & 63) == 0) fin_column<FIN>(a.st[c], acc, a, k);
    }
}

// The finishing step in the kernel to 1024 totals (workgroups by columns), else k_final: the
// one workgroup that sums them is then slower than the launch it saves.  One column, 7-point
// 10^3 1390 -> 1340 us a solve with its setup, 50^3 5.06 -> 4.83 ms, 160^3 (FP32 cycle) 67.2 -> 66.7
// ms; 5 columns in 1024 workgroups (CG, 131150 rows) 9.5 -> 9.9 ms, so they keep k_final.
constexpr int FIN_MAX_TOTALS = 1024;
static FinArgs fin_args(const FcgBufs& f, int phase = 0) {
    return FinArgs{f.st, f.all_done, f.all_done + 1, f.nblk * f.k <= FIN_MAX_TOTALS ? f.tickets : nullptr, f.rtol, f.itnlim, phase};
}
template <int FIN>
static void fin_launch(Context* c, const FcgBufs& f, int nblk, const FinArgs& a) {
    k_final<FIN><<<f.k, WG, 0, c->stream>>>(f.partials, nblk, f.k, a);
    BCMGX_LAUNCHED();
}

// NV dot products per column over a row range; partials[(blk*k + c)*3 + m]
template <int NV, int FIN = FIN_NONE>
__global__ __launch_bounds__(WG) void k_dots(int n, int k, const double* __restrict__ a0, const double* __restrict__ b0,
                                             const double* __restrict__ a1, const double* __restrict__ b1,
                                             const double* __restrict__ a2, const double* __restrict__ b2,
                                             double* __restrict__ partials, const int* all_done, FinArgs fa) {
    if (all_done && *all_done) return;
    __shared__ double s[NV][WG];
    int tid = threadIdx.x;
    const RowSplit sp(k);
    int c = sp.c;
    double acc[NV];
#pragma unroll
    for (int m = 0; m < NV; m++) acc[m] = 0.0;
    if (sp.active()) {
        for (long long i = (long long)blockIdx.x * sp.R + sp.rl; i < n; i += (long long)gridDim.x * sp.R) {
            long long o = i * k + c;
            acc[0] += a0[o] * b0[o];
            if (NV > 1) acc[1] += a1[o] * b1[o];
            if (NV > 2) acc[2] += a2[o] * b2[o];
        }
    }
#pragma unroll
    for (int m = 0; m < NV; m++) s[m][tid] = acc[m];
    __syncthreads();
    sp.sum<NV>(s, k);
    if constexpr (FIN != FIN_NONE) {
        block_end<FIN>(s, partials, k, fa);
    } else if (tid < k) {
#pragma unroll
        for (int m = 0; m < NV; m++) partials[((long long)blockIdx.x * k + tid) * 3 + m] = s[m][tid];
    }
}

// mode 0: initial residual norm (delta0); mode 1: post-initial-step norm
__global__ __launch_bounds__(WG) void k_norm_final(const double* __restrict__ partials, int nblk, int k, FcgState* st,
                                                   int mode, int* all_done, int* ndone) {
    __shared__ double s[1][WG];
    double tot[1];
    int c = blockIdx.x;
    sum_partials<1>(partials, nblk, k, c, tot, s);
    if (threadIdx.x == 0) {
        double l2 = sqrt(tot[0]);
        st[c].l2 = l2;
        if (mode == 0) {
            st[c].delta0 = l2;
            st[c].iter = 0;
            st[c].done = 0;
            st[c].pend = 0.0;
            st[c].pad1 = 0;
            if (l2 == 0.0) {  // b == A x already: nothing to iterate on
                st[c].done = 1;
                if (atomicAdd(ndone, 1) + 1 == k) *all_done = 1;
            }
        }
    }
}

// ||r||^2 partials in k_dots<1>'s blocks and order, with the cycle's
// level-0 entry (FP32: F = (float) r, X = F/M) written on the way, as k_update does
__global__ __launch_bounds__(WG) void k_norm_entry(int n, int k, const double* __restrict__ r,
                                                   double* __restrict__ partials, FcgEntry e) {
    __shared__ double s[1][WG];
    int tid = threadIdx.x;
    const RowSplit sp(k);
    int c = sp.c;
    double acc = 0.0;
    if (sp.active()) {
        for (long long i = (long long)blockIdx.x * sp.R + sp.rl; i < n; i += (long long)gridDim.x * sp.R) {
            long long o = i * k + c;
            double rr = r[o];
            acc += rr * rr;
            e.put(o, i, rr);
        }
    }
    s[0][tid] = acc;
    __syncthreads();
    sp.sum<1>(s, k);
    if (tid < k) partials[((long long)blockIdx.x * k + tid) * 3] = s[0][tid];
}

void fcg_norm_entry(Context* c, const FcgBufs& f, const double* r, int mode, const FcgEntry& e) {
    k_norm_entry<<<f.nblk, WG, 0, c->stream>>>(f.n, f.k, r, f.partials, e);
    BCMGX_LAUNCHED();
    k_norm_final<<<f.k, WG, 0, c->stream>>>(f.partials, f.nblk, f.k, f.st, mode, f.all_done, f.all_done + 1);
    BCMGX_LAUNCHED();
}

void fcg_norm(Context* c, const FcgBufs& f, const double* v, int mode) {
    k_dots<1><<<f.nblk, WG, 0, c->stream>>>(f.n, f.k, v, v, nullptr, nullptr, nullptr, nullptr, f.partials, nullptr, FinArgs());
    BCMGX_LAUNCHED();
    k_norm_final<<<f.k, WG, 0, c->stream>>>(f.partials, f.nblk, f.k, f.st, mode, f.all_done, f.all_done + 1);
    BCMGX_LAUNCHED();
}

__global__ __launch_bounds__(WG) void k_init_scalars(const double* __restrict__ partials, int nblk, int k, FcgState* st) {
    __shared__ double s[2][WG];
    double tot[2];
    int c = blockIdx.x;
    sum_partials<2>(partials, nblk, k, c, tot, s);
    if (threadIdx.x == 0) {
        FcgState& S = st[c];
        S.alpha = tot[0];
        S.beta = tot[1];
        S.delta = S.beta;                // FCG.cu:84
        S.theta = S.done ? 0.0 : S.alpha / S.delta;  // FCG.cu:85
        S.gamma = 0.0;
    }
}

void fcg_init_dots(Context* c, const FcgBufs& f, const double* r, const double* v, const double* w) {
    k_dots<2><<<f.nblk, WG, 0, c->stream>>>(f.n, f.k, r, v, w, v, nullptr, nullptr, f.partials, nullptr, FinArgs());
    BCMGX_LAUNCHED();
    fcg_init_scalars(c, f, f.nblk);
}

void fcg_init_scalars(Context* c, const FcgBufs& f, int nblk) {
    k_init_scalars<<<f.k, WG, 0, c->stream>>>(f.partials, nblk, f.k, f.st);
    BCMGX_LAUNCHED();
}

// v in FP64, or the FP32 cycle result widened exactly
template <typename VT>
__global__ __launch_bounds__(WG) void k_init_update(int n, int k, const FcgState* __restrict__ st, double* __restrict__ x,
                                                    double* __restrict__ r, const VT* __restrict__ v,
                                                    const double* __restrict__ w, double* __restrict__ d,
                                                    double* __restrict__ q, FcgEntry e) {
    long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (long long)n * k) return;
    int i = (int)(t / k);
    int c = (int)(t - (long long)i * k);
    double th = st[c].theta;
    double vv = (double)v[t], ww = w[t];
    double rr = r[t];
    if (!st[c].done) {
        x[t] += th * vv;      // my_axpby(v, x, theta, 1): y += a x  (basic.cu:114-130)
        rr += -th * ww;       // my_axpby(w, r, -theta, 1)
        r[t] = rr;
    }
    d[t] = vv;                // d = clone(v), q = clone(w)  (FCG.cu:98-99)
    q[t] = ww;
    e.put(t, i, rr);
}

void fcg_init_update(Context* c, const FcgBufs& f, double* x, double* r, const double* v, const double* w, double* d, double* q,
                     const FcgEntry& e) {
    long long nk = (long long)f.n * f.k;
    if (!nk) return;
    k_init_update<double><<<grid_for(nk, WG), WG, 0, c->stream>>>(f.n, f.k, f.st, x, r, v, w, d, q, e);
    BCMGX_LAUNCHED();
}

void fcg_init_update_z32(Context* c, const FcgBufs& f, double* x, double* r, const float* z, const double* w, double* d,
                         double* q, const FcgEntry& e) {
    long long nk = (long long)f.n * f.k;
    if (!nk) return;
    k_init_update<float><<<grid_for(nk, WG), WG, 0, c->stream>>>(f.n, f.k, f.st, x, r, z, w, d, q, e);
    BCMGX_LAUNCHED();
}

void fcg_scalars3(Context* c, const FcgBufs& f, int nblk, int phase) { fin_launch<FIN_SCALARS>(c, f, nblk, fin_args(f, phase)); }

void fcg_dots3(Context* c, const FcgBufs& f, const double* r, const double* p0, const double* w0, const double* w1, int phase) {
    FinArgs a = fin_args(f, phase);
    k_dots<3, FIN_SCALARS><<<f.nblk, WG, 0, c->stream>>>(f.n, f.k, r, p0, w0, p0, w1, p0, f.partials, f.all_done, a);
    BCMGX_LAUNCHED();
    if (!a.tickets) fin_launch<FIN_SCALARS>(c, f, f.nblk, a);
}

// double_merged_axpy(P1, P0, x, -theta, theta2); double_merged_axpy(W1, W0, r, -theta, -theta2)
// (double_merged_axpy.cu:28-39), fused, with the partial sums of r.r.  The x
// step is taken every second iteration: phase 0 leaves x alone (its theta2
// waits in pend, its direction stays in the buffer that is p1 next time),
// phase 1 forms x = theta2' t' + (pend p1 + x) -- the two steps in the
// reference's order, so x has the same bits -- and saves one x read and write.
template <int PHASE>
__global__ __launch_bounds__(WG) void k_update(int n, int k, const FcgState* st,
                                               double* __restrict__ p0, const double* __restrict__ p1,
                                               double* __restrict__ w0, const double* __restrict__ w1,
                                               double* __restrict__ x, double* __restrict__ r,
                                               double* __restrict__ partials, const int* all_done,
                                               FcgEntry e, FinArgs fa) {
    if (*all_done) return;
    __shared__ double s[1][WG];
    int tid = threadIdx.x;
    const RowSplit sp(k);
    int c = sp.c;
    double acc = 0.0;
    if (sp.active()) {
        const FcgState S = st[c];
        double mth = -S.theta, th2 = S.theta2, mth2 = -S.theta2;
        bool waiting = PHASE == 1 && S.pad1;  // the pair's first step, still to be added
        double pend = S.pend;
        for (long long i = (long long)blockIdx.x * sp.R + sp.rl; i < n; i += (long long)gridDim.x * sp.R) {
            long long o = i * k + c;
            double rr;
            if (!S.done) {
                double p1o = p1[o];
                double t = mth * p1o + p0[o];
                if constexpr (PHASE == 1) {
                    double xo = x[o];
                    double xw = pend * p1o + xo;
                    x[o] = th2 * t + (waiting ? xw : xo);
                }
                p0[o] = t;
                double u = mth * w1[o] + w0[o];
                rr = mth2 * u + r[o];
                r[o] = rr;
                w0[o] = u;
            } else {
                rr = r[o];
                if (waiting) x[o] = pend * p1[o] + x[o];
            }
            acc += rr * rr;
            e.put(o, i, rr);
        }
    }
    s[0][tid] = acc;
    __syncthreads();
    sp.sum<1>(s, k);
    block_end<FIN_STEP>(s, partials, k, fa);
}

void fcg_update(Context* c, const FcgBufs& f, double* p0, const double* p1, double* w0, const double* w1, double* x, double* r,
                int phase, const FcgEntry& e) {
    FinArgs a = fin_args(f, phase);
    if (phase == 0) k_update<0><<<f.nblk, WG, 0, c->stream>>>(f.n, f.k, f.st, p0, p1, w0, w1, x, r, f.partials, f.all_done, e, a);
    else k_update<1><<<f.nblk, WG, 0, c->stream>>>(f.n, f.k, f.st, p0, p1, w0, w1, x, r, f.partials, f.all_done, e, a);
    BCMGX_LAUNCHED();
    if (!a.tickets) fin_launch<FIN_STEP>(c, f, f.nblk, a);
}

// k_update with z in FP32 (widened exactly) and p, w updated in place
template <int PHASE>
__global__ __launch_bounds__(WG) void k_update_z32(int n, int k, const FcgState* st,
                                                   const float* __restrict__ z, double* __restrict__ p,
                                                   const double* __restrict__ w0, double* __restrict__ w,
                                                   double* __restrict__ x, double* __restrict__ r,
                                                   double* __restrict__ partials, const int* all_done,
                                                   FcgEntry e, FinArgs fa) {
    if (*all_done) return;
    __shared__ double s[1][WG];
    int tid = threadIdx.x;
    const RowSplit sp(k);
    int c = sp.c;
    double acc = 0.0;
    if (sp.active()) {
        const FcgState S = st[c];
        double mth = -S.theta, th2 = S.theta2, mth2 = -S.theta2;
        bool waiting = PHASE == 1 && S.pad1;
        double pend = S.pend;
        for (long long i = (long long)blockIdx.x * sp.R + sp.rl; i < n; i += (long long)gridDim.x * sp.R) {
            long long o = i * k + c;
            double rr;
            if (!S.done) {
                double po = p[o];
                double t = mth * po + (double)z[o];
                if constexpr (PHASE == 1) {
                    double xo = x[o];
                    double xw = pend * po + xo;
                    x[o] = th2 * t + (waiting ? xw : xo);
                }
                p[o] = t;
                double u = mth * w[o] + w0[o];
                rr = mth2 * u + r[o];
                r[o] = rr;
                w[o] = u;
            } else {
                rr = r[o];
                if (waiting) x[o] = pend * p[o] + x[o];
            }
            acc += rr * rr;
            e.put(o, i, rr);
        }
    }
    s[0][tid] = acc;
    __syncthreads();
    sp.sum<1>(s, k);
    block_end<FIN_STEP>(s, partials, k, fa);
}

void fcg_update_z32(Context* c, const FcgBufs& f, const float* z, double* p, const double* w0, double* w, double* x, double* r,
                    int phase, const FcgEntry& e) {
    FinArgs a = fin_args(f, phase);
    if (phase == 0) k_update_z32<0><<<f.nblk, WG, 0, c->stream>>>(f.n, f.k, f.st, z, p, w0, w, x, r, f.partials, f.all_done, e, a);
    else k_update_z32<1><<<f.nblk, WG, 0, c->stream>>>(f.n, f.k, f.st, z, p, w0, w, x, r, f.partials, f.all_done, e, a);
    BCMGX_LAUNCHED();
    if (!a.tickets) fin_launch<FIN_STEP>(c, f, f.nblk, a);
}

__global__ __launch_bounds__(WG) void k_flush_pending(int n, int k, FcgState* st, const double* __restrict__ t,
                                                      double* __restrict__ x) {
    const RowSplit sp(k);
    int c = sp.c;
    if (!sp.active() || !st[c].pad1) return;
    double pend = st[c].pend;
    for (long long i = (long long)blockIdx.x * sp.R + sp.rl; i < n; i += (long long)gridDim.x * sp.R) {
        long long o = i * k + c;
        x[o] = pend * t[o] + x[o];
    }
}

__global__ void k_clear_pending(int k, FcgState* st) {
    int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c < k) st[c].pad1 = 0;
}

void fcg_clear_pending(Context* c, const FcgBufs& f) {
    k_clear_pending<<<1, 64, 0, c->stream>>>(f.k, f.st);
    BCMGX_LAUNCHED();
}

void fcg_flush_pending(Context* c, const FcgBufs& f, const double* t, double* x) {
    k_flush_pending<<<f.nblk, WG, 0, c->stream>>>(f.n, f.k, f.st, t, x);
    BCMGX_LAUNCHED();
    k_clear_pending<<<1, 64, 0, c->stream>>>(f.k, f.st);
    BCMGX_LAUNCHED();
}

// ---- CG (Hestenes-Stiefel), cg_hs (src/solver/cghs/CG_HS.cu:24-172) ---------
// FcgState fields as used by CG: alpha = rho = r.u of the current iteration,
// delta = rho of the previous one, theta = beta, gamma = p.s, theta2 = alpha
// (the step), pad0 = 1 once the column converged.

// delta0 = ||r|| (stop_criterion 1) or 1 (CG_HS.cu:74-79); a zero initial
// residual stops the column at once (the reference would divide 0 by 0)
__global__ __launch_bounds__(WG) void k_cg_init(const double* __restrict__ partials, int nblk, int k, FcgState* st,
                                                int stopcrit, int* all_done, int* ndone) {
    __shared__ double s[1][WG];
    double tot[1];
    int c = blockIdx.x;
    sum_partials<1>(partials, nblk, k, c, tot, s);
    if (threadIdx.x == 0) {
        FcgState& S = st[c];
        double l2 = sqrt(tot[0]);
        S.l2 = l2;
        S.delta0 = stopcrit == 1 ? l2 : 1.0;
        S.iter = 0;
        S.done = 0;
        S.pad0 = 0;
        S.delta = 0.0;
        if (l2 == 0.0) {
            S.done = 1;
            S.pad0 = 1;
            if (atomicAdd(ndone, 1) + 1 == k) *all_done = 1;
        }
    }
}

void cg_init(Context* c, const FcgBufs& f, const double* r, int stopcrit) {
    k_dots<1><<<f.nblk, WG, 0, c->stream>>>(f.n, f.k, r, r, nullptr, nullptr, nullptr, nullptr, f.partials, nullptr, FinArgs());
    BCMGX_LAUNCHED();
    k_cg_init<<<f.k, WG, 0, c->stream>>>(f.partials, f.nblk, f.k, f.st, stopcrit, f.all_done, f.all_done + 1);
    BCMGX_LAUNCHED();
}

// p = 1 u + beta p  (my_axpby, basic.cu:114-130; CG_HS.cu:103-107)
__global__ __launch_bounds__(WG) void k_cg_direction(int n, int k, const FcgState* __restrict__ st,
                                                     const double* __restrict__ u, double* __restrict__ p,
                                                     const int* __restrict__ all_done) {
    if (*all_done) return;
    const RowSplit sp(k);
    int c = sp.c;
    if (!sp.active() || st[c].done) return;
    double be = st[c].theta;
    for (long long i = (long long)blockIdx.x * sp.R + sp.rl; i < n; i += (long long)gridDim.x * sp.R) {
        long long o = i * k + c;
        p[o] = 1.0 * u[o] + be * p[o];
    }
}

void cg_beta_direction(Context* c, const FcgBufs& f, const double* r, const double* u, double* p) {
    FinArgs a = fin_args(f);
    k_dots<1, FIN_BETA><<<f.nblk, WG, 0, c->stream>>>(f.n, f.k, r, u, nullptr, nullptr, nullptr, nullptr, f.partials, f.all_done, a);
    BCMGX_LAUNCHED();
    if (!a.tickets) fin_launch<FIN_BETA>(c, f, f.nblk, a);
    k_cg_direction<<<f.nblk, WG, 0, c->stream>>>(f.n, f.k, f.st, u, p, f.all_done);
    BCMGX_LAUNCHED();
}

void cg_alpha(Context* c, const FcgBufs& f, const double* p, const double* s, const double* u, const double* r, bool first) {
    FinArgs a = fin_args(f);
    if (first) {
        k_dots<2, FIN_ALPHA0><<<f.nblk, WG, 0, c->stream>>>(f.n, f.k, p, s, u, r, nullptr, nullptr, f.partials, f.all_done, a);
        BCMGX_LAUNCHED();
        if (!a.tickets) fin_launch<FIN_ALPHA0>(c, f, f.nblk, a);
    } else {
        k_dots<1, FIN_ALPHA><<<f.nblk, WG, 0, c->stream>>>(f.n, f.k, p, s, nullptr, nullptr, nullptr, nullptr, f.partials, f.all_done, a);
        BCMGX_LAUNCHED();
        if (!a.tickets) fin_launch<FIN_ALPHA>(c, f, f.nblk, a);
    }
}

// x = alpha p + 1 x; r = -alpha s + 1 r (CG_HS.cu:131-132), with the ||r||^2 partials
__global__ __launch_bounds__(WG) void k_cg_update(int n, int k, const FcgState* st,
                                                  const double* __restrict__ p, const double* __restrict__ sv,
                                                  double* __restrict__ x, double* __restrict__ r,
                                                  double* __restrict__ partials, const int* all_done, FinArgs fa) {
    if (*all_done) return;
    __shared__ double s[1][WG];
    int tid = threadIdx.x;
    const RowSplit sp(k);
    int c = sp.c;
    double acc = 0.0;
    if (sp.active()) {
        const FcgState S = st[c];
        double al = S.theta2;
        for (long long i = (long long)blockIdx.x * sp.R + sp.rl; i < n; i += (long long)gridDim.x * sp.R) {
            long long o = i * k + c;
            double rr;
            if (!S.done) {
                x[o] = al * p[o] + 1.0 * x[o];
                rr = -al * sv[o] + 1.0 * r[o];
                r[o] = rr;
            } else {
                rr = r[o];
            }
            acc += rr * rr;
        }
    }
    s[0][tid] = acc;
    __syncthreads();
    sp.sum<1>(s, k);
    block_end<FIN_CG>(s, partials, k, fa);
}

void cg_update_finish(Context* c, const FcgBufs& f, const double* p, const double* s, double* x, double* r) {
    FinArgs a = fin_args(f);
    k_cg_update<<<f.nblk, WG, 0, c->stream>>>(f.n, f.k, f.st, p, s, x, r, f.partials, f.all_done, a);
    BCMGX_LAUNCHED();
    if (!a.tickets) fin_launch<FIN_CG>(c, f, f.nblk, a);
}

}  // namespace bcmgx
