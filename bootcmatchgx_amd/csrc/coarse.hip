// coarse.hip -- all the l1-Jacobi sweeps of the coarsest level in one launch
// (relaxCoarsest, GAMG_cycle.cu:186; _jacobi_it_full<0>, l1jacobi.cu:344-379).
//
// The coarsest operator has a few thousand rows (max_coarse_size: 40 cbrt(N))
// and the cycle sweeps it 20 times.  As 20 launches each sweep costs 2.4-4.6 us
// of dispatch and dependent memory round trips for 0.1-0.5 us of data (about 90 us
// per cycle at 27-point 128^3, one right-hand side).  Here one launch does them
// all: every lane keeps its matrix entries in registers, and the iterate moves
// between the workgroups through memory, or through LDS when one workgroup
// holds the level.  Measured for 20 sweeps, the launches it replaces -> here:
// 4096 rows (27-point 128^3) 92 -> 42 us, 1954 rows (7-point 50^3) 55 -> 28 us,
// 250 rows (7-point 10^3) 50 -> 12 us, 11270 rows (7-point diffusion 160^3)
// 102 -> 77 us.  What is left is the latency of a store and of the loads that
// find it, 2 us a sweep across the XCDs' L2s.
//
// Same bits as the launches it replaces: a row is summed by the same number of
// lanes with the same stride and the same shuffle tree as k_spmv1, and the
// update is the same expression.
#include "kernels.h"

namespace bcmgx {

constexpr int CO_ROWS = 32;          // rows per workgroup of the exchanging kernel
constexpr int CO_FETCH = 4;          // listed columns a thread of it fetches
constexpr int CO_COLS = 8;           // columns per workgroup of the k-column kernel
constexpr int CO_COL_PLACES = 512;   // its LDS places: distinct columns of a tile, and a zero
constexpr int CO_COL_FETCH = 8;      // elements a thread of it has in flight
constexpr size_t CO_SLOT_WORDS = size_t(8) << 20;  // 64 MB
constexpr int CO_SMALL_T = 1024;    // threads of the one-workgroup kernel
constexpr int CO_SMALL_N = 1024;    // rows it holds in LDS
constexpr int CO_SMALL_RR = 4;      // rows per lane group there
constexpr int CO_SMALL_E = 4;       // entries per lane and row there

typedef unsigned long long u64;

// the sum over a row's L lanes, in every lane
template <int L>
__device__ __forceinline__ double group_sum(double t) {
#pragma unroll
    for (int o = L / 2; o > 0; o >>= 1) t += __shfl_xor(t, o, L);
    return t;
}

// a row's entries of this lane: lane, lane + L, ... from the row's start
template <int L, int E>
struct RowPart {
    double a[E];
    int c[E];  // -1: no entry
    __device__ __forceinline__ void load(bool on, int r, int lane, const int* __restrict__ row, const int* __restrict__ col,
                                         const double* __restrict__ val) {
        int s = 0, e = 0;
        if (on) {
            s = row[r];
            e = row[r + 1];
        }
#pragma unroll
        for (int q = 0; q < E; q++) {
            int j = s + lane + q * L;
            c[q] = j < e ? col[j] : -1;
            a[q] = j < e ? val[j] : 0.0;
        }
    }
    __device__ __forceinline__ double sum(const double* xv) const {
        double t = 0;
#pragma unroll
        for (int q = 0; q < E; q++)
            if (c[q] >= 0) t += a[q] * xv[q];
        return group_sum<L>(t);
    }
};

// Thread 0 of a workgroup that has passed its waits: 0, or for the last of them 1, or 2 when
// one gave up.  A workgroup's word of that (ctl[2]) is stored by its own thread 0, so the fence
// here has it visible before the ticket is counted, and no such store is left to land
// after the last workgroup has cleared the word.
__device__ __forceinline__ int coarse_ticket(unsigned* ctl, unsigned workgroups) {
    __threadfence();
    if (atomicAdd(ctl + 1, 1u) != workgroups - 1) return 0;
    __threadfence();
    return __hip_atomic_load(ctl + 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ? 2 : 1;
}

// The exchanging kernel: a workgroup owns CO_ROWS rows, L lanes each.  An
// iterate's element travels as two 64-bit words, each half of the double with a
// 32-bit tag beside it, written and read with device scope: a reader that finds
// both tags has the value, so there is no barrier over the grid and no separate
// flag to wait for.  A workgroup fetches each distinct column of its rows once
// per sweep (the list made at setup, sorted, so neighbouring threads read
// neighbouring elements) and its lanes take them from LDS: with every lane
// fetching its own entries' elements a sweep of the 4096 rows of 27-point 128^3
// took 4 us, bound by the 100 K scattered requests (2.1 us with the list).  Each sweep has its own
// slots, so a workgroup that runs ahead overwrites nothing, and tags rise from
// launch to launch (ctl[0]), so nothing is cleared.  The first sweep from zero,
// f / D, is formed by every reader itself.
//
// The waits need the workgroups to run at the same time.  The launcher keeps the
// grid to half of what the device holds; whatever else occupies it, each
// wait is bounded: a workgroup that waits longer than `patience` clock ticks
// raises ctl[2], all give up, and the workgroup that finishes last computes the
// sweeps alone.  Workgroups that had their values wrote the same ones.  It says
// so in *gave_up (the host's memory), and the host goes back to a launch a sweep:
// whatever holds the device would have every cycle wait.
template <typename V, int L, int E>
__global__ __launch_bounds__(CO_ROWS * L) void k_coarse_exchange(
    int n, const int* __restrict__ row, const int* __restrict__ col, const double* __restrict__ val,
    const double* __restrict__ D, const V* __restrict__ f, const V* __restrict__ x0, V* __restrict__ out, int sweeps,
    const int* __restrict__ ucnt, const int* __restrict__ ucol, const unsigned short* __restrict__ upos, u64* slots,
    double* scratch, unsigned* ctl, unsigned* gave_up, const int* __restrict__ stop, long long patience, RowProlong<V> up) {
    constexpr int T = CO_ROWS * L, NU = CO_FETCH;
    if (stop && *stop) return;
    __shared__ double xs[2][TILE_MAX_COLS];
    __shared__ int s_late, s_last;
    int tid = threadIdx.x, lane = tid % L;
    int r = blockIdx.x * CO_ROWS + tid / L;
    bool on = r < n;
    unsigned base = ctl[0];
    if (tid == 0) s_late = 0;
    int rs = on ? row[r] : 0, re = on ? row[r + 1] : 0;
    // the listed columns this thread fetches (-1: none) and its entries' places among them;
    // a tile without a list (too many entries or columns) has every lane fetch its own
    // entries' elements, one after another
    int U = ucnt[blockIdx.x];
    bool listed = U > 0 && U <= NU * T;
    int uc[NU], at[E];
    double a[E];
#pragma unroll
    for (int w = 0; w < NU; w++)
        uc[w] = listed && tid + w * T < U ? ucol[(size_t)blockIdx.x * TILE_MAX_COLS + tid + w * T] : -1;
#pragma unroll
    for (int q = 0; q < E; q++) {
        int j = rs + lane + q * L;
        at[q] = listed && j < re ? upos[j] : -1;
        a[q] = listed && j < re ? val[j] : 0.0;
    }
    double fr = on ? (double)f[r] : 0.0, Dr = on ? D[r] : 1.0;
    double xr;
    int done = x0 ? 0 : 1;
    // the iterate that costs no exchange: the guess, or the sweep from zero ((-0 + f) / D) + 0
    auto first = [&](int c) { return x0 ? (double)x0[c] : (double)f[c] / D[c]; };
    xr = x0 ? (on ? (double)x0[r] : 0.0) : fr / Dr;
    bool given_up = false;  // uniform over the workgroup
    for (int s = done; s < sweeps; s++) {
        double* xc = xs[s & 1];
        double t = 0;
        if (s == done) {
            if (listed) {
#pragma unroll
                for (int w = 0; w < NU; w++)
                    if (uc[w] >= 0) xc[tid + w * T] = first(uc[w]);
            } else {
                for (int j = rs + lane; j < re; j += L) t += val[j] * first(col[j]);
            }
        } else {  // the elements that sweep s - 1 published
            const u64* p = slots + (size_t)(s - 1) * n * 2;
            unsigned tag = base + (unsigned)s;
            auto fetch = [&](int c, double& v) {
                u64 lo = __hip_atomic_load(p + (size_t)c * 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                u64 hi = __hip_atomic_load(p + (size_t)c * 2 + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                v = __hiloint2double((int)(unsigned)hi, (int)(unsigned)lo);
                return (unsigned)(lo >> 32) == tag && (unsigned)(hi >> 32) == tag;
            };
            long long t0 = 0;
            bool late = patience < 0;  // negative: no waiting at all
            int j = rs + lane;         // without a list: the entry waited for
            for (int poll = 0; !late; poll++) {
                bool ready = true;
                if (listed) {
                    double v[NU];
                    bool ok[NU];
#pragma unroll
                    for (int w = 0; w < NU; w++) ok[w] = uc[w] < 0 || fetch(uc[w], v[w]);
#pragma unroll
                    for (int w = 0; w < NU; w++) {
                        if (uc[w] >= 0 && ok[w]) xc[tid + w * T] = v[w];
                        ready = ready && ok[w];
                    }
                } else {
                    double v;
                    while (j < re && fetch(col[j], v)) {
                        t += val[j] * v;
                        j += L;
                    }
                    ready = j >= re;
                }
                if (ready) break;
                if ((poll & 15) == 15) {
                    if (poll == 15) t0 = wall_clock64();
                    else if (wall_clock64() - t0 > patience) late = true;
                    if (__hip_atomic_load(&s_late, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) == s + 1 ||
                        __hip_atomic_load(ctl + 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
                        late = true;
                }
            }
            if (late) __hip_atomic_store(&s_late, s + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
        __syncthreads();  // the other half of xs is written before the next one
        if (s_late == s + 1) {  // not a faster wave's of the next sweep
            given_up = true;
            if (tid == 0) __hip_atomic_store(ctl + 2, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            break;
        }
        if (listed) {
#pragma unroll
            for (int q = 0; q < E; q++)
                if (at[q] >= 0) t += a[q] * xc[at[q]];
        }
        t = group_sum<L>(t);
        xr = ((-t + fr) / Dr) + xr;
        if (s + 1 < sweeps && on && lane == 0) {
            u64* p = slots + ((size_t)s * n + r) * 2;
            u64 tag = (u64)(base + (unsigned)s + 1u) << 32;
            __hip_atomic_store(p, tag | (unsigned)__double2loint(xr), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(p + 1, tag | (unsigned)__double2hiint(xr), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    if (!given_up && on) {
        if (up.out) up.template put<L>(r, lane, (V)xr);
        else if (lane == 0) out[r] = (V)xr;
    }
    __syncthreads();
    if (tid == 0) s_last = coarse_ticket(ctl, gridDim.x);
    __syncthreads();
    if (!s_last) return;
    // the last workgroup: every other one has passed its waits for good
    if (s_last == 2) {
        if (tid == 0) __hip_atomic_store(gave_up, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        double* cur = scratch;
        double* nxt = scratch + n;
        for (int i = tid; i < n; i += T) cur[i] = first(i);
        __threadfence();
        __syncthreads();
        for (int s = done; s < sweeps; s++) {
            for (int i0 = 0; i0 < n; i0 += CO_ROWS) {
                int i = i0 + tid / L;
                double t = 0;
                if (i < n)
                    for (int j = row[i] + lane; j < row[i + 1]; j += L) t += val[j] * cur[col[j]];
                t = group_sum<L>(t);
                if (i < n && lane == 0) nxt[i] = ((-t + (double)f[i]) / D[i]) + cur[i];
            }
            __threadfence();
            __syncthreads();
            double* w = cur;
            cur = nxt;
            nxt = w;
        }
        for (int i = tid; i < n; i += T) {
            if (up.out) up.template put<1>(i, 0, (V)cur[i]);
            else out[i] = (V)cur[i];
        }
        __syncthreads();
    }
    if (tid == 0) {
        ctl[0] = base + (unsigned)sweeps + 1u;
        ctl[1] = 0;
        ctl[2] = 0;
    }
}

// The one-workgroup kernel: the iterate in LDS, one barrier per sweep.
template <typename V, int L>
__global__ __launch_bounds__(CO_SMALL_T) void k_coarse_small(int n, const int* __restrict__ row, const int* __restrict__ col,
                                                             const double* __restrict__ val, const double* __restrict__ D,
                                                             const V* __restrict__ f, const V* __restrict__ x0,
                                                             V* __restrict__ out, int sweeps, const int* __restrict__ stop,
                                                             RowProlong<V> up) {
    if (stop && *stop) return;
    constexpr int RR = CO_SMALL_RR, E = CO_SMALL_E, G = CO_SMALL_T / L;
    __shared__ double xs[2][CO_SMALL_N];
    int lane = threadIdx.x % L, g = threadIdx.x / L;
    RowPart<L, E> part[RR];
    double fr[RR], Dr[RR], xr[RR];
#pragma unroll
    for (int w = 0; w < RR; w++) {
        int r = w * G + g;
        bool on = r < n;
        part[w].load(on, r, lane, row, col, val);
        fr[w] = on ? (double)f[r] : 0.0;
        Dr[w] = on ? D[r] : 1.0;
        xr[w] = x0 ? (on ? (double)x0[r] : 0.0) : fr[w] / Dr[w];
        if (on && lane == 0) xs[0][r] = xr[w];
    }
    __syncthreads();
    int cur = 0;
    for (int s = x0 ? 0 : 1; s < sweeps; s++) {
#pragma unroll
        for (int w = 0; w < RR; w++) {
            if (w * G >= n) break;  // uniform
            double xv[E];
#pragma unroll
            for (int q = 0; q < E; q++) xv[q] = part[w].c[q] >= 0 ? xs[cur][part[w].c[q]] : 0.0;
            double t = part[w].sum(xv);
            xr[w] = ((-t + fr[w]) / Dr[w]) + xr[w];
            int r = w * G + g;
            if (r < n && lane == 0) xs[cur ^ 1][r] = xr[w];
        }
        cur ^= 1;
        __syncthreads();
    }
#pragma unroll
    for (int w = 0; w < RR; w++) {
        int r = w * G + g;
        if (r >= n) continue;
        if (up.out) up.template put<L>(r, lane, (V)xr[w]);
        else if (lane == 0) out[r] = (V)xr[w];
    }
}

template <typename V, int L, int E>
static bool launch_exchange(Context* c, const DCsr& A, const double* D, const V* f, const V* x0, V* out, int sweeps,
                            const CoarseIndex& ix, CoarseSync& cs, const int* stop, const RowProlong<V>& up) {
    auto kern = k_coarse_exchange<V, L, E>;
    static int resident = 0;  // workgroups the device holds, per instantiation; identical devices assumed within a process
    if (!resident) {
        int per_cu = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, CO_ROWS * L, 0) != hipSuccess) per_cu = 0;
        resident = c->num_cus * per_cu + 1;
    }
    unsigned grid = grid_for(A.n, CO_ROWS);
    if ((long long)grid * 2 > resident) return false;
    kern<<<grid, CO_ROWS * L, 0, c->stream>>>(A.n, A.row.get(), A.col.get(), A.val.get(), D, f, x0, out, sweeps,
                                              ix.ucnt.get(), ix.ucol.get(), ix.upos.get(), cs.slots.get(),
                                              cs.scratch.get(), cs.ctl.get(), c->mailbox() + MAIL_GAVE_UP, stop, c->coarse_patience, up);
    BCMGX_LAUNCHED();
    return true;
}

void CoarseIndex::build(Context* c, const DCsr& A) {
    if (A.n <= 0 || A.n > CO_MAX_N) return;
    unsigned nt = grid_for(A.n, CO_ROWS);
    ucnt.reset(c, nt);
    ucol.reset(c, (size_t)nt * TILE_MAX_COLS);
    upos.reset(c, (size_t)std::max(A.nnz, 2));
    tile_columns_strided(c, A, CO_ROWS, ucnt.get(), ucol.get(), upos.get());
}

void CoarseSync::reserve(Context* c, int n, int sweeps, int k) {
    size_t words = (size_t)std::max(sweeps, 1) * 2, need = n * words;
    if (k > 1) {
        // as many groups of columns as launch_columns takes, a workgroup a CU, whatever k is: a wide
        // solve's slots serve the narrow ones after it (20 sweeps of 4096 rows: 21 MB)
        size_t rows = (size_t)c->num_cus * CO_ROWS, groups = (k + CO_COLS - 1) / CO_COLS;
        size_t all = std::min(n * groups, rows) * words * CO_COLS;
        if ((size_t)n <= rows && all <= CO_SLOT_WORDS) need = std::max(need, all);
    }
    if (slots.size() >= need && scratch.size() >= (size_t)n * 2) return;
    slots.reset(c, need);
    scratch.reset(c, (size_t)n * 2);
    ctl.reset(c, 4);
    fill<long long>(c, (long long*)slots.get(), (long long)need, 0);
    fill<int>(c, (int*)ctl.get(), 4, 0);
}

static bool coarse_one_workgroup(const DCsr& A, int L) {
    return A.n <= CO_SMALL_N && (long long)A.n * L <= (long long)CO_SMALL_RR * CO_SMALL_T && A.maxrow <= CO_SMALL_E * L;
}

bool coarse_sweeps_fit(int n, int sweeps) { return n > 0 && n <= CO_MAX_N && sweeps >= 2 && sweeps <= CO_MAX_SWEEPS; }

template <typename V>
bool coarse_sweeps(Context* c, const DCsr& A, int lanes, const double* D, const V* f, const V* x0, V* out, int sweeps,
                   const CoarseIndex& ix, CoarseSync& cs, const int* stop, const RowProlong<V>& up) {
    int L = lanes != 0 ? lanes : default_lanes(A.nnz, A.n);
    if (!coarse_sweeps_fit(A.n, sweeps) || A.maxrow < 0 || L < 2 || L > 32 || (const void*)out == (const void*)x0) return false;
    // One workgroup while it holds the level's entries in registers (n <= 4096 / L): a
    // sweep is then a barrier and LDS reads, 0.5 us against 1.4-2 us for the exchange.
    if (coarse_one_workgroup(A, L)) {
#define BCMGX_CS(LL)                                                                                                     \
    case LL:                                                                                                             \
        k_coarse_small<V, LL><<<1, CO_SMALL_T, 0, c->stream>>>(A.n, A.row.get(), A.col.get(), A.val.get(), D, f, x0, out, \
                                                               sweeps, stop, up);                                          \
        break;
        switch (L) { BCMGX_CS(2) BCMGX_CS(4) BCMGX_CS(8) BCMGX_CS(16) BCMGX_CS(32) }
#undef BCMGX_CS
        BCMGX_LAUNCHED();
        return true;
    }
    if (cs.off || !ix.ucnt || cs.slots.size() < (size_t)A.n * sweeps * 2 || cs.scratch.size() < (size_t)A.n * 2) return false;
#define BCMGX_CX(LL)                                                                                         \
    case LL:                                                                                                 \
        if (A.maxrow <= 2 * LL) return launch_exchange<V, LL, 2>(c, A, D, f, x0, out, sweeps, ix, cs, stop, up);     \
        if (A.maxrow <= 4 * LL) return launch_exchange<V, LL, 4>(c, A, D, f, x0, out, sweeps, ix, cs, stop, up);     \
        if (A.maxrow <= 8 * LL) return launch_exchange<V, LL, 8>(c, A, D, f, x0, out, sweeps, ix, cs, stop, up);     \
        return false;
    switch (L) { BCMGX_CX(2) BCMGX_CX(4) BCMGX_CX(8) BCMGX_CX(16) BCMGX_CX(32) }
#undef BCMGX_CX
    return false;
}
template bool coarse_sweeps<double>(Context*, const DCsr&, int, const double*, const double*, const double*, double*, int,
                                    const CoarseIndex&, CoarseSync&, const int*, const RowProlong<double>&);
template bool coarse_sweeps<float>(Context*, const DCsr&, int, const double*, const float*, const float*, float*, int,
                                   const CoarseIndex&, CoarseSync&, const int*, const RowProlong<float>&);

// The exchanging kernel for k columns: CC of them per workgroup, a thread per row and column, the row
// summed in order as the k-column kernels do (the same bits).  Slots: [group of CC columns][sweep][row][CC][2],
// so the columns of an element are fetched together; a group past k carries zeros.  The entries' values
// and places are in registers, one LDS buffer holds the tile's distinct elements (place U: zero).
// 8 columns of 4096 rows (27-point 128^3), 20 sweeps: 186 us as launches (130 in a replayed graph), 60 here;
// 3 us a sweep, two rounds of loads through the memory side and the row sums from LDS.
template <typename V, int E>
__global__ __launch_bounds__(CO_ROWS * CO_COLS, E > 32 ? 2 : E > 16 ? 3 : 4) void k_coarse_columns(
    int n, int k, const int* __restrict__ row, const int* __restrict__ col, const double* __restrict__ val,
    const double* __restrict__ D, const V* __restrict__ f, const V* __restrict__ x0, V* __restrict__ out, int sweeps,
    const int* __restrict__ ucnt, const int* __restrict__ ucol, const unsigned short* __restrict__ upos, u64* slots,
    double* scratch, unsigned* ctl, unsigned* gave_up, const int* __restrict__ stop, long long patience) {
    constexpr int CC = CO_COLS, T = CO_ROWS * CC, NU = CO_COL_FETCH;
    if (stop && *stop) return;
    __shared__ double xs[CO_COL_PLACES * CC];
    __shared__ int s_late, s_last;
    int tid = threadIdx.x, cl = tid % CC;
    int r = blockIdx.x * CO_ROWS + tid / CC;
    int c = (int)blockIdx.y * CC + cl;
    bool on = r < n, act = c < k;
    unsigned base = ctl[0];
    u64* mine = slots + (size_t)blockIdx.y * sweeps * n * CC * 2;
    int U = ucnt[blockIdx.x];
    bool listed = U > 0 && U < CO_COL_PLACES;
    const int* list = ucol + (size_t)blockIdx.x * TILE_MAX_COLS;
    if (tid == 0) s_late = 0;
    if (listed && tid < CC) xs[U * CC + tid] = 0.0;
    int rs = on ? row[r] : 0, re = on ? row[r + 1] : 0;
    double a[E];
    unsigned at[E / 2];
#pragma unroll
    for (int q = 0; q < E; q += 2) {
        bool i0 = listed && rs + q < re, i1 = listed && rs + q + 1 < re;
        a[q] = i0 ? val[rs + q] : 0.0;
        a[q + 1] = i1 ? val[rs + q + 1] : 0.0;
        at[q / 2] = (i0 ? upos[rs + q] : (listed ? U : 0)) | (unsigned)(i1 ? upos[rs + q + 1] : (listed ? U : 0)) << 16;
    }
    double fr = on && act ? (double)f[(size_t)r * k + c] : 0.0, Dr = on ? D[r] : 1.0;
    auto first = [&](int i) {
        return !act ? 0.0 : x0 ? (double)x0[(size_t)i * k + c] : (double)f[(size_t)i * k + c] / D[i];
    };
    int done = x0 ? 0 : 1;
    double xr = x0 ? (on && act ? (double)x0[(size_t)r * k + c] : 0.0) : fr / Dr;
    bool given_up = false;  // uniform over the workgroup
    for (int s = done; s < sweeps; s++) {
        double t = 0;
        if (s == done) {
            if (listed) {
                for (int u = tid / CC; u < U; u += CO_ROWS) xs[u * CC + cl] = first(list[u]);
            } else {
                for (int j = rs; j < re; j++) t += val[j] * first(col[j]);
            }
        } else {  // the elements that sweep s - 1 published
            const u64* p = mine + (size_t)(s - 1) * n * CC * 2;
            unsigned tag = base + (unsigned)s;
            auto fetch = [&](unsigned o, double& v) {  // o: bytes, below 2^32 (one register an address)
                const u64* e = (const u64*)((const char*)p + o);
                u64 lo = __hip_atomic_load(e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                u64 hi = __hip_atomic_load(e + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                v = __hiloint2double((int)(unsigned)hi, (int)(unsigned)lo);
                return (unsigned)(lo >> 32) == tag && (unsigned)(hi >> 32) == tag;
            };
            long long t0 = 0;
            bool late = patience < 0;  // negative: no waiting at all
            int j = rs;                // without a list: the entry waited for
            int u0 = tid / CC;         // with one: the first place of the NU waited for
            for (int poll = 0; !late; poll++) {
                if (listed) {
                    while (u0 < U) {
                        double v[NU];
                        unsigned o[NU];
                        bool ok = true;
#pragma unroll
                        for (int w = 0; w < NU; w++) o[w] = ((unsigned)list[min(u0 + w * CO_ROWS, U - 1)] * CC + cl) * 16u;
#pragma unroll
                        for (int w = 0; w < NU; w++) ok = fetch(o[w], v[w]) & ok;
                        if (!ok) break;
#pragma unroll
                        for (int w = 0; w < NU; w++) xs[min(u0 + w * CO_ROWS, U - 1) * CC + cl] = v[w];
                        u0 += NU * CO_ROWS;
                    }
                    if (u0 >= U) break;
                } else {
                    double v;
                    while (j < re && fetch(((unsigned)col[j] * CC + cl) * 16u, v)) t += val[j++] * v;
                    if (j >= re) break;
                }
                if ((poll & 15) == 15) {
                    if (poll == 15) t0 = wall_clock64();
                    else if (wall_clock64() - t0 > patience) late = true;
                    if (__hip_atomic_load(&s_late, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) == s + 1 ||
                        __hip_atomic_load(ctl + 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
                        late = true;
                }
            }
            if (late) __hip_atomic_store(&s_late, s + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
        __syncthreads();
        if (s_late == s + 1) {
            given_up = true;
            if (tid == 0) __hip_atomic_store(ctl + 2, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            break;
        }
        if (listed) {
#pragma unroll
            for (int q = 0; q < E; q += 4) {
                if (!__any(rs + q < re)) break;
                unsigned p01 = at[q / 2], p23 = at[q / 2 + 1];
                asm("" : "+v"(p01), "+v"(p23));  // unpacked here: E addresses kept over the sweeps would spill
                double v0 = xs[(p01 & 0xffffu) * CC + cl], v1 = xs[(p01 >> 16) * CC + cl];
                double v2 = xs[(p23 & 0xffffu) * CC + cl], v3 = xs[(p23 >> 16) * CC + cl];
                t += a[q] * v0;
                t += a[q + 1] * v1;
                t += a[q + 2] * v2;
                t += a[q + 3] * v3;
            }
        }
        xr = ((-t + fr) / Dr) + xr;
        if (s + 1 < sweeps && on) {
            u64* p = mine + (((size_t)s * n + r) * CC + cl) * 2;
            u64 tag = (u64)(base + (unsigned)s + 1u) << 32;
            __hip_atomic_store(p, tag | (unsigned)__double2loint(xr), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(p + 1, tag | (unsigned)__double2hiint(xr), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __syncthreads();  // xs is read: the next elements take its place
    }
    if (!given_up && on && act) out[(size_t)r * k + c] = (V)xr;
    __syncthreads();
    if (tid == 0) s_last = coarse_ticket(ctl, gridDim.x * gridDim.y);
    __syncthreads();
    if (!s_last) return;
    // the last workgroup: every other one has passed its waits for good
    if (s_last == 2) {
        if (tid == 0) __hip_atomic_store(gave_up, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        for (int q = 0; q < k; q++) {
            double* cur = scratch;
            double* nxt = scratch + n;
            for (int i = tid; i < n; i += T) cur[i] = x0 ? (double)x0[(size_t)i * k + q] : (double)f[(size_t)i * k + q] / D[i];
            __threadfence();
            __syncthreads();
            for (int s = done; s < sweeps; s++) {
                for (int i = tid; i < n; i += T) {
                    double t = 0;
                    for (int j = row[i]; j < row[i + 1]; j++) t += val[j] * cur[col[j]];
                    nxt[i] = ((-t + (double)f[(size_t)i * k + q]) / D[i]) + cur[i];
                }
                __threadfence();
                __syncthreads();
                double* w = cur;
                cur = nxt;
                nxt = w;
            }
            for (int i = tid; i < n; i += T) out[(size_t)i * k + q] = (V)cur[i];
            __syncthreads();
        }
    }
    if (tid == 0) {
        ctl[0] = base + (unsigned)sweeps + 1u;
        ctl[1] = 0;
        ctl[2] = 0;
    }
}

template <typename V, int E>
static bool launch_columns(Context* c, const DCsr& A, const double* D, const V* f, const V* x0, V* out, int k, int sweeps,
                           const CoarseIndex& ix, CoarseSync& cs, const int* stop) {
    auto kern = k_coarse_columns<V, E>;
    static int resident = 0;  // workgroups the device holds, per instantiation; identical devices assumed within a process
    if (!resident) {
        int per_cu = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, CO_ROWS * CO_COLS, 0) != hipSuccess) per_cu = 0;
        resident = c->num_cus * per_cu + 1;
    }
    int tiles = (int)grid_for(A.n, CO_ROWS), groups = (k + CO_COLS - 1) / CO_COLS;
    // to one workgroup a CU: beyond, the fetches of 128 bytes an element and row of columns bound a sweep (32
    // columns of 4096 rows, 512 workgroups: 114 us, and the same as 20 launches)
    if (tiles * groups > c->num_cus || tiles * groups * 2 > resident ||
        (size_t)A.n * sweeps * groups * CO_COLS * 2 > cs.slots.size())
        return false;
    kern<<<dim3(tiles, groups), CO_ROWS * CO_COLS, 0, c->stream>>>(
        A.n, k, A.row.get(), A.col.get(), A.val.get(), D, f, x0, out, sweeps, ix.ucnt.get(), ix.ucol.get(), ix.upos.get(),
        cs.slots.get(), cs.scratch.get(), cs.ctl.get(), c->mailbox() + MAIL_GAVE_UP, stop, c->coarse_patience);
    BCMGX_LAUNCHED();
    return true;
}

template <typename V>
bool coarse_sweeps_columns(Context* c, const DCsr& A, const double* D, const V* f, const V* x0, V* out, int k, int sweeps,
                           const CoarseIndex& ix, CoarseSync& cs, const int* stop) {
    if (cs.off || k < 2 || !coarse_sweeps_fit(A.n, sweeps) || A.maxrow < 0 || !ix.ucnt || (const void*)out == (const void*)x0 ||
        (const void*)out == (const void*)f || cs.scratch.size() < (size_t)A.n * 2)
        return false;
    if (A.maxrow <= 16) return launch_columns<V, 16>(c, A, D, f, x0, out, k, sweeps, ix, cs, stop);
    if (A.maxrow <= 32) return launch_columns<V, 32>(c, A, D, f, x0, out, k, sweeps, ix, cs, stop);
    if (A.maxrow <= 64) return launch_columns<V, 64>(c, A, D, f, x0, out, k, sweeps, ix, cs, stop);
    return false;
}
template bool coarse_sweeps_columns<double>(Context*, const DCsr&, const double*, const double*, const double*, double*, int, int,
                                            const CoarseIndex&, CoarseSync&, const int*);
template bool coarse_sweeps_columns<float>(Context*, const DCsr&, const double*, const float*, const float*, float*, int, int,
                                           const CoarseIndex&, CoarseSync&, const int*);

}  // namespace bcmgx
