// afsai.hip -- adaptive factorized sparse approximate inverse, M^-1 = G^T G.
//
// Restates afsai_setup (src/preconditioner/afsai/afsai.cu:287-1090) for one
// GPU.  The reference runs its loop step by step over all rows with separate
// kernels (d_kapGrad_merge, kapGradCUDA_WiP.cu:189-368; d_gatherFullSysAdapt,
// d_gFSA.cu:8-79; cudacholdcMix, choldc.cu:24-77; multiscalar_product;
// check_done, afsai.cu:261-280).  Rows never interact, so here 16 or 32 lanes of
// a wave64 own one row for all steps and keep its pattern, coefficients and
// dense system in LDS and registers:
//   * Kaporin gradient over the columns < i of the rows {i} u P (factor 1, then
//     the current coefficients), each column's value summed in lane order (row
//     i, then the pattern rows in column order); the largest |gradient| outside
//     P wins, ties to the smallest column; a zero maximum adds nothing and the
//     row is done.  Two ways to the same sums:
//       - column table (first launch, k_afsai_table): a row's columns get slots of
//         a hash table in LDS once, when the row joins; each step then adds each
//         row's products into the slots, one row after the other in lane order,
//         and reduces the table for the largest entry.  Rows whose entries left
//         of the diagonal are more than 30, not strictly increasing, or would
//         take the table past 192 columns are handed to
//       - the merge (second launch, k_afsai_rows, those rows only): lane r walks
//         row r, the columns merged in ascending order with a wave min, a column's
//         contributions summed over the lanes in order.
//   * dense system A_s[P,P] and rhs -A_s[i,P]; Cholesky with the reference's
//     operation order (diagonal stored as its reciprocal), triangular solves and
//     DKap = b.x.
//   * stop when |DKap - DKap_old| < 1e-3 DKap_old or DKap == 0; at most 30
//     entries (AFSAISTEP = 30, AFSAILFIL = 1, AFSAIEPSILON, afsai.cu:41-45).
// A_s = D^-1/2 A D^-1/2 (scalediag + CSRscaleA_0).  createprc (:165-202):
// row i of G = (a_s,ii - DKap_i)^-1/2 [x, 1].
#include "kernels.h"

#include <climits>
#include <utility>

namespace bcmgx {

constexpr int AF_MMAX = 30;
constexpr int AF_PACK = AF_MMAX * (AF_MMAX + 1) / 2;
constexpr double AF_EPS = 0.001;
constexpr int AF_WAVES = 2;  // waves per workgroup
constexpr int AF_TS = 256;   // column-table slots per row (slot indices are bytes)
constexpr int AF_TLIM = 192; // columns a table takes before its row goes to the merge
constexpr int AF_EMAX = 30;  // entries left of the diagonal a row may bring into the table
static_assert(AF_TS == 256 && AF_TLIM < AF_TS && AF_TS <= AF_PACK, "table slots: bytes, never full, sums in L_s");

// 8-bit multiplicative hash of a column
__device__ __forceinline__ int af_hash(int c) { return (int)(((unsigned)c * 2654435761u) >> 24); }

__global__ void k_scale_diag(int n, const double* __restrict__ val, const int* __restrict__ dind, double* __restrict__ d) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) d[i] = 1.0 / sqrt(val[dind[i]]);
}
__global__ void k_scale_A(int n, const int* __restrict__ row, const int* __restrict__ col, const double* __restrict__ val,
                          const double* __restrict__ d, double* __restrict__ cs) {
    // 16 lanes a row: coalesced (27-point 128^3: 2.4 ms with one thread a row, 0.29 ms)
    int i = (int)(((long long)blockIdx.x * blockDim.x + threadIdx.x) / 16);
    if (i >= n) return;
    double di = d[i];
    for (int j = row[i] + (int)threadIdx.x % 16; j < row[i + 1]; j += 16) cs[j] = (val[j] * d[col[j]]) * di;
}

// order LDS accesses of the lanes of one wave (no hardware barrier needed)
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// s - P(0) Q(0) - P(1) Q(1) - ... (s + ... when ADD) over cnt terms, each product rounded and
// then subtracted (added) in term order; the operands of eight terms are loaded before their
// eight dependent updates, so the chain waits for the LDS once per eight terms, not per term
template <bool ADD, typename FP, typename FQ>
__device__ __forceinline__ double af_chain(double s, int cnt, FP P, FQ Q) {
    int t = 0;
    for (; t + 8 <= cnt; t += 8) {
        double p[8], q[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            p[u] = P(t + u);
            q[u] = Q(t + u);
        }
#pragma unroll
        for (int u = 0; u < 8; u++) s = ADD ? s + p[u] * q[u] : s - p[u] * q[u];
    }
    for (; t < cnt; t++) s = ADD ? s + P(t) * Q(t) : s - P(t) * Q(t);
    return s;
}

// min over the 32 lanes of a half wave
__device__ __forceinline__ int half_min_int(int v) {
#pragma unroll
    for (int o = 16; o > 0; o >>= 1) {
        int u = __shfl_xor(v, o, 32);
        v = u < v ? u : v;
    }
    return v;
}

// ---------------------------------------------------------------- table ----
// f(0), f(1), ..., f(N - 1) with compile-time indices
template <int... I, typename F>
__device__ __forceinline__ void af_each(std::integer_sequence<int, I...>, F&& f) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void af_for(F&& f) {
    af_each(std::make_integer_sequence<int, N>{}, f);
}
// lane LN's value in all 16 lanes of its group (DPP, no LDS)
template <int LN>
__device__ __forceinline__ double af_bc(double v) {
    return __longlong_as_double(__builtin_amdgcn_update_dpp(0ll, __double_as_longlong(v), 0x150 + LN, 0xf, 0xf, true));
}
// system row R's value: rows 0-15 in lo, 16-29 in hi of lane R % 16
template <int R>
__device__ __forceinline__ double af_row(double lo, double hi) {
    if constexpr (R < 16) return af_bc<R>(lo);
    else return af_bc<R - 16>(hi);
}

// a fresh copy of a wave-uniform (lane) value, so that comparisons with it are
// made where they are used and not kept in registers from another place
__device__ __forceinline__ int af_uniform(int v) {
    asm volatile("" : "+s"(v));
    return v;
}
__device__ __forceinline__ int af_lane(int v) {
    asm volatile("" : "+v"(v));
    return v;
}

// The dense part of a step for the four rows of a wave, in registers: lane hl of
// a group holds rows hl (lo) and hl + 16 (hi) of its row's system, entry c in
// lo[c] / hi[c].  Every element is formed by the operations of the packed
// one-lane formulation in its order (Cholesky terms ascending, forward
// substitution from the newest term down, backward from the newest up).  m is
// the wave's; rows past it hold anything and reach no valid row.  The steps nest
// (each tests m once and leaves all the rest), four columns to a test.
struct AfSystem {
    static constexpr int NC = AF_MMAX;
    double lo[16], hi[NC];
    double bl, bh, xl, xh;  // right-hand side and solution, rows hl and hl + 16
    double dl, dh;          // reciprocal pivots of those rows in the last factorisation
    double inv;             // the current one
    bool fail;
    int hl;

    template <int C>
    __device__ __forceinline__ void column(double ll, double lh) {
        if constexpr (C < NC) {
            double lc = af_row<C>(ll, lh);
            if constexpr (C < 16) lo[C] = lo[C] - lc * ll;
            hi[C] = hi[C] - lc * lh;
        }
    }
    template <int C>
    __device__ __forceinline__ void columns(int m, double ll, double lh) {
        if constexpr (C < NC) {
            if (C < m) {
                column<C>(ll, lh);
                column<C + 1>(ll, lh);
                column<C + 2>(ll, lh);
                column<C + 3>(ll, lh);
                columns<C + 4>(m, ll, lh);
            }
        }
    }
    // step K: rows and columns before q are the last factorisation's (the new entry sits at q),
    // so its pivot is too; the column's own elements are formed again
    template <int K>
    __device__ __forceinline__ void pivot(int m, int q) {
        if constexpr (K < NC) {
            if (K < m) {
                if (K < q) {
                    inv = af_row<K>(dl, dh);
                } else {
                    double d;
                    if constexpr (K < 16) d = af_bc<K % 16>(lo[K < 16 ? K : 0]);
                    else d = af_bc<K % 16>(hi[K]);
                    fail = fail || d <= 0.0;
                    inv = 1. / sqrt(d);
                }
                double ll = 0.0, lh = hi[K] * inv;
                int h = af_lane(hl);
                if constexpr (K < 16) {
                    ll = lo[K < 16 ? K : 0] * inv;
                    lo[K < 16 ? K : 0] = h == K ? inv : ll;
                    dl = h == K ? inv : dl;
                    hi[K] = lh;
                } else {
                    hi[K] = h == K - 16 ? inv : lh;
                    dh = h == K - 16 ? inv : dh;
                }
                columns<K + 1>(m, ll, lh);
                pivot<K + 1>(m, q);
            }
        }
    }
    // L y = b: a row's products with the known y, subtracted newest first
    template <int A>
    __device__ __forceinline__ void forward(int m, double (&pl)[15], double (&ph)[NC - 1]) {
        if constexpr (A < NC) {
            if (A < m) {
                int h = af_lane(hl);
                if constexpr (A < 16) {
                    double s = xl;
                    af_for<A>([&](auto t) { s = s - pl[A - 1 - t]; });
                    s = s * lo[A < 16 ? A : 0];
                    xl = h == A ? s : xl;
                    double y = af_bc<A % 16>(s);
                    if constexpr (A < 15) pl[A < 15 ? A : 0] = lo[A < 16 ? A : 0] * y;
                    ph[A < NC - 1 ? A : 0] = hi[A] * y;
                } else {
                    double s = xh;
                    af_for<A>([&](auto t) { s = s - ph[A - 1 - t]; });
                    s = s * hi[A];
                    xh = h == A - 16 ? s : xh;
                    if constexpr (A < NC - 1) ph[A < NC - 1 ? A : 0] = hi[A] * af_bc<A % 16>(s);
                }
                forward<A + 1>(m, pl, ph);
            }
        }
    }
    template <int B>
    __device__ __forceinline__ void terms(int m, double& s, double p, double q) {
        if constexpr (B < NC) {
            if (B < m) {  // rows past m count zero
                s = s - af_row<B>(p, q);
                if constexpr (B + 1 < NC) s = s - af_row<(B + 1 < NC ? B + 1 : 0)>(p, q);
                if constexpr (B + 2 < NC) s = s - af_row<(B + 2 < NC ? B + 2 : 0)>(p, q);
                if constexpr (B + 3 < NC) s = s - af_row<(B + 3 < NC ? B + 3 : 0)>(p, q);
                terms<B + 4>(m, s, p, q);
            }
        }
    }
    // L^T x = y: column A's products lie across the lanes
    template <int A>
    __device__ __forceinline__ void backward(int m, bool inl, bool inh) {
        if constexpr (A >= 0) {
            if (A < m) {
                double p = 0.0, q = inh ? hi[A] * xh : 0.0, s, iv;
                if constexpr (A < 15) p = inl ? lo[A < 16 ? A : 0] * xl : 0.0;
                if constexpr (A < 16) {
                    s = af_bc<A % 16>(xl);
                    iv = af_bc<A % 16>(lo[A < 16 ? A : 0]);
                } else {
                    s = af_bc<A % 16>(xh);
                    iv = af_bc<A % 16>(hi[A]);
                }
                terms<A + 1>(m, s, p, q);
                s = s * iv;
                int h = af_lane(hl);
                if constexpr (A < 16) xl = h == A ? s : xl;
                else xh = h == A - 16 ? s : xh;
            }
            backward<A - 1>(m, inl, inh);
        }
    }
    template <int E>
    __device__ __forceinline__ void dot(int m, double& dk, double p, double q) {
        if constexpr (E < NC) {
            if (E < m) {
                dk = dk + af_row<E>(p, q);
                if constexpr (E + 1 < NC) dk = dk + af_row<(E + 1 < NC ? E + 1 : 0)>(p, q);
                dot<E + 2>(m, dk, p, q);
            }
        }
    }
    // x and DKap; q: where the step's new entry went, the least over the wave's rows (0: factor anew)
    __device__ __forceinline__ double solve(int m, int q) {
        fail = false;
        pivot<0>(af_uniform(m), af_uniform(q));
        xl = bl;
        xh = bh;
        {
            double pl[15], ph[NC - 1];
            forward<0>(af_uniform(m), pl, ph);
        }
        bool inl = hl < m, inh = hl + 16 < m;
        backward<NC - 1>(af_uniform(m), inl, inh);
        if (fail) {  // breakdown: x = b, as the reference leaves it
            xl = bl;
            xh = bh;
        }
        double dk = 0.0;
        dot<0>(af_uniform(m), dk, inl ? bl * xl : 0.0, inh ? bh * xh : 0.0);
        return dk;
    }
};

// Four rows per wave, 16 lanes each; a workgroup is one wave.  The rows of a wave
// take their steps together, so the pattern size m is the wave's and the dense
// part runs from registers with compile-time indices (AfSystem).  A half-wave
// per row with the system in LDS and the substitutions on one lane spent two
// thirds of its time in those serial chains, each term two LDS operands and
// address arithmetic: 525 ms at 27-point 128^3 against 140 ms here, the factor bit
// for bit the same.  Now the vector units issue 57% of the kernel's cycles; the
// rest is latency that two waves a SIMD (registers, LDS) do not hide.
// LDS per row, 5 KB, so that eight waves (32 rows) fit a CU: the slots' sums of
// the gradient share their space with the dense system, which goes to registers
// in two parts (rows 0-15, then 16-29); the coefficients lie behind the sums, the
// right-hand side behind the first part.
// A row's entries are walked two to a lane with no test of their number: the
// places past it name slots of their own (AF_SLOTS + lane) that hold no column,
// and the values there are read from the padded end of cs or from the next row.
constexpr int AF4_ROWS = 4;
constexpr int AF_U = 8;              // pattern rows whose entries are in flight together
constexpr int AF_SLOTS = AF_TS - 16; // slots that hold columns
constexpr int AF_NONE = AF_MMAX + 1; // the entry list of no row
constexpr int AF_LO = 16 * 17 / 2;   // elements of rows 0-15
constexpr int AF_X0 = AF_TS;
constexpr int AF_PAD = 32;           // elements of cs past the last entry
struct alignas(16) AfRow {
    int hcol[AF_TS];               // slot columns: -1 empty, sign bit set once in the pattern
    double dense[AF_PACK - AF_LO];  // sums [0, AF_TS) and factors [AF_X0, + 31), or a part of the system
    int2 rb[AF_MMAX + 1];          // row i, then the pattern rows in column order: first entry, slot << 16 | place of the list in es
    unsigned char es[AF_MMAX + 2][AF_EMAX];  // entries' slots by the order rows joined (0: row i; AF_NONE: none)
    unsigned char pos[AF_TS];      // slot -> 1 + place in the pattern, 0 outside it
};
static_assert(AF_X0 + AF_MMAX + 1 <= AF_PACK - AF_LO && AF_LO + AF_MMAX <= AF_PACK - AF_LO && AF_EMAX % 2 == 0, "shared space");
static_assert(AF_TLIM < AF_SLOTS && sizeof(AfRow) * AF4_ROWS <= 160 * 1024 / 8, "eight waves per CU");

__global__ __launch_bounds__(64, 2) void k_afsai_table(int n, const int* __restrict__ row, const int* __restrict__ col,
                                                       const double* __restrict__ cs, int* __restrict__ pat_out,
                                                       double* __restrict__ x_out, int* __restrict__ mrow_out,
                                                       double* __restrict__ dk_out, int* __restrict__ redo,
                                                       int* __restrict__ nredo) {
    typedef double D2 __attribute__((ext_vector_type(2), aligned(8)));
    __shared__ AfRow rows_s[AF4_ROWS];
    int lane = threadIdx.x, grp = lane >> 4, hl = lane & 15;
    long long ri = (long long)xcd_remap(blockIdx.x, gridDim.x) * AF4_ROWS + grp;
    bool live = ri < n;
    int i = live ? (int)ri : 0;
    AfRow& R = rows_s[grp];
    double* xs = R.dense + AF_X0;  // the factors of rb's rows: 1, then x
    unsigned char* es = &R.es[0][0];
    // 16 bits of a ballot: this group's lanes
    auto bits = [&](bool v) { return (unsigned)(__ballot(v) >> (16 * grp)) & 0xffffu; };
    int hcnt = 0;  // columns in the table (uniform per group)
    // row r's entries left of column i into the table as joining index q: lane hl takes entries
    // hl and hl + 16 (`on` uniform per group); false when the table cannot take them
    auto table_row = [&](bool on, int q, int r, int& beg) -> bool {
        int end = 0;
        beg = 0;
        if (on) {
            beg = row[r];
            end = row[r + 1];
        }
        int cc[2];
#pragma unroll
        for (int h = 0; h < 2; h++) cc[h] = (on && beg + hl + 16 * h < end) ? col[beg + hl + 16 * h] : INT_MAX;
        unsigned ge = bits(cc[0] >= i) | bits(cc[1] >= i) << 16;
        int cnt = ge ? __ffs(ge) - 1 : 32;
        int nx0 = __shfl_down(cc[0], 1, 16), nx1 = __shfl_down(cc[1], 1, 16), first1 = __shfl(cc[1], 0, 16);
        if (hl == 15) nx0 = first1;
        unsigned bad = bits(hl + 1 < cnt && nx0 <= cc[0]) | bits(hl + 17 < cnt && nx1 <= cc[1]) << 16;
        bool ok = on && bad == 0 && cnt <= AF_EMAX && hcnt + cnt <= AF_TLIM;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            bool added = false;
            int e = hl + 16 * h;
            if (ok && e < AF_EMAX) {
                int s = AF_SLOTS + (e >> 1);  // the lane that walks this place
                if (e < cnt) {
                    // an empty slot always remains (at most AF_TLIM < AF_SLOTS columns): the probe ends
                    s = af_hash(cc[h]) * AF_SLOTS >> 8;
                    while (true) {
                        int v = R.hcol[s];
                        if ((v & INT_MAX) == cc[h]) break;
                        if (v == -1) {
                            int old = atomicCAS(&R.hcol[s], -1, cc[h]);
                            if (old == -1) {
                                added = true;
                                break;
                            }
                            if ((old & INT_MAX) == cc[h]) break;
                        }
                        s = s + 1 < AF_SLOTS ? s + 1 : 0;
                    }
                }
                R.es[q][e] = (unsigned char)s;
            }
            hcnt += __popc(bits(added));
        }
        wave_sync();
        return ok;
    };
    for (int u = hl; u < AF_TS; u += 16) {
        R.hcol[u] = -1;
        R.pos[u] = 0;
    }
    for (int u = hl; u <= AF_MMAX; u += 16) R.rb[u] = make_int2(0, AF_NONE * AF_EMAX);
    for (int e = hl; e < AF_EMAX; e += 16) R.es[AF_NONE][e] = (unsigned char)(AF_SLOTS + (e >> 1));
    if (hl == 0) xs[0] = 1.0;
    wave_sync();
    int ibeg;
    bool handed = !table_row(live, 0, i, ibeg) && live;  // the row goes to the merge
    bool active = live && !handed;  // the group's row still grows
    if (active && hl == 0) R.rb[0] = make_int2(ibeg, 0);
    wave_sync();
    int mrow = 0;
    double dko = 0.0;  // DKap of the last step
    // entries 2 hl and 2 hl + 1 of rb's row l: the values and the slots.  Lane 15's places are
    // past every list (AF_EMAX = 30 entries): it takes its own empty slot
    struct Pair {
        D2 v;
        int s0, s1;
    };
    auto load_pair = [&](int2 w) {
        Pair p;
        p.v = *(const D2*)(cs + w.x + 2 * hl);
        unsigned u = *(const unsigned short*)(es + (w.y & 0xffff) + 2 * hl);
        u = hl == 15 ? (AF_TS - 1) * 0x101u : u;
        p.s0 = u & 255;
        p.s1 = u >> 8;
        return p;
    };
    AfSystem sys;
    sys.hl = hl;
    sys.fail = false;
    sys.dl = sys.dh = 0.0;
    for (int step = 0; step < AF_MMAX; step++) {
        // every active row has `step` pattern entries here
        if (__ballot(active) == 0) break;
        // ---------------- Kaporin gradient
        double ba = -1.0;
        int best = INT_MAX, bslot = -1;
        if (active) {
            double2* z = (double2*)R.dense;
#pragma unroll
            for (int u = 0; u < AF_TS / 32; u++) z[hl + 16 * u] = make_double2(0.0, 0.0);
            // each row's products into its columns' slots, the rows in lane order; LDS operations of
            // a wave complete in order, so the adds to one slot keep that order
#pragma unroll 1
            for (int l0 = 0; l0 <= step; l0 += AF_U) {
                Pair p[AF_U];
                double fac[AF_U];
#pragma unroll
                for (int u = 0; u < AF_U; u++) {  // (rows past the pattern have no list)
                    int l = l0 + u <= AF_MMAX ? l0 + u : AF_MMAX;
                    fac[u] = xs[l];
                    p[u] = load_pair(R.rb[l]);
                }
#pragma unroll
                for (int u = 0; u < AF_U; u++) {
                    if (l0 + u > AF_MMAX) break;  // uniform
                    __hip_atomic_fetch_add(&R.dense[p[u].s0], p[u].v.x * fac[u], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                    __hip_atomic_fetch_add(&R.dense[p[u].s1], p[u].v.y * fac[u], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                }
            }
            // the largest |sum| outside the pattern, ties to the smallest column (a NaN never wins)
#pragma unroll
            for (int t = 0; t < AF_TS / 64; t++) {
                int u = 4 * (hl + 16 * t);
                int4 c4 = *(const int4*)&R.hcol[u];
                double2 h0 = *(const double2*)&R.dense[u], h1 = *(const double2*)&R.dense[u + 2];
                int cv[4] = {c4.x, c4.y, c4.z, c4.w};
                double hv[4] = {h0.x, h0.y, h1.x, h1.y};
#pragma unroll
                for (int w = 0; w < 4; w++) {
                    double a = fabs(hv[w]);
                    bool wins = (cv[w] >= 0) & ((a > ba) | ((a == ba) & (cv[w] < best)));
                    ba = wins ? a : ba;
                    best = wins ? cv[w] : best;
                    bslot = wins ? u + w : bslot;
                }
            }
        }
#pragma unroll
        for (int o = 8; o > 0; o >>= 1) {
            double oa = __shfl_xor(ba, o, 16);
            int oc = __shfl_xor(best, o, 16), os = __shfl_xor(bslot, o, 16);
            bool wins = (oa > ba) | ((oa == ba) & (oc < best));
            ba = wins ? oa : ba;
            best = wins ? oc : best;
            bslot = wins ? os : bslot;
        }
        if (!(ba > 0.0)) active = false;  // no new entry: the row is done
        if (__ballot(active) == 0) break;
        // ---------------- insert it into the sorted pattern
        int pa[2];
        int2 pr[2];
#pragma unroll
        for (int h = 0; h < 2; h++) {
            int e = hl + 16 * h;
            pr[h] = active && e < step ? R.rb[e + 1] : make_int2(0, 0);
            pa[h] = active && e < step ? R.hcol[pr[h].y >> 16] & INT_MAX : INT_MAX;
        }
        int q = __popc(bits(pa[0] < best)) + __popc(bits(pa[1] < best));
        int nbeg;
        bool ok = table_row(active, step + 1, best, nbeg);
        if (active) {
#pragma unroll
            for (int h = 0; h < 2; h++) {
                int e = hl + 16 * h;
                if (e >= q && e < step) R.rb[e + 2] = pr[h];
            }
            if (hl == 0) {
                R.rb[q + 1] = make_int2(nbeg, bslot << 16 | (step + 1) * AF_EMAX);
                R.hcol[bslot] |= INT_MIN;
            }
            mrow = step + 1;
            if (!ok) {
                handed = true;
                active = false;
            }
        }
        wave_sync();
        int m = step + 1;
        // ---------------- dense system A_s[P,P] (packed, row p from column 0) and rhs
        double* bb = R.dense + AF_LO;
        int jh = hl + 16 < AF_MMAX ? hl + 16 : AF_MMAX - 1;
#pragma unroll
        for (int c = 0; c < AF_MMAX; c++) sys.hi[c] = 0.0;
        if (active) {
#pragma unroll
            for (int h = 0; h < 2; h++) {
                int e = hl + 16 * h;
                if (e < m) {
                    R.pos[R.rb[e + 1].y >> 16] = (unsigned char)(e + 1);
                    bb[e] = 0.0;
                }
            }
            wave_sync();
            {
                Pair p = load_pair(R.rb[0]);
                int r0 = R.pos[p.s0], r1 = R.pos[p.s1];
                if (r0) bb[r0 - 1] = -p.v.x;
                if (r1) bb[r1 - 1] = -p.v.y;
            }
            // the system's rows [0, 16), then [16, m): scattered from the pattern rows' entries, and loaded
#pragma unroll 1
            for (int p0 = 0; p0 < m; p0 += 16) {
                int p1 = m < p0 + 16 ? m : p0 + 16, off = p0 == 0 ? 0 : AF_LO;
                for (int t = hl; t < p1 * (p1 + 1) / 2 - off; t += 16) R.dense[t] = 0.0;
                wave_sync();
#pragma unroll 1
                for (int a0 = 0; a0 < p1; a0 += AF_U) {
                    Pair p[AF_U];
#pragma unroll
                    for (int u = 0; u < AF_U; u++) p[u] = load_pair(R.rb[a0 + u < AF_MMAX ? a0 + u + 1 : AF_MMAX]);
#pragma unroll
                    for (int u = 0; u < AF_U; u++) {
                        int a = a0 + u, lim = a > p0 ? a : p0;
                        int r0 = R.pos[p[u].s0] - 1, r1 = R.pos[p[u].s1] - 1;
                        if (r0 >= lim && r0 < p1) R.dense[r0 * (r0 + 1) / 2 + a - off] = p[u].v.x;
                        if (r1 >= lim && r1 < p1) R.dense[r1 * (r1 + 1) / 2 + a - off] = p[u].v.y;
                    }
                }
                wave_sync();
                if (p0 == 0) {
                    const double* dl = R.dense + hl * (hl + 1) / 2;
#pragma unroll
                    for (int c = 0; c < 16; c++) sys.lo[c] = dl[c];
                    sys.bl = bb[hl];
                    sys.bh = bb[jh];
                } else {
                    const double* dh = R.dense + jh * (jh + 1) / 2 - AF_LO;
#pragma unroll
                    for (int c = 0; c < AF_MMAX; c++) sys.hi[c] = dh[c];
                }
                wave_sync();
            }
        }
        // the factorisation's first columns are the last step's up to where the new entries went
        int qw = sys.fail ? 0 : active ? q : AF_MMAX;
#pragma unroll
        for (int o = 16; o < 64; o <<= 1) qw = min(qw, __shfl_xor(qw, o, 64));
        double dk = sys.solve(m, __builtin_amdgcn_readfirstlane(qw));
        wave_sync();
        if (active) {
            if (hl == 0) xs[0] = 1.0;
            if (hl < m) xs[hl + 1] = sys.xl;
            if (hl + 16 < m) xs[hl + 17] = sys.xh;
            bool stop = (fabs(dk - dko) < AF_EPS * dko) || dk == 0.0;
            dko = dk;
            if (stop) active = false;
        }
        wave_sync();
    }
    if (handed) {
        if (hl == 0) redo[atomicAdd(nredo, 1)] = i;
        return;
    }
    if (!live) return;
#pragma unroll
    for (int h = 0; h < 2; h++) {
        int e = hl + 16 * h;
        if (e < mrow) {
            pat_out[(long long)i * AF_MMAX + e] = R.hcol[R.rb[e + 1].y >> 16] & INT_MAX;
            x_out[(long long)i * AF_MMAX + e] = xs[e + 1];
        }
    }
    if (hl == 0) {
        mrow_out[i] = mrow;
        dk_out[i] = dko;
    }
}

// Two rows per wave, one per half (32 lanes: the row and its at most 30 pattern
// rows in the gradient), the rows of rows_in: the ones the column table cannot
// take.  The serial parts (Cholesky diagonals, triangular solves, DKap) run for
// both rows in one instruction stream.  Cross-lane operations are always executed
// by the whole wave; a half whose row is done (or past n) only idles through them.
__global__ __launch_bounds__(64 * AF_WAVES) void k_afsai_rows(int n, const int* __restrict__ rows_in, int nrows,
                                                            const int* __restrict__ row, const int* __restrict__ col,
                                                            const double* __restrict__ cs, int* __restrict__ pat_out,
                                                            double* __restrict__ x_out, int* __restrict__ mrow_out,
                                                            double* __restrict__ dk_out) {
    constexpr int NH = 2 * AF_WAVES;
    __shared__ int pat_s[NH][AF_MMAX];
    __shared__ double x_s[NH][AF_MMAX];
    __shared__ double b_s[NH][AF_MMAX];
    __shared__ double L_s[NH][AF_PACK];
    int wid = threadIdx.x >> 6, lane = threadIdx.x & 63;
    int half = lane >> 5, hl = lane & 31;
    int slot = 2 * wid + half;
    long long ri = 2 * ((long long)blockIdx.x * AF_WAVES + wid) + half;
    bool live = ri < (rows_in ? (long long)nrows : (long long)n);
    if (__ballot(live) == 0) return;  // whole wave (LDS is per half; only wave-level sync below)
    int i = live ? (rows_in ? rows_in[ri] : (int)ri) : 0;
    int* pat = pat_s[slot];
    double* xs = x_s[slot];
    double* bb = b_s[slot];
    double* Lp = L_s[slot];
    int mrow = 0;
    double dk = 0.0, dko = 0.0;
    bool active = live;  // the half's row still grows (uniform within the half)
    for (int step = 0; step < AF_MMAX; step++) {
        if (__ballot(active) == 0) break;
        int best = -1;
        {
            // ---------------- Kaporin gradient over columns < i, by merging the rows
            int rr = -1;
            double fac = 0.0;
            if (active) {
                if (hl == 0) { rr = i; fac = 1.0; }
                else if (hl <= mrow) { rr = pat[hl - 1]; fac = xs[hl - 1]; }
            }
            int ptr = 0, end = 0;
            if (rr >= 0) { ptr = row[rr]; end = row[rr + 1]; }
            int pp = 0;  // pattern cursor (uniform within the half)
            double bestabs = -1.0, bestval = 0.0;
            while (true) {
                int cc = (rr >= 0 && ptr < end) ? col[ptr] : INT_MAX;
                if (cc >= i) cc = INT_MAX;
                int jmin = half_min_int(cc);
                bool more = jmin != INT_MAX;
                if (__ballot(more) == 0) break;
                bool hit = more && cc == jmin;
                double contrib = hit ? cs[ptr] * fac : 0.0;
                if (hit) ptr++;
                unsigned mh = (unsigned)(__ballot(hit) >> (32 * half));
                // the column's value: the contributions summed in lane order (both halves
                // take as many shuffles as the larger count)
                int cnt = __popc(mh);
                int c0 = __shfl(cnt, 0, 64), c1 = __shfl(cnt, 32, 64);
                int cmax = c0 > c1 ? c0 : c1;
                double acc = 0.0;
                for (int q = 0; q < cmax; q++) {
                    int b = mh ? __ffs(mh) - 1 : 0;
                    double v = __shfl(contrib, b, 32);
                    if (mh) {
                        acc += v;
                        mh &= mh - 1;
                    }
                }
                if (more) {
                    while (pp < mrow && pat[pp] < jmin) pp++;
                    bool inpat = pp < mrow && pat[pp] == jmin;
                    double a = inpat ? 0.0 : fabs(acc);
                    if (a > bestabs) {
                        bestabs = a;
                        best = jmin;
                        bestval = inpat ? 0.0 : acc;
                    }
                }
            }
            if (active && (best < 0 || bestval == 0.0)) active = false;  // no new entry: the row is done
        }
        if (__ballot(active) == 0) break;
        // insert `best` into the sorted pattern (the half's lane 0)
        if (active && hl == 0) {
            int q = mrow;
            while (q > 0 && pat[q - 1] > best) {
                pat[q] = pat[q - 1];
                q--;
            }
            pat[q] = best;
        }
        wave_sync();
        if (active) mrow++;
        // ---------------- dense system A_s[P,P] and rhs
        if (active) {
            for (int t = hl; t < mrow * (mrow + 1) / 2; t += 32) Lp[t] = 0.0;
            if (hl < mrow) bb[hl] = 0.0;
        }
        wave_sync();
        if (active && hl < mrow) {
            int a = hl;
            int r2 = pat[a];
            int jj = row[r2], je = row[r2 + 1];
            for (int b = a; b < mrow; b++) {
                while (jj < je && col[jj] < pat[b]) jj++;
                if (jj == je) break;
                if (col[jj] == pat[b]) Lp[b * (b + 1) / 2 + a] = cs[jj];
            }
        }
        if (active && hl == 0) {
            int jj = row[i], je = row[i + 1], ii = 0;
            while (jj < je && col[jj] < i && ii < mrow) {
                if (pat[ii] > col[jj]) jj++;
                else if (pat[ii] == col[jj]) { bb[ii] = -cs[jj]; jj++; ii++; }
                else ii++;
            }
        }
        wave_sync();
        // ---------------- Cholesky (cudacholdcMix order)
        bool fail = false;
        int mh0 = __shfl(active ? mrow : 0, 0, 64), mh1 = __shfl(active ? mrow : 0, 32, 64);
        int mmax = mh0 > mh1 ? mh0 : mh1;
        for (int ci = 0; ci < mmax; ci++) {
            bool on = active && !fail && ci < mrow;  // uniform within the half
            // diagonal
            const double* lc = Lp + ci * (ci + 1) / 2;
            double sum = 0.0;
            if (on && hl == 0) {
                auto Lc = [&](int k) { return lc[k]; };
                sum = af_chain<false>(lc[ci], ci, Lc, Lc);
                if (!(sum <= 0.0)) Lp[ci * (ci + 1) / 2 + ci] = 1. / sqrt(sum);
            }
            sum = __shfl(sum, 0, 32);
            if (on && sum <= 0.0) {
                fail = true;
                on = false;
            }
            wave_sync();
            int j = ci + 1 + hl;
            if (on && j < mrow) {
                const double* lj = Lp + j * (j + 1) / 2;
                double s2 = af_chain<false>(lj[ci], ci, [&](int k) { return lc[k]; }, [&](int k) { return lj[k]; });
                Lp[j * (j + 1) / 2 + ci] = s2 * lc[ci];
            }
            wave_sync();
        }
        // b kept for DKap; x solved in x_s (on breakdown x = b, as the reference leaves it)
        if (active && hl == 0) {
            for (int t = 0; t < mrow; t++) xs[t] = bb[t];
            if (!fail) {
                // L y = b, row a's terms b = a-1 down to 0; then L^T x = y, terms b = a+1 up
                for (int a = 0; a < mrow; a++) {
                    const double* la = Lp + a * (a + 1) / 2;
                    double s = af_chain<false>(xs[a], a, [&](int t) { return la[a - 1 - t]; },
                                               [&](int t) { return xs[a - 1 - t]; });
                    xs[a] = s * la[a];
                }
                for (int a = mrow - 1; a >= 0; a--) {
                    double s = af_chain<false>(xs[a], mrow - 1 - a,
                                               [&](int t) { return Lp[(a + 1 + t) * (a + 2 + t) / 2 + a]; },
                                               [&](int t) { return xs[a + 1 + t]; });
                    xs[a] = s * Lp[a * (a + 1) / 2 + a];
                }
            }
            dk = af_chain<true>(0.0, mrow, [&](int e) { return bb[e]; }, [&](int e) { return xs[e]; });
        }
        wave_sync();
        dk = __shfl(dk, 0, 32);
        if (active) {
            bool stop = (fabs(dk - dko) < AF_EPS * dko) || dk == 0.0;
            dko = dk;
            if (stop) active = false;
        }
    }
    if (live && hl < mrow) {
        pat_out[(long long)i * AF_MMAX + hl] = pat[hl];
        x_out[(long long)i * AF_MMAX + hl] = xs[hl];
    }
    if (live && hl == 0) {
        mrow_out[i] = mrow;
        dk_out[i] = dk;
    }
}

__global__ void k_g_rowlen(int n, const int* __restrict__ mrow, int* __restrict__ len) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) len[i] = mrow[i] + 1;
}

// createprc (afsai.cu:165-202)
__global__ void k_createprc(int n, const double* __restrict__ cs, const int* __restrict__ dind, const int* __restrict__ pat,
                            const double* __restrict__ xs, const int* __restrict__ mrow, const double* __restrict__ dk,
                            const int* __restrict__ grow, int* __restrict__ gcol, double* __restrict__ gval) {
    // 32 lanes a row, one entry each (27-point 128^3: 3.3 ms with one thread a row, 0.54 ms)
    static_assert(AF_MMAX < 32, "a lane for every entry");
    int i = (int)(((long long)blockIdx.x * blockDim.x + threadIdx.x) / 32);
    int k = (int)threadIdx.x % 32;
    if (i >= n) return;
    int o = grow[i], m = mrow[i];
    if (k > m) return;
    double sc = cs[dind[i]] - dk[i];
    // a negative scaling factor (afsai.cu:187): off-diagonals left at their zero initialisation
    bool pos = sc > 0.0;
    sc = pos ? 1.0 / sqrt(sc) : 1.0;
    if (k < m) {
        gval[o + k] = pos ? sc * xs[(long long)i * AF_MMAX + k] : 0.0;
        gcol[o + k] = pos ? pat[(long long)i * AF_MMAX + k] : 0;
    } else {
        gval[o + m] = sc;
        gcol[o + m] = i;
    }
}

void afsai_build(Context* c, const DCsr& A, DCsr& G, DCsr& GT) {
    int n = A.n;
    BCMGX_CHECK(A.n == A.m, BCMGX_ERR_ARG, "AFSAI needs a square matrix");
    DBuf<int> dind(c, std::max(n, 1));
    diag_index(c, n, A.row.get(), A.col.get(), dind.get());
    BCMGX_CHECK(count_missing_diagonals(c, n, dind.get()) == 0, BCMGX_ERR_ARG, "AFSAI: row without diagonal entry");
    DBuf<double> d(c, std::max(n, 1)), cs(c, (size_t)A.nnz + AF_PAD);
    k_scale_diag<<<grid_for(n, WG), WG, 0, c->stream>>>(n, A.val.get(), dind.get(), d.get());
    BCMGX_LAUNCHED();
    k_scale_A<<<grid_for((long long)n * 16, WG), WG, 0, c->stream>>>(n, A.row.get(), A.col.get(), A.val.get(), d.get(), cs.get());
    BCMGX_LAUNCHED();
    DBuf<int> pat(c, (size_t)std::max(n, 1) * AF_MMAX), mrow(c, std::max(n, 1));
    DBuf<double> xs(c, (size_t)std::max(n, 1) * AF_MMAX), dk(c, std::max(n, 1));
    DBuf<int> redo(c, std::max(n, 1)), nredo(c, 1);
    fill<int>(c, nredo.get(), 1, 0);
    k_afsai_table<<<grid_for(n, AF4_ROWS), 64, 0, c->stream>>>(n, A.row.get(), A.col.get(), cs.get(), pat.get(), xs.get(),
                                                               mrow.get(), dk.get(), redo.get(), nredo.get());
    BCMGX_LAUNCHED();
    int nr = c->read1(nredo.get());  // rows the column table could not take
    if (nr > 0) {
        k_afsai_rows<<<grid_for(nr, 2 * AF_WAVES), 64 * AF_WAVES, 0, c->stream>>>(
            n, redo.get(), nr, A.row.get(), A.col.get(), cs.get(), pat.get(), xs.get(), mrow.get(), dk.get());
        BCMGX_LAUNCHED();
    }
    DBuf<int> len(c, std::max(n, 1));
    k_g_rowlen<<<grid_for(n, WG), WG, 0, c->stream>>>(n, mrow.get(), len.get());
    BCMGX_LAUNCHED();
    G.n = G.m = n;
    G.row.reset(c, (size_t)n + 1);
    long long nnz = scan_exclusive(c, len.get(), G.row.get(), n);
    G.nnz = (int)nnz;
    G.col.reset(c, std::max<long long>(nnz, 1));
    G.val.reset(c, std::max<long long>(nnz, 1));
    k_createprc<<<grid_for((long long)n * 32, WG), WG, 0, c->stream>>>(n, cs.get(), dind.get(), pat.get(), xs.get(), mrow.get(), dk.get(),
                                                      G.row.get(), G.col.get(), G.val.get());
    BCMGX_LAUNCHED();
    transpose(c, G, GT);
    c->sync();
}

}  // namespace bcmgx
