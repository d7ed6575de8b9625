// tiled.hip -- k-column products straight from column-major columns over the row-tile index.
//
// The public product takes its k columns column-major.  Through the interleaved
// kernels that is three passes (columns in, product, columns out), and the product
// gathers one row of x per entry through the L1.  Here a workgroup owns a tile of 64
// consecutive rows.  It keeps the tile's entries in registers, one row a lane (the
// four waves each hold all 64 rows), brings the tile's distinct columns of x into LDS
// 4 vector columns at a time (runs of consecutive columns: coalesced in the
// column-major layout) and each wave sums one of those columns from LDS; the next
// ones are in flight meanwhile.  y leaves 64 rows of a column at a time.  x goes
// through the L1 once per tile and distinct column (9.3 per row on the 27-point
// grid, not 27), and nothing is transposed.
//
// Whole calls, transposed columns and this: 27-point 128^3, k = 32: 1210 and 695 us
// (memory 374 us), k = 8: 527 and 270, k = 2: 963 and 177; 7-point 128^3, k = 32: 838
// and 563; 27-point 10^3, any k: 27 and 16.  Bound by the latency of a step (load,
// barrier, 27 dependent sums; a test of the row length per 4 entries, not 8, 727): 8 columns
// a step, with 3 waves a SIMD where 4 columns
// have 4, gave 912 us; loads under branches, waited for one by one, 1547.
//
// Each column's sum runs over the row in order, product and sum rounded apart, as in
// the interleaved kernels: the same bits.
#include "kernels.h"

namespace bcmgx {

constexpr int CM_WAVES = WG / 64;
constexpr int CM_ORDER = 32;  // tiles of a super-block dealt to an XCD
constexpr int cm_waves_simd(int E) { return E > 28 ? 3 : 4; }  // as many as the entries' registers leave
static_assert(TILE_ROWS == 64, "a row of the tile per lane");

template <SpOp OP>
__device__ __forceinline__ void cm_store(double* __restrict__ y, double t, double beta) {
    if (OP == SpOp::RES) t = *y - t;
    else if (OP == SpOp::AXPBY) t = t + beta * *y;
    __builtin_nontemporal_store(t, y);
}

// y = op(A x) on column-major columns; rows of at most E entries, tiles of fewer than S distinct
// columns; C vector columns at a time.  blockIdx.y: its share of the columns.  Loads are
// unconditional (indices clamped), so that those of a phase are in flight together.
template <int E, int C, int S, SpOp OP>
__global__ __launch_bounds__(WG, cm_waves_simd(E)) void k_spmm_cm(int n, int k, int ld, int share, const int* __restrict__ row,
                                                         const double* __restrict__ val, const int* __restrict__ tu,
                                                         const int* __restrict__ tucol,
                                                         const unsigned short* __restrict__ tlidx, const double* __restrict__ x,
                                                         double* __restrict__ y, double alpha, double beta, int sb) {
    constexpr int CW = C / CM_WAVES, P = (S + WG - 1) / WG < TILE_MAX_COLS / WG ? (S + WG - 1) / WG : TILE_MAX_COLS / WG;
    constexpr int NE = E * TILE_ROWS, Q = NE / WG;  // a tile's entries, per thread
    static_assert(E % 4 == 0 && C % CM_WAVES == 0, "four entries at a time, as many columns for every wave");
    // the entries (values, then positions), then C columns of S places; a row's unused places may read E past its entries
    constexpr int POOL = C * S * 8 > (NE + E) * 10 ? C * S : (NE + E) * 10 / 8;
    __shared__ double pool[POOL];
    unsigned short* sl = (unsigned short*)(pool + NE + E);
    int blk = xcd_order(blockIdx.x, gridDim.x, sb);
    int tid = threadIdx.x, lane = tid & 63, w = tid / 64;
    int r0 = blk * TILE_ROWS, rend = r0 + TILE_ROWS < n ? r0 + TILE_ROWS : n;
    int base = row[r0], cnt = row[rend] - base;
    int u0 = tu[blk], U = tu[blk + 1] - u0;
    int c0 = blockIdx.y * share, c1 = c0 + share < k ? c0 + share : k;
    int r = r0 + lane;
    if (cnt == 0) {  // nothing to load
        for (int c = c0 + w; r < n && c < c1; c += CM_WAVES) cm_store<OP>(y + (long long)c * ld + r, 0.0, beta);
        return;
    }
    int s = row[r < n ? r : n] - base, len = row[r < n ? r + 1 : n] - base - s;
    int uc[P];
#pragma unroll
    for (int p = 0; p < P; p++) uc[p] = tucol[u0 + (tid + p * WG < U ? tid + p * WG : U - 1)];
    double ev[Q];
    unsigned short el[Q];
#pragma unroll
    for (int q = 0; q < Q; q++) {
        int t = base + (tid + q * WG < cnt ? tid + q * WG : cnt - 1);
        ev[q] = ldg_nt(val + t);
        el[q] = tlidx[t];
    }
    double xv[C][P];
    auto fetch = [&](int c) {
#pragma unroll
        for (int q = 0; q < C; q++) {
            const double* xc = x + (long long)(c + q < c1 ? c + q : c1 - 1) * ld;
#pragma unroll
            for (int p = 0; p < P; p++) xv[q][p] = xc[uc[p]];
        }
    };
    fetch(c0);
#pragma unroll
    for (int q = 0; q < Q; q++) {
        pool[tid + q * WG] = OP == SpOp::AXPBY ? alpha * ev[q] : ev[q];
        sl[tid + q * WG] = el[q];
    }
    __syncthreads();
    // this lane's row; unused places: value 0 at the zero place U
    double a[E];
    unsigned l2[E / 2];
#pragma unroll
    for (int j = 0; j < E; j += 2) {
        double a0 = pool[s + j], a1 = pool[s + j + 1];
        unsigned lo = sl[s + j], hi = sl[s + j + 1];
        a[j] = j < len ? a0 : 0.0;
        a[j + 1] = j + 1 < len ? a1 : 0.0;
        l2[j / 2] = (j < len ? lo : U) | (j + 1 < len ? hi : U) << 16;
    }
    for (int c = c0; c < c1; c += C) {
        __syncthreads();  // the entries, or the columns before, are read
#pragma unroll
        for (int q = 0; q < C; q++)
#pragma unroll
            for (int p = 0; p < P; p++) {
                int u = tid + p * WG;  // past the list: zeros to the zero place
                pool[q * S + (u < U ? u : U)] = u < U ? xv[q][p] : 0.0;
            }
        if (tid < C) pool[tid * S + U] = 0.0;  // (no thread is past a list of P * WG)
        __syncthreads();
        if (c + C < c1) fetch(c + C);
        const double* xs = pool + w * CW * S;
        double t[CW];
#pragma unroll
        for (int q = 0; q < CW; q++) t[q] = 0.0;
#pragma unroll
        for (int j = 0; j < E; j += 4) {
            if (j % 8 == 0 && !__any(j < len)) break;
            unsigned p01 = l2[j / 2], p23 = l2[j / 2 + 1];
            asm("" : "+v"(p01), "+v"(p23));  // unpacked here: E addresses kept over the columns would spill
            const double* x0 = xs + (p01 & 0xffffu);
            const double* x1 = xs + (p01 >> 16);
            const double* x2 = xs + (p23 & 0xffffu);
            const double* x3 = xs + (p23 >> 16);
            double v[CW][4];
#pragma unroll
            for (int q = 0; q < CW; q++) v[q][0] = x0[q * S], v[q][1] = x1[q * S], v[q][2] = x2[q * S], v[q][3] = x3[q * S];
#pragma unroll
            for (int u = 0; u < 4; u++)
#pragma unroll
                for (int q = 0; q < CW; q++) t[q] += a[j + u] * v[q][u];
        }
#pragma unroll
        for (int q = 0; q < CW; q++) {
            int cc = c + w * CW + q;
            if (r < n && cc < c1) cm_store<OP>(y + (long long)cc * ld + r, t[q], beta);
        }
    }
}

template <int E, int C, int S>
static void launch_cm(Context* c, SpOp op, const DCsr& A, const double* x, double* y, int k, int ld, double alpha, double beta) {
    int nt = (int)grid_for(A.n, TILE_ROWS);
    // small matrices: the columns shared out so that the device has work
    int parts = std::min((k + C - 1) / C, std::max(1, 1024 / nt));
    int share = ((k + parts - 1) / parts + C - 1) / C * C;
    dim3 g(nt, (k + share - 1) / share);
#define BCMGX_CM(OO)                                                                                              \
    k_spmm_cm<E, C, S, OO><<<g, WG, 0, c->stream>>>(A.n, k, ld, share, A.row.get(), A.val.get(), A.tu.get(),      \
                                                    A.tucol.get(), A.tlidx.get(), x, y, alpha, beta, CM_ORDER)
    if (op == SpOp::AX) BCMGX_CM(SpOp::AX);
    else if (op == SpOp::RES) BCMGX_CM(SpOp::RES);
    else BCMGX_CM(SpOp::AXPBY);
#undef BCMGX_CM
    BCMGX_LAUNCHED();
}

bool spmm_colmajor(Context* c, SpOp op, const DCsr& A, const double* x, double* y, int k, int ld, double alpha, double beta) {
    if (k < 2 || !A.tiled() || A.tiles_left_out != 0 || A.maxrow < 1 || A.maxrow > 32 || op == SpOp::JACOBI) return false;
    // runs of 8 consecutive columns on average, whole 64-byte pieces of x: grids of 5 points a side have 15; with
    // scattered columns a load here brings 8 bytes where the interleaved rows bring all k columns
    if (A.tile_cols < 8 * A.tile_runs) return false;
    bool wide = A.tile_widest >= 640;
#define BCMGX_E(EE)                                                                        \
    if (A.maxrow <= EE) {                                                                  \
        if (wide) launch_cm<EE, 4, TILE_MAX_COLS + 64>(c, op, A, x, y, k, ld, alpha, beta); \
        else launch_cm<EE, 4, 640>(c, op, A, x, y, k, ld, alpha, beta);                    \
        return true;                                                                       \
    }
    BCMGX_E(8) BCMGX_E(16) BCMGX_E(28) BCMGX_E(32)
#undef BCMGX_E
    return false;
}

}  // namespace bcmgx
