// blocked.hip -- k-column products on the matrix cores from a 16-row block form.
//
// The k-column SpMM gathers one row of x (k values) per matrix entry; on the
// 27-point grid that is 27 row loads per row, and the L1 and texture path that
// carry them bound k_spmmp (88-96% busy, memory at half its rate).  But rows share
// columns: 16 rows that the first coarsening puts into the same aggregates (a
// 4 x 2 x 2 brick there) touch 101 distinct ones for 426 entries.  Here a wave
// owns 16 rows and loads each distinct column's x once, straight into the B
// operand of a 16x16x4 MFMA (lane l: column l / 16 of a group of four, vector
// columns l % 16), against the 16 x 4 block of the matrix as A operand (lane l:
// row l % 16, column l / 16 of the group).  4.2 times fewer x loads; the zeros of
// a block cost matrix-core time that is otherwise idle.
//
// Measured on 27-point 128^3, FP32 columns, k = 32: y = A x 373 -> 185 us, the
// level-0 residual (r read in FP64) 430 -> 284 us, FCG's fused FP64 product 672 ->
// 517 us; the last two now move 1.7 and 3.0 GB at 5.9 TB/s, above the copy rate.
// Sixteen consecutive rows instead of aggregated ones (164 columns) gave 270, 348
// and 690 us: bound by the L1's outstanding misses.
//
// Block form, built once per pattern (1.5 ms at 128^3) and kept with the matrix:
// per tile of 16 rows the sorted distinct columns in groups of four; per group a
// 64-bit mask of the entries present (bit l: lane l's) and the entries' values in
// bit order.  A lane finds its value at the group's offset plus the number of
// mask bits below its own, so the form reads 4 (8) bytes per entry, 8 per group
// and 4 per column: 144 bytes per row in FP32 against CSR's 216.  Columns are
// stored 16 groups at a time, [column of the group][group], so one load per 16
// groups brings them and a DPP broadcast hands them out.
//
// Sums are fused multiply-adds in column order (MFMA), not the separate
// products and sums of the CSR kernels: the FP32 V-cycle and the fused FCG
// product use them, the public products keep theirs.
#include "kernels.h"

#include <climits>
#include <utility>

namespace bcmgx {

typedef unsigned long long u64;
constexpr int BT = BLK_ROWS;
constexpr int BLK_ORDER = 32;           // workgroups (64 rows each) of a super-block dealt to an XCD
constexpr int BLK_MAX_ENTRIES = 512;  // entries of a tile (rows of up to 32)
constexpr int BLK_STAGE = BLK_MAX_ENTRIES + 4;  // a wave's share of LDS
constexpr int BLK_HASH = 1024;
constexpr int BLK_LOADS = 4;             // x loads in flight together (8: no faster, more registers)

__device__ __forceinline__ void blk_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// One wave per tile: its distinct columns (hashed, compacted, sorted) into
// list[t * stride ...], their number, its entries' number, and each entry's
// place among the columns.
__global__ __launch_bounds__(64) void k_blk_columns(int n, const int* __restrict__ rows, const int* __restrict__ row,
                                                    const int* __restrict__ col, int stride, int* __restrict__ ucnt,
                                                    int* __restrict__ vcnt, int* __restrict__ list,
                                                    unsigned short* __restrict__ upos) {
    __shared__ int hkey[BLK_HASH];
    __shared__ int keys[BLK_MAX_ENTRIES];
    __shared__ unsigned short rank[BLK_HASH];
    int t = blockIdx.x, lane = threadIdx.x;
    // 16 lanes to a row, four rows at a time: f(entry) for all lanes at once, -1 past a row's end
    auto each_entry = [&](auto f) {
        for (int q = lane / 16; q < BT; q += 4) {
            int s = 0, e = 0;
            if (t * BT + q < n) {
                int r = rows[t * BT + q];
                s = row[r];
                e = row[r + 1];
            }
            for (int j = s + lane % 16; __any(j < e); j += 16) f(j < e ? j : -1);
        }
    };
    int cnt = 0;
    if (lane < BT && t * BT + lane < n) {
        int r = rows[t * BT + lane];
        cnt = row[r + 1] - row[r];
    }
    for (int o = 1; o < 64; o <<= 1) cnt += __shfl_xor(cnt, o, 64);
    int H = 128;  // a power of two, at least twice the entries
    while (H < 2 * cnt) H <<= 1;
    auto slot_of = [&](int c) { return (int)(((unsigned)c * 2654435761u) >> 16) & (H - 1); };
    for (int u = lane; u < H; u += 64) hkey[u] = -1;
    blk_sync();
    int U = 0;
    each_entry([&](int j) {
        int c = -1;
        bool fresh = false;
        if (j >= 0) {
            c = col[j];
            int s = slot_of(c);
            while (true) {  // at most H / 2 columns: an empty slot ends the probe
                int old = atomicCAS(&hkey[s], -1, c);
                if (old == -1) fresh = true;
                if (old == -1 || old == c) break;
                s = (s + 1) & (H - 1);
            }
        }
        u64 m = __ballot(fresh);
        if (fresh) keys[U + __popcll(m & ((1ull << lane) - 1ull))] = c;
        U += __popcll(m);
    });
    int P = 1;
    while (P < U) P <<= 1;
    for (int u = U + lane; u < P; u += 64) keys[u] = INT_MAX;
    blk_sync();
    for (int kk = 2; kk <= P; kk <<= 1)
        for (int j = kk >> 1; j > 0; j >>= 1) {
            for (int p = lane; p < P / 2; p += 64) {
                int a = ((p & ~(j - 1)) << 1) | (p & (j - 1)), b = a | j;
                int x = keys[a], y = keys[b];
                if ((x > y) == ((a & kk) == 0)) {
                    keys[a] = y;
                    keys[b] = x;
                }
            }
            blk_sync();
        }
    for (int u = lane; u < U; u += 64) {
        int c = keys[u], s = slot_of(c);
        while (hkey[s] != c) s = (s + 1) & (H - 1);
        rank[s] = (unsigned short)u;
        list[(long long)t * stride + u] = c;
    }
    if (lane == 0) {
        ucnt[t] = U;
        vcnt[t] = cnt;
    }
    blk_sync();
    each_entry([&](int j) {
        if (j < 0) return;
        int c = col[j], s = slot_of(c);
        while (hkey[s] != c) s = (s + 1) & (H - 1);
        upos[j] = rank[s];
    });
}

__global__ void k_blk_counts(int nt, const int* __restrict__ ucnt, int* __restrict__ groups, int* __restrict__ blocks) {
    int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nt) return;
    int g = (ucnt[t] + 3) / 4;
    groups[t] = g;
    blocks[t] = (g + 15) / 16;
}

// per tile: its columns 16 groups at a time (the tail repeats the last column) and its masks; twice
// counts the entries whose column the row has already listed
__global__ __launch_bounds__(64) void k_blk_masks(int n, const int* __restrict__ rows, const int* __restrict__ row, int stride, const int* __restrict__ ucnt,
                                                  const int* __restrict__ list, const unsigned short* __restrict__ upos,
                                                  const int* __restrict__ gptr, const int* __restrict__ bptr,
                                                  int* __restrict__ bcol, u64* __restrict__ bmask, int* __restrict__ twice) {
    __shared__ u64 mask[BLK_MAX_ENTRIES / 4];
    int t = blockIdx.x, lane = threadIdx.x;
    int U = ucnt[t], G = (U + 3) / 4, NB = (G + 15) / 16;
    for (int g = lane; g < G; g += 64) mask[g] = 0;
    blk_sync();
    for (int b = 0; b < NB; b++) {
        int u = 4 * (16 * b + lane % 16) + lane / 16;
        bcol[64ll * (bptr[t] + b) + lane] = list[(long long)t * stride + (u < U ? u : U - 1)];
    }
    for (int q = lane / 16; q < BT; q += 4) {
        if (t * BT + q >= n) break;
        int r = rows[t * BT + q];
        for (int j = row[r] + lane % 16; j < row[r + 1]; j += 16) {
            int u = upos[j];
            u64 bit = 1ull << ((u & 3) * 16 + q);
            if (atomicOr(&mask[u >> 2], bit) & bit) atomicAdd(twice, 1);
        }
    }
    blk_sync();
    for (int g = lane; g < G; g += 64) bmask[gptr[t] + g] = mask[g];
}

// values into block order
template <typename T>
__global__ __launch_bounds__(64) void k_blk_values(int n, const int* __restrict__ rows, const int* __restrict__ row, const int* __restrict__ vptr, const double* __restrict__ val,
                                                   const unsigned short* __restrict__ upos, const int* __restrict__ gptr,
                                                   const u64* __restrict__ bmask, T* __restrict__ bval) {
    __shared__ u64 mask[BLK_MAX_ENTRIES / 4];
    __shared__ int off[BLK_MAX_ENTRIES / 4];
    int t = blockIdx.x, lane = threadIdx.x;
    int g0 = gptr[t], G = gptr[t + 1] - g0;
    int base = vptr[t], carry = 0;
    for (int c0 = 0; c0 < G; c0 += 64) {
        u64 m = c0 + lane < G ? bmask[g0 + c0 + lane] : 0;
        int p = __popcll(m), s = p;
        for (int o = 1; o < 64; o <<= 1) {
            int v = __shfl_up(s, o, 64);
            if (lane >= o) s += v;
        }
        if (c0 + lane < G) {
            mask[c0 + lane] = m;
            off[c0 + lane] = carry + s - p;
        }
        carry += __shfl(s, 63, 64);
    }
    blk_sync();
    for (int q = lane / 16; q < BT; q += 4) {
        if (t * BT + q >= n) break;
        int r = rows[t * BT + q];
        for (int j = row[r] + lane % 16; j < row[r + 1]; j += 16) {
            int u = upos[j], bit = (u & 3) * 16 + q;
            bval[base + off[u >> 2] + __popcll(mask[u >> 2] & ((1ull << bit) - 1ull))] = (T)val[j];
        }
    }
}

template <typename T>
static void block_values(Context* c, const DCsr& A, DBuf<T>& out) {
    // a tile's last 16-byte load may reach three elements past the array
    if (!out) out.reset(c, (size_t)A.nnz + 4);
    k_blk_values<T><<<grid_for(A.n, BT), 64, 0, c->stream>>>(A.n, A.blk.rows.get(), A.row.get(), A.blk.vptr.get(), A.val.get(), A.blk.upos.get(), A.blk.gptr.get(),
                                                             A.blk.mask.get(), out.get());
    BCMGX_LAUNCHED();
}

static bool form_blocks(Context* c, DCsr& A, const int* order, double min_reuse) {
    if (A.blk.refused || A.n <= 0 || A.maxrow < 1 || A.maxrow * BT > BLK_MAX_ENTRIES) return false;
    int nt = (A.n + BT - 1) / BT, stride = A.maxrow * BT;
    DBuf<int> ucnt(c, nt), vcnt(c, nt), groups(c, nt), blocks(c, nt), gptr(c, (size_t)nt + 1), bptr(c, (size_t)nt + 1),
        vptr(c, (size_t)nt + 1), rows(c, A.n);
    copy_d2d(c, rows.get(), order, sizeof(int) * (size_t)A.n);
    DBuf<int> list(c, (size_t)nt * stride);
    DBuf<unsigned short> upos(c, (size_t)std::max(A.nnz, 1));
    k_blk_columns<<<nt, 64, 0, c->stream>>>(A.n, rows.get(), A.row.get(), A.col.get(), stride, ucnt.get(), vcnt.get(),
                                              list.get(), upos.get());
    BCMGX_LAUNCHED();
    k_blk_counts<<<grid_for(nt, WG), WG, 0, c->stream>>>(nt, ucnt.get(), groups.get(), blocks.get());
    BCMGX_LAUNCHED();
    scan_exclusive_async(c, vcnt.get(), vptr.get(), nt);
    long long ng = scan_exclusive(c, groups.get(), gptr.get(), nt), nb = scan_exclusive(c, blocks.get(), bptr.get(), nt);
    A.blk.groups = ng;
    A.blk.m = A.m;
    // the blocks pay when they bring down the x rows loaded (4 per group) well below one per entry
    if ((double)A.nnz < min_reuse * 4.0 * (double)ng) {
        A.blk.refused = true;
        return false;
    }
    DBuf<int> bcol(c, (size_t)(nb + 1) * 64);
    DBuf<u64> mask(c, (size_t)ng + 16);
    DBuf<int> twice(c, 1);
    fill<int>(c, twice.get(), 1, 0);
    k_blk_masks<<<nt, 64, 0, c->stream>>>(A.n, rows.get(), A.row.get(), stride, ucnt.get(), list.get(), upos.get(), gptr.get(), bptr.get(),
                                          bcol.get(), mask.get(), twice.get());
    BCMGX_LAUNCHED();
    // a block has one place per row and column: a matrix that lists a column twice in a row, which
    // the CSR products add up, stays with them
    if (c->read1(twice.get()) != 0) {
        A.blk.refused = true;
        return false;
    }
    A.blk.rows = std::move(rows);
    A.blk.vptr = std::move(vptr);
    A.blk.gptr = std::move(gptr);
    A.blk.bptr = std::move(bptr);
    A.blk.col = std::move(bcol);
    A.blk.mask = std::move(mask);
    A.blk.upos = std::move(upos);
    return true;
}

bool build_blocks(Context* c, DCsr& A, const int* order, double min_reuse) {
    if (A.blk.built()) return true;
    try {
        return form_blocks(c, A, order, min_reuse);
    } catch (const Error& e) {  // no memory for it now: the products run from CSR as before
        if (e.code != BCMGX_ERR_ALLOC) throw;
        A.blk = BlockForm();
        return false;
    }
}

template <typename T>
static bool have_values(Context* c, DCsr& A, DBuf<T>& out) {
    if (!A.blk.built()) return false;
    try {
        if (!out) block_values<T>(c, A, out);
        return true;
    } catch (const Error& e) {
        if (e.code != BCMGX_ERR_ALLOC) throw;
        return false;
    }
}
bool block_values32(Context* c, DCsr& A) { return have_values(c, A, A.blk.val32); }
bool block_values64(Context* c, DCsr& A) { return have_values(c, A, A.blk.val64); }
void refresh_blocks(Context* c, DCsr& A) {
    if (A.blk.val32) block_values<float>(c, A, A.blk.val32);
    if (A.blk.val64) block_values<double>(c, A, A.blk.val64);
}

// ------------------------------------------------------------- products ---
struct BlkOps {
    const int* gptr;
    const int* bptr;
    const int* col;
    const u64* mask;
    const int* vptr;  // tile -> its first value
    const int* rows;  // tile's rows
    int n;
};

template <int... J, typename F>
__device__ __forceinline__ void blk_each(std::integer_sequence<int, J...>, F&& f) {
    (f(std::integral_constant<int, J>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void blk_for(F&& f) {
    blk_each(std::make_integer_sequence<int, N>{}, f);
}
// old, with the lanes of the banks (4 lanes each) of BANKS taking src through the DPP control CTRL
template <int CTRL, int BANKS>
__device__ __forceinline__ int blk_dpp(int old, int src) {
    return __builtin_amdgcn_update_dpp(old, src, CTRL, 0xf, BANKS, false);
}
template <int CTRL, int BANKS>
__device__ __forceinline__ float blk_dpp(float old, float src) {
    return __int_as_float(blk_dpp<CTRL, BANKS>(__float_as_int(old), __float_as_int(src)));
}
template <int CTRL, int BANKS>
__device__ __forceinline__ double blk_dpp(double old, double src) {
    int lo = blk_dpp<CTRL, BANKS>(__double2loint(old), __double2loint(src));
    return __hiloint2double(blk_dpp<CTRL, BANKS>(__double2hiint(old), __double2hiint(src)), lo);
}
constexpr int DPP_BCAST = 0x150, DPP_ROR = 0x120;

typedef float blk_f4 __attribute__((ext_vector_type(4)));
typedef double blk_d4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ blk_f4 blk_mfma(float a, float b, blk_f4 acc) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, acc, 0, 0, 0); }
__device__ __forceinline__ blk_d4 blk_mfma(double a, double b, blk_d4 acc) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, acc, 0, 0, 0); }

// k = 4 P vector columns.  An x row is loaded by P lanes, four columns (16
// bytes) each: the texture path takes four lanes at a time, so 16-byte loads move
// twice the bytes of 8-byte ones (k = 32 with 8-byte loads: no faster than
// k_spmmp).  One load thus brings R = 16 / P groups: of the 16 lanes that carry
// column kk of a group in the MFMA, lanes [P e, P e + P) hold it for group e.
// split() moves the four values between those lanes (DPP rotations) into the
// operands of the R groups; the vector column of lane n in operand b follows
// from that, and join() undoes it for the rows of the result.  k = 8 fills half
// of an operand; the other lanes carry another group's values into result
// columns that are never written.
template <int P>
struct BlkCols {
    static constexpr int R = 16 / P, K = 4 * P;
    static constexpr int NB = P < 4 ? 1 : P / 4;   // operands per group
    static constexpr int STEPS = R < 4 ? 4 / R : 1;  // rows of its four that a lane writes
    // operand B of group E from the four loaded values
    template <int E, int B>
    static __device__ __forceinline__ float split(const blk_f4& r) {
        if constexpr (R == 1) return r[B];
        else if constexpr (R == 2) {
            if constexpr (E == 0) return blk_dpp<DPP_ROR + 8, 0xc>(r[2 * B], r[2 * B + 1]);
            else return blk_dpp<DPP_ROR + 8, 0x3>(r[2 * B + 1], r[2 * B]);
        } else {  // bank b takes value b
            constexpr int b0 = P * E % 4 == 0 ? P * E / 4 : -1;  // the bank that holds its own
            float v = r[b0 < 0 ? 0 : b0];
            blk_for<4>([&](auto bc) {
                constexpr int b = bc;
                if constexpr (b != b0) v = blk_dpp<DPP_ROR + ((4 * b - P * E) & 15), 1 << b>(v, r[b]);
            });
            return v;
        }
    }
    // columns 4 quad(lane) + C of the row this lane writes in step S, row_of(lane, S) of its four
    static __device__ __forceinline__ int quad(int lane) { return R < 4 ? lane % P : lane % 4; }
    static __device__ __forceinline__ bool writes(int lane) { return quad(lane) < P; }
    static __device__ __forceinline__ int row_of(int lane, int s) { return R < 4 ? R * s + lane % 16 / P : lane % 16 / 4; }
    template <int S, int C, typename A>
    static __device__ __forceinline__ auto join(const A (&acc)[NB]) {
        if constexpr (R == 1) return acc[C][S];
        else if constexpr (R == 2) {
            if constexpr (C % 2 == 0) return blk_dpp<DPP_ROR + 8, 0xc>(acc[C / 2][2 * S], acc[C / 2][2 * S + 1]);
            else return blk_dpp<DPP_ROR + 8, 0x3>(acc[C / 2][2 * S + 1], acc[C / 2][2 * S]);
        } else {
            auto v = acc[0][C];
            blk_for<4>([&](auto bc) {
                constexpr int b = bc;
                if constexpr (b != C) v = blk_dpp<DPP_ROR + ((4 * (b - C)) & 15), 1 << b>(v, acc[0][b]);
            });
            return v;
        }
    }
    // the column of this lane's x row in load J of a block (groups R J .. R J + R - 1)
    template <int J>
    static __device__ __forceinline__ int column(int cv, int lane) {
        if constexpr (R > 4) return __shfl(cv, (lane & 48) + R * J + lane % 16 / P, 64);
        int c = blk_dpp<DPP_BCAST + (R * J & 15), 0xf>(cv, cv);
        if constexpr (R == 2) c = blk_dpp<DPP_BCAST + (2 * J + 1 & 15), 0xc>(c, cv);
        if constexpr (R == 4) {
            c = blk_dpp<DPP_BCAST + (4 * J + 1 & 15), 0x2>(c, cv);
            c = blk_dpp<DPP_BCAST + (4 * J + 2 & 15), 0x4>(c, cv);
            c = blk_dpp<DPP_BCAST + (4 * J + 3 & 15), 0x8>(c, cv);
        }
        return c;
    }
};

// The tile's product into acc.  The tile's values go through LDS (`stage`, this
// wave's BLK_MAX_ENTRIES): they come in with 16-byte loads, and each lane picks
// the one below its mask bit.  BLK_LOADS x loads are in flight together.
template <typename T, int P, typename A4>
__device__ __forceinline__ void blk_tile(int t, int lane, const BlkOps& m, const T* __restrict__ val,
                                         const float* __restrict__ x, T* stages, int wave, A4 (&acc)[BlkCols<P>::NB]) {
    typedef BlkCols<P> Cols;
    constexpr int R = Cols::R, NB = Cols::NB, V = 16 / (int)sizeof(T), SL = BLK_MAX_ENTRIES / (64 * V);
    constexpr int L = BLK_LOADS < 16 / R ? BLK_LOADS : 16 / R;  // loads together, L R groups
    typedef T VT __attribute__((ext_vector_type(V), aligned(sizeof(T))));
    typedef T VTA __attribute__((ext_vector_type(V)));
    int g = m.gptr[t], g1 = m.gptr[t + 1];
    int base = m.vptr[t], cnt = m.vptr[t + 1] - base;
    const int* cb = m.col + 64ll * m.bptr[t];
    T* stage = stages + wave * BLK_STAGE;  // 16-byte aligned
    VT sv[SL];
#pragma unroll
    for (int q = 0; q < SL; q++)
        if ((q * 64 + lane) * V < cnt) sv[q] = *(const VT*)(val + base + (q * 64 + lane) * V);
    // columns as byte offsets of their x rows (n k < 2^30: the launcher's check)
    unsigned cv = g < g1 ? (unsigned)cb[lane] * (Cols::K * 4u) : 0u;
#pragma unroll
    for (int q = 0; q < SL; q++)
        if ((q * 64 + lane) * V < cnt) *(VTA*)(stage + (q * 64 + lane) * V) = sv[q];
    blk_sync();
    unsigned lo16 = 16u * (unsigned)(lane % P);
    unsigned o = (unsigned)(wave * BLK_STAGE);  // the group's first value
    // the loads H .. H + L - 1 of a block; ALL: every group is the tile's
    auto chunk = [&](auto hc, auto all, unsigned& next) {
        constexpr int h = hc;
        constexpr bool ALL = all;
        auto on = [&](int u) { return ALL || g + (h + u) * R < g1; };  // uniform
        blk_f4 xv[L];
        u64 mk[L * R];
        blk_for<L * R>([&](auto uc) {
            constexpr int u = uc;
            mk[u] = m.mask[g + h * R + u];  // (padded past the last tile's)
        });
        blk_for<L>([&](auto uc) {
            constexpr int u = uc;
            if (on(u)) xv[u] = *(const blk_f4*)((const char*)x + (unsigned)((unsigned)Cols::template column<h + u>((int)cv, lane) + lo16));
        });
        if constexpr (ALL && h == 0) next = (unsigned)cb[64 + lane] * (Cols::K * 4u);  // the next block's columns (padded past the last)
        __builtin_amdgcn_sched_barrier(0);  // every load issued before the first is waited for
        blk_for<L>([&](auto uc) {
            constexpr int u = uc;
            if (on(u)) {
                blk_for<R>([&](auto ec) {
                    constexpr int e = ec;
                    u64 mm = ALL || g + (h + u) * R + e < g1 ? mk[u * R + e] : 0;
                    // past the last entry: the element behind the tile's values
                    T a = stages[__builtin_amdgcn_mbcnt_hi((unsigned)(mm >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)mm, o))];
                    a = __builtin_amdgcn_inverse_ballot_w64(mm) ? a : (T)0;
                    o += (unsigned)__popcll(mm);
                    blk_for<NB>([&](auto bc) {
                        constexpr int b = bc;
                        acc[b] = blk_mfma(a, (T)Cols::template split<e, b>(xv[u]), acc[b]);
                    });
                });
            }
        });
    };
    for (; g + 16 <= g1; g += 16, cb += 64) {
        unsigned next = 0;
        blk_for<16 / (L * R)>([&](auto hc) { chunk(std::integral_constant<int, hc * L>{}, std::true_type{}, next); });
        cv = next;
    }
    blk_for<16 / (L * R)>([&](auto hc) {
        unsigned next;
        if (g + hc * (L * R) < g1) chunk(std::integral_constant<int, hc * L>{}, std::false_type{}, next);
    });
}

// y = A x (AX), b - A x (RES; b in FP32 or, rounded as it is read, FP64) or the
// Jacobi sweep on 4 P interleaved FP32 columns; four tiles per workgroup, the
// workgroups dealt to the XCDs in super-blocks of BLK_ORDER.
template <int P, SpOp OP>
__global__ __launch_bounds__(WG) void k_blk_f32(int nt, BlkOps m, const float* __restrict__ val,
                                                const float* __restrict__ x, float* __restrict__ y,
                                                const float* __restrict__ b, const double* __restrict__ b64,
                                                const float* __restrict__ D, const int* __restrict__ stop) {
    if (stop && *stop) return;
    typedef BlkCols<P> Cols;
    __shared__ __attribute__((aligned(16))) float stage[WG / 64 * BLK_STAGE];
    int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
    int t = __builtin_amdgcn_readfirstlane(xcd_order(blockIdx.x, gridDim.x, BLK_ORDER) * (WG / 64) + wave);
    if (t >= nt) return;
    blk_f4 acc[Cols::NB];
#pragma unroll
    for (int q = 0; q < Cols::NB; q++) acc[q] = (blk_f4)0.f;
    blk_tile<float, P>(t, lane, m, val, x, stage, wave, acc);
    blk_for<Cols::STEPS>([&](auto sc) {
        constexpr int st = sc;
        blk_f4 s;
        blk_for<4>([&](auto cc) {
            constexpr int c = cc;
            s[c] = Cols::template join<st, c>(acc);
        });
        int i = t * BT + 4 * (lane / 16) + Cols::row_of(lane, st);
        if (i < m.n && Cols::writes(lane)) {
            int r = m.rows[i];
            size_t o = (size_t)r * Cols::K + 4 * Cols::quad(lane);
            if (OP == SpOp::RES) {
                blk_f4 bv = b64 ? __builtin_convertvector(*(const blk_d4*)(b64 + o), blk_f4) : *(const blk_f4*)(b + o);
                s = bv - s;
            } else if (OP == SpOp::JACOBI) {
                s = ((-s + *(const blk_f4*)(b + o)) / D[r]) + *(const blk_f4*)(x + o);
            }
            *(blk_f4*)(y + o) = s;
        }
    });
}

// FCG's fused product: w = A z, z in FP32 widened exactly, FP64 sums, with the
// three dot products (r.z, w.z, wold.z) per column, reduced per workgroup in a
// fixed order into partials[(block * k + column) * 3 + m].  A fixed persistent
// grid: each XCD's workgroups walk its share of the rows (k_spmmp's two orders).
template <int P>
__global__ __launch_bounds__(WG, P == 16 ? 3 : 5) void k_blk_dots(int nt, BlkOps m, const double* __restrict__ val,
                                                                 const float* __restrict__ z, double* __restrict__ w,
                                                                 const double* __restrict__ r,
                                                                 const double* __restrict__ wold,
                                                                 double* __restrict__ partials,
                                                                 const int* __restrict__ stop) {
    if (stop && *stop) return;
    typedef BlkCols<P> Cols;
    constexpr int W = WG / 64, X = 8, K = Cols::K;
    // the values of each wave's tile; at the end the partial sums
    __shared__ __attribute__((aligned(32))) double stage[W * BLK_STAGE];
    static_assert(4 * WG <= W * BLK_STAGE, "one dot product's sums fit");
    int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
    int xcd = blockIdx.x % X, local = blockIdx.x / X, nloc = gridDim.x / X;
    int ngroups = (nt + W - 1) / W;
    blk_d4 da = (blk_d4)0.0, db = (blk_d4)0.0, dc = (blk_d4)0.0;
    for (int q = local;; q += nloc) {
        long long grp = ((long long)(q / BLK_ORDER) * X + xcd) * BLK_ORDER + q % BLK_ORDER;
        if (grp >= ngroups) break;
        int t = __builtin_amdgcn_readfirstlane((int)grp * W + wave);
        if (t >= nt) continue;
        blk_d4 acc[Cols::NB];
#pragma unroll
        for (int b = 0; b < Cols::NB; b++) acc[b] = (blk_d4)0.0;
        blk_sync();  // the last tile's values are read
        blk_tile<double, P>(t, lane, m, val, z, stage, wave, acc);
        blk_for<Cols::STEPS>([&](auto sc) {
            constexpr int st = sc;
            blk_d4 s;
            blk_for<4>([&](auto cc) {
                constexpr int c = cc;
                s[c] = Cols::template join<st, c>(acc);
            });
            int i = t * BT + 4 * Cols::row_of(lane, st) + lane / 16;
            if (i < m.n && Cols::writes(lane)) {
                int rr = m.rows[i];
                size_t o = (size_t)rr * K + 4 * Cols::quad(lane);
                blk_d4 zw = __builtin_convertvector(*(const blk_f4*)(z + o), blk_d4);
                *(blk_d4*)(w + o) = s;
                da += *(const blk_d4*)(r + o) * zw;
                db += s * zw;
                dc += *(const blk_d4*)(wold + o) * zw;
            }
        });
    }
    // lanes S apart hold the same columns; one dot product at a time through LDS
    constexpr int S = P < 4 ? 4 : P;
    double* red = stage;
    blk_for<3>([&](auto mc) {
        constexpr int mm = mc;
        blk_d4 v = mm == 0 ? da : mm == 1 ? db : dc;
        __syncthreads();
        *(blk_d4*)(red + 4 * threadIdx.x) = v;
        __syncthreads();
        for (int st = WG / 2; st >= S; st >>= 1) {
            if ((int)threadIdx.x < st) *(blk_d4*)(red + 4 * threadIdx.x) += *(const blk_d4*)(red + 4 * (threadIdx.x + st));
            __syncthreads();
        }
        if (threadIdx.x < K) partials[((long long)blockIdx.x * K + threadIdx.x) * 3 + mm] = red[threadIdx.x];
    });
}

static BlkOps ops_of(const SpmvArgs& a) {
    return {a.blk->gptr.get(), a.blk->bptr.get(), a.blk->col.get(), a.blk->mask.get(), a.blk->vptr.get(), a.blk->rows.get(), a.n};
}


static bool blk_applies(const SpmvArgs& a) {
    return a.blk && a.blk->built() && a.kchunk == BLK_CODE && blk_width(a.k) && (long long)a.blk->m * a.k < (1ll << 30);
}

#define BCMGX_BLK(K, CALL)              \
    switch (K) {                        \
    case 8: { CALL(2); break; }         \
    case 16: { CALL(4); break; }        \
    case 32: { CALL(8); break; }        \
    default: { CALL(16); break; }       \
    }

bool spmm_blocked_f32(Context* c, SpOp op, const SpmvArgs& a) {
    if (!blk_applies(a) || !a.blk->val32 || a.y64 || a.x0 || op == SpOp::AXPBY || a.alpha != 1.0) return false;
    int nt = (a.n + BT - 1) / BT;
    unsigned grid = grid_for(nt, WG / 64);
#define BCMGX_B(P, OP)                                                                                                \
    k_blk_f32<P, OP><<<grid, WG, 0, c->stream>>>(nt, ops_of(a), a.blk->val32.get(), (const float*)a.x, (float*)a.y, \
                                                 (const float*)a.b, a.b64, (const float*)a.D, a.stop)
#define BCMGX_AX(P) BCMGX_B(P, SpOp::AX)
#define BCMGX_RES(P) BCMGX_B(P, SpOp::RES)
#define BCMGX_JAC(P) BCMGX_B(P, SpOp::JACOBI)
    if (op == SpOp::AX) BCMGX_BLK(a.k, BCMGX_AX)
    else if (op == SpOp::RES) BCMGX_BLK(a.k, BCMGX_RES)
    else BCMGX_BLK(a.k, BCMGX_JAC)
#undef BCMGX_AX
#undef BCMGX_RES
#undef BCMGX_JAC
#undef BCMGX_B
    BCMGX_LAUNCHED();
    return true;
}

template <int P>
static int dots_grid(Context* c) {
    int per_cu = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_blk_dots<P>, WG, 0) != hipSuccess || per_cu < 1) per_cu = 1;
    return std::max(8, c->num_cus * per_cu / 8 * 8);
}
int spmm_blocked_dots_blocks(Context* c, int k) {
    if (!blk_width(k)) return 0;
    int g = 0;
#define BCMGX_G(P) g = dots_grid<P>(c)
    BCMGX_BLK(k, BCMGX_G)
#undef BCMGX_G
    return g;
}

bool spmm_blocked_dots(Context* c, const SpmvArgs& a, const double* r, const double* wold, double* partials, int nblk,
                       const int* all_done) {
    if (!blk_applies(a) || !a.blk->val64 || nblk <= 0 || nblk % 8) return false;
    int nt = (a.n + BT - 1) / BT;
#define BCMGX_D(P)                                                                                                       \
    k_blk_dots<P><<<nblk, WG, 0, c->stream>>>(nt, ops_of(a), a.blk->val64.get(), (const float*)a.x, (double*)a.y, r, wold, \
                                              partials, all_done)
    BCMGX_BLK(a.k, BCMGX_D)
#undef BCMGX_D
    BCMGX_LAUNCHED();
    return true;
}
#undef BCMGX_BLK

}  // namespace bcmgx
