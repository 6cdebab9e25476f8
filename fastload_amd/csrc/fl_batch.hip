// Multi-right-hand-side SpMM (ROW schedule), block-diagonal batching of many matrices, zero
// fill and hipGraph capture. No reference counterpart: the reference multiplies one matrix by
// one vector per call (src/FastLoad_GPU.h:275-409).
//
// ROW: Y (m x k, row-major) = A * X (n x k, row-major, original column order). With k >= 8 a
// FastLoad-style column sweep would need k scattered y updates per non-zero (global atomics run
// at ~20 G cache lines/s on MI355X); instead the entries are re-ordered by row once, a row is
// owned by k lanes, X rows are gathered whole (k*4 bytes, a full 128-byte line at k = 32) and
// each Y row is written once, without atomics.
#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <type_traits>
#include <vector>

#include "fl_matrix.h"

namespace fl {

static unsigned sgb(long long count) { return std::max(1u, std::min<unsigned>(grid_for(count), 65536u)); }

#define GSTRIDE(i, count) \
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < (count); i += (long long)gridDim.x * blockDim.x)

// length of every original column
__global__ void k_col_lengths(const int *__restrict__ perm, const int *__restrict__ sortnnz, int n, int *__restrict__ len) {
    GSTRIDE(i, n) len[perm[i]] = sortnnz[i];
}

__global__ void k_rows_fill(const int *__restrict__ order, const ColEntry *__restrict__ ents, int *__restrict__ rcol,
                            double *__restrict__ rv64, float *__restrict__ rv32, int count) {
    GSTRIDE(i, count) {
        const ColEntry e = ents[order[i]];
        rcol[i] = e.col;
        rv64[i] = e.val;
        rv32[i] = (float)e.val;
    }
}

// The row arrays end with kRowPad entries that belong to no row: the row kernels load entries up to four at a time.
constexpr int kRowPad = 4;

void row_prepare(fl_matrix *A, hipStream_t s) {
    if (A->row_ready) return;
    const int nnz = A->nnz, m = A->m, n = A->n;
    A->row_ptr.alloc((size_t)m + 1);
    A->row_col.alloc((size_t)nnz + kRowPad);
    A->row_val32.alloc((size_t)nnz + kRowPad);
    A->row_val64.alloc((size_t)nnz + kRowPad);
    if (nnz == 0) {
        FL_HIP(hipMemsetAsync(A->row_ptr.p, 0, sizeof(int) * ((size_t)m + 1), s));
        A->row_ready = true;
        return;
    }
    // (row, original column) order: the entries in original column order (columns_from_tiles), then stable by
    // row. The order inside a row then depends only on A, not on the column sort, so a block of a batch
    // sums exactly as the same matrix alone.
    TmpBuf<int> len(n, s), colptr((size_t)n + 1, s), order(nnz, s);
    TmpBuf<uint32_t> key(nnz, s);
    TmpBuf<ColEntry> ents(nnz, s);
    k_col_lengths<<<sgb(n), kBlock, 0, s>>>(A->perm.p, A->sortnnz.p, n, len.p);
    FL_LAUNCH_CHECK();
    exclusive_scan_i32(len.p, colptr.p, n, s);
    columns_from_tiles(A, 0, colptr.p, 0, A->perm.p, key.p, ents.p, s);
    radix_sort_positions(key.p, key.p, order.p, nnz, bits_for((uint32_t)std::max(m - 1, 0)), s);
    k_rows_fill<<<sgb(nnz), kBlock, 0, s>>>(order.p, ents.p, A->row_col.p, A->row_val64.p, A->row_val32.p, nnz);
    FL_LAUNCH_CHECK();
    key_bounds(key.p, nnz, m, A->row_ptr.p, s);
    HostInts longest(s);
    max_step_begin(A->row_ptr.p, m, longest, s);
    (void)longest.wait();
    A->row_longest = max_i32_end(longest);
    A->row_ready = true;
}

__global__ void k_row_val32(const double *__restrict__ v64, float *__restrict__ v32, int count) {
    GSTRIDE(i, count) v32[i] = (float)v64[i];
}

// The row order read back from a file: row_ptr [m+1] must be a pointer array over nnz and every
// column inside [0, n) before the kernels may index with them.
int row_install(fl_matrix *A, const int *row_ptr, const int *row_col, const double *row_val, hipStream_t s) {
    const int m = A->m, n = A->n, nnz = A->nnz;
    bool ok = row_ptr[0] == 0 && row_ptr[m] == nnz;
    int longest = 0;
    for (int r = 0; ok && r < m; ++r) {
        ok = row_ptr[r] <= row_ptr[r + 1];
        longest = std::max(longest, row_ptr[r + 1] - row_ptr[r]);
    }
    for (long long i = 0; ok && i < nnz; ++i) ok = row_col[i] >= 0 && row_col[i] < n;
    if (!ok) {
        set_error("fl_matrix_load: row order invalid (row pointers or columns out of range)");
        return FL_ERR_INVALID;
    }
    A->row_ptr.alloc((size_t)m + 1);
    A->row_col.alloc((size_t)nnz + kRowPad);
    A->row_val64.alloc((size_t)nnz + kRowPad);
    A->row_val32.alloc((size_t)nnz + kRowPad);
    FL_HIP(hipMemcpyAsync(A->row_ptr.p, row_ptr, sizeof(int) * ((size_t)m + 1), hipMemcpyHostToDevice, s));
    if (nnz) {
        FL_HIP(hipMemcpyAsync(A->row_col.p, row_col, sizeof(int) * (size_t)nnz, hipMemcpyHostToDevice, s));
        FL_HIP(hipMemcpyAsync(A->row_val64.p, row_val, sizeof(double) * (size_t)nnz, hipMemcpyHostToDevice, s));
        k_row_val32<<<sgb(nnz), kBlock, 0, s>>>(A->row_val64.p, A->row_val32.p, nnz);
        FL_LAUNCH_CHECK();
    }
    A->row_longest = longest;
    A->row_ready = true;
    return FL_OK;
}

// Vector of VEC consecutive T (VEC = 1, 2 or 4), loaded and stored as one access.
template <typename T, int VEC>
struct RowVec;
template <> struct RowVec<float, 1> { using type = float; };
template <> struct RowVec<float, 2> { using type = float2; };
template <> struct RowVec<float, 4> { using type = float4; };
template <> struct RowVec<double, 1> { using type = double; };
template <> struct RowVec<double, 2> { using type = double2; };

// The value of lane U0 of each group of L consecutive lanes, in all lanes of the group (which must
// all be active). DPP moves for up to 16 lanes: quad permutes, and row broadcasts (for 8 lanes
// one per half row, selected by the bank mask).
template <int L, int U0>
__device__ __forceinline__ uint32_t bcast_u32(uint32_t v) {
    if constexpr (L == 1) return v;
    else if constexpr (L == 2) return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, U0 | (U0 << 2) | ((2 + U0) << 4) | ((2 + U0) << 6), 0xf, 0xf, true);
    else if constexpr (L == 4) return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, U0 * 0x55, 0xf, 0xf, true);
    else if constexpr (L == 16) return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x150 + U0, 0xf, 0xf, true);
    else if constexpr (L == 8) {
        const int lo = __builtin_amdgcn_update_dpp(0, (int)v, 0x150 + U0, 0xf, 0x3, false);
        return (uint32_t)__builtin_amdgcn_update_dpp(lo, (int)v, 0x150 + 8 + U0, 0xf, 0xc, false);
    } else return (uint32_t)__builtin_amdgcn_ds_bpermute((int)(((__lane_id() & ~(uint32_t)(L - 1)) + U0) * 4), (int)v);
}
template <int L, int U0>
__device__ __forceinline__ float bcast(float v) { return __uint_as_float(bcast_u32<L, U0>(__float_as_uint(v))); }
template <int L, int U0>
__device__ __forceinline__ double bcast(double v) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    const uint32_t lo = bcast_u32<L, U0>((uint32_t)b), hi = bcast_u32<L, U0>((uint32_t)(b >> 32));
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
template <int I, int N, typename F>
__device__ __forceinline__ void static_for(F &&f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<I + 1, N>(f);
    }
}

// L = K / VEC lanes own one row (64 / L rows per wave, one group of rows per wave); lane j
// accumulates columns [j*VEC, j*VEC + VEC) of the row's Y block, gathering them from X as one
// VEC-wide load per entry. Every Y element sums its row's entries in entry order whatever VEC is.
//
// Bound by the vector memory path: every distinct line an instruction touches takes a turn in
// the L1, and a gather touches one per row. So the entries are not loaded once per row and entry
// (which cost as many turns as the X rows themselves): each lane of a row loads Q consecutive ones of the
// next L * Q entries, up to four with a load (at the alignment of an entry), and the lanes hand them to each
// other with DPP moves while the next step's are in flight. Every L-th entry per lane instead, Q loads that touch
// the same lines while the first is still on its way, fetches each line once per load (us; consecutive
// entries / every L-th / all loaded by every lane of the row as they are used): k = 2 in FP32, 100 K uniform rows of 32
// 19.0 / 28.3 / 23.2, 50^3 grid 7.1 / 11.8 / 10.7; k = 8 in FP64, 40^3 grid 9.4 / 10.9 / 9.9.
// X rows come in groups of U, unconditionally: past the row's end the lanes read X row 0
// (one line for all of them) and drop it, since a branch around the loads would drain them.
// Consecutive groups run on one XCD in chunks of kRowChunk rows, dealt round-robin: rows with local
// columns (bands, grids, block-diagonal batches) share X lines in that XCD's L2, and no XCD gets
// all of the large blocks of a batch. One group per wave: waves that loop over several groups
// end unevenly (grid of 64^3, k = 16 in FP64: 58 us with one group, 78 with eight).
// HUB: for matrices whose longest row takes longer than all others (hub_rows), where one wave's chain of loads and
// instructions is the time: 16 X rows in flight, the next step's entries loaded after them (loads come back in order,
// so loaded before them they would delay every use of X), and no test per entry in whole steps. FP32, 400 K rows of
// Zipf(2) length up to 50,000, k = 2, 8, 32: 1.05, 1.23, 1.90 ms, without 2.32, 4.60, 6.29, and with four entries ahead
// loaded by every lane of the row 2.30, 3.91, 4.28. It takes 64 to 124 registers instead of 26 to 84, which costs where
// rows are of one length: uniform rows of 32, k = 8 in FP64 28 and 40 us.
// Y rows of at least a line are stored with the streaming hint: they are written whole and leave the L2
// to X (k = 32: 287 -> 274 us).
// Measured, before (one entry load per row, four entries ahead, contiguous row ranges) -> after, still with every
// L-th entry per lane: 128 stacked Zipf(2) matrices (5.2 M rows, 37 M entries) k = 8: 398 -> 291 us; 64 of them, k = 32:
// 395 -> 273 us; 64^3 27-point grid, k = 16 in FP64: 79 -> 58 us. With every gather
// sent to 64 lines of X the k = 8 product takes 238 us, without gathers 121 us. Measured and not
// kept: the columns that recur in a block of rows staged in LDS (k = 8: 290 us, k = 32: 332 us and
// more, grid: 104 us and more: the entry loop grows by the choice of source and LDS costs waves);
// rows ordered by length in windows of 256 (k = 8: 409 us: entries of a wave's rows no longer share
// lines).
constexpr int kRowChunk = 1024;
template <typename T, typename ACC, int K, int VEC, bool HUB>
__global__ __launch_bounds__(kBlock) void k_spmm_row(int m, int chunk, const int *__restrict__ row_ptr,
                                                     const int *__restrict__ row_col, const T *__restrict__ row_val,
                                                     const T *__restrict__ X, T *__restrict__ Y, int accumulate) {
    using V = typename RowVec<T, VEC>::type;
    constexpr int L = K / VEC, RPW = 64 / L;  // lanes per row, rows per wave
    constexpr int Q = L < 16 ? 16 / L : 1;    // entries per lane of a step
    constexpr int U = HUB ? 16 : 4;           // X rows in flight together
    constexpr bool kStreamY = K * sizeof(T) >= 128;
    const int idx = blockIdx.x >> 3;
    const long long wg = (long long)(idx / chunk * 8 + (int)(blockIdx.x & 7)) * chunk + idx % chunk;
    const int lane = threadIdx.x & 63, sub = lane / L, j = lane % L;
    const long long r = (wg * (kBlock / 64) + (threadIdx.x >> 6)) * RPW + sub;
    if (r >= m) return;
    const V *__restrict__ Xv = reinterpret_cast<const V *>(X);
    const int e0 = row_ptr[r];
    const int *__restrict__ pc = row_col + e0 + j * Q;
    const T *__restrict__ pv = row_val + e0 + j * Q;
    ACC acc[VEC];
#pragma unroll
    for (int q = 0; q < VEC; ++q) acc[q] = 0;
    int c[Q], nc[Q];
    T v[Q], nv[Q];
    auto fetch = [&](int left, int *cc, T *vv) {  // the next entries of the row, `left` of them to come
        constexpr int G = Q < 4 ? Q : 4;           // per load: at most G - 1 < kRowPad past the row's end
#pragma unroll
        for (int q = 0; q < Q; q += G) {
#pragma unroll
            for (int g = 0; g < G; ++g) {
                cc[q + g] = 0;
                vv[q + g] = T(0);
            }
            if (j * Q + q < left) {
                __builtin_memcpy(cc + q, pc + q, sizeof(int) * G);
                __builtin_memcpy(vv + q, pv + q, sizeof(T) * G);
            }
        }
        pc += L * Q;
        pv += L * Q;
    };
    int left = row_ptr[r + 1] - e0;
    fetch(left, c, v);
    auto step = [&](auto whole) {  // whole: the row has all L * Q entries of the step
        constexpr bool W = decltype(whole)::value;
        if constexpr (!HUB) fetch(left - L * Q, nc, nv);
        static_for<0, L * Q / U>([&](auto h) {
            constexpr int H = decltype(h)::value * U;
            if (W || H < left) {
                V x[U];
                static_for<0, U>([&](auto u) {
                    constexpr int k = H + decltype(u)::value;
                    x[u] = Xv[(long long)bcast_u32<L, k / Q>((uint32_t)c[k % Q]) * L + j];
                });
                if constexpr (HUB && H == L * Q - U) fetch(left - L * Q, nc, nv);
                static_for<0, U>([&](auto u) {
                    constexpr int k = H + decltype(u)::value;
                    const T a = bcast<L, k / Q>(v[k % Q]);
                    if (W || k < left) {
                        const T *xs = reinterpret_cast<const T *>(&x[u]);
#pragma unroll
                        for (int q = 0; q < VEC; ++q) acc[q] += (ACC)a * (ACC)xs[q];
                    }
                });
            }
        });
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            c[q] = nc[q];
            v[q] = nv[q];
        }
        left -= L * Q;
    };
    if constexpr (HUB) {
        while (left >= L * Q) step(std::true_type{});
    }
    while (left > 0) {
#pragma unroll
        for (int q = 0; q < Q; ++q) c[q] = j * Q + q < left ? c[q] : 0;
        step(std::false_type{});
    }
    V *out = reinterpret_cast<V *>(Y) + r * L + j;
    V o;
    if (accumulate) o = *out;
    T *os = reinterpret_cast<T *>(&o);
#pragma unroll
    for (int q = 0; q < VEC; ++q) os[q] = accumulate ? (T)((ACC)os[q] + acc[q]) : (T)acc[q];
    if constexpr (kStreamY) st_stream(out, o);
    else *out = o;
}

// k = 1: four lanes share a row (16 rows per wave, one group per wave); lane j adds the sums of entries
// 4j..4j+3 of every sixteen, and a butterfly adds the four lanes' sums. The order depends only on the row, so a
// block of a stacked batch equals its matrix run alone bit for bit.
// Bound by the L1's turns, one per distinct line of an instruction (see k_spmm_row): a lane's four
// entries come in one 16-byte load of columns and one or two of values (at the alignment of an
// entry), instead of four loads that each touch the lines of all 16 rows. Loads past the row's end stay
// inside the arrays (kRowPad); those entries gather the lane's first column again and are dropped.
// kRowPre: the next sixteen entries are loaded before the gathers. That pays where rows have more than
// sixteen entries (100^3 grid: 47 against 50 us) and costs where they do not, since the
// gathers then wait for loads of few rows (60 stacked Zipf(2) matrices: 85 against 75 us).
// Measured, before (four entries ahead, every fourth entry per lane) -> after: 524 K rows of diagonal
// blocks, 24 entries each, FP32: 38 -> 26 us; 100^3 27-point grid: 70 -> 47; 80^3 in FP64: 51 -> 38; 500 K
// uniform rows of 8: 26 -> 21; 1 M power-law rows: 117 -> 97; 60 stacked Zipf(2) matrices: 113 -> 75.
// Two lanes per row: 32, 63, 52 us for the first three, 8 for short rows of 6 entries (10); eight: 31, 52,
// 37 and 17 us.
// kRowHub: for matrices whose longest row takes longer than all others (hub_rows): four steps of it at a time, 16 gathers
// of a lane in flight and the next entries loaded after them. FP32, 400 K rows of Zipf(2.2) and Zipf(2) length up to
// 50,000: 177 and 351 us; plain 374 and 738, four loads of every fourth entry 347 and 703, two lanes per row 634 for the
// first. Its 100 to 144 registers (plain: 36 to 48) cost 1.4 times the time where the longest row does not decide
// (800 K rows of 3).
template <typename T>
__device__ __forceinline__ void load_quad(const T *p, T *out) {
    __builtin_memcpy(out, p, 4 * sizeof(T));
}

constexpr int kRowLanes = 4;
enum RowAhead { kRowPlain, kRowPre, kRowHub };
template <typename T, typename ACC, RowAhead MODE>
__global__ __launch_bounds__(kBlock) void k_spmv_row1(int m, int chunk, const int *__restrict__ row_ptr,
                                                      const int *__restrict__ row_col, const T *__restrict__ row_val,
                                                      const T *__restrict__ X, T *__restrict__ Y, int accumulate) {
    constexpr int RPW = 64 / kRowLanes, kStep = 4 * kRowLanes;
    const int idx = blockIdx.x >> 3;
    const long long wg = (long long)(idx / chunk * 8 + (int)(blockIdx.x & 7)) * chunk + idx % chunk;
    const int lane = threadIdx.x & 63, sub = lane / kRowLanes, j = lane % kRowLanes;
    const long long r = (wg * (kBlock / 64) + (threadIdx.x >> 6)) * RPW + sub;
    const bool live = r < m;  // all lanes reach the butterfly
    int e0 = 0, left = 0;     // entries from this lane's next one to the row's end
    if (live) {
        e0 = row_ptr[r];
        left = row_ptr[r + 1] - e0 - 4 * j;
    }
    const int *__restrict__ pc = row_col + e0 + 4 * j;
    const T *__restrict__ pv = row_val + e0 + 4 * j;
    ACC acc = 0;
    if constexpr (MODE == kRowHub) {
        constexpr int S = 4;  // of the row's steps at a time, while the lane's part of them is whole
        const auto whole = [](int l) { return l >= (S - 1) * kStep + 4; };
        const auto load = [&](int(*cc)[4], T(*vv)[4]) {
#pragma unroll
            for (int i = 0; i < S; ++i) {
                load_quad(pc + i * kStep, cc[i]);
                load_quad(pv + i * kStep, vv[i]);
            }
        };
        int c[S][4], nc[S][4];
        T v[S][4], nv[S][4], x[S][4];
        if (whole(left)) load(c, v);
        while (whole(left)) {
#pragma unroll
            for (int i = 0; i < S; ++i)
#pragma unroll
                for (int u = 0; u < 4; ++u) x[i][u] = X[c[i][u]];
            pc += S * kStep;
            pv += S * kStep;
            left -= S * kStep;
            if (whole(left)) load(nc, nv);
#pragma unroll
            for (int i = 0; i < S; ++i) {
                ACC q = 0;
#pragma unroll
                for (int u = 0; u < 4; ++u) q += (ACC)v[i][u] * (ACC)x[i][u];
                acc += q;
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    c[i][u] = nc[i][u];
                    v[i][u] = nv[i][u];
                }
            }
        }
    }
    int c[4], nc[4];
    T v[4], nv[4];
    if (left > 0) {
        load_quad(pc, c);
        load_quad(pv, v);
    }
    while (left > 0) {
        pc += kStep;
        pv += kStep;
        if (MODE == kRowPre && left > kStep) {
            load_quad(pc, nc);
            load_quad(pv, nv);
        }
        T x[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) x[u] = X[u < left ? c[u] : c[0]];
        ACC q = 0;  // four at a time: shorter chains of roundings
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (u < left) q += (ACC)v[u] * (ACC)x[u];
        acc += q;
        left -= kStep;
        if (MODE != kRowPre && left > 0) {
            load_quad(pc, nc);
            load_quad(pv, nv);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            c[u] = nc[u];
            v[u] = nv[u];
        }
    }
#pragma unroll
    for (int o = kRowLanes / 2; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
    if (live && j == 0) Y[r] = accumulate ? (T)((ACC)Y[r] + acc) : (T)acc;
}

// The same sums for short rows, two lanes per row (32 rows per wave): lane j takes the fours j and j + 2 of every
// sixteen, so each sum and their order are those of the four lanes above, bit for bit. Of rows of up to four
// entries one lane in four has work there, and a wave half as many rows.
template <typename T, typename ACC>
__global__ __launch_bounds__(kBlock) void k_spmv_row1_short(int m, int chunk, const int *__restrict__ row_ptr,
                                                            const int *__restrict__ row_col,
                                                            const T *__restrict__ row_val, const T *__restrict__ X,
                                                            T *__restrict__ Y, int accumulate) {
    constexpr int RPW = 32;
    const int idx = blockIdx.x >> 3;
    const long long wg = (long long)(idx / chunk * 8 + (int)(blockIdx.x & 7)) * chunk + idx % chunk;
    const int lane = threadIdx.x & 63, j = lane & 1;
    const long long r = (wg * (kBlock / 64) + (threadIdx.x >> 6)) * RPW + (lane >> 1);
    const bool live = r < m;  // all lanes reach the exchange
    int e0 = 0, left = 0;     // entries from this lane's next four to the row's end
    if (live) {
        e0 = row_ptr[r];
        left = row_ptr[r + 1] - e0 - 4 * j;
    }
    const int *__restrict__ pc = row_col + e0 + 4 * j;
    const T *__restrict__ pv = row_val + e0 + 4 * j;
    ACC acc[2] = {0, 0};
    auto four = [&](ACC &a) {
        int c[4];
        T v[4], x[4];
        load_quad(pc, c);
        load_quad(pv, v);
#pragma unroll
        for (int u = 0; u < 4; ++u) x[u] = X[u < left ? c[u] : c[0]];
        ACC q = 0;
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (u < left) q += (ACC)v[u] * (ACC)x[u];
        a += q;
        left -= 8;
        pc += 8;
        pv += 8;
    };
    while (left > 0) {
        four(acc[0]);
        if (left > 0) four(acc[1]);
    }
    ACC sum = acc[0] + acc[1];
    sum += __shfl_xor(sum, 1, 64);
    if (live && j == 0) Y[r] = accumulate ? (T)((ACC)Y[r] + sum) : (T)sum;
}

// A launch has fewer than 2^32 work-items, so the rows run in slices of at most 2^31 lanes each (one launch for all up to
// 2^25 rows at 64 lanes a row). launch(rows of the slice, their pointers, their Y).
template <typename T, typename F>
static void row_slices(const fl_matrix *A, int lanes, int k, T *Y, F &&launch) {
    const long long most = (1LL << 31) / lanes;
    for (long long r = 0; r < A->m; r += most) {
        launch((int)std::min<long long>(most, A->m - r), A->row_ptr.p + r, Y + r * k);
        FL_LAUNCH_CHECK();
    }
}

// Workgroups of `rows` rows each for m rows: chunks of kRowChunk rows, shorter where that would leave an
// XCD fewer than eight of them, and a grid of whole chunks for each XCD.
struct RowGrid {
    int chunk, grid;
};
static RowGrid row_grid(int m, int rows) {
    const int wgs = div_up(m, rows);
    const int chunk = std::max(1, std::min(kRowChunk / rows, wgs / 64));
    return {chunk, 8 * chunk * div_up(wgs, 8 * chunk)};
}

// Whether the longest row is more than 1 / part of the entries and far from the others' length: its chain, one step
// after another, then outlasts the rest of the matrix, spread over the chip. With k >= 2 the line lies where the
// chain of the ordinary kernel begins to show (400 K rows of 4 and one of 100 entries, a 16,000th of all, k = 8 in FP32:
// ordinary 35.7 us, HUB 26.8, every lane of a row loading its entries 32.0; one of 400, a 4,000th: 73, 30 and 59).
constexpr long long kHubPart = 24576;
static bool hub_rows(const fl_matrix *A, long long part) {
    return A->row_longest * part > A->nnz && (long long)A->row_longest * A->m > 8LL * A->nnz;
}

// Entries per row, on average, up to which rows take two lanes. Two lanes / four (every fourth entry per lane, before both), us:
// 800 K rows in diagonal blocks, FP32, 3 entries 9.0 / 12.8 (9.8), 6 12.2 / 15.2 (17.1), 9 15.4 / 17.0 (21.5), FP64 at 9
// 20.3 / 19.7 (34.3); 800 K rows of 3 uniform entries 16.1 / 17.8 (18.6), 6 28.7 / 26.5 (31.3), FP64 51.4 / 47.2 (58.3);
// 60 stacked Zipf(2) matrices, 7 entries, 64.6 / 61.1 (75.9). From 7 on four lanes are ahead of both
// on all of them but the blocks in FP32.
// A row longer than 1 / kShortPart of the entries takes four lanes all the same: two take twice as long over it (800 K rows
// of 3, one of 200 entries, a 12,000th, FP32 17.7 / 16.9, FP64 29.8 / 25.5; one of 100 15.4 / 16.9 and 25.5 / 25.4; 100 K
// rows of 4, 300 of 200 10.7 / 7.0). From kHubPart1 on it is kRowHub's (four lanes / kRowHub: one of 400, a
// 6,000th, 20.0 / 23.8; one of 1,000, a 2,400th, 29.2 / 24.0).
constexpr long long kShortRow = 6, kShortPart = 16384, kHubPart1 = 3072;
template <typename T, typename ACC>
static void launch_row_k1(const fl_matrix *A, const T *val, const T *X, T *Y, int accumulate, hipStream_t s) {
    const bool small = (long long)A->nnz <= kShortRow * A->m && !hub_rows(A, kShortPart);
    const bool pre = (long long)A->nnz > 4LL * kRowLanes * A->m;  // rows of more than one step on average
    const int lanes = small ? 2 : kRowLanes;
    auto k = small                     ? k_spmv_row1_short<T, ACC>
             : hub_rows(A, kHubPart1) ? k_spmv_row1<T, ACC, kRowHub>
             : pre                     ? k_spmv_row1<T, ACC, kRowPre>
                                       : k_spmv_row1<T, ACC, kRowPlain>;
    row_slices(A, lanes, 1, Y, [&](int m, const int *row_ptr, T *y) {
        const RowGrid g = row_grid(m, kBlock / lanes);
        k<<<g.grid, kBlock, 0, s>>>(m, g.chunk, row_ptr, A->row_col.p, val, X, y, accumulate);
    });
}

template <typename T, typename ACC, int K, int VEC>
static void launch_row_v(const fl_matrix *A, const T *val, const T *X, T *Y, int accumulate, hipStream_t s) {
    auto k = hub_rows(A, kHubPart) ? k_spmm_row<T, ACC, K, VEC, true> : k_spmm_row<T, ACC, K, VEC, false>;
    row_slices(A, K / VEC, K, Y, [&](int m, const int *row_ptr, T *y) {
        const RowGrid g = row_grid(m, kBlock * VEC / K);
        k<<<g.grid, kBlock, 0, s>>>(m, g.chunk, row_ptr, A->row_col.p, val, X, y, accumulate);
    });
}

// Widest vector that keeps at least 4 lanes per row (k >= 4), is at most 16 bytes and that X
// and Y are aligned for. With 1 or 2 lanes per row instead (16-byte loads from k = 4 on) 40 Zipf(2)
// matrices at k = 4 took 86 us against 76, 128 of them at k = 8 294 against 291.
template <typename T, typename ACC, int K>
static void launch_row(const fl_matrix *A, const T *val, const T *X, T *Y, int accumulate, hipStream_t s) {
    constexpr int VT = 16 / (int)sizeof(T);
    constexpr int VK = K / 4 > 1 ? K / 4 : 1;
    constexpr int VMAX = VT < VK ? VT : VK;
    const uintptr_t mis = reinterpret_cast<uintptr_t>(X) | reinterpret_cast<uintptr_t>(Y);
    if constexpr (VMAX >= 4) {
        if ((mis & 15) == 0) return launch_row_v<T, ACC, K, 4>(A, val, X, Y, accumulate, s);
    }
    if constexpr (VMAX >= 2) {
        if ((mis & (2 * sizeof(T) - 1)) == 0) return launch_row_v<T, ACC, K, 2>(A, val, X, Y, accumulate, s);
    }
    launch_row_v<T, ACC, K, 1>(A, val, X, Y, accumulate, s);
}

template <typename T, typename ACC>
static int dispatch_row(const fl_matrix *A, const T *val, int k, const T *X, T *Y, int acc, hipStream_t s) {
    switch (k) {
        case 1: launch_row_k1<T, ACC>(A, val, X, Y, acc, s); return FL_OK;
        case 2: launch_row<T, ACC, 2>(A, val, X, Y, acc, s); return FL_OK;
        case 4: launch_row<T, ACC, 4>(A, val, X, Y, acc, s); return FL_OK;
        case 8: launch_row<T, ACC, 8>(A, val, X, Y, acc, s); return FL_OK;
        case 16: launch_row<T, ACC, 16>(A, val, X, Y, acc, s); return FL_OK;
        case 32: launch_row<T, ACC, 32>(A, val, X, Y, acc, s); return FL_OK;
        case 64: launch_row<T, ACC, 64>(A, val, X, Y, acc, s); return FL_OK;
        default:
            set_error("fl_spmm: k must be 1, 2, 4, 8, 16, 32 or 64");
            return FL_ERR_INVALID;
    }
}

int spmm_row(const fl_matrix *A, int kind, int k, const void *X, void *Y, int accumulate, hipStream_t s) {
    if (!A->row_ready) {
        set_error("fl_spmm: row order not prepared (fl_matrix_prepare_rows)");
        return FL_ERR_INVALID;
    }
    if (A->m == 0) return FL_OK;
    if (kind == FL_VAL_F64) return dispatch_row<double, double>(A, A->row_val64.p, k, (const double *)X, (double *)Y, accumulate, s);
    if (kind == FL_VAL_F32) return dispatch_row<float, float>(A, A->row_val32.p, k, (const float *)X, (float *)Y, accumulate, s);
    set_error("fl_spmm: FL_VAL_F64 or FL_VAL_F32 only");
    return FL_ERR_INVALID;
}

// ------------------------------------------------------------------------- zero fill
// 16-byte stores, then words, then bytes, each from where the one before ends. One launch: a second one for the odd
// 4 to 12 bytes of a y took as long as the first (1.3 us and the gap before it, 45^3 FP32 rows).
__global__ void k_zero(unsigned char *__restrict__ p, long long quads, long long words, int bytes) {
    GSTRIDE(i, quads) reinterpret_cast<uint4 *>(p)[i] = make_uint4(0u, 0u, 0u, 0u);
    p += 16 * quads;
    GSTRIDE(i, words) reinterpret_cast<uint32_t *>(p)[i] = 0u;
    if (blockIdx.x == 0 && (int)threadIdx.x < bytes) p[4 * words + threadIdx.x] = 0;
}

// Zero fill with a kernel (graph-capturable; no memset node).
void zero_fill(void *d, size_t bytes, hipStream_t s) {
    if (!bytes) return;
    const long long quads = (reinterpret_cast<uintptr_t>(d) & 15) == 0 ? (long long)(bytes / 16) : 0;
    const long long words = ((long long)bytes - 16 * quads) / 4;
    k_zero<<<sgb(std::max(std::max(quads, words), 1LL)), kBlock, 0, s>>>((unsigned char *)d, quads, words,
                                                                        (int)(bytes & 3));
    FL_LAUNCH_CHECK();
}

}  // namespace fl

using namespace fl;

extern "C" {

int fl_matrix_prepare_rows(fl_matrix *A, void *stream) {
    FL_API_BEGIN
    if (!A) {
        set_error("fl_matrix_prepare_rows: NULL");
        return FL_ERR_INVALID;
    }
    row_prepare(A, (hipStream_t)stream);
    FL_HIP(hipStreamSynchronize((hipStream_t)stream));  // products may follow on any stream
    return FL_OK;
    FL_API_END
}

int fl_spmm(fl_matrix *A, int val_kind, int k, const void *d_X, void *d_Y, int accumulate, void *stream) {
    FL_API_BEGIN
    if (!A || (A->m && (!d_X || !d_Y))) {
        set_error("fl_spmm: NULL");
        return FL_ERR_INVALID;
    }
    return spmm_row(A, val_kind, k, d_X, d_Y, accumulate, (hipStream_t)stream);
    FL_API_END
}

int fl_zero_device(void *d, size_t bytes, void *stream) {
    FL_API_BEGIN
    if (bytes && !d) {
        set_error("fl_zero_device: NULL");
        return FL_ERR_INVALID;
    }
    zero_fill(d, bytes, (hipStream_t)stream);
    return FL_OK;
    FL_API_END
}

int fl_batch_assemble(int count, const int *m, const int *n, const int *const *colptr, const int *const *rowidx,
                      const double *const *val, int *M, int *N, int **colptr_out, int **rowidx_out, double **val_out,
                      int *row_off, int *col_off) {
    if (count < 0 || !m || !n || !colptr || !rowidx || !val || !M || !N || !colptr_out || !rowidx_out || !val_out ||
        !row_off || !col_off) {
        set_error("fl_batch_assemble: NULL or negative count");
        return FL_ERR_INVALID;
    }
    long long MM = 0, NN = 0, NZ = 0;
    row_off[0] = col_off[0] = 0;
    for (int i = 0; i < count; ++i) {
        if (m[i] < 0 || n[i] < 0 || !colptr[i]) {
            set_error("fl_batch_assemble: matrix %d invalid", i);
            return FL_ERR_INVALID;
        }
        // colptr[i] must be a column pointer (starts at 0, never decreases) before its last entry
        // sizes the output and its ranges are copied
        const int *cpi = colptr[i];
        bool ok = cpi[0] == 0;
        for (int c = 0; ok && c < n[i]; ++c) ok = cpi[c] <= cpi[c + 1];
        if (!ok) {
            set_error("fl_batch_assemble: matrix %d colptr is not a column pointer (colptr[0] != 0 or decreasing)", i);
            return FL_ERR_INVALID;
        }
        if (cpi[n[i]] > 0 && (!rowidx[i] || !val[i])) {
            set_error("fl_batch_assemble: matrix %d has entries but NULL rowidx/val", i);
            return FL_ERR_INVALID;
        }
        MM += m[i];
        NN += n[i];
        NZ += colptr[i][n[i]];
        if (MM > 0x7fffffffLL || NN > 0x7fffffffLL || NZ > 0x7fffffffLL) {
            set_error("fl_batch_assemble: batch exceeds int32 indexing");
            return FL_ERR_SIZE;
        }
        row_off[i + 1] = (int)MM;
        col_off[i + 1] = (int)NN;
    }
    int *cp = (int *)malloc(sizeof(int) * ((size_t)NN + 1));
    int *ri = (int *)malloc(sizeof(int) * (size_t)std::max<long long>(NZ, 1));
    double *vv = (double *)malloc(sizeof(double) * (size_t)std::max<long long>(NZ, 1));
    if (!cp || !ri || !vv) {
        free(cp); free(ri); free(vv);
        set_error("fl_batch_assemble: out of memory");
        return FL_ERR_ALLOC;
    }
    long long pos = 0;
    for (int i = 0; i < count; ++i) {
        const int ro = row_off[i], co = col_off[i];
        for (int c = 0; c < n[i]; ++c) {
            cp[co + c] = (int)pos;
            for (int e = colptr[i][c]; e < colptr[i][c + 1]; ++e, ++pos) {
                if (rowidx[i][e] < 0 || rowidx[i][e] >= m[i]) {
                    free(cp); free(ri); free(vv);
                    set_error("fl_batch_assemble: matrix %d row index out of range", i);
                    return FL_ERR_RANGE;
                }
                ri[pos] = ro + rowidx[i][e];
                vv[pos] = val[i][e];
            }
        }
    }
    cp[NN] = (int)pos;
    *M = (int)MM;
    *N = (int)NN;
    *colptr_out = cp;
    *rowidx_out = ri;
    *val_out = vv;
    return FL_OK;
}

// ---------------------------------------------------------------------------- hipGraph
int fl_graph_begin_capture(void *stream) {
    FL_API_BEGIN
    if (!stream) {
        set_error("fl_graph_begin_capture: capture needs a created stream, not the default stream");
        return FL_ERR_INVALID;
    }
    FL_HIP(hipStreamBeginCapture((hipStream_t)stream, hipStreamCaptureModeRelaxed));
    return FL_OK;
    FL_API_END
}

int fl_graph_end_capture(void *stream, void **graph_exec) {
    FL_API_BEGIN
    if (!stream || !graph_exec) {
        set_error("fl_graph_end_capture: NULL");
        return FL_ERR_INVALID;
    }
    hipGraph_t g = nullptr;
    FL_HIP(hipStreamEndCapture((hipStream_t)stream, &g));
    hipGraphExec_t ge = nullptr;
    const hipError_t e = hipGraphInstantiate(&ge, g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    FL_HIP(e);
    *graph_exec = ge;
    return FL_OK;
    FL_API_END
}

int fl_graph_launch(void *graph_exec, void *stream) {
    FL_API_BEGIN
    FL_HIP(hipGraphLaunch((hipGraphExec_t)graph_exec, (hipStream_t)stream));
    return FL_OK;
    FL_API_END
}

int fl_graph_destroy(void *graph_exec) {
    FL_API_BEGIN
    if (graph_exec) FL_HIP(hipGraphExecDestroy((hipGraphExec_t)graph_exec));
    return FL_OK;
    FL_API_END
}

}  // extern "C"
