// HYB schedule: heavy columns from LDS, the rest through propagation blocking.
//
// A power-law matrix keeps most of its entries in few columns: on the 4M-column, 67M-entry
// workload the 32768 longest columns hold 70 % of them. Their x values (128 KB in FP32) fit in one
// workgroup's LDS, so those entries can be summed row by row with x gathered from LDS: each entry
// costs its value and a 16-bit column, and y is written once per row, with no product buffer and
// no row index. The other columns keep the PB schedule (a product and a 16-bit row per entry
// moved twice through the Infinity Cache), run on a sub-matrix of their own.
//
// Layout of the heavy part (all built on the GPU by hyb_prepare):
//   - rows are ordered by heavy entry count, longest first, inside windows of hyb_win rows, the
//     sub-matrix's PB bands (hyb_iperm[r] = position of row r inside its window), so the 64 rows of
//     a slice have nearly the same count;
//   - slice s = sorted positions [64 s, 64 s + 64) is an ELL block of hyb_np[s] pair rows: slot
//     (q, lane), at hyb_sb[s] + 64 q + lane, holds entries 2q and 2q + 1 of the lane's row as a
//     value pair and one word of two 16-bit columns; rows shorter than the slice's longest are
//     padded with value 0 and column H, which reads the zero stored after x in LDS. On the
//     power-law workload the padding adds 5 % to the heavy entries. A wave reads one slot per
//     lane per pair row: 8 (16 in FP64) + 4 contiguous bytes, with no per-entry index math;
//   - the heavy kernel writes y by sorted position (hyb_ys), and the sub-matrix's first PB phase 2
//     adds it to y: a band is a window, so it reads hyb_ys in order and adds hyb_ys[p] to row
//     hyb_perm[p] of its LDS sums (a gather through hyb_iperm would move a 128-byte line per
//     4-byte value: 14 of phase 2's 42 us on the power-law workload).
// The column sort is ascending, so the heavy columns are the last H sorted columns: heavy x is
// sortx + (n - H), and the sub-matrix's sorted columns are the first n - H sorted columns in the
// same order (its own column sort of already ascending counts is the identity, so it is not run),
// so the sub-matrix reads sortx directly.
#include <algorithm>

#include "fl_matrix.h"

namespace fl {

void pb_prepare(fl_matrix *A, int bt, int R, hipStream_t s);
void prepare_values(fl_matrix *A, int kind, hipStream_t s);
void zero_fill(void *d, size_t bytes, hipStream_t s);

#define HSTRIDE(i, count) \
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < (count); i += (long long)gridDim.x * blockDim.x)

// pair rows per load group of the heavy kernel (two groups in flight per wave)
constexpr int kHybPairs = 2;

static unsigned hg(long long threads) { return std::max(1u, std::min<unsigned>(grid_for(threads), 65536u)); }

// ------------------------------------------------------------------------ preparation
__global__ void k_hyb_iota(int *__restrict__ v, int count) {
    HSTRIDE(i, count) v[i] = (int)i;
}

// Rows by (window, heavy count descending, row), and the pair rows of every slice (half its first, longest
// row, rounded up). One workgroup per window: a stable radix sort of the counts in LDS, 8 bits at a time, the
// second pass only where a row has 256 heavy entries or more. Each wave ranks a contiguous part of the rows, as in
// the radix sort of the whole device; one sort of all rows there, by count and then by window, was
// 17 launches and 75 us for 600 K rows, this is one of 9 us.
constexpr int kOrderThreads = 1024, kOrderWaves = kOrderThreads / 64;
constexpr int kOrderRounds = 16;  // of 64 rows per wave: windows of up to 16,384 rows
__global__ __launch_bounds__(kOrderThreads) void k_hyb_order(const int *__restrict__ hptr, int m, int win, int rounds,
                                                             int *__restrict__ rows, uint16_t *__restrict__ iperm,
                                                             uint16_t *__restrict__ perm, int *__restrict__ np,
                                                             int *__restrict__ pairs) {
    extern __shared__ double order_lds[];
    const int cap = rounds * kOrderThreads;
    uint16_t *ka = reinterpret_cast<uint16_t *>(order_lds), *ia = ka + cap, *kb = ia + cap, *ib = kb + cap;
    int(*wcnt)[256] = reinterpret_cast<int(*)[256]>(ib + cap);  // a wave's rows per digit, then where they go
    __shared__ int wsum[4];
    const int base = (int)blockIdx.x * win, n = min(win, m - base);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int big = 0;
    for (int i = threadIdx.x; i < n; i += kOrderThreads) {
        const int c = hptr[base + i + 1] - hptr[base + i];
        big |= c >= 256;
        ka[i] = (uint16_t)(65535 - c);
        ia[i] = (uint16_t)i;
    }
    const int passes = __syncthreads_or(big) ? 2 : 1;
    const uint64_t lt_mask = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    for (int p = 0; p < passes; ++p) {
        const int shift = 8 * p;
        for (int i = threadIdx.x; i < kOrderWaves * 256; i += kOrderThreads) wcnt[i >> 8][i & 255] = 0;
        __syncthreads();
        int at[kOrderRounds];  // rank among the wave's rows of the same digit
#pragma unroll
        for (int r = 0; r < kOrderRounds; ++r) {
            if (r >= rounds) break;
            const int i = (w * rounds + r) * 64 + lane;
            const bool valid = i < n;
            const int d = valid ? (ka[i] >> shift) & 255 : 0;
            uint64_t peers = ballot64(valid);
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const bool bit = (d >> k) & 1;
                const uint64_t b = ballot64(bit);
                peers &= bit ? b : ~b;
            }
            const int rank = __popcll(peers & lt_mask);
            int o = 0;
            if (valid && rank == 0) o = atomicAdd(&wcnt[w][d], __popcll(peers));
            at[r] = __shfl(o, valid ? __ffsll((unsigned long long)peers) - 1 : lane, 64) + rank;
        }
        __syncthreads();
        // where each wave's rows of a digit start
        int sum = 0, v = 0;
        if (w < 4) {
            for (int q = 0; q < kOrderWaves; ++q) sum += wcnt[q][threadIdx.x];
            v = wave_inclusive_scan(sum);
            if (lane == 63) wsum[w] = v;
        }
        __syncthreads();
        if (w < 4) {
            int before = v - sum;
            for (int q = 0; q < w; ++q) before += wsum[q];
            for (int q = 0; q < kOrderWaves; ++q) {
                const int t = wcnt[q][threadIdx.x];
                wcnt[q][threadIdx.x] = before;
                before += t;
            }
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kOrderRounds; ++r) {
            if (r >= rounds) break;
            const int i = (w * rounds + r) * 64 + lane;
            if (i < n) {
                const int pos = wcnt[w][(ka[i] >> shift) & 255] + at[r];
                kb[pos] = ka[i];
                ib[pos] = ia[i];
            }
        }
        __syncthreads();
        uint16_t *t = ka;
        ka = kb, kb = t;
        t = ia, ia = ib, ib = t;
    }
    for (int p = threadIdx.x; p < n; p += kOrderThreads) {
        const int r = ia[p];
        rows[base + p] = base + r;
        perm[base + p] = (uint16_t)r;
        iperm[base + r] = (uint16_t)p;
        if ((p & 63) == 0) {
            const int q = (65535 - ka[p] + 1) / 2;
            np[(base + p) / 64] = q;
            pairs[(base + p) / 64] = q;
        }
    }
}

// One lane per sorted position writes its row's slots: the heavy entries in column order, then
// the padding (value 0, column H) up to the slice's pair rows (all padding past the last row). Bound by the
// gathers of the entries, one line each; two pair rows at a time keep four in flight per lane.
__global__ void k_hyb_fill(int m, int nslice, int H, const int *__restrict__ rows, const int *__restrict__ np,
                           const long long *__restrict__ sb, const int *__restrict__ hptr, const int *__restrict__ ridx,
                           const ColEntry *__restrict__ ents, uint32_t *__restrict__ col2, double2 *__restrict__ val2,
                           float2 *__restrict__ val2f) {
    // one position per thread; consecutive workgroups of an XCD take consecutive slices, so the lines of the
    // entries that a sorting window's rows share are fetched once (7.4 M heavy entries: 195 us with the slices dealt round-robin, 148 so; the three
    // dependent reads per entry before that took 545)
    const long long p = ((long long)(blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3)) * kBlock + threadIdx.x;
    if (p < (long long)nslice * 64) {
        const long long s = p >> 6;
        const int lane = (int)(p & 63);
        int base = 0, L = 0;
        if (p < m) {
            const int r = rows[p];
            base = hptr[r];
            L = hptr[r + 1] - base;
        }
        const int P = np[s];
        for (int q = 0; q < P; q += 2) {
            int at[4];
            ColEntry e[4];
#pragma unroll
            for (int h = 0; h < 4; ++h) at[h] = 2 * q + h < L ? ridx[base + 2 * q + h] : -1;
#pragma unroll
            for (int h = 0; h < 4; ++h) {
                e[h] = ColEntry{0.0, H, 0};
                if (at[h] >= 0) e[h] = ents[at[h]];
            }
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                if (q + h >= P) break;
                const long long slot = sb[s] + 64LL * (q + h) + lane;
                col2[slot] = (uint32_t)e[2 * h].col | ((uint32_t)e[2 * h + 1].col << 16);
                val2[slot] = make_double2(e[2 * h].val, e[2 * h + 1].val);
                if (val2f) val2f[slot] = make_float2((float)e[2 * h].val, (float)e[2 * h + 1].val);
            }
        }
    }
}

__global__ void k_hyb_fill_u32(uint32_t *__restrict__ d, uint32_t v, long long count) {
    HSTRIDE(i, count) d[i] = v;
}

__global__ void k_hyb_slot_base(const int *__restrict__ pscan, int count, long long *__restrict__ sb) {
    HSTRIDE(i, (long long)count + 1) sb[i] = 64LL * pscan[i];
}

// the entries of the nl light columns (cps: entries before each sorted column) and the longest one, to the host
__global__ void k_hyb_light(const int *__restrict__ cps, const int *__restrict__ sortnnz, int nl,
                            int *__restrict__ host) {
    if (threadIdx.x == 0) {
        host[0] = cps[nl];
        host[1] = sortnnz[nl - 1];
    }
}

__global__ void k_hyb_f32(const double *__restrict__ in, float *__restrict__ out, long long count) {
    HSTRIDE(i, count) out[i] = (float)in[i];
}

static int cu_count() {
    int dev = 0, cus = 0;
    FL_HIP(hipGetDevice(&dev));
    FL_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    return std::max(cus, 1);
}

void hyb_values(fl_matrix *A, int kind, hipStream_t s) {
    fl_matrix *L = A->hyb_light.get();
    if (!L) return;
    if ((kind == FL_VAL_F32 || kind == FL_VAL_PACKED) && !A->hyb_val32.p) {
        const long long c = 2 * (A->hyb_slots + 2LL * kHybPairs * 64);
        A->hyb_val32.alloc((size_t)c);
        k_hyb_f32<<<hg(c), kBlock, 0, s>>>(A->hyb_val64.p, A->hyb_val32.p, c);
        FL_LAUNCH_CHECK();
    }
    if (kind == FL_VAL_F32 || kind == FL_VAL_PACKED) prepare_values(L, kind, s);
}

void hyb_prepare(fl_matrix *A, int H, int bt, int R, hipStream_t s) {
    if (A->hyb_ready && A->hyb_H == H && A->hyb_bt == bt && A->hyb_R == R) return;
    ++A->built;
    A->hyb_ready = false;
    A->hyb_light.reset();
    A->hyb_val32.release();
    A->hyb_ys32.release();
    A->hyb_ys64.release();
    const int m = A->m, n = A->n, nnz = A->nnz, nl = n - H;
    TmpBuf<int> cps((size_t)n + 1, s);  // entries of the sorted columns before each
    exclusive_scan_i32(A->sortnnz.p, cps.p, n, s);
    HostInts h(s);  // light entries, longest light column; pair rows
    if (nl > 0) {
        k_hyb_light<<<1, 64, 0, s>>>(cps.p, A->sortnnz.p, nl, h.out(0));
        FL_LAUNCH_CHECK();
    }
    const int nnz_l = h.wait()[0];
    const int nnz_h = nnz - nnz_l;

    // light sub-matrix: sorted columns [0, nl) in the same order, its own tiles and PB schedule
    auto L = std::make_unique<fl_matrix>();
    L->m = m;
    L->n = nl;
    L->nnz = nnz_l;
    L->W = 64;
    L->perm.alloc(std::max(nl, 1));
    L->sortnnz.alloc(std::max(nl, 1));
    if (nl > 0) {
        k_hyb_iota<<<hg(nl), kBlock, 0, s>>>(L->perm.p, nl);
        FL_LAUNCH_CHECK();
        FL_HIP(hipMemcpyAsync(L->sortnnz.p, A->sortnnz.p, sizeof(int) * (size_t)nl, hipMemcpyDeviceToDevice, s));
        L->max_col_nnz = h[1];
    }
    {
        ElemSource src;
        src.parent = A;
        transform_device(L.get(), L->sortnnz.p, src, s, nullptr, nullptr, false);
    }
    pb_prepare(L.get(), bt, R & ~63, s);  // bands of whole slices: they are the sorting windows
    const int win = A->hyb_win = L->pb_R;

    // heavy part
    const int nslice = (m + 63) / 64;
    A->hyb_nslice = nslice;
    A->hyb_nnz = nnz_h;
    A->hyb_sb.alloc((size_t)nslice + 1);
    A->hyb_np.alloc(std::max(nslice, 1));
    A->hyb_iperm.alloc(std::max(m, 1));
    A->hyb_perm.alloc(std::max(m, 1));
    long long slots = 0;
    TmpBuf<int> hptr((size_t)m + 1, s), rows(std::max(m, 1), s);
    TmpBuf<uint32_t> rkey(std::max(nnz_h, 1), s);
    TmpBuf<int> ridx(std::max(nnz_h, 1), s);
    TmpBuf<ColEntry> ents(std::max(nnz_h, 1), s);
    FL_HIP(hipMemsetAsync(A->hyb_sb.p, 0, sizeof(long long) * ((size_t)nslice + 1), s));
    if (m > 0) {
        if (nnz_h > 0) {  // heavy entries by row (stable: inside a row by column)
            columns_from_tiles(A, nl, cps.p, nnz_l, nullptr, rkey.p, ents.p, s);
            radix_sort_positions(rkey.p, rkey.p, ridx.p, nnz_h, bits_for((uint32_t)(m - 1)), s);
        }
        key_bounds(rkey.p, nnz_h, m, hptr.p, s);
        // rows by (window, heavy count descending, row)
        TmpBuf<int> pairs(std::max(nslice, 1), s), pscan((size_t)nslice + 1, s);
        const int rounds = div_up(win, kOrderThreads);
        const size_t lds = sizeof(uint16_t) * 4 * rounds * kOrderThreads + sizeof(int) * kOrderWaves * 256;
        FL_HIP(hipFuncSetAttribute((const void *)k_hyb_order, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        k_hyb_order<<<div_up(m, win), kOrderThreads, lds, s>>>(hptr.p, m, win, rounds, rows.p, A->hyb_iperm.p,
                                                              A->hyb_perm.p, A->hyb_np.p, pairs.p);
        FL_LAUNCH_CHECK();
        exclusive_scan_i32(pairs.p, pscan.p, nslice, s, h.out(2));
        k_hyb_slot_base<<<hg((long long)nslice + 1), kBlock, 0, s>>>(pscan.p, nslice, A->hyb_sb.p);
        FL_LAUNCH_CHECK();
        slots = 64LL * h.wait()[2];
    }
    // slots past the last slice: the kernel's look-ahead loads past a wave's last slice read
    // kHybPairs pair rows at hyb_slots, and those past a slice's end up to kHybPairs - 1 pair
    // rows beyond the last slice
    const long long padded = slots + 2LL * kHybPairs * 64;
    A->hyb_slots = slots;
    A->hyb_col2.alloc((size_t)padded);
    A->hyb_val64.alloc((size_t)padded * 2);
    k_hyb_fill_u32<<<hg(padded - slots), kBlock, 0, s>>>(A->hyb_col2.p + slots, (uint32_t)H | ((uint32_t)H << 16),
                                                         padded - slots);
    FL_LAUNCH_CHECK();
    FL_HIP(hipMemsetAsync(A->hyb_val64.p + 2 * slots, 0, sizeof(double) * 2 * (size_t)(padded - slots), s));
    if (A->val32.p) {  // FP32 values along with the others
        A->hyb_val32.alloc((size_t)padded * 2);
        FL_HIP(hipMemsetAsync(A->hyb_val32.p + 2 * slots, 0, sizeof(float) * 2 * (size_t)(padded - slots), s));
    }
    if (slots > 0) {
        k_hyb_fill<<<(grid_for((long long)nslice * 64) + 7u) & ~7u, kBlock, 0, s>>>(m, nslice, H, rows.p, A->hyb_np.p, A->hyb_sb.p, hptr.p,
                                                                 ridx.p, ents.p, A->hyb_col2.p,
                                                                 (double2 *)A->hyb_val64.p,
                                                                 (float2 *)A->hyb_val32.p);
        FL_LAUNCH_CHECK();
    }
    A->hyb_light = std::move(L);
    A->hyb_H = H;
    A->hyb_bt = bt;
    A->hyb_R = R;
    A->hyb_grid = cu_count();
    if (A->val32.p) hyb_values(A, FL_VAL_F32, s);
    if (A->pack_wanted) hyb_values(A, FL_VAL_PACKED, s);
    A->hyb_ready = true;
}

// --------------------------------------------------------------------------- SpMV
// One load group: U pair rows q0 .. q0+U-1 of slice s (P pair rows), and whether it is the
// slice's last group; valid = false past the wave's last slice (its loads read padding).
template <typename V2, int U>
struct HybGroup {
    V2 v[U];
    uint32_t c[U];
    long long s;
    int q0, P;
    bool last, valid;
};

// Per wave: the slices it takes, in snake order (round k: slice k * nw + g0, or k * nw + nw - 1 -
// g0 when k is odd), so that its long and short slices (long first inside every sorting window)
// even out, and the position of the next load group.
struct HybCursor {
    long long s, slot;  // current slice, its first slot + lane
    int k, q, P;        // round, next pair row to load, pair rows of the slice
};

__device__ __forceinline__ long long hyb_slice_of(int k, int nw, int g0) {
    return (long long)k * nw + ((k & 1) ? nw - 1 - g0 : g0);
}

__device__ __forceinline__ void hyb_enter(HybCursor &c, int nslice, const long long *__restrict__ sb,
                                          const int *__restrict__ np, long long pad_slot, int lane) {
    if (c.s < nslice) {
        c.P = np[c.s];
        c.slot = sb[c.s] + lane;
    } else {
        c.P = 0;
        c.slot = pad_slot + lane;
    }
    c.q = 0;
}

// Issues the loads of the cursor's next group (always: past the last slice, or past a slice's pair
// rows, they read padding or the next slice's slots, which hyb_consume skips) and advances the
// cursor, entering the next slice after a slice's last group.
template <typename V2, int U, bool S>
__device__ __forceinline__ void hyb_load(HybGroup<V2, U> &g, HybCursor &c, int nw, int g0, int nslice,
                                         const long long *__restrict__ sb, const int *__restrict__ np,
                                         long long pad_slot, int lane, const V2 *__restrict__ val2,
                                         const uint32_t *__restrict__ col2) {
    g.s = c.s;
    g.q0 = c.q;
    g.P = c.P;
    g.valid = c.s < nslice;
    const long long slot = g.valid ? c.slot + 64LL * c.q : pad_slot + lane;
#pragma unroll
    for (int u = 0; u < U; ++u) {
        if constexpr (S) {
            g.v[u] = ld_stream(&val2[slot + 64 * u]);
            g.c[u] = ld_stream(&col2[slot + 64 * u]);
        } else {
            g.v[u] = val2[slot + 64 * u];
            g.c[u] = col2[slot + 64 * u];
        }
    }
    c.q += U;
    g.last = c.q >= c.P;
    if (g.last && g.valid) {
        ++c.k;
        c.s = hyb_slice_of(c.k, nw, g0);
        hyb_enter(c, nslice, sb, np, pad_slot, lane);
    }
}

// Adds the group's pair rows below P (wave-uniform test: the rest belong to the next slice);
// padding entries multiply value 0 with the zero at xs[H]. After a slice's last group, writes its
// 64 sums by sorted position.
template <typename V2, typename X, typename Y, int U>
__device__ __forceinline__ void hyb_consume(double &acc, const HybGroup<V2, U> &g, const X *xs, int m, int lane,
                                            Y *__restrict__ ys) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
        if (g.q0 + u < g.P) {
            const X x0 = xs[g.c[u] & 0xffffu], x1 = xs[g.c[u] >> 16];
            if constexpr (sizeof(X) == 4) acc += (double)__builtin_fmaf(g.v[u].x, x0, g.v[u].y * x1);  // FP32 pair
            else acc = fma(g.v[u].x, x0, fma(g.v[u].y, x1, acc));
        }
    }
    if (g.last) {
        const long long p = g.s * 64 + lane;
        if (p < m) ys[p] = (Y)acc;
        acc = 0.0;
    }
}

// Persistent workgroups of 16 waves: x of the H heavy columns (and a zero after them) is staged
// in LDS once; then every wave runs through its slices as one stream of load groups, the loads
// of the next group (possibly the next slice's first) in flight while the current one is summed.
// Every group's loads are unconditional, since a conditional load would make the compiler wait
// for all loads in flight before each sum.
// S: read the slots with the streaming hint (stream_reads).
template <typename V2, typename X, typename Y, int U, bool S>
__global__ __launch_bounds__(1024) void k_hyb(int m, int H, int nslice, const long long *__restrict__ sb,
                                              const int *__restrict__ np, long long pad_slot,
                                              const V2 *__restrict__ val2, const uint32_t *__restrict__ col2,
                                              const X *__restrict__ xh, Y *__restrict__ ys) {
    extern __shared__ double hyb_lds[];
    X *xs = reinterpret_cast<X *>(hyb_lds);
    // stage x: 8 loads in flight per thread before their LDS stores (one load-store round trip
    // per element would keep every wave waiting on L2 latency about 10 us before its first slice)
    constexpr int kStage = 8;
    for (int base = 0; base <= H; base += 1024 * kStage) {
        X r[kStage];
#pragma unroll
        for (int j = 0; j < kStage; ++j) {
            const int i = base + j * 1024 + (int)threadIdx.x;
            r[j] = i < H ? xh[i] : X(0);
        }
#pragma unroll
        for (int j = 0; j < kStage; ++j) {
            const int i = base + j * 1024 + (int)threadIdx.x;
            if (i <= H) xs[i] = r[j];
        }
    }
    __syncthreads();
    const int wave = uni((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    const int nw = (int)gridDim.x * 16, g0 = (int)blockIdx.x * 16 + wave;
    HybCursor c;
    c.k = 0;
    c.s = hyb_slice_of(0, nw, g0);
    hyb_enter(c, nslice, sb, np, pad_slot, lane);
    HybGroup<V2, U> a, b;
    double acc = 0.0;
    hyb_load<V2, U, S>(a, c, nw, g0, nslice, sb, np, pad_slot, lane, val2, col2);
    while (a.valid) {
        hyb_load<V2, U, S>(b, c, nw, g0, nslice, sb, np, pad_slot, lane, val2, col2);
        hyb_consume<V2, X, Y, U>(acc, a, xs, m, lane, ys);
        if (!b.valid) break;
        hyb_load<V2, U, S>(a, c, nw, g0, nslice, sb, np, pad_slot, lane, val2, col2);
        hyb_consume<V2, X, Y, U>(acc, b, xs, m, lane, ys);
    }
}

// y = ys in row order (assign) or y += it: the HYB schedule when no light entries exist
template <typename Y, bool ASSIGN>
__global__ void k_hyb_unperm(int m, int win, const uint16_t *__restrict__ iperm, const Y *__restrict__ ys, Y *__restrict__ y) {
    HSTRIDE(r, m) {
        const Y v = ys[(int)r / win * win + iperm[r]];
        if constexpr (ASSIGN) y[r] = v;
        else y[r] += v;
    }
}

int hyb_check(const fl_matrix *A, int kind) {
    if (!A->hyb_ready) {
        set_error("fl_spmv: HYB schedule not prepared");
        return FL_ERR_INVALID;
    }
    if (kind != FL_VAL_F64 && kind != FL_VAL_F32 && kind != FL_VAL_PACKED) {
        set_error("fl_spmv: the HYB schedule supports FL_VAL_F64, FL_VAL_F32 and FL_VAL_PACKED");
        return FL_ERR_INVALID;
    }
    if (kind == FL_VAL_F64 && A->hyb_nnz > 0 && A->hyb_H > kHybMaxH64) {
        set_error("fl_spmv: FL_VAL_F64 with the HYB schedule needs at most %d heavy columns (prepared: %d)",
                  kHybMaxH64, A->hyb_H);
        return FL_ERR_INVALID;
    }
    if (kind != FL_VAL_F64 && A->hyb_nnz > 0 && !A->hyb_val32.p) {
        set_error("fl_spmv: FP32 values not prepared");
        return FL_ERR_INVALID;
    }
    const fl_matrix *L = A->hyb_light.get();
    if (L->tilenum > 0) {
        if (kind == FL_VAL_F32 && !L->val32.p) {
            set_error("fl_spmv: FP32 values not prepared");
            return FL_ERR_INVALID;
        }
        if (kind == FL_VAL_PACKED && !L->pb_pack.p) {
            set_error("fl_spmv: no packed values for the HYB schedule's PB part (fl_matrix_prepare_values("
                      "FL_VAL_PACKED) not called, or fewer than 12 mantissa bits would remain)");
            return FL_ERR_INVALID;
        }
    }
    return FL_OK;
}

static size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

size_t hyb_scratch_bytes(const fl_matrix *A, int kind) {
    const size_t ysz = kind == FL_VAL_F64 ? sizeof(double) : sizeof(float);
    const fl_matrix *L = A->hyb_light.get();
    const size_t bins = (L && L->tilenum > 0) ? (size_t)L->pb_ring * ysz : 0;
    return align256((size_t)A->m * ysz) + bins;
}

template <typename V2, typename X, typename Y>
static void launch_hyb(const fl_matrix *A, const V2 *val2, const X *xh, Y *ys, bool stream, hipStream_t s) {
    constexpr int U = kHybPairs;
    const size_t lds = ((size_t)A->hyb_H + 1) * sizeof(X);
    auto k = stream ? k_hyb<V2, X, Y, U, true> : k_hyb<V2, X, Y, U, false>;
    FL_HIP(hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    // two workgroups per compute unit (32 waves) when their LDS fits, else one
    const int per_cu = lds <= 80 * 1024 ? 2 : 1;
    const int grid = std::max(1, std::min(A->hyb_grid * per_cu, (A->hyb_nslice + 15) / 16));
    k<<<grid, 1024, lds, s>>>(A->m, A->hyb_H, A->hyb_nslice, A->hyb_sb.p, A->hyb_np.p, A->hyb_slots, val2,
                              A->hyb_col2.p, xh, ys);
    FL_LAUNCH_CHECK();
}

// Called by spmv after hyb_check. x = sortx (n entries).
int spmv_hyb(fl_matrix *A, int kind, const void *x, void *y, bool assign, hipStream_t s, void *scratch) {
    fl_matrix *L = A->hyb_light.get();
    const bool dbl = kind == FL_VAL_F64;
    const int m = A->m, nl = L->n;
    void *ys = nullptr, *bins = nullptr;
    if (scratch) {
        ys = scratch;
        bins = (char *)scratch + align256((size_t)m * (dbl ? 8 : 4));
    } else if (A->hyb_nnz > 0) {
        if (dbl) {
            if (!A->hyb_ys64.p) A->hyb_ys64.alloc(std::max(m, 1));
            ys = A->hyb_ys64.p;
        } else {
            if (!A->hyb_ys32.p) A->hyb_ys32.alloc(std::max(m, 1));
            ys = A->hyb_ys32.p;
        }
    }
    const bool heavy = A->hyb_nnz > 0;
    // one streaming decision for the three kernels, which share the caches
    const long long heavy_bytes = heavy ? A->hyb_slots * (long long)(dbl ? 16 + 4 : 8 + 4) : 0;
    const bool stream =
        stream_reads(heavy_bytes + (L->tilenum > 0 ? batched_stream_bytes(L, FL_KERNEL_PB, kind) : 0));
    if (heavy) {
        if (dbl) launch_hyb<double2, double, double>(A, (const double2 *)A->hyb_val64.p, (const double *)x + nl, (double *)ys, stream, s);
        else launch_hyb<float2, float, float>(A, (const float2 *)A->hyb_val32.p, (const float *)x + nl, (float *)ys, stream, s);
    }
    if (L->tilenum > 0) {
        PbFold fold;
        if (heavy) {
            fold.ys = ys;
            fold.perm = A->hyb_perm.p;
        }
        return spmv_batched(L, FL_KERNEL_PB, kind, x, y, assign, s, bins, &fold, stream ? 1 : 0);
    }
    if (heavy) {
        if (dbl) {
            if (assign) k_hyb_unperm<double, true><<<hg(m), kBlock, 0, s>>>(m, A->hyb_win, A->hyb_iperm.p, (const double *)ys, (double *)y);
            else k_hyb_unperm<double, false><<<hg(m), kBlock, 0, s>>>(m, A->hyb_win, A->hyb_iperm.p, (const double *)ys, (double *)y);
        } else {
            if (assign) k_hyb_unperm<float, true><<<hg(m), kBlock, 0, s>>>(m, A->hyb_win, A->hyb_iperm.p, (const float *)ys, (float *)y);
            else k_hyb_unperm<float, false><<<hg(m), kBlock, 0, s>>>(m, A->hyb_win, A->hyb_iperm.p, (const float *)ys, (float *)y);
        }
        FL_LAUNCH_CHECK();
    } else if (assign) {
        zero_fill(y, (size_t)m * (dbl ? 8 : 4), s);
    }
    return FL_OK;
}

}  // namespace fl
