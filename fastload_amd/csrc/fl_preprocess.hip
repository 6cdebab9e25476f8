// FastLoad preprocessing on the GPU: CSR->CSC, stable column sort, level table, tile
// enumeration, tile data layout, segment detection and tile classification.
//
// Reference pipeline (skyler-ruiter/FastLoad): csr_to_csc (src/csr2csc_cuda.h:51-135),
// ColSort (src/ColSort_GPU.h:46-137), formatTransform (src/formatTransform_GPU.h:289-596).
// The reference's quadratic prefix loops (ColSort_GPU.h:30-33, formatTransform_GPU.h:41-47,
// 123-129) and per-tile serial loops are replaced by scans and closed forms:
//   level k   : sorted position col_k where the length steps up; base_k = length before the
//               step; tall_k = step size
//   tiles     : level k has T_k = ceil((n-col_k)/W) chunks x tall_k depths, ordered
//               (level, chunk, depth); tile t in level k: j = local / tall_k, e = local % tall_k
//   tile_ptr  : nnzoff_k + j*tall_k*W + e*len  (only the last chunk of a level is short)
//   element   : (sorted column colidx+l, depth base_k+e)
#include <algorithm>
#include <vector>

#include "fl_matrix.h"

namespace fl {

// ----------------------------------------------------------------------- small kernels
template <typename T>
__global__ void k_gather(const T *__restrict__ src, const int *__restrict__ idx, T *__restrict__ dst, int count) {
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += (long long)gridDim.x * blockDim.x)
        dst[i] = src[idx[i]];
}

static unsigned stride_grid(long long count) { return std::max(1u, std::min<unsigned>(grid_for(count), 65536u)); }

// ---------------------------------------------------------------------- input checks
// bad[0] (host memory): ptr not monotone / wrong ends; bad[1]: index out of range. Nothing is written for a
// sound matrix.
__global__ void k_check(const int *__restrict__ ptr, int count, const int *__restrict__ idx, int nnz, int limit,
                        int *__restrict__ bad) {
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x, step = (long long)gridDim.x * blockDim.x;
    for (long long i = t; i < count; i += step) {
        const int a = ptr[i], b = ptr[i + 1];
        if (a > b || a < 0 || b > nnz) bad[0] = 1;
    }
    if (t == 0 && (ptr[0] != 0 || ptr[count] != nnz)) bad[0] = 1;
    for (long long i = t; i < nnz; i += step) {
        const int r = idx[i];
        if (r < 0 || r >= limit) bad[1] = 1;
    }
}

// Starts the check that ptr[0]==0, ptr[count]==nnz, ptr is monotone and every idx in [0, limit); after h.wait(),
// check_result is 0 if so, else bit 0: ptr, bit 1: idx.
void check_begin(const int *d_ptr, int count, const int *d_idx, int nnz, int limit, HostInts &h, hipStream_t s) {
    k_check<<<stride_grid(std::max(count, nnz)), kBlock, 0, s>>>(d_ptr, count, d_idx, nnz, limit, h.out());
    FL_LAUNCH_CHECK();
}

int check_result(const HostInts &h) { return (h[0] ? 1 : 0) | (h[1] ? 2 : 0); }

int check_compressed(const int *d_ptr, int count, const int *d_idx, int nnz, int limit, hipStream_t s) {
    HostInts h(s);
    check_begin(d_ptr, count, d_idx, nnz, limit, h, s);
    (void)h.wait();
    return check_result(h);
}

// ------------------------------------------------------------------------------ csr2csc
__global__ void k_row_of(const int *__restrict__ rowptr, int m, int *__restrict__ row_of) {
    for (long long r = (long long)blockIdx.x * blockDim.x + threadIdx.x; r < m; r += (long long)gridDim.x * blockDim.x)
        for (int j = rowptr[r]; j < rowptr[r + 1]; ++j) row_of[j] = (int)r;
}

__global__ void k_count(const uint32_t *__restrict__ keys, int count, int *__restrict__ counts) {
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += (long long)gridDim.x * blockDim.x)
        atomicAdd(&counts[keys[i]], 1);
}

__global__ void k_csc_fill(const int *__restrict__ order, const int *__restrict__ row_of, const double *__restrict__ val,
                           int *__restrict__ cscrow, double *__restrict__ cscval, int count) {
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += (long long)gridDim.x * blockDim.x) {
        const int o = order[i];
        cscrow[i] = row_of[o];
        cscval[i] = val[o];
    }
}

// CSR -> CSC: stable LSD radix sort of the column indices with the CSR position as payload;
// stability keeps rows ascending inside each column (CSR positions ascend with the row).
void csr2csc_device(int m, int n, int nnz, const int *d_rowptr, const int *d_colind, const double *d_val,
                    double *d_cscval, int *d_cscrow, int *d_colptr, int *d_nnzpercol, hipStream_t s) {
    FL_HIP(hipMemsetAsync(d_nnzpercol, 0, sizeof(int) * std::max(n, 1), s));
    if (nnz > 0) {
        TmpBuf<uint32_t> keys(nnz, s);
        TmpBuf<int> order(nnz, s), row_of(nnz, s);
        k_row_of<<<stride_grid(m), kBlock, 0, s>>>(d_rowptr, m, row_of.p);
        FL_LAUNCH_CHECK();
        radix_sort_positions((const uint32_t *)d_colind, keys.p, order.p, nnz,
                             bits_for((uint32_t)std::max(n - 1, 0)), s);
        k_csc_fill<<<stride_grid(nnz), kBlock, 0, s>>>(order.p, row_of.p, d_val, d_cscrow, d_cscval, nnz);
        k_count<<<stride_grid(nnz), kBlock, 0, s>>>(keys.p, nnz, d_nnzpercol);
        FL_LAUNCH_CHECK();
    }
    exclusive_scan_i32(d_nnzpercol, d_colptr, n, s);
    FL_HIP(hipStreamSynchronize(s));
}

// ------------------------------------------------------------------------ column sort
void colsort_device(int n, const int *d_counts, int *d_perm, int *d_sortnnz, int max_key, hipStream_t s) {
    if (n <= 0) return;
    radix_sort_positions((const uint32_t *)d_counts, (uint32_t *)d_sortnnz, d_perm, n, bits_for((uint32_t)max_key), s);
}

// Concatenate the sorted columns (Pre4SortIdxVal, ColSort_GPU.h:21-43): one lane per column
// for short columns; columns at or beyond `long_from` (lengths are ascending) get a wave each.
__global__ void k_sorted_copy_short(int n, int long_from, const int *__restrict__ perm, const int *__restrict__ P,
                                    const int *__restrict__ colptr, const int *__restrict__ rowidx,
                                    const double *__restrict__ val, int *__restrict__ tmp_row,
                                    double *__restrict__ tmp_val) {
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < long_from; i += (long long)gridDim.x * blockDim.x) {
        const int c = perm[i], src = colptr[c], len = colptr[c + 1] - src, dst = P[i];
        for (int d = 0; d < len; ++d) {
            tmp_row[dst + d] = rowidx[src + d];
            tmp_val[dst + d] = val[src + d];
        }
    }
}

__global__ void k_sorted_copy_long(int n, int long_from, const int *__restrict__ perm, const int *__restrict__ P,
                                   const int *__restrict__ colptr, const int *__restrict__ rowidx,
                                   const double *__restrict__ val, int *__restrict__ tmp_row,
                                   double *__restrict__ tmp_val) {
    const int lane = threadIdx.x & 63;
    const long long wave0 = ((long long)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const long long nwaves = ((long long)gridDim.x * blockDim.x) >> 6;
    for (long long i = long_from + wave0; i < n; i += nwaves) {
        const int c = perm[i], src = colptr[c], len = colptr[c + 1] - src, dst = P[i];
        for (int d = lane; d < len; d += 64) {
            tmp_row[dst + d] = rowidx[src + d];
            tmp_val[dst + d] = val[src + d];
        }
    }
}

__global__ void k_lower_bound(const int *__restrict__ sorted, int n, int key, int *__restrict__ out) {
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        int lo = 0, hi = n;
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if (sorted[mid] < key) lo = mid + 1; else hi = mid;
        }
        *out = lo;
    }
}

void sorted_copy(int n, const int *d_perm, const int *d_sortnnz, const int *d_P, const int *d_colptr,
                 const int *d_rowidx, const double *d_val, int *d_tmp_row, double *d_tmp_val, hipStream_t s) {
    if (n <= 0) return;
    HostInts lf(s);
    k_lower_bound<<<1, 64, 0, s>>>(d_sortnnz, n, 64, lf.out());
    FL_LAUNCH_CHECK();
    const int long_from = *lf.wait();
    if (long_from > 0) {
        k_sorted_copy_short<<<stride_grid(long_from), kBlock, 0, s>>>(n, long_from, d_perm, d_P, d_colptr, d_rowidx,
                                                                       d_val, d_tmp_row, d_tmp_val);
        FL_LAUNCH_CHECK();
    }
    if (long_from < n) {
        const long long waves = n - long_from;
        const unsigned g = std::max(1u, std::min<unsigned>(grid_for(waves * 64), 16384u));
        k_sorted_copy_long<<<g, kBlock, 0, s>>>(n, long_from, d_perm, d_P, d_colptr, d_rowidx, d_val, d_tmp_row,
                                                d_tmp_val);
        FL_LAUNCH_CHECK();
    }
}

// --------------------------------------------------------------------- level table
__global__ void k_level_flags(const int *__restrict__ s, int n, int *__restrict__ flags) {
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
        flags[i] = (i == 0) ? (s[0] != 0) : (s[i] != s[i - 1]);
}

__global__ void k_level_fill(const int *__restrict__ s, int n, int W, const int *__restrict__ lidx,
                             int *__restrict__ lvl_col, int *__restrict__ lvl_base, int *__restrict__ lvl_tall,
                             int *__restrict__ lvl_tiles, int *__restrict__ lvl_nnz) {
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
        const int k = lidx[i];
        if (lidx[i + 1] == k) continue;  // not a level start
        const int base = (i == 0) ? 0 : s[i - 1];
        const int tall = s[i] - base;
        const long long width = n - i;
        lvl_col[k] = (int)i;
        lvl_base[k] = base;
        lvl_tall[k] = tall;
        lvl_tiles[k] = (int)(((width + W - 1) / W) * tall);
        lvl_nnz[k] = (int)(width * tall);
    }
}

// Level of tile t: the k with tileoff[k] <= t < tileoff[k+1].
__device__ __forceinline__ int find_level(const int *__restrict__ tileoff, int L, int t) {
    int lo = 0, hi = L - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (tileoff[mid] <= t) lo = mid; else hi = mid - 1;
    }
    return lo;
}

__global__ void k_tiles(int T, int L, int n, int nnz, int W, const int *__restrict__ lvl_col,
                        const int *__restrict__ lvl_base, const int *__restrict__ lvl_tall,
                        const int *__restrict__ tileoff, const int *__restrict__ nnzoff, int *__restrict__ tile_ptr,
                        int *__restrict__ tile_len, int *__restrict__ tile_colidx, int *__restrict__ tile_depth) {
    for (long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x; t < T; t += (long long)gridDim.x * blockDim.x) {
        const int k = find_level(tileoff, L, (int)t);
        const int local = (int)t - tileoff[k];
        const int tall = lvl_tall[k], col = lvl_col[k];
        const int j = local / tall, e = local - j * tall;
        const int width = n - col;
        const int chunks = (width + W - 1) / W;
        const int len = (j == chunks - 1) ? width - (chunks - 1) * W : W;
        tile_len[t] = len;
        tile_colidx[t] = col + W * j;
        tile_depth[t] = lvl_base[k] + e;
        tile_ptr[t] = nnzoff[k] + j * tall * W + e * len;
        if (t == T - 1) tile_ptr[T] = nnz;
    }
}

// ------------------------------------------------------------------- columns <-> tiles
// The levels as kernels read them: element (sorted column i, depth d) is at
//   nnzoff_k + j * tall_k * W + (d - base_k) * len + lane,  j, lane = divmod(i - col_k, W),
// in level k (base_k <= d < base_k + tall_k), len = W except in the level's last chunk.
struct Levels {
    const int *__restrict__ col;
    const int *__restrict__ base;
    const int *__restrict__ tall;
    const int *__restrict__ nnzoff;
    int L, n, W;
};

struct Level {
    int col, base, tall, off, chunks, last;  // last = length of the tiles of the last chunk

    __device__ __forceinline__ void load(const Levels &lv, int k) {
        set(lv, uni(lv.col[k]), uni(lv.base[k]), uni(lv.tall[k]), uni(lv.nnzoff[k]));
    }
    __device__ __forceinline__ void set(const Levels &lv, int c, int b, int t, int o) {
        col = c;
        base = b;
        tall = t;
        off = o;
        const int width = lv.n - col;
        chunks = (width + lv.W - 1) / lv.W;
        last = width - (chunks - 1) * lv.W;
    }
    __device__ __forceinline__ int at(const Levels &lv, int i, int d) const {
        const int w = i - col, lg = lv.W == 64 ? 6 : 5;
        const int j = w >> lg;
        return off + ((j * tall) << lg) + (d - base) * (j == chunks - 1 ? last : lv.W) + (w & (lv.W - 1));
    }
};

// Walks between column order and tile order: a wave takes 64 consecutive sorted columns, a lane each, and
// kWalkDepth consecutive depths; on the tile side its lanes touch one or two runs of consecutive positions
// for each depth. One thread per element in tile order instead fetched a whole line of the column for
// each entry, level after level. A long column is spread over many waves: item q of group g is its depths
// from q * kWalkDepth on.
// Tiles from columns, 10 M power-law entries: one thread per element 193 us, this with a lane per column on both
// sides 139, with 16-byte pieces through LDS 121, with the levels in lanes 112 (67 M entries: 690; 4 M
// entries of uniform columns of 8: 149 -> 56). Columns from tiles, 7.4 M entries: 242, 98 and 89 us.
constexpr int kWalkDepth = 32;

__global__ void k_walk_items(const int *__restrict__ sortnnz, int n, int groups, int *__restrict__ items) {
    for (long long g = (long long)blockIdx.x * blockDim.x + threadIdx.x; g < groups; g += (long long)gridDim.x * blockDim.x)
        items[g] = (sortnnz[min((int)g * 64 + 63, n - 1)] + kWalkDepth - 1) / kWalkDepth;
}

struct Walk {
    const int *__restrict__ start;     // [groups + 1] items before each group
    const int *__restrict__ level_of;  // [depths]
    int groups, first_group, depths;
};

// level_of[d] = the level of depth d
__global__ void k_depth_levels(const int *__restrict__ base, int L, int depths, int *__restrict__ level_of) {
    for (long long d = (long long)blockIdx.x * blockDim.x + threadIdx.x; d < depths; d += (long long)gridDim.x * blockDim.x)
        level_of[d] = find_level(base, L, (int)d);
}

// The levels of a wave's depths, those of d0 + u in lane u: read with readlane, so the walk does not wait for
// memory where the level changes with every depth or two (long columns).
struct LaneLevels {
    int col, base, tall, off;
    __device__ __forceinline__ void load(const Levels &lv, const int *__restrict__ level_of, int depths, int d0) {
        const int k = level_of[min(d0 + (int)(threadIdx.x & (kWalkDepth - 1)), depths - 1)];
        col = lv.col[k];
        base = lv.base[k];
        tall = lv.tall[k];
        off = lv.nnzoff[k];
    }
    __device__ __forceinline__ Level get(const Levels &lv, int u) const {
        Level l;
        l.set(lv, __builtin_amdgcn_readlane(col, u), __builtin_amdgcn_readlane(base, u),
              __builtin_amdgcn_readlane(tall, u), __builtin_amdgcn_readlane(off, u));
        return l;
    }
};

// The wave's item -> its group and first depth; false past the last item.
__device__ __forceinline__ bool walk_item(const Walk &w, int &g, int &d0) {
    const long long wave = ((long long)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const long long item = wave + uni(w.start[w.first_group]);
    if (item >= uni(w.start[w.groups])) return false;
    int lo = w.first_group, hi = w.groups - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (uni(w.start[mid]) <= item) lo = mid; else hi = mid - 1;
    }
    g = uni(lo);
    d0 = ((int)item - uni(w.start[g])) * kWalkDepth;
    return true;
}

// A wave's stage: kStageDepth entries of each of its 64 columns. The column side is accessed by pieces of 16
// bytes, consecutive lanes on consecutive pieces of a column (a lane per column and entry makes as many
// requests, each for a line of its own); the tile side by a lane per column.
constexpr int kStageDepth = 8;
struct WalkStage {
    alignas(16) double val[64][kStageDepth];
    alignas(16) int row[64][kStageDepth];
    long long at[64];  // column side: position of the column's first entry
    int len[64], col[64];
};

// Tile data layout (dataTrans, formatTransform_GPU.h:152-171) from columns: column i's entries start at
// start[i] (start of perm[i] in colptr when start is null) of src rows and values, count entries in all.
__global__ __launch_bounds__(kBlock) void k_fill_tiles(Walk w, Levels lv, const int *__restrict__ sortnnz,
                                                       const int *__restrict__ start, const int *__restrict__ colptr,
                                                       const int *__restrict__ perm, const int *__restrict__ src_row,
                                                       const double *__restrict__ src_val, int count,
                                                       int *__restrict__ sortrowidx, double *__restrict__ sortval) {
    __shared__ WalkStage stage[kBlock / 64];
    int g, d0;
    if (!walk_item(w, g, d0)) return;
    WalkStage &st = stage[threadIdx.x >> 6];
    const int lane = (int)(threadIdx.x & 63), i = g * 64 + lane;
    const int len = i < lv.n ? sortnnz[i] : 0;
    st.len[lane] = len;
    st.at[lane] = len > d0 ? (start ? start[i] : colptr[perm[i]]) : 0;
    LaneLevels ll;
    ll.load(lv, w.level_of, w.depths, d0);
    for (int d = d0; d < d0 + kWalkDepth; d += kStageDepth) {
        if (!ballot64(d < len)) break;
        // pieces of 4 rows or 2 values; whole loads also past the column's end, up to the arrays' end
#pragma unroll
        for (int q = 0; q < kStageDepth / 4; ++q) {
            const int t = q * 64 + lane, c = t / (kStageDepth / 4), o = t % (kStageDepth / 4) * 4;
            const long long at = st.at[c] + d + o;
            const int left = st.len[c] - d - o;
            alignas(16) int row[4] = {0, 0, 0, 0};
            if (left > 0) {
                if (at + 4 <= count) {
                    __builtin_memcpy(row, src_row + at, sizeof row);
                } else {
                    for (int u = 0; u < 4 && u < left; ++u) row[u] = src_row[at + u];
                }
            }
            *reinterpret_cast<int4 *>(&st.row[c][o]) = *reinterpret_cast<int4 *>(row);
        }
#pragma unroll
        for (int q = 0; q < kStageDepth / 2; ++q) {
            const int t = q * 64 + lane, c = t / (kStageDepth / 2), o = t % (kStageDepth / 2) * 2;
            const long long at = st.at[c] + d + o;
            const int left = st.len[c] - d - o;
            alignas(16) double val[2] = {0.0, 0.0};
            if (left > 0) {
                if (at + 2 <= count) __builtin_memcpy(val, src_val + at, sizeof val);
                else val[0] = src_val[at];
            }
            *reinterpret_cast<double2 *>(&st.val[c][o]) = *reinterpret_cast<double2 *>(val);
        }
        __builtin_amdgcn_wave_barrier();  // the wave's own LDS accesses are in order
#pragma unroll
        for (int u = 0; u < kStageDepth; ++u) {
            if (!ballot64(d + u < len)) break;
            const Level l = ll.get(lv, d - d0 + u);
            if (d + u < len) {
                const int p = l.at(lv, i, d + u);
                sortrowidx[p] = st.row[lane][u];
                sortval[p] = st.val[lane][u];
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
}

__global__ __launch_bounds__(kBlock) void k_columns_from_tiles(Walk w, Levels lv, const int *__restrict__ sortnnz,
                                                               int first, const int *__restrict__ dst, int base,
                                                               const int *__restrict__ col_of,
                                                               const int *__restrict__ sortrowidx,
                                                               const double *__restrict__ sortval,
                                                               uint32_t *__restrict__ rows, ColEntry *__restrict__ ents) {
    __shared__ WalkStage stage[kBlock / 64];
    int g, d0;
    if (!walk_item(w, g, d0)) return;
    WalkStage &st = stage[threadIdx.x >> 6];
    const int lane = (int)(threadIdx.x & 63), i = g * 64 + lane;
    const int len = i >= first && i < lv.n ? sortnnz[i] : 0;
    st.len[lane] = len;
    if (len > d0) {
        const int col = col_of ? col_of[i] : i - first;
        st.col[lane] = col;
        st.at[lane] = (long long)dst[col_of ? col : i] - base;
    }
    LaneLevels ll;
    ll.load(lv, w.level_of, w.depths, d0);
    for (int d = d0; d < d0 + kWalkDepth; d += kStageDepth) {
        if (!ballot64(d < len)) break;
        int p[kStageDepth];
#pragma unroll
        for (int u = 0; u < kStageDepth; ++u) {
            const Level l = ll.get(lv, d - d0 + u);
            p[u] = d + u < len ? l.at(lv, i, d + u) : -1;
        }
        int row[kStageDepth];
        double val[kStageDepth];
#pragma unroll
        for (int u = 0; u < kStageDepth; ++u) {
            row[u] = p[u] >= 0 ? sortrowidx[p[u]] : 0;
            val[u] = p[u] >= 0 ? sortval[p[u]] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < kStageDepth; ++u) {
            st.row[lane][u] = row[u];
            st.val[lane][u] = val[u];
        }
        __builtin_amdgcn_wave_barrier();  // the wave's own LDS accesses are in order
#pragma unroll
        for (int q = 0; q < kStageDepth; ++q) {  // kStageDepth lanes write a column's entries
            const int t = q * 64 + lane, c = t / kStageDepth, o = t % kStageDepth;
            if (d + o < st.len[c]) {
                const long long at = st.at[c] + d + o;
                rows[at] = (uint32_t)st.row[c][o];
                ents[at] = ColEntry{st.val[c][o], st.col[c], 0};
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
}

// Tile data of a sub-matrix of the parent's first n sorted columns (parent mode): one thread per (tile, lane).
__global__ void k_copy_tiles(int T, int W, const int *__restrict__ tile_ptr, const int *__restrict__ tile_len,
                             const int *__restrict__ tile_colidx, const int *__restrict__ tile_depth,
                             const int *__restrict__ tileoff, Levels pl, const int *__restrict__ prow,
                             const double *__restrict__ pval, int L, int *__restrict__ sortrowidx,
                             double *__restrict__ sortval) {
    const long long total = (long long)T * W;
    for (long long g = (long long)blockIdx.x * blockDim.x + threadIdx.x; g < total; g += (long long)gridDim.x * blockDim.x) {
        const int t = uni((int)(g / W));  // W = 64: a wave per tile
        const int l = (int)(g - (long long)t * W);
        Level lev;
        lev.load(pl, find_level(tileoff, L, t));
        if (l >= tile_len[t]) continue;
        const int at = lev.at(pl, tile_colidx[t] + l, tile_depth[t]);
        const int dst = tile_ptr[t] + l;
        sortrowidx[dst] = prow[at];
        sortval[dst] = pval[at];
    }
}

static Levels levels_of(const fl_matrix *A) {
    return {A->lvl_col.p, A->lvl_base.p, A->lvl_tall.p, A->lvl_nnzoff.p, A->L, A->n, A->W};
}

// start[g] = items of the groups before g. At most walk_bound items in all: a group has as many as its longest
// column needs, which is no longer than any column of the next group; the last two groups are bounded by
// the longest column (the last one may have fewer than 64 columns).
struct WalkPlan {
    TmpBuf<int> start, level_of;
    Walk w;
    WalkPlan(const fl_matrix *A, const int *sortnnz, int first, hipStream_t s) : start(s), level_of(s) {
        const int groups = div_up(A->n, 64), depths = std::max(A->max_col_nnz, 1);
        TmpBuf<int> items(groups, s);
        start.alloc((size_t)groups + 1);
        level_of.alloc(depths);
        k_walk_items<<<stride_grid(groups), kBlock, 0, s>>>(sortnnz, A->n, groups, items.p);
        k_depth_levels<<<stride_grid(depths), kBlock, 0, s>>>(A->lvl_base.p, A->L, depths, level_of.p);
        FL_LAUNCH_CHECK();
        exclusive_scan_i32(items.p, start.p, groups, s);
        w = {start.p, level_of.p, groups, first / 64, depths};
    }
};

static long long walk_bound(int columns, long long entries, int longest) {
    return div_up(columns, 64) + 1 + (entries / 64 + 2LL * longest) / kWalkDepth + 1;
}

static unsigned walk_grid(long long items) { return (unsigned)((items + kBlock / 64 - 1) / (kBlock / 64)); }

void columns_from_tiles(const fl_matrix *A, int first, const int *dst, int base, const int *col_of, uint32_t *rows,
                        ColEntry *ents, hipStream_t s) {
    if (A->nnz == 0 || first >= A->n) return;
    const WalkPlan plan(A, A->sortnnz.p, first, s);
    k_columns_from_tiles<<<walk_grid(walk_bound(A->n - first + 64, A->nnz, A->max_col_nnz)), kBlock, 0, s>>>(
        plan.w, levels_of(A), A->sortnnz.p, first, dst, base, col_of, A->sortrowidx.p, A->val64.p, rows, ents);
    FL_LAUNCH_CHECK();
}

// Segments + tile format (Pre4CountRow .. Pre4tileclass, formatTransform_GPU.h:188-285):
// one wave holds 64/W tiles; heads from a neighbour compare; run lengths from the head mask.
// Each wave takes kClassTiles of them, all loads before their use: 8.8 M entries 41 -> 23 us,
// k_segoff 38 -> 20.
constexpr int kClassTiles = 4;
template <int W>
__global__ __launch_bounds__(kBlock) void k_classify(int T, const int *__restrict__ tile_ptr,
                                                     const int *__restrict__ tile_len,
                                                     const int *__restrict__ sortrowidx,
                                                     int *__restrict__ sortrowindex, int *__restrict__ seg_count,
                                                     int *__restrict__ tile_format) {
    constexpr int S = 64 / W;
    const int lane = threadIdx.x & 63;
    const long long wave = ((long long)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int sub = lane / W, l = lane % W;
    const long long t0 = wave * (S * kClassTiles) + sub;
    int len[kClassTiles], ptr[kClassTiles], row[kClassTiles];
#pragma unroll
    for (int u = 0; u < kClassTiles; ++u) {
        const long long t = t0 + u * S;
        len[u] = t < T ? tile_len[t] : 0;
        ptr[u] = t < T ? tile_ptr[t] : 0;
    }
#pragma unroll
    for (int u = 0; u < kClassTiles; ++u) row[u] = l < len[u] ? sortrowidx[ptr[u] + l] : -1;
#pragma unroll
    for (int u = 0; u < kClassTiles; ++u) {
        const long long t = t0 + u * S;
        const bool act = l < len[u];
        const int prev = __shfl_up(row[u], 1);
        const bool head = act && (l == 0 || row[u] != prev);
        const uint64_t hm = ballot64(head);
        const uint64_t tmask = (W == 64) ? hm : ((hm >> (sub * 32)) & 0xffffffffull);
        if (act) {
            int run = 0;
            if (head) {
                const uint64_t above = (l + 1 >= 64) ? 0ull : (tmask >> (l + 1));
                const int nh = above ? (l + 1 + __ffsll((long long)above) - 1) : len[u];
                run = min(nh, len[u]) - l;
            }
            sortrowindex[ptr[u] + l] = run;
        }
        if (t < T && l == 0) {
            const int cnt = __popcll(tmask);
            seg_count[t] = cnt;
            tile_format[t] = (len[u] == W) ? (cnt == 1 ? 1 : 2) : 0;
        }
    }
}

template <int W>
__global__ __launch_bounds__(kBlock) void k_segoff(int T, const int *__restrict__ tile_ptr,
                                                   const int *__restrict__ tile_len,
                                                   const int *__restrict__ sortrowindex,
                                                   const int *__restrict__ countrow, int *__restrict__ segoff) {
    constexpr int S = 64 / W;
    const int lane = threadIdx.x & 63;
    const long long wave = ((long long)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int sub = lane / W, l = lane % W;
    const long long t0 = wave * (S * kClassTiles) + sub;
    int len[kClassTiles], ptr[kClassTiles], at[kClassTiles], run[kClassTiles];
#pragma unroll
    for (int u = 0; u < kClassTiles; ++u) {
        const long long t = t0 + u * S;
        len[u] = t < T ? tile_len[t] : 0;
        ptr[u] = t < T ? tile_ptr[t] : 0;
        at[u] = t < T ? countrow[t] : 0;
    }
#pragma unroll
    for (int u = 0; u < kClassTiles; ++u) run[u] = l < len[u] ? sortrowindex[ptr[u] + l] : 0;
#pragma unroll
    for (int u = 0; u < kClassTiles; ++u) {
        const uint64_t hm = ballot64(run[u] != 0);
        const uint64_t tmask = (W == 64) ? hm : ((hm >> (sub * 32)) & 0xffffffffull);
        if (run[u] != 0) {
            const uint64_t below = (l == 0) ? 0ull : (tmask & ((1ull << l) - 1ull));
            segoff[at[u] + __popcll(below)] = run[u];
        }
    }
}

// Level of the first tile of each group of 64 tiles (for the FAST kernel).
__global__ void k_group_level(int T, int L, const int *__restrict__ tileoff, int *__restrict__ group_level) {
    const long long groups = ((long long)T + 63) / 64;
    for (long long gidx = (long long)blockIdx.x * blockDim.x + threadIdx.x; gidx < groups; gidx += (long long)gridDim.x * blockDim.x)
        group_level[gidx] = find_level(tileoff, L, (int)(gidx * 64));
}

void transform_device(fl_matrix *A, const int *d_sortnnz, const ElemSource &src, hipStream_t s, float *t_tran_ms,
                      float *t_clas_ms, bool classify) {
    const int n = A->n, nnz = A->nnz, W = A->W;
    HostInts h(s);  // levels; tiles and entries they cover; segments
    const bool timed = t_tran_ms || t_clas_ms;
    hipEvent_t e0 = nullptr, e1 = nullptr, e2 = nullptr;
    if (timed) {
        FL_HIP(hipEventCreate(&e0));
        FL_HIP(hipEventCreate(&e1));
        FL_HIP(hipEventCreate(&e2));
        FL_HIP(hipEventRecord(e0, s));
    }

    // levels
    TmpBuf<int> flags(std::max(n, 1), s), lidx((size_t)n + 1, s);
    if (n > 0) {
        k_level_flags<<<stride_grid(n), kBlock, 0, s>>>(d_sortnnz, n, flags.p);
        FL_LAUNCH_CHECK();
    }
    exclusive_scan_i32(flags.p, lidx.p, n, s, h.out(0));
    const int L = h.wait()[0];
    A->L = L;
    A->lvl_col.alloc(std::max(L, 1));
    A->lvl_base.alloc(std::max(L, 1));
    A->lvl_tall.alloc(std::max(L, 1));
    A->lvl_tileoff.alloc((size_t)L + 1);
    A->lvl_nnzoff.alloc((size_t)L + 1);
    TmpBuf<int> lvl_tiles(std::max(L, 1), s), lvl_nnz(std::max(L, 1), s);
    if (n > 0) {
        k_level_fill<<<stride_grid(n), kBlock, 0, s>>>(d_sortnnz, n, W, lidx.p, A->lvl_col.p, A->lvl_base.p,
                                                       A->lvl_tall.p, lvl_tiles.p, lvl_nnz.p);
        FL_LAUNCH_CHECK();
    }
    exclusive_scan_i32(lvl_tiles.p, A->lvl_tileoff.p, L, s, h.out(1));
    exclusive_scan_i32(lvl_nnz.p, A->lvl_nnzoff.p, L, s, h.out(2));
    const int T = h.wait()[1];
    const int total = h[2];
    if (total != nnz) {
        set_error("formatTransform: level table covers %d elements, expected nnz=%d", total, nnz);
        throw HipError{hipErrorInvalidValue};
    }
    A->tilenum = T;

    // tiles + data
    A->tile_ptr.alloc((size_t)T + 1);
    A->tile_len.alloc(std::max(T, 1));
    A->tile_colidx.alloc(std::max(T, 1));
    if (classify) A->tile_format.alloc(std::max(T, 1));
    TmpBuf<int> tile_depth(std::max(T, 1), s);
    if (!src.tiled) {
        A->sortrowidx.alloc(std::max(nnz, 1));
        A->val64.alloc(std::max(nnz, 1));
    }
    if (classify) A->sortrowindex.alloc(std::max(nnz, 1));
    if (T > 0) {
        k_tiles<<<stride_grid(T), kBlock, 0, s>>>(T, L, n, nnz, W, A->lvl_col.p, A->lvl_base.p, A->lvl_tall.p,
                                                  A->lvl_tileoff.p, A->lvl_nnzoff.p, A->tile_ptr.p, A->tile_len.p,
                                                  A->tile_colidx.p, tile_depth.p);
        FL_LAUNCH_CHECK();
        if (src.parent) {
            k_copy_tiles<<<stride_grid((long long)T * W), kBlock, 0, s>>>(
                T, W, A->tile_ptr.p, A->tile_len.p, A->tile_colidx.p, tile_depth.p, A->lvl_tileoff.p,
                levels_of(src.parent), src.parent->sortrowidx.p, src.parent->val64.p, L, A->sortrowidx.p, A->val64.p);
            FL_LAUNCH_CHECK();
        } else if (!src.tiled) {
            const WalkPlan plan(A, d_sortnnz, 0, s);
            k_fill_tiles<<<walk_grid(walk_bound(n, nnz, A->max_col_nnz)), kBlock, 0, s>>>(
                plan.w, levels_of(A), d_sortnnz, src.P, src.colptr, src.perm, src.rowidx, src.val, nnz, A->sortrowidx.p,
                A->val64.p);
            FL_LAUNCH_CHECK();
        }
    } else {
        FL_HIP(hipMemsetAsync(A->tile_ptr.p, 0, sizeof(int), s));
    }
    if (timed) FL_HIP(hipEventRecord(e1, s));

    // classification
    if (classify) {
        TmpBuf<int> seg_count(std::max(T, 1), s);
        A->countrow.alloc((size_t)T + 1);
        if (T > 0) {
            const unsigned g = grid_for(((long long)T + 64 / W * kClassTiles - 1) / (64 / W * kClassTiles) * 64);
            if (W == 32)
                k_classify<32><<<g, kBlock, 0, s>>>(T, A->tile_ptr.p, A->tile_len.p, A->sortrowidx.p, A->sortrowindex.p,
                                                    seg_count.p, A->tile_format.p);
            else
                k_classify<64><<<g, kBlock, 0, s>>>(T, A->tile_ptr.p, A->tile_len.p, A->sortrowidx.p, A->sortrowindex.p,
                                                    seg_count.p, A->tile_format.p);
            FL_LAUNCH_CHECK();
        }
        exclusive_scan_i32(seg_count.p, A->countrow.p, T, s, h.out(3));
        A->segsum = h.wait()[3];
        A->segmentoffset.alloc((size_t)A->segsum + 1);
        FL_HIP(hipMemsetAsync(A->segmentoffset.p + A->segsum, 0, sizeof(int), s));
        if (T > 0) {
            const unsigned g = grid_for(((long long)T + 64 / W * kClassTiles - 1) / (64 / W * kClassTiles) * 64);
            if (W == 32)
                k_segoff<32><<<g, kBlock, 0, s>>>(T, A->tile_ptr.p, A->tile_len.p, A->sortrowindex.p, A->countrow.p,
                                                  A->segmentoffset.p);
            else
                k_segoff<64><<<g, kBlock, 0, s>>>(T, A->tile_ptr.p, A->tile_len.p, A->sortrowindex.p, A->countrow.p,
                                                  A->segmentoffset.p);
            FL_LAUNCH_CHECK();
        }
    }
    if (timed) FL_HIP(hipEventRecord(e2, s));

    // group -> level hints for the FAST kernel
    const long long groups = ((long long)T + 63) / 64;
    A->group_level.alloc((size_t)std::max<long long>(groups, 1));
    if (groups > 0 && L > 0) {
        k_group_level<<<stride_grid(groups), kBlock, 0, s>>>(T, L, A->lvl_tileoff.p, A->group_level.p);
        FL_LAUNCH_CHECK();
    }
    if (!timed) return;
    FL_HIP(hipEventSynchronize(e2));
    FL_HIP(hipStreamSynchronize(s));
    float a = 0.f, b = 0.f;
    FL_HIP(hipEventElapsedTime(&a, e0, e1));
    FL_HIP(hipEventElapsedTime(&b, e1, e2));
    if (t_tran_ms) *t_tran_ms = a;
    if (t_clas_ms) *t_clas_ms = b;
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    (void)hipEventDestroy(e2);
}

}  // namespace fl
