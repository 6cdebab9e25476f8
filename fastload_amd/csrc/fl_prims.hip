// Device primitives for the preprocessing pipeline: exclusive scan, stable LSD radix sort of
// (key, index) pairs, max reduction. These replace the reference's CUB DeviceScan calls
// (src/formatTransform_GPU.h:402-496) and thrust::sort_by_key (src/ColSort_GPU.h:101).
#include <algorithm>
#include <atomic>
#include <cstdarg>
#include <map>
#include <mutex>
#include <vector>

#include "fl_common.h"

namespace fl {

// --------------------------------------------------------------------------------- scan
// A scan is bound by its launches: the largest of a preparation, 8.8 M flags, moves 105 MB in 23 us, most have
// below 100 K elements, and a launch and the gap before it take about 5 us. One workgroup scans up to
// kScanSmall elements; above that the tiles' sums are one launch, and each tile then adds up the sums before
// its own itself, instead of a third launch that scans them (up to kScanTiles tiles; 4,096 sums are 16 loads per
// thread). A radix pass: 5 launches -> 4, and 3 for up to 262,144 keys.
constexpr int kScanItems = 8;
constexpr int kScanTile = kBlock * kScanItems;  // 2048 elements per block
constexpr int kScanTiles = 4096;
constexpr int kScanBig = 1024, kScanBigItems = 16;
constexpr int kScanSmall = kScanBig * kScanBigItems;

template <int NT>
__device__ __forceinline__ int block_exclusive_scan(int v, int *lds_wave, int &block_total) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int incl = wave_inclusive_scan(v);
    if (lane == 63) lds_wave[w] = incl;
    __syncthreads();
    int prefix = 0, total = 0;
#pragma unroll
    for (int i = 0; i < NT / kWave; ++i) {
        const int x = lds_wave[i];
        prefix += (i < w) ? x : 0;
        total += x;
    }
    block_total = total;
    return prefix + incl - v;
}

// ITEMS consecutive elements from i on, 0 past count; 16 bytes at a time where all are there and in is aligned
template <int ITEMS>
__device__ __forceinline__ void scan_load(const int *__restrict__ in, long long i, int count, int *v) {
    if (i + ITEMS <= count && (reinterpret_cast<uintptr_t>(in) & 15) == 0) {
#pragma unroll
        for (int k = 0; k < ITEMS; k += 4) {
            const int4 q = *reinterpret_cast<const int4 *>(in + i + k);
            v[k] = q.x, v[k + 1] = q.y, v[k + 2] = q.z, v[k + 3] = q.w;
        }
    } else {
#pragma unroll
        for (int k = 0; k < ITEMS; ++k) v[k] = (i + k < count) ? in[i + k] : 0;
    }
}

__global__ __launch_bounds__(kBlock) void k_tile_sums(const int *__restrict__ in, int count, int *__restrict__ partial) {
    __shared__ int lds_wave[kBlock / kWave];
    const long long base = (long long)blockIdx.x * kScanTile + (long long)threadIdx.x * kScanItems;
    int v[kScanItems], s = 0;
    scan_load<kScanItems>(in, base, count, v);
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) s += v[k];
    int total;
    (void)block_exclusive_scan<kBlock>(s, lds_wave, total);
    if (threadIdx.x == 0) partial[blockIdx.x] = total;
}

// sums: the tiles' sums, scanned (SCANNED) or as they are; null with one tile. host: also gets the total, or null.
template <int NT, int ITEMS, bool SCANNED>
__global__ __launch_bounds__(NT) void k_scan_tiles(const int *__restrict__ in, int *__restrict__ out, int count,
                                                   const int *__restrict__ sums, int *__restrict__ host) {
    __shared__ int lds_wave[NT / kWave], lds_carry[NT / kWave];
    const long long base = ((long long)blockIdx.x * NT + threadIdx.x) * ITEMS;
    int v[ITEMS], s = 0;
    scan_load<ITEMS>(in, base, count, v);
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) s += v[k];
    int carry = 0;
    if (SCANNED) {
        carry = sums[blockIdx.x];
    } else if (sums) {
        int c = 0;
        for (int i = threadIdx.x; i < (int)blockIdx.x; i += NT) c += sums[i];
        (void)block_exclusive_scan<NT>(c, lds_carry, carry);
    }
    int total;
    const int excl = block_exclusive_scan<NT>(s, lds_wave, total);
    int run = carry + excl;
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
        const int t = v[k];
        v[k] = run;
        run += t;
    }
    if (base + ITEMS <= count && (reinterpret_cast<uintptr_t>(out) & 15) == 0) {
#pragma unroll
        for (int k = 0; k < ITEMS; k += 4)
            *reinterpret_cast<int4 *>(out + base + k) = make_int4(v[k], v[k + 1], v[k + 2], v[k + 3]);
    } else {
#pragma unroll
        for (int k = 0; k < ITEMS; ++k)
            if (base + k < count) out[base + k] = v[k];
    }
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) {
        out[count] = carry + total;
        if (host) *host = carry + total;
    }
}

void exclusive_scan_i32(const int *in, int *out, int count, hipStream_t s, int *total) {
    if (count <= 0) {
        FL_HIP(hipMemsetAsync(out, 0, sizeof(int), s));
        return;
    }
    const int nb = div_up(count, kScanTile);
    if (count <= kScanSmall) {
        if (nb == 1) k_scan_tiles<kBlock, kScanItems, false><<<1, kBlock, 0, s>>>(in, out, count, nullptr, total);
        else k_scan_tiles<kScanBig, kScanBigItems, false><<<1, kScanBig, 0, s>>>(in, out, count, nullptr, total);
        FL_LAUNCH_CHECK();
        return;
    }
    TmpBuf<int> partial(nb, s);
    k_tile_sums<<<nb, kBlock, 0, s>>>(in, count, partial.p);
    FL_LAUNCH_CHECK();
    if (nb <= kScanTiles) {
        k_scan_tiles<kBlock, kScanItems, false><<<nb, kBlock, 0, s>>>(in, out, count, partial.p, total);
        FL_LAUNCH_CHECK();
        return;
    }
    TmpBuf<int> partial_scan((size_t)nb + 1, s);
    exclusive_scan_i32(partial.p, partial_scan.p, nb, s);
    k_scan_tiles<kBlock, kScanItems, true><<<nb, kBlock, 0, s>>>(in, out, count, partial_scan.p, total);
    FL_LAUNCH_CHECK();
}

// ------------------------------------------------------------------------------ ints read by the host
namespace {
struct HostBlocks {
    std::mutex mu;
    std::vector<int *> idle;
};
// never destroyed: see block_store
HostBlocks &host_blocks() {
    static HostBlocks &b = *new HostBlocks();
    return b;
}
}  // namespace

HostInts::HostInts(hipStream_t st) : s(st) {
    {
        HostBlocks &b = host_blocks();
        std::lock_guard<std::mutex> g(b.mu);
        if (!b.idle.empty()) {
            p = b.idle.back();
            b.idle.pop_back();
        }
    }
    if (!p) FL_HIP(hipHostMalloc((void **)&p, sizeof(int) * kHostInts, hipHostMallocPortable));
    std::fill_n(p, kHostInts, 0);
}

HostInts::~HostInts() {
    // kernels may still be writing when an error took the caller past its wait
    bool keep = !pending || hipStreamSynchronize(s) == hipSuccess;
    if (keep) {
        HostBlocks &b = host_blocks();
        std::lock_guard<std::mutex> g(b.mu);
        keep = b.idle.size() < (size_t)kHostBlocks;
        if (keep) try {
                b.idle.push_back(p);
            } catch (...) {
                keep = false;
            }
    }
    if (!keep) (void)hipHostFree(p);
}

// ------------------------------------------------------------------------------ max-reduce
// One value per workgroup, at most kHostInts workgroups, and the host takes the largest.
template <bool STEP>
__global__ __launch_bounds__(kBlock) void k_max_i32(const int *__restrict__ in, int count, int *__restrict__ out) {
    __shared__ int part[kBlock / kWave];
    int m = 0;
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += (long long)gridDim.x * blockDim.x)
        m = max(m, STEP ? in[i + 1] - in[i] : in[i]);
    for (int off = 32; off > 0; off >>= 1) m = max(m, __shfl_xor(m, off));
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kBlock / kWave; ++w) m = max(m, part[w]);
        out[blockIdx.x] = m;
    }
}

template <bool STEP>
static void max_begin(const int *in, int count, HostInts &h, hipStream_t s) {
    if (count <= 0) return;
    const unsigned g = std::min<unsigned>(grid_for(count), (unsigned)kHostInts);
    k_max_i32<STEP><<<g, kBlock, 0, s>>>(in, count, h.out());
    FL_LAUNCH_CHECK();
}

void max_i32_begin(const int *in, int count, HostInts &h, hipStream_t s) { max_begin<false>(in, count, h, s); }

void max_step_begin(const int *in, int count, HostInts &h, hipStream_t s) { max_begin<true>(in, count, h, s); }

int max_i32_end(const HostInts &h) {
    int m = 0;
    for (int i = 0; i < kHostInts; ++i) m = std::max(m, h[i]);
    return m;
}

int device_max_i32(const int *in, int count, hipStream_t s) {
    if (count <= 0) return 0;
    HostInts h(s);
    max_i32_begin(in, count, h, s);
    (void)h.wait();
    return max_i32_end(h);
}

int bits_for(uint32_t v) {
    int b = 0;
    while (b < 32 && (v >> b) != 0) ++b;
    return b;
}

// ------------------------------------------------------------------------ radix sort
// One 8-bit LSD pass = histogram per block -> scan (digit-major) -> stable scatter.
// Block tile: kSortRounds rounds of 256 keys in index order; inside a round the rank of a key
// among equal digits is (earlier waves' counts) + (lower lanes of its wave with that digit),
// the latter from a ballot-based match over the 8 digit bits. The scatter stages the tile in
// LDS in digit order before writing it out.
constexpr int kRadixBits = 8;
constexpr int kRadix = 1 << kRadixBits;
constexpr int kSortRounds = 16;
constexpr int kSortTile = kBlock * kSortRounds;  // 4096 keys per block

// The tile of this workgroup: the workgroups of an XCD (blockIdx % 8) take consecutive tiles, so the counts of
// neighbouring tiles, next to each other in the digit-major histogram, and the ends of their runs in the
// output are completed in one L2. The grid is a multiple of 8; tiles from nblocks on do not exist.
__device__ __forceinline__ int sort_tile() { return (int)((blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3)); }
static unsigned sort_grid(int nblocks) { return ((unsigned)nblocks + 7u) & ~7u; }

// 7.4 M keys: 11 us (12 to 17 with tiles dealt out in turn and a load at a time).
__global__ __launch_bounds__(kBlock) void k_radix_hist(const uint32_t *__restrict__ keys, int count, int shift,
                                                       int nblocks, int *__restrict__ hist) {
    __shared__ int cnt[kRadix];
    const int b = sort_tile();
    if (b >= nblocks) return;
    cnt[threadIdx.x] = 0;
    const long long base = (long long)b * kSortTile + threadIdx.x;
    uint32_t key[kSortRounds];
#pragma unroll
    for (int r = 0; r < kSortRounds; ++r) key[r] = base + r * kBlock < count ? keys[base + r * kBlock] : 0u;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kSortRounds; ++r) {
        const bool valid = base + r * kBlock < count;
        const int d = (int)((key[r] >> shift) & (kRadix - 1));
        // the high digits of nearly sorted keys are the same in a whole wave: one add instead of 64 in turn
        const uint64_t all = ballot64(valid);
        if (all == ballot64(valid && d == __builtin_amdgcn_readfirstlane(d))) {
            if (all && (threadIdx.x & 63) == 0) atomicAdd(&cnt[d], __popcll(all));
        } else if (valid) {
            atomicAdd(&cnt[d], 1);
        }
    }
    __syncthreads();
    hist[(long long)threadIdx.x * nblocks + b] = cnt[threadIdx.x];
}

// The tile's keys are first placed in LDS in (digit, input order) order, each at its digit's
// local offset plus its stable rank; then they are written out from LDS position i to
// global_base[d] + (i - local_base[d]): consecutive threads write consecutive positions of one
// digit's run, instead of every key going straight to one of 256 scattered buckets. The tile's
// digit counts are the differences of the scanned histogram (offsets).
// Each wave ranks its own 1,024 consecutive keys: in a round of 64 the lowest lane of each digit adds the
// number of its peers to the wave's counter of the digit and hands the old value to them. The rounds'
// adds are in order, so the ranks are stable, and nothing waits for another wave until all are ranked.
// 7.4 M pairs: 33 us, 3.6 TB/s (62 with rounds of 256 keys and the waves' counts put together after each, three
// barriers a round; 49 with the tiles dealt to the XCDs in turn). The old value is handed on inside the round:
// kept for a second loop, its lanes' masks took the kernel past 256 registers.
// PAIRS: the values move with the keys (vals_in null: the values are the input positions); else keys alone
// (vals_in and vals_out unused).
template <bool PAIRS>
__global__ __launch_bounds__(kBlock, 4) void k_radix_scatter(const uint32_t *__restrict__ keys_in,
                                                          const int *__restrict__ vals_in,
                                                          uint32_t *__restrict__ keys_out, int *__restrict__ vals_out,
                                                          int count, int shift, int nblocks,
                                                          const int *__restrict__ offsets) {
    static_assert(kRadix == kBlock, "one digit per thread");
    constexpr int kWaves = kBlock / kWave;
    __shared__ uint32_t skey[kSortTile];
    __shared__ int sval[PAIRS ? kSortTile : 1];
    __shared__ int lbase[kRadix], gbase[kRadix];
    __shared__ int wsum[kWaves];
    __shared__ int wcnt[kWaves][kRadix];  // the wave's keys per digit, then where they start in the tile
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, b = sort_tile();
    if (b >= nblocks) return;
    const long long tile = (long long)b * kSortTile;
    const long long first = tile + (long long)w * kWave * kSortRounds + lane;
    uint32_t key[kSortRounds];
    int val[kSortRounds], old[kSortRounds];
#pragma unroll
    for (int r = 0; r < kSortRounds; ++r) {
        const long long i = first + r * kWave;
        key[r] = i < count ? keys_in[i] : 0u;
        if constexpr (PAIRS) val[r] = !vals_in ? (int)i : i < count ? vals_in[i] : 0;
    }
    const long long idx = (long long)threadIdx.x * nblocks + b;
    const int g = offsets[idx];
    const int c = offsets[idx + 1] - g;  // keys of digit threadIdx.x in this tile
    for (int q = 0; q < kWaves; ++q) wcnt[q][threadIdx.x] = 0;
    __syncthreads();
    const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
#pragma unroll
    for (int r = 0; r < kSortRounds; ++r) {
        const bool valid = first + r * kWave < count;
        const int d = (int)((key[r] >> shift) & (kRadix - 1));
        uint64_t peers = ballot64(valid);
#pragma unroll
        for (int k = 0; k < kRadixBits; ++k) {
            const bool bit = (d >> k) & 1;
            const uint64_t m = ballot64(bit);
            peers &= bit ? m : ~m;
        }
        const int rank = __popcll(peers & lt_mask);
        int o = 0;
        if (valid && rank == 0) o = atomicAdd(&wcnt[w][d], __popcll(peers));
        old[r] = __shfl(o, valid ? __ffsll((unsigned long long)peers) - 1 : lane, 64) + rank;
    }
    {
        gbase[threadIdx.x] = g;
        // exclusive scan of the 256 counts: inside each wave, then across the 4 waves
        const int v = wave_inclusive_scan(c);
        if (lane == 63) wsum[w] = v;
        __syncthreads();
        int before = v - c;
        for (int q = 0; q < w; ++q) before += wsum[q];
        lbase[threadIdx.x] = before;
        for (int q = 0; q < kWaves; ++q) {
            const int t = wcnt[q][threadIdx.x];
            wcnt[q][threadIdx.x] = before;
            before += t;
        }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kSortRounds; ++r) {
        if (first + r * kWave < count) {
            const int pos = wcnt[w][(key[r] >> shift) & (kRadix - 1)] + old[r];
            skey[pos] = key[r];
            if constexpr (PAIRS) sval[pos] = val[r];
        }
    }
    __syncthreads();
    const int n_tile = (int)min((long long)kSortTile, (long long)count - tile);
    for (int i = threadIdx.x; i < n_tile; i += kBlock) {
        const uint32_t k = skey[i];
        const int d = (int)((k >> shift) & (kRadix - 1));
        const int o = gbase[d] + (i - lbase[d]);
        keys_out[o] = k;
        if constexpr (PAIRS) vals_out[o] = sval[i];
    }
}

__global__ void k_positions(int *__restrict__ v, int count) {
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += (long long)gridDim.x * blockDim.x)
        v[i] = (int)i;
}

__global__ void k_copy_pairs(const uint32_t *__restrict__ k, const int *__restrict__ v, uint32_t *__restrict__ keys,
                             int *__restrict__ vals, int count) {
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += (long long)gridDim.x * blockDim.x) {
        keys[i] = k[i];
        vals[i] = v[i];
    }
}

// in: the keys, in another array than `keys` or in it. From another array the passes alternate between the scratch pair
// and the caller's arrays so that the last one ends there; in place that takes a third pair for an odd
// number of passes, and a copy for a single one.
static void sort_pairs(const uint32_t *in, uint32_t *keys, int *vals, int count, int bits, bool positions, hipStream_t s) {
    const bool inplace = in == keys;
    if (count <= 1 || bits <= 0) {
        if (positions && count > 0) {
            k_positions<<<std::min(grid_for(count), 65536u), kBlock, 0, s>>>(vals, count);
            FL_LAUNCH_CHECK();
        }
        if (!inplace && count > 0)
            FL_HIP(hipMemcpyAsync(keys, in, sizeof(uint32_t) * (size_t)count, hipMemcpyDeviceToDevice, s));
        return;
    }
    const int nb = div_up(count, kSortTile);
    const long long hcount = (long long)nb * kRadix;
    if (hcount > 0x7fffffffLL) {
        set_error("radix sort: histogram too large");
        throw HipError{hipErrorInvalidValue};
    }
    TmpBuf<int> hist((size_t)hcount, s), offs((size_t)hcount + 1, s);
    const int passes = (bits + kRadixBits - 1) / kRadixBits;
    const bool third = inplace && passes >= 3 && passes % 2 == 1;
    const bool scratch = inplace || passes > 1;
    TmpBuf<uint32_t> k2(scratch ? count : 0, s), k3(third ? count : 0, s);
    TmpBuf<int> v2(scratch ? count : 0, s), v3(third ? count : 0, s);
    const uint32_t *kin = in;
    const int *vin = vals;
    for (int p = 0; p < passes; ++p) {
        const int shift = p * kRadixBits;
        uint32_t *kout = (passes - 1 - p) % 2 == 0 ? keys : k2.p;
        int *vout = (passes - 1 - p) % 2 == 0 ? vals : v2.p;
        if (third && p == 1) kout = k3.p, vout = v3.p;
        if (inplace && p == 0) kout = k2.p, vout = v2.p;
        k_radix_hist<<<sort_grid(nb), kBlock, 0, s>>>(kin, count, shift, nb, hist.p);
        FL_LAUNCH_CHECK();
        exclusive_scan_i32(hist.p, offs.p, (int)hcount, s);
        k_radix_scatter<true><<<sort_grid(nb), kBlock, 0, s>>>(kin, positions && p == 0 ? nullptr : vin, kout, vout, count, shift, nb, offs.p);
        FL_LAUNCH_CHECK();
        kin = kout;
        vin = vout;
    }
    if (kin != keys) {  // one pass in place
        k_copy_pairs<<<std::min(grid_for(count), 65536u), kBlock, 0, s>>>(kin, vin, keys, vals, count);
        FL_LAUNCH_CHECK();
    }
    // no wait here: the temporaries are freed in stream order, and the caller's later work on s
    // (or its own readback) comes after the sort
}

void radix_sort_pairs(uint32_t *keys, int *vals, int count, int bits, hipStream_t s) {
    sort_pairs(keys, keys, vals, count, bits, false, s);
}

void radix_sort_positions(const uint32_t *in, uint32_t *keys, int *order, int count, int bits, hipStream_t s) {
    sort_pairs(in, keys, order, count, bits, true, s);
}

__global__ void k_bin_starts(const int *__restrict__ offs, int nblocks, int count, int *__restrict__ start) {
    start[threadIdx.x] = threadIdx.x < kRadix ? offs[(long long)threadIdx.x * nblocks] : count;
}

// out = keys grouped by bits [shift, shift + 8) in ascending order (keys above them must be zero), start[b]
// = first position of group b (257 entries).
void radix_partition(const uint32_t *keys, uint32_t *out, int count, int shift, int *start, hipStream_t s) {
    const int nb = std::max(1, div_up(count, kSortTile));
    const long long hcount = (long long)nb * kRadix;
    if (hcount > 0x7fffffffLL) {
        set_error("radix partition: histogram too large");
        throw HipError{hipErrorInvalidValue};
    }
    TmpBuf<int> hist((size_t)hcount, s), offs((size_t)hcount + 1, s);
    k_radix_hist<<<sort_grid(nb), kBlock, 0, s>>>(keys, count, shift, nb, hist.p);
    FL_LAUNCH_CHECK();
    exclusive_scan_i32(hist.p, offs.p, (int)hcount, s);
    k_radix_scatter<false><<<sort_grid(nb), kBlock, 0, s>>>(keys, nullptr, out, nullptr, count, shift, nb, offs.p);
    k_bin_starts<<<1, kRadix + 1, 0, s>>>(offs.p, nb, count, start);
    FL_LAUNCH_CHECK();
}

// ------------------------------------------------------------------------------ key bounds
// A search for every b, two to a thread so that the loads of one hide those of the other. Bound by the chain of
// dependent loads. A thread per key that writes the b up to the next key takes less where every b has keys
// (2 M of 55 M keys: 84 us against 108; 600 K of 7.4 M: 17 and 15) but writes a run of b without keys alone:
// 100 ms for 4 M of them at the end, here 59 us for all 8 M. One search to a thread: 83, 19 and 101 us.
__global__ void k_key_bounds(const uint32_t *__restrict__ keys, int count, int nb, int *__restrict__ start) {
    constexpr int U = 2;
    const long long total = (long long)nb + 1;
    for (long long b = (long long)blockIdx.x * (kBlock * U) + threadIdx.x; b < total; b += (long long)gridDim.x * (kBlock * U)) {
        int at[U] = {};
        for (int len = count; len > 0;) {  // the answers are in [at, at + len]
            const int half = (len + 1) / 2;
            uint32_t k[U];
#pragma unroll
            for (int u = 0; u < U; ++u) k[u] = keys[at[u] + half - 1];
#pragma unroll
            for (int u = 0; u < U; ++u) at[u] += (long long)k[u] < b + u * kBlock ? half : 0;
            len -= half;
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (b + u * kBlock < total) start[b + u * kBlock] = at[u];
    }
}

void key_bounds(const uint32_t *keys, int count, int nb, int *start, hipStream_t s) {
    k_key_bounds<<<std::min(grid_for((long long)nb + 1, kBlock * 2), 65536u), kBlock, 0, s>>>(keys, count, nb, start);
    FL_LAUNCH_CHECK();
}

// --------------------------------------------------------------------- kept device blocks
namespace {
struct Kept {
    void *p;
    unsigned long long since;  // requests made when it was put back
};
struct BlockStore {
    std::mutex mu;
    std::multimap<std::pair<int, size_t>, Kept> blocks;  // by (device, bytes)
    unsigned long long held = 0, requests = 0;
};
// never destroyed: objects may be released while the process ends
BlockStore &block_store() {
    static BlockStore &b = *new BlockStore();
    return b;
}

size_t block_size(size_t bytes) {
    const size_t grain = bytes < (1u << 20) ? 256 : 1u << 16;
    return (bytes + grain - 1) / grain * grain;
}

// whether a block serves a request of `want` bytes (a block_size)
bool block_fits(size_t bytes, size_t want) { return bytes >= want && bytes - bytes / 8 <= want; }

// Takes the blocks that have waited longest out of the store until `room` more bytes fit, and those past
// kBlockAge; the caller frees them without the lock.
std::vector<void *> drop_blocks(BlockStore &b, unsigned long long room) {
    std::vector<void *> out;
    while (!b.blocks.empty()) {
        auto oldest = b.blocks.begin();
        for (auto it = b.blocks.begin(); it != b.blocks.end(); ++it)
            if (it->second.since < oldest->second.since) oldest = it;
        if (b.held + room <= kBlockKeep && b.requests - oldest->second.since <= kBlockAge) break;
        out.push_back(oldest->second.p);
        b.held -= oldest->first.second;
        b.blocks.erase(oldest);
    }
    return out;
}

// Keeps an idle block.
void keep_block(const DevBlock &d) {
    if (d.bytes > kBlockKeep / 2) {
        (void)hipFree(d.p);
        return;
    }
    BlockStore &b = block_store();
    std::vector<void *> out;
    try {
        std::lock_guard<std::mutex> g(b.mu);
        out = drop_blocks(b, d.bytes);
        b.blocks.emplace(std::make_pair(d.dev, d.bytes), Kept{d.p, b.requests});
        b.held += d.bytes;
    } catch (...) {  // no host memory to note it (called from destructors)
        (void)hipFree(d.p);
    }
    for (void *p : out) (void)hipFree(p);
}

// This thread's released temporaries, whose kernels may still run.
struct Pending {
    DevBlock block;
    hipStream_t s;
};
thread_local std::vector<Pending> t_pending;
thread_local int t_depth = 0;

// Waits for the temporaries' streams, then keeps the blocks (keep) or frees them.
void settle_pending(bool keep) {
    std::vector<Pending> done;
    done.swap(t_pending);
    for (size_t i = 0; i < done.size(); ++i) {
        bool waited = false;  // for this stream
        for (size_t k = 0; k < i && !waited; ++k) waited = done[k].s == done[i].s;
        if (!waited && hipStreamSynchronize(done[i].s) != hipSuccess) {
            (void)hipGetLastError();
            keep = false;
        }
    }
    for (const Pending &q : done) {
        if (keep) keep_block(q.block);
        else (void)hipFree(q.block.p);
    }
}
}  // namespace

size_t dev_blocks_release() {
    BlockStore &b = block_store();
    std::vector<void *> out;
    size_t bytes = 0;
    {
        std::lock_guard<std::mutex> g(b.mu);
        for (auto &k : b.blocks) out.push_back(k.second.p);
        bytes = (size_t)b.held;
        b.blocks.clear();
        b.held = 0;
    }
    for (void *p : out) (void)hipFree(p);
    return bytes;
}

DevBlock dev_block_get(size_t bytes) {
    DevBlock d;
    FL_HIP(hipGetDevice(&d.dev));
    d.bytes = block_size(bytes);
    BlockStore &b = block_store();
    {
        std::lock_guard<std::mutex> g(b.mu);
        ++b.requests;
        auto it = b.blocks.lower_bound({d.dev, d.bytes});
        if (it != b.blocks.end() && it->first.first == d.dev && block_fits(it->first.second, d.bytes)) {
            d.p = it->second.p;
            d.bytes = it->first.second;
            b.held -= d.bytes;
            b.blocks.erase(it);
            return d;
        }
    }
    if (hipMalloc(&d.p, d.bytes) != hipSuccess) {
        (void)hipGetLastError();
        dev_blocks_release();
        if (hipMalloc(&d.p, d.bytes) != hipSuccess) {
            (void)hipGetLastError();
            settle_pending(false);
            d.p = nullptr;
            FL_HIP(hipMalloc(&d.p, d.bytes));
        }
    }
    return d;
}

void dev_block_put(const DevBlock &d) {
    int cur = d.dev;
    (void)hipGetDevice(&cur);
    if (cur != d.dev) (void)hipSetDevice(d.dev);
    const bool idle = hipDeviceSynchronize() == hipSuccess;  // not while this thread captures, or after a fault
    if (cur != d.dev) (void)hipSetDevice(cur);
    if (!idle) {
        (void)hipGetLastError();
        (void)hipFree(d.p);
        return;
    }
    keep_block(d);
}

DevBlock tmp_block_get(size_t bytes, hipStream_t s) {
    const size_t want = block_size(bytes);
    int dev = 0;
    FL_HIP(hipGetDevice(&dev));
    size_t best = t_pending.size();
    for (size_t i = 0; i < t_pending.size(); ++i) {
        const Pending &q = t_pending[i];
        if (q.s == s && q.block.dev == dev && block_fits(q.block.bytes, want) &&
            (best == t_pending.size() || q.block.bytes < t_pending[best].block.bytes))
            best = i;
    }
    if (best < t_pending.size()) {
        const DevBlock d = t_pending[best].block;
        t_pending[best] = t_pending.back();
        t_pending.pop_back();
        return d;
    }
    return dev_block_get(bytes);
}

void tmp_block_put(const DevBlock &d, hipStream_t s) {
    if (t_depth > 0) {
        try {
            t_pending.push_back({d, s});
            return;
        } catch (...) {
        }
    }
    dev_block_put(d);
}

TmpScope::TmpScope() { ++t_depth; }

TmpScope::~TmpScope() {
    if (--t_depth == 0 && !t_pending.empty()) settle_pending(true);
}

// ------------------------------------------------------------------------------- errors
static thread_local char g_err[512] = {0};

void set_error(const char *fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof g_err, fmt, ap);
    va_end(ap);
}

}  // namespace fl

extern "C" const char *fl_last_error(void) { return fl::g_err; }
