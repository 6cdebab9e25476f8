// Internal helpers shared by the FastLoad HIP translation units (gfx950, wave64).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <cstdio>
#include <string>

#include "../../include/fastload.h"

// ---------------------------------------------------------------------------------- errors
namespace fl {

void set_error(const char *fmt, ...);

struct HipError {
    hipError_t err;
};

// The extent of an entry point, during which this thread's released temporaries wait for their stream.
struct TmpScope {
    TmpScope();
    ~TmpScope();
    TmpScope(const TmpScope &) = delete;
    TmpScope &operator=(const TmpScope &) = delete;
};

}  // namespace fl

#define FL_HIP(call)                                                                                  \
    do {                                                                                              \
        hipError_t fl_e_ = (call);                                                                    \
        if (fl_e_ != hipSuccess) {                                                                    \
            fl::set_error("%s:%d: %s failed: %s", __FILE__, __LINE__, #call, hipGetErrorString(fl_e_)); \
            throw fl::HipError{fl_e_};                                                                \
        }                                                                                             \
    } while (0)

#define FL_LAUNCH_CHECK() FL_HIP(hipGetLastError())

// Entry-point wrapper: converts thrown HIP errors / bad_alloc into status codes.
#define FL_API_BEGIN \
    try {            \
        fl::TmpScope fl_tmp_scope_;
#define FL_API_END                                                         \
    }                                                                      \
    catch (const fl::HipError &) { return FL_ERR_HIP; }                   \
    catch (const std::bad_alloc &) {                                       \
        fl::set_error("host allocation failed");                           \
        return FL_ERR_ALLOC;                                               \
    }                                                                      \
    catch (...) {                                                          \
        fl::set_error("unexpected exception");                             \
        return FL_ERR_INVALID;                                             \
    }

namespace fl {

constexpr int kWave = 64;
constexpr int kBlock = 256;  // 4 waves

inline int div_up(long long a, long long b) { return (int)((a + b - 1) / b); }

// A load with the nontemporal (streaming) cache hint, for data a kernel reads exactly once: the
// matrix's value and index streams, and products written by the previous kernel. Those lines
// are then the first to be evicted, so the L2 and the Infinity Cache keep what is reused (x, the
// products still to be read, the heavy part's y); on the power-law workload the HYB schedule's
// three kernels take 137 instead of 146 us with it. T is a 2-, 4-, 8- or 16-byte type.
template <typename T>
__device__ __forceinline__ T ld_stream(const T *p) {
    typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
    typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
    static_assert(sizeof(T) == 2 || sizeof(T) == 4 || sizeof(T) == 8 || sizeof(T) == 16, "ld_stream: size");
    T out;
    if constexpr (sizeof(T) == 16) {
        const u32x4 r = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(p));
        __builtin_memcpy(&out, &r, 16);
    } else if constexpr (sizeof(T) == 8) {
        const u32x2 r = __builtin_nontemporal_load(reinterpret_cast<const u32x2 *>(p));
        __builtin_memcpy(&out, &r, 8);
    } else if constexpr (sizeof(T) == 4) {
        const unsigned r = __builtin_nontemporal_load(reinterpret_cast<const unsigned *>(p));
        __builtin_memcpy(&out, &r, 4);
    } else {
        const unsigned short r = __builtin_nontemporal_load(reinterpret_cast<const unsigned short *>(p));
        __builtin_memcpy(&out, &r, 2);
    }
    return out;
}

// A store with the same hint, for data the kernel does not read again. T is 4 to 16 bytes.
template <typename T>
__device__ __forceinline__ void st_stream(T *p, const T &v) {
    typedef unsigned int W __attribute__((ext_vector_type(sizeof(T) / 4)));
    W w;
    __builtin_memcpy(&w, &v, sizeof(T));
    __builtin_nontemporal_store(w, reinterpret_cast<W *>(p));
}

inline unsigned grid_for(long long threads, int block = kBlock) { return (unsigned)((threads + block - 1) / block); }

// Device memory of the library's own objects (matrices, solvers, networks), kept for the next object
// when one is destroyed: on this runtime a hipFree of 160 MB takes 0.55 ms and a hipMalloc 0.06, and
// preparing a matrix of 10 M entries and dropping it spent 7 of its 19 ms in them.
//   - dev_block_put waits for the device, as hipFree does, so a kept block is idle: any stream and
//     any thread may get it next.
//   - A block serves requests of its own device of 7/8 of its size or more.
//   - At most kBlockKeep bytes are kept. The block that has waited longest goes first, and one that
//     kBlockAge later requests passed over goes too; when the device has no memory left, all
//     kept blocks are freed and the allocation is tried again.
constexpr unsigned long long kBlockKeep = 8ull << 30;
constexpr unsigned long long kBlockAge = 4096;
struct DevBlock {
    void *p = nullptr;
    size_t bytes = 0;
    int dev = 0;
};
DevBlock dev_block_get(size_t bytes);  // throws HipError
void dev_block_put(const DevBlock &b);
size_t dev_blocks_release();  // frees every kept block, returns their bytes

// RAII device buffer (a device block, put back on scope exit).
template <typename T>
struct DevBuf {
    T *p = nullptr;
    size_t count = 0;
    DevBuf() = default;
    explicit DevBuf(size_t c) { alloc(c); }
    void alloc(size_t c) {
        release();
        if (c) {
            block = dev_block_get(c * sizeof(T));
            p = (T *)block.p;
        }
        count = c;
    }
    void release() {
        if (p) dev_block_put(block);
        p = nullptr;
        count = 0;
    }
    ~DevBuf() { release(); }
    DevBuf(const DevBuf &) = delete;
    DevBuf &operator=(const DevBuf &) = delete;

  private:
    DevBlock block;
};

// Temporary device buffer of a preparation step on stream s. When it is released its kernels may still be
// running: the block goes to a list of this thread, for later temporaries on the same stream (which
// run after them), and to the kept blocks when the entry point ends (TmpScope), after the
// stream has been waited for.
DevBlock tmp_block_get(size_t bytes, hipStream_t s);
void tmp_block_put(const DevBlock &b, hipStream_t s);
template <typename T>
struct TmpBuf {
    T *p = nullptr;
    size_t count = 0;
    hipStream_t s = nullptr;
    explicit TmpBuf(hipStream_t st) : s(st) {}
    TmpBuf(size_t c, hipStream_t st) : s(st) { alloc(c); }
    void alloc(size_t c) {
        release();
        if (c) {
            block = tmp_block_get(c * sizeof(T), s);
            p = (T *)block.p;
        }
        count = c;
    }
    void release() {
        if (p) tmp_block_put(block, s);
        p = nullptr;
        count = 0;
    }
    ~TmpBuf() { release(); }
    TmpBuf(const TmpBuf &) = delete;
    TmpBuf &operator=(const TmpBuf &) = delete;

  private:
    DevBlock block;
};

// Up to kHostInts ints in pinned host memory, zero at first, for what a preparation step has to know on the
// host: kernels on stream s write them, wait() returns them after the stream. A copy of one int to
// ordinary memory costs a copy kernel and a wait of its own, 15 to 20 us; 46 of them took a quarter of the
// 2.9 ms that a new matrix of 8.8 M entries needs. The blocks are kept for later (one per thread in
// preparation, and never more than kHostBlocks idle ones).
constexpr int kHostInts = 256;
constexpr int kHostBlocks = 64;
class HostInts {
  public:
    explicit HostInts(hipStream_t st);
    ~HostInts();
    HostInts(const HostInts &) = delete;
    HostInts &operator=(const HostInts &) = delete;
    // for a kernel's argument: where int i goes
    int *out(int i = 0) {
        pending = true;
        return p + i;
    }
    const int *wait() {
        if (pending) FL_HIP(hipStreamSynchronize(s));
        pending = false;
        return p;
    }
    int operator[](int i) const { return p[i]; }  // after wait()

  private:
    int *p = nullptr;
    hipStream_t s;
    bool pending = false;
};

// ----------------------------------------------------------------- device-side primitives
// Exclusive prefix sum: out[0]=0, out[i]=sum(in[0..i-1]), out[count]=total. in may equal out
// only when in has count+1 entries. Returns nothing; total is on the device at out[count], and
// in *total (of a HostInts) when that is given.
void exclusive_scan_i32(const int *in, int *out, int count, hipStream_t s, int *total = nullptr);

// Stable LSD radix sort of (key, value) pairs by the low `bits` bits of key.
// keys/vals are sorted in place (ping-pong through internal scratch).
void radix_sort_pairs(uint32_t *keys, int *vals, int count, int bits, hipStream_t s);
// The same with the values 0 .. count - 1: order[i] = input position of the i-th key (order is output only).
// The keys come from in, which may be keys itself.
void radix_sort_positions(const uint32_t *in, uint32_t *keys, int *order, int count, int bits, hipStream_t s);

// Keys grouped by their top 8 bits [shift, shift + 8), and where each of the 256 groups starts.
void radix_partition(const uint32_t *keys, uint32_t *out, int count, int shift, int *start, hipStream_t s);

// start[b] = first position of a key >= b in the ascending keys, b in [0, nb] (start[nb] = count when all are below nb).
void key_bounds(const uint32_t *keys, int count, int nb, int *start, hipStream_t s);

// Device reduction helpers.
int device_max_i32(const int *in, int count, hipStream_t s);
// The same in two steps: the kernel, and the maximum after h.wait().
void max_i32_begin(const int *in, int count, HostInts &h, hipStream_t s);
// the same of in[i + 1] - in[i], i < count
void max_step_begin(const int *in, int count, HostInts &h, hipStream_t s);
int max_i32_end(const HostInts &h);
int bits_for(uint32_t v);

}  // namespace fl

// --------------------------------------------------------------- wave64 device helpers
namespace fl {

__device__ __forceinline__ int lane_id() { return (int)__lane_id(); }

// DPP move with compile-time control. old=0 for lanes outside row_mask or reading out of range.
template <int CTRL, int ROW_MASK = 0xf>
__device__ __forceinline__ int dpp_i32(int v) {
    return __builtin_amdgcn_update_dpp(0, v, CTRL, ROW_MASK, 0xf, false);
}

template <int CTRL, int ROW_MASK = 0xf>
__device__ __forceinline__ float dpp_f32(float v) {
    return __int_as_float(dpp_i32<CTRL, ROW_MASK>(__float_as_int(v)));
}

template <int CTRL, int ROW_MASK = 0xf>
__device__ __forceinline__ double dpp_f64(double v) {
    int2 a = *reinterpret_cast<int2 *>(&v);
    int2 r;
    r.x = dpp_i32<CTRL, ROW_MASK>(a.x);
    r.y = dpp_i32<CTRL, ROW_MASK>(a.y);
    return *reinterpret_cast<double *>(&r);
}

template <int CTRL, int ROW_MASK, typename T>
struct Dpp;
template <int CTRL, int ROW_MASK>
struct Dpp<CTRL, ROW_MASK, float> {
    static __device__ __forceinline__ float mov(float v) { return dpp_f32<CTRL, ROW_MASK>(v); }
};
template <int CTRL, int ROW_MASK>
struct Dpp<CTRL, ROW_MASK, double> {
    static __device__ __forceinline__ double mov(double v) { return dpp_f64<CTRL, ROW_MASK>(v); }
};
template <int CTRL, int ROW_MASK>
struct Dpp<CTRL, ROW_MASK, int> {
    static __device__ __forceinline__ int mov(int v) { return dpp_i32<CTRL, ROW_MASK>(v); }
};

// DPP control codes (GFX9 encoding).
constexpr int kRowShr1 = 0x111, kRowShr2 = 0x112, kRowShr4 = 0x114, kRowShr8 = 0x118;
constexpr int kRowBcast15 = 0x142, kRowBcast31 = 0x143, kWaveShr1 = 0x138;

// Segmented inclusive scan across the 64 lanes of a wave.
// start = index of the first lane of this lane's segment (start <= lane). On return each lane
// holds the sum of v over [start, lane]. All 64 lanes must execute this call (DPP reads other
// lanes' registers); lanes outside any tile should pass v = 0 and start = lane.
// In-row phase: row_shr 1,2,4,8 inside each 16-lane row; cross-row phase: row_bcast:15
// (lane 15 -> row 1, lane 47 -> row 3) then row_bcast:31 (lane 31 -> rows 2,3).
template <typename T>
__device__ __forceinline__ T wave_segscan(T v, int start, int lane) {
    const int lr = lane & 15;
    T t;
    t = Dpp<kRowShr1, 0xf, T>::mov(v);
    if (lr >= 1 && lane - 1 >= start) v += t;
    t = Dpp<kRowShr2, 0xf, T>::mov(v);
    if (lr >= 2 && lane - 2 >= start) v += t;
    t = Dpp<kRowShr4, 0xf, T>::mov(v);
    if (lr >= 4 && lane - 4 >= start) v += t;
    t = Dpp<kRowShr8, 0xf, T>::mov(v);
    if (lr >= 8 && lane - 8 >= start) v += t;
    t = Dpp<kRowBcast15, 0xa, T>::mov(v);
    if ((lane & 16) && start <= (lane & ~15) - 1) v += t;
    t = Dpp<kRowBcast31, 0xc, T>::mov(v);
    if ((lane & 32) && start <= 31) v += t;
    return v;
}

// Plain inclusive wave scan of ints (segment = whole wave).
__device__ __forceinline__ int wave_inclusive_scan(int v) { return wave_segscan<int>(v, 0, (int)__lane_id()); }

// Start lane of the segment containing `lane`, given the 64-bit mask of segment heads.
__device__ __forceinline__ int segment_start(uint64_t heads, int lane) {
    const uint64_t upto = (lane == 63) ? ~0ull : ((2ull << lane) - 1ull);
    return 63 - __clzll((long long)(heads & upto));
}

__device__ __forceinline__ uint64_t ballot64(bool p) { return (uint64_t)__ballot(p); }

}  // namespace fl
