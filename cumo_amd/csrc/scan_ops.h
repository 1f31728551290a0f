// What the scan kernels share: the operators, the description of many runs, lanes of a wave talking to each other.
#ifndef CUMO_HIP_SCAN_OPS_H
#define CUMO_HIP_SCAN_OPS_H

#include "common.h"

namespace cumo_hip {
namespace {

template <class T> __device__ __forceinline__ bool scan_is_nan(T x) { return x != x; }
template <> __device__ __forceinline__ bool scan_is_nan<int32_t>(int32_t) { return false; }

template <class T> struct scan_is_int { static constexpr bool value = false; };
template <> struct scan_is_int<int32_t> { static constexpr bool value = true; };

// OP: 0 sum, 1 prod. NANF: NaN is skipped.
template <class T, int OP, bool NANF>
struct ScanOp {
    __device__ __forceinline__ static T apply(T a, T b) {
        if (NANF) {
            if (scan_is_nan(a)) return b;
            if (scan_is_nan(b)) return a;
        }
        if constexpr (scan_is_int<T>::value) {
            // Int32: wrapping arithmetic done in unsigned
            return OP == 0 ? (T)((uint32_t)a + (uint32_t)b) : (T)((uint32_t)a * (uint32_t)b);
        } else {
            return OP == 0 ? a + b : a * b;
        }
    }
};

// sixteen bytes of a run
template <class T>
struct ScanVec {
    typedef uint32_t u4 __attribute__((ext_vector_type(4)));
    static constexpr int V = 16 / (int)sizeof(T);
    union { u4 q; T e[V]; };
};

// many runs of n elements: where each starts (outer dimensions), and the byte step along it
struct ScanRowsParams {
    int nouter;
    uint64_t rows, n;
    uint64_t oshape[CUMO_NA_MAX_DIMENSION];
    int64_t ostep_in[CUMO_NA_MAX_DIMENSION], ostep_out[CUMO_NA_MAX_DIMENSION];
    int64_t s_in, s_out;
    const char* in;
    char* out;
    bool through;   // see StoreRows (scan_rows_whole_kernel)
};

// where run `row` starts on either side, in bytes from the first one
__device__ __forceinline__ void scan_run_offsets(const ScanRowsParams& p, uint64_t row, int64_t& oi, int64_t& oo) {
    oi = oo = 0;
#pragma unroll 1
    for (int d = p.nouter - 1; d >= 0; --d) {
        const uint64_t m = p.oshape[d];
        const uint64_t q = row / m;
        const int64_t k = (int64_t)(row - q * m);
        row = q;
        oi += k * p.ostep_in[d];
        oo += k * p.ostep_out[d];
    }
}
__device__ __forceinline__ void scan_run_start(const ScanRowsParams& p, uint64_t row, const char*& in, char*& out) {
    int64_t oi, oo;
    scan_run_offsets(p, row, oi, oo);
    in = p.in + oi;
    out = p.out + oo;
}

// v of another lane by data-parallel primitive (no trip through the LDS unit that shuffles take); lanes without a source keep their own
template <int CTRL, class T>
__device__ __forceinline__ T scan_dpp(T v) {
    constexpr int W = (int)(sizeof(T) / 4);
    union { T t; int w[W]; } a, b;
    a.t = v;
#pragma unroll
    for (int i = 0; i < W; ++i) b.w[i] = __builtin_amdgcn_update_dpp(a.w[i], a.w[i], CTRL, 0xf, 0xf, false);
    return b.t;
}

// v of one lane, the same lane for the whole wave
template <class T>
__device__ __forceinline__ T scan_read_lane(T v, uint32_t lane) {
    constexpr int W = (int)(sizeof(T) / 4);
    union { T t; int w[W]; } a;
    a.t = v;
#pragma unroll
    for (int i = 0; i < W; ++i) a.w[i] = __builtin_amdgcn_readlane(a.w[i], (int)lane);
    return a.t;
}

}  // namespace

// scan_short.hip: runs of up to 4 KiB, as many to a wave as it holds. False when they are not what it takes; nothing is launched then.
bool scan_short_launch(int type, int prod, int nan, const cumo_hip_scan_rows_t* d);

}  // namespace cumo_hip

#endif
