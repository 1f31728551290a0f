// Row-wise composites that a Cumo program writes as a chain of array operations,
// done in one pass over each row:
//
//   softmax     m = x.max(axis:-1, keepdims:true); e = NMath.exp(x - m); e / e.sum(axis:-1, keepdims:true)
//   layernorm   (x - x.mean(axis:-1, keepdims:true)) / NMath.sqrt(x.var(axis:-1, keepdims:true) + eps)
//
// (the shapes of bench/transformer_bench.rb:110-124 of the reference). As separate
// launches the first moves 9 x the array (5 launches), the second 6.5 x (6
// launches); here a row is read once into registers, reduced across the lanes that
// share it with wave64 shuffles (and four LDS slots when a block shares it), and the
// result written once: 2 x the array. Every elementwise step is the same single
// IEEE operation the separate launches perform (float subtraction, the sqrt that is
// the double-precision function rounded once, float division); the SFloat softmax's
// exponential is the double-precision 2^(x log2 e) of the table-driven core rounded
// once, which differs from NMath.exp's float in the last place at about one argument
// in 10^4. Results differ from the chain through that and the order of the two row sums.
//
// The reference has no such entry point; the host layer (cumo_hip_na_softmax /
// cumo_hip_na_layernorm) uses these for contiguous rows and composes the chain
// otherwise.
#include "common.h"
#include "ew_ops.h"

#include <cstring>

namespace cumo_hip {
namespace {

constexpr int kFrBlock = 256;

template <class T>
__device__ __forceinline__ T fr_shfl_xor(T v, int m) {
    if constexpr (sizeof(T) == 8) {
        union { T t; uint32_t w[2]; } a, b;
        a.t = v;
        b.w[0] = __shfl_xor(a.w[0], m);
        b.w[1] = __shfl_xor(a.w[1], m);
        return b.t;
    } else {
        union { T t; uint32_t w; } a, b;
        a.t = v;
        b.w = __shfl_xor(a.w, m);
        return b.t;
    }
}

// Combines one value per lane over the TPR lanes that share a row; every lane gets
// the result. The order is fixed (butterfly within the wave, then the block's waves in
// index order), so results do not vary from launch to launch.
template <class T, int TPR, int BLOCK = kFrBlock, class F>
__device__ __forceinline__ T fr_allreduce(T v, F f) {
    constexpr int SPAN = TPR < 64 ? TPR : 64;
#pragma unroll
    for (int m = SPAN >> 1; m > 0; m >>= 1) v = f(v, fr_shfl_xor(v, m));
    if constexpr (TPR > 64) {
        __shared__ T slot[BLOCK / 64];
        __syncthreads();  // the slots may still be read from the previous use
        if ((threadIdx.x & 63) == 0) slot[threadIdx.x >> 6] = v;
        __syncthreads();
        v = slot[0];
#pragma unroll
        for (int w = 1; w < BLOCK / 64; ++w) v = f(v, slot[w]);
    }
    return v;
}

// The lanes' parts of a row's sum. DFloat carries what each addition rounds off (the two-sum of Knuth, The Art of Computer
// Programming 2, 4.2.2) beside the sum: sixteen waves' parts one after the other would cost most of a last place. An infinite
// sum has no such rest.
template <class T, int LANES>
__device__ __forceinline__ double fr_allsum(double v) {
    if constexpr (sizeof(T) == 4) {
        return fr_allreduce<double, LANES, LANES>(v, [](double a, double b) { return a + b; });
    } else {
        struct Sum { double s, r; };
        auto add = [](Sum a, Sum b) {
            const double s = a.s + b.s, bb = s - a.s;
            return Sum{s, (a.r + b.r) + ((a.s - (s - bb)) + (b.s - bb))};
        };
        Sum t = {v, 0.0};
#pragma unroll
        for (int m = 32; m > 0; m >>= 1) t = add(t, Sum{fr_shfl_xor(t.s, m), fr_shfl_xor(t.r, m)});
        __shared__ Sum slot[LANES / 64];
        __syncthreads();  // the slots may still be read from the previous use
        if ((threadIdx.x & 63) == 0) slot[threadIdx.x >> 6] = t;
        __syncthreads();
        t = slot[0];
#pragma unroll
        for (int w = 1; w < LANES / 64; ++w) t = add(t, slot[w]);
        return t.s - t.s == 0.0 ? t.s + t.r : t.s;
    }
}

template <class T> __device__ __forceinline__ T fr_exp(T x);
// SFloat: 2^(x log2 e) from the table-driven core of ew_ops.h (2^-39 relative before the rounding to float; the
// element operator's polynomial form is good to 2^-50, which a softmax, divided by a sum of 2^-24 terms, cannot
// show): eight double operations fewer an element in a kernel that the exponential's arithmetic bounds.
// A NaN passes through the arithmetic; the clamp keeps the exponent in the core's range.
template <> __device__ __forceinline__ float fr_exp<float>(float x) {
    float xc = (x < -105.0f) ? -105.0f : x;
    xc = (xc > 89.0f) ? 89.0f : xc;
    return (float)exp2_by_table(1.44269504088896338700e+00 * (double)xc, float_tables());
}
template <> __device__ __forceinline__ double fr_exp<double>(double x) { return exp(x); }
template <class T> __device__ __forceinline__ T fr_sqrt(T x) { return (T)sqrt((double)x); }

// max that answers NaN when any element is NaN, as the reduction does (all-NaN or
// any-NaN max is NaN on the device: narray_test.rb:2551-2560)
template <class T> __device__ __forceinline__ T fr_max_nan(T a, T b) { return (a != a) ? a : ((b != b) ? b : (a > b ? a : b)); }

template <class T> __device__ __forceinline__ T fr_fmax(T a, T b);
template <> __device__ __forceinline__ float fr_fmax<float>(float a, float b) { return __builtin_fmaxf(a, b); }
template <> __device__ __forceinline__ double fr_fmax<double>(double a, double b) { return __builtin_fmax(a, b); }

// x / s for many x and one s, with the result of the IEEE division in T where s is a T.
// float: x / s = float(double(x) * (1.0 / double(s))). The product is within 2^-52 of
// the quotient, while the quotient of two 24-bit numbers is never closer than 2^-49
// (relative) to the midpoint of two floats unless it is a float itself, so the one
// rounding to float lands where the division's does; zero, infinity and NaN behave
// alike on both routes, and a subnormal quotient is rounded once by the conversion.
template <class T> struct FrDivisor;
template <> struct FrDivisor<float> {
    double r;
    __device__ __forceinline__ explicit FrDivisor(double s) : r(1.0 / s) {}
    __device__ __forceinline__ float divide(float x) const { return (float)((double)x * r); }
};
template <> struct FrDivisor<double> {
    double s;
    __device__ __forceinline__ explicit FrDivisor(double s_) : s(s_) {}
    __device__ __forceinline__ double divide(double x) const { return x / s; }
};

struct FusedRowsParams {
    uint64_t rows, n;
    int64_t in_row_step, out_row_step;  // bytes
    const char* in;
    char* out;
    double eps;
    bool through;  // see StoreRows
};

// whether rows of the result are written through (StoreRows)
__device__ __forceinline__ bool fr_pieces(const FusedRowsParams& p) {
    return p.through && store_pieces(p.out, p.out_row_step);
}

// MODE 0 softmax, 1 layernorm. TPR lanes share a row, each holding NV vectors of V
// elements (TPR * NV * V >= n). Rows, vectors and the elements of a row's last vector beyond the data are masked.
// NT: non-temporal accesses, for arrays larger than the last-level cache.
template <class T, int MODE, int TPR, int NV, bool NT>
__global__ __launch_bounds__(kFrBlock) void fused_rows_kernel(FusedRowsParams p) {
    constexpr int V = 16 / (int)sizeof(T);
    constexpr int RPB = kFrBlock / TPR;  // rows per block
    typedef uint32_t u4 __attribute__((ext_vector_type(4)));
    union Vec { u4 q; T t[V]; __device__ Vec() {} };
    const unsigned lane_r = threadIdx.x % TPR;
    const unsigned row_in_block = threadIdx.x / TPR;
    const uint64_t n_row_blocks = (p.rows + RPB - 1) / RPB;
    if constexpr (MODE == 0 && sizeof(T) == 4) float_tables_prepare();  // (the SFloat softmax reads the 2^x table)
    for (uint64_t rb = blockIdx.x; rb < n_row_blocks; rb += gridDim.x) {
        const uint64_t row = rb * RPB + row_in_block;
        const bool row_ok = row < p.rows;
        const char* src = p.in + (int64_t)(row_ok ? row : 0) * p.in_row_step;
        char* dst = p.out + (int64_t)(row_ok ? row : 0) * p.out_row_step;
        Vec x[NV];
        int cnt[NV];  // how many elements of the vector exist: V, none, or (the row's last vector) fewer
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            const uint64_t col = ((uint64_t)k * TPR + lane_r) * V;
            const int64_t left = (int64_t)p.n - (int64_t)col;
            cnt[k] = row_ok ? (left >= V ? V : (left > 0 ? (int)left : 0)) : 0;
            // a lane without a whole vector re-reads the row's first one: no branch between the loads
            const u4* ld = reinterpret_cast<const u4*>(src + (cnt[k] == V ? col : 0) * sizeof(T));
            x[k].q = NT ? __builtin_nontemporal_load(ld) : *ld;
        }
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            if (cnt[k] > 0 && cnt[k] < V) {
                // part of a vector at the row's end: element by element, nothing read past the row
                const uint64_t col = ((uint64_t)k * TPR + lane_r) * V;
#pragma unroll
                for (int j = 0; j < V; ++j)
                    if (j < cnt[k]) x[k].t[j] = reinterpret_cast<const T*>(src)[col + j];
            }
        }
        auto put = [&](int k) {
            const uint64_t col = ((uint64_t)k * TPR + lane_r) * V;
            if (cnt[k] == V) {
                store_vector<NT>(reinterpret_cast<u4*>(dst + col * sizeof(T)), x[k].q, fr_pieces(p));
            } else {
#pragma unroll
                for (int j = 0; j < V; ++j)
                    if (j < cnt[k]) reinterpret_cast<T*>(dst)[col + j] = x[k].t[j];
            }
        };
        if constexpr (MODE == 0) {
            // Lanes without data hold -inf: neutral in the max, and exp(-inf - m) adds 0 to the sum.
            // The max keeps the larger non-NaN value per element and notes NaN apart (one maximum and
            // one compare per element); a NaN anywhere then replaces the row's max, as in the reduction.
            T m = -INFINITY;
            bool any_nan = false;
#pragma unroll
            for (int k = 0; k < NV; ++k) {
#pragma unroll
                for (int j = 0; j < V; ++j) {
                    const T v = j < cnt[k] ? x[k].t[j] : (T)-INFINITY;
                    x[k].t[j] = v;
                    any_nan |= (v != v);
                    m = fr_fmax(m, v);
                }
            }
            if (any_nan) m = (T)NAN;
            m = fr_allreduce<T, TPR>(m, [](T a, T b) { return fr_max_nan(a, b); });
            T s = 0;
#pragma unroll
            for (int k = 0; k < NV; ++k) {
#pragma unroll
                for (int j = 0; j < V; ++j) {
                    const T e = fr_exp<T>(x[k].t[j] - m);
                    x[k].t[j] = e;
                    s += e;
                }
            }
            s = fr_allreduce<T, TPR>(s, [](T a, T b) { return a + b; });
            const FrDivisor<T> by_s((double)s);
#pragma unroll
            for (int k = 0; k < NV; ++k) {
                if (cnt[k] > 0) {
#pragma unroll
                    for (int j = 0; j < V; ++j) x[k].t[j] = by_s.divide(x[k].t[j]);
                    put(k);
                }
            }
        } else {
            // mean, then the squared deviations from it: two passes over registers
            T s = 0;
#pragma unroll
            for (int k = 0; k < NV; ++k) {
#pragma unroll
                for (int j = 0; j < V; ++j)
                    if (j < cnt[k]) s += x[k].t[j];
            }
            s = fr_allreduce<T, TPR>(s, [](T a, T b) { return a + b; });
            const T mean = s / (T)p.n;
            T q = 0;
#pragma unroll
            for (int k = 0; k < NV; ++k) {
#pragma unroll
                for (int j = 0; j < V; ++j) {
                    const T c = x[k].t[j] - mean;
                    x[k].t[j] = c;
                    if (j < cnt[k]) q += c * c;
                }
            }
            q = fr_allreduce<T, TPR>(q, [](T a, T b) { return a + b; });
            const T var = q / ((T)p.n - (T)1);
            const T sd = fr_sqrt<T>(var + (T)p.eps);
#pragma unroll
            for (int k = 0; k < NV; ++k) {
                if (cnt[k] > 0) {
#pragma unroll
                    for (int j = 0; j < V; ++j) x[k].t[j] = x[k].t[j] / sd;
                    put(k);
                }
            }
        }
    }
}

// ---- rows that the registers of 256 lanes do not hold --------------------------------
// One stretch of a row in the registers of a block: whole vectors, lane l holding vectors l, l + LANES, ..., and, one to a lane,
// the elements behind the last whole one. A vector is there or not: one compare, whose outcome is not kept, since counts and
// masks would be registers beside those that hold the row (64 of a lane's 128 with sixteen vectors).
template <class T, int LANES, int NV>
struct FrStretch {
    static constexpr int V = 16 / (int)sizeof(T);
    static constexpr uint32_t kElements = LANES * NV * V;
    typedef uint32_t u4 __attribute__((ext_vector_type(4)));
    union Vec { u4 q; T t[V]; __device__ Vec() {} };
    Vec x[NV];
    T last;
    uint32_t vectors, rest;  // whole vectors of the stretch, elements behind them

    __device__ __forceinline__ bool has(int k) const { return (uint32_t)k * LANES + threadIdx.x < vectors; }
    __device__ __forceinline__ bool has_last() const { return threadIdx.x < rest; }

    // `row`: the start of the row, which has one whole vector at least. A lane without a vector reads the stretch's first one, or
    // the row's: no branch between the loads, and an address every lane of the block shares.
    template <bool NT>
    __device__ __forceinline__ void load(const char* row, uint64_t start, uint32_t held) {
        const char* src = row + start * sizeof(T);
        vectors = held / V;
        rest = held % V;
        const char* whole = vectors ? src : row;
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            const u4* ld = reinterpret_cast<const u4*>(whole + (has(k) ? ((uint32_t)k * LANES + threadIdx.x) * 16u : 0u));
            x[k].q = NT ? __builtin_nontemporal_load(ld) : *ld;
        }
        last = *reinterpret_cast<const T*>(src + (has_last() ? (vectors * V + threadIdx.x) * (uint32_t)sizeof(T) : 0u));
    }
    __device__ __forceinline__ void fill(T none) {
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            const bool there = has(k);
#pragma unroll
            for (int j = 0; j < V; ++j) x[k].t[j] = there ? x[k].t[j] : none;
        }
        last = has_last() ? last : none;
    }
    template <class F>
    __device__ __forceinline__ void each(F f) {
#pragma unroll
        for (int k = 0; k < NV; ++k) {
#pragma unroll
            for (int j = 0; j < V; ++j) f(x[k].t[j]);
            if constexpr (NV > 8) __builtin_amdgcn_sched_barrier(0);
        }
        f(last);
    }
    // every element that is there less `by`; absent ones, which are 0, stay so. (A second fill() after taking `by` from every element
    // kept both copies of a vector: 26 registers of a lane of doubles were spilled.)
    __device__ __forceinline__ void lessen(T by) {
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            const T mine = has(k) ? by : (T)0;
#pragma unroll
            for (int j = 0; j < V; ++j) x[k].t[j] -= mine;
            if constexpr (NV > 8) __builtin_amdgcn_sched_barrier(0);
        }
        last -= has_last() ? by : (T)0;
    }
    // f of every element that is there, to memory
    template <bool NT, class F>
    __device__ __forceinline__ void store(char* row, uint64_t start, bool pieces, F f) {
        char* dst = row + start * sizeof(T);
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            if (has(k)) {
#pragma unroll
                for (int j = 0; j < V; ++j) x[k].t[j] = f(x[k].t[j]);
                store_vector<NT>(reinterpret_cast<u4*>(dst + ((uint32_t)k * LANES + threadIdx.x) * 16u), x[k].q, pieces);
            }
            if constexpr (NV > 8) __builtin_amdgcn_sched_barrier(0);
        }
        if (has_last()) reinterpret_cast<T*>(dst)[vectors * V + threadIdx.x] = f(last);
    }
    // the largest element, NaN where there is one; wants absent elements to be -inf
    __device__ __forceinline__ T maximum() {
        T m = -INFINITY;
        bool any_nan = false;
        each([&](T& v) {
            any_nan |= (v != v);
            m = fr_fmax(m, v);
        });
        if (any_nan) m = (T)NAN;
        return fr_allreduce<T, LANES, LANES>(m, [](T a, T b) { return fr_max_nan(a, b); });
    }
    // `part` gives what an element adds, which is 0 for one that is not there. A lane adds its elements as pairs of pairs in T,
    // the lanes' sums meet in double.
    template <class F>
    __device__ __forceinline__ double sum(F part) {
        T s = pairs<0, NV>(part);
        s += part(last);
        return fr_allsum<T, LANES>((double)s);
    }
    template <int FROM, int N, class F>
    __device__ __forceinline__ T pairs(F& part) {
        if constexpr (N == 1) {
            T a[V];
#pragma unroll
            for (int j = 0; j < V; ++j) a[j] = part(x[FROM].t[j]);
            if constexpr (NV > 8) __builtin_amdgcn_sched_barrier(0);
            if constexpr (V == 4) return (a[0] + a[1]) + (a[2] + a[3]);
            else return a[0] + a[1];
        } else {
            const T low = pairs<FROM, N / 2>(part);
            return low + pairs<FROM + N / 2, N / 2>(part);
        }
    }
};

template <class T, int MODE, int LANES, bool NT>
__global__ __launch_bounds__(LANES, 4) void fused_wide_rows_kernel(FusedRowsParams p) {
    if constexpr (MODE == 0 && sizeof(T) == 4) float_tables_prepare();
    const bool pieces = fr_pieces(p);
    FrStretch<T, LANES, 16> a;
    a.template load<NT>(p.in + (int64_t)blockIdx.x * p.in_row_step, 0, (uint32_t)p.n);
    char* dst = p.out + (int64_t)blockIdx.x * p.out_row_step;
    if constexpr (MODE == 0) {
        a.fill(-INFINITY);
        const T m = a.maximum();
        const double s = a.sum([&](T& v) { return v = fr_exp<T>(v - m); });
        const FrDivisor<T> by_s(s);
        a.template store<NT>(dst, 0, pieces, [&](T v) { return by_s.divide(v); });
    } else {
        a.fill((T)0);
        const T mean = (T)(a.sum([](T& v) { return v; }) / (double)p.n);
        a.lessen(mean);
        const T var = (T)(a.sum([](T& v) { return v * v; }) / ((double)p.n - 1.0));
        const T sd = fr_sqrt<T>(var + (T)p.eps);
        a.template store<NT>(dst, 0, pieces, [&](T v) { return v / sd; });
    }
}

// Longer rows, and few of them, are cut into pieces of 32 KiB, a block each, in two launches: the first leaves what the row
// needs of every piece, the second folds a row's parts in every block again (sixteen bytes a piece, from the second-level cache)
// and reads the piece once more, in the opposite order, since the pieces read last are still in the last-level cache.
//   softmax    part {maximum of the piece, sum of exp(x - that maximum)}
//   layernorm  part {sum of the piece, squared deviations from the piece's own mean}
// Sums within a piece are the type's; parts are folded in double.
template <class T> using FrPiece = FrStretch<T, kFrBlock, 8>;

struct FusedSplitParams : FusedRowsParams {
    uint32_t pieces;  // of a row
    double* parts;    // two for each piece, row after row
};

template <class T>
__device__ __forceinline__ uint32_t fr_piece_held(const FusedSplitParams& p, uint32_t piece) {
    const uint64_t left = p.n - (uint64_t)piece * FrPiece<T>::kElements;
    return left < FrPiece<T>::kElements ? (uint32_t)left : FrPiece<T>::kElements;
}

template <class T, int MODE>
__global__ __launch_bounds__(kFrBlock) void fused_parts_kernel(FusedSplitParams p) {
    if constexpr (MODE == 0 && sizeof(T) == 4) float_tables_prepare();
    const uint32_t row = blockIdx.x / p.pieces, piece = blockIdx.x - row * p.pieces;
    const uint32_t held = fr_piece_held<T>(p, piece);
    FrPiece<T> a;
    a.template load<false>(p.in + (int64_t)row * p.in_row_step, (uint64_t)piece * FrPiece<T>::kElements, held);
    double* part = p.parts + 2 * (uint64_t)blockIdx.x;
    if constexpr (MODE == 0) {
        a.fill(-INFINITY);
        const T m = a.maximum();
        const double s = a.sum([&](T& v) { return fr_exp<T>(v - m); });
        if (threadIdx.x == 0) {
            part[0] = (double)m;
            part[1] = m == (T)-INFINITY ? 0.0 : s;  // (nothing but -inf: adds 0 to a row that has more than that)
        }
    } else {
        a.fill((T)0);
        const T mean = (T)(a.sum([](T& v) { return v; }) / (double)held);
        a.lessen(mean);
        const double q = a.sum([](T& v) { return v * v; });
        const double r = a.sum([](T& v) { return v; });  // what rounding left of the sum: the deviations do not quite cancel
        if (threadIdx.x == 0) {
            part[0] = (double)mean * (double)held + r;
            part[1] = q;
        }
    }
}

template <class T, int MODE, bool NT>
__global__ __launch_bounds__(kFrBlock) void fused_apply_kernel(FusedSplitParams p) {
    const uint32_t at = gridDim.x - 1 - blockIdx.x;
    const uint32_t row = at / p.pieces, piece = at - row * p.pieces;
    const uint64_t start = (uint64_t)piece * FrPiece<T>::kElements;
    FrPiece<T> a;
    a.template load<NT>(p.in + (int64_t)row * p.in_row_step, start, fr_piece_held<T>(p, piece));
    if constexpr (MODE == 0 && sizeof(T) == 4) float_tables_prepare();
    const double* part = p.parts + 2 * (uint64_t)row * p.pieces;
    char* dst = p.out + (int64_t)row * p.out_row_step;
    const bool pieces = fr_pieces(p);
    if constexpr (MODE == 0) {
        double m = -INFINITY;
        for (uint32_t c = threadIdx.x; c < p.pieces; c += kFrBlock) m = fr_max_nan(m, part[2 * c]);
        m = fr_allreduce<double, kFrBlock>(m, [](double u, double w) { return fr_max_nan(u, w); });
        double s = 0.0;
        for (uint32_t c = threadIdx.x; c < p.pieces; c += kFrBlock) s += part[2 * c + 1] * exp(part[2 * c] - m);
        s = fr_allsum<T, kFrBlock>(s);
        const T mt = (T)m;  // (a maximum of T's)
        const FrDivisor<T> by_s(s);
        a.template store<NT>(dst, start, pieces, [&](T v) { return by_s.divide(fr_exp<T>(v - mt)); });
    } else {
        const double n = (double)p.n;
        double s = 0.0;
        for (uint32_t c = threadIdx.x; c < p.pieces; c += kFrBlock) s += part[2 * c];
        s = fr_allsum<T, kFrBlock>(s);
        const double mean = s / n;
        double q = 0.0;
        for (uint32_t c = threadIdx.x; c < p.pieces; c += kFrBlock) {
            const double held = (double)fr_piece_held<T>(p, c);
            const double away = part[2 * c] / held - mean;
            q += part[2 * c + 1] + held * away * away;
        }
        q = fr_allsum<T, kFrBlock>(q);
        const T var = (T)(q / (n - 1.0));
        const T sd = fr_sqrt<T>(var + (T)p.eps);
        const T mt = (T)mean;
        a.template store<NT>(dst, start, pieces, [&](T v) { return (v - mt) / sd; });
    }
}

// one read and one write of the array: beyond the 256 MB last-level cache, stream past it
template <class T>
bool fr_store_form(FusedRowsParams& p) {
    const bool nt = stream_past_caches(2 * p.rows * p.n * sizeof(T));
    StoreRows out_rows(p.out, p.n * sizeof(T));
    out_rows.dimension(p.rows, p.out_row_step);
    p.through = out_rows.through(nt);
    return nt;
}

template <class T, int MODE, int TPR, int NV>
void fr_launch_one(FusedRowsParams p, hipStream_t stream) {
    constexpr int RPB = kFrBlock / TPR;
    uint64_t grid = (p.rows + RPB - 1) / RPB;
    if (grid > 256u * 64u) grid = 256u * 64u;
    if (fr_store_form<T>(p)) hipLaunchKernelGGL((fused_rows_kernel<T, MODE, TPR, NV, true>), dim3((unsigned)grid), dim3(kFrBlock), 0, stream, p);
    else hipLaunchKernelGGL((fused_rows_kernel<T, MODE, TPR, NV, false>), dim3((unsigned)grid), dim3(kFrBlock), 0, stream, p);
}

// (a launch's lanes number less than 2^32; 2^22 blocks write 128 GiB and more)
constexpr uint64_t kFrMostBlocks = 1u << 22;

template <class T, int MODE, int LANES>
void fr_launch_wide(FusedRowsParams p, hipStream_t stream) {
    const dim3 grid((unsigned)p.rows), block(LANES);
    if (fr_store_form<T>(p)) hipLaunchKernelGGL((fused_wide_rows_kernel<T, MODE, LANES, true>), grid, block, 0, stream, p);
    else hipLaunchKernelGGL((fused_wide_rows_kernel<T, MODE, LANES, false>), grid, block, 0, stream, p);
}

template <class T, int MODE>
bool fr_launch_split(FusedRowsParams p, hipStream_t stream) {
    const uint64_t pieces = (p.n + FrPiece<T>::kElements - 1) / FrPiece<T>::kElements;
    if (pieces > kFrMostBlocks / p.rows) return false;
    const bool nt = fr_store_form<T>(p);
    char* parts = cumo_cuda_runtime_malloc(2 * sizeof(double) * p.rows * pieces);
    if (!parts) return true;  // the pool has reported it
    const FusedSplitParams q = {p, (uint32_t)pieces, reinterpret_cast<double*>(parts)};
    const dim3 grid((unsigned)(p.rows * pieces)), block(kFrBlock);
    hipLaunchKernelGGL((fused_parts_kernel<T, MODE>), grid, block, 0, stream, q);
    cumo_cuda_runtime_check_kernel_launch();
    if (nt) hipLaunchKernelGGL((fused_apply_kernel<T, MODE, true>), grid, block, 0, stream, q);
    else hipLaunchKernelGGL((fused_apply_kernel<T, MODE, false>), grid, block, 0, stream, q);
    cumo_cuda_runtime_free(parts);
    return true;
}

// Rows of more than 64 KiB (DFloat 32) were taken to the chain, which has no trouble with a result that overlaps its operand in some other
// way than element on element; what takes them here leaves those to it.
template <class T>
bool fr_apart(const FusedRowsParams& p) {
    if (p.in == p.out && p.in_row_step == p.out_row_step) return true;
    auto reach = [&](const char* at, int64_t step, uintptr_t* low, uintptr_t* high) {
        const int64_t far = step * (int64_t)(p.rows - 1);
        *low = (uintptr_t)at + (far < 0 ? far : 0);
        *high = (uintptr_t)at + (far > 0 ? far : 0) + p.n * sizeof(T);
    };
    uintptr_t in_low, in_high, out_low, out_high;
    reach(p.in, p.in_row_step, &in_low, &in_high);
    reach(p.out, p.out_row_step, &out_low, &out_high);
    return in_high <= out_low || out_high <= in_low;
}

// Picks lanes per row and vectors per lane for the row length (four vectors per lane
// where the row allows, so that a lane has four loads in flight). Beyond 64 KiB (DFloat 32) lanes hold sixteen vectors, 64
// registers: rows up to 128 KiB take 512 lanes, two blocks to a compute unit, so that one computes while the other's loads and
// stores are under way; up to 256 KiB 1024 lanes, if there are rows enough; longer ones are cut. us, softmax / layernorm, the
// chain that all of these took before, then 512 or 1024 lanes, then cut:
//   SFloat [588,27696]  91.2 / 76.5, 32.1 / 26.3, 46.7 / 39.1     [8,20000]   19.6 / 22.0, 10.5 / 7.4, 11.4 / 10.3
//   SFloat [400,65000]  211 / 190, 62.4 / 46.8, 63.6 / 55.0       [20,65000]  22.5 / 22.4, 19.2 / 12.7, 13.4 / 10.5
//   DFloat [762,29665]  230 / 178, 91.6 / 82.1, 99.7 / 95.1       [33,29738]  24.6 / 26.4, -, 14.6 / 12.5
//   DFloat [588,27696]  69.2 / 57.0 and 69.0 / 66.4 cut, [2000,10000] 63.6 / 55.0 and 90.1 / 86.2, [200,32768] 25.8 / 21.8 and 33.3 / 33.3,
//   [70,20000] 16.3 / 12.0 and 14.4 / 12.4
//   cut: SFloat [76,440000] 165 / 139, -, 80.0 / 67.0;  DFloat [108,128807] 146 / 123, -, 64.9 / 58.4
// (1024 lanes with eight vectors each for [588,27696]: 45.5 / 32.1.) false when the shape is left to the chain.
template <class T, int MODE>
bool fr_launch(const FusedRowsParams& p, hipStream_t stream) {
    constexpr int V = 16 / (int)sizeof(T);
    const uint64_t nv = (p.n + V - 1) / V;  // vectors per row, the last one maybe partly there
    if (nv <= 8) fr_launch_one<T, MODE, 8, 1>(p, stream);
    else if (nv <= 16) fr_launch_one<T, MODE, 8, 2>(p, stream);
    else if (nv <= 32) fr_launch_one<T, MODE, 8, 4>(p, stream);
    else if (nv <= 64) fr_launch_one<T, MODE, 16, 4>(p, stream);
    else if (nv <= 128) fr_launch_one<T, MODE, 32, 4>(p, stream);
    else if (nv <= 256) fr_launch_one<T, MODE, 64, 4>(p, stream);
    else if (nv <= 512) fr_launch_one<T, MODE, 256, 2>(p, stream);
    else if (nv <= 1024) fr_launch_one<T, MODE, 256, 4>(p, stream);
    else if (nv <= 2048) fr_launch_one<T, MODE, 256, 8>(p, stream);
    else if (nv <= 4096 && sizeof(T) == 4) fr_launch_one<T, MODE, 256, 16>(p, stream);
    else if (p.rows > kFrMostBlocks || !fr_apart<T>(p)) return false;
    else if (nv <= 8192) fr_launch_wide<T, MODE, 512>(p, stream);
    else if (nv <= 16384 && p.rows > 64) fr_launch_wide<T, MODE, 1024>(p, stream);
    else return fr_launch_split<T, MODE>(p, stream);
    return true;
}

}  // namespace
}  // namespace cumo_hip

using namespace cumo_hip;

// type: 0 SFloat, 1 DFloat. mode: 0 softmax, 1 layernorm. Returns 1 when the launch
// was made, 0 when the shape is outside what the kernels take (rows shorter than one
// 128-bit vector, not aligned as their elements are, or too long): the caller
// composes the operations instead.
extern "C" int cumo_hip_fused_rows_kernel_launch(int type, int mode, const cumo_hip_fused_rows_t* d) {
    if (!d || d->rows == 0 || d->n == 0) return 1;
    const int es = type == 0 ? 4 : 8;
    const uint64_t v = 16 / es;
    if (type < 0 || type > 1 || mode < 0 || mode > 1) return 0;
    // rows need their element's alignment only (128-bit accesses work on any 4-byte boundary) and may end in
    // part of a vector, which goes element by element
    if (d->n < v) return 0;
    if (((uintptr_t)d->in % es) || ((uintptr_t)d->out % es) || (d->in_row_step % es) || (d->out_row_step % es)) return 0;
    FusedRowsParams p;
    p.rows = d->rows;
    p.n = d->n;
    p.in_row_step = d->in_row_step;
    p.out_row_step = d->out_row_step;
    p.in = d->in;
    p.out = d->out;
    p.eps = d->eps;
    p.through = false;  // (fr_store_form says)
    hipStream_t stream = current_stream();
    bool ok;
    if (type == 0) ok = mode == 0 ? fr_launch<float, 0>(p, stream) : fr_launch<float, 1>(p, stream);
    else ok = mode == 0 ? fr_launch<double, 0>(p, stream) : fr_launch<double, 1>(p, stream);
    if (ok) cumo_cuda_runtime_check_kernel_launch();
    return ok ? 1 : 0;
}
