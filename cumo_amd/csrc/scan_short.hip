// cumsum / cumprod along many short runs (up to 4 KiB each): as many whole runs to a wave as its registers hold.
//
// Runs that follow one another in memory are one stretch of elements, and a scan of each is a scan of the stretch that starts anew
// where a run starts. A wave takes R rows of 64 vectors of such a stretch (whole runs, 2048 elements of four bytes at most), lane l
// holding vector l of every row, as the scan of long runs does (scan.hip), and scans them with one more condition: a lane takes
// on what a lane d vectors before it holds when the offset of its last element in its run says that the run reaches back that far.
// No lane has to know where another's runs start, nothing goes through LDS and waves do not meet. Runs with gaps between
// them, or whose elements have gaps, go element by element through the same steps.
// Bound by memory on the way in and out. Before, a block of 256 lanes took one run at a time, most of them idle, with two barriers:
//   us, before / now: SFloat [400001,83] 662 / 46, [200000,16] 314 / 6.3, [40000,51] 73 / 5.9, [562,18] 4.3 / 2.9, columns 3 to 79 of
//   [100000,100] 161 / 21; DFloat [400001,83] 869 / 85 (a copy of it: 86), [200000,16] 395 / 10.9, [40000,51] 90 / 8.6.
#include "scan_ops.h"

#include <cstring>

namespace cumo_hip {
namespace {

constexpr int kShortBlock = 256, kShortRows = 8;

struct ScanShortParams {
    const char* in;
    char* out;
    uint64_t runs;
    uint32_t n, per_wave;        // elements of a run, runs of a wave
    uint32_t magic;              // ceil(2^32 / n): positions below 2^16 divided by n > 1
    int64_t step_in, step_out;   // bytes from run to run
    int64_t s_in, s_out;         // and from element to element (DENSE: of their size, the runs without gaps)
    bool through;                // see StoreRows
};

template <class T, class Op, bool NT, bool DENSE>
__global__ __launch_bounds__(kShortBlock) void scan_short_kernel(ScanShortParams p) {
    typedef typename ScanVec<T>::u4 u4;
    constexpr int V = ScanVec<T>::V, R = kShortRows;
    const uint32_t lane = threadIdx.x & 63u, n = p.n;
    const uint64_t run0 = ((uint64_t)blockIdx.x * (kShortBlock / 64) + (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6))) * p.per_wave;
    if (run0 >= p.runs) return;
    const uint32_t runs = p.runs - run0 < p.per_wave ? (uint32_t)(p.runs - run0) : p.per_wave;
    const uint32_t nelem = runs * n;
    const char* in = p.in + (int64_t)run0 * p.step_in;
    char* out = p.out + (int64_t)run0 * p.step_out;
    ScanVec<T> v[R];
    uint32_t off[R];  // of the vector's first element in its run
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const u4 zero = {0u, 0u, 0u, 0u};
        v[r].q = zero;   // what does not exist lies after everything that does
        const uint32_t pos = ((uint32_t)r * 64u + lane) * V;
        uint32_t run = n == 1 ? pos : __umulhi(pos, p.magic);
        off[r] = pos - run * n;
        if ((uint32_t)r * 64u * V >= nelem) continue;
        if constexpr (DENSE) {
            const u4* src = reinterpret_cast<const u4*>(in) + r * 64 + lane;
            if (pos + V <= nelem) {
                v[r].q = NT ? __builtin_nontemporal_load(src) : *src;
            } else {
#pragma unroll
                for (int e = 0; e < V; ++e)
                    if (pos + e < nelem) v[r].e[e] = reinterpret_cast<const T*>(src)[e];
            }
        } else {
            uint32_t o = off[r];
#pragma unroll
            for (int e = 0; e < V; ++e) {
                if (pos + e < nelem) v[r].e[e] = *reinterpret_cast<const T*>(in + (int64_t)run * p.step_in + (int64_t)o * p.s_in);
                if (++o == n) { o = 0; ++run; }
            }
        }
    }
    T before = T();  // the running value after the rows so far
#pragma unroll
    for (int r = 0; r < R; ++r) {
        if ((uint32_t)r * 64u * V >= nelem) break;
        const uint32_t pos = ((uint32_t)r * 64u + lane) * V;
        uint32_t o[V];
        o[0] = off[r];
#pragma unroll
        for (int e = 1; e < V; ++e) {
            o[e] = o[e - 1] + 1 == n ? 0 : o[e - 1] + 1;
            v[r].e[e] = o[e] == 0 ? v[r].e[e] : Op::apply(v[r].e[e - 1], v[r].e[e]);
        }
        T x = v[r].e[V - 1];
        const uint32_t reach = o[V - 1];  // elements of its run before the lane's last one
#define CUMO_SHORT_STEP(CTRL, COND, LANES)                                        \
    {                                                                             \
        const T w = scan_dpp<CTRL>(x);                                            \
        x = (COND) && reach >= (uint32_t)(LANES) * V ? Op::apply(w, x) : x;       \
    }
        CUMO_SHORT_STEP(0x111, (lane & 15u) >= 1, 1)   // row_shr:1
        CUMO_SHORT_STEP(0x112, (lane & 15u) >= 2, 2)   // row_shr:2
        CUMO_SHORT_STEP(0x114, (lane & 15u) >= 4, 4)   // row_shr:4
        CUMO_SHORT_STEP(0x118, (lane & 15u) >= 8, 8)   // row_shr:8
        CUMO_SHORT_STEP(0x142, (lane & 16u) != 0, (lane & 15u) + 1u)   // row_bcast:15
        CUMO_SHORT_STEP(0x143, lane >= 32, lane - 31u)                 // row_bcast:31
#undef CUMO_SHORT_STEP
        // runs that began in an earlier row
        if (reach >= (lane + 1u) * V) x = Op::apply(before, x);
        T pre = scan_dpp<0x138>(x);  // the lane before (wave_shr:1)
        pre = lane == 0 ? before : pre;
        before = scan_read_lane(x, 63);
#pragma unroll
        for (int e = 0; e < V; ++e)
            if (o[e] > (uint32_t)e) v[r].e[e] = Op::apply(pre, v[r].e[e]);
        if constexpr (DENSE) {
            u4* dst = reinterpret_cast<u4*>(out) + r * 64 + lane;
            if (pos + V <= nelem) {
                store_vector<NT>(dst, v[r].q, p.through && store_pieces(out));
            } else {
#pragma unroll
                for (int e = 0; e < V; ++e)
                    if (pos + e < nelem) reinterpret_cast<T*>(dst)[e] = v[r].e[e];
            }
        } else {
            uint32_t run = n == 1 ? pos : __umulhi(pos, p.magic);
#pragma unroll
            for (int e = 0; e < V; ++e) {
                if (e > 0 && o[e] == 0) ++run;
                if (pos + e < nelem) *reinterpret_cast<T*>(out + (int64_t)run * p.step_out + (int64_t)o[e] * p.s_out) = v[r].e[e];
            }
        }
    }
}

template <class T, class Op>
void scan_short_run(ScanShortParams& p, bool dense, hipStream_t stream) {
    constexpr uint64_t V = ScanVec<T>::V, CAP = kShortRows * 64 * V;
    // As many runs to a wave as fit, or as leave a wave to every SIMD; then, if that costs no more than an eighth of them, as many as
    // make whole 64-byte pieces (or the next smaller power of two), so that waves do not share those.
    uint64_t per = CAP / p.n, fair = (p.runs + 1023) / 1024;
    if (per > fair) per = fair;
    if (dense) {
        for (uint64_t m = kStorePiece / sizeof(T); m > 1; m >>= 1) {
            const uint64_t whole = per / m * m;
            if (whole > 0 && whole * 8 >= per * 7) {
                per = whole;
                break;
            }
        }
    }
    p.per_wave = (uint32_t)per;
    const uint64_t waves = (p.runs + per - 1) / per, grid = (waves + kShortBlock / 64 - 1) / (kShortBlock / 64);
    const bool nt = stream_past_caches(2 * p.runs * p.n * sizeof(T));
    p.through = true;
    const dim3 g((unsigned)grid), b(kShortBlock);
    if (!dense) hipLaunchKernelGGL((scan_short_kernel<T, Op, false, false>), g, b, 0, stream, p);
    else if (nt) hipLaunchKernelGGL((scan_short_kernel<T, Op, true, true>), g, b, 0, stream, p);
    else hipLaunchKernelGGL((scan_short_kernel<T, Op, false, true>), g, b, 0, stream, p);
}

template <class T>
void scan_short_dispatch(int prod, int nan, ScanShortParams& p, bool dense, hipStream_t stream) {
    if (prod) {
        if (nan) scan_short_run<T, ScanOp<T, 1, true> >(p, dense, stream);
        else scan_short_run<T, ScanOp<T, 1, false> >(p, dense, stream);
    } else {
        if (nan) scan_short_run<T, ScanOp<T, 0, true> >(p, dense, stream);
        else scan_short_run<T, ScanOp<T, 0, false> >(p, dense, stream);
    }
}

}  // namespace

bool scan_short_launch(int type, int prod, int nan, const cumo_hip_scan_rows_t* d) {
    if (type < 0 || type > 2) return false;
    const int64_t es = type == 1 ? 8 : 4;
    if (d->n > 4096 / (uint64_t)es || d->rows < 2) return false;
    if ((((uintptr_t)d->in | (uintptr_t)d->out) % es) != 0 || d->s_in % es != 0 || d->s_out % es != 0) return false;
    // the runs, one step apart on either side; outer dimensions that are more than that go elsewhere
    uint64_t runs = 1;
    int64_t step_in = 0, step_out = 0;
    for (int k = d->nouter - 1; k >= 0; --k) {
        if (d->oshape[k] == 1) continue;
        if (d->ostep_in[k] % es != 0 || d->ostep_out[k] % es != 0) return false;
        if (runs == 1) {
            step_in = d->ostep_in[k];
            step_out = d->ostep_out[k];
        } else if (d->ostep_in[k] != step_in * (int64_t)runs || d->ostep_out[k] != step_out * (int64_t)runs) {
            return false;
        }
        runs *= d->oshape[k];
    }
    if (runs != d->rows) return false;
    ScanShortParams p;
    std::memset(&p, 0, sizeof(p));
    p.in = d->in;
    p.out = d->out;
    p.runs = runs;
    p.n = (uint32_t)d->n;
    p.magic = d->n > 1 ? (uint32_t)(((1ull << 32) + d->n - 1) / d->n) : 0;
    p.step_in = step_in;
    p.step_out = step_out;
    p.s_in = d->s_in;
    p.s_out = d->s_out;
    const int64_t run_bytes = (int64_t)d->n * es;
    const bool unit = d->n == 1 || (d->s_in == es && d->s_out == es);
    const bool dense = unit && step_in == run_bytes && step_out == run_bytes;
    // A block to a run / this form, us: runs of SFloat 300 in 5000 6.7 / 5.1, 400 in 60000 64 / 32, 700 in 30000 37 / 29, 1000 in 30000
    // 40.1 / 38.5, 1100 in 20000 33.7 / 31.3, 1500 in 10000 21.5 / 23.4; DFloat 300 in 5000 8.2 / 7.0, 501 in 30000 48.9 / 43.4, 700 51.8 / 54.0.
    // From 64 vectors on that form reads runs with gaps between them by vectors and this one does not.
    if (unit && !dense && d->n * (uint64_t)es >= 1024) return false;
    hipStream_t stream = current_stream();
    switch (type) {
        case 0: scan_short_dispatch<float>(prod, nan, p, dense, stream); break;
        case 1: scan_short_dispatch<double>(prod, nan, p, dense, stream); break;
        default: scan_short_dispatch<int32_t>(prod, 0, p, dense, stream); break;
    }
    return true;
}

}  // namespace cumo_hip
