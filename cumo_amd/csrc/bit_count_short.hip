// Counts of set (or clear) bits of many short runs along memory, on word boundaries or not: the rows of the masks of tables. (The
// reference walks the outputs on the host and launches one kernel each: narray/ndloop.c:1569-1613 under
// gen/tmpl_bit/bit_count.c:9-36.)
//
// Bound by the trip to memory of one wave after another, so 2^k lanes take a run, as many as give each at most four words,
// and a wave takes 64 / 2^k runs with all of their words in flight; a wave for every run had a word in each of a few lanes and a
// 64-lane sum behind it, and a launch in front that cleared the results. us a call, a wave a run / this, whose calls the host
// bounds at 3.1: [180232,137] 67.7 / 3.2, [24304,1066] 15.4 / 3.3, [32768,1024] 18.4 / 3.3, [1000000,8] 298 / 4.4, [2000,1000] 6.1 / 3.2.
#include "bit_common.h"
#include "div31.h"

#include <cstring>

using namespace cumo_hip;

namespace {

constexpr int kRgBlock = 256;
constexpr int kRgWords = 4;   // words of a lane

struct ShortRows {
    const uint32_t* in;
    char* out;
    uint64_t pos;
    int64_t in_step[CUMO_NA_MAX_DIMENSION], out_step[CUMO_NA_MAX_DIMENSION];   // bits, bytes
    uint32_t shape[CUMO_NA_MAX_DIMENSION];
    Div31 div[CUMO_NA_MAX_DIMENSION];
    uint32_t rows, n;
    int ndim, count_false, overwrite;
};

// LPR lanes share a row of up to LPR * kRgWords words
template <int LPR>
__global__ __launch_bounds__(kRgBlock) void bit_count_short_rows_kernel(ShortRows p) {
    const uint32_t at = (blockIdx.x * (uint32_t)kRgBlock + threadIdx.x) / LPR;
    const uint32_t lane = threadIdx.x % LPR;
    const uint32_t row = at < p.rows ? at : p.rows - 1;
    int64_t bit = (int64_t)p.pos, off = 0;
    uint32_t r = row;
    for (int d = p.ndim - 1; d >= 0; --d) {
        uint32_t k = r;
        if (d > 0) {
            const uint32_t q = div31(r, p.div[d]);
            k = r - q * p.shape[d];
            r = q;
        }
        bit += (int64_t)k * p.in_step[d];
        off += (int64_t)k * p.out_step[d];
    }
    const uint64_t first = (uint64_t)bit >> 5;
    const uint32_t lead = (uint32_t)bit & 31u;
    const uint32_t last = (lead + p.n - 1) >> 5;          // the row's last word, counted from its first
    const uint32_t end = (lead + p.n - 1) & 31u;          // the row's last bit in it
    uint32_t x[kRgWords];
#pragma unroll
    for (int k = 0; k < kRgWords; ++k) {
        const uint32_t w = (uint32_t)k * LPR + lane;
        x[k] = p.in[first + (w < last ? w : last)];
    }
    uint32_t c = 0;
#pragma unroll
    for (int k = 0; k < kRgWords; ++k) {
        const uint32_t w = (uint32_t)k * LPR + lane;
        uint32_t v = p.count_false ? ~x[k] : x[k];
        if (w == 0) v &= 0xffffffffu << lead;
        if (w == last) v &= 0xffffffffu >> (31u - end);
        c += w <= last ? (uint32_t)__popc(v) : 0u;
    }
#pragma unroll
    for (int m = LPR >> 1; m > 0; m >>= 1) c += __shfl_xor(c, m);
    if (lane == 0 && at < p.rows) {
        unsigned long long* dst = reinterpret_cast<unsigned long long*>(p.out + off);
        *dst = p.overwrite ? (unsigned long long)c : *dst + c;
    }
}

template <int LPR>
void launch_short(const ShortRows& p, hipStream_t stream) {
    const uint64_t lanes = (uint64_t)p.rows * LPR;
    hipLaunchKernelGGL((bit_count_short_rows_kernel<LPR>), dim3((unsigned)((lanes + kRgBlock - 1) / kRgBlock)), dim3(kRgBlock), 0, stream, p);
    cumo_cuda_runtime_check_kernel_launch();
}

}  // namespace

namespace cumo_hip {

// Runs of up to 8161 bits that lie along memory, anywhere (256 words, with the first bit the last of its word). 1 when launched (counts
// stored or added as d->overwrite says), 0 when the loop is another.
int bit_count_short_rows_launch(const cumo_hip_bit_count_nd_t* d) {
    if (d->red_ndim != 1 || d->in_red_step[0] != 1 || d->out_ndim < 1 || force_wide_indices()) return 0;
    const uint64_t n = d->red_shape[0];
    const uint64_t words = (n + 62) / 32;   // as many as a run can touch
    if (n == 0 || words > 64 * kRgWords) return 0;
    ShortRows p;
    std::memset(&p, 0, sizeof(p));
    uint64_t rows = 1;
    for (int k = 0; k < d->out_ndim; ++k) {
        if (d->out_shape[k] == 0 || d->out_shape[k] >= (1ull << 31)) return 0;
        rows *= d->out_shape[k];
        if (rows >= (1ull << 31)) return 0;
        p.shape[k] = (uint32_t)d->out_shape[k];
        p.div[k] = div31_make(p.shape[k]);
        p.in_step[k] = d->in_out_step[k];
        p.out_step[k] = d->out_step[k];
    }
    int lpr = 1;
    while ((uint64_t)lpr * kRgWords < words) lpr *= 2;
    if (rows * lpr >= (1ull << 31)) return 0;
    p.in = d->in;
    p.out = d->out;
    p.pos = d->pos;
    p.rows = (uint32_t)rows;
    p.n = (uint32_t)n;
    p.ndim = d->out_ndim;
    p.count_false = d->count_false;
    p.overwrite = d->overwrite;
    hipStream_t stream = current_stream();
    switch (lpr) {
        case 1: launch_short<1>(p, stream); break;
        case 2: launch_short<2>(p, stream); break;
        case 4: launch_short<4>(p, stream); break;
        case 8: launch_short<8>(p, stream); break;
        case 16: launch_short<16>(p, stream); break;
        case 32: launch_short<32>(p, stream); break;
        default: launch_short<64>(p, stream); break;
    }
    return 1;
}

}  // namespace cumo_hip
