// Bit#where and Bit#mask: the positions of the set (or clear) bits of a run,
// compacted in ascending order.
//
// Replaces narray/gen/tmpl_bit/where_kernel.cu and mask_kernel.cu of the reference
// with the same launcher ABI and the same scratch layout (two running cursors, then
// up to 1024 block counts), so that the host iterators (tmpl_bit/where.c:34-52,
// mask.c) bind unchanged: a cursor in the scratch carries the output position from
// one run of a view to the next on the device, and nothing is read back.
//
// Three launches per run: every block counts the set bits of its contiguous range
// of 32-bit chunks; one block turns the counts into output positions (and advances
// the cursor); every block walks its range again, 256 chunks a round: an exclusive
// scan over the block places each chunk's hits in a list in LDS, and consecutive
// lanes then write the list out, so the stores of a wave are adjacent. Blocks are 256
// threads (4 wave64): the scan inside a block is a wave scan by DPP steps plus four LDS
// slots.
// A contiguous run reads whole words (two per chunk when the run starts inside a
// word); strided and index-array runs gather bit by bit.
#include "common.h"
#include "div31.h"

#include <type_traits>

#include <chrono>
#include <cstring>

namespace cumo_hip {
namespace {

constexpr int kWhBlock = 256;
constexpr uint64_t kWhMaxBlocks = 1024;  // the scratch holds this many block counts (where_kernel.cu:11)

// the 32 bits [c*32, c*32+32) of the run, bits beyond n cleared
__device__ __forceinline__ uint32_t wh_chunk(const CUMO_BIT_DIGIT* a, uint64_t p, int64_t s, const size_t* idx, uint64_t n, uint64_t c,
                                             int contiguous, int invert) {
    const uint64_t first = c * 32;
    const uint64_t left = n - first;
    const uint32_t valid = left >= 32 ? 0xffffffffu : ((1u << left) - 1u);
    uint32_t z;
    if (contiguous) {
        const uint64_t q = p + first;
        const uint64_t w = q >> 5;
        const unsigned sh = (unsigned)(q & 31);
        z = a[w] >> sh;
        // the second word only exists when the chunk reaches into it
        if (sh && (uint64_t)(32 - sh) < left) z |= a[w + 1] << (32 - sh);
    } else {
        z = 0;
        const unsigned m = left >= 32 ? 32u : (unsigned)left;
        for (unsigned k = 0; k < m; ++k) {
            const uint64_t q = idx ? (p + idx[first + k]) : (uint64_t)((int64_t)p + (int64_t)(first + k) * s);
            z |= ((a[q >> 5] >> (q & 31)) & 1u) << k;
        }
    }
    if (invert) z = ~z;
    return z & valid;
}

// exclusive scan of one value per thread over the block; *total gets the block's sum
// in every thread. Two barriers; safe to call again right away.
__device__ __forceinline__ uint64_t wh_block_exscan(uint64_t v, uint64_t* total) {
    __shared__ uint64_t wave_sum[kWhBlock / 64];
    const unsigned lane = threadIdx.x & 63;
    uint64_t inc = v;
    for (unsigned d = 1; d < 64; d <<= 1) {
        const uint32_t lo = __shfl_up((uint32_t)inc, d);
        const uint32_t hi = __shfl_up((uint32_t)(inc >> 32), d);
        if (lane >= d) inc += ((uint64_t)hi << 32) | lo;
    }
    __syncthreads();  // the slots may still be read from the previous call
    if (lane == 63) wave_sum[threadIdx.x >> 6] = inc;
    __syncthreads();
    uint64_t before = 0, all = 0;
    for (unsigned w = 0; w < kWhBlock / 64; ++w) {
        if (w < (threadIdx.x >> 6)) before += wave_sum[w];
        all += wave_sum[w];
    }
    *total = all;
    return before + inc - v;
}

// A barrier for the LDS traffic only: loads from global memory that were sent ahead stay
// in flight across it (__syncthreads() waits for them as well).
__device__ __forceinline__ void wh_lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// inclusive scan over the 64 lanes of a wave: four shifts within the rows of 16 lanes,
// then lane 15 of a row into the next row and lane 31 into the upper half
__device__ __forceinline__ uint32_t wh_wave_scan(uint32_t v) {
    int x = (int)v;
    x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, true);   // row_shr:1
    x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, true);   // row_shr:2
    x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, true);   // row_shr:4
    x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, true);   // row_shr:8
    x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);  // row_bcast:15 into rows 1 and 3
    x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);  // row_bcast:31 into rows 2 and 3
    return (uint32_t)x;
}

// exclusive scan of one small value per thread over the block (the sum fits 32 bits); *total
// gets the block's sum in every thread. Two LDS-only barriers; safe to call again right away.
__device__ __forceinline__ uint32_t wh_block_exscan32(uint32_t v, uint32_t* total) {
    __shared__ uint32_t wave_sum32[kWhBlock / 64];
    const uint32_t inc = wh_wave_scan(v);
    wh_lds_barrier();  // the slots may still be read from the previous call
    if ((threadIdx.x & 63) == 63) wave_sum32[threadIdx.x >> 6] = inc;
    wh_lds_barrier();
    uint32_t before = 0, all = 0;
#pragma unroll
    for (unsigned w = 0; w < kWhBlock / 64; ++w) {
        const uint32_t ws = wave_sum32[w];
        before += (w < (threadIdx.x >> 6)) ? ws : 0u;
        all += ws;
    }
    *total = all;
    return before + inc - v;
}

// The hits of every placing block's share of the chunks: a block counts for kWhGroups of them, 256 lanes each, four words in
// flight a lane. host_sums: pinned host memory that the caller looks at, which gets a copy of each count, one up so that no count
// is the 0 the host looks for. Measured with x.where and x[mask] of 2^25 SFloat, the host's time, us a call: blocks of one share
// and one word in flight a lane 27.3 and (a hit in a thousand) 22.8, this 23.7 and 18.9; the total of a block's four counts to
// the host in their place, a quarter of the words, 24.5 and 19.7. (Masks of a few thousand bits: 14.5 against 14.3; blocks of no
// more waves than there are shares changed nothing there.)
constexpr int kWhGroups = 4;
__global__ __launch_bounds__(kWhBlock * kWhGroups) void where_count_kernel(const CUMO_BIT_DIGIT* a, uint64_t p, int64_t s, const size_t* idx, uint64_t n,
                                                                           int contiguous, int invert, uint64_t nchunks, uint64_t cpb, uint64_t nshares,
                                                                           uint64_t* sums, uint64_t* host_sums) {
    __shared__ uint64_t wave_sum[kWhBlock * kWhGroups / 64];
    const unsigned t = threadIdx.x % kWhBlock;
    const uint64_t share = (uint64_t)blockIdx.x * kWhGroups + threadIdx.x / kWhBlock;
    uint64_t start = share * cpb;
    if (start > nchunks) start = nchunks;
    const uint64_t end = (nchunks - start < cpb) ? nchunks : start + cpb;
    uint64_t cnt = 0;
    uint64_t c = start + t;
    if (contiguous && (p & 31) == 0) {
        // whole words, four in flight a lane; a run's last chunk, partly there, comes below
        const uint64_t whole = (end == nchunks && (n & 31) != 0) ? end - 1 : end;
        const uint32_t* w = reinterpret_cast<const uint32_t*>(a) + (p >> 5);
        const uint32_t flip = invert ? 0xffffffffu : 0u;
        for (; c + 3 * kWhBlock < whole; c += 4 * kWhBlock) {
            uint32_t v[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) v[k] = w[c + k * kWhBlock];
#pragma unroll
            for (int k = 0; k < 4; ++k) cnt += (uint64_t)__popc(v[k] ^ flip);
        }
    }
    for (; c < end; c += kWhBlock) cnt += (uint64_t)__popc(wh_chunk(a, p, s, idx, n, c, contiguous, invert));
    for (int m = 32; m > 0; m >>= 1) {
        const uint32_t lo = __shfl_xor((uint32_t)cnt, m), hi = __shfl_xor((uint32_t)(cnt >> 32), m);
        cnt += ((uint64_t)hi << 32) | lo;
    }
    if ((threadIdx.x & 63) == 0) wave_sum[threadIdx.x >> 6] = cnt;
    __syncthreads();
    constexpr unsigned WPS = kWhBlock / 64;   // waves of a share
    if (threadIdx.x < kWhGroups) {
        uint64_t mine = 0;
        for (unsigned k = 0; k < WPS; ++k) mine += wave_sum[threadIdx.x * WPS + k];
        const uint64_t at = (uint64_t)blockIdx.x * kWhGroups + threadIdx.x;
        if (at < nshares) {
            sums[at] = mine;
            if (host_sums) __hip_atomic_store(host_sums + at, mine + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
}
inline unsigned wh_count_grid(uint64_t nblocks) { return (unsigned)((nblocks + kWhGroups - 1) / kWhGroups); }

// block_sums[b] becomes the output position of block b's first hit; *running moves on
__global__ __launch_bounds__(kWhBlock) void where_scan_kernel(uint64_t* block_sums, uint64_t nblocks, uint64_t* running) {
    uint64_t acc = *running;
    for (uint64_t t0 = 0; t0 < nblocks; t0 += kWhBlock) {
        const uint64_t t = t0 + threadIdx.x;
        const uint64_t v = t < nblocks ? block_sums[t] : 0;
        uint64_t total;
        const uint64_t pre = wh_block_exscan(v, &total);
        if (t < nblocks) block_sums[t] = acc + pre;
        acc += total;
    }
    __syncthreads();  // every thread has read *running before it is rewritten
    if (threadIdx.x == 0) *running = acc;
}

// MODE 0: out[o] = count + position in the run, as ES-byte integers (where).
// MODE 1: out[o] = the masked array's element position p2 + j*s2 (or p2 + idx2[j]), as size_t (mask; ES 8).
// MODE 2: out[o] = the masked array's element itself, ES (4 or 8) bytes read at p2 + j*s2 where p2 is
//         its address (the compaction the reference reaches through a view over the positions of mode 1).
// COUNTS: block_sums holds the blocks' plain counts (no scan launch ran): the block adds up
// the counts of the blocks before it.
template <int MODE, int ES, bool COUNTS>
__global__ __launch_bounds__(kWhBlock) void where_scatter_kernel(const CUMO_BIT_DIGIT* a, uint64_t p, int64_t s, const size_t* idx, uint64_t n,
                                                                 int contiguous, int invert, uint64_t nchunks, uint64_t cpb, char* out,
                                                                 uint64_t count, size_t p2, int64_t s2, const size_t* idx2,
                                                                 const uint64_t* block_sums) {
    typedef typename std::conditional<ES == 4, uint32_t, uint64_t>::type E;
    uint64_t start = (uint64_t)blockIdx.x * cpb;
    if (start > nchunks) start = nchunks;
    const uint64_t end = (nchunks - start < cpb) ? nchunks : start + cpb;
    // hits of one round (256 chunks, up to 8192 bits) are listed in LDS by their bit
    // position within the round, then written out by consecutive lanes
    __shared__ uint16_t hit[kWhBlock * 32];
    uint64_t off;
    if (COUNTS) {
        uint64_t before = 0;
        for (uint64_t t = threadIdx.x; t < blockIdx.x; t += kWhBlock) before += block_sums[t];
        wh_block_exscan(before, &off);
    } else {
        off = block_sums[blockIdx.x];
    }
    // the next round's bits are loaded before this round's are placed
    uint32_t znext = start + threadIdx.x < end ? wh_chunk(a, p, s, idx, n, start + threadIdx.x, contiguous, invert) : 0u;
    for (uint64_t c0 = start; c0 < end; c0 += kWhBlock) {
        uint32_t z = znext;
        const uint64_t cn = c0 + kWhBlock + threadIdx.x;
        znext = cn < end ? wh_chunk(a, p, s, idx, n, cn, contiguous, invert) : 0u;
        uint32_t total;
        // the first barrier inside the scan also ends the previous round's reads of hit[]
        uint32_t o = wh_block_exscan32((uint32_t)__popc(z), &total);
        const uint32_t mine = threadIdx.x * 32;
        while (z) {
            hit[o++] = (uint16_t)(mine + (unsigned)__builtin_ctz(z));
            z &= z - 1;
        }
        wh_lds_barrier();
        const uint64_t j0 = c0 * 32;             // the round's first bit, and where its hits go
        E* const dst = reinterpret_cast<E*>(out) + off;
#pragma unroll 4
        for (uint32_t k = threadIdx.x; k < total; k += kWhBlock) {
            const uint32_t h = hit[k];
            if (MODE == 2) {
                dst[k] = *reinterpret_cast<const E*>(reinterpret_cast<const char*>(p2) + (int64_t)(j0 + h) * s2);
            } else if (MODE == 1) {
                const uint64_t j = j0 + h;
                dst[k] = (E)(idx2 ? (p2 + idx2[j]) : (size_t)((int64_t)p2 + (int64_t)j * s2));
            } else {
                dst[k] = (E)(count + j0) + (E)h;
            }
        }
        off += total;
    }
}

// The elements of a contiguous run where the mask is set, as whole vectors of the run: a wave takes 1024 elements (32
// chunks) at a time, a lane the VEC neighbours of each of U rows, reads a vector only where one of them is a hit, and
// lists the hits in the wave's stretch of LDS by their rank: what the chunk's earlier bits and the scan over the
// chunks count. Consecutive lanes then write the list out. The waves of a block meet once per tile, over their totals, in an
// LDS-only barrier, so the next tile's vectors stay in flight while this one's hits are written.
// Bound by memory: where_scatter_kernel asks for one element per hit and lane, which is a third of the cache lines' worth
// of bytes at a hit in three: 2^25 SFloat at 33 % hits, fresh operands, 45.5 -> 35.8 us. NT (arrays that no cache is to hold): the call
// 49 us, with plain loads 52; on an array that lies in the last-level cache all the same 49.5 and 43 (one by one 46), but a pass of
// mask, counts, values, positions and rows of 8192 x 4096 takes 173 us with NT and 181 without. Of sparse masks both read the lines
// that hold a hit, and what a wave does for every 1024 elements here costs more than its few hits do there: where_place.
template <int ES, bool NT>
__global__ __launch_bounds__(kWhBlock) void mask_pack_kernel(const CUMO_BIT_DIGIT* a, uint64_t p, uint64_t n, int invert, uint64_t nchunks, uint64_t cpb,
                                                             char* out, const char* x, const uint64_t* block_sums) {
    typedef typename std::conditional<ES == 4, uint32_t, uint64_t>::type E;
    typedef uint32_t u4 __attribute__((ext_vector_type(4)));
    constexpr int VEC = 16 / ES;              // elements of a vector
    constexpr int U = 16 / VEC;               // rows of 64 vectors: 1024 elements
    constexpr unsigned WAVES = kWhBlock / 64;
    constexpr unsigned TILE = WAVES * 32;     // chunks of a block's tile
    union V { u4 q; E e[VEC]; __device__ V() {} };
    __shared__ E list[WAVES][1024];
    __shared__ uint32_t totals[2][WAVES];
    const unsigned lane = threadIdx.x & 63u;
    const unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    uint64_t start = (uint64_t)blockIdx.x * cpb;
    if (start > nchunks) start = nchunks;
    const uint64_t end = (nchunks - start < cpb) ? nchunks : start + cpb;
    uint64_t off;
    {
        uint64_t before = 0;
        for (uint64_t t = threadIdx.x; t < blockIdx.x; t += kWhBlock) before += block_sums[t];
        wh_block_exscan(before, &off);
    }
    const unsigned bit = (lane * VEC) & 31u;        // where the lane's vector starts in its chunk
    const unsigned chunk0 = (lane * VEC) >> 5;      // ... of row 0; a row is 2 * VEC chunks
    // lane l < 32 holds chunk l of the wave's next 1024 bits
    auto chunk_at = [&](uint64_t c0) -> uint32_t {
        const uint64_t c = c0 + wave * 32 + lane;
        return (lane < 32 && c < end) ? wh_chunk(a, p, 1, nullptr, n, c, 1, invert) : 0u;
    };
    V v[U];
    uint32_t w[U];
    auto load = [&](uint64_t c0, uint32_t z) {
        const uint64_t e0 = (c0 + wave * 32) * 32 + lane * VEC;
#pragma unroll
        for (int u = 0; u < U; ++u) w[u] = __shfl(z, (int)(chunk0 + u * 2 * VEC));
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint64_t e = e0 + (uint64_t)u * 64 * VEC;
            const uint32_t mine = (w[u] >> bit) & ((1u << VEC) - 1u);
            if (mine) {
                if (e + VEC <= n) {
                    const u4* src = reinterpret_cast<const u4*>(x + e * ES);
                    v[u].q = NT ? __builtin_nontemporal_load(src) : *src;
                } else {
#pragma unroll
                    for (int j = 0; j < VEC; ++j)
                        if (e + j < n) v[u].e[j] = reinterpret_cast<const E*>(x)[e + j];
                }
            }
        }
    };
    uint32_t z = chunk_at(start);
    load(start, z);
    uint32_t znext = chunk_at(start + TILE);
    unsigned turn = 0;
    for (uint64_t c0 = start; c0 < end; c0 += TILE, turn ^= 1u) {
        const uint32_t cnt = (uint32_t)__popc(z);
        const uint32_t inc = wh_wave_scan(cnt);
        const uint32_t mine = __builtin_amdgcn_readlane((int)inc, 63);
        if (lane == 0) totals[turn][wave] = mine;
        const uint32_t ex = inc - cnt;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            uint32_t r = __shfl(ex, (int)(chunk0 + u * 2 * VEC)) + (uint32_t)__popc(w[u] & ((1u << bit) - 1u));
#pragma unroll
            for (int j = 0; j < VEC; ++j) {
                if ((w[u] >> (bit + j)) & 1u) list[wave][r++] = v[u].e[j];
            }
        }
        z = znext;
        load(c0 + TILE, z);
        znext = chunk_at(c0 + 2 * TILE);
        wh_lds_barrier();   // (the other half of totals[] is what the waves still behind read: one barrier a tile is enough)
        uint32_t before = 0, all = 0;
#pragma unroll
        for (unsigned k = 0; k < WAVES; ++k) {
            const uint32_t t = totals[turn][k];
            before += k < wave ? t : 0u;
            all += t;
        }
        E* const dst = reinterpret_cast<E*>(out) + off + before;
        for (uint32_t k = lane; k < mine; k += 64) dst[k] = list[wave][k];
        off += all;
    }
}

// a run of n bits as 32-bit chunks shared out over the blocks, a contiguous range each
struct WhGeometry {
    uint64_t nchunks, nblocks, cpb;
};
WhGeometry wh_geometry(uint64_t n) {
    WhGeometry g;
    g.nchunks = (n + 31) / 32;
    g.nblocks = (g.nchunks + kWhBlock - 1) / kWhBlock;
    if (g.nblocks > kWhMaxBlocks) g.nblocks = kWhMaxBlocks;
    g.cpb = g.nblocks ? (g.nchunks + g.nblocks - 1) / g.nblocks : 0;
    return g;
}

template <int MODE>
void where_launch(CUMO_BIT_DIGIT* a, size_t p, ssize_t s, size_t* idx, uint64_t n, int invert, char* out, size_t elmsz, uint64_t count, size_t p2,
                  ssize_t s2, size_t* idx2, uint64_t* running, uint64_t* block_sums) {
    if (n == 0) return;  // a grid of no blocks is an invalid launch
    const WhGeometry g = wh_geometry(n);
    const uint64_t nchunks = g.nchunks, nblocks = g.nblocks, cpb = g.cpb;
    const int contiguous = (idx == nullptr && s == 1) ? 1 : 0;
    hipStream_t st = current_stream();
    hipLaunchKernelGGL(where_count_kernel, dim3(wh_count_grid(nblocks)), dim3(kWhBlock * kWhGroups), 0, st, a, (uint64_t)p, (int64_t)s, (const size_t*)idx, n,
                       contiguous, invert, nchunks, cpb, nblocks, block_sums, (uint64_t*)nullptr);
    hipLaunchKernelGGL(where_scan_kernel, dim3(1), dim3(kWhBlock), 0, st, block_sums, nblocks, running);
#define WH_SCATTER(ES)                                                                                                                      \
    hipLaunchKernelGGL((where_scatter_kernel<MODE, ES, false>), dim3((unsigned)nblocks), dim3(kWhBlock), 0, st, a, (uint64_t)p, (int64_t)s,     \
                       (const size_t*)idx, n, contiguous, invert, nchunks, cpb, out, count, p2, (int64_t)s2, (const size_t*)idx2,               \
                       (const uint64_t*)block_sums)
    if (elmsz == 4) {
        if constexpr (MODE != 1) WH_SCATTER(4);
    } else {
        WH_SCATTER(8);
    }
#undef WH_SCATTER
    cumo_cuda_runtime_check_kernel_launch();
}

// a tiny fill instead of a memset node, so that a caller may capture the stream
__global__ void where_zero_kernel(uint64_t* p) {
    if (threadIdx.x < 2) p[threadIdx.x] = 0;
}

// z[i] = the element of x at flat (row-major) position pos[i]
struct GatherParams {
    int ndim;
    uint64_t n;
    uint64_t shape[CUMO_NA_MAX_DIMENSION];
    Div31 div[CUMO_NA_MAX_DIMENSION];
    int64_t step[CUMO_NA_MAX_DIMENSION];
    const char* in;
    char* out;
    const char* pos;
};
// PW, EW: bytes per position and per element (4 or 8). SMALL: the view has fewer than
// 2^31 elements, so a position splits over the dimensions with 32-bit multiplies.
template <int PW, int EW, bool SMALL>
__global__ __launch_bounds__(256) void gather_flat_kernel(GatherParams g) {
    typedef typename std::conditional<PW == 4, uint32_t, uint64_t>::type P;
    typedef typename std::conditional<EW == 4, uint32_t, uint64_t>::type E;
    for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < g.n; i += (uint64_t)gridDim.x * 256) {
        const uint64_t r0 = (uint64_t)reinterpret_cast<const P*>(g.pos)[i];
        int64_t off = 0;
        if (SMALL) {
            uint32_t r = (uint32_t)r0;
            for (int d = g.ndim - 1; d > 0; --d) {
                const uint32_t q = div31(r, g.div[d]);
                off += (int64_t)(r - q * (uint32_t)g.shape[d]) * g.step[d];
                r = q;
            }
            off += (int64_t)r * g.step[0];
        } else {
            uint64_t r = r0;
            for (int d = g.ndim - 1; d > 0; --d) {
                const uint64_t m = g.shape[d];
                const uint64_t q = r / m;
                off += (int64_t)(r - q * m) * g.step[d];
                r = q;
            }
            off += (int64_t)r * g.step[0];
        }
        reinterpret_cast<E*>(g.out)[i] = *reinterpret_cast<const E*>(g.in + off);
    }
}

}  // namespace
// What cumo_hip_bit_where_place_kernel_launch does, for a mask that is known to have `hits` of them.
// Elements of a contiguous run are packed as vectors from one hit in 40 on: 2^25 SFloat, fresh operands, at 3 % hits 37.4 us one by one,
// 36.4 packed; at 2 % 33.7 and 35.0, at 0.1 % 25.2 and 30.7 (DFloat 2^24: 30.2 / 30.5, 26.8 / 29.6, 23.0 / 25.3).
void where_place(CUMO_BIT_DIGIT* a, size_t p, ssize_t s, uint64_t n, int invert, const uint64_t* counts, uint64_t hits, const char* x, ssize_t sx,
                 size_t elmsz, char* out) {
    if (n == 0) return;
    const WhGeometry g = wh_geometry(n);
    const int contiguous = s == 1 ? 1 : 0;
    hipStream_t st = current_stream();
#define WH_PLACE(MODE, ES, P2, S2)                                                                                                     \
    hipLaunchKernelGGL((where_scatter_kernel<MODE, ES, true>), dim3((unsigned)g.nblocks), dim3(kWhBlock), 0, st, a, (uint64_t)p, (int64_t)s, \
                       (const size_t*)nullptr, n, contiguous, invert, g.nchunks, g.cpb, out, (uint64_t)0, (size_t)(P2), (int64_t)(S2),      \
                       (const size_t*)nullptr, counts)
    if (x && contiguous && sx == (ssize_t)elmsz && ((uintptr_t)x & (elmsz - 1)) == 0 && hits >= n / 40) {
        const bool nt = stream_past_caches(n * elmsz);
#define WH_PACK(ES, NT)                                                                                                                 \
    hipLaunchKernelGGL((mask_pack_kernel<ES, NT>), dim3((unsigned)g.nblocks), dim3(kWhBlock), 0, st, a, (uint64_t)p, n, invert, g.nchunks, g.cpb, \
                       out, x, counts)
        if (elmsz == 4) { if (nt) WH_PACK(4, true); else WH_PACK(4, false); }
        else { if (nt) WH_PACK(8, true); else WH_PACK(8, false); }
#undef WH_PACK
    } else if (x) {
        if (elmsz == 4) WH_PLACE(2, 4, (uintptr_t)x, sx);
        else WH_PLACE(2, 8, (uintptr_t)x, sx);
    } else {
        if (elmsz == 4) WH_PLACE(0, 4, 0, 0);
        else WH_PLACE(0, 8, 0, 0);
    }
#undef WH_PLACE
    cumo_cuda_runtime_check_kernel_launch();
}

}  // namespace cumo_hip

using namespace cumo_hip;

extern "C" {

// reference: where_kernel.cu:83-89
char* cumo_bit_where_scratch_new(void) {
    char* scratch = cumo_cuda_runtime_malloc((2 + kWhMaxBlocks) * sizeof(uint64_t));
    if (!scratch) return nullptr;
    hipLaunchKernelGGL(where_zero_kernel, dim3(1), dim3(64), 0, current_stream(), reinterpret_cast<uint64_t*>(scratch));
    cumo_cuda_runtime_check_kernel_launch();
    return scratch;
}

// reference: where_kernel.cu:91-107
void cumo_bit_where_kernel_launch(CUMO_BIT_DIGIT* a, size_t p, ssize_t s, size_t* idx, uint64_t n, int invert, char* out, size_t elmsz, uint64_t count,
                                  char* scratch) {
    uint64_t* running = reinterpret_cast<uint64_t*>(scratch) + (invert ? 1 : 0);
    where_launch<0>(a, p, s, idx, n, invert, out, elmsz, count, 0, 0, nullptr, running, reinterpret_cast<uint64_t*>(scratch) + 2);
}

// reference: mask_kernel.cu:36-54
void cumo_bit_mask_kernel_launch(CUMO_BIT_DIGIT* a, size_t p, ssize_t s, size_t* idx, uint64_t n, size_t* out, size_t p2, ssize_t s2, size_t* idx2,
                                 char* scratch) {
    where_launch<1>(a, p, s, idx, n, 0, reinterpret_cast<char*>(out), sizeof(size_t), 0, p2, s2, idx2, reinterpret_cast<uint64_t*>(scratch),
                       reinterpret_cast<uint64_t*>(scratch) + 2);
}

// The same compaction for a caller that sizes the result in between: the blocks' counts of one run
// (cumo_hip_bit_where_blocks(n) of them, every one written), which the caller reads back and adds
// up, then the placement, where every block adds up the counts before it. Two launches instead of
// a count for the size plus the three above.
size_t cumo_hip_bit_where_blocks(uint64_t n) { return (size_t)wh_geometry(n).nblocks; }

void cumo_hip_bit_where_count_kernel_launch(CUMO_BIT_DIGIT* a, size_t p, ssize_t s, uint64_t n, int invert, uint64_t* counts) {
    if (n == 0) return;
    const WhGeometry g = wh_geometry(n);
    hipLaunchKernelGGL(where_count_kernel, dim3(wh_count_grid(g.nblocks)), dim3(kWhBlock * kWhGroups), 0, current_stream(), a, (uint64_t)p, (int64_t)s,
                       (const size_t*)nullptr, n, s == 1 ? 1 : 0, invert, g.nchunks, g.cpb, g.nblocks, counts, (uint64_t*)nullptr);
    cumo_cuda_runtime_check_kernel_launch();
}

// The same, and the counts on the host when the call returns: the kernel writes them into pinned host memory of the
// calling thread as well, and the host looks at that memory until every share's count is there. They are the last thing
// the stream has been given, so nothing earlier is still running then. A stream that has not come this far within
// kWhLookNs is waited for instead, which also reports what may have gone wrong on it. Looking costs the caller's core
// what the runtime's own wait costs it, and saves the wait's way through a signal: SFloat 104 x 96 x[mask]
// 20.9 -> 15.8 us, mask.where() 20.0 -> 15.2 us.
// host_counts: cumo_hip_bit_where_blocks(n) words of ordinary host memory.
constexpr int64_t kWhLookNs = 2000000;
int cumo_hip_bit_where_count_to_host(CUMO_BIT_DIGIT* a, size_t p, ssize_t s, uint64_t n, int invert, uint64_t* counts, uint64_t* host_counts) {
    if (n == 0) return CUMO_HIP_OK;
    const WhGeometry g = wh_geometry(n);
    static thread_local uint64_t* pinned = nullptr;   // kWhMaxBlocks words, kept for the thread's lifetime
    if (pinned == nullptr) {
        void* m = nullptr;
        if (!hip_ok(hipHostMalloc(&m, kWhMaxBlocks * sizeof(uint64_t), hipHostMallocMapped | hipHostMallocPortable | hipHostMallocCoherent), "hipHostMalloc"))
            return CUMO_HIP_ERROR_RUNTIME;
        pinned = static_cast<uint64_t*>(m);
    }
    std::memset(pinned, 0, g.nblocks * sizeof(uint64_t));
    hipStream_t st = current_stream();
    // The launch's own status: hipGetLastError would answer for an earlier call of the thread as well, and a kernel that has been
    // queued must be waited for, or its counts could be taken for the next call's.
    uint64_t first = p, words = n, *host = pinned;
    int64_t step = s;
    const size_t* idx = nullptr;
    int contiguous = s == 1 ? 1 : 0;
    WhGeometry kg = g;
    void* args[] = {&a, &first, &step, &idx, &words, &contiguous, &invert, &kg.nchunks, &kg.cpb, &kg.nblocks, &counts, &host};
    const hipError_t launched = hipLaunchKernel(reinterpret_cast<const void*>(where_count_kernel), dim3(wh_count_grid(g.nblocks)), dim3(kWhBlock * kWhGroups), args, 0, st);
    if (launched != hipSuccess) {
        (void)hipGetLastError();
        report_hip_error(launched, "kernel launch");
        return CUMO_HIP_ERROR_RUNTIME;
    }
    // (under capture nothing has been queued that could leave a count: the runtime's wait refuses at once, as it always has)
    hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(st, &capturing) != hipSuccess) {
        (void)hipGetLastError();
        capturing = hipStreamCaptureStatusActive;
    }
    if (capturing != hipStreamCaptureStatusNone && !hip_ok(hipStreamSynchronize(st), "hipStreamSynchronize")) return CUMO_HIP_ERROR_RUNTIME;
    const auto begin = std::chrono::steady_clock::now();
    uint64_t b = 0;
    for (unsigned looks = 0; b < g.nblocks; ++looks) {
        while (b < g.nblocks && __atomic_load_n(pinned + b, __ATOMIC_ACQUIRE) != 0) ++b;
        if (b == g.nblocks) break;
        __builtin_ia32_pause();
        if ((looks & 63u) == 63u && (std::chrono::steady_clock::now() - begin) > std::chrono::nanoseconds(kWhLookNs)) {
            if (!hip_ok(hipStreamSynchronize(st), "hipStreamSynchronize")) return CUMO_HIP_ERROR_RUNTIME;
            break;
        }
    }
    if (!wait_trouble_check()) return CUMO_HIP_ERROR_RUNTIME;
    for (b = 0; b < g.nblocks; ++b) {
        const uint64_t word = __atomic_load_n(pinned + b, __ATOMIC_RELAXED);
        if (word == 0) {
            report_error(CUMO_HIP_ERROR_RUNTIME, 0, "where: a block left no count");
            return CUMO_HIP_ERROR_RUNTIME;
        }
        host_counts[b] = word - 1;
    }
    cumo_cuda_runtime_check_kernel_launch();   // (what an earlier call left on the thread, as behind every other launch)
    return CUMO_HIP_OK;
}

// x == NULL: out[o] = the position in the run of the o-th hit, as an elmsz-byte integer (4 or 8);
// otherwise out[o] = the element (elmsz 4 or 8 bytes) at x + j*sx of the o-th hit j.
void cumo_hip_bit_where_place_kernel_launch(CUMO_BIT_DIGIT* a, size_t p, ssize_t s, uint64_t n, int invert, const uint64_t* counts, const char* x,
                                            ssize_t sx, size_t elmsz, char* out) {
    where_place(a, p, s, n, invert, counts, n, x, sx, elmsz, out);   // (as of a mask with many hits)
}

void cumo_hip_gather_flat_kernel_launch(const cumo_hip_gather_flat_t* d) {
    if (!d || d->n == 0) return;
    GatherParams g;
    std::memset(&g, 0, sizeof(g));
    // dimensions that follow one another in memory count as one; size-1 dimensions drop out
    uint64_t total = 1;
    int nd = 0;
    for (int k = 0; k < d->ndim && k < CUMO_NA_MAX_DIMENSION; ++k) {
        total *= d->shape[k];
        if (d->shape[k] == 1) continue;
        if (nd > 0 && g.step[nd - 1] == (int64_t)d->step[k] * (int64_t)d->shape[k]) {
            g.shape[nd - 1] *= d->shape[k];
            g.step[nd - 1] = d->step[k];
        } else {
            g.shape[nd] = d->shape[k];
            g.step[nd] = d->step[k];
            ++nd;
        }
    }
    if (nd == 0) {
        g.shape[0] = 1;
        nd = 1;
    }
    g.ndim = nd;
    const bool small = total < (1ull << 31);
    if (small) {
        for (int k = 0; k < nd; ++k) g.div[k] = div31_make((uint32_t)g.shape[k]);
    }
    g.n = d->n;
    g.in = d->in;
    g.out = d->out;
    g.pos = d->pos;
    uint64_t grid = (d->n + 255) / 256;
    if (grid > 65536) grid = 65536;
    hipStream_t st = current_stream();
#define WH_GATHER(PW, EW)                                                                                              \
    do {                                                                                                               \
        if (small) hipLaunchKernelGGL((gather_flat_kernel<PW, EW, true>), dim3((unsigned)grid), dim3(256), 0, st, g);  \
        else hipLaunchKernelGGL((gather_flat_kernel<PW, EW, false>), dim3((unsigned)grid), dim3(256), 0, st, g);       \
    } while (0)
    if (d->pos_elmsz == 4 && d->elmsz == 4) WH_GATHER(4, 4);
    else if (d->pos_elmsz == 4) WH_GATHER(4, 8);
    else if (d->elmsz == 4) WH_GATHER(8, 4);
    else WH_GATHER(8, 8);
#undef WH_GATHER
    cumo_cuda_runtime_check_kernel_launch();
}

}  // extern "C"
