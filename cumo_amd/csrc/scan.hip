// cumsum / cumprod: inclusive scans along one run of a view.
//
// Replaces narray/gen/tmpl/cum_kernel.cu of the reference, which hands each run
// to thrust::inclusive_scan (one call per run, walked on the host:
// narray/gen/tmpl/cum.c:12-46). The operators are the reference's
// (types/real_accum_kernel.h:12-26, xint_macro_kernel.h:46-47); the nan forms
// treat NaN as "nothing yet", which makes them associative like the plain ones.
// Like a sum, a parallel float scan does not add strictly left to right.
//
// The forms, by layout:
//   scan_rows_kernel        one block per run, tile after tile with the running value
//                           carried along: many runs (an axis of a matrix), or short ones;
//   scan_short_kernel       many short runs, as many to a wave as its registers hold (scan_short.hip);
//   scan_rows_whole_kernel  the same for contiguous runs of 64 vectors or more, a chunk of them at a time held in
//                           registers wave by wave, the last chunk maybe partly there;
//   scan_chain_kernel       one contiguous run, or a few long ones, in one pass: tiles hand their
//                           totals on through words in memory (read once, written once);
//   scan_chain_alone_kernel those few, a block to each, where the stream keeps no such words: the same bits;
//   three launches          one long run that is strided: per-tile totals, a scan of the
//                           totals, then every tile scans itself from its offset (reads the
//                           input twice);
//   scan_cols_chain_kernel  runs that lie across memory (down the rows of a matrix) in one
//                           pass, tiles of 256 rows or more handing on their column totals;
//   scan_cols_kernel        other runs across memory, in segments and two passes.
// Inside a tile each lane owns 8 consecutive elements: it scans them in registers,
// the lane totals are scanned across the wave with shuffles and the four wave
// totals through LDS. Everything is in a fixed order, so results do not change
// from launch to launch.
#include "common.h"
#include "scan_ops.h"
#include "wait_ctl.h"

#include <cstdlib>
#include <cstring>
#include <mutex>

namespace cumo_hip {
namespace {

constexpr int kScanBlock = 256;
constexpr int kScanPer = 8;                         // elements per lane
constexpr int kScanTile = kScanBlock * kScanPer;    // 2048

template <class T>
__device__ __forceinline__ T scan_shfl_up(T v, unsigned d) {
    if constexpr (sizeof(T) == 8) {
        union { T t; uint32_t w[2]; } a, b;
        a.t = v;
        b.w[0] = __shfl_up(a.w[0], d);
        b.w[1] = __shfl_up(a.w[1], d);
        return b.t;
    } else {
        union { T t; uint32_t w; } a, b;
        a.t = v;
        b.w = __shfl_up(a.w, d);
        return b.t;
    }
}

// Inclusive scan of one tile held as v[kScanPer] per lane (element k of lane t is
// tile position t * kScanPer + k; cnt = how many positions of the tile exist).
// `carry` is the running value before the tile and has_carry says whether there is
// one. Returns the running value after the tile in every lane (has_carry becomes true
// when the tile is not empty).
template <class T, class Op>
__device__ __forceinline__ void scan_tile(T (&v)[kScanPer], int cnt, T& carry, bool& has_carry) {
    constexpr int NWAVES = kScanBlock / 64;
    __shared__ T wave_tot[NWAVES];
    __shared__ int wave_has[NWAVES];
    const int t = threadIdx.x;
    const int base = t * kScanPer;
    int mine = cnt - base;  // how many of this lane's elements exist
    mine = mine < 0 ? 0 : (mine > kScanPer ? kScanPer : mine);
    // lane-local inclusive scan
#pragma unroll
    for (int k = 1; k < kScanPer; ++k)
        if (k < mine) v[k] = Op::apply(v[k - 1], v[k]);
    T tot = mine > 0 ? v[mine - 1] : T();
    bool has = mine > 0;
    // inclusive scan of the lane totals across the wave
    const int lane = t & 63;
#pragma unroll
    for (unsigned d = 1; d < 64; d <<= 1) {
        const T o = scan_shfl_up(tot, d);
        const int oh = __shfl_up((int)has, d);
        if (lane >= (int)d && oh) {
            tot = has ? Op::apply(o, tot) : o;
            has = true;
        }
    }
    const int w = t >> 6;
    if (lane == 63) {
        wave_tot[w] = tot;
        wave_has[w] = has ? 1 : 0;
    }
    __syncthreads();
    // what precedes this lane: the carry, the earlier waves, the earlier lanes of its wave
    T pre = carry;
    bool pre_has = has_carry;
    for (int j = 0; j < w; ++j) {
        if (wave_has[j]) {
            pre = pre_has ? Op::apply(pre, wave_tot[j]) : wave_tot[j];
            pre_has = true;
        }
    }
    T run = carry;          // the running value after the whole tile, for every lane
    bool run_has = has_carry;
#pragma unroll
    for (int j = 0; j < NWAVES; ++j) {
        if (wave_has[j]) {
            run = run_has ? Op::apply(run, wave_tot[j]) : wave_tot[j];
            run_has = true;
        }
    }
    const T lane_excl = scan_shfl_up(tot, 1);
    const int lane_excl_has = __shfl_up((int)has, 1);
    if (lane > 0 && lane_excl_has) {
        pre = pre_has ? Op::apply(pre, lane_excl) : lane_excl;
        pre_has = true;
    }
    if (pre_has) {
#pragma unroll
        for (int k = 0; k < kScanPer; ++k)
            if (k < mine) v[k] = Op::apply(pre, v[k]);
    }
    __syncthreads();  // wave_tot is written again by the next tile
    carry = run;
    has_carry = run_has;
}

template <class T>
__device__ __forceinline__ void scan_load(const char* p, int64_t s, uint64_t first, int cnt, T (&v)[kScanPer]) {
    const int base = threadIdx.x * kScanPer;
    if (s == (int64_t)sizeof(T) && base + kScanPer <= cnt && ((reinterpret_cast<uintptr_t>(p) + (first + base) * sizeof(T)) & 15) == 0) {
        typedef uint32_t u4 __attribute__((ext_vector_type(4)));
        constexpr int NV = (int)(kScanPer * sizeof(T) / 16);
        union { T t[kScanPer]; u4 q[NV]; } u;
        const u4* src = reinterpret_cast<const u4*>(p + (first + base) * sizeof(T));
#pragma unroll
        for (int i = 0; i < NV; ++i) u.q[i] = src[i];
#pragma unroll
        for (int k = 0; k < kScanPer; ++k) v[k] = u.t[k];
        return;
    }
#pragma unroll
    for (int k = 0; k < kScanPer; ++k)
        if (base + k < cnt) v[k] = *reinterpret_cast<const T*>(p + (int64_t)(first + base + k) * s);
}

template <class T>
__device__ __forceinline__ void scan_store(char* p, int64_t s, uint64_t first, int cnt, const T (&v)[kScanPer]) {
    const int base = threadIdx.x * kScanPer;
    if (s == (int64_t)sizeof(T) && base + kScanPer <= cnt && ((reinterpret_cast<uintptr_t>(p) + (first + base) * sizeof(T)) & 15) == 0) {
        typedef uint32_t u4 __attribute__((ext_vector_type(4)));
        constexpr int NV = (int)(kScanPer * sizeof(T) / 16);
        union { T t[kScanPer]; u4 q[NV]; } u;
#pragma unroll
        for (int k = 0; k < kScanPer; ++k) u.t[k] = v[k];
        u4* dst = reinterpret_cast<u4*>(p + (first + base) * sizeof(T));
#pragma unroll
        for (int i = 0; i < NV; ++i) dst[i] = u.q[i];
        return;
    }
#pragma unroll
    for (int k = 0; k < kScanPer; ++k)
        if (base + k < cnt) *reinterpret_cast<T*>(p + (int64_t)(first + base + k) * s) = v[k];
}

template <class T, class Op>
__global__ __launch_bounds__(kScanBlock) void scan_rows_kernel(ScanRowsParams p) {
    for (uint64_t row = blockIdx.x; row < p.rows; row += gridDim.x) {
        const char* in;
        char* out;
        scan_run_start(p, row, in, out);
        T carry = T();
        bool has_carry = false;
        for (uint64_t first = 0; first < p.n; first += kScanTile) {
            const uint64_t left = p.n - first;
            const int cnt = left < (uint64_t)kScanTile ? (int)left : kScanTile;
            T v[kScanPer];
            scan_load<T>(in, p.s_in, first, cnt, v);
            scan_tile<T, Op>(v, cnt, carry, has_carry);
            scan_store<T>(out, p.s_out, first, cnt, v);
        }
    }
}

template <class T>
__device__ __forceinline__ T scan_shfl_xor(T v, unsigned m) {
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

// phase 1 of the three-launch form: the total of each tile, by a plain fold (the
// operators are associative and commutative: lane-local fold, wave butterfly, four LDS
// slots), which is lighter than the scan of the tile. A tile of nothing but NaN under a
// nan operator has the total NaN, which the operator reads as "nothing". The last tile
// may be partial; nothing comes after it, so its total is never used and none is formed.
template <class T, class Op>
__global__ __launch_bounds__(kScanBlock) void scan_tile_totals_kernel(const char* in, int64_t s_in, uint64_t n, T* totals) {
    __shared__ T wave_tot[kScanBlock / 64];
    const uint64_t first = (uint64_t)blockIdx.x * kScanTile;
    const uint64_t left = n - first;
    if (left < (uint64_t)kScanTile) {
        if (threadIdx.x == 0) totals[blockIdx.x] = T();
        return;
    }
    T v[kScanPer];
    scan_load<T>(in, s_in, first, kScanTile, v);
    T t = v[0];
#pragma unroll
    for (int k = 1; k < kScanPer; ++k) t = Op::apply(t, v[k]);
#pragma unroll
    for (unsigned m = 32; m > 0; m >>= 1) t = Op::apply(t, scan_shfl_xor(t, m));
    if ((threadIdx.x & 63) == 0) wave_tot[threadIdx.x >> 6] = t;
    __syncthreads();
    if (threadIdx.x == 0) {
        T tot = wave_tot[0];
#pragma unroll
        for (int w = 1; w < kScanBlock / 64; ++w) tot = Op::apply(tot, wave_tot[w]);
        totals[blockIdx.x] = tot;
    }
}

// phase 3: every block scans its tiles, starting from the scanned total of the blocks before it
template <class T, class Op>
__global__ __launch_bounds__(kScanBlock) void scan_apply_kernel(const char* in, int64_t s_in, char* out, int64_t s_out, uint64_t n, uint64_t per,
                                                                const T* scanned_totals) {
    bool hc = blockIdx.x > 0;
    T carry = hc ? scanned_totals[blockIdx.x - 1] : T();
    const uint64_t begin = (uint64_t)blockIdx.x * per * kScanTile;
    for (uint64_t k = 0; k < per; ++k) {
        const uint64_t first = begin + k * kScanTile;
        if (first >= n) break;
        const uint64_t left = n - first;
        const int cnt = left < (uint64_t)kScanTile ? (int)left : kScanTile;
        T v[kScanPer];
        scan_load<T>(in, s_in, first, cnt, v);
        scan_tile<T, Op>(v, cnt, carry, hc);
        scan_store<T>(out, s_out, first, cnt, v);
    }
}

// ---- one long run in one pass ----------------------------------------------------
// Every block takes the next tile from a ticket (so a tile only ever waits for tiles whose
// blocks are already running), scans it in registers, publishes the tile's total and then
// needs the total of everything before it. That comes in a fixed shape, so that results
// do not change from launch to launch: tiles form groups of 64 and groups form supergroups
// of 64; the last tile of a group also publishes the group's total and the last tile of a
// supergroup the supergroup's. A tile folds, each with one scan across a wave, the totals
// of the earlier tiles of its group, of the earlier groups of its supergroup and of the
// earlier supergroups. Reads the input once and writes the output once.
// A published value travels as 64-bit words {the launch's number, 32 bits of the value},
// stored and loaded with agent-scope atomics: a word is there when its upper half is the
// launch's number, no fence needed. The words live in a region that the stream keeps from
// launch to launch (chain_words_acquire below), so nothing is cleared: what an earlier launch
// left carries another number, and the ticket word just counts on (a launch takes exactly one
// ticket per block; the host knows where it stood). A wait gives up after kChainSpinLimit polls
// (it cannot be reached while every tile before this one has a running block); it then counts
// that and raises the host's give-up word (wait_ctl.h), so the next point where the host waits
// for the device reports the launch as failed.
// The ticket is a relaxed add on purpose: it hands out tile numbers and publishes nothing; what
// a tile publishes travels whole in its tagged words.
constexpr uint32_t kChainSpinLimit = 1u << 22;
constexpr uint64_t kChainMaxTiles = 64ull * 64ull * 64ull;
constexpr uint64_t kChainSmallBytes = 16 << 10;

template <class T>
struct ScanChain {
    static constexpr int W = (int)(sizeof(T) / 4);
    WaitCtl* wait;     // where a look-back that gives up reports it
    uint32_t* ticket;
    uint64_t* tile;    // [run][n_tiles][W]
    uint64_t* group;   // [run][n_groups][W]
    uint64_t* super;   // [run][n_supers][W]
    uint32_t n_tiles, n_groups, n_supers;  // of one run
    uint32_t flag;         // the upper half of a word of this launch
    uint32_t ticket_base;  // what the ticket word held before this launch
};

template <class T>
__device__ __forceinline__ void chain_publish(uint64_t* slot, T value, uint32_t flag) {
    constexpr int W = ScanChain<T>::W;
    union { T t; uint32_t w[W]; } u;
    u.t = value;
#pragma unroll
    for (int i = 0; i < W; ++i)
        __hip_atomic_store(slot + i, ((uint64_t)flag << 32) | u.w[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// one look at a published value: true when all of it is there
template <class T>
__device__ __forceinline__ bool chain_peek(const uint64_t* slot, T& value, uint32_t flag) {
    constexpr int W = ScanChain<T>::W;
    union { T t; uint32_t w[W]; } u;
    uint64_t x[W];
#pragma unroll
    for (int i = 0; i < W; ++i) x[i] = __hip_atomic_load(slot + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    bool all = true;
#pragma unroll
    for (int i = 0; i < W; ++i) {
        all = all && (uint32_t)(x[i] >> 32) == flag;
        u.w[i] = (uint32_t)x[i];
    }
    value = u.t;
    return all;
}

template <class T, class Op>
__device__ __forceinline__ void chain_join(T& a, bool& a_has, T b, bool b_has) {  // a = a (+) b, a the earlier
    if (b_has) {
        a = a_has ? Op::apply(a, b) : b;
        a_has = true;
    }
}

// Inclusive scan of K values of every lane across the wave, side by side: inside quarters of 16 lanes, then the
// quarters' totals from lane 15 of the first and third, then the half's from lane 31.
template <class T, class Op, int K>
__device__ __forceinline__ void scan_across_wave(T (&x)[K]) {
    const unsigned lane = threadIdx.x & 63u;
#define CUMO_SCAN_STEP(CTRL, COND)                        \
    _Pragma("unroll") for (int k = 0; k < K; ++k) {       \
        const T o = scan_dpp<CTRL>(x[k]);                 \
        x[k] = (COND) ? Op::apply(o, x[k]) : x[k];        \
    }
    CUMO_SCAN_STEP(0x111, (lane & 15u) >= 1)   // row_shr:1
    CUMO_SCAN_STEP(0x112, (lane & 15u) >= 2)   // row_shr:2
    CUMO_SCAN_STEP(0x114, (lane & 15u) >= 4)   // row_shr:4
    CUMO_SCAN_STEP(0x118, (lane & 15u) >= 8)   // row_shr:8
    CUMO_SCAN_STEP(0x142, (lane & 16u) != 0)   // row_bcast:15
    CUMO_SCAN_STEP(0x143, lane >= 32)          // row_bcast:31
#undef CUMO_SCAN_STEP
}

// x of the first `count` lanes folded in a fixed shape, the same for the whole wave; has: whether there is one
template <class T, class Op>
__device__ __forceinline__ void chain_fold_lanes(T& x, bool& has, uint32_t count) {
    has = count > 0;
    if (!has) return;
    T k[1] = {x};
    scan_across_wave<T, Op, 1>(k);
    x = scan_read_lane(k[0], count - 1);
}

// What a tile needs from the tiles before it, through the published totals (wave 0 of the
// block; every lane returns the same). Lane l wants the l-th earlier tile of this group, the
// l-th earlier group of this supergroup and the l-th supergroup. Whatever this tile waits
// for, the tile just before it publishes last, so one lane first polls that one word, with
// pauses (64 lanes of every running block polling would flood the memory system); then every
// lane looks at its own words, all in flight together, until they are there.
template <class T, class Op>
__device__ __forceinline__ void chain_look_back(const ScanChain<T>& c, uint32_t t, T total, T& prefix, bool& prefix_has) {
    constexpr int W = ScanChain<T>::W;
    const unsigned lane = threadIdx.x & 63u;
    t = (uint32_t)__builtin_amdgcn_readfirstlane(t);
    const uint32_t pos = t & 63u, g = t >> 6, gpos = g & 63u, sg = g >> 6;
    if (lane == 0) chain_publish<T>(c.tile + (size_t)t * W, total, c.flag);
    T x = T(), y = T(), z = T();
    const bool has_x = lane < pos, has_y = lane < gpos, has_z = lane < sg;
    bool need_x = has_x, need_y = has_y, need_z = has_z;
    const uint64_t* px = c.tile + (size_t)(g * 64u + lane) * W;
    const uint64_t* py = c.group + (size_t)(sg * 64u + lane) * W;
    const uint64_t* pz = c.super + (size_t)lane * W;
    uint32_t polls = 0;
    const uint32_t spin_limit = wait_limit(c.wait, kChainSpinLimit);
    if (t > 0) {
        // the last word that the tile before this one publishes
        const uint64_t* latest = pos > 0 ? c.tile + (size_t)(t - 1) * W + (W - 1)
                                         : (gpos > 0 ? c.group + (size_t)(g - 1) * W + (W - 1) : c.super + (size_t)(sg - 1) * W + (W - 1));
        if (lane == 0) {
            // (running out of looks here is not yet a failure: the loop below looks again and reports)
            while ((uint32_t)(__hip_atomic_load(latest, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >> 32) != c.flag) {
                if (++polls > spin_limit) break;
                __builtin_amdgcn_s_sleep(16);
            }
        }
    }
    // A tile that closes its group publishes the group's total as soon as the group's tiles
    // are in, before it has everything it needs itself (and likewise the supergroup's):
    // otherwise every group would wait for the group before it, one memory round trip each.
    const bool closes_group = pos == 63u, closes_super = closes_group && gpos == 63u;
    bool group_out = !closes_group, super_out = !closes_super;
    bool xh = false, yh = false, zh = false;
    bool x_folded = false, y_folded = false;
    T gt = T();
    for (;;) {
        if (need_x) need_x = !chain_peek<T>(px, x, c.flag);
        if (need_y) need_y = !chain_peek<T>(py, y, c.flag);
        if (need_z) need_z = !chain_peek<T>(pz, z, c.flag);
        if (!x_folded && __ballot(need_x) == 0) {
            chain_fold_lanes<T, Op>(x, xh, pos);
            x_folded = true;
            if (!group_out) {
                gt = Op::apply(x, total);
                if (lane == 0) chain_publish<T>(c.group + (size_t)g * W, gt, c.flag);
                group_out = true;
            }
        }
        if (!y_folded && x_folded && __ballot(need_y) == 0) {
            chain_fold_lanes<T, Op>(y, yh, gpos);
            y_folded = true;
            if (!super_out) {
                if (lane == 0) chain_publish<T>(c.super + (size_t)sg * W, Op::apply(y, gt), c.flag);
                super_out = true;
            }
        }
        if (__ballot(need_x || need_y || need_z) == 0) break;
        if (++polls > spin_limit) {
            if (lane == 0) wait_gave_up(c.wait, WAIT_SCAN);
            break;
        }
        __builtin_amdgcn_s_sleep(16);
    }
    if (!x_folded) chain_fold_lanes<T, Op>(x, xh, pos);  // (only after giving up)
    if (!y_folded) chain_fold_lanes<T, Op>(y, yh, gpos);
    chain_fold_lanes<T, Op>(z, zh, sg);
    chain_join<T, Op>(z, zh, y, yh);
    chain_join<T, Op>(z, zh, x, xh);
    prefix = z;
    prefix_has = zh;
}

// Both sides are contiguous and aligned as their elements are. A tile goes wave by wave: each of the block's
// four or eight waves owns a part of the tile as R rows of 64 vectors, lane l holding vector l of every
// row (each load and store covers 1 KiB without gaps); the rows are scanned side by side, the
// waves meet once, in LDS, and what is left to add after the look-back is one value per
// wave, so only the tile's elements stay in registers while the block waits. The ragged last
// tile of a run goes the same way with what it lacks read as zeros (sub-tile by sub-tile through the block-wide
// scan, its input read twice, it took as long as everything before it: SFloat 1975200 19.1 -> 8.9 us, 7489984 28.8 -> 14.0; and
// without that code a block of doubles needs 110 registers a lane instead of 165, so two wide ones share a compute unit: DFloat 2^24
// 58.3 -> 54.6, 7489984 29.8 -> 25.7).
// Several runs (MANY) go level by level: the first tile of every run, then the second of every run, so that a tile waits only for
// tiles whose blocks are running, as with one run. Bound by what a block waits for with nothing in flight: its ticket and the look-back. The
// steps across a wave go by data-parallel primitives: shuffles put 16 rows times six steps through
// the LDS unit (64 KiB tiles: 2^24 DFloat 75 -> 63 us, 2^22 24.1 -> 20.2, 2^26 SFloat 114 -> 109; 128 KiB
// tiles: 72 -> 57, 20.5 -> 16.4, 111 -> 103). The three launches take 155 us for 2^26 SFloat. Slower, measured: 32 KiB
// tiles; persistent blocks that stage the next tile into LDS with a wave of their own for tickets
// and look-backs (2^24 DFloat 67 us with 64 KiB tiles, 89 with 32, 141 with 16: the tickets; with
// tiles dealt out by block index, which could wait for a block that is not running, 63 with 32).
struct ChainShared {
    uint32_t tile;
    int prefix_has;
};

// RAGGED: only the first nelem elements from `first` on exist; the others read as zeros (they lie
// after everything that exists, so what they add to never reaches an element that is stored).
// The one vector that is partly there goes element by element: nothing is read past the run.
template <class T, bool NT, int R, bool RAGGED = false>
__device__ __forceinline__ void chain_issue_loads(const char* in, uint64_t first, ScanVec<T> (&v)[R], uint32_t nelem = 0, int w = threadIdx.x >> 6) {
    typedef typename ScanVec<T>::u4 u4;
    constexpr int V = ScanVec<T>::V;
    const unsigned lane = threadIdx.x & 63u;
    const u4* src = reinterpret_cast<const u4*>(in + (first + (uint64_t)w * (R * 64 * V)) * sizeof(T)) + lane;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        if (RAGGED) {
            const u4 zero = {0u, 0u, 0u, 0u};
            v[r].q = zero;
            const uint32_t e0 = ((uint32_t)(w * R * 64 + r * 64) + lane) * V;
            if (e0 + V <= nelem) {
                v[r].q = NT ? __builtin_nontemporal_load(src + r * 64) : src[r * 64];
            } else if (e0 < nelem) {
                const T* s1 = reinterpret_cast<const T*>(src + r * 64);
#pragma unroll
                for (int e = 0; e < V; ++e)
                    if (e0 + e < nelem) v[r].e[e] = s1[e];
            }
        } else {
            v[r].q = NT ? __builtin_nontemporal_load(src + r * 64) : src[r * 64];
        }
    }
}

// The rows of one wave in v (already loaded) scanned by themselves; returns their total. Eight rows at a time, so that what
// is in flight beside the tile stays in registers (a lane of doubles has 168 of them; none is spilled).
template <class T, class Op, int R>
__device__ __forceinline__ T chain_scan_wave(ScanVec<T> (&v)[R]) {
    constexpr int V = ScanVec<T>::V;
    constexpr int K = R < 8 ? R : 8;
    static_assert(R % K == 0, "rows in whole groups");
    const unsigned lane = threadIdx.x & 63u;
    T run = T();  // the rows so far
#pragma unroll
    for (int r0 = 0; r0 < R; r0 += K) {
        T inc[K];
#pragma unroll
        for (int k = 0; k < K; ++k) {
#pragma unroll
            for (int e = 1; e < V; ++e) v[r0 + k].e[e] = Op::apply(v[r0 + k].e[e - 1], v[r0 + k].e[e]);
            inc[k] = v[r0 + k].e[V - 1];
        }
        scan_across_wave<T, Op, K>(inc);   // the lane totals of each row (the rows are independent)
        // every element takes on what precedes its vector inside the wave's part
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const T ex = scan_dpp<0x138>(inc[k]);        // the lanes before, in this row (wave_shr:1)
            const T row = scan_read_lane(inc[k], 63);    // the whole row
            T before = ex;
            if (r0 + k > 0) before = lane > 0 ? Op::apply(run, ex) : run;
            if (r0 + k > 0 || lane > 0) {
#pragma unroll
                for (int e = 0; e < V; ++e) v[r0 + k].e[e] = Op::apply(before, v[r0 + k].e[e]);
            }
            run = r0 + k == 0 ? row : Op::apply(run, row);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    return run;
}

// the total of a tile from its waves' totals, and what precedes wave w in it (for wave 0: nothing)
template <class T, class Op, int NW>
__device__ __forceinline__ void chain_fold_waves(const T* s_wave_tot, int w, T& total, T& wave_pre) {
    total = s_wave_tot[0];
    wave_pre = T();
#pragma unroll
    for (int j = 1; j < NW; ++j) {
        if (j == w) wave_pre = total;
        total = Op::apply(total, s_wave_tot[j]);
    }
}

// The tile in v (already loaded) scanned by itself: afterwards every element holds the running
// value from the start of its wave's part, `total` is the tile's total and `wave_pre` the
// total of the waves before this one (for wave 0: nothing). One barrier, met by every thread.
template <class T, class Op, int R>
__device__ __forceinline__ void chain_scan_tile(ScanVec<T> (&v)[R], T* s_wave_tot, T& total, T& wave_pre) {
    const int w = threadIdx.x >> 6;
    const T run = chain_scan_wave<T, Op, R>(v);
    if ((threadIdx.x & 63u) == 0) s_wave_tot[w] = run;
    __syncthreads();
    chain_fold_waves<T, Op, kScanBlock / 64>(s_wave_tot, w, total, wave_pre);
}

// adds what precedes the tile (if anything) and the earlier waves' total, and stores (pieces: see store_form.h)
template <class T, class Op, bool NT, int R, bool RAGGED = false>
__device__ __forceinline__ void chain_store_tile(char* out, uint64_t first, ScanVec<T> (&v)[R], T head, bool head_has, T wave_pre, bool pieces,
                                                 uint32_t nelem = 0, int w = threadIdx.x >> 6) {
    typedef typename ScanVec<T>::u4 u4;
    constexpr int V = ScanVec<T>::V;
    const unsigned lane = threadIdx.x & 63u;
    if (w > 0) {
        head = head_has ? Op::apply(head, wave_pre) : wave_pre;
        head_has = true;
    }
    u4* dst = reinterpret_cast<u4*>(out + (first + (uint64_t)w * (R * 64 * V)) * sizeof(T)) + lane;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        if (head_has) {
#pragma unroll
            for (int e = 0; e < V; ++e) v[r].e[e] = Op::apply(head, v[r].e[e]);
        }
        if (RAGGED) {
            const uint32_t e0 = ((uint32_t)(w * R * 64 + r * 64) + lane) * V;
            if (e0 >= nelem) continue;
            if (e0 + V > nelem) {
                T* d1 = reinterpret_cast<T*>(dst + r * 64);
#pragma unroll
                for (int e = 0; e < V; ++e)
                    if (e0 + e < nelem) d1[e] = v[r].e[e];
                continue;
            }
        }
        store_vector<NT>(dst + r * 64, v[r].q, pieces);
    }
}

// Many runs, each contiguous on both sides (64 vectors at least, aligned as their elements are):
// one block per run, chunk after chunk of R * 256 vectors in the same wave-by-wave form,
// the running value handed on in a register; the last chunk may be partly there.
template <class T, class Op, bool NT, int R>
__global__ __launch_bounds__(kScanBlock) void scan_rows_whole_kernel(ScanRowsParams p) {
    constexpr int V = ScanVec<T>::V;
    constexpr uint64_t CHUNK = (uint64_t)R * kScanBlock * V;
    __shared__ T s_wave_tot[kScanBlock / 64];
    for (uint64_t row = blockIdx.x; row < p.rows; row += gridDim.x) {
        int64_t oi, oo;
        scan_run_offsets(p, row, oi, oo);
        T carry = T();
        bool has_carry = false;
        const bool pieces = p.through && store_pieces(p.out + oo);
        for (uint64_t first = 0; first < p.n; first += CHUNK) {
            ScanVec<T> v[R];
            T total, wave_pre;
            if (p.n - first >= CHUNK) {
                chain_issue_loads<T, NT, R>(p.in + oi, first, v);
                chain_scan_tile<T, Op, R>(v, s_wave_tot, total, wave_pre);
                chain_store_tile<T, Op, NT, R>(p.out + oo, first, v, carry, has_carry, wave_pre, pieces);
            } else {
                // the run's last chunk, partly there
                const uint32_t nelem = (uint32_t)(p.n - first);
                chain_issue_loads<T, NT, R, true>(p.in + oi, first, v, nelem);
                chain_scan_tile<T, Op, R>(v, s_wave_tot, total, wave_pre);
                chain_store_tile<T, Op, NT, R, true>(p.out + oo, first, v, carry, has_carry, wave_pre, pieces, nelem);
            }
            carry = has_carry ? Op::apply(carry, total) : total;
            has_carry = true;
            __syncthreads();  // s_wave_tot is written again by the next chunk
        }
    }
}

template <class T, class Op, bool NT, int NW, int R, bool MANY>
__global__ __launch_bounds__(NW * 64, sizeof(T) == 8 ? 3 : 4) void scan_chain_kernel(ScanRowsParams p, ScanChain<T> c) {
    constexpr int V = ScanVec<T>::V;
    constexpr int TILE = NW * R * 64 * V;
    __shared__ ChainShared sh;
    __shared__ T s_prefix;
    __shared__ T s_wave_tot[NW];
    if (threadIdx.x == 0) sh.tile = __hip_atomic_fetch_add(c.ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) - c.ticket_base;
    __syncthreads();
    // the first tile of every run, then the second of every run: runs come along side by side
    uint32_t t = sh.tile;
    const char* in = p.in;
    char* out = p.out;
    if constexpr (MANY) {
        const uint32_t rows = (uint32_t)p.rows, row = t % rows;
        t /= rows;
        c.tile += (size_t)row * c.n_tiles * ScanChain<T>::W;
        c.group += (size_t)row * c.n_groups * ScanChain<T>::W;
        c.super += (size_t)row * c.n_supers * ScanChain<T>::W;
        scan_run_start(p, row, in, out);
    }
    const uint64_t first = (uint64_t)t * TILE;
    if (first >= p.n) return;  // (the grid is exactly the tiles; a stray ticket does nothing)
    ScanVec<T> v[R];
    // A run's last tile may be partly there. Loads and the scan stand in one branch each: where the branches met between them the
    // compiler waited for all loads before the first addition (2^24 SFloat 28.4 -> 30.0 us). The look-back stands once: a second
    // copy of it took registers that the tile needs.
    const bool whole = p.n - first >= (uint64_t)TILE;
    const uint32_t nelem = (uint32_t)(p.n - first);
    T total, wave_pre;
    if (whole) {
        chain_issue_loads<T, NT, R>(in, first, v);
        total = chain_scan_wave<T, Op, R>(v);
    } else {
        chain_issue_loads<T, NT, R, true>(in, first, v, nelem);
        total = chain_scan_wave<T, Op, R>(v);
    }
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63u) == 0) s_wave_tot[w] = total;
    __syncthreads();
    chain_fold_waves<T, Op, NW>(s_wave_tot, w, total, wave_pre);
    if (threadIdx.x < 64) {
        T pre;
        bool pre_has;
        chain_look_back<T, Op>(c, t, total, pre, pre_has);
        if (threadIdx.x == 0) {
            s_prefix = pre;
            sh.prefix_has = pre_has ? 1 : 0;
        }
    }
    __syncthreads();
    const bool pieces = p.through && store_pieces(out);
    if (whole) chain_store_tile<T, Op, NT, R>(out, first, v, s_prefix, sh.prefix_has != 0, wave_pre, pieces);
    else chain_store_tile<T, Op, NT, R, true>(out, first, v, s_prefix, sh.prefix_has != 0, wave_pre, pieces, nelem);
}

// a barrier for what is in LDS: __syncthreads() also waits for the block's loads and stores
__device__ __forceinline__ void chain_meet() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// The same without words in memory, for streams that keep none (a stream under capture: a replay would repeat the launch's number): a
// block has a run to itself, STEP tiles at a time, and keeps the totals of its tiles, groups and supergroups in LDS. Tiles, and the order
// in which their totals are folded, are those of the one pass, and so is every bit of the result; a few compute units do all the work.
// us, this in a graph / scan_rows_whole_kernel there, whose bits are others / the one pass: SFloat [8,20000] 6.4 / 7.4 / 6.1, one run of
// 65000 11.1 / 14.9 / 5.7, [100,40000] 11.9 / 11.1 / 10.9, [72,438001] 70 / 135 / 53; DFloat 10.0 / 11.6 / 6.3, 22.6 / 30.1 / 6.2,
// 20.8 / 27.6 / 19.3, 200 / 300 / 101. Bound by what a step takes from its loads to its stores, some 1.5 us; tiles asked for a step
// ahead did not shorten it, four small tiles or two of 64 KiB to a step did (one run of 65000: 23.1 and 47.6 with one).
template <class T, class Op, int NW, int R, int STEP>
__global__ __launch_bounds__(STEP * NW * 64) void scan_chain_alone_kernel(ScanRowsParams p) {
    constexpr uint32_t TILE = NW * R * 64 * ScanVec<T>::V;
    static_assert(64 % STEP == 0, "the tiles of a step are of one group");
    __shared__ T s_tile[64], s_group[64], s_super[64];
    __shared__ T s_wave_tot[STEP][NW];
    const unsigned lane = threadIdx.x & 63u;
    const uint32_t q = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x / (NW * 64)));   // this wave's tile of a step
    const int w = (int)(threadIdx.x >> 6) % NW;                                                     // and its place in the tile
    const char* in;
    char* out;
    scan_run_start(p, blockIdx.x, in, out);
    const bool pieces = p.through && store_pieces(out);
    uint32_t t = q;
    for (uint64_t step = 0; step < p.n; step += (uint64_t)STEP * TILE, t += STEP) {
        const uint64_t first = step + q * TILE;
        ScanVec<T> v[R];
        // (a tile that lies behind the run's end holds nothing)
        const bool whole = first + TILE <= p.n;
        const uint32_t nelem = first < p.n ? (uint32_t)(p.n - first) : 0;
        T total, wave_pre;
        if (whole) {
            chain_issue_loads<T, false, R>(in, first, v, 0, w);
            total = chain_scan_wave<T, Op, R>(v);
        } else {
            chain_issue_loads<T, false, R, true>(in, first, v, nelem, w);
            total = chain_scan_wave<T, Op, R>(v);
        }
        if (lane == 0) s_wave_tot[q][w] = total;
        chain_meet();
        chain_fold_waves<T, Op, NW>(s_wave_tot[q], w, total, wave_pre);
        const uint32_t pos = t & 63u, g = t >> 6, gpos = g & 63u, sg = g >> 6;
        if (w == 0 && lane == 0) s_tile[pos] = total;
        chain_meet();
        T x = lane < pos ? s_tile[lane] : T(), y = lane < gpos ? s_group[lane] : T(), z = lane < sg ? s_super[lane] : T();
        bool xh, yh, zh;
        chain_fold_lanes<T, Op>(x, xh, pos);
        chain_fold_lanes<T, Op>(y, yh, gpos);
        chain_fold_lanes<T, Op>(z, zh, sg);
        // (read from the step after the next barrier on)
        if (pos == 63u && w == 0 && lane == 0) {
            const T sum = Op::apply(x, total);
            s_group[gpos] = sum;
            if (gpos == 63u) s_super[sg] = Op::apply(y, sum);
        }
        chain_join<T, Op>(z, zh, y, yh);
        chain_join<T, Op>(z, zh, x, xh);
        if (whole) chain_store_tile<T, Op, false, R>(out, first, v, z, zh, wave_pre, pieces, 0, w);
        else chain_store_tile<T, Op, false, R, true>(out, first, v, z, zh, wave_pre, pieces, nelem, w);
    }
}

__global__ __launch_bounds__(256) void scan_chain_clear_kernel(uint64_t* words, uint64_t n) {
    for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (uint64_t)gridDim.x * 256) words[i] = 0;
}

// The words of one launch: the ticket word first, the published totals from word kChainHead on.
// A stream that is not being captured keeps a region of its own (per device and stream slot,
// allocated from the driver at first use, grown when a launch needs more, never cleared after
// that): launches on it are numbered, and a launch's words carry its number. Under capture (a
// replay would repeat the number), without a slot, or beyond kChainKeptWords the words come from
// the pool and a small kernel clears them first; the number is 1 then.
constexpr uint64_t kChainHead = 32;
constexpr uint64_t kChainKeptWords = 8ull << 20;  // 64 MiB
constexpr int kChainDevices = 16;
struct ChainRegion {
    uint64_t* ptr;
    uint64_t cap;
    uint32_t launch, ticket;
};
ChainRegion g_chain_region[kChainDevices][kStreamSlots];
std::mutex g_chain_lock;

struct ChainWords {
    uint64_t* ws;
    uint32_t flag, ticket_base;
    bool pooled;
};

// CUMO_HIP_SCAN_KEEP_WORDS=0 (read once): always the pool and the clearing kernel
static bool chain_keep_enabled() {
    static const bool on = [] {
        const char* e = std::getenv("CUMO_HIP_SCAN_KEEP_WORDS");
        return !(e && e[0] == '0');
    }();
    return on;
}

// words counts the head; tickets = blocks of the launch. False: no memory (the error is set), or, with kept_only, no region to keep them in.
static bool chain_words_acquire(hipStream_t stream, uint64_t words, uint32_t tickets, ChainWords* w, bool kept_only = false) {
    w->flag = 1;
    w->ticket_base = 0;
    w->pooled = true;
    hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &capturing) != hipSuccess) {
        (void)hipGetLastError();
        capturing = hipStreamCaptureStatusActive;
    }
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess) {
        (void)hipGetLastError();
        dev = -1;
    }
    const int slot = stream_slot(stream);
    if (chain_keep_enabled() && capturing == hipStreamCaptureStatusNone && slot >= 0 && dev >= 0 && dev < kChainDevices && words <= kChainKeptWords) {
        // held until chain_words_release, that is across the launch itself: launches that share a
        // stream must reach it in the order of their numbers and tickets
        g_chain_lock.lock();
        ChainRegion& r = g_chain_region[dev][slot];
        bool ok = true;
        if (r.cap < words) {
            if (r.ptr) {
                // only this stream's launches use the region
                ok = hipStreamSynchronize(stream) == hipSuccess && hipFree(r.ptr) == hipSuccess;
                r.ptr = nullptr;
                r.cap = 0;
            }
            uint64_t cap = 1ull << 16;
            while (cap < words) cap <<= 1;
            void* p = nullptr;
            if (ok && hipMalloc(&p, cap * sizeof(uint64_t)) == hipSuccess) {
                if (hipMemsetAsync(p, 0, cap * sizeof(uint64_t), stream) == hipSuccess) {
                    r.ptr = static_cast<uint64_t*>(p);
                    r.cap = cap;
                    r.launch = 0;
                    r.ticket = 0;
                } else {
                    (void)hipFree(p);
                    ok = false;
                }
            } else {
                ok = false;
            }
            if (!ok) (void)hipGetLastError();
        }
        if (ok && r.launch == 0xffffffffu) {
            // every number has been used once: start over from cleared words
            ok = hipMemsetAsync(r.ptr, 0, r.cap * sizeof(uint64_t), stream) == hipSuccess;
            r.launch = 0;
            r.ticket = 0;
            if (!ok) (void)hipGetLastError();
        }
        if (ok) {
            r.launch += 1;
            w->ws = r.ptr;
            w->flag = r.launch;
            w->ticket_base = r.ticket;
            r.ticket += tickets;
            w->pooled = false;
            return true;
        }
        g_chain_lock.unlock();
    }
    if (kept_only) return false;
    w->ws = reinterpret_cast<uint64_t*>(cumo_cuda_runtime_malloc(words * sizeof(uint64_t)));
    if (!w->ws) return false;
    uint64_t clear_grid = (words + 255) / 256;
    if (clear_grid > 2048) clear_grid = 2048;
    hipLaunchKernelGGL(scan_chain_clear_kernel, dim3((unsigned)clear_grid), dim3(256), 0, stream, w->ws, words);
    return true;
}

// after the launch that uses the words has been issued
static void chain_words_release(const ChainWords& w) {
    // stream-ordered reuse: whoever gets the block next can only touch it from later work on this stream
    if (w.pooled) cumo_cuda_runtime_free(reinterpret_cast<char*>(w.ws));
    else g_chain_lock.unlock();
}

// Whether the one pass is the better form for `rows` runs of `bytes` bytes than a block to each run: fewer runs than compute units,
// and each longer than two small tiles and a KiB for every run that shares the device with it. A block to a run / one pass, us:
// one run: SFloat 20000 6.4 / 4.7, 65013 14.6 / 4.9; several: SFloat [8,20000] 7.3 / 5.3, [100,40000] 12.2 / 10.7, [72,438001] 134 / 54;
// DFloat [8,20000] 11.2 / 5.8, [32,10000] 7.7 / 6.5, [72,438001] 297 / 102, [200,40000] 33.0 / 30.6. On the other side SFloat [16,5001]
// 4.3 / 5.4, [200,40000] 16.0 / 19.4, [256,30000] 15.8 / 15.8; DFloat [100,10000] 8.2 / 9.0, [250,20000] 20.5 / 22.6, [500,20000] 29 / 36.
static bool scan_chain_pays(uint64_t rows, uint64_t bytes) { return rows < 256 && bytes > 2 * kChainSmallBytes + rows * 1024; }

// The runs of p, contiguous and aligned as their elements are (p.through is set), in one pass; kept_only: with words that the stream
// keeps, or, where it keeps none, tile after tile by one block a run, to the same bits.
enum ChainLaunch { CHAIN_NOT_TAKEN, CHAIN_LAUNCHED, CHAIN_NO_MEMORY };
template <class T, class Op>
ChainLaunch scan_chain_launch(const ScanRowsParams& p, bool nt, bool kept_only, hipStream_t stream) {
    constexpr int W = ScanChain<T>::W;
    constexpr uint64_t E = 1024 / sizeof(T);  // elements of a row of 64 vectors
    // Blocks of eight waves and 128 KiB tiles wherever that leaves 64 tiles of four-byte elements or 128 of eight-byte ones (half
    // the tickets, which one word hands out at about 10 ns each, and half the look-backs per byte), else blocks of four waves and
    // 64 KiB tiles, or 16 KiB ones where that makes 128 of them or fewer, so that a short run has more than a few blocks. One run,
    // us on fresh operands, wide / narrow (small, where it is taken): SFloat 2^18 7.7 / 6.1 (4.9), 2^20 7.9 / 6.4 (256 small tiles 7.9), 2^22
    // 10.4 / 10.9, 2^24 28.2 / 34.0, 2^26 96.5 / 102; DFloat 2^18 9.1 / 6.5 (6.2), 2^20 10.0 / 9.5, 2^21 11.2 / 11.0, 2^22 15.8 / 19.6,
    // 2^24 54.2 / 60.7, 2^26 190 / 201.
    // CUMO_HIP_SCAN_CHAIN_WAVES=4 or 8, read once, fixes the choice.
    static const int forced_waves = [] {
        const char* e = std::getenv("CUMO_HIP_SCAN_CHAIN_WAVES");
        return e ? std::atoi(e) : 0;
    }();
    constexpr uint64_t kSmall = kChainSmallBytes / sizeof(T), kNarrow = 4 * 16 * E, kWide = 8 * 16 * E;
    const uint64_t wide_tiles = p.rows * ((p.n + kWide - 1) / kWide);
    const bool wide = forced_waves == 8 || (forced_waves != 4 && wide_tiles >= (sizeof(T) == 4 ? 64u : 128u));
    const bool small = !wide && forced_waves == 0 && p.rows * ((p.n + kSmall - 1) / kSmall) <= 128;
    const uint64_t tile = wide ? kWide : small ? kSmall : kNarrow;
    const uint64_t n_tiles = (p.n + tile - 1) / tile;
    if (n_tiles < 2 || n_tiles > kChainMaxTiles || p.rows * n_tiles > 0x7fffffffull) return CHAIN_NOT_TAKEN;
    const uint64_t n_groups = (n_tiles + 63) / 64, n_supers = (n_groups + 63) / 64;
    const uint64_t words = kChainHead + p.rows * (n_tiles + n_groups + n_supers) * W;
    WaitCtl* wait = wait_ctl();
    if (wait == nullptr && !kept_only) return CHAIN_NOT_TAKEN;  // nowhere to report a wait that gives up: the form without waits
    ChainWords cw;
    if (wait == nullptr || !chain_words_acquire(stream, words, (uint32_t)(p.rows * n_tiles), &cw, kept_only)) {
        if (!kept_only) return CHAIN_NO_MEMORY;
        const dim3 rows((unsigned)p.rows);
        if (small) hipLaunchKernelGGL((scan_chain_alone_kernel<T, Op, 4, 4, 4>), rows, dim3(1024), 0, stream, p);
        else if (wide) hipLaunchKernelGGL((scan_chain_alone_kernel<T, Op, 8, 16, 1>), rows, dim3(512), 0, stream, p);
        else hipLaunchKernelGGL((scan_chain_alone_kernel<T, Op, 4, 16, 2>), rows, dim3(512), 0, stream, p);
        return CHAIN_LAUNCHED;
    }
    ScanChain<T> c;
    c.wait = wait;
    c.ticket = reinterpret_cast<uint32_t*>(cw.ws);
    c.n_tiles = (uint32_t)n_tiles;
    c.n_groups = (uint32_t)n_groups;
    c.n_supers = (uint32_t)n_supers;
    c.tile = cw.ws + kChainHead;
    c.group = c.tile + p.rows * n_tiles * W;
    c.super = c.group + p.rows * n_groups * W;
    c.flag = cw.flag;
    c.ticket_base = cw.ticket_base;
    const dim3 g((unsigned)(p.rows * n_tiles));
#define CUMO_SCAN_CHAIN(NT_, NW_, R_)                                                                                                   \
    do {                                                                                                                                \
        if (p.rows > 1) hipLaunchKernelGGL((scan_chain_kernel<T, Op, NT_, NW_, R_, true>), g, dim3(NW_ * 64), 0, stream, p, c);        \
        else hipLaunchKernelGGL((scan_chain_kernel<T, Op, NT_, NW_, R_, false>), g, dim3(NW_ * 64), 0, stream, p, c);                  \
    } while (0)
    if (small) CUMO_SCAN_CHAIN(false, 4, 4);
    else if (wide && nt) CUMO_SCAN_CHAIN(true, 8, 16);
    else if (wide) CUMO_SCAN_CHAIN(false, 8, 16);
    else if (nt) CUMO_SCAN_CHAIN(true, 4, 16);
    else CUMO_SCAN_CHAIN(false, 4, 16);
#undef CUMO_SCAN_CHAIN
    chain_words_release(cw);
    return CHAIN_LAUNCHED;
}

// ---- runs that lie across memory (the scan goes down the rows of a matrix) ------
// Lanes sit along the dimension that is contiguous in memory and each lane walks
// its VEC columns down the run, so every load is coalesced across the wave. A run
// is cut into segments to fill the device: phase 0 leaves each segment's total per
// column and phase 2 scans each segment from what the segments before it add up to:
// with up to 32 segments it folds their totals itself, with more the totals are first
// turned into running totals by a column scan of their own (they form a small matrix).
// With enough columns there is one segment and only phase 2 runs (one read, one write).
struct ScanColsParams {
    int nouter;               // dimensions outside the run and the column dimension
    uint64_t planes, cols, n; // planes = product of those dimensions
    uint64_t oshape[CUMO_NA_MAX_DIMENSION];
    int64_t ostep_in[CUMO_NA_MAX_DIMENSION], ostep_out[CUMO_NA_MAX_DIMENSION];
    int64_t s_in, s_out;      // byte step along the run
    uint64_t seg_len, n_seg;
    int tx_bits;              // 2^tx_bits lanes along the columns, the rest of the block along segments
    const char* in;
    char* out;
};

template <class T, int VEC, bool NT = false>
__device__ __forceinline__ void scan_cols_load(const char* p, T (&v)[VEC]) {
    if constexpr (VEC * sizeof(T) == 16) {
        typedef uint32_t u4 __attribute__((ext_vector_type(4)));
        union { u4 q; T t[VEC]; } u;
        u.q = NT ? __builtin_nontemporal_load(reinterpret_cast<const u4*>(p)) : *reinterpret_cast<const u4*>(p);
#pragma unroll
        for (int j = 0; j < VEC; ++j) v[j] = u.t[j];
    } else {
#pragma unroll
        for (int j = 0; j < VEC; ++j) v[j] = reinterpret_cast<const T*>(p)[j];
    }
}
template <class T, int VEC, bool NT = false>
__device__ __forceinline__ void scan_cols_store(char* p, const T (&v)[VEC]) {
    if constexpr (VEC * sizeof(T) == 16) {
        typedef uint32_t u4 __attribute__((ext_vector_type(4)));
        union { u4 q; T t[VEC]; } u;
#pragma unroll
        for (int j = 0; j < VEC; ++j) u.t[j] = v[j];
        if (NT) __builtin_nontemporal_store(u.q, reinterpret_cast<u4*>(p));
        else *reinterpret_cast<u4*>(p) = u.q;
    } else {
#pragma unroll
        for (int j = 0; j < VEC; ++j) reinterpret_cast<T*>(p)[j] = v[j];
    }
}

// PHASE 0: totals[(plane * n_seg + seg) * cols + col] = total of the segment.
// PHASE 2: scan the segment, starting from what the segments before it add up to:
//   LOOKBACK false  totals holds running totals already: one load of totals[.. seg - 1 ..]
//   LOOKBACK true   totals holds each segment's own total: they are folded here, in
//                   segment order (few segments: cheaper than a launch that does it)
template <class T, class Op, int VEC, int PHASE, bool LOOKBACK, bool NT>
__global__ __launch_bounds__(kScanBlock) void scan_cols_kernel(ScanColsParams p, T* totals) {
    constexpr int UNR = 4;  // four rows in flight per lane (more open more rows at once in memory and measured slower)
    const unsigned TX = 1u << p.tx_bits, TY = (unsigned)kScanBlock >> p.tx_bits;
    const unsigned tx = threadIdx.x & (TX - 1), ty = threadIdx.x >> p.tx_bits;
    const uint64_t col_groups = p.cols / VEC;
    const uint64_t strips = (col_groups + TX - 1) / TX;
    const uint64_t seg_blocks = (p.n_seg + TY - 1) / TY;
    const uint64_t n_blocks = strips * seg_blocks * p.planes;
    for (uint64_t b = blockIdx.x; b < n_blocks; b += gridDim.x) {
        const uint64_t strip = b % strips;
        const uint64_t sb = (b / strips) % seg_blocks;
        const uint64_t plane = b / (strips * seg_blocks);
        const uint64_t cg = strip * TX + tx;
        const uint64_t seg = sb * TY + ty;
        if (cg >= col_groups || seg >= p.n_seg) continue;
        int64_t oi = 0, oo = 0;
        uint64_t r = plane;
        for (int d = p.nouter - 1; d >= 0; --d) {
            const uint64_t m = p.oshape[d];
            const uint64_t q = r / m;
            const int64_t k = (int64_t)(r - q * m);
            r = q;
            oi += k * p.ostep_in[d];
            oo += k * p.ostep_out[d];
        }
        const uint64_t col = cg * VEC;
        const uint64_t begin = seg * p.seg_len;
        uint64_t end = begin + p.seg_len;
        if (end > p.n) end = p.n;
        const char* src = p.in + oi + (int64_t)col * (int64_t)sizeof(T);
        char* dst = p.out + oo + (int64_t)col * (int64_t)sizeof(T);
        T acc[VEC];
        bool has = false;
        if (PHASE == 2 && seg > 0) {
            if (LOOKBACK) {
                const T* t = totals + plane * p.n_seg * p.cols + col;
                scan_cols_load<T, VEC>(reinterpret_cast<const char*>(t), acc);
#pragma unroll 4
                for (uint64_t q = 1; q < seg; ++q) {
                    T v[VEC];
                    scan_cols_load<T, VEC>(reinterpret_cast<const char*>(t + q * p.cols), v);
#pragma unroll
                    for (int j = 0; j < VEC; ++j) acc[j] = Op::apply(acc[j], v[j]);
                }
            } else {
                scan_cols_load<T, VEC>(reinterpret_cast<const char*>(totals + (plane * p.n_seg + seg - 1) * p.cols + col), acc);
            }
            has = true;
        }
        uint64_t i = begin;
        for (; i + UNR <= end; i += UNR) {
            T v[UNR][VEC];
#pragma unroll
            for (int u = 0; u < UNR; ++u) scan_cols_load<T, VEC, NT>(src + (int64_t)(i + u) * p.s_in, v[u]);
            __builtin_amdgcn_sched_barrier(0);  // the step's loads go out before anything is folded
#pragma unroll
            for (int u = 0; u < UNR; ++u) {
#pragma unroll
                for (int j = 0; j < VEC; ++j) acc[j] = has ? Op::apply(acc[j], v[u][j]) : v[u][j];
                has = true;
                if (PHASE == 2) scan_cols_store<T, VEC, NT>(dst + (int64_t)(i + u) * p.s_out, acc);
            }
        }
        for (; i < end; ++i) {
            T v[VEC];
            scan_cols_load<T, VEC, NT>(src + (int64_t)i * p.s_in, v);
#pragma unroll
            for (int j = 0; j < VEC; ++j) acc[j] = has ? Op::apply(acc[j], v[j]) : v[j];
            has = true;
            if (PHASE == 2) scan_cols_store<T, VEC, NT>(dst + (int64_t)i * p.s_out, acc);
        }
        if (PHASE == 0) scan_cols_store<T, VEC>(reinterpret_cast<char*>(totals + (plane * p.n_seg + seg) * p.cols + col), acc);
    }
}

constexpr uint64_t kScanLookbackSegs = 32;
constexpr uint64_t kScanColsThreads = 256ull * 8 * kScanBlock;  // lanes that the segments are to make

// Two passes over the data with the segment totals between them. With few segments
// the second pass folds the totals of the segments before its own by itself (two
// launches); with many, the totals, a [segments x columns] matrix per plane, are
// scanned in place by this same routine first (a column scan of a much smaller array).
template <class T, class Op, int VEC>
void scan_cols_launch_vec(ScanColsParams& p, hipStream_t stream) {
    const uint64_t col_groups = p.cols / VEC;
    int txb = 0;
    while (txb < 8 && (1ull << txb) < col_groups) ++txb;
    p.tx_bits = txb;
    const uint64_t TX = 1ull << txb, TY = (uint64_t)kScanBlock >> txb;
    // segments: enough threads for eight blocks on every compute unit, at least 16 rows each;
    // no more than the second pass folds by itself when those already give every compute unit four
    // blocks (with one block each, SFloat [8192,8192] ran its first pass at half the bandwidth)
    const uint64_t want_threads = kScanColsThreads;
    const uint64_t lanes_per_seg = col_groups * p.planes;
    uint64_t n_seg = (want_threads + lanes_per_seg - 1) / lanes_per_seg;
    const uint64_t max_seg = (p.n + 15) / 16;
    if (n_seg > kScanLookbackSegs && lanes_per_seg * kScanLookbackSegs >= 1024ull * kScanBlock) n_seg = kScanLookbackSegs;
    if (n_seg > max_seg) n_seg = max_seg;
    if (n_seg > 1024) n_seg = 1024;
    if (n_seg < 1) n_seg = 1;
    p.seg_len = (p.n + n_seg - 1) / n_seg;
    p.n_seg = (p.n + p.seg_len - 1) / p.seg_len;
    const uint64_t strips = (col_groups + TX - 1) / TX;
    uint64_t grid = strips * ((p.n_seg + TY - 1) / TY) * p.planes;
    if (grid > 0x7fffffffull) grid = 0x7fffffffull;
    const dim3 g((unsigned)grid), b(kScanBlock);
    const bool nt = stream_past_caches(2 * p.planes * p.n * p.cols * sizeof(T));
#define CUMO_SCAN_COLS(PHASE_, LB_, TOTALS_)                                                                                  \
    do {                                                                                                                      \
        if (nt) hipLaunchKernelGGL((scan_cols_kernel<T, Op, VEC, PHASE_, LB_, true>), g, b, 0, stream, p, TOTALS_);           \
        else hipLaunchKernelGGL((scan_cols_kernel<T, Op, VEC, PHASE_, LB_, false>), g, b, 0, stream, p, TOTALS_);             \
    } while (0)
    if (p.n_seg == 1) {
        CUMO_SCAN_COLS(2, false, (T*)nullptr);
        return;
    }
    T* totals = reinterpret_cast<T*>(cumo_cuda_runtime_malloc(sizeof(T) * p.planes * p.n_seg * p.cols));
    if (!totals) return;
    CUMO_SCAN_COLS(0, false, totals);
    if (p.n_seg <= kScanLookbackSegs) {
        CUMO_SCAN_COLS(2, true, totals);
    } else {
        ScanColsParams q;
        std::memset(&q, 0, sizeof(q));
        q.nouter = 1;
        q.planes = p.planes;
        q.oshape[0] = p.planes;
        q.ostep_in[0] = q.ostep_out[0] = (int64_t)(p.n_seg * p.cols * sizeof(T));
        q.cols = p.cols;
        q.n = p.n_seg;
        q.s_in = q.s_out = (int64_t)(p.cols * sizeof(T));
        q.in = reinterpret_cast<const char*>(totals);
        q.out = reinterpret_cast<char*>(totals);
        scan_cols_launch_vec<T, Op, VEC>(q, stream);  // at most 1024 rows: the next level has at most 64 segments
        CUMO_SCAN_COLS(2, false, totals);
    }
#undef CUMO_SCAN_COLS
    // stream-ordered reuse: whoever gets the block next can only touch it from later work on this stream
    cumo_cuda_runtime_free(reinterpret_cast<char*>(totals));
}

// ---- long runs across memory in one pass ---------------------------------------
// The matrix is cut into tiles of NW * 16 rows by 64 vectors (1 KiB of a row): wave w of
// a block holds 16 rows of the tile, lane l their vector l, all in registers. Of narrower
// matrices a wave holds two, four or eight bands of 16 rows side by side. A tile adds
// up its columns (in the lane, from band to band by shuffles, then across the waves through LDS), publishes the column
// totals, gathers what the tiles above it published, and scans its rows from there: the
// data is read once and written once. The published words are {the launch's number, 32 bits of
// the value}, in the region the stream keeps (see above). Tiles take their places by ticket, level by level
// (all strips of one band of rows, then the next band), so whatever a tile waits for
// belongs to a block that is already running, and no tile waits before it has published
// its own totals. What a tile gathers has a fixed shape, so results do not change from
// launch to launch: tiles come in groups of 8 and groups in supergroups of 8; a tile folds
// the supergroups before its own, then the groups before its own, then the tiles before it
// in its group, each in order. The tile that closes a group publishes the group's total,
// the one that closes a supergroup the supergroup's.
constexpr int kColsChainRows = 16;
constexpr uint32_t kColsChainFan = 8;

template <class T>
struct ScanColsChain {
    static constexpr int W = (int)(sizeof(T) / 4);
    WaitCtl* wait;     // where a look-back that gives up reports it
    uint32_t* ticket;
    uint64_t* tile;    // [strip][level][column][W]
    uint64_t* group;   // [strip][group][column][W]
    uint64_t* super;   // [strip][supergroup][column][W]
    uint32_t depth, n_groups, n_supers;  // per strip; nothing is published or waited for where depth is 1
    uint32_t strips;                     // per plane
    uint32_t all_strips;                 // planes * strips
    uint32_t flag;                       // the upper half of a word of this launch
    uint32_t ticket_base;                // what the ticket word held before this launch
};

// Up to seven published values, `stride` words apart, the earliest first: all are asked for at
// once (eight-byte types: four, then three; seven would not fit the registers beside the tile),
// asked for again until they are there, then folded in order. False when count is 0.
template <class T, class Op>
__device__ __forceinline__ bool cols_chain_gather(const uint64_t* base, size_t stride, uint32_t count, uint32_t flag, WaitCtl* ctl, T& out) {
    constexpr int W = ScanColsChain<T>::W;
    constexpr uint32_t N = kColsChainFan - 1, C = sizeof(T) == 8 ? 4 : N;
    uint32_t polls = 0;
    const uint32_t spin_limit = wait_limit(ctl, kChainSpinLimit);
    bool has = false;
#pragma unroll
    for (uint32_t c0 = 0; c0 < N; c0 += C) {
        uint64_t x[C][W];
#pragma unroll
        for (uint32_t i = 0; i < C; ++i)
#pragma unroll
            for (int h = 0; h < W; ++h)
                x[i][h] = c0 + i < count ? __hip_atomic_load(base + (c0 + i) * stride + h, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : ((uint64_t)flag << 32);
        for (;;) {
            bool all = true;
#pragma unroll
            for (uint32_t i = 0; i < C; ++i)
#pragma unroll
                for (int h = 0; h < W; ++h) all = all && (uint32_t)(x[i][h] >> 32) == flag;
            if (all) break;
            if (++polls > spin_limit) {
                wait_gave_up(ctl, WAIT_SCAN);
                break;
            }
            __builtin_amdgcn_s_sleep(8);
#pragma unroll
            for (uint32_t i = 0; i < C; ++i)
#pragma unroll
                for (int h = 0; h < W; ++h)
                    if ((uint32_t)(x[i][h] >> 32) != flag) x[i][h] = __hip_atomic_load(base + (c0 + i) * stride + h, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
#pragma unroll
        for (uint32_t i = 0; i < C; ++i) {
            if (c0 + i < count) {
                union { T t; uint32_t w[W]; } u;
#pragma unroll
                for (int h = 0; h < W; ++h) u.w[h] = (uint32_t)x[i][h];
                out = has ? Op::apply(out, u.t) : u.t;
                has = true;
            }
        }
    }
    return has;
}

// v of the lane `step` rows' lanes before this one
template <class T>
__device__ __forceinline__ T cols_chain_up(T v, int step) {
    constexpr int N = (int)(sizeof(T) / 4);
    union { T t; int w[N]; } u;
    u.t = v;
#pragma unroll
    for (int i = 0; i < N; ++i) u.w[i] = __shfl_up(u.w[i], step);
    return u.t;
}

// LPR lanes to a row of the tile, so 64 / LPR bands of 16 rows to a wave. ONE: one tile holds every row, nothing is published or
// waited for. DEEP: more than 512 tiles down a column.
template <class T, class Op, bool NT, int NW, int LPR, bool ONE, bool DEEP>
__global__ __launch_bounds__(NW * 64) void scan_cols_chain_kernel(ScanColsParams p, ScanColsChain<T> c) {
    constexpr int V = 16 / (int)sizeof(T), R = kColsChainRows, SW = LPR * V, SUB = 64 / LPR, W = ScanColsChain<T>::W;
    __shared__ T part[NW][SW];
    __shared__ T s_groups[SW], s_supers[SW];
    __shared__ uint32_t s_ticket;
    static_assert(NW * 64 >= (ONE ? 1 : 3) * SW, "three roles of SW threads each");
    const unsigned w = threadIdx.x >> 6, l = threadIdx.x % LPR, sub = (threadIdx.x & 63u) / LPR;
    uint32_t id = blockIdx.x;
    if constexpr (!ONE) {
        if (threadIdx.x == 0) s_ticket = __hip_atomic_fetch_add(c.ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) - c.ticket_base;
        __syncthreads();
        id = s_ticket;
    }
    const uint32_t k = id / c.all_strips, ps = id - k * c.all_strips;
    const uint32_t plane = ps / c.strips, strip = ps - plane * c.strips;
    int64_t oi = 0, oo = 0;
    if (p.nouter > 0) {
        uint64_t r = plane;
#pragma unroll 1
        for (int d = p.nouter - 1; d >= 0; --d) {
            const uint64_t m = p.oshape[d];
            const uint64_t q = r / m;
            const int64_t i = (int64_t)(r - q * m);
            r = q;
            oi += i * p.ostep_in[d];
            oo += i * p.ostep_out[d];
        }
    }
    const int64_t row0 = (int64_t)k * (NW * SUB * R) + (int64_t)(w * SUB + sub) * R;
    const int64_t colb = ((int64_t)strip * SW + (int64_t)l * V) * (int64_t)sizeof(T);
    char* dst = p.out + oo + row0 * p.s_out + colb;
    // A tile at the lower edge has fewer rows and one at the right edge fewer columns: this lane's first `rows` rows exist, and of
    // its columns the first ncol. What such a tile reads as missing is zeros; the totals they enter are only ever used by
    // rows or columns that do not exist either. A lane that has anything sends all of its loads, from inside the array: a row that
    // does not exist is read again from the last one, a vector that is partly there as the one that ends with the row. They go by
    // the second-level cache: the lines hold the start of the next row as well, which another block reads (SFloat [131072,257] 66.5 us
    // with non-temporal loads here).
    const int64_t rows_left = (int64_t)p.n - row0;
    const int rows = rows_left >= R ? R : (rows_left > 0 ? (int)rows_left : 0);
    const int64_t cols_left = (int64_t)p.cols - (int64_t)((uint64_t)strip * SW + (uint64_t)l * V);
    const int ncol = cols_left >= V ? V : (cols_left > 0 ? (int)cols_left : 0);  // this lane's columns that exist
    const bool all_there = __builtin_amdgcn_ballot_w64(rows != R || ncol != V) == 0;
    T raw[R][V];
    if (all_there) {
        const char* src = p.in + oi + row0 * p.s_in + colb;
#pragma unroll
        for (int r = 0; r < R; ++r) scan_cols_load<T, V, NT>(src + (int64_t)r * p.s_in, raw[r]);
    } else {
        const char* src = p.in + oi + (ncol == V ? colb : ((int64_t)p.cols - V) * (int64_t)sizeof(T));
        if (rows > 0 && ncol > 0) {
            const int64_t last = (int64_t)p.n - 1;
#pragma unroll
            for (int r = 0; r < R; ++r) scan_cols_load<T, V>(src + (row0 + r < last ? row0 + r : last) * p.s_in, raw[r]);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            T v[V];
#pragma unroll
            for (int j = 0; j < V; ++j) v[j] = raw[r][j];
#pragma unroll
            for (int j = 0; j < V; ++j) {
                // column j is element j + V - ncol of the vector
                T e = T();
#pragma unroll
                for (int n = 1; n <= V; ++n)
                    if (j < n) e = ncol == n ? v[j + V - n] : e;
                raw[r][j] = r < rows ? e : T();
            }
        }
    }
    // This lane's rows are scanned by themselves, here, and take what lies above them when it is known: a value is rounded at the size
    // of the whole sum once, not at every row, and nothing is left to do one after the other behind the wait. Their total, and, of
    // a wave that holds several bands, that of the bands before, follow.
#pragma unroll
    for (int r = 1; r < R; ++r)
#pragma unroll
        for (int j = 0; j < V; ++j) raw[r][j] = Op::apply(raw[r - 1][j], raw[r][j]);
    T above_lane[V];
    {
        T tot[V];
#pragma unroll
        for (int j = 0; j < V; ++j) tot[j] = raw[R - 1][j];
        if constexpr (SUB > 1) {
#pragma unroll
            for (int d = 1; d < SUB; d *= 2) {
#pragma unroll
                for (int j = 0; j < V; ++j) {
                    const T before = cols_chain_up(tot[j], d * LPR);
                    if ((int)sub >= d) tot[j] = Op::apply(before, tot[j]);
                }
            }
#pragma unroll
            for (int j = 0; j < V; ++j) above_lane[j] = cols_chain_up(tot[j], LPR);
        }
        if (sub == SUB - 1) {
#pragma unroll
            for (int j = 0; j < V; ++j) part[w][l * V + j] = tot[j];
        }
    }
    __syncthreads();
    // Threads 0 .. SW-1 see to the tile's own totals and to the tiles before it in its group,
    // the next SW threads to the groups before its group, the SW after those to the supergroups:
    // the three waits run side by side in different waves, each with seven loads in flight.
    const unsigned col = threadIdx.x % SW, role = threadIdx.x / SW;
    if constexpr (ONE) {
        if (role == 0) {
            T above = part[0][col];
#pragma unroll
            for (int ww = 1; ww < NW; ++ww) {
                const T mine = part[ww][col];
                part[ww][col] = above;
                above = Op::apply(above, mine);
            }
        }
        __syncthreads();
    } else {
    const uint32_t pos = k % kColsChainFan, g = k / kColsChainFan, gpos = g % kColsChainFan, sg = g / kColsChainFan;
    // (supergroups are as many as there are: they are gathered seven at a time)
    const size_t cw = (size_t)SW * W;  // words from one tile's (group's) totals to the next one's
    T gt = T();
    if (role == 0) {
        // part[ww][col] becomes what the waves above ww add up to; gt, the tile's total
        gt = part[0][col];
#pragma unroll
        for (int ww = 1; ww < NW; ++ww) {
            const T e = gt;
            gt = Op::apply(gt, part[ww][col]);
            part[ww][col] = e;
        }
        chain_publish<T>(c.tile + (((size_t)ps * c.depth + k) * SW + col) * W, gt, c.flag);
    }
    const uint64_t* from = c.tile + (((size_t)ps * c.depth + (size_t)g * kColsChainFan) * SW + col) * W;
    uint32_t count = pos;
    if (role == 1) {
        from = c.group + (((size_t)ps * c.n_groups + (size_t)sg * kColsChainFan) * SW + col) * W;
        count = gpos;
    } else if (role == 2) {
        from = c.super + ((size_t)ps * c.n_supers * SW + col) * W;
        count = sg;
    } else if (role > 2) {
        count = 0;
    }
    T xs = T();
    const bool xh = cols_chain_gather<T, Op>(from, cw, DEEP && count > kColsChainFan - 1 ? kColsChainFan - 1 : count, c.flag, c.wait, xs);
    if constexpr (DEEP) {
        for (uint32_t at = kColsChainFan - 1; at < count; at += kColsChainFan - 1) {
            T more = T();
            const uint32_t left = count - at;
            cols_chain_gather<T, Op>(from + at * cw, cw, left < kColsChainFan - 1 ? left : kColsChainFan - 1, c.flag, c.wait, more);
            xs = Op::apply(xs, more);
        }
    }
    if (role == 0) {
        if (xh) gt = Op::apply(xs, gt);  // the group's total so far
        if (pos == kColsChainFan - 1) chain_publish<T>(c.group + (((size_t)ps * c.n_groups + g) * SW + col) * W, gt, c.flag);
    } else if (role == 1) {
        s_groups[col] = xs;
    } else if (role == 2) {
        s_supers[col] = xs;
    }
    __syncthreads();
    if (role == 0 && k > 0) {
        const bool yh = gpos > 0;
        T ys = T();
        if (yh) ys = s_groups[col];
        if (pos == kColsChainFan - 1 && gpos == kColsChainFan - 1) {
            const T st = yh ? Op::apply(ys, gt) : gt;
            chain_publish<T>(c.super + (((size_t)ps * c.n_supers + sg) * SW + col) * W, st, c.flag);
        }
        bool ph = sg > 0;
        T pre = T();
        if (ph) pre = s_supers[col];
        if (yh) { pre = ph ? Op::apply(pre, ys) : ys; ph = true; }
        if (xh) { pre = ph ? Op::apply(pre, xs) : xs; ph = true; }
        // k > 0: something lies above, so ph holds
        part[0][col] = pre;
#pragma unroll
        for (int ww = 1; ww < NW; ++ww) part[ww][col] = Op::apply(pre, part[ww][col]);
    }
    __syncthreads();
    }
    const bool first_wave = k == 0 && w == 0, topmost = first_wave && sub == 0;   // (nothing above it)
    T above[V];
#pragma unroll
    for (int j = 0; j < V; ++j) {
        above[j] = first_wave ? T() : part[w][l * V + j];
        if constexpr (SUB > 1) {
            if (sub > 0) above[j] = first_wave ? above_lane[j] : Op::apply(above[j], above_lane[j]);
        }
    }
    if (all_there) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            T out[V];
#pragma unroll
            for (int j = 0; j < V; ++j) out[j] = topmost ? raw[r][j] : Op::apply(above[j], raw[r][j]);
            scan_cols_store<T, V, NT>(dst + (int64_t)r * p.s_out, out);
        }
    } else {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            T out[V];
#pragma unroll
            for (int j = 0; j < V; ++j) out[j] = topmost ? raw[r][j] : Op::apply(above[j], raw[r][j]);
            if (r < rows && ncol == V) {
                scan_cols_store<T, V, NT>(dst + (int64_t)r * p.s_out, out);
            } else if (r < rows) {
#pragma unroll
                for (int j = 0; j < V; ++j)
                    if (j < ncol) reinterpret_cast<T*>(dst + (int64_t)r * p.s_out)[j] = out[j];
            }
        }
    }
}

static bool scan_cols_chain_enabled() {
    static const bool on = [] {
        const char* e = std::getenv("CUMO_HIP_SCAN_COLS_CHAIN");
        return !(e && e[0] == '0');
    }();
    return on;
}

// true when the launch was made (or failed: the error is left for the caller's check)
template <class T, class Op, int NW, int LPR, bool MAY_NT, bool ONE, bool DEEP>
bool scan_cols_chain_go(const ScanColsParams& p, hipStream_t stream) {
    constexpr int V = 16 / (int)sizeof(T), W = ScanColsChain<T>::W;
    constexpr uint64_t SW = LPR * V, TR = (uint64_t)NW * (64 / LPR) * kColsChainRows;
    constexpr uint64_t F = kColsChainFan;
    const uint64_t depth = (p.n + TR - 1) / TR, strips = (p.cols + SW - 1) / SW;
    if (depth > F * F * F * (DEEP ? 8 : 1)) return false;
    const uint64_t all_strips = strips * p.planes;
    const uint64_t n_tiles = all_strips * depth;
    if (n_tiles > 0x3fffffull) return false;
    const uint64_t n_groups = (depth + F - 1) / F, n_supers = (n_groups + F - 1) / F;
    ScanColsChain<T> c;
    std::memset(&c, 0, sizeof(c));
    ChainWords cw;
    if constexpr (!ONE) {
        const uint64_t words = kChainHead + all_strips * (depth + n_groups + n_supers) * SW * W;
        c.wait = wait_ctl();
        if (c.wait == nullptr) return false;  // nowhere to report a wait that gives up: the form without waits
        if (!chain_words_acquire(stream, words, (uint32_t)n_tiles, &cw)) return true;
        c.ticket = reinterpret_cast<uint32_t*>(cw.ws);
        c.tile = cw.ws + kChainHead;
        c.flag = cw.flag;
        c.ticket_base = cw.ticket_base;
        c.group = c.tile + all_strips * depth * SW * W;
        c.super = c.group + all_strips * n_groups * SW * W;
    }
    c.depth = (uint32_t)depth;
    c.n_groups = (uint32_t)n_groups;
    c.n_supers = (uint32_t)n_supers;
    c.strips = (uint32_t)strips;
    c.all_strips = (uint32_t)all_strips;
    const bool nt = MAY_NT && stream_past_caches(2 * p.planes * p.n * p.cols * sizeof(T));
    const dim3 g((unsigned)n_tiles), b(NW * 64);
    if (nt) hipLaunchKernelGGL((scan_cols_chain_kernel<T, Op, MAY_NT, NW, LPR, ONE, DEEP>), g, b, 0, stream, p, c);
    else hipLaunchKernelGGL((scan_cols_chain_kernel<T, Op, false, NW, LPR, ONE, DEEP>), g, b, 0, stream, p, c);
    if constexpr (!ONE) chain_words_release(cw);
    return true;
}

// Matrices whose rows hold a vector: what this leaves to the segments is rows of less than that, more than 4096 tiles down, and
// what the tests below say. Up to 256 rows are one tile, in blocks of four waves up to 64
// rows. us, two passes / this:
//   rows that are few    SFloat [208,53952] 29.2 / 15.4, [64,500000] 68.6 / 46.8, [31,32000] 8.3 / 5.5; DFloat [76,440000] 149 / 100
//   columns that are few SFloat [234385,93] 94.5 / 39.2, [20000,130] 25.0 / 14.2, [1000000,16] 416 / 39.9; DFloat [131072,33] 44 / 20
//   matrices of few tiles SFloat [619,640] 14.2 / 9.0, [3036,248] 15.5 / 10.5, DFloat [20,700] 6.1 / 4.3
template <class T, class Op>
bool scan_cols_chain_launch(ScanColsParams& p, hipStream_t stream) {
    constexpr int V = 16 / (int)sizeof(T);
    if (!scan_cols_chain_enabled() || p.cols < (uint64_t)V || p.n < 2) return false;
    const uint64_t vectors = (p.cols + V - 1) / V;
    // Up to sixteen rows, or columns enough for a lane each: the segments are one, a launch that reads and writes once (us, that /
    // this: [12,100000] 4.3 / 5.1, [3,20] 3.3 / 5.7); rows of 64 vectors keep to the tiles where there are two of them.
    const bool one_segment = p.n <= (uint64_t)kColsChainRows || vectors * p.planes >= kScanColsThreads;
    if (one_segment && (vectors < 64 || p.n <= 16 * kColsChainRows)) return false;
    // Up to 512 rows are two launches in segments, which small arrays are done with sooner than tiles hand on their totals ([300,200]
    // 7.5 / 9.3, [500,130] 8.2 / 10.1; [300,3000] 9.3 / 8.6): one tile or a MiB of them.
    const bool one_tile = vectors > 32 && p.n <= 16 * kColsChainRows;
    if (!one_tile && p.n <= kScanLookbackSegs * 16 && p.planes * p.n * p.cols * sizeof(T) < (1u << 20)) return false;
    if (vectors > 32) {
        if (p.n <= 4 * kColsChainRows) return scan_cols_chain_go<T, Op, 4, 64, true, true, false>(p, stream);
        if (p.n <= 16 * kColsChainRows) return scan_cols_chain_go<T, Op, 16, 64, true, true, false>(p, stream);
        if (p.n <= 512 * 16 * kColsChainRows) return scan_cols_chain_go<T, Op, 16, 64, true, false, false>(p, stream);
        return scan_cols_chain_go<T, Op, 16, 64, true, false, true>(p, stream);
    }
    // (many planes of fewer rows than a quarter of a tile would be tiles, and words, of nothing)
    const uint64_t bands = vectors > 16 ? 2 : vectors > 8 ? 4 : 8;
    if (p.n < 4 * bands * kColsChainRows) return false;
    if (vectors > 16) return scan_cols_chain_go<T, Op, 16, 32, true, false, true>(p, stream);
    if (vectors > 8) return scan_cols_chain_go<T, Op, 16, 16, false, false, true>(p, stream);
    return scan_cols_chain_go<T, Op, 16, 8, false, false, true>(p, stream);
}

template <class T, class Op>
void scan_cols_launch(ScanColsParams& p, hipStream_t stream) {
    constexpr int V = 16 / (int)sizeof(T);
    bool vec = (p.cols % V) == 0 && ((uintptr_t)p.in % 16) == 0 && ((uintptr_t)p.out % 16) == 0 && (p.s_in % 16) == 0 && (p.s_out % 16) == 0;
    for (int d = 0; d < p.nouter && vec; ++d) vec = (p.ostep_in[d] % 16) == 0 && (p.ostep_out[d] % 16) == 0;
    // the one-pass form needs the elements' alignment only (128-bit accesses work on any 4-byte boundary)
    // and takes a last vector of a row that is partly there
    bool elem = ((uintptr_t)p.in % sizeof(T)) == 0 && ((uintptr_t)p.out % sizeof(T)) == 0 && (p.s_in % (int64_t)sizeof(T)) == 0 &&
                (p.s_out % (int64_t)sizeof(T)) == 0;
    for (int d = 0; d < p.nouter && elem; ++d) elem = (p.ostep_in[d] % (int64_t)sizeof(T)) == 0 && (p.ostep_out[d] % (int64_t)sizeof(T)) == 0;
    if (elem && scan_cols_chain_launch<T, Op>(p, stream)) return;
    if (vec) scan_cols_launch_vec<T, Op, V>(p, stream);
    else scan_cols_launch_vec<T, Op, 1>(p, stream);
}

template <class T>
void scan_cols_dispatch(int prod, int nan, ScanColsParams& p, hipStream_t stream) {
    if (prod) {
        if (nan) scan_cols_launch<T, ScanOp<T, 1, true> >(p, stream);
        else scan_cols_launch<T, ScanOp<T, 1, false> >(p, stream);
    } else {
        if (nan) scan_cols_launch<T, ScanOp<T, 0, true> >(p, stream);
        else scan_cols_launch<T, ScanOp<T, 0, false> >(p, stream);
    }
}

// CUMO_HIP_SCAN_CHAIN=0 (read once): long runs take the three launches instead of the one pass
static bool scan_chain_enabled() {
    static const bool on = [] {
        const char* e = std::getenv("CUMO_HIP_SCAN_CHAIN");
        return !(e && e[0] == '0');
    }();
    return on;
}

template <class T, class Op>
void scan_rows_launch(ScanRowsParams& p, hipStream_t stream) {
    if (p.rows == 0 || p.n == 0) return;
    uint64_t grid = p.rows;
    if (grid > 65536) grid = 65536;
    constexpr uint64_t V = 16 / sizeof(T);
    // (runs need their element's alignment only: 128-bit accesses work on any 4-byte boundary)
    bool whole = p.s_in == (int64_t)sizeof(T) && p.s_out == (int64_t)sizeof(T) && p.n >= 64 * V &&
                 (((uintptr_t)p.in | (uintptr_t)p.out) % sizeof(T)) == 0;
    for (int d = 0; d < p.nouter && whole; ++d) whole = (p.ostep_in[d] % (int64_t)sizeof(T)) == 0 && (p.ostep_out[d] % (int64_t)sizeof(T)) == 0;
    if (whole) {
        const uint64_t vec_rows = (p.n + kScanBlock * V - 1) / (kScanBlock * V);  // rows of 256 vectors in a run, the last one maybe partly there
        const bool nt = stream_past_caches(2 * p.rows * p.n * sizeof(T));
        StoreRows out_rows(p.out, p.n * sizeof(T));
        for (int d = 0; d < p.nouter; ++d) out_rows.dimension(p.oshape[d], p.ostep_out[d]);
        p.through = out_rows.through(nt);
        // (the blocks that take a run each need no memory from the pool: neither does this call, under capture or on a stream without a slot)
        if (scan_chain_enabled() && scan_chain_pays(p.rows, p.n * sizeof(T)) && scan_chain_launch<T, Op>(p, nt, true, stream) == CHAIN_LAUNCHED) return;
        const dim3 g((unsigned)grid), b(kScanBlock);
#define CUMO_SCAN_WHOLE(R_) do { if (nt) hipLaunchKernelGGL((scan_rows_whole_kernel<T, Op, true, R_>), g, b, 0, stream, p); \
                                 else hipLaunchKernelGGL((scan_rows_whole_kernel<T, Op, false, R_>), g, b, 0, stream, p); } while (0)
        // chunks of 8, 4, 2 or 1 such rows: the largest that the run fills at least once, or that holds all of it
        if (vec_rows > 4) CUMO_SCAN_WHOLE(8);
        else if (vec_rows > 2) CUMO_SCAN_WHOLE(4);
        else if (vec_rows > 1) CUMO_SCAN_WHOLE(2);
        else CUMO_SCAN_WHOLE(1);
#undef CUMO_SCAN_WHOLE
        return;
    }
    hipLaunchKernelGGL((scan_rows_kernel<T, Op>), dim3((unsigned)grid), dim3(kScanBlock), 0, stream, p);
}

// One run of n elements: the one pass where it is contiguous; else one block where it is short, and three launches (also for runs
// beyond 2^30 elements, and with the knob above).
template <class T, class Op>
int scan_run_launch(const char* p1, char* p2, ssize_t s1, ssize_t s2, uint64_t n) {
    if (n == 0) return 0;
    hipStream_t stream = current_stream();
    const uint64_t n_tiles = (n + kScanTile - 1) / kScanTile;
    const bool contiguous = s1 == (ssize_t)sizeof(T) && s2 == (ssize_t)sizeof(T) && (((uintptr_t)p1 | (uintptr_t)p2) % sizeof(T)) == 0;
    ScanRowsParams p;
    std::memset(&p, 0, sizeof(p));
    p.rows = 1;
    p.n = n;
    p.s_in = s1;
    p.s_out = s2;
    p.in = p1;
    p.out = p2;
    p.through = true;
    if (n_tiles <= 8) {
        scan_rows_launch<T, Op>(p, stream);
        return (int)hipGetLastError();
    }
    if (contiguous && scan_chain_enabled()) {
        const ChainLaunch how = scan_chain_launch<T, Op>(p, stream_past_caches(2 * n * sizeof(T)), false, stream);
        if (how != CHAIN_NOT_TAKEN) return how == CHAIN_NO_MEMORY ? (int)hipErrorOutOfMemory : (int)hipGetLastError();
    }
    // One tile per block keeps the most loads in flight (a block that walks a stretch of
    // tiles waits at two barriers per tile: measured 15 % slower). The totals are scanned
    // in place by this same routine, so a long run never leaves many tiles to one block.
    const uint64_t per = 1;
    const uint64_t n_blocks = n_tiles;
    if (n_blocks > 0x7fffffffull) return (int)hipErrorInvalidValue;
    T* totals = reinterpret_cast<T*>(cumo_cuda_runtime_malloc(sizeof(T) * n_blocks));
    if (!totals) return (int)hipErrorOutOfMemory;
    hipLaunchKernelGGL((scan_tile_totals_kernel<T, Op>), dim3((unsigned)n_blocks), dim3(kScanBlock), 0, stream, p1, (int64_t)s1, n, totals);
    const int inner = scan_run_launch<T, Op>(reinterpret_cast<const char*>(totals), reinterpret_cast<char*>(totals), (ssize_t)sizeof(T),
                                             (ssize_t)sizeof(T), n_blocks);
    if (inner) {
        cumo_cuda_runtime_free(reinterpret_cast<char*>(totals));
        return inner;
    }
    hipLaunchKernelGGL((scan_apply_kernel<T, Op>), dim3((unsigned)n_blocks), dim3(kScanBlock), 0, stream, p1, (int64_t)s1, p2, (int64_t)s2, n, per,
                       (const T*)totals);
    const int st = (int)hipGetLastError();
    // stream-ordered reuse: whoever gets the block next can only touch it from later work on this stream
    cumo_cuda_runtime_free(reinterpret_cast<char*>(totals));
    return st;
}

template <class T>
void scan_rows_dispatch(int prod, int nan, ScanRowsParams& p, hipStream_t stream) {
    if (prod) {
        if (nan) scan_rows_launch<T, ScanOp<T, 1, true> >(p, stream);
        else scan_rows_launch<T, ScanOp<T, 1, false> >(p, stream);
    } else {
        if (nan) scan_rows_launch<T, ScanOp<T, 0, true> >(p, stream);
        else scan_rows_launch<T, ScanOp<T, 0, false> >(p, stream);
    }
}

}  // namespace

// The kept regions go back to the driver when their stream is retired and when the caller asks
// the pool to give back what it holds (they are not the pool's blocks -- they must outlive a
// launch without being handed to anybody else -- but they are memory the library holds:
// up to kChainKeptWords * 8 bytes per stream that has run a one-pass scan).
// The stream of the slot must have finished its work.
void scan_chain_words_drop_slot(int slot) {
    if (slot < 0 || slot >= kStreamSlots) return;
    std::lock_guard<std::mutex> hold(g_chain_lock);
    for (int dev = 0; dev < kChainDevices; ++dev) {
        ChainRegion& r = g_chain_region[dev][slot];
        if (!r.ptr) continue;
        if (hipFree(r.ptr) != hipSuccess) (void)hipGetLastError();
        r = ChainRegion{nullptr, 0, 0, 0};
    }
}

// every region, after waiting for the device (a launch that still uses one may be queued)
void scan_chain_words_drop_all() {
    std::lock_guard<std::mutex> hold(g_chain_lock);
    bool any = false;
    for (int dev = 0; dev < kChainDevices && !any; ++dev)
        for (int slot = 0; slot < kStreamSlots && !any; ++slot) any = g_chain_region[dev][slot].ptr != nullptr;
    if (!any) return;
    if (hipDeviceSynchronize() != hipSuccess) {
        (void)hipGetLastError();
        return;
    }
    for (int dev = 0; dev < kChainDevices; ++dev)
        for (int slot = 0; slot < kStreamSlots; ++slot) {
            ChainRegion& r = g_chain_region[dev][slot];
            if (!r.ptr) continue;
            if (hipFree(r.ptr) != hipSuccess) (void)hipGetLastError();
            r = ChainRegion{nullptr, 0, 0, 0};
        }
}

size_t scan_chain_words_held_bytes() {
    std::lock_guard<std::mutex> hold(g_chain_lock);
    size_t total = 0;
    for (int dev = 0; dev < kChainDevices; ++dev)
        for (int slot = 0; slot < kStreamSlots; ++slot) total += (size_t)g_chain_region[dev][slot].cap * sizeof(uint64_t);
    return total;
}

}  // namespace cumo_hip

using namespace cumo_hip;

extern "C" {

#define CUMO_DEF_CUM(t, c, name, OP, NANF)                                                                        \
    int cumo_##t##_##name##_kernel_launch(char* p1, char* p2, ssize_t s1, ssize_t s2, uint64_t n) {               \
        return scan_run_launch<c, ScanOp<c, OP, NANF> >(p1, p2, s1, s2, n);                                       \
    }
CUMO_DEF_CUM(sfloat, float, cumsum, 0, false)
CUMO_DEF_CUM(sfloat, float, cumsum_nan, 0, true)
CUMO_DEF_CUM(sfloat, float, cumprod, 1, false)
CUMO_DEF_CUM(sfloat, float, cumprod_nan, 1, true)
CUMO_DEF_CUM(dfloat, double, cumsum, 0, false)
CUMO_DEF_CUM(dfloat, double, cumsum_nan, 0, true)
CUMO_DEF_CUM(dfloat, double, cumprod, 1, false)
CUMO_DEF_CUM(dfloat, double, cumprod_nan, 1, true)
CUMO_DEF_CUM(int32, int32_t, cumsum, 0, false)
CUMO_DEF_CUM(int32, int32_t, cumprod, 1, false)

void cumo_hip_scan_rows_kernel_launch(int type, int prod, int nan, const cumo_hip_scan_rows_t* d) {
    if (!d || d->rows == 0 || d->n == 0) return;
    ScanRowsParams p;
    std::memset(&p, 0, sizeof(p));
    p.nouter = d->nouter;
    p.rows = d->rows;
    p.n = d->n;
    for (int k = 0; k < d->nouter && k < CUMO_NA_MAX_DIMENSION; ++k) {
        p.oshape[k] = d->oshape[k];
        p.ostep_in[k] = d->ostep_in[k];
        p.ostep_out[k] = d->ostep_out[k];
    }
    p.s_in = d->s_in;
    p.s_out = d->s_out;
    p.in = d->in;
    p.out = d->out;
    if (scan_short_launch(type, prod, nan, d)) {
        cumo_cuda_runtime_check_kernel_launch();
        return;
    }
    hipStream_t stream = current_stream();
    switch (type) {
        case 0: scan_rows_dispatch<float>(prod, nan, p, stream); break;
        case 1: scan_rows_dispatch<double>(prod, nan, p, stream); break;
        case 2: scan_rows_dispatch<int32_t>(prod, 0, p, stream); break;
        default: report_error(CUMO_HIP_ERROR_TYPE, 0, "scan: element type is not SFloat, DFloat or Int32"); return;
    }
    cumo_cuda_runtime_check_kernel_launch();
}

void cumo_hip_scan_cols_kernel_launch(int type, int prod, int nan, const cumo_hip_scan_rows_t* d, uint64_t cols) {
    if (!d || d->rows == 0 || d->n == 0 || cols == 0) return;
    ScanColsParams p;
    std::memset(&p, 0, sizeof(p));
    p.nouter = d->nouter;
    p.planes = d->rows;
    p.cols = cols;
    p.n = d->n;
    for (int k = 0; k < d->nouter && k < CUMO_NA_MAX_DIMENSION; ++k) {
        p.oshape[k] = d->oshape[k];
        p.ostep_in[k] = d->ostep_in[k];
        p.ostep_out[k] = d->ostep_out[k];
    }
    p.s_in = d->s_in;
    p.s_out = d->s_out;
    p.in = d->in;
    p.out = d->out;
    hipStream_t stream = current_stream();
    switch (type) {
        case 0: scan_cols_dispatch<float>(prod, nan, p, stream); break;
        case 1: scan_cols_dispatch<double>(prod, nan, p, stream); break;
        case 2: scan_cols_dispatch<int32_t>(prod, 0, p, stream); break;
        default: report_error(CUMO_HIP_ERROR_TYPE, 0, "scan: element type is not SFloat, DFloat or Int32"); return;
    }
    cumo_cuda_runtime_check_kernel_launch();
}

}  // extern "C"
