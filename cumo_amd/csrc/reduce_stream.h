// Lean reduction kernels for the layouts that carry nearly all the bytes: the
// reduce axis is ONE run of elements (after merging), the outputs span at most two
// dimensions, every access is a whole 128-bit vector and all totals fit 32 bits.
// Included by reduce_kernels.h, which keeps the general kernels for everything else.
//
//  red_srow_kernel        the reduce axis runs along memory; 2^k lanes share an output.
//  red_srow_split_kernel  the same with the axis cut over several blocks per output, in
//                         ONE launch: every block leaves its accumulator in a scratch
//                         array and counts in on a ticket; the block that counts in last
//                         folds the accumulators of its output in index order. The order
//                         of the fold does not depend on which block that is, so results
//                         are the same bits on every run, as with a second launch.
//  red_scol_kernel        the outputs run along memory; a lane owns VEC neighbouring
//                         outputs and walks the axis; with SHARE, lanes of a block share
//                         the rows and combine through LDS; with PARTIAL, the axis is also
//                         cut across blocks and red_fold_parts_kernel folds their parts.
//
// What makes them lean: a 136-byte argument block instead of 620 bytes; every load of
// an unrolled step is unconditional (a position past the end is pulled back inside the
// run and its value not used), so the four 128-bit loads of a lane are in flight
// together; no per-element index decomposition at all; non-temporal loads for inputs
// that no cache level could hold anyway.
#ifndef CUMO_HIP_REDUCE_STREAM_H
#define CUMO_HIP_REDUCE_STREAM_H

namespace cumo_hip {

constexpr int kRsUnroll = 4;            // 128-bit loads a lane keeps in flight
constexpr int kRsWide = 1024;           // lanes of a block that has a long row to itself when there are a few hundred of them
constexpr int kRsGroup = 32;            // blocks that count in on one first-level ticket when an output has more than kRsOneLevel
constexpr int kRsOneLevel = 128;        // up to this many blocks per output count in on a single ticket
constexpr uint32_t kRsTicketWords = 16384;  // ticket words per stream slot

// An Impl whose accumulate_columns<U, VEC>(x[U][VEC], acc[VEC]) folds U positions of VEC neighbouring outputs at once,
// all of which have seen the same number of positions before, and whose combine_columns<VEC>(next, acc) folds two
// lanes' accumulators of such outputs
template <class I, class = void> struct folds_columns_together { static constexpr bool value = false; };
template <class I> struct folds_columns_together<I, decltype((void)I::COLUMNS_TOGETHER)> { static constexpr bool value = I::COLUMNS_TOGETHER; };

// An Impl whose combine() goes without branches and that has a form with them, combine_seldom(), for parts that mostly change nothing.
template <class I, class = void> struct combines_in_two_forms { static constexpr bool value = false; };
template <class I> struct combines_in_two_forms<I, decltype((void)&I::combine_seldom)> { static constexpr bool value = true; };

// An Impl whose accumulate_step<U, VEC>(x[U][VEC], vectors, acc) folds a step's elements, of which the first `vectors` vectors are
// there, among themselves before they join the accumulator: what a long row's sum rounds off does not depend on how few lanes share it.
template <class I, class = void> struct folds_steps { static constexpr bool value = false; };
template <class I> struct folds_steps<I, decltype((void)I::STEPS)> { static constexpr bool value = I::STEPS; };

// An Impl whose accumulate_columns_by_position<U, VEC>(x[U][VEC], first position, acc[VEC]) folds U consecutive
// positions of VEC neighbouring outputs without a branch
template <class I, class = void> struct folds_columns_by_position { static constexpr bool value = false; };
template <class I> struct folds_columns_by_position<I, decltype((void)I::COLUMNS_BY_POSITION)> { static constexpr bool value = I::COLUMNS_BY_POSITION; };

// An Impl whose accumulator is rounded by every ROUNDS_EVERY rows of a column (0, or none given: not at all, or it does not matter)
template <class I, class = void> struct rounds_every { static constexpr int value = 0; };
template <class I> struct rounds_every<I, decltype((void)I::ROUNDS_EVERY)> { static constexpr int value = I::ROUNDS_EVERY; };

struct RedSParams {
    const char* in;
    char* out;
    char* out2;
    uint64_t n;            // length of the reduce axis in elements (row form: of its whole vectors)
    uint32_t tail;         // row form: elements of the axis past its last whole vector (fewer than a vector)
    int64_t red_step;      // column form: byte step along the reduce axis
    int64_t in_step[2];    // input byte steps over the (at most two) output dimensions, outer first
    int64_t out_step[2];
    int64_t out2_step[2];
    uint32_t n_out;        // outputs
    uint32_t out_inner;    // extent of the inner output dimension (= n_out when there is one dimension)
    uint32_t n_split;      // split form: blocks per output
    uint64_t chunk;        // column form cut across blocks: positions of the axis a block takes 
    uint32_t group;        // split form: blocks that count in on one first-level ticket
    uint32_t tstride;      // split form: words between two tickets (tickets in one cache line serialise in one memory channel)
    uint32_t tpr_bits;     // row form: 2^tpr_bits lanes share an output
    uint32_t width;        // column form: output groups side by side in a block
    uint32_t slots;        // column form: lanes of a block that share an output group's part of the axis
    uint32_t run;          // column form: steps of kRcRows rows that a lane folds by themselves (where the Impl rounds)
    uint32_t fold_bits;    // fold of the column form's parts: 2^fold_bits lanes share an output
    int32_t index_mode;    // what accumulate() gets as idx: 1 = position along the axis, 2 = element offset from `in`
    char* partial;         // split form: n_out * n_split accumulators
    uint32_t* tickets;     // split form: n_out + n_out * ceil(n_split / group) words, zero between launches
    WaitCtl* wait;         // hand-over form: where a wait that gives up reports it
};

template <class In, int VEC, bool NT>
__device__ __forceinline__ void rs_load(const char* p, In (&x)[VEC]) {
    static_assert(sizeof(In) * VEC == 16, "whole 128-bit vectors");
    typedef uint32_t u4 __attribute__((ext_vector_type(4)));
    union V {
        u4 q;
        In v[VEC];
        __device__ V() {}
    } t;
    if constexpr (NT) t.q = __builtin_nontemporal_load(reinterpret_cast<const u4*>(p));
    else t.q = *reinterpret_cast<const u4*>(p);
#pragma unroll
    for (int j = 0; j < VEC; ++j) x[j] = t.v[j];
}

__device__ __forceinline__ void rs_split_out(const RedSParams& p, uint32_t o, uint32_t& o0, uint32_t& o1) {
    if (p.out_inner == p.n_out) {
        o0 = 0;
        o1 = o;
    } else {
        o0 = o / p.out_inner;
        o1 = o - o0 * p.out_inner;
    }
}

// The 2^tpr_bits lanes of a group fold the tiles first, first + every, first + 2 * every, ...
// of the run [0, end) (base = its element 0); a tile is what the group loads in one step,
// kRsUnroll vectors per lane. end is a multiple of VEC. Every lane of the group runs the
// same number of steps. The run may go on for `tail` more elements, fewer than a vector: the
// group's first lane folds those one by one when the group has the run's first tile (first == 0).
// In a wide block sums go step by step as pairs of pairs: its lanes are fewer than those of the blocks that would share the row, so
// that one element after the other a lane's chain was up to four times as long. Error in norm, rows of zero mean, cut across
// blocks / a wide block, one after the other / as pairs: SFloat 128 x 262144 1.5e-7 / 3.0e-7 / 1.3e-7, 200 x 100000 1.5e-7 / 2.0e-7 / 1.2e-7,
// DFloat 200 x 100000 2.8e-16 / 3.7e-16 / 2.3e-16; the times are the same.
template <class Impl, int VEC, bool NT, int BLOCK = kRedBlock>
__device__ __forceinline__ typename Impl::Acc rs_row_scan(const Impl& impl, const char* base, uint64_t first, uint64_t every, uint64_t end,
                                                          uint32_t tail, unsigned lane_r, unsigned tpr_bits, int64_t idx_base) {
    typedef typename Impl::In In;
    typename Impl::Acc acc = impl.identity();
    const uint64_t stride = (uint64_t)VEC << tpr_bits;
    const uint64_t per_step = stride * kRsUnroll;
    const uint64_t tiles = (end + per_step - 1) / per_step;
    if (first >= tiles) return acc;
    const uint64_t steps = (tiles - first + every - 1) / every;
    const uint64_t advance = per_step * every;
    const uint64_t last = end - VEC;
    uint64_t i0 = first * per_step + (uint64_t)lane_r * VEC;
    for (uint64_t s = 0; s < steps; ++s, i0 += advance) {
        In x[kRsUnroll][VEC];
#pragma unroll
        for (int u = 0; u < kRsUnroll; ++u) {
            const uint64_t i = i0 + (uint64_t)u * stride;
            const uint64_t ic = i < end ? i : last;
            rs_load<In, VEC, NT>(base + ic * sizeof(In), x[u]);
        }
        // every load of the step is issued before anything is folded (the scheduler would
        // otherwise start folding the first vector and hold the later loads back behind it)
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (BLOCK > kRedBlock && folds_steps<Impl>::value) {
            uint32_t vectors = 0;
#pragma unroll
            for (int u = 0; u < kRsUnroll; ++u) vectors += i0 + (uint64_t)u * stride < end ? 1u : 0u;
            impl.template accumulate_step<kRsUnroll, VEC>(x, vectors, acc);
            continue;
        }
        if constexpr (has_group<Impl>::value) {
            if (i0 + (uint64_t)(kRsUnroll - 1) * stride < end) {
                int64_t idx[kRsUnroll];
#pragma unroll
                for (int u = 0; u < kRsUnroll; ++u) idx[u] = idx_base + (int64_t)(i0 + (uint64_t)u * stride);
                impl.template accumulate_group<kRsUnroll, VEC>(x, idx, acc);
                continue;
            }
        }
#pragma unroll
        for (int u = 0; u < kRsUnroll; ++u) {
            const uint64_t i = i0 + (uint64_t)u * stride;
            if (i < end) impl.template accumulate_n<VEC>(x[u], idx_base + (int64_t)i, acc);
        }
    }
    // (after the lane's other elements: a lane folds in the order of the axis, which an impl may rely on)
    if (tail != 0 && first == 0 && lane_r == 0) {
        const In* rest = reinterpret_cast<const In*>(base) + end;
        for (uint32_t e = 0; e < tail; ++e) impl.accumulate(rest[e], idx_base + (int64_t)(end + e), acc);
    }
    return acc;
}

// Lanes of one output combine; the group's first lane (thread 0 when a block shares the
// output) ends up with everything, later lanes folded into earlier ones in a fixed order.
template <class Impl, int BLOCK = kRedBlock>
__device__ __forceinline__ void rs_group_combine(const Impl& impl, typename Impl::Acc& acc, unsigned tpr_bits,
                                                 typename Impl::Acc* wave_slots) {
    typedef typename Impl::Acc Acc;
    constexpr unsigned WAVES = BLOCK / 64;
    const unsigned TPR = 1u << tpr_bits;
    const unsigned span = TPR < 64 ? TPR : 64;
    for (unsigned d = span >> 1; d > 0; d >>= 1) {
        const Acc other = shfl_down_any(acc, d);
        impl.combine(other, acc);
    }
    if (TPR > 64) {
        if ((threadIdx.x & 63) == 0) wave_slots[threadIdx.x >> 6] = acc;
        __syncthreads();
        if constexpr (WAVES > 4) {
            // the far half onto the near one, as within the wave
            if (threadIdx.x < 64) {
                acc = wave_slots[threadIdx.x & (WAVES - 1)];
                for (unsigned d = WAVES >> 1; d > 0; d >>= 1) {
                    const Acc other = shfl_down_any(acc, d);
                    impl.combine(other, acc);
                }
            }
        } else if (threadIdx.x == 0) {
            for (unsigned w = 1; w < WAVES; ++w) impl.combine(wave_slots[w], acc);
        }
        __syncthreads();
    }
}

// scan + combine (+ the exact second fold where the impl asks for one)
template <class Impl, int VEC, bool NT, int BLOCK = kRedBlock>
__device__ __forceinline__ typename Impl::Acc rs_row_reduce(const Impl& impl, const char* base, uint64_t first, uint64_t every, uint64_t end,
                                                            uint32_t tail, unsigned lane_r, unsigned tpr_bits, int64_t idx_base,
                                                            typename Impl::Acc* wave_slots, int* s_need) {
    typedef typename Impl::Acc Acc;
    Acc acc = rs_row_scan<Impl, VEC, NT, BLOCK>(impl, base, first, every, end, tail, lane_r, tpr_bits, idx_base);
    rs_group_combine<Impl, BLOCK>(impl, acc, tpr_bits, wave_slots);
    if constexpr (has_exact<Impl>::value) {
        const unsigned TPR = 1u << tpr_bits;
        bool need;
        if (TPR > 64) {
            if (threadIdx.x == 0) *s_need = impl.needs_exact(acc) ? 1 : 0;
            __syncthreads();
            need = *s_need != 0;
            __syncthreads();
        } else {
            const int mine = impl.needs_exact(acc) ? 1 : 0;
            need = __shfl(mine, (int)((threadIdx.x & 63u) & ~(TPR - 1))) != 0;
        }
        if (need) {
            typedef typename Impl::Exact Exact;
            const Exact ex = impl.exact();
            // the exact accumulator is wider: its own LDS slots
            __shared__ typename Exact::Acc exact_slots[BLOCK / 64];
            typename Exact::Acc e = rs_row_scan<Exact, VEC, false>(ex, base, first, every, end, tail, lane_r, tpr_bits, 0);
            rs_group_combine<Exact, BLOCK>(ex, e, tpr_bits, exact_slots);
            acc = impl.from_exact(e);
        }
    }
    return acc;
}

// BLOCK: kRedBlock lanes, or kRsWide of them for a few hundred long rows (red_rows_wide)
template <class Impl, int VEC, bool NT, int BLOCK = kRedBlock>
__global__ __launch_bounds__(BLOCK) void red_srow_kernel(RedSParams p, Impl impl) {
    typedef typename Impl::In In;
    typedef typename Impl::Acc Acc;
    __shared__ Acc wave_slots[BLOCK / 64];
    __shared__ int s_need;
    const unsigned TPR = 1u << p.tpr_bits;
    const unsigned RPB = (unsigned)BLOCK >> p.tpr_bits;
    const unsigned lane_r = threadIdx.x & (TPR - 1);
    const unsigned row_in_block = threadIdx.x >> p.tpr_bits;
    const uint32_t n_rb = (p.n_out + RPB - 1) / RPB;
    for (uint32_t rb = blockIdx.x; rb < n_rb; rb += gridDim.x) {
        const uint32_t row = rb * RPB + row_in_block;
        const bool ok = row < p.n_out;
        uint32_t o0, o1;
        rs_split_out(p, ok ? row : p.n_out - 1, o0, o1);
        const int64_t in_off = (int64_t)o0 * p.in_step[0] + (int64_t)o1 * p.in_step[1];
        const int64_t idx_base = p.index_mode == 2 ? in_off / (int64_t)sizeof(In) : 0;
        const Acc acc = rs_row_reduce<Impl, VEC, NT, BLOCK>(impl, p.in + in_off, 0, 1, p.n, p.tail, lane_r, p.tpr_bits, idx_base, wave_slots, &s_need);
        if (ok && lane_r == 0) {
            const int64_t a = (int64_t)o0 * p.out_step[0] + (int64_t)o1 * p.out_step[1];
            const int64_t b = (Impl::NOUT > 1) ? (int64_t)o0 * p.out2_step[0] + (int64_t)o1 * p.out2_step[1] : 0;
            impl.store(acc, p.out + a, (Impl::NOUT > 1) ? (p.out2 + b) : nullptr);
        }
    }
}

// accumulators cross between blocks as 32-bit words written through to memory
template <class Acc>
__device__ __forceinline__ void rs_publish(char* dst, const Acc& acc) {
    static_assert(sizeof(Acc) % 4 == 0, "accumulator must be a whole number of 32-bit words");
    constexpr int W = sizeof(Acc) / 4;
    union U {
        Acc a;
        uint32_t w[W];
        __device__ U() {}
    } u;
    u.a = acc;
#pragma unroll
    for (int i = 0; i < W; ++i)
        __hip_atomic_store(reinterpret_cast<uint32_t*>(dst) + i, u.w[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// read after the acquire fence of the block that counted in last: plain loads, all in flight together
template <class Acc>
__device__ __forceinline__ Acc rs_fetch(const char* src) {
    return *reinterpret_cast<const Acc*>(src);
}

// One block per (output, chunk of the axis). blockIdx.x = output * n_split + chunk.
template <class Impl, int VEC, bool NT>
__global__ __launch_bounds__(kRedBlock) void red_srow_split_kernel(RedSParams p, Impl impl) {
    typedef typename Impl::In In;
    typedef typename Impl::Acc Acc;
    __shared__ Acc wave_slots[kRedBlock / 64];
    __shared__ int s_need;
    __shared__ int s_last;
    const uint32_t vrow = blockIdx.x;
    const uint32_t i_out = vrow / p.n_split;
    const uint32_t i_split = vrow - i_out * p.n_split;
    uint32_t o0, o1;
    rs_split_out(p, i_out, o0, o1);
    const int64_t in_off = (int64_t)o0 * p.in_step[0] + (int64_t)o1 * p.in_step[1];
    const int64_t idx_base = p.index_mode == 2 ? in_off / (int64_t)sizeof(In) : 0;
    // the blocks of an output take its 16 KiB tiles in turn, so that together they read one window
    // of the run at a time (memory sees a few long streams instead of n_split short ones)
    Acc acc = rs_row_reduce<Impl, VEC, NT>(impl, p.in + in_off, i_split, p.n_split, p.n, p.tail, threadIdx.x, 8, idx_base, wave_slots, &s_need);

    if (threadIdx.x == 0) {
        // The accumulator is written through to memory and has arrived there before
        // this block counts in. Blocks count in on their group's ticket; the last of a
        // group counts in on the output's ticket; the last there finds every
        // accumulator of the output in memory. Tickets go back to zero on the way.
        // What orders the publication before the count:
        //  * the hardware: rs_publish stores with agent scope, which on this device writes through
        //    the compute die's second-level cache to the memory all dies share, and the wait below
        //    returns when those stores are acknowledged; the ticket add is issued after that;
        //  * the compiler: the fence. At workgroup scope it costs nothing beyond that same wait,
        //    but no memory operation may be moved across it.
        // A release on the ticket add itself (agent scope) would be the textbook form; on this
        // device it also writes back the whole second-level cache of the die, once per block:
        // measured on T.sum() of 2^25 SFloat with tickets, 25.2 -> 107 us. The emitted order
        // (store sc1 ... s_waitcnt vmcnt(0) ... atomic add) is pinned by tests/test_emitted_ordering.py.
        rs_publish<Acc>(p.partial + (size_t)vrow * sizeof(Acc), acc);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __builtin_amdgcn_s_waitcnt(0);  // vmcnt(0) expcnt(0) lgkmcnt(0): the stores are acknowledged
        const uint32_t groups = (p.n_split + p.group - 1) / p.group;
        const uint32_t g = i_split / p.group;
        const uint32_t g_size = (g + 1 == groups) ? p.n_split - g * p.group : p.group;
        uint32_t* t1 = p.tickets + (size_t)(p.n_out + i_out * groups + g) * p.tstride;
        uint32_t* t0 = p.tickets + (size_t)i_out * p.tstride;
        int last = 0;
        if (__hip_atomic_fetch_add(t1, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == g_size - 1) {
            __hip_atomic_store(t1, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (groups == 1) {
                last = 1;  // one group: its last block is the output's last
            } else if (__hip_atomic_fetch_add(t0, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == groups - 1) {
                __hip_atomic_store(t0, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                last = 1;
            }
        }
        s_last = last;
    }
    __syncthreads();
    if (!s_last) return;
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");

    // fold the output's accumulators in index order: thread t takes chunks t, t + 256, ...
    const char* mine = p.partial + (size_t)i_out * p.n_split * sizeof(Acc);
    const int64_t o_a = (int64_t)o0 * p.out_step[0] + (int64_t)o1 * p.out_step[1];
    const int64_t o_b = (Impl::NOUT > 1) ? (int64_t)o0 * p.out2_step[0] + (int64_t)o1 * p.out2_step[1] : 0;
    if constexpr (has_exact<Impl>::value) {
        // the accumulators are values in axis order: the fast fold first, and only where
        // it cannot decide (which of two equal values came first) the exact rule over the same values
        typedef typename Impl::Exact Exact;
        Acc total = impl.identity();
        for (uint32_t k = threadIdx.x; k < p.n_split; k += kRedBlock) impl.combine(rs_fetch<Acc>(mine + (size_t)k * sizeof(Acc)), total);
        rs_group_combine(impl, total, 8, wave_slots);
        if (threadIdx.x == 0) s_need = impl.needs_exact(total) ? 1 : 0;
        __syncthreads();
        if (s_need) {
            const Exact ex = impl.exact();
            __shared__ typename Exact::Acc exact_slots[kRedBlock / 64];
            typename Exact::Acc e = ex.identity();
            for (uint32_t k = threadIdx.x; k < p.n_split; k += kRedBlock) ex.accumulate_acc(rs_fetch<Acc>(mine + (size_t)k * sizeof(Acc)), (int64_t)k, e);
            rs_group_combine(ex, e, 8, exact_slots);
            total = impl.from_exact(e);
        }
        if (threadIdx.x == 0) impl.store(total, p.out + o_a, (Impl::NOUT > 1) ? (p.out2 + o_b) : nullptr);
    } else {
        Acc total = impl.identity();
        for (uint32_t k = threadIdx.x; k < p.n_split; k += kRedBlock) impl.combine(rs_fetch<Acc>(mine + (size_t)k * sizeof(Acc)), total);
        rs_group_combine(impl, total, 8, wave_slots);
        if (threadIdx.x == 0) impl.store(total, p.out + o_a, (Impl::NOUT > 1) ? (p.out2 + o_b) : nullptr);
    }
}

// Second launch of the column form cut across blocks: folds partial[part][output] (rows of rs_parts_row
// accumulators) into the results. A lane has one output and a run of its parts in axis order, up to eight in
// flight; the 2^fold_bits lanes of an output combine pairwise through LDS, earlier parts on the left. What bounds
// it is one chain of memory round trips (parts that another die wrote, the LDS rounds, the store), not bytes, so a
// lane has at most eight parts however wide the accumulator is: with a group of four outputs per lane the
// running moments of 512 parts of 257 columns took 12.4 us (four divisions in turn, eight times over), one
// output per lane 5.0 us.
__host__ __device__ __forceinline__ size_t rs_parts_row(uint32_t n_out, uint32_t out_inner, int vec) {
    const uint32_t gpo = (out_inner + vec - 1) / vec;
    return (size_t)gpo * vec * (n_out / out_inner);
}

// one output's parts through the fold of I; E(impl, part, k, acc) folds part k
template <class I, class Part, class F>
__device__ __forceinline__ typename I::Acc rs_fold_output(const I& impl, const Part* base, size_t row, uint32_t k0, uint32_t k1, unsigned pg, unsigned PG,
                                                          unsigned OV, typename I::Acc* slots, F fold) {
    constexpr int B = 8;
    typename I::Acc total = impl.identity();
    for (uint32_t k = k0; k < k1; k += B) {
        Part v[B];
#pragma unroll
        for (int b = 0; b < B; ++b) v[b] = base[(size_t)(k + b < k1 ? k + b : k1 - 1) * row];
        if constexpr (rounds_every<I>::value != 0) {
            // neighbours first: one behind the other, a lane's eight lose as much as all before them have (error of the column
            // sums of 1677 x 20001, 12 parts, in norm: 4.2e-8 that way, 3.9e-8 this way)
#pragma unroll
            for (int b = 0; b < B; ++b)
                if (k + b >= k1) v[b] = impl.identity();
#pragma unroll
            for (int d = 1; d < B; d <<= 1) {
#pragma unroll
                for (int b = 0; b < B; b += 2 * d) impl.combine(v[b + d], v[b]);
            }
            impl.combine(v[0], total);
        } else {
#pragma unroll
            for (int b = 0; b < B; ++b)
                if (k + b < k1) fold(v[b], k + b, total);
        }
    }
    for (unsigned d = 1; d < PG; d <<= 1) {
        slots[threadIdx.x] = total;
        __syncthreads();
        if ((pg & (2 * d - 1)) == 0) impl.combine(slots[threadIdx.x + d * OV], total);
        __syncthreads();
    }
    return total;
}

template <class Impl>
__global__ __launch_bounds__(kRedBlock) void red_fold_parts_kernel(RedSParams p, Impl impl, size_t row) {
    typedef typename Impl::Acc Acc;
    __shared__ Acc slots[kRedBlock];
    const unsigned PG = 1u << p.fold_bits, OV = (unsigned)kRedBlock >> p.fold_bits;
    const unsigned ov = threadIdx.x & (OV - 1), pg = threadIdx.x / OV;
    const uint32_t o = blockIdx.x * OV + ov;
    const bool ok = o < p.n_out;
    const uint32_t per = (p.n_split + PG - 1) / PG;
    const uint32_t k0 = pg * per < p.n_split ? pg * per : p.n_split;
    const uint32_t k1 = k0 + per < p.n_split ? k0 + per : p.n_split;
    const Acc* base = reinterpret_cast<const Acc*>(p.partial) + (ok ? o : p.n_out - 1);
    Acc total = rs_fold_output(impl, base, row, k0, k1, pg, PG, OV, slots, [&](const Acc& v, uint32_t, Acc& t) {
        if constexpr (combines_in_two_forms<Impl>::value) impl.combine_seldom(v, t);
        else impl.combine(v, t);
    });
    if constexpr (has_exact<Impl>::value) {
        // the parts are plain values in axis order: where the fast fold cannot tell which of two equal
        // values came first, the exact rule over the same values, by the same lanes
        typedef typename Impl::Exact Exact;
        if (__syncthreads_or(ok && pg == 0 && impl.needs_exact(total))) {
            __shared__ typename Exact::Acc exact_slots[kRedBlock];
            const Exact ex = impl.exact();
            const typename Exact::Acc e = rs_fold_output(ex, base, row, k0, k1, pg, PG, OV, exact_slots,
                                                         [&](const Acc& v, uint32_t k, typename Exact::Acc& t) { ex.accumulate_acc(v, (int64_t)k, t); });
            if (impl.needs_exact(total)) total = impl.from_exact(e);
        }
    }
    if (pg != 0 || !ok) return;
    const uint32_t q0 = p.out_inner == p.n_out ? 0u : o / p.out_inner;
    const uint32_t q1 = o - q0 * p.out_inner;
    const int64_t a = (int64_t)q0 * p.out_step[0] + (int64_t)q1 * p.out_step[1];
    const int64_t b = (Impl::NOUT > 1) ? (int64_t)q0 * p.out2_step[0] + (int64_t)q1 * p.out2_step[1] : 0;
    impl.store(total, p.out + a, (Impl::NOUT > 1) ? (p.out2 + b) : nullptr);
}

// The exact second fold by ONE wave over the tiles that a whole block (tpr_bits 8) folded: the
// tiles first, first + every, ... of kRedBlock * VEC * kRsUnroll elements each, every vector of
// them taken by one of the 64 lanes. For the streaming blocks of the kernel below, where only
// the first wave learns (by a shuffle, no barrier, no LDS) that the block's result needs it:
// it is rare (a minimum or maximum that is a zero), and asking the whole block cost every
// launch 0.7 us. Lane 0 returns the result.
template <class Impl, int VEC>
__device__ __attribute__((noinline)) typename Impl::Acc rs_exact_refold_wave(const Impl& impl, const char* base, uint64_t first, uint64_t every,
                                                                              uint64_t end, uint32_t tail) {
    typedef typename Impl::In In;
    typedef typename Impl::Exact Exact;
    const Exact ex = impl.exact();
    typename Exact::Acc e = ex.identity();
    const uint64_t per_tile = (uint64_t)kRedBlock * VEC * kRsUnroll;
    const uint64_t tiles = (end + per_tile - 1) / per_tile;
    const unsigned lane = threadIdx.x & 63u;
    for (uint64_t t = first; t < tiles; t += every) {
        const uint64_t t0 = t * per_tile;
        const uint64_t t1 = t0 + per_tile < end ? t0 + per_tile : end;
        for (uint64_t i = t0 + (uint64_t)lane * VEC; i < t1; i += 64u * VEC) {
            In x[VEC];
            rs_load<In, VEC, false>(base + i * sizeof(In), x);
            ex.template accumulate_n<VEC>(x, (int64_t)i, e);
        }
    }
    if (tail != 0 && first == 0 && lane == 0) {
        const In* rest = reinterpret_cast<const In*>(base) + end;
        for (uint32_t k = 0; k < tail; ++k) ex.accumulate(rest[k], (int64_t)(end + k), e);
    }
    for (unsigned d = 32; d > 0; d >>= 1) {
        const typename Exact::Acc other = shfl_down_any(e, d);
        ex.combine(other, e);
    }
    return impl.from_exact(e);
}

// Few outputs, the axis of each cut over n_split blocks, one launch, no tickets: the first n_out
// blocks read nothing of the input; each waits for the accumulators of its output's other blocks,
// which arrive as 64-bit words {launch number, 32 bits of the accumulator} written with agent-scope
// atomic stores, and folds them in index order as the split form above does. The chain after
// the last block has finished its part is then one store becoming visible and one look at it,
// instead of store, acknowledgement, two tickets in turn, fence and loads (C3 T.sum() on fresh
// operands: 25.0 -> 22.4 us; a sum of 4 MiB: 5.9 -> 4.0 us). A streaming block never waits for
// anything, so the waiting blocks (which the dispatcher starts first) cannot hold the others up;
// a wait gives up after kRsPollLimit looks, counts that and raises the host's give-up word (wait_ctl.h).
constexpr uint32_t kRsHandoverWords = 8192;
constexpr uint32_t kRsHandoverOutputs = 256;
constexpr uint32_t kRsPollLimit = 1u << 24;

template <class Acc>
__device__ __forceinline__ Acc rs_await(const uint64_t* slot, uint32_t launch, WaitCtl* ctl) {
    constexpr int W = sizeof(Acc) / 4;
    union U {
        Acc a;
        uint32_t w[W];
        __device__ U() {}
    } u;
    uint64_t x[W];
#pragma unroll
    for (int i = 0; i < W; ++i) x[i] = __hip_atomic_load(slot + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    uint32_t looks = 0;
    const uint32_t limit = wait_limit(ctl, kRsPollLimit);
    for (;;) {
        bool all = true;
#pragma unroll
        for (int i = 0; i < W; ++i) all = all && (uint32_t)(x[i] >> 32) == launch;
        if (all) break;
        if (++looks > limit) {
            wait_gave_up(ctl, WAIT_REDUCE);
            break;
        }
        __builtin_amdgcn_s_sleep(4);
#pragma unroll
        for (int i = 0; i < W; ++i)
            if ((uint32_t)(x[i] >> 32) != launch) x[i] = __hip_atomic_load(slot + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
#pragma unroll
    for (int i = 0; i < W; ++i) u.w[i] = (uint32_t)x[i];
    return u.a;
}

template <class Impl, int VEC, bool NT>
__global__ __launch_bounds__(kRedBlock) void red_srow_poll_kernel(RedSParams p, Impl impl, uint64_t* words, uint32_t launch) {
    typedef typename Impl::In In;
    typedef typename Impl::Acc Acc;
    constexpr int W = sizeof(Acc) / 4;
    static_assert(sizeof(Acc) % 4 == 0, "accumulator must be a whole number of 32-bit words");
    __shared__ Acc wave_slots[kRedBlock / 64];
    __shared__ int s_need;
    if (blockIdx.x >= p.n_out) {
        const uint32_t vrow = blockIdx.x - p.n_out;
        const uint32_t i_out = vrow / p.n_split;
        const uint32_t i_split = vrow - i_out * p.n_split;
        uint32_t o0, o1;
        rs_split_out(p, i_out, o0, o1);
        const int64_t in_off = (int64_t)o0 * p.in_step[0] + (int64_t)o1 * p.in_step[1];
        const int64_t idx_base = p.index_mode == 2 ? in_off / (int64_t)sizeof(In) : 0;
        Acc acc = rs_row_scan<Impl, VEC, NT>(impl, p.in + in_off, i_split, p.n_split, p.n, p.tail, threadIdx.x, 8, idx_base);
        rs_group_combine(impl, acc, 8, wave_slots);
        if constexpr (has_exact<Impl>::value) {
            // thread 0 holds the block's result; its wave alone repeats the fold where that is needed
            if (threadIdx.x >= 64) return;
            const int mine = impl.needs_exact(acc) ? 1 : 0;
            if (__shfl(mine, 0) != 0) acc = rs_exact_refold_wave<Impl, VEC>(impl, p.in + in_off, i_split, p.n_split, p.n, p.tail);
        }
        if (threadIdx.x == 0) {
            union U {
                Acc a;
                uint32_t w[W];
                __device__ U() {}
            } u;
            u.a = acc;
#pragma unroll
            for (int i = 0; i < W; ++i)
                __hip_atomic_store(words + (size_t)vrow * W + i, ((uint64_t)launch << 32) | u.w[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        return;
    }
    // fold the output's accumulators in index order: thread t takes chunks t, t + 256, ...
    const uint32_t i_out = blockIdx.x;
    uint32_t o0, o1;
    rs_split_out(p, i_out, o0, o1);
    const uint64_t* mine = words + (size_t)i_out * p.n_split * W;
    const int64_t o_a = (int64_t)o0 * p.out_step[0] + (int64_t)o1 * p.out_step[1];
    const int64_t o_b = (Impl::NOUT > 1) ? (int64_t)o0 * p.out2_step[0] + (int64_t)o1 * p.out2_step[1] : 0;
    if constexpr (has_exact<Impl>::value) {
        typedef typename Impl::Exact Exact;
        Acc total = impl.identity();
        for (uint32_t k = threadIdx.x; k < p.n_split; k += kRedBlock) impl.combine(rs_await<Acc>(mine + (size_t)k * W, launch, p.wait), total);
        rs_group_combine(impl, total, 8, wave_slots);
        if (threadIdx.x == 0) s_need = impl.needs_exact(total) ? 1 : 0;
        __syncthreads();
        if (s_need) {
            const Exact ex = impl.exact();
            __shared__ typename Exact::Acc exact_slots[kRedBlock / 64];
            typename Exact::Acc e = ex.identity();
            for (uint32_t k = threadIdx.x; k < p.n_split; k += kRedBlock) ex.accumulate_acc(rs_await<Acc>(mine + (size_t)k * W, launch, p.wait), (int64_t)k, e);
            rs_group_combine(ex, e, 8, exact_slots);
            total = impl.from_exact(e);
        }
        if (threadIdx.x == 0) impl.store(total, p.out + o_a, (Impl::NOUT > 1) ? (p.out2 + o_b) : nullptr);
    } else {
        Acc total = impl.identity();
        for (uint32_t k = threadIdx.x; k < p.n_split; k += kRedBlock) impl.combine(rs_await<Acc>(mine + (size_t)k * W, launch, p.wait), total);
        rs_group_combine(impl, total, 8, wave_slots);
        if (threadIdx.x == 0) impl.store(total, p.out + o_a, (Impl::NOUT > 1) ? (p.out2 + o_b) : nullptr);
    }
}

// Column form: a lane owns VEC neighbouring outputs (a group) and walks the reduce axis, four rows in flight.
//
// What bounds it is how memory sees the reads, so that is what the split is for. A block is `width` groups side by
// side (as equal a share of the row as whole blocks give, 256 groups at most) times `slots` lanes that share the
// rows: slot s takes four rows, then the four that come slots * 4 later, so the whole block moves down one window
// of slots * 4 rows at a time. Neither number is a power of two: 65 groups of a 257-column row are one
// block of 65 x 7 lanes (blocks of 64 groups left a second block beside the first with one lane of 64 at work), and
// a slot that kept a stretch of the axis to itself opened one stream per slot (131072 x 64: 27.1 -> 22 us).
// PARTIAL: the axis is also cut across blocks, p.n_split ways, so that 256 blocks run: one on each compute unit, half of
// what fits, reads faster than a full device (131072 x 256, this launch alone: 20.7 us against 21.9 for 512 blocks and 22.3
// for 1024). Neighbouring blocks are neighbouring parts of the same columns: with the columns going first, 4096 x 4095
// DFloat took 28.5 us instead of 24.9 and 2048 x 16384 SFloat 32.9 instead of 25.4, since block numbers go round the eight dies
// and each die then has the same columns of every row.
// Column sums of 128 MiB of SFloat, fresh operands, the fold included, before and after: 131072 x 257 41.6 -> 25.2 us,
// 8192 x 4096 26.5 -> 24.5, 8192 x 4095 27.9 -> 24.3, 2048 x 16384 30.4 -> 22.0, 65536 x 500 30.0 -> 24.2; stddev of
// 131072 x 257 51.7 -> 28.4; 500 x 500 (one launch instead of two) 6.7 -> 4.1.
constexpr int kRcBlock = 512;   // SHARE: lanes of a block (slots * width of them at work)
constexpr int kRcRows = 4;      // rows a lane has in flight

// two accumulators of VEC outputs each, `next` of later rows
template <class I, int VEC>
__device__ __forceinline__ void rc_combine(const I& impl, const typename I::Acc (&next)[VEC], typename I::Acc (&acc)[VEC]) {
    if constexpr (folds_columns_together<I>::value) {
        impl.template combine_columns<VEC>(next, acc);
    } else {
#pragma unroll
        for (int j = 0; j < VEC; ++j) impl.combine(next[j], acc[j]);
    }
}

// Steps of a run of a lane that walks `rows` rows (see rc_walk) and rounds every `every` of them. m roundings in runs of L leave
// an error that goes with the root of L^2 / 3m inside the runs and of m / 3L between them: least at L^3 = m^2 / 2. Few rows stay one
// run (var of 500 x 500, eight rows a lane, costs 0.4 of its 6.6 us more in runs).
static inline uint32_t rc_run_steps(uint64_t rows, int every) {
    if (rows <= 32) return 0xffffffffu;
    const double m = (double)rows / every;
    const uint64_t steps = ((uint64_t)std::ceil(std::cbrt(m * m / 2)) * every + kRcRows - 1) / kRcRows;
    return steps < 1 ? 1u : (steps > 0xffffffffull ? 0xffffffffu : (uint32_t)steps);
}

// The lane's rows [begin, end) in steps of `step`, kRcRows at a time, through the fold of I.
// Where that rounds, it goes in runs of p.run steps, each folded by itself and then into what the lane has: all rows in one chain
// would lose the more the fewer lanes share them. Error of the sum of uniform SFloat columns, in norm, one chain / runs:
// 128 x 262144 1.6e-7 / 5.4e-8, 4096 x 262144 8.4e-7 / 8.2e-8 (a lane per group); 4096 x 65536 1.1e-7 / 4.5e-8 (eight slots).
// The times stay what they are: it is memory that a lane waits for.
template <class I, int VEC, bool NT>
__device__ __forceinline__ void rc_walk(const I& impl, const RedSParams& p, int64_t in_off, uint64_t begin, uint64_t end, uint64_t step,
                                        typename I::Acc (&acc)[VEC]) {
    typedef typename I::In In;
    typedef typename I::Acc Acc;
    constexpr int U = kRcRows;
    constexpr bool RUNS = rounds_every<I>::value != 0;
    const char* base = p.in + in_off;
    Acc own[VEC];
    Acc(&to)[VEC] = RUNS ? own : acc;
    uint32_t left = p.run;
    bool several = false;
#pragma unroll
    for (int j = 0; j < VEC; ++j) acc[j] = own[j] = impl.identity();
    for (uint64_t i0 = begin; i0 < end; i0 += step) {
        In x[U][VEC];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint64_t i = i0 + u;
            const uint64_t ic = i < end ? i : end - 1;
            rs_load<In, VEC, NT>(base + (int64_t)ic * p.red_step, x[u]);
        }
        __builtin_amdgcn_sched_barrier(0);  // all loads of the step issued before the first fold
        if (i0 + U <= end && p.index_mode != 2) {
            // a whole block of consecutive positions along the axis for each output
            if constexpr (folds_columns_together<I>::value) {
                // (the lane's outputs have had the same positions so far: what depends on the count alone is worked out once)
                impl.template accumulate_columns<U, VEC>(x, to);
            } else if constexpr (folds_columns_by_position<I>::value) {
                impl.template accumulate_columns_by_position<U, VEC>(x, (int64_t)i0, to);
            } else {
#pragma unroll
                for (int j = 0; j < VEC; ++j) {
                    In t[U];
#pragma unroll
                    for (int u = 0; u < U; ++u) t[u] = x[u][j];
                    impl.template accumulate_n<U>(t, (int64_t)i0, to[j]);
                }
            }
        } else {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const uint64_t i = i0 + u;
                if (i < end) {
#pragma unroll
                    for (int j = 0; j < VEC; ++j) {
                        int64_t idx = 0;
                        if (I::USES_INDEX)
                            idx = (p.index_mode == 2) ? ((in_off + (int64_t)i * p.red_step) / (int64_t)sizeof(In) + j) : (int64_t)i;
                        impl.accumulate(x[u][j], idx, to[j]);
                    }
                }
            }
        }
        if constexpr (RUNS) {
            if (--left == 0) {
                left = p.run;
                several = true;
                rc_combine<I, VEC>(impl, own, acc);
#pragma unroll
                for (int j = 0; j < VEC; ++j) own[j] = impl.identity();
            }
        }
    }
    if constexpr (RUNS) {
        if (several) {
            rc_combine<I, VEC>(impl, own, acc);
        } else {
#pragma unroll
            for (int j = 0; j < VEC; ++j) acc[j] = own[j];
        }
    }
}

// The slots' accumulators of every group meet pairwise through LDS: log2(slots) rounds in which every left-hand
// lane works. Slot 0 ends up with everything. (Slots hold interleaved rows: what depends on the order of the
// axis rides in the accumulator as a position.)
template <class I, int VEC>
__device__ __forceinline__ void rc_meet(const I& impl, typename I::Acc (&acc)[VEC], unsigned s, unsigned slots, unsigned width, char* lds) {
    typedef typename I::Acc Acc;
    Acc(*part)[VEC] = reinterpret_cast<Acc(*)[VEC]>(lds);
#pragma unroll
    for (int j = 0; j < VEC; ++j) part[threadIdx.x][j] = acc[j];
    __syncthreads();
    for (unsigned d = 1; d < slots; d <<= 1) {
        if ((s & (2u * d - 1u)) == 0 && s + d < slots) {
            Acc next[VEC];
#pragma unroll
            for (int j = 0; j < VEC; ++j) next[j] = part[threadIdx.x + d * width][j];
            rc_combine<I, VEC>(impl, next, acc);
            if (2u * d < slots) {
#pragma unroll
                for (int j = 0; j < VEC; ++j) part[threadIdx.x][j] = acc[j];
            }
        }
        __syncthreads();
    }
}

// LDS of a SHARE block: the wider of the accumulators that meet there
template <class Impl, int VEC>
constexpr size_t rc_lds_bytes() {
    if constexpr (has_exact<Impl>::value) {
        constexpr size_t a = sizeof(typename Impl::Acc), e = sizeof(typename Impl::Exact::Acc);
        return (a > e ? a : e) * VEC * kRcBlock;
    } else {
        return sizeof(typename Impl::Acc) * VEC * kRcBlock;
    }
}

template <class Impl, int VEC, bool NT, bool SHARE, bool PARTIAL = false>
__global__ __launch_bounds__(SHARE ? kRcBlock : kRedBlock) void red_scol_kernel(RedSParams p, Impl impl) {
    typedef typename Impl::Acc Acc;
    static_assert(rc_lds_bytes<Impl, VEC>() <= 65536, "the accumulators of a block fit its share of LDS");
    __shared__ __align__(16) char lds[SHARE ? rc_lds_bytes<Impl, VEC>() : 16];
    const unsigned width = SHARE ? p.width : (unsigned)kRedBlock;
    const unsigned slots = SHARE ? p.slots : 1u;
    const unsigned s = SHARE ? threadIdx.x / width : 0u;
    const unsigned c = threadIdx.x - s * width;
    // (the inner output dimension need not be a whole number of vectors: its last group is pulled
    // back to its last VEC outputs and stores only those the group before it does not)
    const uint32_t gpo = (p.out_inner + VEC - 1) / VEC;            // groups per position of the outer output dimension
    const uint32_t groups = (p.n_out / p.out_inner) * gpo;
    const uint32_t n_cb = (groups + width - 1) / width;
    // this block's stretch of the axis
    const uint32_t cb_first = PARTIAL ? blockIdx.x / p.n_split : blockIdx.x;
    const uint32_t part_no = PARTIAL ? blockIdx.x - cb_first * p.n_split : 0u;
    uint64_t b0 = 0, b1 = p.n;
    if (PARTIAL) {
        b0 = (uint64_t)part_no * p.chunk;
        if (b0 > p.n) b0 = p.n;
        b1 = b0 + p.chunk;
        if (b1 > p.n) b1 = p.n;
    }
    for (uint32_t cb = cb_first; cb < n_cb; cb += gridDim.x) {
        const uint32_t g = cb * width + c;
        const bool ok = g < groups && s < slots;
        const uint32_t gg = g < groups ? g : groups - 1;
        const uint32_t o0 = p.out_inner == p.n_out ? 0u : gg / gpo;
        const uint32_t own1 = (gg - o0 * gpo) * VEC;
        const uint32_t o1 = own1 + VEC <= p.out_inner ? own1 : p.out_inner - VEC;  // where the group's vector starts
        const uint32_t own0 = o0 * p.out_inner + own1;                // the group's first output
        const uint32_t i_out0 = o0 * p.out_inner + o1;
        const int64_t in_off = (int64_t)o0 * p.in_step[0] + (int64_t)o1 * p.in_step[1];
        // (a lane without a group or a slot walks nothing)
        const uint64_t begin = ok ? b0 + (uint64_t)s * kRcRows : b1;
        const uint64_t step = (uint64_t)slots * kRcRows;
        Acc acc[VEC];
        rc_walk<Impl, VEC, NT>(impl, p, in_off, begin, b1, step, acc);
        if constexpr (SHARE) rc_meet<Impl, VEC>(impl, acc, s, slots, width, lds);
        if constexpr (has_exact<Impl>::value) {
            // folded by value; where an output may have lost which of two equal elements came first, its rows
            // are walked again with the rule that carries the position (whole blocks together when lanes share rows)
            bool again = false;
            if (ok && s == 0) {
#pragma unroll
                for (int j = 0; j < VEC; ++j) again = again || impl.needs_exact(acc[j]);
            }
            if (SHARE ? __syncthreads_or(again ? 1 : 0) != 0 : again) {
                typedef typename Impl::Exact Exact;
                const Exact ex = impl.exact();
                typename Exact::Acc e[VEC];
                rc_walk<Exact, VEC, false>(ex, p, in_off, begin, b1, step, e);
                if constexpr (SHARE) rc_meet<Exact, VEC>(ex, e, s, slots, width, lds);
#pragma unroll
                for (int j = 0; j < VEC; ++j)
                    if (impl.needs_exact(acc[j])) acc[j] = impl.from_exact(e[j]);
            }
        }
        if (!ok || s != 0) continue;
        if (PARTIAL) {
            // partial[part][output], a part's outputs padded to whole groups: the lanes of a block write one run
            Acc* mine = reinterpret_cast<Acc*>(p.partial) + (size_t)part_no * ((size_t)gpo * VEC * (p.n_out / p.out_inner)) + i_out0;
#pragma unroll
            for (int j = 0; j < VEC; ++j)
                if (i_out0 + j >= own0) mine[j] = acc[j];
            continue;
        }
#pragma unroll
        for (int j = 0; j < VEC; ++j) {
            if (i_out0 + j < own0) continue;  // (the pulled-back last group: the group before it has these)
            // the VEC outputs of a group are neighbours along the inner output dimension
            const int64_t a = (int64_t)o0 * p.out_step[0] + (int64_t)(o1 + j) * p.out_step[1];
            const int64_t b = (Impl::NOUT > 1) ? (int64_t)o0 * p.out2_step[0] + (int64_t)(o1 + j) * p.out2_step[1] : 0;
            impl.store(acc[j], p.out + a, (Impl::NOUT > 1) ? (p.out2 + b) : nullptr);
        }
    }
}

}  // namespace cumo_hip

#endif
