// Vector stores of results, 128 bits a lane: the form, and the rule that picks it.
// Where the lanes of a wave fill whole 64-byte pieces of memory (`pieces`: the result, and each of its rows, starts on
// one) they are written through the second-level cache at device scope (`sc1`): the last-level cache has the line as it
// is written, so the operation that reads the result next finds up to about 200 MB of it there, and the second-level
// cache keeps nothing dirty that it would write back later, in an order of its own, beside what the next operation
// reads. Measured with a 1R+1W kernel (four vectors in flight a lane, operands loaded non-temporally, every launch on
// fresh operands), us a launch on the MI355X:
//   array      copy, plain / nt / sc1    a copy and a copy of its result    a copy and a sum of its result
//   1 MiB      2.8 / 2.9 / 2.4           5.1 / 5.4 / 4.7                    4.7 / 5.0 / 4.4
//   16 MiB     7.4 / 6.6 / 7.0           14.1 / 13.3 / 12.9                 10.8 / 10.5 / 10.5
//   128 MiB    46.8 / 44.2 / 43.4        85.8 / 88.3 / 82.0                 59.6 / 64.4 / 58.0
//   512 MiB    185 / 175.5 / 175.8       371 / 349 / 351                    248 / 253 / 236
// For a call on its own it is no gain in every kernel; its reader is the faster for it (the library's calls, us, non-temporal / sc1):
//   SFloat x.clip(-1,1), x ** 3, [8192,4096]                    43.2 / 42.1, 44.5 / 42.6
//   two operands, flat: SFloat.maximum [8192,4096], 2^26 t + b  63.5 / 65.0, 125.1 / 126.3
//   DFloat [4096,4096] + [1,4096], alone and with the sum and the maximum of its rows  43.2 / 42.2, 89.0 / 82.6
//   SFloat [32768,1024] + [32768,1], alone, then times 2, then the sum of its rows     43.5 / 43.8, 86.7 / 82.9, 64.7 / 60.8
//   SFloat [8192,4096] transposed (from `nt sc1`), alone and with a copy of it  47.8 / 48.6, 91.2 / 85.3
//   SFloat [8192,4112] transposed, whose rows end inside a line                 50.8 / 54.6, 94.2 / 90.0
//   512 MiB of SFloat: S - m, e / z, Fused.softmax(S)           169.3 / 170.0, 166.8 / 170.4, 189.6 / 191.9
// From other boundaries every wave would leave part of a piece at each end (128 MiB, 32 bytes off: 47.6 / 45.5 /
// 49.9), so those results go non-temporally where NT, from stream_past_caches, says so, else plainly.
#pragma once
#ifndef CUMO_HIP_HOST_CHECK  // (a CPU build checks the rule alone)
#include <hip/hip_runtime.h>
#endif

#include <cstdint>

namespace cumo_hip {

constexpr uint64_t kStorePiece = 64;

// whether every one of these (an address, byte steps) is a whole number of pieces
template <class... S>
constexpr bool store_pieces(uint64_t address, S... steps) {
    return ((address | ... | (uint64_t)steps) & (kStorePiece - 1)) == 0;
}

// Kernels that write rows ask on the host as well whether the rows may be written through at all (`through`). Rows that follow
// one another may: what a row leaves of its last line the next one fills. Rows with gaps between them (a window, z[:, :w] = x)
// may where they are whole 128-byte lines of the second-level cache, start and length. Else each leaves parts of lines, and
// the call costs 5 to 30 % more; a reader right behind it gets that back where rows end inside a piece, and not where they
// are whole pieces. 2^24 SFloat in z, us, non-temporal / written through (in brackets with a copy of the window after it):
//   w 36 of 64      20.5 / 25.9 (38.9 / 35.1)        w 48 of 64       18.8 / 23.0 (39.4 / 40.2)
//   w 1004 of 1040  23.5 / 27.4 (47.1 / 42.2)        w 1008 of 1040   23.0 / 25.6 (45.9 / 46.9)
//   w 4100 of 4160  23.7 / 25.1 (47.8 / 42.3)        w 4080 of 4160   23.5 / 24.7 (47.0 / 46.2)
//   whole lines: w 4096 of 4160  23.3 / 23.8 (46.4 / 44.4);  no gaps: [33288,1008] + [33288,1]  44.3 / 44.6 (87.6 / 83.6)
// Below the size of the non-temporal forms writing through wins either way (6 * 2^20 SFloat, plain / through: w 36 of 64
// 9.8 / 8.7, w 1008 of 1040 12.3 / 11.3).
struct StoreRows {
    uint64_t bytes, reach, bits;  // what the rows hold; from the first byte to the last; address, steps and length or-ed

    StoreRows(const void* p, uint64_t row_bytes) : bytes(row_bytes), reach(row_bytes), bits((uint64_t)(uintptr_t)p | row_bytes) {}
    void dimension(uint64_t n, int64_t step) {
        if (n <= 1) return;
        bytes *= n;
        reach += (n - 1) * (step < 0 ? 0 - (uint64_t)step : (uint64_t)step);
        bits |= (uint64_t)step;
    }
    bool through(bool nt) const { return !nt || bytes == reach || (bits & 127) == 0; }
};

#ifndef CUMO_HIP_HOST_CHECK
template <class... S>
__device__ __forceinline__ bool store_pieces(const void* p, S... steps) {
    return store_pieces((uint64_t)(uintptr_t)p, steps...);
}

typedef uint32_t store_u4 __attribute__((ext_vector_type(4)));

template <bool NT>
__device__ __forceinline__ void store_vector(store_u4* p, store_u4 v, bool pieces) {
    if (pieces) __builtin_amdgcn_global_store_b128((__attribute__((address_space(1))) store_u4*)p, v, "agent");
    else if (NT) __builtin_nontemporal_store(v, p);
    else *p = v;
}

// The same for kernels that write a tile of many rows at a time: where the pieces are not whole, non-temporal stores of large
// results are written through at device scope as well (`nt sc1`), so that the second-level cache does not collect the partly
// written lines of many rows before it lets them go (windows of z written with a transposed SFloat, w 36 of 64 23.6 us with
// `nt`, 22.9 so; 1004 of 1040 28.2, 27.6; 4100 of 4160 27.0, 26.5). No builtin spells the pair, and what the compiler does
// not know for a store it does not guard: the registers of a 128-bit store may be written again two wait states later,
// which the s_nop behind it gives.
template <bool NT>
__device__ __forceinline__ void store_tile_vector(store_u4* p, store_u4 v, bool pieces) {
    if (!NT || pieces) store_vector<NT>(p, v, pieces);
    else asm volatile("global_store_dwordx4 %0, %1, off nt sc1\n\ts_nop 1" ::"v"(p), "v"(v) : "memory");
}
#endif

}  // namespace cumo_hip
