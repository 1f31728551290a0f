// Compares the rules that pick the written-through form of vector stores (cumo_amd/csrc/store_form.h) with a look at
// every row of a result: which rows start on whole pieces, which leave gaps, which are whole lines. Prints the number
// of results compared; exits 1 at the first difference.
#define CUMO_HIP_HOST_CHECK
#include "../cumo_amd/csrc/store_form.h"

#include <algorithm>
#include <cstdio>
#include <initializer_list>
#include <utility>
#include <vector>

using cumo_hip::StoreRows;
using cumo_hip::store_pieces;

typedef std::pair<int64_t, int64_t> Extent;

int main() {
    long compared = 0;
    for (int64_t start : {0, 4, 16, 32, 48, 64, 128, 192})
        for (int64_t bytes : {16, 48, 64, 112, 128, 144, 192, 256, 4032, 4096, 4100})
            for (int64_t gap : {0, 4, 16, 64, 128, 144, 8192})
                for (int64_t outer_gap : {0, 16, 64, 128, 4096})
                    for (int r0 : {1, 3})
                        for (int r1 : {1, 2, 5})
                            for (int sign : {1, -1}) {
                                const int64_t step = sign * (bytes + gap);
                                const int64_t outer = (bytes + gap) * r1 + outer_gap;
                                const int64_t base = (1 << 20) + start;
                                std::vector<Extent> rows;
                                for (int i = 0; i < r0; ++i)
                                    for (int j = 0; j < r1; ++j) rows.push_back(Extent(base + i * outer + j * step, base + i * outer + j * step + bytes));
                                bool pieces = true, lines = true, dense = true;
                                for (const Extent& r : rows) {
                                    pieces = pieces && r.first % 64 == 0;
                                    lines = lines && r.first % 128 == 0 && r.second % 128 == 0;
                                }
                                std::sort(rows.begin(), rows.end());
                                for (size_t k = 1; k < rows.size(); ++k) dense = dense && rows[k].first == rows[k - 1].second;
                                StoreRows s(reinterpret_cast<const void*>(base), (uint64_t)bytes);
                                s.dimension((uint64_t)r1, step);
                                s.dimension((uint64_t)r0, outer);
                                const bool starts = store_pieces((uint64_t)base, r1 > 1 ? step : 0, r0 > 1 ? outer : 0);
                                if (starts != pieces || s.through(true) != (dense || lines) || !s.through(false)) {
                                    std::printf("start %ld bytes %ld step %ld outer %ld rows %d x %d\n", (long)start, (long)bytes, (long)step, (long)outer, r0, r1);
                                    return 1;
                                }
                                ++compared;
                            }
    std::printf("%ld\n", compared);
    return 0;
}
