// Orders of training samples against their definition, Fisher-Yates with
// rng() % (k + 1), over several epochs of one generator, at sizes around the
// reciprocal table's end; the table's memory whatever the size.
#include <algorithm>
#include <cstdio>
#include <utility>
#include <vector>

#include "../opendynamo_amd/csrc/od_order.hpp"

int main() {
    const size_t cap = od::SampleOrder::kTable;
    long wrong = 0, most = 0;
    for (size_t n : {(size_t)1, (size_t)2, (size_t)1000, cap - 1, cap, cap + 1, 3 * cap + 17})
        for (bool table : {false, true}) {
            od::SampleOrder order(n, 7, table);
            std::mt19937_64 rng(7);
            std::vector<int> got(n), want(n);
            for (int epoch = 0; epoch < 3; ++epoch) {
                order.next(got.data());
                for (size_t k = 0; k < n; ++k) want[k] = (int)k;
                for (size_t k = n - 1; k > 0; --k) std::swap(want[k], want[rng() % (k + 1)]);
                wrong += got != want;
            }
            if ((long)order.table_bytes() > most) most = (long)order.table_bytes();
        }
    // as many samples as a training run takes: only the table is allocated here
    most = std::max(most, (long)od::SampleOrder((size_t)0x7fffffff, 1, true).table_bytes());
    std::printf("wrong %ld table_bytes %ld\n", wrong, most);
    return wrong != 0;
}
