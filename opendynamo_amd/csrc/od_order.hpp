// Order of the samples in a training epoch: Fisher-Yates from the identity with
// one seeded generator for all epochs (od_mlp_train).
#pragma once
#include <cstddef>
#include <cstdint>
#include <cstdlib>
#include <random>
#include <utility>

namespace od {

class SampleOrder {
   public:
    // Divisors up to here have their reciprocal in a table, 2 MB at most: x mod d
    // without a 64-bit division, as an epoch takes one modulus per sample, with
    // the same divisors every time.  Larger sample sets take x % d beyond it, no
    // slower there (the table and the order then both miss the caches: 16 million
    // samples 206 ms with % alone, 201 with this table, 225 with one of all
    // divisors) and in no more memory than their order needs.
    static constexpr size_t kTable = (size_t)1 << 18;

    // n samples; table: worth filling (more than one epoch).
    SampleOrder(size_t n, uint64_t seed, bool table) : n_(n), rng_(seed) {
        if (!table) return;
        const size_t m = n < kTable ? n : kTable;
        inv_ = (uint64_t*)std::malloc((m + 1) * sizeof(uint64_t));
        if (!inv_) return;
        for (size_t d = 1; d <= m; ++d) inv_[d] = ~(uint64_t)0 / d;
        n_inv_ = m;
    }
    ~SampleOrder() { std::free(inv_); }
    SampleOrder(const SampleOrder&) = delete;
    SampleOrder& operator=(const SampleOrder&) = delete;

    // The next epoch's order -> perm[n].
    void next(int* perm) {
        for (size_t k = 0; k < n_; ++k) perm[k] = (int)k;
        for (size_t k = n_ - 1; k > 0; --k) std::swap(perm[k], perm[mod(rng_(), k + 1)]);
    }
    size_t table_bytes() const { return n_inv_ * sizeof(uint64_t); }

   private:
    // q = the high half of x floor((2^64 - 1) / d) is floor(x / d) or one less.
    size_t mod(uint64_t x, size_t d) const {
        if (d > n_inv_) return (size_t)(x % d);
        const uint64_t r = x - (uint64_t)(((unsigned __int128)x * inv_[d]) >> 64) * d;
        return (size_t)(r >= d ? r - d : r);
    }
    size_t n_, n_inv_ = 0;
    std::mt19937_64 rng_;
    uint64_t* inv_ = nullptr;
};

}  // namespace od
