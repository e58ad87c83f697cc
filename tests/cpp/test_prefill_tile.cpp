// The key tile's row arithmetic of the flash prefill (csrc/prefill_tile.hpp)
// against 64-bit arithmetic: contiguous caches of up to several times 4 GiB and
// paged ones, every row of the tiles around the places where 32 bits end.
#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <random>
#include <vector>

#include "../../runtherder_amd/csrc/prefill_tile.hpp"

namespace {

long long checked = 0;

// Row r of the tile at key0, as the copies address it, against the row that
// key min(key0 + r, total - 1) has.
template <bool kPaged>
bool check(int key0, int total, uint32_t stride, const int* bt, int shift) {
    using Rows = rth::TileRows<kPaged>;
    const Rows t(key0, total, Rows::entries(key0, total, bt, shift), shift);
    const int from = std::min(key0, (total - 1) / rth::kBN * rth::kBN);
    for (int r = 0; r < rth::kBN; ++r) {
        const bool     hi   = r >= 32;
        const uint32_t off  = t.offset(hi, static_cast<uint32_t>(r & 31) * stride, stride);
        const int64_t  got  = static_cast<int64_t>(t.base(hi, stride)) + off;
        const int64_t  key  = std::min<int64_t>(from + r, total - 1);
        const int64_t  row  = kPaged ? (static_cast<int64_t>(bt[key >> shift]) << shift) +
                                           (key & ((1 << shift) - 1))
                                     : key;
        ++checked;
        if (got != row * stride) {
            std::printf("%s total %d stride %u tile %d row %d: %lld, not %lld\n",
                        kPaged ? "paged" : "contiguous", total, stride, key0, r,
                        static_cast<long long>(got), static_cast<long long>(row * stride));
            return false;
        }
    }
    return true;
}

}  // namespace

int main() {
    for (int hkv : {1, 2, 4, 7, 8, 16, 24, 32, 64, 128}) {
        for (uint32_t stride : {128u * hkv, 4u * hkv}) {   // codes, scales
            for (int wraps = 0; wraps < 4; ++wraps) {
                // Cache lengths around wraps * 2^32 bytes.
                const int64_t around = (static_cast<int64_t>(wraps) << 32) / stride;
                for (int64_t d = -70; d <= 70; ++d) {
                    const int64_t total = around + d;
                    if (total < 1 || total > 0x7fff0000) {
                        continue;
                    }
                    const int last = static_cast<int>((total - 1) / rth::kBN) * rth::kBN;
                    for (int key0 : {0, 64, 4096, last - 64, last, last + 64, last + 256}) {
                        if (key0 >= 0 &&
                            !check<false>(key0, static_cast<int>(total), stride, nullptr, 0)) {
                            return 1;
                        }
                    }
                }
            }
        }
    }
    std::mt19937 rng(5);
    for (int shift : {5, 6, 7, 10}) {
        for (int total : {1, 31, 32, 33, 64, 65, 97, 1000, 5000}) {
            const int        blocks = (total + (1 << shift) - 1) >> shift;
            std::vector<int> bt(blocks + 3);
            for (size_t i = 0; i < bt.size(); ++i) {
                bt[i] = static_cast<int>(i);
            }
            std::shuffle(bt.begin(), bt.end(), rng);
            for (int hkv : {1, 8, 64}) {
                for (int key0 = 0; key0 < total + 192; key0 += rth::kBN) {
                    if (!check<true>(key0, total, 128u * hkv, bt.data(), shift) ||
                        !check<true>(key0, total, 4u * hkv, bt.data(), shift)) {
                        return 1;
                    }
                }
            }
        }
    }
    std::printf("%lld rows\n", checked);
    return checked > 1000000 ? 0 : 2;
}
