// Where the rows of a flash prefill's key tile lie: host and device, so that
// the arithmetic is checked on the CPU at slab sizes past 32 bits.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace rth {

constexpr int kBN = 64;   // keys per tile

// Where the rows of a key tile are: base(hi) is the byte offset of the first row
// of its first or second half (32 keys), offset(hi, x) that of a lane whose row
// lies x bytes into the half, as far as there are keys: a row past the last key
// reads the last one. Products of rows within a tile, 32 bits whatever the cache
// holds. A tile past the last one repeats it.
// Contiguous: both halves count from the tile's first row.
template <bool kPaged>
struct TileRows {
    struct Entries {};
    static __host__ __device__ __forceinline__ Entries entries(int, int, const int*, int) {
        return {};
    }

    int key0, rem;   // the tile's first key, its last row that exists
    __host__ __device__ __forceinline__ TileRows(int key, int total, Entries, int) {
        const int last_tile = (total - 1) & ~(kBN - 1);
        key0                = key < last_tile ? key : last_tile;
        rem                 = total - 1 - key0 < kBN - 1 ? total - 1 - key0 : kBN - 1;
    }
    __host__ __device__ __forceinline__ uint64_t base(bool, uint32_t stride) const {
        return static_cast<uint64_t>(static_cast<uint32_t>(key0)) * stride;
    }
    __host__ __device__ __forceinline__ uint32_t offset(bool hi, uint32_t x, uint32_t stride) const {
        const uint32_t row = x + (hi ? kBN / 2 * stride : 0u);
        const uint32_t lim = static_cast<uint32_t>(rem) * stride;
        return row < lim ? row : lim;
    }
};

// Paged: each half lies in one block (blocks hold a power of two >= 32 keys); a
// half without keys takes the last key's row. The block table's entries come in
// by themselves (Entries), so that a kernel can load them ahead.
template <>
struct TileRows<true> {
    struct Entries {
        uint32_t lo, hi;
    };
    struct Keys {
        uint32_t lo, hi;   // the halves' first keys
    };
    static __host__ __device__ __forceinline__ Keys keys(int key, int total) {
        const uint32_t end = static_cast<uint32_t>(total - 1), k = static_cast<uint32_t>(key);
        const uint32_t last_tile = end & ~static_cast<uint32_t>(kBN - 1);
        const uint32_t k0        = k < last_tile ? k : last_tile;
        return {k0, k0 + kBN / 2 < end ? k0 + kBN / 2 : end};
    }
    static __host__ __device__ __forceinline__ Entries entries(int key, int total,
                                                               const int* __restrict__ bt,
                                                               int bshift) {
        const Keys k = keys(key, total);
        return {static_cast<uint32_t>(bt[k.lo >> bshift]), static_cast<uint32_t>(bt[k.hi >> bshift])};
    }

    uint32_t row_lo, row_hi;   // physical rows of the halves' first keys
    uint32_t rem;              // the tile's last row that exists
    __host__ __device__ __forceinline__ TileRows(int key, int total, Entries e, int bshift) {
        const Keys     k   = keys(key, total);
        const uint32_t in  = (1u << bshift) - 1u;   // mask: a key's place in its block
        const uint32_t end = static_cast<uint32_t>(total - 1);
        row_lo             = (e.lo << bshift) | (k.lo & in);
        row_hi             = (e.hi << bshift) | (k.hi & in);
        rem                = end - k.lo < kBN - 1 ? end - k.lo : kBN - 1;
    }
    __host__ __device__ __forceinline__ uint64_t base(bool hi, uint32_t stride) const {
        return static_cast<uint64_t>(hi ? row_hi : row_lo) * stride;
    }
    __host__ __device__ __forceinline__ uint32_t offset(bool hi, uint32_t x, uint32_t stride) const {
        // The half's last row that exists (without keys: its only one).
        constexpr uint32_t kHalf = kBN / 2;
        const uint32_t last = hi ? (rem > kHalf ? rem : kHalf) - kHalf : rem < kHalf - 1 ? rem : kHalf - 1;
        const uint32_t lim  = last * stride;
        return x < lim ? x : lim;
    }
};

}  // namespace rth
