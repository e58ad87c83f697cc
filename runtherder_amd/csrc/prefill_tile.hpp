// Where the rows of a flash prefill's key tile lie: host and device, so that
// the arithmetic is checked on the CPU at slab sizes past 32 bits.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace rth {

constexpr int kBN = 64;   // keys per tile

// Where a tile's rows are: key0 (clamped to the last tile, so that a copy past
// the end repeats it), the tile's last row that exists (within the tile, so that
// it times a row's bytes fits 32 bits whatever the cache holds), and, paged, the
// offsets (physical - logical key) of its two 32-key halves, each of which lies
// in one block (blocks hold a power of two >= 32 keys).
template <bool kPaged>
struct TileRows {
    int key0, rem, d_lo, d_hi;
    __host__ __device__ __forceinline__ TileRows(int key0_, int total, const int* __restrict__ bt,
                                                 int bshift)
        : key0(key0_), d_lo(0), d_hi(0) {
        const int last_tile = (total - 1) & ~(kBN - 1);
        key0                = key0 < last_tile ? key0 : last_tile;
        rem                 = total - 1 - key0 < kBN - 1 ? total - 1 - key0 : kBN - 1;
        if constexpr (kPaged) {
            d_lo = (bt[key0 >> bshift] << bshift) - (key0 & ~((1 << bshift) - 1));
            d_hi = d_lo;
            if (rem >= 32) {
                const int k1 = key0 + 32;
                d_hi         = (bt[k1 >> bshift] << bshift) - (k1 & ~((1 << bshift) - 1));
            }
        }
    }
    // Byte offset of the tile's row 0 as half `hi` counts its rows. Signed when
    // paged: the second half's block can lie at physical row 0, so that its
    // row 0 counted from the tile's start is row -32.
    __host__ __device__ __forceinline__ int64_t base(bool hi, uint32_t stride) const {
        if constexpr (kPaged) {
            return static_cast<int64_t>(key0 + (hi ? d_hi : d_lo)) * static_cast<int64_t>(stride);
        } else {
            return static_cast<int64_t>(static_cast<uint64_t>(static_cast<uint32_t>(key0)) * stride);
        }
    }
    // Byte offset of the tile's last row that exists: a lane whose row (at byte
    // offset row * stride) lies past it reads it instead, by the smaller of the
    // two offsets.
    __host__ __device__ __forceinline__ uint32_t last_row(uint32_t stride) const {
        return static_cast<uint32_t>(rem) * stride;
    }
};

}  // namespace rth
