// Causal flash prefill over an OCP E4M3 KV cache, gfx950.
//
// Math follows flash_prefill_bf16 (reference src/kernels/flash_prefill.cu:
// 34-241): causal rule "query t at position cache_len + t sees keys
// 0 .. cache_len + t" (:127-139), online softmax in fp32, bf16 RNE output of
// O / l. head_dim is 128, as in the reference (:226).
//
// MI355X design:
//  * Rows: the q heads of one kv head are packed token by token (row r of a
//    kv head: token r / G, head r % G), so a block of rows holds few tokens,
//    its waves reach the diagonal in the same tile or the next, and the blocks
//    of one kv head (on one XCD) share its K/V tiles in L2. 32 rows per wave;
//    workgroups of 8 waves (256 rows, one per compute unit) or 4 (128 rows,
//    two per compute unit). Longest (last) row blocks first.
//  * Keys go in 64-key tiles, copied by LDS-DMA (global_load_lds) one and a
//    half tiles or more ahead: K codes unchanged into a ring of three (16-byte
//    chunks XOR-swizzled by row, so the operand reads are bank-conflict free),
//    V codes into a ring of two that each wave copies and reads back for
//    itself, scales into a ring of four. No load of the tile loop goes through
//    registers, and the waits are explicit: the compiler would wait for every
//    outstanding LDS-DMA before each LDS read.
//  * Scores S^T = K Q^T run on the fp8 MFMA v_mfma_scale_f32_32x32x64_f8f6f4
//    with A = the raw K codes from LDS and B = Q split into two E4M3
//    parts: q * 2^a = hi + lo / 16 (a per row, so the row maximum lands in
//    [128, 256)), the MFMA's per-lane E8M0 scales undoing 2^a and 16. A bf16
//    q has 8 significant bits and hi takes the top 4, so for scaled elements
//    |y| >= 2^-6 the split is exact and every product is the exact code * q
//    product, accumulated in fp32. Below 2^-6 (elements more than ~13
//    binades under their row maximum) lo falls into E4M3 subnormals and the
//    split errs by at most 2^-14 in scaled units, 2^-21 of the row maximum
//    (tests/test_prefill_q_split.py checks both over every bf16 value).
//  * Each lane owns one query row (the S^T column), so the softmax needs no
//    cross-lane step except on a rebase. t = s * (k_scale * scale * log2 e)
//    - m_ref against a lazy reference maximum; p = 2^t rounded to f16, the
//    row sum taken from the fp32 2^t.
//  * V is dequantized into LDS as f16(code * v_scale), transposed to V^T in
//    registers (v_perm) before the LDS write, and O^T += V^T P^T runs on
//    v_mfma_f32_32x32x16_f16 with P^T straight from the score registers.
//  * The tile loop is software pipelined by half tiles (32 keys) and written
//    in issue order (sched_barrier between the pieces): the P V MFMAs of one
//    half alternate with the score MFMAs of the half a tile later (which are a
//    dependent chain of four), and both run over the softmax of the half
//    between them, the staging of the next V tile and the operand reads of the
//    MFMAs ahead. Before, a wave did scores, softmax and P V one after the
//    other, and the compiler put a wait for all outstanding copies in front of
//    each tile's reads. What bounds it: one wave per SIMD (4-wave grids of up
//    to one workgroup per compute unit) takes ~2410 cycles a tile, 1.02 us at
//    2.36 GHz (1.6 us before): ~340 instructions, 1024 cycles of MFMAs and the
//    softmax and staging, which one wave overlaps in part only; two waves per
//    SIMD run at 60 % of the MFMA rate at ~1.9 GHz, where the part's power
//    holds it (a large bf16 matrix product: 1.23 PFLOP/s; this kernel at 16384
//    tokens, 32 heads 1.15-1.18). Measured, before -> now, us, both built and
//    timed in turn: 24 heads 1021 / 1700 / 3000 tokens 27.0 -> 23.4, 39.6 -> 35.4,
//    86.3 -> 69.2; 28 heads 1700 48.0 -> 36.8; 32 heads 1021 / 2048 / 3000 / 4096
//    27.0 -> 23.4, 55.3 -> 45.3, 96.1 -> 84.4, 141 -> 133; 8192 / 16384 tokens 511 ->
//    493, 1927 -> 1883, 4096 after 32K / 127K keys 1977 -> 1946, 7449 -> 7283.
//  * Key runs (flash_prefill_keysplit_launch, kPart): for chunks after a long
//    cache, each row block of the 4-wave kernel is split over gridDim.y
//    workgroups, each walking one run of key tiles and storing partials in the
//    split-K decode layout for a merge of its own.
#include <algorithm>
#include <climits>
#include <type_traits>

#include "device_common.hpp"
#include "launch.hpp"
#include "prefill_tile.hpp"

namespace rth {
namespace {

typedef int      i32x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

constexpr int kHD     = 128;         // head_dim
constexpr int kKTile  = kBN * kHD;   // bytes of E4M3 K codes per tile
constexpr int kVPitch = kBN + 8;     // f16 per V^T row in LDS (144 B)
constexpr int kE8M0One = 127;        // E8M0 encoding of 1.0

// LDS column of key o (0..63) in the V^T tile: within each group of 16 keys,
// offset 8a + 4h + b is stored at 8h + 4a + b, so the 8 keys one MFMA lane
// feeds are contiguous.
__device__ __forceinline__ int vt_pos(int o) {
    const int grp = o & ~15;
    const int a   = (o >> 3) & 1;
    const int h   = (o >> 2) & 1;
    return grp + 8 * h + 4 * a + (o & 3);
}

// Row of q / out ([n_new, hq] rows of kHD) that row r of virtual head vhead's
// packed rows holds: token r / pack, q head vhead * pack + r % pack.
__device__ __forceinline__ int64_t packed_row(int r, int pack, int hq, int vhead) {
    const int t = r / pack;
    return static_cast<int64_t>(t) * hq + vhead * pack + (r - t * pack);
}

// Byte offset of 16-byte chunk c (0..7) of K row r (0..63) in an LDS K tile.
__device__ __forceinline__ int k_chunk(int r, int c) {
    return r * kHD + 16 * (c ^ (r & 7));
}

// A lane's part of the tile copies, as byte offsets from the first row of the
// tile's half that the copy lies in (TileRows).
template <int kWaves>
struct TileLane {
    uint32_t kstride, sstride;   // bytes per key: codes, scales
    uint32_t krow, kcol;         // K copy: row offset of slot tid (4 waves: in each half), its chunk
    uint32_t vrow, vcol;         // V copy: row offset of its (even) key, its chunk
    uint32_t srow;               // scale copy: offset of its key

    // The wave's key pairs p (8 of 4 waves, 4 of 8): first key of pair p. Eight
    // waves take the pairs whose V^T words are consecutive (vt_pos).
    static __device__ __forceinline__ int pair_key(int wave, int p) {
        return kWaves == 4 ? 16 * wave + 2 * p
                           : 16 * (wave >> 1) + 4 * (wave & 1) + 2 * (p & 1) + 8 * (p >> 1);
    }

    __device__ __forceinline__ TileLane(int tid, int wave, int lane, int hkv) {
        const int r = tid >> 3;
        const int c = (tid & 7) ^ (r & 7);
        kstride     = static_cast<uint32_t>(hkv) * kHD;
        sstride     = static_cast<uint32_t>(hkv) * 4u;
        krow        = static_cast<uint32_t>(r & (kBN / 2 - 1)) * kstride;
        kcol        = 16u * static_cast<uint32_t>(c);
        // V rows of a wave in LDS: the even keys of its pairs, then the odd ones.
        const int vr = lane >> 3;
        const int vk = kWaves == 4 ? pair_key(wave, vr) : pair_key(wave, vr & 3) + (vr >> 2);
        vrow         = static_cast<uint32_t>(vk & (kBN / 2 - 1)) * kstride;
        vcol         = 16u * static_cast<uint32_t>(lane & 7);
        // Scales of a wave in LDS: v_scale of its keys pair by pair, then k_scale.
        const int sk = lane & (kWaves == 4 ? 15 : 7);
        srow = static_cast<uint32_t>((pair_key(wave, sk >> 1) + (sk & 1)) & (kBN / 2 - 1)) * sstride;
    }
};

// One LDS-DMA of 16 (or 4) bytes per lane: lane l's bytes land at LDS address
// to + 16 l (4 l). In assembly, because the compiler waits for every
// outstanding LDS-DMA before any LDS read; the waits here are explicit. The
// base is the same in every lane: scalar arithmetic on arguments and on what a
// v_readfirstlane gave (the base itself through one, built by the vector ALU,
// cost 0.04 us a tile). A vector-memory read of a scalar register needs five
// wait states after a VALU write of it, which the hardware does not check and
// the compiler does not count inside an asm. The s_mov_b64 makes the scalar ALU
// the last to write it (scalar reads and writes are ordered by the hardware),
// and is the one wait state between the write of m0 and the copy.
__device__ __forceinline__ void dma16(uint32_t to, const uint8_t* base, uint32_t off) {
    to = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(to)));
    asm volatile("s_mov_b32 m0, %1\n\ts_mov_b64 %0, %0\n\tglobal_load_lds_dwordx4 %2, %0"
                 : "+s"(base)
                 : "s"(to), "v"(off)
                 : "memory");
}
// Lanes 0 .. kLanes - 1 only (the wave's lanes are all active).
template <int kLanes>
__device__ __forceinline__ void dma4_low(uint32_t to, const uint8_t* at) {
    static_assert(kLanes >= 16 && kLanes < 64, "");
    constexpr int kLo = kLanes >= 32 ? -1 : (1 << (kLanes & 31)) - 1;
    constexpr int kHi = kLanes > 32 ? (1 << (kLanes & 31)) - 1 : 0;
    to = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(to)));
    asm volatile("s_mov_b32 m0, %0\n\ts_mov_b32 exec_hi, %3\n\ts_mov_b32 exec_lo, %2\n\t"
                 "s_nop 0\n\tglobal_load_lds_dword %1, off\n\ts_mov_b64 exec, -1"
                 :
                 : "s"(to), "v"(at), "i"(kLo), "i"(kHi)
                 : "memory");
}

// K tile: slot s (16 bytes) holds chunk (s & 7) ^ (row & 7) of row s >> 3, so
// that k_chunk() finds it. kh: k + kvh rows. Slots of one copy lie in one
// 32-row half.
template <int kWaves, bool kPaged>
__device__ __forceinline__ void k_tile_dma(uint32_t dst, const uint8_t* __restrict__ kh,
                                           const TileRows<kPaged>& rows,
                                           const TileLane<kWaves>& ln, int wave) {
#pragma unroll
    for (int rep = 0; rep < 8 / kWaves; ++rep) {
        const bool hi = kWaves == 8 ? wave >= 4 : rep == 1;
        dma16(dst + 1024u * static_cast<uint32_t>(wave + rep * kWaves),
              kh + rows.base(hi, ln.kstride), rows.offset(hi, ln.krow, ln.kstride) + ln.kcol);
    }
}

// V tile: each wave copies its own 64 / kWaves keys (8 lanes per key), the
// even keys of its pairs first, and later reads back only those.
template <int kWaves, bool kPaged>
__device__ __forceinline__ void v_tile_dma(uint32_t dst, const uint8_t* __restrict__ vh,
                                           const TileRows<kPaged>& rows,
                                           const TileLane<kWaves>& ln, int wave) {
    const bool     hi   = wave >= kWaves / 2;
    const uint8_t* base = vh + rows.base(hi, ln.kstride);
    const uint32_t to   = dst + static_cast<uint32_t>(wave * (kKTile / kWaves));
    dma16(to, base, rows.offset(hi, ln.vrow, ln.kstride) + ln.vcol);
    if constexpr (kWaves == 4) {
        dma16(to + 1024u, base, rows.offset(hi, ln.vrow + ln.kstride, ln.kstride) + ln.vcol);
    }
}

// A wave's floats of one tile in the scales' ring: v_scale of its keys, k_scale,
// and (paged) the block-table entries of the tile three further on, which come
// with the same copy.
template <int kWaves, bool kPaged>
constexpr int kScaleWave = 128 / kWaves + (kPaged ? 2 : 0);
template <int kWaves, bool kPaged>
constexpr int kScaleTile = kWaves * kScaleWave<kWaves, kPaged>;

// The scales of the wave's keys: v_scale, then k_scale. key3: the first key of
// the tile three further on.
template <int kWaves, bool kPaged>
__device__ __forceinline__ void scale_dma(uint32_t dst, const float* __restrict__ ksh,
                                          const float* __restrict__ vsh,
                                          const TileRows<kPaged>& rows,
                                          const TileLane<kWaves>& ln, int wave, int lane, int key3,
                                          int total, const int* __restrict__ bt, int bshift) {
    constexpr int  kKeys = 64 / kWaves;
    const bool     hi    = wave >= kWaves / 2;
    const uint64_t at    = rows.base(hi, ln.sstride) + rows.offset(hi, ln.srow, ln.sstride);
    const uint8_t* from  = reinterpret_cast<const uint8_t*>(lane < kKeys ? vsh : ksh) + at;
    const uint32_t to    = dst + static_cast<uint32_t>(wave * kScaleWave<kWaves, kPaged> * 4);
    if constexpr (kPaged) {   // lanes 2 kKeys (even) and 2 kKeys + 1: the entries
        const auto     k     = TileRows<kPaged>::keys(key3, total);
        const uint32_t block = ((lane & 1) != 0 ? k.hi : k.lo) >> bshift;
        const uint8_t* e     = reinterpret_cast<const uint8_t*>(bt + block);
        dma4_low<2 * kKeys + 2>(to, lane < 2 * kKeys ? from : e);
    } else {
        dma4_low<2 * kKeys>(to, from);
    }
}

// Exponent field of x alone: 2^floor(log2 x) for normal x > 0, 0 for 0.
__device__ __forceinline__ uint32_t pow2_bits(float x) {
    return __float_as_uint(x) & 0x7f800000u;
}

// V'^T = f16(code * v_scale) of the staged units: the two keys of a unit share
// the larger power of two 2^e of their scales, applied exactly by the
// converter; the f16 factors v_scale / 2^e (rounded once per key, a relative
// error below 2^-11 that enters O linearly) are applied with one packed f16
// multiply.
struct VFactor {
    float p;   // 2^e
    f16x2 m;
};
__device__ __forceinline__ VFactor v_factor(float sa, float sb) {
    const uint32_t e   = max(pow2_bits(sa), pow2_bits(sb));
    const float    inv = __uint_as_float(0x7f000000u - e);   // 2^-e
    return {__uint_as_float(e),
            f16x2{static_cast<_Float16>(sa * inv), static_cast<_Float16>(sb * inv)}};
}

// Word of V^T row d in LDS: rows of kVPitch f16 (conflict-free for the operand
// reads, 32 consecutive rows), 16 words further per 32 rows, which spreads the
// staging writes of lanes 16 d apart.
__device__ __forceinline__ constexpr int vt_row(int d) {
    return d * (kVPitch / 2) + 16 * (d >> 5);
}
constexpr int kVtWords = kHD * (kVPitch / 2) + 16 * (kHD / 32);

// Stages four d of a key pair: wa, wb hold their codes of the two keys, col the
// pair's V^T column at the first of them. swap: the lane writes d + 2, d + 3
// first, so that lanes an odd multiple of 16 d apart use other banks.
struct VOrder {
    uint32_t sel0, sel1;   // byte selectors of the first and the second two d
    int      at0, at1;     // their word offsets
    __device__ __forceinline__ explicit VOrder(bool swap)
        // [a0 b0 a1 b1] and [a2 b2 a3 b3]: the two keys of one d per word.
        : sel0(swap ? 0x07030602u : 0x05010400u), sel1(swap ? 0x05010400u : 0x07030602u),
          at0(swap ? kVPitch : 0), at1(swap ? 0 : kVPitch) {}
};
__device__ __forceinline__ void v_stage4(uint32_t wa, uint32_t wb, const VFactor& f,
                                         const VOrder& v, uint32_t* col0, uint32_t* col1) {
    const uint32_t w0 = __builtin_amdgcn_perm(wb, wa, v.sel0);
    const uint32_t w1 = __builtin_amdgcn_perm(wb, wa, v.sel1);
    const f16x2    x0 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w0, f.p, false) * f.m;
    const f16x2    x1 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w0, f.p, true) * f.m;
    const f16x2    x2 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w1, f.p, false) * f.m;
    const f16x2    x3 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w1, f.p, true) * f.m;
    col0[0]           = __builtin_bit_cast(uint32_t, x0);
    col0[kVPitch / 2] = __builtin_bit_cast(uint32_t, x1);
    col1[0]           = __builtin_bit_cast(uint32_t, x2);
    col1[kVPitch / 2] = __builtin_bit_cast(uint32_t, x3);
}

// Four fp32 -> four E4M3 bytes (RNE; inputs within range).
__device__ __forceinline__ uint32_t pack_e4m3x4(float a, float b, float c, float d) {
    const int lo = __builtin_amdgcn_cvt_pk_fp8_f32(a, b, 0, false);
    return static_cast<uint32_t>(__builtin_amdgcn_cvt_pk_fp8_f32(c, d, lo, true));
}

// Workgroup barrier that orders LDS accesses only: waits for this wave's LDS
// operations, not for its outstanding global loads.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// s_waitcnt immediate (gfx9 encoding: vmcnt in bits 3:0 and 15:14, expcnt
// 6:4, lgkmcnt 11:8) waiting until at most n vector-memory operations are
// outstanding, and for nothing else.
constexpr int waitcnt_vm(int n) {
    return (n & 0xf) | (0x7 << 4) | (0xf << 8) | ((n >> 4) << 14);
}

// Keeps the instruction scheduler from moving anything across: the tile loop
// below is written in the order it is meant to issue.
__device__ __forceinline__ void pin() { __builtin_amdgcn_sched_barrier(0); }

// kPart (4-wave workgroups): the keys are split over gridDim.y workgroups per
// row block; workgroup y takes the y-th run of max(ceil(tiles / S),
// run_min) key tiles and stores its rows' partials (m in log2 units, l,
// unnormalized O) in the split-K decode layout ([rows, S] m, [rows, S] l,
// [rows, S, D] O, rows t * Hq + h) for the merge; a row with no key in
// the run stores m = -inf, l = 0 and, in a workgroup that has keys, O = 0 (a
// workgroup without keys leaves O unwritten; the merge drops slots with m =
// -inf). When run 0 holds every key (at most run_min tiles in all), it stores
// the normalized output instead and the merge returns at once.

template <int kWaves, bool kPaged, bool kPart>
__global__ __launch_bounds__(kWaves * kWave, 2) void flash_prefill_kernel(
    uint16_t* __restrict__ out, const uint16_t* __restrict__ q,
    const uint8_t* __restrict__ k, const uint8_t* __restrict__ v,
    const float* __restrict__ ks, const float* __restrict__ vs, int n_new,
    const int* __restrict__ cache_len, int pack, int share, int hkv, float scale_log2,
    const int* __restrict__ block_table, int block_shift, int first_wgs,
    float* __restrict__ partial, int num_splits, int run_min) {
    constexpr int kBM = 32 * kWaves;   // query rows per workgroup
    // LDS-DMA operations of one tile: K and V 8 / kWaves each, scales 1.
    constexpr int kCopies = 8 / kWaves;
    constexpr int kOps    = 2 * kCopies + 1;

    __shared__ __attribute__((aligned(16))) uint8_t  sK[3 * kKTile];    // K codes: ring of three
    __shared__ __attribute__((aligned(16))) uint8_t  sV[2 * kKTile];    // V codes: ring of two
    __shared__ __attribute__((aligned(16))) uint32_t sVt[2 * kVtWords]; // V^T: ring of two
    __shared__ __attribute__((aligned(16))) float    sKf[4 * kBN];      // k-factors: ring of four
    constexpr int kScTile = kScaleTile<kWaves, kPaged>, kScWave = kScaleWave<kWaves, kPaged>;
    __shared__ __attribute__((aligned(16))) float    sSc[4 * kScTile];  // scales: ring of four

    const int tid  = static_cast<int>(threadIdx.x);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int lane = tid & (kWave - 1);
    const int qn   = lane & 31;   // query row of this lane within the wave
    const int h    = lane >> 5;   // k-group

    // Virtual head vhead: `pack` q heads of one kv head, whose rows are packed
    // token by token (row r: token r / pack, head r % pack); each kv head has
    // `share` of them. Heavy (last) row blocks first, the virtual heads of one
    // kv head on one XCD.
    const int n_rows  = n_new * pack;   // of one virtual head
    const int n_heads = hkv * share;
    const int n_blk   = (n_rows + kBM - 1) / kBM;
    const int bid     = static_cast<int>(blockIdx.x);
    const int blk     = bid >= first_wgs ? (bid - first_wgs) / n_heads : n_blk - 1 - bid / n_heads;
    const int hb      = bid % n_heads;
    const int vhead   = ((n_heads & 7) == 0) ? ((hb & 7) * (n_heads >> 3) + (hb >> 3)) : hb;
    const int kvh     = vhead / share;
    const int hq      = n_heads * pack;

    const int clen    = *cache_len;
    const int total   = clen + n_new;
    const int q0      = blk * kBM;
    const int last    = (min(q0 + kBM, n_rows) - 1) / pack;   // the block's last token
    const int n_tiles = min((total + kBN - 1) / kBN, (clen + last) / kBN + 1);
    // kPart: this workgroup's run of key tiles [kt_lo, kt_hi).
    int                   kt_lo   = 0;
    int                   kt_hi   = n_tiles;
    [[maybe_unused]] bool one_run = false;   // kPart: run 0 holds every key
    if constexpr (kPart) {
        const int tiles_all = (total + kBN - 1) / kBN;
        const int per       = max((tiles_all + num_splits - 1) / num_splits, run_min);
        one_run             = tiles_all <= per;
        kt_lo               = static_cast<int>(blockIdx.y) * per;
        kt_hi               = min(kt_lo + per, n_tiles);
        if (kt_hi <= kt_lo) {   // no key of this run for any row of the block: m, l only
            const int r = q0 + tid;
            if (!one_run && tid < kBM && r < n_rows) {
                const int64_t rows = static_cast<int64_t>(n_new) * hq;
                const int64_t slot = packed_row(r, pack, hq, vhead) * num_splits +
                                     static_cast<int64_t>(blockIdx.y);
                partial[slot]                     = -INFINITY;
                partial[rows * num_splits + slot] = 0.0f;
            }
            return;
        }
    }

    const int  wq0     = q0 + wave * 32;              // first row of this wave
    const int  wlast   = min(wq0 + 31, n_rows - 1);   // may be < wq0 (idle wave)
    const int  w_tiles = (wlast < wq0) ? 0 : (clen + wlast / pack) / kBN + 1;
    // A half tile from a key past this one on crosses the diagonal of the wave's
    // first row or the end of the keys.
    const int  mask_from = min(clen + wq0 / pack - 31, total - 32);
    const int  my_row  = wq0 + qn;                    // row of this lane
    const bool has     = my_row < n_rows;
    // The last key it sees, less 4 h (mask).
    const int my_lim = min(clen + my_row / pack, total - 1) - 4 * h;

    const TileLane<kWaves> ln(tid, wave, lane, hkv);
    const uint8_t* kh  = k + static_cast<int64_t>(kvh) * kHD;
    const uint8_t* vh  = v + static_cast<int64_t>(kvh) * kHD;
    const float*   ksh = ks + kvh;
    const float*   vsh = vs + kvh;
    const uint32_t sk_at = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(sK));   // LDS addresses
    const uint32_t sv_at = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(sV));
    const uint32_t ss_at = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(sSc));
    // Rows of tile i of the run, from its block-table entries.
    using Rows = TileRows<kPaged>;
    auto entries_of = [&](int i) {
        return Rows::entries((kt_lo + i) * kBN, total, block_table, block_shift);
    };
    auto rows_of = [&](int i, const typename Rows::Entries& e) {
        return Rows((kt_lo + i) * kBN, total, e, block_shift);
    };

    auto scales = [&](int i, const Rows& rows) {   // of tile i
        scale_dma<kWaves, kPaged>(ss_at + static_cast<uint32_t>((i & 3) * kScTile * 4), ksh, vsh,
                                  rows, ln, wave, lane, (kt_lo + i + 3) * kBN, total, block_table,
                                  block_shift);
    };

    // Prologue: the first tiles' copies and q all go out before anything
    // waits. The copies of tiles 0 and 1 (and the scales of 2 and 3) first; the
    // block-table entries of the first five tiles in one round trip.
    const typename Rows::Entries e0 = entries_of(0), e1 = entries_of(1), e2 = entries_of(2);
    const typename Rows::Entries e3 = entries_of(3), e4 = entries_of(4);
    const Rows                   r2  = rows_of(2, e2);
    // Rows of the tiles three and four ahead of the loop's.
    Rows rn3 = rows_of(3, e3), rn4 = rows_of(4, e4);
    {
        const Rows r0 = rows_of(0, e0), r1 = rows_of(1, e1);
        scales(0, r0);
        v_tile_dma<kWaves, kPaged>(sv_at, vh, r0, ln, wave);
        k_tile_dma<kWaves, kPaged>(sk_at, kh, r0, ln, wave);
        scales(1, r1);
        k_tile_dma<kWaves, kPaged>(sk_at + kKTile, kh, r1, ln, wave);
        v_tile_dma<kWaves, kPaged>(sv_at + kKTile, vh, r1, ln, wave);
        scales(2, r2);
        scales(3, rn3);
        k_tile_dma<kWaves, kPaged>(sk_at + 2 * kKTile, kh, r2, ln, wave);
    }
    // Q^T (B operand) as hi + lo E4M3 parts. Lane (row my_row, group h) holds,
    // for k-step j, d = 64j + 32h .. +32 (the same d the K operand lanes of
    // group h hold, so the MFMA pairs matching d).
    i32x8 qhi[2], qlo[2];
    int   sc_hi, sc_lo;
    u32x4 qraw[2][4];
    {
        const uint16_t* qr = q + packed_row(has ? my_row : 0, pack, hq, vhead) * kHD;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                qraw[j][c] = *reinterpret_cast<const u32x4*>(qr + 64 * j + 32 * h + 8 * c);
            }
        }
    }
    pin();
    {
        float x[2][32];
        float amax = 0.0f;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                u32x4 w = qraw[j][c];
                if (!has) {
                    w = u32x4{0u, 0u, 0u, 0u};
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    x[j][8 * c + 2 * i]     = __uint_as_float(w[i] << 16);
                    x[j][8 * c + 2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
                    amax = fmaxf(amax, fmaxf(fabsf(x[j][8 * c + 2 * i]),
                                             fabsf(x[j][8 * c + 2 * i + 1])));
                }
            }
        }
        amax = wave_xor_max(amax, 32);
        // 2^a with amax * 2^a in [128, 256); a zero row keeps a = 0.
        // (a is clamped so that 2^a, 2^-a and 2^(-a-4) stay normal: only rows
        // with max |q| below 2^-116 land under 128.)
        const int a = (amax > 0.0f)
                          ? min(max(7 - (static_cast<int>(pow2_bits(amax) >> 23) - 127), -120), 123)
                          : 0;
        const float s2a = __uint_as_float(static_cast<uint32_t>(127 + a) << 23);
        sc_hi = kE8M0One - a;
        sc_lo = kE8M0One - a - 4;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
#pragma unroll
            for (int w = 0; w < 8; ++w) {
                float y[4], r[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    y[i] = x[j][4 * w + i] * s2a;
                }
                const uint32_t hw = pack_e4m3x4(y[0], y[1], y[2], y[3]);
                const f32x2    h0 = __builtin_amdgcn_cvt_pk_f32_fp8(static_cast<int>(hw), false);
                const f32x2    h1 = __builtin_amdgcn_cvt_pk_f32_fp8(static_cast<int>(hw), true);
                r[0] = (y[0] - h0.x) * 16.0f;
                r[1] = (y[1] - h0.y) * 16.0f;
                r[2] = (y[2] - h1.x) * 16.0f;
                r[3] = (y[3] - h1.y) * 16.0f;
                qhi[j][w] = static_cast<int>(hw);
                qlo[j][w] = static_cast<int>(pack_e4m3x4(r[0], r[1], r[2], r[3]));
            }
        }
    }

    f32x16 o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        o[i] = f32x16{};
    }
    float m_ref = 0.0f;   // lazy reference maximum of this lane's row (log2 units)
    float l_run = 0.0f;

    // V staging: this lane's key pair is pair lane / (4 kWaves / 2) of its wave,
    // its d the kD following kD * (lane % (128 / kD)).
    constexpr int   kD     = kWaves == 4 ? 16 : 8;
    constexpr int   kParts = kD / 4;   // staged four d at a time
    const int       vp     = lane / (kHD / kD);
    const int       vd     = kD * (lane % (kHD / kD));
    const VOrder    vorder((vd & 16) != 0);
    uint32_t* const vcol   = sVt + vt_row(vd) + vt_pos(TileLane<kWaves>::pair_key(wave, vp)) / 2;
    uint32_t* const vcol0  = vcol + vorder.at0;
    uint32_t* const vcol1  = vcol + vorder.at1;
    const uint8_t*  vraw   = sV + wave * (kKTile / kWaves) + vp * kHD + vd;
    const float* const sc  = sSc + wave * kScWave;
    const float*    vsc    = sc + 2 * vp;
    constexpr int   kKeys  = 64 / kWaves;
    const int       kk     = lane & (kKeys - 1);
    const float*    ksc    = sc + kKeys + kk;
    float* const    kfw    = sKf + TileLane<kWaves>::pair_key(wave, kk >> 1) + (kk & 1);
    struct VRaw {
        uint32_t a[kParts], b[kParts];
        f32x2    s;
        float    ks;
        u32x2    e;
    };
    // V codes and v_scales of tile i, k_scale of tile i + 1.
    auto read_raw = [&](int i) {
        using Codes      = std::conditional_t<kWaves == 4, u32x4, u32x2>;
        const uint8_t* p = vraw + (i & 1) * kKTile;
        const Codes    a = *reinterpret_cast<const Codes*>(p);
        const Codes    b = *reinterpret_cast<const Codes*>(p + kKeys / 2 * kHD);
        VRaw           r;
#pragma unroll
        for (int c = 0; c < kParts; ++c) {
            r.a[c] = a[c];
            r.b[c] = b[c];
        }
        r.s  = *reinterpret_cast<const f32x2*>(vsc + (i & 3) * kScTile);
        r.ks = ksc[((i + 1) & 3) * kScTile];
        if constexpr (kPaged) {   // entries of tile i + 4, with the scales of i + 1
            r.e = *reinterpret_cast<const u32x2*>(sc + ((i + 1) & 3) * kScTile + 2 * kKeys);
        }
        return r;
    };
    auto stage = [&](const VRaw& r, const VFactor& f, int i, int c) {   // d 4c .. 4c + 3
        if (c < kParts) {
            const int at = (i & 1) * kVtWords + 4 * c * (kVPitch / 2);
            v_stage4(r.a[c], r.b[c], f, vorder, vcol0 + at, vcol1 + at);
        }
    };
    auto stage_kf = [&](float k_scale, int i) { kfw[(i & 3) * kBN] = k_scale * scale_log2; };

    // Tile 0's and 1's copies have landed; behind them are the scales of tiles
    // 2 and 3 and K(2).
    __builtin_amdgcn_s_waitcnt(waitcnt_vm(2 + kCopies));
    pin();
    {
        const VRaw    r = read_raw(0);
        const VFactor f = v_factor(r.s.x, r.s.y);
#pragma unroll
        for (int c = 0; c < kParts; ++c) {
            stage(r, f, 0, c);
        }
        stage_kf(ksc[0], 0);
        stage_kf(r.ks, 1);
    }
    pin();
    lds_barrier();
    // V(2) over V(0), which this wave alone has read.
    v_tile_dma<kWaves, kPaged>(sv_at, vh, r2, ln, wave);
    pin();

    // ---- operand reads and pieces of a tile --------------------------------
    // The K operand of one 32-key half: k-steps j = 0, 1.
    const uint32_t k_at = k_chunk(qn, 2 * h);   // the other chunks: bits 4 and 6 flipped
    auto read_k = [&](uint32_t at_ring, int half, int j, i32x8& ka) {
        const uint8_t* b  = sK + half * 32 * kHD;
        const uint32_t at = (at_ring + k_at) ^ (j ? 64u : 0u);
        const u32x4    lo = *reinterpret_cast<const u32x4*>(b + at);
        const u32x4    hi = *reinterpret_cast<const u32x4*>(b + (at ^ 16u));
        ka = i32x8{static_cast<int>(lo.x), static_cast<int>(lo.y), static_cast<int>(lo.z),
                   static_cast<int>(lo.w), static_cast<int>(hi.x), static_cast<int>(hi.y),
                   static_cast<int>(hi.z), static_cast<int>(hi.w)};
    };
    // MFMA c (0..3) of a half's scores: k-step c / 2, hi then lo part of q.
    auto qk = [&](const i32x8 (&ka)[2], f32x16& s, int c) {
        const f32x16 z = c == 0 ? f32x16{} : s;
        s = (c & 1) ? __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(
                          ka[c >> 1], qlo[c >> 1], z, 0, 0, 0, kE8M0One, 0, sc_lo)
                    : __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(
                          ka[c >> 1], qhi[c >> 1], z, 0, 0, 0, kE8M0One, 0, sc_hi);
        // Keeps the compiler from sinking the MFMA below a later branch.
        asm volatile("" : "+v"(s));
        pin();
    };
    auto read_kf = [&](int i, int half, f32x4 (&f)[4]) {
        const float* b = sKf + (i & 3) * kBN + 32 * half + 4 * h;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            f[g] = *reinterpret_cast<const f32x4*>(b + 8 * g);
        }
    };
    const uint32_t* const vrow = sVt + vt_row(qn) + 4 * h;
    f16x8                 va[8];
    // Operand of MFMA c (0..7) of a half's P V: d block c & 3, k-step c / 4.
    auto read_v = [&](int i, int half, int c) {
        const uint32_t* p = vrow + (i & 1) * kVtWords + (vt_row(32) * (c & 3)) + 8 * (2 * half + (c >> 2));
        va[c] = __builtin_bit_cast(f16x8, *reinterpret_cast<const u32x4*>(p));
    };
    auto scale4 = [&](f32x16& s, const f32x4 (&f)[4], int g) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            s[4 * g + e] = fmaf(s[4 * g + e], f[g][e], -m_ref);
        }
    };
    // Register r of a half is its key 8 (r / 4) + 4 h + r % 4; key0: the half's
    // first key. Masks past the diagonal and past the last key.
    auto mask = [&](f32x16& s, int key0) {
        if (key0 > mask_from) {
            const int lim = my_lim - key0;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                if (8 * (r >> 2) + (r & 3) > lim) {
                    s[r] = -INFINITY;
                }
            }
        }
    };
    struct Sum {
        float a, b;
    };
    // Four of a half's exponentials: p into the P^T operands, the fp32 sums.
    auto exp4 = [&](const f32x16& s, int g, f16x8 (&p)[2], Sum& sum) {
        const float e0 = __builtin_amdgcn_exp2f(s[4 * g]);
        const float e1 = __builtin_amdgcn_exp2f(s[4 * g + 1]);
        const float e2 = __builtin_amdgcn_exp2f(s[4 * g + 2]);
        const float e3 = __builtin_amdgcn_exp2f(s[4 * g + 3]);
        sum.a = g == 0 ? e0 + e1 : sum.a + (e0 + e1);
        sum.b = g == 0 ? e2 + e3 : sum.b + (e2 + e3);
        p[g >> 1][4 * (g & 1) + 0] = static_cast<_Float16>(e0);
        p[g >> 1][4 * (g & 1) + 1] = static_cast<_Float16>(e1);
        p[g >> 1][4 * (g & 1) + 2] = static_cast<_Float16>(e2);
        p[g >> 1][4 * (g & 1) + 3] = static_cast<_Float16>(e3);
    };
    // Lazy reference maximum (exact): m_ref moves to the row maximum of the
    // half only on the run's first half tile or when a row's sum of a half
    // exceeds 2^15 (some score more than 15 above m_ref); otherwise the half
    // needs no max reduction, no cross-lane step and no rescale of l and O.
    // Every p and l use the same m_ref, and p <= 2^15 keeps every p inside the
    // f16 range.
    auto settle = [&](f32x16& s, f16x8 (&p)[2], Sum& sum, bool first) {
        if (__any(first || !(sum.a + sum.b <= 0x1p15f))) {
            float tmax = -INFINITY;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                tmax = fmaxf(tmax, s[r]);
            }
            tmax = wave_xor_max(tmax, 32);
            // The first tile sets the reference; later tiles only raise it. A
            // row that is here because another row of the wave overflowed may
            // sit far below its reference: lowering it would scale O and l by
            // 2^-tmax, which overflows.
            const float delta = first ? ((tmax == -INFINITY) ? 0.0f : tmax) : fmaxf(tmax, 0.0f);
            const float alpha = first ? 1.0f : __builtin_amdgcn_exp2f(-delta);
            s -= delta;
            m_ref += delta;
            l_run *= alpha;
#pragma unroll
            for (int db = 0; db < 4; ++db) {
                o[db] *= alpha;
            }
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                exp4(s, g, p, sum);
            }
        }
        l_run += sum.a + sum.b;
    };
    auto pv = [&](const f16x8 (&p)[2], int c) {   // MFMA c (0..7) of a half's P V
        o[c & 3] = __builtin_amdgcn_mfma_f32_32x32x16_f16(va[c], p[c >> 2], o[c & 3], 0, 0, 0);
        pin();
    };

    // Entering tile i, a wave holds P of its first half, the scores and the
    // k-factors of its second, and the operands of the MFMAs ahead: V^T of the
    // first half, K of the next tile's first half.
    f32x16 sa, sb;
    f16x8  pa[2], pb[2];
    f32x4  kf[4];
    Sum    sum;
    i32x8  ka[2];
    const int n_steps = kt_hi - kt_lo;
    const int mine    = max(0, min(w_tiles - kt_lo, n_steps));
    if (mine > 0) {
        i32x8 kb[2];
        read_k(0, 0, 0, ka[0]);
        read_k(0, 0, 1, ka[1]);
        read_k(0, 1, 0, kb[0]);
        read_k(0, 1, 1, kb[1]);
        read_kf(0, 0, kf);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            qk(ka, sa, c);
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            qk(kb, sb, c);
        }
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            scale4(sa, kf, g);
        }
        mask(sa, kt_lo * kBN);
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            exp4(sa, g, pa, sum);
        }
        settle(sa, pa, sum, true);
    }
    uint32_t ring = 0;   // byte offset of K(i) in its ring
    // The copies of a tile: K(i + 3) over K(i), whose last reads a barrier has
    // closed; V(i + 3) over V(i + 1), once this wave has read it; the scales
    // of tile i + 4.
    auto next_k = [&]() {
        pin();
        k_tile_dma<kWaves, kPaged>(sk_at + ring, kh, rn3, ln, wave);
        pin();
    };
    // (raw: read_raw(i + 1). Paged: the block-table entries come through LDS, two
    // tiles behind the copy that brought them, and are taken in front of the
    // barrier, where the wave waits in any case. As scalar loads in the tile, the
    // second one behind a branch, two round trips stood in every tile: 400 tokens
    // after 4K keys x 32 heads 96 us, now 86, contiguous 76.)
    auto next_v = [&](int i, const VRaw& raw) {
        pin();
        v_tile_dma<kWaves, kPaged>(sv_at + ((i + 1) & 1) * kKTile, vh, rn3, ln, wave);
        scales(i + 4, rn4);
        rn3 = rn4;
        typename Rows::Entries e{};
        if constexpr (kPaged) {
            e.lo = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(raw.e.x)));
            e.hi = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(raw.e.y)));
        }
        rn4 = rows_of(i + 5, e);
        pin();
    };
    // The copies of the tile before must have landed and the staged LDS writes
    // be visible; this tile's copies stay in flight.
    auto tile_barrier = [&]() {
        pin();
        __builtin_amdgcn_s_waitcnt(waitcnt_vm(kOps));
        lds_barrier();
        pin();
    };
    auto ring_next = [](uint32_t r) {
        return r == 2u * kKTile ? 0u : r + static_cast<uint32_t>(kKTile);
    };
    // K(0) is overwritten by the first tile's copy: its operand reads are done.
    pin();
    __builtin_amdgcn_s_waitcnt(waitcnt_vm(kCopies));
    lds_barrier();
    pin();
    // (In the order of the loop's reads, so that its waits count the same.)
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        read_v(0, 0, c);
        pin();
        if (c == 3) {
            read_k(kKTile, 0, 0, ka[0]);
            pin();
        }
        if (c == 5) {
            read_kf(0, 1, kf);
            read_k(kKTile, 0, 1, ka[1]);
            pin();
        }
    }

    // A tile that is not the workgroup's last.
    auto tile = [&](int i) {
        const uint32_t k1 = ring_next(ring);   // K(i + 1)
        const uint32_t k2 = ring_next(k1);     // K(i + 2)
        // P V of the first half and the next tile's first scores, under the
        // softmax of the second half and the staging of V(i + 1); the operands
        // of the part after this one are read as their registers come free.
        pin();
        scale4(sb, kf, 0);
        scale4(sb, kf, 1);
        pin();
        if constexpr (kWaves == 8) {
            __builtin_amdgcn_s_setprio(1);
        }
        pv(pa, 0);
        read_v(i, 1, 0);
        scale4(sb, kf, 2);
        scale4(sb, kf, 3);
        pin();
        pv(pa, 1);
        read_v(i, 1, 1);
        const VRaw raw = read_raw(i + 1);
        mask(sb, (kt_lo + i) * kBN + 32);
        pin();
        qk(ka, sa, 0);
        exp4(sb, 0, pb, sum);
        pin();
        pv(pa, 2);
        read_v(i, 1, 2);
        pin();
        pv(pa, 3);
        read_v(i, 1, 3);
        pin();
        qk(ka, sa, 1);
        read_k(k1, 1, 0, ka[0]);
        exp4(sb, 1, pb, sum);
        pin();
        pv(pa, 4);
        read_v(i, 1, 4);
        const VFactor f = v_factor(raw.s.x, raw.s.y);
        pin();
        pv(pa, 5);
        read_v(i, 1, 5);
        exp4(sb, 2, pb, sum);
        pin();
        // Priority over the first two thirds of the half: held to its end, the SIMD's
        // other wave got its own MFMAs in too late (4096 tokens after 64K / 127K keys,
        // priority to the end of the half -> to here 3910 -> 3828, 7497 -> 7335 us,
        // 16384 tokens 1949 -> 1910, 4096 136.6 -> 133.7; two MFMAs earlier or later
        // gains half of that, none at all costs 1.6 %).
        if constexpr (kWaves == 8) {
            __builtin_amdgcn_s_setprio(0);
        }
        qk(ka, sa, 2);
        exp4(sb, 3, pb, sum);
        pin();
        pv(pa, 6);
        read_v(i, 1, 6);
        pin();
        pv(pa, 7);
        read_v(i, 1, 7);
        stage(raw, f, i + 1, 0);
        pin();
        qk(ka, sa, 3);
        read_k(k1, 1, 1, ka[1]);
        stage(raw, f, i + 1, 1);
        pin();
        settle(sb, pb, sum, false);
        // P V of the second half and the next tile's second scores, under the
        // softmax of the next tile's first half.
        pin();
        pv(pb, 0);
        read_kf(i + 1, 0, kf);
        stage(raw, f, i + 1, 2);
        pin();
        qk(ka, sb, 0);
        stage(raw, f, i + 1, 3);
        stage_kf(raw.ks, i + 2);
        pin();
        pv(pb, 1);
        next_k();
        scale4(sa, kf, 0);
        scale4(sa, kf, 1);
        pin();
        pv(pb, 2);
        scale4(sa, kf, 2);
        scale4(sa, kf, 3);
        pin();
        mask(sa, (kt_lo + i + 1) * kBN);
        pin();
        qk(ka, sb, 1);
        exp4(sa, 0, pa, sum);
        pin();
        pv(pb, 3);
        next_v(i, raw);
        tile_barrier();
        // V^T(i + 1) and K(i + 2) are there.
        qk(ka, sb, 2);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            read_v(i + 1, 0, c);
        }
        read_k(k2, 0, 0, ka[0]);
        exp4(sa, 1, pa, sum);
        pin();
        pv(pb, 4);
        read_v(i + 1, 0, 4);
        pin();
        pv(pb, 5);
        read_v(i + 1, 0, 5);
        read_kf(i + 1, 1, kf);
        exp4(sa, 2, pa, sum);
        pin();
        qk(ka, sb, 3);
        read_k(k2, 0, 1, ka[1]);
        exp4(sa, 3, pa, sum);
        pin();
        pv(pb, 6);
        read_v(i + 1, 0, 6);
        pin();
        pv(pb, 7);
        read_v(i + 1, 0, 7);
        pin();
        settle(sa, pa, sum, false);
        ring = k1;
    };
    // Tiles with keys for this wave that are not the workgroup's last.
    const int n_a = min(mine, n_steps - 1);
    for (int i = 0; i < n_a; ++i) {
        tile(i);
    }
    if (mine == n_steps) {   // the last tile
        const int i = n_steps - 1;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            scale4(sb, kf, g);
        }
        mask(sb, (kt_lo + i) * kBN + 32);
        pin();
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            pv(pa, c);
            read_v(i, 1, c);
            if (c & 1) {
                exp4(sb, c >> 1, pb, sum);
                pin();
            }
        }
        settle(sb, pb, sum, false);
        pin();
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            pv(pb, c);
        }
    } else {   // rows that see no further key: copy and stage for the other waves
        for (int i = n_a; i < n_steps - 1; ++i) {
            next_k();
            const VRaw    raw = read_raw(i + 1);
            const VFactor f   = v_factor(raw.s.x, raw.s.y);
#pragma unroll
            for (int c = 0; c < kParts; ++c) {
                stage(raw, f, i + 1, c);
            }
            stage_kf(raw.ks, i + 2);
            next_v(i, raw);
            tile_barrier();
            ring = ring_next(ring);
        }
    }

    // The copies past the last tile must have landed before the workgroup's LDS
    // is given back.
    __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
    const float l_tot = wave_xor_sum(l_run, 32);
    // (The lane's row afresh, so that it takes no register over the loop.)
    const int lane_e = static_cast<int>(
        __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)));
    const int he    = lane_e >> 5;
    const int row_e = wq0 + (lane_e & 31);
    // kPart with a single live run (short caches): run 0 stores the output
    // itself, as the plain kernel does, and the merge skips the call.
    if (kPart && !one_run) {
        if (row_e >= n_rows) {
            return;
        }
        const int64_t row    = packed_row(row_e, pack, hq, vhead);
        const int64_t rows   = static_cast<int64_t>(n_new) * hq;
        const int64_t slot   = row * num_splits + static_cast<int64_t>(blockIdx.y);
        const bool    any    = !(l_tot == 0.0f);   // (a NaN row is one with keys)
        float*        part_o = partial + 2 * rows * num_splits + slot * kHD;
        if (he == 0) {
            partial[slot]                     = any ? m_ref : -INFINITY;
            partial[rows * num_splits + slot] = l_tot;
        }
#pragma unroll
        for (int db = 0; db < 4; ++db) {
#pragma unroll
            for (int rg = 0; rg < 4; ++rg) {
                *reinterpret_cast<f32x4_a4*>(part_o + 32 * db + 8 * rg + 4 * he) =
                    any ? f32x4{o[db][4 * rg], o[db][4 * rg + 1], o[db][4 * rg + 2],
                                o[db][4 * rg + 3]}
                        : f32x4{0.f, 0.f, 0.f, 0.f};
            }
        }
        return;
    }
    // O / l in bf16 through LDS (every wave is past its last tile and every copy
    // has landed), 64 d at a time, so that the stores are whole 128-byte runs
    // of a row (16-byte pieces of 32 rows each before; per call, 32 heads: 128 /
    // 300 / 4096 tokens 9.4 -> 8.6, 12.7 -> 11.9, 139.5 -> 136.5 us).
    lds_barrier();
    constexpr int kOPitch = 64 + 8;   // bf16 per row
    static_assert(kWaves * 32 * kOPitch * 2 <= sizeof(sVt), "a wave's rows fit V^T's LDS");
    uint16_t* const so    = reinterpret_cast<uint16_t*>(sVt) + wave * 32 * kOPitch;
    const float     inv_l = 1.0f / l_tot;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
#pragma unroll
        for (int db = 0; db < 2; ++db) {
            const f32x16& od = o[2 * half + db];
#pragma unroll
            for (int rg = 0; rg < 4; ++rg) {
                u32x2 w;
                w.x = pack_bf16x2(od[4 * rg + 0] * inv_l, od[4 * rg + 1] * inv_l);
                w.y = pack_bf16x2(od[4 * rg + 2] * inv_l, od[4 * rg + 3] * inv_l);
                *reinterpret_cast<u32x2*>(so + (lane_e & 31) * kOPitch + 32 * db + 8 * rg +
                                          4 * he) = w;
            }
        }
        // (One wave's LDS operations run in order.)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int   r = 8 * j + (lane_e >> 3);
            const u32x4 w = *reinterpret_cast<const u32x4*>(so + r * kOPitch + 8 * (lane_e & 7));
            if (wq0 + r < n_rows) {
                *reinterpret_cast<u32x4*>(out + packed_row(wq0 + r, pack, hq, vhead) * kHD +
                                          64 * half + 8 * (lane_e & 7)) = w;
            }
        }
    }
}

// Merges the key runs' partials: out = sum_s 2^(m_s - M) O_s / sum_s 2^(m_s -
// M) l_s over the live runs (derived as the prefill kernel does). kSub groups
// of 32 lanes per row (16 bytes of each O_s per lane; group i takes runs i, i +
// kSub, ...). Many rows (few runs each) are bound by the partials' bytes, 520
// per row and run, few rows by the loads' round trips; only the live runs are
// read. Per call at 32 q heads / 8 kv heads, 64 / 160 / 250 tokens, with the
// decode's whole-row merge (a workgroup of 128 per row, 32 slots read whatever
// the count) -> with this one: empty cache 10.3 / 15.1 / 18.7 -> 9.0 / 11.1 /
// 12.4 us, 1K keys 17.6 / 26.0 / 30.0 -> 13.6 / 22.9 / 26.0, 8K keys 26.5 /
// 40.5 / 53.8 -> 23.5 / 41.0 / 51.6.
// ways > 1: the run kernel's workgroups of a kv head lie on one XCD (kv heads a
// multiple of 8: way_heads q heads on each) or on the 8 / ways XCDs x with x %
// ways = the kv head (1, 2 or 4 kv heads): a merge workgroup (on XCD blockIdx.x
// % 8) merges rows of its own XCD's heads, whose partials that XCD's L2 holds
// (of 4 kv heads half, of 2 a quarter). Rows in order reach the right XCD only
// where a workgroup's four rows are one kv head's (groups of 4); the others read
// every partial across XCDs, 41-80 tokens slower than the decode route at
// 300-2K keys. Per call, 64 tokens after 700 / 1K / 2K keys, rows in order ->
// by XCD (decode route): 24 heads 15.6 / 16.4 / 18.6 -> 14.3 / 14.1 / 15.6 us
// (14.9 / 16.0 / 18.4), 64 heads 21.1 / 24.1 / 28.8 -> 17.4 / 20.0 / 23.7 (19.5 /
// 20.9 / 25.8), 32 heads 14.1 / 14.1 / 15.8 -> 14.2 / 14.2 / 15.8; 28 heads on 4
// kv heads 15.1 / 15.9 / 18.1 -> 14.3 / 14.5 / 16.1 (14.8 / 16.3 / 18.5), at 41
// tokens 14.3 / 14.8 / 16.9 -> 13.6 / 13.6 / 15.0 (14.2 / 14.2 / 16.3).
constexpr int kMergeThreads = 256;
template <int kSub>
__global__ __launch_bounds__(kMergeThreads) void flash_prefill_merge_kernel(
    uint16_t* __restrict__ out, const float* __restrict__ partial, int num_splits,
    const int* __restrict__ cache_len, int rows, int n_new, int run_min, int ways, int way_heads) {
    constexpr int kRows = kMergeThreads / (32 * kSub);
    static_assert(kSub == 1 || kSub == 2, "a row's lanes lie in one wave");
    const int tiles = (*cache_len + n_new + kBN - 1) / kBN;
    const int per   = max((tiles + num_splits - 1) / num_splits, run_min);
    const int live  = (tiles + per - 1) / per;
    if (live == 1) {   // run 0 stored the output itself
        return;
    }
    const int     hl  = static_cast<int>(threadIdx.x) & 31;
    const int     sub = static_cast<int>(threadIdx.x) / 32 % kSub;
    const int64_t hs  = static_cast<int64_t>(rows) * num_splits;
    // The rows of this workgroup's way (its XCD's, or all): row j of them is head
    // j % way_heads of the way's heads, token j / way_heads.
    const int bid = static_cast<int>(blockIdx.x);
    for (int j = bid / ways * kRows + static_cast<int>(threadIdx.x) / (32 * kSub);
         j < rows / ways; j += static_cast<int>(gridDim.x) / ways * kRows) {
        const int row =
            ways > 1 ? (j / way_heads * ways + bid % ways) * way_heads + j % way_heads : j;
        const int64_t slot0 = static_cast<int64_t>(row) * num_splits;
        const float*  pm    = partial + slot0;
        const float*  pl    = partial + hs + slot0;
        const float*  po    = partial + 2 * hs + slot0 * kHD + 4 * hl;
        float         m[8], ls[8];
        f32x4         os[8];
        auto load8 = [&](int s0) {   // runs s0 + u kSub, clamped to the live ones
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int i = min(s0 + u * kSub, live - 1);
                m[u]        = pm[i];
                ls[u]       = pl[i];
                os[u]       = *reinterpret_cast<const f32x4_a4*>(po + static_cast<int64_t>(i) * kHD);
            }
        };
        float big = pm[min(hl, live - 1)];   // M
        load8(sub);
        for (int i = hl + 32; i < live; i += 32) {
            big = fmaxf(big, pm[i]);
        }
#pragma unroll
        for (int x = 1; x < 32; x <<= 1) {
            big = fmaxf(big, __shfl_xor(big, x, 32));
        }
        float l   = 0.0f;
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        for (int s0 = sub;;) {
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                // A run without keys of the row (m = -inf) may hold no O at all.
                const bool  use = s0 + u * kSub < live && m[u] != -INFINITY;
                const float f   = use ? __builtin_amdgcn_exp2f(m[u] - big) : 0.0f;
                acc += (use ? os[u] : f32x4{0.f, 0.f, 0.f, 0.f}) * f;
                l += (use ? ls[u] : 0.0f) * f;
            }
            s0 += 8 * kSub;
            if (s0 >= live) {
                break;
            }
            load8(s0);
        }
        if constexpr (kSub == 2) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                acc[e] += __shfl_xor(acc[e], 32);
            }
            l += __shfl_xor(l, 32);
        }
        if (sub == 0) {
            const float inv = __builtin_amdgcn_rcpf(l);   // 1 ulp; the output is bf16
            u32x2       w;
            w.x = pack_bf16x2(acc[0] * inv, acc[1] * inv);
            w.y = pack_bf16x2(acc[2] * inv, acc[3] * inv);
            *reinterpret_cast<u32x2*>(out + static_cast<int64_t>(row) * kHD + 4 * hl) = w;
        }
    }
}

template <int kWaves>
void launch_prefill(uint16_t* out, const uint16_t* q, const uint8_t* k, const uint8_t* v,
                    const float* k_scale, const float* v_scale, int n_new, const int* cache_len,
                    int hq, int hkv, int pack, float scale_log2, hipStream_t stream,
                    const int* block_table, int block_shift, int first_wgs) {
    constexpr int kBM   = 32 * kWaves;
    const int     share = hq / hkv / pack;
    const int     n_blk = (n_new * pack + kBM - 1) / kBM;
    const dim3    grid(static_cast<unsigned>(n_blk * hkv * share));
    if (block_table != nullptr) {
        hipLaunchKernelGGL((flash_prefill_kernel<kWaves, true, false>), grid,
                           dim3(kWaves * kWave), 0, stream, out, q, k, v, k_scale, v_scale,
                           n_new, cache_len, pack, share, hkv, scale_log2, block_table,
                           block_shift, first_wgs, nullptr, 1, 1);
    } else {
        hipLaunchKernelGGL((flash_prefill_kernel<kWaves, false, false>), grid,
                           dim3(kWaves * kWave), 0, stream, out, q, k, v, k_scale, v_scale,
                           n_new, cache_len, pack, share, hkv, scale_log2, nullptr, 0, first_wgs,
                           nullptr, 1, 1);
    }
}

// The flash prefill with its keys split over num_splits workgroups per row
// block, then the merge of the n_new * Hq rows.
template <bool kPaged>
hipError_t launch_prefill_part(uint16_t* out, const uint16_t* q, const uint8_t* k,
                               const uint8_t* v, const float* k_scale, const float* v_scale,
                               float* partial, int num_splits, int n_new, const int* cache_len,
                               int hq, int hkv, float scale_log2, hipStream_t stream,
                               const int* block_table, int block_shift) {
    // A run's minimum of tiles, so that short caches use few runs: what another
    // run saves (1.02 us a tile) against the partials it writes for its rows
    // and the merge reads, by the tokens up to 64 and from 81 on, by the rows
    // between (where the runs took the decode route's place: that is the figure
    // in brackets). After 300 / 1K / 2K keys, minimum 2 / 4 / 8, us: 64 tokens x 32
    // heads 13.1 / 14.7 / 14.3, 13.7 / 15.1 / 19.0, 15.2 / 16.0 / 19.5; 80 x 24 heads
    // 13.2 / 15.0 / 14.3 [14.1], 14.0 / 15.5 / 19.4 [17.5], 15.5 / 16.4 / 19.8 [21.6];
    // 80 x 32 heads (2560 rows) 13.9 / 15.3 / 14.3 [14.7], 14.7 / 15.9 / 19.6 [18.2],
    // 17.6 / 16.8 / 20.3 [22.3]; 80 x 64 heads 14.4 / 15.7 / 14.3 [19.3], 20.7 / 17.0 /
    // 20.3 [25.6], 23.9 / 24.9 / 21.2 [35.4]; 128 x 32 heads 15.5 / 16.9 / 15.6, 20.4 /
    // 17.8 / 21.2, 23.0 / 21.8 / 22.2; 200 x 32 heads 16.1 / 17.4 / 17.1, 21.8 / 20.3 /
    // 21.4, 26.3 / 26.0 / 22.6.
    const bool short_runs = n_new <= 64 || (n_new <= 80 && n_new * hq <= 2560);
    const int  run_min    = short_runs ? 2 : n_new <= 128 ? 4 : 8;
    constexpr int kBM     = 32 * 4;
    const int     group = hq / hkv;
    const int     n_blk = (n_new * group + kBM - 1) / kBM;
    const dim3    grid(static_cast<unsigned>(n_blk * hkv), static_cast<unsigned>(num_splits));
    hipLaunchKernelGGL((flash_prefill_kernel<4, kPaged, true>), grid,
                       dim3(4 * kWave), 0, stream, out, q, k, v, k_scale, v_scale, n_new,
                       cache_len, group, 1, hkv, scale_log2, block_table, block_shift, INT_MAX, partial,
                       num_splits, run_min);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        return e;
    }
    const int rows = n_new * hq;
    // At most eight workgroups per compute unit (256), 32 waves: all resident. A
    // whole wave per row up to 4096 rows; the line at 8192 instead, 160 / 200
    // tokens x 32 heads: empty cache 11.0 / 11.3 -> 11.3 / 11.6 us, 8K keys 41.4 /
    // 47.2 -> 40.6 / 47.9, 32K 100.4 / 123.8 -> 101.6 / 126.3.
    const bool wide = rows <= 4096;
    const int wgs = std::min((rows * (wide ? 64 : 32) + kMergeThreads - 1) / kMergeThreads, 2048);
    const int ways = hkv % 8 == 0 ? 8 : 8 % hkv == 0 ? hkv : 1;
    // (A multiple of 8 workgroups: as many on each XCD.)
    hipLaunchKernelGGL(wide ? flash_prefill_merge_kernel<2> : flash_prefill_merge_kernel<1>,
                       dim3(static_cast<unsigned>((wgs + 7) & ~7)), dim3(kMergeThreads), 0, stream,
                       out, partial, num_splits, cache_len, rows, n_new, run_min, ways, hq / ways);
    return hipGetLastError();
}

}  // namespace

hipError_t flash_prefill_keysplit_launch(uint16_t* out, const uint16_t* q, const uint8_t* k,
                                         const uint8_t* v, const float* k_scale,
                                         const float* v_scale, float* partial, int num_splits,
                                         int n_new, const int* cache_len, int num_q_heads,
                                         int num_kv_heads, int head_dim, float scale,
                                         hipStream_t stream, const int* block_table,
                                         int block_shift) {
    if (head_dim != kHD) {
        return hipErrorInvalidValue;
    }
    const float sl = scale * kLog2e;
    return block_table != nullptr
               ? launch_prefill_part<true>(out, q, k, v, k_scale, v_scale, partial, num_splits,
                                           n_new, cache_len, num_q_heads, num_kv_heads, sl,
                                           stream, block_table, block_shift)
               : launch_prefill_part<false>(out, q, k, v, k_scale, v_scale, partial, num_splits,
                                            n_new, cache_len, num_q_heads, num_kv_heads, sl,
                                            stream, nullptr, 0);
}

hipError_t flash_prefill_launch(uint16_t* out, const uint16_t* q,
                                const uint8_t* k, const uint8_t* v,
                                const float* k_scale, const float* v_scale,
                                int n_new, const int* cache_len,
                                int num_q_heads, int num_kv_heads,
                                int head_dim, float scale, hipStream_t stream,
                                const int* block_table, int block_shift) {
    if (head_dim != kHD) {
        return hipErrorInvalidValue;
    }
    int        cus = 0;
    hipError_t ce  = device_cu_count(&cus);
    if (ce != hipSuccess) {
        return ce;
    }
    const float sl    = scale * kLog2e;
    const int   group = num_q_heads / num_kv_heads;
    // The q heads of a kv head share blocks (packed rows) except in calls of up
    // to 64 tokens, whose few blocks finish sooner one head each, spread over
    // more compute units (17 x 32 heads 7.0 -> 6.4 us, 64 x 24 heads 8.2 -> 7.7).
    const int pack   = n_new <= 64 ? 1 : group;
    const int heads  = num_q_heads / pack;
    const int rows   = n_new * pack;
    const int wgs128 = (rows + 127) / 128 * heads;
    // 8-wave workgroups (256 rows, one per compute unit, V staged once for all)
    // when the grid takes 1.6 rounds of them or more; below that 4-wave
    // workgroups (128 rows, two per compute unit), whose finer blocks balance
    // the causal work better (8 / 4 waves, us: 24 heads 3600 tokens, 1.3
    // rounds, 98.5 / 89.7; 32 heads 3000, 1.5 rounds, 85.5 / 85.5; 3600, 1.8
    // rounds, 111.6 / 121.9; 4096, 2 rounds, 137 / 151).
    if (5 * ((rows + 255) / 256) * heads >= 8 * cus) {
        launch_prefill<8>(out, q, k, v, k_scale, v_scale, n_new, cache_len, num_q_heads,
                          num_kv_heads, pack, sl, stream, block_table, block_shift, INT_MAX);
    } else {
        // A grid that is resident in one round: one workgroup per compute unit,
        // heaviest first, then the lightest blocks in ascending order, so that
        // the workgroups that share a compute unit are a heavy and a light one.
        const int per = cus / heads * heads;
        launch_prefill<4>(out, q, k, v, k_scale, v_scale, n_new, cache_len, num_q_heads,
                          num_kv_heads, pack, sl, stream, block_table, block_shift,
                          per > 0 && wgs128 <= 2 * cus ? per : INT_MAX);
    }
    return hipGetLastError();
}

}  // namespace rth
