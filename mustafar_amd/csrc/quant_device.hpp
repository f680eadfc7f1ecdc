// Device-side building blocks of the quantised consumers (quant_spmv.hip, fused_quant.hip): staging sizes,
// dequantisation of a staged run of tiles into an fp16 tile image in LDS, expansion of that image.
#pragma once
#include "rank_whole.hpp"
#include "spmv_device.hpp"

#ifndef MSTF_IMG_STRIDE
#define MSTF_IMG_STRIDE 144
#endif

namespace mstf {

#pragma clang fp contract(off)

template <int BIT>
struct QFmt {
    static constexpr int kCap = 32 / BIT;                       // codes per packed word
    static constexpr int kCapShift = BIT == 2 ? 4 : (BIT == 4 ? 3 : 2);
    static constexpr int kSlots = 64 / kCap;                    // words of a full tile = lanes per tile in a pass
    static constexpr int kTilesPerPass = 64 / kSlots;
    static constexpr int kPasses = kSubTiles / kTilesPerPass;
    static constexpr int kWordsMax = kSubTiles * kSlots;        // words of a stage, every tile full
    static constexpr int kWordBuf = kWordsMax * 4 + 64;         // + room for the lanes past a tile's last word
};
// fp16 image of a stage: 64 two-byte slots per tile, the tiles kImgStride bytes apart.  128 would do; with 144 the
// sixteen-byte writes of the lanes that dequantise different tiles at the same time (tiles 128 bytes apart start in
// one of two banks) and the gathers spread over all LDS banks.
constexpr int kImgStride = MSTF_IMG_STRIDE;
constexpr int kImgBytes = kSubTiles * kImgStride;
// Staged metadata of a stage.  One (scale, zero) pair per tile: 32 word offsets, 32 scales, 32 zero-points (256 bytes,
// one LDS-direct load).  Two pairs per tile (G32: pair g for the elements 32g .. 32g+31): 32 word offsets, 32 x 2
// scales, 32 x 2 zero-points and the upper halves of the 32 bitmaps (their popcount is the number of codes that
// belong to the first pair), 128 bytes each, two LDS-direct loads.
template <bool G32>
constexpr int meta_bytes()
{
    return G32 ? 512 : 256;
}
template <int BIT, bool G32 = false>
constexpr int q_lds_bytes()
{
    return kImgBytes + 2 * QFmt<BIT>::kWordBuf + 2 * meta_bytes<G32>();
}

__device__ __forceinline__ float half_bits_to_float(uint32_t bits) { return (float)as_h((uint16_t)bits); }

// The literal arithmetic of the two dequantisation modes for one code.
__device__ __forceinline__ _Float16 dequant_exact(uint32_t q, uint32_t scale_bits, uint32_t zero_bits, int mode)
{
    if (mode == 1) {
        const _Float16 d = (_Float16)(int)q - as_h((uint16_t)zero_bits);  // fp16 arithmetic, rounded after each step
        return d * as_h((uint16_t)scale_bits);
    }
    return (_Float16)(((float)q - half_bits_to_float(zero_bits)) * half_bits_to_float(scale_bits));
}

// fp16x2 ( (q_lo - zero) * scale, (q_hi - zero) * scale ) from two codes held in bytes 0 and 2 of `codes`.
__device__ __forceinline__ uint32_t dequant_pair(uint32_t codes, h2_t neg_bias, h2_t scale2)
{
    const h2_t x = as_h2(codes | 0x64006400u);  // (1024 + q_lo, 1024 + q_hi)
    return as_u32((x + neg_bias) * scale2);
}

// The values of one packed word into the tile image at dst.  sc / zp: the (scale, zero) pair of its tile (low half) or, G32,
// both pairs (first in the low half), kb: the codes of the word that belong to the first pair.
template <int BIT, bool G32>
__device__ __forceinline__ void dequant_word(uint32_t w, uint32_t sc, uint32_t zp, int kb, uint32_t dst, int mode)
{
    using F = QFmt<BIT>;
    typedef short s2_t __attribute__((ext_vector_type(2)));
    const bool small_zero = G32 ? ((zp & 0x7fffu) <= 0x6400u && ((zp >> 16) & 0x7fffu) <= 0x6400u)
                                : ((zp & 0x7fffu) <= 0x6400u);
    if (small_zero) {
        const _Float16 nb = (_Float16)(-1024.0f) - as_h((uint16_t)zp);  // exact: |zero| <= 1024
        const _Float16 sh = as_h((uint16_t)sc);
        const h2_t nb_a = {nb, nb};
        const h2_t sc_a = {sh, sh};
        uint32_t nb_b = 0u, sc_b = 0u, kb2 = 0u;
        if (G32) {
            const _Float16 nb1 = (_Float16)(-1024.0f) - as_h((uint16_t)(zp >> 16));
            const _Float16 sh1 = as_h((uint16_t)(sc >> 16));
            nb_b = as_u32(h2_t{nb1, nb1});
            sc_b = as_u32(h2_t{sh1, sh1});
            kb2 = (uint32_t)kb | ((uint32_t)kb << 16);
        }
        // dequantises codes 2n, 2n+1 of the word (held in bytes 0 and 2 of `codes`); G32: each of the two takes the
        // first pair if its index is below kb - a packed 16-bit subtract and arithmetic shift give the halfword
        // masks, two bit-field inserts the parameters
        auto deq = [&](uint32_t codes, int n) -> uint32_t {
            if (!G32) return dequant_pair(codes, nb_a, sc_a);
            const s2_t d = __builtin_bit_cast(s2_t, (uint32_t)(2 * n) | ((uint32_t)(2 * n + 1) << 16)) -
                           __builtin_bit_cast(s2_t, kb2);                       // < 0 <=> first pair
            const uint32_t m = __builtin_bit_cast(uint32_t, (s2_t)(d >> 15));
            const uint32_t nbx = (m & as_u32(nb_a)) | (~m & nb_b);
            const uint32_t scx = (m & as_u32(sc_a)) | (~m & sc_b);
            return dequant_pair(codes, as_h2(nbx), as_h2(scx));
        };
        if constexpr (BIT == 2 && !G32) {
            // Four values are all that a tile's codes stand for: their low and their high bytes make two registers, out
            // of which one byte permute per pair of codes looks both values up - its selector holds a code, and the
            // code + 4 for the high byte - instead of a subtraction and a product for each pair.  Fused attention,
            // 256 heads x 4096 tokens: 51.3 -> 50.7 us.
            const uint32_t v01 = dequant_pair(0x00010000u, nb_a, sc_a), v23 = dequant_pair(0x00030002u, nb_a, sc_a);
            const uint32_t low = __builtin_amdgcn_perm(v23, v01, 0x06040200u);
            const uint32_t high = __builtin_amdgcn_perm(v23, v01, 0x07050301u);
            uint32_t code = 0x03030303u;
            asm("" : "+v"(code));  // (in a register: and-or takes one constant only)
            const uint32_t w1 = w >> 2, w2 = w >> 4, w3 = w >> 6;
            auto look = [&](uint32_t odd, uint32_t even, uint32_t byte) {
                const uint32_t c = __builtin_amdgcn_perm(odd, even, 0x04040000u + byte * 0x01010101u);
                return (uint32_t)__builtin_amdgcn_perm(high, low, (c & code) | 0x04000400u);
            };
            u32x4_t lo, hi;
            lo[0] = look(w1, w, 0), lo[1] = look(w3, w2, 0);  // code k sits in byte k / 4, at bit 2 (k % 4) of it
            lo[2] = look(w1, w, 1), lo[3] = look(w3, w2, 1);
            hi[0] = look(w1, w, 2), hi[1] = look(w3, w2, 2);
            hi[2] = look(w1, w, 3), hi[3] = look(w3, w2, 3);
            *(MSTF_LDS u32x4_t*)(uintptr_t)dst = lo;
            *(MSTF_LDS u32x4_t*)(uintptr_t)(dst + 16u) = hi;
        } else if (BIT == 2) {
            // E[k % 4] holds code k in byte k / 4
            const uint32_t e0 = w & 0x03030303u, e1 = (w >> 2) & 0x03030303u;
            const uint32_t e2 = (w >> 4) & 0x03030303u, e3 = (w >> 6) & 0x03030303u;
            u32x4_t lo, hi;
            lo[0] = deq(__builtin_amdgcn_perm(e1, e0, 0x0c040c00u), 0);  // codes 0, 1
            lo[1] = deq(__builtin_amdgcn_perm(e3, e2, 0x0c040c00u), 1);  // codes 2, 3
            lo[2] = deq(__builtin_amdgcn_perm(e1, e0, 0x0c050c01u), 2);
            lo[3] = deq(__builtin_amdgcn_perm(e3, e2, 0x0c050c01u), 3);
            hi[0] = deq(__builtin_amdgcn_perm(e1, e0, 0x0c060c02u), 4);
            hi[1] = deq(__builtin_amdgcn_perm(e3, e2, 0x0c060c02u), 5);
            hi[2] = deq(__builtin_amdgcn_perm(e1, e0, 0x0c070c03u), 6);
            hi[3] = deq(__builtin_amdgcn_perm(e3, e2, 0x0c070c03u), 7);
            *(MSTF_LDS u32x4_t*)(uintptr_t)dst = lo;
            *(MSTF_LDS u32x4_t*)(uintptr_t)(dst + 16u) = hi;
        } else if (BIT == 4) {
            // e0 holds codes 0, 2, 4, 6 in its bytes, e1 codes 1, 3, 5, 7
            const uint32_t e0 = w & 0x0f0f0f0fu, e1 = (w >> 4) & 0x0f0f0f0fu;
            u32x4_t v;
            v[0] = deq(__builtin_amdgcn_perm(e1, e0, 0x0c040c00u), 0);
            v[1] = deq(__builtin_amdgcn_perm(e1, e0, 0x0c050c01u), 1);
            v[2] = deq(__builtin_amdgcn_perm(e1, e0, 0x0c060c02u), 2);
            v[3] = deq(__builtin_amdgcn_perm(e1, e0, 0x0c070c03u), 3);
            *(MSTF_LDS u32x4_t*)(uintptr_t)dst = v;
        } else {
            u32x2_t v;
            v[0] = deq(__builtin_amdgcn_perm(w, w, 0x0c010c00u), 0);
            v[1] = deq(__builtin_amdgcn_perm(w, w, 0x0c030c02u), 1);
            *(MSTF_LDS u32x2_t*)(uintptr_t)dst = v;
        }
    } else {
    #pragma unroll 1
        for (int k = 0; k < F::kCap; k++) {
            const uint32_t q = (w >> (k * BIT)) & ((1u << BIT) - 1u);
            const uint32_t sel = (G32 && k >= kb) ? 16u : 0u;
            *(MSTF_LDS _Float16*)(uintptr_t)(dst + 2u * (uint32_t)k) =
                dequant_exact(q, (sc >> sel) & 0xffffu, (zp >> sel) & 0xffffu, mode);
        }
    }
}
// One code by the arithmetic of dequant_word.
__device__ __forceinline__ _Float16 dequant_code(uint32_t q, uint32_t scale_bits, uint32_t zero_bits, int mode)
{
    if ((zero_bits & 0x7fffu) <= 0x6400u) {
        const _Float16 nb = (_Float16)(-1024.0f) - as_h((uint16_t)zero_bits);  // exact: |zero| <= 1024
        return (as_h((uint16_t)(0x6400u | q)) + nb) * as_h((uint16_t)scale_bits);
    }
    return dequant_exact(q, scale_bits, zero_bits, mode);
}

// The lane's places in the first buffers of staged metadata and words of a wavefront, and in its image.
template <int BIT>
struct StageLane {
    uint32_t meta4, meta2;  // LDS address of the metadata of the lane's tile (of the first pass): 4 and 2 bytes a tile
    uint32_t word, dst;     // of the lane's word of a tile that starts the buffer; of its values in the image
    // (opaque: every access is one of these registers and an immediate offset)
    __device__ __forceinline__ StageLane(uint32_t meta0, uint32_t words0, uint32_t img, int lane)
    {
        constexpr int kLanes = QFmt<BIT>::kSlots / 2;
        const uint32_t tl = (uint32_t)(lane / kLanes), slot = (uint32_t)(lane % kLanes);
        meta4 = meta0 + tl * 4u;
        meta2 = meta0 + tl * 2u;
        word = words0 + slot * 4u;
        dst = img + tl * (uint32_t)kImgStride + slot * (uint32_t)(QFmt<BIT>::kCap * 2);
        asm volatile("" : "+v"(meta4), "+v"(meta2), "+v"(word), "+v"(dst));
    }
};
// A stage that lies `meta` and `words` bytes behind the first buffers at meta0 and words0; its words are those from start_word to
// end_word.
struct StageAt {
    uint32_t meta0, words0, meta, words, start_word, end_word;
};
// Tiles of the stage with more than 32 survivors, whose words are more than the first halves (dequant_halves): bit of the lane
// that speaks for the tile.  That follows from the word offsets: a lane compares its tile's with the next one's; with 2 bits that is
// the tile that it dequantises.
template <int BIT>
struct LongTiles {
    static constexpr int kHalfSlots = QFmt<BIT>::kSlots / 2;
    static constexpr bool kOwn = kHalfSlots * kSubTiles == 64;
    static constexpr int kLanes = kOwn ? kHalfSlots : 1;  // lanes that speak for a tile
    uint32_t off;   // word offset of the lane's tile
    uint64_t mask;
    __device__ __forceinline__ LongTiles(const StageLane<BIT>& at, const StageAt& s, int lane)
    {
        static_assert(kHalfSlots * QFmt<BIT>::kCap == 32, "the first half holds 32 codes of every tile");
        const uint32_t tl = kOwn ? (uint32_t)(lane / kHalfSlots) : (uint32_t)lane % kSubTiles;
        const uint32_t a = kOwn ? at.meta4 + s.meta : s.meta0 + s.meta + tl * 4u;
        off = lds_load_u32(a);
        const uint32_t next = lds_load_u32(a + 4u);
        mask = __ballot((tl == kSubTiles - 1 ? s.end_word : next) - off > (uint32_t)kHalfSlots) &
               (kOwn ? 0x5555555555555555ull : 0xFFFFFFFFull);
    }
    __device__ __forceinline__ int count() const
    {
        int n = __builtin_popcountll(mask);
        asm("" : "+s"(n));  // (compared as 32 bits: the compiler makes a 64-bit vector comparison of it)
        return n;
    }
    // bit t: tile t is a long one
    __device__ __forceinline__ uint32_t tiles() const
    {
        if (!kOwn) return (uint32_t)mask;
        uint64_t x = mask;
        x = (x | x >> 1) & 0x3333333333333333ull;
        x = (x | x >> 2) & 0x0F0F0F0F0F0F0F0Full;
        x = (x | x >> 4) & 0x00FF00FF00FF00FFull;
        x = (x | x >> 8) & 0x0000FFFF0000FFFFull;
        return (uint32_t)(x | x >> 16);
    }
};
// Every lane owns one packed word and writes that word's values to the tile image, `shift` bytes behind its place (StageLane).  A
// tile's words are visited in two halves: first words 0 .. kSlots/2 - 1 of every tile (kSlots/2 lanes per tile: all there is for a
// tile with at most 32 survivors), then, with `high`, words kSlots/2 .. kSlots - 1.  Lanes past a tile's last word decode whatever
// follows in the staged buffer into image slots no rank ever points to.
// Returns the (scale, zero) pairs of the lane's tile of the last pass.
template <int BIT, bool G32>
__device__ __forceinline__ uint2 dequant_halves(const StageLane<BIT>& at, const StageAt& s, const LongTiles<BIT>& lt, uint32_t shift,
                                                bool high, int lane, int mode)
{
    using F = QFmt<BIT>;
    constexpr int kHalfSlots = F::kSlots / 2;
    constexpr int kTilesPerHalfPass = 64 / kHalfSlots;
    constexpr int kHalfPasses = kSubTiles / kTilesPerHalfPass;
    static_assert(kSubTiles == 32, "lanes 0..31 test the 32 tiles of the stage");
    uint2 pair = make_uint2(0u, 0u);
#pragma unroll
    for (int hp = 0; hp < 2 * kHalfPasses; hp++) {
        const int half = hp / kHalfPasses, p = hp % kHalfPasses;
        if (half == 1 && !high) break;
        const uint32_t m4 = at.meta4 + s.meta + (uint32_t)(p * kTilesPerHalfPass * 4);
        const uint32_t m2 = at.meta2 + s.meta + (uint32_t)(p * kTilesPerHalfPass * 2);
        const uint32_t slot = (uint32_t)(half * kHalfSlots + lane % kHalfSlots);
        const uint32_t off = lt.kOwn ? lt.off : lds_load_u32(m4);
        const uint32_t sc = G32 ? lds_load_u32(m4 + 128u) : lds_load_u16(m2 + 128u);
        const uint32_t zp = G32 ? lds_load_u32(m4 + 256u) : lds_load_u16(m2 + 192u);
        if (half == 0) pair = make_uint2(sc, zp);
        // G32: the codes of this word that belong to the first pair, 0 .. kCap (codes are in rank order over the whole
        // tile; the first popcount(upper bitmap half) of them sit in elements 0 .. 31)
        int kb = F::kCap;
        if (G32) {
            const int c0 = __builtin_popcount(lds_load_u32(m4 + 384u));
            kb = c0 - (int)slot * F::kCap;
            kb = kb < 0 ? 0 : (kb > F::kCap ? F::kCap : kb);
        }
        const uint32_t w = lds_load_u32(at.word + s.words + (uint32_t)(half * kHalfSlots * 4) + (off - s.start_word) * 4u);
        dequant_word<BIT, G32>(w, sc, zp, kb,
                               at.dst + shift + (uint32_t)(p * kTilesPerHalfPass * kImgStride + half * kHalfSlots * F::kCap * 2), mode);
    }
    return pair;
}
// The value of rank r (of the lane) of long tile `bit` of the mask.  pair: dequant_halves.
template <int BIT, bool G32>
__device__ __forceinline__ _Float16 dequant_long(const StageAt& s, const LongTiles<BIT>& lt, uint2 pair, uint32_t bit, uint32_t r,
                                                 int mode)
{
    using F = QFmt<BIT>;
    const uint32_t tl = bit / LongTiles<BIT>::kLanes, m = s.meta0 + s.meta;
    uint32_t off, sc, zp;
    if constexpr (LongTiles<BIT>::kOwn) {  // (out of a lane's registers instead of by two reads in a row)
        off = (uint32_t)__builtin_amdgcn_readlane((int)lt.off, (int)bit);
        sc = (uint32_t)__builtin_amdgcn_readlane((int)pair.x, (int)bit);
        zp = (uint32_t)__builtin_amdgcn_readlane((int)pair.y, (int)bit);
    } else {
        off = lds_load_u32(m + tl * 4u);
        sc = G32 ? lds_load_u32(m + 128u + tl * 4u) : lds_load_u16(m + 128u + tl * 2u);
        zp = G32 ? lds_load_u32(m + 256u + tl * 4u) : lds_load_u16(m + 192u + tl * 2u);
    }
    const uint32_t word0 = s.words0 + s.words + (off - s.start_word) * 4u;
    const uint32_t w = lds_load_u32(word0 + (r >> F::kCapShift) * 4u);
    const uint32_t q = __builtin_amdgcn_ubfe(w, r * (uint32_t)BIT, (uint32_t)BIT);  // (the place counts modulo 32)
    uint32_t sel = 0u;  // G32: the first popcount(upper bitmap half) codes belong to the first pair
    if (G32) sel = r >= (uint32_t)__builtin_popcount(lds_load_u32(m + 384u + tl * 4u)) ? 16u : 0u;
    return dequant_code(q, G32 ? (sc >> sel) & 0xffffu : sc, G32 ? (zp >> sel) & 0xffffu : zp, mode);
}
// Up to this many long tiles of a stage are finished one by one (a key stage typically holds one channel of outliers, which
// keeps all 64 tokens); with more of them the stage takes the second halves.  (With four at 55 % pruned, where stages have three or
// four: 2 bits 8 heads x 1024 tokens 17.5 us, with two 16.6; at 70 % no difference.)
constexpr int kDirectMax = 2;

// One stage into the image, all of every tile: the long tiles, lane = rank, where they are few.
template <int BIT, bool G32>
__device__ __forceinline__ void dequant_stage(const StageLane<BIT>& at, const StageAt& s, uint32_t img, int lane, int mode)
{
    const LongTiles<BIT> lt(at, s, lane);
    const bool high = lt.count() > kDirectMax;
    const uint2 pair = dequant_halves<BIT, G32>(at, s, lt, 0u, high, lane, mode);
    if (high) return;
    // (the slots of the first half are written again with the same values; ranks beyond the tile's count land in slots no
    // gather points to)
    for (uint64_t left = lt.mask; left != 0ull; left &= left - 1ull) {
        const uint32_t bit = (uint32_t)__builtin_ctzll(left), tl = bit / LongTiles<BIT>::kLanes;
        uint32_t r = (uint32_t)lane;
        asm volatile("" : "+v"(r));  // (what follows from it is made here and holds no registers elsewhere)
        const _Float16 val = dequant_long<BIT, G32>(s, lt, pair, bit, r, mode);
        *(MSTF_LDS _Float16*)(uintptr_t)(img + tl * (uint32_t)kImgStride + r * 2u) = val;
    }
}

// LDS-direct loads of a stage's packed words without control flow (see sub_issue_flat in spmv_device.hpp): piece i
// of lane l is word 64 * i + l of src, issued for the lanes with 64 * i + l < nw by setting exec by hand; the
// wavefront must have all 64 lanes active.  dst_lds: LDS byte address of the word buffer; lane4 = lane * 4.
template <int PIECES>
__device__ __forceinline__ void words_issue_flat(const uint32_t* src, uint32_t nw, uint32_t dst_lds, uint32_t lane,
                                                 uint32_t lane4)
{
    static_assert(PIECES == 2 || PIECES == 4 || PIECES == 8, "pieces of 64 words");
    uint32_t t, m0_kept;
    uint64_t sv;  // exec as found, handed back
#define MSTF_WPIECE(I)                                                     \
    "s_sub_i32 %[t], %[n], " #I " * 64\n\t"                                \
    "v_cmp_gt_i32 vcc, %[t], %[l]\n\t"                                     \
    "s_mov_b64 exec, vcc\n\t"                                              \
    "global_load_lds_dword %[l4], %[src] offset:" #I " * 256\n\t"
#define MSTF_WHEAD "s_mov_b32 %[keep], m0\n\ts_mov_b64 %[sv], exec\n\ts_mov_b32 m0, %[dst]\n\t"
#define MSTF_WTAIL "s_mov_b64 exec, %[sv]\n\ts_mov_b32 m0, %[keep]"
#define MSTF_WOPS                                                                                      \
    : [t] "=&s"(t), [keep] "=&s"(m0_kept), [sv] "=&s"(sv)                                              \
    : [dst] "s"(dst_lds), [n] "s"(nw), [l] "v"(lane), [l4] "v"(lane4), [src] "s"(src)                  \
    : "vcc", "scc", "memory"
    if constexpr (PIECES == 2)
        asm volatile(MSTF_WHEAD MSTF_WPIECE(0) MSTF_WPIECE(1) MSTF_WTAIL MSTF_WOPS);
    else if constexpr (PIECES == 4)
        asm volatile(MSTF_WHEAD MSTF_WPIECE(0) MSTF_WPIECE(1) MSTF_WPIECE(2) MSTF_WPIECE(3) MSTF_WTAIL MSTF_WOPS);
    else
        asm volatile(MSTF_WHEAD MSTF_WPIECE(0) MSTF_WPIECE(1) MSTF_WPIECE(2) MSTF_WPIECE(3) MSTF_WPIECE(4)
                         MSTF_WPIECE(5) MSTF_WPIECE(6) MSTF_WPIECE(7) MSTF_WTAIL MSTF_WOPS);
#undef MSTF_WPIECE
#undef MSTF_WHEAD
#undef MSTF_WTAIL
#undef MSTF_WOPS
}

// Where a lane fetches its 4 bytes of a stage's metadata from (lanes 0..31 the word offsets of the 32 tiles, 32..47
// the scales, 48..63 the zero-points, two per lane): the address for tile 0 and the shift that turns a tile index
// into the lane's byte offset, formed once, so that a stage needs one shift and one 64-bit add.
struct MetaLane {
    const char* p0;
    uint32_t shift;
    __device__ __forceinline__ const void* at(uint32_t t) const { return p0 + ((size_t)t << shift); }
    // the stage behind the one p0 is at
    __device__ __forceinline__ void advance() { p0 += (uint32_t)kSubTiles << shift; }
};
__device__ __forceinline__ MetaLane meta_lane(const uint32_t* off_dma, const uint16_t* scales, const uint16_t* zeros, int lane)
{
    MetaLane m;
    m.p0 = lane < 32 ? reinterpret_cast<const char*>(off_dma + lane)
                     : lane < 48 ? reinterpret_cast<const char*>(reinterpret_cast<const uint32_t*>(scales) + (lane - 32))
                                 : reinterpret_cast<const char*>(reinterpret_cast<const uint32_t*>(zeros) + (lane - 48));
    m.shift = lane < 32 ? 2u : 1u;
    return m;
}
// Two pairs per tile: two loads.  First: lanes 0..31 the word offsets, 32..63 the scales (4 bytes per tile).  Second:
// lanes 0..31 the zero-points (4 bytes per tile), 32..63 the upper halves of the bitmaps (elements 0 .. 31 of a tile
// are bits 63 .. 32, i.e. the second 4 bytes of the little-endian 8).
struct MetaLanes {
    MetaLane a, b;
};
__device__ __forceinline__ MetaLanes meta_lanes_g32(const uint32_t* off_dma, const uint16_t* scales, const uint16_t* zeros,
                                                    const uint64_t* bmp, int lane)
{
    MetaLanes m;
    const int l = lane & 31;
    m.a.p0 = lane < 32 ? reinterpret_cast<const char*>(off_dma + l)
                       : reinterpret_cast<const char*>(reinterpret_cast<const uint32_t*>(scales) + l);
    m.a.shift = 2u;
    m.b.p0 = lane < 32 ? reinterpret_cast<const char*>(reinterpret_cast<const uint32_t*>(zeros) + l)
                       : reinterpret_cast<const char*>(bmp + l) + 4;
    m.b.shift = lane < 32 ? 2u : 3u;
    return m;
}
// Issues the metadata of the stage the pointers are at and moves them on to the next one (consecutive stages).
template <bool G32>
__device__ __forceinline__ void meta_issue_next(MetaLanes& m, char* metabuf)
{
    dma4(m.a.p0, metabuf);
    m.a.advance();
    if (G32) {
        dma4(m.b.p0, metabuf + 256);
        m.b.advance();
    }
}
// Issues the metadata of the stage starting at tile t (relative to the pointers the lanes were built from).
template <bool G32>
__device__ __forceinline__ void meta_issue(const MetaLanes& m, uint32_t t, char* metabuf)
{
    dma4(m.a.at(t), metabuf);
    if (G32) dma4(m.b.at(t), metabuf + 256);
}
template <bool G32>
__device__ __forceinline__ MetaLanes meta_lanes(const uint32_t* off_dma, const uint16_t* scales, const uint16_t* zeros,
                                                const uint64_t* bmp, int lane)
{
    if (G32) return meta_lanes_g32(off_dma, scales, zeros, bmp, lane);
    MetaLanes m;
    m.a = meta_lane(off_dma, scales, zeros, lane);
    m.b = m.a;
    return m;
}

// The C operand of the address products: where the image starts (of the lane half's first tile; img), in all sixteen
// registers; the tiles behind it are immediate offsets of the gather.  Made anew for every stage by eight 64-bit moves
// (written out: the compiler makes sixteen of 32 bits): kept, the sixteen registers would not fit beside the dequantisation's.
__device__ __forceinline__ i32x16_t image_base(uint32_t img)
{
    typedef uint64_t u64x8_t __attribute__((ext_vector_type(8)));
    u64x8_t b;
    const uint64_t pair = ((uint64_t)img << 32) | img;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        uint64_t x;
        asm volatile("v_mov_b64 %0, %1" : "=v"(x) : "v"(pair));
        b[i] = x;
    }
    return __builtin_bit_cast(i32x16_t, b);
}
// How the 32 tiles of a stage are dequantised and expanded: half of two tiles per LDS read (HALVES, rank_device.hpp), as for more
// than eight weight rows always, or a whole tile (rank_whole.hpp).  bits: bits_load of the stage; w, wgroup: see RowSums.
// With whole tiles a batch has fewer scalar instructions but twice as many reads of weights: less where the scalar unit's share
// is on the way of the vector unit's, as in the fused kernels, more where a wavefront waits for its own reads, as in the key
// products (us, 70 %, halves / whole: 256 heads x 4096 tokens, keys, 2 bits, four rows 32.6 / 33.3, eight 33.6 / 37.5; 4 bits 33.5
// / 34.5, 35.6 / 39.5; 32 x 1024, 4 bits, eight rows 7.61 / 8.15).  The value products: value_whole (quant_spmv.hip).
template <int NW, int BIT, bool G32, bool HALVES>
struct StageRank;
// The bitmaps of the first batch are requested behind the products and arrive while those run (nothing scalar is
// carried across the lane-dependent branches of the dequantisation in front), the others one batch ahead.
template <int NW, int BIT, bool G32>
struct StageRank<NW, BIT, G32, true> {
    using Sums = RowSums<NW>;
    RankConst rank;
    StageLane<BIT> at;
    uint32_t image, img;
    __device__ __forceinline__ StageRank(uint32_t meta0, uint32_t words0, uint32_t image, int lane)
        : rank(rank_const(lane)), at(meta0, words0, image, lane), image(image), img(image + (uint32_t)(lane >> 5) * 4u * kImgStride) {}
    // The stage's bitmaps in front of the address products (bm: of its first tile): bitmap of tile lane & 31.
    static __device__ __forceinline__ uint32_t bits_at(int lane) { return (uint32_t)(lane & (kSubTiles - 1)) * 8u; }
    static __device__ __forceinline__ uint2 bits_load(const uint64_t* bm, uint32_t at)
    {
        return *reinterpret_cast<const uint2*>(reinterpret_cast<const char*>(bm) + at);
    }
    __device__ __forceinline__ void stage(const StageAt& s, const uint64_t* bm, uint2 bits, uint32_t w, uint32_t wgroup, Sums& sums,
                                          int lane, int mode) const
    {
        dequant_stage<BIT, G32>(at, s, image, lane, mode);
        constexpr int G = kSubTiles / 8;
        RankAddr a = rank_addresses(rank, bits, image_base(img));
        u32x16_t cur;
        rank_settle_load(a, cur, bm);
        static_for<G>([&](auto gc) {
            constexpr int g = decltype(gc)::value;
            u32x16_t nxt;
            sums.template batch<(g + 1 < G), g, (g + 1) * 64, g * 8 * kImgStride, kImgStride>(cur, nxt, bm, a, w, wgroup);
            cur = nxt;
        });
    }
};
// Whole tiles.  kZeros: tiles of up to 32 survivors lie behind zeros in the image and are read without masks (rank_whole.hpp); the few
// others' rows count as empty there, and the lanes fetch their values out of the staged words.  A stage with more than kDirectMax of
// those goes under exec masks, from an image without zeros, and so do the stages behind it up to one that has none: clearing the
// zeros again costs a third of a stage.  With 2 bits, one group and up to four rows only: the wider formats, whose long tiles take three LDS reads in a
// row, gain nothing by it (4 bits, 8 heads x 1024 tokens, 70 %: 16.2 under masks, 16.8 without; two groups 16.7 and 17.7), and with eight
// rows there are no registers for both forms (128 x 4096, 70 %: 38.4 under masks, 38.8 with both; 50 % 43.1 and 44.0).
template <int NW, int BIT, bool G32>
struct StageRank<NW, BIT, G32, false> {
    using Sums = WholeSums<NW>;
    static constexpr bool kZeros = BIT == 2 && !G32 && NW <= 4;
    WholeRank rank;
    StageLane<BIT> at;
    uint32_t image;
    uint32_t direct = kDirectMax;  // long tiles that a stage may have; 0: the zeros in the image have been written over
    __device__ __forceinline__ StageRank(uint32_t meta0, uint32_t words0, uint32_t image, int lane)
        : rank(whole_rank(lane)), at(meta0, words0, image, lane), image(image)
    {
        if (kZeros) clear_zeros(lane);
    }
    static __device__ __forceinline__ uint32_t bits_at(int lane) { return whole_bits_at(lane); }
    static __device__ __forceinline__ uint2 bits_load(const uint64_t* bm, uint32_t at) { return whole_bits_load(bm, at); }
    __device__ __forceinline__ void clear_zeros(int lane) const
    {
        constexpr int kPieces = kWholeZeros / 16;
        uint32_t z = 0u;
        asm volatile("" : "+v"(lane), "+v"(z));  // (addresses and zeros are made here and hold no registers elsewhere)
        static_assert(kWholeZeros % 16 == 0 && kWholeZeros >= 2 * 33 && kWholeZeros + 64 <= kImgStride, "zeros, then 32 values");
#pragma unroll
        for (int i = 0; i < (kSubTiles * kPieces + 63) / 64; i++) {
            const int e = i * 64 + lane;
            if (e < kSubTiles * kPieces)
                *(MSTF_LDS u32x4_t*)(uintptr_t)(image + (uint32_t)(e / kPieces) * kImgStride + (uint32_t)(e % kPieces) * 16u) =
                    u32x4_t{z, z, z, z};
        }
    }
    template <bool FIRST>
    __device__ __forceinline__ void expand_masked(const uint64_t* bm, uint2 bits, uint32_t w, uint32_t wgroup, Sums& sums) const
    {
        if (FIRST) sums.clear();
        whole_masked_stage<Sums::NM, kImgStride>(rank, bm, bits, image, w, w + wgroup, sums.acc);
    }
    // FIRST: the stage starts the sums.
    template <bool FIRST = false>
    __device__ __forceinline__ void stage(const StageAt& s, const uint64_t* bm, uint2 bits, uint32_t w, uint32_t wgroup, Sums& sums,
                                          int lane, int mode)
    {
        if constexpr (!kZeros) {
            dequant_stage<BIT, G32>(at, s, image, lane, mode);
            expand_masked<FIRST>(bm, bits, w, wgroup, sums);
        } else {
            const LongTiles<BIT> lt(at, s, lane);
            if (lt.count() > (int)direct) {
                dequant_halves<BIT, G32>(at, s, lt, 0u, true, lane, mode);
                expand_masked<FIRST>(bm, bits, w, wgroup, sums);
                direct = 0u;
                return;
            }
            if (direct == 0u) clear_zeros(lane);
            direct = kDirectMax;
            const uint2 pair = dequant_halves<BIT, G32>(at, s, lt, (uint32_t)kWholeZeros, false, lane, mode);
            static_assert(Sums::NM == 1, "four rows");
            whole_stage<kImgStride, FIRST>(rank, lt.mask != 0ull ? whole_without(bits, lt.tiles(), lane) : bits, image, w, sums.acc[0]);
            for (uint64_t left = lt.mask; left != 0ull; left &= left - 1ull) {
                const uint32_t bit = (uint32_t)__builtin_ctzll(left), tl = bit / LongTiles<BIT>::kLanes;
                const uint64_t there = lanes_of(whole_bitmap(bits, tl));
                const _Float16 v = dequant_long<BIT, G32>(s, lt, pair, bit, rank_below(there), mode);
                const uint32_t x = select_lane(there, (uint32_t)as_u16(v), 0u);
                const uint32_t wt = lds_load_u16(w + tl * 2u);
                sums.acc[0][0] = __builtin_amdgcn_mfma_f32_4x4x4f16(as_h4(x, 0u), as_h4(wt, 0u), sums.acc[0][0], 0, 0, 0);
            }
        }
    }
};

}  // namespace mstf
