// Expansion of bitmap tiles a whole tile per LDS read, for images of tiles at a fixed stride and up to eight weight rows: the
// quantised fused kernels and value products over many blocks (quant_device.hpp, StageRank).
//
// In rank_device.hpp a register of the address products holds the same half of two tiles, so that an exec mask is put
// together from two 32-bit pieces and the lane halves' sums have to be joined.  Here the rows of a product are the two halves
// of sixteen tiles - row 8 g + 4 P + j for half P of a tile - so that a register holds a tile whole, lane = element: one
// 64-bit reversal sets its exec mask, two products (three there) make the addresses of 32 tiles, and nothing is joined.
// A product sums over 64 bits: the elements of the row's own half in front of the column's position (lanes 0 .. 31),
// and for the second half of a tile all of the first (lanes 32 .. 63; masked off for the first half).
// The bits are 4-bit floats and the sums 32-bit floats below the normal range, whose bits are the integer they hold: with the
// products' unit at twice the smallest 32-bit float every bit adds 2 to the LDS byte address in C, all of it exact.  (Where the
// tiles' addresses differ - the fp16 format - C would be read from a table for 32 tiles instead of for 16 pairs, and the
// longer chain of these products costs the single wavefronts of small calls 2 %: those kernels keep the other layout.)
// 2 bits, 70 %, 256 heads x 4096 tokens, fused attention: 48.3 -> 46.9 us (exec masks 3.5 us of it before, rank products 3.4).
#pragma once
#include "rank_device.hpp"

namespace mstf {

typedef uint64_t u64x8_t __attribute__((ext_vector_type(8)));

struct WholeRank {
    i32x4_t before;    // B: register r, number i is bit 4 i + r of a half, element 31 - (4 i + r)
    uint32_t keep;     // all bits, none in the lanes that add nothing to a tile's first half
    bool second, mix;  // the lane's row belongs to a tile's second half; that, or (not both) the lane is one of 32 .. 63
};
__device__ __forceinline__ WholeRank whole_rank(int lane)
{
    WholeRank c;
    const int n = lane & 31, all = lane >> 5;  // column (position); lanes 32 .. 63: the whole first half counts
    c.second = (lane & 4) != 0;                // row n
    c.mix = c.second != (all != 0);
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const uint32_t one = r == 0 ? 4u : (r == 1 ? 2u : 1u);  // 2, 1, 0.5 as 4-bit numbers
        uint32_t b = 0u;
#pragma unroll
        for (int i = 0; i < 8; i++) b |= (all || 31 - (4 * i + r) < n ? one : 0u) << (4 * i);
        c.before[r] = (int)b;
    }
    c.keep = all && !c.second ? 0u : ~0u;
    return c;
}
// at[p][4 g + j]: LDS address, in the image at base, of the lane's element of tile 8 g + 4 p + j less the tile's place in the
// image.  bits: bitmap of tile lane & 31 (see rank_addresses).  Lanes n and n ^ 4 hold the bitmaps of the two tiles whose rows
// they are, so that each sends the other the half it wants: the first half is bits.y.
__device__ __forceinline__ RankAddr whole_addresses(const WholeRank& c, uint2 bits, const i32x16_t& base)
{
    typedef int i32x8_t __attribute__((ext_vector_type(8)));
    constexpr int kFp4 = 4, kScale = 127 - 74;  // (the two scales together: 2^-148)
    constexpr int kHalfMirror = 0x141, kQuadReverse = 0x1b;  // lane 7 - n of eight, then 3 - n of four: n ^ 4
    const uint32_t send = c.mix ? bits.y : bits.x, own = c.mix ? bits.x : bits.y;
    const uint32_t got = (uint32_t)__builtin_amdgcn_mov_dpp(__builtin_amdgcn_mov_dpp((int)send, kHalfMirror, 0xf, 0xf, true),
                                                            kQuadReverse, 0xf, 0xf, true);
    const uint32_t w[2] = {(c.second ? got : own) & c.keep, (c.second ? own : got) & c.keep};
    const i32x8_t before = {c.before[0], c.before[1], c.before[2], c.before[3], 0, 0, 0, 0};  // (this type reads four)
    RankAddr a;
#pragma unroll
    for (int p = 0; p < 2; p++) {
        // as 4-bit numbers the bits are worth 0.5, 1, 2 where they stand (and 2, shifted down by one)
        const i32x8_t x = {(int)(w[p] & 0x11111111u), (int)(w[p] & 0x22222222u), (int)(w[p] & 0x44444444u),
                           (int)((w[p] >> 1) & 0x44444444u), 0, 0, 0, 0};
        a.at[p] = __builtin_bit_cast(i32x16_t, __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(
                                                   x, before, __builtin_bit_cast(f16x_t, base), kFp4, kFp4, 0, kScale, 0, kScale));
    }
    return a;
}
// rank_settle_load of rank_device.hpp.
__device__ __forceinline__ void whole_settle_load(RankAddr& a, u64x8_t& first, const uint64_t* bm)
{
    asm volatile("s_load_dwordx16 %[f], %[bm], 0\n\ts_nop 15\n\ts_waitcnt lgkmcnt(0)"
                 : [f] "=&s"(first), "+v"(a.at[0]), "+v"(a.at[1])
                 : [bm] "s"(bm)
                 : "memory");
}

// Batch G (tiles 8 G .. 8 G + 7): eight LDS reads, each under its tile's bitmap, the first four tiles into acc[m][0] and the
// others into acc[m][1] by 4x4x4 products; see rank_batch (rank_device.hpp) for registers, waits and the other arguments.
//   wa, wb : LDS address of w[lane & 3][0] of the first tile of the stage, for the accumulators 0 .. 3 and (NM = 2) 4 .. 7
#define MSTF_WG(LD, H, M, A, I) "s_brev_b64 exec, %[" M "]\n\t" LD " " H ", %[" A "] offset:%[" I "]\n\t"
#define MSTF_WLO "ds_read_u16"
#define MSTF_WHI "ds_read_u16_d16_hi"
#define MSTF_WGATHER                                                                                                 \
    MSTF_WG(MSTF_WLO, MSTF_GV0, "m0", "a0", "i0") MSTF_WG(MSTF_WHI, MSTF_GV2, "m1", "a1", "i1")                       \
    MSTF_WG(MSTF_WLO, MSTF_GV1, "m2", "a2", "i2") MSTF_WG(MSTF_WHI, MSTF_GV3, "m3", "a3", "i3")                       \
    MSTF_WG(MSTF_WLO, MSTF_GV4, "m4", "a4", "i4") MSTF_WG(MSTF_WHI, MSTF_GV6, "m5", "a5", "i5")                       \
    MSTF_WG(MSTF_WLO, MSTF_GV5, "m6", "a6", "i6") MSTF_WG(MSTF_WHI, MSTF_GV7, "m7", "a7", "i7")                       \
    "s_mov_b64 exec, -1\n\ts_waitcnt lgkmcnt(4)\n\t"
#define MSTF_WCLEAR                                                                                                  \
    "v_mov_b64 " MSTF_GV0_1 ", 0\n\tv_mov_b64 " MSTF_GV2_3 ", 0\n\tv_mov_b64 " MSTF_GV4_5 ", 0\n\tv_mov_b64 " MSTF_GV6_7 ", 0\n\t"
#define MSTF_WIN                                                                                                     \
    [m0] "s"(mv[0]), [m1] "s"(mv[1]), [m2] "s"(mv[2]), [m3] "s"(mv[3]), [m4] "s"(mv[4]), [m5] "s"(mv[5]), [m6] "s"(mv[6]), \
        [m7] "s"(mv[7]), [a0] "v"(x[R]), [a1] "v"(x[R + 1]), [a2] "v"(x[R + 2]), [a3] "v"(x[R + 3]), [a4] "v"(y[R]),             \
        [a5] "v"(y[R + 1]), [a6] "v"(y[R + 2]), [a7] "v"(y[R + 3]), [i0] "i"(I0), [i1] "i"(I0 + IS), [i2] "i"(I0 + 2 * IS), \
        [i3] "i"(I0 + 3 * IS), [i4] "i"(I0 + 4 * IS), [i5] "i"(I0 + 5 * IS), [i6] "i"(I0 + 6 * IS), [i7] "i"(I0 + 7 * IS),  \
        [wa] "v"(wa), [woff] "i"(G * 16)
#define MSTF_WLOAD "s_load_dwordx16 %[nm], %[nb], %[boff]\n\t"
#define MSTF_WM(ACC, A, W) "v_mfma_f32_4x4x4_16b_f16 %[" ACC "], " A ", %[" W "], %[" ACC "]\n\t"
// (the weights of four tiles are half of a register quadruple, which an operand cannot name: two 8-byte reads)
#define MSTF_WONE                                                                                                    \
    MSTF_WCLEAR "ds_read_b64 %[w], %[wa] offset:%[woff]\n\tds_read_b64 %[v], %[wa] offset:%[woff]+8\n\t" MSTF_WGATHER   \
    MSTF_WM("p0", MSTF_GV0_1, "w") "s_waitcnt lgkmcnt(0)\n\t" MSTF_WM("p1", MSTF_GV4_5, "v")                           \
    MSTF_WM("p0", MSTF_GV2_3, "w") "s_nop 0\n\t" MSTF_WM("p1", MSTF_GV6_7, "v") "s_nop 4"
#define MSTF_WTWO                                                                                                    \
    MSTF_WCLEAR "ds_read_b64 %[w], %[wa] offset:%[woff]\n\tds_read_b64 %[v], %[wa] offset:%[woff]+8\n\t"                \
    "ds_read_b64 %[w2], %[wb] offset:%[woff]\n\tds_read_b64 %[v2], %[wb] offset:%[woff]+8\n\t" MSTF_WGATHER             \
    "v_or_b32 " MSTF_GV0 ", " MSTF_GV0 ", " MSTF_GV2 "\n\tv_or_b32 " MSTF_GV1 ", " MSTF_GV1 ", " MSTF_GV3 "\n\t"        \
    "s_nop 1\n\t" MSTF_WM("p0", MSTF_GV0_1, "w") MSTF_WM("q0", MSTF_GV0_1, "w2") "s_waitcnt lgkmcnt(0)\n\t"          \
    "v_or_b32 " MSTF_GV4 ", " MSTF_GV4 ", " MSTF_GV6 "\n\tv_or_b32 " MSTF_GV5 ", " MSTF_GV5 ", " MSTF_GV7 "\n\t"        \
    "s_nop 1\n\t" MSTF_WM("p1", MSTF_GV4_5, "v") MSTF_WM("q1", MSTF_GV4_5, "v2") "s_nop 4"
template <int NM, bool PREFETCH, int G, int BOFF, int IS>
__device__ __forceinline__ void whole_batch(const u64x8_t& mv, u64x8_t& nxt, const uint64_t* nbm, const RankAddr& at, uint32_t wa,
                                            uint32_t wb, f4_t (&acc)[NM][2])
{
    static_assert(NM == 1 || NM == 2, "four or eight accumulators");
    constexpr int R = G * 4, I0 = G * 8 * IS;
    const i32x16_t &x = at.at[0], &y = at.at[1];
    u32x2_t w, v, w2, v2;
    if constexpr (NM == 1) {
        if constexpr (PREFETCH)
            asm volatile(MSTF_WLOAD MSTF_WONE
                         : [p0] "+v"(acc[0][0]), [p1] "+v"(acc[0][1]), [w] "=&v"(w), [v] "=&v"(v), [nm] "=&s"(nxt)
                         : MSTF_WIN, [nb] "s"(nbm), [boff] "i"(BOFF)
                         : MSTF_GV_CLOBBER, "memory");
        else
            asm volatile(MSTF_WONE
                         : [p0] "+v"(acc[0][0]), [p1] "+v"(acc[0][1]), [w] "=&v"(w), [v] "=&v"(v)
                         : MSTF_WIN
                         : MSTF_GV_CLOBBER, "memory");
    } else {
        if constexpr (PREFETCH)
            asm volatile(MSTF_WLOAD MSTF_WTWO
                         : [p0] "+v"(acc[0][0]), [p1] "+v"(acc[0][1]), [q0] "+v"(acc[1][0]), [q1] "+v"(acc[1][1]),
                           [w] "=&v"(w), [v] "=&v"(v), [w2] "=&v"(w2), [v2] "=&v"(v2), [nm] "=&s"(nxt)
                         : MSTF_WIN, [wb] "v"(wb), [nb] "s"(nbm), [boff] "i"(BOFF)
                         : MSTF_GV_CLOBBER, "memory");
        else
            asm volatile(MSTF_WTWO
                         : [p0] "+v"(acc[0][0]), [p1] "+v"(acc[0][1]), [q0] "+v"(acc[1][0]), [q1] "+v"(acc[1][1]),
                           [w] "=&v"(w), [v] "=&v"(v), [w2] "=&v"(w2), [v2] "=&v"(v2)
                         : MSTF_WIN, [wb] "v"(wb)
                         : MSTF_GV_CLOBBER, "memory");
    }
    if constexpr (!PREFETCH) nxt = mv;
}
#undef MSTF_WG
#undef MSTF_WLO
#undef MSTF_WHI
#undef MSTF_WGATHER
#undef MSTF_WCLEAR
#undef MSTF_WIN
#undef MSTF_WLOAD
#undef MSTF_WM
#undef MSTF_WONE
#undef MSTF_WTWO

// The sums of NW <= 8 weight rows; see RowSums (rank_device.hpp).
template <int NW>
struct WholeSums {
    static_assert(!wide_rows(NW), "at most eight rows");
    static constexpr bool kWide = false;
    static constexpr int NM = (NW + 3) / 4, kRows = NM * 4;
    f4_t acc[NM][2];

    __device__ __forceinline__ void clear()
    {
#pragma unroll
        for (int m = 0; m < NM; m++) acc[m][0] = acc[m][1] = f4_t{0.f, 0.f, 0.f, 0.f};
    }
    static __device__ __forceinline__ uint32_t waddr(uint32_t rows_lds, uint32_t row_bytes, int lane)
    {
        return rows_lds + (uint32_t)(lane & 3) * row_bytes;
    }
    static __device__ __forceinline__ uint32_t advance(uint32_t w, uint32_t bytes) { return w + bytes; }
    // lane 4 b + j: positions 4 b .. 4 b + 3 of row 4 m + j
    __device__ __forceinline__ f4_t joined(int m) const { return acc[m][0] + acc[m][1]; }
    template <class F>
    __device__ __forceinline__ void each4(int lane, F&& f) const
    {
#pragma unroll
        for (int m = 0; m < NM; m++) {
            const f4_t v = joined(m);
            if (4 * m + (lane & 3) < NW) f(4 * m + (lane & 3), lane & ~3, v);
        }
    }
};

}  // namespace mstf
