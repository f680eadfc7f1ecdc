// Expansion of bitmap tiles with the ranks computed by the matrix cores.
//
// Element p of a tile sits at rank(p) = number of bits set in front of p in the tile's packed values, so that expanding
// a tile means one LDS read per lane at base + 2 * rank.  As a prefix count that rank is a product of the bitmap with a
// triangular matrix of twos, and a run of 32 bitmaps makes it a matrix product: three v_mfma_i32_32x32x32_i8 per 32
// tiles leave the finished LDS byte addresses of all 2048 elements - the tile's base is the product's C operand - in
// the registers of the lanes that read them.  The vector unit, which the decode kernels keep busiest, is left with
// spreading the bitmaps into byte operands (twelve instructions per 32 tiles) instead of two v_mbcnt and one v_lshl_add
// per tile.
//
// Layout of a product: a register of the result holds, in lanes 0 .. 31, the 32 positions of one half (P) of tile
// 8 * (r / 4) + r % 4 and, in lanes 32 .. 63, the same positions of the tile four further on.  One LDS read therefore
// gathers half of two tiles, under an exec mask put together from a 32-bit half of each bitmap (elements of a tile are
// MSB first, so the mask is the half with its bits reversed); four consecutive registers are four consecutive tiles of
// the lane, which is what the A operand of the accumulating product wants: the lane multiplies its four tiles with
// their weights, the two lane halves add up different tiles of the same positions, and join_halves folds them at the end.
//
// Against ranks on the vector unit (two v_mbcnt, address, one tile per LDS read): vector instructions of the 2-bit fused
// kernel 30.4 -> 21.7 M per launch (256 KV heads x 4096 tokens), LDS busy cycles 23.0 -> 17.8 M (weights as 8-byte reads
// and no reads to clear registers), 69.4 -> 64.8 us; fp16 fused kernel at 64 heads x 4096 tokens 14.8 -> 14.5 us under
// rocprofv3, 18.7 -> 17.8 us per step with its merge - it waits for memory more than for instructions.
#pragma once
#include "spmv_device.hpp"

namespace mstf {

// The fixed vector registers of the gather statements: the top of the budget of 128 that four wavefronts per SIMD leave.
#define MSTF_GV0 "v120"
#define MSTF_GV1 "v121"
#define MSTF_GV2 "v122"
#define MSTF_GV3 "v123"
#define MSTF_GV4 "v124"
#define MSTF_GV5 "v125"
#define MSTF_GV6 "v126"
#define MSTF_GV7 "v127"
#define MSTF_GV0_1 "v[120:121]"
#define MSTF_GV2_3 "v[122:123]"
#define MSTF_GV4_5 "v[124:125]"
#define MSTF_GV6_7 "v[126:127]"
#define MSTF_GV_CLOBBER MSTF_GV0, MSTF_GV1, MSTF_GV2, MSTF_GV3, MSTF_GV4, MSTF_GV5, MSTF_GV6, MSTF_GV7

typedef float f16x_t __attribute__((ext_vector_type(16)));
typedef int i32x4_t __attribute__((ext_vector_type(4)));
typedef int i32x16_t __attribute__((ext_vector_type(16)));

// The constant B operands.  A lane's sixteen bytes of a bitmap operand are, for lane half s, register r and byte i, the
// bit 8 i + 4 s + r of the 32-bit bitmap half; it is left where the mask finds it, so registers 0 and 2 hold it as 1
// and registers 1 and 3 as 2, and the constants make up for that: tri counts the bits of the elements in front of the
// lane's position (element e of a half is bit 31 - e), full counts all of them.
struct RankConst {
    i32x4_t tri, full;
    uint32_t shift;  // 4 * lane half
};
__device__ __forceinline__ RankConst rank_const(int lane)
{
    RankConst c;
    const int p = lane & 31, s = lane >> 5;
    c.shift = (uint32_t)s * 4u;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const uint32_t unit = (r & 1) ? 1u : 2u;
        uint32_t t = 0u;
#pragma unroll
        for (int i = 0; i < 4; i++) t |= (31 - (8 * i + 4 * s + r) < p ? unit : 0u) << (8 * i);
        c.tri[r] = (int)t;
        c.full[r] = (int)(unit * 0x01010101u);
    }
    return c;
}
__device__ __forceinline__ i32x4_t rank_bits(uint32_t half, uint32_t shift)
{
    const uint32_t a = half >> shift, b = a >> 2;
    return i32x4_t{(int)(a & 0x01010101u), (int)(a & 0x02020202u), (int)(b & 0x01010101u), (int)(b & 0x02020202u)};
}

// LDS addresses of the elements of 32 tiles: at[P] for the positions of half P.  bits: bitmap of tile lane & 31 (x: the
// low 32 bits, elements 32 .. 63; y: elements 0 .. 31).  base: LDS byte address of the first value of the register's
// tile (see the layout above).
struct RankAddr {
    i32x16_t at[2];
};
__device__ __forceinline__ RankAddr rank_addresses(const RankConst& c, uint2 bits, const i32x16_t& base)
{
    RankAddr a;
    const i32x4_t front = rank_bits(bits.y, c.shift), back = rank_bits(bits.x, c.shift);
    a.at[0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(front, c.tri, base, 0, 0, 0);
    a.at[1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(front, c.full, base, 0, 0, 0);
    a.at[1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(back, c.tri, a.at[1], 0, 0, 0);
    return a;
}
// Requests the bitmaps of the stage's first batch (8 tiles from bm) and waits for them and for the products of
// rank_addresses, whose results an LDS read that the compiler cannot see must not use earlier (twelve wait states
// after an eight-pass product).
__device__ __forceinline__ void rank_settle_load(RankAddr& a, u32x16_t& first, const uint64_t* bm)
{
    asm volatile("s_load_dwordx16 %[f], %[bm], 0\n\ts_nop 15\n\ts_waitcnt lgkmcnt(0)"
                 : [f] "=&s"(first), "+v"(a.at[0]), "+v"(a.at[1])
                 : [bm] "s"(bm)
                 : "memory");
}

// The same without a load.
__device__ __forceinline__ void rank_settle(RankAddr& a)
{
    asm volatile("s_nop 15" : "+v"(a.at[0]), "+v"(a.at[1])::"memory");
}
// The bitmaps of the first eight tiles of a chain of rank_batch statements, requested and waited for in one statement.
__device__ __forceinline__ u32x16_t load_bitmaps_scalar(const uint64_t* bm)
{
    u32x16_t m;
    asm volatile("s_load_dwordx16 %0, %1, 0\n\ts_waitcnt lgkmcnt(0)" : "=&s"(m) : "s"(bm) : "memory");
    return m;
}

// A wavefront's table of the LDS addresses at which the 32 tiles of a stage start, and its way into the C operand: a
// lane puts the address of tile lane & 31 and gets back those of the tiles of its sixteen result registers, four
// neighbours per LDS read.
struct RankTable {
    uint32_t mine, four;
    __device__ __forceinline__ void put(uint32_t a) const { *(MSTF_LDS uint32_t*)(uintptr_t)mine = a; }
    __device__ __forceinline__ i32x16_t get() const
    {
        i32x16_t b;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const u32x4_t v = *(MSTF_LDS const u32x4_t*)(uintptr_t)(four + (uint32_t)i * 32u);
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const uint32_t x = v[k];
                b[4 * i + k] = (int)x;
            }
        }
        return b;
    }
};
__device__ __forceinline__ RankTable rank_table(const char* room, int lane)
{
    const uint32_t a = lds_addr(room);
    return {a + (uint32_t)(lane & 31) * 4u, a + (uint32_t)(lane >> 5) * 16u};
}

// Pieces of the gather statements below.  They gather batch G (tiles 8 G .. 8 G + 7) of a stage: per half P four LDS
// reads, each under the exec mask of its two half tiles, the first and third into the low half of a register, the second
// and fourth into the high half of another (cleared registers: a lane without an element multiplies zero).  One
// statement on fixed registers, as nothing of the compiler's may be scheduled while exec is partial; the wavefront has
// all 64 lanes active in front of and behind it.  The weights are requested first and LDS reads return in order, so
// lgkmcnt(4) waits for them and the first half P (a scalar load in flight can only make that wait longer).
#define MSTF_RG(LD, H, D, X, Y, I) \
    "s_brev_b32 exec_lo, %[" X "]\n\ts_brev_b32 exec_hi, %[" Y "]\n\t" LD " " H ", %[" D "] offset:%[" I "]\n\t"
#define MSTF_RLO "ds_read_u16"
#define MSTF_RHI "ds_read_u16_d16_hi"
#define MSTF_RGATHER                                                                                                  \
    MSTF_RG(MSTF_RLO, MSTF_GV0, "a0", "h0", "h4", "i0") MSTF_RG(MSTF_RHI, MSTF_GV2, "a1", "h1", "h5", "i1")           \
    MSTF_RG(MSTF_RLO, MSTF_GV1, "a2", "h2", "h6", "i2") MSTF_RG(MSTF_RHI, MSTF_GV3, "a3", "h3", "h7", "i3")           \
    MSTF_RG(MSTF_RLO, MSTF_GV4, "b0", "l0", "l4", "i0") MSTF_RG(MSTF_RHI, MSTF_GV6, "b1", "l1", "l5", "i1")           \
    MSTF_RG(MSTF_RLO, MSTF_GV5, "b2", "l2", "l6", "i2") MSTF_RG(MSTF_RHI, MSTF_GV7, "b3", "l3", "l7", "i3")           \
    "s_mov_b64 exec, -1\n\ts_waitcnt lgkmcnt(4)\n\t"
#define MSTF_RCLEAR                                                                                                   \
    "v_mov_b64 " MSTF_GV0_1 ", 0\n\tv_mov_b64 " MSTF_GV2_3 ", 0\n\tv_mov_b64 " MSTF_GV4_5 ", 0\n\tv_mov_b64 " MSTF_GV6_7 ", 0\n\t"
#define MSTF_RIN                                                                                                      \
    [l0] "s"(mv[0]), [h0] "s"(mv[1]), [l1] "s"(mv[2]), [h1] "s"(mv[3]), [l2] "s"(mv[4]), [h2] "s"(mv[5]),             \
        [l3] "s"(mv[6]), [h3] "s"(mv[7]), [l4] "s"(mv[8]), [h4] "s"(mv[9]), [l5] "s"(mv[10]), [h5] "s"(mv[11]),       \
        [l6] "s"(mv[12]), [h6] "s"(mv[13]), [l7] "s"(mv[14]), [h7] "s"(mv[15]), [a0] "v"(a.at[0][4 * G]),             \
        [a1] "v"(a.at[0][4 * G + 1]), [a2] "v"(a.at[0][4 * G + 2]), [a3] "v"(a.at[0][4 * G + 3]),                     \
        [b0] "v"(a.at[1][4 * G]), [b1] "v"(a.at[1][4 * G + 1]), [b2] "v"(a.at[1][4 * G + 2]),                         \
        [b3] "v"(a.at[1][4 * G + 3]), [i0] "i"(I0), [i1] "i"(I0 + IS), [i2] "i"(I0 + 2 * IS), [i3] "i"(I0 + 3 * IS),  \
        [wa] "v"(wa), [woff] "i"(WOFF)
#define MSTF_RLOAD "s_load_dwordx16 %[nm], %[nb], %[boff]\n\t"

// Batch G into acc[m][P] for at most eight accumulators, by 4x4x4 products.  Four: the register pair (t0, 0, t2, 0) and
// the pair (0, t1, 0, t3) both against the weights (w0 .. w3) of the lane's four tiles, so that no vector instruction
// packs - and an infinite weight makes a NaN of a tile's neighbour as it does of an absent element, 0 x inf.  Eight: the
// pairs are merged first, two vector instructions for two products less; only absent elements meet a zero then.
//   mv      : the batch's eight bitmaps;  PREFETCH: those of the coming batch are requested at nbm + BOFF bytes
//   I0, IS  : immediate offset of the batch's first tile and bytes between two tiles (0, 0: `a` holds full addresses)
//   wa, wb  : LDS address of w[lane & 3][4 * (lane >> 5)] of the first tile of the stage, for the accumulators 0 .. 3
//             and (NM = 2) 4 .. 7;  WOFF: + bytes to the batch's first tile
// Two products of one accumulator are at least two instructions apart, and the statement ends
// with the wait states that an ordinary vector instruction needs before it may read a sum.
template <int NM, bool PREFETCH, int G, int BOFF, int I0, int IS, int WOFF>
__device__ __forceinline__ void rank_batch(const u32x16_t& mv, u32x16_t& nxt, const uint64_t* nbm, const RankAddr& a,
                                           uint32_t wa, uint32_t wb, f4_t (&acc)[NM][2])
{
    static_assert(NM == 1 || NM == 2, "four or eight accumulators");
    u32x2_t w, w2;
#define MSTF_RM(ACC, A, W) "v_mfma_f32_4x4x4_16b_f16 %[" ACC "], " A ", %[" W "], %[" ACC "]\n\t"
#define MSTF_RONE                                                                                                     \
    MSTF_RCLEAR "ds_read_b64 %[w], %[wa] offset:%[woff]\n\t" MSTF_RGATHER MSTF_RM("p0", MSTF_GV0_1, "w")              \
    "s_waitcnt lgkmcnt(0)\n\t" MSTF_RM("p1", MSTF_GV4_5, "w") MSTF_RM("p0", MSTF_GV2_3, "w") "s_nop 0\n\t"            \
    MSTF_RM("p1", MSTF_GV6_7, "w") "s_nop 4"
#define MSTF_RTWO                                                                                                     \
    MSTF_RCLEAR "ds_read_b64 %[w], %[wa] offset:%[woff]\n\tds_read_b64 %[w2], %[wb] offset:%[woff]\n\t" MSTF_RGATHER  \
    "v_or_b32 " MSTF_GV0 ", " MSTF_GV0 ", " MSTF_GV2 "\n\tv_or_b32 " MSTF_GV1 ", " MSTF_GV1 ", " MSTF_GV3 "\n\t"        \
    "s_nop 1\n\t" MSTF_RM("p0", MSTF_GV0_1, "w") MSTF_RM("q0", MSTF_GV0_1, "w2") "s_waitcnt lgkmcnt(0)\n\t"          \
    "v_or_b32 " MSTF_GV4 ", " MSTF_GV4 ", " MSTF_GV6 "\n\tv_or_b32 " MSTF_GV5 ", " MSTF_GV5 ", " MSTF_GV7 "\n\t"        \
    "s_nop 1\n\t" MSTF_RM("p1", MSTF_GV4_5, "w") MSTF_RM("q1", MSTF_GV4_5, "w2") "s_nop 4"
    if constexpr (NM == 1) {
        if constexpr (PREFETCH)
            asm volatile(MSTF_RLOAD MSTF_RONE
                         : [p0] "+v"(acc[0][0]), [p1] "+v"(acc[0][1]), [w] "=&v"(w), [nm] "=&s"(nxt)
                         : MSTF_RIN, [nb] "s"(nbm), [boff] "i"(BOFF)
                         : MSTF_GV_CLOBBER, "memory");
        else
            asm volatile(MSTF_RONE
                         : [p0] "+v"(acc[0][0]), [p1] "+v"(acc[0][1]), [w] "=&v"(w)
                         : MSTF_RIN
                         : MSTF_GV_CLOBBER, "memory");
    } else {
        if constexpr (PREFETCH)
            asm volatile(MSTF_RLOAD MSTF_RTWO
                         : [p0] "+v"(acc[0][0]), [p1] "+v"(acc[0][1]), [q0] "+v"(acc[1][0]), [q1] "+v"(acc[1][1]),
                           [w] "=&v"(w), [w2] "=&v"(w2), [nm] "=&s"(nxt)
                         : MSTF_RIN, [wb] "v"(wb), [nb] "s"(nbm), [boff] "i"(BOFF)
                         : MSTF_GV_CLOBBER, "memory");
        else
            asm volatile(MSTF_RTWO
                         : [p0] "+v"(acc[0][0]), [p1] "+v"(acc[0][1]), [q0] "+v"(acc[1][0]), [q1] "+v"(acc[1][1]),
                           [w] "=&v"(w), [w2] "=&v"(w2)
                         : MSTF_RIN, [wb] "v"(wb)
                         : MSTF_GV_CLOBBER, "memory");
    }
    if constexpr (!PREFETCH) nxt = mv;
#undef MSTF_RM
#undef MSTF_RONE
#undef MSTF_RTWO
}

// Batch G into the 32 accumulators of acc[P] by one 32x32x8 product per half P: the result layout of the address
// products is also the A layout of that shape (row = position, the lane half's four tiles the k index).  The two
// registers of a pair are merged first (one vector instruction per two reads), since the product, not the vector unit,
// bounds this form.  wa: LDS address of w[lane & 31][8 G + 4 * (lane >> 5)].
template <bool PREFETCH, int G, int BOFF, int I0, int IS>
__device__ __forceinline__ void rank_batch_wide(const u32x16_t& mv, u32x16_t& nxt, const uint64_t* nbm, const RankAddr& a,
                                                uint32_t wa, f16x_t (&acc)[2])
{
    constexpr int WOFF = 0;
    u32x2_t w;
#define MSTF_RWIDE                                                                                                    \
    MSTF_RCLEAR "ds_read_b64 %[w], %[wa] offset:%[woff]\n\t" MSTF_RGATHER                                             \
    "v_or_b32 " MSTF_GV0 ", " MSTF_GV0 ", " MSTF_GV2 "\n\tv_or_b32 " MSTF_GV1 ", " MSTF_GV1 ", " MSTF_GV3 "\n\t"        \
    "s_nop 1\n\tv_mfma_f32_32x32x8_f16 %[p0], " MSTF_GV0_1 ", %[w], %[p0]\n\t"                                        \
    "s_waitcnt lgkmcnt(0)\n\t"                                                                                        \
    "v_or_b32 " MSTF_GV4 ", " MSTF_GV4 ", " MSTF_GV6 "\n\tv_or_b32 " MSTF_GV5 ", " MSTF_GV5 ", " MSTF_GV7 "\n\t"        \
    "s_nop 1\n\tv_mfma_f32_32x32x8_f16 %[p1], " MSTF_GV4_5 ", %[w], %[p1]\n\t"                                        \
    "s_nop 15"
    if constexpr (PREFETCH) {
        asm volatile(MSTF_RLOAD MSTF_RWIDE
                     : [p0] "+v"(acc[0]), [p1] "+v"(acc[1]), [w] "=&v"(w), [nm] "=&s"(nxt)
                     : MSTF_RIN, [nb] "s"(nbm), [boff] "i"(BOFF)
                     : MSTF_GV_CLOBBER, "memory");
    } else {
        asm volatile(MSTF_RWIDE
                     : [p0] "+v"(acc[0]), [p1] "+v"(acc[1]), [w] "=&v"(w)
                     : MSTF_RIN
                     : MSTF_GV_CLOBBER, "memory");
        nxt = mv;
    }
#undef MSTF_RWIDE
}
#undef MSTF_RG
#undef MSTF_RLO
#undef MSTF_RHI
#undef MSTF_RGATHER
#undef MSTF_RCLEAR
#undef MSTF_RIN
#undef MSTF_RLOAD

// The sums of both lane halves over both position halves as the rest of the kernels wants them: lane 4 b + j holds
// positions 4 b .. 4 b + 3 (b = 0 .. 15) of accumulator j.
__device__ __forceinline__ f4_t join_halves(const f4_t (&acc)[2])
{
    f4_t out;
#pragma unroll
    for (int c = 0; c < 4; c++) {
        const float x = acc[0][c], y = acc[1][c];
        typedef uint32_t pair_t __attribute__((ext_vector_type(2)));
        const pair_t r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, x), __builtin_bit_cast(uint32_t, y),
                                                          false, false);
        const uint32_t r0 = r[0], r1 = r[1];  // (a bit cast applied to a vector element directly reads element 0)
        out[c] = __builtin_bit_cast(float, r0) + __builtin_bit_cast(float, r1);
    }
    return out;
}

// Adds the sums of a stage to those of the stages before and clears them.  The key phase does so after every stage, in
// order: a score then is the same number - bit for bit, and with it the fp16 score behind it - however the stages are
// dealt out over wavefronts (fused.hip), and in the SpMV kernel as in the fused ones.
template <int NM>
__device__ __forceinline__ void fold_stage(f4_t (&total)[NM], f4_t (&acc)[NM][2])
{
#pragma unroll
    for (int m = 0; m < NM; m++) {
        total[m] += join_halves(acc[m]);
        acc[m][0] = acc[m][1] = f4_t{0.f, 0.f, 0.f, 0.f};
    }
}

// The sums of NW weight rows (the SpMV kernels): at most eight by the 4x4x4 products, more by the 32x32x8 ones.
constexpr bool wide_rows(int nw) { return nw > 8; }
// With more than eight rows every lane reads another row, 64 or 256 bytes apart: the 16-byte chunks of a row are
// stored at chunk ^ weight_swizzle(row), which spreads the reads of sixteen (eight for rows of 128 bytes) rows over all
// LDS banks.  chunks: 16-byte chunks of a row, 4, 8 or 16.
__device__ __forceinline__ uint32_t weight_swizzle(int row, int chunks)
{
    return chunks == 4 ? (uint32_t)(row >> 2) & 3u : (uint32_t)row & (uint32_t)(chunks - 1);
}

// FOLD: sums of at most eight rows are folded stage by stage (fold_stage, called as stage_done).
template <int NW, bool FOLD = false>
struct RowSums {
    static constexpr bool kWide = wide_rows(NW);
    static constexpr int kRows = kWide ? 32 : (NW + 3) / 4 * 4;  // rows the weights have room for
    static constexpr int NM = kWide ? 1 : (NW + 3) / 4;
    f4_t narrow[kWide ? 1 : NM][2];
    f4_t total[NM];
    f16x_t wide[2];

    __device__ __forceinline__ void clear()
    {
        if constexpr (kWide) {
#pragma unroll
            for (int i = 0; i < 16; i++) wide[0][i] = wide[1][i] = 0.f;
        } else {
#pragma unroll
            for (int m = 0; m < NM; m++) narrow[m][0] = narrow[m][1] = total[m] = f4_t{0.f, 0.f, 0.f, 0.f};
        }
    }
    // row_bytes: 64 or 128 or 256; `rows_lds`: LDS address of row 0 (a multiple of row_bytes)
    static __device__ __forceinline__ uint32_t waddr(uint32_t rows_lds, uint32_t row_bytes, int lane)
    {
        const uint32_t side = (uint32_t)(lane >> 5) * 8u;
        if constexpr (kWide) {
            const int row = lane & 31;
            return rows_lds + (uint32_t)row * row_bytes + weight_swizzle(row, (int)row_bytes / 16) * 16u + side;
        } else {
            return rows_lds + (uint32_t)(lane & 3) * row_bytes + side;
        }
    }
    // w of a stage whose first weight sits `bytes` further on in its row
    static __device__ __forceinline__ uint32_t advance(uint32_t w, uint32_t bytes) { return kWide ? w ^ bytes : w + bytes; }

    template <bool PREFETCH, int G, int BOFF, int I0, int IS>
    __device__ __forceinline__ void batch(const u32x16_t& mv, u32x16_t& nxt, const uint64_t* nbm, const RankAddr& a,
                                          uint32_t w, uint32_t wgroup)
    {
        if constexpr (kWide)
            rank_batch_wide<PREFETCH, G, BOFF, I0, IS>(mv, nxt, nbm, a, w ^ (uint32_t)(G * 16), wide);
        else
            rank_batch<NM, PREFETCH, G, BOFF, I0, IS, G * 16>(mv, nxt, nbm, a, w, w + wgroup, narrow);
    }
    __device__ __forceinline__ void stage_done()
    {
        if constexpr (FOLD && !kWide) fold_stage(total, narrow);
    }
    // f(row, position, sums): the sums of four consecutive positions of a row
    template <class F>
    __device__ __forceinline__ void each4(int lane, F&& f) const
    {
        if constexpr (kWide) {
            const int row = lane & 31;
            if (row < NW) {
#pragma unroll
                for (int p = 0; p < 2; p++)
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        f(row, p * 32 + r * 8 + (lane >> 5) * 4,
                          f4_t{wide[p][4 * r], wide[p][4 * r + 1], wide[p][4 * r + 2], wide[p][4 * r + 3]});
            }
        } else {
#pragma unroll
            for (int m = 0; m < NM; m++) {
                const f4_t v = FOLD ? total[m] : join_halves(narrow[m]);
                if (4 * m + (lane & 3) < NW) f(4 * m + (lane & 3), lane & ~3, v);
            }
        }
    }
};

__device__ __forceinline__ h4_t round_h4(const f4_t& v)
{
    h4_t o;
#pragma unroll
    for (int i = 0; i < 4; i++) o[i] = (_Float16)v[i];
    return o;
}
// Stores the sums of more than eight rows as fp16, 64 positions of row r at out + r * stride.  The wide layout has every
// lane hold another row, sixteen bytes of it per store instruction; through `room` (4 KB of the wavefront's own, free by
// now) the rows leave as whole 128-byte lines instead.
template <int NW, bool FOLD>
__device__ __forceinline__ void store_rows_wide(const RowSums<NW, FOLD>& sums, char* room, _Float16* out, size_t stride,
                                                int lane)
{
    static_assert(NW % 8 == 0, "eight rows per store instruction");
    const uint32_t base = lds_addr(room);
    // (the sixteen-byte pieces of a row at piece ^ row, so that the rows spread over the LDS banks)
    sums.each4(lane, [=](int row, int pos, const f4_t& v) {
        *(MSTF_LDS h4_t*)(uintptr_t)(base + (uint32_t)row * 128u + (uint32_t)(((pos >> 3) ^ (row & 7)) * 16 + (pos & 4) * 2)) =
            round_h4(v);
    });
    const int piece = lane & 7, sub = lane >> 3;
#pragma unroll
    for (int i = 0; i < NW / 8; i++) {
        const int row = i * 8 + sub;
        const u32x4_t v = *(MSTF_LDS const u32x4_t*)(uintptr_t)(base + (uint32_t)row * 128u + (uint32_t)((piece ^ sub) * 16));
        *reinterpret_cast<u32x4_t*>(out + (size_t)row * stride + piece * 8) = v;
    }
}

// The four wavefronts of a workgroup took a channel stage each of one token block: adds their sums of more than eight rows,
// in the order of the stages, and stores them as store_rows_wide does.  Wavefront w adds up the positions 8 w .. 8 w + 7 of
// both halves and parks the others at its `my` (6 KB, its reads are over; the others' are at area + i * bytes); the fp16
// rows pass through `room` (4 KB that no wavefront reads any more behind the first barrier).
constexpr int kParkShares = 3 * 2 * 1024;
template <int NW, bool FOLD>
__device__ __forceinline__ void store_rows_shared(const RowSums<NW, FOLD>& sums, char* area, int bytes, char* room, _Float16* out,
                                                  size_t stride, int wave, int lane)
{
    static_assert(NW % 8 == 0 && wide_rows(NW), "eight rows per store instruction");
    const uint32_t mine = lds_addr(area) + (uint32_t)(wave * bytes) + (uint32_t)lane * 16u;
    f4_t own[2];
#pragma unroll
    for (int r = 0; r < 4; r++)
#pragma unroll
        for (int p = 0; p < 2; p++) {
            const f4_t v = {sums.wide[p][4 * r], sums.wide[p][4 * r + 1], sums.wide[p][4 * r + 2], sums.wide[p][4 * r + 3]};
            if (r == wave)
                own[p] = v;
            else  // (slot r, or r - 1 behind the wavefront's own)
                *(MSTF_LDS f4_t*)(uintptr_t)(mine + (uint32_t)((r - (r > wave ? 1 : 0)) * 2 + p) * 1024u) = v;
        }
    __syncthreads();
    f4_t sum[2];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int p = 0; p < 2; p++) {
            const uint32_t slot = (uint32_t)((wave - (wave > i ? 1 : 0)) * 2 + p) * 1024u;
            const f4_t v = i == wave ? own[p]
                                     : *(MSTF_LDS const f4_t*)(uintptr_t)(lds_addr(area) + (uint32_t)(i * bytes) + slot + (uint32_t)lane * 16u);
            sum[p] = i == 0 ? v : sum[p] + v;
        }
    const uint32_t base = lds_addr(room);
    const uint32_t row = (uint32_t)lane & 31u;
#pragma unroll
    for (int p = 0; p < 2; p++)  // (pieces as in store_rows_wide)
        *(MSTF_LDS h4_t*)(uintptr_t)(base + row * 128u + (((uint32_t)(4 * p + wave) ^ (row & 7u)) * 16u) +
                                     (uint32_t)(lane >> 5) * 8u) = round_h4(sum[p]);
    __syncthreads();
    if (wave < NW / 8) {
        const uint32_t piece = (uint32_t)lane & 7u, sub = (uint32_t)lane >> 3, at = (uint32_t)wave * 8u + sub;
        const u32x4_t v = *(MSTF_LDS const u32x4_t*)(uintptr_t)(base + at * 128u + ((piece ^ sub) * 16u));
        *reinterpret_cast<u32x4_t*>(out + (size_t)at * stride + piece * 8u) = v;
    }
}

// Requests the weights of the 32 tiles of a stage for more than eight rows of a value product: 64 bytes each of rows
// `stride` apart into [row][32] at dst, the sixteen-byte pieces where weight_swizzle wants them.  Sixteen rows per
// instruction; with four bytes a lane the sixteen instructions a stage took kept a CU's address unit busy as well
// (32 rows, 128 heads x 4096 tokens, value product and merge: 41.7 -> 39.3 us).
template <int NW>
__device__ __forceinline__ void stage_rows_wide(const _Float16* src, size_t stride, char* dst, int lane)
{
    static_assert(NW % 16 == 0 && kSubTiles * 2 == 64, "sixteen rows of 64 bytes per instruction");
#pragma unroll
    for (int i = 0; i < NW / 16; i++) {
        const int row = 16 * i + (lane >> 2);
        const uint32_t piece = ((uint32_t)lane & 3u) ^ weight_swizzle(row, 4);
        dma16(src + (size_t)row * stride + piece * 8u, dst + i * 1024);
    }
}

// Requests the NW query rows of a key product, rbytes each and contiguous at src, into [row][rbytes] at dst.  SHARED: the
// WAVES wavefronts of the workgroup fetch equal shares, and the sixteen-byte pieces go where weight_swizzle wants them.
// Rows that do not start at a multiple of sixteen bytes come four bytes a lane.
template <int NW, int WAVES, bool SHARED>
__device__ __forceinline__ void stage_key_rows(const char* src, uint32_t rbytes, char* dst, int wave, int lane)
{
    constexpr int kPieces = (NW * 128 * 2 + 1023) / 1024, kMine = SHARED ? (kPieces + WAVES - 1) / WAVES : kPieces;
    static_assert(!SHARED || kPieces % WAVES == 0 || kMine == 1, "equal shares, or a piece each for some wavefronts");
    const uint32_t bytes = (uint32_t)NW * rbytes;
    auto from = [=](uint32_t o) {
        return SHARED ? o ^ weight_swizzle((int)(o / rbytes), (int)rbytes / 16) * 16u : o;
    };
    const bool whole = ((uintptr_t)src & 15u) == 0;  // (wave-uniform)
#pragma unroll
    for (int k = 0; k < kMine; k++) {
        const int i = SHARED ? wave * kMine + k : k;
        if (__builtin_expect(whole, 1)) {
            const uint32_t o = (uint32_t)(i * 64 + lane) * 16u;
            if (o < bytes) dma16(src + from(o), dst + i * 1024);
        } else {
#pragma unroll 1
            for (int part = 0; part < 4; part++) {
                const uint32_t o = (uint32_t)(i * 1024 + part * 256 + lane * 4);
                if (o < bytes) dma4(src + from(o), dst + i * 1024 + part * 256);
            }
        }
    }
}

// Walks `nsubs` sub-chunks of one KV head with a two-deep pipeline: while sub-chunk n is being
// decompressed out of one LDS buffer, sub-chunk n+1 streams from HBM into the other.
//   tile_of(n)    : first tile of sub-chunk n
//   stage_w(n)    : issues the LDS-direct loads of the weights sub-chunk n needs (may be a no-op)
//   SHARED        : the weights of all sub-chunks are staged by the workgroup in stage_w(0): a barrier behind those loads
//   waddr_of(n)   : the lane's weights of sub-chunk n (RowSums::waddr / advance);  wgroup: bytes between four rows
template <bool SHARED, class Sums, class TileOf, class StageW, class WAddrOf>
__device__ __forceinline__ void walk_subs(int nsubs, TileOf tile_of, StageW stage_w, WAddrOf waddr_of, uint32_t wgroup,
                                          const uint64_t* bmk, const uint32_t* ixk, const char* nzk, char* my, int lane,
                                          Sums& sums)
{
    // stage_w must be free of lane-dependent branches: the coming scalar batch is live across it (see sub_issue_flat)
    if (nsubs <= 0) return;
    const uint32_t lbase = lds_addr(my);
    const RankConst rank = rank_const(lane);
    const RankTable table = rank_table(my + 2 * kSubBytes, lane);
    const uint32_t lane16 = (uint32_t)lane * 16u;
    const uint32_t off8 = (uint32_t)(lane & (kSubTiles - 1)) * 8u;
    const uint32_t off4 = (uint32_t)(lane & (kSubTiles - 1)) * 4u;
    size_t t_cur = tile_of(0), t_nxt = nsubs > 1 ? tile_of(1) : t_cur;
    // Where the values of the coming sub-chunk start and end (even and odd lanes), requested in front of the sub-chunk before
    // it, whose wait completes the load: by scalar loads, waited for in the middle of a sub-chunk, each of these had a round trip
    // to HBM of its own (70 %, 256 heads x 4096 tokens, eight blocks a wavefront, four rows: value product 34.7 -> 24.5 us, key
    // product 31.3 -> 29.2).
    const uint32_t bnd4 = (uint32_t)(lane & 1) * (kSubTiles * 4u);
    auto bounds = [&](size_t t) { return *reinterpret_cast<const uint32_t*>(reinterpret_cast<const char*>(ixk + t) + bnd4); };
    uint32_t bnd = bounds(t_nxt);
    // (the offsets may come back through a vector load; the statement below wants them in scalar registers)
    auto uni = [](uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); };
    uint32_t s_cur = uni(ixk[t_cur]);
    sub_issue_flat(nzk + (size_t)s_cur * 4u, sub_bytes(s_cur, uni(ixk[t_cur + kSubTiles])), lbase, lane16);
    stage_w(0);
    Touch touch = touch_sub_flat(bmk + t_cur, ixk + t_cur, off8, off4);
    if constexpr (SHARED) {
        wait_vm0_keep(touch);
        __syncthreads();
    }
    u32x16_t cur = load_bitmaps_scalar(bmk + t_cur);
    constexpr int G = kSubTiles / 8;
    for (int n = 0; n < nsubs; n++) {
        set_wave_priority_uniform(3u - ((uint32_t)n & 3u));  // falls from stage to stage (see set_wave_priority)
        wait_vm0_keep(touch);  // sub-chunk n (values, weights) has landed
        asm volatile("" : "+v"(bnd));  // (and the bounds of the coming one)
        // Buffer (n+1)&1 is refilled now.  Its last reader was sub-chunk n-1, and every LDS read of that sub-chunk
        // fed an MFMA issued before this point, so the reads have returned.
        __builtin_amdgcn_sched_barrier(0);
        const uint2 bits = touch.bm;
        table.put(touch.ix * 4u + (lbase + (uint32_t)(n & 1) * kSubBytes - s_cur * 4u));
        const uint64_t* bm_now = bmk + t_cur;
        if (n + 1 < nsubs) {
            t_cur = t_nxt;
            s_cur = (uint32_t)__builtin_amdgcn_readlane((int)bnd, 0);
            const uint32_t e_cur = (uint32_t)__builtin_amdgcn_readlane((int)bnd, 1);
            sub_issue_flat(nzk + (size_t)s_cur * 4u, sub_bytes(s_cur, e_cur), lbase + (uint32_t)((n + 1) & 1) * kSubBytes,
                           lane16);
            stage_w(n + 1);
            touch = touch_sub_flat(bmk + t_cur, ixk + t_cur, off8, off4);
            if (n + 2 < nsubs) {
                t_nxt = tile_of(n + 2);
                bnd = bounds(t_nxt);
            }
        }
        RankAddr at = rank_addresses(rank, bits, table.get());
        rank_settle(at);
        const uint32_t w = waddr_of(n);
        static_for<G>([&](auto gc) {
            constexpr int g = decltype(gc)::value;
            u32x16_t nxt;
            if constexpr (g + 1 < G)
                sums.template batch<true, g, (g + 1) * 64, 0, 0>(cur, nxt, bm_now, at, w, wgroup);
            else  // the first batch of the coming sub-chunk (of this one again after the last: loaded, never used)
                sums.template batch<true, g, 0, 0, 0>(cur, nxt, bmk + t_cur, at, w, wgroup);
            cur = nxt;
        });
        sums.stage_done();
        __builtin_amdgcn_sched_barrier(0);
    }
    wait_lgkm0();
}

}  // namespace mstf
