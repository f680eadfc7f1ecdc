// Expansion of bitmap tiles a whole tile per LDS read, for images of tiles at a fixed stride and up to eight weight rows: the
// quantised fused kernels and value products over many blocks (quant_device.hpp, StageRank).
//
// In rank_device.hpp a register of the address products holds the same half of two tiles, so that an exec mask is put
// together from two 32-bit pieces and the lane halves' sums have to be joined.  Here the rows of a product are the two halves
// of sixteen tiles - row 8 g + 4 P + j for half P of a tile - so that a register holds a tile whole, lane = element: one
// 64-bit reversal sets its exec mask, two products (three there) make the addresses of 32 tiles, and nothing is joined.
// A product sums over 64 bits: the elements of the row's own half in front of the column's position and at it (lanes 0 .. 31),
// and for the second half of a tile all of the first (lanes 32 .. 63; masked off for the first half).
// The bits are 4-bit floats and the sums 32-bit floats below the normal range, whose bits are the integer they hold: with the
// products' unit at an eighth of twice the smallest 32-bit float every bit adds 2 to the LDS byte address in C, all of it exact.  (Where the
// tiles' addresses differ - the fp16 format - C would be read from a table for 32 tiles instead of for 16 pairs, and the
// longer chain of these products costs the single wavefronts of small calls 2 %: those kernels keep the other layout.)
//
// A stage of 32 tiles is one statement on fixed registers.  Under exec masks, eight tiles a batch (whole_masked_stage); or, for
// tiles of up to 32 survivors, without any: all lanes read, those of elements that are not there from zeros in front of the
// tile's values, into the registers that held the addresses, and a batch is on its way while the one in front of it is multiplied
// (whole_stage).  Fused attention, 70 %, 256 heads x 4096 tokens / 48 x 2048 / 8 x 1024 and eight 2-bit decode steps of 128 heads x 60
// blocks + window, us: the statements batch by batch with the compiler's moves between them 46.9 / 16.4 / 15.3, 262; masked stages 45.7
// / 16.1 / 15.0, 262 (4 bits, 128 x 4096 34.7 -> 32.5); without masks 44.2 / 15.5 / 14.4, 255.  The vector unit stays the bound (74 % busy).
#pragma once
#include "rank_device.hpp"

namespace mstf {

typedef int i32x6_t __attribute__((ext_vector_type(6)));

// An element that is there has this much added to its address on top of its rank.  A tile of up to 32 values may so lie behind as
// many bytes of zeros in the image, which the lanes of the other elements read by their own rank: no exec mask, no register cleared.
constexpr int kWholeZeros = 80;

struct WholeRank {
    i32x6_t factor;     // B, 6-bit numbers (e3m2): number 8 r + i is bit 4 i + r of a half, element 31 - (4 i + r)
    uint32_t one;       // every fourth bit from bit 0 on; none in the lanes that add nothing to a tile's first half
};
// Row n of a product belongs to this tile of eight or to the one four further on (second product): the tiles of a register
// quadruple stand in the order 0, 2, 1, 3, in which pairs of registers hold what a 4x4x4 product takes (whole_stage).
__device__ __forceinline__ uint32_t whole_row(uint32_t t) { return (t & 1u) << 1 | (t >> 1 & 1u); }
__device__ __forceinline__ uint32_t whole_tile(int lane)
{
    const uint32_t n = (uint32_t)lane & 31u;
    return (n >> 3) * 8u + whole_row(n & 3u);
}
// A lane's words of the bitmaps: lanes 0 .. 31 the half of a tile whose row they are, lanes 32 .. 63 the first half of that tile
// (elements 0 .. 31 are the upper word); of the first product's tile and of the second's.  Fetched as they are wanted: with a
// whole bitmap per lane the halves changed hands between lanes n and n ^ 4 by ten vector instructions a stage.
__device__ __forceinline__ uint32_t whole_bits_at(int lane)
{
    const bool upper = lane >= 32 || (lane & 4) == 0;
    return whole_tile(lane) * 8u + (upper ? 4u : 0u);
}
__device__ __forceinline__ uint2 whole_bits_load(const uint64_t* bm, uint32_t at)
{
    asm volatile("" : "+v"(at));  // (one register beside a scalar base, and no address per place)
    const char* p = reinterpret_cast<const char*>(bm) + at;
    return make_uint2(*reinterpret_cast<const uint32_t*>(p), *reinterpret_cast<const uint32_t*>(p + 32));
}
// The bitmap of (wave-uniform) tile t out of the lanes' words.
__device__ __forceinline__ uint64_t whole_bitmap(uint2 bits, uint32_t t)
{
    const int n = (int)((t >> 3) * 8u + whole_row(t & 3u));
    uint32_t hi, lo;
    if (t & 4u) {
        hi = (uint32_t)__builtin_amdgcn_readlane((int)bits.y, n), lo = (uint32_t)__builtin_amdgcn_readlane((int)bits.y, n + 4);
        asm volatile("" : "+s"(hi), "+s"(lo));  // (a scalar branch: both words of either product are two more vector instructions)
    } else {
        hi = (uint32_t)__builtin_amdgcn_readlane((int)bits.x, n), lo = (uint32_t)__builtin_amdgcn_readlane((int)bits.x, n + 4);
        asm volatile("" : "+s"(hi), "+s"(lo));
    }
    return u64_of(lo, hi);
}
// The words with the tiles of the mask as empty ones.
__device__ __forceinline__ uint2 whole_without(uint2 bits, uint32_t tiles, int lane)
{
    asm volatile("" : "+v"(lane));
    const uint32_t t = whole_tile(lane);
    return make_uint2(bits.x & (uint32_t)__builtin_amdgcn_sbfe((int)~tiles, t, 1u),
                      bits.y & (uint32_t)__builtin_amdgcn_sbfe((int)~tiles, t + 4u, 1u));
}
__device__ __forceinline__ WholeRank whole_rank(int lane)
{
    WholeRank c;
    const int n = lane & 31, all = lane >> 5;  // column (position); lanes 32 .. 63: the whole first half counts
    const bool second = (lane & 4) != 0;       // row n belongs to a tile's second half
    uint32_t f[6] = {0u, 0u, 0u, 0u, 0u, 0u};
#pragma unroll
    for (int k = 0; k < 32; k++) {
        const int r = k / 8, e = 31 - (4 * (k % 8) + r);
        // Two bytes are worth 0.125: a bit of registers 0 and 1 is 0.5 there, times 0.25, of the others 2, times 0.0625; and the
        // element itself, kWholeZeros bytes, 10 and 2.5.
        static_assert(kWholeZeros == 80, "10 x 0.5 = 2.5 x 2 = 40 x 0.125");
        const uint32_t before = r < 2 ? 4u : 1u, itself = r < 2 ? 25u : 17u;  // 0.25, 0.0625, 10, 2.5 as 6-bit numbers
        const uint32_t v = all || e < n ? before : (e == n ? itself : 0u);
        const int at = 6 * k, w = at / 32, b = at % 32;
        f[w] |= v << b;
        if (b > 26) f[w + 1] |= v >> (32 - b);
    }
    c.factor = i32x6_t{(int)f[0], (int)f[1], (int)f[2], (int)f[3], (int)f[4], (int)f[5]};
    c.one = all && !second ? 0u : 0x11111111u;
    return c;
}
constexpr int kWholeScales = (127 - 73) | (127 - 72) << 8;  // of A and B: together 2^-145
// The base for an image without zeros in front of a tile's values (an integer as a 32-bit float below the normal range).
__device__ __forceinline__ uint32_t whole_base(uint32_t image)
{
    return image >= (uint32_t)kWholeZeros ? image - (uint32_t)kWholeZeros : 0x80000000u | ((uint32_t)kWholeZeros - image);
}
// A stage of tiles of up to 32 survivors behind zeros (kWholeZeros; the tiles IS bytes apart in the image): address products, a
// gather into the register of each address, all lanes active, and the 4x4x4 products, in one statement on fixed registers.  Eight
// gathers are in flight while the products of the eight in front of them run, and nothing is scalar: under exec masks, eight tiles
// at a time, a wavefront waited for its own reads and for the masks of the coming tiles.
// A gather into an upper half clears the lower one, where the tile's address was: so it is with SRAM-ECC on, for which alone this library
// is built (build.py).  With the half kept, address bits would be multiplied by a weight.
// v[96:111], v[112:127]: addresses, then values, of the two products; v87, v[88:95]: the products' scales and rows, then the weights of two batches.
//   wa : LDS address of w[lane & 3][0] of the first tile of the stage (up to four rows)
#define MSTF_SG(H, R, T) "ds_read_u16" H " v" R ", v" R " offset:%[is]*" T "\n\t"
#define MSTF_SQUAD(R0, R1, R2, R3, T0, T1, T2, T3)                                                                  \
    MSTF_SG("", R0, T0) MSTF_SG("", R1, T2) MSTF_SG("_d16_hi", R2, T1) MSTF_SG("_d16_hi", R3, T3)
#define MSTF_SG0 MSTF_SQUAD("96", "97", "98", "99", "0", "1", "2", "3") MSTF_SQUAD("112", "113", "114", "115", "4", "5", "6", "7")
#define MSTF_SG1 \
    MSTF_SQUAD("100", "101", "102", "103", "8", "9", "10", "11") MSTF_SQUAD("116", "117", "118", "119", "12", "13", "14", "15")
#define MSTF_SG2 \
    MSTF_SQUAD("104", "105", "106", "107", "16", "17", "18", "19") MSTF_SQUAD("120", "121", "122", "123", "20", "21", "22", "23")
#define MSTF_SG3 \
    MSTF_SQUAD("108", "109", "110", "111", "24", "25", "26", "27") MSTF_SQUAD("124", "125", "126", "127", "28", "29", "30", "31")
#define MSTF_SBASE                                                                                                  \
    "v_mov_b64 v[112:113], %[base]\n\tv_mov_b64 v[114:115], %[base]\n\tv_mov_b64 v[116:117], %[base]\n\t"            \
    "v_mov_b64 v[118:119], %[base]\n\tv_mov_b64 v[120:121], %[base]\n\tv_mov_b64 v[122:123], %[base]\n\t"            \
    "v_mov_b64 v[124:125], %[base]\n\tv_mov_b64 v[126:127], %[base]\n\t"
#define MSTF_SROWS(A, B, C, D, X)                                                                                    \
    "v_lshrrev_b32 " D ", 1, %[" X "]\n\tv_and_b32 " A ", %[" X "], %[one]\n\tv_and_b32 " B ", " D ", %[one]\n\t"           \
    "v_and_b32 " C ", %[" X "], v96\n\tv_and_b32 " D ", " D ", v96\n\t"  // bits 0, 2 where they stand, the others one down
#define MSTF_SADDR(D, X, S)                                                                                         \
    "v_mfma_scale_f32_32x32x64_f8f6f4 " D ", " X ", %[f], v[112:127], " S ", " S " op_sel:[0,1,0] op_sel_hi:[0,0,0] cbsz:4 "  \
    "blgp:3\n\t"
#define MSTF_SADDRS                                                                                                 \
    "v_lshlrev_b32 v96, 2, %[one]\n\t" MSTF_SROWS("v88", "v89", "v90", "v91", "x") MSTF_SROWS("v92", "v93", "v94", "v95", "y")             \
    "v_mov_b32 v87, %[sc]\n\t" MSTF_SBASE "s_nop 1\n\t"                                                              \
    MSTF_SADDR("v[96:111]", "v[88:91]", "v87") MSTF_SADDR("v[112:127]", "v[92:95]", "v87") "s_nop 15\n\t"
#define MSTF_SW(W, R, OFF) "ds_read_b128 " R ", %[" W "] offset:" OFF "\n\t"
#define MSTF_SM(ACC, A, W) "v_mfma_f32_4x4x4_16b_f16 %[" ACC "], " A ", " W ", %[" ACC "]\n\t"
#define MSTF_SM0(ACC, A, W) "v_mfma_f32_4x4x4_16b_f16 %[" ACC "], " A ", " W ", 0\n\t"
#define MSTF_SONE0(A0, A1, B0, B1, W0, W1)                                                                          \
    MSTF_SM0("p0", A0, W0) MSTF_SM0("p1", B0, W1) MSTF_SM("p0", A1, W0) "s_nop 0\n\t" MSTF_SM("p1", B1, W1)
#define MSTF_SONE(A0, A1, B0, B1, W0, W1)                                                                           \
    MSTF_SM("p0", A0, W0) MSTF_SM("p1", B0, W1) MSTF_SM("p0", A1, W0) "s_nop 0\n\t" MSTF_SM("p1", B1, W1)
#define MSTF_SREGS                                                                                                  \
    "v87", "v88", "v89", "v90", "v91", "v92", "v93", "v94", "v95", "v96", "v97", "v98", "v99", "v100", "v101", "v102", "v103", "v104", "v105", "v106", "v107", "v108", "v109", "v110", "v111", "v112",  \
        "v113", "v114", "v115", "v116", "v117", "v118", "v119", "v120", "v121", "v122", "v123", "v124", "v125", "v126", "v127"
template <int IS, bool FIRST>
__device__ __forceinline__ void whole_stage(const WholeRank& c, uint2 bits, uint32_t image, uint32_t wa, f4_t (&acc)[2])
{
    const uint64_t base = (uint64_t)image << 32 | image;
#define MSTF_SSTAGE(M0)                                                                                             \
    MSTF_SADDRS MSTF_SW("wa", "v[88:91]", "0") MSTF_SG0 MSTF_SW("wa", "v[92:95]", "16")                                \
    MSTF_SG1 "s_waitcnt lgkmcnt(9)\n\t" M0("v[96:97]", "v[98:99]", "v[112:113]", "v[114:115]", "v[88:89]", "v[90:91]")  \
    MSTF_SW("wa", "v[88:91]", "32") MSTF_SG2 "s_waitcnt lgkmcnt(9)\n\t"                                               \
    MSTF_SONE("v[100:101]", "v[102:103]", "v[116:117]", "v[118:119]", "v[92:93]", "v[94:95]")                           \
    MSTF_SW("wa", "v[92:95]", "48") MSTF_SG3 "s_waitcnt lgkmcnt(9)\n\t"                                               \
    MSTF_SONE("v[104:105]", "v[106:107]", "v[120:121]", "v[122:123]", "v[88:89]", "v[90:91]") "s_waitcnt lgkmcnt(0)\n\t" \
    MSTF_SONE("v[108:109]", "v[110:111]", "v[124:125]", "v[126:127]", "v[92:93]", "v[94:95]") "s_nop 4"
#define MSTF_SIN                                                                                                    \
    [x] "v"(bits.x), [y] "v"(bits.y), [one] "v"(c.one), [f] "v"(c.factor), [base] "s"(base),         \
        [sc] "i"(kWholeScales), [wa] "v"(wa), [is] "i"(IS)
    if constexpr (FIRST)
        asm volatile(MSTF_SSTAGE(MSTF_SONE0) : [p0] "=&v"(acc[0]), [p1] "=&v"(acc[1]) : MSTF_SIN : MSTF_SREGS, "memory");
    else
        asm volatile(MSTF_SSTAGE(MSTF_SONE) : [p0] "+v"(acc[0]), [p1] "+v"(acc[1]) : MSTF_SIN : MSTF_SREGS, "memory");
}

// The same for tiles of any number of survivors, without zeros in the image, under the tiles' masks: eight tiles at a time, each
// read under its bitmap into cleared registers, the bitmaps from scalar loads one batch ahead.  bm: of the first tile.
// v[96:127]: addresses; v[88:95]: values; v[84:87] (and v[80:83], eight rows): weights; s[64:79], s[80:95]: bitmaps.
//   wa, wb : LDS address of w[lane & 3][0] of the first tile of the stage, for the accumulators 0 .. 3 and (NM = 2) 4 .. 7
#define MSTF_XG(H, R, A, M, T) "s_brev_b64 exec, s[" M "]\n\tds_read_u16" H " " R ", " A " offset:%[is]*" T "\n\t"
#define MSTF_XCLEAR "v_mov_b64 v[88:89], 0\n\tv_mov_b64 v[90:91], 0\n\tv_mov_b64 v[92:93], 0\n\tv_mov_b64 v[94:95], 0\n\t"
#define MSTF_XGATHER(M0, M1, M2, M3, M4, M5, M6, M7, A0, A1, A2, A3, B0, B1, B2, B3, T0, T1, T2, T3, T4, T5, T6, T7)  \
    MSTF_XG("", "v88", A0, M0, T0) MSTF_XG("_d16_hi", "v90", A2, M1, T1) MSTF_XG("", "v89", A1, M2, T2)                \
    MSTF_XG("_d16_hi", "v91", A3, M3, T3) MSTF_XG("", "v92", B0, M4, T4) MSTF_XG("_d16_hi", "v94", B2, M5, T5)         \
    MSTF_XG("", "v93", B1, M6, T6) MSTF_XG("_d16_hi", "v95", B3, M7, T7) "s_mov_b64 exec, -1\n\t"
#define MSTF_XG_EVEN(...) MSTF_XGATHER("64:65", "66:67", "68:69", "70:71", "72:73", "74:75", "76:77", "78:79", __VA_ARGS__)
#define MSTF_XG_ODD(...) MSTF_XGATHER("80:81", "82:83", "84:85", "86:87", "88:89", "90:91", "92:93", "94:95", __VA_ARGS__)
#define MSTF_XG0 MSTF_XG_EVEN("v96", "v97", "v98", "v99", "v112", "v113", "v114", "v115", "0", "1", "2", "3", "4", "5", "6", "7")
#define MSTF_XG1 \
    MSTF_XG_ODD("v100", "v101", "v102", "v103", "v116", "v117", "v118", "v119", "8", "9", "10", "11", "12", "13", "14", "15")
#define MSTF_XG2 \
    MSTF_XG_EVEN("v104", "v105", "v106", "v107", "v120", "v121", "v122", "v123", "16", "17", "18", "19", "20", "21", "22", "23")
#define MSTF_XG3 \
    MSTF_XG_ODD("v108", "v109", "v110", "v111", "v124", "v125", "v126", "v127", "24", "25", "26", "27", "28", "29", "30", "31")
#define MSTF_XMASKS(S, OFF) "s_load_dwordx16 s[" S "], %[bm], " OFF "\n\t"
#define MSTF_XONE                                                                                                   \
    "s_waitcnt lgkmcnt(4)\n\t" MSTF_SM("p0", "v[88:89]", "v[84:85]") "s_waitcnt lgkmcnt(0)\n\t"                       \
    MSTF_SM("p1", "v[92:93]", "v[86:87]") MSTF_SM("p0", "v[90:91]", "v[84:85]") "s_nop 0\n\t"                         \
    MSTF_SM("p1", "v[94:95]", "v[86:87]") "s_nop 4\n\t"
// (eight rows: the pairs merged first, half the products)
#define MSTF_SOR(D, S) "v_or_b32 " D ", " D ", " S "\n\t"
#define MSTF_XTWO                                                                                                   \
    "s_waitcnt lgkmcnt(4)\n\t" MSTF_SOR("v88", "v90") MSTF_SOR("v89", "v91") "s_nop 1\n\t"                           \
    MSTF_SM("p0", "v[88:89]", "v[84:85]") MSTF_SM("q0", "v[88:89]", "v[80:81]") "s_waitcnt lgkmcnt(0)\n\t"           \
    MSTF_SOR("v92", "v94") MSTF_SOR("v93", "v95") "s_nop 1\n\t" MSTF_SM("p1", "v[92:93]", "v[86:87]")                \
    MSTF_SM("q1", "v[92:93]", "v[82:83]") "s_nop 4\n\t"
#define MSTF_XW1(OFF) MSTF_XCLEAR MSTF_SW("wa", "v[84:87]", OFF)
#define MSTF_XW2(OFF) MSTF_XCLEAR MSTF_SW("wa", "v[84:87]", OFF) MSTF_SW("wb", "v[80:83]", OFF)
#define MSTF_XSTAGE(W, M)                                                                                           \
    MSTF_XMASKS("64:79", "0") MSTF_SADDRS "s_waitcnt lgkmcnt(0)\n\t" MSTF_XMASKS("80:95", "64") W("0") MSTF_XG0 M        \
    MSTF_XMASKS("64:79", "128") W("16") MSTF_XG1 M MSTF_XMASKS("80:95", "192") W("32") MSTF_XG2 M W("48") MSTF_XG3 M
#define MSTF_XSREGS                                                                                                 \
    "s64", "s65", "s66", "s67", "s68", "s69", "s70", "s71", "s72", "s73", "s74", "s75", "s76", "s77", "s78", "s79", "s80", "s81", \
        "s82", "s83", "s84", "s85", "s86", "s87", "s88", "s89", "s90", "s91", "s92", "s93", "s94", "s95"
template <int NM, int IS>
__device__ __forceinline__ void whole_masked_stage(const WholeRank& c, const uint64_t* bm, uint2 bits, uint32_t image, uint32_t wa,
                                                   uint32_t wb, f4_t (&acc)[NM][2])
{
    static_assert(NM == 1 || NM == 2, "four or eight accumulators");
    const uint64_t base = u64_of(whole_base(image), whole_base(image));
    if constexpr (NM == 1)
        asm volatile(MSTF_XSTAGE(MSTF_XW1, MSTF_XONE)
                     : [p0] "+v"(acc[0][0]), [p1] "+v"(acc[0][1])
                     : MSTF_SIN, [bm] "s"(bm)
                     : MSTF_SREGS, MSTF_XSREGS, "v84", "v85", "v86", "memory");
    else
        asm volatile(MSTF_XSTAGE(MSTF_XW2, MSTF_XTWO)
                     : [p0] "+v"(acc[0][0]), [p1] "+v"(acc[0][1]), [q0] "+v"(acc[1][0]), [q1] "+v"(acc[1][1])
                     : MSTF_SIN, [wb] "v"(wb), [bm] "s"(bm)
                     : MSTF_SREGS, MSTF_XSREGS, "v80", "v81", "v82", "v83", "v84", "v85", "v86", "memory");
}

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
