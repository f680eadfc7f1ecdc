// Key / value SpMV over the quantised bitmap format, with dequantisation fused into the decompression.
//
// Same work decomposition, LDS-direct staging and MFMA accumulation as the fp16 kernels (spmv.hip); what
// differs is how a staged run of 32 tiles becomes fp16 values:
//   1. the run's packed words (contiguous in `packed`) and its per-tile metadata (word offsets, scales,
//      zero-points) stream HBM -> LDS one stage ahead;
//   2. dequantisation happens in the packed domain: one lane per packed word unpacks its 16 / 8 / 4 codes
//      and writes the fp16 values, in rank order, into a fixed-stride tile image in LDS, so the cost is per
//      non-zero word, not per dense position;
//   3. the image is expanded like the fp16 format (bitmap rank -> LDS gather -> MFMA; rank_whole.hpp, rank_device.hpp),
//      with the tile base a constant instead of idx.
// Dequantised value = fp16( (q - zero) * scale ).  For |zero| <= 1024 this is computed with packed fp16
// arithmetic and is the same number the reference's fp32 (dequant_mode 0) and fp16 (dequant_mode 1)
// sequences give: 0x6400 | q is the fp16 number 1024 + q, subtracting 1024 + zero is exact, and the one
// remaining multiplication by scale rounds the exact product once.  Tiles with a larger zero-point take
// the literal per-mode arithmetic.
#include "quant_device.hpp"
#include "spmv_common.hpp"

namespace mstf {

#pragma clang fp contract(off)

// Pointers of one KV-head-agnostic quantised cache.  `off_dma`, `scales`, `zeros`, `packed` feed LDS-direct
// loads; `off` is the same array as `off_dma`, kept as a separate, never-escaping pointer so that the stage
// boundaries are still fetched with scalar loads.
struct QCache {
    const uint64_t* bmp;
    const uint32_t* off;
    const uint32_t* off_dma;
    const uint16_t* scales;
    const uint16_t* zeros;
    const uint32_t* packed;
};

// Walks `nsubs` stages of 32 tiles with a two-deep pipeline (see walk_subs).  Tile indices are global
// (KV head included): tile_off / scales / zeros / bmp are flat over [Bkv, T].
template <bool SHARED, int BIT, bool G32, class Rank, class TileOf, class StageW, class WAddrOf>
__device__ __forceinline__ void walk_subs_q(int nsubs, TileOf tile_of, StageW stage_w, WAddrOf waddr_of, uint32_t wgroup,
                                            const QCache& c, char* my, int lane, int mode, typename Rank::Sums& sums)
{
    using F = QFmt<BIT>;
    if (nsubs <= 0) return;
    const uint32_t lbase = lds_addr(my);
    char* wordbuf = my + kImgBytes;
    char* metabuf = wordbuf + 2 * F::kWordBuf;

    // words of the stage starting at tile t: [tile_off[t], tile_off[t + 31] + words of tile t + 31)
    auto bounds = [&](size_t t, uint32_t& s, uint32_t& e) {
        s = c.off[t];
        const uint32_t cnt = (uint32_t)__builtin_popcountll(c.bmp[t + kSubTiles - 1]);
        e = c.off[t + kSubTiles - 1] + ((cnt + (uint32_t)F::kCap - 1u) >> F::kCapShift);
    };
    constexpr int kMetaBytes = meta_bytes<G32>();
    const MetaLanes meta = meta_lanes<G32>(c.off_dma, c.scales, c.zeros, c.bmp, lane);
    const uint32_t lane4 = (uint32_t)lane * 4u;
    const uint32_t bits_at = Rank::bits_at(lane);
    const uint32_t wordbuf_lds = lds_addr(wordbuf);
    Rank rank(lds_addr(metabuf), wordbuf_lds, lbase, lane);
    auto uni = [](uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); };
    // (no lane-dependent branches in the word and metadata loads: exec set by hand, clamped touch address)
    auto issue = [&](int n, size_t t, uint32_t s, uint32_t e) {
        uint32_t nw = uni(e) - uni(s);
        nw = nw > (uint32_t)F::kWordsMax ? (uint32_t)F::kWordsMax : nw;  // never true for a well-formed cache
        words_issue_flat<F::kWordsMax / 64>(c.packed + uni(s), nw, wordbuf_lds + (uint32_t)(n & 1) * F::kWordBuf,
                                            (uint32_t)lane, lane4);
        // metadata: lanes 0..31 the word offsets, 32..47 the scales, 48..63 the zero-points (two per lane); two loads
        // when a tile has two (scale, zero) pairs
        meta_issue<G32>(meta, (uint32_t)t, metabuf + (n & 1) * kMetaBytes);
        stage_w(n);
        // the stage's bitmaps (and the scalar loads of the expansion find them in L2)
        return Rank::bits_load(c.bmp + t, bits_at);
    };

    size_t t_cur = tile_of(0), t_nxt = nsubs > 1 ? tile_of(1) : t_cur;
    // The bounds of the coming stage: even lanes the first tile's offset, odd ones the last tile's and, with its bitmap, where
    // its words end.  Requested in front of the stage before it, whose wait completes the loads (see walk_subs).
    const uint32_t bnd4 = (uint32_t)(lane & 1) * ((kSubTiles - 1) * 4u);
    struct Raw {
        uint32_t off;
        uint2 last;
    };
    auto bounds_of = [&](size_t t) {
        Raw r;
        r.off = *reinterpret_cast<const uint32_t*>(reinterpret_cast<const char*>(c.off + t) + bnd4);
        r.last = *reinterpret_cast<const uint2*>(c.bmp + t + kSubTiles - 1);
        return r;
    };
    Raw bnd = bounds_of(t_nxt);
    uint32_t s_cur, e_cur;
    bounds(t_cur, s_cur, e_cur);
    uint2 touch = issue(0, t_cur, s_cur, e_cur);
    if constexpr (SHARED) {
        asm volatile("s_waitcnt vmcnt(0)" : "+v"(touch.x), "+v"(touch.y)::"memory");
        __syncthreads();
    }
    for (int n = 0; n < nsubs; n++) {
        set_wave_priority_uniform(3u - ((uint32_t)n & 3u));  // falls from stage to stage (see set_wave_priority)
        // stage n has landed, and the bounds of the coming one
        asm volatile("s_waitcnt vmcnt(0)"
                     : "+v"(touch.x), "+v"(touch.y), "+v"(bnd.off), "+v"(bnd.last.x), "+v"(bnd.last.y)::"memory");
        const uint2 bits = touch;
        const size_t t_now = t_cur;
        const uint32_t s_now = s_cur, e_now = e_cur;
        if (n + 1 < nsubs) {
            t_cur = t_nxt;
            const uint32_t words = ((uint32_t)__builtin_popcount(bnd.last.x) + (uint32_t)__builtin_popcount(bnd.last.y) +
                                    (uint32_t)F::kCap - 1u) >> F::kCapShift;
            s_cur = (uint32_t)__builtin_amdgcn_readlane((int)bnd.off, 0);
            e_cur = (uint32_t)__builtin_amdgcn_readlane((int)(bnd.off + words), 1);
            touch = issue(n + 1, t_cur, s_cur, e_cur);
            if (n + 2 < nsubs) {
                t_nxt = tile_of(n + 2);
                bnd = bounds_of(t_nxt);
            }
        }
        const StageAt here = {lds_addr(metabuf), wordbuf_lds, (uint32_t)(n & 1) * kMetaBytes, (uint32_t)(n & 1) * F::kWordBuf, s_now, e_now};
        rank.stage(here, c.bmp + t_now, bits, waddr_of(n), wgroup, sums, lane, mode);
        wait_lgkm0();  // every read of the image and of the staged buffers is done before they are rewritten
    }
}

// ------------------------------------------------------------------------------- key
// One wavefront per (KV head, token block); see key_spmv_kernel (more than eight rows are shared by the workgroup, whose
// wavefronts then work on one head, or, SHARE, on one block: see kKeyShareQuant).
template <int NW, int BIT, bool G32>
constexpr int key_quant_lds()
{
    constexpr int rows = RowSums<NW>::kRows * 128 * 2;
    return 4 * q_lds_bytes<BIT, G32>() + (RowSums<NW>::kWide ? rows : 4 * rows);
}
template <int NW, int BIT, bool G32, bool SHARE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(resident_waves(key_quant_lds<NW, BIT, G32>(), 4)))) void key_spmv_quant_kernel(
    const uint64_t* __restrict__ bmp, const uint32_t* packed, const uint32_t* __restrict__ tile_off,
    const uint32_t* tile_off_dma, const uint16_t* scales, const uint16_t* zeros, const _Float16* Bm,
    _Float16* __restrict__ C, int Lc, int D, int nblk, int ntasks, int rows_per_kv, int row0, int mode)
{
    using Rank = StageRank<NW, BIT, G32, true>;
    using Sums = typename Rank::Sums;
    constexpr bool kShared = Sums::kWide;
    constexpr int kMaxD = 128;
    constexpr int kQ = q_lds_bytes<BIT, G32>();
    constexpr int kRowsLds = Sums::kRows * kMaxD * 2;
    constexpr int kWaveLds = kQ + (kShared ? 0 : kRowsLds);
    __shared__ __attribute__((aligned(256))) char lds[key_quant_lds<NW, BIT, G32>()];
    const int lane = lane_id();
    const int wave = wave_id();
    const int quads = (nblk + 3) / 4;  // workgroups of a head when they may not span two
    const int nwg = SHARE ? ntasks : (kShared ? ntasks / nblk * quads : (ntasks + 3) / 4);
    static_assert(!SHARE || (kShared && kWaveLds >= kParkShares), "rows and sums of the workgroup");
    // neighbouring token blocks on the same XCD: their packed words share cache lines
    const int wg = xcd_contiguous((int)blockIdx.x, nwg);
    if (wg >= nwg) return;  // (the whole workgroup: no barrier is left waiting)
    const int task = SHARE ? wg : wg * 4 + wave;
    if (!kShared && task >= ntasks) return;
    const int kv = kShared && !SHARE ? wg / quads : task / nblk;
    const int tb = kShared && !SHARE ? (wg - kv * quads) * 4 + wave : task - kv * nblk;
    const int first = SHARE ? wave : 0;  // channel stage
    const size_t T = (size_t)Lc * D / 64;
    const QCache c = {bmp, tile_off, tile_off_dma, scales, zeros, packed};
    const char* wsrc = reinterpret_cast<const char*>(Bm + ((size_t)kv * rows_per_kv + row0) * D);
    char* my = lds + (kShared ? kRowsLds : 0) + wave * kWaveLds;
    char* wl = kShared ? lds : my + kQ;             // the rows; what lies behind row NW - 1 stays unwritten

    Sums sums;
    sums.clear();
    const size_t tile0 = (size_t)kv * T + (size_t)tb * D + (size_t)first * kSubTiles;
    const uint32_t rbytes = (uint32_t)D * 2u;
    const uint32_t wrow = Sums::waddr(lds_addr(wl), rbytes, lane);
    auto stage_rows = [=](int n) {
        if (n != 0) return;  // the query rows are staged once per task
        stage_key_rows<NW, 4, kShared>(wsrc, rbytes, wl, wave, lane);
    };
    if (kShared && !SHARE && tb >= nblk) {  // (wave-uniform) no block left, but a share of the rows
        stage_rows(0);
        wait_vm0();
        __syncthreads();
        return;
    }
    walk_subs_q<kShared, BIT, G32, Rank>(
        SHARE ? 1 : D / kSubTiles, [=](int n) { return tile0 + (size_t)n * kSubTiles; }, stage_rows,
        [=](int n) { return Sums::advance(wrow, (uint32_t)(first + n) * kSubTiles * 2u); }, (uint32_t)D * 8u, c, my, lane, mode, sums);
    _Float16* out = C + ((size_t)kv * rows_per_kv + row0) * Lc + (size_t)tb * 64;
    if constexpr (SHARE) {
        store_rows_shared(sums, lds + kRowsLds, kWaveLds, lds, out, (size_t)Lc, wave, lane);
    } else if constexpr (Sums::kWide) {
        store_rows_wide<NW>(sums, my, out, (size_t)Lc, lane);
    } else {
        sums.each4(lane, [=](int row, int pos, const f4_t& v) {
            *reinterpret_cast<h4_t*>(out + (size_t)row * Lc + pos) = round_h4(v);
        });
    }
}

// ------------------------------------------------------------------------------- value
// grid = xcd_grid(token splits x D/64 halves x KV heads), halves fastest in the logical index: the two halves of a
// token range read the same weights and interleaved cache lines, so they run on the same XCD; see value_spmv_kernel.
template <int NW, int BIT, bool G32>
constexpr int value_quant_wave_lds()
{
    // the rows start at a multiple of their length (64 bytes); the per-wave sums are parked in the room at the end
    constexpr int need = ((q_lds_bytes<BIT, G32>() + 63) & ~63) + 2 * RowSums<NW>::kRows * kSubTiles * 2;
    return need > NW * 256 ? need : NW * 256;
}
template <int NW, int WAVES, int BIT, bool G32, bool WHOLE>
__global__ __launch_bounds__(WAVES * 64) __attribute__((amdgpu_waves_per_eu(resident_waves(WAVES * value_quant_wave_lds<NW, BIT, G32>(), WAVES)))) void value_spmv_quant_kernel(
    const uint64_t* __restrict__ bmp, const uint32_t* packed, const uint32_t* __restrict__ tile_off,
    const uint32_t* tile_off_dma, const uint16_t* scales, const uint16_t* zeros, const _Float16* P,
    _Float16* __restrict__ C, float* __restrict__ part, int Lc, int D, int nblk, int nbpw, int nsplit, int rows_per_kv,
    int row0, int mode, int nwg, uint32_t per_split)
{
    using Rank = StageRank<NW, BIT, G32, !WHOLE>;
    using Sums = typename Rank::Sums;
    static_assert(Sums::kRows == RowSums<NW>::kRows, "LDS of a wavefront");
    constexpr int kWRow = kSubTiles * 2;
    constexpr int kWBuf = Sums::kRows * kWRow;
    constexpr int kQ = (q_lds_bytes<BIT, G32>() + 63) & ~63;
    constexpr int kWaveLds = value_quant_wave_lds<NW, BIT, G32>();
    __shared__ __attribute__((aligned(64))) char lds[WAVES][kWaveLds];
    const int lane = lane_id();
    const int wave = wave_id();
    const int nhalf = D / 64;
    const int logical = xcd_contiguous((int)blockIdx.x, nwg);
    if (logical >= nwg) return;  // (the whole workgroup: no barrier is left waiting)
    const ValueIndex at = value_index(logical, nhalf, nsplit, per_split);
    const int half = at.half, split = at.split, kv = at.kv;
    const size_t T = (size_t)Lc * D / 64;
    const QCache c = {bmp, tile_off, tile_off_dma, scales, zeros, packed};
    const _Float16* wk = P + ((size_t)kv * rows_per_kv + row0) * Lc;
    char* my = lds[wave];
    char* wl = my + kQ;

    Sums sums;
    sums.clear();

    const int first = (split * WAVES + wave) * nbpw;
    int last = first + nbpw;
    if (last > nblk) last = nblk;
    constexpr int subs_per_blk = 64 / kSubTiles;
    const uint32_t wrow = Sums::waddr(lds_addr(wl), kWRow, lane);
    const size_t thead = (size_t)kv * T + (size_t)half * 64;
    walk_subs_q<false, BIT, G32, Rank>(
        (last - first) * subs_per_blk,
        [=](int n) { return thead + (size_t)(first + n / subs_per_blk) * D + (size_t)(n % subs_per_blk) * kSubTiles; },
        [=](int n) {
            const size_t tok0 = (size_t)(first + n / subs_per_blk) * 64 + (size_t)(n % subs_per_blk) * kSubTiles;
            if constexpr (Sums::kWide) {
                stage_rows_wide<NW>(wk + tok0, (size_t)Lc, wl + (n & 1) * kWBuf, lane);
                return;
            }
            constexpr int kDwPerRow = kSubTiles / 2, kRowsPer = 64 / kDwPerRow;
#pragma unroll
            for (int i = 0; i < (NW + kRowsPer - 1) / kRowsPer; i++) {
                const int row = kRowsPer * i + lane / kDwPerRow;
                const int dw = lane % kDwPerRow;
                if (row < NW) dma4(wk + (size_t)row * Lc + tok0 + 2 * dw, wl + (n & 1) * kWBuf + i * 256);
            }
        },
        [=](int n) { return wrow + (uint32_t)(n & 1) * kWBuf; }, 4u * kWRow, c, my, lane, mode, sums);
    // workgroup reduction: every wavefront parks its sums [accumulator][channel] in its own LDS area
    __syncthreads();
    float* mine = reinterpret_cast<float*>(my);
    // (the four-float pieces of a row at piece ^ row, so that lanes of different rows do not all write to one bank)
    sums.each4(lane, [=](int row, int pos, const f4_t& v) {
        *reinterpret_cast<f4_t*>(mine + row * 64 + (((pos >> 2) ^ (row & 15)) << 2)) = v;
    });
    __syncthreads();
    for (int o = (int)threadIdx.x; o < NW * 64; o += WAVES * 64) {
        const int n = o >> 6, ch = o & 63;
        float s = 0.f;
#pragma unroll
        for (int wv = 0; wv < WAVES; wv++)
            s += reinterpret_cast<const float*>(lds[wv])[(n << 6) + (((ch >> 2) ^ (n & 15)) << 2) + (ch & 3)];
        const size_t row = (size_t)kv * rows_per_kv + row0 + n;
        if (nsplit == 1)
            C[row * D + (size_t)half * 64 + ch] = (_Float16)s;
        else
            part[(row * nsplit + split) * D + (size_t)half * 64 + ch] = s;
    }
}

// ------------------------------------------------------------------------------- host
static int check_quant_spmv(const void* bmp, const void* packed, const void* tile_off, const void* scales,
                            const void* zeros, const void* Bm, const void* C, int tokens, int head_dim, int Bq,
                            int groups, int n_rows, int bit, int capacity, int dequant_mode)
{
    if (!bmp || !packed || !tile_off || !scales || !zeros || !Bm || !C) return MSTF_EINVAL;
    if (tokens <= 0 || head_dim <= 0 || Bq <= 0 || groups <= 0 || n_rows <= 0 || Bq % groups != 0) return MSTF_EINVAL;
    if (dequant_mode != 0 && dequant_mode != 1) return MSTF_EINVAL;
    if (bit != 2 && bit != 4 && bit != 8) return MSTF_EUNSUPPORTED;
    if (capacity != 32 / bit) return MSTF_EINVAL;
    if (tokens % 64 != 0 || head_dim % 64 != 0 || head_dim > 128) return MSTF_EUNSUPPORTED;
    if (!aligned_to(bmp, 8) || !aligned_to(packed, 4) || !aligned_to(tile_off, 4) || !aligned_to(scales, 4) ||
        !aligned_to(zeros, 4) || !aligned_to(Bm, 4) || !aligned_to(C, 2))
        return MSTF_EALIGN;
    return MSTF_OK;
}

struct QArgs {
    const uint64_t* bmp;
    const uint32_t* packed;
    const uint32_t* tile_off;
    const uint16_t* scales;
    const uint16_t* zeros;
    int mode;
    int group_size;  // 64: one (scale, zero) pair per tile; 32: two
};

// Whether the four wavefronts of a workgroup share a token block of a key product with more than eight rows, a channel stage
// each, instead of taking a block each: a quarter of the chain, and as many wavefronts four times over.  1024 such workgroups
// fit the chip; a few more still pay.  32 rows, 4 bits, 70 %, heads x blocks, a block each / shared: 1 x 1 7.06 / 3.95 us,
// 8 x 33 7.97 / 4.88, 32 x 24 8.33 / 5.91, 32 x 33 9.33 / 8.36, 32 x 48 9.84 / 10.02, 64 x 64 13.0 / 21.0 (2 bits 6.64 / 3.89,
// 7.43 / 4.78, 7.72 / 5.74, 8.70 / 7.91, 9.25 / 9.66, 12.5 / 20.5).  Up to the line no call of 16, 24 or 32 rows, 2, 4 or 8 bits, one
// group per tile or two, is slower for it (32 x 40, 8 bits, 32 rows 10.85 / 10.57).
constexpr int kKeyShareQuant = 1280;
template <int NW, int BIT>
static void launch_key_q(hipStream_t st, const QArgs& a, const _Float16* Bm, _Float16* C, int Lc, int D, int Bkv,
                         int rows_per_kv, int row0)
{
    const int nblk = Lc / 64;
    const int ntasks = Bkv * nblk;
    const bool share = wide_rows(NW) && D == 128 && ntasks <= kKeyShareQuant;
    const int wgs = xcd_grid(share ? ntasks : (wide_rows(NW) ? Bkv * ((nblk + 3) / 4) : (ntasks + 3) / 4));
#define MSTF_KQ_LAUNCH(G32, SHARE)                                                                                            \
    hipLaunchKernelGGL((key_spmv_quant_kernel<NW, BIT, G32, SHARE>), dim3(wgs), dim3(256), 0, st, a.bmp, a.packed, a.tile_off, \
                       a.tile_off, a.scales, a.zeros, Bm, C, Lc, D, nblk, ntasks, rows_per_kv, row0, a.mode)
    constexpr bool kShare = wide_rows(NW);
    if (a.group_size == 32) {
        if (share) MSTF_KQ_LAUNCH(true, kShare); else MSTF_KQ_LAUNCH(true, false);
    } else {
        if (share) MSTF_KQ_LAUNCH(false, kShare); else MSTF_KQ_LAUNCH(false, false);
    }
#undef MSTF_KQ_LAUNCH
}
template <int NW>
static void launch_key_q_bit(int bit, hipStream_t st, const QArgs& a, const _Float16* Bm, _Float16* C, int Lc, int D,
                             int Bkv, int rows_per_kv, int row0)
{
    if (bit == 2)
        launch_key_q<NW, 2>(st, a, Bm, C, Lc, D, Bkv, rows_per_kv, row0);
    else if (bit == 4)
        launch_key_q<NW, 4>(st, a, Bm, C, Lc, D, Bkv, rows_per_kv, row0);
    else
        launch_key_q<NW, 8>(st, a, Bm, C, Lc, D, Bkv, rows_per_kv, row0);
}

// Whether a value product of up to eight rows reads whole tiles (StageRank): with more blocks of all heads than this there is more
// than one to a wavefront all over the chip.  70 %, heads x blocks, whole / halves, over rows 1, 4 and 8, 2, 4 and 8 bits, one
// group per tile or two: 256 x 64 0.96 - 1.00 (4 bits, four rows 29.4 -> 28.3 us), 64 x 256 0.96 - 1.01, 40 x 256 0.97 - 1.01; but
// 128 x 64 0.98 - 1.05, 256 x 32 0.99 - 1.06, 32 x 256 0.98 - 1.05, 256 x 16 0.99 - 1.07, 32 x 16 1.00 - 1.04.
static bool value_whole(int nw, int nblk, int Bkv) { return !wide_rows(nw) && (long long)Bkv * nblk > 8192; }
template <int NW, int WAVES, int BIT>
static void launch_value_q(hipStream_t st, const ValuePlan& pl, const QArgs& a, const _Float16* P, _Float16* C,
                           float* part, int Lc, int D, int Bkv, int rows_per_kv, int row0)
{
    const int nwg = pl.nsplit * (D / 64) * Bkv;
    const bool whole = value_whole(NW, Lc / 64, Bkv);
#define MSTF_VQ_LAUNCH(G32, WHOLE)                                                                                           \
    hipLaunchKernelGGL((value_spmv_quant_kernel<NW, WAVES, BIT, G32, WHOLE>), dim3(xcd_grid(nwg)), dim3(WAVES * 64), 0, st, \
                       a.bmp, a.packed, a.tile_off, a.tile_off, a.scales, a.zeros, P, C, part, Lc, D, Lc / 64, pl.nbpw,       \
                       pl.nsplit, rows_per_kv, row0, a.mode, nwg, split_inverse(pl.nsplit))
    constexpr bool kWhole = !wide_rows(NW);
    if (a.group_size == 32) {
        if (whole) MSTF_VQ_LAUNCH(true, kWhole); else MSTF_VQ_LAUNCH(true, false);
    } else {
        if (whole) MSTF_VQ_LAUNCH(false, kWhole); else MSTF_VQ_LAUNCH(false, false);
    }
#undef MSTF_VQ_LAUNCH
}
template <int NW, int WAVES>
static void launch_value_q_bit(int bit, hipStream_t st, const ValuePlan& pl, const QArgs& a, const _Float16* P,
                               _Float16* C, float* part, int Lc, int D, int Bkv, int rows_per_kv, int row0)
{
    if (bit == 2)
        launch_value_q<NW, WAVES, 2>(st, pl, a, P, C, part, Lc, D, Bkv, rows_per_kv, row0);
    else if (bit == 4)
        launch_value_q<NW, WAVES, 4>(st, pl, a, P, C, part, Lc, D, Bkv, rows_per_kv, row0);
    else
        launch_value_q<NW, WAVES, 8>(st, pl, a, P, C, part, Lc, D, Bkv, rows_per_kv, row0);
}

}  // namespace mstf

using namespace mstf;

static int key_spmv_quant_impl(void* stream, const uint64_t* bmp, const uint32_t* packed, const uint32_t* tile_off,
                               const mstf_half* scales, const mstf_half* zeros, const mstf_half* Bm, mstf_half* C, int M,
                               int K, int Bq, int groups, int n_rows, int bit, int capacity, int dequant_mode,
                               int group_size)
{
    if (group_size != 64 && group_size != 32) return MSTF_EUNSUPPORTED;
    int rc = check_quant_spmv(bmp, packed, tile_off, scales, zeros, Bm, C, M, K, Bq, groups, n_rows, bit, capacity,
                              dequant_mode);
    if (rc != MSTF_OK) return rc;
    hipStream_t st = as_stream(stream);
    const int Bkv = Bq / groups, rows_per_kv = groups * n_rows;
    const _Float16* b = reinterpret_cast<const _Float16*>(Bm);
    _Float16* c = reinterpret_cast<_Float16*>(C);
    const QArgs a = {bmp, packed, tile_off, scales, zeros, dequant_mode, group_size};
    const bool lines = aligned_to(C, 16);     // (the rows of a wide pass leave as whole lines)
    for (int row0 = 0; row0 < rows_per_kv;) {
        const int nw = pick_nw(rows_per_kv - row0, lines);
        switch (nw) {
            case 32: launch_key_q_bit<32>(bit, st, a, b, c, M, K, Bkv, rows_per_kv, row0); break;
            case 16: launch_key_q_bit<16>(bit, st, a, b, c, M, K, Bkv, rows_per_kv, row0); break;
            case 8: launch_key_q_bit<8>(bit, st, a, b, c, M, K, Bkv, rows_per_kv, row0); break;
            case 4: launch_key_q_bit<4>(bit, st, a, b, c, M, K, Bkv, rows_per_kv, row0); break;
            case 2: launch_key_q_bit<2>(bit, st, a, b, c, M, K, Bkv, rows_per_kv, row0); break;
            default: launch_key_q_bit<1>(bit, st, a, b, c, M, K, Bkv, rows_per_kv, row0); break;
        }
        if ((rc = check_launch()) != MSTF_OK) return rc;
        row0 += nw;
    }
    return MSTF_OK;
}

extern "C" int mstf_key_spmv_quant(void* stream, const uint64_t* bmp, const uint32_t* packed, const uint32_t* tile_off,
                                   const uint32_t* counts, const uint32_t* units, const mstf_half* scales,
                                   const mstf_half* zeros, const mstf_half* Bm, mstf_half* C, int M, int K, int Bq,
                                   int groups, int n_rows, int bit, int capacity, int dequant_mode)
{
    (void)counts;  // raw counts and units follow from the bitmaps; accepted for interface compatibility
    (void)units;
    return key_spmv_quant_impl(stream, bmp, packed, tile_off, scales, zeros, Bm, C, M, K, Bq, groups, n_rows, bit, capacity,
                               dequant_mode, 64);
}

extern "C" int mstf_key_spmv_quant_grouped(void* stream, const uint64_t* bmp, const uint32_t* packed,
                                           const uint32_t* tile_off, const mstf_half* scales, const mstf_half* zeros,
                                           const mstf_half* Bm, mstf_half* C, int M, int K, int Bq, int groups, int n_rows,
                                           int bit, int capacity, int dequant_mode, int group_size)
{
    return key_spmv_quant_impl(stream, bmp, packed, tile_off, scales, zeros, Bm, C, M, K, Bq, groups, n_rows, bit, capacity,
                               dequant_mode, group_size);
}

extern "C" size_t mstf_value_spmv_quant_workspace_bytes(int M, int K, int Bq, int groups, int n_rows)
{
    if (M <= 0 || K <= 0 || Bq <= 0 || groups <= 0 || n_rows <= 0 || K % 64 != 0 || M % 64 != 0 || Bq % groups != 0)
        return 0;
    return value_workspace_bytes(M, K, Bq, groups, n_rows);
}

static int value_spmv_quant_impl(void* stream, const uint64_t* bmp, const uint32_t* packed, const uint32_t* tile_off,
                                 const mstf_half* scales, const mstf_half* zeros, const mstf_half* P, mstf_half* C, int M,
                                 int K, int Bq, int groups, int n_rows, int bit, int capacity, int dequant_mode,
                                 int group_size, void* workspace, size_t workspace_bytes)
{
    if (group_size != 64 && group_size != 32) return MSTF_EUNSUPPORTED;
    // M = head_dim, K = compressed tokens (the operator's GEMM naming)
    int rc = check_quant_spmv(bmp, packed, tile_off, scales, zeros, P, C, K, M, Bq, groups, n_rows, bit, capacity,
                              dequant_mode);
    if (rc != MSTF_OK) return rc;
    const size_t need = mstf_value_spmv_quant_workspace_bytes(M, K, Bq, groups, n_rows);
    if (need > 0 && (!workspace || workspace_bytes < need)) return MSTF_EWORKSPACE;
    if (workspace && !aligned_to(workspace, 16)) return MSTF_EALIGN;
    hipStream_t st = as_stream(stream);
    const int Bkv = Bq / groups, rows_per_kv = groups * n_rows;
    const _Float16* p = reinterpret_cast<const _Float16*>(P);
    _Float16* c = reinterpret_cast<_Float16*>(C);
    float* part = reinterpret_cast<float*>(workspace);
    const QArgs a = {bmp, packed, tile_off, scales, zeros, dequant_mode, group_size};
    const bool pieces = aligned_to(P, 16);    // (a wide pass fetches the weights in pieces of sixteen bytes)
    const int most = pieces ? kAnySplits : splits_that_fit(workspace ? workspace_bytes : 0, M, Bq, n_rows);
    for (int row0 = 0; row0 < rows_per_kv;) {
        const int nw = pick_nw(rows_per_kv - row0, pieces);
        const ValuePlan pl = plan_value(K, M, Bkv, nw, most);
        switch (nw) {
            case 32: launch_value_q_bit<32, 4>(bit, st, pl, a, p, c, part, K, M, Bkv, rows_per_kv, row0); break;
            case 16: launch_value_q_bit<16, 4>(bit, st, pl, a, p, c, part, K, M, Bkv, rows_per_kv, row0); break;
            case 8: launch_value_q_bit<8, 8>(bit, st, pl, a, p, c, part, K, M, Bkv, rows_per_kv, row0); break;
            case 4: launch_value_q_bit<4, 8>(bit, st, pl, a, p, c, part, K, M, Bkv, rows_per_kv, row0); break;
            case 2: launch_value_q_bit<2, 8>(bit, st, pl, a, p, c, part, K, M, Bkv, rows_per_kv, row0); break;
            default: launch_value_q_bit<1, 8>(bit, st, pl, a, p, c, part, K, M, Bkv, rows_per_kv, row0); break;
        }
        if ((rc = check_launch()) != MSTF_OK) return rc;
        if (pl.nsplit > 1) {
            launch_value_merge(st, part, c, pl.nsplit, M, rows_per_kv, row0, nw, Bkv);
            if ((rc = check_launch()) != MSTF_OK) return rc;
        }
        row0 += nw;
    }
    return MSTF_OK;
}

extern "C" int mstf_value_spmv_quant(void* stream, const uint64_t* bmp, const uint32_t* packed,
                                     const uint32_t* tile_off, const uint32_t* counts, const uint32_t* units,
                                     const mstf_half* scales, const mstf_half* zeros, const mstf_half* P, mstf_half* C,
                                     int M, int K, int Bq, int groups, int n_rows, int bit, int capacity,
                                     int dequant_mode, void* workspace, size_t workspace_bytes)
{
    (void)counts;
    (void)units;
    return value_spmv_quant_impl(stream, bmp, packed, tile_off, scales, zeros, P, C, M, K, Bq, groups, n_rows, bit, capacity,
                                 dequant_mode, 64, workspace, workspace_bytes);
}

extern "C" int mstf_value_spmv_quant_grouped(void* stream, const uint64_t* bmp, const uint32_t* packed,
                                             const uint32_t* tile_off, const mstf_half* scales, const mstf_half* zeros,
                                             const mstf_half* P, mstf_half* C, int M, int K, int Bq, int groups, int n_rows,
                                             int bit, int capacity, int dequant_mode, int group_size, void* workspace,
                                             size_t workspace_bytes)
{
    return value_spmv_quant_impl(stream, bmp, packed, tile_off, scales, zeros, P, C, M, K, Bq, groups, n_rows, bit, capacity,
                                 dequant_mode, group_size, workspace, workspace_bytes);
}
