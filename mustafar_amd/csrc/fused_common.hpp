// Pieces shared by the fused decode-attention kernels (fused.hip: fp16 format and dense window; fused_quant.hip:
// quantised format): block softmax statistics, the workgroup combine and the layout of the split partials.
#pragma once
#include "spmv_common.hpp"
#include "spmv_device.hpp"

namespace mstf {

constexpr int kFusedD = 128;
constexpr int kFusedWaves = 8;    // token blocks (= wavefronts) per workgroup: 512 tokens per split
constexpr int kKeySubs = kFusedD / kSubTiles;       // sub-chunks of the key phase
constexpr int kValSubs = kFusedD / kSubTiles;       // sub-chunks of the value phase (both halves)

constexpr int kFusedResident = 1024 * 4;  // wavefronts of the fused kernel the 256 CUs hold at once
constexpr int kFusedMaxBpw = 8;           // token blocks that a wavefront walks at most, on average over its workgroup

// (The planning helpers below are constexpr, hence usable from device code as well as from the launchers.)
// How the token blocks of a KV head are dealt out.  While every block finds a resident wavefront of its own, a workgroup
// takes eight; beyond that the blocks are spread evenly over as many workgroups per head as the chip holds at once, and a
// wavefront walks the ones it gets, so that only its first block waits for memory.
// (A fixed number of blocks per wavefront instead left a few workgroups to a second generation - 528 of them for the 512
// that the chip holds at 24 heads x 511 blocks - or a part of the chip without work.  fp16, 70 %, launch + merge: 24 x 511
// blocks 58.2 -> 45.1 us, 304 x 64 94.7 -> 66.3, 384 x 64 112 -> 70, 64 x 66 27.1 -> 26.0; 2 bits: 24 x 511 71.6 -> 52.0,
// 1024 x 16 80.9 -> 56.2; a 2-bit decode step of 8 layers at 128 heads x 60 blocks + window 300 -> 264 us, where the
// wavefronts with a block less now take the window's; one head of 4200 blocks, whose merge got twice the splits, 32.5 -> 34.8,
// 30.5 since the merge takes its runs in groups.)
struct FusedFill {
    int once;  // workgroups per KV head up to which a launch takes eight blocks each
    int full;  // workgroups per KV head that fill the chip
};
// Where the heads do not divide the chip's room (300 of 512 workgroups), two or more generations of workgroups fill it
// better than one: the first count of at most four that leaves less than a quarter of the room empty, or the best of them.
// One generation still is the better one (at two or more workgroups per head) while there are too few blocks for all of them.
constexpr FusedFill fused_fill(int Bkv, int resident = kFusedResident)
{
    const int room = resident / kFusedWaves;
    const int first = (Bkv + room - 1) / room;
    int best = 1;
    long long best_num = 0, best_den = 1;
    for (int g = first; g < first + 4; g++) {
        const long long slots = (long long)g * room, wgs = slots / Bkv;
        const long long used = wgs * Bkv;
        if (used * best_den > best_num * slots) {
            best = (int)wgs;
            best_num = used;
            best_den = slots;
        }
        if (used * 4 > slots * 3) break;
    }
    return {room / Bkv >= 2 ? room / Bkv : best, best};
}
// (as a kernel argument)
constexpr int fused_fill_pack(FusedFill f) { return (f.once < 0x7FFF ? f.once : 0x7FFF) << 16 | (f.full < 0x7FFF ? f.full : 0x7FFF); }
constexpr FusedFill fused_fill_unpack(int v) { return {v >> 16, v & 0xFFFF}; }
// Split slots (= workgroups) per KV head at eight token blocks each.
constexpr int fused_nsplit(int tokens)
{
    return (tokens / 64 + kFusedWaves - 1) / kFusedWaves;
}
// Split slots of a launch over nblk blocks per head; grows with nblk, so that the count for a cache's capacity has room for
// every smaller one.
constexpr int fused_splits(int nblk, FusedFill fill)
{
    const int one = (nblk + kFusedWaves - 1) / kFusedWaves;
    const long long most = (long long)fill.full * (kFusedWaves * kFusedMaxBpw);
    if (one <= fill.full) return one <= fill.once ? one : fill.once;
    return nblk <= most ? fill.full : fill.full * (int)((nblk + most - 1) / most);
}
// The same for a decode step, whose wavefronts also take a block of the dense window each: at least as many workgroups as
// have wavefronts for all of them (or kFusedWaves compressed blocks each, where the window is the longer part).
constexpr int fused_splits_step(int nblk, FusedFill fill, int window)
{
    const int one = (nblk + kFusedWaves - 1) / kFusedWaves, ns = fused_splits(nblk, fill);
    const int need = (window + kFusedWaves - 1) / kFusedWaves;
    return need <= ns ? ns : (need < one ? need : one);
}
// The share of a split: blocks per split in the low byte and, above, the number of leading splits that take one more.
constexpr int fused_deal(int nblk, int ns)
{
    return ns == (nblk + kFusedWaves - 1) / kFusedWaves ? kFusedWaves : (nblk / ns | nblk % ns << 8);
}
struct BlockRange {
    int first, count;
};
// The blocks of a split.
constexpr BlockRange fused_blocks_of_split(int nblk, int deal, int split)
{
    const int base = deal & 255, more = deal >> 8;
    const int b0 = split * base + (split < more ? split : more);
    const int n = base + (split < more ? 1 : 0), there = nblk - b0 < n ? nblk - b0 : n;
    return {b0, there > 0 ? there : 0};
}
// The blocks of a wavefront: those of its split dealt out evenly over the eight wavefronts, the last of them take one less.
constexpr BlockRange fused_blocks_of(int nblk, int deal, int split, int wave)
{
    const BlockRange all = fused_blocks_of_split(nblk, deal, split);
    const int each = (int)((unsigned)all.count / kFusedWaves), left = (int)((unsigned)all.count % kFusedWaves);
    return {all.first + wave * each + (wave < left ? wave : left), each + (wave < left ? 1 : 0)};
}
// The wavefronts of a split in the order in which they take a block of the dense window behind their compressed ones: from the
// last one on where those have a block less (128 heads x 60 blocks, 2 bits: 300 -> 264 us per eight layers; 64 x 60, 8 bits, four
// layers: 150 -> 134), else from the first one on, which is the first to start (16 heads x 24 blocks, eight query heads, 8 bits:
// 102 -> 98 us, 4 bits 93.5 -> 90).  Where the last ones have no block at all, they may still
// be too few for the split's share of the window (rows: those there are, ns: splits of a head).  A short block - the window's
// last one - then follows onto a wavefront with a compressed block, but a longer one would come to it with the new token's row
// still behind it: from the first wavefront on the new row's block finds an idle one (156 heads x 4 blocks, four layers, 2 bits:
// a window of 257 rows 77.7 us from the last one on, 100.6 from the first; 320 rows 95.9, 93.9; 429 98.4, 93.4; 511 103.8, 95.3).
constexpr int fused_window_order(int nblk, int deal, int split, int wave, int rows, int ns)
{
    const int n = fused_blocks_of_split(nblk, deal, split).count, left = n % kFusedWaves;
    const bool last_first = left != 0 && (n > kFusedWaves || rows <= ((kFusedWaves - left) * ns + split) * 64 + 32);
    return last_first ? kFusedWaves - 1 - wave : wave;
}

// Whether the four wavefronts of a workgroup share a token block instead of walking blocks of their own: with few blocks a
// launch lasts as long as one wavefront's chain of eight dependent stages, and idle SIMDs take three quarters of it off.
// More workgroups (extra: of the dense window) than the chip holds at once run one after the other and lose it again: four per
// CU, three with eight query heads, whose rows take more LDS.  Measured, fp16, 70 %, launch + merge: 128 blocks 12.2 -> 8.1 us,
// 512 12.8 -> 9.8, 1024 12.9 -> 11.6 us; two wavefronts per block at 1536 and 2048 blocks 13.9 -> 14.2 and 13.8 -> 14.6.
// The merge has a split per block then, eight times as many: beyond 128 blocks per head its round trips outweigh the gain
// (3 heads x 256 blocks 14.6 -> 15.3, 1 x 512 17.0 -> 20.2).
constexpr int kShareMaxBlocks = 128;                                            // token blocks of a head
constexpr int fused_share_launch(int groups) { return groups <= 4 ? 1024 : 768; }  // of all heads
constexpr bool fused_shares_blocks(int tokens, int Bkv, int groups, int extra = 0)
{
    return tokens <= kShareMaxBlocks * 64 && (long long)Bkv * (tokens / 64) + extra <= fused_share_launch(groups);
}

// Calls over up to eight blocks a head have no split, and their workgroups write the output.  Sharing makes the call two
// launches: recorded into a graph, where a launch behind another takes 2 us, it is the faster form all the same up to this many
// blocks of all heads, from five blocks a head on or with more than four query heads (fp16, 70 %, pairs or a wavefront per
// block / shared and merged: 8 heads x 8 blocks 8.4 / 6.6 us, 64 x 8 8.9 / 8.1, 128 x 8 9.0 / 10.2; eight query heads, 8 x 4
// 9.6 / 7.1, 64 x 8 11.2 / 9.6); launched call by call it is not (8 x 8 8.4 / 9.5).  With more than four query heads the
// rows that the merge has to launch for outweigh few blocks a head (recorded, eight query heads: 128 x 1 9.04 / 8.24, 256 x 1 9.31 /
// 9.80, 128 x 2 9.43 / 8.93, 160 x 2 9.46 / 10.00, 96 x 3 9.60 / 9.40, 128 x 3 9.71 / 9.93, 96 x 4 10.16 / 9.47, 160 x 4 10.25 / 10.98;
// but 80 x 8 11.3 / 10.9; five: 256 x 1 9.24 / 8.96, 160 x 2 9.34 / 9.49), unless there are more heads than workgroups fit the
// chip at once (five, 512 x 1 17.2 / 11.5).
constexpr int kShareOneSplit = 640;
constexpr bool fused_share_one_split(int nblk, int Bkv, int groups, bool recorded)
{
    if (!recorded || Bkv * nblk > kShareOneSplit) return false;
    if (nblk > 4 || groups <= 4) return nblk > 4;
    return Bkv > 256 || (nblk == 1 ? Bkv * groups <= 1280 : Bkv <= (nblk == 2 ? 128 : 112));
}
// Whether a workgroup of sixteen wavefronts takes a whole head, with up to four query heads, and writes its output, so that
// no merge follows: heads of up to eight blocks, two wavefronts per block (a wavefront per block / this: 8 heads x 1 block 7.6 /
// 5.5 us, 8 x 4 8.0 / 6.2, 256 x 4 8.7 / 7.1, 8 x 8 8.8 / 8.4, 256 x 8 9.7 / 9.5: eight blocks keep a CU busy), and heads of two
// splits where these are as many as fill the chip (two splits and merge / this: 256 x 16 16.4 / 14.6, 256 x 64 48.8 / 47.3,
// 224 x 64 44.9 / 43.4, 200 x 64 41.5 / 40.2, 2 bits 256 x 64 50.5 / 48.1; but 176 x 64 41.5 / 41.9, 64 x 16 9.9 / 11.8), with one
// to four query heads alike, and longer heads no slower (200 and 256 x 128: from 0.96 to 1.03 of the two splits', by the card).
constexpr bool fused_whole_head(int nblk, int ns, int Bkv, int groups, bool pairs)
{
    if (groups > 4 || Bkv > 256) return false;
    return nblk <= kFusedWaves ? pairs : ns == 2 && Bkv >= 200;
}

constexpr int window_blocks(int win_len) { return (win_len + 63) / 64; }
// Bytes of `slots` split slots: kFusedD outputs and (max, sum) each, fp32.
constexpr size_t fused_slot_bytes(size_t slots) { return (slots * (kFusedD + 2) * sizeof(float) + 255) / 256 * 256; }
// What a call over `tokens` compressed tokens and a window demands of its workspace: a slot per query row, kFusedWaves blocks
// and window block.  Grows with every argument, so that a workspace made for the largest call serves the others.
constexpr size_t fused_workspace_need(int tokens, int window, int Bq)
{
    return fused_slot_bytes((size_t)Bq * (fused_nsplit(tokens) + window_blocks(window)));
}
// Whether a workspace has room for wavefronts to share blocks, a slot per block; without it a call goes without sharing (the
// results are the same numbers).
constexpr bool fused_share_fits(int tokens, int window, int Bq, size_t workspace_bytes)
{
    return fused_slot_bytes((size_t)Bq * (tokens / 64 + window_blocks(window))) <= workspace_bytes;
}
// The size that the queries answer: what the call demands, or has use for where its wavefronts may share blocks.
constexpr size_t fused_workspace_room(int tokens, int window, int Bq, int groups)
{
    return fused_shares_blocks(tokens, Bq / groups, groups)
               ? fused_slot_bytes((size_t)Bq * (tokens / 64 + window_blocks(window)))
               : fused_workspace_need(tokens, window, Bq);
}

// Launches the merge of ns split slots per query row out of a workspace in the layout of the fused kernels
// (defined beside the merge kernel).  The first `blocks` slots hold one token block each (wavefronts shared blocks).
int merge_splits(hipStream_t st, const void* workspace, mstf_half* out, float* lse_out, int ns, int head_dim, int Bq,
                 int blocks = 0);

// Launches the dense-window kernel: the (max, sum, output) triples of the window's 64-token blocks go into split
// slots split0 .. of a workspace with nst slots per query row (defined beside the kernel).
int window_launch(hipStream_t st, const mstf_half* k_win, const mstf_half* v_win, const mstf_half* q, void* workspace,
                  int win_len, const int32_t* win_len_dev, int win_stride, int head_dim, int Bq, int groups, int nst,
                  int split0);

// Reductions over the sixteen lanes 4b+j (b = 0..15) that hold column j, without LDS round trips: inside a row of
// sixteen lanes by two rotations (DPP row_ror 4 and 8, folded into the combining instruction), across the four rows by
// v_permlane16_swap / v_permlane32_swap (a and b copies of v: afterwards a holds the even rows / the lower half twice,
// b the odd rows / the upper half twice).  Every lane ends up with the maximum; of the sum, lanes 4b+j of one column may
// differ in the last bit (the rotations add in a different order per lane), and lanes 0..3 are the ones that are used.
typedef uint32_t u32x2v_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ float dpp_row_ror(float v, int n4)
{
    const int x = __builtin_bit_cast(int, v);
    return __builtin_bit_cast(float, n4 == 4 ? __builtin_amdgcn_update_dpp(x, x, 0x124, 0xf, 0xf, false)
                                               : __builtin_amdgcn_update_dpp(x, x, 0x128, 0xf, 0xf, false));
}
__device__ __forceinline__ void rows_swapped(float v, bool halves, float& a, float& b)
{
    const uint32_t x = __builtin_bit_cast(uint32_t, v);
    const u32x2v_t r = halves ? __builtin_amdgcn_permlane32_swap(x, x, false, false)
                              : __builtin_amdgcn_permlane16_swap(x, x, false, false);
    const uint32_t r0 = r[0], r1 = r[1];  // (a bit cast applied to a vector element directly reads element 0)
    a = __builtin_bit_cast(float, r0);
    b = __builtin_bit_cast(float, r1);
}
__device__ __forceinline__ float wave_max_same_column(float v)
{
    float a, b;
    v = fmaxf(v, dpp_row_ror(v, 4));
    v = fmaxf(v, dpp_row_ror(v, 8));
    rows_swapped(v, false, a, b);
    v = fmaxf(a, b);
    rows_swapped(v, true, a, b);
    return fmaxf(a, b);
}
__device__ __forceinline__ float wave_sum_same_column(float v)
{
    float a, b;
    v += dpp_row_ror(v, 4);
    v += dpp_row_ror(v, 8);
    rows_swapped(v, false, a, b);
    v = a + b;
    rows_swapped(v, true, a, b);
    return a + b;
}

// x / c for |x| up to the fp16 range and c = sqrt(head_dim), r = 1 / c rounded: the quotient estimate and one
// correction by the exact remainder - the correctly rounded quotient, as the full division sequence gives it, without
// that sequence's scaling and special cases (a dozen instructions per value), which these operands never need.
__device__ __forceinline__ float div_small(float x, float c, float r)
{
    const float q = x * r;
    return __builtin_fmaf(__builtin_fmaf(-c, q, x), r, q);
}

// Softmax statistics of one 64-token block from its scores; lane 4b+j holds tokens 4b..4b+3 of head 4m+j in acc_k[m].
// Scores are rounded to fp16 and divided by sqrt(d) in fp16 (as the reference's glue does); the un-normalised
// weights exp(w - max) go to LDS as fp16 rows of 64 tokens, kPRow bytes apart, (the B operand of the value phase) and the block's
// (max, sum of the fp16 weights) stay in m_run / l_run.  Tokens >= nt (nt < 64 only in a partial block) get weight 0.
template <int NM, int kPRow = 64 * 2>
__device__ __forceinline__ void block_softmax(const f4_t (&acc_k)[NM], float sqrt_d, int nt, char* pl, int lane,
                                              float (&m_run)[NM], float (&l_run)[NM])
{
    const int j = lane & 3;
    const float rcp_d = 1.0f / sqrt_d;
#pragma unroll
    for (int m = 0; m < NM; m++) {
        float w[4];
        float mx = -INFINITY;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const _Float16 s16 = (_Float16)acc_k[m][r];
            w[r] = ((lane & ~3) + r < nt) ? (float)(_Float16)div_small((float)s16, sqrt_d, rcp_d) : -INFINITY;
            mx = fmaxf(mx, w[r]);
        }
        mx = wave_max_same_column(mx);
        float sum = 0.f;
        h4_t e16;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const float e = w[r] == -INFINITY ? 0.f : __expf(w[r] - mx);
            e16[r] = (_Float16)e;
            sum += (float)e16[r];  // the sum matches the fp16 weights that multiply V
        }
        sum = wave_sum_same_column(sum);
        m_run[m] = mx;
        l_run[m] = sum;
        *reinterpret_cast<h4_t*>(pl + (m * 4 + j) * kPRow + (lane & ~3) * 2) = e16;
    }
}

// Folds a block's (max, sum, output) into the running one of the wavefront (lane 4b+j: head j in every register).  In two
// steps: what the running output and the block's are worth beside each other follows from the maxima, before the block's is there.
struct Folded {
    float fa, fb;
    __device__ __forceinline__ Folded(float& m_run, float& l_run, float m_blk, float l_blk)
    {
        const float mn = fmaxf(m_run, m_blk);
        fa = m_run == -INFINITY ? 0.f : __expf(m_run - mn);
        fb = m_blk == -INFINITY ? 0.f : __expf(m_blk - mn);
        l_run = l_run * fa + l_blk * fb;
        m_run = mn;
    }
};
__device__ __forceinline__ void fold_block(f4_t (&acc)[2], float& m_run, float& l_run, const f4_t (&blk)[2], float m_blk,
                                           float l_blk)
{
    const Folded f(m_run, l_run, m_blk, l_blk);
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
        for (int c = 0; c < 4; c++) acc[h][c] = acc[h][c] * f.fa + blk[h][c] * f.fb;
}

// Workgroup combine of the kFusedWaves blocks of a split: every wavefront parks (output[4*NM][D], max, sum) in its
// own LDS area (`lds_base + wave * wave_stride`, at least fused_park_bytes), then one thread per (head, channel)
// folds them and writes either the final fp16 output (write_final, one split only) or the split's partial:
//   part_o[((kv*groups + h)*nsplit + split)*D + d] (un-normalised), part_ml[..][2] = (max, sum).
// An inactive wavefront parks (-inf, 0, 0).
template <int NM>
constexpr int fused_park_bytes()
{
    return NM * 4 * kFusedD * 4 + 64;
}
// (BOTH: both halves of the channels, or only half `half`, which is in acc_v[m][0])
template <int NM, bool BOTH = true>
__device__ __forceinline__ void park(char* area, int lane, const f4_t (&acc_v)[NM][2], const float (&m_run)[NM],
                                     const float (&l_run)[NM], int half = 0)
{
    constexpr int D = kFusedD;
    const int j = lane & 3;
    float* po = reinterpret_cast<float*>(area);
#pragma unroll
    for (int m = 0; m < NM; m++) {
        if constexpr (BOTH) {
            *reinterpret_cast<f4_t*>(po + (m * 4 + j) * D + (lane & ~3)) = acc_v[m][0];
            *reinterpret_cast<f4_t*>(po + (m * 4 + j) * D + 64 + (lane & ~3)) = acc_v[m][1];
        } else {
            *reinterpret_cast<f4_t*>(po + (m * 4 + j) * D + half * 64 + (lane & ~3)) = acc_v[m][0];
        }
        if (lane < 4) {
            po[NM * 4 * D + (m * 4 + j) * 2] = m_run[m];
            po[NM * 4 * D + (m * 4 + j) * 2 + 1] = l_run[m];
        }
    }
}
struct Triple {
    float M, so, sl;
};
// (head h, channel c) of kFusedWaves parked triples, stride bytes apart.
template <int NM>
__device__ __forceinline__ Triple combined(const char* area0, int stride, int h, int c)
{
    constexpr int D = kFusedD;
    Triple t = {-INFINITY, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < kFusedWaves; w++)
        t.M = fmaxf(t.M, reinterpret_cast<const float*>(area0 + w * stride)[NM * 4 * D + h * 2]);
#pragma unroll
    for (int w = 0; w < kFusedWaves; w++) {
        const float* pw = reinterpret_cast<const float*>(area0 + w * stride);
        const float mw = pw[NM * 4 * D + h * 2];
        const float f = mw == -INFINITY ? 0.f : __expf(mw - t.M);
        t.so = __builtin_fmaf(f, pw[h * D + c], t.so);
        t.sl = __builtin_fmaf(f, pw[NM * 4 * D + h * 2 + 1], t.sl);
    }
    return t;
}
template <int NM>
__device__ __forceinline__ void workgroup_combine(char* lds_base, int wave_stride, int wave, int lane,
                                                  const f4_t (&acc_v)[NM][2], const float (&m_run)[NM],
                                                  const float (&l_run)[NM], int kv, int groups, int split, int nsplit,
                                                  int write_final, _Float16* out, float* part_o, float* part_ml)
{
    constexpr int D = kFusedD;
    // (the wavefront parks its triple in its own LDS region, which only it has used so far: no barrier in front)
    park<NM>(lds_base + wave * wave_stride, lane, acc_v, m_run, l_run);
    __syncthreads();
    for (int o = (int)threadIdx.x; o < groups * D; o += kFusedWaves * 64) {
        const int h = o / D, c = o - h * D;
        const Triple t = combined<NM>(lds_base, wave_stride, h, c);
        const size_t row = (size_t)kv * groups + h;
        if (write_final) {
            out[row * D + c] = (_Float16)(t.so / t.sl);
        } else {
            part_o[(row * nsplit + split) * D + c] = t.so;
            if (c == 0) {
                part_ml[(row * nsplit + split) * 2] = t.M;
                part_ml[(row * nsplit + split) * 2 + 1] = t.sl;
            }
        }
    }
}

// A run of eight splits into a running (max, output, sum) (decode_merge_kernel).
constexpr int kMergeRun = 8;
__device__ __forceinline__ void merge_run(Triple& s, const float (&m)[kMergeRun], const float (&l)[kMergeRun],
                                          const float (&o)[kMergeRun], int valid, bool alone = false)
{
    float gm = s.M;
#pragma unroll
    for (int u = 0; u < kMergeRun; u++)
        if (u < valid) gm = fmaxf(gm, m[u]);
    const float fr = s.M == -INFINITY ? 0.f : __expf(s.M - gm);
    s.so *= fr;
    s.sl *= fr;
#pragma unroll
    for (int u = 0; u < kMergeRun; u++) {
        const bool there = u < valid;
        const float f = (there && m[u] != -INFINITY) ? __expf(m[u] - gm) : 0.f;
        // (alone: one split, which no merge would follow without sharing; its infinite outputs must not meet the zero)
        s.so = __builtin_fmaf(f, there || !alone ? o[u] : 0.f, s.so);  // (written out: the same numbers in every kernel)
        s.sl = __builtin_fmaf(f, there || !alone ? l[u] : 0.f, s.sl);
    }
    s.M = gm;
}

// ---- One workgroup of sixteen wavefronts takes a whole head, and no merge follows (fused_whole_head).
constexpr int kWholeWaves = 16;
constexpr int kWholeLds = 160 * 1024;  // what a workgroup may have
// Behind the parked triples of its wavefronts: both splits combined as workgroup_combine does it, and merged as
// decode_merge_kernel does it - the same numbers bit for bit - into the output.
template <int NM>
__device__ __forceinline__ void combine_whole_head(char* lds_base, int stride, int wave, int lane, const f4_t (&acc_v)[NM][2],
                                                   const float (&m_run)[NM], const float (&l_run)[NM], int kv, int groups,
                                                   _Float16* out)
{
    constexpr int D = kFusedD, kHalf = kFusedWaves * 64;
    park<NM>(lds_base + wave * stride, lane, acc_v, m_run, l_run);
    __syncthreads();
    const int side = (int)threadIdx.x / kHalf, first = (int)threadIdx.x % kHalf;
    // (the second split's triples, behind three of the parked ones: max, output, sum)
    auto other = [=](int part, int o) {
        return reinterpret_cast<float*>(lds_base + (kFusedWaves + part) * stride + fused_park_bytes<NM>()) + o;
    };
    Triple mine[NM];
#pragma unroll
    for (int m = 0; m < NM; m++) {
        const int o = first + m * kHalf, h = o / D, c = o % D;
        if (o >= groups * D) break;
        mine[m] = combined<NM>(lds_base + side * kFusedWaves * stride, stride, h, c);
        if (side == 1) *other(0, o) = mine[m].M, *other(1, o) = mine[m].so, *other(2, o) = mine[m].sl;
    }
    __syncthreads();
    if (side == 1) return;
#pragma unroll
    for (int m = 0; m < NM; m++) {
        const int o = first + m * kHalf;
        if (o >= groups * D) break;
        const Triple b = {*other(0, o), *other(1, o), *other(2, o)};
        float M[kMergeRun], l[kMergeRun], v[kMergeRun];
#pragma unroll
        for (int u = 0; u < kMergeRun; u++) {  // (the merge kernel repeats the last split)
            M[u] = u == 0 ? mine[m].M : b.M;
            l[u] = u == 0 ? mine[m].sl : b.sl;
            v[u] = u == 0 ? mine[m].so : b.so;
        }
        Triple s = {-INFINITY, 0.f, 0.f};
        merge_run(s, M, l, v, 2);
        out[(size_t)kv * groups * D + o] = (_Float16)(s.so / s.sl);
    }
}

// ---- Four wavefronts - a workgroup - share a token block (fused_shares_blocks): one key stage and one value stage each.
// What they exchange goes through LDS.  Every stage's sums start at zero and are added up in the order of the stages, with
// one wavefront per block as with four, so the results are the same numbers bit for bit.
constexpr int kShare = 4;
// (Only LDS traffic is waited for, loads stay in flight.)
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
// The scores of the block out of the sums of its four key stages: every wavefront leaves its stage's in LDS (room `sub` of
// four, `stride` bytes apart, NM KB each) and adds up those of all.
template <int NM>
__device__ __forceinline__ void shared_scores(char* room0, int stride, int sub, int lane, const f4_t (&stage)[NM], f4_t (&acc)[NM])
{
#pragma unroll
    for (int m = 0; m < NM; m++) *reinterpret_cast<f4_t*>(room0 + sub * stride + m * 1024 + lane * 16) = stage[m];
    lds_barrier();
#pragma unroll
    for (int m = 0; m < NM; m++) {
        f4_t got[kShare];
#pragma unroll
        for (int s = 0; s < kShare; s++) got[s] = *reinterpret_cast<const f4_t*>(room0 + s * stride + m * 1024 + lane * 16);
        acc[m] = ((got[0] + got[1]) + got[2]) + got[3];
    }
}
// The (max, sum, un-normalised output) of the block into its split slot (slot0 + h * nsplit for query row h of the head):
// the two wavefronts of a half of the channels add their stages up (room as above; nothing else may still be read there)
// and the first of them writes.
template <int NM>
__device__ __forceinline__ void shared_store(char* room0, int stride, int sub, int lane, f4_t (&half)[NM],
                                             const float (&m_run)[NM], const float (&l_run)[NM], int groups, size_t slot0,
                                             int nsplit, float* part_o, float* part_ml)
{
    constexpr int D = kFusedD;
    const int j = lane & 3;
    if (sub & 1) {
#pragma unroll
        for (int m = 0; m < NM; m++) *reinterpret_cast<f4_t*>(room0 + sub * stride + m * 1024 + lane * 16) = half[m];
    }
    lds_barrier();
    if (sub & 1) return;
#pragma unroll
    for (int m = 0; m < NM; m++) {
        half[m] += *reinterpret_cast<const f4_t*>(room0 + (sub + 1) * stride + m * 1024 + lane * 16);
        const int h = 4 * m + j;
        if (h < groups) {
            const size_t slot = slot0 + (size_t)h * nsplit;
            *reinterpret_cast<f4_t*>(part_o + slot * D + sub * 32 + (lane & ~3)) = half[m];
            if (lane < 4 && sub == 0) {
                part_ml[slot * 2] = m_run[m];
                part_ml[slot * 2 + 1] = l_run[m];
            }
        }
    }
}
// Pairs of wavefronts with a half of their block's channels each (pair_scores): as workgroup_combine, final output.
template <int NM>
__device__ __forceinline__ void combine_pairs(char* lds_base, int stride, int wave, int lane, const f4_t (&acc_v)[NM][2],
                                              const float (&m_run)[NM], const float (&l_run)[NM], int kv, int groups, _Float16* out)
{
    constexpr int D = kFusedD;
    park<NM, false>(lds_base + wave * stride, lane, acc_v, m_run, l_run, wave & 1);
    __syncthreads();
    for (int o = (int)threadIdx.x; o < groups * D; o += kWholeWaves * 64) {
        const int h = o / D, c = o % D;
        const Triple t = combined<NM>(lds_base + (c / 64) * stride, 2 * stride, h, c);
        out[(size_t)kv * groups * D + o] = (_Float16)(t.so / t.sl);
    }
}

// ---- Two wavefronts share a block inside a workgroup that takes a whole head of at most eight: two key stages and a half of
// the channels each.  The scores out of the sums of the four stages (stage[]: the wavefront's two), by way of `room` (3 KB * NM
// of the block's own).  The barrier is the whole workgroup's: idle wavefronts wait at it too.
template <int NM>
__device__ __forceinline__ void pair_scores(char* room, int sub, int lane, const f4_t (&stage)[2][NM], f4_t (&acc)[NM])
{
    auto at = [=](int piece, int m) { return reinterpret_cast<f4_t*>(room + (piece * NM + m) * 1024 + lane * 16); };
#pragma unroll
    for (int m = 0; m < NM; m++) {
        if (sub == 0) {
            *at(0, m) = stage[0][m] + stage[1][m];
        } else {
            *at(1, m) = stage[0][m];
            *at(2, m) = stage[1][m];
        }
    }
    lds_barrier();
#pragma unroll
    for (int m = 0; m < NM; m++) acc[m] = (*at(0, m) + *at(1, m)) + *at(2, m);
}
// The neutral triple in the slot of a block that holds no tokens (a launch sized for more than there are); by one wavefront.
template <int NM>
__device__ __forceinline__ void store_neutral(int lane, int groups, size_t slot0, int nsplit, float* part_o, float* part_ml)
{
    constexpr int D = kFusedD;
    const int j = lane & 3;
#pragma unroll
    for (int m = 0; m < NM; m++) {
        const int h = 4 * m + j;
        if (h < groups) {
            const size_t slot = slot0 + (size_t)h * nsplit;
            *reinterpret_cast<f4_t*>(part_o + slot * D + (lane & ~3)) = f4_t{0.f, 0.f, 0.f, 0.f};
            *reinterpret_cast<f4_t*>(part_o + slot * D + 64 + (lane & ~3)) = f4_t{0.f, 0.f, 0.f, 0.f};
            if (lane < 4) {
                part_ml[slot * 2] = -INFINITY;
                part_ml[slot * 2 + 1] = 0.f;
            }
        }
    }
}

}  // namespace mstf
