// Host-side planning and the split-merge kernel shared by the fp16 and the quantised SpMV files.
#pragma once
#include "common.hpp"

namespace mstf {

// Adds the token-split partials of rows [row0, row0+nw) of every KV head and rounds to fp16.  A column of a row is added up
// by PARTS wavefronts of its workgroup, consecutive splits each, with eight loads on their way at a time; their sums are added
// in order.  (D is a multiple of 64: the 64 columns of a wavefront are one row's.)
// One thread for each column, one load after the other, waited for memory once per split.  Four wavefronts a column, from
// nine splits on, 32 rows, 70 %, value product and merge: 1 head x 40000 tokens (157 splits) 46.2 -> 10.5 us, 8 x 32768
// 29.8 -> 18.7, 8 x 4096 12.6 -> 8.3.  With few splits and many rows they only wait for each other: 128 x 4096 (3 splits)
// 28.5 with one, 32.9 with four.
constexpr int kMergeParts = 4, kMergeRow = 8;
template <int PARTS>
__global__ __launch_bounds__(256) void value_merge_kernel(const float* __restrict__ part, _Float16* __restrict__ C,
                                                          int nsplit, int D, int rows_per_kv, int row0, int nw,
                                                          size_t total)
{
    constexpr int kColumns = 256 / PARTS;
    __shared__ float sums[PARTS > 1 ? PARTS - 1 : 1][kColumns];
    const int column = (int)threadIdx.x % kColumns, mine = (int)threadIdx.x / kColumns;
    const size_t i = (size_t)blockIdx.x * kColumns + column;
    if (i >= total) return;  // (PARTS > 1: never, total is a multiple of 64)
    const size_t d = i % D;
    const size_t r = i / D;
    const size_t row = (r / nw) * rows_per_kv + row0 + (r % nw);
    const int per = (nsplit + PARTS - 1) / PARTS;
    const int first = mine * per;
    const int last = first + per < nsplit ? first + per : nsplit;
    const float* src = part + row * nsplit * D + d;
    float s = 0.f;
    for (int k = first; k < last; k += kMergeRow) {
        float v[kMergeRow];
#pragma unroll
        for (int j = 0; j < kMergeRow; j++) v[j] = src[(size_t)(k + j < last ? k + j : last - 1) * D];
#pragma unroll
        for (int j = 0; j < kMergeRow; j++) s += k + j < last ? v[j] : 0.f;
    }
    if constexpr (PARTS > 1) {
        if (mine > 0) sums[mine - 1][column] = s;
        __syncthreads();
        if (mine > 0) return;
#pragma unroll
        for (int j = 0; j < PARTS - 1; j++) s += sums[j][column];
    }
    C[row * D + d] = (_Float16)s;
}

// Largest accumulator count with an instantiated kernel that fits in `left`; wide: whether more than eight may be taken.
inline int pick_nw(int left, bool wide = true)
{
    const int opts[] = {32, 16, 8, 4, 2, 1};
    for (int o : opts)
        if (o <= left && (wide || o <= 8)) return o;
    return 1;
}

// Workgroups are handed to the chip's eight XCDs round-robin by their linear index, and every XCD has an L2 of its
// own: two workgroups that share cache lines - neighbours in memory - fetch them twice when they sit on different
// XCDs.  xcd_contiguous turns the linear index `id` of a launch of xcd_grid(n) workgroups into a logical index such
// that every XCD works through one contiguous eighth of the n logical workgroups; indices >= n are surplus
// workgroups that leave at once.  (Only traffic depends on the round-robin assumption, never results.)
inline int xcd_grid(int n) { return 8 * ((n + 7) / 8); }
#ifdef __HIPCC__
__device__ __forceinline__ int xcd_contiguous(int id, int n) { return (id & 7) * ((n + 7) >> 3) + (id >> 3); }
#endif

// Workgroup `index` of a value product over KV heads x nsplit token splits x nhalf (one or two) halves of the channels, the
// halves fastest; per_split: split_inverse(nsplit).  By general divisions, three in a row in front of a wavefront's first load,
// the indices took 0.2 - 0.4 us: four rows, 70 %, 2 heads x 512 tokens 4.63 -> 4.37 us, 64 x 4096 with 2 bits 12.04 -> 11.45.
struct ValueIndex {
    int half, split, kv;
};
inline uint32_t split_inverse(int nsplit) { return nsplit == 1 ? 0u : 0xFFFFFFFFu / (uint32_t)nsplit + 1u; }
#ifdef __HIPCC__
__device__ __forceinline__ ValueIndex value_index(int index, int nhalf, int nsplit, uint32_t per_split)
{
    const int rest = index >> (nhalf - 1);
    // rest / nsplit, exact while rest * nsplit < 2^32: plan_value gives all heads together at most 3072 splits more than there
    // are heads, so that 3000 splits of one head or two of each of 2^29 pass
    const int kv = nsplit == 1 ? rest : (int)__umulhi((uint32_t)rest, per_split);
    return {index & (nhalf - 1), rest - kv * nsplit, kv};
}
#endif

struct ValuePlan {
    int waves;   // wavefronts per workgroup
    int nbpw;    // token blocks per wavefront
    int nsplit;  // workgroups along the token axis
};

// most: splits that there is room for.
constexpr int kAnySplits = 0x7FFFFFFF;
inline ValuePlan plan_value(int Lc, int D, int Bkv, int nw, int most_splits = kAnySplits)
{
    ValuePlan p;
    const int nblk = Lc / 64;
    const long chunks = (long)nblk * (D / 64) * Bkv;
    p.waves = nw > 8 ? 4 : 8;
    if (nw > 8) {
        // 768 workgroups of four wavefronts fit the chip (their LDS leaves three per CU).  One to four turns of it, the
        // number with the shortest chain: the blocks that a wavefront walks in every turn, and about one more for the
        // turn's start and end.  Against as many blocks as 4096 wavefronts need at once (32 rows, 70 %, value product and
        // merge): 24 heads x 32704 tokens 57.4 -> 39.1 us, 128 x 4096 39.3 -> 34.9, 340 x 576 27.4 -> 15.5.
        const long heads = (long)(D / 64) * Bkv, most = (nblk + 3) / 4;
        long best = -1;
        for (long turns = 1; turns <= 4; turns++) {
            long ns = 768 * turns / heads;
            if (ns > most) ns = most;
            if (ns < 1) ns = 1;
            const long nb = (nblk + 4 * ns - 1) / (4 * ns);
            ns = (nblk + 4 * nb - 1) / (4 * nb);
            const long cost = (heads * ns + 767) / 768 * (nb + 1);
            if (best < 0 || cost < best) {
                best = cost;
                p.nbpw = (int)nb;
                p.nsplit = (int)ns;
            }
        }
        return p;
    }
    // aim at ~4096 resident wavefronts on 256 CUs, at least two token blocks each to pipeline
    long nb = (chunks + 4095) / 4096;
    if (nb < 1) nb = 1;
    if (nb > nblk) nb = nblk;
    const long room = ((long)nblk + (long)p.waves * most_splits - 1) / ((long)p.waves * most_splits);
    p.nbpw = (int)(nb > room ? nb : room);
    p.nsplit = (nblk + p.waves * p.nbpw - 1) / (p.waves * p.nbpw);
    return p;
}

// Launches the merge of rows [row0, row0+nw) of every KV head.
inline void launch_value_merge(hipStream_t st, const float* part, _Float16* C, int nsplit, int D, int rows_per_kv,
                               int row0, int nw, int Bkv)
{
    const size_t total = (size_t)Bkv * nw * D;
    if (nsplit > kMergeRow)
        hipLaunchKernelGGL(value_merge_kernel<kMergeParts>, dim3((unsigned)(total / (256 / kMergeParts))), dim3(256), 0, st, part,
                           C, nsplit, D, rows_per_kv, row0, nw, total);
    else
        hipLaunchKernelGGL(value_merge_kernel<1>, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, part, C, nsplit, D,
                           rows_per_kv, row0, nw, total);
}

// Splits of a value product that a workspace has room for, at least the one that takes none.
inline int splits_that_fit(size_t workspace_bytes, int head_dim, int Bq, int n_rows)
{
    const size_t fit = workspace_bytes / ((size_t)Bq * n_rows * head_dim * sizeof(float));
    return fit < 1 ? 1 : (fit < 1024 ? (int)fit : 1024);
}
// Workspace of a token-split value product (fp32 partials), 0 when no pass splits.  (Passes of eight rows in the place of a
// wide one, for unaligned weights, take no more splits than fit.)
inline size_t value_workspace_bytes(int head_dim, int tokens, int Bq, int groups, int n_rows)
{
    const int rows_per_kv = groups * n_rows;
    size_t worst = 0;
    for (int row0 = 0; row0 < rows_per_kv;) {
        const int nw = pick_nw(rows_per_kv - row0);
        const ValuePlan pl = plan_value(tokens, head_dim, Bq / groups, nw);
        const size_t need = pl.nsplit > 1 ? (size_t)Bq * n_rows * pl.nsplit * head_dim * sizeof(float) : 0;
        if (need > worst) worst = need;
        row0 += nw;
    }
    return round_up(worst, 256);
}

}  // namespace mstf
