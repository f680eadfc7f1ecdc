// Fused sparse decode attention over the quantised format: key SpMV -> scale + softmax -> value SpMV in one
// launch, with the work decomposition, softmax and combine of the fp16 kernel (fused.hip) and the staged
// dequantisation of the quantised SpMVs (quant_spmv.hip).
//
// A wavefront walks (KV head, 64-token) blocks: four stages of 32 key tiles, then four stages of 32 value
// tiles.  A stage's packed words and metadata arrive by LDS-direct loads one stage ahead (double buffers, across the
// blocks); the stage is dequantised into the wavefront's fp16 tile image and expanded from there.
#include "fused_common.hpp"
#include "step_device.hpp"

#ifndef MSTF_QPAD
#define MSTF_QPAD 16
#endif
#include "quant_device.hpp"

namespace mstf {

#pragma clang fp contract(off)

// Rows of the query and of the block weights sit 16 bytes further apart than their length: the four rows that the lanes
// of a group read together then start in different LDS banks.
constexpr int kQuantQRow = kFusedD * 2 + MSTF_QPAD;
// (Block weights as far apart as query rows where the LDS has room: the lanes' places in both are then one register.)
template <int NM>
constexpr int quant_prow()
{
    return NM == 1 ? kQuantQRow : 64 * 2 + MSTF_QPAD;
}
template <int NM, int BIT, bool G32>
constexpr int quant_wave_lds()
{
    // image, two word buffers, two metadata buffers; query rows; block weights; or the parked triple at the end
    constexpr int need = q_lds_bytes<BIT, G32>() + NM * 4 * (kQuantQRow + quant_prow<NM>());
    constexpr int park = NM * 4 * kFusedD * 4 + 64;
    return need > park ? need : park;
}
// Whether a wavefront may walk several blocks: with eight query heads the running output of the blocks before (sixteen
// registers) does not fit beside the rest.
template <int NM>
constexpr bool quant_multi()
{
    return NM == 1;
}
template <int NM, int BIT, bool G32>
constexpr int quant_occupancy()
{
    return resident_waves(kFusedWaves * quant_wave_lds<NM, BIT, G32>(), kFusedWaves);
}

// grid = (token splits, KV heads), kFusedWaves wavefronts, or (KV heads, token splits) with tokens_dev: the workgroups
// beyond the valid blocks are then dispatched last instead of standing in front of working ones.  Every wavefront walks
// the consecutive blocks that fused_blocks_of deals to it: with one each, a launch of more blocks than resident wavefronts paid the first memory round
// trips, the combine and the wait at its barrier once per block (256 heads x 4096 tokens, 2 bits: 64.8 -> 51.1 us).
// See decode_attention_kernel for the rest.  STEP: the launch is a whole
// decode step (st, the last argument; QuantKernargs mirrors the argument list and tells where it sits in the
// kernel-argument segment; step_device.hpp).
struct QuantKernargs {
    const void* first_ptrs[4];
    size_t tstride;
    const void* tokens_dev;
    int nblk, deal;
    const void* ptrs[12];
    int groups, nsplit, write_final;
    float sqrt_d;
    int mode;
    StepArgs st;
};
constexpr size_t kQuantStepArgsAt = offsetof(QuantKernargs, st);
// WHOLE: a workgroup of sixteen wavefronts takes both splits of a head and writes the output (fused_whole_head).
template <int NM, int BIT, bool G32>
constexpr bool quant_whole_fits()
{
    return NM == 1 && kWholeWaves * quant_wave_lds<NM, BIT, G32>() <= kWholeLds;
}
// SHARE (few blocks): workgroups of four wavefronts that share a block, a key stage and a value stage each (shared_scores,
// shared_store, fused_common.hpp); every block has a split slot then.  FOLDED: the sums of a stage start at zero and are added up in
// the order of the stages, as the wavefronts that share a block do it - the same numbers bit for bit - for a call that would share
// blocks and has no room for a slot per block.
constexpr int quant_waves(bool share, bool whole) { return whole ? kWholeWaves : (share ? kShare : kFusedWaves); }
template <int NM, int BIT, bool G32, bool MULTI, bool STEP = false, bool WHOLE = false, bool SHARE = false, bool FOLDED = false>
__global__ __launch_bounds__(quant_waves(SHARE, WHOLE) * 64) __attribute__((amdgpu_waves_per_eu(WHOLE ? 4 : quant_occupancy<NM, BIT, G32>()))) void decode_attention_quant_kernel(
    const uint32_t* __restrict__ k_off, const uint32_t* __restrict__ v_off, const uint64_t* __restrict__ k_bmp,
    const uint64_t* __restrict__ v_bmp, size_t tstride, const int* __restrict__ tokens_dev, int nblk, int deal,
    const uint32_t* k_packed, const uint32_t* k_off_dma, const uint16_t* k_scales, const uint16_t* k_zeros,
    const uint32_t* v_packed, const uint32_t* v_off_dma, const uint16_t* v_scales, const uint16_t* v_zeros,
    const _Float16* q, _Float16* __restrict__ out, float* __restrict__ part_o, float* __restrict__ part_ml, int groups,
    int nsplit, int write_final, float sqrt_d, int mode, StepArgs st)
{
    // Argument order: the first fourteen 32-bit words - what a wavefront's first loads need - are in scalar registers
    // when it starts (kernel-argument preload, a compile option of this library).
    // tstride: tiles between the per-tile rows of two heads - the tile count of the cached tokens unless the arrays are
    // pre-allocated for more.  tokens_dev (nullable): the number of cached tokens is read from device memory, at most
    // nblk blocks of it; the launch is then sized for the capacity.
    using F = QFmt<BIT>;
    const int blocks_room = nblk;  // (SHARE: split slots of blocks)
    if (tokens_dev) {
        const int valid = *tokens_dev / 64;
        nblk = valid < nblk ? valid : nblk;
        // the blocks a wavefront walks follow from the tokens that are there now, as a launch sized for exactly them
        // would choose; the workgroups behind the last block leave neutral partials
        if (MULTI) deal = fused_deal(nblk, fused_splits(nblk, fused_fill_unpack(deal)));
    }
    constexpr int D = kFusedD;
    constexpr int kQRow = kQuantQRow, kPRow = quant_prow<NM>();
    constexpr int kQLds = NM * 4 * kQRow;
    constexpr int kMetaBytes = meta_bytes<G32>();
    constexpr int kStage = q_lds_bytes<BIT, G32>();  // image, two word buffers, two metadata buffers
    constexpr int kWaveLds = quant_wave_lds<NM, BIT, G32>();
    // one array on purpose (LDS-direct loads into several LDS objects make the compiler serialise them)
    __shared__ __attribute__((aligned(16))) char lds_all[quant_waves(SHARE, WHOLE) * kWaveLds];
    static_assert(!SHARE || (!MULTI && !WHOLE && kKeySubs == kShare), "a stage of each side per wavefront of a shared block");
    static_assert(!SHARE || (kQLds >= NM * 1024 && kImgBytes >= NM * 1024), "room for the sums that the wavefronts exchange");
    static_assert(!WHOLE || (!STEP && fused_park_bytes<NM>() + NM * 2048 <= kWaveLds), "room behind the parked triples");
    const int lane = lane_id();
    const int wave = wave_id();
    // (WHOLE: the first eight wavefronts do what the workgroup of the first split would, the others the second's)
    const int split = WHOLE ? wave / kFusedWaves : (tokens_dev ? (int)blockIdx.y : (int)blockIdx.x);
    const int kv = tokens_dev ? (int)blockIdx.x : (int)blockIdx.y;
    const int slot = WHOLE ? wave % kFusedWaves : wave;
    const int sub = SHARE ? wave : 0;                                 // its stages of the block
    BlockRange mine = {SHARE ? split : split * kFusedWaves + slot, 0};  // the token blocks of this wavefront
    if constexpr (MULTI) mine = fused_blocks_of(nblk, deal, split, slot);
    const int tb = mine.first, nb = MULTI ? mine.count : nblk - tb;   // (wave-uniform)
    const bool active = nb > 0;
    const size_t T = tstride;
    char* my = lds_all + wave * kWaveLds;
    char* wordbuf = my + kImgBytes;
    char* metabuf = wordbuf + 2 * F::kWordBuf;
    char* ql = my + kStage;
    char* pl = ql + kQLds;
    const uint32_t lbase = lds_addr(my);

    if constexpr (STEP && SHARE) {
        // (the blocks of the dense window get workgroups of their own behind the splits, see decode_attention_kernel)
        if (split >= st.wg0) {
            const int wblk = (split - st.wg0) * kShare + wave;
            if (wblk < (st.win_len + 63) / 64) {
                stage_query_rotated<kQRow>(ql, st, kv, groups, lane);
                step_window_wave<NM, kQRow, kPRow, 8>(my, ql, pl, st, part_o, part_ml, kv, groups, nsplit, wblk, step_window_count(st),
                                                      sqrt_d, lane);
            }
            return;  // (the whole workgroup: no barrier is left waiting)
        }
    }
    if constexpr (SHARE) {
        if (!active) {  // (wave-uniform, and the same for the workgroup)
            if (wave == 0 && tb < blocks_room)
                store_neutral<NM>(lane, groups, (size_t)kv * groups * nsplit + tb, nsplit, part_o, part_ml);
            return;
        }
    }

    f4_t acc_v[NM][2];
    float m_run[NM], l_run[NM];
#pragma unroll
    for (int m = 0; m < NM; m++) {
        acc_v[m][0] = f4_t{0.f, 0.f, 0.f, 0.f};
        acc_v[m][1] = f4_t{0.f, 0.f, 0.f, 0.f};
        m_run[m] = -INFINITY;
        l_run[m] = 0.f;
    }

    if (active) {
        const size_t tile0 = (size_t)kv * T + (size_t)tb * D;  // tile_off / scales / zeros / bmp are flat over [Bkv, T]
        constexpr size_t kPairs = G32 ? 2 : 1;  // (scale, zero) pairs per tile
        const uint64_t *bmK = k_bmp + tile0, *bmV = v_bmp + tile0;
        const uint32_t *offK = k_off + tile0, *offV = v_off + tile0;
        // Word offsets at the stage boundaries of both sides of a block by one vector load (lanes 0 .. 3 keys, 16 .. 19
        // values, each side's last tile one lane further on); the block's last stage ends where its last tile's words
        // end, which takes that tile's bitmap: a second load.  Requested for the coming block while the current one is
        // expanded; bound() makes the boundaries of it.
        const int bnd_l = lane & 15;
        const int bnd_i = bnd_l < kKeySubs ? bnd_l * kSubTiles : (bnd_l == kKeySubs ? D - 1 : 0);
        static_assert(kKeySubs == kValSubs && kKeySubs < 15, "boundary lanes");
        struct Raw {
            uint32_t off;
            uint2 last;
        };
        auto bounds_of = [&](const uint32_t* ok, const uint32_t* ov, const uint64_t* bk, const uint64_t* bv) {
            Raw r;
            r.off = *((lane < 16 ? ok : ov) + bnd_i);
            r.last = *reinterpret_cast<const uint2*>((lane < 16 ? bk : bv) + (D - 1));
            return r;
        };
        auto bound = [&](const Raw& r) {
            const uint32_t words = ((uint32_t)__builtin_popcount(r.last.x) + (uint32_t)__builtin_popcount(r.last.y) +
                                    (uint32_t)F::kCap - 1u) >> F::kCapShift;
            return r.off + (bnd_l == kKeySubs ? words : 0u);
        };
        uint32_t bnd = bound(bounds_of(offK, offV, bmK, bmV));
        const size_t tile1 = tile0 + (size_t)sub * kSubTiles;
        MetaLanes metaK = meta_lanes<G32>(k_off_dma + tile1, k_scales + tile1 * kPairs, k_zeros + tile1 * kPairs, k_bmp + tile1, lane);
        MetaLanes metaV = meta_lanes<G32>(v_off_dma + tile1, v_scales + tile1 * kPairs, v_zeros + tile1 * kPairs, v_bmp + tile1, lane);
        const uint32_t lane4 = (uint32_t)lane * 4u;
        using Rank = StageRank<4 * NM, BIT, G32, false>;
        const uint32_t bits_at = Rank::bits_at(lane);
        const uint32_t wordbuf_lds = lds_addr(wordbuf);
        auto start_of = [&](int n) { return (uint32_t)__builtin_amdgcn_readlane(bnd, n < kKeySubs ? n : 16 + n - kKeySubs); };
        auto end_of = [&](int n) { return (uint32_t)__builtin_amdgcn_readlane(bnd, n < kKeySubs ? n + 1 : 17 + n - kKeySubs); };
        // (no lane-dependent branches: every piece is issued with exec set by hand or from a clamped address)
        auto issue = [&](int n) {
            const uint64_t* bm = n < kKeySubs ? bmK : bmV;
            const int t = (n < kKeySubs ? n : n - kKeySubs) * kSubTiles;
            const uint32_t s = start_of(n);
            uint32_t nw = end_of(n) - s;
            nw = nw > (uint32_t)F::kWordsMax ? (uint32_t)F::kWordsMax : nw;  // never true for a well-formed cache
            words_issue_flat<F::kWordsMax / 64>((n < kKeySubs ? k_packed : v_packed) + s, nw,
                                                wordbuf_lds + (uint32_t)(n & 1) * F::kWordBuf, (uint32_t)lane, lane4);
            // metadata: lanes 0..31 the word offsets, 32..47 the scales, 48..63 the zero-points (two per lane)
            meta_issue_next<G32>(n < kKeySubs ? metaK : metaV, metabuf + (n & 1) * kMetaBytes);
            // the stage's bitmaps (and the scalar loads of the expansion find them in L2)
            return Rank::bits_load(bm + t, bits_at);
        };

        Rank rank(lds_addr(metabuf), wordbuf_lds, lbase, lane);

        // the query rows of this KV head: groups x D fp16, contiguous (STEP: rotated out of the projection output)
        if constexpr (STEP) {
            stage_query_rotated<kQRow>(ql, st, kv, groups, lane);
        } else {
            const char* qsrc = reinterpret_cast<const char*>(q + (size_t)kv * groups * D);
            // a row per load: sixteen lanes fetch the 256 bytes of query row `row`, four rows per pass
            const int row_in_pass = lane >> 4;
#pragma unroll
            for (int i = 0; i < NM; i++) {
                const int row = i * 4 + row_in_pass;
                const uint4 v = row < groups ? *reinterpret_cast<const uint4*>(qsrc + row * (D * 2) + (lane & 15) * 16)
                                             : make_uint4(0u, 0u, 0u, 0u);
                *reinterpret_cast<uint4*>(ql + row * kQRow + (lane & 15) * 16) = v;
            }
        }
        typename Rank::Sums sums;  // of the phase (keys, one half of the values, the other half)
        const uint32_t qrow = sums.waddr(lds_addr(ql), kQRow, lane);
        const uint32_t prow = kPRow == kQRow ? qrow + (uint32_t)kQLds : sums.waddr(lds_addr(pl), kPRow, lane);
        if constexpr (SHARE) {
            // Both stages are requested at once: one round trip behind the boundaries'.
            const uint64_t* bm[2] = {k_bmp + tile1, v_bmp + tile1};
            uint32_t start[2], end[2];
            uint2 bits[2];
#pragma unroll
            for (int i = 0; i < 2; i++) {
                start[i] = (uint32_t)__builtin_amdgcn_readlane((int)bnd, 16 * i + sub);
                end[i] = (uint32_t)__builtin_amdgcn_readlane((int)bnd, 16 * i + sub + 1);
                uint32_t nw = end[i] - start[i];
                nw = nw > (uint32_t)F::kWordsMax ? (uint32_t)F::kWordsMax : nw;  // never true for a well-formed cache
                words_issue_flat<F::kWordsMax / 64>((i == 0 ? k_packed : v_packed) + start[i], nw,
                                                    wordbuf_lds + (uint32_t)i * F::kWordBuf, (uint32_t)lane, lane4);
                meta_issue_next<G32>(i == 0 ? metaK : metaV, metabuf + i * kMetaBytes);
                bits[i] = Rank::bits_load(bm[i], bits_at);
            }
            asm volatile("s_waitcnt vmcnt(0)" : "+v"(bits[0].x), "+v"(bits[0].y), "+v"(bits[1].x), "+v"(bits[1].y)::"memory");
            f4_t part[NM], acc_k[NM];
            float m_blk[NM], l_blk[NM];
            auto stage = [&](int i, uint32_t w, uint32_t wgroup) {
                const StageAt here = {lds_addr(metabuf), wordbuf_lds, (uint32_t)i * kMetaBytes, (uint32_t)i * F::kWordBuf, start[i],
                                      end[i]};
                rank.template stage<true>(here, bm[i], bits[i], w, wgroup, sums, lane, mode);
#pragma unroll
                for (int m = 0; m < NM; m++) part[m] = sums.joined(m);
                wait_lgkm0();
            };
            stage(0, qrow + (uint32_t)(sub * kSubTiles * 2), 4u * kQRow);
            shared_scores<NM>(lds_all + kStage, kWaveLds, sub, lane, part, acc_k);  // (the query rows have been read)
            block_softmax<NM, kPRow>(acc_k, sqrt_d, 64, pl, lane, m_blk, l_blk);
            stage(1, prow + (uint32_t)((sub & 1) * kSubTiles * 2), 4u * kPRow);
            shared_store<NM>(lds_all, kWaveLds, sub, lane, part, m_blk, l_blk, groups, (size_t)kv * groups * nsplit + tb, nsplit,
                             part_o, part_ml);  // (the image has been read, and only by this wavefront)
            return;
        }
        uint2 touch = issue(0);

#pragma unroll 1
        for (int r = 0; r < (MULTI ? nb : 1); r++) {
            const bool more = MULTI && r + 1 < nb;
            float fb[NM];
            f4_t acc_k[NM], blk[NM];  // scores; a half of the block's output
            Raw coming;
            uint32_t bnd_next = bnd;
            static_for<kKeySubs + kValSubs>([&](auto nc) {
                constexpr int n = decltype(nc)::value;
                // 3, 2, 1, 0 over the key stages and again over the value stages (keeping the wavefronts that also take a
                // block of the dense window at 3, as the fp16 kernel does, measured slower here)
                set_wave_priority(3 - n % 4);
                asm volatile("s_waitcnt vmcnt(0)" : "+v"(touch.x), "+v"(touch.y)::"memory");  // stage n has landed
                const uint2 bits = touch;
                const uint32_t start = start_of(n), end = end_of(n);
                const uint64_t* bm = (n < kKeySubs ? bmK : bmV) + (n < kKeySubs ? n : n - kKeySubs) * kSubTiles;
                if (n + 1 < kKeySubs + kValSubs) {
                    touch = issue(n + 1);
                } else if (MULTI) {
                    // the coming block of this wavefront: its boundaries have arrived, its first stage goes out while the
                    // last one of this block is expanded
                    bnd_next = bound(coming);
                    if (more) {
                        bnd = bnd_next;
                        bmK += D, bmV += D, offK += D, offV += D;
                        touch = issue(0);
                    }
                }
                if (n == kKeySubs) {
                    if constexpr (!FOLDED) {
#pragma unroll
                        for (int m = 0; m < NM; m++) acc_k[m] = sums.joined(m);
                    }
                    float m_blk[NM], l_blk[NM];
                    block_softmax<NM, kPRow>(acc_k, sqrt_d, 64, pl, lane, m_blk, l_blk);
                    // (the fold of the block begins here, so that nothing of it waits in registers beside the running output)
#pragma unroll
                    for (int m = 0; m < NM; m++) {
                        if constexpr (MULTI) {
                            const Folded f(m_run[m], l_run[m], m_blk[m], l_blk[m]);
                            fb[m] = f.fb;
#pragma unroll
                            for (int h = 0; h < 2; h++)
#pragma unroll
                                for (int c = 0; c < 4; c++) acc_v[m][h][c] *= f.fa;
                        } else {
                            m_run[m] = m_blk[m];
                            l_run[m] = l_blk[m];
                        }
                    }
                    const int adv = more ? D : 0;
                    if (MULTI) coming = bounds_of(offK + adv, offV + adv, bmK + adv, bmV + adv);
                }
                constexpr int vs = n - kKeySubs;  // value stage: half = vs / 2, tokens (vs % 2) * 32..
                constexpr int kSubsPerHalf = 64 / kSubTiles;
                const uint32_t w = n < kKeySubs ? qrow + (uint32_t)n * kSubTiles * 2u
                                                : prow + (uint32_t)(vs % kSubsPerHalf) * kSubTiles * 2u;
                const StageAt here = {lds_addr(metabuf), wordbuf_lds, (uint32_t)(n & 1) * kMetaBytes, (uint32_t)(n & 1) * F::kWordBuf,
                                      start, end};
                constexpr bool kStarts = FOLDED || n == 0 || n == kKeySubs || n == kKeySubs + kSubsPerHalf;
                rank.template stage<kStarts>(here, bm, bits, w, n < kKeySubs ? 4u * kQRow : 4u * kPRow, sums, lane, mode);
                if constexpr (FOLDED) {
                    f4_t(&to)[NM] = n < kKeySubs ? acc_k : blk;
#pragma unroll
                    for (int m = 0; m < NM; m++) {
                        if constexpr (n == 0 || (n >= kKeySubs && vs % kSubsPerHalf == 0)) to[m] = sums.joined(m);
                        else to[m] += sums.joined(m);
                    }
                }
                if (n >= kKeySubs && vs % kSubsPerHalf == kSubsPerHalf - 1) {  // the half is complete
#pragma unroll
                    for (int m = 0; m < NM; m++) {
                        if constexpr (!FOLDED) blk[m] = sums.joined(m);
                        f4_t& out_v = acc_v[m][vs / kSubsPerHalf];
#pragma unroll
                        for (int c = 0; c < 4; c++) out_v[c] = MULTI ? out_v[c] + blk[m][c] * fb[m] : blk[m][c];
                    }
                }
                wait_lgkm0();  // every read of the image and of the staged buffers is done before they are rewritten
            });
        }
    }
    if constexpr (STEP && !SHARE) {
        // The dense window: block i goes to wavefront number i / ns of split i % ns, behind its compressed block (see
        // decode_attention_kernel); the value rows pass through the room of the tile image, eight at a time.  The
        // step's arguments are fetched again here, through a pointer the compiler cannot see through, so that they
        // hold no scalar registers above.
        static_assert(2 * 8 * D * 2 <= kImgBytes, "two buffers of eight value rows in the room of the image");
        const StepArgs __attribute__((address_space(4)))* sp = (const StepArgs __attribute__((address_space(4)))*)(
            (const char __attribute__((address_space(4)))*)__builtin_amdgcn_kernarg_segment_ptr() + kQuantStepArgsAt);
        asm volatile("" : "+s"(sp));
        StepArgs sw;
        sw.q_in = sp->q_in, sw.k_in = sp->k_in, sw.v_in = sp->v_in;
        sw.q_stride = sp->q_stride, sw.k_stride = sp->k_stride, sw.v_stride = sp->v_stride;
        sw.cos = sp->cos, sw.sin = sp->sin, sw.rope_stride = sp->rope_stride;
        sw.k_win = sp->k_win, sw.v_win = sp->v_win, sw.win_len_dev = sp->win_len_dev, sw.overflow = sp->overflow;
        sw.win_len = sp->win_len, sw.win_stride = sp->win_stride, sw.n_kv = sp->n_kv, sw.ns = sp->ns;
        const int count = step_window_count(sw);
        const int order = fused_window_order(nblk, MULTI ? deal : kFusedWaves, split, wave, step_window_rows(sw, count), sw.ns);
        const int wblk = step_window_block(sw.ns, order, split);
        if (wblk < (sw.win_len + 63) / 64) {
            if (!active) stage_query_rotated<kQRow>(ql, sw, kv, groups, lane);
            step_window_wave<NM, kQRow, kPRow, 8>(my, ql, pl, sw, part_o, part_ml, kv, groups, nsplit, wblk, count, sqrt_d, lane);
        }
    }
    if constexpr (WHOLE)
        combine_whole_head<NM>(lds_all, kWaveLds, wave, lane, acc_v, m_run, l_run, kv, groups, out);
    else
        workgroup_combine<NM>(lds_all, kWaveLds, wave, lane, acc_v, m_run, l_run, kv, groups, split, nsplit, write_final, out,
                              part_o, part_ml);
}

template <int NM, int BIT>
static void launch_decode_quant(hipStream_t st, dim3 grid, const uint64_t* k_bmp, const uint32_t* k_packed,
                                const uint32_t* k_off, const uint16_t* k_scales, const uint16_t* k_zeros,
                                const uint64_t* v_bmp, const uint32_t* v_packed, const uint32_t* v_off,
                                const uint16_t* v_scales, const uint16_t* v_zeros, const _Float16* q, _Float16* out,
                                float* part_o, float* part_ml, int tokens, int groups, int ns, int write_final, float sq,
                                int mode, int group_size, size_t tstride, const int32_t* tokens_dev, int deal,
                                bool one_block, const StepArgs* step, bool whole, bool shared, bool folded)
{
    const StepArgs sa = step ? *step : StepArgs{};
    const unsigned threads = 64 * (unsigned)quant_waves(shared, whole);
#define MSTF_FQ_LAUNCH(...)                                                                                              \
    hipLaunchKernelGGL((decode_attention_quant_kernel<NM, BIT, __VA_ARGS__>), grid, dim3(threads), 0, st, k_off, \
                       v_off, k_bmp, v_bmp, tstride, tokens_dev, tokens / 64, deal, k_packed, k_off, k_scales, k_zeros,   \
                       v_packed, v_off, v_scales, v_zeros, q, out, part_o, part_ml, groups, ns, write_final, sq, mode, sa)
    // With one block per wavefront the form for one where it is the faster one: 280 to 1696 blocks, 70 - 75 %, fused attention in
    // the form for several / for one: 4 bits 16.4 / 15.4 us (two groups per tile 18.4 / 17.7), 8 bits 17.8 / 17.5 (20.1 / 20.6),
    // 2 bits 14.4 / 14.6 (17.4 / 16.5; 4096 blocks, one group: 17.9 / 18.3).
    constexpr bool kMulti = quant_multi<NM>(), kOne = kMulti && BIT == 2, kOneG32 = kMulti && BIT == 8;
    if (shared) {
        if (step) MSTF_FQ_LAUNCH(false, false, true, false, true);
        else if (group_size == 32) MSTF_FQ_LAUNCH(true, false, false, false, true);
        else MSTF_FQ_LAUNCH(false, false, false, false, true);
        return;
    }
    if (folded) {  // (so few blocks that no wavefront has more than one)
        if (step) MSTF_FQ_LAUNCH(false, false, true, false, false, true);
        else if (group_size == 32) MSTF_FQ_LAUNCH(true, false, false, false, false, true);
        else MSTF_FQ_LAUNCH(false, false, false, false, false, true);
        return;
    }
    if constexpr (quant_whole_fits<NM, BIT, false>()) {
        if (whole && group_size == 64) {
            if (one_block) MSTF_FQ_LAUNCH(false, kOne, false, true); else MSTF_FQ_LAUNCH(false, kMulti, false, true);
            return;
        }
    }
    if constexpr (quant_whole_fits<NM, BIT, true>()) {
        if (whole) {
            if (one_block) MSTF_FQ_LAUNCH(true, kOneG32, false, true); else MSTF_FQ_LAUNCH(true, kMulti, false, true);
            return;
        }
    }
    if (step) {  // (group_size is 64 there: quant_launch has checked it)
        if (one_block) MSTF_FQ_LAUNCH(false, kOne, true); else MSTF_FQ_LAUNCH(false, kMulti, true);
    } else if (group_size == 32) {
        if (one_block) MSTF_FQ_LAUNCH(true, kOneG32); else MSTF_FQ_LAUNCH(true, kMulti);
    } else {
        if (one_block) MSTF_FQ_LAUNCH(false, kOne); else MSTF_FQ_LAUNCH(false, kMulti);
    }
#undef MSTF_FQ_LAUNCH
}

}  // namespace mstf

using namespace mstf;

// Shared argument checks of the quantised fused entry points.
static int quant_check(const void* k_bmp, const void* k_packed, const void* k_tile_off, const void* k_scales,
                       const void* k_zeros, const void* v_bmp, const void* v_packed, const void* v_tile_off,
                       const void* v_scales, const void* v_zeros, const void* q, int tokens, int head_dim, int Bq,
                       int groups, int bit, int capacity, int dequant_mode)
{
    if (!k_bmp || !k_packed || !k_tile_off || !k_scales || !k_zeros || !v_bmp || !v_packed || !v_tile_off || !v_scales ||
        !v_zeros || !q)
        return MSTF_EINVAL;
    if (tokens <= 0 || Bq <= 0 || groups <= 0 || Bq % groups != 0) return MSTF_EINVAL;
    if (dequant_mode != 0 && dequant_mode != 1) return MSTF_EINVAL;
    if (bit != 2 && bit != 4 && bit != 8) return MSTF_EUNSUPPORTED;
    if (capacity != 32 / bit) return MSTF_EINVAL;
    if (head_dim != kFusedD || tokens % 64 != 0 || groups > 8) return MSTF_EUNSUPPORTED;
    if (!aligned_to(k_bmp, 8) || !aligned_to(v_bmp, 8) || !aligned_to(k_packed, 4) || !aligned_to(v_packed, 4) ||
        !aligned_to(k_tile_off, 4) || !aligned_to(v_tile_off, 4) || !aligned_to(k_scales, 4) || !aligned_to(v_scales, 4) ||
        !aligned_to(k_zeros, 4) || !aligned_to(v_zeros, 4) || !aligned_to(q, 16))
        return MSTF_EALIGN;
    return MSTF_OK;
}

// Wavefronts of the quantised kernel that the chip holds at once (its LDS differs by width and group size), or more than
// any launch has where a wavefront walks one block only.
static int quant_resident(int groups, int bit, int group_size)
{
    if (groups > 4) return 0x40000000;
    static_assert(quant_multi<1>() && !quant_multi<2>(), "groups of more than four heads: one block per wavefront");
    const bool g32 = group_size == 32;
    return 1024 * (bit == 2   ? (g32 ? quant_occupancy<1, 2, true>() : quant_occupancy<1, 2, false>())
                   : bit == 4 ? (g32 ? quant_occupancy<1, 4, true>() : quant_occupancy<1, 4, false>())
                              : (g32 ? quant_occupancy<1, 8, true>() : quant_occupancy<1, 8, false>()));
}
// Whether sixteen wavefronts of the kernel fit a workgroup (up to four query heads).
static bool quant_whole(int bit, int group_size)
{
    const bool g32 = group_size == 32;
    return bit == 2   ? (g32 ? quant_whole_fits<1, 2, true>() : quant_whole_fits<1, 2, false>())
           : bit == 4 ? (g32 ? quant_whole_fits<1, 4, true>() : quant_whole_fits<1, 4, false>())
                      : (g32 ? quant_whole_fits<1, 8, true>() : quant_whole_fits<1, 8, false>());
}
// Split slots its launch fills for `tokens` tokens, or for any count up to that many (at most fused_nsplit(tokens), which
// is what workspaces are sized for).  window: blocks of the dense window.
static int quant_nsplit(int tokens, int Bkv, int groups, int bit, int group_size, int window = 0)
{
    return fused_splits_step(tokens / 64, fused_fill(Bkv, quant_resident(groups, bit, group_size)), window);
}

// KV heads whose blocks, up to eight of each, the chip holds at once with a wavefront per block: its workgroups of kFusedWaves.
static int quant_heads_at_once(int groups, int bit, int group_size)
{
    if (groups <= 4) return quant_resident(groups, bit, group_size) / kFusedWaves;
    const bool g32 = group_size == 32;
    return 1024 / kFusedWaves * (bit == 2   ? (g32 ? quant_occupancy<2, 2, true>() : quant_occupancy<2, 2, false>())
                                 : bit == 4 ? (g32 ? quant_occupancy<2, 4, true>() : quant_occupancy<2, 4, false>())
                                            : (g32 ? quant_occupancy<2, 8, true>() : quant_occupancy<2, 8, false>()));
}
// Whether four wavefronts share a block, where blocks are few (fused_shares_blocks).  merged: the call has splits to merge
// without that too: a window, or (max, sum) asked for.
// Nearly always, also where one split would leave no merge to launch behind it: with three quarters of the stages gone from a
// wavefront's chain the two launches are the faster form, call by call and recorded alike (us, 70 %, a wavefront per block / shared;
// recorded unless said: 2 bits, 8 heads x 2 blocks 12.2 / 9.1, call by call 10.9 / 10.3, 8 x 8 13.2 / 9.1, 12.0 / 10.5, 8 x 16 15.3 / 9.2, 24 x 32
// 15.3 / 11.8, 16 x 64 15.5 / 13.5, 8 x 128 15.8 / 15.1, eight query heads 8 x 16 16.8 / 10.1, 8 x 96 17.3 / 14.8; 8 bits, two groups, eight
// query heads 22.3 / 11.5; a step with a window of 300: 2 bits 8 x 8 21.6 / 11.7, 24 x 32 19.8 / 15.6, 8 bits 8 x 60 23.3 / 15.0).
// Not for many heads of one to four blocks that are all there at once anyway: workgroups of all blocks come one behind the other then,
// and the merge launches for every query row.  The more query heads and the fewer bits, the sooner that is so (a wavefront
// per block / shared: 2 bits, four query heads 256 x 4 10.9 / 11.7, 448 x 2 11.7 / 12.2, but 192 x 4 10.8 / 10.4; eight 512 x 1 12.2 / 14.2, 384 x 1
// 12.2 / 12.4, 256 x 3 12.0 / 13.2, 192 x 3 11.9 / 12.3, but 128 x 4 12.0 / 10.3, 160 x 3 11.8 / 10.8; 8 bits, four 256 x 4 14.1 / 14.9; 4 bits, eight
// 256 x 3 13.2 / 13.6, 192 x 3 12.9 / 12.7; a 2-bit step of 384 heads of one block, eight query heads, window of 256 23.1 / 25.6), while heads for
// which the chip has no room at once gain by a factor (8 bits, 300 x 1 24.3 / 9.9).
static bool quant_shares(int tokens, int Bkv, int groups, int bit, int group_size, int window, bool merged)
{
    const int nblk = tokens / 64, wgs = Bkv * (nblk + (window_blocks(window) + kShare - 1) / kShare);
    if (nblk > 4 || Bkv > quant_heads_at_once(groups, bit, group_size)) return true;
    if (merged) return nblk > 1 || bit > 2 || window_blocks(window) < 4 || groups * wgs < 4608;
    if (groups <= 4) return bit == 4 || wgs <= 768 || groups == 1 || (groups == 2 && bit == 2);
    if (bit == 8 || (group_size == 32 && (bit == 4 || nblk > 1))) return true;
    const bool least = bit == 2 && group_size == 64;
    const int most = least ? 4096 : 5376;  // query heads x blocks
    return nblk == 1 ? 3 * groups * wgs < 2 * most : groups * wgs <= most && (!least || wgs <= 640);
}
// How a launch takes its blocks: shared by four wavefronts, a split slot each, where they are few; without room for those slots, or
// where the shared form is the slower one (folded), the same numbers come from a wavefront per block, in no more time than from sums
// that run through the stages (8 heads x 16 blocks, running / folded: 2 / 4 / 8 bits 13.4 / 14.6 / 16.5, 12.4 / 14.5 / 16.4; eight query heads
// 15.1 / 16.1 / 18.1, 15.2 / 16.0 / 17.9) but with 2 bits, two groups and more than four query heads, whose folded form spills registers (16.9,
// 17.8; the half of the output that is done parked in LDS, the metadata's addresses made late or anew: three to eleven still spill).
// window: tokens of the dense window behind them.
struct QuantPlan {
    bool shared, folded;
    int ns;
    int merge_blocks() const { return shared ? ns : 0; }
};
static QuantPlan quant_plan(int tokens, int Bq, int groups, int bit, int group_size, int window, int window_in_launch,
                            bool merged, size_t workspace_bytes)
{
    const int Bkv = Bq / groups;
    const bool few = fused_shares_blocks(tokens, Bkv, groups, Bkv * ((window_blocks(window) + kShare - 1) / kShare));
    if (few && quant_shares(tokens, Bkv, groups, bit, group_size, window, merged) && fused_share_fits(tokens, window, Bq, workspace_bytes))
        return {true, false, tokens / 64};
    return {false, few, quant_nsplit(tokens, Bkv, groups, bit, group_size, window_blocks(window_in_launch))};
}

// The quantised kernel over the compressed tokens: fills split slots 0 .. ns-1 (ns: quant_nsplit) of a workspace
// with nst slots per query row (or writes the final output when write_final).
static int quant_launch(hipStream_t st, const uint64_t* k_bmp, const uint32_t* k_packed, const uint32_t* k_tile_off,
                        const mstf_half* k_scales, const mstf_half* k_zeros, const uint64_t* v_bmp,
                        const uint32_t* v_packed, const uint32_t* v_tile_off, const mstf_half* v_scales,
                        const mstf_half* v_zeros, const mstf_half* q, mstf_half* out, int tokens, int head_dim, int Bq,
                        int groups, int bit, int dequant_mode, void* workspace, int ns, int nst, int write_final,
                        int group_size = 64, size_t tile_stride = 0, const int32_t* tokens_dev = nullptr,
                        const StepArgs* step = nullptr, bool whole = false, bool shared = false, bool folded = false)
{
    const int Bkv = Bq / groups;
    // (token count in device memory: the kernel deals the blocks out itself, from the number of workgroups that fill the chip)
    const FusedFill fill = fused_fill(Bkv, quant_resident(groups, bit, group_size));
    const int deal = tokens_dev ? fused_fill_pack(fill) : fused_deal(tokens / 64, ns);
    // no wavefront has more than one block (and none has with fewer tokens, should their number be in device memory)
    const bool one_block = fused_splits(tokens / 64, fill) == fused_nsplit(tokens);
    // step: the launch is a whole decode step; its window blocks are dealt out over the wavefronts of a head
    // (or get workgroups of their own behind those of shared blocks, which a call may go without: they take no longer windows)
    const int window = step ? window_blocks(step->win_len) : 0;
    const int walks = shared && step ? quant_nsplit(tokens, Bkv, groups, bit, group_size, window) : ns;
    if (step && (group_size != 64 || window > walks * kFusedWaves)) return MSTF_EUNSUPPORTED;
    const int wgs = ns + (shared ? (window + kShare - 1) / kShare : 0);
    // tile_stride / tokens_dev: a cache pre-allocated for `tokens` tokens that holds *tokens_dev of them (see the kernel)
    float* part_o = reinterpret_cast<float*>(workspace);
    float* part_ml = part_o + (size_t)Bq * nst * head_dim;
    const dim3 grid = tokens_dev ? dim3((unsigned)Bkv, (unsigned)wgs) : dim3(whole ? 1u : (unsigned)wgs, (unsigned)Bkv);
    const size_t tstride = tile_stride ? tile_stride : (size_t)tokens * head_dim / 64;
    const _Float16* qh = reinterpret_cast<const _Float16*>(q);
    _Float16* oh = reinterpret_cast<_Float16*>(out);
    const float sq = sqrtf((float)head_dim);
    const uint16_t* ks = reinterpret_cast<const uint16_t*>(k_scales);
    const uint16_t* kz = reinterpret_cast<const uint16_t*>(k_zeros);
    const uint16_t* vs = reinterpret_cast<const uint16_t*>(v_scales);
    const uint16_t* vz = reinterpret_cast<const uint16_t*>(v_zeros);
#define MSTF_FQ(NMV, BITV)                                                                                             \
    launch_decode_quant<NMV, BITV>(st, grid, k_bmp, k_packed, k_tile_off, ks, kz, v_bmp, v_packed, v_tile_off, vs, vz, \
                                   qh, oh, part_o, part_ml, tokens, groups, nst, write_final, sq, dequant_mode, group_size, \
                                   tstride, tokens_dev, deal, one_block, step, whole, shared, folded)
    if (groups <= 4) {
        if (bit == 2) MSTF_FQ(1, 2); else if (bit == 4) MSTF_FQ(1, 4); else MSTF_FQ(1, 8);
    } else {
        if (bit == 2) MSTF_FQ(2, 2); else if (bit == 4) MSTF_FQ(2, 4); else MSTF_FQ(2, 8);
    }
#undef MSTF_FQ
    return check_launch();
}

static int decode_attention_quant_impl(void* stream, const uint64_t* k_bmp, const uint32_t* k_packed,
                                       const uint32_t* k_tile_off, const mstf_half* k_scales, const mstf_half* k_zeros,
                                       const uint64_t* v_bmp, const uint32_t* v_packed, const uint32_t* v_tile_off,
                                       const mstf_half* v_scales, const mstf_half* v_zeros, const mstf_half* q,
                                       mstf_half* out, float* lse_out, int tokens, int head_dim, int Bq, int groups,
                                       int bit, int capacity, int dequant_mode, int group_size, void* workspace,
                                       size_t workspace_bytes)
{
    if (!out) return MSTF_EINVAL;
    if (group_size != 64 && group_size != 32) return MSTF_EUNSUPPORTED;
    int rc = quant_check(k_bmp, k_packed, k_tile_off, k_scales, k_zeros, v_bmp, v_packed, v_tile_off, v_scales, v_zeros, q,
                         tokens, head_dim, Bq, groups, bit, capacity, dequant_mode);
    if (rc != MSTF_OK) return rc;
    if (!aligned_to(out, 2) || (lse_out && !aligned_to(lse_out, 4))) return MSTF_EALIGN;
    if (!workspace || workspace_bytes < fused_workspace_need(tokens, 0, Bq)) return MSTF_EWORKSPACE;
    if (!aligned_to(workspace, 16)) return MSTF_EALIGN;
    hipStream_t st = as_stream(stream);
    const QuantPlan plan = quant_plan(tokens, Bq, groups, bit, group_size, 0, 0, lse_out || tokens > kFusedWaves * 64, workspace_bytes);
    const int ns = plan.ns;
    // with one split and no (max, sum) requested the kernel writes the final output itself
    // (and with a workgroup per head)
    const bool whole = !plan.shared && !lse_out && quant_whole(bit, group_size) && fused_whole_head(tokens / 64, ns, Bq / groups, groups, false);
    const int write_final = whole || (!plan.shared && ns == 1 && !lse_out) ? 1 : 0;
    rc = quant_launch(st, k_bmp, k_packed, k_tile_off, k_scales, k_zeros, v_bmp, v_packed, v_tile_off, v_scales, v_zeros, q,
                      out, tokens, head_dim, Bq, groups, bit, dequant_mode, workspace, ns, ns, write_final, group_size, 0, nullptr,
                      nullptr, whole, plan.shared, plan.folded);
    if (rc != MSTF_OK || write_final) return rc;
    return merge_splits(st, workspace, out, lse_out, ns, head_dim, Bq, plan.merge_blocks());
}

extern "C" int mstf_decode_attention_quant(void* stream, const uint64_t* k_bmp, const uint32_t* k_packed,
                                           const uint32_t* k_tile_off, const mstf_half* k_scales,
                                           const mstf_half* k_zeros, const uint64_t* v_bmp, const uint32_t* v_packed,
                                           const uint32_t* v_tile_off, const mstf_half* v_scales,
                                           const mstf_half* v_zeros, const mstf_half* q, mstf_half* out, float* lse_out,
                                           int tokens, int head_dim, int Bq, int groups, int bit, int capacity,
                                           int dequant_mode, void* workspace, size_t workspace_bytes)
{
    return decode_attention_quant_impl(stream, k_bmp, k_packed, k_tile_off, k_scales, k_zeros, v_bmp, v_packed, v_tile_off,
                                       v_scales, v_zeros, q, out, lse_out, tokens, head_dim, Bq, groups, bit, capacity,
                                       dequant_mode, 64, workspace, workspace_bytes);
}

extern "C" int mstf_decode_attention_quant_grouped(void* stream, const uint64_t* k_bmp, const uint32_t* k_packed,
                                                   const uint32_t* k_tile_off, const mstf_half* k_scales,
                                                   const mstf_half* k_zeros, const uint64_t* v_bmp,
                                                   const uint32_t* v_packed, const uint32_t* v_tile_off,
                                                   const mstf_half* v_scales, const mstf_half* v_zeros,
                                                   const mstf_half* q, mstf_half* out, float* lse_out, int tokens,
                                                   int head_dim, int Bq, int groups, int bit, int capacity,
                                                   int dequant_mode, int group_size, void* workspace,
                                                   size_t workspace_bytes)
{
    return decode_attention_quant_impl(stream, k_bmp, k_packed, k_tile_off, k_scales, k_zeros, v_bmp, v_packed, v_tile_off,
                                       v_scales, v_zeros, q, out, lse_out, tokens, head_dim, Bq, groups, bit, capacity,
                                       dequant_mode, group_size, workspace, workspace_bytes);
}

extern "C" int mstf_decode_attention_window_quant(
    void* stream, const uint64_t* k_bmp, const uint32_t* k_packed, const uint32_t* k_tile_off, const mstf_half* k_scales,
    const mstf_half* k_zeros, const uint64_t* v_bmp, const uint32_t* v_packed, const uint32_t* v_tile_off,
    const mstf_half* v_scales, const mstf_half* v_zeros, const mstf_half* q, const mstf_half* k_win,
    const mstf_half* v_win, int win_len, const int32_t* win_len_dev, int win_stride, mstf_half* out, float* lse_out,
    int tokens, int head_dim, int Bq, int groups, int bit, int capacity, int dequant_mode, void* workspace,
    size_t workspace_bytes)
{
    if (!q || !k_win || !v_win || !out) return MSTF_EINVAL;
    if (tokens < 0 || win_len <= 0 || win_stride < win_len || Bq <= 0 || groups <= 0 || Bq % groups != 0)
        return MSTF_EINVAL;
    if (head_dim != kFusedD || tokens % 64 != 0 || groups > 8) return MSTF_EUNSUPPORTED;
    if (!aligned_to(q, 16) || !aligned_to(k_win, 16) || !aligned_to(v_win, 16) || !aligned_to(out, 2) ||
        (lse_out && !aligned_to(lse_out, 4)) || (win_len_dev && !aligned_to(win_len_dev, 4)))
        return MSTF_EALIGN;
    if (!workspace || workspace_bytes < fused_workspace_need(tokens, win_len, Bq)) return MSTF_EWORKSPACE;
    if (!aligned_to(workspace, 16)) return MSTF_EALIGN;
    hipStream_t st = as_stream(stream);
    int rc;
    QuantPlan plan = {false, false, 0};
    if (tokens > 0) {
        rc = quant_check(k_bmp, k_packed, k_tile_off, k_scales, k_zeros, v_bmp, v_packed, v_tile_off, v_scales, v_zeros, q,
                         tokens, head_dim, Bq, groups, bit, capacity, dequant_mode);
        if (rc != MSTF_OK) return rc;
        plan = quant_plan(tokens, Bq, groups, bit, 64, win_len, 0, true, workspace_bytes);
    }
    const int ns = plan.ns, nst = ns + window_blocks(win_len);
    if (tokens > 0) {
        rc = quant_launch(st, k_bmp, k_packed, k_tile_off, k_scales, k_zeros, v_bmp, v_packed, v_tile_off, v_scales,
                          v_zeros, q, nullptr, tokens, head_dim, Bq, groups, bit, dequant_mode, workspace, ns, nst, 0, 64, 0, nullptr,
                          nullptr, false, plan.shared, plan.folded);
        if (rc != MSTF_OK) return rc;
    }
    if ((rc = window_launch(st, k_win, v_win, q, workspace, win_len, win_len_dev, win_stride, head_dim, Bq, groups, nst,
                            ns)) != MSTF_OK)
        return rc;
    return merge_splits(st, workspace, out, lse_out, nst, head_dim, Bq, plan.merge_blocks());
}

extern "C" int mstf_decode_attention_window_quant_pool(
    void* stream, const uint64_t* k_bmp, const uint32_t* k_packed, const uint32_t* k_tile_off, const mstf_half* k_scales,
    const mstf_half* k_zeros, const uint64_t* v_bmp, const uint32_t* v_packed, const uint32_t* v_tile_off,
    const mstf_half* v_scales, const mstf_half* v_zeros, const mstf_half* q, const mstf_half* k_win,
    const mstf_half* v_win, int win_len, const int32_t* win_len_dev, int win_stride, mstf_half* out, float* lse_out,
    int max_tokens, const int32_t* tokens_dev, int64_t tile_capacity, int head_dim, int Bq, int groups, int bit,
    int capacity, int dequant_mode, void* workspace, size_t workspace_bytes)
{
    if (!q || !k_win || !v_win || !out || !tokens_dev) return MSTF_EINVAL;
    if (max_tokens <= 0 || win_len <= 0 || win_stride < win_len || Bq <= 0 || groups <= 0 || Bq % groups != 0)
        return MSTF_EINVAL;
    if (head_dim != kFusedD || max_tokens % 64 != 0 || groups > 8) return MSTF_EUNSUPPORTED;
    if (tile_capacity < (int64_t)max_tokens * head_dim / 64) return MSTF_EINVAL;
    if (!aligned_to(q, 16) || !aligned_to(k_win, 16) || !aligned_to(v_win, 16) || !aligned_to(out, 2) ||
        (lse_out && !aligned_to(lse_out, 4)) || (win_len_dev && !aligned_to(win_len_dev, 4)) || !aligned_to(tokens_dev, 4))
        return MSTF_EALIGN;
    // rows of the per-tile arrays start tile_capacity entries apart: the two-byte ones keep their four-byte alignment
    if (tile_capacity % 2 != 0) return MSTF_EALIGN;
    if (!workspace || workspace_bytes < fused_workspace_need(max_tokens, win_len, Bq)) return MSTF_EWORKSPACE;
    if (!aligned_to(workspace, 16)) return MSTF_EALIGN;
    hipStream_t st = as_stream(stream);
    int rc = quant_check(k_bmp, k_packed, k_tile_off, k_scales, k_zeros, v_bmp, v_packed, v_tile_off, v_scales, v_zeros, q,
                         max_tokens, head_dim, Bq, groups, bit, capacity, dequant_mode);
    if (rc != MSTF_OK) return rc;
    const int wblk = window_blocks(win_len);
    const QuantPlan plan = quant_plan(max_tokens, Bq, groups, bit, 64, win_len, win_len, true, workspace_bytes);
    const int ns = plan.ns, nst = ns + wblk;
    rc = quant_launch(st, k_bmp, k_packed, k_tile_off, k_scales, k_zeros, v_bmp, v_packed, v_tile_off, v_scales, v_zeros, q,
                      nullptr, max_tokens, head_dim, Bq, groups, bit, dequant_mode, workspace, ns, nst, 0, 64,
                      (size_t)tile_capacity, tokens_dev, nullptr, false, plan.shared, plan.folded);
    if (rc != MSTF_OK) return rc;
    if ((rc = window_launch(st, k_win, v_win, q, workspace, win_len, win_len_dev, win_stride, head_dim, Bq, groups, nst,
                            ns)) != MSTF_OK)
        return rc;
    return merge_splits(st, workspace, out, lse_out, nst, head_dim, Bq, plan.merge_blocks());
}

extern "C" int mstf_decode_step_quant_pool(
    void* stream, const uint64_t* k_bmp, const uint32_t* k_packed, const uint32_t* k_tile_off, const mstf_half* k_scales,
    const mstf_half* k_zeros, const uint64_t* v_bmp, const uint32_t* v_packed, const uint32_t* v_tile_off,
    const mstf_half* v_scales, const mstf_half* v_zeros, const mstf_half* q_in, int64_t q_stride, const mstf_half* k_in,
    int64_t k_stride, const mstf_half* v_in, int64_t v_stride, int bs, int n_q, int n_kv, const mstf_half* cos,
    const mstf_half* sin, int64_t rope_stride, mstf_half* k_win, mstf_half* v_win, int win_stride, int win_len,
    const int32_t* win_len_dev, uint32_t* overflow, mstf_half* out, float* lse_out, int max_tokens,
    const int32_t* tokens_dev, int64_t tile_capacity, int head_dim, int bit, int capacity, int dequant_mode,
    void* workspace, size_t workspace_bytes)
{
    if (!q_in || !k_in || !v_in || !k_win || !v_win || !out || !tokens_dev) return MSTF_EINVAL;
    if ((cos == nullptr) != (sin == nullptr)) return MSTF_EINVAL;
    if (bs <= 0 || n_q <= 0 || n_kv <= 0 || n_q % n_kv != 0) return MSTF_EINVAL;
    if (max_tokens <= 0 || win_len <= 0 || win_stride < win_len) return MSTF_EINVAL;
    const int groups = n_q / n_kv;
    const int64_t Bq64 = (int64_t)bs * n_q;
    if (Bq64 > 0x7FFFFFF0) return MSTF_EUNSUPPORTED;
    const int Bq = (int)Bq64;
    if (head_dim != kFusedD || max_tokens % 64 != 0 || groups > 8) return MSTF_EUNSUPPORTED;
    if (tile_capacity < (int64_t)max_tokens * head_dim / 64) return MSTF_EINVAL;
    if (tile_capacity % 2 != 0) return MSTF_EALIGN;  // (rows of the two-byte per-tile arrays stay four-byte aligned)
    if (q_stride % 8 != 0 || k_stride % 8 != 0 || v_stride % 8 != 0 || rope_stride % 8 != 0) return MSTF_EALIGN;
    if (!aligned_to(q_in, 16) || !aligned_to(k_in, 16) || !aligned_to(v_in, 16) || !aligned_to(cos, 16) ||
        !aligned_to(sin, 16) || !aligned_to(k_win, 16) || !aligned_to(v_win, 16) || !aligned_to(out, 2) ||
        (lse_out && !aligned_to(lse_out, 4)) || (win_len_dev && !aligned_to(win_len_dev, 4)) ||
        !aligned_to(tokens_dev, 4) || !aligned_to(overflow, 4))
        return MSTF_EALIGN;
    if (!workspace || workspace_bytes < fused_workspace_need(max_tokens, win_len, Bq)) return MSTF_EWORKSPACE;
    if (!aligned_to(workspace, 16)) return MSTF_EALIGN;
    int rc = quant_check(k_bmp, k_packed, k_tile_off, k_scales, k_zeros, v_bmp, v_packed, v_tile_off, v_scales, v_zeros,
                         q_in, max_tokens, head_dim, Bq, groups, bit, capacity, dequant_mode);
    if (rc != MSTF_OK) return rc;
    hipStream_t st = as_stream(stream);
    const int wblk = window_blocks(win_len);
    const QuantPlan plan = quant_plan(max_tokens, Bq, groups, bit, 64, win_len, win_len, true, workspace_bytes);
    const int ns = plan.ns, nst = ns + wblk;
    StepArgs sa = {};
    sa.q_in = reinterpret_cast<const _Float16*>(q_in);
    sa.k_in = reinterpret_cast<const _Float16*>(k_in);
    sa.v_in = reinterpret_cast<const _Float16*>(v_in);
    sa.q_stride = q_stride;
    sa.k_stride = k_stride;
    sa.v_stride = v_stride;
    sa.cos = reinterpret_cast<const _Float16*>(cos);
    sa.sin = reinterpret_cast<const _Float16*>(sin);
    sa.rope_stride = rope_stride;
    sa.k_win = reinterpret_cast<_Float16*>(k_win);
    sa.v_win = reinterpret_cast<_Float16*>(v_win);
    sa.win_len_dev = win_len_dev;
    sa.overflow = overflow;
    sa.win_len = win_len;
    sa.win_stride = win_stride;
    sa.n_kv = n_kv;
    sa.ns = ns;
    sa.wg0 = ns;
    rc = quant_launch(st, k_bmp, k_packed, k_tile_off, k_scales, k_zeros, v_bmp, v_packed, v_tile_off, v_scales, v_zeros,
                      q_in, nullptr, max_tokens, head_dim, Bq, groups, bit, dequant_mode, workspace, ns, nst, 0, 64,
                      (size_t)tile_capacity, tokens_dev, &sa, false, plan.shared, plan.folded);
    if (rc != MSTF_OK) return rc;
    return merge_splits(st, workspace, out, lse_out, nst, head_dim, Bq, plan.merge_blocks());
}
