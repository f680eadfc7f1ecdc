// Quantised variant of the bitmap format: the producer (bitmaps, per-tile scale / zero-point, packed
// 2/4/8-bit codes).  The consumers are in quant_spmv.hip.
//
// Same tiles, bitmaps and work units as the fp16 format; per tile the non-zeros are replaced by
// codes  q = clamp(floor(v / scale + 0.5) + zero, 0, 2^bit - 1)  packed `capacity = 32 / bit` to a
// 4-byte word (code j of a tile at bits bit*(j % capacity) of word j / capacity), and tile_off[b][t]
// is the GLOBAL word offset of the tile inside the flat `packed` buffer.
//
#include "compress_common.hpp"
#include "spmv_common.hpp"

namespace mstf {

#pragma clang fp contract(off)

__device__ __forceinline__ float half_bits_to_float(uint32_t bits) { return (float)as_h((uint16_t)bits); }

// ------------------------------------------------------------------------------- producer: count
// grid = B * M/64 units, 64 threads.  Lane l owns tiles l and 64+l of the unit: bitmap, raw count,
// units, scale, zero; tile_off gets the unit-local exclusive word offset, unit_tot the unit total.
// G32: two (scale, zero) pairs per tile, pair g from the kept elements 32g .. 32g+31 of the tile; scales / zeros are
// then [B][T][2].
template <bool IS_VALUE, bool G32>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) void quant_count_kernel(const _Float16* __restrict__ x, int M, int kth, int bit,
                                                         uint64_t* __restrict__ bmp, uint32_t* __restrict__ counts,
                                                         uint32_t* __restrict__ units, uint32_t* __restrict__ tile_off,
                                                         _Float16* __restrict__ scales, _Float16* __restrict__ zeros,
                                                         uint32_t* __restrict__ unit_tot)
{
    __shared__ uint32_t slab[kHalfSlabDw];
    const int lane = lane_id();
    const int nblk = M / 64;
    const int unit = (int)blockIdx.x;
    const int b = unit / nblk, tb = unit - b * nblk;
    const size_t T = (size_t)M * kD / 64;
    uint32_t r[64];  // this lane's token: 128 fp16 values
    unit_rows(x + (size_t)b * M * kD, (int64_t)tb * 64, (int64_t)M, slab, lane, r);

    uint64_t bm[2];
    uint32_t thr;
    {
        uint32_t mag[64];
#pragma unroll
        for (int j = 0; j < 64; j++) mag[j] = r[j] & 0x7FFF7FFFu;
        thr = unit_keep<IS_VALUE>(mag, kth, lane, bm[0], bm[1]);
    }
    // The pruned elements become NaN (exponent and mantissa all ones under the element's own sign), which the
    // minimum / maximum instructions pass over: no per-element test of the bitmap is needed afterwards.
    typedef short s2_t __attribute__((ext_vector_type(2)));
    const us2_t t2 = as_us2(thr | (thr << 16));
#pragma unroll
    for (int j = 0; j < 64; j++) {
        const s2_t d = __builtin_bit_cast(s2_t, (us2_t)(as_us2(r[j] & 0x7FFF7FFFu) - t2));   // < 0 <=> pruned
        r[j] |= __builtin_bit_cast(uint32_t, (s2_t)(d >> 15)) & 0x7FFF7FFFu;
    }
    const _Float16* sh = reinterpret_cast<const _Float16*>(slab);
    const int cap = 32 / bit;
    const float maxq = (float)((1 << bit) - 1);
    const size_t tile0 = (size_t)b * T + (size_t)tb * kD;
    uint32_t u[2];
#pragma unroll
    for (int h = 0; h < 2; h++) {
        constexpr int NG = G32 ? 2 : 1;
        float mn[NG], mx[NG];
        const uint64_t m = bm[h];
        if (IS_VALUE) {
            // tile (h, token = lane): the lane's own 64 channels, two per register; group g = registers 16g .. 16g+15
            typedef _Float16 h2v_t __attribute__((ext_vector_type(2)));
#pragma unroll
            for (int g = 0; g < NG; g++) {
                h2v_t mn2 = {(_Float16)INFINITY, (_Float16)INFINITY}, mx2 = {(_Float16)-INFINITY, (_Float16)-INFINITY};
#pragma unroll
                for (int j = g * (32 / NG); j < (g + 1) * (32 / NG); j++) {
                    const h2v_t v = __builtin_bit_cast(h2v_t, r[32 * h + j]);
                    mn2 = __builtin_elementwise_min(mn2, v);
                    mx2 = __builtin_elementwise_max(mx2, v);
                }
                mn[g] = fminf((float)mn2[0], (float)mn2[1]);
                mx[g] = fmaxf((float)mx2[0], (float)mx2[1]);
            }
        } else {
            // tile = channel 64h + lane over the 64 tokens: the half-slab back into LDS, the lane walks its column;
            // group g = tokens 32g .. 32g+31
#pragma unroll
            for (int j = 0; j < 32; j++) slab[lane * kHalfRowDw + j] = r[32 * h + j];
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int g = 0; g < NG; g++) {
                float a = INFINITY, z = -INFINITY;
#pragma unroll 8
                for (int i = g * (64 / NG); i < (g + 1) * (64 / NG); i++) {
                    const float v = (float)sh[i * (2 * kHalfRowDw) + lane];
                    a = fminf(a, v);
                    z = fmaxf(z, v);
                }
                mn[g] = a;
                mx[g] = z;
            }
            __builtin_amdgcn_wave_barrier();
        }
        const uint32_t cnt = (uint32_t)__popcll(m);
        const size_t ti = tile0 + (size_t)h * 64 + lane;
#pragma unroll
        for (int g = 0; g < NG; g++) {
            // an empty group leaves the minimum at +inf: scale 1, zero 0, as for an empty tile
            float scale = 1.f, zero = 0.f;
            if (mn[g] <= mx[g]) {
                scale = (mx[g] - mn[g]) / maxq;
                if (scale == 0.f) scale = 1.f;
                zero = floorf(-mn[g] / scale + 0.5f);
            }
            scales[ti * NG + g] = (_Float16)scale;
            zeros[ti * NG + g] = (_Float16)zero;
        }
        bmp[ti] = m;
        counts[ti] = cnt;
        u[h] = (cnt + (uint32_t)cap - 1u) / (uint32_t)cap;
        units[ti] = u[h];
    }
    uint32_t totA, totB;
    const uint32_t eA = wave_excl_scan(u[0], lane, totA);
    const uint32_t eB = wave_excl_scan(u[1], lane, totB);
    tile_off[tile0 + lane] = eA;
    tile_off[tile0 + 64 + lane] = totA + eB;
    if (lane == 0) unit_tot[(size_t)b * nblk + tb] = totA + totB;
}

// grid = B, 256 threads: exclusive scan of the head's unit totals into unit_base; head_base[b] = words of all earlier
// heads (summed from their unit totals, which spares a launch for a scan over heads); the last head's workgroup
// writes the grand total.
__global__ __launch_bounds__(256) void quant_scan_kernel(const uint32_t* __restrict__ unit_tot,
                                                         uint32_t* __restrict__ unit_base,
                                                         uint32_t* __restrict__ head_base,
                                                         uint64_t* __restrict__ total_words, int nblk)
{
    extern __shared__ uint32_t base[];
    const int b = (int)blockIdx.x;
    const uint32_t total = units_scan(unit_tot + (size_t)b * nblk, base, nblk);
    for (int i = (int)threadIdx.x; i < nblk; i += 256) unit_base[(size_t)b * nblk + i] = base[i];
    const uint64_t pre = sum_before(unit_tot, (size_t)b * nblk);
    if (threadIdx.x == 0) {
        head_base[b] = (uint32_t)pre;
        if (b == (int)gridDim.x - 1) *total_words = pre + total;
    }
}

// tile_off[b][t] += head base + unit base  (global word offsets, as the reference returns them): the sizing-only call.
__global__ __launch_bounds__(256) void quant_finalize_kernel(uint32_t* __restrict__ tile_off,
                                                             const uint32_t* __restrict__ unit_base,
                                                             const uint32_t* __restrict__ head_base, int nblk, size_t T)
{
    const int b = (int)blockIdx.y;
    const size_t t = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= T) return;
    tile_off[(size_t)b * T + t] += head_base[b] + unit_base[(size_t)b * nblk + t / kD];
}

// ------------------------------------------------------------------------------- producer: one pass
// (scale, zero-point) of a group of values as the consumers will read them - rounded to fp16 - and what a value is
// quantised with.  v / scale is the quotient estimate by the reciprocal and one correction by the exact remainder: for
// fp16 values and scales the correctly rounded quotient, in three instructions instead of the full division sequence.
struct QuantGroup {
    float scale, rcp, zero;
};
__device__ __forceinline__ QuantGroup quant_group(float mn, float mx, float maxq, _Float16& s16, _Float16& z16)
{
    // an empty group leaves the minimum at +inf: scale 1, zero 0, as for an empty tile
    float scale = 1.f, zero = 0.f;
    if (mn <= mx) {
        scale = (mx - mn) / maxq;
        if (scale == 0.f) scale = 1.f;
        zero = floorf(-mn / scale + 0.5f);
    }
    s16 = (_Float16)scale;
    z16 = (_Float16)zero;
    QuantGroup g;
    g.scale = (float)s16 == 0.f ? 1.f : (float)s16;
    g.rcp = 1.0f / g.scale;
    // an infinite scale makes every finite value 0: the reciprocal does, the remainder has to stay finite for it
    g.scale = g.scale == INFINITY ? 1.f : g.scale;
    g.zero = (float)z16;
    return g;
}
__device__ __forceinline__ uint32_t quant_code(float v, float scale, float rcp, float zero, float maxq)
{
    const float e = v * rcp;
    const float d = __builtin_fmaf(__builtin_fmaf(-e, scale, v), rcp, e);
    const float q = floorf(d + 0.5f) + zero;
    return (uint32_t)fminf(fmaxf(q, 0.f), maxq);  // (a NaN becomes 0)
}
__device__ __forceinline__ float lane_of(float x, int src4)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(src4, __builtin_bit_cast(int, x)));
}
// Quantises and packs the values of half a unit, a lane per word.  The image at img holds the kept values of tile t
// (= lane t's) from word e of the half on, 32 / BIT values per word, NaN in the places without one - their codes are 0.
//   tot: words of the half;  u: words of the lane's tile;  c0: G32: how many of its values belong to the first group
//   map: LDS room for 64 words;  dst: where the half's words go;  room: words there is room for (a tile that would
//   not fit is left untouched)
template <int BIT, bool G32>
__device__ __forceinline__ void quant_words(uint32_t img, uint32_t map, uint32_t tot, uint32_t e, uint32_t u, uint32_t c0,
                                            const QuantGroup (&grp)[G32 ? 2 : 1], float maxq, uint32_t* dst, uint64_t room,
                                            int lane)
{
    constexpr int CAP = 32 / BIT;
    uint32_t carry = 0;  // tile of the word in front of the pass
#pragma unroll 1
    for (uint32_t w0 = 0; w0 < tot; w0 += 64) {
        // tile of word w0 + lane: the last one that starts at or in front of it
        const uint32_t rel = e - w0;
        *(MSTF_LDS uint32_t*)(uintptr_t)(map + (uint32_t)lane * 4u) = 0u;
        asm volatile("" ::: "memory");
        if (u != 0u && rel < 64u) *(MSTF_LDS uint32_t*)(uintptr_t)(map + rel * 4u) = (uint32_t)lane + 1u;
        asm volatile("" ::: "memory");
        __builtin_amdgcn_wave_barrier();
        const uint32_t first = *(MSTF_LDS const uint32_t*)(uintptr_t)(map + (uint32_t)lane * 4u);
        const uint64_t before = __ballot(first != 0u) & (~0ull >> (63 - lane));
        const uint32_t found = (uint32_t)__builtin_amdgcn_ds_bpermute((63 - (int)__builtin_clzll(before | 1ull)) * 4, (int)first);
        const uint32_t tile = before != 0ull ? found - 1u : carry;
        carry = (uint32_t)__builtin_amdgcn_readlane((int)tile, 63);
        const int t4 = (int)tile * 4;
        const uint32_t w = w0 + (uint32_t)lane;
        uint32_t v[CAP / 2];
#pragma unroll
        for (int i = 0; i < CAP / 2; i += CAP / 2 < 4 ? 2 : 4) {
            const uint32_t a = img + w * (uint32_t)(CAP * 2) + (uint32_t)i * 4u;
            if constexpr (CAP / 2 < 4) {
                const u32x2_t x = *(MSTF_LDS const u32x2_t*)(uintptr_t)a;
                v[i] = x[0], v[i + 1] = x[1];
            } else {
                const u32x4_t x = *(MSTF_LDS const u32x4_t*)(uintptr_t)a;
                v[i] = x[0], v[i + 1] = x[1], v[i + 2] = x[2], v[i + 3] = x[3];
            }
        }
        float sc[2], rc[2], zp[2];
#pragma unroll
        for (int g = 0; g < (G32 ? 2 : 1); g++) {
            sc[g] = lane_of(grp[g].scale, t4);
            rc[g] = lane_of(grp[g].rcp, t4);
            zp[g] = lane_of(grp[g].zero, t4);
        }
        int left = CAP;  // G32: values of the word in front of the second group
        if (G32)
            left = __builtin_amdgcn_ds_bpermute(t4, (int)c0) -
                   (int)(w - (uint32_t)__builtin_amdgcn_ds_bpermute(t4, (int)e)) * CAP;
        uint32_t cur = 0;
#pragma unroll
        for (int k = CAP - 1; k >= 0; k--) {
            const float x = half_bits_to_float((k & 1) ? v[k >> 1] >> 16 : v[k >> 1] & 0xFFFFu);
            const bool second = G32 && k >= left;
            cur = (cur << BIT) | quant_code(x, second ? sc[1] : sc[0], second ? rc[1] : rc[0], second ? zp[1] : zp[0], maxq);
        }
        bool store = w < tot;
        if (room < tot) {  // (wave-uniform: the exchange needs every lane)
            const uint32_t end = (uint32_t)__builtin_amdgcn_ds_bpermute(t4, (int)(e + u));
            store = store && end <= room;
        }
        if (store) dst[w] = cur;
    }
}

// Everything with one read of the input, for the calls that produce the packed words: threshold, bitmaps, the word
// counts, which need nothing but those, and the workgroup's word total published as a status word; then, half a unit
// at a time, the kept values compacted into an LDS image (compact_half, as the fp16 compressor does), the minimum and
// maximum of every tile out of the image, and the image's words quantised by one lane each (quant_words), at the final
// global word offsets from the totals of the workgroups in front (the one-pass ordering of compress.hip).
// grid = units / W workgroups of W wavefronts, W divides M / 64.
// total_words reads as all ones when a wait ran out of its polls.
// Bound by vector instructions: with a lane quantising the values of its own tile one after the other - as long as the
// longest tile of 64, a full division each, words stored one by one - 40.7 / 35.7 us for 64 heads x 4096 tokens of
// keys / values, 2 bits, 70 %; 34.8 / 30.4 us like this (rocprofv3).
template <bool IS_VALUE, bool G32, int W>
__global__ __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(4))) void quant_onepass_kernel(
    const _Float16* __restrict__ x, int M, int kth, int bit, uint64_t* __restrict__ bmp, uint32_t* __restrict__ counts,
    uint32_t* __restrict__ units, uint32_t* __restrict__ tile_off, _Float16* __restrict__ scales,
    _Float16* __restrict__ zeros, uint32_t* __restrict__ packed, uint64_t capacity_words,
    uint64_t* __restrict__ total_words, uint64_t* state, int nunits, int groups_total, uint32_t spin_limit, Handover how)
{
    // staging buffer of a half-slab, then image of half a unit's kept values (at most 64 tiles x 128 bytes), behind it
    // the 64 words that quant_words looks tiles up in
    __shared__ __attribute__((aligned(16))) uint32_t slabs[W][kHalfSlabDw];
    constexpr uint32_t kImage = 64 * 128;
    static_assert(kHalfSlabDw * 4 >= kImage + 64 * 4, "image and tile look-up fit the staging buffer");
    __shared__ uint32_t wave_total[W];
    __shared__ uint64_t bases[W][2];
    const int lane = lane_id();
    const int wave = wave_id();
    const int nblk = M / 64;
    const int g = (int)blockIdx.x;
    const int unit = g * W + wave;
    const int b = unit / nblk, tb = unit - b * nblk;
    const size_t T = (size_t)M * kD / 64;
    uint32_t* slab = slabs[wave];
    uint32_t r[64];  // this lane's token: 128 fp16 values
    {
        UnitRaw raw;
        unit_fetch(x + (size_t)b * M * kD, (int64_t)tb * 64, lane, raw);
        unit_rows_parked(raw, slab, lane, r);  // r[32 .. 64) stays in the slab during the search
    }
    uint32_t kept[4];
    if (kth > 0) {
        select_kth_planes_parked<true>(r, slab, lane, kth, kept);  // the sign bits become planes the search never looks at
    } else {
        parked_rows_take(slab, lane, r);
        kept_nonzero(r, kept);
    }
    __builtin_amdgcn_wave_barrier();
    uint64_t bm[2];
    if (IS_VALUE) {
        bm[0] = spread_bitmap(kept[0], kept[1]);
        bm[1] = spread_bitmap(kept[2], kept[3]);
    } else {
        key_bitmaps_from_kept(kept, lane, bm[0], bm[1]);
    }
    const uint32_t cap_shift = bit == 2 ? 4u : (bit == 4 ? 3u : 2u);
    const float maxq = (float)((1 << bit) - 1);
    const size_t tile0 = (size_t)b * T + (size_t)tb * kD;
    constexpr int NG = G32 ? 2 : 1;
    uint32_t cnt[2], c0[2], u[2], e[2], tot[2];
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const size_t ti = tile0 + (size_t)h * 64 + lane;
        cnt[h] = (uint32_t)__popcll(bm[h]);
        c0[h] = (uint32_t)__builtin_popcount((uint32_t)(bm[h] >> 32));  // of elements 0 .. 31
        u[h] = (cnt[h] + (1u << cap_shift) - 1u) >> cap_shift;
        bmp[ti] = bm[h];
        counts[ti] = cnt[h];
        units[ti] = u[h];
        e[h] = wave_excl_scan(u[h], lane, tot[h]);
        tot[h] = __builtin_amdgcn_readfirstlane(tot[h]);
    }
    if (lane == 0) wave_total[wave] = tot[0] + tot[1];
    __syncthreads();
    uint32_t in_group = 0, group_total = 0;
#pragma unroll
    for (int w = 0; w < W; w++) {
        const uint32_t t = wave_total[w];
        in_group += w < wave ? t : 0u;
        group_total += t;
    }
    if (threadIdx.x == 0) agent_store(state + g, kWordReady | group_total);

    const uint32_t img = lds_addr(slab);
    uint64_t before = 0;
#pragma unroll
    for (int h = 0; h < 2; h++) {  // unrolled: everything indexed by h stays in registers
        const uint32_t own = e[h] << (cap_shift + 1);  // where the lane's tile starts in the image
        image_fill(img, tot[h] << (cap_shift + 1), 0xFFFFFFFFu, lane);  // NaN between tiles
        compact_half<IS_VALUE>(r, kept, h, own / 4u, img, lane);
        float mn[NG], mx[NG];
        // four values per read (a word holds at least that many)
        h2_t mn2[NG], mx2[NG];
#pragma unroll
        for (int gq = 0; gq < NG; gq++) {
            mn2[gq] = h2_t{(_Float16)INFINITY, (_Float16)INFINITY};
            mx2[gq] = h2_t{(_Float16)-INFINITY, (_Float16)-INFINITY};
        }
        auto take = [&](int gq, u32x2_t v) {
            const h2_t va = as_h2(v[0]), vb = as_h2(v[1]);
            mn2[gq] = __builtin_elementwise_min(__builtin_elementwise_min(mn2[gq], va), vb);
            mx2[gq] = __builtin_elementwise_max(__builtin_elementwise_max(mx2[gq], va), vb);
        };
        auto four = [&](uint32_t k) { return *(MSTF_LDS const u32x2_t*)(uintptr_t)(img + own + 2u * k); };
        if constexpr (G32) {
            // Two groups: the whole fours of the first one, the four that the second one starts in - the other group's
            // values made NaN - and the rest.  (Value by value with a select for either group, as long as the longest tile
            // of the wavefront: keys of 256 heads x 4096 tokens, 2 bits, 70 %: 146.5 us, 113.0 like this;
            // values 116.0, 104.0.)
            const uint32_t mid = c0[h] & ~3u;
            for (uint32_t k = 0; k < mid; k += 4) take(0, four(k));
            if (mid < cnt[h]) {
                const u32x2_t v = four(mid);
                const uint64_t first = (1ull << (16u * (c0[h] & 3u))) - 1ull;
                const uint32_t f0 = (uint32_t)first, f1 = (uint32_t)(first >> 32);
                take(0, u32x2_t{v[0] | ~f0, v[1] | ~f1});
                take(NG - 1, u32x2_t{v[0] | f0, v[1] | f1});
            }
            for (uint32_t k = mid + 4; k < cnt[h]; k += 4) take(NG - 1, four(k));
        } else {
            for (uint32_t k = 0; k < cnt[h]; k += 4) take(0, four(k));
        }
#pragma unroll
        for (int gq = 0; gq < NG; gq++) {
            mn[gq] = fminf((float)mn2[gq][0], (float)mn2[gq][1]);
            mx[gq] = fmaxf((float)mx2[gq][0], (float)mx2[gq][1]);
        }
        QuantGroup grp[NG];
        const size_t ti = tile0 + (size_t)h * 64 + lane;
#pragma unroll
        for (int gq = 0; gq < NG; gq++) {
            _Float16 s16, z16;
            grp[gq] = quant_group(mn[gq], mx[gq], maxq, s16, z16);
            scales[ti * NG + gq] = s16;
            zeros[ti * NG + gq] = z16;
        }
        if (h == 0) {
            uint64_t lo = 0, hi = 0;
            const bool ok0 = wait_for_words<W>(state, 0, 0, g, wave, lane, spin_limit, lo, hi);
            if (lane == 0) {
                bases[wave][0] = hi;
                bases[wave][1] = ok0 ? 1ull : 0ull;
            }
            __syncthreads();
            before = in_group;
            bool ok = true;
#pragma unroll
            for (int w = 0; w < W; w++) {
                before += bases[w][0];
                ok = ok && bases[w][1] != 0ull;
            }
            // (the unit's place is the same for the whole wavefront, and so are the addresses made from it)
            before = u64_of(__builtin_amdgcn_readfirstlane((uint32_t)before),
                            __builtin_amdgcn_readfirstlane((uint32_t)(before >> 32)));
            if (!ok && threadIdx.x == 0) mark_gave_up(how.flag, how.kept ? nullptr : total_words, nullptr);
            if (how.counted()) {
                if (g == groups_total - 1)
                    hand_over(how, total_words, before - in_group + group_total, ok, state, groups_total, spin_limit, wave_total);
                else if (threadIdx.x == 0)
                    count_through(counter_of(how, state, groups_total, g), ok);
            }
            if (lane == 0 && unit == nunits - 1 && ok && !how.kept)
                atomicMax(reinterpret_cast<unsigned long long*>(total_words), before + tot[0] + tot[1]);
            tile_off[tile0 + lane] = (uint32_t)(before + e[0]);
            tile_off[tile0 + 64 + lane] = (uint32_t)(before + tot[0] + e[1]);
            if (!ok) return;
        }
        const uint64_t off = before + (h == 0 ? 0u : tot[0]);
        const uint64_t room = capacity_words > off ? capacity_words - off : 0ull;
        const uint32_t map = img + kImage;
        if (bit == 2)
            quant_words<2, G32>(img, map, tot[h], e[h], u[h], c0[h], grp, maxq, packed + off, room, lane);
        else if (bit == 4)
            quant_words<4, G32>(img, map, tot[h], e[h], u[h], c0[h], grp, maxq, packed + off, room, lane);
        else
            quant_words<8, G32>(img, map, tot[h], e[h], u[h], c0[h], grp, maxq, packed + off, room, lane);
        __builtin_amdgcn_wave_barrier();
    }
}

// ------------------------------------------------------------------------------- host
static int cap_shift_of(int bit)
{
    switch (bit) {
        case 2: return 4;
        case 4: return 3;
        case 8: return 2;
        default: return -1;
    }
}

// workspace: unit totals, unit bases (both [B][M/64]) and the head bases [B]
static size_t quant_ws_bytes(int B, int M)
{
    return 2 * round_up((size_t)B * (M / 64) * 4, 256) + round_up((size_t)B * 4 + 64, 256);  // also the one-pass status words
}

template <bool IS_VALUE, bool G32>
static int compress_quant_impl(void* stream, const mstf_half* x, int B, int M, int N, int kth, int bit, uint64_t* bmp,
                               uint32_t* tile_off, uint32_t* counts, uint32_t* units, mstf_half* scales,
                               mstf_half* zeros, uint64_t* total_words, uint32_t* packed, uint64_t cap_words, void* ws,
                               size_t ws_bytes, uint64_t* landing, uint64_t* status)
{
    if (!x || !bmp || !tile_off || !counts || !units || !scales || !zeros || !total_words) return MSTF_EINVAL;
    if (B <= 0 || M <= 0 || N <= 0 || kth < 0 || kth > N) return MSTF_EINVAL;
    if (cap_shift_of(bit) < 0) return MSTF_EUNSUPPORTED;
    if (N != kD || M % 64 != 0 || M / 64 > 8192 || (int64_t)B * (M / 64) > 0x7FFFFFFF) return MSTF_EUNSUPPORTED;
    // tile offsets are 32-bit word offsets into one buffer (the reference's format): the worst case has to fit
    if ((uint64_t)B * (uint64_t)M * (uint64_t)N / 64u * (uint64_t)(64 * bit / 32) > 0xFFFFFFFFull) return MSTF_EUNSUPPORTED;
    if (!aligned_to(x, 16) || !aligned_to(bmp, 8) || !aligned_to(tile_off, 4) || !aligned_to(counts, 4) ||
        !aligned_to(units, 4) || !aligned_to(scales, G32 ? 4 : 2) || !aligned_to(zeros, G32 ? 4 : 2) || !aligned_to(total_words, 8) ||
        (packed && !aligned_to(packed, 4)))
        return MSTF_EALIGN;
    if (!ws || ws_bytes < quant_ws_bytes(B, M)) return MSTF_EWORKSPACE;
    if (!aligned_to(ws, 256)) return MSTF_EALIGN;
    hipStream_t st = as_stream(stream);
    const int nblk = M / 64;
    const size_t T = (size_t)M * kD / 64;
    char* w = reinterpret_cast<char*>(ws);
    const size_t ub = round_up((size_t)B * nblk * 4, 256);
    uint32_t* unit_tot = reinterpret_cast<uint32_t*>(w);
    uint32_t* unit_base = reinterpret_cast<uint32_t*>(w + ub);
    uint32_t* head_base = reinterpret_cast<uint32_t*>(w + 2 * ub);
    const _Float16* xh = reinterpret_cast<const _Float16*>(x);
    int rc;
    if (packed) {
        const int units_all = B * nblk;
        const int W = nblk % 4 == 0 ? 4 : (nblk % 2 == 0 ? 2 : 1);
        const int groups = units_all / W;
        uint64_t* state = status ? status + kKeptHead : reinterpret_cast<uint64_t*>(ws);
        const int counters = status ? kCounters : counters_within(quant_ws_bytes(B, M) / 8, groups);
        const Handover how = {landing, status ? status : state + groups, status != nullptr, counters};
        const int words = status_words(groups, counters);
        const uint32_t spin_limit = onepass_spin_limit();
        if (!status) {
            hipLaunchKernelGGL(onepass_init_kernel, dim3((unsigned)((words + 255) / 256 < 256 ? (words + 255) / 256 : 256)),
                               dim3(256), 0, st, state, words, total_words, static_cast<uint64_t*>(nullptr));
            if ((rc = check_launch()) != MSTF_OK) return rc;
        }
#define MSTF_QOP(WV)                                                                                                  \
    hipLaunchKernelGGL((quant_onepass_kernel<IS_VALUE, G32, WV>), dim3((unsigned)groups), dim3(64 * WV), 0, st, xh, M, kth, \
                       bit, bmp, counts, units, tile_off, reinterpret_cast<_Float16*>(scales),                          \
                       reinterpret_cast<_Float16*>(zeros), packed, cap_words, total_words, state, units_all, groups,    \
                       spin_limit, how)
        if (W == 4)
            MSTF_QOP(4);
        else if (W == 2)
            MSTF_QOP(2);
        else
            MSTF_QOP(1);
#undef MSTF_QOP
        return check_launch();
    }
    hipLaunchKernelGGL((quant_count_kernel<IS_VALUE, G32>), dim3((unsigned)(B * nblk)), dim3(64), 0, st, xh, M, kth, bit, bmp,
                       counts, units, tile_off, reinterpret_cast<_Float16*>(scales), reinterpret_cast<_Float16*>(zeros),
                       unit_tot);
    if ((rc = check_launch()) != MSTF_OK) return rc;
    hipLaunchKernelGGL(quant_scan_kernel, dim3((unsigned)B), dim3(256), (size_t)nblk * 4, st, unit_tot, unit_base,
                       head_base, total_words, nblk);
    if ((rc = check_launch()) != MSTF_OK) return rc;
    hipLaunchKernelGGL(quant_finalize_kernel, dim3((unsigned)((T + 255) / 256), (unsigned)B), dim3(256), 0, st, tile_off,
                       unit_base, head_base, nblk, T);
    if ((rc = check_launch()) != MSTF_OK) return rc;
    return MSTF_OK;
}

}  // namespace mstf

using namespace mstf;

extern "C" size_t mstf_compress_quant_workspace_bytes(int B, int M, int N)
{
    if (B <= 0 || M <= 0 || N <= 0 || M % 64 != 0) return 0;
    return quant_ws_bytes(B, M);
}

// group_size 64: one (scale, zero) pair per tile (the reference); 32: two, scales / zeros [B][T][2].
template <bool IS_VALUE>
static int compress_quant_group(int group_size, void* stream, const mstf_half* x, int B, int M, int N, int kth, int bit,
                                uint64_t* bmp, uint32_t* tile_off, uint32_t* counts, uint32_t* units, mstf_half* scales,
                                mstf_half* zeros, uint64_t* total_words, uint32_t* packed, uint64_t cap_words, void* ws,
                                size_t ws_bytes, uint64_t* landing = nullptr, uint64_t* status = nullptr)
{
    if (group_size == 64)
        return compress_quant_impl<IS_VALUE, false>(stream, x, B, M, N, kth, bit, bmp, tile_off, counts, units, scales, zeros,
                                                    total_words, packed, cap_words, ws, ws_bytes, landing, status);
    if (group_size == 32)
        return compress_quant_impl<IS_VALUE, true>(stream, x, B, M, N, kth, bit, bmp, tile_off, counts, units, scales, zeros,
                                                   total_words, packed, cap_words, ws, ws_bytes, landing, status);
    return MSTF_EUNSUPPORTED;
}

extern "C" int mstf_compress_key_quant(void* stream, const mstf_half* x, int B, int M, int N, int kth, int bit,
                                       uint64_t* bmp, uint32_t* tile_off, uint32_t* counts, uint32_t* units,
                                       mstf_half* scales, mstf_half* zeros, uint64_t* total_words, uint32_t* packed,
                                       uint64_t packed_capacity_words, void* workspace, size_t workspace_bytes)
{
    return compress_quant_group<false>(64, stream, x, B, M, N, kth, bit, bmp, tile_off, counts, units, scales, zeros,
                                       total_words, packed, packed_capacity_words, workspace, workspace_bytes);
}

extern "C" int mstf_compress_value_quant(void* stream, const mstf_half* x, int B, int M, int N, int kth, int bit,
                                         uint64_t* bmp, uint32_t* tile_off, uint32_t* counts, uint32_t* units,
                                         mstf_half* scales, mstf_half* zeros, uint64_t* total_words, uint32_t* packed,
                                         uint64_t packed_capacity_words, void* workspace, size_t workspace_bytes)
{
    return compress_quant_group<true>(64, stream, x, B, M, N, kth, bit, bmp, tile_off, counts, units, scales, zeros,
                                      total_words, packed, packed_capacity_words, workspace, workspace_bytes);
}

extern "C" int mstf_compress_quant_grouped(void* stream, const mstf_half* x, int is_value, int B, int M, int N, int kth,
                                           int bit, int group_size, uint64_t* bmp, uint32_t* tile_off, uint32_t* counts,
                                           uint32_t* units, mstf_half* scales, mstf_half* zeros, uint64_t* total_words,
                                           uint32_t* packed, uint64_t packed_capacity_words, void* workspace,
                                           size_t workspace_bytes)
{
    if (is_value)
        return compress_quant_group<true>(group_size, stream, x, B, M, N, kth, bit, bmp, tile_off, counts, units, scales,
                                          zeros, total_words, packed, packed_capacity_words, workspace, workspace_bytes);
    return compress_quant_group<false>(group_size, stream, x, B, M, N, kth, bit, bmp, tile_off, counts, units, scales,
                                       zeros, total_words, packed, packed_capacity_words, workspace, workspace_bytes);
}

extern "C" int mstf_compress_quant_sized(void* stream, const mstf_half* x, int is_value, int B, int M, int N, int kth, int bit,
                                         int group_size, uint64_t* bmp, uint32_t* tile_off, uint32_t* counts, uint32_t* units,
                                         mstf_half* scales, mstf_half* zeros, uint64_t* total_words, uint32_t* packed,
                                         uint64_t packed_capacity_words, void* workspace, size_t workspace_bytes,
                                         uint64_t* status, size_t status_bytes, int64_t* landing, int64_t* value)
{
    if (!packed) return MSTF_EINVAL;
    hipStream_t st = as_stream(stream);
    int rc = status_check(status, status_bytes, B, M, 1);
    if (rc == MSTF_OK) rc = landing_ready(st, landing, value);
    if (rc != MSTF_OK) return rc;
    rc = (is_value ? compress_quant_group<true> : compress_quant_group<false>)(
        group_size, stream, x, B, M, N, kth, bit, bmp, tile_off, counts, units, scales, zeros, total_words, packed,
        packed_capacity_words, workspace, workspace_bytes, reinterpret_cast<uint64_t*>(landing), status);
    return rc != MSTF_OK ? rc : total_wait(st, landing, value);
}
