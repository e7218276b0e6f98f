// dxt5a_gpu.hip -- DXT5 alpha-block endpoint search (crnlib's
// dxt5_endpoint_optimizer, crnlib/crn_dxt5a.cpp:40-262) on gfx950.
//
// A wavefront takes a run of blocks (16 values of one channel each), one per
// lane; blocks of one or two values are answered there, and the others are
// searched one after another by the whole wave, 64 candidate pairs at a time.
// The search is pure integer work and gives what the reference's sequence gives:
// unique values in first-appearance order, all unique pairs, then (quality >=
// better, error > 0) the +-16 / +-8 probe box whose centre follows every
// improvement -- the wave takes the first candidate of a batch that improves
// and goes on from the one after it.
//
// The reference skips box pairs already visited in either order
// (crn_dxt5a.cpp:131-137).  Skipping them cannot change the result: the
// 8-value and 6-value palettes of (l, h) and (h, l) hold the same values, so
// both orders have the same per-value minima and the same total, and a pair
// that was evaluated once has an error no smaller than the current best,
// which only decreases; re-evaluating it never replaces the best (strict <).
// So every box pair is evaluated and no visited set is kept.
//
// What bounds it: vector integer work, 14 value distances per candidate and
// distinct value, two per 16-bit packed operation.  One lane per block with
// the state in scratch took 35.6 ms for the alpha elements of 16 textures of
// 64^2 to 1024^2 with mips (one slow lane held 63 up), now 2.6 ms.
//
// Block gather for whole images follows crnlib/crn_dxt_image.cpp:330-344
// (4x4 texels with edge clamp) and :1491-1523 (component index, quality and
// both-block-types flag); the block is written as DXT5 alpha bytes
// {first, second, 48 bits of 3-bit selectors, texel 0 in the low bits}.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "autotune.h"
#include "crn2_internal.h"
#include "encode_set.h"

namespace {

__device__ __constant__ uint8_t k_six_invert[8] = {1, 0, 5, 4, 3, 2, 6, 7};
__device__ __constant__ uint8_t k_eight_invert[8] = {1, 0, 7, 6, 5, 4, 3, 2};

struct E2Result {
    uint64_t err;
    uint32_t first, second, type, reordered;
    uint64_t sel48;   // 3-bit selectors of texels 0..15
};

typedef short s16x2 __attribute__((ext_vector_type(2)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

__device__ inline uint32_t lane_id() { return threadIdx.x & 63u; }
__device__ inline uint32_t at_lane(uint32_t v, uint32_t l) { return (uint32_t)__builtin_amdgcn_readlane((int)v, (int)l); }

// x / 7 for x <= 1785 and x / 5 for x <= 1275 (exact there, 24-bit products)
__device__ inline uint32_t div7(uint32_t x) { return (x * 9363u) >> 16; }
__device__ inline uint32_t div5(uint32_t x) { return (x * 13108u) >> 16; }

__device__ inline u16x2 abs_diff(u16x2 v, u16x2 p)
{
    const s16x2 d = __builtin_bit_cast(s16x2, v) - __builtin_bit_cast(s16x2, p);
    return __builtin_bit_cast(u16x2, __builtin_elementwise_max(d, -d));
}

__device__ inline u16x2 two(uint32_t a, uint32_t b) { return u16x2{(unsigned short)a, (unsigned short)b}; }

// A lane's candidate pair: errors of the 8-value and the 6-value palette over
// the nu distinct values (lane i of uval / uw: value i and its count).
__device__ inline void pair_errors(uint32_t uval, uint32_t uw, uint32_t nu, uint32_t lo, uint32_t hi, uint32_t& e8,
                                   uint32_t& e6)
{
    const u16x2 ends = two(lo, hi);
    const u16x2 a0 = two(div7(lo * 6 + hi), div7(lo * 5 + hi * 2)), a1 = two(div7(lo * 4 + hi * 3), div7(lo * 3 + hi * 4)),
                a2 = two(div7(lo * 2 + hi * 5), div7(lo + hi * 6));
    const u16x2 b0 = two(div5(lo * 4 + hi), div5(lo * 3 + hi * 2)), b1 = two(div5(lo * 2 + hi * 3), div5(lo + hi * 4));
    e8 = e6 = 0;
    for (uint32_t i = 0; i < nu; i++) {
        const uint32_t v = at_lane(uval, i), w = at_lane(uw, i);
        const u16x2 x = two(v, v);
        const u16x2 de = abs_diff(x, ends);
        const u16x2 m8 = __builtin_elementwise_min(__builtin_elementwise_min(de, abs_diff(x, a0)),
                                                   __builtin_elementwise_min(abs_diff(x, a1), abs_diff(x, a2)));
        const u16x2 m6 = __builtin_elementwise_min(__builtin_elementwise_min(de, abs_diff(x, b0)), abs_diff(x, b1));
        const uint32_t d8 = min((uint32_t)m8.x, (uint32_t)m8.y);
        const uint32_t d6 = min(min((uint32_t)m6.x, (uint32_t)m6.y), min(v, 255u - v));   // 0 and 255
        e8 += __umul24(__umul24(d8, d8), w);
        e6 += __umul24(__umul24(d6, d6), w);
    }
}

// The block of values w[0..3] (four bytes each, the same on all lanes) with
// at least two distinct ones; the result is the same on all lanes.
__device__ inline E2Result dxt5a_search(const uint32_t (&w)[4], int quality, bool both)
{
    const uint32_t lane = lane_id(), t = lane & 15u;
    // (values, not places: an array read at a lane's index would live in LDS, and each
    // wave would read the launch packet in host memory for its place there, 10 us)
    const uint32_t w0 = w[0], w1 = w[1], w2 = w[2], w3 = w[3];
    const uint32_t word = t < 8 ? (t < 4 ? w0 : w1) : (t < 12 ? w2 : w3);
    const uint32_t mine = (word >> (8 * (t & 3u))) & 0xFFu;
    // distinct values in first-appearance order: lane u < nu holds value u
    uint32_t before = 0, count = 0;
#pragma unroll
    for (uint32_t k = 0; k < 16; k++) {
        const bool eq = ((w[k >> 2] >> (8 * (k & 3u))) & 0xFFu) == mine;
        before |= eq && k < t ? 1u : 0u;
        count += eq ? 1u : 0u;
    }
    const uint64_t firsts = __ballot(!before && lane < 16);
    const uint32_t nu = (uint32_t)__popcll(firsts);
    const uint32_t to = !before && lane < 16 ? (uint32_t)__popcll(firsts & ((1ull << lane) - 1ull)) : 63u;
    const uint32_t uval = (uint32_t)__builtin_amdgcn_ds_permute((int)(4 * to), (int)mine);
    const uint32_t uw = (uint32_t)__builtin_amdgcn_ds_permute((int)(4 * to), (int)count);

    uint32_t best = 0xFFFFFFFFu, best_first = 0, best_second = 0, best_type = 0;
    // every pair i < j in order, type 0 before type 1: the smallest error, the
    // earliest on ties
    for (uint32_t p0 = 0, pairs = nu * (nu - 1) / 2; p0 < pairs; p0 += 64) {
        const uint32_t p = min(p0 + lane, pairs - 1);
        uint32_t i = 0, left = p;
        for (uint32_t k = 0; k + 1 < nu; k++) {   // row i holds the nu - 1 - i pairs (i, j > i)
            const bool next = i == k && left >= nu - 1 - k;
            left -= next ? nu - 1 - k : 0u;
            i += next ? 1u : 0u;
        }
        const uint32_t lo = (uint32_t)__shfl((int)uval, (int)i), hi = (uint32_t)__shfl((int)uval, (int)(i + 1 + left));
        uint32_t e8, e6;
        pair_errors(uval, uw, nu, lo, hi, e8, e6);
        const uint32_t type = both && e6 < e8 ? 1u : 0u;
        // error (below 2^21), then place
        uint32_t key = ((type ? e6 : e8) << 6) | lane, m = key;
        for (int off = 32; off > 0; off >>= 1) m = min(m, (uint32_t)__shfl_xor((int)m, off));
        m = (uint32_t)__builtin_amdgcn_readfirstlane((int)m);
        if (m >> 6 < best) {
            best = m >> 6;
            const uint32_t k = m & 63u;
            best_first = at_lane(lo, k);
            best_second = at_lane(hi, k);
            best_type = at_lane(type, k);
        }
    }
    if (quality >= 3 && best) {
        const uint32_t probe = quality == 4 ? 16 : 8, side = 2 * probe + 1, all = side * side;
        // a row's low end is fixed where the row starts: row `row` keeps `row_lo`
        uint32_t row = ~0u, row_lo = 0, next = 0;
        while (next < all && best) {
            const uint32_t c = next + lane, dl = c / side, dh = c - dl * side;
            const uint32_t lo = dl == row ? row_lo : best_first + dl - probe, hi = best_second + dh - probe;
            uint32_t e8, e6;
            pair_errors(uval, uw, nu, lo & 0xFFu, hi & 0xFFu, e8, e6);
            const uint32_t type = both && e6 < e8 && e8 ? 1u : 0u, e = type ? e6 : e8;
            const uint64_t mask = __ballot(c < all && lo <= 255u && hi <= 255u && e < best);
            next += 64;
            if (mask) {
                const uint32_t k = (uint32_t)__builtin_ctzll(mask);
                best = at_lane(e, k);
                best_first = row_lo = at_lane(lo, k);
                best_second = at_lane(hi, k);
                best_type = at_lane(type, k);
                row = at_lane(dl, k);
                next = at_lane(c, k) + 1;
            }
        }
    }
    // the texels' selectors (the first nearest entry), one texel per lane
    uint32_t sel = 0, nearest = 0xFFFFFFFFu;
    for (uint32_t j = 0; j < 8; j++) {
        const uint32_t l = best_first, h = best_second;
        uint32_t p;
        if (j < 2) p = j ? h : l;
        else if (!best_type) p = (l * (8 - j) + h * (j - 1)) / 7;
        else p = j < 6 ? (l * (6 - j) + h * (j - 1)) / 5 : j == 6 ? 0u : 255u;
        const int d = (int)mine - (int)p;
        const uint32_t e = (uint32_t)(d * d);
        if (e < nearest) {
            nearest = e;
            sel = j;
        }
    }
    E2Result r;
    uint32_t f = best_first, sc = best_second;
    r.reordered = 0;
    if (f == sc) {
        sel = 0;
    } else if (best_type) {
        if (f > sc) {
            const uint32_t x = f; f = sc; sc = x;
            r.reordered = 1;
            sel = k_six_invert[sel];
        }
    } else if (f <= sc) {
        const uint32_t x = f; f = sc; sc = x;
        r.reordered = 1;
        sel = k_eight_invert[sel];
    }
    const uint64_t mine48 = (uint64_t)sel << (3 * t);
    uint32_t s0 = (uint32_t)mine48, s1 = (uint32_t)(mine48 >> 32);
    for (int off = 8; off > 0; off >>= 1) {
        s0 |= (uint32_t)__shfl_xor((int)s0, off);
        s1 |= (uint32_t)__shfl_xor((int)s1, off);
    }
    r.err = best;
    r.first = f;
    r.second = sc;
    r.type = best_type;
    r.sel48 = (uint64_t)at_lane(s0, 0) | ((uint64_t)at_lane(s1, 0) << 32);
    return r;
}

// The wave's blocks, lane k < n holding block k's values in w: every lane's
// result.
__device__ inline E2Result dxt5a_wave(const uint32_t (&w)[4], uint32_t n, int quality, bool both)
{
    const uint32_t lane = lane_id();
    E2Result r;
    r.err = 0;
    r.first = r.second = w[0] & 0xFFu;
    r.type = 0;
    r.reordered = 0;
    r.sel48 = 0;
    // one value, or two: the first pair is exact (the 8-value palette holds
    // both ends), in canonical order the larger value first
    const uint32_t a = w[0] & 0xFFu;
    uint32_t other = a;
    uint64_t is_a = 0;
    bool more = false;
#pragma unroll
    for (uint32_t t = 0; t < 16; t++) {
        const uint32_t v = (w[t >> 2] >> (8 * (t & 3u))) & 0xFFu;
        other = other == a ? v : other;
        more |= v != a && v != other;
        is_a |= v == a ? 1ull << (3 * t) : 0ull;
    }
    if (!more && other != a) {
        constexpr uint64_t kOnes = 0x249249249249ull;   // selector 1 on every texel
        r.first = max(a, other);
        r.second = min(a, other);
        r.reordered = a < other ? 1u : 0u;
        r.sel48 = a < other ? is_a : is_a ^ kOnes;      // the second end's texels
    }
    uint64_t todo = __ballot(lane < n && more);
    while (todo) {
        const uint32_t k = (uint32_t)__builtin_ctzll(todo);
        todo &= todo - 1;
        const uint32_t wk[4] = {at_lane(w[0], k), at_lane(w[1], k), at_lane(w[2], k), at_lane(w[3], k)};
        const E2Result q = dxt5a_search(wk, quality, both);
        if (lane == k) r = q;
    }
    return r;
}

// Blocks per wave: one up to 43,690 blocks, then as many as keep the waves to
// about 21,845 (a wave searches its blocks in turn, but one with nothing to
// search costs little more than its start), up to one per lane.  Measured at
// 1024^2 (65,536 blocks), runs of 2 / 3 / 4: a normal map 1,289 / 1,320 / 1,354
// us, a flat channel 10.2 / 7.8 / 7.8 (one lane per block: 8.5).
inline uint32_t blocks_per_wave(uint64_t n) { return (uint32_t)std::min<uint64_t>(64, std::max<uint64_t>(1, n * 3 >> 16)); }

// The wave's first block and its number of blocks.
__device__ inline uint32_t wave_blocks(uint32_t per, uint32_t total, uint32_t& first)
{
    const uint64_t f = (uint64_t)(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) * per;
    first = (uint32_t)min(f, (uint64_t)total);
    first = (uint32_t)__builtin_amdgcn_readfirstlane((int)first);
    return min(per, total - first);
}

__device__ inline uint32_t pack4(uint32_t a, uint32_t b, uint32_t c, uint32_t d) { return a | b << 8 | c << 16 | d << 24; }

// values: 16 bytes per block; outputs per block: sel48 (u64), err (u64),
// meta = first | second << 8 | type << 16 | reordered << 24
__global__ void __launch_bounds__(256) dxt5a_blocks_kernel(const uint8_t* __restrict__ values, uint32_t nblocks,
                                                           uint32_t per, int quality, int use_both,
                                                           uint64_t* __restrict__ sel, uint64_t* __restrict__ err,
                                                           uint32_t* __restrict__ meta)
{
    uint32_t first;
    const uint32_t n = wave_blocks(per, nblocks, first), lane = lane_id();
    if (!n) return;
    const uint32_t b = first + min(lane, n - 1);
    const uint4 raw = reinterpret_cast<const uint4*>(values)[b];
    const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
    const E2Result r = dxt5a_wave(w, n, quality, use_both != 0);
    if (lane >= n) return;
    sel[b] = r.sel48;
    err[b] = r.err;
    meta[b] = r.first | (r.second << 8) | (r.type << 16) | (r.reordered << 24);
}

// Whole image: RGBA8 texels, one channel, DXT5 alpha blocks out (8 bytes each).
__global__ void __launch_bounds__(256) dxt5a_image_kernel(const uint8_t* __restrict__ rgba, uint32_t width,
                                                          uint32_t height, uint32_t comp, uint32_t blocks_x,
                                                          uint32_t blocks_y, uint32_t per, int quality, int use_both,
                                                          uint64_t* __restrict__ out, uint32_t out_stride,
                                                          uint64_t* __restrict__ err)
{
    uint32_t first;
    const uint32_t n = wave_blocks(per, blocks_x * blocks_y, first), lane = lane_id();
    if (!n) return;
    const uint32_t b = first + min(lane, n - 1);
    const uint32_t bx = b % blocks_x, by = b / blocks_x;
    uint32_t w[4];
    for (uint32_t y = 0; y < 4; y++) {
        const size_t row = (size_t)min(by * 4 + y, height - 1) * width;
        uint32_t v[4];
        for (uint32_t x = 0; x < 4; x++) v[x] = rgba[4 * (row + min(bx * 4 + x, width - 1)) + comp];
        w[y] = pack4(v[0], v[1], v[2], v[3]);
    }
    const E2Result r = dxt5a_wave(w, n, quality, use_both != 0);
    if (lane >= n) return;
    out[(size_t)b * out_stride] = (uint64_t)r.first | ((uint64_t)r.second << 8) | (r.sel48 << 16);
    if (err) err[b] = r.err;
}

// Texture-set encode, alpha elements (DXT5 alpha, DXN channels, DXT5A) of
// many level images in one flat order, each wave taking runs of `per`
// elements with a grid stride; a run may reach over a job's end.
__global__ void __launch_bounds__(256) dxt5a_set_kernel(const crn2::SetJob* __restrict__ jobs, uint32_t njobs,
                                                        uint64_t begin, uint64_t end, uint32_t per, int quality)
{
    const uint32_t lane = lane_id();
    const uint64_t waves = (uint64_t)gridDim.x * (blockDim.x >> 6);
    const uint64_t wave = (uint64_t)blockIdx.x * (blockDim.x >> 6) +
                          (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    for (uint64_t i0 = begin + wave * per; i0 < end; i0 += waves * per) {
        const uint32_t n = (uint32_t)min((uint64_t)per, end - i0);
        const uint64_t i = i0 + min(lane, n - 1);
        const crn2::SetJob j = jobs[crn2::set_job_of(jobs, njobs, i)];
        const uint32_t b = (uint32_t)(i - j.first);
        const uint32_t bx = b % j.blocks_x, by = b / j.blocks_x;
        uint32_t w[4];
        for (uint32_t y = 0; y < 4; y++) {
            const size_t row = (size_t)min(by * 4 + y, j.height - 1) * j.width;
            uint32_t v[4];
            for (uint32_t x = 0; x < 4; x++) v[x] = (j.rgba[row + min(bx * 4 + x, j.width - 1)] >> (8 * j.comp)) & 0xFFu;
            w[y] = pack4(v[0], v[1], v[2], v[3]);
        }
        // one set has one flag for its alpha elements (crn2_encode_set_create)
        const bool both = (uint32_t)__builtin_amdgcn_readfirstlane((int)j.flags) != 0;
        const E2Result r = dxt5a_wave(w, n, quality, both);
        if (lane < n) j.out[(size_t)b * j.stride] = (uint64_t)r.first | ((uint64_t)r.second << 8) | (r.sel48 << 16);
    }
}

}  // namespace

extern "C" int crn2_dxt5a_blocks_device(const void* values, uint32_t nblocks, int quality, int use_both,
                                        void* selectors48, void* errors, void* meta, void* stream)
{
    if (!values || !selectors48 || !errors || !meta || quality < 0 || quality > 4) return CRN2_EINVAL;
    if (reinterpret_cast<uintptr_t>(values) & 15) return CRN2_EINVAL;
    if (!nblocks) return CRN2_OK;
    hipStream_t s = static_cast<hipStream_t>(stream);
    // launch shapes (threads per workgroup; identical results): 256, 64, 128
    auto launch = [&](int shape) -> hipError_t {
        const uint32_t tb = shape == 1 ? 64 : shape == 2 ? 128 : 256, per = blocks_per_wave(nblocks);
        const uint32_t wg = tb / 64 * per, nb = (uint32_t)(((uint64_t)nblocks + wg - 1) / wg);
        hipLaunchKernelGGL(dxt5a_blocks_kernel, dim3(nb), dim3(tb), 0, s, static_cast<const uint8_t*>(values),
                           nblocks, per, quality, use_both, static_cast<uint64_t*>(selectors48),
                           static_cast<uint64_t*>(errors), static_cast<uint32_t*>(meta));
        return hipGetLastError();
    };
    const int shape = crn2::tuner().pick(crn2::TUNE_DXT5A, nblocks, 3, 0, s, launch);
    return launch(shape) == hipSuccess ? CRN2_OK : CRN2_EHIP;
}

extern "C" int crn2_encode_dxt5a_image_device(const void* rgba, uint32_t width, uint32_t height, uint32_t comp,
                                              int quality, int use_both, void* blocks, uint32_t block_stride_u64,
                                              void* errors, void* stream)
{
    if (!rgba || !blocks || !width || !height || comp > 3 || quality < 0 || quality > 4 || !block_stride_u64)
        return CRN2_EINVAL;
    const uint32_t bx = (width + 3) / 4, by = (height + 3) / 4;
    const uint32_t n = bx * by, tb = 256, per = blocks_per_wave(n), wg = tb / 64 * per;
    const uint32_t nb = (uint32_t)(((uint64_t)n + wg - 1) / wg);
    hipLaunchKernelGGL(dxt5a_image_kernel, dim3(nb), dim3(tb), 0, static_cast<hipStream_t>(stream),
                       static_cast<const uint8_t*>(rgba), width, height, comp, bx, by, per, quality, use_both,
                       static_cast<uint64_t*>(blocks), block_stride_u64, static_cast<uint64_t*>(errors));
    return hipGetLastError() == hipSuccess ? CRN2_OK : CRN2_EHIP;
}

extern "C" uint32_t crn2_dxt5a_set_per_wave(uint64_t elements) { return blocks_per_wave(elements); }

extern "C" int crn2_dxt5a_set_launch(const crn2::SetJob* jobs, uint32_t njobs, uint64_t begin, uint64_t end,
                                     int quality, uint32_t per, uint32_t grid, uint32_t tb, hipStream_t stream)
{
    if (!jobs || !njobs || !grid || !per || per > 64 || (tb != 64 && tb != 128 && tb != 256) || quality < 0 ||
        quality > 4)
        return CRN2_EINVAL;
    if (begin >= end) return CRN2_OK;
    hipLaunchKernelGGL(dxt5a_set_kernel, dim3(grid), dim3(tb), 0, stream, jobs, njobs, begin, end, per, quality);
    return hipGetLastError() == hipSuccess ? CRN2_OK : CRN2_EHIP;
}
