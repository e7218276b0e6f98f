// mip_gpu.hip -- mip generation on the GPU: mipmapped_texture::
// generate_mipmaps (crnlib/crn_mipmapped_texture.cpp:2140-2220) with
// image_utils::resample (crnlib/crn_image_utils.cpp:478-865) and crnlib's
// separable Resampler (crnlib/crn_resampler.cpp), bit-exact.
//
// Every level is resampled from level 0 in two passes.  A pass is a set of
// sequential dot products: output o of line k is
//     s = 0;  s += in[k][p] * w  for (p, w) in list(o), in list order,
// (the reference's Y pass starts from the first product, which differs from
// 0 + it only in the sign of a zero) with separate float multiplies and adds
// (-ffp-contract=off), so every sum rounds exactly as the reference's.  A
// list is stored as runs of contributors: a run of one texel repeated (the
// clamped edge of a wide filter: most of the contributors of the deepest
// levels) or a run of consecutive texels.  An output's longest consecutive run
// is its main one (all there is, away from the edges).
// Neighbouring outputs share most of their texels (5.4 outputs each with the
// default Kaiser filter), so a wave sums kGroup = 4 outputs at once: the runs
// before their main ones, output by output; then the texels of all four main
// runs in order, each loaded and converted once for four products, with
// weight 0 where it is outside an output's run (s + v * 0 == s up to the sign
// of a zero sum, which nothing later tells apart); then the runs behind.
// What bounds it: the loads and table look-ups of samples where lists are
// short, one output's serial chain where they are long (dot_long).  3840x2160
// with the default filter, one output at a time and a texel per load: pass 1
// 595 us, pass 2 272 us; now 245 and 119 us.  Eight outputs at once would load a
// quarter less, and multiply by more zeros.
// The order of the passes is the reference's choice per level: X then Y
// (always, for the multithreaded resampler) or, where the single-thread
// Resampler delays X, Y then X.  Y then X is run as X then Y on the
// transposed image -- the same sums in the same order.
//
// Layout in HBM (one plane per component c):
//   level-0 planes ... bytes, four texels of a line in a word: lx[c][x / 4][y]
//                      (the lanes of a wave are 64 consecutive rows, so a
//                      load is 256 coalesced bytes) and/or ly[c][y / 4][x];
//                      every level re-reads them, so bytes rather than floats
//                      (the sRGB table sits in LDS) cut the dominant traffic
//                      4x;
//   pass-1 output .... inter[c][line][o], o along the first pass's axis;
//   pass 2 ........... lanes = 64 consecutive o, one wave per component, the
//                      contributor lists of the block's four output lines in
//                      scalar registers; clamp to [0, 1], (int)(255 x + .5) or the
//                      linear-to-sRGB table, optional renorm_normal_map, one
//                      RGBA8 texel per lane.
// Both passes cover every level in one launch, the deepest levels first:
// their sums are the longest serial chains (level l has about 5.4 * 2^l
// contributors per output with the default Kaiser filter) and start while the
// wide levels fill the rest of the GPU.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <new>
#include <type_traits>
#include <vector>

#include "crn2_internal.h"
#include "mip_plan.h"

namespace {

// outputs that a wave sums at once
constexpr uint32_t kGroup = 4;
// groups per pass-1 wave, one after the other: 16 outputs (64 bytes of each
// lane's line) where lists are shorter than kMidList, one group where they are
// longer (shorter serial chains, more waves)
constexpr uint32_t kGroupsPerWave = 4;
constexpr uint32_t kMidList = 64;
// Lists of at least this many contributors per output take a wave for each
// output (dot_long): the deepest levels' sums are the longest chains of the
// launch.  Pass 1 has a wave for every 64 lines all the same, and a level of 690
// contributors takes 17 us in groups; pass 2 has few waves, and the same level
// takes 44 us in groups and 2 us a wave for each output.
// So where the waves of single outputs are few, they are taken from much shorter
// lists on: then nothing hides a chain of four outputs' texels (pass 1 up to
// 1,024 waves a level, pass 2 up to 256 blocks; with the limits for any number of
// waves alone, 100x37 with the default filter 36 us before groups, 40 with them,
// 26 so; 256^2 92 / 57 / 36; 1000x700 box 89 / 106 / 84; with twice as many
// waves 2048^2 takes 2 % longer again).  Not with wrapped edges, whose lists are
// many runs: a single sum starts afresh with each (16x16: 18 us in groups, 20
// singly).
constexpr uint32_t kLongList = 1024, kLongList2 = 256;
constexpr uint32_t kFewList = 64, kFewWaves = 1024, kFewList2 = 32, kFewBlocks2 = 256;
constexpr uint32_t kChunk = 256;   // weights that dot_long fetches at once
constexpr uint32_t kRunPad = 16;   // a run's weights are padded with zeros to a multiple of this (so that runs start at 16-byte steps)

struct Pass1Level {
    uint32_t unit0;   // first wave of this level
    uint32_t nlb;     // blocks of 64 lines
    uint32_t single;  // 1: a wave sums one output, 0: `per` groups
    uint32_t per;
    uint32_t runs;    // waves per line block
    uint32_t lines;   // lines (rows for X first, columns for Y first)
    uint32_t d;       // outputs per line
    uint32_t s;       // source samples per line
    uint32_t list;    // index of the list's first group
    uint32_t layout;  // 0 = lx, 1 = ly
    uint64_t inter;   // float offset of this level's pass-1 output
};

struct Pass2Level {
    uint32_t block0;  // first block of this level
    uint32_t nxb;     // blocks of 64 pass-1 outputs
    uint32_t d2;      // output lines of pass 2
    uint32_t single;  // 1: a block makes one of them, 0: kGroup
    uint32_t lines;   // contributors' range (pass-1 lines)
    uint32_t d;       // pass-1 outputs per line = lanes
    uint32_t list;
    uint32_t os_lane, os_o;  // texel strides of the output: per lane, per pass-2 line
    uint64_t inter;
    uint64_t out;  // texel offset of this level in the chain
};

// contributors pix[k] .. pix[k] + (n - 1) * step with weights wt[w .. w + n)
struct Run {
    uint32_t pix, n, step, w;
};

// kGroup neighbouring outputs, output i the sum of the runs [run[i], end[i]);
// unless the list is long: texel pre_pix with pre_n weights per output at
// wt[pre_w + kGroup * k + i] and then the runs [run[i], before[i]) (one of the
// two is empty); texels pix .. pix + n - 1 (pix a multiple of 4)
// with weights wt[w + kGroup * k + i] of output i stand for its runs
// [before[i], after[i]); then texel post_pix and the runs [after[i], end[i]) in
// the same way.  Outputs past the list's
// last have no runs and weights 0.
struct alignas(16) Group {
    uint32_t pix, n, w;
    uint32_t pre_pix, pre_n, pre_w, post_pix, post_n, post_w, pad[3];
    uint32_t run[kGroup], before[kGroup], after[kGroup], end[kGroup];
};

struct Tables {
    const Pass1Level* p1;
    const Pass2Level* p2;
    const Group* groups;
    const Run* runs;
    const float* wt;
    const float* s2l;
    const uint8_t* l2s;
};

// The tables stay as they are while a kernel runs, and say so: what is the same
// for a whole wave is then loaded by scalar loads, whatever else the kernel
// writes or orders (with wave barriers in dot_long and plain pointers the
// 3840x2160 chain took 562 us instead of 391).
typedef __attribute__((address_space(4))) const Pass1Level cPass1Level;
typedef __attribute__((address_space(4))) const Pass2Level cPass2Level;
typedef __attribute__((address_space(4))) const Group cGroup;
typedef __attribute__((address_space(4))) const Run cRun;
typedef __attribute__((address_space(4))) const float cfloat;
typedef float f4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(4))) const f4 cf4;

__device__ __forceinline__ uint32_t uni(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ float unif(float v) { return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v))); }

// Source samples: float (the intermediate), or level-0 bytes converted as
// resample_single_thread does (crn_image_utils.cpp:575-590): colour through
// srgb_to_linear when sRGB (the 256 floats staged in LDS), alpha and linear
// colour v * (1/255).
enum Src { kFloat, kLinear8, kTable8 };

template <Src S>
__device__ __forceinline__ float convert8(uint32_t v, const float* tab)
{
    if constexpr (S == kTable8) return tab[v];
    else return __fmul_rn((float)v, 1.0f / 255.0f);
}

// Texel p of the lane's line.
template <Src S>
__device__ __forceinline__ float sample(const void* base, uint32_t p, uint32_t lane, uint32_t stride, const float* tab)
{
    if constexpr (S == kFloat) return static_cast<const float*>(base)[p * stride + lane];
    else return convert8<S>(static_cast<const uint8_t*>(base)[4 * ((p >> 2) * stride + lane) + (p & 3u)], tab);
}

// s + src(p) * w over the runs [rb, re) of one output, in order.  Runs and
// weights are wave-uniform (scalar loads).  A batch past the end of a run
// repeats its last texel with weight 0; the weights of a batch are read as 16
// consecutive floats (the table buffer continues past the last list).
template <Src S>
__device__ __forceinline__ float dot_runs(const Tables& t, uint32_t rb, uint32_t re, const void* base,
                                          uint32_t lane, uint32_t stride, float s, const float* tab)
{
    for (uint32_t g = rb; g < re; g++) {
        const cRun* r = (cRun*)t.runs + g;
        const uint32_t n = uni(r->n), p = uni(r->pix);
        const cfloat* wp = (cfloat*)t.wt + uni(r->w);
        if (uni(r->step) == 0) {
            const float v = sample<S>(base, p, lane, stride, tab);
            uint32_t k = 0;
            for (; k + 16 <= n; k += 16) {
#pragma unroll
                for (int i = 0; i < 16; i++) s = __fadd_rn(s, __fmul_rn(v, unif(wp[k + i])));
            }
            for (; k < n; k++) s = __fadd_rn(s, __fmul_rn(v, unif(wp[k])));
        } else {
            for (uint32_t k = 0; k < n; k += 16) {
                float v[16];
#pragma unroll
                for (int i = 0; i < 16; i++) v[i] = sample<S>(base, p + min(k + i, n - 1), lane, stride, tab);
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    const float w = unif(wp[k + i]);
                    s = __fadd_rn(s, __fmul_rn(v[i], k + i < n ? w : 0.0f));
                }
            }
        }
    }
    return s;
}

// kGroup sums over one texel repeated: n weights per output, a multiple of 4.
template <Src S>
__device__ __forceinline__ void dot_repeat(const cfloat* wp, uint32_t n, const void* base, uint32_t p, uint32_t lane,
                                           uint32_t stride, float (&s)[kGroup], const float* tab)
{
    if (!n) return;
    const float v = sample<S>(base, p, lane, stride, tab);
    for (uint32_t k = 0; k < n; k += 4) {
#pragma unroll
        for (uint32_t b = 0; b < 4; b++) {
#pragma unroll
            for (uint32_t i = 0; i < kGroup; i++)
                s[i] = __fadd_rn(s[i], __fmul_rn(v, unif(wp[kGroup * (k + b) + i])));
        }
    }
}

// The kGroup sums of group G.  Its texels come in batches of 8, the next
// batch's loads in flight while one is summed; a batch past the end repeats
// the last texels with weights 0 (the table holds them).
template <Src S>
__device__ __forceinline__ void dot_group(const Tables& t, const cGroup* G, const void* base, uint32_t lane,
                                          uint32_t stride, float (&s)[kGroup], const float* tab)
{
#pragma unroll
    for (uint32_t i = 0; i < kGroup; i++)
        s[i] = dot_runs<S>(t, uni(G->run[i]), uni(G->before[i]), base, lane, stride, 0.0f, tab);
    dot_repeat<S>((cfloat*)t.wt + uni(G->pre_w), uni(G->pre_n), base, uni(G->pre_pix), lane, stride, s, tab);
    const uint32_t p = uni(G->pix), n = uni(G->n);
    const cfloat* wp = (cfloat*)t.wt + uni(G->w);
    constexpr uint32_t kBatch = 8, kWords = S == kFloat ? kBatch : kBatch / 4;
    typedef typename std::conditional<S == kFloat, float, uint32_t>::type Word;
    const Word* src = static_cast<const Word*>(base) + (size_t)(S == kFloat ? p : p >> 2) * stride + lane;
    const uint32_t words = S == kFloat ? n : (n + 3) >> 2;
    Word v[kWords];
#pragma unroll
    for (uint32_t i = 0; i < kWords; i++) v[i] = words ? src[min(i, words - 1) * stride] : Word(0);
    for (uint32_t k = 0, w = 0; k < n; k += kBatch) {
        w += kWords;
        Word x[kWords];
#pragma unroll
        for (uint32_t i = 0; i < kWords; i++) x[i] = src[min(w + i, words - 1) * stride];
#pragma unroll
        for (uint32_t b = 0; b < kBatch; b++) {
            float f;
            if constexpr (S == kFloat) f = v[b];
            else f = convert8<S>((v[b / 4] >> (8 * (b % 4))) & 0xFFu, tab);
#pragma unroll
            for (uint32_t i = 0; i < kGroup; i++)
                s[i] = __fadd_rn(s[i], __fmul_rn(f, unif(wp[kGroup * (k + b) + i])));
        }
#pragma unroll
        for (uint32_t i = 0; i < kWords; i++) v[i] = x[i];
    }
    dot_repeat<S>((cfloat*)t.wt + uni(G->post_w), uni(G->post_n), base, uni(G->post_pix), lane, stride, s, tab);
#pragma unroll
    for (uint32_t i = 0; i < kGroup; i++)
        s[i] = dot_runs<S>(t, uni(G->after[i]), uni(G->end[i]), base, lane, stride, s[i], tab);
}

// One output's sum where its list is long: a serial chain of thousands of
// products and adds, which nothing overlaps at the end of the launch, so all
// that it reads is under way long before.  The weights come 256 at a time,
// four to a lane, one to two chunks ahead of the sum, and are handed round
// through `wl` (two chunks of LDS, this wave's own; the wave barriers, which
// emit nothing, keep the lanes' stores and each other's reads in order); a
// consecutive run's texels come 32 (of the byte planes 64, four to a load) at a
// time, a batch ahead.  With scalar loads of the weights, and waits for each
// batch of 16 texels, a contributor took some 60 cycles, and the one sum of the
// deepest level of a 2160-row image all of pass 2's 272 us.
template <Src S>
__device__ float dot_long(const Tables& t, uint32_t rb, uint32_t re, const void* base, uint32_t lane,
                          uint32_t stride, const float* tab, float* wl)
{
    const uint32_t me = threadIdx.x & 63u;
    float s = 0.0f;
    for (uint32_t g = rb; g < re; g++) {
        const cRun* r = (cRun*)t.runs + g;
        const uint32_t n = uni(r->n), p = uni(r->pix), step = uni(r->step);
        const cf4* wp = (cf4*)((cfloat*)t.wt + uni(r->w)) + me;
        f4* mine = reinterpret_cast<f4*>(wl) + me;
        // chunk 0 in place, chunk 1 under way
        __builtin_amdgcn_wave_barrier();
        mine[0] = wp[0];
        __builtin_amdgcn_wave_barrier();
        f4 ahead = wp[kChunk / 4];
        auto chunk = [&](uint32_t c) {   // halfway through chunk c: puts chunk c + 1 in place
            __builtin_amdgcn_wave_barrier();
            mine[kChunk / 4 * ((c + 1) & 1u)] = ahead;
            __builtin_amdgcn_wave_barrier();
            ahead = wp[kChunk / 4 * (c + 2)];
        };
        auto read16 = [&](uint32_t k, float (&w)[16]) {
            const f4* q = reinterpret_cast<const f4*>(wl + (k & (2 * kChunk - 1)));
#pragma unroll
            for (uint32_t i = 0; i < 4; i++) {
                const f4 v = q[i];
                w[4 * i] = v.x;
                w[4 * i + 1] = v.y;
                w[4 * i + 2] = v.z;
                w[4 * i + 3] = v.w;
            }
        };
        float w[16];
        read16(0, w);
        if (step == 0) {
            const float v = sample<S>(base, p, lane, stride, tab);
            auto add16 = [&](const float (&w)[16]) {
#pragma unroll
                for (uint32_t i = 0; i < 16; i++) s = __fadd_rn(s, __fmul_rn(v, w[i]));
            };
            float wn[16];
            const uint32_t n16 = (n + 15) & ~15u;
            uint32_t k = 0;
            for (; k + 32 <= n16; k += 32) {   // (16 at a time: pass 2 of the 3840x2160 chain 117 -> 141 us)
                if ((k & (kChunk - 1)) == kChunk / 2) chunk(k / kChunk);
                read16(k + 16, wn);
                add16(w);
                read16(k + 32, w);
                add16(wn);
            }
            if (k < n16) add16(w);
        } else {
            // (a run in the byte planes starts at a word: add_list)
            typedef typename std::conditional<S == kFloat, float, uint32_t>::type Word;
            constexpr uint32_t kPer = S == kFloat ? 1 : 4, kWords = S == kFloat ? 32 : 16, kBatch = kPer * kWords;
            const Word* src = static_cast<const Word*>(base) + (size_t)(p / kPer) * stride + lane;
            const uint32_t words = (n + kPer - 1) / kPer;
            Word v[kWords];
#pragma unroll
            for (uint32_t i = 0; i < kWords; i++) v[i] = src[min(i, words - 1) * stride];
            for (uint32_t k = 0, q = 0; k < n; k += kBatch) {
                q += kWords;
                Word vn[kWords];
#pragma unroll
                for (uint32_t i = 0; i < kWords; i++) vn[i] = src[min(q + i, words - 1) * stride];
#pragma unroll
                for (uint32_t h = 0; h < kBatch / 16; h++) {
                    const uint32_t at = k + 16 * h;
                    if (at < n) {
                        if ((at & (kChunk - 1)) == kChunk / 2) chunk(at / kChunk);
                        float wn[16];
                        read16(at + 16, wn);
#pragma unroll
                        for (uint32_t i = 0; i < 16; i++) {
                            float f;
                            if constexpr (S == kFloat) f = v[16 * h + i];
                            else f = convert8<S>((v[4 * h + i / 4] >> (8 * (i % 4))) & 0xFFu, tab);
                            s = __fadd_rn(s, __fmul_rn(f, w[i]));
                        }
#pragma unroll
                        for (uint32_t i = 0; i < 16; i++) w[i] = wn[i];
                    }
                }
#pragma unroll
                for (uint32_t i = 0; i < kWords; i++) v[i] = vn[i];
            }
        }
    }
    return s;
}

// ------------------------------------------------------------ level-0 planes

// RGBA8 -> byte planes per component, a word for four texels along x (lx) and/or
// along y (ly), zero past the edge; also copies the image to `copy` (level 0 of
// the chain) where that is another buffer.  32x32 tiles.
__global__ void __launch_bounds__(256) mip_planes_kernel(const uint32_t* __restrict__ rgba, uint32_t w, uint32_t h,
                                                         uint32_t* __restrict__ lx, uint32_t* __restrict__ ly,
                                                         uint32_t ncomp, uint32_t* __restrict__ copy)
{
    __shared__ uint32_t tile[32][33];
    const uint32_t tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    const uint32_t x0 = blockIdx.x * 32, y0 = blockIdx.y * 32;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const uint32_t y = y0 + ty + 8 * i, x = x0 + tx;
        const bool in = x < w && y < h;
        const uint32_t p = in ? rgba[(size_t)y * w + x] : 0;
        tile[ty + 8 * i][tx] = p;
        if (copy && in) copy[(size_t)y * w + x] = p;
    }
    __syncthreads();
    const uint32_t w4 = (w + 3) / 4, h4 = (h + 3) / 4;
    auto gather = [](uint32_t a, uint32_t b, uint32_t c, uint32_t d, uint32_t comp) {
        const uint32_t k = 8 * comp;
        return ((a >> k) & 0xFFu) | ((b >> k) & 0xFFu) << 8 | ((c >> k) & 0xFFu) << 16 | (d >> k) << 24;
    };
    if (lx) {
        const uint32_t q = x0 / 4 + ty, y = y0 + tx;
        if (q < w4 && y < h) {
            const uint32_t* r = &tile[tx][4 * ty];
            for (uint32_t c = 0; c < ncomp; c++) lx[((size_t)c * w4 + q) * h + y] = gather(r[0], r[1], r[2], r[3], c);
        }
    }
    if (ly) {
        const uint32_t q = y0 / 4 + ty, x = x0 + tx;
        if (q < h4 && x < w) {
            const uint32_t a = tile[4 * ty][tx], b = tile[4 * ty + 1][tx], c2 = tile[4 * ty + 2][tx],
                           d = tile[4 * ty + 3][tx];
            for (uint32_t c = 0; c < ncomp; c++) ly[((size_t)c * h4 + q) * w + x] = gather(a, b, c2, d, c);
        }
    }
}

// ------------------------------------------------------------------- pass 1

// One wave per (level, component, 64 lines, `per` groups or one
// output); lanes are lines.
__global__ void __launch_bounds__(256) mip_pass1_kernel(Tables t, const uint32_t* __restrict__ lx,
                                                        const uint32_t* __restrict__ ly, float* __restrict__ inter,
                                                        uint32_t nlevels, uint32_t units, uint32_t ncomp, int srgb)
{
    __shared__ float tab[256];
    __shared__ __align__(16) float wl[4][2 * kChunk];
    tab[threadIdx.x] = t.s2l[threadIdx.x];
    __syncthreads();
    const uint32_t u = uni(blockIdx.x * 4 + (threadIdx.x >> 6));
    if (u >= units) return;
    uint32_t l = 0;
    const cPass1Level* L = (cPass1Level*)t.p1;
    while (l + 1 < nlevels && L[1].unit0 <= u) {
        l++;
        L++;
    }
    uint32_t rem = u - L->unit0;
    const uint32_t run = rem % L->runs;
    rem /= L->runs;
    const uint32_t lb = rem % L->nlb, c = rem / L->nlb;
    const uint32_t line = lb * 64 + (threadIdx.x & 63);
    const bool valid = line < L->lines;
    const uint32_t rl = valid ? line : L->lines - 1;
    const uint32_t* base = (L->layout ? ly : lx) + (size_t)c * ((L->s + 3) / 4) * L->lines;
    const bool table = srgb && c < 3;
    if (L->single) {
        const cGroup* G = (cGroup*)t.groups + L->list + run / kGroup;
        const uint32_t rb = uni(G->run[run % kGroup]), re = uni(G->end[run % kGroup]);
        float* mine = wl[threadIdx.x >> 6];
        const float s = table ? dot_long<kTable8>(t, rb, re, base, rl, L->lines, tab, mine)
                              : dot_long<kLinear8>(t, rb, re, base, rl, L->lines, tab, mine);
        if (valid) inter[L->inter + ((size_t)c * L->lines + rl) * L->d + run] = s;
        return;
    }
    const uint32_t ngroups = (L->d + kGroup - 1) / kGroup;
    for (uint32_t g = run * L->per; g < min(ngroups, (run + 1) * L->per); g++) {
        float s[kGroup];
        const cGroup* G = (cGroup*)t.groups + L->list + g;
        if (table) dot_group<kTable8>(t, G, base, rl, L->lines, s, tab);
        else dot_group<kLinear8>(t, G, base, rl, L->lines, s, tab);
        float* out = inter + L->inter + ((size_t)c * L->lines + rl) * L->d + kGroup * g;
        if (!valid) continue;
        if (!(L->d & 3u)) {
            *reinterpret_cast<float4*>(out) = make_float4(s[0], s[1], s[2], s[3]);
        } else {
#pragma unroll
            for (uint32_t i = 0; i < kGroup; i++)
                if (kGroup * g + i < L->d) out[i] = s[i];
        }
    }
}

// ------------------------------------------------------------------- pass 2

__device__ __forceinline__ float clamp01(float x)
{
    if (x < 0.0f) x = 0.0f;
    else if (x > 1.0f) x = 1.0f;
    return x;
}

// image_utils::renorm_normal_map for one texel (crn_image_utils.cpp:369-420)
__device__ void renorm(uint32_t* c)
{
    if (c[0] == 128 && c[1] == 128 && c[2] == 128) return;
    float v[3];
#pragma unroll
    for (int i = 0; i < 3; i++) {
        float f = (float)c[i];
        f = __fmul_rn(f, 1.0f / 255.0f);
        f = __fmul_rn(f, 2.0f);
        f = f - 1.0f;
        if (f < -1.0f) f = -1.0f;
        else if (f > 1.0f) f = 1.0f;
        v[i] = f;
    }
    float sum = __fmul_rn(v[0], v[0]);
    sum = __fadd_rn(sum, __fmul_rn(v[1], v[1]));
    sum = __fadd_rn(sum, __fmul_rn(v[2], v[2]));
    const float len = sqrtf(sum);
    if (len < .077f) {
        c[0] = c[1] = c[2] = 128;
    } else if (fabsf(len - 1.0f) > .077f) {
#pragma unroll
        for (int i = 0; i < 3; i++) {
            const float n = v[i] / len;
            float f = floorf(__fadd_rn(__fmul_rn(__fmul_rn(n + 1.0f, .5f), 255.0f), .5f));
            f = f < 0.0f ? 0.0f : (f > 255.0f ? 255.0f : f);
            c[i] = (uint32_t)f;
        }
        if (c[0] == 128 && c[1] == 128) c[2] = c[2] < 128 ? 0 : 255;
    }
}

// One block per (level, kGroup output lines of pass 2 or one, 64 lanes), one
// wave per component; wave i packs the texels of line i.
__global__ void __launch_bounds__(256, 4) mip_pass2_kernel(Tables t, const float* __restrict__ inter,
                                                        uint32_t* __restrict__ out, uint32_t nlevels,
                                                        uint32_t ncomp, int srgb, int renormalize)
{
    __shared__ uint32_t px[kGroup][4][64];
    __shared__ __align__(16) float wl[4][2 * kChunk];
    const uint32_t b = blockIdx.x;
    uint32_t l = 0;
    const cPass2Level* L = (cPass2Level*)t.p2;
    while (l + 1 < nlevels && L[1].block0 <= b) {
        l++;
        L++;
    }
    const uint32_t rem = b - L->block0;
    const uint32_t xb = rem % L->nxb, g = rem / L->nxb;
    const uint32_t c = uni(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const uint32_t x = xb * 64 + lane;
    const bool valid = x < L->d;
    const uint32_t rx = valid ? x : L->d - 1;
    float s[kGroup] = {0.0f, 0.0f, 0.0f, 0.0f};
    const uint32_t nout = L->single ? 1 : kGroup;
    if (c < ncomp) {
        const float* base = inter + L->inter + (size_t)c * L->lines * L->d;
        if (L->single) {
            const cGroup* G = (cGroup*)t.groups + L->list + g / kGroup;
            s[0] = dot_long<kFloat>(t, uni(G->run[g % kGroup]), uni(G->end[g % kGroup]), base, rx, L->d, nullptr, wl[c]);
        } else {
            dot_group<kFloat>(t, (cGroup*)t.groups + L->list + g, base, rx, L->d, s, nullptr);
        }
    }
#pragma unroll
    for (uint32_t i = 0; i < kGroup; i++) {
        uint32_t val = 255;
        const float v = clamp01(s[i]);
        if (c >= ncomp) {
        } else if (!srgb || c == 3) {
            val = (uint32_t)min(255, max(0, (int)__fadd_rn(__fmul_rn(255.0f, v), .5f)));
        } else {
            val = t.l2s[min(8191, max(0, (int)__fadd_rn(__fmul_rn(8192.0f, v), .5f)))];
        }
        px[i][c][lane] = val;
    }
    __syncthreads();
    const uint32_t o2 = nout * g + c;
    if (c < nout && o2 < L->d2 && valid) {
        uint32_t q[4] = {px[c][0][lane], px[c][1][lane], px[c][2][lane], px[c][3][lane]};
        if (renormalize) renorm(q);
        out[L->out + (size_t)o2 * L->os_o + (size_t)x * L->os_lane] = q[0] | q[1] << 8 | q[2] << 16 | q[3] << 24;
    }
}

bool hip_ok(hipError_t e) { return e == hipSuccess; }

}  // namespace

struct crn2_mip_plan {
    uint32_t magic;
    uint32_t width, height, levels, ncomp;
    crn2_mip_params params;
    std::vector<uint64_t> level_ofs;  // bytes
    std::vector<uint8_t> y_first;
    uint64_t chain_bytes;
    // device
    void* tables = nullptr;
    void* scratch = nullptr;
    Tables t{};
    uint32_t *lx = nullptr, *ly = nullptr;  // level-0 planes, four texels a word
    float* inter = nullptr;
    uint32_t units1 = 0, blocks2 = 0;
    // stage timing (HIP events on the run stream): planes, pass 1, pass 2
    bool prof = false;
    hipEvent_t ev[4] = {};
    double ms[3] = {};
    uint64_t runs = 0;
};

namespace {

constexpr uint32_t kPlanMagic = 0x4d495032u;

bool plan_ok(const crn2_mip_plan* p) { return p && p->magic == kPlanMagic; }

void plan_free(crn2_mip_plan* p)
{
    if (p->tables) (void)hipFree(p->tables);
    if (p->scratch) (void)hipFree(p->scratch);
    for (hipEvent_t& e : p->ev)
        if (e) (void)hipEventDestroy(e);
    p->magic = 0;
    delete p;
}

size_t align_up(size_t v, size_t a) { return (v + a - 1) / a * a; }

}  // namespace

extern "C" {

uint32_t crn2_mip_level_count(uint32_t width, uint32_t height, uint32_t min_mip_size, uint32_t max_levels)
{
    if (!width || !height) return 0;
    return crn2mip::level_count(width, height, min_mip_size, max_levels);
}

int crn2_mip_contributors(uint32_t src, uint32_t dst, int wrap, uint32_t filter, float filter_scale, uint32_t* offs,
                          uint32_t* pix, float* weight, uint32_t cap)
{
    if (!src || !dst || src > 16384 || dst > 16384 || (cap && (!pix || !weight))) return CRN2_EINVAL;
    crn2mip::List L;
    if (!crn2mip::make_list(src, dst, wrap != 0, filter, filter_scale, L)) return CRN2_EINVAL;
    if (offs) std::memcpy(offs, L.offs.data(), L.offs.size() * sizeof(uint32_t));
    const size_t n = std::min<size_t>(cap, L.pix.size());
    if (n) {
        std::memcpy(pix, L.pix.data(), n * sizeof(uint32_t));
        std::memcpy(weight, L.wt.data(), n * sizeof(float));
    }
    return (int)L.pix.size();
}

int crn2_mip_gamma_tables(float gamma, float* srgb_to_linear, uint8_t* linear_to_srgb)
{
    if (!srgb_to_linear || !linear_to_srgb || !(gamma > 0.0f)) return CRN2_EINVAL;
    crn2mip::gamma_tables(gamma, srgb_to_linear, linear_to_srgb);
    return CRN2_OK;
}

int crn2_mip_plan_create(uint32_t width, uint32_t height, const crn2_mip_params* params, crn2_mip_plan** out)
{
    if (!out || !params) return CRN2_EINVAL;
    *out = nullptr;
    if (params->flags & ~31u) return CRN2_EINVAL;
    std::vector<crn2mip::Level> lv;
    if (!crn2mip::plan_levels(width, height, *params, lv)) return CRN2_EINVAL;
    crn2_mip_plan* p = new (std::nothrow) crn2_mip_plan;
    if (!p) return CRN2_ENOMEM;
    p->magic = kPlanMagic;
    p->width = width;
    p->height = height;
    p->params = *params;
    p->levels = (uint32_t)lv.size() + 1;
    p->ncomp = (params->flags & CRN2_MIP_ALPHA) ? 4 : 3;
    p->level_ofs.assign(1, 0);
    p->y_first.assign(1, 0);
    uint64_t ofs = (uint64_t)width * height * 4;
    for (const auto& v : lv) {
        p->level_ofs.push_back(ofs);
        p->y_first.push_back(v.xfirst ? 0 : 1);
        ofs += (uint64_t)v.width * v.height * 4;
    }
    p->chain_bytes = ofs;
    if (lv.empty()) {
        *out = p;
        return CRN2_OK;
    }
    const uint32_t nl = (uint32_t)lv.size();
    const uint32_t nc = p->ncomp;
    // host image of the device tables
    std::vector<Pass1Level> p1(nl);
    std::vector<Pass2Level> p2(nl);
    std::vector<Group> groups;
    std::vector<Run> runs;
    std::vector<float> wt;
    bool need_lx = false, need_ly = false;
    uint64_t inter_floats = 0;
    uint32_t units = 0, blocks = 0;
    // a list as runs (one texel repeated, step 0, or consecutive texels, step 1)
    // and groups of outputs
    // Every output's texels in one piece, edge texels perhaps repeated (no wrapped edges)
    auto one_piece = [](const crn2mip::List& L) {
        for (size_t o = 0; o + 1 < L.offs.size(); o++)
            for (uint32_t k = L.offs[o] + 1; k < L.offs[o + 1]; k++)
                if (L.pix[k] != L.pix[k - 1] && L.pix[k] != L.pix[k - 1] + 1) return false;
        return true;
    };
    auto add_list = [&](const crn2mip::List& L, bool single) {
        const uint32_t at = (uint32_t)groups.size();
        const size_t n = L.offs.size() - 1;
        for (size_t o0 = 0; o0 < n; o0 += kGroup) {
            Group G;
            std::memset(&G, 0, sizeof(G));
            uint32_t lo = 0xFFFFFFFFu, hi = 0;
            Run main[kGroup] = {};
            for (uint32_t i = 0; i < kGroup && o0 + i < n; i++) {
                G.run[i] = (uint32_t)runs.size();
                uint32_t best = 0xFFFFFFFFu;
                for (uint32_t k = L.offs[o0 + i], end = L.offs[o0 + i + 1]; k < end;) {
                    const uint32_t p = L.pix[k];
                    uint32_t m = 1, step = 1;
                    if (k + 1 < end && L.pix[k + 1] == p) {
                        step = 0;
                        while (k + m < end && L.pix[k + m] == p) m++;
                    } else {
                        while (k + m < end && L.pix[k + m] == p + m) m++;
                    }
                    if (step && (best == 0xFFFFFFFFu || m > runs[best].n)) best = (uint32_t)runs.size();
                    // a consecutive run starts at a multiple of 4, from there on with weights 0
                    const uint32_t lead = step ? p & 3u : 0;
                    runs.push_back(Run{p - lead, m + lead, step, (uint32_t)wt.size()});
                    wt.resize(wt.size() + lead, 0.0f);
                    wt.insert(wt.end(), L.wt.begin() + k, L.wt.begin() + k + m);
                    wt.resize((wt.size() - runs.back().w + kRunPad - 1) / kRunPad * kRunPad + runs.back().w, 0.0f);
                    k += m;
                }
                G.end[i] = (uint32_t)runs.size();
                G.before[i] = G.after[i] = G.end[i];
                if (best == 0xFFFFFFFFu) continue;
                G.before[i] = best;
                G.after[i] = best + 1;
                main[i] = runs[best];
                lo = std::min(lo, main[i].pix);
                hi = std::max(hi, main[i].pix + main[i].n);
            }
            // Outputs whose texels lie far apart (box filters, narrow ones) are summed
            // each by its own runs: a texel loaded once for four products, most of
            // weight 0, costs about as much as a contributor of a run, which loads
            // 16 at a time (2048^2, filter scale 0.1: 99 us, all in groups 103).
            if (hi && !single) {
                uint32_t own = 0;
                for (uint32_t i = 0; i < kGroup; i++) own += (main[i].n + 15) & ~15u;
                if (hi - (lo & ~3u) > own) {
                    for (uint32_t i = 0; i < kGroup; i++) G.before[i] = G.after[i] = G.end[i];
                    hi = 0;
                }
            }
            if (hi && !single) {
                G.pix = lo & ~3u;
                G.n = hi - G.pix;
                G.w = (uint32_t)wt.size();
                wt.resize(wt.size() + (size_t)kGroup * ((G.n + 7) & ~7u), 0.0f);
                for (uint32_t i = 0; i < kGroup; i++)
                    for (uint32_t k = 0; k < main[i].n; k++)
                        wt[G.w + kGroup * (size_t)(main[i].pix - G.pix + k) + i] = wt[main[i].w + k];
            }
            // the runs on one side of the main ones, where each is at most one
            // texel repeated, the same for all outputs: the shorter ones with
            // weights 0 on the side away from the main runs
            auto repeats = [&](uint32_t* from, uint32_t* to, bool before, uint32_t& pix, uint32_t& cnt, uint32_t& at_w) {
                uint32_t n_max = 0, texel = 0;
                for (uint32_t i = 0; i < kGroup; i++) {
                    if (from[i] == to[i]) continue;
                    const Run& r = runs[from[i]];
                    if (to[i] - from[i] > 1 || r.step || (n_max && r.pix != texel)) return;
                    texel = r.pix;
                    n_max = std::max(n_max, r.n);
                }
                if (!n_max) return;
                n_max = (n_max + 3) & ~3u;
                pix = texel;
                cnt = n_max;
                at_w = (uint32_t)wt.size();
                wt.resize(wt.size() + (size_t)kGroup * n_max, 0.0f);
                for (uint32_t i = 0; i < kGroup; i++) {
                    if (from[i] == to[i]) continue;
                    const Run r = runs[from[i]];
                    for (uint32_t k = 0; k < r.n; k++)
                        wt[at_w + kGroup * (size_t)(before ? n_max - r.n + k : k) + i] = wt[r.w + k];
                    if (before) from[i] = to[i];
                    else to[i] = from[i];
                }
            };
            if (hi && !single) {
                repeats(G.run, G.before, true, G.pre_pix, G.pre_n, G.pre_w);
                repeats(G.after, G.end, false, G.post_pix, G.post_n, G.post_w);
            }
            groups.push_back(G);
        }
        return at;
    };
    // deepest level first in both launches
    for (uint32_t i = 0; i < nl; i++) {
        const crn2mip::Level& v = lv[nl - 1 - i];
        const uint32_t level = nl - i;  // 1-based chain index
        Pass1Level& a = p1[i];
        Pass2Level& b = p2[i];
        const crn2mip::List& first = v.xfirst ? v.lx : v.ly;
        const crn2mip::List& second = v.xfirst ? v.ly : v.lx;
        a.lines = v.xfirst ? height : width;
        a.s = v.xfirst ? width : height;
        a.d = v.xfirst ? v.width : v.height;
        a.layout = v.xfirst ? 0 : 1;
        (v.xfirst ? need_lx : need_ly) = true;
        a.nlb = (a.lines + 63) / 64;
        const uint32_t list = first.ops() / a.d;
        a.single = list >= kLongList ||
                   (list >= kFewList && nc * a.nlb * a.d <= kFewWaves && one_piece(first)) ? 1 : 0;
        a.per = list >= kMidList ? 1 : kGroupsPerWave;
        a.runs = a.single ? a.d : ((a.d + kGroup - 1) / kGroup + a.per - 1) / a.per;
        a.unit0 = units;
        units += nc * a.nlb * a.runs;
        a.list = add_list(first, a.single);
        a.inter = inter_floats;
        inter_floats += ((uint64_t)nc * a.lines * a.d + 3) & ~3ull;   // (16-byte stores)
        b.lines = a.lines;
        b.d = a.d;
        b.d2 = v.xfirst ? v.height : v.width;
        b.nxb = (b.d + 63) / 64;
        b.block0 = blocks;
        const uint32_t list2 = second.ops() / b.d2;
        b.single = list2 >= kLongList2 ||
                   (list2 >= kFewList2 && b.d2 * b.nxb <= kFewBlocks2 && one_piece(second)) ? 1 : 0;
        blocks += (b.single ? b.d2 : (b.d2 + kGroup - 1) / kGroup) * b.nxb;
        b.list = add_list(second, b.single);
        b.inter = a.inter;
        b.out = p->level_ofs[level] / 4;
        b.os_lane = v.xfirst ? 1 : v.width;
        b.os_o = v.xfirst ? v.width : 1;
    }
    p->units1 = units;
    p->blocks2 = blocks;
    float s2l[256];
    std::vector<uint8_t> l2s(8192);
    crn2mip::gamma_tables(params->source_gamma, s2l, l2s.data());
    // one device buffer: level descriptors, lists, gamma tables
    size_t at = 0;
    const size_t o_p1 = at;
    at = align_up(at + nl * sizeof(Pass1Level), 256);
    const size_t o_p2 = at;
    at = align_up(at + nl * sizeof(Pass2Level), 256);
    const size_t o_groups = at;
    at = align_up(at + groups.size() * sizeof(Group), 256);
    const size_t o_runs = at;
    at = align_up(at + runs.size() * sizeof(Run), 256);
    const size_t o_wt = at;
    at = align_up(at + wt.size() * 4 + 4 * 3 * kChunk, 256);  // chunks read fewer than 3 * kChunk weights past a run
    const size_t o_s2l = at;
    at = align_up(at + sizeof(s2l), 256);
    const size_t o_l2s = at;
    at = align_up(at + l2s.size(), 256);
    std::vector<uint8_t> host(at, 0);
    std::memcpy(host.data() + o_p1, p1.data(), nl * sizeof(Pass1Level));
    std::memcpy(host.data() + o_p2, p2.data(), nl * sizeof(Pass2Level));
    std::memcpy(host.data() + o_groups, groups.data(), groups.size() * sizeof(Group));
    std::memcpy(host.data() + o_runs, runs.data(), runs.size() * sizeof(Run));
    std::memcpy(host.data() + o_wt, wt.data(), wt.size() * 4);
    std::memcpy(host.data() + o_s2l, s2l, sizeof(s2l));
    std::memcpy(host.data() + o_l2s, l2s.data(), l2s.size());
    const uint64_t plane_x = align_up((uint64_t)nc * ((width + 3) / 4) * height * 4, 256);  // bytes
    const uint64_t plane_y = align_up((uint64_t)nc * ((height + 3) / 4) * width * 4, 256);
    const uint64_t scratch_bytes = (need_lx ? plane_x : 0) + (need_ly ? plane_y : 0) + inter_floats * sizeof(float);
    int rc = CRN2_OK;
    if (!hip_ok(hipMalloc(&p->tables, at)) || !hip_ok(hipMalloc(&p->scratch, scratch_bytes)))
        rc = CRN2_ENOMEM;
    else if (!hip_ok(hipMemcpy(p->tables, host.data(), at, hipMemcpyHostToDevice)))
        rc = CRN2_EHIP;
    if (rc != CRN2_OK) {
        plan_free(p);
        return rc;
    }
    const uint8_t* d = static_cast<const uint8_t*>(p->tables);
    p->t.p1 = reinterpret_cast<const Pass1Level*>(d + o_p1);
    p->t.p2 = reinterpret_cast<const Pass2Level*>(d + o_p2);
    p->t.groups = reinterpret_cast<const Group*>(d + o_groups);
    p->t.runs = reinterpret_cast<const Run*>(d + o_runs);
    p->t.wt = reinterpret_cast<const float*>(d + o_wt);
    p->t.s2l = reinterpret_cast<const float*>(d + o_s2l);
    p->t.l2s = d + o_l2s;
    uint8_t* f = static_cast<uint8_t*>(p->scratch);
    if (need_lx) { p->lx = reinterpret_cast<uint32_t*>(f); f += plane_x; }
    if (need_ly) { p->ly = reinterpret_cast<uint32_t*>(f); f += plane_y; }
    p->inter = reinterpret_cast<float*>(f);
    *out = p;
    return CRN2_OK;
}

int crn2_mip_plan_info(const crn2_mip_plan* p, uint32_t* levels, uint64_t* chain_bytes, uint64_t* level_offsets,
                       uint8_t* y_first)
{
    if (!plan_ok(p)) return CRN2_EINVAL;
    if (levels) *levels = p->levels;
    if (chain_bytes) *chain_bytes = p->chain_bytes;
    if (level_offsets) std::memcpy(level_offsets, p->level_ofs.data(), p->levels * sizeof(uint64_t));
    if (y_first) std::memcpy(y_first, p->y_first.data(), p->levels);
    return CRN2_OK;
}

int crn2_mip_plan_run(crn2_mip_plan* p, const void* rgba, void* out, uint64_t out_size, void* stream)
{
    if (!plan_ok(p) || !rgba || !out || out_size < p->chain_bytes) return CRN2_EINVAL;
    if ((reinterpret_cast<uintptr_t>(rgba) | reinterpret_cast<uintptr_t>(out)) & 3) return CRN2_EINVAL;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const uint64_t l0 = (uint64_t)p->width * p->height * 4;
    if (p->levels == 1) {
        if (out != rgba && !hip_ok(hipMemcpyAsync(out, rgba, l0, hipMemcpyDeviceToDevice, st))) return CRN2_EHIP;
        return CRN2_OK;
    }
    const int srgb = (p->params.flags & CRN2_MIP_SRGB) != 0;
    if (p->prof) (void)hipEventRecord(p->ev[0], st);
    hipLaunchKernelGGL(mip_planes_kernel, dim3((p->width + 31) / 32, (p->height + 31) / 32), dim3(256), 0, st,
                       static_cast<const uint32_t*>(rgba), p->width, p->height, p->lx, p->ly, p->ncomp,
                       out != rgba ? static_cast<uint32_t*>(out) : nullptr);
    if (p->prof) (void)hipEventRecord(p->ev[1], st);
    hipLaunchKernelGGL(mip_pass1_kernel, dim3((p->units1 + 3) / 4), dim3(256), 0, st, p->t, p->lx, p->ly, p->inter,
                       p->levels - 1, p->units1, p->ncomp, srgb);
    if (p->prof) (void)hipEventRecord(p->ev[2], st);
    hipLaunchKernelGGL(mip_pass2_kernel, dim3(p->blocks2), dim3(256), 0, st, p->t, p->inter,
                       static_cast<uint32_t*>(out), p->levels - 1, p->ncomp, srgb,
                       (p->params.flags & CRN2_MIP_RENORMALIZE) ? 1 : 0);
    if (p->prof) {
        (void)hipEventRecord(p->ev[3], st);
        if (hipEventSynchronize(p->ev[3]) == hipSuccess) {
            for (int s = 0; s < 3; s++) {
                float ms = 0;
                if (hipEventElapsedTime(&ms, p->ev[s], p->ev[s + 1]) == hipSuccess) p->ms[s] += ms;
            }
            p->runs++;
        }
    }
    return hip_ok(hipGetLastError()) ? CRN2_OK : CRN2_EHIP;
}

int crn2_mip_plan_destroy(crn2_mip_plan* p)
{
    if (!plan_ok(p)) return CRN2_EINVAL;
    (void)hipDeviceSynchronize();
    plan_free(p);
    return CRN2_OK;
}

/* Stage timing of a plan's runs: on != 0 records HIP events around the three
 * launches of every run (and waits for them); ms[0..2] = planes, pass 1,
 * pass 2 totals since it was switched on. */
int crn2_mip_plan_profile(crn2_mip_plan* p, int on, double* ms, uint64_t* runs)
{
    if (!plan_ok(p)) return CRN2_EINVAL;
    if (on && !p->prof) {
        for (hipEvent_t& e : p->ev)
            if (!e && hipEventCreate(&e) != hipSuccess) return CRN2_EHIP;
        p->ms[0] = p->ms[1] = p->ms[2] = 0;
        p->runs = 0;
    }
    p->prof = on != 0;
    if (ms) std::memcpy(ms, p->ms, sizeof(p->ms));
    if (runs) *runs = p->runs;
    return CRN2_OK;
}

int crn2_generate_mipmaps_device(const void* rgba, uint32_t width, uint32_t height, const crn2_mip_params* params,
                                 void* out, uint64_t out_size, void* stream)
{
    crn2_mip_plan* p = nullptr;
    int rc = crn2_mip_plan_create(width, height, params, &p);
    if (rc != CRN2_OK) return rc;
    rc = crn2_mip_plan_run(p, rgba, out, out_size, stream);
    if (hipStreamSynchronize(static_cast<hipStream_t>(stream)) != hipSuccess && rc == CRN2_OK) rc = CRN2_EHIP;
    plan_free(p);
    return rc;
}

int crn2_generate_mipmaps(const void* rgba, uint32_t width, uint32_t height, const crn2_mip_params* params,
                          void* out, uint64_t out_size)
{
    if (!rgba || !out) return CRN2_EINVAL;
    crn2_mip_plan* p = nullptr;
    int rc = crn2_mip_plan_create(width, height, params, &p);
    if (rc != CRN2_OK) return rc;
    if (out_size < p->chain_bytes) {
        plan_free(p);
        return CRN2_EINVAL;
    }
    const uint64_t l0 = (uint64_t)width * height * 4;
    void *d_in = nullptr, *d_out = nullptr;
    if (!hip_ok(hipMalloc(&d_in, l0)) || !hip_ok(hipMalloc(&d_out, p->chain_bytes))) rc = CRN2_ENOMEM;
    if (rc == CRN2_OK && !hip_ok(hipMemcpy(d_in, rgba, l0, hipMemcpyHostToDevice))) rc = CRN2_EHIP;
    if (rc == CRN2_OK) rc = crn2_mip_plan_run(p, d_in, d_out, p->chain_bytes, nullptr);
    if (rc == CRN2_OK && !hip_ok(hipMemcpy(out, d_out, p->chain_bytes, hipMemcpyDeviceToHost))) rc = CRN2_EHIP;
    if (d_in) (void)hipFree(d_in);
    if (d_out) (void)hipFree(d_out);
    plan_free(p);
    return rc;
}

}  // extern "C"
