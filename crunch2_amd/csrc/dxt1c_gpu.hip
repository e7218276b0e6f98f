// dxt1c_gpu.hip -- DXT1 endpoint search for pixel clusters of any size, one
// workgroup per cluster (the dxt_hc endpoint-cluster case).
//
// Reference: dxt1_endpoint_optimizer::compute (crnlib/crn_dxt1.cpp:2081-2246)
// at uber quality.  Without 3-colour blocks (the path dxt_hc uses for its
// endpoint clusters, determine_color_endpoint_codebook_task,
// crn_dxt_hc.cpp:663-754) the hc evaluators (evaluate_solution_hc_*,
// compute_selectors_hc, crn_dxt1.cpp:1759-1869) judge every candidate; with
// them (qdxt1's clusters, crn_qdxt1.cpp:616-626) evaluate_solution_uber
// (:1370-1592) scores both block types, and the solid-block tries, the
// one-colour shortcut and return_solution take their 3-colour branches
// (:119, :143, :2220, :263-365).  Unique colours (first-appearance order), the error planes,
// PCA, the probe sweeps, refine_solution, try_median4,
// optimize_endpoint_comps and the special cases follow crn_dxt1.cpp as in the
// per-block kernel (dxt1_gpu.hip).
//
// Layout: one workgroup per cluster; the cluster's unique colours, weights,
// selectors and per-channel error tables live in LDS.  Wave 0 runs the search
// (its state is wave-uniform); the other waves wait for batches of candidates
// and score their share.
//
// Scoring is a contraction and runs on the matrix cores.  The distance of
// colour c to palette entry p is |c|^2 - 2 c.p + |p|^2 under the channel
// weights; |c|^2 is the same for every candidate and summed once, and the
// rest is a product of [r, g, g, g, b, 1, 1, 1] with
// [-16 pr, -32 pg, -16 pg, -2 pg, -2 pb, K2, K1, K0] (K = |p|^2 in three 8-bit
// limbs): every factor is an integer of at most 8 significant bits times a
// power of two, exact in bfloat16, and every partial sum an integer below
// 2^24, exact in float32.  One v_mfma_f32_32x32x16_bf16 gives 32 colours x 8
// palettes x 4 entries; a lane takes the minimum of its four entries and adds
// weight x minimum in double (integers below 2^53 for clusters of up to 2^30
// texels).  So a candidate's error is the exact integer, whatever the order.
//
// Candidates are scored in batches and taken in the reference's order:
// evaluate_solution (:1312-1340) keeps a candidate when its error-plane bound
// and then its error are below the best at its turn.  A batch holds candidates
// whose bound is below the best at the gather; the ordered scan over
// max(bound, error) then takes what the reference takes.  Lists that read the
// current best (the lattice moves, optimize_endpoint_comps) are gathered again
// after each candidate taken.
//
// Float sums (means, covariance, 4-means) keep the reference's sequential
// order: a chunk of 64 colours' terms is computed by all lanes into LDS, then
// one lane per sum adds them one after another.
//
// What bounds it: the chain of lists of the largest clusters, and for the many
// small ones the vector work around the matrix instructions.  Scored by 64
// lanes with 60 integer operations per colour and candidate, one candidate at a
// time on one wave, the classes took 91 / 25 / 17 / 8 ms side by side on the
// 2048^2 DXT1 chain at quality 128 (2,415 clusters, 1,388 of 2,049 to 4,096
// texels); now 3.2 ms for the longest class.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <mutex>
#include <type_traits>

#include "crn2_internal.h"

namespace {

// Largest cluster kept in LDS: 4096 unique colours.  The kernel comes in four
// sizes by texel count (512, 1024, 2048 and 4096), so that small clusters, the
// common case, share a CU, and a fifth for more texels of at most 4096 colours.
constexpr uint32_t kMaxU = 4096;

__device__ __constant__ int16_t c_uber_probe[15] = {0, 1, 2, 3, 5, 7, 9, 10, 13, 15, 19, 27, 43, 59, 91};
__device__ __constant__ int8_t c_adj[26][3] = {
    {-1, -1, -1}, {0, -1, -1}, {1, -1, -1}, {-1, 0, -1}, {0, 0, -1}, {1, 0, -1}, {-1, 1, -1}, {0, 1, -1},
    {1, 1, -1}, {-1, -1, 0}, {0, -1, 0}, {1, -1, 0}, {-1, 0, 0}, {1, 0, 0}, {-1, 1, 0}, {0, 1, 0},
    {1, 1, 0}, {-1, -1, 1}, {0, -1, 1}, {1, -1, 1}, {-1, 0, 1}, {0, 0, 1}, {1, 0, 1}, {-1, 1, 1},
    {0, 1, 1}, {1, 1, 1}};
__device__ uint8_t g_c_om5[256][2], g_c_om6[256][2], g_c_om5_3[256][2], g_c_om6_3[256][2];

// Candidates scored together: 32, or 64 (one per lane) where eight waves share them.
template <uint32_t W>
constexpr uint32_t kBatchOf = W >= 8 ? 64 : 32;
constexpr uint32_t kMaxBatch = 64;
struct Pal {
    int r[4], g[4], b[4];
};

constexpr uint32_t kRow = 68;       // floats per staged sum: 64 terms, the rows on different LDS banks
constexpr uint32_t kRowD = 66;      // doubles per staged sum

// Per-channel error of one selector class as a function of the class's value
// p: W p^2 - WP2 p + WPP (the reference's compute_endpoint_component_errors
// tables, crn_dxt1.cpp:369-418, evaluated where they are read).
struct QErr {
    uint64_t W[4], WP2[4], WPP[4];
    __device__ inline uint64_t at(int sl, uint64_t p) const { return W[sl] * p * p - WP2[sl] * p + WPP[sl]; }
};

// The search's working set in LDS.
struct SearchLds {
    uint32_t cmd;                // candidates to score | alternate rounding << 8; 0: the search has ended
    Pal end_pal;                 // the result, for the texels' selectors
    uint32_t end_alpha, end_inv, end_enforce, end_enforced;
    uint32_t cand[kMaxBatch];       // low | high << 16
    uint32_t cidx[kMaxBatch];       // the candidate's place in its list
    uint64_t bnd[kMaxBatch];        // its error-plane bound
    uint64_t err[2 * kMaxBatch];    // palette sums: one per candidate, or four-colour and three-colour
    union {
        float f[6][kRow];
        double d[6][kRowD];
    } stage;                     // terms of the sequential float sums
    uint32_t list[2][64];        // the list's colours (sweep ends, combinatorial set, means)
    QErr q;                      // optimize_endpoint_comps
    uint64_t brem[4], qbest;
    int fixed[2][3];             // refine_solution's rounded endpoints / the components not being optimised
};

// Error planes (count, sum, sum of squares per quantised value) are dead once
// the per-value bounds are made; the search's working set takes their space.
union PlanesOrSearch {
    unsigned long long pl[3][64][3];
    SearchLds q;
};

struct Bounds {
    uint64_t rlo[32], rhi[32], glo[64], ghi[64], blo[32], bhi[32];
    uint64_t base;       // sum of weight x |colour|^2
};

// Store of the size classes whose texel count never exceeds the colour
// capacity.  The unique-colour pass sorts (colour, texel index) pairs in a
// buffer that overlays the search's tables (dead until the search starts):
// 13, 15, 24 and 49 KiB.
template <uint32_t MaxU>
struct LdsS {
    static constexpr uint32_t kSearch = MaxU + sizeof(PlanesOrSearch) + sizeof(Bounds);
    static constexpr uint32_t kSort = 6 * MaxU;   // u32 colours + u16 texel indices
    uint32_t col[MaxU];      // r | g << 8 | b << 16
    uint16_t w[MaxU];
    uint32_t fbits[MaxU / 32];           // first texel of each colour
    uint32_t fbase[MaxU / 32];           // first texels before each word of fbits
    uint32_t nuniq, nopaque;
    int scan[8];                         // per wave
    uint8_t sel[MaxU];                   // from here on: the sort buffers' space
    PlanesOrSearch u;
    Bounds b;
    uint8_t pad[kSort > kSearch ? kSort - kSearch : 4];
};

// Store of clusters of more texels but at most MaxU distinct colours: a colour
// hash with the first texel and the count of each colour, whose space the
// search takes over (128 KiB).
template <uint32_t MaxU>
struct LdsT {
    static constexpr uint32_t kCapH = 2 * MaxU;    // colour hash slots (power of two)
    uint32_t col[MaxU];          // during the unique-colour pass: first texels ...
    uint32_t w[MaxU];            // ... and hash slots (u16) being sorted
    uint32_t nuniq, nopaque, nsort, pad;
    union {
        struct {
            uint32_t hkey[kCapH];        // colour | 0xFF000000, 0 = empty
            uint32_t hval[kCapH];        // first texel
            uint32_t hcnt[kCapH];
        };
        struct {
            uint8_t sel[MaxU];
            PlanesOrSearch u;
            Bounds b;
        };
    };
};

// A colour store tagged with the evaluator: kUber -- evaluate_solution_uber
// with both block types (3-colour blocks allowed); else the hc evaluators.
template <class Base, bool U>
struct LdsU : Base {
    using Base::Base;
    static constexpr bool kUber = U;
};

struct Best {
    uint32_t lo, hi;
    uint64_t err;
    int alt, enforce, enforced, alpha;
};

struct St {
    int perceptual;
    int have_alpha;      // DXT1A: texels below the alpha threshold are transparent (3-colour blocks only)
    uint32_t nu, total_w;
    uint64_t base;       // sum of weight x |colour|^2
    float mean[3], meanw[3], pw[3], axis[3];
    Best best;
    bool sel_valid;      // L.sel holds the selectors of the current best solution
    bool sel_nonempty;   // selectors have been computed at least once (results::m_selectors not empty)
};

__device__ inline uint32_t lane_id() { return threadIdx.x & 63u; }

__device__ inline uint32_t uni(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }
__device__ inline uint64_t uni64(uint64_t v) { return (uint64_t)uni((uint32_t)v) | ((uint64_t)uni((uint32_t)(v >> 32)) << 32); }
__device__ inline bool unib(bool v) { return uni(v ? 1u : 0u) != 0; }
__device__ inline float unif(float v) { return __builtin_bit_cast(float, uni(__builtin_bit_cast(uint32_t, v))); }
__device__ inline uint32_t lane_u32(uint32_t v, uint32_t l) { return (uint32_t)__builtin_amdgcn_readlane((int)v, (int)l); }
__device__ inline uint64_t lane_u64(uint64_t v, uint32_t l)
{
    return (uint64_t)lane_u32((uint32_t)v, l) | ((uint64_t)lane_u32((uint32_t)(v >> 32), l) << 32);
}
__device__ inline float lane_f32(float v, uint32_t l) { return __builtin_bit_cast(float, lane_u32(__builtin_bit_cast(uint32_t, v), l)); }
__device__ inline double lane_f64(double v, uint32_t l) { return __builtin_bit_cast(double, lane_u64(__builtin_bit_cast(uint64_t, v), l)); }

template <int Ctrl, int RowMask>
__device__ inline uint64_t dpp_add(uint64_t v)
{
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)v, Ctrl, RowMask, 0xF, false);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(v >> 32), Ctrl, RowMask, 0xF, false);
    return v + ((uint64_t)lo | ((uint64_t)hi << 32));
}

// Sums over each half of the wave, in lanes 31 and 63.
__device__ inline uint64_t half_sums(uint64_t v)
{
    v = dpp_add<0x111, 0xF>(v);   // row_shr 1, 2, 4, 8
    v = dpp_add<0x112, 0xF>(v);
    v = dpp_add<0x114, 0xF>(v);
    v = dpp_add<0x118, 0xF>(v);
    return dpp_add<0x142, 0xA>(v);   // row_bcast15 into rows 1 and 3
}

__device__ inline uint64_t wave_sum(uint64_t v)
{
    return lane_u64(dpp_add<0x143, 0xC>(half_sums(v)), 63);   // row_bcast31 into rows 2 and 3
}

__device__ inline uint32_t hash32(uint32_t x)
{
    x ^= x >> 16;
    x *= 0x7FEB352Du;
    x ^= x >> 15;
    x *= 0x846CA68Bu;
    x ^= x >> 16;
    return x;
}

__device__ inline void unpack565(uint32_t p, int scaled, int& r, int& g, int& b)
{
    uint32_t bb = p & 31u, gg = (p >> 5) & 63u, rr = (p >> 11) & 31u;
    if (scaled) {
        bb = (bb << 3) | (bb >> 2);
        gg = (gg << 2) | (gg >> 4);
        rr = (rr << 3) | (rr >> 2);
    }
    r = (int)rr;
    g = (int)gg;
    b = (int)bb;
}

__device__ inline uint32_t pack565(int r, int g, int b, int scaled)
{
    uint32_t R = (uint32_t)min(max(r, 0), 255), G = (uint32_t)min(max(g, 0), 255), B = (uint32_t)min(max(b, 0), 255);
    if (scaled) {
        R = (R * 31u + 127u) / 255u;
        G = (G * 63u + 127u) / 255u;
        B = (B * 31u + 127u) / 255u;
    }
    R = min(R, 31u);
    G = min(G, 63u);
    B = min(B, 31u);
    return B | (G << 5) | (R << 11);
}

__device__ inline void canon(uint32_t& lo, uint32_t& hi)
{
    const uint32_t a = max(lo, hi), b = min(lo, hi);
    lo = a;
    hi = b;
}

__device__ inline uint32_t cdist(int perceptual, uint32_t px, int r, int g, int b)
{
    const int dr = (int)(px & 255u) - r, dg = (int)((px >> 8) & 255u) - g, db = (int)((px >> 16) & 255u) - b;
    return perceptual ? (uint32_t)(dr * dr * 8 + dg * dg * 25 + db * db) : (uint32_t)(dr * dr + dg * dg + db * db);
}

__device__ inline Pal palette4(uint32_t lo, uint32_t hi, int alt)
{
    Pal p;
    unpack565(lo, 1, p.r[0], p.g[0], p.b[0]);
    unpack565(hi, 1, p.r[1], p.g[1], p.b[1]);
    p.r[2] = (p.r[0] * 2 + p.r[1] + alt) / 3;
    p.g[2] = (p.g[0] * 2 + p.g[1] + alt) / 3;
    p.b[2] = (p.b[0] * 2 + p.b[1] + alt) / 3;
    p.r[3] = (p.r[1] * 2 + p.r[0] + alt) / 3;
    p.g[3] = (p.g[1] * 2 + p.g[0] + alt) / 3;
    p.b[3] = (p.b[1] * 2 + p.b[0] + alt) / 3;
    return p;
}

// get_block_colors3 with the alternate rounding (crn_dxt1.cpp:1432-1440)
__device__ inline Pal palette3(uint32_t lo, uint32_t hi, int alt)
{
    Pal p;
    unpack565(lo, 1, p.r[0], p.g[0], p.b[0]);
    unpack565(hi, 1, p.r[1], p.g[1], p.b[1]);
    p.r[2] = (p.r[0] + p.r[1] + alt) >> 1;
    p.g[2] = (p.g[0] + p.g[1] + alt) >> 1;
    p.b[2] = (p.b[0] + p.b[1] + alt) >> 1;
    p.r[3] = p.g[3] = p.b[3] = 0;
    return p;
}

// ------------------------------------------------------------- scoring
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// Two integers of at most 8 significant bits (times a power of two) as bfloat16.
__device__ inline uint32_t bf2(float a, float b)
{
    return (__float_as_uint(a) >> 16) | (__float_as_uint(b) & 0xFFFF0000u);
}

// Row `row` (palette row / 4, entry row % 4) of the palettes' operand.
template <bool Uber>
__device__ inline bf16x8 palette_row(const SearchLds& q, uint32_t pal, uint32_t entry, uint32_t n, int alt,
                                     int perceptual)
{
    const uint32_t cand = Uber ? pal >> 1 : pal;
    const bool three = Uber && (pal & 1u);
    const uint32_t c = q.cand[min(cand, n - 1)];
    int a[3], b[3], p[3];
    unpack565(c & 0xFFFFu, 1, a[0], a[1], a[2]);
    unpack565(c >> 16, 1, b[0], b[1], b[2]);
    for (int k = 0; k < 3; k++) {
        const int far = entry == 2 ? a[k] : b[k], near = entry == 2 ? b[k] : a[k];
        const int mid = three ? (a[k] + b[k] + alt) >> 1 : (far * 2 + near + alt) / 3;
        p[k] = entry == 0 ? a[k] : entry == 1 ? b[k] : mid;
    }
    const float r = (float)p[0], g = (float)p[1], bl = (float)p[2];
    const uint32_t K = perceptual ? (uint32_t)(8 * p[0] * p[0] + 25 * p[1] * p[1] + p[2] * p[2])
                                  : (uint32_t)(p[0] * p[0] + p[1] * p[1] + p[2] * p[2]);
    u32x4 v;
    v.x = perceptual ? bf2(-16.0f * r, -32.0f * g) : bf2(-2.0f * r, -2.0f * g);
    v.y = perceptual ? bf2(-16.0f * g, -2.0f * g) : 0u;
    v.z = bf2(-2.0f * bl, (float)(K & 0xFF0000u));
    v.w = bf2((float)(K & 0xFF00u), (float)(K & 0xFFu));
    return __builtin_bit_cast(bf16x8, v);
}

// Sums of weight x smallest distance for the batch's palettes, groups of
// eight dealt to the W waves; Lds::kUber scores two palettes per candidate.
template <class Lds, uint32_t W>
__device__ void score(Lds& L, SearchLds& q, uint32_t nu, uint64_t base, int perceptual, uint32_t n, int alt,
                      uint32_t wave)
{
    constexpr uint32_t kPer = Lds::kUber ? 2 : 1;
    constexpr uint32_t kShare = kBatchOf<W> * kPer / 8 / W;
    constexpr uint32_t G = kShare >= 2 ? 2 : 1;   // groups that share a pass over the colours
    const uint32_t groups = (n * kPer + 7) / 8;
    const uint32_t col = lane_id() & 31u, half = lane_id() >> 5;
    for (uint32_t g0 = wave * G; g0 < groups; g0 += W * G) {
        bf16x8 A[G];
        double acc[G][4];
#pragma unroll
        for (uint32_t t = 0; t < G; t++) {
            A[t] = palette_row<Lds::kUber>(q, 8 * (g0 + t) + (col >> 2), col & 3u, n, alt, perceptual);
            if (half) A[t] = __builtin_bit_cast(bf16x8, u32x4{0u, 0u, 0u, 0u});
#pragma unroll
            for (int j = 0; j < 4; j++) acc[t][j] = 0.0;
        }
        for (uint32_t i0 = 0; i0 < nu; i0 += 32) {
            const uint32_t i = min(i0 + col, nu - 1);
            const uint32_t px = L.col[i];
            const double w = i0 + col < nu ? (double)L.w[i] : 0.0;
            const float r = (float)(px & 255u), g = (float)((px >> 8) & 255u), b = (float)((px >> 16) & 255u);
            const u32x4 v = {bf2(r, g), bf2(g, g), bf2(b, 1.0f), bf2(1.0f, 1.0f)};
            const bf16x8 B = __builtin_bit_cast(bf16x8, v);
#pragma unroll
            for (uint32_t t = 0; t < G; t++) {
                const f32x16 zero = {0};
                const f32x16 d = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A[t], B, zero, 0, 0, 0);
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const float m = fminf(fminf(d[4 * j], d[4 * j + 1]), fminf(d[4 * j + 2], d[4 * j + 3]));
                    acc[t][j] = __builtin_fma(w, (double)m, acc[t][j]);
                }
            }
        }
#pragma unroll
        for (uint32_t t = 0; t < G; t++)
#pragma unroll
            for (uint32_t j = 0; j < 4; j++) {
                const uint64_t e = base + half_sums((uint64_t)(int64_t)acc[t][j]);
                const uint32_t pal = 8 * (g0 + t) + 2 * j + half;
                if (col == 31u && pal < kPer * n) q.err[pal] = e;
            }
    }
}

// The waves beside wave 0: score their share of each batch until the search ends.
template <class Lds, uint32_t W>
__device__ void score_loop(Lds& L, uint32_t nu, uint64_t base, int perceptual, uint32_t wave)
{
    SearchLds& q = L.u.q;
    for (;;) {
        __syncthreads();
        const uint32_t cmd = uni(q.cmd);
        if (!cmd) return;
        score<Lds, W>(L, q, nu, base, perceptual, cmd & 0xFFu, (int)(cmd >> 8), wave);
        __syncthreads();
    }
}

// evaluate_solution's plane lower bound (crn_dxt1.cpp:1312-1340)
__device__ inline uint64_t plane_bound(const Bounds& B, uint32_t lo, uint32_t hi)
{
    int ar, ag, ab, br, bg, bb;
    unpack565(lo, 0, ar, ag, ab);
    unpack565(hi, 0, br, bg, bb);
    return B.rlo[min(ar, br)] + B.rhi[max(ar, br)] + B.glo[min(ag, bg)] + B.ghi[max(ag, bg)] + B.blo[min(ab, bb)] +
           B.bhi[max(ab, bb)];
}

__device__ inline int clampi(int v, int hi) { return v < 0 ? 0 : (v > hi ? hi : v); }

// ------------------------------------------------------------ candidate lists
enum ListKind : uint32_t {
    kListPair,      // list[0][0..3]: the six pairs of four colours, canonical order
    kListRefine,    // refine_solution level 1: 27 moves of either endpoint
    kListSweep,     // list[0] x list[1], canonical order; index low * 32 + high
    kListAdj0,      // 26 neighbours of the low / high end (the other end is the current best's)
    kListAdj1,
    kListAxis0,     // +-2 on each component of the low / high end
    kListAxis1,
    kListSolid,     // the average colour (list[0][0]) and each colour as a solid block
    kListComb,      // list[0][i], list[0][j], i < j < fixed[0][0]; index i * 64 + j
    kListComp0,     // optimize_endpoint_comps, one component: c0 * 64 + c1
    kListComp1,
    kListComp2,
};

__device__ inline uint32_t expand_comp(int comp, uint32_t c)
{
    return comp == 1 ? (((c << 2) | (c >> 4)) & 0xFF) : (((c << 3) | (c >> 2)) & 0xFF);
}

// Candidate `i` of the list; false: the list has none there.
template <class Lds>
__device__ inline bool list_candidate(const St& s, const Lds& L, const SearchLds& q, uint32_t kind, uint32_t i,
                                      uint32_t from, uint32_t& lo, uint32_t& hi)
{
    switch (kind) {
    case kListPair: {
        const uint32_t a = i < 3 ? 0 : i < 5 ? 1 : 2, b = i < 3 ? i + 1 : i < 5 ? i - 1 : 3;
        lo = q.list[0][a];
        hi = q.list[0][b];
        canon(lo, hi);
        return true;
    }
    case kListRefine: {
        const uint32_t e = i >= 27 ? 1 : 0, m = i - 27 * e;
        uint32_t c[2];
        for (uint32_t k = 0; k < 2; k++) {
            const int d = e == k ? 1 : 0;
            c[k] = pack565(clampi(q.fixed[k][0] + d * ((int)(m / 9) - 1), 31),
                           clampi(q.fixed[k][1] + d * ((int)(m / 3 % 3) - 1), 63),
                           clampi(q.fixed[k][2] + d * ((int)(m % 3) - 1), 31), 0);
        }
        lo = c[0];
        hi = c[1];
        canon(lo, hi);
        return true;
    }
    case kListSweep:
        if ((i & 31u) >= (uint32_t)q.fixed[0][0]) return false;
        lo = q.list[0][i >> 5];
        hi = q.list[1][i & 31u];
        canon(lo, hi);
        return true;
    case kListAdj0:
    case kListAdj1:
    case kListAxis0:
    case kListAxis1: {
        int c[3];
        unpack565(from, 0, c[0], c[1], c[2]);
        if (kind <= kListAdj1) {
            for (int k = 0; k < 3; k++) c[k] += c_adj[min(i, 25u)][k];
        } else {
            const int d = (i & 1u) ? 2 : -2;
            for (uint32_t k = 0; k < 3; k++) c[k] += i >> 1 == k ? d : 0;
        }
        if (c[0] < 0 || c[0] > 31 || c[1] < 0 || c[1] > 63 || c[2] < 0 || c[2] > 31) return false;
        lo = pack565(c[0], c[1], c[2], 0);
        hi = kind == kListAdj0 || kind == kListAxis0 ? s.best.hi : s.best.lo;
        canon(lo, hi);
        return true;
    }
    case kListSolid: {
        const uint32_t k = Lds::kUber ? i >> 1 : i;
        const uint32_t avg = q.list[0][0];
        const uint32_t c = k ? L.col[min(k, s.nu) - 1] : avg;
        if (k && c == avg) return false;
        const uint32_t r = c & 255u, g = (c >> 8) & 255u, b = (c >> 16) & 255u;
        const uint8_t(*o5)[2] = Lds::kUber && (i & 1u) ? g_c_om5_3 : g_c_om5;
        const uint8_t(*o6)[2] = Lds::kUber && (i & 1u) ? g_c_om6_3 : g_c_om6;
        lo = ((uint32_t)o5[r][0] << 11) | ((uint32_t)o6[g][0] << 5) | o5[b][0];
        hi = ((uint32_t)o5[r][1] << 11) | ((uint32_t)o6[g][1] << 5) | o5[b][1];
        return true;
    }
    case kListComb:
        if ((i & 63u) <= i >> 6 || (i & 63u) >= (uint32_t)q.fixed[0][0]) return false;
        lo = q.list[0][i >> 6];
        hi = q.list[0][i & 63u];
        return true;
    default: {
        // optimize_endpoint_comps (crn_dxt1.cpp:420-486), one component
        const int comp = (int)(kind - kListComp0);
        const uint32_t c0 = i >> 6, c1 = i & 63u, lim = comp == 1 ? 64 : 32;
        if (c1 >= lim) return false;
        const uint32_t p0 = expand_comp(comp, c0), p1 = expand_comp(comp, c1);
        const uint64_t best = q.qbest, e0 = q.q.at(0, p0);
        if (e0 + q.brem[1] >= best) return false;
        uint64_t e = e0 + q.q.at(1, p1);
        if (e + q.brem[2] >= best) return false;
        e += q.q.at(2, (p0 * 2 + p1) / 3);
        if (e + q.brem[3] >= best) return false;
        e += q.q.at(3, (p0 + p1 * 2) / 3);
        if (e >= best) return false;
        int a[3], b[3];
        for (int k = 0; k < 3; k++) {
            a[k] = k == comp ? (int)c0 : q.fixed[0][k];
            b[k] = k == comp ? (int)c1 : q.fixed[1][k];
        }
        lo = pack565(a[0], a[1], a[2], 0);
        hi = pack565(b[0], b[1], b[2], 0);
        return true;
    }
    }
}

// Tries the list's candidates [first, n) in order from `first`: gathers a
// batch, scores it, takes what the reference takes.  With `again`, returns at
// the first candidate taken (first: the place after it).  True: one was taken.
template <class Lds, uint32_t W>
__device__ bool try_list(St& s, Lds& L, uint32_t kind, uint32_t n, int alt, bool again, uint32_t from, uint32_t& first)
{
    constexpr uint32_t kBatch = kBatchOf<W>;
    SearchLds& q = L.u.q;
    const uint32_t lane = lane_id();
    bool took = false;
    while (first < n && s.best.err) {
        uint32_t cnt = 0, next = first;
        __builtin_amdgcn_wave_barrier();   // the last batch has been read
        while (next < n && cnt < kBatch) {
            const uint32_t i = next + lane;
            uint32_t lo = 0, hi = 0;
            bool ok = i < n && list_candidate(s, L, q, kind, i, from, lo, hi);
            uint64_t b = 0;
            if (ok) {
                b = plane_bound(L.b, lo, hi);
                ok = b < s.best.err;
            }
            const uint64_t mask = __ballot(ok);
            const uint32_t at = cnt + (uint32_t)__popcll(mask & ((1ull << lane) - 1ull));
            if (ok && at < kBatch) {
                q.cand[at] = lo | (hi << 16);
                q.cidx[at] = i;
                q.bnd[at] = b;
            }
            cnt += (uint32_t)__popcll(mask);
            next += 64;
        }
        if (!cnt) {
            first = n;
            break;
        }
        if (cnt > kBatch) cnt = kBatch;
        if (lane == 0) q.cmd = cnt | ((uint32_t)alt << 8);
        __builtin_amdgcn_wave_barrier();
        if (cnt == kBatch) next = uni(q.cidx[kBatch - 1]) + 1;
        if constexpr (W > 1) __syncthreads();
        score<Lds, W>(L, q, s.nu, s.base, s.perceptual, cnt, alt, 0);
        if constexpr (W > 1) __syncthreads();
        else __builtin_amdgcn_wave_barrier();
        // lane k: candidate k's error, block type and the larger of error and bound
        const uint32_t k = min(lane, cnt - 1);
        uint64_t e;
        uint32_t alpha = 0;
        if constexpr (Lds::kUber) {
            const uint64_t e4 = q.err[2 * k], e3 = q.err[2 * k + 1];
            alpha = s.have_alpha || e3 < e4 ? 1u : 0u;
            e = alpha ? e3 : e4;
        } else {
            e = q.err[k];
        }
        const uint64_t bk = q.bnd[k];
        const uint64_t m = e > bk ? e : bk;
        const uint32_t c = q.cand[k];
        uint64_t left = ~0ull;
        first = next;
        for (;;) {
            const uint64_t mask = __ballot(lane < cnt && m < s.best.err) & left;
            if (!mask) break;
            const uint32_t t = (uint32_t)__builtin_ctzll(mask);
            const uint32_t lh = lane_u32(c, t);
            s.best.lo = lh & 0xFFFFu;
            s.best.hi = lh >> 16;
            s.best.err = lane_u64(e, t);
            s.best.alt = alt;
            s.best.alpha = Lds::kUber ? (int)lane_u32(alpha, t) : 0;
            s.best.enforce = !s.best.alpha && s.best.lo == s.best.hi;
            if (s.best.enforce) {
                if ((s.best.lo & 31) != 31) {
                    s.best.lo++;
                    s.best.enforced = 1;
                } else {
                    s.best.hi--;
                    s.best.enforced = 0;
                }
            }
            s.sel_valid = false;
            if (Lds::kUber) s.sel_nonempty = true;
            took = true;
            if (again) {
                first = uni(q.cidx[t]) + 1;
                return true;
            }
            left = t == 63 ? 0ull : ~0ull << (t + 1);
        }
    }
    return took;
}

// The selector of a colour: compute_selectors_hc (crn_dxt1.cpp:1837-1869), or
// with `three` the 3-colour palette's first nearest entry (evaluate_solution_uber).
__device__ inline uint32_t nearest(const Pal& p, int perceptual, bool three, uint32_t px)
{
    const uint32_t e0 = cdist(perceptual, px, p.r[0], p.g[0], p.b[0]);
    const uint32_t e1 = cdist(perceptual, px, p.r[1], p.g[1], p.b[1]);
    const uint32_t e2 = cdist(perceptual, px, p.r[2], p.g[2], p.b[2]);
    if (three) return e1 < e0 ? (e2 < e1 ? 2 : 1) : (e2 < e0 ? 2 : 0);
    const uint32_t e3 = cdist(perceptual, px, p.r[3], p.g[3], p.b[3]);
    const uint32_t e01 = min(e0, e1), e23 = min(e2, e3);
    return e01 <= e23 ? (e01 == e0 ? 0 : 1) : (e23 == e2 ? 2 : 3);
}

// The best solution's selectors of the unique colours.
template <class Lds>
__device__ void compute_selectors(St& s, Lds& L)
{
    if (s.sel_valid) return;
    const bool three = Lds::kUber && s.best.alpha;
    const Pal p = three ? palette3(s.best.lo, s.best.hi, s.best.alt) : palette4(s.best.lo, s.best.hi, s.best.alt);
    for (uint32_t i = lane_id(); i < s.nu; i += 64)
        L.sel[i] = (uint8_t)(s.best.enforce ? (uint32_t)s.best.enforced : nearest(p, s.perceptual, three, L.col[i]));
    __builtin_amdgcn_wave_barrier();
    s.sel_valid = true;
    s.sel_nonempty = true;
}

// --------------------------------------------------- sequential float sums
// Lane k < K adds row k's 64 staged terms to its sum, one after another.
__device__ inline float add_row(const float* row, float a)
{
#pragma unroll
    for (uint32_t j = 0; j < 64; j += 4) {
        const float4 v = *reinterpret_cast<const float4*>(row + j);
        a += v.x;
        a += v.y;
        a += v.z;
        a += v.w;
    }
    return a;
}

__device__ inline double add_row(const double* row, double a)
{
#pragma unroll
    for (uint32_t j = 0; j < 64; j += 2) {
        const double2 v = *reinterpret_cast<const double2*>(row + j);
        a += v.x;
        a += v.y;
    }
    return a;
}

// normalised (and perceptually weighted) colour minus the mean, as
// compute_vectors stores it (crn_dxt1.cpp:155-189)
__device__ inline void norm_of(const St& s, uint32_t c, float* n, float* nw)
{
    for (int k = 0; k < 3; k++) {
        const float v = (float)((c >> (8 * k)) & 255u) * 1.0f / 255.0f;
        n[k] = v - s.mean[k];
        nw[k] = s.pw[k] * v - s.meanw[k];
    }
}

template <class Lds>
__device__ void compute_vectors(St& s, Lds& L)
{
    const uint32_t lane = lane_id();
    float(*f)[kRow] = L.u.q.stage.f;
    float acc = 0.0f;
    for (uint32_t i0 = 0; i0 < s.nu; i0 += 64) {
        const uint32_t i = min(i0 + lane, s.nu - 1), c = L.col[i];
        const bool in = i0 + lane < s.nu;
        const float w = (float)L.w[i];
        for (int k = 0; k < 3; k++) {
            const float v = (float)((c >> (8 * k)) & 255u) * 1.0f / 255.0f;
            f[k][lane] = in ? v * w : 0.0f;
            f[3 + k][lane] = in ? (s.pw[k] * v) * w : 0.0f;
        }
        __builtin_amdgcn_wave_barrier();
        acc = add_row(f[min(lane, 5u)], acc);
        __builtin_amdgcn_wave_barrier();
    }
    for (uint32_t k = 0; k < 3; k++) {
        s.mean[k] = lane_f32(acc, k);
        s.meanw[k] = lane_f32(acc, 3 + k);
    }
    if (s.total_w) {
        const float inv = 1.0f / (float)s.total_w;
        for (int k = 0; k < 3; k++) {
            s.mean[k] = unif(s.mean[k] * inv);
            s.meanw[k] = unif(s.meanw[k] * inv);
        }
    }
}

// compute_pca (crn_dxt1.cpp:192-256) over the weighted vectors
template <class Lds>
__device__ void compute_pca(St& s, Lds& L, float* axis)
{
    const uint32_t lane = lane_id();
    double(*d)[kRowD] = L.u.q.stage.d;
    double acc = 0.0;
    for (uint32_t i0 = 0; i0 < s.nu; i0 += 64) {
        const uint32_t i = min(i0 + lane, s.nu - 1), wi = L.w[i];
        const bool in = i0 + lane < s.nu;
        float n[3], nw[3];
        norm_of(s, L.col[i], n, nw);
        const float r = nw[0], g = nw[1], b = nw[2];
        const float t[6] = {r * r, r * g, r * b, g * g, g * b, b * b};
        const double w = (double)wi;
        for (int k = 0; k < 6; k++) d[k][lane] = !in ? 0.0 : wi > 1 ? t[k] * w : (double)t[k];
        __builtin_amdgcn_wave_barrier();
        acc = add_row(d[min(lane, 5u)], acc);
        __builtin_amdgcn_wave_barrier();
    }
    double cov[6];
    for (uint32_t k = 0; k < 6; k++) cov[k] = lane_f64(acc, k);
    double vr = .9f, vg = 1.0f, vb = .7f;
    for (int it = 0; it < 8; it++) {
        double r = vr * cov[0] + vg * cov[1] + vb * cov[2];
        double g = vr * cov[1] + vg * cov[3] + vb * cov[4];
        double b = vr * cov[2] + vg * cov[4] + vb * cov[5];
        double m = fabs(r);
        if (fabs(g) > m) m = fabs(g);
        if (fabs(b) > m) m = fabs(b);
        if (m > 1e-10) {
            m = 1.0f / m;
            r *= m;
            g *= m;
            b *= m;
        }
        const double dd = (vr - r) * (vr - r) + (vg - g) * (vg - g) + (vb - b) * (vb - b);
        vr = r;
        vg = g;
        vb = b;
        if (it > 2 && dd < 1e-8) break;
    }
    double len = vr * vr + vg * vg + vb * vb;
    if (len < 1e-10) {
        axis[0] = .2837149f;
        axis[1] = 0.9540631f;
        axis[2] = 0.096277453f;
        return;
    }
    len = 1.0f / sqrt(len);
    axis[0] = (float)(vr * len);
    axis[1] = (float)(vg * len);
    axis[2] = (float)(vb * len);
}

// ray-box intersection (crn_intersect.h:44-120) for the unit cube
__device__ bool ray_unit_box(float* coord, const float* org, const float* dir)
{
    bool inside = true;
    int quad[3];
    float cand[3], maxt[3];
    for (int i = 0; i < 3; i++) {
        cand[i] = 0.0f;
        if (org[i] < 0.0f) { quad[i] = 1; cand[i] = 0.0f; inside = false; }
        else if (org[i] > 1.0f) { quad[i] = 0; cand[i] = 1.0f; inside = false; }
        else quad[i] = 2;
    }
    if (inside) return false;
    for (int i = 0; i < 3; i++) maxt[i] = (quad[i] != 2 && dir[i] != 0.0f) ? (cand[i] - org[i]) / dir[i] : -1.0f;
    int wp = 0;
    float wt = maxt[0];
    for (int i = 1; i < 3; i++)
        if (wt < maxt[i]) {
            wp = i;
            wt = maxt[i];
        }
    if (wt < 0.0f) return false;
    float c[3];
    for (int i = 0; i < 3; i++) {
        if (i != wp) {
            c[i] = org[i] + wt * dir[i];
            if (c[i] < 0.0f || c[i] > 1.0f) return false;
        } else {
            c[i] = cand[i];
        }
    }
    for (int i = 0; i < 3; i++) coord[i] = c[i];
    return true;
}

// refine_solution's least squares (crn_dxt1.cpp:525-600): the rounded
// endpoints into q.fixed; false when the system has no solution.  The sums are
// of integers times integer weights (exact in double), so a lane-split sum is
// the reference's value.
template <class Lds>
__device__ bool refine_fit(St& s, Lds& L)
{
    compute_selectors(s, L);
    uint64_t A0 = 0, A1 = 0, A2 = 0, T1[3] = {0, 0, 0}, T2[3] = {0, 0, 0};
    for (uint32_t i = lane_id(); i < s.nu; i += 64) {
        const uint32_t c = L.col[i];
        const uint64_t w = L.w[i];
        const int step = L.sel[i] ^ 1;
        const uint32_t w1 = step == 0 ? 3 : step == 1 ? 0 : step == 2 ? 2 : 1;
        const uint32_t q0 = step >= 2 ? 2 : 0;
        const uint32_t q1 = step == 0 ? 0 : step == 1 ? 9 : step == 2 ? 1 : 4;
        const uint32_t q2 = step == 0 ? 9 : step == 1 ? 0 : step == 2 ? 4 : 1;
        A0 += q0 * w;
        A1 += q1 * w;
        A2 += q2 * w;
        for (int k = 0; k < 3; k++) {
            const uint64_t v = ((c >> (8 * k)) & 255u) * w;
            T1[k] += w1 * v;
            T2[k] += v;
        }
    }
    A0 = wave_sum(A0);
    A1 = wave_sum(A1);
    A2 = wave_sum(A2);
    double t1[3], t2[3];
    for (int k = 0; k < 3; k++) {
        t1[k] = (double)wave_sum(T1[k]);
        t2[k] = 3 * (double)wave_sum(T2[k]) - t1[k];
    }
    const double xx = (double)A2, yy = (double)A1, xy = (double)A0;
    const double t = xx * yy - xy * xy;
    if (unib(!yy || !xx || fabs(t) < (double).0000125f)) return false;
    const double frb = (double)(3.0f * 31.0f / 255.0f) / t;
    const double fg = frb * (double)(63.0f / 31.0f);
    int e0[3], e1[3];
    e0[0] = clampi((int)((t1[0] * yy - t2[0] * xy) * frb + (double)0.5f), 31);
    e0[1] = clampi((int)((t1[1] * yy - t2[1] * xy) * fg + (double)0.5f), 63);
    e0[2] = clampi((int)((t1[2] * yy - t2[2] * xy) * frb + (double)0.5f), 31);
    e1[0] = clampi((int)((t2[0] * xx - t1[0] * xy) * frb + (double)0.5f), 31);
    e1[1] = clampi((int)((t2[1] * xx - t1[1] * xy) * fg + (double)0.5f), 63);
    e1[2] = clampi((int)((t2[2] * xx - t1[2] * xy) * frb + (double)0.5f), 31);
    if (lane_id() == 0)
        for (int k = 0; k < 3; k++) {
            L.u.q.fixed[0][k] = e0[k];
            L.u.q.fixed[1][k] = e1[k];
        }
    __builtin_amdgcn_wave_barrier();
    return true;
}

// fast_random (crn_rand.cpp:310-405)
struct FastRandom {
    uint32_t jsr = 0xABCD917Au, jcong = 0x17F3DEADu;
    __device__ uint32_t u32()
    {
        jsr ^= jsr << 17;
        jsr ^= jsr >> 13;
        jsr ^= jsr << 5;
        jcong = 69069u * jcong + 1234567u;
        return jsr ^ jcong;
    }
    __device__ float frand(float l, float h)
    {
        if (l >= h) return l;
        const float v = (float)((double)l + (double)(h - l) * ((double)u32() * (1.0 / 4294967296.0)));
        return v < l ? l : (v > h ? h : v);
    }
};

// try_median4's means (crn_dxt1.cpp:1181-1290): 4-means over the colours with
// sequential float sums (lane 4 j + k: mean j's component k, k = 3 its weight;
// lane 16: the total distance); the four means as 5:6:5 colours into q.list.
template <class Lds>
__device__ void median4(St& s, Lds& L, const float* lo, const float* hi)
{
    const uint32_t lane = lane_id();
    SearchLds& q = L.u.q;
    float means[4][3];
    if (s.nu <= 4) {
        for (uint32_t i = 0; i < 4; i++) {
            float n[3], nw[3];
            norm_of(s, L.col[min(i, s.nu - 1)], n, nw);
            for (int k = 0; k < 3; k++) means[i][k] = n[k];
        }
    } else {
        for (int k = 0; k < 3; k++) {
            means[0][k] = lo[k] - s.mean[k];
            means[3][k] = hi[k] - s.mean[k];
        }
        for (int k = 0; k < 3; k++) {
            means[1][k] = means[0][k] + (means[3][k] - means[0][k]) * (1.0f / 3.0f);
            means[2][k] = means[0][k] + (means[3][k] - means[0][k]) * (2.0f / 3.0f);
        }
        FastRandom rm;
        uint32_t rover = 0;
        float prev = 1.0e+37f;
        float(*f)[kRow] = q.stage.f;
        for (uint32_t it = 0; it < 8; it++) {
            float acc = 0.0f;
            const uint32_t mine = min(lane >> 2, 4u);
            const float* row = f[lane < 16 ? lane & 3u : 4u];
            for (uint32_t i0 = 0; i0 < s.nu; i0 += 64) {
                const uint32_t i = min(i0 + lane, s.nu - 1);
                const bool in = i0 + lane < s.nu;
                float v[3], vw[3];
                norm_of(s, L.col[i], v, vw);
                float bd = 0;
                for (int k = 0; k < 3; k++) {
                    const float d = means[0][k] - v[k];
                    bd += d * d;
                }
                uint32_t bi = 0;
                for (uint32_t jj = 1; jj < 4; jj++) {
                    float dd = 0;
                    for (int k = 0; k < 3; k++) {
                        const float d = means[jj][k] - v[k];
                        dd += d * d;
                    }
                    if (dd < bd) {
                        bd = dd;
                        bi = jj;
                    }
                }
                const float w = (float)L.w[i];
                for (int k = 0; k < 3; k++) f[k][lane] = v[k] * w;
                f[3][lane] = w;
                f[4][lane] = in ? bd : 0.0f;
                f[5][lane] = __builtin_bit_cast(float, in ? bi : 7u);
                __builtin_amdgcn_wave_barrier();
                // a term of another mean adds +0, which changes no sum (none is -0)
#pragma unroll 4
                for (uint32_t j = 0; j < 64; j += 4) {
                    const float4 x = *reinterpret_cast<const float4*>(row + j);
                    const uint4 b = *reinterpret_cast<const uint4*>(&f[5][j]);
                    const bool all = mine == 4u;
                    acc += all || b.x == mine ? x.x : 0.0f;
                    acc += all || b.y == mine ? x.y : 0.0f;
                    acc += all || b.z == mine ? x.z : 0.0f;
                    acc += all || b.w == mine ? x.w : 0.0f;
                }
                __builtin_amdgcn_wave_barrier();
            }
            const float total = lane_f32(acc, 16);
            uint32_t hidx = 0;
            float hw = 0;
            bool empty = false;
            float nwt[4];
            for (uint32_t jj = 0; jj < 4; jj++) {
                nwt[jj] = lane_f32(acc, 4 * jj + 3);
                if (nwt[jj] > 0.0f) {
                    for (uint32_t k = 0; k < 3; k++) means[jj][k] = lane_f32(acc, 4 * jj + k) / nwt[jj];
                    if (nwt[jj] > hw) {
                        hw = nwt[jj];
                        hidx = jj;
                    }
                } else {
                    empty = true;
                }
            }
            if (!empty) {
                if (unib(fabsf(total - prev) < .00001f)) break;
                prev = total;
            } else {
                prev = 1.0e+37f;
            }
            if (unib(empty) && it != 7) {
                const uint32_t ri = (hidx + rover) & 3u;
                rover++;
                for (uint32_t jj = 0; jj < 4; jj++)
                    if (nwt[jj] == 0.0f)
                        for (int k = 0; k < 3; k++) {
                            const float src = ri == 0 ? means[0][k] : ri == 1 ? means[1][k] : ri == 2 ? means[2][k] : means[3][k];
                            means[jj][k] = src + rm.frand(-.00196f, .00196f);
                        }
            }
        }
    }
    if (lane == 0)
        for (int i = 0; i < 4; i++) {
            float a[3];
            for (int k = 0; k < 3; k++) a[k] = means[i][k] + s.mean[k];
            q.list[0][i] = pack565((int)floorf(.5f + a[0] * 31.0f), (int)floorf(.5f + a[1] * 63.0f),
                                   (int)floorf(.5f + a[2] * 31.0f), 0);
        }
    __builtin_amdgcn_wave_barrier();
}

// are_selectors_all_equal (crn_dxt1.h:300-316) on the best solution's
// selector vector as last computed: the hc evaluators leave it untouched, so
// it may belong to an earlier solution, and it is empty before the first
// compute_selectors.
template <class Lds>
__device__ bool sel_all_equal(const St& s, const Lds& L)
{
    if (!s.sel_nonempty) return false;
    bool diff = false;
    for (uint32_t i = lane_id(); i < s.nu; i += 64) diff |= L.sel[i] != L.sel[0];
    return __ballot(diff) == 0;
}

// The average colour of try_average_block_as_solid (crn_dxt1.cpp:93-153)
template <class Lds>
__device__ uint32_t average_colour(St& s, Lds& L)
{
    uint64_t tr = 0, tg = 0, tb = 0, tw = 0;
    for (uint32_t i = lane_id(); i < s.nu; i += 64) {
        const uint32_t c = L.col[i];
        const uint64_t w = L.w[i];
        tw += w;
        tr += (c & 255u) * w;
        tg += ((c >> 8) & 255u) * w;
        tb += ((c >> 16) & 255u) * w;
    }
    tw = wave_sum(tw);
    tr = wave_sum(tr);
    tg = wave_sum(tg);
    tb = wave_sum(tb);
    const uint64_t half = tw >> 1;
    return (uint32_t)((tr + half) / tw) | (uint32_t)((tg + half) / tw) << 8 | (uint32_t)((tb + half) / tw) << 16;
}

// compute_endpoint_component_errors (crn_dxt1.cpp:369-418)
template <class Lds>
__device__ void comp_errors(St& s, Lds& L, int comp)
{
    SearchLds& sq = L.u.q;
    QErr q;
    uint64_t W[4] = {0, 0, 0, 0}, WP2[4] = {0, 0, 0, 0}, WPP[4] = {0, 0, 0, 0};
    for (uint32_t i = lane_id(); i < s.nu; i += 64) {
        const uint32_t p = (L.col[i] >> (8 * comp)) & 255u;
        const uint32_t w = L.w[i];
        const uint32_t sl = L.sel[i];
        const uint64_t w2 = (uint64_t)w * (2 * p), wpp = (uint64_t)w * (p * p);
#pragma unroll
        for (uint32_t k = 0; k < 4; k++) {
            const bool on = k == sl;
            W[k] += on ? w : 0u;
            WP2[k] += on ? w2 : 0ull;
            WPP[k] += on ? wpp : 0ull;
        }
    }
    for (int k = 0; k < 4; k++) {
        q.W[k] = wave_sum(W[k]);
        q.WP2[k] = wave_sum(WP2[k]);
        q.WPP[k] = wave_sum(WPP[k]);
    }
    const uint32_t lane = lane_id();
    const uint32_t lim = comp == 1 ? 64 : 32;
    uint64_t brem[4];
    for (int sl = 0; sl < 4; sl++) {
        const uint32_t n = sl < 2 ? lim : 256;
        uint64_t m = ~0ull;
        for (uint32_t c = lane; c < n; c += 64) m = min(m, q.at(sl, sl < 2 ? expand_comp(comp, c) : c));
        for (int off = 32; off > 0; off >>= 1) {
            const uint32_t lo = (uint32_t)__shfl_xor((int)(uint32_t)m, off);
            const uint32_t hi = (uint32_t)__shfl_xor((int)(uint32_t)(m >> 32), off);
            m = min(m, ((uint64_t)hi << 32) | lo);
        }
        brem[sl] = uni64(m);
    }
    for (int sl = 3; sl; sl--) brem[sl - 1] += brem[sl];
    if (lane == 0) {
        sq.q = q;
        for (int sl = 0; sl < 4; sl++) sq.brem[sl] = brem[sl];
    }
    __builtin_amdgcn_wave_barrier();
}

// The component errors' sum at (p0, p1) into q.qbest.
template <class Lds>
__device__ void comp_best(Lds& L, uint32_t p0, uint32_t p1)
{
    SearchLds& q = L.u.q;
    const uint64_t best = q.q.at(0, p0) + q.q.at(1, p1) + q.q.at(2, (p0 * 2 + p1) / 3) + q.q.at(3, (p0 + p1 * 2) / 3);
    __builtin_amdgcn_wave_barrier();
    if (lane_id() == 0) q.qbest = best;
    __builtin_amdgcn_wave_barrier();
}

__device__ inline uint32_t lerp_color(uint32_t a, uint32_t b, float f, int rounding)
{
    const float rr = rounding ? 1.0f : 0.0f;
    int o[3];
    for (int k = 0; k < 3; k++) {
        const float x = (float)((a >> (8 * k)) & 255u), y = (float)((b >> (8 * k)) & 255u);
        o[k] = clampi((int)(rr + (x + (y - x) * f)), 255);
    }
    return pack565(o[0], o[1], o[2], 1);
}

// The distinct packed colours of try_combinatorial_encoding (crn_dxt1.cpp:
// 1886-1950) for 2 to 4 colours into q.list[0], in the reference's order (the
// colours, then the interpolations; one per lane): their number.
template <class Lds>
__device__ uint32_t combinatorial_colours(St& s, Lds& L)
{
    SearchLds& q = L.u.q;
    const uint32_t lane = lane_id(), nu = s.nu;
    uint32_t n = nu, p = 0;
    if (lane < nu) {
        const uint32_t c = L.col[lane];
        p = pack565((int)(c & 255u), (int)((c >> 8) & 255u), (int)((c >> 16) & 255u), 1);
    }
    if (nu == 2) {
        // rounding (2) x start (2) x ten factors
        n += 40;
        if (lane >= nu && lane < n) {
            const uint32_t i = lane - nu, k = i / 20, a = i / 10 % 2, f = i % 10;
            const float fs[10] = {2.0f, 3.0f, .5f, 1.5f, -1.0f, 2.0f, -.5f, .5f, -2.0f, -1.0f};
            float v = fs[0];
            for (uint32_t t = 1; t < 10; t++) v = t == f ? fs[t] : v;
            p = lerp_color(L.col[a], L.col[a ^ 1u], v, (int)k);
        }
    } else if (nu == 3) {
        // ordered pairs (6) x four factors
        n += 24;
        if (lane >= nu && lane < n) {
            const uint32_t i = lane - nu, pr = i / 4, f = i % 4, a = pr / 2, b0 = pr % 2, b = b0 >= a ? b0 + 1 : b0;
            const float v = f == 0 ? 1.5f : f == 1 ? 2.0f / 3.0f : f == 2 ? 1.0f / 3.0f : -.5f;
            p = lerp_color(L.col[a], L.col[b], v, 1);
        }
    }
    bool dup = lane >= n;
    for (uint32_t k = 0; k + 1 < n; k++) dup |= k < lane && lane_u32(p, k) == p;
    const uint64_t mask = __ballot(!dup);
    if (!dup) q.list[0][__popcll(mask & ((1ull << lane) - 1ull))] = p;
    const uint32_t np = (uint32_t)__popcll(mask);
    if (lane == 0) q.fixed[0][0] = (int)np;
    __builtin_amdgcn_wave_barrier();
    return np;
}

// One end of a probe sweep into `out`: probe i's two signs in order, each
// dropped when it packs as the sign's probe before it did (one probe and sign
// per lane); their number.
__device__ uint32_t sweep(const float* base, const float (*axis2)[3], uint32_t* out)
{
    const uint32_t lane = lane_id();
    uint32_t packed[2] = {0, 0};
    const uint32_t sg = (lane + 1) & 1u;       // lane 0: probe 0, sign 1; lane 2 i - 1, 2 i: probe i, signs 0, 1
    const uint32_t i = (lane + 1) >> 1;
    for (int back = 0; back < 2; back++) {
        const int x = c_uber_probe[min(i - (uint32_t)(back && i ? 1 : 0), 14u)];
        const float a0 = sg ? axis2[1][0] : axis2[0][0], a1 = sg ? axis2[1][1] : axis2[0][1],
                    a2 = sg ? axis2[1][2] : axis2[0][2];
        const float pr = (base[0] + .5f) + a0 * (float)x;
        const float pg = (base[1] + .5f) + a1 * (float)x;
        const float pb = (base[2] + .5f) + a2 * (float)x;
        packed[back] = (uint32_t)(clampi((int)floorf(pb), 31) | (clampi((int)floorf(pg), 63) << 5) |
                                  (clampi((int)floorf(pr), 31) << 11));
    }
    // probe 0 has sign 1 only: nothing lies before it, nor before probe 1 of sign 0
    const bool first = sg ? i == 0 : i == 1;
    const bool keep = lane < 29 && (first || packed[0] != packed[1]);
    const uint64_t mask = __ballot(keep);
    if (keep) out[__popcll(mask & ((1ull << lane) - 1ull))] = packed[0];
    return (uint32_t)__popcll(mask);
}

// handle_multicolor_block up to optimize_endpoints (crn_dxt1.cpp:1069-1178):
// weights, means, axis, and the two ends of the colours' extent on the axis.
template <class Lds>
__device__ void multicolor_ends(St& s, Lds& L, float* lo, float* hi)
{
    const uint32_t lane = lane_id();
    uint32_t npass = 1;
    s.pw[0] = s.pw[1] = s.pw[2] = 1.0f;
    if (s.perceptual) {
        float(*f)[kRow] = L.u.q.stage.f;
        float acc = 0.0f;
        for (uint32_t i0 = 0; i0 < s.nu; i0 += 64) {
            const uint32_t i = min(i0 + lane, s.nu - 1), c = L.col[i];
            const bool in = i0 + lane < s.nu;
            const int r = (int)(c & 255u), g = (int)((c >> 8) & 255u), b = (int)((c >> 16) & 255u);
            const int l = (r + g + b + 1) / 3;
            const float lf = (float)l;
            const float scale = (float)L.w[i] / (lf > 1.0f ? lf : 1.0f);
            f[0][lane] = in ? scale * r : 0.0f;
            f[1][lane] = in ? scale * b : 0.0f;
            f[2][lane] = in ? lf : 0.0f;
            __builtin_amdgcn_wave_barrier();
            acc = add_row(f[min(lane, 2u)], acc);
            __builtin_amdgcn_wave_barrier();
        }
        float red = lane_f32(acc, 0), blue = lane_f32(acc, 1), al = lane_f32(acc, 2);
        red /= s.total_w;
        blue /= s.total_w;
        al /= s.total_w;
        al = al * 16.0f / 255.0f;
        al = 1.0f < al ? 1.0f : al;
        const float m = red > blue ? red : blue;
        float sat = m * 1.0f / 3.0f;
        sat = sat < 0.0f ? 0.0f : (sat > 1.0f ? 1.0f : sat);
        const float p = unif(al * powf(sat, 2.75f));
        if (p >= 1.0f) {
            npass = 1;
        } else {
            npass = 2;
            const float lum[3] = {.212f, .72f, .072f};
            for (int k = 0; k < 3; k++) s.pw[k] = unif(lum[k] + (s.pw[k] - lum[k]) * p);
        }
    }
    for (uint32_t pass = 0; pass < npass; pass++) {
        compute_vectors(s, L);
        compute_pca(s, L, s.axis);
        s.axis[0] /= s.pw[0];
        s.axis[1] /= s.pw[1];
        s.axis[2] /= s.pw[2];
        double n = s.axis[0] * s.axis[0];
        n += s.axis[1] * s.axis[1];
        n += s.axis[2] * s.axis[2];
        if (n != 0) {
            const float k = (float)(1.0f / sqrt(n));
            for (int i = 0; i < 3; i++) s.axis[i] *= k;
        }
        for (int i = 0; i < 3; i++) s.axis[i] = unif(s.axis[i]);
        if (npass > 1) {
            if (fabsf(s.axis[0]) >= .795f) {
                s.pw[0] = .424f; s.pw[1] = .6f; s.pw[2] = .072f;
            } else if (fabsf(s.axis[2]) >= .795f) {
                s.pw[0] = .212f; s.pw[1] = .6f; s.pw[2] = .212f;
            } else {
                break;
            }
        }
    }
    float l = 1e+9f, h = -1e+9f;
    for (uint32_t i = lane; i < s.nu; i += 64) {
        float n[3], nw[3];
        norm_of(s, L.col[i], n, nw);
        float d = n[0] * s.axis[0];
        d += n[1] * s.axis[1];
        d += n[2] * s.axis[2];
        l = d < l ? d : l;
        h = h < d ? d : h;
    }
    for (int off = 32; off > 0; off >>= 1) {
        const float l2 = __shfl_xor(l, off), h2 = __shfl_xor(h, off);
        l = l2 < l ? l2 : l;
        h = h < h2 ? h2 : h;
    }
    l = unif(l);
    h = unif(h);
    for (int k = 0; k < 3; k++) {
        lo[k] = s.mean[k] + l * s.axis[k];
        hi[k] = s.mean[k] + h * s.axis[k];
    }
    bool in = true;
    for (int k = 0; k < 3; k++)
        if (lo[k] < 0.0f || lo[k] > 1.0f) in = false;
    if (!in) {
        float c[3];
        if (ray_unit_box(c, lo, s.axis)) { lo[0] = c[0]; lo[1] = c[1]; lo[2] = c[2]; }
    }
    in = true;
    for (int k = 0; k < 3; k++)
        if (hi[k] < 0.0f || hi[k] > 1.0f) in = false;
    if (!in) {
        float c[3];
        const float nd[3] = {-s.axis[0], -s.axis[1], -s.axis[2]};
        if (ray_unit_box(c, hi, nd)) { hi[0] = c[0]; hi[1] = c[1]; hi[2] = c[2]; }
    }
}

// The search over the cluster's colours (crn_dxt1.cpp:703-1178, 2207-2232):
// the one-colour shortcut, or handle_multicolor_block and optimize_endpoints
// at uber quality.  Every step prepares a list of candidates; one loop tries
// them, so that gathering, scoring and taking exist once.
enum Step : uint32_t {
    kStepOne,         // a single colour
    kStepMedian,      // try_median4: the pairs of means ...
    kStepMedianFit,   // ... and refine_solution
    kStepSweep,       // a pass: probe sweeps, lattice moves of either end, refine_solution
    kStepAdj0,
    kStepAxis0,
    kStepAdj1,
    kStepAxis1,
    kStepPassEnd,
    kStepSolid,       // all selectors equal: solid tries
    kStepComps,       // optimize_endpoint_comps, one component at a time
    kStepCombFirst,   // 2 to 4 colours: try_combinatorial_encoding
    kStepComb,
    kStepCombAlt,
};

template <class Lds, uint32_t W>
__device__ void search(St& s, Lds& L)
{
    SearchLds& q = L.u.q;
    const uint32_t lane = lane_id();
    float lo[3], hi[3], ax[2][3];
    uint32_t step = kStepOne, pass = 0;
    uint64_t prev = 0, comb_err = 0;
    int slo[3] = {0, 0, 0}, shi[3] = {0, 0, 0}, comp = 0;
    if (!(s.nu == 1 && !s.have_alpha)) {
        multicolor_ends(s, L, lo, hi);
        median4(s, L, lo, hi);
        const float dist = .015625f;
        for (int k = 0; k < 3; k++) ax[1][k] = s.axis[k] * dist;
        ax[1][0] *= 31.0f;
        ax[1][1] *= 63.0f;
        ax[1][2] *= 31.0f;
        for (int k = 0; k < 3; k++) ax[0][k] = -ax[1][k];
        const float lim[3] = {31.0f, 63.0f, 31.0f};
        for (int k = 0; k < 3; k++) {
            const float a = lo[k] * lim[k];
            lo[k] = a < 0.0f ? 0.0f : (a > lim[k] ? lim[k] : a);
            const float b = hi[k] * lim[k];
            hi[k] = b < 0.0f ? 0.0f : (b > lim[k] ? lim[k] : b);
        }
        step = kStepMedian;
    }
    for (;;) {
        uint32_t kind = 0, n = 0, from = 0;
        int alt = 0;
        bool again = false;
        switch (step) {
        case kStepOne:
            // evaluated as the average of one colour
            if (lane == 0) q.list[0][0] = L.col[0];
            __builtin_amdgcn_wave_barrier();
            kind = kListSolid;
            n = Lds::kUber ? 2 : 1;
            break;
        case kStepMedian:
            kind = kListPair;
            n = 6;
            break;
        case kStepMedianFit:
        case kStepPassEnd:
            if (refine_fit(s, L)) {
                kind = kListRefine;
                n = 54;
            }
            break;
        case kStepSweep: {
            if (pass == 4 || !s.best.err) {
                step = kStepSolid;
                continue;
            }
            if (pass) {
                int r, g, b;
                unpack565(s.best.lo, 0, r, g, b);
                lo[0] = (float)r; lo[1] = (float)g; lo[2] = (float)b;
                unpack565(s.best.hi, 0, r, g, b);
                hi[0] = (float)r; hi[1] = (float)g; hi[2] = (float)b;
            }
            prev = s.best.err;
            const uint32_t nl = sweep(lo, ax, q.list[0]);
            const uint32_t nh = sweep(hi, ax, q.list[1]);
            if (lane == 0) q.fixed[0][0] = (int)nh;
            __builtin_amdgcn_wave_barrier();
            kind = kListSweep;
            n = nl * 32;
            break;
        }
        case kStepAdj0:
        case kStepAdj1:
            kind = step == kStepAdj0 ? kListAdj0 : kListAdj1;
            from = step == kStepAdj0 ? s.best.lo : s.best.hi;
            n = 26;
            again = true;
            break;
        case kStepAxis0:
        case kStepAxis1:
            kind = step == kStepAxis0 ? kListAxis0 : kListAxis1;
            from = step == kStepAxis0 ? s.best.lo : s.best.hi;
            n = 6;
            again = true;
            break;
        case kStepSolid:
            if (!s.best.err || s.have_alpha) {
                step = kStepCombFirst;
                continue;
            }
            // the uber evaluator keeps the best solution's selectors current
            if (Lds::kUber && s.sel_nonempty) compute_selectors(s, L);
            if (sel_all_equal(s, L)) {
                const uint32_t avg = average_colour(s, L);
                if (lane == 0) q.list[0][0] = avg;
                __builtin_amdgcn_wave_barrier();
                kind = kListSolid;
                n = (s.nu + 1) * (Lds::kUber ? 2 : 1);
            }
            break;
        case kStepComps: {
            if (comp == 0) {
                // the starting values stay those of the solution found so far
                compute_selectors(s, L);
                unpack565(s.best.lo, 1, slo[0], slo[1], slo[2]);
                unpack565(s.best.hi, 1, shi[0], shi[1], shi[2]);
            }
            if (!s.best.err || comp == 3 || (comp == 0 && s.best.alpha)) {
                step = kStepCombFirst;
                continue;
            }
            int a[3], b[3];
            unpack565(s.best.lo, 0, a[0], a[1], a[2]);
            unpack565(s.best.hi, 0, b[0], b[1], b[2]);
            if (lane == 0)
                for (int k = 0; k < 3; k++) {
                    q.fixed[0][k] = a[k];
                    q.fixed[1][k] = b[k];
                }
            compute_selectors(s, L);
            comp_errors(s, L, comp);
            comp_best(L, (uint32_t)(comp == 0 ? slo[0] : comp == 1 ? slo[1] : slo[2]),
                      (uint32_t)(comp == 0 ? shi[0] : comp == 1 ? shi[1] : shi[2]));
            if (uni64(q.brem[0]) < uni64(q.qbest)) {
                kind = kListComp0 + (uint32_t)comp;
                n = (comp == 1 ? 64u : 32u) * 64;
                again = true;
            }
            break;
        }
        case kStepCombFirst:
            if (!s.best.err || s.nu < 2 || s.nu > 4) return;
            combinatorial_colours(s, L);
            step = kStepComb;
            continue;
        case kStepComb:
        case kStepCombAlt:
            kind = kListComb;
            alt = step == kStepCombAlt ? 1 : 0;
            n = uni((uint32_t)q.fixed[0][0]) * 64;
            break;
        }
        bool improved = false;
        uint32_t first = 0;
        while (first < n && try_list<Lds, W>(s, L, kind, n, alt, again, from, first)) {
            improved = true;
            if (kind >= kListComp0 && s.best.err) {
                // the tables and the best of the new solution's selectors
                const uint32_t i = first - 1;
                compute_selectors(s, L);
                comp_errors(s, L, comp);
                comp_best(L, expand_comp(comp, i >> 6), expand_comp(comp, i & 63u));
            }
        }
        switch (step) {
        case kStepOne: return;
        case kStepAxis1:
            step = !s.best.err || (pass && s.best.err == prev) ? (uint32_t)kStepSolid : (uint32_t)kStepPassEnd;
            break;
        case kStepPassEnd:
            pass++;
            step = kStepSweep;
            break;
        case kStepSolid: step = improved ? (uint32_t)kStepCombFirst : (uint32_t)kStepComps; break;
        case kStepComps: comp++; break;
        case kStepComb:
            comb_err = s.best.err;
            if (comb_err) s.best.err = 1;
            step = kStepCombAlt;
            break;
        case kStepCombAlt:
            if (s.best.err) s.best.err = comb_err;
            return;
        default: step++; break;   // kStepMedian, kStepMedianFit, kStepSweep, kStepAdj0, kStepAxis0, kStepAdj1
        }
    }
}

struct ClusterOut {
    uint64_t error;
    uint32_t lo_hi;    // results::m_low_color | m_high_color << 16
    uint32_t nunique;
    uint32_t flags;    // reordered | alternate_rounding << 2 | enforce << 3 | enforced << 4 | too_many_colours << 8
    uint32_t pad;
};
constexpr uint32_t kNotEncoded = 1u << 8;

// Open-addressing colour hash over `cap` slots (a power of two in LDS, any
// size in the global store): first slot and linear probe.
__device__ inline uint32_t hash_next(uint32_t cap, uint32_t h) { return h + 1 == cap ? 0 : h + 1; }

__device__ inline uint32_t hash_find(const uint32_t* hkey, uint32_t cap, uint32_t key)
{
    uint32_t h = hash32(key) % cap;
    while (hkey[h] != key) h = hash_next(cap, h);
    return h;
}

// Ascending bitonic sort of P (a power of two) pairs by (key, idx), T threads.
template <uint32_t T>
__device__ inline void sort_pairs(uint32_t* key, uint16_t* idx, uint32_t P)
{
    for (uint32_t k = 2; k <= P; k <<= 1)
        for (uint32_t j = k >> 1; j > 0; j >>= 1) {
            for (uint32_t t = threadIdx.x; t < P / 2; t += T) {
                const uint32_t a = ((t & ~(j - 1)) << 1) | (t & (j - 1)), b = a + j;
                const uint32_t ka = key[a], kb = key[b];
                const uint32_t ia = idx[a], ib = idx[b];
                const bool gt = ka > kb || (ka == kb && ia > ib);
                if (gt == ((a & k) == 0)) {
                    key[a] = kb;
                    key[b] = ka;
                    idx[a] = (uint16_t)ib;
                    idx[b] = (uint16_t)ia;
                }
            }
            __syncthreads();
        }
}

// Unique colours of a cluster of n <= MaxU texels in first-appearance order
// with their texel counts, without a hash: sorted (colour, texel index) pairs, the first texel of each run of equal
// colours marked in a bitmap, a colour's rank = the number of marked texels
// before its first one.  Each of the T threads then walks its stretch of the
// sorted pairs from the run that reaches into it.
template <uint32_t MaxU, uint32_t T>
__device__ uint32_t unique_sorted(LdsS<MaxU>& L, const uint32_t* __restrict__ px, uint32_t p0, uint32_t n,
                                  uint32_t thresh, uint32_t& opaque)
{
    uint32_t* key = reinterpret_cast<uint32_t*>(L.sel);
    uint16_t* idx = reinterpret_cast<uint16_t*>(key + MaxU);
    const uint32_t tid = threadIdx.x, lane = lane_id(), wave = uni(tid >> 6);
    uint32_t P = 64;
    while (P < n) P <<= 1;   // n <= MaxU, a power of two
    if (tid == 0) L.nopaque = 0;
    __syncthreads();
    for (uint32_t i0 = 0; i0 < P; i0 += T) {
        // transparent texels (DXT1A) sort after every colour, before the padding
        const uint32_t i = i0 + tid;
        const uint32_t p = i < n ? px[p0 + i] : 0u;
        const bool tr = i < n && (p >> 24) < thresh;
        if (i < P) {
            key[i] = i < n ? (tr ? 0xFFFFFFFEu : (p & 0x00FFFFFFu)) : 0xFFFFFFFFu;
            idx[i] = (uint16_t)i;
        }
        const uint64_t mask = __ballot(i < n && !tr);
        if (lane == 0) atomicAdd(&L.nopaque, (uint32_t)__popcll(mask));
    }
    for (uint32_t i = tid; i < MaxU / 32; i += T) L.fbits[i] = 0;
    __syncthreads();
    const uint32_t nop = opaque = uni(L.nopaque);
    sort_pairs<T>(key, idx, P);
    // runs of equal colours (the padding sorts past the n real texels)
    for (uint32_t j = tid; j < nop; j += T)
        if (j == 0 || key[j] != key[j - 1]) atomicOr(&L.fbits[idx[j] >> 5], 1u << (idx[j] & 31u));
    __syncthreads();
    if (wave == 0) {
        uint32_t base = 0;
        for (uint32_t w0 = 0; w0 < MaxU / 32; w0 += 64) {
            const uint32_t w = w0 + lane;
            const uint32_t cnt = w < MaxU / 32 ? (uint32_t)__popc(L.fbits[w]) : 0u;
            uint32_t incl = cnt;
            for (uint32_t off = 1; off < 64; off <<= 1) {
                const uint32_t v = (uint32_t)__shfl_up((int)incl, off);
                if (lane >= off) incl += v;
            }
            if (w < MaxU / 32) L.fbase[w] = base + incl - cnt;
            base += lane_u32(incl, 63);
        }
        if (lane == 0) L.nuniq = base;
    }
    // the last run start in each thread's stretch, and by a scan the one before it
    const uint32_t E = P > T ? P / T : 1u, j0 = min(tid * E, nop), j1 = min(j0 + E, nop);
    int head = -1;
    for (uint32_t j = j0; j < j1; j++)
        if (j == 0 || key[j] != key[j - 1]) head = (int)j;
    int incl = head;
    for (uint32_t off = 1; off < 64; off <<= 1) {
        const int v = __shfl_up(incl, off);
        if (lane >= off) incl = max(incl, v);
    }
    if (lane == 63) L.scan[wave] = incl;
    int before = __shfl_up(incl, 1);
    if (lane == 0) before = -1;
    __syncthreads();
    for (uint32_t w = 0; w < wave; w++) before = max(before, L.scan[w]);
    auto rank = [&](uint32_t j) {
        const uint32_t f = idx[j];   // the colour's first texel
        return L.fbase[f >> 5] + (uint32_t)__popc(L.fbits[f >> 5] & ((1u << (f & 31u)) - 1u));
    };
    if (j0 < j1) {
        int h = before;
        uint32_t r = h >= 0 ? rank((uint32_t)h) : 0u;
        for (uint32_t j = j0; j < j1; j++) {
            if (j == 0 || key[j] != key[j - 1]) {
                if (h >= 0) L.w[r] = (uint16_t)(j - (uint32_t)h);
                h = (int)j;
                r = rank(j);
                L.col[r] = key[j];
            }
        }
        if (j1 == nop) L.w[r] = (uint16_t)(nop - (uint32_t)h);
    }
    __syncthreads();
    return uni(L.nuniq);
}

// The same for a cluster of any number of texels, through a colour hash in
// LDS that keeps each colour's first texel and count; a colour's rank follows
// from sorting the first texels.  More than MaxU colours: returns MaxU + 1.
template <uint32_t MaxU, uint32_t T>
__device__ uint32_t unique_hashed(LdsT<MaxU>& L, const uint32_t* __restrict__ px, uint32_t p0, uint32_t n,
                                  uint32_t thresh, uint32_t& opaque)
{
    constexpr uint32_t kCap = LdsT<MaxU>::kCapH, kPer = MaxU / T;
    const uint32_t tid = threadIdx.x;
    for (uint32_t i = tid; i < kCap; i += T) {
        L.hkey[i] = 0;
        L.hval[i] = 0xFFFFFFFFu;
        L.hcnt[i] = 0;
    }
    if (tid == 0) L.nuniq = L.nopaque = L.nsort = 0;
    __syncthreads();
    uint32_t nop = 0;
    // the table is half empty at MaxU colours and each thread adds at most one
    // more once the count has passed it, so a probe always ends
    static_assert(MaxU + T < kCap, "hash load");
    auto insert = [&](uint32_t key, uint32_t first, uint32_t count) {
        if (__hip_atomic_load(&L.nuniq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) > MaxU) return;
        uint32_t h = hash32(key) % kCap;
        for (;;) {
            const uint32_t prev = atomicCAS(&L.hkey[h], 0u, key);
            if (prev == 0u) atomicAdd(&L.nuniq, 1u);
            if (prev == 0u || prev == key) {
                atomicMin(&L.hval[h], first);
                atomicAdd(&L.hcnt[h], count);
                return;
            }
            h = hash_next(kCap, h);
        }
    };
    // four texels per thread at a time; equal neighbours are added at once
    for (uint32_t i = 4 * tid; i < n; i += 4 * T) {
        uint32_t p[4], run = 0, first = 0, key = 0;
        const uint32_t m = min(4u, n - i);
        for (uint32_t k = 0; k < 4; k++) p[k] = px[p0 + i + min(k, m - 1)];
        for (uint32_t k = 0; k < m; k++) {
            if ((p[k] >> 24) < thresh) continue;   // transparent (DXT1A)
            const uint32_t c = (p[k] & 0x00FFFFFFu) | 0xFF000000u;
            nop++;
            if (run && c == key) {
                run++;
                continue;
            }
            if (run) insert(key, first, run);
            key = c;
            first = i + k;
            run = 1;
        }
        if (run) insert(key, first, run);
    }
    atomicAdd(&L.nopaque, nop);
    __syncthreads();
    opaque = uni(L.nopaque);
    const uint32_t nu = uni(L.nuniq);
    if (nu > MaxU) return MaxU + 1;
    uint32_t* first = L.col;
    uint16_t* slot = reinterpret_cast<uint16_t*>(L.w);
    uint32_t P = 64;
    while (P < nu) P <<= 1;
    for (uint32_t h = tid; h < kCap; h += T)
        if (L.hkey[h]) {
            const uint32_t at = atomicAdd(&L.nsort, 1u);
            first[at] = L.hval[h];
            slot[at] = (uint16_t)h;
        }
    for (uint32_t i = nu + tid; i < P; i += T) {
        first[i] = 0xFFFFFFFFu;
        slot[i] = 0xFFFFu;
    }
    __syncthreads();
    sort_pairs<T>(first, slot, P);
    uint32_t mine[kPer];
#pragma unroll
    for (uint32_t k = 0; k < kPer; k++) mine[k] = tid + k * T < nu ? slot[tid + k * T] : 0u;
    __syncthreads();
#pragma unroll
    for (uint32_t k = 0; k < kPer; k++) {
        const uint32_t r = tid + k * T;
        if (r < nu) {
            L.col[r] = L.hkey[mine[k]] & 0x00FFFFFFu;
            L.w[r] = L.hcnt[mine[k]];
        }
    }
    __syncthreads();
    return nu;
}

// The colour set of a cluster with more distinct colours than the LDS store
// holds: colours, weights, selectors and the hash in global memory (a scratch
// region the cluster owns, sized by its texel count), the search's working
// set and tables in LDS.
struct GTables {
    PlanesOrSearch u;
    Bounds b;
    uint32_t nopaque;
    uint32_t scan[8];    // per wave
};

struct GStore {
    PlanesOrSearch& u;
    Bounds& b;
    uint32_t kCapH = 0;
    uint32_t* col = nullptr;
    uint32_t* w = nullptr;
    uint8_t* sel = nullptr;
    uint32_t* hkey = nullptr;
    uint32_t* hval = nullptr;
    __device__ explicit GStore(GTables& t) : u(t.u), b(t.b) {}
};

// Clusters by texel count into the five classes (any order within a class: each
// cluster's result depends only on its own texels).
__global__ void __launch_bounds__(256) dxt1_cluster_classes_kernel(const uint32_t* __restrict__ ofs,
                                                                  uint32_t nclusters, uint32_t* __restrict__ count,
                                                                  uint32_t* __restrict__ list)
{
    const uint32_t c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= nclusters) return;
    const uint32_t n = ofs[c + 1] - ofs[c];
    const uint32_t k = n <= 512 ? 0 : n <= 1024 ? 1 : n <= 2048 ? 2 : n <= 4096 ? 3 : 4;
    // the last two classes share an array of nclusters entries, filled from its two ends
    const uint32_t at = atomicAdd(&count[k], 1u);
    if (k < 4) list[(size_t)k * nclusters + at] = c;
    else list[4 * (size_t)nclusters - 1 - at] = c;
}

// One channel's bounds: prefix sums of its planes, one value per lane.
__device__ inline uint64_t channel_bounds(const unsigned long long (*pl)[3], uint32_t lim, uint64_t scale, uint64_t* lo,
                                          uint64_t* hi)
{
    const uint32_t lane = lane_id();
    uint64_t p[3];
    for (int k = 0; k < 3; k++) {
        p[k] = lane < lim ? pl[lane][k] * scale : 0ull;
        for (uint32_t off = 1; off < 64; off <<= 1) {
            const uint32_t a = (uint32_t)__shfl_up((int)(uint32_t)p[k], off), b = (uint32_t)__shfl_up((int)(p[k] >> 32), off);
            if (lane >= off) p[k] += (uint64_t)a | ((uint64_t)b << 32);
        }
    }
    const uint64_t C = lim == 64 ? (uint8_t)((lane << 2) | (lane >> 4)) : (uint8_t)((lane << 3) | (lane >> 2));
    const uint64_t t0 = lane_u64(p[0], 63), t1 = lane_u64(p[1], 63), t2 = lane_u64(p[2], 63);
    const uint64_t l = p[2] + C * C * p[0] - 2 * C * p[1];
    if (lane < lim) {
        lo[lane] = l;
        hi[lane] = t2 + C * C * t0 - 2 * C * t1 - l;
    }
    return t2;
}

// Everything after the unique colours: error planes (crn_dxt1.cpp:2134-2203),
// the search, selectors and return_solution, for any colour store.  The
// planes have been cleared.
template <class Lds, uint32_t W>
__device__ void cluster_search(St& s, Lds& L, const uint32_t* __restrict__ px, uint32_t p0, uint32_t n,
                               int flags, uint32_t cl, ClusterOut* __restrict__ out,
                               uint8_t* __restrict__ selectors)
{
    constexpr uint32_t T = 64 * W;
    const uint32_t tid = threadIdx.x, lane = lane_id(), wave = uni(tid >> 6);
    ClusterOut o{};
    const uint32_t thresh = s.have_alpha ? ((uint32_t)flags >> 8) & 255u : 0u;
    if (!s.nu) {
        // no opaque texel (compute_internal, crn_dxt1.cpp:2207-2212): a 3-colour
        // block of zero endpoints, every selector transparent (error 0 here)
        if (selectors)
            for (uint32_t i = tid; i < n; i += T) selectors[p0 + i] = 3;
        if (tid == 0) {
            o.flags = 2;
            out[cl] = o;
        }
        return;
    }
    for (uint32_t i = tid; i < s.nu; i += T) {
        const uint32_t c = L.col[i];
        const unsigned long long w = L.w[i];
        const uint32_t R = c & 255u, G = (c >> 8) & 255u, B = (c >> 16) & 255u;
        const uint32_t r = (R >> 3) + (((R & 7) > (R >> 5)) ? 1 : 0);
        const uint32_t g = (G >> 2) + (((G & 3) > (G >> 6)) ? 1 : 0);
        const uint32_t b = (B >> 3) + (((B & 7) > (B >> 5)) ? 1 : 0);
        auto& pl = L.u.pl;
        atomicAdd(&pl[0][r][0], w); atomicAdd(&pl[0][r][1], w * R); atomicAdd(&pl[0][r][2], w * R * R);
        atomicAdd(&pl[1][g][0], w); atomicAdd(&pl[1][g][1], w * G); atomicAdd(&pl[1][g][2], w * G * G);
        atomicAdd(&pl[2][b][0], w); atomicAdd(&pl[2][b][1], w * B); atomicAdd(&pl[2][b][2], w * B * B);
    }
    __syncthreads();
    if (wave == 0) {
        const uint64_t base = channel_bounds(L.u.pl[0], 32, s.perceptual ? 8u : 1u, L.b.rlo, L.b.rhi) +
                              channel_bounds(L.u.pl[1], 64, s.perceptual ? 25u : 1u, L.b.glo, L.b.ghi) +
                              channel_bounds(L.u.pl[2], 32, 1u, L.b.blo, L.b.bhi);
        if (lane == 0) L.b.base = base;
    }
    __syncthreads();
    s.base = uni64(L.b.base);
    if (wave == 0) {
        s.best.lo = s.best.hi = 0;
        s.best.err = ~0ull;
        s.best.alt = s.best.enforce = s.best.enforced = s.best.alpha = 0;
        s.sel_valid = false;
        s.sel_nonempty = false;
        search<Lds, W>(s, L);
        // return_solution (crn_dxt1.cpp:263-365): four-colour blocks keep low >
        // high (selectors through {1, 0, 3, 2}), 3-colour blocks low <= high
        // (through {1, 0, 2, 3})
        const bool inv = s.best.alpha ? s.best.lo > s.best.hi : s.best.lo < s.best.hi;
        if (lane == 0) {
            const uint32_t lo = inv ? s.best.hi : s.best.lo, hi = inv ? s.best.lo : s.best.hi;
            o.error = s.best.err;
            o.lo_hi = lo | (hi << 16);
            o.nunique = s.nu;
            o.flags = (uint32_t)inv | ((uint32_t)s.best.alpha << 1) | ((uint32_t)s.best.alt << 2) |
                      ((uint32_t)s.best.enforce << 3) | ((uint32_t)s.best.enforced << 4);
            out[cl] = o;
            L.u.q.end_pal = s.best.alpha ? palette3(s.best.lo, s.best.hi, s.best.alt)
                                         : palette4(s.best.lo, s.best.hi, s.best.alt);
            L.u.q.end_alpha = (uint32_t)s.best.alpha;
            L.u.q.end_inv = inv ? 1u : 0u;
            L.u.q.end_enforce = (uint32_t)s.best.enforce;
            L.u.q.end_enforced = (uint32_t)s.best.enforced;
            L.u.q.cmd = 0;
        }
    } else if constexpr (W > 1) {
        score_loop<Lds, W>(L, s.nu, s.base, s.perceptual, wave);
        __syncthreads();
    }
    if (wave == 0) {
        __syncthreads();   // ends the other waves' loop
        if constexpr (W > 1) __syncthreads();
    }
    if (!selectors) return;
    const SearchLds& q = L.u.q;
    const bool alpha = uni(q.end_alpha) != 0, inv = uni(q.end_inv) != 0, enforce = uni(q.end_enforce) != 0;
    const Pal pal = q.end_pal;
    for (uint32_t i = tid; i < n; i += T) {
        const uint32_t p = px[p0 + i];
        uint32_t v = 3;   // transparent (return_solution, crn_dxt1.cpp:300-343)
        if ((p >> 24) >= thresh) {
            v = enforce ? q.end_enforced : nearest(pal, s.perceptual, alpha, p);
            if (inv) v = alpha ? (v < 2 ? v ^ 1u : v) : (v ^ 1u);
        }
        selectors[p0 + i] = (uint8_t)v;
    }
}

// Waves per cluster: the search of one cluster is a chain of lists, so a large
// cluster is shared by several waves (each list's candidates dealt to them)
// and a small one, of which there are thousands, is left to one.  Eight waves
// and batches of 64 serve the last class, whose workgroups have a CU alone.
template <uint32_t Class>
constexpr uint32_t kWavesOf = Class == 0 ? 1 : Class == 1 ? 2 : Class == 4 ? 8 : 4;
constexpr uint32_t kBigWaves = 8;

template <uint32_t Class>
using StoreOf = std::conditional_t<Class == 4, LdsT<kMaxU>, LdsS<(Class < 3 ? 512u << Class : kMaxU)>>;

template <uint32_t Class, bool Uber>
__device__ void cluster_of_class(LdsU<StoreOf<Class>, Uber>& L, const uint32_t* __restrict__ px,
                                 const uint32_t* __restrict__ ofs, uint32_t cl, int flags,
                                 ClusterOut* __restrict__ out, uint8_t* __restrict__ selectors)
{
    constexpr uint32_t W = kWavesOf<Class>, T = 64 * W;
    const uint32_t tid = threadIdx.x;
    const uint32_t p0 = ofs[cl], p1 = ofs[cl + 1];
    const uint32_t n = p1 - p0;
    // DXT1A (qdxt1 with 3-colour blocks): texels with alpha below this are transparent
    const uint32_t thresh = Uber ? ((uint32_t)flags >> 8) & 255u : 0u;
    ClusterOut o{};
    if (!n) {
        if (tid == 0) out[cl] = o;
        return;
    }
    St s;
    s.perceptual = flags & 1;
    uint32_t opaque = n;
    if constexpr (Class < 4) {
        // the class's texel count is at most its colour capacity
        s.nu = unique_sorted<(Class < 3 ? 512u << Class : kMaxU), T>(L, px, p0, n, thresh, opaque);
    } else {
        s.nu = unique_hashed<kMaxU, T>(L, px, p0, n, thresh, opaque);
        if (s.nu > kMaxU) {
            // more distinct colours than this store holds: left to dxt1_cluster_big_kernel
            o.flags = kNotEncoded;
            if (tid == 0) out[cl] = o;
            return;
        }
    }
    s.total_w = opaque;
    s.have_alpha = opaque != n;
    for (uint32_t i = tid; i < 3 * 64 * 3; i += T) (&L.u.pl[0][0][0])[i] = 0;   // over the sort buffers or the hash
    __syncthreads();
    cluster_search<LdsU<StoreOf<Class>, Uber>, W>(s, L, px, p0, n, flags, cl, out, selectors);
}

template <uint32_t Class, bool Uber>
__global__ void __launch_bounds__(64 * kWavesOf<Class>, 4) dxt1_cluster_kernel(const uint32_t* __restrict__ px,
                                                                               const uint32_t* __restrict__ ofs,
                                                                               const uint32_t* __restrict__ list,
                                                                               const uint32_t* __restrict__ count,
                                                                               int flags,
                                                                               ClusterOut* __restrict__ out,
                                                                               uint8_t* __restrict__ selectors)
{
    extern __shared__ __align__(16) uint8_t lds_raw[];
    LdsU<StoreOf<Class>, Uber>& L = *reinterpret_cast<LdsU<StoreOf<Class>, Uber>*>(lds_raw);
    if constexpr (Class < 4) {
        if (blockIdx.x >= *count) return;
        cluster_of_class<Class, Uber>(L, px, ofs, list[blockIdx.x], flags, out, selectors);
    } else {
        // (its list runs downwards)
        const uint32_t num = *count;
        for (uint32_t b = blockIdx.x; b < num; b += gridDim.x) {
            cluster_of_class<Class, Uber>(L, px, ofs, *(list - b), flags, out, selectors);
            __syncthreads();   // the last reads of L
        }
    }
}

// Clusters the LDS pass flagged (more than 4,096 distinct colours), one
// workgroup each, with the colour set in global scratch: the cluster's texels
// own scratch entries [p0, p1) of the texel-sized arrays and [2 p0, 2 p1) of
// the hash.  The first-appearance order is found in parallel: every texel
// inserts its colour with compare-and-swap and keeps the smallest texel index
// and the count per slot, the first texel of each colour is marked, and a
// prefix count over the marks gives each colour its rank.
template <bool Uber>
__global__ void __launch_bounds__(64 * kBigWaves) dxt1_cluster_big_kernel(const uint32_t* __restrict__ px,
                                                                         const uint32_t* __restrict__ ofs,
                                                                         uint32_t nclusters, int perceptual,
                                                                         ClusterOut* __restrict__ out,
                                                                         uint8_t* __restrict__ selectors,
                                                                         uint8_t* __restrict__ work)
{
    constexpr uint32_t W = kBigWaves, T = 64 * W;
    __shared__ GTables G;
    const uint32_t cl = blockIdx.x;
    if (cl >= nclusters || !(out[cl].flags & kNotEncoded)) return;
    const uint32_t tid = threadIdx.x, lane = lane_id(), wave = uni(tid >> 6);
    const uint32_t p0 = ofs[cl], p1 = ofs[cl + 1], n = p1 - p0, total = ofs[nclusters];
    LdsU<GStore, Uber> L(G);
    L.kCapH = 2 * n;
    // scratch layout, 37 bytes per texel of all clusters (`total`): u32
    // arrays col, w, mark of `total` entries, hkey, hval, hcnt of 2 * total,
    // then the u8 selectors of `total`
    uint32_t* base = reinterpret_cast<uint32_t*>(work);
    L.col = base + p0;
    L.w = base + (size_t)total + p0;
    uint32_t* mark = base + 2 * (size_t)total + p0;
    L.hkey = base + 3 * (size_t)total + 2 * (size_t)p0;
    L.hval = base + 5 * (size_t)total + 2 * (size_t)p0;
    uint32_t* hcnt = base + 7 * (size_t)total + 2 * (size_t)p0;
    L.sel = work + 36 * (size_t)total + p0;
    for (uint32_t i = tid; i < L.kCapH; i += T) {
        L.hkey[i] = 0;
        L.hval[i] = 0xFFFFFFFFu;
        hcnt[i] = 0;
    }
    for (uint32_t i = tid; i < n; i += T) mark[i] = 0;
    for (uint32_t i = tid; i < 3 * 64 * 3; i += T) (&G.u.pl[0][0][0])[i] = 0;
    if (tid == 0) G.nopaque = 0;
    __threadfence();
    __syncthreads();
    const uint32_t thresh = Uber ? ((uint32_t)perceptual >> 8) & 255u : 0u;
    uint32_t nop = 0;
    for (uint32_t i = tid; i < n; i += T) {
        if ((px[p0 + i] >> 24) < thresh) continue;   // transparent (DXT1A)
        nop++;
        const uint32_t key = (px[p0 + i] & 0x00FFFFFFu) | 0xFF000000u;
        uint32_t h = hash32(key) % L.kCapH;
        for (;;) {
            const uint32_t prev = atomicCAS(&L.hkey[h], 0u, key);
            if (prev == 0u || prev == key) {
                atomicMin(&L.hval[h], i);
                atomicAdd(&hcnt[h], 1u);
                break;
            }
            h = hash_next(L.kCapH, h);
        }
    }
    atomicAdd(&G.nopaque, nop);
    __threadfence();
    __syncthreads();
    for (uint32_t h = tid; h < L.kCapH; h += T)
        if (L.hkey[h]) mark[L.hval[h]] = 1;
    __threadfence();
    __syncthreads();
    // ranks in texel order: a running count over the marks, T texels per step
    uint32_t base_rank = 0;
    for (uint32_t i0 = 0; i0 < n; i0 += T) {
        const uint32_t i = i0 + tid;
        const bool m = i < n && mark[i];
        const uint64_t bal = __ballot(m);
        if (lane == 0) G.scan[wave] = (uint32_t)__popcll(bal);
        __syncthreads();
        uint32_t before = 0, all = 0;
        for (uint32_t w = 0; w < W; w++) {
            before += w < wave ? G.scan[w] : 0u;
            all += G.scan[w];
        }
        if (m) {
            const uint32_t r = base_rank + before + (uint32_t)__popcll(bal & ((1ull << lane) - 1ull));
            const uint32_t key = (px[p0 + i] & 0x00FFFFFFu) | 0xFF000000u;
            const uint32_t h = hash_find(L.hkey, L.kCapH, key);
            L.col[r] = key & 0x00FFFFFFu;
            L.w[r] = hcnt[h];
        }
        base_rank += all;
        __syncthreads();
    }
    __threadfence();
    __syncthreads();
    St s;
    s.perceptual = perceptual & 1;
    s.nu = uni(base_rank);
    s.total_w = uni(G.nopaque);
    s.have_alpha = s.total_w != n;
    cluster_search<LdsU<GStore, Uber>, W>(s, L, px, p0, n, perceptual, cl, out, selectors);
}

}  // namespace

namespace {
// Helper streams and events for crn2_dxt1_clusters_device, one set per device,
// kept until the process ends.  Callers hold g_side_mu from the fork to the
// join, so concurrent calls queue their work on the shared streams in turn.
std::mutex g_side_mu;

int side_streams(hipStream_t* side, hipEvent_t* fork, hipEvent_t* join)
{
    struct Set {
        bool ready = false;
        hipStream_t s[3];
        hipEvent_t fork, join[3];
    };
    static Set sets[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return CRN2_EHIP;
    Set& set = sets[dev];
    if (!set.ready) {
        for (int i = 0; i < 3; i++)
            if (hipStreamCreateWithFlags(&set.s[i], hipStreamNonBlocking) != hipSuccess) return CRN2_EHIP;
        if (hipEventCreateWithFlags(&set.fork, hipEventDisableTiming) != hipSuccess) return CRN2_EHIP;
        for (int i = 0; i < 3; i++)
            if (hipEventCreateWithFlags(&set.join[i], hipEventDisableTiming) != hipSuccess) return CRN2_EHIP;
        set.ready = true;
    }
    for (int i = 0; i < 3; i++) {
        side[i] = set.s[i];
        join[i] = set.join[i];
    }
    *fork = set.fork;
    return CRN2_OK;
}
}  // namespace

namespace {
// Scratch of crn2_dxt1_clusters_noalloc_device: the class counters, then four
// lists of at most kNoAllocMaxClusters cluster indices (1 MiB + 32 B on every
// GPU the library runs on, held until the process ends).  Host code never
// passes the array's name to a kernel: it takes the device address from
// hipGetSymbolAddress once per device (noalloc_scratch below).
constexpr uint32_t kNoAllocMaxClusters = 65536;
constexpr uint32_t kCountWords = 8;   // class counters, before the lists
__device__ __align__(256) uint32_t scratch[kCountWords + 4 * kNoAllocMaxClusters];

__global__ void clear_class_counts_kernel(uint32_t* __restrict__ count)
{
    if (threadIdx.x < kCountWords) count[threadIdx.x] = 0;
}

constexpr int kMaxDevices = 64;
std::mutex g_init_mu;
bool g_init[kMaxDevices];
uint32_t* g_noalloc_scratch[kMaxDevices];

// Per-device set-up: the single-colour tables in device memory, the kernels'
// LDS limits and the device address of `scratch`.  Idempotent; runs on the
// device that is current.
template <uint32_t Class, bool Uber>
int set_lds_of()
{
    return hipFuncSetAttribute(reinterpret_cast<const void*>(&dxt1_cluster_kernel<Class, Uber>),
                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)sizeof(StoreOf<Class>)) == hipSuccess
               ? CRN2_OK
               : CRN2_EHIP;
}

template <bool Uber>
int set_lds()
{
    if (set_lds_of<0, Uber>() != CRN2_OK || set_lds_of<1, Uber>() != CRN2_OK || set_lds_of<2, Uber>() != CRN2_OK ||
        set_lds_of<3, Uber>() != CRN2_OK || set_lds_of<4, Uber>() != CRN2_OK)
        return CRN2_EHIP;
    return CRN2_OK;
}

int clusters_init(int* dev_out)
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return CRN2_EHIP;
    *dev_out = dev;
    std::lock_guard<std::mutex> lk(g_init_mu);
    if (g_init[dev]) return CRN2_OK;
    // ryg single-colour tables (crn_ryg_dxt.cpp:58-99, 517-535), four- and
    // three-colour
    static uint8_t t5[256][2], t6[256][2], t5_3[256][2], t6_3[256][2];
    static bool tables = false;
    if (!tables) {
        for (int which = 0; which < 4; which++) {
            const int size = (which & 1) ? 64 : 32;
            const bool three = which >= 2;
            uint8_t (*t)[2] = which == 0 ? t5 : which == 1 ? t6 : which == 2 ? t5_3 : t6_3;
            for (int i = 0; i < 256; i++) {
                int best = 256;
                for (int mn = 0; mn < size; mn++)
                    for (int mx = 0; mx < size; mx++) {
                        const int me = size == 32 ? ((mn << 3) | (mn >> 2)) : ((mn << 2) | (mn >> 4));
                        const int xe = size == 32 ? ((mx << 3) | (mx >> 2)) : ((mx << 2) | (mx >> 4));
                        int err = three ? abs(((me + xe) >> 1) - i) : abs(((xe * 2 + me) / 3) - i);
                        err += (abs(xe - me) * 8) >> 8;
                        if (err < best) {
                            t[i][0] = (uint8_t)mx;
                            t[i][1] = (uint8_t)mn;
                            best = err;
                        }
                    }
            }
        }
        tables = true;
    }
    if (hipMemcpyToSymbol(HIP_SYMBOL(g_c_om5), t5, 512) != hipSuccess) return CRN2_EHIP;
    if (hipMemcpyToSymbol(HIP_SYMBOL(g_c_om6), t6, 512) != hipSuccess) return CRN2_EHIP;
    if (hipMemcpyToSymbol(HIP_SYMBOL(g_c_om5_3), t5_3, 512) != hipSuccess) return CRN2_EHIP;
    if (hipMemcpyToSymbol(HIP_SYMBOL(g_c_om6_3), t6_3, 512) != hipSuccess) return CRN2_EHIP;
    if (set_lds<false>() != CRN2_OK || set_lds<true>() != CRN2_OK) return CRN2_EHIP;
    void* p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return CRN2_EHIP;
    g_noalloc_scratch[dev] = static_cast<uint32_t*>(p);
    g_init[dev] = true;
    return CRN2_OK;
}

// One class's launch: a workgroup per cluster of the call, those past the
// class's count ending at once.  The last class has few clusters and nearly a
// CU's LDS per workgroup, so idle ones would hold the other classes up: one
// workgroup per CU takes its clusters in turn.
template <uint32_t Class, bool Uber>
void launch_class(const uint32_t* px, const uint32_t* offsets, uint32_t nclusters, const uint32_t* list,
                  const uint32_t* count, int flags, ClusterOut* o, uint8_t* selectors, hipStream_t st)
{
    const uint32_t grid = Class < 4 ? nclusters : std::min(nclusters, 256u);
    hipLaunchKernelGGL((dxt1_cluster_kernel<Class, Uber>), dim3(grid), dim3(64 * kWavesOf<Class>),
                       sizeof(StoreOf<Class>), st, px, offsets, list, count + Class, flags, o, selectors);
}

template <bool Uber>
void launch_classes(const uint32_t* px, const uint32_t* offsets, uint32_t nclusters, const uint32_t* list,
                    const uint32_t* work, int perceptual, ClusterOut* o, uint8_t* selectors, const hipStream_t* cls)
{
    const size_t n = nclusters;
    launch_class<4, Uber>(px, offsets, nclusters, list + 4 * n - 1, work, perceptual, o, selectors, cls[3]);
    launch_class<3, Uber>(px, offsets, nclusters, list + 3 * n, work, perceptual, o, selectors, cls[3]);
    launch_class<2, Uber>(px, offsets, nclusters, list + 2 * n, work, perceptual, o, selectors, cls[2]);
    launch_class<1, Uber>(px, offsets, nclusters, list + n, work, perceptual, o, selectors, cls[1]);
    launch_class<0, Uber>(px, offsets, nclusters, list, work, perceptual, o, selectors, cls[0]);
}

// The search proper.  work: kCountWords class counters + 4 lists of nclusters
// entries (device memory).  fork: run the classes side by side on helper
// streams; else every class runs on `st`, in turn (identical results).
int clusters_run(const void* rgba, const uint32_t* offsets, uint32_t nclusters, int flags, void* out,
                 uint8_t* selectors, hipStream_t st, uint32_t* work, bool fork)
{
    hipLaunchKernelGGL(clear_class_counts_kernel, dim3(1), dim3(64), 0, st, work);
    uint32_t* list = work + kCountWords;
    const uint32_t* px = static_cast<const uint32_t*>(rgba);
    ClusterOut* o = static_cast<ClusterOut*>(out);
    hipLaunchKernelGGL(dxt1_cluster_classes_kernel, dim3((nclusters + 255) / 256), dim3(256), 0, st, offsets,
                       nclusters, work, list);
    hipStream_t cls[4] = {st, st, st, st};
    hipStream_t side[3];
    hipEvent_t fork_ev, join[3];
    std::unique_lock<std::mutex> lk(g_side_mu, std::defer_lock);
    int rc = CRN2_OK;
    if (fork) {
        // The classes run side by side: the large clusters are few and long, and
        // alone would leave most CUs idle.  Three helper streams
        // (default priority, created once per device) fork from `st` and join
        // back into it.
        lk.lock();
        rc = side_streams(side, &fork_ev, join);
        if (rc == CRN2_OK && hipEventRecord(fork_ev, st) != hipSuccess) rc = CRN2_EHIP;
        for (int i = 0; rc == CRN2_OK && i < 3; i++)
            if (hipStreamWaitEvent(side[i], fork_ev, 0) != hipSuccess) rc = CRN2_EHIP;
        if (rc != CRN2_OK) return rc;
        cls[3] = side[0];
        cls[2] = side[1];
        cls[1] = side[2];
    }
    if (flags & 2)
        launch_classes<true>(px, offsets, nclusters, list, work, flags & 0xFF01, o, selectors, cls);
    else
        launch_classes<false>(px, offsets, nclusters, list, work, flags & 1, o, selectors, cls);
    if (hipGetLastError() != hipSuccess) rc = CRN2_EHIP;
    if (fork)
        for (int i = 0; i < 3; i++)
            if (hipEventRecord(join[i], side[i]) != hipSuccess || hipStreamWaitEvent(st, join[i], 0) != hipSuccess)
                rc = CRN2_EHIP;
    return rc;
}

// Second pass for clusters of more than 4,096 distinct colours (the LDS pass
// marks them kNotEncoded): reads the texel count once (the call waits for the
// stream there), and when some cluster may hold more colours than the largest
// LDS store, runs dxt1_cluster_big_kernel with stream-ordered global scratch.
int clusters_big_pass(const void* rgba, const uint32_t* offsets, uint32_t nclusters, int flags, void* out,
                      uint8_t* selectors, hipStream_t st)
{
    uint32_t total = 0;
    if (hipMemcpyAsync(&total, offsets + nclusters, 4, hipMemcpyDeviceToHost, st) != hipSuccess ||
        hipStreamSynchronize(st) != hipSuccess)
        return CRN2_EHIP;
    if (total <= kMaxU) return CRN2_OK;      // no cluster can hold more colours than the LDS store
    uint8_t* big = nullptr;
    if (hipMallocAsync((void**)&big, 37 * (size_t)total, st) != hipSuccess) return CRN2_ENOMEM;
    if (flags & 2)
        hipLaunchKernelGGL(dxt1_cluster_big_kernel<true>, dim3(nclusters), dim3(64 * kBigWaves), 0, st,
                           static_cast<const uint32_t*>(rgba), offsets, nclusters, flags & 0xFF01,
                           static_cast<ClusterOut*>(out), selectors, big);
    else
        hipLaunchKernelGGL(dxt1_cluster_big_kernel<false>, dim3(nclusters), dim3(64 * kBigWaves), 0, st,
                           static_cast<const uint32_t*>(rgba), offsets, nclusters, flags & 1,
                           static_cast<ClusterOut*>(out), selectors, big);
    const int rc = hipGetLastError() == hipSuccess ? CRN2_OK : CRN2_EHIP;
    (void)hipFreeAsync(big, st);
    return rc;
}
}  // namespace

extern "C" int crn2_dxt1_clusters_device(const void* rgba, const uint32_t* offsets, uint32_t nclusters, int flags,
                                         void* out, uint8_t* selectors, void* stream)
{
    if (!rgba || !offsets || !out || (flags & ~0xFF03) || ((flags & 0xFF00) && !(flags & 2))) return CRN2_EINVAL;
    if (!nclusters) return CRN2_OK;
    int dev = 0;
    int rc = clusters_init(&dev);
    if (rc != CRN2_OK) return rc;
    hipStream_t st = static_cast<hipStream_t>(stream);
    uint32_t* work = nullptr;      // class counts + 4 lists of nclusters
    if (hipMallocAsync((void**)&work, (kCountWords + 4 * (size_t)nclusters) * sizeof(uint32_t), st) != hipSuccess)
        return CRN2_ENOMEM;
    rc = clusters_run(rgba, offsets, nclusters, flags, out, selectors, st, work, true);
    (void)hipFreeAsync(work, st);
    if (rc == CRN2_OK) rc = clusters_big_pass(rgba, offsets, nclusters, flags, out, selectors, st);
    return rc;
}

extern "C" int crn2_dxt1_clusters_noalloc_device(const void* rgba, const uint32_t* offsets, uint32_t nclusters,
                                                 int flags, void* out, uint8_t* selectors, void* stream)
{
    if (!rgba || !offsets || !out || (flags & ~0xFF03) || ((flags & 0xFF00) && !(flags & 2)) ||
        nclusters > kNoAllocMaxClusters)
        return CRN2_EINVAL;
    if (!nclusters) return CRN2_OK;
    int dev = 0;
    const int rc = clusters_init(&dev);
    if (rc != CRN2_OK) return rc;
    return clusters_run(rgba, offsets, nclusters, flags, out, selectors, static_cast<hipStream_t>(stream),
                        g_noalloc_scratch[dev], false);
}
