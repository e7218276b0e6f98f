// hc_endpoints_gpu.hip -- dxt_hc's colour endpoint codebook on gfx950.
//
// Reference: dxt_hc::determine_color_endpoint_codebook_task
// (crnlib/crn_dxt_hc.cpp:663-754) and dxt_endpoint_refiner::refine /
// optimize_dxt1 (crnlib/crn_dxt_endpoint_refiner.cpp:36-144, 203-302).
// Three launches on the caller's stream:
//   1. crn2_dxt1_clusters_device: the uber endpoint search per cluster, one
//      wave per cluster (dxt1c_gpu.hip), with every texel's selector;
//   2. hc_ep_blocks_kernel, one thread per block: the cluster's four colours
//      (rounded middle colours when the search chose alternate rounding), the
//      block's weight and its 16 nearest-colour selectors;
//   3. hc_ep_refine_kernel, one workgroup per cluster: the refiner -- double
//      least-squares sums (certified to give the start that the reference's
//      texel-order sums give), then up to 8 rounds over the +-1 neighbours of
//      either endpoint scored through per-selector histograms with the
//      selectors fixed; its endpoints replace the search's when their error
//      is lower.
// All float and double expressions keep the reference's types and operation
// order; the library is built with -ffp-contract=off and IEEE division.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "crn2_internal.h"

extern "C" int crn2_dxt1_clusters_device(const void* rgba, const uint32_t* offsets, uint32_t nclusters, int flags,
                                         void* out, uint8_t* selectors, void* stream);

namespace {

constexpr uint32_t kNone = 0xFFFFFFFFu;

struct ClusterRes {          // crn2_dxt1_clusters_device output, 24 bytes per cluster
    uint64_t error;
    uint32_t lo_hi;
    uint32_t nunique;
    uint32_t flags;          // bit 0 reordered, bit 2 alternate rounding, bit 8 not encoded
    uint32_t pad;
};

__constant__ uint8_t k_to_linear[4] = {0, 3, 1, 2};
__constant__ uint8_t k_from_linear[4] = {0, 2, 3, 1};

__device__ inline void unpack565(uint32_t p, int* o)
{
    const uint32_t b = p & 31u, g = (p >> 5) & 63u, r = (p >> 11) & 31u;
    o[0] = (int)((r << 3) | (r >> 2));
    o[1] = (int)((g << 2) | (g >> 4));
    o[2] = (int)((b << 3) | (b >> 2));
}

// dxt1_block::get_block_colors4 (crn_dxt.cpp:247-260)
__device__ inline void colors4(uint32_t c0, uint32_t c1, int (*o)[3])
{
    unpack565(c0, o[0]);
    unpack565(c1, o[1]);
    for (int k = 0; k < 3; k++) {
        o[2][k] = (o[0][k] * 2 + o[1][k]) / 3;
        o[3][k] = (o[1][k] * 2 + o[0][k]) / 3;
    }
}

__device__ inline uint32_t color_distance(bool perceptual, const int* a, const int* b)
{
    const int dr = a[0] - b[0], dg = a[1] - b[1], db = a[2] - b[2];
    return perceptual ? (uint32_t)(8 * dr * dr + 25 * dg * dg + db * db) : (uint32_t)(dr * dr + dg * dg + db * db);
}

// The cluster's colours in linear order (crn_dxt_hc.cpp:692-702).
__device__ inline void cluster_colors(const ClusterRes& r, int (*cv)[3], bool rounded)
{
    int bv[4][3];
    colors4(r.lo_hi & 0xFFFFu, r.lo_hi >> 16, bv);
    for (int i = 0; i < 4; i++)
        for (int k = 0; k < 3; k++) cv[i][k] = bv[k_from_linear[i]][k];
    if (rounded && (r.flags & 4u))
        for (int k = 0; k < 3; k++) {
            cv[1][k] = ((cv[0][k] << 1) + cv[3][k] + 1) / 3;
            cv[2][k] = ((cv[3][k] << 1) + cv[0][k] + 1) / 3;
        }
}

__global__ void __launch_bounds__(256) hc_ep_blocks_kernel(const ClusterRes* __restrict__ res,
                                                           const uint32_t* __restrict__ ofs,
                                                           const uint32_t* __restrict__ block_cluster, uint32_t nblocks,
                                                           const uint8_t* __restrict__ blocks,
                                                           const float* __restrict__ weights,
                                                           const uint8_t* __restrict__ encodings, bool perceptual,
                                                           uint64_t* __restrict__ block_selectors)
{
    const uint32_t b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nblocks) return;
    const uint32_t c = block_cluster[b];
    if (c == kNone || ofs[c + 1] == ofs[c]) return;
    const ClusterRes r = res[c];
    if (r.flags & 256u) return;
    int cv[4][3];
    cluster_colors(r, cv, true);
    const uint32_t endpoint_weight = color_distance(perceptual, cv[0], cv[3]) / 2000;
    const float enc_w = 1.15f + (1.0f - 1.15f) * ((float)encodings[b] / 7.0f);
    const uint32_t w0 = (uint32_t)((float)endpoint_weight * weights[b]);
    const uint32_t wc = w0 < 1 ? 1u : (w0 > 2048 ? 2048u : w0);
    const uint32_t weight = (uint32_t)((float)wc * enc_w);
    const bool reordered = (r.flags & 1u) != 0;
    uint32_t selector = 0;
    const uint8_t* px = blocks + (size_t)b * 64;
    for (int p = 0; p < 16; p++) {
        const int x[3] = {px[4 * p], px[4 * p + 1], px[4 * p + 2]};
        uint32_t best = 0xFFFFFFFFu, sb = 0;
        for (int t = 0; t < 4; t++) {
            const uint32_t s = reordered ? 3u - k_to_linear[t] : k_to_linear[t];
            const uint32_t e = color_distance(perceptual, x, cv[s]);
            if (e < best) {
                sb = s;
                best = e;
            }
        }
        selector = selector << 2 | sb;
    }
    block_selectors[b] = (uint64_t)selector << 32 | weight;
}

__device__ inline int clamp_int(int v, int lo, int hi) { return v < lo ? lo : (v > hi ? hi : v); }

// ------------------------------------------ certified least-squares sums
// The refiners take their start from double sums in texel order (alpha, beta:
// the selector's weights; x: the texel's value), which round once per texel.
// A start is then cut to a grid of 32, 64 or 256 steps, so nearly always any
// order of summation gives the same start.  The kernels sum in parallel and
// certify that: every term is >= 0, so a sum of n terms in any order lies
// within n 2^-53 (relative) of the exact one, two orders within twice that,
// and the interval that this gives for the start is compared after the cut.
// Only when its two ends differ (or the 2 x 2 system may be singular) are the
// sums taken again in texel order, on one wave.
struct FitSums {
    double alpha2, beta2, alphabeta;
};

// Relative distance between a sum of n non-negative terms in texel order and
// one in any other order (2 n 2^-53, and room for the bound's own rounding).
__device__ inline double order_error(uint32_t n) { return ((double)n * 2.5 + 16.0) * 1.1102230246251565e-16; }

// The solution a, b of one component and how far a solution from sums in
// another order can lie from it.  False: the system may be singular.
__device__ inline bool fit_interval(const FitSums& f, double ax, double bx, double e, double& a, double& ra, double& b,
                                    double& rb)
{
    constexpr double kU = 1.1102230246251565e-16;
    a = b = ra = rb = 0.0;
    if (f.beta2 == 0.0) {          // exact: no term of the sum is above zero
        a = ax / f.alpha2;
        ra = a * (2.1 * e + 4 * kU);
        return true;
    }
    if (f.alpha2 == 0.0) {
        b = bx / f.beta2;
        rb = b * (2.1 * e + 4 * kU);
        return true;
    }
    const double g = 2.1 * e + 8 * kU;
    const double p = f.alpha2 * f.beta2, q = f.alphabeta * f.alphabeta;
    const double factor = p - q, ef = (p + q) * g;
    if (!(factor > 2 * ef)) return false;
    const double a1 = ax * f.beta2, a2 = bx * f.alphabeta, b1 = bx * f.alpha2, b2 = ax * f.alphabeta;
    a = (a1 - a2) / factor;
    b = (b1 - b2) / factor;
    ra = ((a1 + a2) * g + fabs(a) * ef) / (factor - ef) * 1.01 + fabs(a) * 8 * kU;
    rb = ((b1 + b2) * g + fabs(b) * ef) / (factor - ef) * 1.01 + fabs(b) * 8 * kU;
    return true;
}

// a solution's component on a grid of `steps` (the reference's float clamp and cut)
__device__ inline int fit_cut(double v, float steps, int limit)
{
    float f = (float)v;
    f = f < 0.0f ? 0.0f : (f > 1.0f ? 1.0f : f);
    return clamp_int((int)(f * steps), 0, limit);
}

// The sums in texel order solved as dxt_endpoint_refiner::refine does.
__device__ inline void fit_solve(const FitSums& f, double ax, double bx, double first, double& a, double& b)
{
    if (f.beta2 == 0.0f) {
        a = ax / f.alpha2;
        b = 0.0;
    } else if (f.alpha2 == 0.0f) {
        a = 0.0;
        b = bx / f.beta2;
    } else {
        const double factor = f.alpha2 * f.beta2 - f.alphabeta * f.alphabeta;
        if (factor != 0.0f) {
            a = (ax * f.beta2 - bx * f.alphabeta) / factor;
            b = (bx * f.alpha2 - ax * f.alphabeta) / factor;
        } else {
            a = b = first;
        }
    }
}

// c added n times to 0, one rounding per addition, without n additions: after
// one addition inside a power of two every further one there moves the sum by
// the same multiple of its last place (a tie rounds to an even sum, and from
// an even sum the same way each time), so each power of two takes a few steps.
// A skip ends one to two additions below the next power of two, so that the
// second sum of the next pair is the first one past it: the first of a pair that
// is skipped on is then a sum of two inside (below the power where ties begin,
// every sum is exact).
__device__ inline double repeat_sum(double c, uint32_t n)
{
    double s = 0.0;
    while (n) {
        const double s1 = s + c;
        if (--n == 0 || s1 == s) return s1;
        const double s2 = s1 + c;
        n--;
        s = s2;
        const uint64_t x1 = __builtin_bit_cast(uint64_t, s1) >> 52, x2 = __builtin_bit_cast(uint64_t, s2) >> 52;
        if (x1 != x2 || !n) continue;
        const double d = s2 - s1;
        if (d == 0.0) return s2;
        const double top = __builtin_bit_cast(double, (x2 + 1) << 52);
        const double steps = floor((top - s2) / d) - 1.0;
        if (steps >= 1.0) {
            const uint32_t k = steps < (double)n ? (uint32_t)steps : n;
            s = s2 + (double)k * d;   // below `top` and a multiple of the last place: exact
            n -= k;
        }
    }
    return s;
}

__device__ inline double shfl_xor_d(double v, int off)
{
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = (uint32_t)__shfl_xor((int)(uint32_t)u, off), hi = (uint32_t)__shfl_xor((int)(u >> 32), off);
    return __builtin_bit_cast(double, (uint64_t)lo | ((uint64_t)hi << 32));
}

__device__ inline uint64_t shfl_xor_u64(uint64_t v, int off)
{
    const uint32_t lo = (uint32_t)__shfl_xor((int)(uint32_t)v, off), hi = (uint32_t)__shfl_xor((int)(v >> 32), off);
    return (uint64_t)lo | ((uint64_t)hi << 32);
}

// The wave's smallest (error, key), errors first.
__device__ inline void wave_min_key(uint64_t& err, uint32_t& key)
{
    for (int off = 32; off > 0; off >>= 1) {
        const uint64_t e = shfl_xor_u64(err, off);
        const uint32_t k = (uint32_t)__shfl_xor((int)key, off);
        if (e < err || (e == err && k < key)) {
            err = e;
            key = k;
        }
    }
}

// optimize_dxt1 (crn_dxt_endpoint_refiner.cpp:203-302), one wave: up to eight
// rounds over the 26 neighbours of either endpoint, one candidate per lane.
// The reference sorts a round's candidates, drops repeats and keeps each
// strict improvement, so a round ends at its smallest error, the smallest
// candidate word on ties.
__device__ void optimize_dxt1(const uint64_t* hist, const uint64_t (*D2)[3], const uint64_t (*DD)[3], bool perceptual,
                              const int* l0, const int* h0, uint32_t& out_lo, uint32_t& out_hi, uint64_t& out_err)
{
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t L0 = (uint32_t)(l0[0] << 11 | l0[1] << 5 | l0[2]);
    uint32_t H0 = (uint32_t)(h0[0] << 11 | h0[1] << 5 | h0[2]);
    const bool preserveL = hist[0] + hist[2] > hist[1] + hist[3];
    const uint32_t pass = lane >> 5, m = lane & 31u;
    const int db = (int)(m / 9) - 1, dg = (int)(m / 3 % 3) - 1, dr = (int)(m % 3) - 1;
    out_err = ~0ull;
    for (uint32_t iterations = 8; iterations; iterations--) {
        const uint32_t E = pass ? H0 : L0, O = pass ? L0 : H0;
        const int b = (int)(E & 31u) + db, g = (int)((E >> 5) & 63u) + dg, r = (int)((E >> 11) & 31u) + dr;
        const uint32_t X = (uint32_t)(r << 11 | g << 5 | b);
        const bool ok = m < 27 && m != 13 && b >= 0 && b <= 31 && g >= 0 && g <= 63 && r >= 0 && r <= 31;
        const uint32_t sol = X > O ? X | O << 16 : O | X << 16;
        uint32_t L = sol & 0xFFFFu, H = sol >> 16;
        if (L == H) {
            uint32_t addL, subH;
            if (!preserveL)
                addL = (~L & 0x1Fu) ? 0x1u : (~L & 0xF800u) ? 0x800u : (~L & 0x7E0u) ? 0x20u : 0u;
            else
                addL = !L ? 0x1u : 0u;
            L = (L + addL) & 0xFFFFu;
            if (preserveL)
                subH = (H & 0x1Fu) ? 0x1u : (H & 0xF800u) ? 0x800u : (H & 0x7E0u) ? 0x20u : 0u;
            else
                subH = H == 0xFFFFu ? 0x1u : 0u;
            H = (H - subH) & 0xFFFFu;
        }
        uint64_t error = ~0ull;
        if (ok) {
            int bc[4][3];
            colors4(L, H, bc);
            error = 0;
            for (int s = 0; s < 4; s++) {
                uint64_t d[3];
                for (int c = 0; c < 3; c++) {
                    const uint64_t v = (uint64_t)bc[s][c];
                    d[c] = hist[s] * v * v - D2[s][c] * v + DD[s][c];
                }
                error += perceptual ? d[0] * 8 + d[1] * 25 + d[2] : d[0] + d[1] + d[2];
            }
        }
        uint64_t e = error;
        uint32_t key = ok ? sol : 0xFFFFFFFFu;
        wave_min_key(e, key);
        if (e >= out_err) break;
        // the lane that holds the kept candidate gives its (adjusted) endpoints
        const uint32_t src = (uint32_t)__builtin_ctzll(__ballot(ok && error == e && sol == key));
        const uint32_t lh = (uint32_t)__shfl((int)(L | H << 16), (int)src);
        out_lo = L0 = lh & 0xFFFFu;
        out_hi = H0 = lh >> 16;
        out_err = e;
        if (!e) return;
    }
}

// One workgroup per cluster.  The pass over the texels bounds it; it was a
// serial chain on one wave (2048^2 DXT1 chain at quality 128: 4.07 ms, the
// largest cluster's texels one after another), now 0.18 ms.
constexpr uint32_t kRefineThreads = 256;

__global__ void __launch_bounds__(kRefineThreads) hc_ep_refine_kernel(
    const uint32_t* __restrict__ px_all, const uint32_t* __restrict__ ofs, uint32_t nclusters,
    const ClusterRes* __restrict__ res, const uint8_t* __restrict__ sel_all, bool perceptual,
    uint32_t* __restrict__ endpoints, uint32_t* __restrict__ color_values, uint32_t* __restrict__ not_encoded)
{
    constexpr uint32_t kWaves = kRefineThreads / 64;
    __shared__ uint64_t s_int[kWaves][4][7];   // per wave and selector: texels, value sums, sums of squares
    __shared__ double s_ab[kWaves][6];         // per wave: sums of alpha x, beta x
    const uint32_t c = blockIdx.x, tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    if (c >= nclusters) return;
    const uint32_t o = ofs[c], n = ofs[c + 1] - o;
    if (tid == 0) endpoints[c] = 0;
    if (tid < 4) color_values[4 * c + tid] = 0;
    if (!n) return;
    const ClusterRes r = res[c];
    if (r.flags & 256u) {
        if (tid == 0) atomicAdd(not_encoded, 1u);
        return;
    }
    if (tid == 0) {
        int cv[4][3];
        cluster_colors(r, cv, false);
        for (int i = 0; i < 4; i++)
            color_values[4 * c + i] =
                (uint32_t)cv[i][0] | (uint32_t)cv[i][1] << 8 | (uint32_t)cv[i][2] << 16 | 0xFF000000u;
    }
    // dxt_endpoint_refiner::refine (crn_dxt_endpoint_refiner.cpp:36-144)
    const uint32_t* px = px_all + o;
    const uint8_t* sel = sel_all + o;
    double alpha[4], beta[4];
    for (int s = 0; s < 4; s++) {
        const double k = (double)((float)k_to_linear[s] * 1.0f / 3.0f);
        alpha[s] = 1.0f - k;
        beta[s] = k;
    }
    uint64_t hist[4] = {0, 0, 0, 0}, D2[4][3], DD[4][3];
    double ax[3] = {0, 0, 0}, bx[3] = {0, 0, 0};
    {
        uint32_t cnt[4] = {0, 0, 0, 0}, sum[4][3];
        for (int s = 0; s < 4; s++)
            for (int k = 0; k < 3; k++) {
                sum[s][k] = 0;
                DD[s][k] = 0;
            }
        // a value sum stays below 2^32: at most n / 256 < 2^24 texels of 255 per thread
        for (uint32_t i = tid; i < n; i += kRefineThreads) {
            const uint32_t p = px[i], t = sel[i] & 3u;
            const double al = t == 0 ? alpha[0] : t == 1 ? alpha[1] : t == 2 ? alpha[2] : alpha[3];
            const double be = t == 0 ? beta[0] : t == 1 ? beta[1] : t == 2 ? beta[2] : beta[3];
            const uint32_t pc[3] = {p & 0xFFu, (p >> 8) & 0xFFu, (p >> 16) & 0xFFu};
            for (int q = 0; q < 3; q++) {
                const double x = (double)((float)pc[q] * 1.0f / 255.0f);
                ax[q] += al * x;
                bx[q] += be * x;
            }
#pragma unroll
            for (uint32_t s = 0; s < 4; s++) {
                const uint32_t on = t == s ? 0xFFFFFFFFu : 0u;
                cnt[s] += on & 1u;
                for (int q = 0; q < 3; q++) {
                    sum[s][q] += pc[q] & on;
                    DD[s][q] += (pc[q] * pc[q]) & on;
                }
            }
        }
        for (int s = 0; s < 4; s++) {
            uint64_t v[7] = {cnt[s], sum[s][0], sum[s][1], sum[s][2], DD[s][0], DD[s][1], DD[s][2]};
            for (int q = 0; q < 7; q++) {
                for (int off = 32; off > 0; off >>= 1) v[q] += shfl_xor_u64(v[q], off);
                if (lane == 0) s_int[wave][s][q] = v[q];
            }
        }
        for (int q = 0; q < 3; q++) {
            for (int off = 32; off > 0; off >>= 1) {
                ax[q] += shfl_xor_d(ax[q], off);
                bx[q] += shfl_xor_d(bx[q], off);
            }
            if (lane == 0) {
                s_ab[wave][q] = ax[q];
                s_ab[wave][3 + q] = bx[q];
            }
        }
    }
    __syncthreads();
    if (wave) return;
    for (int q = 0; q < 3; q++) {
        ax[q] = bx[q] = 0;
        for (uint32_t w = 0; w < kWaves; w++) {
            ax[q] += s_ab[w][q];
            bx[q] += s_ab[w][3 + q];
        }
    }
    FitSums f{0, 0, 0};
    for (int s = 0; s < 4; s++) {
        uint64_t v[7] = {0, 0, 0, 0, 0, 0, 0};
        for (uint32_t w = 0; w < kWaves; w++)
            for (int q = 0; q < 7; q++) v[q] += s_int[w][s][q];
        hist[s] = v[0];
        for (int q = 0; q < 3; q++) {
            D2[s][q] = 2 * v[1 + q];
            DD[s][q] = v[4 + q];
        }
        f.alpha2 += (double)v[0] * (alpha[s] * alpha[s]);
        f.beta2 += (double)v[0] * (beta[s] * beta[s]);
        f.alphabeta += (double)v[0] * (alpha[s] * beta[s]);
    }
    int l0[3], h0[3];
    bool sure = true;
    const double e = order_error(n);
    for (int q = 0; q < 3; q++) {
        const float steps = q == 1 ? 64.0f : 32.0f;
        const int limit = q == 1 ? 63 : 31;
        double a, b, ra, rb;
        sure &= fit_interval(f, ax[q], bx[q], e, a, ra, b, rb);
        l0[q] = fit_cut(a - ra, steps, limit);
        h0[q] = fit_cut(b - rb, steps, limit);
        sure &= l0[q] == fit_cut(a + ra, steps, limit) && h0[q] == fit_cut(b + rb, steps, limit);
    }
    if (!sure) {
        double first[3];
        for (int q = 0; q < 3; q++) {
            first[q] = (double)((float)((px[0] >> (8 * q)) & 0xFFu) * 1.0f / 255.0f);
            ax[q] = bx[q] = 0;
        }
        f = FitSums{0, 0, 0};
        uint32_t one = 4;
        for (uint32_t s = 0; s < 4; s++)
            if (hist[s] == n) one = s;
        if (r.nunique == 1 && one < 4) {
            // one colour on one middle selector (a singular system): every sum
            // is of one repeated term; lanes 0-8 take a sum each
            const uint32_t q = lane % 3;
            const double al = one == 0 ? alpha[0] : one == 1 ? alpha[1] : one == 2 ? alpha[2] : alpha[3];
            const double be = one == 0 ? beta[0] : one == 1 ? beta[1] : one == 2 ? beta[2] : beta[3];
            const double x = q == 0 ? first[0] : q == 1 ? first[1] : first[2];
            const double t = lane < 3 ? (q == 0 ? al * al : q == 1 ? be * be : al * be) : lane < 6 ? al * x : be * x;
            const double v = lane < 9 ? repeat_sum(t, n) : 0.0;
            auto from = [&](int l) {
                const uint64_t u = __builtin_bit_cast(uint64_t, v);
                return __builtin_bit_cast(double, (uint64_t)(uint32_t)__shfl((int)(uint32_t)u, l) |
                                                      ((uint64_t)(uint32_t)__shfl((int)(u >> 32), l) << 32));
            };
            f = FitSums{from(0), from(1), from(2)};
            for (int k = 0; k < 3; k++) {
                ax[k] = from(3 + k);
                bx[k] = from(6 + k);
            }
        } else
        // in texel order; every lane holds the sums, 64 texels per load
        for (uint32_t i0 = 0; i0 < n; i0 += 64) {
            const uint32_t mine =
                i0 + lane < n ? (px[i0 + lane] & 0x00FFFFFFu) | ((uint32_t)(sel[i0 + lane] & 3u) << 24) : 0u;
            const uint32_t m = min(64u, n - i0);
            for (uint32_t t = 0; t < m; t++) {
                const uint32_t p = (uint32_t)__builtin_amdgcn_readlane((int)mine, (int)t);
                const uint32_t s = p >> 24;
                const double k = (double)((float)k_to_linear[s] * 1.0f / 3.0f);
                const double al = 1.0f - k, be = k;
                f.alpha2 += al * al;
                f.beta2 += be * be;
                f.alphabeta += al * be;
                for (int q = 0; q < 3; q++) {
                    const double x = (double)((float)((p >> (8 * q)) & 0xFFu) * 1.0f / 255.0f);
                    ax[q] += al * x;
                    bx[q] += be * x;
                }
            }
        }
        for (int q = 0; q < 3; q++) {
            double a, b;
            fit_solve(f, ax[q], bx[q], first[q], a, b);
            l0[q] = fit_cut(a, q == 1 ? 64.0f : 32.0f, q == 1 ? 63 : 31);
            h0[q] = fit_cut(b, q == 1 ? 64.0f : 32.0f, q == 1 ? 63 : 31);
        }
    }
    uint32_t lo = 0, hi = 0;
    uint64_t err;
    optimize_dxt1(hist, D2, DD, perceptual, l0, h0, lo, hi, err);
    if (lane == 0) endpoints[c] = err < r.error ? (lo | hi << 16) : r.lo_hi;
}

// ------------------------------------------------------------ alpha (H.8)
// dxt_hc::determine_alpha_endpoint_codebook_task (crn_dxt_hc.cpp:1014-1130,
// without ETC colour blocks) for one alpha channel:
//   hc_alpha_search_kernel, one wave per cluster: the uber dxt5_endpoint_
//     optimizer (crn_dxt5a.cpp:40-262, 8-value blocks only) over the cluster's
//     values -- distinct values in first-appearance order with their counts
//     (LDS tables over the 256 values), every distinct pair in that order,
//     then the +-16 box around the current best (centre re-read at every
//     step); each candidate is scored by all lanes at once (first minimum per
//     value, wave sum) and kept on a strict improvement, a zero error ends the
//     search; canonical order with the eight-value invert table;
//   hc_alpha_blocks_kernel, one thread per block: values in linear order,
//     encoding weights from the endpoint spread, 3-bit nearest-value selectors;
//   hc_alpha_refine_kernel, one workgroup per cluster: the DXT5 refiner
//     (certified least squares on the alpha values, then the canonical
//     23 x 23 box scored through per-selector histograms).
struct AlphaRes {
    uint64_t error;
    uint32_t first, second, reordered, pad;
};

__constant__ uint8_t k5_to_linear[8] = {0, 7, 1, 2, 3, 4, 5, 6};
__constant__ uint8_t k5_from_linear[8] = {0, 2, 3, 4, 5, 6, 7, 1};
__constant__ uint8_t k5_eight_invert[8] = {1, 0, 7, 6, 5, 4, 3, 2};

__device__ inline void values8(uint32_t l, uint32_t h, uint32_t* v)
{
    v[0] = l;
    v[1] = h;
    for (uint32_t j = 2; j < 8; j++) v[j] = (l * (8 - j) + h * (j - 1)) / 7;
}

// dxt5_block::get_block_values (crn_dxt.cpp:369-455)
__device__ inline void alpha_values_of(uint32_t l, uint32_t h, uint32_t* v)
{
    if (l > h) {
        values8(l, h, v);
    } else {
        v[0] = l;
        v[1] = h;
        for (uint32_t j = 2; j < 6; j++) v[j] = (l * (6 - j) + h * (j - 1)) / 5;
        v[6] = 0;
        v[7] = 255;
    }
}

struct AlphaLds {
    uint32_t count[256];
    uint32_t first[256];
    uint32_t uval[256];
    uint32_t uw[256];
    uint32_t rank[256];
    uint8_t trial[256];
    uint8_t best[256];
};

__device__ inline uint64_t wave_sum64(uint64_t v)
{
    for (int off = 32; off > 0; off >>= 1) {
        const uint32_t lo = (uint32_t)__shfl_xor((int)(uint32_t)v, off), hi = (uint32_t)__shfl_xor((int)(v >> 32), off);
        v += (uint64_t)lo | ((uint64_t)hi << 32);
    }
    return v;
}

__global__ void __launch_bounds__(64) hc_alpha_search_kernel(const uint8_t* __restrict__ vals_all,
                                                             const uint32_t* __restrict__ ofs, uint32_t nclusters,
                                                             AlphaRes* __restrict__ res, uint8_t* __restrict__ sel_all)
{
    __shared__ AlphaLds L;
    const uint32_t c = blockIdx.x, lane = threadIdx.x;
    const uint32_t o = ofs[c], n = ofs[c + 1] - o;
    if (!n) return;
    const uint8_t* vals = vals_all + o;
    for (uint32_t v = lane; v < 256; v += 64) {
        L.count[v] = 0;
        L.first[v] = 0xFFFFFFFFu;
    }
    __syncthreads();
    for (uint32_t i = lane; i < n; i += 64) {
        atomicAdd(&L.count[vals[i]], 1u);
        atomicMin(&L.first[vals[i]], i);
    }
    __syncthreads();
    // rank of each present value by first appearance
    for (uint32_t v = lane; v < 256; v += 64) {
        if (!L.count[v]) continue;
        const uint32_t f = L.first[v];
        uint32_t r = 0;
        for (uint32_t u = 0; u < 256; u++) r += (L.count[u] && L.first[u] < f) ? 1u : 0u;
        L.rank[v] = r;
        L.uval[r] = v;
        L.uw[r] = L.count[v];
    }
    __syncthreads();
    uint32_t nu = 0;
    for (uint32_t v = 0; v < 256; v++) nu += L.count[v] ? 1u : 0u;
    AlphaRes out;
    out.pad = 0;
    if (nu == 1) {
        out.error = 0;
        out.first = out.second = L.uval[0];
        out.reordered = 0;
        if (lane == 0) res[c] = out;
        for (uint32_t i = lane; i < n; i += 64) sel_all[o + i] = 0;
        return;
    }
    uint64_t best_err = ~0ull;
    uint32_t best_first = 0, best_second = 0;
    bool done = false;
    // evaluate_solution (crn_dxt5a.cpp:198-262) with the 8-value palette only
    auto evaluate = [&](uint32_t lo, uint32_t hi) {
        uint32_t pal[8];
        values8(lo, hi, pal);
        uint64_t part = 0;
        for (uint32_t i = lane; i < nu; i += 64) {
            const int val = (int)L.uval[i], w = (int)L.uw[i];
            uint32_t best = 0xFFFFFFFFu, bsel = 0;
            for (uint32_t j = 0; j < 8; j++) {
                int e = val - (int)pal[j];
                e = e * e * w;
                if ((uint32_t)e < best) {
                    best = (uint32_t)e;
                    bsel = j;
                    if (!best) break;
                }
            }
            L.trial[i] = (uint8_t)bsel;
            part += best;
        }
        const uint64_t err = wave_sum64(part);
        if (err < best_err) {
            best_err = err;
            best_first = lo;
            best_second = hi;
            for (uint32_t i = lane; i < nu; i += 64) L.best[i] = L.trial[i];
            if (!err) done = true;
        }
    };
    for (uint32_t i = 0; i + 1 < nu && !done; i++)
        for (uint32_t j = i + 1; j < nu && !done; j++) evaluate(L.uval[i], L.uval[j]);
    if (best_err && !done) {
        for (int dl = -16; dl <= 16 && !done; dl++) {
            const int l = (int)best_first + dl;
            if (l < 0) continue;
            if (l > 255) break;
            for (int dh = -16; dh <= 16 && !done; dh++) {
                const int h = (int)best_second + dh;
                if (h < 0) continue;
                if (h > 255) break;
                evaluate((uint32_t)l, (uint32_t)h);
            }
        }
    }
    // canonical order (crn_dxt5a.cpp:151-184), 8-value blocks
    uint32_t f = best_first, sc = best_second, reordered = 0;
    bool zero = f == sc, invert = false;
    if (!zero && f <= sc) {
        const uint32_t t = f;
        f = sc;
        sc = t;
        reordered = 1;
        invert = true;
    }
    __syncthreads();
    for (uint32_t i = lane; i < n; i += 64) {
        const uint32_t u = L.rank[vals[i]];
        uint32_t s = zero ? 0u : L.best[u];
        if (invert) s = k5_eight_invert[s];
        sel_all[o + i] = (uint8_t)s;
    }
    out.error = best_err;
    out.first = f;
    out.second = sc;
    out.reordered = reordered;
    if (lane == 0) res[c] = out;
}

__global__ void __launch_bounds__(256) hc_alpha_blocks_kernel(const AlphaRes* __restrict__ res,
                                                              const uint32_t* __restrict__ ofs,
                                                              const uint32_t* __restrict__ block_cluster,
                                                              uint32_t nblocks, const uint8_t* __restrict__ block_vals,
                                                              const uint8_t* __restrict__ encodings,
                                                              uint64_t* __restrict__ block_selectors)
{
    const uint32_t b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nblocks) return;
    const uint32_t c = block_cluster[b];
    if (c == kNone || ofs[c + 1] == ofs[c]) return;
    const AlphaRes r = res[c];
    uint32_t bv[8], av[8];
    alpha_values_of(r.first, r.second, bv);
    for (int i = 0; i < 8; i++) av[i] = bv[k5_from_linear[i]];
    const int delta = (int)r.first - (int)r.second;
    const uint32_t dd = (uint32_t)(delta * delta >> 3);
    const uint32_t ew = dd < 1 ? 1u : (dd > 2048 ? 2048u : dd);
    const uint32_t weight = (uint32_t)((float)ew * (1.15f + (1.0f - 1.15f) * ((float)encodings[b] / 7.0f)));
    uint64_t selector = 0;
    const uint8_t* v = block_vals + (size_t)b * 16;
    for (int p = 0; p < 16; p++) {
        uint32_t best = 0xFFFFFFFFu, sb = 0;
        for (int t = 0; t < 8; t++) {
            const uint32_t s = r.reordered ? 7u - k5_to_linear[t] : k5_to_linear[t];
            const int d = (int)v[p] - (int)av[s];
            const uint32_t e = (uint32_t)(d >= 0 ? d : -d);
            if (e < best) {
                sb = s;
                best = e;
            }
        }
        selector = selector << 3 | sb;
    }
    block_selectors[b] = selector << 16 | weight;
}

// One workgroup per cluster: the texels' (selector, value) pairs into a
// histogram in LDS, from which every sum follows (the least-squares ones
// certified as in hc_ep_refine_kernel), then the 23 x 23 box one candidate
// per lane.  It was one serial chain of double sums per cluster, as long as
// the largest cluster (1024^2 DXT5 chain at quality 128, one cluster of most
// of the opaque texels: 102 ms), now
// 0.15 ms.
__global__ void __launch_bounds__(kRefineThreads) hc_alpha_refine_kernel(
    const uint8_t* __restrict__ vals_all, const uint32_t* __restrict__ ofs, uint32_t nclusters,
    const AlphaRes* __restrict__ res, const uint8_t* __restrict__ sel_all, uint32_t* __restrict__ endpoints,
    uint32_t* __restrict__ alpha_values, uint32_t* __restrict__ refined_values)
{
    __shared__ uint32_t s_bin[8 * 256];
    __shared__ uint64_t s_int[8][3];
    __shared__ double s_ab[8][2];
    const uint32_t c = blockIdx.x, tid = threadIdx.x, lane = tid & 63u;
    if (c >= nclusters) return;
    const uint32_t o = ofs[c], n = ofs[c + 1] - o;
    if (tid == 0) {
        endpoints[c] = 0;
        alpha_values[2 * c] = alpha_values[2 * c + 1] = 0;
        refined_values[2 * c] = refined_values[2 * c + 1] = 0;
    }
    if (!n) return;
    const AlphaRes r = res[c];
    uint32_t bv[8], av[8];
    alpha_values_of(r.first, r.second, bv);
    for (int i = 0; i < 8; i++) av[i] = bv[k5_from_linear[i]];
    if (tid == 0) {
        alpha_values[2 * c] = av[0] | av[1] << 8 | av[2] << 16 | av[3] << 24;
        alpha_values[2 * c + 1] = av[4] | av[5] << 8 | av[6] << 16 | av[7] << 24;
    }
    // dxt_endpoint_refiner::refine, DXT5 selectors (crn_dxt_endpoint_refiner.cpp:36-144)
    const uint8_t* vals = vals_all + o;
    const uint8_t* sel = sel_all + o;
    for (uint32_t i = tid; i < 8 * 256; i += kRefineThreads) s_bin[i] = 0;
    __syncthreads();
    // four texels per lane; one LDS add where a lane's four are the same pair,
    // and one per wave where the whole wave's are (flat areas)
    const uint32_t quads = n / 4;
    for (uint32_t q0 = 0; q0 < quads; q0 += kRefineThreads) {
        const uint32_t q = q0 + tid;
        uint32_t v = 0, t = 0;
        if (q < quads) {
            __builtin_memcpy(&v, vals + 4 * (size_t)q, 4);
            __builtin_memcpy(&t, sel + 4 * (size_t)q, 4);
        }
        t &= 0x07070707u;
        const uint32_t k0 = (t & 7u) << 8 | (v & 0xFFu);
        const bool same = q < quads && v == (v & 0xFFu) * 0x01010101u && t == (t & 0xFFu) * 0x01010101u;
        const uint32_t kw = (uint32_t)__builtin_amdgcn_readfirstlane((int)k0);
        if (__all(same && k0 == kw)) {
            if (lane == 0) atomicAdd(&s_bin[kw], 256u);
        } else if (same) {
            atomicAdd(&s_bin[k0], 4u);
        } else if (q < quads) {
            for (int i = 0; i < 4; i++) atomicAdd(&s_bin[((t >> (8 * i)) & 7u) << 8 | ((v >> (8 * i)) & 0xFFu)], 1u);
        }
    }
    if (tid < n - 4 * quads) {
        const uint32_t i = 4 * quads + tid;
        atomicAdd(&s_bin[(uint32_t)(sel[i] & 7u) << 8 | vals[i]], 1u);
    }
    __syncthreads();
    // 32 lanes per selector, eight values each
    {
        const uint32_t s = tid >> 5, sub = tid & 31u;
        const double k = (double)((float)k5_to_linear[s] * 1.0f / 7.0f);
        const double alpha = 1.0f - k, beta = k;
        uint64_t cnt = 0, sum = 0, sq = 0;
        double ax = 0, bx = 0;
        for (uint32_t j = 0; j < 8; j++) {
            const uint32_t a = sub + 32 * j;
            const uint64_t m = s_bin[s << 8 | a];
            const double x = (double)((float)a / 255.0f);
            cnt += m;
            sum += m * a;
            sq += m * a * a;
            ax += (double)m * (alpha * x);
            bx += (double)m * (beta * x);
        }
        for (int off = 16; off > 0; off >>= 1) {
            cnt += shfl_xor_u64(cnt, off);
            sum += shfl_xor_u64(sum, off);
            sq += shfl_xor_u64(sq, off);
            ax += shfl_xor_d(ax, off);
            bx += shfl_xor_d(bx, off);
        }
        if (sub == 0) {
            s_int[s][0] = cnt;
            s_int[s][1] = sum;
            s_int[s][2] = sq;
            s_ab[s][0] = ax;
            s_ab[s][1] = bx;
        }
    }
    __syncthreads();
    if (tid >= 64) return;
    uint64_t hist[8], D2[8], DD[8];
    FitSums f{0, 0, 0};
    double ax = 0, bx = 0;
    for (int s = 0; s < 8; s++) {
        const double k = (double)((float)k5_to_linear[s] * 1.0f / 7.0f);
        const double alpha = 1.0f - k, beta = k;
        hist[s] = s_int[s][0];
        D2[s] = 2 * s_int[s][1];
        DD[s] = s_int[s][2];
        f.alpha2 += (double)hist[s] * (alpha * alpha);
        f.beta2 += (double)hist[s] * (beta * beta);
        f.alphabeta += (double)hist[s] * (alpha * beta);
        ax += s_ab[s][0];
        bx += s_ab[s][1];
    }
    double a, b, ra, rb;
    bool sure = fit_interval(f, ax, bx, order_error(n), a, ra, b, rb);
    uint32_t L0 = (uint32_t)fit_cut(a - ra, 256.0f, 255), H0 = (uint32_t)fit_cut(b - rb, 256.0f, 255);
    sure &= L0 == (uint32_t)fit_cut(a + ra, 256.0f, 255) && H0 == (uint32_t)fit_cut(b + rb, 256.0f, 255);
    if (!sure) {
        f = FitSums{0, 0, 0};
        ax = bx = 0;
        for (uint32_t i0 = 0; i0 < n; i0 += 64) {
            const uint32_t mine = i0 + lane < n ? ((uint32_t)sel[i0 + lane] & 7u) | ((uint32_t)vals[i0 + lane] << 8) : 0u;
            const uint32_t m = min(64u, n - i0);
            for (uint32_t t = 0; t < m; t++) {
                const uint32_t sv = (uint32_t)__builtin_amdgcn_readlane((int)mine, (int)t);
                const double k = (double)((float)k5_to_linear[sv & 7u] * 1.0f / 7.0f);
                const double alpha = 1.0f - k, beta = k, x = (double)((float)(sv >> 8) / 255.0f);
                f.alpha2 += alpha * alpha;
                f.beta2 += beta * beta;
                f.alphabeta += alpha * beta;
                ax += alpha * x;
                bx += beta * x;
            }
        }
        fit_solve(f, ax, bx, (double)((float)vals[0] / 255.0f), a, b);
        L0 = (uint32_t)fit_cut(a, 256.0f, 255);
        H0 = (uint32_t)fit_cut(b, 256.0f, 255);
    }
    // optimize_dxt5 (crn_dxt_endpoint_refiner.cpp:146-201): the start, then
    // the box in (L, H) order; the first smallest error is kept
    auto canon = [](uint32_t L, uint32_t H) -> uint32_t {
        return L == H ? (H ? ((H - 1) << 8 | L) : 1u) : (L > H ? (H << 8 | L) : (L << 8 | H));
    };
    auto score = [&](uint32_t sol) -> uint64_t {
        uint32_t v[8];
        values8(sol & 0xFFu, sol >> 8, v);
        uint64_t error = 0;
        for (int s = 0; s < 8; s++) error += hist[s] * v[s] * v[s] - D2[s] * v[s] + DD[s];
        return error;
    };
    const uint32_t minL = L0 <= 11 ? 0 : L0 - 11, maxL = L0 >= 244 ? 255 : L0 + 11;
    const uint32_t minH = H0 <= 11 ? 0 : H0 - 11, maxH = H0 >= 244 ? 255 : H0 + 11;
    const uint32_t nh = maxH - minH + 1, cands = (maxL - minL + 1) * nh;
    uint64_t rerr = lane == 0 ? score(canon(L0, H0)) : ~0ull;
    uint32_t key = lane == 0 ? 0u : 0xFFFFFFFFu;   // 0: the start; 1 + index: a candidate of the box
    for (uint32_t i = lane; i < cands; i += 64) {
        const uint32_t L = minL + i / nh, H = minH + i % nh;
        if (!((maxH < L || L <= H || H < minL) && (L != L0 || H != H0) && (L != H0 || H != L0))) continue;
        const uint64_t error = score(canon(L, H));
        if (error < rerr) {
            rerr = error;
            key = 1 + i;
        }
    }
    wave_min_key(rerr, key);
    const uint32_t sol = key ? canon(minL + (key - 1) / nh, minH + (key - 1) % nh) : canon(L0, H0);
    const bool refined = rerr < r.error;
    uint32_t first = r.first, second = r.second;
    if (refined) {
        first = sol & 0xFFu;
        second = sol >> 8;
        alpha_values_of(first, second, bv);
        for (int i = 0; i < 8; i++) av[i] = bv[k5_from_linear[i]];
    }
    if (lane == 0) {
        refined_values[2 * c] = av[0] | av[1] << 8 | av[2] << 16 | av[3] << 24;
        refined_values[2 * c + 1] = av[4] | av[5] << 8 | av[6] << 16 | av[7] << 24;
        endpoints[c] = first | second << 8 | (refined ? 1u : 0u) << 16;
    }
}

inline uint32_t grid1(uint64_t n, uint32_t tb) { return (uint32_t)((n + tb - 1) / tb); }

}  // namespace

extern "C" int crn2_hc_color_endpoints_device(const void* cluster_px, const uint32_t* cluster_ofs, uint32_t nclusters,
                                              uint32_t total_px, const uint32_t* block_cluster, uint32_t nblocks,
                                              const void* blocks, const float* block_weights,
                                              const uint8_t* block_encodings, int perceptual, uint32_t* endpoints,
                                              void* color_values, uint64_t* block_selectors, uint32_t* not_encoded,
                                              void* stream)
{
    if (!nclusters) return CRN2_OK;
    if (!cluster_px || !cluster_ofs || !endpoints || !color_values || !not_encoded || (perceptual & ~1) ||
        (nblocks && (!block_cluster || !blocks || !block_weights || !block_encodings || !block_selectors)))
        return CRN2_EINVAL;
    hipStream_t s = static_cast<hipStream_t>(stream);
    ClusterRes* res = nullptr;
    uint8_t* sel = nullptr;
    if (hipMallocAsync(reinterpret_cast<void**>(&res), (size_t)nclusters * sizeof(ClusterRes), s) != hipSuccess)
        return CRN2_ENOMEM;
    if (hipMallocAsync(reinterpret_cast<void**>(&sel), (size_t)total_px + 1, s) != hipSuccess) {
        (void)hipFreeAsync(res, s);
        return CRN2_ENOMEM;
    }
    int rc = CRN2_OK;
    if (hipMemsetAsync(not_encoded, 0, 4, s) != hipSuccess) rc = CRN2_EHIP;
    if (rc == CRN2_OK) rc = crn2_dxt1_clusters_device(cluster_px, cluster_ofs, nclusters, perceptual, res, sel, stream);
    if (rc == CRN2_OK && nblocks) {
        hipLaunchKernelGGL(hc_ep_blocks_kernel, dim3(grid1(nblocks, 256)), dim3(256), 0, s, res, cluster_ofs,
                           block_cluster, nblocks, static_cast<const uint8_t*>(blocks), block_weights, block_encodings,
                           perceptual != 0, block_selectors);
        if (hipGetLastError() != hipSuccess) rc = CRN2_EHIP;
    }
    if (rc == CRN2_OK) {
        hipLaunchKernelGGL(hc_ep_refine_kernel, dim3(nclusters), dim3(kRefineThreads), 0, s,
                           static_cast<const uint32_t*>(cluster_px), cluster_ofs, nclusters, res, sel, perceptual != 0,
                           endpoints, static_cast<uint32_t*>(color_values), not_encoded);
        if (hipGetLastError() != hipSuccess) rc = CRN2_EHIP;
    }
    (void)hipFreeAsync(sel, s);
    (void)hipFreeAsync(res, s);
    return rc;
}

extern "C" int crn2_hc_alpha_endpoints_device(const void* cluster_vals, const uint32_t* cluster_ofs, uint32_t nclusters,
                                              uint32_t total_vals, const uint32_t* block_cluster, uint32_t nblocks,
                                              const void* block_vals, const uint8_t* block_encodings,
                                              uint32_t* endpoints, void* alpha_values, void* refined_values,
                                              uint64_t* block_selectors, void* stream)
{
    if (!nclusters) return CRN2_OK;
    if (!cluster_vals || !cluster_ofs || !endpoints || !alpha_values || !refined_values ||
        (nblocks && (!block_cluster || !block_vals || !block_encodings || !block_selectors)))
        return CRN2_EINVAL;
    hipStream_t s = static_cast<hipStream_t>(stream);
    AlphaRes* res = nullptr;
    uint8_t* sel = nullptr;
    if (hipMallocAsync(reinterpret_cast<void**>(&res), (size_t)nclusters * sizeof(AlphaRes), s) != hipSuccess)
        return CRN2_ENOMEM;
    if (hipMallocAsync(reinterpret_cast<void**>(&sel), (size_t)total_vals + 1, s) != hipSuccess) {
        (void)hipFreeAsync(res, s);
        return CRN2_ENOMEM;
    }
    int rc = CRN2_OK;
    hipLaunchKernelGGL(hc_alpha_search_kernel, dim3(nclusters), dim3(64), 0, s, static_cast<const uint8_t*>(cluster_vals),
                       cluster_ofs, nclusters, res, sel);
    if (hipGetLastError() != hipSuccess) rc = CRN2_EHIP;
    if (rc == CRN2_OK && nblocks) {
        hipLaunchKernelGGL(hc_alpha_blocks_kernel, dim3(grid1(nblocks, 256)), dim3(256), 0, s, res, cluster_ofs,
                           block_cluster, nblocks, static_cast<const uint8_t*>(block_vals), block_encodings,
                           block_selectors);
        if (hipGetLastError() != hipSuccess) rc = CRN2_EHIP;
    }
    if (rc == CRN2_OK) {
        hipLaunchKernelGGL(hc_alpha_refine_kernel, dim3(nclusters), dim3(kRefineThreads), 0, s,
                           static_cast<const uint8_t*>(cluster_vals), cluster_ofs, nclusters, res, sel, endpoints,
                           static_cast<uint32_t*>(alpha_values), static_cast<uint32_t*>(refined_values));
        if (hipGetLastError() != hipSuccess) rc = CRN2_EHIP;
    }
    (void)hipFreeAsync(sel, s);
    (void)hipFreeAsync(res, s);
    return rc;
}
