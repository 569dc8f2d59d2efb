// raster.hip -- tile compositing (replaces gs_rasterize_forward,
// gs_rasterize_backward and gs_rasterize_depth, splatting/rasterize.py:28-290).
//
// Up to 16 channels the forward (k_raster_fwd) has one 256-lane workgroup (4
// wave64) per 16x16 tile; wave w owns the 8x8 pixel quadrant (w&1, w>>1).  The
// tile's depth-sorted Gaussians are staged through LDS in batches (16-byte
// pieces, read as broadcasts).  While staging, each lane tests its Gaussian's
// alpha >= 1/255 ellipse against the four quadrants (exact minimum of the conic
// form over each quadrant's pixel centres, with a margin that covers the float32
// rounding of the per-pixel power), and the workgroup publishes per quadrant a
// bit mask of the Gaussians that can touch it.  Each wave compacts its
// quadrant's bits into a list of record offsets and walks it in list order,
// reading each Gaussian's records while the previous one is evaluated.  Skipped
// pairs are exactly pairs whose alpha is below 1/255, which the reference also
// skips, so every output is unchanged.
//
// Forward: per-pixel front-to-back compositing as rasterize.py:60-96 (same
// skips, same termination before compositing the splat that would drop T
// below 1e-4), branch-free per pair; a wave stops once its 64 pixels have
// terminated and the workgroup stops loading once all 256 have.  Small frames
// give every quadrant a workgroup (k_raster_fwd_split: three waves evaluate
// alphas, one composites); blocks of 17 to 32 channels form the channel sums on
// the matrix cores (k_raster_fwd_mx).
// Backward: back-to-front replay (rasterize.py:147-220) from the largest
// n_contrib of each quadrant; the reference issues one atomic per (pixel,
// Gaussian, component).  Up to four channels (k_raster_bwd) a workgroup has a
// tile and its lanes are pixels: a pair's gradient terms are summed over the
// wave with cross-row swaps and DPP row operations, two Gaussians per
// reduction, and after the batch one lane per Gaussian adds the four waves'
// slots and issues one global atomic per (Gaussian, tile, component).  From
// five channels on (k_raster_bwd_wide) a workgroup is one wave with one
// quadrant, the lanes are Gaussians and the channel work runs on the matrix
// cores.
#include <algorithm>
#include <type_traits>

#include "gsx_device.h"
#include "tile_order.h"

using namespace gsx;

namespace {

template <int V>
using Int = std::integral_constant<int, V>;

constexpr int kThreads = kTilePixels;
constexpr int kWaves = kThreads / kWave;  // 4 quadrant waves

// The compositing loops' exp (stands in for metal::exp at rasterize.py:80,
// 171), nine instructions: k = the integer nearest x log2 e from one fused
// multiply-add with the rounding constant 1.5 * 2^23 (j lies in
// [2^23, 2^24), where floats are spaced 1 apart, so j - 1.5 * 2^23 = k
// exactly); r = x - k ln2 with ln2 rounded to float32 (one multiply-add);
// e^r by the degree-5 polynomial p = 1 + r q(r) whose coefficients were
// fitted for least maximum relative error on |r| <= ln2/2; then 2^k p by
// one shift-and-add of j's encoding into p's (its low nine bits are
// k mod 2^9, so the shift adds k to the exponent field modulo 2^32; for x in
// [-86, 88] the result is normal and the add is the exact scaling).  At
// most 2.02 ulp from exp for x in [-6, 0] (every power that can pass the
// alpha test), 4.75 ulp on [-87, 0], and exp(0) = 1.  splat_exp_core is the
// sequence without range handling (callers that know x lies in [-86, 88]);
// splat_exp_sel adds it with selects: 0 below -86, +inf above 88, NaN
// unchanged.
__device__ __forceinline__ float splat_exp_core(float x) {
    const float j = fmaf(x, 1.44269504088896341f, 12582912.0f);
    const float k = j - 12582912.0f;
    const float r = fmaf(k, -0.693147182464599609375f, x);
    float q = 8.290260538610955e-03f;
    q = fmaf(q, r, 4.189814578274823e-02f);
    q = fmaf(q, r, 1.6667638172664237e-01f);
    q = fmaf(q, r, 4.9999147944277167e-01f);
    q = fmaf(q, r, 9.999997063356061e-01f);
    const float p = fmaf(q, r, 1.0f);
    return __uint_as_float(__float_as_uint(p) + (__float_as_uint(j) << 23));
}

__device__ __forceinline__ float splat_exp_sel(float x) {
    float e = splat_exp_core(fminf(fmaxf(x, -86.0f), 88.0f));
    e = (x < -86.0f) ? 0.0f : e;
    e = (x > 88.0f) ? __builtin_huge_valf() : e;
    return (x != x) ? x : e;
}

// rasterize.py:77-78, power = -0.5 (a dx^2 + c dy^2) - b dx dy, with the
// conic staged pre-scaled to (A, B, C) = (-a/2, -b, -c/2) (exact scalings)
// and factored as power = (A dx + B dy) dx + (C dy) dy: three products and
// two multiply-adds, five roundings whose error is at most
// 2 eps (|A| dx^2 + |B dx dy| + |C| dy^2) + eps |power| (eps = 2^-24).
__device__ __forceinline__ float splat_power(float A, float B, float C, float dx, float dy) {
    return fmaf(fmaf(B, dy, A * dx), dx, (C * dy) * dy);
}

// ln x from the hardware base-2 logarithm (about 1 ulp of log2 x, plus the
// rounding of the product): the culling bounds below carry margins of
// 1e-3 + 1e-4 |L| (alpha_floor_power) and 1% + 1e-3 (quadrant_mask), far
// above that error.  x must be a positive normal number.
__device__ __forceinline__ float ln_fast(float x) {
    return __builtin_amdgcn_logf(x) * 0.693147180559945309f;
}

// Power below which o * exp(power) < 1/255 for certain.  +inf when the
// opacity can never reach 1/255 (o <= 0 or tiny), -inf when no bound is safe
// (o NaN or +inf).
__device__ __forceinline__ float alpha_floor_power(float o) {
    if (o > 0.0f) {
        // ln(1 / (255 o)); below the normal range the bound is 200 anyway
        float L = 255.0f * o >= 1.17549435e-38f ? -ln_fast(255.0f * o) : 200.0f;
        L = fminf(L, 200.0f);
        return L - (1e-3f + 1e-4f * fabsf(L));
    }
    if (o <= 0.0f) return __builtin_huge_valf();
    return -__builtin_huge_valf();
}

// Which of the tile's four 8x8 quadrants (bit q = quadrant (q&1, q>>1)) the
// pixels with alpha >= 1/255 of this Gaussian can lie in.  alpha >= 1/255
// needs q(d) = a dx^2 + 2 b dx dy + c dy^2 <= 2 ln(255 o); a quadrant is
// kept when the minimum of q over its rectangle of pixel centres is within
// that bound: zero if the mean is inside, else the least of the four edge
// minima.  On a row dy = k, q = a (dx + b k / a)^2 + k^2 det / a, so the
// edge minimum is that expression at dx clamped to the edge (columns alike
// with a and c exchanged), and the eight edge lines are shared by the
// quadrants.  Float32 throughout: with det > 1e-3 a c every term carries a
// relative error below 1e-4, and with b^2 < 0.999 a c the float32
// evaluation of the power (splat_power) is within 4.8e-4 relative of the
// exact value, so tau is inflated by 1% (+1e-3); the float32 log of the
// bound and the <= 5 ulp of splat_exp add errors of ~1e-6, well inside
// that.  Ill-conditioned, non-positive or non-finite conics get no culling
// (all four bits).
__device__ __forceinline__ uint32_t quadrant_mask(float x, float y, float4 c, int px0, int py0) {
    const float o = c.w;
    if (!(o >= 0.0039215f)) return (o == o) ? 0u : 0xFu;  // alpha < 1/255 everywhere
    const float A = c.x, B = c.y, C = c.z;
    const float det = fmaf(A, C, -B * B);
    if (!(A > 0.0f && C > 0.0f && det > 1e-3f * A * C)) return 0xFu;
    const float t2 = 2.0f * fmaf(ln_fast(255.0f * o), 1.01f, 1e-3f);
    if (!(t2 < 1e30f && A < 1e30f && C < 1e30f && fabsf(x) < 1e30f && fabsf(y) < 1e30f))
        return 0xFu;
    const float ia = __builtin_amdgcn_rcpf(A), ic = __builtin_amdgcn_rcpf(C);
    const float ba = -B * ia, bc = -B * ic, da = det * ia, dc = det * ic;
    // pixel-centre offsets from the mean: columns [xl0, xl0 + 7] (left
    // quadrants) and [xl0 + 8, xl0 + 15] (right), rows likewise
    const float xl0 = ((float)px0 + 0.5f) - x, xl1 = xl0 + 7.0f;
    const float xr0 = xl0 + 8.0f, xr1 = xl0 + 15.0f;
    const float yt0 = ((float)py0 + 0.5f) - y, yt1 = yt0 + 7.0f;
    const float yb0 = yt0 + 8.0f, yb1 = yt0 + 15.0f;
    // minimum of q on row dy = k over dx in [lo, hi], and on columns
    auto row = [&](float k, float lo, float hi) {
        const float xs = ba * k, u = fminf(fmaxf(xs, lo), hi) - xs;
        return fmaf(A * u, u, k * k * da);
    };
    auto col = [&](float k, float lo, float hi) {
        const float ys = bc * k, u = fminf(fmaxf(ys, lo), hi) - ys;
        return fmaf(C * u, u, k * k * dc);
    };
    const bool inl = xl0 <= 0.0f && xl1 >= 0.0f, inr = xr0 <= 0.0f && xr1 >= 0.0f;
    const bool intp = yt0 <= 0.0f && yt1 >= 0.0f, inb = yb0 <= 0.0f && yb1 >= 0.0f;
    // With the mean outside a rectangle, q's minimum over it lies on an edge
    // whose outer side holds the mean (at a minimiser inside an edge the
    // gradient 2M(p - mean) points into the rectangle, so the mean lies
    // beyond that edge): of each quadrant's two rows and two columns only
    // the one nearer the mean can hold it, and the other edge of the pair
    // is an upper bound, so min(row edge, column edge) is the minimum.
    const float kt = yt1 < 0.0f ? yt1 : yt0, kb = yb1 < 0.0f ? yb1 : yb0;
    const float kl = xl1 < 0.0f ? xl1 : xl0, kr = xr1 < 0.0f ? xr1 : xr0;
    const float q0 = fminf(row(kt, xl0, xl1), col(kl, yt0, yt1));
    const float q1 = fminf(row(kt, xr0, xr1), col(kr, yt0, yt1));
    const float q2 = fminf(row(kb, xl0, xl1), col(kl, yb0, yb1));
    const float q3 = fminf(row(kb, xr0, xr1), col(kr, yb0, yb1));
    return ((inl && intp) || q0 <= t2 ? 1u : 0u) | ((inr && intp) || q1 <= t2 ? 2u : 0u) |
           ((inl && inb) || q2 <= t2 ? 4u : 0u) | ((inr && inb) || q3 <= t2 ? 8u : 0u);
}

// The same test for one quadrant, pixel (px0, py0) its first.
__device__ __forceinline__ bool quadrant_reached(float x, float y, float4 c, int px0, int py0) {
    const float o = c.w;
    if (!(o >= 0.0039215f)) return !(o == o);  // alpha < 1/255 everywhere
    const float A = c.x, B = c.y, C = c.z;
    const float det = fmaf(A, C, -B * B);
    if (!(A > 0.0f && C > 0.0f && det > 1e-3f * A * C)) return true;
    const float t2 = 2.0f * fmaf(ln_fast(255.0f * o), 1.01f, 1e-3f);
    if (!(t2 < 1e30f && A < 1e30f && C < 1e30f && fabsf(x) < 1e30f && fabsf(y) < 1e30f))
        return true;
    const float ia = __builtin_amdgcn_rcpf(A), ic = __builtin_amdgcn_rcpf(C);
    const float x0 = ((float)px0 + 0.5f) - x, x1 = x0 + 7.0f;
    const float y0 = ((float)py0 + 0.5f) - y, y1 = y0 + 7.0f;
    // the row and the column edge nearer the mean
    const float ky = y1 < 0.0f ? y1 : y0, kx = x1 < 0.0f ? x1 : x0;
    const float xs = -B * ia * ky, u = fminf(fmaxf(xs, x0), x1) - xs;
    const float ys = -B * ic * kx, v = fminf(fmaxf(ys, y0), y1) - ys;
    const float q = fminf(fmaf(A * u, u, ky * ky * (det * ia)), fmaf(C * v, v, kx * kx * (det * ic)));
    return (x0 <= 0.0f && x1 >= 0.0f && y0 <= 0.0f && y1 >= 0.0f) || q <= t2;
}

// A staged Gaussian is "plain" when every quantity the per-pixel loop reads
// is finite and small enough that the float32 power is finite and, for a
// pixel that passes the alpha bound, within [-86, 0]: then exp needs no
// range handling and a zero weight leaves the accumulators unchanged.
//
// The conic must also be well conditioned, det > 1e-6 (a + c)^2 with
// a + c in [1e-12, 1e19), and then the float32 power (splat_power) is never
// positive, so the loops need no power > 0 test.  Its rounding error is at
// most eps (a dx^2 + c dy^2 + 2 |b dx dy|) <= 1.25 eps (a + c) |d|^2
// (eps = 2^-24, |b| < (a + c) / 2), while the exact value is at most
// -lambda_min |d|^2 / 2 with lambda_min >= det / (a + c) > 1e-6 (a + c) (the
// float32 det and trace lose far less than the factor 6.7 of margin).  A
// nonzero offset has |d| >= 2^-25 (pixel centres are >= 0.5 and the
// difference of two floats within a factor two of each other is exact), so
// the exact value stays above 4e-34 in magnitude, far from where the
// denormal rounding of the products (<= 2^-150 each) could matter; at d = 0
// the power is a signed zero.
template <int CH>
__device__ __forceinline__ bool plain_gaussian(float x, float y, float4 c, float thr,
                                               const float4* f) {
    const float tr = c.x + c.z, det = fmaf(c.x, c.z, -c.y * c.y);
    bool ok = fabsf(x) < 1e6f && fabsf(y) < 1e6f && tr >= 1e-12f && tr < 1e19f &&
              det > 1e-6f * (tr * tr) && c.w >= 0.0f && c.w < 1e30f && thr >= -86.0f;
    constexpr int F4 = (CH + 3) / 4;
#pragma unroll
    for (int k = 0; k < F4; ++k)
        ok = ok && fabsf(f[k].x) < 1e30f && fabsf(f[k].y) < 1e30f && fabsf(f[k].z) < 1e30f &&
             fabsf(f[k].w) < 1e30f;
    return ok;
}

template <int CTRL, int ROW_MASK, int BANK_MASK>
__device__ __forceinline__ float dpp_f(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, ROW_MASK,
                                                       BANK_MASK, false));
}

// In-place v_permlane32_swap (upper 32 lanes of a[k] <-> lower 32 lanes of
// b[k]) and v_permlane16_swap (odd rows of a[k] <-> even rows of b[k]) for
// K register pairs, up to four per asm block.  Written as asm so the
// operands are swapped where they live (the builtins' two results made the
// register allocator copy both operands first); each block starts with
// s_nop 1, the two wait states a swap needs after a VALU write of its
// operands, since the compiler's hazard check cannot see into the asm (the
// swaps inside a block touch disjoint registers).
#define GSX_SWAP_BLOCK(OP, K, a, b)                                                          \
    do {                                                                                     \
        if constexpr (K >= 4) {                                                              \
            asm("s_nop 1\n\t" OP " %0, %1\n\t" OP " %2, %3\n\t" OP " %4, %5\n\t" OP " %6, %7" \
                : "+v"(a[0]), "+v"(b[0]), "+v"(a[1]), "+v"(b[1]), "+v"(a[2]), "+v"(b[2]),    \
                  "+v"(a[3]), "+v"(b[3]));                                                   \
        } else if constexpr (K == 3) {                                                       \
            asm("s_nop 1\n\t" OP " %0, %1\n\t" OP " %2, %3\n\t" OP " %4, %5"                \
                : "+v"(a[0]), "+v"(b[0]), "+v"(a[1]), "+v"(b[1]), "+v"(a[2]), "+v"(b[2]));   \
        } else if constexpr (K == 2) {                                                       \
            asm("s_nop 1\n\t" OP " %0, %1\n\t" OP " %2, %3"                                 \
                : "+v"(a[0]), "+v"(b[0]), "+v"(a[1]), "+v"(b[1]));                           \
        } else if constexpr (K == 1) {                                                       \
            asm("s_nop 1\n\t" OP " %0, %1" : "+v"(a[0]), "+v"(b[0]));                        \
        }                                                                                    \
    } while (0)

template <int K>
__device__ __forceinline__ void swap_rows32(float (&a)[K], float (&b)[K]) {
    GSX_SWAP_BLOCK("v_permlane32_swap_b32", K, a, b);
}
template <int K>
__device__ __forceinline__ void swap_rows16(float (&a)[K], float (&b)[K]) {
    GSX_SWAP_BLOCK("v_permlane16_swap_b32", K, a, b);
}

// Sums of NVP per-lane values (NVP a multiple of 4) over the four 16-lane
// rows of the wave, spread over the rows: after the two steps every lane of
// row r holds in q[m] its column's total of value 4m + row_value(r).  Step 1
// swaps the upper half of value 2k with the lower half of value 2k + 1 and
// adds, so each half carries one of the two values; step 2 does the same
// between rows.  Values from index NZ on are known zeros: pairs of them skip
// their exchange.  All lanes must be active.
__device__ __forceinline__ int row_value(int row) { return ((row & 1) << 1) | (row >> 1); }

// Step 1 for value pairs K0..K1-1: h[k] = swap32-sum of v[2k], v[2k + 1]
// (values from NZ on are zeros), four pairs per asm block.
template <int K0, int K1, int NVP, int NZ>
__device__ __forceinline__ void reduce_step1(const float (&v)[NVP], float (&h)[NVP / 2]) {
    if constexpr (K0 < K1) {
        constexpr int N = (K1 - K0) < 4 ? (K1 - K0) : 4;
        float a[N], b[N];
#pragma unroll
        for (int k = 0; k < N; ++k) {
            a[k] = v[2 * (K0 + k)];
            b[k] = 2 * (K0 + k) + 1 < NZ ? v[2 * (K0 + k) + 1] : 0.0f;
        }
        swap_rows32<N>(a, b);
#pragma unroll
        for (int k = 0; k < N; ++k) h[K0 + k] = a[k] + b[k];
        reduce_step1<K0 + N, K1, NVP, NZ>(v, h);
    }
}

// Step 2 alone for row groups M0..M1-1: q[m] = swap16-sum of h[2m],
// h[2m + 1] (the row's partial of value 4m + row_value(row)).
template <int M0, int M1, int NVP>
__device__ __forceinline__ void reduce_step2(const float (&h)[NVP / 2], float (&q)[NVP / 4]) {
    if constexpr (M0 < M1) {
        constexpr int N = (M1 - M0) < 4 ? (M1 - M0) : 4;
        float a[N], b[N];
#pragma unroll
        for (int k = 0; k < N; ++k) {
            a[k] = h[2 * (M0 + k)];
            b[k] = h[2 * (M0 + k) + 1];
        }
        swap_rows16<N>(a, b);
#pragma unroll
        for (int k = 0; k < N; ++k) q[M0 + k] = a[k] + b[k];
        reduce_step2<M0 + N, M1, NVP>(h, q);
    }
}

__device__ __forceinline__ uint64_t uniform64(uint64_t v) {
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return ((uint64_t)hi << 32) | lo;
}


// Tile processing order.  Workgroups go round-robin over the 8 XCDs and a
// workgroup slot that frees takes the next workgroup of its XCD, so the
// kernel ends when the last XCD drains its share; tiles differ in work by
// 2-3x (crowded regions of the frame).  xcd_remap gives each XCD a
// contiguous band of tiles (neighbours share its L2: the same Gaussians'
// records).  With an order (k_tile_order) the bands stay contiguous, each
// XCD takes its band's heaviest tiles first (longest-processing-time-first
// list scheduling), and for the backward, whose per-tile work the forward
// recorded exactly, the bands are cut to equal work rather than equal tile
// counts, with up to twice the mean tiles per band: the backward then
// launches 16 ceil(T / 8) workgroups, those past a band's end exit at once.
// Ordering the whole frame instead, heaviest first regardless of bands,
// balanced as well but doubled the rasterizers' HBM traffic (1.05 GB per
// C3 backward instead of 0.47: neighbouring tiles on different XCDs).
// by_block: order is indexed by workgroup (the backward's layout, -1 = no
// tile).  The forward does not know a tile's work beforehand, and a scene's
// crowded region fills a few of its bands: the busiest XCD's lists hold 1.1 to
// 3.5 times the mean.  Its workgroups therefore take the bands' lists in turns of
// eight ranks, each XCD an eighth of every band.  Whole bands -> turns, us, at
// 1200 / 3600 / 8160 / 32400 tiles: a blob (300k) 232 -> 230, 176 -> 161, 197 ->
// 137, 512 -> 279; a box (300k) 82 -> 81, 79 -> 80, 103 -> 97; heavy tails (400k;
// 1M at 32400) 38 -> 37, 69 -> 67, 126 -> 120, 432 -> 418; shells (1M), where
// neighbouring tiles share the most, 85 -> 89, 104 -> 106, 178 -> 170, 457 -> 457;
// 32 channels, 1M in a box at 8160 tiles, 451 -> 381.  Neighbouring tiles on
// different XCDs cost traffic that the balance outweighs: 1M with SH at 1080p
// reads and writes 181 MB instead of 91, of the 1.2 GB that fit in its time.
__device__ __forceinline__ int tile_at(const int* order, uint32_t b, uint32_t nb, bool by_block) {
    if (!order) return (int)xcd_remap(b, nb);
    if (by_block) return order[b];
    const uint32_t q = nb / 8u, r = nb % 8u, i = b / 8u, x = b % 8u;
    const uint32_t band = i < q ? (x + (i >> 3)) & 7u : x;
    return order[band * q + min(band, r) + i];
}

// The workgroup's largest contributor count (n_contrib) into work[tile]:
// the number of list entries the backward replays for the tile.  Every
// thread of the workgroup calls it.
__device__ __forceinline__ void store_tile_work(int* work, int tile, int last, int wave,
                                                int lane) {
    __shared__ int s_wmax[kWaves];
    int m = last;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = max(m, __shfl_xor(m, o, kWave));
    if (lane == 0) s_wmax[wave] = m;
    __syncthreads();
    if (wave == 0 && lane == 0)
        work[tile] = max(max(s_wmax[0], s_wmax[1]), max(s_wmax[2], s_wmax[3]));
}

// The lane's index from the execution hardware, opaque to the compiler:
// values derived from it are formed where they are used instead of being held
// in registers over a whole loop.
__device__ __forceinline__ int lane_again() {
    uint32_t z = 0;
    asm volatile("" : "+s"(z));
    return (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, z));
}

// A quadrant wave's walk list: the staged Gaussians whose bit is set in the
// quadrant's NW mask words (loader wave lw, lane l <-> staged index
// 64 lw + l), compacted in LDS as 32-bit record byte offsets (step x index)
// so the walk is a counted loop over uniform offsets.  Built by the wave
// itself after the workgroup barrier that publishes the masks; ascending
// index order (REV: descending).  list[cnt .. cnt + PADS - 1] are set to
// record pad's offset, for the walks' look-ahead.  Returns cnt
// (uniform).
template <int NW, bool REV, int PADS = 2>
__device__ __forceinline__ int build_list(const uint64_t* words, uint32_t* list, int lane,
                                          int step, int pad) {
    int total = 0;
    const uint64_t below = (1ull << lane) - 1ull;
    const uint64_t above = lane == 63 ? 0ull : ~((2ull << lane) - 1ull);
#pragma unroll
    for (int k = 0; k < NW; ++k) {
        const int lw = REV ? NW - 1 - k : k;
        const uint64_t m = uniform64(words[lw]);
        if ((m >> lane) & 1ull)
            list[total + __popcll(m & (REV ? above : below))] = (uint32_t)((lw * kWave + lane) * step);
        total += __popcll(m);
    }
    if (lane < PADS) list[total + lane] = (uint32_t)(pad * step);
    return total;
}

// The staged record at a byte offset from a list (16 x staged index).
__device__ __forceinline__ const float4& rec_at(const float4* base, int off) {
    return *reinterpret_cast<const float4*>(reinterpret_cast<const char*>(base) + off);
}

template <int CH>
__device__ __forceinline__ void stage_features(float4* dst, const float* f, int nc) {
    constexpr int F4 = (CH + 3) / 4;
    float v[4 * F4];
    if (nc >= CH) {  // uniform: every channel, loads without branches
#pragma unroll
        for (int ch = 0; ch < 4 * F4; ++ch) v[ch] = ch < CH ? f[ch] : 0.0f;
    } else {
#pragma unroll
        for (int ch = 0; ch < 4 * F4; ++ch) v[ch] = (ch < CH && ch < nc) ? f[ch] : 0.0f;
    }
#pragma unroll
    for (int k = 0; k < F4; ++k) dst[k] = make_float4(v[4 * k], v[4 * k + 1], v[4 * k + 2], v[4 * k + 3]);
}

__device__ __forceinline__ float comp4(const float4& v, int e) {
    return e == 0 ? v.x : (e == 1 ? v.y : (e == 2 ? v.z : v.w));
}

// The staged record of the forward's walk: r0 = (mean x, mean y, opacity,
// value 0), r1 = (-a/2, -b, -c/2, value 1) and the values from 2 on, where
// the values are the channels and then the depth.  The walk reads a record
// for every pair of a wave and a Gaussian, and an LDS read costs two cycles
// per register it fills, broadcast or not: a separate log-alpha bound, depth
// and padded channels (12 registers) kept the LDS busy for 82 of the 91
// million cycles in which a CU had work (1M Gaussians, 1080p, 194 us), so a
// record holds nothing the loop can do without (45 of 80 million, 157 us).  Its
// 16-byte pieces lie in arrays of their own, which a walk addresses by one offset
// of 16 x the staged index (whole records of 32 to 96 bytes took up to six more
// registers and 0.5 to 2 % longer, 16 channels 1 % less).
constexpr int kRecords = kThreads + 1;  // the last is the walk lists' padding
template <int NV>
struct FwdRec {
    static constexpr int EX = NV > 2 ? NV - 2 : 0;
    static constexpr int X4 = (EX + 3) / 4;
    static constexpr int kPieces = 2 + X4;
    float4 r0, r1;
    float x[4 * X4 + 1];
    __device__ __forceinline__ float value(int i) const {
        return i == 0 ? r0.w : (i == 1 ? r1.w : x[i - 2]);
    }
    __device__ __forceinline__ void load(const float4* base, uint32_t off) {
        r0 = rec_at(base, off);
        r1 = rec_at(base + kRecords, off);
    }
    __device__ __forceinline__ void load_values(const float4* base, uint32_t off) {
        const float4* const p = &rec_at(base + 2 * kRecords, off);
        if constexpr (EX == 1) {
            x[0] = p->x;
        } else if constexpr (EX == 2) {
            const float2 v = *reinterpret_cast<const float2*>(p);
            x[0] = v.x;
            x[1] = v.y;
        } else if constexpr (EX > 2) {
#pragma unroll
            for (int k = 0; k < X4; ++k) {
                const float4 v = p[k * kRecords];
                x[4 * k] = v.x;
                x[4 * k + 1] = v.y;
                x[4 * k + 2] = v.z;
                x[4 * k + 3] = v.w;
            }
        }
    }
};

// A lane's pixel in the front-to-back loop: its centre, transmittance, sums
// and the record offset of the last Gaussian composited in this batch.
template <int NV>
struct FwdPixel {
    float x, y;
    float T;
    float acc[NV];
    int last_off;
};

// One (pixel, Gaussian) step of the front-to-back loop (rasterize.py:74-87):
// lanes that do not composite keep their state.  PLAIN: the Gaussian passed plain_gaussian(),
// so its power is never positive; powers below -86, where exp would need
// range handling, lie under the alpha bound whatever the opacity
// (plain_gaussian: the log-alpha bound is at least -86).  The updates then
// run under the compositing lanes' exec mask (a branch that no lane takes is
// skipped, and a move costs 2.4 cycles where a select costs 4.2).  Otherwise
// every update is a select; powers below the log-alpha bound need no test of
// their own there either, since o e < 1/255 for each of them (o <= 0 and
// e = 0 included, and a power of NaN passes both ways).
// The per-lane decisions are kept as wave masks (alive: the pixel has not
// stopped): a ballot of one comparison is that comparison's lane mask, the
// masks combine in scalar registers, and inverse_ballot hands one back to
// the lanes as a select condition, so none of it costs vector ALU work.
template <int NV, bool PLAIN>
__device__ __forceinline__ void fwd_pair(const FwdRec<NV>& g, int off, FwdPixel<NV>& px,
                                         uint64_t& alive) {
    const float power = splat_power(g.r1.x, g.r1.y, g.r1.z, g.r0.x - px.x, g.r0.y - px.y);
    const uint64_t live =
        alive & (PLAIN ? __ballot(!(power < -86.0f)) : __ballot(!(power > 0.0f)));
    const float e = PLAIN ? splat_exp_core(power) : splat_exp_sel(power);
    const float alpha = fminf(0.99f, g.r0.z * e);
    const uint64_t pass = live & __ballot(!(alpha < 1.0f / 255.0f));
    const float next_T = px.T * (1.0f - alpha);
    const uint64_t lt = __ballot(next_T < 1e-4f);
    alive &= ~(pass & lt);  // the reference's early stop
    const bool add = __builtin_amdgcn_inverse_ballot_w64(pass & ~lt);
    // acc += rgb * (alpha * T) (rasterize.py:84) as one fused multiply-add,
    // the contraction Metal's default fast-math applies to the reference
    const float w = alpha * px.T;
    if (PLAIN) {
        px.T = add ? next_T : px.T;
        px.last_off = add ? off : px.last_off;
        if (add) {
            // keeps the sums a branch (the compiler would turn them into
            // selects) and w computed before it
            asm volatile("" ::"v"(w) : "memory");
#pragma unroll
            for (int i = 0; i < NV; ++i) px.acc[i] = fmaf(g.value(i), w, px.acc[i]);
        }
    } else {
        px.T = add ? next_T : px.T;
        px.last_off = add ? off : px.last_off;
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const float a2 = fmaf(g.value(i), w, px.acc[i]);
            px.acc[i] = add ? a2 : px.acc[i];
        }
    }
}

// Front-to-back walk of one quadrant wave over its list, four Gaussians per
// round: each Gaussian's record (up to four values past the first two) is
// read while the one before it is evaluated, and list entries two places
// ahead.  list[cnt .. cnt + 3] are the padding record, which no pixel takes,
// so a round may run past the list's end (a stale entry is read only as the
// next round's offsets and never used, since the round count ends first).
// The wave stops once its 64 pixels have terminated.  last_off gets the
// offset of each pixel's last composited Gaussian of this batch.
template <int NV, bool PLAIN>
__device__ __forceinline__ void fwd_walk(const uint32_t* list, int cnt, const float4* rec,
                                         FwdPixel<NV>& px, uint64_t& alive) {
    using Rec = FwdRec<NV>;
    // more values are read just before their pair (registers)
    constexpr bool kAhead = Rec::X4 <= 1;
    if (cnt == 0) return;
    Rec a, b;
    auto load = [&](Rec& g, uint32_t off) {
        g.load(rec, off);
        if (kAhead) g.load_values(rec, off);
    };
    auto pair = [&](Rec& g, uint32_t off) {
        if (!kAhead) g.load_values(rec, off);
        fwd_pair<NV, PLAIN>(g, (int)off, px, alive);
    };
    uint32_t oa = list[0], ob = list[1];
    load(a, oa);
    if (!PLAIN) {
        // rounds of two, which keep the long form short.  One needle that
        // covers the frame makes most batches take it: two of them in 1M
        // Gaussians at 1080p 229 us with one entry at a time, nothing read
        // ahead and the bound's logarithm per pair, 190 us this way.
#pragma unroll 1
        for (int i = 0;; i += 2) {
            const uint32_t na = list[i + 2], nb = list[i + 3];
            load(b, ob);
            pair(a, oa);
            load(a, na);
            pair(b, ob);
            if (alive == 0ull || i + 2 >= cnt) return;
            oa = na;
            ob = nb;
        }
    }
    for (int i = 0;; i += 4) {
        const uint32_t nc = list[i + 2], nd = list[i + 3];
        load(b, ob);
        pair(a, oa);
        load(a, nc);
        pair(b, ob);
        const uint32_t na = list[i + 4], nb = list[i + 5];
        load(b, nd);
        pair(a, nc);
        load(a, na);
        pair(b, nd);
        if (alive == 0ull || i + 4 >= cnt) return;
        oa = na;
        ob = nb;
    }
}

// Occupancy targets.  Up to four channels the kernel fits eight waves per SIMD
// (<= 64 VGPRs) by itself; asking for eight or seven makes the compiler hold
// back scalar registers too and move some through vector lanes in the staging
// (60k on 690 tiles 171 us so, 169.5 without).
constexpr int fwd_min_waves(int ch) { return ch <= 8 ? 6 : 4; }

// The channel of value i in a block of nc of CH channels: groups of four that
// lie inside the row, the last ones overlapping where nc < CH (their channels
// are summed twice, with the same bits).  A group is then one load and no channel
// takes a branch; with a branch per channel each was a load of its own (500k,
// 720p: 16 channels 158 -> 130 us, 12 channels 144 -> 126, 3 channels 95 -> 91).
// Up to four channels a block is whole.
template <int CH>
__device__ __forceinline__ int fwd_channel(int i, int nc) {
    return CH <= 4 ? i : min(i & ~3, nc - 4) + (i & 3);
}

// The arguments of the forward kernels up to 16 channels.
struct FwdArgs {
    const float2* xy;
    const float4* co;
    const float* feat;
    int C, c0, nc;
    const float* depths;
    const int* ids;
    const int2* ranges;
    int64_t n, n_ids;
    const float* bg;
    int W, H, tiles_x;
    float *out, *final_T;
    int* n_contrib;
    float *depth_out, *alpha_out;
    int* work;
};
#define GSX_FWD_PARAMS                                                                            \
    const float2 *__restrict__ xy, const float4 *__restrict__ co, const float *__restrict__ feat, \
        int C, int c0, int nc, const float *__restrict__ depths, const int *__restrict__ ids,     \
        const int2 *__restrict__ ranges, int64_t n, int64_t n_ids, const float *__restrict__ bg,  \
        int W, int H, int tiles_x, float *__restrict__ out, float *__restrict__ final_T,          \
        int *__restrict__ n_contrib, float *__restrict__ depth_out,                               \
        float *__restrict__ alpha_out, const int *__restrict__ order, int *__restrict__ work
#define GSX_FWD_ARGS                                                                              \
    FwdArgs {                                                                                     \
        xy, co, feat, C, c0, nc, depths, ids, ranges, n, n_ids, bg, W, H, tiles_x, out, final_T,  \
            n_contrib, depth_out, alpha_out, work                                                 \
    }

template <int NV>
struct FwdTileLds {
    // record kThreads is the lists' padding: opacity zero, which no pixel takes
    float4 rec[FwdRec<NV>::kPieces * kRecords];
    uint64_t mask[kWaves][kWaves];  // [quadrant][loader wave]
    // one word per wave, written before a barrier and read by every thread
    // after it (a 16-byte read): some pixel of the wave still composites /
    // every Gaussian the wave staged is plain.  Each batch's reads come
    // before the next barrier, and the next batch writes only after it.
    alignas(16) uint32_t alive[kWaves];
    alignas(16) uint32_t plain[kWaves];
    uint32_t list[kWaves][kThreads + 8];  // walk lists (+ look-ahead room)
};

// A tile by one workgroup, a wave per quadrant.
template <int CH, bool DEPTH>
__device__ __forceinline__ void fwd_tile(FwdTileLds<CH + (DEPTH ? 1 : 0)>& s, int tile,
                                         const FwdArgs& A) {
    constexpr int NV = CH + (DEPTH ? 1 : 0);
    using Rec = FwdRec<NV>;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tx = tile % A.tiles_x, ty = tile / A.tiles_x;
    const int px0 = tx * kTile, py0 = ty * kTile;
    const int px = px0 + (wave & 1) * 8 + (lane & 7);
    const int py = py0 + (wave >> 1) * 8 + (lane >> 3);
    const bool inside = px < A.W && py < A.H;

    int start, num;
    tile_span(A.ranges[tile], A.n_ids, start, num);

    FwdPixel<NV> p;
    p.x = (float)px + 0.5f;
    p.y = (float)py + 0.5f;
    p.T = 1.0f;
#pragma unroll
    for (int i = 0; i < NV; ++i) p.acc[i] = 0.0f;
    int last = 0;
    uint64_t alive = __ballot(inside);  // the wave's pixels still compositing
    // the padding record (written before the first barrier)
    if (tid < Rec::kPieces)
        s.rec[tid * kRecords + kThreads] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);

    for (int base = 0; base < num; base += kThreads) {
        const int lane = lane_again(), tid = wave * kWave + lane;
        if (lane == 0) s.alive[wave] = alive != 0ull;
        __syncthreads();
        const uint4 al = *reinterpret_cast<const uint4*>(s.alive);
        if ((al.x | al.y | al.z | al.w) == 0u) break;  // all 256 pixels done
        const int k = base + tid;
        uint32_t qm = 0;
        bool plain = true;
        if (k < num) {
            const int g = A.ids[start + k];
            if ((uint32_t)g < (uint64_t)A.n) {
                // the record, depth and feature loads issue together
                const float2 m = A.xy[g];
                const float4 c = A.co[g];
                float v[4 * Rec::X4 + 2];
#pragma unroll
                for (int i = 0; i < 4 * Rec::X4 + 2; ++i) v[i] = 0.0f;
                const float* const f = A.feat + (int64_t)g * A.C + A.c0;
#pragma unroll
                for (int i = 0; i < CH; ++i) v[i] = f[fwd_channel<CH>(i, A.nc)];
                if (DEPTH) v[CH] = A.depths[g];
                const float thr = alpha_floor_power(c.w);
                float4* const r = s.rec + tid;
                r[0] = make_float4(m.x, m.y, c.w, v[0]);
                r[kRecords] = make_float4(-0.5f * c.x, -c.y, -0.5f * c.z, v[1]);
#pragma unroll
                for (int i = 0; i < Rec::X4; ++i)
                    r[(2 + i) * kRecords] = make_float4(v[2 + 4 * i], v[3 + 4 * i],
                                                        v[4 + 4 * i], v[5 + 4 * i]);
                qm = quadrant_mask(m.x, m.y, c, px0, py0);
                plain = plain_gaussian<0>(m.x, m.y, c, thr, nullptr);
#pragma unroll
                for (int i = 0; i < NV; ++i) plain = plain && fabsf(v[i]) < 1e30f;
            }
        }
#pragma unroll
        for (int q = 0; q < kWaves; ++q) {
            const uint64_t b = __ballot((qm >> q) & 1u);
            if (lane == 0) s.mask[q][wave] = b;
        }
        const uint64_t np = __ballot(!plain);
        if (lane == 0) s.plain[wave] = np == 0ull;
        __syncthreads();
        const uint4 pl = *reinterpret_cast<const uint4*>(s.plain);
        const bool batch_plain = (pl.x & pl.y & pl.z & pl.w) != 0u;
        if (alive == 0ull) continue;
        const int cnt =
            build_list<kWaves, false, 4>(s.mask[wave], s.list[wave], lane, 16, kThreads);
        p.last_off = -1;
        if (batch_plain)
            fwd_walk<NV, true>(s.list[wave], cnt, s.rec, p, alive);
        else
            fwd_walk<NV, false>(s.list[wave], cnt, s.rec, p, alive);
        if (p.last_off >= 0) last = base + (p.last_off >> 4) + 1;
    }
    if (inside) {
        const int64_t pid = (int64_t)py * A.W + px;
        const float T = p.T;
        float* o = A.out + pid * A.C + A.c0;
#pragma unroll
        for (int i = 0; i < CH; ++i) {
            const int ch = fwd_channel<CH>(i, A.nc);
            o[ch] = p.acc[i] + T * (A.bg ? A.bg[A.c0 + ch] : 0.0f);
        }
        if (A.c0 == 0) {
            A.final_T[pid] = T;
            A.n_contrib[pid] = last;
            if (A.alpha_out) A.alpha_out[pid] = 1.0f - T;
            if (DEPTH) {
                const float al = 1.0f - T;
                A.depth_out[pid] = al > 1e-6f ? p.acc[CH] / al : 0.0f;
            }
        }
    }
    if (A.work) store_tile_work(A.work, tile, last, wave, lane);
}

template <int CH, bool DEPTH>
__global__ __launch_bounds__(kThreads, fwd_min_waves(CH)) void k_raster_fwd(GSX_FWD_PARAMS) {
    __shared__ FwdTileLds<CH + (DEPTH ? 1 : 0)> s;
    const int tile = __builtin_amdgcn_readfirstlane(tile_at(order, blockIdx.x, gridDim.x, false));
    fwd_tile<CH, DEPTH>(s, tile, GSX_FWD_ARGS);
}

// The forward of small frames.  One wave composites a quadrant's list serially
// in k_raster_fwd, about 45 instructions an entry, and a wave alone on its
// SIMD issues one every six cycles: the tile with the longest list bounds the
// launch (2221 entries of a 256 x 256 view: 106 us, 82 us here).  Only the chain
// through T is serial, so here a workgroup has one quadrant: three waves evaluate
// alphas, 16 entries of a chunk of 48 each, into LDS (zero where the pixel
// does not take the entry), while wave 0 composites the chunk before.  The
// arithmetic of a pair is fwd_pair's, so every output has its bits: an alpha
// of zero leaves T and the sums of a plain batch as they are.
constexpr int kSplitWaves = 3;                    // evaluating waves
constexpr int kSplitPart = 16;                    // entries of a chunk per wave
constexpr int kSplitChunk = kSplitWaves * kSplitPart;
constexpr int kSplitRead = 8;                     // entries composited per round of reads
static_assert(kSplitPart % kSplitRead == 0, "a round lies in one wave's part");

template <int NV>
struct FwdQuadLds {
    static constexpr int V4 = (NV + 3) / 4;
    // the batch's entries that reach the quadrant, in list order
    float4 r0[kThreads];     // mean x, mean y, opacity, list position (int bits)
    float4 r1[kThreads];     // -a/2, -b, -c/2, log-alpha bound
    float4 v[kThreads][V4];  // channels, then depth
    float alpha[2][kSplitChunk][kWave];
    int cnt[kWaves];
    uint32_t plain[kWaves];
    // chunk c's word c & 1: every pixel has stopped.  Written before the
    // chunk's barrier and read after it; the next write of the word follows
    // the next chunk's barrier, which every reader has reached.
    uint32_t stop[2];
};

// A quadrant of a tile by one workgroup.
template <int CH, bool DEPTH>
__device__ __forceinline__ void fwd_quadrant(FwdQuadLds<CH + (DEPTH ? 1 : 0)>& s, int tile,
                                             int quad, const FwdArgs& A) {
    constexpr int NV = CH + (DEPTH ? 1 : 0);
    constexpr int V4 = (NV + 3) / 4;
    static_assert(kThreads == (kSplitWaves + 1) * kWave, "one compositing wave");
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int qx0 = (tile % A.tiles_x) * kTile + (quad & 1) * 8;
    const int qy0 = (tile / A.tiles_x) * kTile + (quad >> 1) * 8;
    const int px = qx0 + (lane & 7), py = qy0 + (lane >> 3);
    const bool inside = px < A.W && py < A.H;
    const float pxf = (float)px + 0.5f, pyf = (float)py + 0.5f;

    int start, num;
    tile_span(A.ranges[tile], A.n_ids, start, num);

    // wave 0's pixels
    float T = 1.0f, acc[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) acc[i] = 0.0f;
    int last = 0;
    uint64_t alive = __ballot(inside);

    bool stopped = false;
    for (int base = 0; base < num && !stopped; base += kThreads) {
        const int k = base + tid;
        bool keep = false, plain = true;
        float2 m = make_float2(0.0f, 0.0f);
        float4 c = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        float v[4 * V4], thr = 0.0f;
#pragma unroll
        for (int i = 0; i < 4 * V4; ++i) v[i] = 0.0f;
        if (k < num) {
            const int g = A.ids[start + k];
            if ((uint32_t)g < (uint64_t)A.n) {
                // the record, depth and feature loads issue together
                m = A.xy[g];
                c = A.co[g];
                const float* const f = A.feat + (int64_t)g * A.C;
#pragma unroll
                for (int ch = 0; ch < CH; ++ch) v[ch] = f[ch];  // CH == nc == C
                if (DEPTH) v[CH] = A.depths[g];
                keep = quadrant_reached(m.x, m.y, c, qx0, qy0);
                thr = alpha_floor_power(c.w);
                plain = plain_gaussian<0>(m.x, m.y, c, thr, nullptr);
#pragma unroll
                for (int i = 0; i < NV; ++i) plain = plain && fabsf(v[i]) < 1e30f;
            }
        }
        const uint64_t kept = __ballot(keep), odd = __ballot(keep && !plain);
        if (lane == 0) {
            s.cnt[wave] = __popcll(kept);
            s.plain[wave] = odd == 0ull;
        }
        __syncthreads();
        int cnt = 0, at = __popcll(kept & ((1ull << lane) - 1ull));
        bool batch_plain = true;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
            if (w < wave) at += s.cnt[w];
            cnt += s.cnt[w];
            batch_plain = batch_plain && s.plain[w] != 0u;
        }
        cnt = __builtin_amdgcn_readfirstlane(cnt);
        if (keep) {
            s.r0[at] = make_float4(m.x, m.y, c.w, __int_as_float(k));
            s.r1[at] = make_float4(-0.5f * c.x, -c.y, -0.5f * c.z, thr);
#pragma unroll
            for (int i = 0; i < V4; ++i)
                s.v[at][i] = make_float4(v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]);
        }
        __syncthreads();
        const int chunks = (cnt + kSplitChunk - 1) / kSplitChunk;
        for (int ck = 0; ck <= chunks; ++ck) {
            if (wave > 0) {
                const int j0 = (wave - 1) * kSplitPart, e0 = ck * kSplitChunk + j0;
                if (e0 < cnt) {
#pragma unroll 4
                    for (int j = 0; j < kSplitPart; ++j) {
                        const int e = min(e0 + j, cnt - 1);  // past the end: alpha zero
                        const float4 r0 = s.r0[e], r1 = s.r1[e];
                        const float power =
                            splat_power(r1.x, r1.y, r1.z, r0.x - pxf, r0.y - pyf);
                        const bool ok = batch_plain ? !(power < -86.0f)
                                                    : !(power > 0.0f) && !(power < r1.w);
                        const float ex =
                            batch_plain ? splat_exp_core(power) : splat_exp_sel(power);
                        const float alpha = fminf(0.99f, r0.z * ex);
                        const bool take = ok && !(alpha < 1.0f / 255.0f) && e0 + j < cnt;
                        s.alpha[ck & 1][j0 + j][lane] = take ? alpha : 0.0f;
                    }
                }
            } else {
                if (ck > 0) {
                    const int f0 = (ck - 1) * kSplitChunk;
                    const int len = min(kSplitChunk, cnt - f0);
                    const float(*const sa)[kWave] = s.alpha[(ck - 1) & 1];
                    int at_last = -1;
                    auto entry = [&](int j, float a, const float4* val, bool masked) {
                        const float next_T = T * (1.0f - a);
                        // the reference's early stop (a is zero, and next_T
                        // the T of a living pixel, where the entry is not taken)
                        alive &= ~__ballot(next_T < 1e-4f);
                        const bool add = __builtin_amdgcn_inverse_ballot_w64(alive);
                        const float w = add ? a * T : 0.0f;
                        T = add ? next_T : T;
                        at_last = w > 0.0f ? j : at_last;
#pragma unroll
                        for (int i = 0; i < NV; ++i) {
                            const float sum = fmaf(comp4(val[i >> 2], i & 3), w, acc[i]);
                            acc[i] = (!masked || w > 0.0f) ? sum : acc[i];
                        }
                    };
                    if (batch_plain) {
                        // eight at a time, their reads together; entries past
                        // the end have alpha zero and the last one's values
                        for (int j = 0; j < len; j += kSplitRead) {
                            float a[kSplitRead];
                            float4 val[kSplitRead][V4];
#pragma unroll
                            for (int u = 0; u < kSplitRead; ++u) {
                                a[u] = sa[j + u][lane];
#pragma unroll
                                for (int i = 0; i < V4; ++i)
                                    val[u][i] = s.v[min(f0 + j + u, cnt - 1)][i];
                            }
#pragma unroll
                            for (int u = 0; u < kSplitRead; ++u)
                                entry(j + u, a[u], val[u], false);
                        }
                    } else {
#pragma unroll 1
                        for (int j = 0; j < len; ++j) entry(j, sa[j][lane], s.v[f0 + j], true);
                    }
                    if (at_last >= 0) last = __float_as_int(s.r0[f0 + at_last].w) + 1;
                }
                if (lane == 0) s.stop[ck & 1] = alive == 0ull;
            }
            __syncthreads();
            stopped = s.stop[ck & 1] != 0u;
            if (stopped) break;
        }
    }
    if (wave > 0) return;
    if (inside) {
        const int64_t pid = (int64_t)py * A.W + px;
        float* o = A.out + pid * A.C;
#pragma unroll
        for (int ch = 0; ch < CH; ++ch)
            o[ch] = acc[ch] + T * (A.bg ? A.bg[ch] : 0.0f);
        A.final_T[pid] = T;
        A.n_contrib[pid] = last;
        if (A.alpha_out) A.alpha_out[pid] = 1.0f - T;
        if (DEPTH) {
            const float al = 1.0f - T;
            A.depth_out[pid] = al > 1e-6f ? acc[CH] / al : 0.0f;
        }
    }
    if (A.work) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) last = max(last, __shfl_xor(last, o, kWave));
        if (lane == 0) atomicMax(&A.work[tile], last);  // cleared with the order
    }
}

template <int CH, bool DEPTH>
__global__ __launch_bounds__(kThreads) void k_raster_fwd_split(GSX_FWD_PARAMS, int tiles) {
    __shared__ FwdQuadLds<CH + (DEPTH ? 1 : 0)> s;
    // workgroups 32 i + 8 q + x: quadrant q of the tile in slot 8 i + x
    const uint32_t bid = blockIdx.x;
    const int slot = (int)((bid & 7u) | ((bid >> 5) << 3)), quad = (int)(bid >> 3) & 3;
    if (slot >= tiles) return;
    const int tile = __builtin_amdgcn_readfirstlane(tile_at(order, slot, tiles, false));
    fwd_quadrant<CH, DEPTH>(s, tile, quad, GSX_FWD_ARGS);
}

// Frames up to this many tiles take k_raster_fwd_split: all of its four workgroups
// per tile then have a place at once on 256 compute units, whose LDS holds four
// each (37 KB up to four values), or three (41 KB).  k_raster_fwd ->
// k_raster_fwd_split, us, for 10k in a blob, 300k in a box, 1M on shells, 400k
// with heavy tails: 110 tiles 153 -> 121, 268 -> 184, 169 -> 143, 39 -> 35; 169
// tiles 128 -> 103, 176 -> 130, 138 -> 125, 33 -> 34; 256 tiles 106 -> 87, 123 ->
// 97, 114 -> 102, 31 -> 31.
constexpr int split_tiles(int values) { return values <= 4 ? 256 : 192; }

// Beyond that, up to this many, they run in two rounds, which a frame bound by a
// few crowded tiles gains from and an evenly filled one does not: 342 tiles, the
// same scenes, 101 -> 83, 113 -> 96, 110 -> 136, 30 -> 45; 510 tiles 104 -> 85,
// 129 -> 103, 113 -> 145, 32 -> 53.  The workgroups decide by how far the longest
// list exceeds the mean one (the order's builders leave both, per band): from
// eight times on every scene gains (blobs, 10 to 20 times, a fifth).  Between 3.2
// and 8 times (boxes, shells on a wide frame) those gain, up to a seventh, whose
// mean list is short; past about 1500 entries the lists are mostly entries that no
// pixel gets to and every quadrant stages them (1M on shells, 3.9 times, mean 4084: 107
// -> 150).  Below (heavy tails, shells) most lose, 51 us instead of 29 at
// worst.  With the values that leave room for three workgroups only the crowded
// frames gain.
constexpr int kChooseTiles = 512;
__device__ __forceinline__ bool crowded(const int* bands, int tiles, bool narrow) {
    int64_t longest = 0, entries = 0;
#pragma unroll
    for (int x = 0; x < kOrderBands; ++x) {
        longest = max(longest, (int64_t)bands[x]);
        entries += (uint32_t)bands[kOrderBands + x];
    }
    longest *= tiles;
    return longest >= 8 * entries ||
           (narrow && 5 * longest >= 16 * entries && entries <= (int64_t)1500 * tiles);
}

template <int NV>
union FwdChooseLds {
    FwdTileLds<NV> tile;
    FwdQuadLds<NV> quad;
};

template <int CH, bool DEPTH>
__global__ __launch_bounds__(kThreads) void k_raster_fwd_choose(GSX_FWD_PARAMS, int tiles) {
    constexpr int NV = CH + (DEPTH ? 1 : 0);
    __shared__ FwdChooseLds<NV> s;
    // each XCD's tiles with their first workgroup, then the other three
    const int x = (int)blockIdx.x & 7, j = (int)blockIdx.x >> 3, per = (tiles + 7) / 8;
    const int rank = j < per ? j : (j - per) / 3, quad = j < per ? 0 : 1 + (j - per) % 3;
    const int slot = 8 * rank + x;
    if (slot >= tiles) return;
    const bool split = crowded(order + tiles, tiles, NV <= 4);
    if (!split && quad != 0) return;
    const int tile = __builtin_amdgcn_readfirstlane(tile_at(order, slot, tiles, false));
    if (split)
        fwd_quadrant<CH, DEPTH>(s.quad, tile, quad, GSX_FWD_ARGS);
    else
        fwd_tile<CH, DEPTH>(s.tile, tile, GSX_FWD_ARGS);
}

// Per-pixel state of the back-to-front replay.
//
// The reference (rasterize.py:170-195) carries per channel the recursively
// blended colour behind the current Gaussian, accum_c = S_c / T_after with
// S_c = sum over later contributors k of c_k alpha_k T_k, and forms
//   dL/dalpha_i = T_i sum_c g_c (c_i - accum_c) - T_final (bg . g) / (1 - alpha_i).
// Since T_i / T_after = 1 / (1 - alpha_i), the channel sum of g_c accum_c
// collapses into one scalar,
//   Q = T_final (bg . g) + sum over later contributors k of alpha_k T_k (c_k . g),
//   dL/dalpha_i = T_i (c_i . g) - Q / (1 - alpha_i),
// so a pixel holds its cotangent g (CH floats) and Q instead of 3 CH floats.
template <int CH>
struct BwdPixel {
    float T;  // transmittance in front of the current Gaussian
    float Q;
    int last;
    float gpix[CH];
};

// One (pixel, Gaussian) step of the back-to-front replay
// (rasterize.py:162-219).  Returns whether any lane of the wave contributes
// and writes each lane's values to out[S q + O] (all zeros when none does):
//   u = G dx dL/dalpha, w = G dy dL/dalpha, u dx, u dy, w dy, G dL/dalpha,
//   alpha T g_c
// (zero for lanes that do not contribute), whose wave sums the flush turns
// into the reference's means2d, conic, opacity and colour gradients (linear
// in these sums).  power, alpha and the skip tests repeat the forward's
// float32 arithmetic exactly (the replay must take the forward's
// decisions); the gradient arithmetic itself uses fused multiply-adds.  T is
// recovered with one reciprocal of (1 - alpha) per pair.  off is the
// Gaussian's record offset (16 x its staged index) and lim = 16 (n_contrib -
// batch base): the pixel's forward composited it only if off < lim.  PLAIN:
// inputs are finite, so a lane that does not contribute can run the same
// update with a zero weight.
template <int CH, bool PLAIN, int S = 1, int O = 0, int NW>
__device__ __forceinline__ bool bwd_values(const float4& r0, const float4& r1,
                                           const float4* __restrict__ fsrc, int off, int lim,
                                           float pxf, float pyf, BwdPixel<CH>& px,
                                           float (&out)[NW]) {
    static_assert(S * (CH + 5) + O < NW, "strided values fit the output array");
    constexpr int F4 = (CH + 3) / 4;
    constexpr int NV = CH + 6;
    const float dx = r0.x - pxf, dy = r0.y - pyf;
    const float power = splat_power(r1.x, r1.y, r1.z, dx, dy);
    // the wave-wide tests ballot each comparison on its own: a ballot of a
    // single comparison is its lane mask, one of a combined condition is
    // first materialised in a vector register
    // PLAIN: the power is never positive (plain_gaussian's conic bound)
    const bool c1 = off < lim, c2 = PLAIN || !(power > 0.0f), c3 = !(power < r0.z);
    bool ok = c1 && c2 && c3;
    const uint64_t m123 = PLAIN ? __ballot(c1) & __ballot(c3)
                                : __ballot(c1) & __ballot(c2) & __ballot(c3);
    if (m123 == 0ull) {
#pragma unroll
        for (int q = 0; q < NV; ++q) out[S * q + O] = 0.0f;
        return false;
    }
    // PLAIN: lanes that pass have power in [-86, 0]; the others' G is
    // replaced by zero below, whatever its value.
    const float G = PLAIN ? splat_exp_core(power) : splat_exp_sel(power);
    const float alpha = fminf(0.99f, r0.w * G);
    const bool c4 = !(alpha < 1.0f / 255.0f);
    ok = ok && c4;
    if ((m123 & __ballot(c4)) == 0ull) {
        // every output is written on every path, so callers hold no stale
        // values across iterations
#pragma unroll
        for (int q = 0; q < NV; ++q) out[S * q + O] = 0.0f;
        return false;
    }
    float4 fv[F4];
#pragma unroll
    for (int q = 0; q < F4; ++q) fv[q] = fsrc[q];
    float cg = 0.0f;  // c_i . g
    // ga = G dL/dalpha (the opacity factor of G dL/dG = o G dL/dalpha is
    // applied to the sums in the flush), aT = alpha T
    float ga, aT;
    if constexpr (PLAIN) {
        // a lane that does not contribute runs the update with G = alpha = 0:
        // its rcp is 1 (T, Q unchanged) and its dL/dalpha is finite, so
        // every value below is zero for it without further selects
        const float Gs = ok ? G : 0.0f;
        const float as = ok ? alpha : 0.0f;
        const float rcp = __builtin_amdgcn_rcpf(1.0f - as);
        px.T = px.T * rcp;
#pragma unroll
        for (int ch = 0; ch < CH; ++ch) cg = fmaf(comp4(fv[ch >> 2], ch & 3), px.gpix[ch], cg);
        const float dL_dalpha = fmaf(cg, px.T, -(px.Q * rcp));
        aT = as * px.T;
        px.Q = fmaf(aT, cg, px.Q);
        ga = Gs * dL_dalpha;
    } else {
        const float rcp = __builtin_amdgcn_rcpf(1.0f - alpha);
        px.T = ok ? px.T * rcp : px.T;
#pragma unroll
        for (int ch = 0; ch < CH; ++ch) cg = fmaf(comp4(fv[ch >> 2], ch & 3), px.gpix[ch], cg);
        float dL_dalpha = fmaf(cg, px.T, -(px.Q * rcp));
        dL_dalpha = ok ? dL_dalpha : 0.0f;
        aT = ok ? alpha * px.T : 0.0f;
        px.Q = ok ? fmaf(aT, cg, px.Q) : px.Q;
        ga = G * dL_dalpha;
    }
    const float u = ga * dx, w = ga * dy;
    float v[NV];
    v[0] = u;
    v[1] = w;
    v[2] = u * dx;
    v[3] = u * dy;
    v[4] = w * dy;
    v[5] = ga;
#pragma unroll
    for (int ch = 0; ch < CH; ++ch) v[6 + ch] = aT * px.gpix[ch];
#pragma unroll
    for (int q = 0; q < NV; ++q) out[S * q + O] = (PLAIN || ok) ? v[q] : 0.0f;
    return true;
}

// A Gaussian's slot in the wave's LDS sums, from its record offset.
template <int CH>
__device__ __forceinline__ float* slot_at(float4 (*part)[((CH + 6) + 3) / 4], int off) {
    constexpr int NV4 = ((CH + 6) + 3) / 4;
    return reinterpret_cast<float*>(reinterpret_cast<char*>(part) + off * NV4);
}

// The same for two different Gaussians in one reduction (fewer padding
// values and shared exchange steps): value i of Gaussian a sits at 2i and of
// Gaussian b at 2i + 1 of the combined array, so the first exchange pairs
// a's and b's value i; rows with row_value 0 and 2 then finish a's values
// 2m and 2m + 1, rows with 1 and 3 b's, each stored at slot position
// 2m + (row_value >> 1).
template <int CH>
__device__ __forceinline__ void bwd_reduce2(float (&w)[4 * ((CH + 7) / 2)], int oa, int ob,
                                            float4 (*part)[((CH + 6) + 3) / 4], int lane) {
    constexpr int NV = CH + 6;
    constexpr int NH = (NV + 1) / 2;  // value pairs per Gaussian
    static_assert(2 * NH <= 4 * ((NV + 3) / 4), "a Gaussian's slot holds its padded pairs");
    constexpr int K1 = NV;            // value pairs with a non-zero member (of 2 NH)
    constexpr int K2 = (K1 + 1) / 2;  // row groups with a non-zero member
    float h[2 * NH];
#pragma unroll
    for (int k = K1; k < 2 * NH; ++k) h[k] = 0.0f;
    reduce_step1<0, K1, 4 * NH, 2 * NV>(w, h);
    // step 2 (swap16-sum between rows): a[m] holds in
    // row r the row's partial of value 4m + row_value(r)
    float a[NH];
#pragma unroll
    for (int m = K2; m < NH; ++m) a[m] = 0.0f;
    reduce_step2<0, K2, 4 * NH>(h, a);
    // Step 3 within the row with halving exchanges.  A: row_mirror pairs
    // a[2j], a[2j + 1] (lanes 8..15 keep the second); B: row_half_mirror
    // pairs those results (lanes with bit 2 set keep the second); then two
    // quad steps.  Afterwards d[k] holds the total of a[4k + 2 bit2 + bit3],
    // bl (nb odd) that of a[2 (nb - 1) + bit3] and c (NH odd) that of
    // a[NH - 1]: 3 instructions per exchanged pair instead of 2 per value
    // and step.
    const int l = lane & 15;
    const bool hi8 = (l & 8) != 0, hi4 = (l & 4) != 0;
    constexpr int NB = NH / 2, ND = NB / 2;
    float b[NB + 1];
#pragma unroll
    for (int j = 0; j < NB; ++j) {
        const float x = hi8 ? a[2 * j + 1] : a[2 * j];
        const float y = hi8 ? a[2 * j] : a[2 * j + 1];
        b[j] = x + dpp_f<0x140, 0xF, 0xF>(y);  // row_mirror
    }
    float c = 0.0f;
    if constexpr (NH % 2 == 1) {
        c = a[NH - 1];
        c += dpp_f<0x140, 0xF, 0xF>(c);
        c += dpp_f<0x141, 0xF, 0xF>(c);  // row_half_mirror
    }
    float d[ND + 1];
#pragma unroll
    for (int k = 0; k < ND; ++k) {
        const float x = hi4 ? b[2 * k + 1] : b[2 * k];
        const float y = hi4 ? b[2 * k] : b[2 * k + 1];
        d[k] = x + dpp_f<0x141, 0xF, 0xF>(y);  // row_half_mirror
    }
    float bl = 0.0f;
    if constexpr (NB % 2 == 1) {
        bl = b[NB - 1];
        bl += dpp_f<0x141, 0xF, 0xF>(bl);
    }
    auto quad_sum = [](float t) {
        t += dpp_f<0xB1, 0xF, 0xF>(t);  // quad_perm [1,0,3,2]
        t += dpp_f<0x4E, 0xF, 0xF>(t);  // quad_perm [2,3,0,1]
        return t;
    };
#pragma unroll
    for (int k = 0; k < ND; ++k) d[k] = quad_sum(d[k]);
    if constexpr (NB % 2 == 1) bl = quad_sum(bl);
    if constexpr (NH % 2 == 1) c = quad_sum(c);
    // the sums complete before the stores' lane branches (the compiler would
    // move the last add into them and lose its DPP form)
#pragma unroll
    for (int k = 0; k < ND; ++k) asm volatile("" ::"v"(d[k]));
    if constexpr (NB % 2 == 1) asm volatile("" ::"v"(bl));
    if constexpr (NH % 2 == 1) asm volatile("" ::"v"(c));
    const int rv = row_value(lane >> 4);
    float* dst = slot_at<CH>(part, (rv & 1) ? ob : oa) + (rv >> 1);
    const int sel = (hi4 ? 2 : 0) + (hi8 ? 1 : 0);
    if ((l & 3) == 3) {
#pragma unroll
        for (int k = 0; k < ND; ++k) dst[2 * (4 * k + sel)] = d[k];
    }
    if constexpr (NB % 2 == 1) {
        if ((l & 7) == 7) dst[2 * (2 * (NB - 1) + (hi8 ? 1 : 0))] = bl;
    }
    if constexpr (NH % 2 == 1) {
        if (l == 15) dst[2 * (NH - 1)] = c;
    }
}

// The same walk two Gaussians at a time, the pair sharing one reduction (a
// Gaussian without contributions enters it as zeros): their values are
// written interleaved, a's at even and b's at odd positions, which is the
// layout bwd_reduce2 sums.  b's records are read before a is evaluated and
// the next a's before b is.  An odd count pairs the last Gaussian with the
// padding record, which contributes nothing and owns a slot of its own.
template <int CH, bool PLAIN>
__device__ __forceinline__ void bwd_walk(const uint32_t* list, int cnt, int lim,
                                          const float4* s_r0, const float4* s_r1,
                                          const float4 (*s_f)[(CH + 3) / 4],
                                          float4 (*part)[((CH + 6) + 3) / 4], float pxf,
                                          float pyf, int lane, BwdPixel<CH>& px) {
    constexpr int F4 = (CH + 3) / 4;
    constexpr int NV = CH + 6;
    constexpr int NW = 4 * ((NV + 1) / 2);
    const float4* sf = &s_f[0][0];
    int oa = list[0], ob = list[1];
    float4 a0 = rec_at(s_r0, oa), a1 = rec_at(s_r1, oa);
    for (int i = 0; i < cnt; i += 2) {
        const int na = list[i + 2], nb = list[i + 3];
        const float4 b0 = rec_at(s_r0, ob), b1 = rec_at(s_r1, ob);
        float w[NW];
#pragma unroll
        for (int q = 2 * NV; q < NW; ++q) w[q] = 0.0f;
        const bool ha = bwd_values<CH, PLAIN, 2, 0>(a0, a1, &rec_at(sf, oa * F4), oa, lim, pxf,
                                                    pyf, px, w);
        a0 = rec_at(s_r0, na);
        a1 = rec_at(s_r1, na);
        const bool hb = bwd_values<CH, PLAIN, 2, 1>(b0, b1, &rec_at(sf, ob * F4), ob, lim, pxf,
                                                    pyf, px, w);
        if (ha || hb) bwd_reduce2<CH>(w, oa, ob, part, lane);
        oa = na;
        ob = nb;
    }
}

// Waves per SIMD the backward asks for (more waves hide LDS and ballot
// latencies): six at one and three channels (<= 80 VGPRs, 12-16 KB of LDS),
// five at two and four channels (which would spill at 80); no instantiation
// spills (checked with -Rpass-analysis=kernel-resource-usage: ScratchSize 0
// for every one).
constexpr int bwd_min_waves(int ch) { return (ch == 2 || ch == 4) ? 5 : 6; }

template <int CH>
__global__ __launch_bounds__(kThreads, bwd_min_waves(CH)) void k_raster_bwd(
    const float2* __restrict__ xy, const float4* __restrict__ co, const float* __restrict__ feat,
    int C, int c0, int nc, const int* __restrict__ ids, const int2* __restrict__ ranges,
    int64_t n, int64_t n_ids, const float* __restrict__ bg, int W, int H, int tiles_x,
    const float* __restrict__ final_T, const int* __restrict__ n_contrib,
    const float* __restrict__ grad_out, const float* __restrict__ grad_T,
    float* __restrict__ g_xy, float* __restrict__ g_conic, float* __restrict__ g_feat,
    float* __restrict__ g_opac, int gstride, const int* __restrict__ order) {
    constexpr int F4 = (CH + 3) / 4;
    constexpr int NV = CH + 6;             // u, w, u dx, u dy, w dy, opacity term, channels
    constexpr int NV4 = (NV + 3) / 4;
    // Gaussians per batch: 64 keeps the slot LDS at 16 KB up to four
    // channels (more workgroups per CU; measured faster than 128)
    constexpr int BB = 64;
    constexpr int NLW = BB / kWave;  // mask words per quadrant
    // entry BB of the records and slots is the walk lists' padding: a record
    // no pixel can take (alpha bound +inf) whose slot the flush never reads
    __shared__ float4 s_r0[BB + 1];
    __shared__ float4 s_r1[BB + 1];  // -a/2, -b, -c/2 (conic), Gaussian id (int bits)
    __shared__ float4 s_f[BB + 1][F4];
    __shared__ float4 s_part[kWaves][BB + 1][NV4];  // per-wave gradient sums per Gaussian
    __shared__ uint64_t s_mask[kWaves][NLW];
    __shared__ uint32_t s_list[kWaves][BB + 4];  // walk lists (+ look-ahead room)
    __shared__ int s_last[kWaves];
    // per wave: every Gaussian it staged is plain (written before the staging
    // barrier, read by all after it; the loop-top barrier orders batches)
    __shared__ __align__(16) uint32_t s_plain[kWaves];

    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int tile = __builtin_amdgcn_readfirstlane(tile_at(order, blockIdx.x, gridDim.x, true));
    if (tile < 0) return;  // past the end of this XCD's band
    const int tx = tile % tiles_x, ty = tile / tiles_x;
    const int px0 = tx * kTile, py0 = ty * kTile;
    const int px = px0 + (wave & 1) * 8 + (lane & 7);
    const int py = py0 + (wave >> 1) * 8 + (lane >> 3);
    const bool inside = px < W && py < H;
    const float pxf = (float)px + 0.5f, pyf = (float)py + 0.5f;
    const int64_t pid = (int64_t)py * W + px;

    int start, num;
    tile_span(ranges[tile], n_ids, start, num);

    BwdPixel<CH> st;
    // the pixel's loads issue together (clamped indices, masked after)
    const int64_t pidc = inside ? pid : 0;
    const float tf = final_T[pidc];
    const int nct = n_contrib[pidc];
    float gp[CH], bgv[CH];
#pragma unroll
    for (int ch = 0; ch < CH; ++ch) {
        gp[ch] = grad_out[pidc * C + c0 + min(ch, nc - 1)];
        bgv[ch] = bg ? bg[c0 + min(ch, nc - 1)] : 0.0f;
    }
    const float gt = grad_T ? grad_T[pidc] : 0.0f;
    const float T_final = inside ? tf : 1.0f;
    st.T = T_final;
    st.last = inside ? nct : 0;
    float bg_dot = 0.0f;
#pragma unroll
    for (int ch = 0; ch < CH; ++ch) {
        st.gpix[ch] = (inside && ch < nc) ? gp[ch] : 0.0f;
        if (ch < nc) bg_dot = bg_dot + bgv[ch] * st.gpix[ch];
    }
    // The alpha output's cotangent enters once, with the first channel block.
    if (inside && c0 == 0 && grad_T) bg_dot = bg_dot + gt;
    st.Q = T_final * bg_dot;

    // the padding record (written before the barrier below)
    if (tid == 0) {
        s_r0[BB] = make_float4(0.0f, 0.0f, __builtin_huge_valf(), 0.0f);
        s_r1[BB] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
        for (int q = 0; q < F4; ++q) s_f[BB][q] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }

    // Largest n_contrib of each quadrant: later list entries changed no pixel.
    {
        int m = st.last;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) m = max(m, __shfl_xor(m, o, kWave));
        if (lane == 0) s_last[wave] = m;
    }
    __syncthreads();
    int quad_last[kWaves];
#pragma unroll
    for (int q = 0; q < kWaves; ++q) quad_last[q] = s_last[q];
    const int max_last = max(max(quad_last[0], quad_last[1]), max(quad_last[2], quad_last[3]));
    const int n_batches = (max_last + BB - 1) / BB;

    for (int b = n_batches - 1; b >= 0; --b) {
        __syncthreads();
        uint32_t qm = 0;
        bool plain = true;
        if (tid < BB) {
            const int k = b * BB + tid;
            float4 r1 = make_float4(0.0f, 0.0f, 0.0f, __int_as_float(-1));
            if (k < num) {
                const int g = ids[start + k];
                if ((uint32_t)g < (uint64_t)n) {
                    // the record and feature loads issue together
                    const float2 m = xy[g];
                    const float4 c = co[g];
                    stage_features<CH>(s_f[tid], feat + (int64_t)g * C + c0, nc);
                    const float thr = alpha_floor_power(c.w);
                    s_r0[tid] = make_float4(m.x, m.y, thr, c.w);
                    r1 = make_float4(-0.5f * c.x, -c.y, -0.5f * c.z, __int_as_float(g));
                    qm = quadrant_mask(m.x, m.y, c, px0, py0);
#pragma unroll
                    for (int q = 0; q < kWaves; ++q)
                        if (k >= quad_last[q]) qm &= ~(1u << q);
                    plain = plain_gaussian<CH>(m.x, m.y, c, thr, s_f[tid]);
                }
            }
            s_r1[tid] = r1;
        }
        if (wave < NLW) {
#pragma unroll
            for (int q = 0; q < kWaves; ++q) {
                const uint64_t bq = __ballot((qm >> q) & 1u);
                if (lane == 0) s_mask[q][wave] = bq;
            }
        }
        const uint64_t np = __ballot(!plain);
        if (lane == 0) s_plain[wave] = np == 0ull;
        __syncthreads();
        const uint4 pl = *reinterpret_cast<const uint4*>(s_plain);
        const bool batch_plain = (pl.x & pl.y & pl.z & pl.w) != 0u;
        // the wave's slots start at zero: Gaussians it does not walk, or
        // whose sums it does not store, then add nothing in the flush
        {
            float4* p = &s_part[wave][0][0];
#pragma unroll
            for (int k = 0; k < BB * NV4 / kWave; ++k)
                p[k * kWave + lane] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        }
        const int cnt = build_list<NLW, true>(s_mask[wave], s_list[wave], lane, 16, BB);
        const int lim = 16 * max(0, min(st.last - b * BB, BB));
        if (batch_plain)
            bwd_walk<CH, true>(s_list[wave], cnt, lim, s_r0, s_r1, s_f, s_part[wave], pxf, pyf,
                               lane, st);
        else
            bwd_walk<CH, false>(s_list[wave], cnt, lim, s_r0, s_r1, s_f, s_part[wave], pxf, pyf,
                                lane, st);
        __syncthreads();
        // 1. one thread per Gaussian adds the four waves' slots and turns the
        //    sums into the reference's gradient components, kept in its own
        //    wave-0 slot
        if (tid < BB) {
            float4 sum[NV4];
#pragma unroll
            for (int q = 0; q < NV4; ++q) sum[q] = s_part[0][tid][q];
            // one wave's slot at a time (all four in flight would need
            // 4 NV4 float4 registers)
#pragma unroll 1
            for (int w = 1; w < kWaves; ++w) {
#pragma unroll
                for (int q = 0; q < NV4; ++q) {
                    const float4 p = s_part[w][tid][q];
                    sum[q].x += p.x;
                    sum[q].y += p.y;
                    sum[q].z += p.z;
                    sum[q].w += p.w;
                }
            }
            float e[4 * NV4];
#pragma unroll
            for (int q = 0; q < NV4; ++q) {
                e[4 * q] = sum[q].x;
                e[4 * q + 1] = sum[q].y;
                e[4 * q + 2] = sum[q].z;
                e[4 * q + 3] = sum[q].w;
            }
            // rasterize.py:197-218 in terms of the sums (dL/dG = o dL/dalpha);
            // the staged conic is (-a/2, -b, -c/2)
            const float4 c = s_r1[tid];
            const float o = s_r0[tid].w;
            float* fin = reinterpret_cast<float*>(s_part[0][tid]);
            fin[0] = o * (2.0f * c.x * e[0] + c.y * e[1]);
            fin[1] = o * (c.y * e[0] + 2.0f * c.z * e[1]);
            fin[2] = -0.5f * o * e[2];
            fin[3] = -o * e[3];
            fin[4] = -0.5f * o * e[4];
#pragma unroll
            for (int q = 5; q < NV; ++q) fin[q] = e[q];
        }
        __syncthreads();
        // 2. the global atomics, component-major across the lanes: a wave's
        //    atomic instruction covers about 64 / NV Gaussians.  With a
        //    gradient record (gstride > 0) each Gaussian's components are
        //    adjacent words of one record; with separate arrays each
        //    Gaussian touches one cache line per array
        for (int item = tid; item < BB * NV; item += kThreads) {
            const int j = item / NV, k = item - j * NV;
            const int g = __float_as_int(s_r1[j].w);
            const float v = reinterpret_cast<const float*>(s_part[0][j])[k];
            if (g < 0 || v == 0.0f || (k >= 6 && k - 6 >= nc)) continue;
            float* dst = k >= 6 && g_feat ? g_feat + (int64_t)g * C + c0 + (k - 6)
                       : gstride > 0 ? g_xy + (int64_t)gstride * g + (k < 6 ? k : c0 + k)
                       : k < 2 ? g_xy + 2 * (int64_t)g + k
                       : k < 5 ? g_conic + 3 * (int64_t)g + (k - 2)
                                : g_opac + g;
            atomicAdd(dst, v);
        }
    }
}

typedef float mx_floatx4 __attribute__((ext_vector_type(4)));
constexpr int kMxGroup = 16;   // Gaussians per matrix-core group

// --------------------------------------- backward, five channels and more --
// The same replay (a pixel's state is T and Q, BwdPixel) with the Gaussians
// across the lanes.
//
// A quadrant wave takes its list 16 entries at a time (a bucket), lane l
// holding entry l % 16 (0 the backmost), and steps over its 64 pixels four
// at a time, row r = l / 16 of the wave working on one pixel: step s, row r
// is pixel (s & 7, 4 (s >> 3) + r) of the quadrant.  Within a row, T in front
// of each entry is the pixel's T times the inclusive product of the entries'
// 1 / (1 - alpha), and Q behind it the pixel's Q plus the exclusive sum of
// alpha T (c . g): two four-step DPP scans.  The Gaussian's gradient terms
// then stay in its lane's registers over all the pixels, where lanes = pixels
// has to sum every term of every Gaussian over the wave.  A column of steps is
// skipped once its eight pixels have stopped in front of the bucket.
//
// Bound: the dependent instructions of a step (41 per 64 pairs; multiply-adds
// take 2.4 cycles, DPP, compares, selects and minima 4.2 and the reciprocal
// 8.3, measured) with 12 to 20 waves on a compute unit.  Measured against the
// kernels before it (pixels across the lanes with the sums on the VALU up to
// 16 channels; the channel products through an LDS tile, geometric sums
// through LDS atomics, at 32): 500k Gaussians, 32 channels, 720p 509 -> 284
// us; 60k, 12 channels, 641 x 479 182 -> 118 us; 200k surfels, 5 channels,
// 960 x 540 224 -> 147 us (all with the geometric gradients in one record,
// below).  With three channels it gains 5 % where Gaussians are small and
// loses 18 % where they cover many tiles (every quadrant stages the list for
// itself), so k_raster_bwd stays there.
//
// Along a column of the quadrant (steps x and x + 8) dx is shared, and a lane
// only ever meets two rows, so the geometric terms are kept as moments in dx
// per row, sum of h, h dx and h dx^2 (h = G dL/dalpha), and combined with the
// rows' dy once per bucket.
//
// The channel work runs on the matrix cores (v_mfma_f32_16x16x4_f32, operand
// A[row = l % 16][k = l / 16], B[k = l / 16][col = l % 16], result rows
// 4 (l / 16) + i, column l % 16, checked on the GPU), whose layouts are the
// replay's own, so nothing moves between lanes:
//   c . g   A = g (16 pixels x 4 channels), B = c (4 channels x 16 entries):
//           lane l gets its entry's product for the pixel of step i, row l / 16;
//   dL/dc   A = g (16 channels x 4 pixels), B = alpha T of a step (4 pixels x
//           16 entries, the lane's own value), accumulated over the steps.
// No decision depends on them.
constexpr int kBucket = 16;  // list entries per bucket (the lanes of a row)

// Channel blocks of 5 to 8, 9 to 16 and 17 to 32 channels.
template <int CHP>
struct BwdShape {
    static constexpr int BUF = 80;               // buffered entries: 15 left over + 64 new
    static constexpr int KS = CHP / 4;           // k-steps of c . g
    static constexpr int CB = (CHP + 15) / 16;   // 16-channel blocks of dL/dc
    // up to 8 channels the cotangent operands are read from LDS where they
    // are used (20 registers saved; dL/dc's rows past the channels hold
    // copies, which nobody reads), wider blocks keep them in registers
    static constexpr bool kNarrow = CHP <= 8;
    static constexpr int NO = CHP + 8;  // row stride of a bucket's gradients in LDS
};


// The gradient outputs: the geometric ones in one record per Gaussian (xy,
// stride floats) or in three arrays; feat + feat_stride * id + c is channel c
// of the block, in the record or in an array of its own.
//
// Where Gaussians reach many tiles the atomics' lines bind (bwd_send).  Rows of
// C floats straddle 64-byte lines unless C is a multiple of 16, so callers then
// ask for rows of 16, or up to ten channels for a record of 16 that holds all,
// and copy the features out.  Rows of C -> whole lines with the copy, us: 300k with
// heavy tails at 960 x 540 (7 tiles each) 228 -> 159 (5 channels), 273 -> 214
// (12); 500k on shells at 1080p (10) 466 -> 437, 541 -> 502; 60k at 641 x 479
// (8; 0.5M duplicates) 121 -> 120, 142 -> 134; 500k in a box at 720p (3) 202 ->
// 203, 247 -> 246.
struct BwdOut {
    float* xy;
    float* conic;
    float* opac;
    float* feat;
    int64_t feat_stride;
    int stride, nc, C;
    bool record;   // geometric gradients in a record
    bool whole;    // features in it too: sent together
    int per, mul;  // entries per atomic instruction (64 / components), 65536 / components + 1
};

// Inclusive scans over the 16 lanes of each row, for two registers at once:
// v <- v * (v of the lane 1, 2, 4, 8 below), sums likewise; lanes without a
// partner keep their value.  A DPP read needs two wait states after the VALU
// write of its operand, which the other register's step and an s_nop fill.
#define GSX_SCAN_STEP(op, n)                                           \
    op " %0, %0, %0 row_shr:" n " row_mask:0xf bank_mask:0xf\n\t"      \
    op " %1, %1, %1 row_shr:" n " row_mask:0xf bank_mask:0xf\n\t"      \
    "s_nop 0\n\t"
#define GSX_SCAN(op)                                                   \
    "s_nop 1\n\t" GSX_SCAN_STEP(op, "1") GSX_SCAN_STEP(op, "2")        \
    GSX_SCAN_STEP(op, "4")                                             \
    op " %0, %0, %0 row_shr:8 row_mask:0xf bank_mask:0xf\n\t"          \
    op " %1, %1, %1 row_shr:8 row_mask:0xf bank_mask:0xf"
__device__ __forceinline__ void row_scan_mul(float& a, float& b) {
    asm volatile(GSX_SCAN("v_mul_f32_dpp") : "+v"(a), "+v"(b));
}
__device__ __forceinline__ void row_scan_add(float& a, float& b) {
    asm volatile(GSX_SCAN("v_add_f32_dpp") : "+v"(a), "+v"(b));
}

// The value of the lane below in the row (0 in its first lane).
__device__ __forceinline__ float lane_below(float v) {
    return __int_as_float(
        __builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x111, 0xF, 0xF, true));  // row_shr:1
}

// The wave's pixels.  The lanes 4 b .. 4 b + 3 of row r hold T and Q of step
// 4 b + k in registers k: a step reads them with a row broadcast folded into
// the consuming instruction and writes them with one DPP move under a bank
// mask (in LDS, two 16-byte reads per pair of steps made the LDS the bound:
// 66 % of the cycles).
struct BwdPixels {
    float T[4], Q[4];
    int nc;        // n_contrib of step l % 16, row l / 16
    float px[8];   // the columns' centres (scalar registers)
};

// A wave-uniform float in a scalar register (the compiler keeps one that
// vector instructions computed in a vector register).  The lane read needs a
// wait state after the VALU write of its operand and a VALU read of its
// result two, neither of which the compiler's hazard check sees.
__device__ __forceinline__ float scalar_float(float v) {
    float s;
    asm("s_nop 0\n\tv_readfirstlane_b32 %0, %1\n\ts_nop 1" : "=s"(s) : "v"(v));
    return s;
}

template <int LANE>
__device__ __forceinline__ int row_bcast(int v) {
    return __builtin_amdgcn_update_dpp(0, v, 0x150 + LANE, 0xF, 0xF, true);  // row_newbcast
}
template <int LANE>
__device__ __forceinline__ float row_bcast(float v) {
    return __int_as_float(row_bcast<LANE>(__float_as_int(v)));
}
// old, with the lanes of bank B (4 B .. 4 B + 3 of each row) set to the row's lane 15 of v
template <int B>
__device__ __forceinline__ float set_bank(float old, float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(old), __float_as_int(v),
                                                       0x150 + 15, 0xF, 1 << B, false));
}
// the quad's lane K in its four lanes
template <int K>
__device__ __forceinline__ float quad_bcast(float v) {
    return __int_as_float(
        __builtin_amdgcn_update_dpp(0, __float_as_int(v), K * 0x55, 0xF, 0xF, true));
}

// The quadrant's cotangents in the two operand layouts.
template <int CHP>
struct BwdCot {
    // A operand of c . g, per group of 4 x 4 pixels
    float a[BwdShape<CHP>::kNarrow ? 1 : 4][BwdShape<CHP>::KS];
    // A operand of dL/dc, per step
    float b[BwdShape<CHP>::kNarrow ? 1 : 16][BwdShape<CHP>::CB];
};

// The wave's buffered entries, backmost first, and its other pieces of LDS.
struct BwdLds {
    float4* r0;   // mean x, mean y, log-alpha bound, opacity
    float4* r1;   // -a/2, -b, -c/2 (conic), Gaussian id (int bits)
    int* k;       // position in the tile's list
    float* g;     // the pixels' cotangents, rows of CHP (BwdShape::kNarrow)
    float* out;   // a bucket's gradients, rows of NO (6 geometric, then channels)
    int* id;      // its Gaussians (-1: none)
};

// One bucket: the entries b0 .. b0 + 15 of the buffer, of which those below cnt
// are real.  PLAIN: every one passed plain_gaussian and the quadrant's
// cotangents are finite; an entry that a pixel does not composite then runs
// the same arithmetic with alpha = h = 0, and h carries the opacity
// (h = o G dL/dalpha).  FIN: features and cotangents are finite, so the
// matrix cores may multiply them by zero weights; otherwise the channel work
// is done pair by pair and only where a pixel composites the Gaussian.
// next: called before the gradients are reduced, to issue the loads that
// follow the bucket.  The gradients stay in LDS until bwd_send.
template <int CHP, bool PLAIN, bool FIN, class Next>
__device__ __forceinline__ void bwd_bucket(const BwdLds& L, int b0, int cnt, BwdPixels& P,
                                           const BwdCot<CHP>& g,
                                           const float (&fb)[BwdShape<CHP>::KS],
                                           const BwdOut& O, const float* __restrict__ gout,
                                           const float* __restrict__ feat, int qx0, int qy0, int W,
                                           int H, Next&& next) {
    using S = BwdShape<CHP>;
    const int lane = lane_again();  // the bucket's forms share no registers derived from it
    const int j = lane & 15, r = lane >> 4, C = O.C;
    const float py0 = (float)(qy0 + r) + 0.5f, py1 = (float)(qy0 + 4 + r) + 0.5f;
    {
        const float4 r0 = L.r0[b0 + j], r1 = L.r1[b0 + j];
        const int k = L.k[b0 + j];
        // the columns whose pixels (any of eight) composited past the
        // bucket's frontmost entry
        const int front = __builtin_amdgcn_readfirstlane(L.k[min(b0 + kBucket, cnt) - 1]);
        uint64_t live = __ballot(P.nc > front);
        live |= live >> 32;
        live |= live >> 16;
        const uint32_t cols = (uint32_t)(live | (live >> 8)) & 0xFFu;
        const float dya = r0.y - py0, dyb = r0.y - py1;
        const float cya = (r1.z * dya) * dya, cyb = (r1.z * dyb) * dyb;
        float ha0 = 0.0f, ha1 = 0.0f, ha2 = 0.0f, hb0 = 0.0f, hb1 = 0.0f, hb2 = 0.0f;
        mx_floatx4 dc[S::CB];
#pragma unroll
        for (int cb = 0; cb < S::CB; ++cb) dc[cb] = mx_floatx4{0.0f, 0.0f, 0.0f, 0.0f};

        // A operand of c . g for group q (columns 4 (q & 1).., rows 4 (q >> 1)..)
        auto cota = [&](int q, int ks) {
            if constexpr (S::kNarrow)
                return L.g[(4 * (4 * (q & 1) + (j & 3) + 8 * (q >> 1)) + (j >> 2)) * CHP +
                           4 * ks + r];
            else
                return g.a[q][ks];
        };
        // A operand of dL/dc at step s
        auto cot = [&](int s, int cb) {
            if constexpr (S::kNarrow)
                return L.g[(4 * s + r) * CHP + (j & (CHP - 1))];
            else
                return g.b[s][cb];
        };
        // cotangent of channel c of the lane's pixel at step s (a pixel outside
        // the image has no contributor)
        auto pix = [&](int s, int c) {
            int rr = r;  // opaque: no step's address is kept in registers
            asm volatile("" : "+v"(rr));
            if constexpr (S::kNarrow)
                return L.g[(4 * s + rr) * CHP + c];
            else
                return gout[((int64_t)min(qy0 + 4 * (s >> 3) + rr, H - 1) * W +
                             min(qx0 + (s & 7), W - 1)) * C + c];
        };
        // column x: steps x (row group a) and x + 8 (b)
        auto column = [&](auto xc, float cga, float cgb) {
            constexpr int x = decltype(xc)::value, K = x & 3, B = x >> 2;
            const float dx = r0.x - P.px[x];
            const float adx = r1.x * dx;
            // splat_power with the products of dx alone and dy alone shared
            const float pa = fmaf(fmaf(r1.y, dya, adx), dx, cya);
            const float pb = fmaf(fmaf(r1.y, dyb, adx), dx, cyb);
            const float Ga = PLAIN ? splat_exp_core(pa) : splat_exp_sel(pa);
            const float Gb = PLAIN ? splat_exp_core(pb) : splat_exp_sel(pb);
            const float oa = r0.w * Ga, ob = r0.w * Gb;
            // min(0.99, o G) < 1/255 exactly when o G < 1/255
            uint64_t ma = __ballot(k < row_bcast<x>(P.nc)) & __ballot(!(pa < r0.z)) &
                          __ballot(!(oa < 1.0f / 255.0f));
            uint64_t mb = __ballot(k < row_bcast<x + 8>(P.nc)) & __ballot(!(pb < r0.z)) &
                          __ballot(!(ob < 1.0f / 255.0f));
            if (!PLAIN) {
                ma &= __ballot(!(pa > 0.0f));
                mb &= __ballot(!(pb > 0.0f));
            }
            const bool ka = __builtin_amdgcn_inverse_ballot_w64(ma);
            const bool kb = __builtin_amdgcn_inverse_ballot_w64(mb);
            const float va = ka ? (PLAIN ? oa : fminf(0.99f, oa)) : 0.0f;
            const float vb = kb ? (PLAIN ? ob : fminf(0.99f, ob)) : 0.0f;
            const float ala = PLAIN ? fminf(0.99f, va) : va;
            const float alb = PLAIN ? fminf(0.99f, vb) : vb;
            const float ra = __builtin_amdgcn_rcpf(1.0f - ala);
            const float rb = __builtin_amdgcn_rcpf(1.0f - alb);
            float Ta = ra, Tb = rb;
            row_scan_mul(Ta, Tb);
            Ta *= row_bcast<4 * B>(P.T[K]);
            Tb *= row_bcast<4 * B + 8>(P.T[K]);
            const float wa = ala * Ta, wb = alb * Tb;
            if (!FIN) {
                // c . g pair by pair
                cga = cgb = 0.0f;
#pragma unroll 1
                for (int c = 0; c < O.nc; ++c) {
                    const float fc = feat[(int64_t)max(__float_as_int(r1.w), 0) * C + c];
                    cga = fmaf(fc, pix(x, c), cga);
                    cgb = fmaf(fc, pix(x + 8, c), cgb);
                }
            }
            const float xa = (PLAIN || ka) ? wa * cga : 0.0f, xb = (PLAIN || kb) ? wb * cgb : 0.0f;
            // Q behind each entry: the sums start one lane up, so that the
            // entry's own term is never in them.  Taking it back out of an
            // inclusive sum leaves that sum's rounding, which 1 / (1 - alpha)
            // multiplies by up to 100 (three-entry stacks with an opaque one:
            // 5.7e-6 of the gradient's terms off, 2e-7 this way; 283 -> 284 us
            // at 32 channels, 500k, 720p).
            float Qa = lane_below(xa), Qb = lane_below(xb);
            row_scan_add(Qa, Qb);
            Qa += row_bcast<4 * B>(P.Q[K]);
            Qb += row_bcast<4 * B + 8>(P.Q[K]);
            // the frontmost entry's lane carries the pixel on
            P.T[K] = set_bank<B>(P.T[K], Ta);
            P.T[K] = set_bank<B + 2>(P.T[K], Tb);
            P.Q[K] = set_bank<B>(P.Q[K], Qa + xa);
            P.Q[K] = set_bank<B + 2>(P.Q[K], Qb + xb);
            const float da = fmaf(cga, Ta, -(Qa * ra));
            const float db = fmaf(cgb, Tb, -(Qb * rb));
            const float ha = PLAIN ? va * da : (ka ? Ga * da : 0.0f);
            const float hb = PLAIN ? vb * db : (kb ? Gb * db : 0.0f);
            const float dx2 = dx * dx;
            ha0 += ha;
            hb0 += hb;
            if (PLAIN) {
                ha1 = fmaf(ha, dx, ha1);
                hb1 = fmaf(hb, dx, hb1);
                ha2 = fmaf(ha, dx2, ha2);
                hb2 = fmaf(hb, dx2, hb2);
            } else {
                // an infinite offset of an entry that is not composited must not enter
                ha1 = ka ? fmaf(ha, dx, ha1) : ha1;
                hb1 = kb ? fmaf(hb, dx, hb1) : hb1;
                ha2 = ka ? fmaf(ha, dx2, ha2) : ha2;
                hb2 = kb ? fmaf(hb, dx2, hb2) : hb2;
            }
            if (FIN) {
#pragma unroll
                for (int cb = 0; cb < S::CB; ++cb) {
                    // rows channels, columns entries
                    dc[cb] = __builtin_amdgcn_mfma_f32_16x16x4f32(cot(x, cb), wa, dc[cb], 0, 0, 0);
                    dc[cb] =
                        __builtin_amdgcn_mfma_f32_16x16x4f32(cot(x + 8, cb), wb, dc[cb], 0, 0, 0);
                }
            } else if (ka || kb) {
                float* const dst = O.feat + O.feat_stride * __float_as_int(r1.w);
#pragma unroll 1
                for (int c = 0; c < O.nc; ++c)
                    atomicAdd(dst + c, (ka ? wa * pix(x, c) : 0.0f) +
                                           (kb ? wb * pix(x + 8, c) : 0.0f));
            }
        };
        // a 4-column half: its c . g products, then its columns
        auto half = [&](auto gxc) {
            constexpr int gx = decltype(gxc)::value;
            if (((cols >> (4 * gx)) & 15u) == 0u) return;
            mx_floatx4 ca = {0.0f, 0.0f, 0.0f, 0.0f}, cc = {0.0f, 0.0f, 0.0f, 0.0f};
            if constexpr (FIN) {
#pragma unroll
                for (int ks = 0; ks < S::KS; ++ks) {
                    ca = __builtin_amdgcn_mfma_f32_16x16x4f32(cota(gx, ks), fb[ks], ca, 0, 0, 0);
                    cc = __builtin_amdgcn_mfma_f32_16x16x4f32(cota(gx + 2, ks), fb[ks], cc, 0, 0,
                                                              0);
                }
            }
            if ((cols >> (4 * gx)) & 1u) column(Int<4 * gx>{}, ca[0], cc[0]);
            if ((cols >> (4 * gx)) & 2u) column(Int<4 * gx + 1>{}, ca[1], cc[1]);
            if ((cols >> (4 * gx)) & 4u) column(Int<4 * gx + 2>{}, ca[2], cc[2]);
            if ((cols >> (4 * gx)) & 8u) column(Int<4 * gx + 3>{}, ca[3], cc[3]);
        };
        half(Int<0>{});
        half(Int<1>{});
        next();

        // the moments over the lane's two rows, as the reference's gradients
        // (rasterize.py:197-218, dL/dG = o dL/dalpha; the staged conic is
        // (-a/2, -b, -c/2)), then summed over the wave's four: row r of the
        // wave ends with values row_value(r) and 4 + row_value(r)
        const float ya = PLAIN || ha0 != 0.0f || ha1 != 0.0f ? dya : 0.0f;
        const float yb = PLAIN || hb0 != 0.0f || hb1 != 0.0f ? dyb : 0.0f;
        const float s0 = ha0 + hb0, sx = ha1 + hb1, sy = fmaf(ha0, ya, hb0 * yb);
        const float o = PLAIN ? 1.0f : r0.w;
        float v[8], h[4], q[2];
        v[0] = 2.0f * r1.x * sx + r1.y * sy;
        v[1] = r1.y * sx + 2.0f * r1.z * sy;
        v[2] = -0.5f * (ha2 + hb2);
        v[3] = -fmaf(ha1, ya, hb1 * yb);
        v[4] = -0.5f * fmaf(ha0 * ya, ya, (hb0 * yb) * yb);
        v[5] = PLAIN ? (s0 != 0.0f ? s0 / r0.w : 0.0f) : s0;
        v[6] = v[7] = 0.0f;
        if (!PLAIN) {
#pragma unroll
            for (int i = 0; i < 5; ++i) v[i] = (s0 != 0.0f || v[i] != 0.0f) ? o * v[i] : 0.0f;
        }
        reduce_step1<0, 3, 8, 6>(v, h);
        h[3] = 0.0f;
        reduce_step2<0, 2, 8>(h, q);
        const int rv = row_value(r);
        float* const row = L.out + j * S::NO;
        row[rv] = q[0];
        if (rv < 2) row[4 + rv] = q[1];
#pragma unroll
        for (int cb = 0; cb < S::CB; ++cb) {
            // dc: channels 16 cb + 4 r + i of entry j (sent pair by pair if not FIN)
            if (16 * cb + 4 * r < CHP) {
#pragma unroll
                for (int i = 0; i < 4; ++i) row[6 + 16 * cb + 4 * r + i] = FIN ? dc[cb][i] : 0.0f;
            }
        }
        if (r == 0) L.id[j] = __float_as_int(r1.w);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    }
}

// The atomics of the bucket whose gradients lie in LDS.  An instruction's lanes
// take whole entries, component by component: the atomics execute at 20 to 21 G
// 64-byte lines/s whatever a line holds (measured over 2 to 256 MiB, 4 to 16
// floats of a line), so an entry's components go out together and lie in as few
// lines as possible.  Memory operations complete in order, and a load issued
// behind atomics waits for them too: the caller sends a bucket's gradients
// once the loads of the next bucket have arrived, so that they drain under
// its arithmetic.
template <int CHP>
__device__ __forceinline__ void bwd_send(const BwdLds& L, const BwdOut& O) {
    using S = BwdShape<CHP>;
    const int lane = lane_again();
    auto part = [&](int first, int count, int per, int mul, float* base, int64_t stride) {
        const int e0 = (int)((uint32_t)(lane * mul) >> 16), c = lane - e0 * count;
        if (e0 >= per) return;
        for (int e = e0; e < kBucket; e += per) {
            const float val = L.out[e * S::NO + first + c];
            const int64_t id = L.id[e];
            if (id >= 0 && val != 0.0f) {
                float* dst = base + stride * id + c;
                if (first == 0 && !O.record)
                    dst = c < 2   ? O.xy + 2 * id + c
                          : c < 5 ? O.conic + 3 * id + (c - 2)
                                  : O.opac + id;
                atomicAdd(dst, val);
            }
        }
    };
    if (O.whole) {
        part(0, 6 + O.nc, O.per, O.mul, O.xy, O.stride);
    } else {
        part(0, 6, 10, 65536 / 6 + 1, O.xy, O.stride);
        part(6, O.nc, O.per, O.mul, O.feat, O.feat_stride);
    }
    // the next bucket's gradients overwrite these
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
}

constexpr float kTame = 1e15f;  // 32 products of two below it stay far inside float

constexpr int bwd_wide_waves(int chp) { return chp == 8 ? 5 : (chp == 16 ? 4 : 3); }

// One wave per quadrant, with no barrier and nothing shared between the
// quadrants of a tile: the wave reads the tile's list backmost first in
// chunks of 64, keeps the Gaussians that can reach its quadrant in a buffer
// in LDS (compacted, so every bucket but the last is full) and replays the
// buffer 16 entries at a time.  A needed list entry reaches 1.0 to 1.5 of a
// tile's four quadrants (1.06 with 1M Gaussians at 1080p), so summing the
// quadrants' gradients before the atomics would save little, while batches
// shared by the four waves cost four barriers each and leave 16 % of the
// bucket lanes empty (32 channels: 367 us, against 283).
//
// A Gaussian's sums take up to four float atomics per tile this way, a few more
// float32 steps for those that cover many tiles.  Against 64 bits, 48 passes of
// 8 and 16 channels over four scenes: 1.03 to 1.06 times the error of one atomic
// per tile in the mean; the most where a few large Gaussians carry the norm
// (scales 0.8e-6 -> 2.6e-6, quaternions 3.2e-6 -> 7.5e-6, features 0.8e-6 ->
// 1.8e-6); surfels and 32 channels as before.
template <int CHP>
__global__ __launch_bounds__(kWave, bwd_wide_waves(CHP)) void k_raster_bwd_wide(
    const float2* __restrict__ xy, const float4* __restrict__ co, const float* __restrict__ feat,
    int C, int c0, int nc, const int* __restrict__ ids, const int2* __restrict__ ranges,
    int64_t n, int64_t n_ids, const float* __restrict__ bg, int W, int H, int tiles_x, int slots,
    const float* __restrict__ final_T, const int* __restrict__ n_contrib,
    const float* __restrict__ grad_out, const float* __restrict__ grad_T,
    float* __restrict__ g_xy, float* __restrict__ g_conic, float* __restrict__ g_feat,
    float* __restrict__ g_opac, int gstride, int fstride, const int* __restrict__ order) {
    using S = BwdShape<CHP>;
    constexpr int GS = CHP < 16 ? CHP : 16;
    // wide blocks' cotangents pass through the records' space, 16 channels of
    // 64 pixels at a time, before the first entries are buffered
    constexpr int kRec = 9 * S::BUF;
    constexpr int kBuf = S::kNarrow || kRec >= kWave * GS ? kRec : kWave * GS;
    __shared__ __align__(16) float s_buf[kBuf];
    __shared__ __align__(16) float s_g[S::kNarrow ? kWave * CHP : 4];
    __shared__ __align__(16) float s_out[kBucket * S::NO];
    __shared__ int s_id[kBucket];
    const BwdLds L{reinterpret_cast<float4*>(s_buf), reinterpret_cast<float4*>(s_buf) + S::BUF,
                   reinterpret_cast<int*>(s_buf + 8 * S::BUF), s_g, s_out, s_id};

    // workgroups 32 i + 8 q + x: quadrant q of the tile in slot 8 i + x, so
    // a tile's quadrants run on one XCD close together
    const uint32_t bid = blockIdx.x;
    const int slot = (int)((bid & 7u) | ((bid >> 5) << 3)), quad = (int)(bid >> 3) & 3;
    if (slot >= slots) return;
    const int tile = __builtin_amdgcn_readfirstlane(tile_at(order, slot, slots, true));
    if (tile < 0) return;  // past the end of this XCD's band
    const int tx = tile % tiles_x, ty = tile / tiles_x;
    const int qx0 = tx * kTile + (quad & 1) * 8, qy0 = ty * kTile + (quad >> 1) * 8;
    const float* const gout = grad_out + c0;

    int start, num;
    tile_span(ranges[tile], n_ids, start, num);
    start = __builtin_amdgcn_readfirstlane(start);
    num = __builtin_amdgcn_readfirstlane(num);

    // the lane's own pixel (step lane % 16, row lane / 16): T and Q behind
    // the list's end and its contributor count
    BwdPixels P;
    BwdCot<CHP> g;
    bool fin = true;
    int top;  // list entries not read yet; later ones changed no pixel
    {
        const int lane = threadIdx.x, j = lane & 15, r = lane >> 4;
        const int opx = qx0 + (j & 7), opy = qy0 + 4 * (j >> 3) + r;
        const bool inside = opx < W && opy < H;
        // the pixel's loads issue together (clamped indices, masked after)
        const int64_t pid = inside ? (int64_t)opy * W + opx : 0;
        const float tf = final_T[pid];
        const int nct = n_contrib[pid];
        const float gt = grad_T ? grad_T[pid] : 0.0f;
        P.nc = inside ? nct : 0;
        int m = P.nc;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) m = max(m, __shfl_xor(m, o, kWave));
        top = min(__builtin_amdgcn_readfirstlane(m), num);
        if (top <= 0) return;
        // the quadrant's cotangents, from the lanes that own the pixels into
        // the operand layouts (zero outside the image or the block)
        float bg_dot = 0.0f;
        float* const buf = S::kNarrow ? s_g : s_buf;
#pragma unroll
        for (int cb = 0; cb < S::CB; ++cb) {
#pragma unroll
            for (int q = 0; q < GS; q += 4) {
                float v[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int ch = 16 * cb + q + i;
                    v[i] = (inside && ch < nc) ? gout[pid * C + min(ch, nc - 1)] : 0.0f;
                    fin = fin && fabsf(v[i]) < kTame;
                    if (bg && ch < nc) bg_dot = bg_dot + bg[c0 + ch] * v[i];
                }
                *reinterpret_cast<float4*>(buf + (4 * j + r) * GS + q) =
                    make_float4(v[0], v[1], v[2], v[3]);
            }
            // the wave's LDS accesses complete in order; the fence keeps the
            // compiler from moving the reads above the writes
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            if constexpr (!S::kNarrow) {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int s = 4 * (q & 1) + (j & 3) + 8 * (q >> 1);
#pragma unroll
                    for (int ks = 0; ks < GS / 4; ++ks)
                        g.a[q][4 * cb + ks] = buf[(4 * s + (j >> 2)) * GS + 4 * ks + r];
                }
#pragma unroll
                for (int s = 0; s < 16; ++s) g.b[s][cb] = buf[(4 * s + r) * GS + j];
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        }
        // The alpha output's cotangent enters once, with the first channel block.
        if (c0 == 0 && grad_T) bg_dot = bg_dot + gt;
        const float T = inside ? tf : 1.0f, Q = inside ? tf * bg_dot : 0.0f;
        fin = fin && fabsf(T) < 1e30f && fabsf(Q) < 1e30f;
        P.T[0] = quad_bcast<0>(T);
        P.T[1] = quad_bcast<1>(T);
        P.T[2] = quad_bcast<2>(T);
        P.T[3] = quad_bcast<3>(T);
        P.Q[0] = quad_bcast<0>(Q);
        P.Q[1] = quad_bcast<1>(Q);
        P.Q[2] = quad_bcast<2>(Q);
        P.Q[3] = quad_bcast<3>(Q);
#pragma unroll
        for (int x = 0; x < 8; ++x) P.px[x] = scalar_float((float)(qx0 + x) + 0.5f);
    }
    // No channel or cotangent so far reaches kTame: no c . g, and so no Q that a
    // pixel carries on, is infinite.  Once one does, every later bucket masks
    // each pair, for an infinite Q must not meet a weight of zero.
    bool tame = __ballot(!fin) == 0ull;
    BwdOut O;
    O.record = gstride > 0;
    O.xy = g_xy;
    O.conic = g_conic;
    O.opac = g_opac;
    O.feat = g_feat + c0;
    O.feat_stride = fstride;
    O.stride = gstride;
    O.nc = nc;
    O.C = C;
    // a block's channels follow the geometric gradients in its record
    O.whole = O.record && g_feat == g_xy + 6 && c0 == 0;
    const int comps = O.whole ? 6 + nc : nc;
    O.per = kWave / comps;
    O.mul = 65536 / comps + 1;

    // the next 64 list entries, backmost first: the lane's Gaussian (-1: none)
    // and its record and channels
    auto load_id = [&]() {
        const int k = top - 1 - lane_again();
        int id = -1;
        if (k >= 0) id = ids[start + k];
        return (uint32_t)id < (uint64_t)n ? id : -1;
    };
    int id = -1;
    float2 m;
    float4 c;
    auto load_record = [&]() {
        const int64_t at = max(id, 0);
        m = xy[at];
        c = co[at];
    };
    id = load_id();
    load_record();

    int cnt = 0;             // buffered entries
    bool all_plain = true;   // every one of them is plain
    bool pending = false;    // a bucket's gradients wait in LDS
    do {
        // buffer those that reach the quadrant
        {
            const int lane = lane_again();
            const bool keep = id >= 0 && quadrant_reached(m.x, m.y, c, qx0, qy0);
            const uint64_t kept = __ballot(keep);
            bool plain = true;
            if (keep) {
                const float thr = alpha_floor_power(c.w);
                const int at = cnt + __popcll(kept & ((1ull << lane) - 1ull));
                L.r0[at] = make_float4(m.x, m.y, thr, c.w);
                L.r1[at] = make_float4(-0.5f * c.x, -c.y, -0.5f * c.z, __int_as_float(id));
                L.k[at] = top - 1 - lane;
                plain = plain_gaussian<0>(m.x, m.y, c, thr, nullptr);
            }
            all_plain = (cnt == 0 || all_plain) && __ballot(!plain) == 0ull;
            cnt += __popcll(kept);
            top -= kWave;
        }
        const bool end = top <= 0;
        const int used = end ? cnt : cnt & ~(kBucket - 1);
        if (end && (cnt & (kBucket - 1)) != 0) {
            // fill the last bucket with records no pixel can take (alpha bound
            // +inf)
            const int at = cnt + lane_again();
            if (at < ((cnt + kBucket - 1) & ~(kBucket - 1))) {
                L.r0[at] = make_float4(0.0f, 0.0f, __builtin_huge_valf(), 0.0f);
                L.r1[at] = make_float4(0.0f, 0.0f, 0.0f, __int_as_float(-1));
                L.k[at] = 0x7fffffff;
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        if (!end) id = load_id();
        if (!end && used == 0) load_record();
#pragma unroll 1
        for (int b0 = 0; b0 < used; b0 += kBucket) {
            const int lane = lane_again(), j = lane & 15, r = lane >> 4;
            // the next entries' records are loaded by the chunk's last bucket
            const bool fetch = !end && b0 + kBucket >= used;
            auto next = [&]() {
                if (fetch) {
                    load_record();
                } else {  // not read; no register holds a value over the bucket
                    asm volatile("" : "=v"(m.x), "=v"(m.y), "=v"(c.x), "=v"(c.y), "=v"(c.z),
                                      "=v"(c.w));
                }
            };
            // the entry's channels 4 ks + r, the B operand of c . g
            float fb[S::KS];
            bool ffin = true;
            {
                const float* const fp =
                    feat + (int64_t)max(__float_as_int(L.r1[b0 + j].w), 0) * C + c0;
#pragma unroll
                for (int ks = 0; ks < S::KS; ++ks) fb[ks] = fp[min(4 * ks + r, nc - 1)];
#pragma unroll
                for (int ks = 0; ks < S::KS; ++ks) {
                    fb[ks] = 4 * ks + r < nc ? fb[ks] : 0.0f;
                    ffin = ffin && fabsf(fb[ks]) < kTame;
                }
            }
            tame = tame && __ballot(!ffin) == 0ull;
            if (pending) bwd_send<CHP>(L, O);
            pending = true;
            const float* const ft = feat + c0;
            if (tame && all_plain)
                bwd_bucket<CHP, true, true>(L, b0, cnt, P, g, fb, O, gout, ft, qx0, qy0, W, H,
                                            next);
            else if (tame)
                bwd_bucket<CHP, false, true>(L, b0, cnt, P, g, fb, O, gout, ft, qx0, qy0, W, H,
                                            next);
            else
                bwd_bucket<CHP, false, false>(L, b0, cnt, P, g, fb, O, gout, ft, qx0, qy0, W, H,
                                            next);
        }
        if (end) break;
        // the entries left over move to the front
        if (used > 0) {
            const int j = lane_again(), left = cnt - used;
            if (j < left) {
                const float4 a = L.r0[used + j], b = L.r1[used + j];
                const int k = L.k[used + j];
                L.r0[j] = a;
                L.r1[j] = b;
                L.k[j] = k;
            }
            cnt = left;
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        }
    } while (true);
    if (pending) bwd_send<CHP>(L, O);
}

// Matrix-core forward for 32-channel blocks.  The per-pixel loop keeps every
// decision of fwd_pair on the vector ALU (power, exp, alpha, the early stop,
// T, depth, the last contributor), so final_T, n_contrib, alpha and depth
// are the VALU path's bits; only the channel sums move.  For a group of 16
// list entries the replay writes each pair's weight w = alpha T (zero where
// the pixel does not composite) into a per-wave LDS tile, then
//   out[c][p] += sum over the group of f[g][c] w[g][p]
// runs as 32 v_mfma_f32_16x16x4_f32 (A = features, 16 channels x 4 entries;
// B = weights, 4 entries x 16 pixels; 2 channel blocks x 4 pixel blocks of
// accumulators).  Lane l holds channels 16 cb + 4 (l / 16) + i of quadrant
// pixel 16 pb + l % 16.  The features are staged row-major with a row
// stride of 48 floats (rows four slots apart share no bank window) and the
// tile with a row stride of 80 (the four rows one operand read touches hit
// disjoint banks).  The sums add in another order than the sequential
// multiply-adds of fwd_pair: channels agree with it to float32 rounding.
// Batches holding a non-finite (or |f| >= 1e30) feature add their groups on
// the vector ALU into the same accumulators, pair by pair in list order and
// only where w != 0, so 0 * inf never reaches a pixel that skipped the
// Gaussian.
constexpr int kMfBatch = 128;  // list entries staged per batch
constexpr int kMfFeat = 48;    // feature row stride (floats)
constexpr int kMfTile = 80;    // weight tile row stride (floats)

// One (pixel, Gaussian) step of fwd_pair without the channel sums: returns
// the weight the pixel gives the Gaussian (zero unless it composites).
template <bool DEPTH, bool PLAIN>
__device__ __forceinline__ float fwd_weight(const float4& r0, const float4& r1, int off,
                                            float pxf, float pyf, float& T, float& dacc,
                                            int& last_off, uint64_t& alive) {
    const float dx = r0.x - pxf, dy = r0.y - pyf;
    const float power = splat_power(r1.x, r1.y, r1.z, dx, dy);
    const uint64_t live =
        PLAIN ? alive & __ballot(!(power < r0.z))
              : alive & __ballot(!(power > 0.0f)) & __ballot(!(power < r0.z));
    const float e = PLAIN ? splat_exp_core(power) : splat_exp_sel(power);
    const float alpha = fminf(0.99f, r0.w * e);
    const uint64_t pass = live & __ballot(!(alpha < 1.0f / 255.0f));
    const float next_T = T * (1.0f - alpha);
    const uint64_t lt = __ballot(next_T < 1e-4f);
    alive &= ~(pass & lt);
    const bool add = __builtin_amdgcn_inverse_ballot_w64(pass & ~lt);
    const float w = alpha * T;
    const float wa = add ? w : 0.0f;
    if (DEPTH) {
        if (PLAIN) {
            dacc = fmaf(r1.w, wa, dacc);
        } else {
            const float d2 = fmaf(r1.w, w, dacc);
            dacc = add ? d2 : dacc;
        }
    }
    T = add ? next_T : T;
    last_off = add ? off : last_off;
    return wa;
}

// The walk of one quadrant wave for the matrix-core forward, in groups of
// 16 list entries: the replay (two entries per round, the next pair's
// records read before this pair is evaluated) fills the weight tile; rows
// past the entries replayed (the group's end, or the wave's early stop)
// are zero.  FINITE: every staged feature is finite and below 1e30.
template <bool DEPTH, bool PLAIN, bool FINITE>
__device__ __forceinline__ void fwd_walk_mx(const uint32_t* list, int cnt, const float4* s_r0,
                                            const float4* s_r1, const float* s_feat,
                                            int pad_slot, float (*tile)[kMfTile], float pxf,
                                            float pyf, int lane, float& T, float& dacc,
                                            int& last_off, uint64_t& alive,
                                            mx_floatx4 (&acc)[2][4]) {
    const int pad = pad_slot * 16;
    const int row = lane & 15, kq = lane >> 4;
#pragma unroll 1
    for (int i0 = 0; i0 < cnt; i0 += kMxGroup) {
        const int ng = min(kMxGroup, cnt - i0);
        int oa = list[i0], ob = 1 < ng ? list[i0 + 1] : pad;
        float4 a0 = rec_at(s_r0, oa), a1 = rec_at(s_r1, oa);
        int j = 0;
#pragma unroll 1
        while (j < ng) {
            const int na = j + 2 < ng ? list[i0 + j + 2] : pad;
            const int nb = j + 3 < ng ? list[i0 + j + 3] : pad;
            const float4 b0 = rec_at(s_r0, ob), b1 = rec_at(s_r1, ob);
            tile[j][lane] =
                fwd_weight<DEPTH, PLAIN>(a0, a1, oa, pxf, pyf, T, dacc, last_off, alive);
            a0 = rec_at(s_r0, na);
            a1 = rec_at(s_r1, na);
            tile[j + 1][lane] =
                fwd_weight<DEPTH, PLAIN>(b0, b1, ob, pxf, pyf, T, dacc, last_off, alive);
            oa = na;
            ob = nb;
            j += 2;
            if (alive == 0ull) break;
        }
#pragma unroll 1
        for (; j < kMxGroup; ++j) tile[j][lane] = 0.0f;
        // the wave's LDS accesses complete in order; the fence keeps the
        // compiler from moving the reads below above the writes
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        if constexpr (FINITE) {
#pragma unroll 1
            for (int ks = 0; ks < 4; ++ks) {
                const int r = 4 * ks + kq;
                const int slot = r < ng ? (list[i0 + r] >> 4) : pad_slot;
                const float fa0 = s_feat[slot * kMfFeat + row];
                const float fa1 = s_feat[slot * kMfFeat + 16 + row];
#pragma unroll
                for (int pb = 0; pb < 4; ++pb) {
                    const float wb = tile[r][16 * pb + row];
                    acc[0][pb] = __builtin_amdgcn_mfma_f32_16x16x4f32(fa0, wb, acc[0][pb], 0, 0, 0);
                    acc[1][pb] = __builtin_amdgcn_mfma_f32_16x16x4f32(fa1, wb, acc[1][pb], 0, 0, 0);
                }
            }
        } else {
#pragma unroll 1
            for (int r = 0; r < ng; ++r) {
                const int slot = list[i0 + r] >> 4;
                float wv[4];
#pragma unroll
                for (int pb = 0; pb < 4; ++pb) wv[pb] = tile[r][16 * pb + row];
#pragma unroll
                for (int cb = 0; cb < 2; ++cb) {
                    const float4 f =
                        *reinterpret_cast<const float4*>(s_feat + slot * kMfFeat + 16 * cb + 4 * kq);
#pragma unroll
                    for (int pb = 0; pb < 4; ++pb) {
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const float v = fmaf(comp4(f, i), wv[pb], acc[cb][pb][i]);
                            acc[cb][pb][i] = wv[pb] != 0.0f ? v : acc[cb][pb][i];
                        }
                    }
                }
            }
        }
        // the next group's replay overwrites the tile
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        if (alive == 0ull) return;
    }
}

template <bool DEPTH>
__global__ __launch_bounds__(kThreads, 3) void k_raster_fwd_mx(
    const float2* __restrict__ xy, const float4* __restrict__ co, const float* __restrict__ feat,
    int C, int c0, int nc, const float* __restrict__ depths, const int* __restrict__ ids,
    const int2* __restrict__ ranges, int64_t n, int64_t n_ids, const float* __restrict__ bg,
    int W, int H, int tiles_x, float* __restrict__ out, float* __restrict__ final_T,
    int* __restrict__ n_contrib, float* __restrict__ depth_out, float* __restrict__ alpha_out,
    const int* __restrict__ order, int* __restrict__ work) {
    constexpr int BB = kMfBatch;
    constexpr int NLW = BB / kWave;  // waves that stage records
    constexpr int F4 = 8;            // float4 pieces of a 32-channel row
    // entry BB of the records (and feature row BB, zeros) is the padding
    __shared__ float4 s_r0[BB + 1];  // mean x, mean y, log-alpha bound, opacity
    __shared__ float4 s_r1[BB + 1];  // -a/2, -b, -c/2 (conic), depth
    __shared__ __align__(16) float s_feat[(BB + 1) * kMfFeat];
    __shared__ float s_tile[kWaves][kMxGroup][kMfTile];
    __shared__ uint64_t s_mask[kWaves][NLW];
    __shared__ uint32_t s_list[kWaves][BB + 4];
    __shared__ __align__(16) uint32_t s_alive[kWaves];
    __shared__ __align__(16) uint32_t s_plain[kWaves];
    __shared__ __align__(16) uint32_t s_finite[kWaves];

    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int tile = __builtin_amdgcn_readfirstlane(tile_at(order, blockIdx.x, gridDim.x, false));
    const int tx = tile % tiles_x, ty = tile / tiles_x;
    const int px0 = tx * kTile, py0 = ty * kTile;
    const int qx0 = px0 + (wave & 1) * 8, qy0 = py0 + (wave >> 1) * 8;
    const int px = qx0 + (lane & 7);
    const int py = qy0 + (lane >> 3);
    const bool inside = px < W && py < H;
    const float pxf = (float)px + 0.5f, pyf = (float)py + 0.5f;

    int start, num;
    tile_span(ranges[tile], n_ids, start, num);

    float T = 1.0f, dacc = 0.0f;
    mx_floatx4 acc[2][4];
#pragma unroll
    for (int cb = 0; cb < 2; ++cb)
#pragma unroll
        for (int pb = 0; pb < 4; ++pb) acc[cb][pb] = mx_floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    int last = 0;
    uint64_t alive = __ballot(inside);
    if (tid == 0) {
        s_r0[BB] = make_float4(0.0f, 0.0f, __builtin_huge_valf(), 0.0f);
        s_r1[BB] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
    if (tid < kMfFeat) s_feat[BB * kMfFeat + tid] = 0.0f;
    // rows of 32 channels at 16-byte aligned addresses: float4 loads
    const bool vec4 = nc >= 4 * F4 && ((C | c0) & 3) == 0 && ((uintptr_t)feat & 15u) == 0;

    for (int base = 0; base < num; base += BB) {
        if (lane == 0) s_alive[wave] = alive != 0ull;
        __syncthreads();
        const uint4 al = *reinterpret_cast<const uint4*>(s_alive);
        if ((al.x | al.y | al.z | al.w) == 0u) break;  // all 256 pixels done
        uint32_t qm = 0;
        bool plain = true, finite = true;
        if (tid < BB) {
            const int k = base + tid;
            if (k < num) {
                const int g = ids[start + k];
                if ((uint32_t)g < (uint64_t)n) {
                    const float2 m = xy[g];
                    const float4 c = co[g];
                    const float thr = alpha_floor_power(c.w);
                    s_r0[tid] = make_float4(m.x, m.y, thr, c.w);
                    const float dz = DEPTH ? depths[g] : 0.0f;
                    s_r1[tid] = make_float4(-0.5f * c.x, -c.y, -0.5f * c.z, dz);
                    qm = quadrant_mask(m.x, m.y, c, px0, py0);
                    plain = plain_gaussian<0>(m.x, m.y, c, thr, nullptr) && fabsf(dz) < 1e30f;
                }
            }
        }
        // the features: thread t stages piece t % 8 of entries t / 8 + 32 i
        constexpr int NIT = BB * F4 / kThreads;
        if (vec4) {
            // whole aligned rows: the id loads, then the 16-byte feature
            // loads, each issued together (invalid entries read row 0 and
            // are dropped)
            int g[NIT];
            float4 v[NIT];
#pragma unroll
            for (int it = 0; it < NIT; ++it) {
                const int k = base + (tid >> 3) + (kThreads / F4) * it;
                g[it] = ids[start + min(k, num - 1)];
                if (k >= num) g[it] = -1;
            }
#pragma unroll
            for (int it = 0; it < NIT; ++it) {
                const int64_t gi = (uint32_t)g[it] < (uint64_t)n ? g[it] : 0;
                v[it] = *reinterpret_cast<const float4*>(feat + gi * C + c0 + 4 * (tid & 7));
            }
#pragma unroll
            for (int it = 0; it < NIT; ++it) {
                if ((uint32_t)g[it] < (uint64_t)n) {
                    const int j = (tid >> 3) + (kThreads / F4) * it;
                    *reinterpret_cast<float4*>(s_feat + j * kMfFeat + 4 * (tid & 7)) = v[it];
                    finite = finite && fabsf(v[it].x) < 1e30f && fabsf(v[it].y) < 1e30f &&
                             fabsf(v[it].z) < 1e30f && fabsf(v[it].w) < 1e30f;
                }
            }
        } else {
#pragma unroll
        for (int it = 0; it < NIT; ++it) {
            const int j = (tid >> 3) + (kThreads / F4) * it, q = tid & 7;
            const int k = base + j;
            if (k < num) {
                const int g = ids[start + k];
                if ((uint32_t)g < (uint64_t)n) {
                    const float* f = feat + (int64_t)g * C + c0 + 4 * q;
                    float4 v;
                    v.x = 4 * q < nc ? f[0] : 0.0f;
                    v.y = 4 * q + 1 < nc ? f[1] : 0.0f;
                    v.z = 4 * q + 2 < nc ? f[2] : 0.0f;
                    v.w = 4 * q + 3 < nc ? f[3] : 0.0f;
                    *reinterpret_cast<float4*>(s_feat + j * kMfFeat + 4 * q) = v;
                    finite = finite && fabsf(v.x) < 1e30f && fabsf(v.y) < 1e30f &&
                             fabsf(v.z) < 1e30f && fabsf(v.w) < 1e30f;
                }
            }
        }
        }
        if (wave < NLW) {
#pragma unroll
            for (int q = 0; q < kWaves; ++q) {
                const uint64_t b = __ballot((qm >> q) & 1u);
                if (lane == 0) s_mask[q][wave] = b;
            }
        }
        const uint64_t np = __ballot(!plain), nf = __ballot(!finite);
        if (lane == 0) {
            s_plain[wave] = np == 0ull;
            s_finite[wave] = nf == 0ull;
        }
        __syncthreads();
        const uint4 pl = *reinterpret_cast<const uint4*>(s_plain);
        const uint4 fi = *reinterpret_cast<const uint4*>(s_finite);
        const bool batch_plain = (pl.x & pl.y & pl.z & pl.w) != 0u;
        const bool batch_finite = (fi.x & fi.y & fi.z & fi.w) != 0u;
        if (alive == 0ull) continue;
        const int cnt = build_list<NLW, false>(s_mask[wave], s_list[wave], lane, 16, BB);
        int last_off = -1;
        if (batch_finite) {
            if (batch_plain)
                fwd_walk_mx<DEPTH, true, true>(s_list[wave], cnt, s_r0, s_r1, s_feat, BB,
                                               s_tile[wave], pxf, pyf, lane, T, dacc, last_off,
                                               alive, acc);
            else
                fwd_walk_mx<DEPTH, false, true>(s_list[wave], cnt, s_r0, s_r1, s_feat, BB,
                                                s_tile[wave], pxf, pyf, lane, T, dacc, last_off,
                                                alive, acc);
        } else {
            fwd_walk_mx<DEPTH, false, false>(s_list[wave], cnt, s_r0, s_r1, s_feat, BB,
                                             s_tile[wave], pxf, pyf, lane, T, dacc, last_off,
                                             alive, acc);
        }
        if (last_off >= 0) last = base + (last_off >> 4) + 1;
    }
    if (inside && c0 == 0) {
        const int64_t pid = (int64_t)py * W + px;
        final_T[pid] = T;
        n_contrib[pid] = last;
        if (alpha_out) alpha_out[pid] = 1.0f - T;
        if (DEPTH) {
            const float al = 1.0f - T;
            depth_out[pid] = al > 1e-6f ? dacc / al : 0.0f;
        }
    }
    if (work) store_tile_work(work, tile, last, wave, lane);
    // channel results: lane l holds quadrant pixel 16 pb + l % 16, channels
    // 16 cb + 4 (l / 16) + i; that pixel's T is lane (16 pb + l % 16)'s
    const int row = lane & 15, kq = lane >> 4;
    // whole 16-byte pieces when the block is 32 aligned channels
    const bool vec_out = nc == 32 && (C & 3) == 0 && (c0 & 3) == 0 &&
                         (reinterpret_cast<uintptr_t>(out) & 15u) == 0;
#pragma unroll
    for (int pb = 0; pb < 4; ++pb) {
        const int q = 16 * pb + row;
        const float Tq = __shfl(T, q, kWave);
        const int bx = qx0 + (q & 7), by = qy0 + (q >> 3);
        if (bx < W && by < H) {
            float* o = out + ((int64_t)by * W + bx) * C + c0;
#pragma unroll
            for (int cb = 0; cb < 2; ++cb) {
                const int ch0 = 16 * cb + 4 * kq;
                float v[4];
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    v[i] = acc[cb][pb][i] + Tq * (bg && ch0 + i < nc ? bg[c0 + ch0 + i] : 0.0f);
                if (vec_out) {
                    *reinterpret_cast<float4*>(o + ch0) = make_float4(v[0], v[1], v[2], v[3]);
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (ch0 + i < nc) o[ch0 + i] = v[i];
                }
            }
        }
    }
}

// One workgroup per band (the forward's order, or the backward's).
template <bool BWD>
__global__ __launch_bounds__(kOrderThreads) void k_tile_order(const int2* __restrict__ ranges,
                                                              const int* __restrict__ work,
                                                              int64_t n_ids, int tiles,
                                                              int* __restrict__ order) {
    __shared__ uint32_t s_order[tile_order_lds_words<kOrderThreads>()];
    tile_order_band<BWD>(blockIdx.x, ranges, work, n_ids, tiles, order, s_order);
}

// The gradient outputs to clear: one record (p[0], n[0] floats, 16-byte
// aligned, n[0] a multiple of 4) and perhaps the features' array (p[2]), or
// four arrays.
struct ZeroGrads {
    float* p[4];
    int64_t n[4];
    bool record;
};

// The backward's prologue in one launch: workgroups [0, bands) build the
// backward's tile order from the forward's per-tile work (bands = 0 without
// one), the others clear the gradient outputs (a fill kernel rather than
// hipMemsetAsync, so the call can sit inside a captured graph).  The order's
// few long-lived workgroups run beside the clearing instead of after it.
__global__ __launch_bounds__(kOrderThreads) void k_bwd_prologue(ZeroGrads z, int bands,
                                                                const int* __restrict__ work,
                                                                int64_t n_ids, int tiles,
                                                                int* __restrict__ order) {
    __shared__ uint32_t s_order[tile_order_lds_words<kOrderThreads>()];
    if ((int)blockIdx.x < bands) {
        tile_order_band<true>(blockIdx.x, nullptr, work, n_ids, tiles, order, s_order);
        return;
    }
    const int64_t b = (int64_t)blockIdx.x - bands;
    const int64_t stride = ((int64_t)gridDim.x - bands) * kOrderThreads;
    if (z.record) {
        float4* a = reinterpret_cast<float4*>(z.p[0]);
        for (int64_t i = b * kOrderThreads + threadIdx.x; i < z.n[0] / 4; i += stride)
            a[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        z.n[0] = 0;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r)
        for (int64_t i = b * kOrderThreads + threadIdx.x; i < z.n[r]; i += stride) z.p[r][i] = 0.0f;
}

// The geometric part of a gradient record as separate arrays, a lane per
// Gaussian: 32 bytes read (the record's first two 16-byte pieces) and 24
// written; bound by the launch (5 us at 200k Gaussians, which the record
// saves many times over in the backward's atomics).
__global__ __launch_bounds__(256) void k_split_grads(int64_t n, const float* __restrict__ rec,
                                                     int stride, float2* __restrict__ g_xy,
                                                     float* __restrict__ g_conic,
                                                     float* __restrict__ g_opac) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const float4* const r = reinterpret_cast<const float4*>(rec + i * stride);
    const float4 a = r[0], b = r[1];
    g_xy[i] = make_float2(a.x, a.y);
    g_conic[3 * i] = a.z;
    g_conic[3 * i + 1] = a.w;
    g_conic[3 * i + 2] = b.x;
    g_opac[i] = b.y;
}

int pick_ch(int nc) {
    if (nc <= 1) return 1;
    if (nc <= 2) return 2;
    if (nc <= 3) return 3;
    if (nc <= 4) return 4;
    if (nc <= 8) return 8;
    if (nc <= 16) return 16;
    return 32;
}
constexpr int kMaxChunk = 32;

template <int CH>
void launch_fwd(dim3 grid, hipStream_t st, bool depth, const float2* xy, const float4* co,
                const float* feat, int C, int c0, int nc, const float* depths, const int* ids,
                const int2* ranges, int64_t n, int64_t n_ids, const float* bg, int W, int H,
                int tiles_x, float* out, float* fT, int* ncon, float* dout, float* aout,
                const int* order, int* work) {
    if constexpr (CH == 32) {
        if (depth)
            hipLaunchKernelGGL((k_raster_fwd_mx<true>), grid, dim3(kThreads), 0, st, xy, co, feat,
                               C, c0, nc, depths, ids, ranges, n, n_ids, bg, W, H, tiles_x, out,
                               fT, ncon, dout, aout, order, work);
        else
            hipLaunchKernelGGL((k_raster_fwd_mx<false>), grid, dim3(kThreads), 0, st, xy, co,
                               feat, C, c0, nc, depths, ids, ranges, n, n_ids, bg, W, H, tiles_x,
                               out, fT, ncon, dout, aout, order, work);
        return;
    }
    if constexpr (CH <= 4) {
        const int tiles = (int)grid.x;
        const bool all = tiles <= split_tiles(CH + (depth ? 1 : 0));
        if (C <= 4 && (all || (order && tiles <= kChooseTiles))) {
            auto* const kernel = all ? (depth ? k_raster_fwd_split<CH, true>
                                              : k_raster_fwd_split<CH, false>)
                                     : (depth ? k_raster_fwd_choose<CH, true>
                                              : k_raster_fwd_choose<CH, false>);
            hipLaunchKernelGGL(kernel, dim3(32u * (((unsigned)tiles + 7u) / 8u)), dim3(kThreads),
                               0, st, xy, co, feat, C, c0, nc, depths, ids, ranges, n, n_ids, bg,
                               W, H, tiles_x, out, fT, ncon, dout, aout, order, work, tiles);
            return;
        }
    }
    if constexpr (CH < 32) {
        if (depth)
            hipLaunchKernelGGL((k_raster_fwd<CH, true>), grid, dim3(kThreads), 0, st, xy, co,
                               feat, C, c0, nc, depths, ids, ranges, n, n_ids, bg, W, H, tiles_x,
                               out, fT, ncon, dout, aout, order, work);
        else
            hipLaunchKernelGGL((k_raster_fwd<CH, false>), grid, dim3(kThreads), 0, st, xy, co,
                               feat, C, c0, nc, depths, ids, ranges, n, n_ids, bg, W, H, tiles_x,
                               out, fT, ncon, dout, aout, order, work);
    }
}

template <int CH>
void launch_bwd(int slots, hipStream_t st, const float2* xy, const float4* co, const float* feat,
                int C, int c0, int nc, const int* ids, const int2* ranges, int64_t n,
                int64_t n_ids, const float* bg, int W, int H, int tiles_x, const float* fT,
                const int* ncon, const float* gout, const float* gT, float* gxy, float* gcon,
                float* gfeat, float* gop, int gstride, int fstride, const int* order) {
    if constexpr (CH > 4)
        // four quadrant workgroups per tile slot, slots in groups of eight (XCDs)
        hipLaunchKernelGGL((k_raster_bwd_wide<CH>), dim3(32u * (((unsigned)slots + 7u) / 8u)),
                           dim3(kWave), 0, st, xy, co, feat, C, c0, nc, ids, ranges, n, n_ids, bg,
                           W, H, tiles_x, slots, fT, ncon, gout, gT, gxy, gcon,
                           gfeat ? gfeat : gxy + 6, gop, gstride, fstride, order);
    else
        hipLaunchKernelGGL((k_raster_bwd<CH>), dim3((unsigned)slots), dim3(kThreads), 0, st, xy,
                           co, feat, C, c0, nc, ids, ranges, n, n_ids, bg, W, H, tiles_x, fT,
                           ncon, gout, gT, gxy, gcon, gfeat, gop, gstride, order);
}

inline bool aligned16(const void* p) { return ((uintptr_t)p & 15u) == 0; }
inline bool aligned8(const void* p) { return ((uintptr_t)p & 7u) == 0; }

// The backward into the outputs that the entry points accept; feature_stride:
// floats from one Gaussian's feature gradient to the next.
int raster_bwd(int64_t n, int32_t C, const float* means2d, const float* conic_opacity,
                   const float* features, const int32_t* sorted_ids, int64_t num_ids,
                   const int32_t* tile_ranges,
                   const float* background, int32_t width, int32_t height, const float* final_T,
                   const int32_t* n_contrib, const float* grad_out, const float* grad_final_T,
                   float* g_means2d, float* g_conics, float* g_features, float* g_opacities,
                   int32_t grad_stride, int32_t feature_stride, int32_t* tile_order,
                   void* stream) {
    if (n < 0 || num_ids < 0 || C <= 0 || width <= 0 || height <= 0) return GSX_ERR_INVALID;
    if (!tile_ranges || !final_T || !n_contrib || !grad_out) return GSX_ERR_INVALID;
    const bool rec = grad_stride > 0;
    if (n > 0 && (!means2d || !conic_opacity || !features || !g_means2d ||
                  (!rec && (!g_conics || !g_features || !g_opacities))))
        return GSX_ERR_INVALID;
    if (num_ids > 0 && !sorted_ids) return GSX_ERR_INVALID;
    if (!aligned8(means2d) || !aligned16(conic_opacity) || !aligned8(tile_ranges))
        return GSX_ERR_INVALID;
    hipStream_t st = (hipStream_t)stream;
    if (n == 0) return GSX_OK;
    const int tiles_x = (width + kTile - 1) / kTile;
    const int tiles_y = (height + kTile - 1) / kTile;
    const int tiles = tiles_x * tiles_y;
    // tile_order: [0, T) the forward's bounds, [T, T + 16 ceil(T / 8)) this
    // call's order, one entry per workgroup
    int* const order = tile_order ? tile_order + tiles : nullptr;
    const int slots = order ? (int)(tile_order_words(tiles) - tiles) : tiles;
    {
        // gradient clearing and the tile order in one launch
        ZeroGrads z{};
        z.record = rec;
        if (rec) {
            z.p[0] = g_means2d;
            z.n[0] = (int64_t)grad_stride * n;
            z.p[2] = g_features;
            z.n[2] = g_features ? (int64_t)feature_stride * n : 0;
        } else {
            z.p[0] = g_means2d;
            z.n[0] = 2 * n;
            z.p[1] = g_conics;
            z.n[1] = 3 * n;
            z.p[2] = g_features;
            z.n[2] = (int64_t)C * n;
            z.p[3] = g_opacities;
            z.n[3] = n;
        }
        const int64_t most =
            rec ? std::max(z.n[0] / 4, z.n[2]) : std::max<int64_t>((int64_t)C, 3) * n;
        const int bands = order ? kOrderBands : 0;
        const unsigned blocks =
            (unsigned)std::min<int64_t>((most + kOrderThreads - 1) / kOrderThreads, 2048);
        hipLaunchKernelGGL(k_bwd_prologue, dim3(blocks + (unsigned)bands), dim3(kOrderThreads), 0,
                           st, z, bands, (const int*)tile_order, num_ids, tiles, order);
        GSX_LAUNCH_CHECK();
    }
    for (int c0 = 0; c0 < C; c0 += kMaxChunk) {
        const int nc = (C - c0 < kMaxChunk) ? C - c0 : kMaxChunk;
        switch (pick_ch(nc)) {
#define GSX_BWD_CASE(V)                                                                          \
    case V:                                                                                      \
        launch_bwd<V>(slots, st, (const float2*)means2d, (const float4*)conic_opacity, features, \
                      C, c0, nc, sorted_ids, (const int2*)tile_ranges, n, num_ids, background,   \
                      width, height, tiles_x, final_T, n_contrib, grad_out, grad_final_T,        \
                      g_means2d, g_conics, g_features, g_opacities, grad_stride, feature_stride, \
                      order);                                                                    \
        break;
            GSX_BWD_CASE(1)
            GSX_BWD_CASE(2)
            GSX_BWD_CASE(3)
            GSX_BWD_CASE(4)
            GSX_BWD_CASE(8)
            GSX_BWD_CASE(16)
            GSX_BWD_CASE(32)
#undef GSX_BWD_CASE
            default:
                return GSX_ERR_INVALID;
        }
        GSX_LAUNCH_CHECK();
    }
    return GSX_OK;
}

}  // namespace

extern "C" {

int gsx_raster_fwd(int64_t n, int32_t C, const float* means2d, const float* conic_opacity,
                   const float* features, const float* depths, const int32_t* sorted_ids,
                   int64_t num_ids, const int32_t* tile_ranges, const float* background,
                   int32_t width,
                   int32_t height, float* out, float* final_T, int32_t* n_contrib,
                   float* depth_out, float* alpha_out, int32_t* tile_order, int32_t order_ready,
                   void* stream) {
    if (n < 0 || num_ids < 0 || C <= 0 || width <= 0 || height <= 0) return GSX_ERR_INVALID;
    if (!tile_ranges || !out || !final_T || !n_contrib) return GSX_ERR_INVALID;
    if (n > 0 && (!means2d || !conic_opacity || !features)) return GSX_ERR_INVALID;
    if (num_ids > 0 && !sorted_ids) return GSX_ERR_INVALID;
    if (n == 0) num_ids = 0;
    if (depths && !depth_out) return GSX_ERR_INVALID;
    if (!aligned8(means2d) || !aligned16(conic_opacity) || !aligned8(tile_ranges))
        return GSX_ERR_INVALID;
    hipStream_t st = (hipStream_t)stream;
    const int tiles_x = (width + kTile - 1) / kTile;
    const int tiles_y = (height + kTile - 1) / kTile;
    const dim3 grid((unsigned)(tiles_x * tiles_y));
    const int tiles = tiles_x * tiles_y;
    // tile_order: [0, T) the bounds this call writes, [T, 2T) its order
    // (order_ready: gsx_bin_tiles_async wrote it for these ranges)
    int* const order = tile_order ? tile_order + tiles : nullptr;
    if (order && !order_ready) {
        hipLaunchKernelGGL(k_tile_order<false>, dim3(kOrderBands), dim3(kOrderThreads), 0, st,
                           (const int2*)tile_ranges, (const int*)nullptr, num_ids, tiles, order);
        GSX_LAUNCH_CHECK();
    }
    for (int c0 = 0; c0 < C; c0 += kMaxChunk) {
        const int nc = (C - c0 < kMaxChunk) ? C - c0 : kMaxChunk;
        const bool depth = depths && c0 == 0;
        int* work = (tile_order && c0 == 0) ? tile_order : nullptr;
        switch (pick_ch(nc)) {
#define GSX_FWD_CASE(V)                                                                          \
    case V:                                                                                      \
        launch_fwd<V>(grid, st, depth, (const float2*)means2d, (const float4*)conic_opacity,     \
                      features, C, c0, nc, depths, sorted_ids, (const int2*)tile_ranges, n,      \
                      num_ids, background, width, height, tiles_x, out, final_T, n_contrib,      \
                      depth_out, alpha_out, order, work);                                        \
        break;
            GSX_FWD_CASE(1)
            GSX_FWD_CASE(2)
            GSX_FWD_CASE(3)
            GSX_FWD_CASE(4)
            GSX_FWD_CASE(8)
            GSX_FWD_CASE(16)
            GSX_FWD_CASE(32)
#undef GSX_FWD_CASE
            default:
                return GSX_ERR_INVALID;
        }
        GSX_LAUNCH_CHECK();
    }
    return GSX_OK;
}

int64_t gsx_tile_order_words(int32_t width, int32_t height) {
    if (width <= 0 || height <= 0) return 0;
    const int64_t tiles =
        (int64_t)((width + kTile - 1) / kTile) * (int64_t)((height + kTile - 1) / kTile);
    return tile_order_words(tiles);
}

int gsx_raster_bwd(int64_t n, int32_t C, const float* means2d, const float* conic_opacity,
                   const float* features, const int32_t* sorted_ids, int64_t num_ids,
                   const int32_t* tile_ranges, const float* background, int32_t width,
                   int32_t height, const float* final_T, const int32_t* n_contrib,
                   const float* grad_out, const float* grad_final_T, float* g_means2d,
                   float* g_conics, float* g_features, float* g_opacities, int32_t grad_stride,
                   int32_t* tile_order, void* stream) {
    const bool rec = grad_stride > 0;
    if (grad_stride < 0 || (rec && (grad_stride % 4 != 0 || grad_stride < 6 + C ||
                                    !aligned16(g_means2d) || g_conics || g_features ||
                                    g_opacities)))
        return GSX_ERR_INVALID;
    return raster_bwd(n, C, means2d, conic_opacity, features, sorted_ids, num_ids, tile_ranges,
                      background, width, height, final_T, n_contrib, grad_out, grad_final_T,
                      g_means2d, g_conics, g_features, g_opacities, grad_stride,
                      rec ? grad_stride : C, tile_order, stream);
}

int gsx_raster_bwd_geometry(int64_t n, int32_t C, const float* means2d, const float* conic_opacity,
                            const float* features, const int32_t* sorted_ids, int64_t num_ids,
                            const int32_t* tile_ranges, const float* background, int32_t width,
                            int32_t height, const float* final_T, const int32_t* n_contrib,
                            const float* grad_out, const float* grad_final_T, float* g_geometry,
                            float* g_features, int32_t grad_stride, int32_t* tile_order,
                            void* stream) {
    if (grad_stride < 8 || grad_stride % 4 != 0 || !aligned16(g_geometry)) return GSX_ERR_INVALID;
    if (n > 0 && !g_features) return GSX_ERR_INVALID;
    return raster_bwd(n, C, means2d, conic_opacity, features, sorted_ids, num_ids, tile_ranges,
                      background, width, height, final_T, n_contrib, grad_out, grad_final_T,
                      g_geometry, nullptr, g_features, nullptr, grad_stride, C, tile_order, stream);
}

int gsx_raster_bwd_rows(int64_t n, int32_t C, const float* means2d, const float* conic_opacity,
                        const float* features, const int32_t* sorted_ids, int64_t num_ids,
                        const int32_t* tile_ranges, const float* background, int32_t width,
                        int32_t height, const float* final_T, const int32_t* n_contrib,
                        const float* grad_out, const float* grad_final_T, float* g_geometry,
                        int32_t grad_stride, float* g_features, int32_t feature_stride,
                        int32_t* tile_order, void* stream) {
    if (C < 5 || C > kMaxChunk || grad_stride < 8 || grad_stride % 4 != 0 ||
        !aligned16(g_geometry))
        return GSX_ERR_INVALID;
    const bool inside = !g_features;  // the features' gradient follows in the record
    if (inside ? grad_stride < 6 + C : feature_stride < C) return GSX_ERR_INVALID;
    return raster_bwd(n, C, means2d, conic_opacity, features, sorted_ids, num_ids, tile_ranges,
                      background, width, height, final_T, n_contrib, grad_out, grad_final_T,
                      g_geometry, nullptr, g_features, nullptr, grad_stride,
                      inside ? grad_stride : feature_stride, tile_order, stream);
}

int gsx_split_raster_grads(int64_t n, const float* record, int32_t grad_stride, float* g_means2d,
                           float* g_conics, float* g_opacities, void* stream) {
    if (n < 0 || grad_stride < 8 || grad_stride % 4 != 0) return GSX_ERR_INVALID;
    if (n == 0) return GSX_OK;
    if (!record || !g_means2d || !g_conics || !g_opacities || !aligned16(record) ||
        !aligned8(g_means2d))
        return GSX_ERR_INVALID;
    const int64_t blocks = (n + 255) / 256;
    if (blocks > 0x7fffffff) return GSX_ERR_TOO_LARGE;
    hipLaunchKernelGGL(k_split_grads, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, n,
                       record, (int)grad_stride, (float2*)g_means2d, g_conics, g_opacities);
    GSX_LAUNCH_CHECK();
    return GSX_OK;
}

}  // extern "C"
