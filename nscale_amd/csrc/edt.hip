// Exact Euclidean distance transform of a u8 image: distance of every nonzero pixel to the
// nearest zero pixel (pixels outside the image are not zeros), as cv::distanceTransform(src, dst,
// CV_DIST_L2, CV_DIST_MASK_PRECISE) is called at HistologicalEntities.cpp:359.
//
// Output value = sqrtf(float(dx^2) + float(g^2)) for the minimising column offset dx, where g is
// the vertical distance of that column to its nearest zero: the same float expression OpenCV's
// precise transform evaluates (sqr_tab[|q-p|] + f[p]); rows without any zero in any column give
// sqrtf(0 + 1e15f) as OpenCV's "infinite" column value does.
//
// 1. k_edt_masks: the zero pixels of every column as 64-bit words, one per 64 rows.
// 2. k_edt_tiles: 64 x 64 pixels per workgroup, with 32 columns more on either side.  A thread turns
//    its column's words (its own and the two next to it) into the vertical distances g of its 64
//    rows, capped at 63, in LDS; then each pair of pixels looks outward, both sides and both pixels in
//    one packed 16-bit operation, while dx^2 is below its best squared distance (four pairs per thread
//    at once: with one, a turn is a round trip to LDS and 512^2 took 40 us).  A result of at most
//    32^2 is exact: every candidate it has not seen is larger (dx > 32, or g > 32 where the cap or the
//    missing words hide it).  Pixels further away flag their row.  Two waves that the first step leaves
//    idle find the last zero above and the first below the segment in each of its columns.
// 3. k_edt_rows: flagged rows (the others' workgroups leave at once).  g of the whole row from the
//    words and those zeros; each flagged pixel searches outward over the row; a search that would exceed SEARCH_CAP
//    columns has the row recomputed with the exact integer lower-envelope algorithm.
// The masks are 1/8 byte per pixel, the zeros beyond the segments 1/16, so little but the image and the result
// moves: 4096^2 nuclei mask, whose rows all leave at once in step 3, 44 us.  (With the vertical distances as a
// 16-bit plane, segments' carries, one pixel per lane and 32-bit squares in the search, six launches: 190 us, of
// which the search 78, bound by its instructions.)  Masks with distances past 32 pay for their flagged rows: 4096^2
// with a hole of radius 8 every 128 pixels 1080 us, of radius 4 every 300 1940 (1690 and 2520 when every
// flagged row walked its columns' words to the next zero).
#include "common.hpp"

namespace nsc {
namespace {

constexpr int SEG = 64;
constexpr uint16_t NONE = 0xFFFF;
constexpr int SEARCH_CAP = 1024;
constexpr int E_COLS = 64, E_HALO = 32, E_WIDE = E_COLS + 2 * E_HALO, E_THREADS = 256;
constexpr int E_CAP = 63;  // largest g of the tile pass

// zero pixels of 64 rows of a column, bit = row; the flags of the segment's rows are cleared for the
// passes that follow
__global__ __launch_bounds__(64) void k_edt_masks(const uint8_t* __restrict__ img, int w, int h, uint64_t* __restrict__ zm,
                                                  int* __restrict__ rowflag) {
    const int sg = blockIdx.y, y0 = sg * SEG, n = min(h, y0 + SEG) - y0;
    if (blockIdx.x == 0 && (int)threadIdx.x < n) rowflag[y0 + threadIdx.x] = 0;
    const int x = blockIdx.x * 64 + threadIdx.x;
    if (x >= w) return;
    // 64 loads in flight (rows past the image read the last row and are masked off), a bit per zero row
    uint32_t v[SEG];
#pragma unroll
    for (int j = 0; j < SEG; ++j) v[j] = img[(size_t)min(y0 + j, h - 1) * w + x];
    uint32_t lo = 0, hi = 0;
#pragma unroll
    for (int j = 0; j < 32; ++j) lo |= (v[j] == 0 ? 1u : 0u) << j;
#pragma unroll
    for (int j = 0; j < 32; ++j) hi |= (v[32 + j] == 0 ? 1u : 0u) << j;
    uint64_t m = (uint64_t)lo | (uint64_t)hi << 32;
    if (n < SEG) m &= (1ull << n) - 1ull;
    zm[(size_t)sg * w + x] = m;
}

typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ u16x2 pk(uint32_t v) { return __builtin_bit_cast(u16x2, v); }

__global__ __launch_bounds__(E_THREADS) void k_edt_tiles(const uint64_t* __restrict__ zm, int w, int h, int nseg,
                                                      float* __restrict__ out, int* __restrict__ rowflag,
                                                      uint16_t* __restrict__ above, uint16_t* __restrict__ below) {
    __shared__ uint16_t G[SEG][E_WIDE];
    const int sg = blockIdx.y, y0 = sg * SEG, x0 = blockIdx.x * E_COLS;
    int row = -1;
    if (threadIdx.x < E_WIDE) {
        const int x = x0 - E_HALO + (int)threadIdx.x;
        // all three words from clamped (always valid) addresses; what lies outside the image holds no zero
        const size_t xc = (size_t)clampi(x, 0, w - 1);
        const uint64_t a = zm[(size_t)max(sg - 1, 0) * w + xc], m = zm[(size_t)sg * w + xc],
                       b = zm[(size_t)min(sg + 1, nseg - 1) * w + xc];
        const bool in = x >= 0 && x < w;
        const uint64_t up = in && sg > 0 ? a : 0ull, own = in ? m : 0ull, dn = in && sg + 1 < nseg ? b : 0ull;
        // distance of the row before the first to its nearest zero above it, of the row after the last below
        uint32_t d = up ? (uint32_t)min((int)__clzll((long long)up), E_CAP) : (uint32_t)E_CAP;
        uint32_t g[SEG];
#pragma unroll
        for (int j = 0; j < SEG; ++j) {
            d = ((uint32_t)(own >> (j & 32)) >> (j & 31) & 1u) ? 0u : min(d + 1u, (uint32_t)E_CAP);
            g[j] = d;
        }
        d = dn ? (uint32_t)min((int)__ffsll((long long)dn) - 1, E_CAP) : (uint32_t)E_CAP;
#pragma unroll
        for (int j = SEG - 1; j >= 0; --j) {
            d = min(d + 1u, g[j]);  // g[j] is 0 at a zero
            G[j][threadIdx.x] = (uint16_t)d;
        }
    } else {
        // waves 2 and 3: the row of the column's last zero above, first zero below the segment
        static_assert(E_WIDE == 128 && E_THREADS == 256 && E_COLS == 64, "a wave each, a lane per column");
        const bool up = threadIdx.x < 192;  // wave-uniform
        const int x = x0 + (int)(threadIdx.x & 63), step = up ? -1 : 1, n = up ? sg : nseg - 1 - sg;
        const uint64_t* const col = zm + min(x, w - 1);
        // the next segment's word, which nearly always holds one, then eight words' loads at a time
        auto hit = [&](uint64_t q, int s) { return s * SEG + (up ? 63 - (int)__clzll((long long)q) : (int)__ffsll((long long)q) - 1); };
        if (n > 0)
            if (const uint64_t q = col[(size_t)(sg + step) * w]) row = hit(q, sg + step);
        for (int k0 = 2; k0 <= n && row < 0; k0 += 8) {
            uint64_t q[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) q[j] = col[(size_t)(sg + step * min(k0 + j, n)) * w];
#pragma unroll
            for (int j = 0; j < 8; ++j)
                if (row < 0 && q[j]) row = hit(q[j], sg + step * min(k0 + j, n));
        }
    }
    __syncthreads();
    if (threadIdx.x >= E_WIDE && x0 + (int)(threadIdx.x & 63) < w)  // (a store the barrier need not wait for)
        (threadIdx.x < 192 ? above : below)[(size_t)sg * w + x0 + (threadIdx.x & 63)] = row < 0 ? NONE : (uint16_t)row;
    constexpr int NP = E_COLS / 2, STEP = E_THREADS / NP, K = 4;  // pairs per row, rows per step
    const int c = 2 * ((int)threadIdx.x % NP), x = x0 + c;
    for (int yb = (int)threadIdx.x / NP; yb < SEG; yb += K * STEP) {
        if (y0 + yb - (int)threadIdx.x / NP >= h) break;  // the same for the whole workgroup
        uint32_t lc[K], rc[K];
        u16x2 best[K];
        auto pair_at = [&](int k, int o) {
            return *reinterpret_cast<const uint32_t*>(&G[yb + k * STEP][E_HALO + c + o]);  // 4-byte aligned
        };
#pragma unroll
        for (int k = 0; k < K; ++k) {
            lc[k] = rc[k] = pair_at(k, 0);
            best[k] = pk(lc[k]) * pk(lc[k]);
        }
        // two steps a turn: an odd one straddles the words of its even neighbours
        for (int dx = 1; dx < E_HALO; dx += 2) {
            u16x2 worst = best[0];
#pragma unroll
            for (int k = 1; k < K; ++k) worst = __builtin_elementwise_max(worst, best[k]);
            const uint32_t b = __builtin_bit_cast(uint32_t, worst);
            if (!__any((int)max(b & 0xFFFFu, b >> 16) > dx * dx)) break;
            uint32_t ln[K], rn[K];
#pragma unroll
            for (int k = 0; k < K; ++k) {
                ln[k] = pair_at(k, -dx - 1);
                rn[k] = pair_at(k, dx + 1);
            }
            const unsigned short s1 = (unsigned short)(dx * dx), s2 = (unsigned short)((dx + 1) * (dx + 1));
#pragma unroll
            for (int k = 0; k < K; ++k) {
                const u16x2 m1 = __builtin_elementwise_min(pk(lc[k] << 16 | ln[k] >> 16), pk(rc[k] >> 16 | rn[k] << 16));
                const u16x2 m2 = __builtin_elementwise_min(pk(ln[k]), pk(rn[k]));
                best[k] = __builtin_elementwise_min(best[k], m1 * m1 + u16x2{s1, s1});
                best[k] = __builtin_elementwise_min(best[k], m2 * m2 + u16x2{s2, s2});
                lc[k] = ln[k];
                rc[k] = rn[k];
            }
        }
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int y = y0 + yb + k * STEP;
            if (y >= h || x >= w) continue;
            const uint32_t b = __builtin_bit_cast(uint32_t, best[k]), d0 = b & 0xFFFFu, d1 = b >> 16;
            float* const o = out + (size_t)y * w + x;
            // the squared distance is an integer below 2^24: one exact float whatever dx and g it came from
            const float f0 = d0 <= E_HALO * E_HALO ? sqrtf((float)d0) : -1.0f;
            const float f1 = d1 <= E_HALO * E_HALO ? sqrtf((float)d1) : -1.0f;
            bool far = f0 < 0.0f;
            if (x + 1 < w) {
                const float2 f = make_float2(f0, f1);
                __builtin_memcpy(o, &f, 8);
                far = far || f1 < 0.0f;
            } else {
                o[0] = f0;
            }
            if (far) rowflag[y] = 1;
        }
    }
}

__device__ __forceinline__ float edt_value(long long dx2, long long g) {
    const float fg = (g == NONE) ? 1e15f : (float)(g * g);
    return sqrtf((float)dx2 + fg);
}

__global__ __launch_bounds__(256) void k_edt_rows(const uint64_t* __restrict__ zm, int w, int h, int nseg,
                                                  float* __restrict__ out, const int* __restrict__ rowflag,
                                                  const uint16_t* __restrict__ above, const uint16_t* __restrict__ below) {
    extern __shared__ uint16_t lds[];
    const int y = blockIdx.x;
    if (!rowflag[y]) return;
    uint16_t* const grow = lds;  // vertical distances of the row (NONE: no zero in the column)
    const int sg = y / SEG, j = y % SEG;
    for (int x = threadIdx.x; x < w; x += blockDim.x) {
        const size_t i = (size_t)sg * w + x;
        const uint64_t m = zm[i], le = m & ((2ull << j) - 1ull), ge = m >> j;
        const uint32_t a = above[i], b = below[i];
        const uint32_t du = le ? (uint32_t)(j - 63 + (int)__clzll((long long)le)) : (a != NONE ? (uint32_t)y - a : NONE);
        const uint32_t dd = ge ? (uint32_t)__ffsll((long long)ge) - 1u : (b != NONE ? b - (uint32_t)y : NONE);
        grow[x] = (uint16_t)min(du, dd);
    }
    __shared__ int need, kk;
    if (threadIdx.x == 0) need = 0;
    __syncthreads();
    for (int x = threadIdx.x; x < w; x += blockDim.x) {
        if (!(out[(size_t)y * w + x] < 0.0f)) continue;
        // squared distances in 32 bits, exactly: g <= 65534 so g^2 < 2^32 and UINT_MAX marks "no
        // zero"; a candidate dx^2 + v^2 is compared as v^2 < best - dx^2 (dx^2 < best), which can
        // neither overflow nor underflow, and a winner is below the old best
        const uint32_t gx = grow[x];
        uint32_t best = (gx == NONE) ? UINT_MAX : gx * gx;
        int bdx = 0;
        uint32_t bg = gx;
        if (best != 0) {
            int dx = 1;
            for (; dx <= SEARCH_CAP; ++dx) {
                const uint32_t dx2 = (uint32_t)(dx * dx);
                if (dx2 >= best) break;
                if (x - dx < 0 && x + dx >= w) { dx = SEARCH_CAP + 2; break; }
                if (x - dx >= 0) {
                    const uint32_t v = grow[x - dx];
                    if (v != NONE && v * v < best - dx2) { best = dx2 + v * v; bdx = dx; bg = v; }
                }
                if (x + dx < w) {
                    const uint32_t v = grow[x + dx];
                    if (v != NONE && v * v < best - dx2) { best = dx2 + v * v; bdx = dx; bg = v; }
                }
            }
            if (dx == SEARCH_CAP + 1) need = 1;  // search cut short: exact envelope below
        }
        float o;
        if (best == UINT_MAX) o = sqrtf(1e15f);
        else o = edt_value((long long)bdx * bdx, bg);
        out[(size_t)y * w + x] = o;
    }
    __syncthreads();
    if (!need) return;
    // exact lower envelope of the parabolas (x - p)^2 + g(p)^2 over the columns with a zero
    // (Felzenszwalb-Huttenlocher with exact integer intersection tests), the apex stack in LDS (a column
    // fits 16 bits), built by one lane and evaluated by all
    uint16_t* const v = lds + w;
    auto f = [&](int p) { return (long long)grow[p] * grow[p]; };
    if (threadIdx.x == 0) {
        int k = -1;
        for (int q = 0; q < w; ++q) {
            if (grow[q] == NONE) continue;
            while (k >= 1) {
                const int p = v[k], r = v[k - 1];
                // drop p when the (r, q) intersection is not right of the (r, p) intersection
                const long long nq = (f(q) + (long long)q * q) - (f(r) + (long long)r * r);
                const long long np = (f(p) + (long long)p * p) - (f(r) + (long long)r * r);
                if (nq * (long long)(p - r) <= np * (long long)(q - r)) --k;
                else break;
            }
            v[++k] = (uint16_t)q;
        }
        kk = k;
    }
    __syncthreads();
    const int k = kk;
    for (int x = threadIdx.x; x < w; x += blockDim.x) {
        if (k < 0) { out[(size_t)y * w + x] = sqrtf(1e15f); continue; }
        // binary search for the apex whose parabola is lowest at x (the envelope order is monotone)
        int lo = 0, hi = k;
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            const int p = v[mid], q = v[mid + 1];
            const long long dp = (long long)(x - p) * (x - p) + f(p);
            const long long dq = (long long)(x - q) * (x - q) + f(q);
            if (dq <= dp) lo = mid + 1;
            else hi = mid;
        }
        const int p = v[lo];
        out[(size_t)y * w + x] = edt_value((long long)(x - p) * (x - p), grow[p]);
    }
}

}  // namespace

int edt_impl(const uint8_t* img, float* out, int w, int h, hipStream_t s) {
    // size limits are checked before anything is queued on the stream
    if (h >= 0xFFFF) {
        set_error("distance transform supports heights below 65535");
        return NSC_ERR_LIMIT;
    }
    if (w > 32768) {
        set_error("distance transform supports widths up to 32768");
        return NSC_ERR_LIMIT;
    }
    const int nseg = (int)cdiv(h, SEG);
    Carver measure(nullptr);
    measure.take<uint64_t>((size_t)nseg * w);
    measure.take<int>(h);
    measure.take<uint16_t>((size_t)nseg * w);
    measure.take<uint16_t>((size_t)nseg * w);
    Scratch sc;
    NSC_CHECK(sc.alloc(measure.size(), s));
    Carver cut(sc.p);
    uint64_t* zm = cut.take<uint64_t>((size_t)nseg * w);
    int* rowflag = cut.take<int>(h);
    uint16_t* above = cut.take<uint16_t>((size_t)nseg * w);
    uint16_t* below = cut.take<uint16_t>((size_t)nseg * w);
    hipLaunchKernelGGL(k_edt_masks, dim3(cdiv(w, 64), nseg), dim3(64), 0, s, img, w, h, zm, rowflag);
    hipLaunchKernelGGL(k_edt_tiles, dim3(cdiv(w, E_COLS), nseg), dim3(E_THREADS), 0, s, zm, w, h, nseg, out, rowflag, above, below);
    // the launch is unconditional and the workgroups of unflagged rows leave at once (no host sync)
    const size_t lds = 2 * sizeof(uint16_t) * (size_t)w;
    if (lds > 64 * 1024)
        NSC_HIP(hipFuncSetAttribute((const void*)k_edt_rows, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(k_edt_rows, dim3(h), dim3(256), lds, s, zm, w, h, nseg, out, rowflag, above, below);
    NSC_HIP(hipGetLastError());
    return NSC_OK;
}

}  // namespace nsc

using namespace nsc;

extern "C" int nsc_dist_transform_u8(const uint8_t* img, float* out, int w, int h, void* stream) {
    NSC_ARG(img && out && w > 0 && h > 0, "dist_transform_u8");
    NSC_CHECK(ensure_init());
    return edt_impl(img, out, w, h, as_stream(stream));
}
