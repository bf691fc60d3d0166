// Colour normalization of src/normalization/Normalization.cpp: Reinhard's transfer in the
// l-alpha-beta space of the foreground that a fixed linear discriminant separates from the
// background (normalization, Normalization.cpp:436-499), and the foreground statistics alone
// (targetParameters, Normalization.cpp:502-582).
//
// The reference builds seven full-size float planes; here every pixel's result depends on its
// own colour and six statistics only, so the work is two streaming passes over the BGR image:
//   1. k_norm_stats: discriminant, LAB, and per-workgroup double sums of the selected pixels'
//      values and float squares;
//   2. k_norm_apply: sums the partials in a fixed order (every workgroup for itself: mean / std in
//      double, the float transfer factors), then LAB again, the transfer for foreground pixels, back
//      to BGR.  (k_norm_finish does the sum for the statistics call.)
// Both passes are bound by instruction issue (about 0.4 us per instruction and pixel of a 4096^2
// tile), so each workgroup first gives every pixel of its chunk the few instructions that decide
// what it needs, and then works through a dense list of the pixels that need the transform: the
// statistics only the foreground (20-30% of an H&E tile; without the list nearly every wave held a
// foreground pixel and all its lanes paid), the result the foreground and the few background pixels
// that norm_bg_fast cannot decide.
// Arithmetic follows the reference operation by operation: the discriminant is the double
// arithmetic of OpenCV 2.4's float addWeighted rounded to float twice, the RGB->LMS products are
// double (the constants are double literals) rounded to float, everything else is float.  log10f
// follows the fdlibm formula C libraries use (float operations around a correctly rounded logf);
// powf(10, x) is correctly rounded.  Both evaluate their core in double with relative error near
// 2^-48, so they differ from a C library only where that library's own logf / powf is not
// correctly rounded (under 1% / 0.1% of arguments for glibc 2.35).
#include <cfloat>
#include <cmath>

#include "common.hpp"
#include "normalize_rules.hpp"
#include "normalize_tables.hpp"

namespace nsc {
namespace {

constexpr int kNormThreads = 512;
constexpr int kNormChunk = 4 * kNormThreads;  // pixels per work item (at most)
// statistics partials (8 doubles each): two workgroups per CU, few enough that every workgroup of
// k_norm_apply can sum them itself
constexpr int kNormMaxBlocks = 512;
// three workgroups per CU, which its registers allow (20 KB of LDS each would allow eight); a fourth per CU ran
// after them: 4096^2 white 66 us with 1024, 64 with 768, 512 x 3900 crop 36 and 35, H&E and noise alike
constexpr int kApplyMaxBlocks = 768;

struct NormConsts {
    float k3, k6, k2;  // 1/sqrtf(3), 1/sqrtf(6), 1/sqrtf(2) (Normalization.cpp:112-114, 172-174)
    float s255;        // the float factor convertTo uses for "/= 255" (Normalization.cpp:331)
};

// Fisher discriminant coefficients (Normalization.cpp:451): rows background, foreground over R G B 1
struct NormDisc {
    float m[8];
};

struct NormParams {
    float meanI[3], ratio[3];  // image statistics and target_std / image_std (float division)
};

// segFG (Normalization.cpp:19-56): addWeighted(addWeighted(R, m0, G, m1, 0), 1, B, m2, m3) for
// each discriminant; each addWeighted evaluates in double and stores float.  With the decimal
// coefficients, d_fg - d_bg = (97 R - 852 G + 621 B - 4169) / 1000 exactly; the float coefficients
// and the float roundings of values below 300 move it by less than 1e-4, so wherever that integer
// is not zero its sign decides, and only exact ties (75 of the 2^24 colours) take the float path.
__device__ __forceinline__ int norm_num(uint32_t b, uint32_t g, uint32_t r) {
    return 97 * (int)r - 852 * (int)g + 621 * (int)b - 4169;
}
__device__ __forceinline__ bool norm_fg(const NormDisc& D, uint32_t b, uint32_t g, uint32_t r) {
    const int num = norm_num(b, g, r);
    if (num != 0) return num > 0;
    float d[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const float* m = D.m + 4 * k;
        const float t = (float)((double)r * (double)m[0] + (double)g * (double)m[1] + 0.0);
        d[k] = (float)((double)t * 1.0 + (double)b * (double)m[2] + (double)m[3]);
    }
    return d[0] < d[1];
}

// The logarithm and exponential tables, staged per workgroup: neighbouring pixels look up different
// entries, which LDS serves at once.
struct NormTabs {
    double2 lg[kLogTabN];
    double ex[kExpTabN];
};
__device__ __forceinline__ void load_log_tab(double2* lg) {
    for (int i = threadIdx.x; i < kLogTabN; i += kNormThreads) lg[i] = kLogTab[i];
}

// Natural logarithm of m in [0.5, 2) in double, m of 24 significant bits: r = m c - 1 with the
// tabled reciprocal c is exact and |r| <= 2^-8, log m = -log c + log(1 + r), series to r^6 (the
// first omitted term is below 2^-50 of the result: where -log c is 0 the terms are relative to r,
// elsewhere they are smaller still).  Relative error about 2^-50, so the float rounding of the
// result is the correct rounding except within that distance of a rounding boundary (this is not an
// operation of the reference, only its accuracy matters).  8 double operations and one LDS read
// instead of 19 for the atanh series without a table.
__device__ __forceinline__ double log_unit(const double2* lg, uint32_t mbits) {
    const double2 T = lg[(mbits - 0x3f000000u) >> 15];
    const double r = fma((double)__uint_as_float(mbits), T.x, -1.0);
    double p = -1.0 / 6;
    p = fma(p, r, 1.0 / 5);
    p = fma(p, r, -1.0 / 4);
    p = fma(p, r, 1.0 / 3);
    p = fma(p, r, -1.0 / 2);
    return T.y + fma(p, r * r, r);
}

// log10f as the fdlibm-derived C libraries compute it (glibc's e_log10f.c, the function the
// reference calls at Normalization.cpp:92-94): x = 2^y m with m in [1, 2) (in [0.5, 1) when the
// exponent is negative), log10 x = y lo + ivln10 logf(m) + y hi in float operations with fdlibm's
// constants; logf(m) is the correctly rounded natural logarithm.
// x is a weighted mean of byte / 255 values: 0, or a normal number between 9e-5 and 1.004.
__device__ __forceinline__ float log10f_lib(const double2* lg, float x) {
    constexpr float kIvln10 = 0x1.bcb7b2p-2f;  // 4.3429449201e-01
    constexpr float kHi = 0x1.344100p-2f;      // 3.0102920532e-01
    constexpr float kLo = 0x1.a84fb6p-21f;     // 7.9034151668e-07
    const uint32_t hx = __float_as_uint(x);
    const bool lt1 = hx < 0x3f800000u;
    const uint32_t mbits = (hx & 0x007fffffu) | (lt1 ? 0x3f000000u : 0x3f800000u);
    const float y = (float)((int)(hx >> 23) - (lt1 ? 126 : 127));
    const float lnm = (float)log_unit(lg, mbits);
    const float z = y * kLo + kIvln10 * lnm;
    return x == 0.0f ? -INFINITY : z + y * kHi;
}

// 10^y rounded to float, evaluated in double: y log2(10) = k / 128 + f with the constant split so
// that y * hi is exact, 2^(k / 128) = 2^(k >> 7) times a tabled value, 2^f by its Taylor series to
// f^4 (|f ln2| <= 0.0028, truncation below 2^-49, fused multiply-adds); relative error about 2^-49
// before the final rounding.  11 double operations instead of 17 without a table.
__device__ __forceinline__ float exp10f_rn(const double* ex, float y) {
    const float yc = fminf(fmaxf(y, -46.0f), 40.0f);  // NaN, and what lies outside, decided below
    const double yd = (double)yc;
    const double z = yd * 0x1.a934f09p+1;  // log2(10) to 29 bits: exact product
    const double kd = rint(z * 128.0);
    const int k = (int)kd;
    const double f = fma(kd, -1.0 / 128, z) + yd * 0x1.e68dc57f24960p-29;
    const double t = ex[k & (kExpTabN - 1)];
    double p = 0x1.3b2ab6fba4e77p-7;           // ln2^4 / 24
    p = fma(p, f, 0x1.c6b08d704a0bfp-5);       // ln2^3 / 6
    p = fma(p, f, 0x1.ebfbdff82c58ep-3);       // ln2^2 / 2
    p = fma(p, f, 0x1.62e42fefa39efp-1);       // ln2
    const float v = (float)__builtin_amdgcn_ldexp(fma(t * f, p, t), k >> 7);
    if (y != y) return y;
    return y > 40.0f ? INFINITY : (y < -46.0f ? 0.0f : v);
}

// bgr2Lab of one pixel (Normalization.cpp:64-146) after PixelClass's scaling (:328-333)
__device__ __forceinline__ void norm_lab(const NormConsts& C, const double2* lg, uint32_t b8, uint32_t g8, uint32_t r8, float lab[3]) {
    const float b = (float)b8 * C.s255, g = (float)g8 * C.s255, r = (float)r8 * C.s255;
    const float L = (float)(0.3811 * r + 0.5783 * g + 0.0402 * b);
    const float M = (float)(0.1967 * r + 0.7244 * g + 0.0782 * b);
    const float S = (float)(0.0241 * r + 0.1288 * g + 0.8444 * b);
    const float l = log10f_lib(lg, L), m = log10f_lib(lg, M), s = log10f_lib(lg, S);
    lab[0] = l * C.k3 + m * C.k3 + s * C.k3;
    lab[1] = l * C.k6 + m * C.k6 + s * (-2.0f * C.k6);
    lab[2] = l * C.k2 + m * (-C.k2) + s * 0.0f;  // s * 0 keeps the NaN of a black pixel
}

// lab2BGR of one pixel (Normalization.cpp:162-306): back to log LMS, 10^x (non-finite -> 0), the
// LMS->RGB matrix, x 255 in double, clamp, round half up; a NaN channel gives 0
__device__ __forceinline__ void norm_bgr(const NormConsts& C, const double* ex, const float lab[3],
                                         uint8_t out[3]) {
    const float ll = lab[0] * C.k3 + lab[1] * C.k6 + lab[2] * C.k2;
    const float lm = lab[0] * C.k3 + lab[1] * C.k6 + lab[2] * (-C.k2);
    const float ls = lab[0] * C.k3 + lab[1] * (-2.0f * C.k6) + lab[2] * (0.0f * C.k2);
    float L = exp10f_rn(ex, ll), M = exp10f_rn(ex, lm), S = exp10f_rn(ex, ls);
    if (!(fabsf(L) <= FLT_MAX)) L = 0.0f;
    if (!(fabsf(M) <= FLT_MAX)) M = 0.0f;
    if (!(fabsf(S) <= FLT_MAX)) S = 0.0f;
    const float bgrf[3] = {L * 0.0585f + M * -0.2611f + S * 1.2057f,
                           L * -1.2197f + M * 2.3831f + S * -0.1626f,
                           L * 4.4687f + M * -3.5887f + S * 0.1196f};
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        float v = (float)((double)bgrf[k] * 255.0);
        v = v < 0.0f ? 0.0f : v;
        v = v > 255.0f ? 255.0f : v;
        const float f = floorf(v);
        int q = (int)f + ((v - f >= 0.5f) ? 1 : 0);
        out[k] = (v == v) ? (uint8_t)q : (uint8_t)0;
    }
}

// A background pixel's result straight from its colour.  Without the transfer, logarithm and
// exponential cancel: v = 255 (LMS->RGB)(RGB->LMS) rgb / 255, here in float from the product of the
// two matrices.  The reference's chain of float operations (and its four-digit matrices' product)
// stays within kBgMargin of v: its logarithms and l-alpha-beta sums carry about ten float roundings
// of values below 8 (at most 2.4e-6 in log10 LMS, 5.5e-6 relative in LMS), which the inverse matrix
// (coefficients summing to below 8.2 a row, LMS below 1.004) turns into at most 0.0115 levels, plus
// 0.0006 of its own roundings.  The value is decided unless v comes within kBgMargin of a rounding
// boundary k + 1/2; the tests compare every colour.
constexpr float kBgMargin = 0.0156f;
struct NormBg {
    float m[9];  // rows: b, g, r of the result; columns: b, g, r of the pixel
};
__device__ __forceinline__ bool norm_bg_fast(const NormBg& G, float b, float g, float r, uint32_t o[3]) {
    bool sure = true;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        float t = fmaf(G.m[3 * k], b, fmaf(G.m[3 * k + 1], g, fmaf(G.m[3 * k + 2], r, 0.5f)));
        t = fminf(fmaxf(t, 0.5f), 255.5f);
        const float f = floorf(t), d = t - f;
        sure = sure && d > kBgMargin && d < 1.0f - kBgMargin;
        o[k] = (uint32_t)f;
    }
    return sure;
}

// The image as groups of four consecutive pixels of a row (a row's last group may hold fewer), numbered row by
// row; an image without gaps between its rows is taken as one long row.  The passes take groups in turn, so
// the lanes of a workgroup have work whatever the rows' length.  (With a row's chunks of 2048 pixels to a workgroup,
// a crop of width 100 kept 25 of its 512 threads busy: 100 x 3900 pixels 53 us a call, by groups 18.)
struct NormImage {
    const uint8_t* bgr;
    size_t ld;
    size_t w;                    // pixels per row
    unsigned long long per_row;  // groups per row
    unsigned long long magic;    // of per_row (normalize_rules.hpp)
    unsigned long long groups;
    bool one_row;
};

// work items: a group per thread of a workgroup
__host__ __device__ inline long long norm_items(const NormImage& I) { return (long long)((I.groups + kNormThreads - 1) / kNormThreads); }

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// group q: byte offset of its first pixel in a plane of row stride ld, and its pixel count (0 past the last).
__device__ __forceinline__ int norm_group(const NormImage& I, unsigned long long q, size_t ld, size_t* off) {
    *off = 0;
    if (q >= I.groups) return 0;
    const unsigned long long y = I.one_row ? 0ull : row_of(q, I.magic);
    const size_t x0 = 4 * (size_t)(q - y * I.per_row);
    *off = (size_t)y * ld + 3 * x0;
    return (int)std::min<size_t>(4, I.w - x0);
}

// the thread's four pixels (12 bytes; n of them exist) as three words, by words where p is aligned
__device__ __forceinline__ void norm_load4(const uint8_t* p, int n, uint32_t wd[3]) {
    if (n == 4 && (reinterpret_cast<uintptr_t>(p) & 3) == 0) {
        const uint32_t* q = reinterpret_cast<const uint32_t*>(p);
        wd[0] = q[0];
        wd[1] = q[1];
        wd[2] = q[2];
    } else {
        uint8_t by[12];
#pragma unroll
        for (int j = 0; j < 12; ++j) by[j] = j < 3 * n ? p[j] : 0;
#pragma unroll
        for (int k = 0; k < 3; ++k)
            wd[k] = by[4 * k] | (uint32_t)by[4 * k + 1] << 8 | (uint32_t)by[4 * k + 2] << 16 | (uint32_t)by[4 * k + 3] << 24;
    }
}
// pixel k's three bytes of those words: b | g << 8 | r << 16
__device__ __forceinline__ uint32_t norm_px(const uint32_t wd[3], int k) {
    return (k == 0 ? wd[0] : k == 1 ? (wd[0] >> 24 | wd[1] << 8) : k == 2 ? (wd[1] >> 16 | wd[2] << 16) : wd[2] >> 8) &
           0xFFFFFFu;
}

// one listed pixel (foreground, or one of the discriminant's ties) into the thread's sums
__device__ __forceinline__ void stats_add(const NormConsts& C, const NormDisc& D, const double2* lg, uint32_t px,
                                          double acc[7]) {
    const uint32_t b = px & 255u, g = px >> 8 & 255u, r = px >> 16;
    if (!norm_fg(D, b, g, r)) return;  // a tie that the float path decides against
    float lab[3];
    norm_lab(C, lg, b, g, r, lab);
    if (!((lab[0] * lab[1]) * lab[2] > 0.0f)) return;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        acc[c] += (double)lab[c];
        acc[3 + c] += (double)(lab[c] * lab[c]);
    }
    acc[6] += 1.0;
}

// Per-workgroup sums over the selected pixels: [sum L, sum a, sum b, sq L, sq a, sq b, count, 0].
// Every wave goes through its own pieces of 64 groups (256 pixels at most) and keeps a list of the
// foreground pixels it met; whenever the list holds 64 it takes 64 off, so all lanes work, nothing
// waits on another wave, and the order of the additions depends on the grid alone.  The next
// piece's words are on their way while the current one is listed.
// 4096^2 H&E tile: 36 us (95 us with the series logarithm on every wave that held a foreground
// pixel).
constexpr int kStatsPiece = 256;
__global__ __launch_bounds__(kNormThreads) void k_norm_stats(NormImage I, NormConsts C, NormDisc D,
                                                             double* __restrict__ part) {
    constexpr int kWaves = kNormThreads / 64;
    __shared__ double2 lg[kLogTabN];
    __shared__ uint32_t lists[kWaves][64 + kStatsPiece];
    const int wv = threadIdx.x >> 6, ln = threadIdx.x & 63;
    uint32_t* const list = lists[wv];
    double acc[7] = {0, 0, 0, 0, 0, 0, 0};
    const long long pieces = (long long)((I.groups + 63) / 64), step = (long long)gridDim.x * kWaves;
    // a piece's words and the number of pixels the lane has of it (past the last group: none)
    auto load = [&](long long pc, uint32_t wd[3]) {
        size_t off;
        const int mine = norm_group(I, 64ull * (unsigned long long)pc + (unsigned)ln, I.ld, &off);
        wd[0] = wd[1] = wd[2] = 0;
        if (mine) norm_load4(I.bgr + off, mine, wd);
        return mine;
    };
    int held = 0;  // wave-uniform
    uint32_t wd[3], nx[3];
    long long pc = (long long)blockIdx.x * kWaves + wv;
    int mine = load(pc, wd);
    load_log_tab(lg);
    __syncthreads();
    for (; pc < pieces; pc += step) {
        const int nmine = load(pc + step, nx);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const uint32_t px = norm_px(wd, k);
            const bool take = k < mine && norm_num(px & 255u, px >> 8 & 255u, px >> 16) >= 0;
            const unsigned long long m = __ballot(take);
            if (take) list[held + __popcll(m & ((1ull << ln) - 1ull))] = px;
            held += __popcll(m);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        while (held >= 64) {
            held -= 64;
            stats_add(C, D, lg, list[held + ln], acc);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        mine = nmine;
#pragma unroll
        for (int k = 0; k < 3; ++k) wd[k] = nx[k];
    }
    if (ln < held) stats_add(C, D, lg, list[ln], acc);
    __shared__ double red[kNormThreads / 64][8];
#pragma unroll
    for (int c = 0; c < 7; ++c) {
        const double v = wave_sum(acc[c]);
        if (ln == 0) red[wv][c] = v;
    }
    __syncthreads();
    if (threadIdx.x < 8) {
        double v = 0.0;
        if (threadIdx.x < 7)
            for (int k = 0; k < kNormThreads / 64; ++k) v += red[k][threadIdx.x];
        part[(size_t)blockIdx.x * 8 + threadIdx.x] = v;
    }
}

// Sums the partials in a fixed order (deterministic; every workgroup that calls it gets the same
// bits): tot[0..6] in LDS, valid for all threads afterwards.
__device__ __forceinline__ void norm_totals(const double* __restrict__ part, int nblocks, double (*red)[8], double* tot) {
    double acc[7] = {0, 0, 0, 0, 0, 0, 0};
    for (int b = threadIdx.x; b < nblocks; b += kNormThreads)
#pragma unroll
        for (int c = 0; c < 7; ++c) acc[c] += part[(size_t)b * 8 + c];
    const int wv = threadIdx.x >> 6, ln = threadIdx.x & 63;
#pragma unroll
    for (int c = 0; c < 7; ++c) {
        const double v = wave_sum(acc[c]);
        if (ln == 0) red[wv][c] = v;
    }
    __syncthreads();
    if (threadIdx.x < 7) {
        double v = 0.0;
        for (int k = 0; k < kNormThreads / 64; ++k) v += red[k][threadIdx.x];
        tot[threadIdx.x] = v;
    }
    __syncthreads();
}
// TransferI's statistics (Normalization.cpp:383-394): mean = sum / count, var = sq / count - mean^2,
// std = sqrt(var), each stored as float by the caller
__device__ __forceinline__ void norm_moments(const double* tot, int c, double* mean, double* sd) {
    const double n = tot[6];
    *mean = tot[c] / n;
    const double var = tot[3 + c] / n - *mean * *mean;
    *sd = sqrt(var);
}

// the statistics call's result: double mean[3], std[3], count
__global__ __launch_bounds__(kNormThreads) void k_norm_finish(const double* __restrict__ part, int nblocks,
                                                              double* __restrict__ stats) {
    __shared__ double red[kNormThreads / 64][8], tot[8];
    norm_totals(part, nblocks, red, tot);
    if (threadIdx.x < 3) norm_moments(tot, threadIdx.x, &stats[threadIdx.x], &stats[3 + threadIdx.x]);
    if (threadIdx.x == 0) stats[6] = tot[6];
}

// normalization's per-pixel part (Normalization.cpp:479-496): foreground LAB values become
// (x - meanI) * ratio + target_mean in float, background ones stay, then lab2BGR.  The transfer
// factor is target_std / std in float (Normalization.cpp:402).
// A chunk's bytes pass through LDS: each thread takes its four pixels as words, settles the
// background pixels that norm_bg_fast decides and lists the others; the list is then worked
// through densely, and the chunk leaves as words again.
// 4096^2 H&E tile: 81 us (185 us with the full transform, by series, on every pixel).
// Six waves per SIMD: three workgroups of a CU work while another waits at its barrier.
__global__ __launch_bounds__(kNormThreads, 6) void k_norm_apply(NormImage I, NormConsts C, NormDisc D, NormBg G,
                                                             const double* __restrict__ part, int nblocks,
                                                             NormParams target, uint8_t* out, size_t out_ld) {
    __shared__ NormTabs T;
    __shared__ uint32_t buf[3 * kNormThreads];  // the chunk's bytes, input then result
    __shared__ uint16_t list[kNormChunk];       // pixel | foreground << 15
    __shared__ int count[2];
    __shared__ double red[kNormThreads / 64][8], tot[8];
    __shared__ NormParams sP;
    static_assert(kNormChunk <= 1 << 15, "list entries hold a pixel and a flag");
    // an item's words and the number of pixels the thread has of it; the first item's are on their way
    // while the tables and the totals are made
    auto load = [&](long long it, uint32_t wd[3]) {
        size_t off;
        const int mine = norm_group(I, (unsigned long long)it * kNormThreads + threadIdx.x, I.ld, &off);
        norm_load4(I.bgr + off, mine, wd);
        return mine;
    };
    const long long items = norm_items(I);
    uint32_t wd[3];
    int mine = load(blockIdx.x, wd);  // the grid has at most one workgroup per item
    load_log_tab(T.lg);
    for (int i = threadIdx.x; i < kExpTabN; i += kNormThreads) T.ex[i] = kExpTab[i];
    if (threadIdx.x < 2) count[threadIdx.x] = 0;
    norm_totals(part, nblocks, red, tot);
    if (threadIdx.x < 3) {
        double mean, sd;
        norm_moments(tot, threadIdx.x, &mean, &sd);
        sP.meanI[threadIdx.x] = (float)mean;
        sP.ratio[threadIdx.x] = target.ratio[threadIdx.x] / (float)sd;
    }
    __syncthreads();
    const NormParams P = sP;
    uint8_t* const by = reinterpret_cast<uint8_t*>(buf);
    int turn = 0;
    for (long long it = blockIdx.x; it < items; it += gridDim.x, turn ^= 1) {
        if (it != (long long)blockIdx.x) mine = load(it, wd);
        uint32_t px[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            px[k] = norm_px(wd, k);
            const uint32_t b = px[k] & 255u, g = px[k] >> 8 & 255u, r = px[k] >> 16;
            const bool fg = norm_fg(D, b, g, r);
            uint32_t o[3];
            const bool sure = norm_bg_fast(G, (float)b, (float)g, (float)r, o);
            const bool full = k < mine && (fg || !sure);
            if (!full) px[k] = o[0] | o[1] << 8 | o[2] << 16;
            const unsigned long long m = __ballot(full);
            if (m) {
                const int lane = threadIdx.x & 63, lead = __ffsll((long long)m) - 1;
                int base = 0;
                if (lane == lead) base = atomicAdd(&count[turn], __popcll(m));
                base = __shfl(base, lead);
                if (full)
                    list[base + __popcll(m & ((1ull << lane) - 1ull))] =
                        (uint16_t)((4 * threadIdx.x + k) | (fg ? 1u << 15 : 0u));
            }
        }
        buf[3 * threadIdx.x] = px[0] | px[1] << 24;
        buf[3 * threadIdx.x + 1] = px[1] >> 8 | px[2] << 16;
        buf[3 * threadIdx.x + 2] = px[2] >> 16 | px[3] << 8;
        if (threadIdx.x == 0) count[turn ^ 1] = 0;  // the next item's counter (nobody reads it here)
        __syncthreads();
        const int m = count[turn];
        for (int q = threadIdx.x; q < m; q += kNormThreads) {
            const uint32_t e = list[q];
            uint8_t* p = by + 3 * (e & 0x7FFFu);
            float lab[3];
            norm_lab(C, T.lg, p[0], p[1], p[2], lab);
            if (e >> 15) {
#pragma unroll
                for (int c = 0; c < 3; ++c) lab[c] = (lab[c] - P.meanI[c]) * P.ratio[c] + target.meanI[c];
            }
            uint8_t o[3];
            norm_bgr(C, T.ex, lab, o);
            p[0] = o[0];
            p[1] = o[1];
            p[2] = o[2];
        }
        __syncthreads();
        size_t ooff;
        (void)norm_group(I, (unsigned long long)it * kNormThreads + threadIdx.x, out_ld, &ooff);
        uint8_t* q = out + ooff;
        if (mine == 4 && (reinterpret_cast<uintptr_t>(q) & 3) == 0) {
            uint32_t* qw = reinterpret_cast<uint32_t*>(q);
            qw[0] = buf[3 * threadIdx.x];
            qw[1] = buf[3 * threadIdx.x + 1];
            qw[2] = buf[3 * threadIdx.x + 2];
        } else {
            for (int j = 0; j < 3 * mine; ++j) q[j] = by[12 * threadIdx.x + j];
        }
        // a thread rewrites only its own bytes of buf before the next barrier, and the list only
        // after every thread has passed the one above
    }
}

NormConsts host_consts() {
    NormConsts C;
    C.k3 = 1 / sqrtf(3.0f);
    C.k6 = 1 / sqrtf(6.0f);
    C.k2 = 1 / sqrtf(2.0f);
    C.s255 = (float)(1. / 255);
    return C;
}

NormDisc host_disc() {
    return NormDisc{{-0.154f, 0.035f, 0.549f, -45.718f, -0.057f, -0.817f, 1.170f, -49.887f}};
}

// (LMS->RGB)(RGB->LMS) in double (Normalization.cpp:83-88, 250-262): bytes to levels
NormBg host_bg() {
    const double a[3][3] = {{0.0402, 0.5783, 0.3811}, {0.0782, 0.7244, 0.1967}, {0.8444, 0.1288, 0.0241}};
    const double m[3][3] = {{0.0585, -0.2611, 1.2057}, {-1.2197, 2.3831, -0.1626}, {4.4687, -3.5887, 0.1196}};
    NormBg G;
    for (int i = 0; i < 3; ++i)
        for (int j = 0; j < 3; ++j) G.m[3 * i + j] = (float)(m[i][0] * a[0][j] + m[i][1] * a[1][j] + m[i][2] * a[2][j]);
    return G;
}

// images as one row where both planes' rows follow each other without a gap
NormImage image_of(const uint8_t* bgr, int w, int h, size_t ld, bool dense) {
    NormImage I;
    I.bgr = bgr;
    I.ld = ld;
    I.w = dense ? (size_t)w * h : (size_t)w;
    I.one_row = dense;
    I.per_row = (I.w + 3) / 4;
    I.magic = row_magic(I.per_row);
    I.groups = I.per_row * (dense ? 1ull : (unsigned long long)h);
    return I;
}

int stats_blocks(const NormImage& I) { return (int)std::min<long long>(norm_items(I), kNormMaxBlocks); }

size_t norm_scratch_bytes(int nblocks) { return sizeof(double) * 8 * ((size_t)nblocks + 1); }

int check_image(const uint8_t* bgr, int w, int h, size_t ld) {
    NSC_ARG(bgr && w > 0 && h > 0, "normalization: image");
    NSC_ARG(ld >= (size_t)3 * w, "normalization: row stride below 3 * width");
    return NSC_OK;
}

}  // namespace
}  // namespace nsc

using namespace nsc;

extern "C" int nsc_normalization_target_parameters(const uint8_t* bgr, int w, int h, size_t ld, float* mean3,
                                                   float* std3, int64_t* count, void* stream) {
    NSC_CHECK(ensure_init());
    NSC_CHECK(check_image(bgr, w, h, ld));
    NSC_ARG(mean3 && std3, "normalization_target_parameters: outputs");
    const hipStream_t s = as_stream(stream);
    const NormImage I = image_of(bgr, w, h, ld, ld == (size_t)3 * w);
    const int nb = stats_blocks(I);
    Scratch sc;
    NSC_CHECK(sc.alloc(norm_scratch_bytes(nb), s));
    double* part = sc.as<double>();
    double* stats = part + 8 * (size_t)nb;
    hipLaunchKernelGGL(k_norm_stats, dim3(nb), dim3(kNormThreads), 0, s, I, host_consts(), host_disc(), part);
    hipLaunchKernelGGL(k_norm_finish, dim3(1), dim3(kNormThreads), 0, s, part, nb, stats);
    NSC_HIP(hipGetLastError());
    double host[8];
    NSC_HIP(hipMemcpyAsync(host, stats, sizeof(host), hipMemcpyDeviceToHost, s));
    NSC_HIP(stream_sync(s));
    for (int k = 0; k < 3; ++k) {
        mean3[k] = (float)host[k];
        std3[k] = (float)host[3 + k];
    }
    if (count) *count = (int64_t)host[6];
    return NSC_OK;
}

extern "C" int nsc_normalization(const uint8_t* bgr, int w, int h, size_t ld, const float* target_mean3,
                                 const float* target_std3, uint8_t* out, size_t out_ld, void* stream) {
    NSC_CHECK(ensure_init());
    NSC_CHECK(check_image(bgr, w, h, ld));
    NSC_ARG(target_mean3 && target_std3 && out, "normalization: targets / output");
    NSC_ARG(out_ld >= (size_t)3 * w, "normalization: output row stride below 3 * width");
    // in place is fine (a chunk is read before it is written, by the same workgroup, after the
    // statistics pass); any other overlap is not
    const size_t in_bytes = ld * (size_t)(h - 1) + (size_t)3 * w, out_bytes = out_ld * (size_t)(h - 1) + (size_t)3 * w;
    NSC_ARG(out == bgr ? out_ld == ld
                       : ((const uint8_t*)out + out_bytes <= bgr || bgr + in_bytes <= (const uint8_t*)out),
            "normalization: output overlaps the input (only exact in-place use is allowed)");
    const hipStream_t s = as_stream(stream);
    const NormImage I = image_of(bgr, w, h, ld, ld == (size_t)3 * w && out_ld == ld);
    const int nb = stats_blocks(I);
    Scratch sc;
    NSC_CHECK(sc.alloc(norm_scratch_bytes(nb), s));
    double* part = sc.as<double>();
    NormParams T{};
    for (int k = 0; k < 3; ++k) {
        T.meanI[k] = target_mean3[k];
        T.ratio[k] = target_std3[k];  // k_norm_apply divides it by the image's
    }
    hipLaunchKernelGGL(k_norm_stats, dim3(nb), dim3(kNormThreads), 0, s, I, host_consts(), host_disc(), part);
    const int nbx = (int)std::min<long long>(norm_items(I), kApplyMaxBlocks);
    hipLaunchKernelGGL(k_norm_apply, dim3(nbx), dim3(kNormThreads), 0, s, I, host_consts(), host_disc(), host_bg(), part, nb,
                       T, out, out_ld);
    NSC_HIP(hipGetLastError());
    return NSC_OK;
}
