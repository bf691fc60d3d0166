// Per-nucleus features of src/features/ObjFeatures.cpp (geometric: area, perimeter, ellipse axes
// and eccentricity, extent ratio, circularity; histogram statistics of an intensity plane and of
// its gradient magnitude, Operators.cpp) from a label image and the reference's box block
// (5 x n, column stride n: [label | minx | maxx | miny | maxy]).
//
// One workgroup per nucleus walks its box (the boxes hold a few hundred pixels) once: the moment
// sums of the ellipse fit are exact (offsets from the box centre are multiples of 1/2, their products
// of 1/4, summed in double), so they do not depend on the order of the additions; the perimeter
// counts the 2x2 cells of the box padded by one empty pixel per table class (identical to the
// reference's interior, edge and corner cells), the histograms are integer counts in LDS, and the
// gradient is taken at the nucleus's own pixels.  Then one wave each evaluates the intensity and the
// gradient statistics from the histograms, four bins a lane.
// A launch is bound by the latency of a workgroup's few dependent steps: 2601 nuclei of a 2048^2
// tile: 28 us (210 us with a gradient plane, the histograms in memory and one thread per nucleus
// running over 2 x 256 bins, which alone took 177 us).
#include <cfloat>
#include <cmath>

#include "common.hpp"
#include "features_rules.hpp"

namespace nsc {
namespace {

constexpr double kHalfDiag = 0.70710678118;  // ObjFeatures.cpp:151-166 table values
constexpr double kDiag = 1.41421356237;
constexpr double kPi = 3.14159265359;         // ObjFeatures.cpp:10

// table class of a marching-squares cell code: 0 none, 1 half diagonal, 2 straight, 3 two diagonals
__device__ __forceinline__ int cell_class(int m) {
    // codes 1 2 4 8 7 11 13 14 -> 1; 3 6 9 12 -> 2; 5 10 -> 3; 0 15 -> 0
    constexpr uint32_t lo = 0x6DB6;  // bit c set: class is odd  (1 or 3)
    constexpr uint32_t hi = 0x1668;  // bit c set: class >= 2    (2 or 3)
    return (int)(((lo >> m) & 1u) | (((hi >> m) & 1u) << 1));
}

// Operators::gradient (Operators.cpp:568-640) at one pixel: central differences [-0.5 0 0.5] with
// replicated borders, one-sided on the first / last column and row, float magnitude, rounded half up,
// clamped to 0..255.  Every value is exact before the square root (multiples of 1/4 below 2^17),
// and the float square root is correctly rounded, so the value is exact.
__device__ __forceinline__ int gradient_at(const uint8_t* __restrict__ img, int stride, int w, int h, int x, int y) {
    const int xl = max(x - 1, 0), xr = min(x + 1, w - 1), yu = max(y - 1, 0), yd = min(y + 1, h - 1);
    const float l = img[((size_t)y * w + xl) * stride], r = img[((size_t)y * w + xr) * stride];
    const float u = img[((size_t)yu * w + x) * stride], d = img[((size_t)yd * w + x) * stride];
    float dx = 0.5f * r - 0.5f * l;
    if (x == 0 || x == w - 1) dx *= 2.0f;
    float dy = 0.5f * d - 0.5f * u;
    if (y == 0 || y == h - 1) dy *= 2.0f;
    const float mag = __fsqrt_rn(dx * dx + dy * dy);
    const float fl = floorf(mag);
    return min((int)fl + ((mag - fl >= 0.5f) ? 1 : 0), 255);
}

struct FeatOut {
    int32_t* area;
    double *perimeter, *major, *minor, *ecc, *extent, *circ;
    float *intensity, *gradient;  // either may be null
};

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// Histogram statistics of Operators.cpp:281-505 by one wave, lane l holding the counts c[0..3] of
// bins 4 l .. 4 l + 3: f[0..] = mean, (max, min when with_minmax), std, entropy, energy, skewness,
// kurtosis.  The reference accumulates some of these in float bin by bin; here every sum is double
// and is rounded to float once.
__device__ __forceinline__ void hist_stats(const int c[4], float* f, bool with_minmax) {
    const int lane = threadIdx.x & 63;
    double ne = 0.0, hm = 0.0;  // exact: integers
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        ne += (double)c[j];
        hm += (double)c[j] * (double)(4 * lane + j);
    }
    ne = wave_sum(ne);
    hm = wave_sum(hm);
    const double mean = ne == 0.0 ? 0.0 : hm / ne, mid = hm / ne;  // mid: NaN for an empty histogram
    double s2 = 0.0, s3 = 0.0, s4 = 0.0, ent = 0.0, energy = 0.0;
    int top = -1, low = 256;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int i = 4 * lane + j;
        const double n = (double)c[j], d = (double)i - mid, p = n / ne;
        s2 += d * d * n;
        s3 += d * d * d * n;
        s4 += (d * d) * (d * d) * n;
        energy += p * p;
        if (c[j] != 0) {
            ent += p * log2(p);
            top = i;
            low = min(low, i);
        }
    }
    s2 = wave_sum(s2);
    s3 = wave_sum(s3);
    s4 = wave_sum(s4);
    ent = wave_sum(ent);
    energy = wave_sum(energy);
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        top = max(top, __shfl_xor(top, o, 64));
        low = min(low, __shfl_xor(low, o, 64));
    }
    if (lane != 0) return;
    const double var = s2 / ne, sd = sqrt(var);
    const double skew = (s3 != 0 && s2 != 0 && ne != 0) ? (s3 / ne) / (sd * sd * sd) : 0.0;
    const double kurt = (s4 != 0 && s2 != 0 && ne != 0) ? (s4 / ne) / (var * var) : 0.0;
    int k = 0;
    f[k++] = (float)mean;
    if (with_minmax) {
        f[k++] = (float)max(top, 0);
        f[k++] = (float)low;
    }
    f[k++] = (float)sd;
    f[k++] = -1.0f * (float)ent;
    f[k++] = (float)energy;
    f[k++] = (float)skew;
    f[k++] = (float)kurt;
}

// One workgroup per nucleus (grid-stride): area, moment sums, cell classes, histograms, statistics.
__global__ __launch_bounds__(256) void k_object_features(const int32_t* __restrict__ L, int w, int h,
                                                         const int32_t* __restrict__ box, int n,
                                                         const uint8_t* __restrict__ img, int stride, FeatOut F) {
    // a histogram pair per wave: a nucleus's values crowd into a few bins, and four waves' atomics on
    // the same words wait for one another
    __shared__ int hist[4][512];
    __shared__ double red[5][4];
    __shared__ int ired[4][4];
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    const bool hists = F.intensity || F.gradient;
    for (int i = blockIdx.x; i < n; i += gridDim.x) {
        const int label = box[i], minx = box[n + i], maxx = box[2 * n + i], miny = box[3 * n + i], maxy = box[4 * n + i];
        const int bw = maxx - minx + 1, bh = maxy - miny + 1;
        const float midX = (float)(minx + maxx) / 2.0f, midY = (float)(miny + maxy) / 2.0f;
        if (hists) {
            for (int k = lane; k < 512; k += 64) hist[wv][k] = 0;  // the wave's own pair
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        }
        int area = 0, c1 = 0, c2 = 0, c3 = 0;
        double sx = 0, sy = 0, sxy = 0, ssqx = 0, ssqy = 0;
        // the 2x2 marching-squares cells of the box padded by one empty pixel, (bw + 1) x (bh + 1):
        // cell (cx, cy) has pixel (minx + cx, miny + cy) as its last corner, so the walk over the cells
        // meets every pixel of the box once.  A thread's cells lie 256 apart; the position advances by
        // that step instead of being divided out.
        const CellWalk cells = cell_walk(bw, bh);  // no cells in an empty box: nothing is read for it
        const int cw = cells.cw, ch = cells.ch, dy = 256 / cw, dx = 256 - dy * cw;
        for (int cy = t / cw, cx = t - cy * cw; cy < ch; cy += dy, cx += dx, cy += cx >= cw ? 1 : 0, cx -= cx >= cw ? cw : 0) {
            const int x = minx + cx, y = miny + cy;
            // the four labels from clamped (always valid) addresses, all issued together
            const int xc = min(x, maxx), xm = max(x - 1, minx);
            const size_t rc = (size_t)min(y, maxy) * w, rm = (size_t)max(y - 1, miny) * w;
            const int l00 = L[rm + xm], l10 = L[rm + xc], l11 = L[rc + xc], l01 = L[rc + xm];
            const bool in11 = cx < bw && cy < bh && l11 == label;
            const int m = ((cx > 0 && cy > 0 && l00 == label) ? 8 : 0) | ((cx < bw && cy > 0 && l10 == label) ? 4 : 0) |
                          (in11 ? 2 : 0) | ((cx > 0 && cy < bh && l01 == label) ? 1 : 0);
            const int c = cell_class(m);
            c1 += c == 1;
            c2 += c == 2;
            c3 += c == 3;
            if (in11) {
                ++area;
                const float fx = (float)x - midX, fy = (float)y - midY;
                sx += fx;
                sy += fy;
                sxy += fx * fy;
                ssqx += fx * fx;
                ssqy += fy * fy;
                if (F.intensity) atomicAdd(&hist[wv][img[((size_t)y * w + x) * stride]], 1);
                if (F.gradient) atomicAdd(&hist[wv][256 + gradient_at(img, stride, w, h, x, y)], 1);
            }
        }
        // workgroup sums (double sums are exact: see the file comment)
        double dv[5] = {sx, sy, sxy, ssqx, ssqy};
        int iv[4] = {area, c1, c2, c3};
        for (int off = 32; off > 0; off >>= 1) {
#pragma unroll
            for (int q = 0; q < 5; ++q) dv[q] += __shfl_down(dv[q], off);
#pragma unroll
            for (int q = 0; q < 4; ++q) iv[q] += __shfl_down(iv[q], off);
        }
        if (lane == 0) {
            for (int q = 0; q < 5; ++q) red[q][wv] = dv[q];
            for (int q = 0; q < 4; ++q) ired[q][wv] = iv[q];
        }
        __syncthreads();
        if (wv < 2) {
            float* const f = wv == 0 ? F.intensity : F.gradient;
            if (f) {
                int c[4] = {0, 0, 0, 0};
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const int4 q = *reinterpret_cast<const int4*>(&hist[k][256 * wv + 4 * lane]);
                    c[0] += q.x;
                    c[1] += q.y;
                    c[2] += q.z;
                    c[3] += q.w;
                }
                hist_stats(c, f + (wv == 0 ? 8 : 6) * (size_t)i, wv == 0);
            }
        }
        if (t == 128) {  // beside the waves of the statistics
            double S[5] = {0, 0, 0, 0, 0};
            int I[4] = {0, 0, 0, 0};
            for (int k = 0; k < 4; ++k) {
                for (int q = 0; q < 5; ++q) S[q] += red[q][k];
                for (int q = 0; q < 4; ++q) I[q] += ired[q][k];
            }
            const double a = I[0];
            F.area[i] = I[0];
            // ObjFeatures::ellipse (ObjFeatures.cpp:96-110)
            const double frac = 1.0 / 12.0, root = sqrt(8.0);
            const double xbar = S[0] / a, ybar = S[1] / a;
            const double mxx = ((S[3] + a * xbar * xbar - 2.0 * xbar * S[0]) / a) + frac;
            const double myy = ((S[4] + a * ybar * ybar - 2.0 * ybar * S[1]) / a) + frac;
            const double mxy = (S[2] - ybar * S[0] - xbar * S[1] + xbar * ybar * a) / a;
            const double delta = sqrt((mxx - myy) * (mxx - myy) + 4.0 * mxy * mxy);
            const double maj = root * sqrt(mxx + myy + delta), mnr = root * sqrt(mxx + myy - delta);
            F.major[i] = maj;
            F.minor[i] = mnr;
            F.ecc[i] = (2.0 * sqrt(fabs(maj * maj - mnr * mnr) / 4.0)) / maj;
            // perimeter (ObjFeatures.cpp:144-278) from the cell class counts, extent (:118-141),
            // circularity (:281-293)
            const double per = (double)I[1] * kHalfDiag + (double)I[2] * 1.0 + (double)I[3] * kDiag;
            F.perimeter[i] = per;
            F.extent[i] = a / (double)(bw * bh);
            F.circ[i] = (4.0 * kPi * a) / (per * per);
        }
        __syncthreads();  // hist and the reduction buffers are reused by the next nucleus
    }
}

}  // namespace
}  // namespace nsc

using namespace nsc;

extern "C" int nsc_object_features(const int32_t* labels, int w, int h, const int32_t* bbox5, int n, const uint8_t* img,
                                   int channels, int channel, nsc_object_features_out* out, void* stream) {
    NSC_ARG(labels && bbox5 && out && w > 0 && h > 0 && n >= 0, "object_features");
    NSC_ARG(!img || (channels >= 1 && channel >= 0 && channel < channels), "object_features: channels");
    NSC_ARG(out->area && out->perimeter && out->major_axis && out->minor_axis && out->eccentricity &&
                out->extent_ratio && out->circularity, "object_features: geometric outputs");
    NSC_ARG(img || (!out->intensity && !out->gradient), "object_features: intensity outputs need an image");
    NSC_LABEL_SIZE(w, h);
    NSC_CHECK(ensure_init());
    if (n == 0) return NSC_OK;
    hipStream_t s = as_stream(stream);
    const FeatOut F{out->area,         out->perimeter, out->major_axis, out->minor_axis, out->eccentricity,
                    out->extent_ratio, out->circularity, out->intensity, out->gradient};
    hipLaunchKernelGGL(k_object_features, dim3(std::min(n, 8192)), dim3(256), 0, s, labels, w, h, bbox5, n,
                       img ? img + channel : nullptr, channels, F);
    NSC_HIP(hipGetLastError());
    return NSC_OK;
}
