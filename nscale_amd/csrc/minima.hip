// imhmin<float> (MorphologicOperations.cpp:3342-3364) and localMaxima / localMinima<float>
// (MorphologicOperations.cpp:3763-3845).
//
// localMaxima(img, conn):
//   candidate  = !(img - 1 < imreconstruct(img - 1, img, conn))     (float arithmetic as the reference)
//   a candidate is a regional maximum unless its plateau -- the conn-connected set of candidates
//   with the same value, which is exactly the region cv::floodFill(FIXED_RANGE, lo = up = 0,
//   MASK_ONLY) marks from a seed -- holds a pixel with a strictly greater conn-neighbour (pixels
//   outside the image count as -FLT_MAX, the reference's padding).
// The flood fills become: CCL over (candidate, equal value) + OR of the "has a greater neighbour"
// flag per component root.
#include <algorithm>
#include <cfloat>
#include <vector>

#include "common.hpp"

namespace nsc {

int ccl_plateaus_without(const uint8_t* fg, const float* vals, const uint8_t* src, uint8_t* out, int w, int h, int conn,
                         int32_t* forest, uint8_t* flag, hipStream_t s);

namespace {

// For c = img, or -img (minima): cand = recon <= c - 1 (i.e. not c - 1 < recon); greater[i] = some
// conn-neighbour is > c[i].  rec is the reconstruction, negated for minima.
template <int CONN, bool MIN>
__global__ void k_lmax_cand(const float* __restrict__ c, const float* __restrict__ rec, uint8_t* __restrict__ cand,
                            uint8_t* __restrict__ greater, int w, int h) {
    const size_t n = (size_t)w * h;
    const auto gc = as_global(c);
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const int x = (int)(i % w), y = (int)(i / w);
        // all nine values from clamped (always valid) addresses, issued together; a neighbour
        // outside the image reads the pixel itself, which is never greater
        const int xl = x > 0 ? x - 1 : x, xr = x + 1 < w ? x + 1 : x;
        const size_t ru = (size_t)(y > 0 ? y - 1 : y) * w, r0 = (size_t)y * w, rd = (size_t)(y + 1 < h ? y + 1 : y) * w;
        const float rc = MIN ? -rec[i] : rec[i], v = gc[i];
        const float n0 = gc[r0 + xl], n1 = gc[r0 + xr], n2 = gc[ru + x], n3 = gc[rd + x];
        auto above = [&](float q) -> int { return MIN ? q < v : v < q; };
        int g = above(n0) | above(n1) | above(n2) | above(n3);
        if (CONN == 8) {
            const float n4 = gc[ru + xl], n5 = gc[ru + xr], n6 = gc[rd + xl], n7 = gc[rd + xr];
            g = g | above(n4) | above(n5) | above(n6) | above(n7);
        }
        const float mk = (MIN ? -v : v) - 1.0f;
        const bool cd = !(mk < rc);
        cand[i] = cd ? 1 : 0;
        greater[i] = (cd && g) ? 1 : 0;
    }
}

inline dim3 grid1(size_t n) { return dim3(std::min<unsigned>(cdiv(n, 256), 8192u)); }

// an address range that a batch reads or writes
struct Extent {
    uintptr_t lo, hi;
    bool out;
};
// whether any output's range overlaps any input's: a sweep over the ranges by their start, keeping the
// furthest end met of either kind
bool outputs_meet_inputs(std::vector<Extent>& ex) {
    std::sort(ex.begin(), ex.end(), [](const Extent& a, const Extent& b) { return a.lo < b.lo; });
    uintptr_t end[2] = {0, 0};
    for (const Extent& e : ex) {
        if (e.lo < end[e.out ? 0 : 1]) return true;
        end[e.out ? 1 : 0] = std::max(end[e.out ? 1 : 0], e.hi);
    }
    return false;
}

}  // namespace

int imhmin_impl(const float* img, float* out, int w, int h, float hval, int conn, hipStream_t s) {
    return recon_hdome_impl(img, out, w, h, conn, hval, true, false, s);
}

// scratch: float plane + int32 plane + 3 byte planes
size_t local_max_scratch(int w, int h) { return (size_t)w * h * (sizeof(float) + sizeof(int32_t) + 3); }

int local_max_impl(const float* img, uint8_t* out, int w, int h, int conn, bool minima, void* scratch, hipStream_t s) {
    const size_t n = (size_t)w * h;
    float* rec = static_cast<float*>(scratch);
    int32_t* L = reinterpret_cast<int32_t*>(rec + n);
    uint8_t* cand = reinterpret_cast<uint8_t*>(L + n);
    uint8_t* greater = cand + n;
    uint8_t* flag = greater + n;
    NSC_CHECK(recon_hdome_impl(img, rec, w, h, conn, 1.0f, minima, false, s));
    if (minima) {
        if (conn == 8) hipLaunchKernelGGL((k_lmax_cand<8, true>), grid1(n), dim3(256), 0, s, img, rec, cand, greater, w, h);
        else hipLaunchKernelGGL((k_lmax_cand<4, true>), grid1(n), dim3(256), 0, s, img, rec, cand, greater, w, h);
    } else {
        if (conn == 8) hipLaunchKernelGGL((k_lmax_cand<8, false>), grid1(n), dim3(256), 0, s, img, rec, cand, greater, w, h);
        else hipLaunchKernelGGL((k_lmax_cand<4, false>), grid1(n), dim3(256), 0, s, img, rec, cand, greater, w, h);
    }
    // plateaus of equal values: the same pixels whichever sign the values carry
    NSC_HIP(hipGetLastError());
    return ccl_plateaus_without(cand, img, greater, out, w, h, conn, L, flag, s);
}

}  // namespace nsc

using namespace nsc;

extern "C" {

int nsc_imhmin_f32_batched(const nsc_recon_desc* descs, int n, float hval, void* stream) {
    NSC_ARG(descs && n > 0, "imhmin_f32_batched");
    // before the sizes and pointers are used
    for (int i = 0; i < n; ++i)
        NSC_ARG(descs[i].mask && descs[i].out && descs[i].w > 0 && descs[i].h > 0 && valid_conn(descs[i].conn),
                "imhmin_f32_batched: descriptor");
    NSC_CHECK(ensure_init());
    hipStream_t s = as_stream(stream);
    // Every image is read until the last pass: where an output overlaps an input (in place, or another
    // image of the batch), all images are taken from copies.
    std::vector<Extent> ex;
    for (int i = 0; i < n; ++i) {
        const size_t bytes = sizeof(float) * (size_t)descs[i].w * descs[i].h;
        ex.push_back(Extent{(uintptr_t)descs[i].mask, (uintptr_t)descs[i].mask + bytes, false});
        ex.push_back(Extent{(uintptr_t)descs[i].out, (uintptr_t)descs[i].out + bytes, true});
    }
    if (!outputs_meet_inputs(ex)) return recon_hmin_batched_impl(descs, n, hval, s);
    size_t total = 0;
    for (int i = 0; i < n; ++i) total += ((size_t)descs[i].w * descs[i].h + 63) / 64 * 64;
    Scratch copy;
    NSC_CHECK(copy.alloc(sizeof(float) * total, s));
    std::vector<nsc_recon_desc> d(descs, descs + n);
    float* p = copy.as<float>();
    for (int i = 0; i < n; ++i) {
        const size_t px = (size_t)d[i].w * d[i].h;
        NSC_HIP(hipMemcpyAsync(p, d[i].mask, sizeof(float) * px, hipMemcpyDeviceToDevice, s));
        d[i].mask = p;
        p += (px + 63) / 64 * 64;
    }
    return recon_hmin_batched_impl(d.data(), n, hval, s);
}

int nsc_imhmin_f32(const float* img, float* out, int w, int h, float hval, int conn, void* stream) {
    NSC_ARG(img && out && w > 0 && h > 0 && valid_conn(conn), "imhmin_f32");
    NSC_CHECK(ensure_init());
    hipStream_t s = as_stream(stream);
    const size_t bytes = sizeof(float) * (size_t)w * h;
    const uintptr_t a = (uintptr_t)img, b = (uintptr_t)out;
    Scratch copy;
    if (a < b + bytes && b < a + bytes) {  // in place: the image is read until the last pass
        NSC_CHECK(copy.alloc(bytes, s));
        NSC_HIP(hipMemcpyAsync(copy.p, img, bytes, hipMemcpyDeviceToDevice, s));
        img = copy.as<float>();
    }
    return imhmin_impl(img, out, w, h, hval, conn, s);
}

int nsc_local_maxima_f32(const float* img, uint8_t* out, int w, int h, int conn, void* stream) {
    NSC_ARG(img && out && w > 0 && h > 0 && valid_conn(conn), "local_maxima_f32");
    NSC_LABEL_SIZE(w, h);
    NSC_CHECK(ensure_init());
    hipStream_t s = as_stream(stream);
    Scratch sc;
    NSC_CHECK(sc.alloc(local_max_scratch(w, h), s));
    return local_max_impl(img, out, w, h, conn, false, sc.p, s);
}

int nsc_local_minima_f32(const float* img, uint8_t* out, int w, int h, int conn, void* stream) {
    NSC_ARG(img && out && w > 0 && h > 0 && valid_conn(conn), "local_minima_f32");
    NSC_LABEL_SIZE(w, h);
    NSC_CHECK(ensure_init());
    hipStream_t s = as_stream(stream);
    Scratch sc;
    NSC_CHECK(sc.alloc(local_max_scratch(w, h), s));
    return local_max_impl(img, out, w, h, conn, true, sc.p, s);
}

}  // extern "C"
