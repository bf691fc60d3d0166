// Connected components and everything built on them:
//   ConnComponents::label / bwlabel2 / relabel / areaThresholdLabeled / boundingBox
//   (ConnComponents.cpp:24-284, MorphologicOperations.cpp:3092-3117, 3281-3314), and the binary
//   reconstruction family imreconstructBinary / imfill / imfillHoles / bwselect
//   (MorphologicOperations.cpp:2768-3031), which are component selections: a pixel of the
//   passable set is reached iff its component contains a seed.
//
// Labelling is union-find with the smallest raster index as root (the reference's merge links
// the larger root under the smaller, ConnComponents.cpp:34-43, so its labels are also the
// smallest index of each component).  It works on runs, not pixels: a run is a maximal stretch of
// left-joined pixels within one row of a 64 x 64 tile, and a row of a tile is two 64-bit words, the
// foreground F and the run starts S.
//   1. ccl_tile: one wave per tile, lane = row.  Bit operations on F and S give the joins to unite
//      (a run's own joins need no union), the runs, numbered in raster order, unite in LDS with
//      atomicMin on their numbers, and the tile leaves behind its F and S words, a code for every run
//      (two bytes: the number of its tile-local root, whether that root is closed, and if so whether it is
//      selected), the places of the roots along its four edges, and for each open root its entry in the
//      forest P (the root's own global index) with what the caller needs of it: pixel count or flag.  A
//      component that meets no other tile is closed: its root, count and flag are final there;
//   2. ccl_seams: two waves per tile unite the runs that meet across its left and its top edge, in P;
//   3. ccl_roots (selections): each open root, found along the edges, finds its final root and hands its
//      count or flag over;
//   4. ccl_select writes the selected pixels, ccl_label the labels: both expand the words again.
// P is indexed by pixel but only the entries of open roots exist; no other per-pixel label is
// stored on the way.  Bytes moved per pixel: about 0.4 for the words and roots, the image in and the
// result out.  Labelling per pixel instead (labels in LDS, stored, seams from the stored labels, a
// flattening pass, a consumer pass) moved 17 and was bound by instruction issue in its tile pass.
// Only what crosses an edge is followed through memory: an image may have as many components as pixels.  With an
// entry, a walk and a lookup for every tile-local root, area opening of 4096 x 4096 differing pixels took 1365 us
// (183 with codes), hole filling of a checkerboard 573 (82), labels of 50 % noise 600 x 600 44 (31).
// Pixel classes: FG_NEQ  -> foreground = value != key; neighbours join when both foreground
//                FG_EQ   -> foreground = value != 0; neighbours join when values are equal
//                FG_FEQ  -> foreground = cls != 0; neighbours join when float values are equal
#include <algorithm>
#include <climits>
#include <type_traits>

#include "common.hpp"

namespace nsc {
namespace {

constexpr int CT = 64;  // tile side: lanes of a wave, bits of a word
enum { FG_NEQ = 0, FG_EQ = 1, FG_FEQ = 2 };

struct Px {
    const uint8_t* img;
    const float* fv;
    uint8_t key;
};

// find with intermediate pointer jumping (each visited node is re-pointed to its grandparent).
// Parents are always smaller than children, and a non-root never becomes a root again, so
// re-pointing a non-root to any ancestor keeps every set intact; a concurrent union that lowers
// the same pointer continues its own loop with the value it replaced (see unite), so a lost
// update only shortens a path.
// relaxed atomic accesses: other threads update the forest concurrently, so no access may be
// kept in a register by the compiler
__device__ __forceinline__ int ld_wg(const int* a) { return __hip_atomic_load(a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); }

// A run's node in LDS: its number's parent in the low half, the place of its first pixel in the tile
// (row * 64 + column) in the high one.
__device__ __forceinline__ int parent_of(const uint32_t* N, int x) {
    return (int)(__hip_atomic_load(&N[x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) & 0xFFFFu);
}
__device__ __forceinline__ uint32_t node_of(const uint32_t* N, int x) {
    return __hip_atomic_load(&N[x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Unites the sets of a and b.  Both walk to their roots together (each step's two reads in one round
// trip), re-pointing what they pass to its grandparent, and stop as soon as they meet.
__device__ __forceinline__ void lunite(uint32_t* N, int a, int b) {
    while (true) {
        uint32_t na = node_of(N, a), nb = node_of(N, b);
        int pa = (int)(na & 0xFFFFu), pb = (int)(nb & 0xFFFFu);
        while (pa != a || pb != b) {
            if (pa == pb) return;
            const uint32_t qa = node_of(N, pa), qb = node_of(N, pb);
            const int ga = (int)(qa & 0xFFFFu), gb = (int)(qb & 0xFFFFu);
            if (ga != pa) __hip_atomic_store(&N[a], (na & 0xFFFF0000u) | ga, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            if (gb != pb) __hip_atomic_store(&N[b], (nb & 0xFFFF0000u) | gb, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            a = pa;
            na = qa;
            pa = ga;
            b = pb;
            nb = qb;
            pb = gb;
        }
        if (a == b) return;
        if (a > b) {
            const int t = a;
            a = b;
            b = t;
            nb = na;
        }
        // the high halves are equal, so the minimum is that of the parents
        const int old = (int)(atomicMin(&N[b], (nb & 0xFFFF0000u) | (uint32_t)a) & 0xFFFFu);
        if (old == b) return;
        b = old;
    }
}

// Orders LDS accesses between the lanes of one wave (they execute in program order).
__device__ __forceinline__ void wave_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// relaxed device-scope accesses: unions from every workgroup of the launch update the forest
__device__ __forceinline__ int ld_rel(const int* a) { return __hip_atomic_load(a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ void st_rel(int* a, int v) { __hip_atomic_store(a, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

// The same union in global memory, of two tile-local roots.  What bounds the seams of a component that
// spans the image is the chain of dependent round trips to the forest (about a microsecond each, past
// the XCDs' own L2s), so both walks advance together and end where they meet.
__device__ __forceinline__ void gunite(int32_t* L, int a, int b) {
    int pa = ld_rel(&L[a]), pb = ld_rel(&L[b]);
    while (true) {
        while (pa != a || pb != b) {
            if (pa == pb) return;
            const int ga = ld_rel(&L[pa]), gb = ld_rel(&L[pb]);
            if (ga != pa) st_rel(&L[a], ga);
            if (gb != pb) st_rel(&L[b], gb);
            a = pa;
            pa = ga;
            b = pb;
            pb = gb;
        }
        if (a == b) return;
        if (a > b) { const int t = a; a = b; b = t; }
        const int old = atomicMin(&L[b], a);
        if (old == b) return;
        b = old;
        pa = ld_rel(&L[a]);
        pb = ld_rel(&L[b]);
    }
}

// ---- the words of a tile -------------------------------------------------------------------
struct RowWords {
    uint64_t S, F;  // run starts, foreground
};

// What a labelling leaves per tile: the words of its 64 rows, the number of runs before each row, the
// code of every run (the number of its tile-local root; kClosed where the component meets no other tile,
// and then kSelected where a selection takes it), the places of the roots along the four edges (kNoRoot
// for background), and, for the equal-value modes, the values of its first and last column (the seams
// compare them).
constexpr uint16_t kNoRoot = 0xFFFF;
constexpr uint32_t kRunRoot = 0x0FFF, kSelected = 0x4000, kClosed = 0x8000;
enum { E_LEFT = 0, E_RIGHT = 1, E_TOP = 2, E_BOTTOM = 3 };
struct CclBufs {
    RowWords* rows;
    uint16_t *off, *roots;
    uint16_t* edge_roots;  // [tile][4][64]
    void* edge;            // uint8_t or float, [tile][2][64]
    int cap;               // run slots of a tile (a multiple of 8)
};

__device__ __forceinline__ int popc64(uint64_t v) { return (int)__popcll(v); }
__device__ __forceinline__ uint64_t upto(int x) { return (2ull << x) - 1ull; }  // bits 0..x (x <= 63: 2 << 63 wraps to 0)
// number, within its row, of the run that holds the foreground pixel at column x
__device__ __forceinline__ int run_index(uint64_t S, int x) { return popc64(S & upto(x)) - 1; }
// first column after the run that starts at a
__device__ __forceinline__ int run_end(uint64_t S, uint64_t F, int a) {
    const uint64_t stop = (S | ~F) & ~upto(a);
    return stop ? __ffsll((long long)stop) - 1 : 64;
}
__device__ __forceinline__ uint64_t run_bits(int a, int end) { return (end < 64 ? 1ull << end : 0ull) - (1ull << a); }

__device__ __forceinline__ uint64_t shfl_up64(uint64_t v) {  // from lane - 1; lane 0 receives 0
    return (uint64_t)(uint32_t)dpp_from_left(0, (int)(uint32_t)v) |
           (uint64_t)(uint32_t)dpp_from_left(0, (int)(uint32_t)(v >> 32)) << 32;
}

// 0x80 in every nonzero byte
__device__ __forceinline__ uint32_t nonzero_bytes(uint32_t x) { return (((x & 0x7f7f7f7fu) + 0x7f7f7f7fu) | x) & 0x80808080u; }
// The flags of eight bytes (as 0x80) as one byte: byte products with the bits' weights, summed
__device__ __forceinline__ uint32_t gather_bits(uint32_t t0, uint32_t t1) {
    return __builtin_amdgcn_udot4(t1, 0x80402010u, __builtin_amdgcn_udot4(t0, 0x08040201u, 0u, false), false) >> 7;
}
// four bits as four bytes of 0 / 255
__device__ __forceinline__ uint32_t spread_bits(uint32_t b) { return ((b * 0x00204081u) & 0x01010101u) * 255u; }

// 16 bytes of a row from column x of `cols` (any alignment; whole when `full`, else the bytes past the
// row repeat its last one)
__device__ __forceinline__ uint4 load16(const uint8_t* row, int x, int cols, bool full) {
    uint4 v;
    if (full) {
        __builtin_memcpy(&v, row + x, 16);
    } else {
        uint32_t wd[4] = {0, 0, 0, 0};
#pragma unroll
        for (int j = 0; j < 16; ++j) wd[j >> 2] |= (uint32_t)row[min(x + j, cols - 1)] << (8 * (j & 3));
        v = make_uint4(wd[0], wd[1], wd[2], wd[3]);
    }
    return v;
}

// Bit x of lane y's result: pixel (x0 + x, y0 + y) lies in the image and differs from key.  A lane
// loads four 16-byte pieces (a row is four lanes), turns each into 16 bits, and the rows come
// together through LDS.
__device__ __forceinline__ uint64_t tile_bits(const uint8_t* __restrict__ img, int w, int h, int x0, int y0, uint32_t key,
                                              uint16_t* stage) {
    const int lane = threadIdx.x & 63, r = lane >> 2, x = 16 * (lane & 3);
    const int cols = min(CT, w - x0);
    const bool full = cols == CT;
    uint4 v[4];
#pragma unroll
    for (int g = 0; g < 4; ++g)
        v[g] = load16(img + (size_t)min(y0 + 16 * g + r, h - 1) * w + x0, x, cols, full);
    const uint32_t k4 = key * 0x01010101u;
    const uint32_t inside = full ? 0xFFFFu : (x >= cols ? 0u : (uint32_t)((2u << min(cols - 1 - x, 15)) - 1u));
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        const uint32_t bits = gather_bits(nonzero_bytes(v[g].x ^ k4), nonzero_bytes(v[g].y ^ k4)) |
                              gather_bits(nonzero_bytes(v[g].z ^ k4), nonzero_bytes(v[g].w ^ k4)) << 8;
        stage[4 * (16 * g + r) + (lane & 3)] = (uint16_t)(y0 + 16 * g + r < h ? bits & inside : 0u);
    }
    wave_order();
    const uint64_t m = *reinterpret_cast<const uint64_t*>(stage + 4 * lane);
    wave_order();
    return m;
}

// The joins of a row to unite with the row above.  A vertical or diagonal join is united only where no
// join further left already connects the same two runs (F, jl: this row's foreground and left joins;
// ju, jul, jur: joins with the pixel above, above left, above right; jlu: left joins of the row above):
//   up:        skipped when the pixel joins its left one, that one joins up, and the pixels above join;
//   up-left:   skipped when the pixel joins up and the pixels above join, or it joins its left one and
//              that one joins up;
//   up-right:  skipped when the pixel joins up and the pixels above join, or the pixel to its right
//              joins it and joins up.
// Every skipped join is implied by a path through joins that are united or skipped only by a rule
// that looks further left, so the components are those of all joins.
struct JoinWords {
    uint64_t up, ul, ur;
};
template <int CONN>
__device__ __forceinline__ JoinWords joins_to_unite(uint64_t jl, uint64_t ju, uint64_t jul, uint64_t jur, uint64_t jlu) {
    JoinWords J;
    J.up = ju & ~(jl & (ju << 1) & jlu);
    J.ul = CONN == 8 ? jul & ~((ju & jlu) | (jl & (ju << 1))) : 0ull;
    J.ur = CONN == 8 ? jur & ~((ju & (jlu >> 1)) | ((jl >> 1) & (ju >> 1))) : 0ull;
    return J;
}

// The words and joins of a tile where equal byte values join: the tile's bytes come to LDS, each lane
// takes its row as 16 dwords (and the row above from the lane before it), and every comparison with a
// neighbour is byte arithmetic on four pixels at a time.  (One ballot per row and comparison took 51 us
// for a 4096 x 3071 mask, this 23 us.)  Returns the row's first and last byte, one above the other.
constexpr int kBytePitch = 17;  // dwords per staged row: the lanes' rows start in different banks
template <int CONN>
__device__ __forceinline__ uint32_t tile_words_eq(const uint8_t* __restrict__ img, int w, int h, int x0, int y0, RowWords& R,
                                              JoinWords& J, uint32_t* stage) {
    const int lane = threadIdx.x & 63, r = lane >> 2, x = 16 * (lane & 3);
    const int cols = min(CT, w - x0);
    const bool full = cols == CT;
    uint4 v[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) v[g] = load16(img + (size_t)min(y0 + 16 * g + r, h - 1) * w + x0, x, cols, full);
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        uint32_t* q = stage + (16 * g + r) * kBytePitch + 4 * (lane & 3);
        q[0] = v[g].x;
        q[1] = v[g].y;
        q[2] = v[g].z;
        q[3] = v[g].w;
    }
    wave_order();
    uint32_t c[16], u[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) c[j] = stage[lane * kBytePitch + j];
    wave_order();
#pragma unroll
    for (int j = 0; j < 16; ++j) u[j] = (uint32_t)dpp_from_left(0, (int)c[j]);
    uint64_t F = 0, nl = 0, nu = 0, nul = 0, nur = 0;  // foreground; pixels that differ from that neighbour
#pragma unroll
    for (int j = 0; j < 16; j += 2) {
        const int sh = 4 * j;
        // the pixels' left, upper left and upper right neighbours: the words shifted by a byte
        const uint32_t l0 = c[j] << 8 | (j ? c[j ? j - 1 : 0] >> 24 : 0u), l1 = c[j + 1] << 8 | c[j] >> 24;
        F |= (uint64_t)gather_bits(nonzero_bytes(c[j]), nonzero_bytes(c[j + 1])) << sh;
        nl |= (uint64_t)gather_bits(nonzero_bytes(c[j] ^ l0), nonzero_bytes(c[j + 1] ^ l1)) << sh;
        nu |= (uint64_t)gather_bits(nonzero_bytes(c[j] ^ u[j]), nonzero_bytes(c[j + 1] ^ u[j + 1])) << sh;
        if (CONN == 8) {
            const uint32_t a0 = u[j] << 8 | (j ? u[j ? j - 1 : 0] >> 24 : 0u), a1 = u[j + 1] << 8 | u[j] >> 24;
            const uint32_t b0 = u[j] >> 8 | u[j + 1] << 24, b1 = u[j + 1] >> 8 | (j < 14 ? u[j < 14 ? j + 2 : 15] << 24 : 0u);
            nul |= (uint64_t)gather_bits(nonzero_bytes(c[j] ^ a0), nonzero_bytes(c[j + 1] ^ a1)) << sh;
            nur |= (uint64_t)gather_bits(nonzero_bytes(c[j] ^ b0), nonzero_bytes(c[j + 1] ^ b1)) << sh;
        }
    }
    if (!full) F &= (1ull << cols) - 1ull;
    if (y0 + lane >= h) F = 0;
    const uint64_t Fu = shfl_up64(F);
    const uint64_t jl = F & (F << 1) & ~nl;
    R = RowWords{F & ~jl, F};
    J = joins_to_unite<CONN>(jl, F & Fu & ~nu, F & (Fu << 1) & ~nul, F & (Fu >> 1) & ~nur, shfl_up64(jl));
    return (c[0] & 255u) | (c[15] >> 24) << 8;
}

// The same where equal floats join (NaN joins nothing): four waves of 16 rows each, lane = column; each
// comparison of a row is one ballot, and row y's words go through LDS to lane y of the first wave.
constexpr int kEqWords = 5;
template <int CONN>
__device__ __forceinline__ void tile_words_feq(const Px& P, int w, int h, int x0, int y0, RowWords& R, JoinWords& J,
                                               float* edge, uint64_t (*words)[kEqWords]) {
    const int lane = threadIdx.x & 63, r0 = 16 * (threadIdx.x >> 6);
    const size_t gxc = (size_t)min(x0 + lane, w - 1);
    const bool in_x = x0 + lane < w;
    uint8_t c[17];
    float f[17];
    // every load first, from clamped (always valid) addresses; entry 0 is the row above the wave's
#pragma unroll
    for (int j = 0; j < 17; ++j) {
        const size_t i = (size_t)min(max(y0 + r0 + j - 1, 0), h - 1) * w + gxc;
        c[j] = as_global(P.img)[i];
        f[j] = as_global(P.fv)[i];
    }
    __builtin_amdgcn_sched_barrier(0);
    const bool above = r0 > 0;  // row 0's neighbours above belong to another tile
    uint64_t pF = __ballot(above && in_x && y0 + r0 - 1 < h && c[0] != 0);
    float pl = from_left(0.0f, f[0]);
    uint64_t pjl = __ballot(f[0] == pl) & pF & (pF << 1);
#pragma unroll
    for (int j = 1; j < 17; ++j) {
        const int y = r0 + j - 1;
        const float v = f[j], l = from_left(0.0f, v);
        const uint64_t F = __ballot(in_x && y0 + y < h && c[j] != 0);
        const uint64_t jl = __ballot(v == l) & F & (F << 1);
        const uint64_t ju = __ballot(v == f[j - 1]) & F & pF;
        uint64_t jul = 0, jur = 0;
        if (CONN == 8) {
            jul = __ballot(v == pl) & F & (pF << 1);
            jur = __ballot(v == from_right(0.0f, f[j - 1])) & F & (pF >> 1);
        }
        const JoinWords q = joins_to_unite<CONN>(jl, ju, jul, jur, pjl);
        const uint64_t word[kEqWords] = {F & ~jl, F, q.up, q.ul, q.ur};
        if (lane < kEqWords) {
            uint64_t v5 = word[0];
#pragma unroll
            for (int k = 1; k < kEqWords; ++k) v5 = lane == k ? word[k] : v5;
            words[y][lane] = v5;
        }
        if (lane == 0) edge[y] = v;
        if (lane == 63) edge[CT + y] = v;
        pl = l;
        pF = F;
        pjl = jl;
    }
    __syncthreads();
    R = RowWords{words[lane][0], words[lane][1]};
    J = JoinWords{words[lane][2], words[lane][3], words[lane][4]};
}

enum { SRC_NONE = 0, SRC_BYTES = 1, SRC_BORDER = 2 };

constexpr int ccl_cap(int mode) { return mode == FG_NEQ ? CT * CT / 2 : CT * CT; }  // most runs of a tile
constexpr int kManyRuns = 512;  // runs from which four waves share a tile: eight a row, a mask of noise
constexpr int kFewRuns = 512;   // codes that the consumers load before they know the run count
constexpr int ccl_tile_threads(int mode, int waves) { return mode == FG_FEQ ? 256 : 64 * waves; }

// global index of the place r of tile (tx, ty)
__device__ __forceinline__ int place_index(int tx, int ty, int r, int w) {
    return (int)((size_t)(ty * CT + (r >> 6)) * w + (tx * CT + (r & 63)));
}
// whether another tile lies across a side of tile (tx, ty)
__device__ __forceinline__ bool side_open(int side, int tx, int ty, int tiles_x, int tiles_y) {
    return side == E_LEFT ? tx > 0 : (side == E_RIGHT ? tx + 1 < tiles_x : (side == E_TOP ? ty > 0 : ty + 1 < tiles_y));
}

// A tile from its words on, by one wave (solo) or by four, each with the runs that start in 16 columns.
struct TileWork {
    CclBufs B;
    int32_t* forest;
    int w, tx, ty, tiles_x, tiles_y;
    int32_t* area;
    int lo, hi;
    uint8_t* flag;
};
template <int SRC, bool solo>
__device__ __forceinline__ void ccl_tile_runs(const TileWork& K, uint32_t* node, const RowWords R, JoinWords J, const uint64_t T,
                                              const int off, const int wv) {
    const CclBufs& B = K.B;
    int32_t* const forest = K.forest;
    int32_t* const area = K.area;
    uint8_t* const flag = K.flag;
    const int w = K.w, tx = K.tx, ty = K.ty, tiles_x = K.tiles_x, tiles_y = K.tiles_y, lo = K.lo, hi = K.hi;
    const int lane = threadIdx.x & 63;
    const int nrun = popc64(R.S), tid = solo ? lane : (int)threadIdx.x;
    constexpr int threads = solo ? 64 : 256;
    // between steps that read in LDS what another lane has written
    auto order = [&] {
        if (solo) wave_order();
        else __syncthreads();
    };
    auto any = [&](bool v) { return solo ? __any(v) != 0 : __syncthreads_or(v ? 1 : 0) != 0; };
    const uint64_t Su = shfl_up64(R.S);
    const int offu = dpp_from_left(0, off);
    const int row = lane * CT, runs = __builtin_amdgcn_readlane(off + nrun, 63);
    // the wave's runs, the number of the first, and their joins
    uint64_t mine = R.S;
    int first = off;
    if (!solo) {
        const uint64_t before = (1ull << (16 * wv)) - 1ull, in = 0xFFFFull << (16 * wv);
        mine = R.S & in;
        first = off + popc64(R.S & before);
        const uint64_t after = R.S & ~(before | in);  // the next wave's first run ends the last of these
        const uint64_t px = mine ? (after ? (after & (0ull - after)) - 1ull : ~0ull) & ~((mine & (0ull - mine)) - 1ull) : 0ull;
        J = JoinWords{J.up & px, J.ul & px, J.ur & px};
    }
    // A run starts out pointing at the run above of one of its joins, if it has any (a smaller number,
    // so this is a forest without any atomics), and the forest is flattened: along a tall component
    // one union per row at once would build a chain that every later find walks.  The joins that
    // are left, where a run meets a second run above it, unite what is flat already.
    {
        int k = first;
        for (uint64_t m = mine; m; m &= m - 1, ++k) {
            const int a = __ffsll((long long)m) - 1;
            const uint64_t rb = run_bits(a, run_end(R.S, R.F, a)), up = J.up & rb, ul = J.ul & rb, ur = J.ur & rb;
            const uint64_t f = up ? up : (ul ? ul : ur);
            const int x = __ffsll((long long)f) - 1;
            int par = k;
            if (f) par = offu + run_index(Su, up ? x : (ul ? x - 1 : x + 1));
            const uint64_t clr = ~(f & (0ull - f));
            if (up) J.up &= clr;
            else if (ul) J.ul &= clr;
            else J.ur &= clr;
            node[k] = (uint32_t)(row + a) << 16 | (uint32_t)par;
        }
    }
    order();
    // every run at its root: pointer doubling, thread = run, four runs' reads in one round trip
    auto flatten = [&]() {
        for (;;) {
            bool changed = false;
            for (int k0 = 0; k0 < runs; k0 += 4 * threads) {
                uint32_t v[4];
                int q[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) v[j] = node_of(node, min(k0 + threads * j + tid, runs - 1));
#pragma unroll
                for (int j = 0; j < 4; ++j) q[j] = parent_of(node, (int)(v[j] & 0xFFFFu));
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int k = k0 + threads * j + tid;
                    if (k < runs && q[j] != (int)(v[j] & 0xFFFFu)) {
                        node[k] = (v[j] & 0xFFFF0000u) | (uint32_t)q[j];
                        changed = true;
                    }
                }
            }
            if (solo) wave_order();
            if (!any(changed)) break;
        }
    };
    flatten();
    if (any((J.up | J.ul | J.ur) != 0)) {
        // one union per lane and turn, straight ones first
        while (J.up | J.ul | J.ur) {
            const uint64_t m = J.up ? J.up : (J.ul ? J.ul : J.ur);
            const int x = __ffsll((long long)m) - 1, xu = J.up ? x : (J.ul ? x - 1 : x + 1);
            const uint64_t clr = ~(m & (0ull - m));
            if (J.up) J.up &= clr;
            else if (J.ul) J.ul &= clr;
            else J.ur &= clr;
            lunite(node, off + run_index(R.S, x), offu + run_index(Su, xu));
        }
        order();
        flatten();
    }
    // edge pixels: left and right of the lane's row, top and bottom of the lane's column.  Roots that they hold
    // on a side with a tile across it are open.
    constexpr uint32_t kOpen = 1u << 30;
    uint16_t* const er = B.edge_roots + (size_t)blockIdx.x * 4 * CT;
    int eroot[4], eplace[4];  // open roots that no pixel before it on the side has: number (else -1), place
    {
        auto edge = [&](int side, bool fg, int k) {
            eroot[side] = -1;
            eplace[side] = 0;
            if (!solo && side != wv) return;  // a side a wave
            const int r = fg ? parent_of(node, k) : 0;
            const int p = (int)(node_of(node, r) >> 16 & 0xFFFu);
            er[side * CT + lane] = fg ? (uint16_t)p : kNoRoot;
            const int o = fg && side_open(side, tx, ty, tiles_x, tiles_y) ? r : -1;
            eroot[side] = o != dpp_from_left(-1, o) ? o : -1;
            eplace[side] = p;
            if (eroot[side] >= 0) atomicOr(&node[o], kOpen);  // (bits that no reader of a place or parent looks at)
        };
        auto word_of = [](uint64_t v, int l) {
            return (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, l) |
                   (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), l) << 32;
        };
        const uint64_t S0 = word_of(R.S, 0), F0 = word_of(R.F, 0), S3 = word_of(R.S, 63), F3 = word_of(R.F, 63);
        const int off3 = __builtin_amdgcn_readlane(off, 63);
        edge(E_LEFT, R.F & 1ull, off);
        edge(E_RIGHT, R.F >> 63, off + nrun - 1);
        edge(E_TOP, (F0 >> lane) & 1ull, run_index(S0, lane));
        edge(E_BOTTOM, (F3 >> lane) & 1ull, off3 + run_index(S3, lane));
    }
    order();
    if (area || SRC != SRC_NONE) {
        // the roots' places are not needed any more: count in bits 16..28, flag in bit 31
        for (int k = tid; k < runs; k += threads) {
            const uint32_t v = node_of(node, k);
            if ((int)(v & 0xFFFFu) == k) node[k] = (v & kOpen) | (uint32_t)k;
        }
        order();
        int k = first;
        for (uint64_t m = mine; m; m &= m - 1, ++k) {
            const int a = __ffsll((long long)m) - 1, end = run_end(R.S, R.F, a), r = parent_of(node, k);
            if (area) atomicAdd(&node[r], (uint32_t)(end - a) << 16);
            if (SRC != SRC_NONE && (T & run_bits(a, end))) atomicOr(&node[r], 0x80000000u);
        }
        order();
    }
    // the runs' codes, four at a time
    uint16_t* const roots = B.roots + (size_t)blockIdx.x * B.cap;
    for (int k0 = 4 * tid; k0 < runs; k0 += 4 * threads) {
        const uint4 q = *reinterpret_cast<const uint4*>(&node[k0]);
        const uint32_t r[4] = {q.x & kRunRoot, q.y & kRunRoot, q.z & kRunRoot, q.w & kRunRoot};
        uint32_t code[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t v = node_of(node, k0 + j < runs ? (int)r[j] : 0);
            const int c = (int)(v >> 16 & 0x1FFFu);
            const bool sel = SRC != SRC_NONE ? (v >> 31) != 0 : area && c >= lo && c < hi;
            code[j] = r[j] | (v & kOpen ? 0u : kClosed | (sel ? kSelected : 0u));
        }
        *reinterpret_cast<uint2*>(roots + k0) = make_uint2(code[0] | code[1] << 16, code[2] | code[3] << 16);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        if (eroot[e] < 0) continue;
        const uint32_t v = node_of(node, eroot[e]);
        const int g = place_index(tx, ty, eplace[e], w);
        forest[g] = g;
        if (area) area[g] = (int)(v >> 16 & 0x1FFFu);
        if (SRC != SRC_NONE) flag[g] = (uint8_t)(v >> 31);
    }
}

// One tile per workgroup, by its first wave once the words are there; where the launch has four waves a tile
// (kFewTiles), a tile of more than kManyRuns runs is shared by all four.  Per open root: P = its own index; area
// (optional) = the pixels of its tile-local component; flag (optional) = whether that holds a source
// pixel: a nonzero pixel of src (SRC_BYTES) or a pixel on the image border (SRC_BORDER).  A closed root is
// selected by its area in [lo, hi), or by its flag.  *zero (optional) is cleared for the passes that follow.
template <int MODE, int CONN, int SRC, int WAVES>
__global__ __launch_bounds__(ccl_tile_threads(MODE, WAVES)) void ccl_tile(Px P, CclBufs B, int32_t* __restrict__ forest, int w, int h,
                                                                   int tiles_x, int32_t* __restrict__ area, int lo,
                                                                   int hi, uint8_t* __restrict__ flag,
                                                                   const uint8_t* __restrict__ src, int* __restrict__ zero) {
    // the runs' nodes (8 KB of LDS for binary masks: every tile of a 4096^2 image is resident at once)
    __shared__ alignas(16) uint32_t node[ccl_cap(MODE)];
    __shared__ union {
        uint16_t bits[4 * CT];
        uint32_t bytes[MODE == FG_EQ ? CT * kBytePitch : 1];
        uint64_t words[MODE == FG_FEQ ? CT : 1][kEqWords];
    } stage;
    __shared__ uint64_t shared_words[WAVES > 1 ? CT : 1][6];
    __shared__ int shared_runs;
    const int tx = blockIdx.x % tiles_x, ty = blockIdx.x / tiles_x, tiles_y = gridDim.x / tiles_x;
    const int x0 = tx * CT, y0 = ty * CT, lane = threadIdx.x & 63;
    const int wv = ccl_tile_threads(MODE, WAVES) == 64 ? 0 : __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    if (zero && blockIdx.x == 0 && threadIdx.x == 0) *zero = 0;
    RowWords R{};
    JoinWords J{};
    uint64_t T = 0;  // source pixels of the row
    uint32_t ends = 0;
    if constexpr (MODE == FG_FEQ) {
        tile_words_feq<CONN>(P, w, h, x0, y0, R, J, static_cast<float*>(B.edge) + (size_t)blockIdx.x * 2 * CT, stage.words);
        if (WAVES == 1 && wv) return;
        if (WAVES > 1) __syncthreads();
        else wave_order();  // the words have been read before their LDS holds bits
    }
    if (wv == 0) {
        if constexpr (MODE == FG_NEQ) {
            R.F = tile_bits(P.img, w, h, x0, y0, P.key, stage.bits);
            const uint64_t jl = R.F & (R.F << 1), Fu = shfl_up64(R.F);
            R.S = R.F & ~jl;
            J = joins_to_unite<CONN>(jl, R.F & Fu, R.F & (Fu << 1), R.F & (Fu >> 1), Fu & (Fu << 1));
        } else if constexpr (MODE == FG_EQ) {
            ends = tile_words_eq<CONN>(P.img, w, h, x0, y0, R, J, stage.bytes);
        }
        if constexpr (SRC == SRC_BYTES) T = tile_bits(src, w, h, x0, y0, 0, stage.bits);
        if constexpr (SRC == SRC_BORDER) {
            const int y = y0 + lane;
            if (y == 0 || y == h - 1) T = ~0ull;
            if (x0 == 0) T |= 1ull;
            if (w - 1 - x0 < CT) T |= 1ull << (w - 1 - x0);
        }
    }
    // the rows' first run numbers: exclusive scan of the run counts
    auto first_runs = [&] {
        int o = popc64(R.S);
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int q = __shfl_up(o, d);
            if (lane >= d) o += q;
        }
        return o - popc64(R.S);
    };
    int off = first_runs();
    bool solo = true;
    if constexpr (WAVES > 1) {
        if (wv == 0) {
            const uint64_t v[6] = {R.S, R.F, J.up, J.ul, J.ur, T};
            const int n = __builtin_amdgcn_readlane(off + popc64(R.S), 63);
            if (lane == 0) shared_runs = n;
            if (n > kManyRuns)
#pragma unroll
                for (int k = 0; k < 6; ++k) shared_words[lane][k] = v[k];
        }
        __syncthreads();
        solo = __builtin_amdgcn_readfirstlane(shared_runs) <= kManyRuns;  // (wave-uniform)
        if (solo && wv) return;
        if (!solo && wv) {
            const uint64_t* v = shared_words[lane];
            R = RowWords{v[0], v[1]};
            J = JoinWords{v[2], v[3], v[4]};
            T = v[5];
            off = first_runs();
        }
    }
    if (wv == 0) {  // (stores after the barrier, which would wait for them)
        B.rows[(size_t)blockIdx.x * CT + lane] = R;
        B.off[(size_t)blockIdx.x * CT + lane] = (uint16_t)off;
        if constexpr (MODE == FG_EQ) {
            uint8_t* const edge = static_cast<uint8_t*>(B.edge) + (size_t)blockIdx.x * 2 * CT;
            edge[lane] = (uint8_t)ends;
            edge[CT + lane] = (uint8_t)(ends >> 8);
        }
    }
    const TileWork K{B, forest, w, tx, ty, tiles_x, tiles_y, area, lo, hi, flag};
    if constexpr (WAVES > 1) {
        if (__builtin_expect(!solo, 0)) {
            ccl_tile_runs<SRC, false>(K, node, R, J, T, off, wv);
            return;
        }
    }
    ccl_tile_runs<SRC, true>(K, node, R, J, T, off, wv);
}

// Unions across tile edges: the tile's first wave takes the pixels of its first column with their left
// neighbours (lane = row), the second its first row with the pixels above (lane = column).  A pixel
// skips a union whose two tile-local roots an adjacent pixel unites by the same kind of join, or that
// its own straight join makes: along an edge, consecutive pixels usually meet the same two components.
template <int MODE, int CONN>
__global__ __launch_bounds__(128) void ccl_seams(Px P, CclBufs B, int32_t* forest, int w, int h, int tiles_x) {
    const int t = blockIdx.x, tx = t % tiles_x, ty = t / tiles_x, lane = threadIdx.x & 63;
    using V = typename std::conditional<MODE == FG_FEQ, float, uint8_t>::type;
    const bool vertical = threadIdx.x < 64;  // wave-uniform
    if (vertical ? tx == 0 : ty == 0) return;
    const uint16_t* er = B.edge_roots;
    const int to = vertical ? t - 1 : t - tiles_x;  // the tile across the edge
    const uint16_t rm = er[((size_t)t * 4 + (vertical ? E_LEFT : E_TOP)) * CT + lane];
    const uint16_t ro = er[((size_t)to * 4 + (vertical ? E_RIGHT : E_BOTTOM)) * CT + lane];
    // this pixel, the one opposite, that one's neighbours along the edge: foreground, tile-local root,
    // value (equal-value modes)
    const bool fm = rm != kNoRoot, fo = ro != kNoRoot;
    const int gm = place_index(tx, ty, rm, w), go = vertical ? place_index(tx - 1, ty, ro, w) : place_index(tx, ty - 1, ro, w);
    V vm = 0, vo = 0;
    if (MODE != FG_NEQ) {
        if (vertical) {
            const V* e = static_cast<const V*>(B.edge);
            vm = e[(size_t)t * 2 * CT + lane];
            vo = e[(size_t)to * 2 * CT + CT + lane];
        } else {
            const size_t xc = (size_t)min(tx * CT + lane, w - 1);
            const V* img;
            if constexpr (MODE == FG_FEQ) img = P.fv;
            else img = P.img;
            vm = img[(size_t)ty * CT * w + xc];
            vo = img[((size_t)ty * CT - 1) * w + xc];
        }
    }
    const bool join = fm && fo && (MODE == FG_NEQ || vm == vo);
    // neighbours along the edge
    const bool pjoin = from_left(0, join ? 1 : 0) != 0, njoin = from_right(0, join ? 1 : 0) != 0;
    const int pgm = from_left(-1, gm), ngm = from_right(-1, gm);
    const int pgo = from_left(-1, go), ngo = from_right(-1, go);
    if (join && !(pjoin && pgm == gm && pgo == go)) gunite(forest, gm, go);
    if (CONN == 4) return;
    bool fol = from_left(0, fo ? 1 : 0) != 0, for_ = from_right(0, fo ? 1 : 0) != 0;
    int gol = pgo, gor = ngo;
    V vol = 0, vor = 0;
    if (MODE == FG_FEQ) {
        vol = (V)from_left(0.0f, (float)vo);
        vor = (V)from_right(0.0f, (float)vo);
    } else if (MODE == FG_EQ) {
        vol = (V)from_left(0, (int)vo);
        vor = (V)from_right(0, (int)vo);
    }
    // the two pixels beyond the ends of the row above belong to the tiles beside it (a column's ends
    // have no such pixel here: the first row's wave takes those joins)
    const int side = lane == 0 ? -1 : 1, tn = t - tiles_x + side;
    if (!vertical && ((lane == 0 && tx > 0) || (lane == 63 && tx + 1 < tiles_x))) {
        const uint16_t r = er[((size_t)tn * 4 + E_BOTTOM) * CT + (side < 0 ? CT - 1 : 0)];
        const bool f = r != kNoRoot;
        const int g = place_index(tx + side, ty - 1, r, w);
        V v = 0;
        if (MODE != FG_NEQ) {
            const V* img;
            if constexpr (MODE == FG_FEQ) img = P.fv;
            else img = P.img;
            v = img[((size_t)ty * CT - 1) * w + (size_t)(tx * CT + (side < 0 ? -1 : CT))];
        }
        if (side < 0) { fol = f; gol = g; vol = v; }
        else { for_ = f; gor = g; vor = v; }
    }
    const bool jl = fm && fol && (MODE == FG_NEQ || vm == vol), jr = fm && for_ && (MODE == FG_NEQ || vm == vor);
    if (jl && !(join && gol == go) && !(pjoin && pgm == gm)) gunite(forest, gm, gol);
    if (jr && !(join && gor == go) && !(njoin && ngm == gm)) gunite(forest, gm, gor);
}

// the final root of a tile-local root.  A read-only walk: a path-jumping find here could re-point an
// entry whose final root another thread has already stored to an intermediate ancestor.  Roots are
// final once the seams are done and every value an entry takes is an ancestor, so cached loads are safe.
__device__ __forceinline__ int final_root(const int32_t* forest, int g) {
    int r = g, nx = ld_wg(&forest[g]);
    while (nx != r) {
        r = nx;
        nx = ld_wg(&forest[r]);
    }
    return r;
}

// A lane's four pixels of a tile's 256 edge pixels (16 lanes a side) and their roots' places; those that are
// open, and not the pixel's before it, are visited.
__device__ __forceinline__ uint2 edge_places(const CclBufs& B, int t) {
    return *reinterpret_cast<const uint2*>(B.edge_roots + ((size_t)t * 4 * CT + 4 * (threadIdx.x & 63)));
}
template <class Visit>
__device__ __forceinline__ void open_edge_roots(uint2 q, int tx, int ty, int tiles_x, int tiles_y, Visit visit) {
    const int lane = threadIdx.x & 63;
    const bool open = side_open(lane >> 4, tx, ty, tiles_x, tiles_y);
    const uint32_t p[4] = {q.x & 0xFFFFu, q.x >> 16, q.y & 0xFFFFu, q.y >> 16};
#pragma unroll
    for (int j = 0; j < 4; ++j) visit((int)p[j], open && p[j] != kNoRoot && (j == 0 || p[j] != p[j ? j - 1 : 0]));
}

// Every open root that is not final hands its count or flag to the final root and points at it.
__global__ __launch_bounds__(256) void ccl_roots(CclBufs B, int32_t* forest, int w, int tiles_x, int ntiles, int32_t* area,
                                                 uint8_t* flag) {
    __shared__ uint32_t seen_s[4][CT * CT / 32];  // by place
    const int t = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (t >= ntiles) return;
    uint32_t* const seen = seen_s[threadIdx.x >> 6];
    const uint2 places = edge_places(B, t);
    seen[lane] = 0;
    seen[64 + lane] = 0;
    wave_order();
    const int tx = t % tiles_x, ty = t / tiles_x;
    open_edge_roots(places, tx, ty, tiles_x, ntiles / tiles_x, [&](int p, bool take) {
        if (!take || (atomicOr(&seen[p >> 5], 1u << (p & 31)) >> (p & 31) & 1u)) return;
        const int g = place_index(tx, ty, p, w), r = final_root(forest, g);
        if (r == g) return;
        forest[g] = r;
        if (area) atomicAdd(&area[r], area[g]);
        if (flag && flag[g]) flag[r] = 1;
    });
}

// What a selection writes per pixel, sel = the pixel's component is selected (by its area in [lo, hi),
// or by its flag):
//   OUT_MASK     255 where sel                           (bwareaopen2)
//   OUT_UNSEL    255 where foreground and not sel         (plateaus without a greater neighbour)
//   OUT_HOLES    0 where sel, else 255                    (imfillHoles: passable and reached from the border)
//   OUT_KEEP     a where sel, else 0                      (bwselect)
//   OUT_BINREC   a where nonzero, else 255 where sel      (imreconstructBinary: a = marker)
//   OUT_FILL     a | (255 - a at the seeds b, else 255 where sel)   (imfill)
enum { OUT_MASK = 0, OUT_UNSEL, OUT_HOLES, OUT_KEEP, OUT_BINREC, OUT_FILL };

template <int OUT>
__device__ __forceinline__ uint32_t select_word(uint32_t sel, uint32_t a, uint32_t b) {
    if (OUT == OUT_HOLES) return ~sel;
    if (OUT == OUT_KEEP) return a & sel;
    if (OUT == OUT_BINREC) return a | (sel & ~((nonzero_bytes(a) >> 7) * 255u));
    if (OUT == OUT_FILL) {
        const uint32_t sd = (nonzero_bytes(b) >> 7) * 255u;
        return a | (sd & ~a) | (sel & ~sd);
    }
    return sel;
}

// One tile per wave: the selected open roots become bits in LDS (by run number), the selected runs bits of the
// rows' words (lane = row; the codes staged in LDS, cap of them a wave), the words bytes (a lane writes four
// 16-byte pieces, a row is four lanes).
// *count (optional) = number of selected components, counted at their final roots; one atomic per
// workgroup, and the grid is at most kSelectBlocks (atomics on one address cost about 10 ns each: one
// per tile of a 4096^2 image took 40 us).
constexpr int kSelectBlocks = 512;
template <int OUT>
__global__ __launch_bounds__(256) void ccl_select(CclBufs B, const int32_t* __restrict__ forest, int w, int h, int tiles_x,
                                                  int ntiles, const int32_t* __restrict__ area, int lo, int hi,
                                                  const uint8_t* __restrict__ flag, const uint8_t* a, const uint8_t* b,
                                                  uint8_t* out, int* count) {
    __shared__ uint32_t keep_s[4][CT * CT / 32];
    __shared__ uint64_t words_s[4][CT];
    extern __shared__ uint4 codes_s[];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    uint4* const codes8 = codes_s + (size_t)wv * (B.cap / 8);
    const uint16_t* const codes = reinterpret_cast<const uint16_t*>(codes8);
    uint32_t* const keep = keep_s[wv];
    uint64_t* const words = words_s[wv];
    int n = 0;
    for (int t = blockIdx.x * 4 + wv; t < ntiles; t += 4 * gridDim.x) {
        const int tx = t % tiles_x, ty = t / tiles_x;
        const RowWords R = B.rows[(size_t)t * CT + lane];
        const int off = B.off[(size_t)t * CT + lane];
        const uint2 places = edge_places(B, t);
        const uint4* roots = reinterpret_cast<const uint4*>(B.roots + (size_t)t * B.cap);
        codes8[lane] = roots[lane];  // a usual tile's codes, without waiting for its run count
        const int runs = __builtin_amdgcn_readlane(off + popc64(R.S), 63);
        for (int k = 64 + lane; 8 * k < runs; k += 64) codes8[k] = roots[k];
        keep[lane] = 0;
        keep[64 + lane] = 0;
        wave_order();
        open_edge_roots(places, tx, ty, tiles_x, ntiles / tiles_x, [&](int p, bool take) {
            // the run that starts there, from its row's words (every lane takes part)
            const int row = take ? p >> 6 : 0;
            const uint64_t S = (uint64_t)(uint32_t)__shfl((int)(uint32_t)R.S, row) |
                               (uint64_t)(uint32_t)__shfl((int)(uint32_t)(R.S >> 32), row) << 32;
            const int k = __shfl(off, row) + run_index(S, p & 63);
            if (!take) return;
            const int g = place_index(tx, ty, p, w), r = forest[g];  // final: ccl_roots has run
            bool s;
            if (OUT == OUT_MASK) {
                const int ar = area[r];
                s = ar >= lo && ar < hi;
            } else {
                s = flag[r] != 0;
            }
            if (!s) return;
            const bool first = !(atomicOr(&keep[k >> 5], 1u << (k & 31)) >> (k & 31) & 1u);
            if (OUT == OUT_MASK) n += (first && r == g) ? 1 : 0;
        });
        wave_order();
        uint64_t sel = 0;
        int k = off;
        for (uint64_t m = R.S; m; m &= m - 1, ++k) {
            const uint32_t c = codes[k], r = c & kRunRoot;
            const bool s = c & kClosed ? (c & kSelected) != 0 : ((keep[r >> 5] >> (r & 31)) & 1u) != 0;
            if (!s) continue;
            const int x = __ffsll((long long)m) - 1;
            sel |= run_bits(x, run_end(R.S, R.F, x));
            if (OUT == OUT_MASK) n += ((c & kClosed) && (int)r == k) ? 1 : 0;
        }
        words[lane] = OUT == OUT_UNSEL ? R.F & ~sel : sel;
        wave_order();
        const int x0 = tx * CT, y0 = ty * CT, cols = min(CT, w - x0), x = 16 * (lane & 3);
        const bool full = cols == CT;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int y = 16 * g + (lane >> 2);
            if (y0 + y >= h || x >= cols) continue;
            const size_t row = (size_t)(y0 + y) * w + x0;
            uint4 va = make_uint4(0, 0, 0, 0), vb = va;
            if (OUT >= OUT_KEEP) va = load16(a + row, x, cols, full);
            if (OUT == OUT_FILL) vb = load16(b + row, x, cols, full);
            const uint32_t bits = (uint32_t)(words[y] >> x);
            const uint4 v = make_uint4(select_word<OUT>(spread_bits(bits & 15u), va.x, vb.x),
                                       select_word<OUT>(spread_bits(bits >> 4 & 15u), va.y, vb.y),
                                       select_word<OUT>(spread_bits(bits >> 8 & 15u), va.z, vb.z),
                                       select_word<OUT>(spread_bits(bits >> 12 & 15u), va.w, vb.w));
            if (full) {
                __builtin_memcpy(out + row + x, &v, 16);
            } else {
                const uint32_t wd[4] = {v.x, v.y, v.z, v.w};
                for (int j = 0; j < min(16, cols - x); ++j) out[row + x + j] = (uint8_t)(wd[j >> 2] >> (8 * (j & 3)));
            }
        }
        wave_order();
    }
    if (count) block_count_add(n, count);  // `count` is the same for every thread
}

// Labels of a tile by run, in LDS: every run's own first pixel (a closed root's label), the open roots' final
// roots (thread = edge pixel), then each run's root's label; then lane = column and a row a step.  forest
// may be the label image itself: an open root's entry is overwritten with its final root, which any walk may
// meet instead of the entry it replaces, and no other entry is read.
__global__ __launch_bounds__(256) void ccl_label(CclBufs B, int32_t* forest, int32_t* L, int w, int h, int tiles_x,
                                                 int32_t bgval) {
    __shared__ int lab[CT * CT];  // by run number
    __shared__ RowWords words[CT];
    __shared__ int offs[CT];
    const int t = blockIdx.x, tx = t % tiles_x, ty = t / tiles_x, lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const RowWords R = B.rows[(size_t)t * CT + lane];
    const int off = B.off[(size_t)t * CT + lane];
    const int p = B.edge_roots[(size_t)t * 4 * CT + threadIdx.x];
    // eight codes at a time, all of a thread's before their use; a usual tile's without waiting for its run count
    const uint4* roots = reinterpret_cast<const uint4*>(B.roots + (size_t)t * B.cap);
    constexpr int kPer = CT * CT / (8 * 256);
    uint4 codes[kPer];
    if (threadIdx.x < kFewRuns / 8) codes[0] = roots[threadIdx.x];
    const int runs = __builtin_amdgcn_readlane(off + popc64(R.S), 63);
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        const int k = threadIdx.x + 256 * j;
        if (k >= kFewRuns / 8 && 8 * k < runs) codes[j] = roots[k];
    }
    if (wv == 0) {
        words[lane] = R;
        offs[lane] = off;
    }
    // the four waves take a row's runs in turn
    {
        int k = off;
        for (uint64_t m = R.S; m; m &= m - 1, ++k)
            if (((k - off) & 3) == wv) lab[k] = place_index(tx, ty, lane * CT + __ffsll((long long)m) - 1, w);
    }
    __syncthreads();
    if (side_open(wv, tx, ty, tiles_x, (int)gridDim.x / tiles_x) && p != kNoRoot && p != dpp_from_left(-1, p))
        lab[offs[p >> 6] + run_index(words[p >> 6].S, p & 63)] = final_root(forest, place_index(tx, ty, p, w));
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        if (8 * ((int)threadIdx.x + 256 * j) >= runs) break;
        const uint32_t c[4] = {codes[j].x, codes[j].y, codes[j].z, codes[j].w};
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int k = 8 * ((int)threadIdx.x + 256 * j) + i, r = (int)(c[i >> 1] >> (16 * (i & 1)) & kRunRoot);
            if (k < runs && r != k) lab[k] = lab[r];  // (roots' entries are only read)
        }
    }
    __syncthreads();
    const int x = tx * CT + lane;
    if (x >= w) return;
#pragma unroll 4
    for (int y = wv; y < CT; y += 4) {
        if (ty * CT + y >= h) break;
        const RowWords W = words[y];
        const bool fg = (W.F >> lane) & 1ull;
        const int v = lab[fg ? offs[y] + run_index(W.S, lane) : 0];
        L[(size_t)(ty * CT + y) * w + x] = fg ? v : bgval;
    }
}

struct CclGrid {
    int tiles_x, nt;
};
CclGrid ccl_grid(int w, int h) {
    const int tx = (int)cdiv(w, CT);
    return CclGrid{tx, tx * (int)cdiv(h, CT)};
}

// scratch of a labelling: run slots for the most runs that a tile of the image can hold (every second pixel of a
// row, or every pixel where equal values join; kFewRuns at least, which the consumers load).  A tile of a
// 64 x 64 image takes 5.8 KB or 10, of an image of one column 2.7.
CclBufs ccl_carve(Carver& c, int nt, int mode, int w, int h) {
    CclBufs B;
    const int cols = std::min(w, CT), most = std::min(h, CT) * (mode == FG_NEQ ? (cols + 1) / 2 : cols);
    B.cap = std::max(kFewRuns, (most + 7) / 8 * 8);
    B.rows = c.take<RowWords>((size_t)nt * CT);
    B.off = c.take<uint16_t>((size_t)nt * CT);
    B.roots = c.take<uint16_t>((size_t)nt * B.cap);
    B.edge_roots = c.take<uint16_t>((size_t)nt * 4 * CT);
    B.edge = mode == FG_NEQ ? nullptr : c.take<uint8_t>((size_t)nt * 2 * CT * (mode == FG_FEQ ? sizeof(float) : 1));
    return B;
}

// LDS of a ccl_select workgroup beside its fixed part: the codes of four tiles
size_t select_lds(const CclBufs& B) { return 4 * sizeof(uint16_t) * (size_t)B.cap; }

struct CclWork {  // a labelling in progress
    Scratch sc;
    CclBufs B;
    CclGrid g;
};

// Launches of at most kFewTiles tiles (two a CU, 1448 x 1448) give a tile four waves: there a tile of many runs lasts
// as long as its own loops over them.  Kernel time at 600 x 600, one wave a tile and four: 50 % noise 24.6 and
// 17.3 us, discs 7.4 and 7.7 (three of the four leave at once).  More tiles fill the chip by themselves, and the
// idle waves take room: hole filling of 4096 x 4096 discs 56 us a call with one wave, 62 with four.
constexpr int kFewTiles = 512;

// the tile and seam passes; flag / src: see ccl_tile
template <int MODE, int CONN, int SRC>
int ccl_forest_t(const Px& P, CclWork& W, int32_t* forest, int w, int h, int32_t* area, int lo, int hi, uint8_t* flag,
                 const uint8_t* src, int* zero, hipStream_t s) {
    W.g = ccl_grid(w, h);
    Carver m(nullptr);
    (void)ccl_carve(m, W.g.nt, MODE, w, h);
    NSC_CHECK(W.sc.alloc(m.size(), s));
    Carver c(W.sc.p);
    W.B = ccl_carve(c, W.g.nt, MODE, w, h);
    auto tiles = [&](auto waves) {
        constexpr int WAVES = decltype(waves)::value;
        hipLaunchKernelGGL((ccl_tile<MODE, CONN, SRC, WAVES>), dim3(W.g.nt), dim3(ccl_tile_threads(MODE, WAVES)), 0, s, P, W.B,
                           forest, w, h, W.g.tiles_x, area, lo, hi, flag, src, zero);
    };
    if (W.g.nt <= kFewTiles) tiles(std::integral_constant<int, 4>{});
    else tiles(std::integral_constant<int, 1>{});
    hipLaunchKernelGGL((ccl_seams<MODE, CONN>), dim3(W.g.nt), dim3(128), 0, s, P, W.B, forest, w, h, W.g.tiles_x);
    NSC_HIP(hipGetLastError());
    return NSC_OK;
}

template <int MODE>
int ccl_labels(const Px& P, int32_t* L, int w, int h, int conn, int32_t bgval, hipStream_t s) {
    CclWork W;
    if (conn == 8) NSC_CHECK((ccl_forest_t<MODE, 8, SRC_NONE>(P, W, L, w, h, nullptr, 0, 0, nullptr, nullptr, nullptr, s)));
    else NSC_CHECK((ccl_forest_t<MODE, 4, SRC_NONE>(P, W, L, w, h, nullptr, 0, 0, nullptr, nullptr, nullptr, s)));
    hipLaunchKernelGGL(ccl_label, dim3(W.g.nt), dim3(256), 0, s, W.B, L, L, w, h, W.g.tiles_x, bgval);
    NSC_HIP(hipGetLastError());
    return NSC_OK;
}

// component selection by a flag: sources = nonzero pixels of src, or the image border when src is null
template <int MODE, int OUT>
int ccl_select_flag(const Px& P, const uint8_t* src, const uint8_t* a, const uint8_t* b, uint8_t* out, int w, int h, int conn,
                    int32_t* forest, uint8_t* flag, hipStream_t s) {
    CclWork W;
    if (src) {
        if (conn == 8) NSC_CHECK((ccl_forest_t<MODE, 8, SRC_BYTES>(P, W, forest, w, h, nullptr, 0, 0, flag, src, nullptr, s)));
        else NSC_CHECK((ccl_forest_t<MODE, 4, SRC_BYTES>(P, W, forest, w, h, nullptr, 0, 0, flag, src, nullptr, s)));
    } else {
        if (conn == 8) NSC_CHECK((ccl_forest_t<MODE, 8, SRC_BORDER>(P, W, forest, w, h, nullptr, 0, 0, flag, src, nullptr, s)));
        else NSC_CHECK((ccl_forest_t<MODE, 4, SRC_BORDER>(P, W, forest, w, h, nullptr, 0, 0, flag, src, nullptr, s)));
    }
    hipLaunchKernelGGL(ccl_roots, dim3(cdiv(W.g.nt, 4)), dim3(256), 0, s, W.B, forest, w, W.g.tiles_x, W.g.nt,
                       (int32_t*)nullptr, flag);
    hipLaunchKernelGGL((ccl_select<OUT>), dim3(cdiv(W.g.nt, 4)), dim3(256), select_lds(W.B), s, W.B, forest, w, h, W.g.tiles_x, W.g.nt,
                       (const int32_t*)nullptr, 0, 0, flag, a, b, out, (int*)nullptr);
    NSC_HIP(hipGetLastError());
    return NSC_OK;
}

template <int MODE>
int ccl_select_area(const Px& P, uint8_t* out, int w, int h, int lo, int hi, int conn, int* dcount, int32_t* forest,
                    int32_t* area, hipStream_t s) {
    CclWork W;
    if (conn == 8) NSC_CHECK((ccl_forest_t<MODE, 8, SRC_NONE>(P, W, forest, w, h, area, lo, hi, nullptr, nullptr, dcount, s)));
    else NSC_CHECK((ccl_forest_t<MODE, 4, SRC_NONE>(P, W, forest, w, h, area, lo, hi, nullptr, nullptr, dcount, s)));
    hipLaunchKernelGGL(ccl_roots, dim3(cdiv(W.g.nt, 4)), dim3(256), 0, s, W.B, forest, w, W.g.tiles_x, W.g.nt, area,
                       (uint8_t*)nullptr);
    const unsigned nb = dcount ? std::min<unsigned>(cdiv(W.g.nt, 4), kSelectBlocks) : cdiv(W.g.nt, 4);
    hipLaunchKernelGGL((ccl_select<OUT_MASK>), dim3(nb), dim3(256), select_lds(W.B), s, W.B, forest, w, h, W.g.tiles_x, W.g.nt, area, lo, hi,
                       (const uint8_t*)nullptr, (const uint8_t*)nullptr, (const uint8_t*)nullptr, out, dcount);
    NSC_HIP(hipGetLastError());
    return NSC_OK;
}

// The per-pixel label consumers below take four pixels per thread and iteration, i, i + S, i + 2S,
// i + 3S (S = threads in the grid): the four labels, then the four per-root gathers, are issued
// together instead of one dependent label -> gather round trip per pixel.
#define NSC_FOR4(n)                                                                                  \
    for (size_t i0 = (size_t)blockIdx.x * blockDim.x + threadIdx.x, S = (size_t)gridDim.x * blockDim.x; \
         i0 < (n); i0 += 4 * S)

// ---- canonical relabel: rank of each root in raster order ----
// A workgroup of 1024 threads covers SCAN_B = 4096 consecutive pixels, four per thread (contiguous,
// so a thread's roots are in raster order after those of the threads before it); few workgroups
// keep the scan of their counts short.
constexpr int SCAN_B = 4096;

// exclusive prefix sum of v over the workgroup (at most 16 waves); *total = the sum of all v
__device__ __forceinline__ int block_scan_excl(int v, int* total) {
    __shared__ int wsum[16];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
    int x = v;  // inclusive scan within the wave
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int y = __shfl_up(x, off);
        if (lane >= off) x += y;
    }
    __syncthreads();  // wsum may still be read by a previous call
    if (lane == 63) wsum[wv] = x;
    __syncthreads();
    int before = 0, tot = 0;
    for (int k = 0; k < nw; ++k) {
        const int t = wsum[k];
        if (k < wv) before += t;
        tot += t;
    }
    if (total) *total = tot;
    return before + x - v;
}

__global__ __launch_bounds__(1024) void k_root_block_count(const int32_t* __restrict__ L, size_t n, int32_t* __restrict__ bsum) {
    const size_t i0 = (size_t)blockIdx.x * SCAN_B + 4 * threadIdx.x;
    int c = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) c += (i0 + j < n && L[i0 + j] == (int32_t)(i0 + j)) ? 1 : 0;
    const int t = block_sum(c);
    if (threadIdx.x == 0) bsum[blockIdx.x] = t;
}
// exclusive scan of nb block sums in place (one workgroup of 1024 threads, a contiguous chunk each)
__global__ __launch_bounds__(1024) void k_scan_small(int32_t* bsum, int nb, int* total) {
    const int per = (nb + 1023) / 1024, start = threadIdx.x * per;
    const int end = min(start + per, nb);
    int acc = 0;
    for (int k = start; k < end; k += 4) {  // four loads in flight
        int v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = k + j < end ? bsum[k + j] : 0;
        acc += v[0] + v[1] + v[2] + v[3];
    }
    int tot = 0;
    int run = block_scan_excl(acc, &tot);
    if (threadIdx.x == 0 && total) *total = tot;
    for (int k = start; k < end; k += 4) {
        int v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = k + j < end ? bsum[k + j] : 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (k + j < end) bsum[k + j] = run;
            run += v[j];
        }
    }
}
// rank[i] (stored in place of area scratch) for roots: 1 + number of roots before i
__global__ __launch_bounds__(1024) void k_root_rank(const int32_t* __restrict__ L, size_t n, const int32_t* __restrict__ boff,
                                                   int32_t* __restrict__ rank) {
    const size_t i0 = (size_t)blockIdx.x * SCAN_B + 4 * threadIdx.x;
    bool root[4];
    int c = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        root[j] = i0 + j < n && L[i0 + j] == (int32_t)(i0 + j);
        c += root[j] ? 1 : 0;
    }
    int k = boff[blockIdx.x] + block_scan_excl(c, nullptr);
#pragma unroll
    for (int j = 0; j < 4; ++j)
        if (root[j]) rank[i0 + j] = ++k;
}
__global__ void k_apply_rank(int32_t* L, const int32_t* __restrict__ rank, size_t n, int32_t bgval) {
    NSC_FOR4(n) {
        int r[4], v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) r[j] = i0 + j * S < n ? L[i0 + j * S] : -1;
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = (r[j] == bgval || r[j] < 0) ? 0 : rank[r[j]];
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (i0 + j * S < n) L[i0 + j * S] = v[j];
    }
}

__global__ void k_bbox_init(int32_t* out5, int32_t* area, int n) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    out5[k] = k + 1;
    out5[n + k] = INT_MAX;
    out5[2 * n + k] = -1;
    out5[3 * n + k] = INT_MAX;
    out5[4 * n + k] = -1;
    if (area) area[k] = 0;
}
// A wave takes 64 consecutive pixels (coalesced loads of the window and of the rows above and
// below it) and visits each run of equal labels in its window once; a row start also starts a
// run.  A run issues an extent atomic only where no pixel of its component is known to beat it:
//   y0: no pixel of the run has its label directly above;      y1: likewise below;
//   x0: the pixels above its first pixel, and left of it in the rows y-1, y and y+1, lack its label;
//   x1: likewise above its last pixel, and right of it in the rows y-1, y and y+1.
// Every skip names a pixel of the component at a smaller row (y0), larger row (y1), smaller
// column or the same column one row up (x0), larger column or the same column one row up (x1).
// The extreme row's runs have no such pixel, and the topmost pixel of the extreme column has none
// either, so each extreme is still issued; the skips drop the ~4 atomics per row of a component to
// the few rows that hold an extreme.  Area stays one atomic per run.  Labels outside 1..n are ignored.
__global__ void k_bbox(const int32_t* __restrict__ L, int w, int h, int n, int32_t* out5, int32_t* area) {
    const size_t total = (size_t)w * h;
    const int lane = threadIdx.x & 63;
    const size_t wave = ((size_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const size_t nwave = ((size_t)gridDim.x * blockDim.x) >> 6;
    constexpr int NONE = INT_MIN;  // never a label in 1..n
    for (size_t base = wave * 64; base < total; base += nwave * 64) {
        const size_t i = base + lane;
        const bool valid = i < total;
        // position: the window's first pixel once per wave, then at most a few row wraps
        int y = (int)(base / w), x = (int)(base - (size_t)y * w) + lane;
        while (x >= w) {
            x -= w;
            ++y;
        }
        // the pixel and its neighbours above and below, and for the window's first / last lane the
        // same three one column further out (same row only; other lanes re-read their own): clamped
        // (always valid) addresses, all six loads issued together, out-of-image values replaced
        // afterwards
        const bool has_l = x > 0, has_r = x < w - 1;
        const bool has_u = valid && y > 0, has_d = valid && y < h - 1;
        const size_t ic = valid ? i : total - 1;
        const bool edge = valid && ((lane == 0 && has_l) || (lane == 63 && has_r));
        const size_t ie = edge ? (lane == 0 ? ic - 1 : ic + 1) : ic;
        const int r0 = L[ic], u0 = L[has_u ? ic - w : ic], d0 = L[has_d ? ic + w : ic];
        const int e0 = L[ie], eu0 = L[has_u ? ie - w : ie], ed0 = L[has_d ? ie + w : ie];
        const int r = valid ? r0 : -1;
        const int ru = has_u ? u0 : NONE, rd = has_d ? d0 : NONE;
        const int ev = edge ? e0 : NONE, evu = (edge && has_u) ? eu0 : NONE, evd = (edge && has_d) ? ed0 : NONE;
        // left and right neighbours: from the adjacent lanes, or the edge lanes' own loads
        int lr = __shfl_up(r, 1), lu = __shfl_up(ru, 1), ld = __shfl_up(rd, 1);
        int rr = __shfl_down(r, 1), ruu = __shfl_down(ru, 1), rdd = __shfl_down(rd, 1);
        if (lane == 0) {
            lr = ev; lu = evu; ld = evd;
        }
        if (lane == 63) {
            rr = ev; ruu = evu; rdd = evd;
        }
        const bool up = valid && ru == r, down = valid && rd == r;
        const bool x1_beaten = valid && (up || (has_r && (rr == r || ruu == r || rdd == r)));
        const unsigned long long m_up = __ballot(up), m_down = __ballot(down), m_x1 = __ballot(x1_beaten);
        const bool head = (lane == 0 || lr != r || x == 0) && valid;
        const unsigned long long heads = __ballot(head);
        if (head && r >= 1 && r <= n) {
            const unsigned long long later = lane == 63 ? 0ull : (heads >> (lane + 1));
            int end = later ? lane + __ffsll((long long)later) : 64;  // first lane after the run
            end = (int)std::min<size_t>((size_t)end, total - base);
            const int k = r - 1, len = end - lane;
            const unsigned long long run = (len == 64 ? ~0ull : ((1ull << len) - 1)) << lane;
            const bool x0_beaten = up || (has_l && (lr == r || lu == r || ld == r));
            if (!x0_beaten) atomicMin(&out5[n + k], x);
            if (!((m_x1 >> (end - 1)) & 1ull)) atomicMax(&out5[2 * n + k], x + len - 1);
            if (!(m_up & run)) atomicMin(&out5[3 * n + k], y);
            if (!(m_down & run)) atomicMax(&out5[4 * n + k], y);
            if (area) atomicAdd(&area[k], len);
        }
    }
}

inline dim3 grid1(size_t n) { return dim3(std::min<unsigned>(cdiv(n, 256), 8192u)); }

// ---- ConnComponents::boundingBox, literally (ConnComponents.cpp:241-284) -----------------------
// The reference scans labels in raster order, skips bgval, stops at the first -1 or 0 label, and
// lists the labels it met in first-seen order.  Here: the stop index, each label's first position
// (atomicMin), a rank of the first positions (the relabel kernels), then the box kernel on the
// ranks.  Labels met before the stop must lie in 1 .. w*h-1 (as ConnComponents::label makes them).
__global__ void k_bb_stop(const int32_t* __restrict__ L, int n, int32_t bgval, int* __restrict__ stop) {
    int best = INT_MAX;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const int32_t v = L[i];
        if (v != bgval && (v == -1 || v == 0)) {  // a thread's first hit in its stride is its smallest
            best = i;
            break;
        }
    }
    for (int off = 32; off > 0; off >>= 1) best = min(best, __shfl_down(best, off));
    __shared__ int part[16];
    const int wv = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
    if ((threadIdx.x & 63) == 0) part[wv] = best;
    __syncthreads();
    if (threadIdx.x == 0) {
        int b = INT_MAX;
        for (int k = 0; k < nw; ++k) b = min(b, part[k]);
        if (b != INT_MAX) atomicMin(stop, b);
    }
}
__global__ void k_bb_first(const int32_t* __restrict__ L, int n, int32_t bgval, const int* __restrict__ stop,
                           int* __restrict__ firstpos, int* __restrict__ bad) {
    const int i0 = min(*stop, n);
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < i0; i += gridDim.x * blockDim.x) {
        const int32_t v = L[i];
        if (v == bgval) continue;
        if (v < 1 || v >= n) atomicOr(bad, 1);
        else atomicMin(&firstpos[v], i);
    }
}
// R[i] = i at first positions (the roots the rank kernels count), -1 elsewhere
__global__ void k_bb_roots(const int32_t* __restrict__ L, int n, int32_t bgval, const int* __restrict__ stop,
                           const int* __restrict__ firstpos, int32_t* __restrict__ R) {
    const int i0 = *stop;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const int32_t v = L[i];
        const bool ok = i < i0 && v != bgval && v >= 1 && v < n;
        const int f = ok ? firstpos[v] : -1;
        R[i] = (ok && f == i) ? i : -1;
    }
}
// canon[i] = rank of the first position of L[i] (1..count) over the scanned pixels, -1 elsewhere
__global__ void k_bb_canon(const int32_t* __restrict__ L, int n, int32_t bgval, const int* __restrict__ stop,
                           const int* __restrict__ firstpos, const int32_t* __restrict__ rank, int32_t* __restrict__ canon) {
    const int i0 = *stop;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const int32_t v = L[i];
        const bool ok = i < i0 && v != bgval && v >= 1 && v < n;
        canon[i] = ok ? rank[firstpos[v]] : -1;
    }
}
// label column: the box of rank k holds the label first seen at the k-th first position
// (rk: the rank at first positions, 0 elsewhere)
__global__ void k_bb_labels(const int32_t* __restrict__ L, int n, const int32_t* __restrict__ rk, int32_t* __restrict__ out5) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const int32_t k = rk[i];
        if (k > 0) out5[k - 1] = L[i];
    }
}
__global__ void k_fill_i32(int32_t* p, int32_t v, size_t n) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = v;
}

}  // namespace

// ------------------------------------------------------------------------------------------
// binary: every nonzero pixel has the same value, so equal-value joins are joins of foreground
int ccl_u8(const uint8_t* img, int32_t* labels, int w, int h, int conn, int32_t bgval, bool binary, hipStream_t s) {
    const Px P{img, nullptr, 0};
    return binary ? ccl_labels<FG_NEQ>(P, labels, w, h, conn, bgval, s) : ccl_labels<FG_EQ>(P, labels, w, h, conn, bgval, s);
}

int ccl_neq(const uint8_t* img, uint8_t key, int32_t* labels, int w, int h, int conn, hipStream_t s) {
    return ccl_labels<FG_NEQ>(Px{img, nullptr, key}, labels, w, h, conn, -1, s);
}

// 255 where the connected set of equal `vals` among the pixels with fg != 0 holds no pixel with
// src != 0, else 0
int ccl_plateaus_without(const uint8_t* fg, const float* vals, const uint8_t* src, uint8_t* out, int w, int h, int conn,
                         int32_t* forest, uint8_t* flag, hipStream_t s) {
    return ccl_select_flag<FG_FEQ, OUT_UNSEL>(Px{fg, vals, 0}, src, nullptr, nullptr, out, w, h, conn, forest, flag, s);
}

int bwareaopen_impl(const uint8_t* img, uint8_t* out, int w, int h, int lo, int hi, int conn, int* dcount, bool binary,
                    int32_t* labels, int32_t* area, hipStream_t s) {
    const Px P{img, nullptr, 0};
    return binary ? ccl_select_area<FG_NEQ>(P, out, w, h, lo, hi, conn, dcount, labels, area, s)
                  : ccl_select_area<FG_EQ>(P, out, w, h, lo, hi, conn, dcount, labels, area, s);
}

int fill_holes_impl(const uint8_t* img, uint8_t* out, int w, int h, int conn, int32_t* labels, uint8_t* flag,
                    hipStream_t s) {
    return ccl_select_flag<FG_NEQ, OUT_HOLES>(Px{img, nullptr, 255}, nullptr, nullptr, nullptr, out, w, h, conn, labels, flag, s);
}

int bwselect_impl(const uint8_t* bw, const uint8_t* seeds, uint8_t* out, int w, int h, int conn, int32_t* labels,
                  uint8_t* flag, hipStream_t s) {
    return ccl_select_flag<FG_NEQ, OUT_KEEP>(Px{bw, nullptr, 0}, seeds, bw, nullptr, out, w, h, conn, labels, flag, s);
}

int relabel_impl(int32_t* labels, int w, int h, int32_t bgval, int* dcount, int32_t* rank, hipStream_t s) {
    const size_t n = (size_t)w * h;
    const int nb = (int)cdiv(n, SCAN_B);
    Scratch sc;
    NSC_CHECK(sc.alloc(sizeof(int32_t) * (nb + 1), s));
    int32_t* bsum = sc.as<int32_t>();
    hipLaunchKernelGGL(k_root_block_count, dim3(nb), dim3(SCAN_B / 4), 0, s, labels, n, bsum);
    hipLaunchKernelGGL(k_scan_small, dim3(1), dim3(1024), 0, s, bsum, nb, dcount);
    hipLaunchKernelGGL(k_root_rank, dim3(nb), dim3(SCAN_B / 4), 0, s, labels, n, bsum, rank);
    hipLaunchKernelGGL(k_apply_rank, grid1(n), dim3(256), 0, s, labels, rank, n, bgval);
    NSC_HIP(hipGetLastError());
    return NSC_OK;
}

// the number of components of a labelling (its roots: label == own index), without relabelling
int root_count_impl(const int32_t* labels, int w, int h, int* dcount, hipStream_t s) {
    const size_t n = (size_t)w * h;
    const int nb = (int)cdiv(n, SCAN_B);
    Scratch sc;
    NSC_CHECK(sc.alloc(sizeof(int32_t) * (nb + 1), s));
    int32_t* bsum = sc.as<int32_t>();
    hipLaunchKernelGGL(k_root_block_count, dim3(nb), dim3(SCAN_B / 4), 0, s, labels, n, bsum);
    hipLaunchKernelGGL(k_scan_small, dim3(1), dim3(1024), 0, s, bsum, nb, dcount);
    NSC_HIP(hipGetLastError());
    return NSC_OK;
}

int bbox_impl(const int32_t* canon, int w, int h, int n, int32_t* out5, int32_t* area, hipStream_t s);

// ConnComponents::boundingBox(w, h, labels, bgval, compcount) with the reference's result block
// (5 x compcount, column stride compcount) in out5 when compcount <= cap.  Scratch: firstpos, R,
// rank (w*h ints each) and cnt (4 ints).  Synchronises the stream (compcount is a host value).
int bbox_literal_impl(const int32_t* L, int w, int h, int32_t bgval, int32_t* out5, int cap, int* compcount,
                      int32_t* firstpos, int32_t* R, int32_t* rank, int* cnt, hipStream_t s) {
    const int n = w * h;
    hipLaunchKernelGGL(k_fill_i32, grid1(n), dim3(256), 0, s, firstpos, INT_MAX, (size_t)n);
    hipLaunchKernelGGL(k_fill_i32, dim3(1), dim3(64), 0, s, cnt, 0, (size_t)4);
    hipLaunchKernelGGL(k_fill_i32, dim3(1), dim3(64), 0, s, cnt, n, (size_t)1);  // stop = n: no stop
    hipLaunchKernelGGL(k_bb_stop, grid1(n), dim3(256), 0, s, L, n, bgval, &cnt[0]);
    hipLaunchKernelGGL(k_bb_first, grid1(n), dim3(256), 0, s, L, n, bgval, &cnt[0], firstpos, &cnt[2]);
    hipLaunchKernelGGL(k_bb_roots, grid1(n), dim3(256), 0, s, L, n, bgval, &cnt[0], firstpos, R);
    // ranks of the first positions (relabel's root rank: 1 + first positions before it)
    NSC_CHECK(relabel_impl(R, w, h, -1, &cnt[1], rank, s));
    int hc[4] = {0, 0, 0, 0};
    NSC_HIP(hipMemcpyAsync(hc, cnt, sizeof(hc), hipMemcpyDeviceToHost, s));
    NSC_HIP(stream_sync(s));
    if (hc[2]) {
        set_error("boundingBox: a label before the first background pixel lies outside 1..w*h-1");
        return NSC_ERR_ARG;
    }
    *compcount = hc[1];
    if (hc[1] == 0 || !out5 || hc[1] > cap) return NSC_OK;
    // R now holds the rank at each first position (0 elsewhere); rank[] becomes the rank image
    hipLaunchKernelGGL(k_bb_canon, grid1(n), dim3(256), 0, s, L, n, bgval, &cnt[0], firstpos, R, rank);
    NSC_CHECK(bbox_impl(rank, w, h, hc[1], out5, nullptr, s));
    hipLaunchKernelGGL(k_bb_labels, grid1(n), dim3(256), 0, s, L, n, R, out5);
    NSC_HIP(hipGetLastError());
    return NSC_OK;
}

int bbox_impl(const int32_t* canon, int w, int h, int n, int32_t* out5, int32_t* area, hipStream_t s) {
    if (n <= 0) return NSC_OK;
    hipLaunchKernelGGL(k_bbox_init, dim3(cdiv(n, 256)), dim3(256), 0, s, out5, area, n);
    hipLaunchKernelGGL(k_bbox, grid1((size_t)w * h), dim3(256), 0, s, canon, w, h, n, out5, area);
    NSC_HIP(hipGetLastError());
    return NSC_OK;
}

}  // namespace nsc

using namespace nsc;

extern "C" {

int nsc_cc_label_u8(const uint8_t* img, int32_t* labels, int w, int h, int32_t bgval, int conn, void* stream) {
    NSC_ARG(img && labels && w > 0 && h > 0 && valid_conn(conn), "cc_label_u8");
    NSC_LABEL_SIZE(w, h);
    NSC_CHECK(ensure_init());
    return ccl_u8(img, labels, w, h, conn, bgval, false, as_stream(stream));
}

int nsc_bwlabel2_u8(const uint8_t* img, int32_t* labels, int w, int h, int conn, void* stream) {
    return nsc_cc_label_u8(img, labels, w, h, -1, conn, stream);
}

int nsc_cc_relabel(int32_t* labels, int w, int h, int32_t bgval, int* count, void* stream) {
    NSC_ARG(labels && w > 0 && h > 0, "cc_relabel");
    NSC_LABEL_SIZE(w, h);
    NSC_CHECK(ensure_init());
    hipStream_t s = as_stream(stream);
    Scratch sc;
    NSC_CHECK(sc.alloc(sizeof(int32_t) * ((size_t)w * h + 1), s));
    int32_t* rank = sc.as<int32_t>();
    int* dcount = reinterpret_cast<int*>(rank + (size_t)w * h);
    NSC_CHECK(relabel_impl(labels, w, h, bgval, dcount, rank, s));
    if (count) {
        NSC_HIP(hipMemcpyAsync(count, dcount, sizeof(int), hipMemcpyDeviceToHost, s));
        NSC_HIP(stream_sync(s));
    }
    return NSC_OK;
}

int nsc_bwareaopen2_u8(const uint8_t* img, uint8_t* out, int w, int h, int minSize, int maxSize, int conn, int* count,
                       void* stream) {
    NSC_ARG(img && out && w > 0 && h > 0 && valid_conn(conn), "bwareaopen2_u8");
    NSC_LABEL_SIZE(w, h);
    NSC_CHECK(ensure_init());
    hipStream_t s = as_stream(stream);
    const size_t n = (size_t)w * h;
    Scratch sc;
    NSC_CHECK(sc.alloc(sizeof(int32_t) * (2 * n + 1), s));
    int32_t* labels = sc.as<int32_t>();
    int32_t* area = labels + n;
    int* dcount = reinterpret_cast<int*>(area + n);
    NSC_CHECK(bwareaopen_impl(img, out, w, h, minSize, maxSize, conn, dcount, false, labels, area, s));
    if (count) {
        NSC_HIP(hipMemcpyAsync(count, dcount, sizeof(int), hipMemcpyDeviceToHost, s));
        NSC_HIP(stream_sync(s));
    }
    return NSC_OK;
}

int nsc_imreconstruct_binary_u8(const uint8_t* marker, const uint8_t* mask, uint8_t* out, int w, int h, int conn,
                                void* stream) {
    NSC_ARG(marker && mask && out && w > 0 && h > 0 && valid_conn(conn), "imreconstruct_binary_u8");
    NSC_LABEL_SIZE(w, h);
    NSC_CHECK(ensure_init());
    hipStream_t s = as_stream(stream);
    const size_t n = (size_t)w * h;
    Scratch sc;
    NSC_CHECK(sc.alloc(sizeof(int32_t) * n + n, s));
    int32_t* labels = sc.as<int32_t>();
    // a component is reached where the marker is nonzero on one of its (mask) pixels
    return ccl_select_flag<FG_NEQ, OUT_BINREC>(Px{mask, nullptr, 0}, marker, marker, nullptr, out, w, h, conn, labels,
                                               reinterpret_cast<uint8_t*>(labels + n), s);
}

int nsc_imfill_u8(const uint8_t* img, const uint8_t* seeds, uint8_t* out, int w, int h, int conn, void* stream) {
    NSC_ARG(img && seeds && out && w > 0 && h > 0 && valid_conn(conn), "imfill_u8");
    NSC_LABEL_SIZE(w, h);
    NSC_CHECK(ensure_init());
    hipStream_t s = as_stream(stream);
    const size_t n = (size_t)w * h;
    Scratch sc;
    NSC_CHECK(sc.alloc(sizeof(int32_t) * n + n, s));
    int32_t* labels = sc.as<int32_t>();
    return ccl_select_flag<FG_NEQ, OUT_FILL>(Px{img, nullptr, 255}, seeds, img, seeds, out, w, h, conn, labels,
                                             reinterpret_cast<uint8_t*>(labels + n), s);
}

int nsc_imfill_holes_u8(const uint8_t* img, uint8_t* out, int w, int h, int conn, void* stream) {
    NSC_ARG(img && out && w > 0 && h > 0 && valid_conn(conn), "imfill_holes_u8");
    NSC_LABEL_SIZE(w, h);
    NSC_CHECK(ensure_init());
    hipStream_t s = as_stream(stream);
    const size_t n = (size_t)w * h;
    Scratch sc;
    NSC_CHECK(sc.alloc(sizeof(int32_t) * n + n, s));
    int32_t* labels = sc.as<int32_t>();
    return fill_holes_impl(img, out, w, h, conn, labels, reinterpret_cast<uint8_t*>(labels + n), s);
}

int nsc_bwselect_u8(const uint8_t* bw, const uint8_t* seeds, uint8_t* out, int w, int h, int conn, void* stream) {
    NSC_ARG(bw && seeds && out && w > 0 && h > 0 && valid_conn(conn), "bwselect_u8");
    NSC_LABEL_SIZE(w, h);
    NSC_CHECK(ensure_init());
    hipStream_t s = as_stream(stream);
    const size_t n = (size_t)w * h;
    Scratch sc;
    NSC_CHECK(sc.alloc(sizeof(int32_t) * n + n, s));
    int32_t* labels = sc.as<int32_t>();
    return bwselect_impl(bw, seeds, out, w, h, conn, labels, reinterpret_cast<uint8_t*>(labels + n), s);
}

int nsc_cc_bounding_box(const int32_t* labels, int w, int h, int32_t bgval, int32_t* out5, int cap, int* compcount,
                        void* stream) {
    NSC_ARG(labels && compcount && w > 0 && h > 0 && cap >= 0, "cc_bounding_box");
    NSC_LABEL_SIZE(w, h);
    NSC_CHECK(ensure_init());
    hipStream_t s = as_stream(stream);
    const size_t n = (size_t)w * h;
    Scratch sc;
    NSC_CHECK(sc.alloc(sizeof(int32_t) * (3 * n + 4), s));
    int32_t* firstpos = sc.as<int32_t>();
    return bbox_literal_impl(labels, w, h, bgval, out5, cap, compcount, firstpos, firstpos + n, firstpos + 2 * n,
                             reinterpret_cast<int*>(firstpos + 3 * n), s);
}

int nsc_bounding_boxes(const int32_t* canon_labels, int w, int h, int n, int32_t* out5, int32_t* area, void* stream) {
    NSC_ARG(canon_labels && out5 && w > 0 && h > 0 && n >= 0, "bounding_boxes");
    NSC_LABEL_SIZE(w, h);
    NSC_CHECK(ensure_init());
    return bbox_impl(canon_labels, w, h, n, out5, area, as_stream(stream));
}

}  // extern "C"
