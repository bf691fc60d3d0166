// Exact parallel decomposition of cv::watershed's sequential flood (OpenCV 2.4.9
// imgproc/segmentation.cpp) for marker images whose unknown region contains a large black
// region B -- the shape watershed2 gets inside segmentNuclei: the background plateau holds label
// 0 (it contains pixel (0,0), MorphologicOperations.cpp:3737 labels a component by its smallest
// index) and is therefore "unknown", and the masked colour image is (0,0,0) there
// (HistologicalEntities.cpp:400-407).  Every other unknown pixel is in F (non-black).
//
// Facts the decomposition rests on (each B-B colour difference is 0, every B-F difference is >0):
//  1. Runs = 4-connected components of F.  Until the first pop of a B pixel that receives a
//     positive label (call it b1, at time T1), runs do not interact: a B pixel popped as -1 changes
//     nothing any other pixel reads.  Each run is flooded by itself ("phase 1": by a wave in LDS, or by a
//     lane in global memory where its frame is too large); B neighbours are recorded as leaf items (when,
//     at what level and by whom they are queued).
//  2. The global pop order of the merged runs is a total order computable from per-run data: for
//     items x, y of different runs, x pops first iff the largest (level, push time) key on x's
//     push chain is smaller than y's, comparing push times recursively through the pushers
//     (a pop can only be delayed by a larger key on its own chain).  `before()` implements it.
//  3. b1 = the earliest B item whose neighbours popped before it agree on one label Y1.  At T1 the
//     level-0 FIFO holds nothing else, so the flood from b1 runs to completion through every B
//     pixel not yet queued that it reaches (label Y1: such a pixel has no labelled F neighbour,
//     which would have queued it) before anything else pops.
//  4. After that, the unresolved pixels fall into 4-connected components that are again
//     independent ("phase 2"), each flooded by a lane, a larger one by a wave, from the queue state at T1.  The only
//     order not known locally is the FIFO order among F pixels queued by the flood from b1 at the
//     same level; for those the lane checks that every permutation gives the same labels.
// Anything outside these assumptions (a capacity, a comparison that does not terminate, a tie
// whose order matters) raises a flag and the caller re-runs the plain sequential flood.
#include <climits>
#include <cstdio>
#include <cstdlib>
#include <vector>

#include <hipcub/hipcub.hpp>

#include "common.hpp"
#include "ws_rules.hpp"

namespace nsc {

int ccl_neq(const uint8_t* img, uint8_t key, int32_t* labels, int w, int h, int conn, hipStream_t s);
int relabel_impl(int32_t* labels, int w, int h, int32_t bgval, int* dcount, int32_t* rank, hipStream_t s);
int bbox_impl(const int32_t* canon, int w, int h, int n, int32_t* out5, int32_t* area, hipStream_t s);

namespace {

constexpr int NQ = 256;
constexpr int IN_QUEUE = -2, WSHED = -1;
constexpr uint16_t NOPUSH = 0xFFFF;
enum { C_FRAME = 0, C_SEED = 1, C_F = 2, C_B = 3 };
enum { FB_LEAF_CAP = 1, FB_CMP = 2, FB_TIES = 4, FB_HEAP = 8, FB_TIEPERM = 16 };
constexpr int CMP_MAX_STEPS = 1 << 22;

struct Dev {
    // image
    const uint8_t* img;
    int W, H, N;
    const int32_t* m0;
    int32_t* m;
    const uint8_t* cls;
    const uint16_t* lvl0;
    const int32_t* run;  // canonical run id (1..R) for F pixels
    // Items: id < N is an F pixel or a B pixel queued in the initial scan, id >= N a leaf slot.  A record is
    // written when the item is queued, its pop index when it pops; records of other ids hold anything.
    // {run, largest-key item of the push chain, level << 24 | pop index, pusher (pixel, -1 = initial push)}
    int4* wr;
    // pop indexes from popcap on (a record then holds popcap); no plane where no run can have so many pops
    int32_t* popx;
    int popcap;
    int32_t* lab;  // F pixel: label decided in its run's flood, 0 = never queued there
    int32_t* qnext;  // FIFO links of the global-memory floods, indexed by item id
    // leaves
    int32_t* head;  // per B pixel: first leaf slot or -1
    int32_t* lf_b;
    int32_t* lf_next;
    int* nleaf;
    int leafcap;
    int* flags;
};

// A value every lane of the wave holds (or the one active lane's), as a wave-uniform value: the
// compiler then keeps it in a scalar register and branches on it with scalar branches.
__device__ __forceinline__ uint32_t uni(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }
__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }

// The label a popped pixel takes from its four neighbours (cv::watershed): the common positive
// label, WSHED where two positive labels differ, 0 where none is positive.  Branch-free: the
// largest label, and the smallest positive one found as the unsigned minimum of t - 1 (0, WSHED and
// IN_QUEUE wrap to the top).
__device__ __forceinline__ int pop_label(int a, int b, int c, int d) {
    const int mx = max(max(a, b), max(c, d));
    const unsigned mn1 = min(min((unsigned)(a - 1), (unsigned)(b - 1)), min((unsigned)(c - 1), (unsigned)(d - 1)));
    return mx <= 0 ? 0 : ((int)mn1 + 1 == mx ? mx : WSHED);
}

__device__ __forceinline__ int c_diff(const uint8_t* a, const uint8_t* b) {
    const int db = abs((int)a[0] - (int)b[0]);
    const int dg = abs((int)a[1] - (int)b[1]);
    const int dr = abs((int)a[2] - (int)b[2]);
    return max(max(db, dg), dr);
}

__device__ __forceinline__ int cdiff_packed(uint32_t a, uint32_t b) {
    const int d0 = abs((int)(a & 255) - (int)(b & 255));
    const int d1 = abs((int)((a >> 8) & 255) - (int)((b >> 8) & 255));
    const int d2 = abs((int)((a >> 16) & 255) - (int)((b >> 16) & 255));
    return max(max(d0, d1), d2);
}

// ---- item accessors ----
constexpr int kPopMax = 1 << 24;
__device__ __forceinline__ int rec_lvl(const int4& r) { return (int)((uint32_t)r.z >> 24); }
__device__ __forceinline__ int rec_pop(const Dev& D, int x, const int4& r) {
    const int q = r.z & (kPopMax - 1);
    return D.popx && q == D.popcap ? D.popx[x] : q;
}
__device__ __forceinline__ int it_lvl(const Dev& D, int x) { return rec_lvl(D.wr[x]); }
__device__ __forceinline__ int it_parent(const Dev& D, int x) { return D.wr[x].w; }

// x pops before y in the merged phase-1 flood (x != y); sets FB_CMP if the walk is too long.
// A step is two dependent loads: the records of x and y, then those of their chains' largest-key items.
__device__ bool before_from(const Dev& D, int x, int y, int step0) {
    for (int step = step0; step < CMP_MAX_STEPS; ++step) {
        if (x == y) return false;
        const int4 rx = D.wr[x], ry = D.wr[y];
        if (rx.x == ry.x) return rec_pop(D, x, rx) < rec_pop(D, y, ry);
        const int a = rx.y, b = ry.y;
        const int4 ra = D.wr[a], rb = D.wr[b];
        const int la = rec_lvl(ra), lb = rec_lvl(rb);
        if (la != lb) return la < lb;
        const int pa = ra.w, pb = rb.w;
        if (pa < 0 && pb < 0) return a < b;  // both queued in the initial raster scan
        if (pa < 0) return true;
        if (pb < 0) return false;
        x = pa;
        y = pb;
    }
    atomicOr(D.flags, FB_CMP);
    return false;
}
__device__ __forceinline__ bool before(const Dev& D, int x, int y) { return before_from(D, x, y, 0); }

// What the first step of before() reads about an item: its run and pop index, its chain's
// largest-key item, that item's level and pusher.  A tournament that compares the same winners
// level after level loads this once per candidate and carries it along.
struct ItemKey {
    int item, run, popidx, top, lvl, par;
};
__device__ __forceinline__ ItemKey item_key(const Dev& D, int x) {
    const int4 rx = D.wr[x];
    const int4 ra = D.wr[rx.y];
    return ItemKey{x, rx.x, rec_pop(D, x, rx), rx.y, rec_lvl(ra), ra.w};
}
// before(D, kx.item, ky.item), its first step taken from the keys
__device__ __forceinline__ bool before_keyed(const Dev& D, const ItemKey& kx, const ItemKey& ky) {
    if (kx.item == ky.item) return false;
    if (kx.run == ky.run) return kx.popidx < ky.popidx;
    if (kx.lvl != ky.lvl) return kx.lvl < ky.lvl;
    if (kx.par < 0 && ky.par < 0) return kx.top < ky.top;
    if (kx.par < 0) return true;
    if (ky.par < 0) return false;
    return before_from(D, kx.par, ky.par, 1);
}

// ---- classification ----
// One pixel: class and initial push level from its marker and colour and its four neighbours' (left, right,
// up, down; pos: the neighbour is a seed off the frame).
struct PixelClass {
    uint8_t cls;
    uint16_t lvl0;
};
__device__ __forceinline__ PixelClass classify(bool frame, int v, uint32_t col, const bool (&pos)[4], const uint32_t (&ncol)[4]) {
    int best = 256;  // smallest colour step to a neighbouring seed
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int d = cdiff_packed(col, ncol[k]);
        best = pos[k] ? min(best, d) : best;
    }
    return {(uint8_t)(frame ? C_FRAME : (v > 0 ? C_SEED : (col == 0 ? C_B : C_F))),
            (uint16_t)(frame || v > 0 || best >= 256 ? NOPUSH : best)};
}

// nF: this workgroup's count goes to partial[blockIdx.x] (summed by k_sum_partials): one atomic
// per workgroup on a single counter would serialise over a grid this large.
// Four pixels in a row (of the plane's linear order) to a thread: their markers and colours and those of
// the rows above and below come in 11 wide loads instead of 80 single ones, and go out in six stores.  The
// first and last row's groups, whose neighbour rows would leave the plane, take pixel by pixel loads.
// Bound by its 23 bytes per pixel; measured, 4098 x 4098: 164 -> 93 us.
// (which groups' loads stay inside both planes: classify_wide, ws_rules.hpp)
typedef int32_t __attribute__((ext_vector_type(4), aligned(4), may_alias)) i32x4_any;
typedef uint32_t __attribute__((ext_vector_type(3), aligned(1), may_alias)) u32x3_any;
typedef uint32_t __attribute__((aligned(1), may_alias)) u32_any;
// the four colours of 12 bytes
__device__ __forceinline__ void colours4(u32x3_any q, uint32_t (&c)[4]) {
    c[0] = q.x & 0xFFFFFFu;
    c[1] = __builtin_amdgcn_alignbit(q.y, q.x, 24) & 0xFFFFFFu;
    c[2] = __builtin_amdgcn_alignbit(q.z, q.y, 16) & 0xFFFFFFu;
    c[3] = q.z >> 8;
}
__device__ __forceinline__ uint32_t colour1(const uint8_t* p) { return p[0] | (uint32_t)p[1] << 8 | (uint32_t)p[2] << 16; }

__global__ void k_classify(Dev D, uint8_t* cls, uint16_t* lvl0, uint8_t* fmask, int* partial) {
    const int W = D.W, H = D.H, N = D.N;
    int local = 0;
    const int groups = (N + 3) / 4;
    for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < groups; t += gridDim.x * blockDim.x) {
        const int i0 = 4 * t;
        if (classify_wide(i0, W, N)) {
            const i32x4_any mo = *reinterpret_cast<const i32x4_any*>(D.m0 + i0), mu = *reinterpret_cast<const i32x4_any*>(D.m0 + i0 - W),
                            md = *reinterpret_cast<const i32x4_any*>(D.m0 + i0 + W);
            const int ml = D.m0[i0 - 1], mr = D.m0[i0 + 4];
            const uint8_t* px = D.img + 3 * (size_t)i0;
            const u32x3_any qo = *reinterpret_cast<const u32x3_any*>(px), qu = *reinterpret_cast<const u32x3_any*>(px - 3 * (size_t)W),
                            qd = *reinterpret_cast<const u32x3_any*>(px + 3 * (size_t)W);
            const uint32_t ql = *reinterpret_cast<const u32_any*>(px - 4), qr = *reinterpret_cast<const u32_any*>(px + 12);
            int y = i0 / W, x = i0 - y * W;
            uint32_t co[4], cu[4], cd[4];
            colours4(qo, co);
            colours4(qu, cu);
            colours4(qd, cd);
            const int m[6] = {ml, mo.x, mo.y, mo.z, mo.w, mr}, up[4] = {mu.x, mu.y, mu.z, mu.w}, dn[4] = {md.x, md.y, md.z, md.w};
            const uint32_t c[6] = {ql >> 8, co[0], co[1], co[2], co[3], qr & 0xFFFFFFu};
            uint32_t ocls = 0, omask = 0, ol[2] = {0, 0};
            i32x4_any om;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const bool frame = x == 0 || y == 0 || x == W - 1 || y == H - 1;
                const bool pos[4] = {x > 1 && m[j] > 0, x < W - 2 && m[j + 2] > 0, y > 1 && up[j] > 0, y < H - 2 && dn[j] > 0};
                const uint32_t nc[4] = {c[j], c[j + 2], cu[j], cd[j]};
                const int v = m[j + 1];
                const PixelClass q = classify(frame, v, c[j + 1], pos, nc);
                ocls |= (uint32_t)q.cls << (8 * j);
                ol[j >> 1] |= (uint32_t)q.lvl0 << (16 * (j & 1));
                omask |= (q.cls == C_F ? 1u : 0u) << (8 * j);
                om[j] = frame ? WSHED : (v < 0 ? 0 : v);
                if (++x == W) {
                    x = 0;
                    ++y;
                }
            }
            local += __popc(omask);
            *reinterpret_cast<u32_any*>(cls + i0) = ocls;
            *reinterpret_cast<u32_any*>(fmask + i0) = omask;
            *reinterpret_cast<u32_any*>(lvl0 + i0) = ol[0];
            *reinterpret_cast<u32_any*>(lvl0 + i0 + 2) = ol[1];
            *reinterpret_cast<i32x4_any*>(D.lab + i0) = i32x4_any{0, 0, 0, 0};
            *reinterpret_cast<i32x4_any*>(D.head + i0) = i32x4_any{-1, -1, -1, -1};
            *reinterpret_cast<i32x4_any*>(D.m + i0) = om;
            continue;
        }
        for (int i = i0; i < min(i0 + 4, N); ++i) {
            const int x = i % W, y = i / W;
            const bool frame = x == 0 || y == 0 || x == W - 1 || y == H - 1;
            // (a frame pixel, whose neighbours may leave the plane, reads itself)
            const int nb[4] = {frame ? i : i - 1, frame ? i : i + 1, frame ? i : i - W, frame ? i : i + W};
            bool pos[4] = {x > 1, x < W - 2, y > 1, y < H - 2};
            uint32_t nc[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                pos[k] = pos[k] && D.m0[nb[k]] > 0;
                nc[k] = colour1(D.img + 3 * (size_t)nb[k]);
            }
            const int v = D.m0[i];
            const PixelClass q = classify(frame, v, colour1(D.img + 3 * (size_t)i), pos, nc);
            cls[i] = q.cls;
            lvl0[i] = q.lvl0;
            fmask[i] = q.cls == C_F ? 1 : 0;
            D.lab[i] = 0;
            D.head[i] = -1;
            D.m[i] = frame ? WSHED : (v < 0 ? 0 : v);
            local += q.cls == C_F;
        }
    }
    const int bs = block_sum(local);
    if (threadIdx.x == 0) partial[blockIdx.x] = bs;
}

// *out = sum of partial[0..n) (one workgroup of 1024 threads)
__global__ __launch_bounds__(1024) void k_sum_partials(const int* __restrict__ partial, int n, int* out) {
    int v = 0;
    for (int i0 = threadIdx.x; i0 < n; i0 += 4 * blockDim.x) {  // four loads in flight per thread
        int p[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) p[j] = i0 + j * (int)blockDim.x < n ? partial[i0 + j * blockDim.x] : 0;
        v += p[0] + p[1] + p[2] + p[3];
    }
    const int t = block_sum(v);
    if (threadIdx.x == 0) *out = t;
}

// ---- phase 1: the flood of one run ----
// in global memory, by one lane, for runs whose frame exceeds the LDS tiers
// (MANY: with the plane of pop indexes beyond the records'; the kernel of the others is 4 % slower with its code)
template <bool MANY>
__device__ void flood_global(const Dev& D, const int32_t* __restrict__ box5, int nrun, int r, int* __restrict__ qh,
                             int* __restrict__ qt) {
    const int W = D.W;
    const int id = r + 1;
    int* head = qh + (size_t)r * NQ;  // per run (run ids are unique across the tiers)
    int* tail = qt + (size_t)r * NQ;
    for (int l = 0; l < NQ; ++l) { head[l] = -1; tail[l] = -1; }
    int active = NQ, popc = 0;
    auto enq = [&](int l, int x) {
        D.qnext[x] = -1;
        if (tail[l] >= 0) D.qnext[tail[l]] = x;
        else head[l] = x;
        tail[l] = x;
        if (l < active) active = l;
    };
    constexpr int QUEUED = -3;  // lab of a pixel that waits in a FIFO
    auto record = [&](int x, int top, int parent, int level) { D.wr[x] = make_int4(id, top, level << 24, parent); };
    const int minx = box5[nrun + r], maxx = box5[2 * nrun + r];
    const int miny = box5[3 * nrun + r], maxy = box5[4 * nrun + r];
    for (int y = miny; y <= maxy; ++y)
        for (int x = minx; x <= maxx; ++x) {
            const int i = y * W + x;
            if (D.cls[i] == C_F && D.run[i] == id && D.lvl0[i] != NOPUSH) {
                record(i, i, -1, D.lvl0[i]);
                D.lab[i] = QUEUED;
                enq(D.lvl0[i], i);
            }
        }
    const int dirs[4] = {-1, 1, -W, W};
    for (;;) {
        if (active >= NQ) break;
        if (head[active] < 0) {
            int l = active + 1;
            while (l < NQ && head[l] < 0) ++l;
            if (l == NQ) break;
            active = l;
        }
        const int x = head[active];
        const int nx = D.qnext[x];
        head[active] = nx;
        if (nx < 0) tail[active] = -1;
        D.wr[x].z |= MANY ? min(popc, D.popcap) : popc;
        if (MANY && popc >= D.popcap) D.popx[x] = popc;
        ++popc;
        if (x >= D.N) continue;  // a leaf: when it pops, nothing else
        const int p = x;
        int lab = 0;
        for (int d = 0; d < 4; ++d) {
            const int s = p + dirs[d];
            int t = 0;
            const uint8_t cs = D.cls[s];
            if (cs == C_SEED) t = D.m0[s];
            else if (cs == C_F) t = D.lab[s];  // positive once popped and labelled
            if (t > 0) { if (lab == 0) lab = t; else if (t != lab) lab = WSHED; }
        }
        D.lab[p] = lab;
        if (lab == WSHED) continue;
        const uint8_t* ptr = D.img + 3 * (size_t)p;
        const int bp = D.wr[p].y;
        const int bl = it_lvl(D, bp);  // a new item's key is the larger one at the same level (pushed later)
        for (int d = 0; d < 4; ++d) {
            const int s = p + dirs[d];
            const uint8_t cs = D.cls[s];
            if (cs == C_F) {
                if (D.lab[s] != 0) continue;
                const int l = c_diff(ptr, D.img + 3 * (size_t)s);
                record(s, bl <= l ? s : bp, p, l);
                D.lab[s] = QUEUED;
                enq(l, s);
            } else if (cs == C_B && D.lvl0[s] == NOPUSH) {
                bool done = false;  // queued already by an earlier labelled neighbour of this run
                for (int e = 0; e < 4; ++e) {
                    const int f2 = s + dirs[e];
                    if (f2 != p && D.cls[f2] == C_F && D.run[f2] == id && D.lab[f2] > 0) done = true;
                }
                if (done) continue;
                const int slot = atomicAdd(D.nleaf, 1);
                if (slot >= D.leafcap) { atomicOr(D.flags, FB_LEAF_CAP); continue; }
                const int l = c_diff(ptr, D.img + 3 * (size_t)s);
                D.lf_b[slot] = s;  // linked into head[s] by k_link_leaves
                const int lid = D.N + slot;
                record(lid, bl <= l ? lid : bp, p, l);
                enq(l, lid);
            }
        }
    }
}

// with the run's neighbourhood staged in LDS, by one wave, for runs whose bounding box plus a 2-pixel
// margin has at most 6400 pixels: the same flood.  The frame is staged into LDS (the 2-pixel margin keeps every neighbour of a leaf
// candidate inside it), the initial items are numbered in raster order with ballots, and the wave pops
// item by item.
// A flood is one chain of pops by one wave, so a pop costs the instructions it issues and the round
// trips it waits for.  With one lane driving it through LDS FIFOs that was 1800 cycles (round trips for
// the head, the neighbours and each pushed FIFO's tail, one per empty level passed over; some fifty
// branches).  Here
//  * everything a pixel holds is 16 bytes of LDS, and lanes 0..3 read the four neighbours and lane 4
//    the pixel itself in one instruction: the pop's only round trip;
//  * the four neighbours are judged, numbered and recorded side by side in their lanes, each item with
//    one 16-byte record;
//  * their FIFOs' entries are read together as soon as the levels are known, behind the label, the
//    numbering and the records; pushes of one level are chained inside the quad;
//  * a level that has run out finds the next queued one in one read of all 256 entries.
//  * labels and pop indexes stay in LDS and leave for the image in one sweep after the last pop.
// Measured: a pop takes 930 cycles; the longest flood of a 512 x 512 tile (704 pops, staging included)
// 509 -> 291 us.
// Each queued F pixel carries the key (level, push sequence) and frame index of its chain's largest-key
// item, so a push compares keys without following pointers.  Leaf slots are reserved per run up front
// (one per B pixel of the frame that could become a leaf), so no atomic sits on the flood's critical
// path; unused slots get lf_b = -1.
constexpr uint16_t NIL16 = 0xFFFF;
// phase-1 FIFO links: an item index below 0x7FFF (frames hold at most 6400 pixels), P1_LEAF when
// the item is a leaf, P1_NIL for none
constexpr uint32_t P1_NIL = 0x7FFF, P1_LEAF = 0x8000, P1_EMPTY = P1_NIL << 16 | P1_NIL;
// the frame pixel's flags: of the run; not queued yet and pushed by a labelled neighbour as an F item /
// as a leaf; queued in the initial scan
enum { K_INRUN = 4, K_CANF = 8, K_CANL = 16, K_LV = 32 };
constexpr int P1_MARGIN = 2;
// parts of a 16-byte entry, accessed beside the whole entry
typedef uint32_t __attribute__((may_alias)) any_u32;
typedef uint16_t __attribute__((may_alias)) any_u16;

// the lane's quad (lanes 4 q .. 4 q + 3) combined by max / min: every lane of it gets the result
__device__ __forceinline__ int quad_swap1(int v) { return __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xF, 0xF, true); }
__device__ __forceinline__ int quad_swap2(int v) { return __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xF, 0xF, true); }
__device__ __forceinline__ int quad_max(int v) {
    v = max(v, quad_swap1(v));
    return max(v, quad_swap2(v));
}
__device__ __forceinline__ uint32_t quad_min(uint32_t v) {
    v = min(v, (uint32_t)quad_swap1((int)v));
    return min(v, (uint32_t)quad_swap2((int)v));
}
// pop_label of the four values in a quad's lanes, at least one of them positive
__device__ __forceinline__ int quad_label(int t) {
    const int mx = quad_max(t);
    const uint32_t mn1 = quad_min((uint32_t)t - 1u);
    return (int)mn1 + 1 == mx ? mx : WSHED;
}
__device__ __forceinline__ uint32_t lane_of(uint32_t v, int lane) {
    return (uint32_t)__builtin_amdgcn_readlane((int)v, lane);
}
__device__ __forceinline__ int lanes_below(unsigned long long m) {
    return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// v of lane (lane + R) & 3 of the lane's quad
template <int R>
__device__ __forceinline__ uint32_t quad_rot(uint32_t v) {
    constexpr int ctrl = R == 1 ? 0x39 : (R == 2 ? 0x4E : 0x93);
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, ctrl, 0xF, 0xF, true);
}
// {level - 4 * lane << 16 | head} of the lowest queued level of a lane's four FIFO entries, P1_NIL for none
__device__ __forceinline__ uint32_t first_queued(uint4 q) {
    const uint32_t h0 = q.x & 0xFFFFu, h1 = q.y & 0xFFFFu, h2 = q.z & 0xFFFFu, h3 = q.w & 0xFFFFu;
    uint32_t v = h3 != P1_NIL ? 3u << 16 | h3 : P1_NIL;
    v = h2 != P1_NIL ? 2u << 16 | h2 : v;
    v = h1 != P1_NIL ? 1u << 16 | h1 : v;
    return h0 != P1_NIL ? h0 : v;
}

// pixels of run r's frame: its box plus the margin
__device__ __forceinline__ int run_frame(const int32_t* __restrict__ box5, int nrun, int r) {
    const long long L = (long long)(box5[2 * nrun + r] - box5[nrun + r] + 1 + 2 * P1_MARGIN) *
                        (box5[4 * nrun + r] - box5[3 * nrun + r] + 1 + 2 * P1_MARGIN);
    return (int)min(L, (long long)INT_MAX);
}

// the wave's n of a counter
__device__ __forceinline__ int wave_take(int* counter, int n) {
    int v = 0;
    if ((threadIdx.x & 63) == 0) v = atomicAdd(counter, n);
    return uni(v);
}

// the wave's own LDS accesses before this point come before those after it
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// qlv (64 entries): per level its FIFO's tail << 16 | head; empty while the head is P1_NIL.
// px (one entry per frame pixel): x = class and flags | push level to the right << 8 | to the lower
// neighbour << 16 | level of its initial push << 24; y = frame index of a queued F pixel's chain's
// largest-key item, or a leaf's index in the run | FIFO link << 16; z = known label (seed label, label of a
// popped F pixel, else 0); w = that largest-key item's key (level << 16 | push seq), then the pixel's pop
// index (and its colour while the frame is staged)
__device__ __forceinline__ void flood_lds(const Dev& D, const int32_t* __restrict__ box5, int nrun, int r, uint4* qlv, uint4* px) {
    any_u32* const word = reinterpret_cast<any_u32*>(px);
    any_u16* const half = reinterpret_cast<any_u16*>(px);  // pixel k's link: half[8 k + 3]
    any_u32* const entry = reinterpret_cast<any_u32*>(qlv);
    any_u16* const head = reinterpret_cast<any_u16*>(qlv);  // head[2 l]
    const int lane = threadIdx.x & 63;
    const int W = D.W, H = D.H, id = r + 1;
    const int ox = uni(box5[nrun + r]) - P1_MARGIN, oy = uni(box5[3 * nrun + r]) - P1_MARGIN;
    const int lw = uni(box5[2 * nrun + r]) - ox + 1 + P1_MARGIN, lh = uni(box5[4 * nrun + r]) - oy + 1 + P1_MARGIN;
    const int L = lw * lh;
    // k / lw by multiply-high (exact for k < 2^16)
    const uint32_t magic = (uint32_t)((0x100000000ull + (unsigned)lw - 1) / (unsigned)lw);
    const int gbase = oy * W + ox, gstep = W - lw;
    auto gidx = [&](int k) { return gbase + k + (int)__umulhi((uint32_t)k, magic) * gstep; };

    qlv[lane] = make_uint4(P1_EMPTY, P1_EMPTY, P1_EMPTY, P1_EMPTY);
    // eight chunks of 64 pixels at a time, every load from a clamped (always valid) pixel before any use
    for (int k0 = 0; k0 < L; k0 += 512) {
        uint8_t c[8], q0[8], q1[8], q2[8];
        uint16_t l0[8];
        int32_t rn[8], m0[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int k = min(k0 + 64 * j + lane, L - 1);
            const int ky = (int)__umulhi((uint32_t)k, magic);
            const size_t g = (size_t)clampi(oy + ky, 0, H - 1) * W + clampi(ox + k - ky * lw, 0, W - 1);
            c[j] = D.cls[g];
            rn[j] = D.run[g];
            m0[j] = D.m0[g];
            l0[j] = D.lvl0[g];
            q0[j] = D.img[3 * g];
            q1[j] = D.img[3 * g + 1];
            q2[j] = D.img[3 * g + 2];
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int k = k0 + 64 * j + lane;
            if (k >= L) continue;
            const int ky = (int)__umulhi((uint32_t)k, magic), gx = ox + k - ky * lw, gy = oy + ky;
            const bool in = gx >= 0 && gx < W && gy >= 0 && gy < H;  // the margin may step one pixel off the image
            const bool lv = l0[j] != NOPUSH;
            uint32_t cd = c[j];
            if (cd == C_F) cd |= K_CANF | (rn[j] == id ? K_INRUN : 0);
            if (cd == C_B && !lv) cd |= K_CANL;
            if (lv) cd |= K_LV | (uint32_t)l0[j] << 24;
            px[k] = make_uint4(in ? cd : (uint32_t)C_FRAME, P1_NIL << 16, in && c[j] == C_SEED ? (uint32_t)m0[j] : 0u,
                               in ? q0[j] | (uint32_t)q1[j] << 8 | (uint32_t)q2[j] << 16 : 0u);
        }
    }
    wave_lds_fence();
    // push levels between 4-neighbours (a pair that wraps around a frame row is never used: pushes
    // start at run pixels, which lie the margin away from the frame's edge)
    for (int k = lane; k < L; k += 64) {
        const uint32_t c = word[4 * k + 3], cr = word[4 * min(k + 1, L - 1) + 3], cl = word[4 * min(k + lw, L - 1) + 3];
        const uint32_t rt = (uint32_t)cdiff_packed(c, cr), dn = (uint32_t)cdiff_packed(c, cl);
        word[4 * k] |= rt << 8 | dn << 16;
    }
    wave_lds_fence();
    // leaf candidates (B, never initially queued, 4-adjacent to the run) and initial items in raster
    // order: a chunk's items of one level are linked in a row behind that level's FIFO (the first of
    // them reads the entry, the last writes it)
    int cnt = 0, seq = 0;
    for (int k0 = 0; k0 < L; k0 += 64) {
        const int k = k0 + lane, kc = min(k, L - 1);
        const int ky = (int)__umulhi((uint32_t)kc, magic), kx = kc - ky * lw;
        const bool inner = k < L && kx > 0 && kx < lw - 1 && ky > 0 && ky < lh - 1;
        const int kn = inner ? kc : min(lw + 1, L - 1);  // a pixel whose neighbours exist (frames are 5 x 5 at least)
        const uint32_t cd = word[4 * kc];
        const uint32_t nb = word[4 * (kn - 1)] | word[4 * (kn + 1)] | word[4 * (kn - lw)] | word[4 * (kn + lw)];
        const bool cand = inner && (cd & K_CANL) && (nb & K_INRUN);
        const bool init = k < L && (cd & K_INRUN) && (cd & K_LV);
        const unsigned long long bi = __ballot(init);
        cnt += __popcll(__ballot(cand));
        if (!bi) continue;
        const int lvl = init ? (int)(cd >> 24) : -1, q = seq + lanes_below(bi);
        int first = -1, prev = -1, next = -1;  // lanes of this chunk's first, previous and next item of the level
        for (unsigned long long m = bi; m; m &= m - 1) {
            const int j = __builtin_ctzll(m);
            const bool same = (int)lane_of((uint32_t)lvl, j) == lvl;
            first = same && first < 0 ? j : first;
            prev = same && j < lane ? j : prev;
            next = same && j > lane && next < 0 ? j : next;
        }
        if (init) {
            const int g = gidx(k);
            px[k] = make_uint4(cd & ~(uint32_t)K_CANF, (next < 0 ? P1_NIL : (uint32_t)(k0 + next)) << 16 | (uint32_t)k, 0u,
                               (uint32_t)lvl << 16 | (uint32_t)q);
            D.wr[g] = make_int4(id, g, lvl << 24, -1);
            const uint32_t e = entry[lvl], h = e & 0xFFFFu;
            if (prev < 0 && h != P1_NIL) half[8 * (e >> 16) + 3] = (uint16_t)k;
            if (next < 0) entry[lvl] = (uint32_t)k << 16 | (h == P1_NIL ? (uint32_t)(k0 + first) : h);
        }
        seq += __popcll(bi);
    }
    if (!seq) return;  // nothing queued initially: the run is not flooded in this phase and takes no leaf slots
    wave_lds_fence();
    const int base = wave_take(D.nleaf, cnt);
    if (base + cnt > D.leafcap) {
        // every reserved slot below the capacity reads as unused
        for (int j = base + lane; j < D.leafcap; j += 64) D.lf_b[j] = -1;
        if (lane == 0) atomicOr(D.flags, FB_LEAF_CAP);
        return;
    }

    // lanes 0..3: the neighbours in push order (left, right, up, down); the others read the pixel itself
    // (queued, so never pushed)
    const int loff = lane == 0 ? -1 : (lane == 1 ? 1 : (lane == 2 ? -lw : (lane == 3 ? lw : 0)));
    const int goff = lane == 0 ? -1 : (lane == 1 ? 1 : (lane == 2 ? -W : (lane == 3 ? W : 0)));
    const int lsh = lane < 2 ? 8 : 16;  // where the level of the push over that edge is, in the pixel itself (lanes
                                        // 1, 3) or in the neighbour (0, 2)
    int popc = 0, nlf = 0, active = 0;
    uint32_t hx = P1_NIL;  // the next item to pop, of level `active`; P1_NIL: of the lowest queued level
    while (popc < L) {  // (a pixel pops at most once)
        if (hx == P1_NIL) {
            const uint32_t f = first_queued(qlv[lane]);
            const unsigned long long m = __builtin_amdgcn_ballot_w64(f != P1_NIL);
            if (!m) break;
            const int l4 = __builtin_ctzll(m);
            const uint32_t v = lane_of(f, l4);
            active = 4 * l4 + (int)(v >> 16);
            hx = v & 0xFFFFu;
        }
        const int x = (int)(hx & P1_NIL);
        const uint4 s = px[x + loff];
        const uint32_t cw = lane_of(s.x, 4), yw = lane_of(s.y, 4), key = lane_of(s.w, 4);
        const uint32_t nx = yw >> 16;
        if (lane == 4) head[2 * active] = (uint16_t)nx;
        const int lvl = (int)(((lane & 1) ? cw : s.x) >> lsh & 255u);
        const uint32_t e = entry[lvl];  // used by the pushes below; everything up to them runs while it loads
        const int ql = uni(quad_label((int)s.z));
        const int lab = hx & P1_LEAF ? 0 : ql;  // a leaf's pop is only counted: no label, no pushes
        // the neighbours to push (none from a leaf or a dam).  A neighbour's state may have changed since the
        // read only through this pop's own pushes, which go to other pixels.  A B pixel queued already is a
        // leaf pushed by an earlier labelled neighbour of this run (every popped F pixel of the run is labelled
        // or a dam, and a labelled one queues its B neighbours)
        const bool isl = s.x & K_CANL, push = lab > 0 && (s.x & (K_CANF | K_CANL));
        const uint32_t m = (uint32_t)__builtin_amdgcn_ballot_w64(push), ml = m & (uint32_t)__builtin_amdgcn_ballot_w64(isl);
        const int sk = x + loff;
        const int sq = (int)__builtin_amdgcn_mbcnt_lo(m, (uint32_t)seq), j = (int)__builtin_amdgcn_mbcnt_lo(ml, (uint32_t)nlf);
        const uint32_t nkey = (uint32_t)lvl << 16 | (uint32_t)sq, bl = yw & 0xFFFFu;
        const bool newer = key < nkey;  // the new item has the larger key on its chain
        if (push || lane == 4) {
            const uint32_t y = P1_NIL << 16 | (isl ? (uint32_t)j : (newer ? (uint32_t)sk : bl));
            px[sk] = make_uint4(s.x & ~(uint32_t)(K_CANF | K_CANL), push ? y : s.y, push ? s.z : (uint32_t)lab,
                                push ? max(key, nkey) : (uint32_t)popc);
        }
        ++popc;
        hx = nx;
        if (!m) continue;
        seq += __popc(m);
        nlf += __popc(ml);
        // pushes of one level go one behind the other, the first of them behind the FIFO's tail; lanes that
        // push nothing hold levels of their own
        const uint32_t pl = push ? (uint32_t)lvl : 256u + (uint32_t)lane, qx = (uint32_t)sk | (isl ? P1_LEAF : 0u);
        const bool s1 = quad_rot<1>(pl) == pl, s2 = quad_rot<2>(pl) == pl, s3 = quad_rot<3>(pl) == pl;
        const uint32_t q1 = quad_rot<1>(qx), q2 = quad_rot<2>(qx), q3 = quad_rot<3>(qx);
        const bool b1 = s3 && lane >= 1, b2 = s2 && lane >= 2, b3 = s1 && lane >= 3;  // one, two, three lanes before
        const bool last = !((s1 && lane <= 2) || (s2 && lane <= 1) || (s3 && lane == 0));
        const uint32_t first = b3 ? q1 : (b2 ? q2 : (b1 ? q3 : qx)), prev = b1 ? q3 : (b2 ? q2 : q1);
        const bool chained = b1 || b2 || b3;
        if (push) {
            const int gp = gidx(x), gs = gp + goff, gt = gidx((int)bl);
            const int me = isl ? D.N + base + j : gs;
            D.wr[me] = make_int4(id, newer ? me : gt, lvl << 24, gp);
        }
        // the level to go on with: a pushed one below the active level, or at it if its FIFO has run out
        const uint32_t lo = (uint32_t)uni((int)quad_min(pl << 2 | (uint32_t)(lane & 3)));
        const int ll = (int)(lo >> 2);
        if (ll + (nx != P1_NIL ? 1 : 0) <= active) {
            active = ll;
            hx = lane_of(qx, (int)(lo & 3u));
        }
        const uint32_t h = e & 0xFFFFu;
        const uint32_t tail = chained ? prev & P1_NIL : e >> 16;
        if (push && (chained || h != P1_NIL)) half[8 * tail + 3] = (uint16_t)qx;
        if (push && last) entry[lvl] = (uint32_t)sk << 16 | (h == P1_NIL ? first : h);
    }
    wave_lds_fence();
    // labels and pop indexes (low half of a record's third word) of the run's queued pixels and of its
    // leaves (every queued item has popped)
    auto pop_of = [&](int item) -> any_u16& { return reinterpret_cast<any_u16*>(D.wr + item)[4]; };
    for (int k = lane; k < L; k += 64) {
        const uint4 s = px[k];
        const int g = gidx(k);
        if ((s.x & (K_INRUN | K_CANF)) == K_INRUN) {
            pop_of(g) = (uint16_t)s.w;
            D.lab[g] = (int)s.z;
        } else if ((s.x & (3 | K_LV | K_CANL)) == C_B) {
            const int j = base + (int)(s.y & 0xFFFFu);
            pop_of(D.N + j) = (uint16_t)s.w;
            D.lf_b[j] = g;
        }
    }
    for (int j = base + nlf + lane; j < base + cnt; j += 64) D.lf_b[j] = -1;
}

// ---- all run floods, from a pool of LDS per CU ----
// One workgroup of 16 waves per CU holds all its LDS; each wave takes the next run, largest frames first,
// and the LDS that run's frame needs, in 1 KB units.  A flood is a chain of dependent steps that leaves most
// issue slots of its SIMD idle, so what counts is how many are in flight: by frame size (launches per size
// tier, each with its tier's LDS, held a third less and each tier ended with its own few longest floods).
// Measured: 363 -> 315 us for a 512 x 512 tile (its longest flood alone is 290), 823 -> 689 us for a
// 4096 x 4096 one.
constexpr int P1_WAVES = 16, P1_UNITS = 158;  // 64 frame pixels a unit
constexpr int kRunTiers = 6;
// runs by the size of their LDS frame: tier b holds frames of at most kRunTier[b] pixels; the last one
// floods from global memory
constexpr int kRunTierMax = 6400;
__constant__ int kRunTier[kRunTiers - 1] = {512, 1024, 2048, 4096, kRunTierMax};

struct LdsPool {
    unsigned long long used[3];
    int lock;
    // the lowest n free units in a row, taken (-1: none now).  Wave-uniform.
    __device__ int take(int n, int lane) {
        enter(lane);
        unsigned long long f[3], r[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            f[k] = ~used[k];
            r[k] = f[k];
        }
        for (int len = 1; len < n;) {  // r: units that start len free ones
            const int sh = min(len, n - len);
            if (sh == 64) {
                r[0] &= r[1]; r[1] &= r[2]; r[2] = 0;
            } else {
                r[0] &= r[0] >> sh | r[1] << (64 - sh);
                r[1] &= r[1] >> sh | r[2] << (64 - sh);
                r[2] &= r[2] >> sh;
            }
            len += sh;
        }
        int at = -1;
#pragma unroll
        for (int k = 2; k >= 0; --k) at = r[k] ? 64 * k + __builtin_ctzll(r[k]) : at;
        at = uni(at);
        if (at >= 0) mark(at, n, lane, true);
        leave(lane);
        return at;
    }
    __device__ void give(int at, int n, int lane) {
        enter(lane);
        mark(at, n, lane, false);
        leave(lane);
    }
    __device__ void mark(int at, int n, int lane, bool on) {
        if (lane < 3) {
            const int lo = max(at - 64 * lane, 0), hi = min(at + n - 64 * lane, 64);
            if (lo < hi) {
                const unsigned long long m = (hi - lo == 64 ? ~0ull : (1ull << (hi - lo)) - 1ull) << lo;
                used[lane] = on ? used[lane] | m : used[lane] & ~m;
            }
        }
    }
    __device__ void enter(int lane) {
        if (lane == 0) {
            int was = 0;
            while (!__hip_atomic_compare_exchange_strong(&lock, &was, 1, __ATOMIC_ACQUIRE, __ATOMIC_RELAXED,
                                                         __HIP_MEMORY_SCOPE_WORKGROUP)) {
                was = 0;
                __builtin_amdgcn_s_sleep(1);
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        __builtin_amdgcn_wave_barrier();
    }
    __device__ void leave(int lane) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __builtin_amdgcn_wave_barrier();
        if (lane == 0) __hip_atomic_store(&lock, 0, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
};

template <bool MANY>
__global__ __launch_bounds__(64 * P1_WAVES) void k_phase1(Dev D, const int32_t* __restrict__ box5, int nrun,
                                                          const int* __restrict__ lists, const int* __restrict__ counts,
                                                          int* __restrict__ next_run, int* __restrict__ qh, int* __restrict__ qt) {
    __shared__ uint4 pool[64 * P1_UNITS];
    __shared__ LdsPool P;
    const int lane = threadIdx.x & 63, wave = uni((int)(threadIdx.x >> 6));
    if (threadIdx.x == 0) {
        P.used[0] = P.used[1] = 0;
        P.used[2] = ~0ull << (P1_UNITS - 128);
        P.lock = 0;
    }
    __syncthreads();  // the only one: the waves go their own ways below
    // first runs spread over the workgroups, further ones from the counter
    int it = wave * (int)gridDim.x + (int)blockIdx.x;
    for (;;) {
        int r = -1, tier = 0, k = it;
        for (int t = kRunTiers - 1; t >= 0 && r < 0; --t) {
            const int c = uni(counts[t]);
            if (k < c) {
                r = uni(lists[(size_t)t * nrun + k]);
                tier = t;
            } else {
                k -= c;
            }
        }
        if (r < 0) break;
        if (tier == kRunTiers - 1) {
            if (lane == 0) flood_global<MANY>(D, box5, nrun, r, qh, qt);
        } else {
            const int L = uni(run_frame(box5, nrun, r));
            const int n = 1 + (L + 63) / 64;  // 102 at most: the pool holds it once the floods in flight are done
            int at;
            while ((at = P.take(n, lane)) < 0) __builtin_amdgcn_s_sleep(64);
            flood_lds(D, box5, nrun, r, pool + 64 * at, pool + 64 * (at + 1));
            P.give(at, n, lane);
        }
        it = wave_take(next_run, 1) + P1_WAVES * (int)gridDim.x;
    }
}


// compute units of the current device (the grid of the run floods)
static int device_cus() {
    static const int n = [] {
        int dev = 0, cus = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) {
            (void)hipGetLastError();
            return 256;
        }
        return std::max(1, cus);
    }();
    return n;
}

// wave-aggregated append of the lanes whose `take` is set
__device__ __forceinline__ void wave_append(bool take, int v, int* __restrict__ list, int* __restrict__ count) {
    const unsigned long long m = __ballot(take);
    if (!m) return;
    const int lane = threadIdx.x & 63;
    const int leader = __ffsll((long long)m) - 1;
    int base = 0;
    if (lane == leader) base = atomicAdd(count, __popcll(m));
    base = __shfl(base, leader);
    if (take) list[base + __popcll(m & ((1ull << lane) - 1ull))] = v;
}

// every used leaf slot joins the list of its B pixel (list order is irrelevant to its readers);
// the first leaf of a pixel also puts the pixel on the list of B pixels with queue entries
// (one append per workgroup and iteration: an atomic per wave on the single list counter
// serialises over tens of thousands of waves)
__global__ void k_link_leaves(Dev D, int* __restrict__ blist, int* __restrict__ bcount) {
    const int n = min(*D.nleaf, D.leafcap);
    const int stride = gridDim.x * blockDim.x;
    for (int k0 = blockIdx.x * blockDim.x; k0 < n; k0 += stride) {  // block-uniform trip count
        const int sl = k0 + threadIdx.x;
        bool first = false;
        int b = -1;
        if (sl < n) {
            b = D.lf_b[sl];
            if (b >= 0 && b < D.N) {
                const int old = atomicExch(&D.head[b], sl);
                D.lf_next[sl] = old;
                first = old < 0;
            }
        }
        block_append(first, b, blist, bcount);
    }
}

// B pixels queued in the initial scan (next to a seed): their list and their records (each a run of its
// own, without a pusher)
__global__ void k_collect_b0(Dev D, int* __restrict__ blist, int* __restrict__ bcount) {
    const int stride = gridDim.x * blockDim.x;
    const int n_up = ((D.N + 63) / 64) * 64;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n_up; i += stride) {
        const int j = min(i, D.N - 1);  // both loads unconditional (clamped), then the test
        const uint8_t c = D.cls[j];
        const uint16_t l0 = D.lvl0[j];
        const bool take = i < D.N && c == C_B && l0 != NOPUSH;
        if (take) D.wr[i] = make_int4(-(i + 2), i, (int)l0 << 24, -1);
        wave_append(take, i, blist, bcount);
    }
}

// (one append per wave and bucket: an atomic per run on the few bucket counters serialises)
__global__ void k_bucket_runs(const int32_t* __restrict__ box5, int nrun, int* __restrict__ lists, int* __restrict__ counts) {
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    int b = -1;
    if (r < nrun) {
        const int L = run_frame(box5, nrun, r);
        b = 0;
        while (b < kRunTiers - 1 && L > kRunTier[b]) ++b;
    }
    for (int t = 0; t < kRunTiers; ++t) wave_append(b == t, r, lists + (size_t)t * nrun, &counts[t]);
}

// Label a B pixel b (never on the frame) takes when its queue entry r pops: the agreeing positive
// label of its seed neighbours and of its F neighbours popped (labelled) before r, WSHED where
// they disagree, 0 for none.  The four neighbours' class, marker, state and label are loaded
// together and used through selects (loads behind the class test were a dependent round trip
// per neighbour); only the pop-order walk stays conditional.
__device__ int b_label(const Dev& D, int b, int r, int W) {
    const int dirs[4] = {-1, 1, -W, W};
    uint8_t cs[4];
    int ms[4], ls[4];
#pragma unroll
    for (int d = 0; d < 4; ++d) {
        const int s = b + dirs[d];
        cs[d] = D.cls[s];
        ms[d] = D.m0[s];
        ls[d] = D.lab[s];
    }
    int lab = 0;
#pragma unroll
    for (int d = 0; d < 4; ++d) {
        const bool seed = cs[d] == C_SEED;
        const bool fcand = cs[d] == C_F && ls[d] > 0;
        int t = seed ? ms[d] : 0;
        if (!seed && fcand && before(D, b + dirs[d], r)) t = ls[d];
        if (t > 0) { if (lab == 0) lab = t; else if (t != lab) lab = WSHED; }
    }
    return lab;
}

// ---- B items: the real queue entry of each B pixel and its label decision at pop time ----
// over the B pixels that have a queue entry (listed by k_collect_b0 / k_link_leaves); real[] of
// every other pixel stays -1
__global__ void k_bresolve(Dev D, int32_t* __restrict__ real, int* __restrict__ cand, int* __restrict__ ncand,
                           const int* __restrict__ blist, const int* __restrict__ bcount) {
    const int W = D.W;
    const int nb = *bcount;
    // block-uniform trip count (block_append synchronises the block)
    for (int k0 = blockIdx.x * blockDim.x; k0 < nb; k0 += gridDim.x * blockDim.x) {
        const int k = k0 + threadIdx.x;
        int b = -1, lab = 0;
        if (k < nb) {
            b = blist[k];
            int r = -1;
            if (D.lvl0[b] != NOPUSH) r = b;
            else {
                for (int sl = D.head[b]; sl >= 0; sl = D.lf_next[sl]) {
                    const int lid = D.N + sl;
                    if (r < 0 || before(D, it_parent(D, lid), it_parent(D, r))) r = lid;
                }
            }
            real[b] = r;
            if (r >= 0) lab = b_label(D, b, r, W);
        }
        block_append(lab > 0, b, cand, ncand);
    }
}

// earliest candidate per block (candidates: B pixels whose earlier-popped neighbours agree on a
// positive label), -1 for a block without candidates
constexpr int B1_BLOCKS = 1024;
__global__ __launch_bounds__(256) void k_b1_partial(Dev D, const int32_t* __restrict__ real, const int* __restrict__ cand,
                                                    const int* __restrict__ ncand, int* __restrict__ partial) {
    __shared__ int best[256];
    __shared__ ItemKey bkey[256];
    const int n = *ncand;
    int mine = -1;
    for (int k = blockIdx.x * 256 + threadIdx.x; k < n; k += B1_BLOCKS * 256) {
        const int b = cand[k];
        if (mine < 0 || before(D, real[b], real[mine])) mine = b;
    }
    best[threadIdx.x] = mine;
    if (mine >= 0) bkey[threadIdx.x] = item_key(D, real[mine]);
    __syncthreads();
    for (int stride = 128; stride > 0; stride >>= 1) {
        if ((int)threadIdx.x < stride) {
            const int a = best[threadIdx.x], c = best[threadIdx.x + stride];
            if (a < 0 || (c >= 0 && before_keyed(D, bkey[threadIdx.x + stride], bkey[threadIdx.x]))) {
                best[threadIdx.x] = c;
                bkey[threadIdx.x] = bkey[threadIdx.x + stride];
            }
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.x] = best[0];
}

// info[0] = b1 pixel (-1 none), info[1] = b1 item, info[2] = Y1; `cand` holds the B1_BLOCKS
// per-block winners (-1 = none)
__global__ __launch_bounds__(1024) void k_b1_reduce(Dev D, const int32_t* __restrict__ real, const int* __restrict__ cand,
                                                    int* __restrict__ info) {
    __shared__ int best[1024];
    __shared__ ItemKey bkey[1024];
    const int n = B1_BLOCKS;
    int mine = -1;
    for (int k = threadIdx.x; k < n; k += blockDim.x) {
        const int b = cand[k];
        if (b < 0) continue;
        if (mine < 0 || before(D, real[b], real[mine])) mine = b;
    }
    best[threadIdx.x] = mine;
    if (mine >= 0) bkey[threadIdx.x] = item_key(D, real[mine]);
    __syncthreads();
    for (int stride = 512; stride > 0; stride >>= 1) {
        if ((int)threadIdx.x < stride) {
            const int a = best[threadIdx.x], c = best[threadIdx.x + stride];
            if (a < 0 || (c >= 0 && before_keyed(D, bkey[threadIdx.x + stride], bkey[threadIdx.x]))) {
                best[threadIdx.x] = c;
                bkey[threadIdx.x] = bkey[threadIdx.x + stride];
            }
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const int b1 = best[0];
        info[0] = b1;
        info[1] = b1 >= 0 ? real[b1] : -1;
        int lab = 0;
        if (b1 >= 0) lab = b_label(D, b1, real[b1], D.W);
        info[2] = lab;
        // a level-0 b1 could share the level-0 FIFO with other items: outside the decomposition
        if (b1 >= 0 && it_lvl(D, real[b1]) == 0) atomicOr(D.flags, FB_TIES);
    }
}

// queue state at T1 (after b1's pop); P pixels (B, never queued) -> pmask
// Four pixels to a thread, their planes in wide loads, and the two dependent record reads of each pixel's
// place in the pop order (its record, its chain's largest-key item's) side by side; b1's are read once.  An F
// pixel popped before b1 has its label, a B pixel is a dam; one whose pusher popped before b1 is queued
// (an item pops after its pusher, so the second question follows a no to the first).
// Bound by 31 bytes per pixel and those reads; measured, 4098 x 4098: 172 -> 132 us.
__global__ void k_t1_state(Dev D, const int32_t* __restrict__ real, const int* __restrict__ info, uint8_t* __restrict__ pmask,
                           uint8_t* __restrict__ kind) {
    const int b1 = info[0], b1i = info[1], Y1 = info[2];
    ItemKey kb{};
    if (b1 >= 0) kb = item_key(D, b1i);
    const int groups = (D.N + 3) / 4;
    for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < groups; t += gridDim.x * blockDim.x) {
        const int p0 = 4 * t, n = min(4, D.N - p0);
        uint8_t c[4];
        int lab[4], r[4], it[4];
        if (n == 4) {
            const uint32_t c4 = *reinterpret_cast<const u32_any*>(D.cls + p0);
            const i32x4_any l4 = *reinterpret_cast<const i32x4_any*>(D.lab + p0), r4 = *reinterpret_cast<const i32x4_any*>(real + p0);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                c[j] = (uint8_t)(c4 >> (8 * j));
                lab[j] = l4[j];
                r[j] = r4[j];
            }
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int p = p0 + min(j, n - 1);
                c[j] = j < n ? D.cls[p] : (uint8_t)C_FRAME;
                lab[j] = D.lab[p];
                r[j] = real[p];
            }
        }
        int4 rec[4], top[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {  // the pixel's queue entry, -1 for none
            const int p = p0 + j;
            it[j] = c[j] == C_F ? (lab[j] != 0 ? p : -1) : (c[j] == C_B && p != b1 ? r[j] : -1);
            if (it[j] >= 0) rec[j] = D.wr[it[j]];
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (it[j] >= 0) top[j] = D.wr[rec[j].y];
        uint32_t pm = 0, kd = 0;
        int v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            v[j] = c[j] == C_B && p0 + j == b1 ? Y1 : 0;
            if (it[j] >= 0) {
                const ItemKey k{it[j], rec[j].x, rec_pop(D, it[j], rec[j]), rec[j].y, rec_lvl(top[j]), top[j].w};
                if (b1 < 0 || before_keyed(D, k, kb)) v[j] = c[j] == C_F ? lab[j] : WSHED;
                else if (rec[j].w < 0 || before(D, rec[j].w, b1i)) {
                    v[j] = IN_QUEUE;
                    kd |= 1u << (8 * j);
                }
            }
            if (c[j] == C_B && v[j] == 0) pm |= 1u << (8 * j);
        }
        const bool all = (c[0] & 2) && (c[1] & 2) && (c[2] & 2) && (c[3] & 2);  // F or B: the others keep their value
        if (all) *reinterpret_cast<i32x4_any*>(D.m + p0) = i32x4_any{v[0], v[1], v[2], v[3]};
        else {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (c[j] & 2) D.m[p0 + j] = v[j];
        }
        if (n == 4) {
            *reinterpret_cast<u32_any*>(pmask + p0) = pm;
            *reinterpret_cast<u32_any*>(kind + p0) = kd;
        } else {
            for (int j = 0; j < n; ++j) {
                pmask[p0 + j] = (uint8_t)(pm >> (8 * j));
                kind[p0 + j] = (uint8_t)(kd >> (8 * j));
            }
        }
    }
}

// flood from b1: the never-queued B pixels it reaches are exactly those at finite geodesic
// distance from b1 through never-queued B pixels; they take Y1.  An F pixel still unqueued next to
// one of them (or to b1) is queued by that flood (kind 2) from its neighbour nearest to b1: the
// FIFO position of that push is ordered first by this distance (the flood's layer).
__global__ void k_geo_init(Dev D, const int* __restrict__ info, uint8_t* __restrict__ pmask, unsigned* __restrict__ dist) {
    const int b1 = info[0];
    for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < D.N; p += gridDim.x * blockDim.x) {
        const bool src = (p == b1);
        if (src) pmask[p] = 1;
        dist[p] = src ? 0u : 0xFFFFFFFFu;
    }
}
__global__ void k_bfs_mark(Dev D, const int* __restrict__ info, const unsigned* __restrict__ dist, uint8_t* __restrict__ kind,
                           int32_t* __restrict__ pdist) {
    const int b1 = info[0], Y1 = info[2];
    const int W = D.W;
    for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < D.N; p += gridDim.x * blockDim.x) {
        if (b1 < 0 || Y1 <= 0) continue;
        if (D.cls[p] != C_F || D.m[p] != 0) continue;
        const int dirs[4] = {-1, 1, -W, W};
        unsigned best = 0xFFFFFFFFu;
        for (int d = 0; d < 4; ++d) {
            const int s = p + dirs[d];
            if (D.cls[s] == C_B) best = min(best, dist[s]);
        }
        if (best != 0xFFFFFFFFu) { kind[p] = 2; pdist[p] = (int)best; }
    }
}
__global__ void k_bfs_commit(Dev D, const int* __restrict__ info, const unsigned* __restrict__ dist, const uint8_t* __restrict__ kind,
                             uint8_t* __restrict__ umask) {
    const int b1 = info[0], Y1 = info[2];
    for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < D.N; p += gridDim.x * blockDim.x) {
        // the four loads first (under the conditions they would wait for one another)
        const int m0 = D.m[p];
        const uint8_t c = D.cls[p], kd = kind[p];
        const unsigned dp = dist[p];
        int v = m0;
        if (b1 >= 0 && Y1 > 0 && c == C_B && v == 0 && dp != 0xFFFFFFFFu) v = Y1;
        if (kd == 2) v = IN_QUEUE;
        if (v != m0) D.m[p] = v;
        umask[p] = (c != C_FRAME && c != C_SEED && (v == 0 || v == IN_QUEUE)) ? 1 : 0;
    }
}

// ---- phase 2: one lane floods one component of unresolved pixels ----
struct P2 {
    const int32_t* comp;
    const int32_t* box5;
    const int32_t* area;
    const int32_t* off;
    const uint8_t* kind;
    int32_t* scratch;  // 3 * area per component: item list, heap, saved labels
    int ncomp;
};

// Order of two queued items of the same level by push time: phase-1 items by pusher order, items
// queued by the flood from b1 after them (their mutual order is not known: they are ordered by the
// b1 flood's layer, then in raster order, and the caller checks that the order does not matter).
// The data this reads of one item is packed once, so that a sort compares cached values:
// bit 63 = queued by the b1 flood (kind 2); then, for kind 2, its label (the layer) in the low 32
// bits; else (pusher + 1) in bits 32..62 and the pusher's direction (its push order) in the low 32 bits.
__device__ __forceinline__ long long push_data(int a, int pa) {
    const int d = a - pa;
    const uint32_t dir = d == -1 ? 0 : (d == 1 ? 1 : (d < 0 ? 2 : 3));  // pushes go left, right, up, down
    return ((long long)(uint32_t)(pa + 1) << 32) | (long long)dir;
}
__device__ long long push_key(const Dev& D, const int32_t* real, const uint8_t* kind, int a) {
    if (kind[a] == 2) return (long long)(1ull << 63) | (long long)(uint32_t)D.lab[a];
    const int ia = D.cls[a] == C_B ? real[a] : a;
    return push_data(a, it_parent(D, ia));
}
// a pushed before b, from their packed data
__device__ bool push_before_key(const Dev& D, const int32_t* real, int a, long long ka, int b, long long kb) {
    const bool ba = ka < 0, bb = kb < 0;
    if (ba != bb) return bb;
    if (ba) {
        const int la = (int)(uint32_t)ka, lb = (int)(uint32_t)kb;
        if (la != lb) return la < lb;
        return a < b;
    }
    const int pa = (int)((ka >> 32) & 0x7FFFFFFF) - 1, pb = (int)((kb >> 32) & 0x7FFFFFFF) - 1;
    if (pa < 0 && pb < 0) {
        const int ia = D.cls[a] == C_B ? real[a] : a;
        const int ib = D.cls[b] == C_B ? real[b] : b;
        return ia < ib;
    }
    if (pa < 0) return true;
    if (pb < 0) return false;
    if (pa == pb) return (int)(uint32_t)ka < (int)(uint32_t)kb;
    return before(D, pa, pb);
}

__device__ int item_level(const Dev& D, const int32_t* real, const uint8_t* kind, int p) {
    if (kind[p] == 2) {
        const uint8_t* c = D.img + 3 * (size_t)p;
        return max(max((int)c[0], (int)c[1]), (int)c[2]);
    }
    return it_lvl(D, D.cls[p] == C_B ? real[p] : p);
}

// binary heap on (level << 24 | seq) packed keys, values = pixel ids
__device__ __forceinline__ void heap_push(long long* hk, int* hv, int& n, long long k, int v) {
    int i = n++;
    while (i > 0) {
        const int pi = (i - 1) >> 1;
        if (hk[pi] <= k) break;
        hk[i] = hk[pi]; hv[i] = hv[pi]; i = pi;
    }
    hk[i] = k; hv[i] = v;
}
__device__ __forceinline__ int heap_pop(long long* hk, int* hv, int& n) {
    const int top = hv[0];
    const long long k = hk[--n];
    const int v = hv[n];
    int i = 0;
    while (true) {
        int c = 2 * i + 1;
        if (c >= n) break;
        if (c + 1 < n && hk[c + 1] < hk[c]) ++c;
        if (hk[c] >= k) break;
        hk[i] = hk[c]; hv[i] = hv[c]; i = c;
    }
    if (n > 0) { hk[i] = k; hv[i] = v; }
    return top;
}

constexpr int MAXG = 8, MAXGL = 5, MAXCOMBO = 4096;
struct TieRec {
    int c, ni, ntie, ncombo;
    long long base;  // offset (ints) of the record's region in the tie pool
    int gfirst[MAXG], glen[MAXG];
};

__device__ __forceinline__ int fact(int n) { int f = 1; for (int k = 2; k <= n; ++k) f *= k; return f; }

// flood one component from its sorted queue `order` (ni items); the state of the component's
// pixels lives either in D.m (st == nullptr) or in a private bbox-indexed array st.  Returns
// false on heap overflow.
__device__ bool flood_component(const Dev& D, const P2& Q, int c, const int* order, int ni, int* st, int* hv,
                                long long* hk, int A, const int32_t* real) {
    const int W = D.W, id = c + 1;
    const int minx = Q.box5[Q.ncomp + c], maxx = Q.box5[2 * Q.ncomp + c];
    const int miny = Q.box5[3 * Q.ncomp + c];
    const int bw = maxx - minx + 1;
    auto loc = [&](int i) -> int* {  // private cell of a component pixel, nullptr otherwise
        if (!st) return nullptr;
        const int x = i % W, y = i / W;
        if (x < minx || x > maxx || y < miny || Q.comp[i] != id) return nullptr;
        return st + (y - miny) * bw + (x - minx);
    };
    auto get = [&](int i) { int* q = loc(i); return q ? *q : D.m[i]; };
    auto put = [&](int i, int v) { int* q = loc(i); if (q) *q = v; else D.m[i] = v; };
    const int dirs[4] = {-1, 1, -W, W};
    int hn = 0;
    long long seqc = 0;
    for (int k = 0; k < ni; ++k)
        heap_push(hk, hv, hn, ((long long)item_level(D, real, Q.kind, order[k]) << 40) | (seqc++), order[k]);
    while (hn > 0) {
        const int p = heap_pop(hk, hv, hn);
        int lab = 0;
        for (int d = 0; d < 4; ++d) {
            const int t = get(p + dirs[d]);
            if (t > 0) { if (lab == 0) lab = t; else if (t != lab) lab = WSHED; }
        }
        put(p, lab);
        if (lab == WSHED) continue;
        const uint8_t* ptr = D.img + 3 * (size_t)p;
        for (int d = 0; d < 4; ++d) {
            const int s2 = p + dirs[d];
            if (get(s2) == 0) {
                if (hn >= A) return false;
                const int l = c_diff(ptr, D.img + 3 * (size_t)s2);
                heap_push(hk, hv, hn, ((long long)l << 40) | (seqc++), s2);
                put(s2, IN_QUEUE);
            }
        }
    }
    return true;
}

// components deferred to the LDS flood: a record per component, a work item per (record, arrangement)
constexpr int FL_SMALL = 1024, FL_BIG = 4096;  // frame pixels (box + 1-pixel margin) of the two LDS tiers
constexpr int FL_MIN_AREA = 24;                // smaller tie-free components flood in their lane
struct FloodQ {
    TieRec* recs;
    int* nrec;
    int reccap;
    int* work[2];
    int* nwork;  // [2]
    int workcap;
    int* res;    // per-arrangement results of tie components (pool)
    int* recbad;  // per record: some arrangement differs from arrangement 0
};

// boxes larger than this are scanned by the whole wave (64 pixels a step) instead of one lane, and
// item lists longer than P2_COOP_SORT (up to 64 * P2_SORT_PER) are sorted by the whole wave
constexpr int P2_COOP_BOX = 512, P2_COOP_SORT = 16, P2_SORT_PER = 8;

// A component's queue in LDS, the lane's column of 64: items, their levels (then heap keys) and push keys.
// Nearly all components have at most FL_MIN_AREA pixels; their lists, sort and flood stay here, and a pop
// reads its neighbours' states and colours from memory in one round trip.  With the lists and the heap in
// memory every step of the sort and of the heap was a round trip of its own.
// Measured, 512 x 512 and 4096 x 4096 chain: 88 -> 70 and 183 -> 163 us.
struct LaneQueue {
    int item[FL_MIN_AREA][64];
    uint32_t lvl[FL_MIN_AREA][64];
    long long key[P2_COOP_SORT][64];
};

// levels and push data (see push_key) of the lane's n items, four items' loads at a time
__device__ __forceinline__ void lane_keys(const Dev& D, const int32_t* real, const uint8_t* kind, LaneQueue& q, int lane, int n) {
    for (int a0 = 0; a0 < n; a0 += 4) {
        int v[4], ia[4], lab[4];
        uint8_t kd[4], c[4], col[4][3];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            v[j] = q.item[min(a0 + j, n - 1)][lane];
            kd[j] = kind[v[j]];
            c[j] = D.cls[v[j]];
            ia[j] = real[v[j]];
            lab[j] = D.lab[v[j]];
#pragma unroll
            for (int ch = 0; ch < 3; ++ch) col[j][ch] = D.img[3 * (size_t)v[j] + ch];
        }
        int4 rec[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (kd[j] != 2) rec[j] = D.wr[c[j] == C_B ? ia[j] : v[j]];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (a0 + j >= n) break;
            if (kd[j] == 2) {
                q.lvl[a0 + j][lane] = (uint32_t)max(max((int)col[j][0], (int)col[j][1]), (int)col[j][2]);
                q.key[a0 + j][lane] = (long long)(1ull << 63) | (long long)(uint32_t)lab[j];
            } else {
                q.lvl[a0 + j][lane] = (uint32_t)rec_lvl(rec[j]);
                q.key[a0 + j][lane] = push_data(v[j], rec[j].w);
            }
        }
    }
}

// flood_component of a component whose sorted queue (n items) is the lane's
__device__ __forceinline__ bool flood_lane(const Dev& D, LaneQueue& q, int lane, int n, int A) {
    const int dirs[4] = {-1, 1, -D.W, D.W};
    for (int a = 0; a < n; ++a) q.lvl[a][lane] = q.lvl[a][lane] << 16 | (uint32_t)a;  // a sorted list is a heap
    uint32_t seq = (uint32_t)n;
    while (n > 0) {
        const int p = q.item[0][lane];
        int t[4];
        uint32_t col[4];
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            t[d] = D.m[p + dirs[d]];
            col[d] = colour1(D.img + 3 * (size_t)(p + dirs[d]));
        }
        const uint32_t own = colour1(D.img + 3 * (size_t)p);
        {  // the last item sinks from the top
            --n;
            const uint32_t k = q.lvl[n][lane];
            const int v = q.item[n][lane];
            int i = 0;
            for (int c = 1; c < n; c = 2 * i + 1) {
                uint32_t kc = q.lvl[c][lane];
                if (c + 1 < n && q.lvl[c + 1][lane] < kc) kc = q.lvl[++c][lane];
                if (kc >= k) break;
                q.lvl[i][lane] = kc;
                q.item[i][lane] = q.item[c][lane];
                i = c;
            }
            q.lvl[i][lane] = k;
            q.item[i][lane] = v;
        }
        const int lab = pop_label(t[0], t[1], t[2], t[3]);
        D.m[p] = lab;
        if (lab == WSHED) continue;
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            if (t[d] != 0) continue;
            if (n >= A) return false;
            const uint32_t k = (uint32_t)cdiff_packed(own, col[d]) << 16 | seq++;
            int i = n++;
            while (i > 0) {
                const int up = (i - 1) >> 1;
                const uint32_t ku = q.lvl[up][lane];
                if (ku <= k) break;
                q.lvl[i][lane] = ku;
                q.item[i][lane] = q.item[up][lane];
                i = up;
            }
            q.lvl[i][lane] = k;
            q.item[i][lane] = p + dirs[d];
            D.m[p + dirs[d]] = IN_QUEUE;
        }
    }
    return true;
}

// One lane per component; launched with 64-thread blocks (one wave), which the cooperative scan of
// large boxes relies on.
__global__ __launch_bounds__(64) void k_phase2(Dev D, P2 Q, const int32_t* __restrict__ real, long long* __restrict__ heapk, TieRec* ties,
                         int* nties, int tiecap, long long* pool_used, long long poolcap, FloodQ F) {
    __shared__ LaneQueue LQ;
    const int lane = threadIdx.x & 63;
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    const bool valid = c < Q.ncomp;
    const int W = D.W;
    const int id = c + 1;
    const int cc = valid ? c : 0;  // a valid index for the loads of lanes without a component
    const int A = Q.area[cc];
    int32_t* items = Q.scratch + 3 * (size_t)Q.off[cc];
    int* hv = items + A;
    long long* hk = heapk + (size_t)Q.off[cc];
    const int minx = Q.box5[Q.ncomp + cc], maxx = Q.box5[2 * Q.ncomp + cc];
    const int miny = Q.box5[3 * Q.ncomp + cc], maxy = Q.box5[4 * Q.ncomp + cc];
    const int bw = maxx - minx + 1, B = bw * (maxy - miny + 1);
    // collect queued items (raster order).  Boxes above P2_COOP_BOX pixels: the wave scans each
    // such box in turn, 64 box pixels a step, and compacts the hits with a ballot (a lane alone
    // would wait on one memory round trip per eight pixels of a box of up to thousands).
    int ni = 0;
    const bool coop = valid && B > P2_COOP_BOX;
    unsigned long long pend = __ballot(coop);
    while (pend) {
        const int src = __ffsll((long long)pend) - 1;
        pend &= pend - 1;
        const int sc = __shfl(c, src), sminx = __shfl(minx, src), sminy = __shfl(miny, src);
        const int sbw = __shfl(bw, src), sB = __shfl(B, src);
        int32_t* sitems = Q.scratch + 3 * (size_t)Q.off[sc];
        int cnt = 0;
        for (int k0 = 0; k0 < sB; k0 += 64) {
            const int k = k0 + lane;
            bool take = false;
            int gi = 0;
            if (k < sB) {
                gi = (sminy + k / sbw) * W + sminx + k % sbw;
                take = Q.comp[gi] == sc + 1 && D.m[gi] == IN_QUEUE;
            }
            const unsigned long long tb = __ballot(take);
            if (take) sitems[cnt + __popcll(tb & ((1ull << lane) - 1ull))] = gi;
            cnt += __popcll(tb);
        }
        if (lane == src) ni = cnt;
    }
    const bool small = valid && !coop && A <= FL_MIN_AREA;  // (at most A items)
    // smaller boxes: the lane scans its own, eight pixels' loads in flight at a time (a load per
    // pixel with its test in the same iteration waits on every pixel in turn)
    if (valid && !coop)
        for (int y = miny; y <= maxy; ++y)
            for (int x0 = minx; x0 <= maxx; x0 += 8) {
                int cv[8], mv[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const int i = y * W + min(x0 + j, maxx);
                    cv[j] = Q.comp[i];
                    mv[j] = D.m[i];
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    if (x0 + j <= maxx && cv[j] == id && mv[j] == IN_QUEUE) {
                        if (small) LQ.item[ni++][lane] = y * W + x0 + j;
                        else items[ni++] = y * W + x0 + j;
                    }
            }
    const bool inlds = small && ni <= P2_COOP_SORT;
    if (small && !inlds)
        for (int a = 0; a < ni; ++a) items[a] = LQ.item[a][lane];
    // Sort by (level, push time): the FIFO pop order, a strict total order.  Each item's level and
    // push data are computed once (into hv[] and hk[], free until the flood below, and ni <= A)
    // and move with the item.  Few items: the lane's own insertion sort.  More (the components of
    // the LDS floods, up to ~100 items): the wave ranks each item by counting the items that
    // precede it (one item per lane, all compared at once) and scatters the items to their ranks
    // -- the same order, without one lane's ~n^2/2 dependent comparisons.
    const bool coopsort = valid && ni > P2_COOP_SORT && ni <= 64 * P2_SORT_PER;
    if (inlds) {
        lane_keys(D, real, Q.kind, LQ, lane, ni);
        for (int a = 1; a < ni; ++a) {
            const int v = LQ.item[a][lane];
            const uint32_t lv = LQ.lvl[a][lane];
            const long long kv = LQ.key[a][lane];
            int b = a - 1;
            for (; b >= 0; --b) {
                const int u = LQ.item[b][lane];
                const uint32_t lu = LQ.lvl[b][lane];
                const long long ku = LQ.key[b][lane];
                if (!(lu > lv || (lu == lv && push_before_key(D, real, v, kv, u, ku)))) break;
                LQ.item[b + 1][lane] = u;
                LQ.lvl[b + 1][lane] = lu;
                LQ.key[b + 1][lane] = ku;
            }
            LQ.item[b + 1][lane] = v;
            LQ.lvl[b + 1][lane] = lv;
            LQ.key[b + 1][lane] = kv;
        }
    } else if (valid && !coopsort) {
        for (int a = 0; a < ni; ++a) {
            const int v = items[a];
            hv[a] = item_level(D, real, Q.kind, v);
            hk[a] = push_key(D, real, Q.kind, v);
        }
        for (int a = 1; a < ni; ++a) {
            const int v = items[a], lv = hv[a];
            const long long kv = hk[a];
            int b = a - 1;
            while (b >= 0) {
                const int u = items[b], lu = hv[b];
                const long long ku = hk[b];
                const bool gt = (lu > lv) || (lu == lv && push_before_key(D, real, v, kv, u, ku));
                if (!gt) break;
                items[b + 1] = u;
                hv[b + 1] = lu;
                hk[b + 1] = ku;
                --b;
            }
            items[b + 1] = v;
            hv[b + 1] = lv;
            hk[b + 1] = kv;
        }
    }
    __syncthreads();  // every item list (stored by every lane in the scans) is complete
    unsigned long long pend_sort = __ballot(coopsort);
    while (pend_sort) {
        const int src = __ffsll((long long)pend_sort) - 1;
        pend_sort &= pend_sort - 1;
        const int sc = __shfl(c, src), sni = __shfl(ni, src), sA = __shfl(A, src);
        int32_t* sitems = Q.scratch + 3 * (size_t)Q.off[sc];
        int* shv = sitems + sA;
        long long* shk = heapk + (size_t)Q.off[sc];
        for (int k = lane; k < sni; k += 64) {
            const int v = sitems[k];
            shv[k] = item_level(D, real, Q.kind, v);
            shk[k] = push_key(D, real, Q.kind, v);
        }
        __syncthreads();
        int rk[P2_SORT_PER], vv[P2_SORT_PER], lvv[P2_SORT_PER];
        long long kvv[P2_SORT_PER];
#pragma unroll
        for (int q = 0; q < P2_SORT_PER; ++q) {
            const int k = lane + 64 * q;
            rk[q] = -1;
            if (k >= sni) continue;
            const int v = sitems[k], lv = shv[k];
            const long long kv = shk[k];
            int rank = 0;
            for (int j = 0; j < sni; ++j) {
                if (j == k) continue;
                const int u = sitems[j], lu = shv[j];
                rank += (lu < lv) || (lu == lv && push_before_key(D, real, u, shk[j], v, kv)) ? 1 : 0;
            }
            rk[q] = rank;
            vv[q] = v;
            lvv[q] = lv;
            kvv[q] = kv;
        }
        __syncthreads();  // every comparison has read the lists before they are overwritten
#pragma unroll
        for (int q = 0; q < P2_SORT_PER; ++q) {
            if (rk[q] < 0) continue;
            sitems[rk[q]] = vv[q];
            shv[rk[q]] = lvv[q];
            shk[rk[q]] = kvv[q];
        }
        __syncthreads();  // the sorted list is complete before its owner reads it
    }
    if (!valid) return;
    // groups of items queued by the b1 flood at the same level and layer: order unknown
    TieRec R;
    R.c = c; R.ni = ni; R.ntie = 0;
    long long ncombo = 1;
    for (int a = 0; a < ni;) {
        int e = a + 1;
        if (inlds) {  // (the push data of an item queued by that flood is its layer)
            const long long kv = LQ.key[a][lane];
            if (kv >= 0) { ++a; continue; }
            while (e < ni && LQ.key[e][lane] == kv && LQ.lvl[e][lane] == LQ.lvl[a][lane]) ++e;
        } else {
            const int v = items[a];
            if (Q.kind[v] != 2) { ++a; continue; }
            const int lv = hv[a];  // cached levels, aligned with the sorted items
            while (e < ni && Q.kind[items[e]] == 2 && hv[e] == lv && D.lab[items[e]] == D.lab[v]) ++e;
        }
        if (e - a >= 2) {
            if (R.ntie == MAXG || e - a > MAXGL) { atomicOr(D.flags, FB_TIES); return; }
            R.gfirst[R.ntie] = a;
            R.glen[R.ntie] = e - a;
            ++R.ntie;
            ncombo *= fact(e - a);
            if (ncombo > MAXCOMBO) { atomicOr(D.flags, FB_TIES); return; }
        }
        a = e;
    }
    R.ncombo = (int)ncombo;
    if (inlds && R.ntie == 0) {
        if (!flood_lane(D, LQ, lane, ni, A)) atomicOr(D.flags, FB_HEAP);
        return;
    }
    if (inlds)  // the list, for the flood of its arrangements
        for (int a = 0; a < ni; ++a) items[a] = LQ.item[a][lane];
    const int L = (maxx - minx + 3) * (maxy - miny + 3);
    if (L <= FL_BIG && (R.ntie > 0 || A > FL_MIN_AREA)) {  // LDS flood, one wave per arrangement
        long long base = 0;
        if (ncombo > 1) {
            const long long need = ncombo * (long long)L;
            base = atomicAdd((unsigned long long*)pool_used, (unsigned long long)need);
            if (base + need > poolcap) { atomicOr(D.flags, FB_TIES); return; }
        }
        R.base = base;
        const int rec = atomicAdd(F.nrec, 1);
        if (rec >= F.reccap) { atomicOr(D.flags, FB_TIES); return; }
        F.recs[rec] = R;
        const int tier = L <= FL_SMALL ? 0 : 1;
        const int w0 = atomicAdd(&F.nwork[tier], (int)ncombo);
        if (w0 + ncombo > F.workcap) { atomicOr(D.flags, FB_TIES); return; }
        for (int k = 0; k < (int)ncombo; ++k) F.work[tier][w0 + k] = rec * MAXCOMBO + k;
        return;
    }
    if (R.ntie == 0) {
        if (!flood_component(D, Q, c, items, ni, nullptr, hv, hk, A, real)) atomicOr(D.flags, FB_HEAP);
        return;
    }
    // defer to the parallel permutation check (one wave per component)
    const long long per = (long long)B + ni + A + 2LL * A + 4;  // B: box pixels
    const long long need = 64 * per + B + 64;
    const long long base = atomicAdd((unsigned long long*)pool_used, (unsigned long long)need);
    const int k = atomicAdd(nties, 1);
    if (k >= tiecap) { atomicOr(D.flags, FB_TIES); return; }
    if (base + need > poolcap) {  // slot taken but no room: leave an empty record
        atomicOr(D.flags, FB_TIES);
        R.c = -1;
    }
    R.base = base;
    ties[k] = R;
}

// one wave per deferred component: lane t floods the arrangements t, t+64, ... of the tie groups
// on a private copy; every result must equal arrangement 0, which is then committed
__global__ __launch_bounds__(64) void k_phase2_ties(Dev D, P2 Q, const int32_t* __restrict__ real, const TieRec* __restrict__ ties,
                                                   const int* __restrict__ nties, int* pool) {
    const int k = blockIdx.x;
    if (k >= min(*nties, (int)gridDim.x)) return;
    const TieRec R = ties[k];
    if (R.c < 0) return;
    const int c = R.c, id = c + 1, W = D.W, lane = threadIdx.x;
    const int A = Q.area[c];
    const int minx = Q.box5[Q.ncomp + c], maxx = Q.box5[2 * Q.ncomp + c];
    const int miny = Q.box5[3 * Q.ncomp + c], maxy = Q.box5[4 * Q.ncomp + c];
    const int bw = maxx - minx + 1, bh = maxy - miny + 1, B = bw * bh;
    const int ni = R.ni;
    const int32_t* items = Q.scratch + 3 * (size_t)Q.off[c];
    const long long per = (long long)B + ni + A + 2LL * A + 4;
    int* mine = pool + R.base + lane * per;
    int* st = mine;
    int* order = st + B;
    int* hv = order + ni;
    long long* hk = reinterpret_cast<long long*>(hv + A + ((reinterpret_cast<uintptr_t>(hv + A) & 7) ? 1 : 0));
    int* canon = pool + R.base + 64 * per;
    __shared__ int bad;
    if (lane == 0) bad = 0;
    __syncthreads();
    const int rounds = (R.ncombo + 63) / 64;
    for (int r = 0; r < rounds; ++r) {
        const int combo = r * 64 + lane;
        const bool act = combo < R.ncombo;
        if (act) {
            for (int q = 0; q < ni; ++q) order[q] = items[q];
            int code = combo;
            for (int g = 0; g < R.ntie; ++g) {  // arrangement = factorial-base digits per group
                const int L = R.glen[g];
                const int f = fact(L);
                int digit = code % f;
                code /= f;
                int pool_el[MAXGL];
                for (int q = 0; q < L; ++q) pool_el[q] = items[R.gfirst[g] + q];
                for (int q = 0; q < L; ++q) {
                    const int fq = fact(L - 1 - q);
                    const int idx = digit / fq;
                    digit %= fq;
                    order[R.gfirst[g] + q] = pool_el[idx];
                    for (int z = idx; z < L - 1 - q; ++z) pool_el[z] = pool_el[z + 1];
                }
            }
            for (int y = 0; y < bh; ++y)
                for (int x = 0; x < bw; ++x) st[y * bw + x] = 0;
            for (int q = 0; q < ni; ++q) {
                const int i = items[q];
                st[(i / W - miny) * bw + (i % W - minx)] = IN_QUEUE;
            }
            if (!flood_component(D, Q, c, order, ni, st, hv, hk, A, real)) atomicOr(&bad, 1);
        }
        if (r == 0) {
            if (lane == 0)
                for (int q = 0; q < B; ++q) canon[q] = st[q];
            __syncthreads();
        }
        if (act) {
            for (int y = 0; y < bh; ++y)
                for (int x = 0; x < bw; ++x) {
                    const int i = (miny + y) * W + (minx + x);
                    if (Q.comp[i] == id && st[y * bw + x] != canon[y * bw + x]) atomicOr(&bad, 1);
                }
        }
    }
    __syncthreads();
    if (lane == 0) {
        if (bad) { atomicOr(D.flags, FB_TIEPERM); return; }
        for (int y = 0; y < bh; ++y)
            for (int x = 0; x < bw; ++x) {
                const int i = (miny + y) * W + (minx + x);
                if (Q.comp[i] == id) D.m[i] = canon[y * bw + x];
            }
    }
}

// one wave floods one arrangement of one deferred component with its frame (box + 1-pixel
// margin) in LDS: the same flood as flood_component (lowest level first, FIFO within a level,
// neighbours in the order left, right, up, down), lane 0 driving it
template <int LCAP>
__global__ __launch_bounds__(64) void k_flood_lds(Dev D, P2 Q, const int32_t* __restrict__ real, FloodQ F, int tier) {
    __shared__ int32_t st[LCAP];
    __shared__ uint32_t col[LCAP];
    __shared__ uint16_t qn[LCAP];
    __shared__ uint8_t inc[LCAP];
    __shared__ uint16_t ord[LCAP];
    __shared__ uint8_t olv[LCAP];
    __shared__ uint16_t qhead[NQ], qtail[NQ];
    __shared__ int bad;
    const int nw = min(F.nwork[tier], F.workcap);
    for (int wi = blockIdx.x; wi < nw; wi += gridDim.x) {
    const int w = F.work[tier][wi];
    const TieRec R = F.recs[w / MAXCOMBO];
    const int combo = w % MAXCOMBO;
    const int c = R.c, id = c + 1, W = D.W, lane = threadIdx.x;
    const int ox = Q.box5[Q.ncomp + c] - 1, oy = Q.box5[3 * Q.ncomp + c] - 1;
    const int lw = Q.box5[2 * Q.ncomp + c] - ox + 2, lh = Q.box5[4 * Q.ncomp + c] - oy + 2;
    const int L = lw * lh;  // <= LCAP; the frame lies inside the image (components avoid the frame)
    const int ni = R.ni;
    const int32_t* items = Q.scratch + 3 * (size_t)Q.off[c];
    auto gidx = [&](int k) { return (oy + k / lw) * W + ox + k % lw; };
    if (lane == 0) bad = 0;
    for (int k = lane; k < L; k += 64) {
        const int g = gidx(k);
        inc[k] = Q.comp[g] == id ? 1 : 0;
        st[k] = D.m[g];
        const uint8_t* q = D.img + 3 * (size_t)g;
        col[k] = (uint32_t)q[0] | ((uint32_t)q[1] << 8) | ((uint32_t)q[2] << 16);
    }
    for (int l = lane; l < NQ; l += 64) { qhead[l] = NIL16; qtail[l] = NIL16; }
    for (int q = lane; q < ni; q += 64) {
        const int v = items[q];
        ord[q] = (uint16_t)((v / W - oy) * lw + (v % W - ox));
        olv[q] = (uint8_t)item_level(D, real, Q.kind, v);
    }
    __syncthreads();
    if (lane == 0) {
        // arrangement `combo`: factorial-base digits, one per tie group (members share their level)
        int code = combo;
        for (int g = 0; g < R.ntie; ++g) {
            const int Lg = R.glen[g], f0 = R.gfirst[g];
            const int f = fact(Lg);
            int digit = code % f;
            code /= f;
            uint16_t pool_el[MAXGL];
            for (int q = 0; q < Lg; ++q) pool_el[q] = ord[f0 + q];
            for (int q = 0; q < Lg; ++q) {
                const int fq = fact(Lg - 1 - q);
                const int idx = digit / fq;
                digit %= fq;
                ord[f0 + q] = pool_el[idx];
                for (int z = idx; z < Lg - 1 - q; ++z) pool_el[z] = pool_el[z + 1];
            }
        }
        int active = NQ;
        int hx = NIL16;  // head of the active level's FIFO (a copy of qhead[active])
        auto enq = [&](int l, int x) {
            qn[x] = NIL16;
            const uint32_t t = uni(qtail[l]);
            if (t != NIL16) qn[t] = (uint16_t)x;
            else qhead[l] = (uint16_t)x;
            qtail[l] = (uint16_t)x;
            if (t == NIL16 && l <= active) {  // nothing is queued below `active`: l was empty
                active = l;
                hx = x;
            }
        };
        for (int q = 0; q < ni; ++q) enq(olv[q], ord[q]);
        const int ld[4] = {-1, 1, -lw, lw};
        for (;;) {
            int p = hx;
            if (p == NIL16) {
                int l = active + 1;
                while (l < NQ && uni(qhead[l]) == NIL16) ++l;
                if (l >= NQ) break;
                active = l;
                p = uni(qhead[l]);
            }
            // everything the pop reads, in one round trip (this pop's own writes go to p and to
            // distinct neighbours, so the values stay current for its pushes)
            uint32_t nx = qn[p], cp = col[p];
            int ns[4];
            uint32_t ninc[4], ncol[4];
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                ns[d] = st[p + ld[d]];
                ninc[d] = inc[p + ld[d]];
                ncol[d] = col[p + ld[d]];
            }
            asm volatile("" : "+v"(nx), "+v"(cp), "+v"(ns[0]), "+v"(ns[1]), "+v"(ns[2]), "+v"(ns[3]), "+v"(ninc[0]),
                         "+v"(ninc[1]), "+v"(ninc[2]), "+v"(ninc[3]), "+v"(ncol[0]), "+v"(ncol[1]), "+v"(ncol[2]),
                         "+v"(ncol[3]));
            // one lane floods: the values are the wave's, kept in scalar registers
            nx = uni(nx);
            cp = uni(cp);
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                ns[d] = uni(ns[d]);
                ninc[d] = uni(ninc[d]);
                ncol[d] = uni(ncol[d]);
            }
            qhead[active] = (uint16_t)nx;
            hx = (int)nx;
            if (nx == NIL16) qtail[active] = NIL16;
            const int lab = pop_label(ns[0], ns[1], ns[2], ns[3]);
            st[p] = lab;
            if (lab == WSHED) continue;
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                const int s2 = p + ld[d];
                if (ns[d] != 0) continue;
                if (!ninc[d]) { bad = 1; continue; }  // an unresolved pixel outside the component
                st[s2] = IN_QUEUE;
                enq(cdiff_packed(cp, ncol[d]), s2);
            }
        }
        if (bad) atomicOr(D.flags, FB_HEAP);
    }
    __syncthreads();
    if (R.ncombo == 1) {
        for (int k = lane; k < L; k += 64)
            if (inc[k]) D.m[gidx(k)] = st[k];
    } else {
        int* out = F.res + R.base + (long long)combo * L;
        for (int k = lane; k < L; k += 64) out[k] = st[k];
    }
    __syncthreads();  // the LDS frame is reused by the next work item
    }
}

// Tie components flooded in LDS: every arrangement must give arrangement 0's labels, which are then
// committed.  The comparison takes one workgroup per (record, arrangement) work item, across the
// device (a workgroup per record would read every arrangement of a record through one CU).
__global__ __launch_bounds__(256) void k_tie_check(P2 Q, FloodQ F, int W) {
    const int n0 = min(F.nwork[0], F.workcap), n1 = min(F.nwork[1], F.workcap);
    for (int t = blockIdx.x; t < n0 + n1; t += gridDim.x) {
        const int w = t < n0 ? F.work[0][t] : F.work[1][t - n0];
        const int ri = w / MAXCOMBO, combo = w % MAXCOMBO;
        const TieRec R = F.recs[ri];
        if (R.ncombo == 1 || combo == 0) continue;
        const int c = R.c, id = c + 1;
        const int ox = Q.box5[Q.ncomp + c] - 1, oy = Q.box5[3 * Q.ncomp + c] - 1;
        const int lw = Q.box5[2 * Q.ncomp + c] - ox + 2, lh = Q.box5[4 * Q.ncomp + c] - oy + 2;
        const int L = lw * lh;
        const int* res = F.res + R.base;
        bool diff = false;
        for (int k = threadIdx.x; k < L; k += blockDim.x) {
            const int g = (oy + k / lw) * W + ox + k % lw;
            if (Q.comp[g] == id && res[(long long)combo * L + k] != res[k]) diff = true;
        }
        if (diff) atomicOr(&F.recbad[ri], 1);
    }
}

__global__ __launch_bounds__(256) void k_tie_commit(Dev D, P2 Q, FloodQ F) {
    const int nr = min(*F.nrec, F.reccap);
    for (int ri = blockIdx.x; ri < nr; ri += gridDim.x) {
        const TieRec R = F.recs[ri];
        if (R.ncombo == 1) continue;
        if (F.recbad[ri]) {
            if (threadIdx.x == 0) atomicOr(D.flags, FB_TIEPERM);
            continue;
        }
        const int c = R.c, id = c + 1, W = D.W;
        const int ox = Q.box5[Q.ncomp + c] - 1, oy = Q.box5[3 * Q.ncomp + c] - 1;
        const int lw = Q.box5[2 * Q.ncomp + c] - ox + 2, lh = Q.box5[4 * Q.ncomp + c] - oy + 2;
        const int L = lw * lh;
        const int* res = F.res + R.base;
        for (int k = threadIdx.x; k < L; k += blockDim.x) {
            const int g = (oy + k / lw) * W + ox + k % lw;
            if (Q.comp[g] == id) D.m[g] = res[k];
        }
    }
}

inline dim3 grid1(size_t n) { return dim3(std::min<unsigned>(cdiv(n, 256), 8192u)); }

}  // namespace

// Returns NSC_OK with *ok = 1 when the decomposition produced the exact result in m, *ok = 0
// when the caller must run the sequential flood instead (m is then undefined).
void ws_last_flags_record(int flags);
void ws_tier_record(const int* runs, int ntiers);

int geodist_impl(const uint8_t* pass, unsigned* dist, int w, int h, hipStream_t s, const int* seed);

int cvws_fast(const uint8_t* img, const int32_t* m0, int32_t* m, int W, int H, int* ok, hipStream_t s) {
    const size_t N = (size_t)W * H;
    const bool dbg = getenv("NSC_WS_DEBUG") != nullptr;
    hipEvent_t ev0 = nullptr;
    auto tick = [&](const char* what, const int* dcount) {
        if (!dbg) return;
        hipEvent_t e;
        (void)hipEventCreate(&e);
        (void)hipEventRecord(e, s);
        (void)hipEventSynchronize(e);
        float ms = 0.f;
        if (ev0) (void)hipEventElapsedTime(&ms, ev0, e);
        int c = -1;
        if (dcount) (void)hipMemcpy(&c, dcount, sizeof(int), hipMemcpyDeviceToHost);
        fprintf(stderr, "[ws] %-12s %8.3f ms  count %d\n", what, ms, c);
        if (ev0) (void)hipEventDestroy(ev0);
        ev0 = e;
    };
    tick("start", nullptr);
    *ok = 0;
    if (N >= (size_t)INT_MAX / 8) return NSC_OK;
    Carver measure(nullptr);
    auto carve = [&](Carver& c, uint8_t*& cls, uint16_t*& lvl0, uint8_t*& fmask, int32_t*& run, int32_t*& lab, int32_t*& head,
                     int32_t*& real, int32_t*& lab2, uint8_t*& kind, int*& small) {
        cls = c.take<uint8_t>(N);
        lvl0 = c.take<uint16_t>(N);
        fmask = c.take<uint8_t>(N);
        run = c.take<int32_t>(N);
        lab = c.take<int32_t>(N);
        head = c.take<int32_t>(N);
        real = c.take<int32_t>(N);
        lab2 = c.take<int32_t>(N);
        kind = c.take<uint8_t>(N);
        small = c.take<int>(64 + B1_BLOCKS);  // counters, then the per-block b1 winners
    };
    uint8_t *cls, *fmask, *kind;
    uint16_t* lvl0;
    int32_t *run, *lab, *head, *real, *lab2;
    int* small;
    carve(measure, cls, lvl0, fmask, run, lab, head, real, lab2, kind, small);
    Scratch sc;
    NSC_CHECK(sc.alloc(measure.size(), s));
    Carver cut(sc.p);
    carve(cut, cls, lvl0, fmask, run, lab, head, real, lab2, kind, small);
    // small[]: 0 nF, 1 nrun, 2 nleaf, 3 flags, 4 ncand, 8..10 info, 16 ncomp, 20 deferred tie components,
    // 24..25 tie pool bump pointer (long long), 26..31 run bucket sizes, 32..34 LDS flood queue counts,
    // 35 B pixels with queue entries, 40 run flood work counter
    NSC_HIP(hipMemsetAsync(small, 0, 64 * sizeof(int), s));

    Dev D{};
    D.img = img; D.W = W; D.H = H; D.N = (int)N; D.m0 = m0; D.m = m; D.cls = cls; D.lvl0 = lvl0; D.run = run;
    D.lab = lab; D.head = head; D.nleaf = &small[2]; D.flags = &small[3];
    // A run's pops are at most the image's inner pixels (a pixel pops once as F, once a run as a leaf), and an F
    // pixel has four neighbours: only runs of larger images can outgrow the records' 24 bits, the largest index
    // standing for itself or, with the plane, for what the plane holds.  NSC_WS_POP_CAP lowers the line (tests of
    // the plane; not below the LDS floods' largest frame, whose indexes are always their records').
    D.popcap = kPopMax - 1;
    if (const char* e = getenv("NSC_WS_POP_CAP")) D.popcap = std::min(std::max(atoi(e), kRunTierMax + 1), kPopMax - 1);
    {  // real[] is unused until B resolution: it holds the per-workgroup counts
        const unsigned nb = (unsigned)std::min<size_t>(cdiv(N, 256), 1u << 14);
        hipLaunchKernelGGL(k_classify, dim3(nb), dim3(256), 0, s, D, cls, lvl0, fmask, real);
        hipLaunchKernelGGL(k_sum_partials, dim3(1), dim3(1024), 0, s, real, (int)nb, &small[0]);
    }
    tick("classify", &small[0]);
    NSC_CHECK(ccl_neq(fmask, 0, run, W, H, 4, s));
    NSC_CHECK(relabel_impl(run, W, H, -1, &small[1], lab2, s));
    tick("runs", &small[1]);
    int hostc[2];
    NSC_HIP(hipMemcpyAsync(hostc, small, 2 * sizeof(int), hipMemcpyDeviceToHost, s));
    NSC_HIP(stream_sync(s));
    const int nF = hostc[0], nrun = hostc[1];
    // phase-1 scratch: run boxes, per-run FIFO heads/tails, queue links, leaf table, item records
    const int leafcap = std::max(1024, std::min((int)std::min(N, (size_t)INT_MAX / 4), 4 * nF + 1024));
    Carver m2(nullptr);
    const bool manypops = std::min((long long)(W - 2) * (H - 2), 5ll * nF) > (long long)D.popcap + 1;
    auto carve2 = [&](Carver& c, int32_t*& box5, int*& qh, int*& qt, int32_t*& qnext, int32_t*& lf, int4*& wr, int32_t*& popx) {
        box5 = c.take<int32_t>(5 * (size_t)std::max(nrun, 1));
        qh = c.take<int>((size_t)std::max(nrun, 1) * (NQ + kRunTiers));  // run buckets, then FIFO heads
        qt = c.take<int>((size_t)std::max(nrun, 1) * NQ);
        qnext = c.take<int32_t>(N + (size_t)leafcap);
        lf = c.take<int32_t>((size_t)leafcap * 2);
        wr = c.take<int4>(N + (size_t)leafcap);
        popx = manypops ? c.take<int32_t>(N + (size_t)leafcap) : nullptr;
    };
    int32_t *box5, *qnext, *lf;
    int *qh, *qt;
    carve2(m2, box5, qh, qt, qnext, lf, D.wr, D.popx);
    Scratch sc2;
    NSC_CHECK(sc2.alloc(m2.size(), s));
    Carver cut2(sc2.p);
    carve2(cut2, box5, qh, qt, qnext, lf, D.wr, D.popx);
    D.qnext = qnext;
    D.leafcap = leafcap;
    D.lf_b = lf;
    D.lf_next = lf + (size_t)leafcap;
    if (nrun > 0) {
        NSC_CHECK(bbox_impl(run, W, H, nrun, box5, nullptr, s));
        int* lists = reinterpret_cast<int*>(qh);  // kRunTiers * nrun ints
        int* bcount = &small[26];                  // kRunTiers counters
        int* qh2 = qh + (size_t)kRunTiers * nrun;  // FIFO heads for the global-flood bucket
        hipLaunchKernelGGL(k_bucket_runs, dim3(cdiv(nrun, 256)), dim3(256), 0, s, box5, nrun, lists, bcount);
        if (dbg) {
            int bc[kRunTiers];
            (void)hipMemcpy(bc, bcount, sizeof(bc), hipMemcpyDeviceToHost);
            fprintf(stderr, "[ws] run tiers %d %d %d %d %d %d\n", bc[0], bc[1], bc[2], bc[3], bc[4], bc[5]);
            std::vector<int32_t> hb((size_t)5 * nrun);
            (void)hipMemcpy(hb.data(), box5, sizeof(int32_t) * hb.size(), hipMemcpyDeviceToHost);
            long long area[kRunTiers] = {}, amax[kRunTiers] = {};
            for (int r = 0; r < nrun; ++r) {
                const long long a = (long long)(hb[2 * (size_t)nrun + r] - hb[nrun + r] + 1 + 2 * P1_MARGIN) *
                                    (hb[4 * (size_t)nrun + r] - hb[3 * (size_t)nrun + r] + 1 + 2 * P1_MARGIN);
                const int tier[kRunTiers - 1] = {512, 1024, 2048, 4096, 6400};
                int b = 0;
                while (b < kRunTiers - 1 && a > tier[b]) ++b;
                area[b] += a;
                amax[b] = std::max(amax[b], a);
            }
            for (int b = 0; b < kRunTiers; ++b)
                fprintf(stderr, "[ws] tier %d: runs %d, box px %lld, max %lld\n", b, bc[b], area[b], amax[b]);
        }
        // four runs a workgroup (one per SIMD) before a further CU is taken whole
        const int g = std::max(1, std::min((int)cdiv(nrun, 4), device_cus()));
        if (D.popx)
            hipLaunchKernelGGL(k_phase1<true>, dim3(g), dim3(64 * P1_WAVES), 0, s, D, box5, nrun, lists, bcount, &small[40], qh2, qt);
        else
            hipLaunchKernelGGL(k_phase1<false>, dim3(g), dim3(64 * P1_WAVES), 0, s, D, box5, nrun, lists, bcount, &small[40], qh2, qt);
    }
    // B pixels with a queue entry: initially queued ones, then those with leaves (the phase-1
    // queue links are dead from here on and hold the list)
    int* blist = qnext;  // N + leafcap ints
    hipLaunchKernelGGL(k_collect_b0, grid1(N), dim3(256), 0, s, D, blist, &small[35]);
    if (nrun > 0) hipLaunchKernelGGL(k_link_leaves, grid1(N), dim3(256), 0, s, D, blist, &small[35]);
    tick("phase1", &small[2]);
    // B resolution and b1
    int* cand = lab2;  // reuse (N ints)
    NSC_HIP(hipMemsetAsync(real, 0xFF, sizeof(int32_t) * N, s));  // -1 everywhere
    hipLaunchKernelGGL(k_bresolve, grid_counted(N), dim3(256), 0, s, D, real, cand, &small[4], blist, &small[35]);
    tick("bresolve", &small[4]);
    {
        int* partial = small + 64;
        hipLaunchKernelGGL(k_b1_partial, dim3(B1_BLOCKS), dim3(256), 0, s, D, real, cand, &small[4], partial);
        hipLaunchKernelGGL(k_b1_reduce, dim3(1), dim3(1024), 0, s, D, real, partial, &small[8]);
    }
    tick("b1", &small[8]);
    hipLaunchKernelGGL(k_t1_state, grid1((N + 3) / 4), dim3(256), 0, s, D, real, &small[8], fmask, kind);
    // flood from b1 over the never-queued B pixels (fmask marks them): geodesic distance from b1
    {
        unsigned* dist = reinterpret_cast<unsigned*>(head);  // head[] is dead after k_bresolve
        hipLaunchKernelGGL(k_geo_init, grid1(N), dim3(256), 0, s, D, &small[8], fmask, dist);
        const int grc = geodist_impl(fmask, dist, W, H, s, &small[8]);  // the seed: b1
        if (grc == NSC_ERR_LIMIT) {  // outside the tile search's range: the sequential flood decides
            clear_error();  // the call still succeeds: no error text left behind
            ws_last_flags_record(FB_CMP);
            return NSC_OK;
        }
        NSC_CHECK(grc);
        tick("geodist", nullptr);
        hipLaunchKernelGGL(k_bfs_mark, grid1(N), dim3(256), 0, s, D, &small[8], dist, kind, lab /* pdist; lab[] is dead */);
        hipLaunchKernelGGL(k_bfs_commit, grid1(N), dim3(256), 0, s, D, &small[8], dist, kind, fmask);
    }
    // phase 2
    NSC_CHECK(ccl_neq(fmask, 0, lab2, W, H, 4, s));
    NSC_CHECK(relabel_impl(lab2, W, H, -1, &small[16], head /* rank scratch: head[] is dead after k_bresolve */, s));
    int sm16[16];  // small[16..31]: ncomp and, at 26..31, the phase-1 run counts per tier
    NSC_HIP(hipMemcpyAsync(sm16, &small[16], sizeof(sm16), hipMemcpyDeviceToHost, s));
    NSC_HIP(stream_sync(s));
    const int ncomp = sm16[0];
    ws_tier_record(sm16 + 10, kRunTiers);
    if (ncomp > 0) {
        Scratch sc3;
        Carver m3(nullptr);
        auto carve3 = [&](Carver& c, int32_t*& b5, int32_t*& area, int32_t*& off, int32_t*& scr, long long*& hk) {
            b5 = c.take<int32_t>(5 * (size_t)ncomp);
            area = c.take<int32_t>(ncomp);
            off = c.take<int32_t>(ncomp);
            scr = c.take<int32_t>(3 * N);
            hk = c.take<long long>(N);
        };
        int32_t *b5, *area, *off, *scr;
        long long* hk;
        carve3(m3, b5, area, off, scr, hk);
        NSC_CHECK(sc3.alloc(m3.size(), s));
        Carver cut3(sc3.p);
        carve3(cut3, b5, area, off, scr, hk);
        NSC_CHECK(bbox_impl(lab2, W, H, ncomp, b5, area, s));
        if (dbg) {  // phase-2 components by where they flood (tie-free ones; a tie moves a small one to LDS)
            std::vector<int32_t> hb(5 * (size_t)ncomp), ha(ncomp);
            (void)hipMemcpy(hb.data(), b5, sizeof(int32_t) * hb.size(), hipMemcpyDeviceToHost);
            (void)hipMemcpy(ha.data(), area, sizeof(int32_t) * ha.size(), hipMemcpyDeviceToHost);
            long long nbig = 0, maxa_big = 0, maxl = 0, nsmall = 0, nlds = 0, n1 = 0, n2 = 0;
            for (int c = 0; c < ncomp; ++c) {
                n1 += ha[c] == 1;
                n2 += ha[c] == 2;
                const long long L = (long long)(hb[2 * ncomp + c] - hb[ncomp + c] + 3) * (hb[4 * ncomp + c] - hb[3 * ncomp + c] + 3);
                maxl = std::max(maxl, L);
                if (L > FL_BIG) { ++nbig; maxa_big = std::max<long long>(maxa_big, ha[c]); }
                else if (ha[c] > FL_MIN_AREA) ++nlds;
                else ++nsmall;
            }
            fprintf(stderr, "[ws] p2 comps %d: lane-flooded %lld (area 1: %lld, 2: %lld), LDS %lld, global %lld (max area %lld), max frame %lld\n",
                    ncomp, nsmall, n1, n2, nlds, nbig, maxa_big, maxl);
        }
        {  // offsets of the components' scratch: exclusive scan of their areas
            size_t tb = 0;
            NSC_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, tb, area, off, ncomp, s));
            Scratch st;
            NSC_CHECK(st.alloc(tb, s));
            NSC_HIP(hipcub::DeviceScan::ExclusiveSum(st.p, tb, area, off, ncomp, s));
        }
        P2 Q{lab2, b5, area, off, kind, scr, ncomp};
        tick("p2 setup", &small[16]);
        const int tiecap = 4096;
        const long long poolcap = std::max<long long>(16ll << 20, 4ll * (long long)N);  // ints
        Scratch sc4;
        NSC_CHECK(sc4.alloc(sizeof(TieRec) * tiecap + sizeof(int) * poolcap + 256, s));
        TieRec* ties = reinterpret_cast<TieRec*>(sc4.p);
        int* pool = reinterpret_cast<int*>(reinterpret_cast<char*>(sc4.p) + ((sizeof(TieRec) * tiecap + 255) & ~size_t(255)));
        long long* pool_used = reinterpret_cast<long long*>(&small[24]);  // 8-byte aligned: small is 256-aligned
        // records and work lists of the LDS flood
        const int workcap = ncomp + (1 << 18);
        Scratch sc5;
        NSC_CHECK(sc5.alloc(sizeof(TieRec) * (size_t)ncomp + 2 * sizeof(int) * (size_t)workcap + sizeof(int) * (size_t)ncomp + 768,
                            s));
        FloodQ F{};
        F.recs = reinterpret_cast<TieRec*>(sc5.p);
        F.reccap = ncomp;
        F.work[0] = reinterpret_cast<int*>(reinterpret_cast<char*>(sc5.p) + ((sizeof(TieRec) * (size_t)ncomp + 255) & ~size_t(255)));
        F.work[1] = F.work[0] + workcap;
        F.workcap = workcap;
        F.nrec = &small[32];
        F.nwork = &small[33];  // [33], [34]
        F.res = pool;
        F.recbad = reinterpret_cast<int*>(reinterpret_cast<char*>(F.work[1] + workcap) + 256 -
                                          (reinterpret_cast<uintptr_t>(F.work[1] + workcap) & 255));
        NSC_HIP(hipMemsetAsync(F.recbad, 0, sizeof(int) * (size_t)ncomp, s));
        hipLaunchKernelGGL(k_phase2, dim3(cdiv(ncomp, 64)), dim3(64), 0, s, D, Q, real, hk, ties, &small[20], tiecap,
                           pool_used, poolcap, F);
        tick("phase2", &small[20]);
        hipLaunchKernelGGL(k_flood_lds<FL_BIG>, dim3(256), dim3(64), 0, s, D, Q, real, F, 1);
        hipLaunchKernelGGL(k_flood_lds<FL_SMALL>, dim3(1024), dim3(64), 0, s, D, Q, real, F, 0);
        hipLaunchKernelGGL(k_tie_check, dim3(2048), dim3(256), 0, s, Q, F, W);
        hipLaunchKernelGGL(k_tie_commit, dim3(1024), dim3(256), 0, s, D, Q, F);
        tick("lds flood", &small[32]);
        hipLaunchKernelGGL(k_phase2_ties, dim3(tiecap), dim3(64), 0, s, D, Q, real, ties, &small[20], pool);
        tick("ties", &small[3]);
    }
    if (ev0) (void)hipEventDestroy(ev0);
    int flags = 0;
    NSC_HIP(hipGetLastError());
    NSC_HIP(hipMemcpyAsync(&flags, &small[3], sizeof(int), hipMemcpyDeviceToHost, s));
    NSC_HIP(stream_sync(s));
    *ok = (flags == 0) ? 1 : 0;
    ws_last_flags_record(flags);
    return NSC_OK;
}

}  // namespace nsc
