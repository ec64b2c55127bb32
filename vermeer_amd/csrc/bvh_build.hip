// QBVH build on the GPU with the reference's output: qbvh.BuildAccel (qbvh/build.go:28-307) node for
// node, with boxes / centroids / indxs permuted into the same leaf order.
//
// The reference recurses depth first.  Each node takes three binary splits (the whole range, then
// its two halves); a split bins the centroids of the longest axis of their bounds into 8 bins
// (k1 = 7.99952 / extent), picks the first strict minimum of the SAH cost and partitions with an
// unstable two-pointer loop; children with at most leafMax elements become leaves.  Every float32
// rounding and every swap decides the leaf order, so the arithmetic here is the reference's, and the
// two-pointer loop is replaced by a closed form of its result that each element computes alone:
//
//   The loop examines elements from two streams, positions 0, 1, ... (the left stream) and n-1,
//   n-2, ... (the right stream): it reads the left stream until it meets a right element (bin >=
//   best), then the right stream until it meets a left element, and so on; left elements land at
//   0, 1, ... and right elements at n-1, n-2, ... in the order examined.  With nl left elements the
//   left stream covers [0, s), s = nl + 1 if position nl holds a right element, else nl.  Then for
//   p < s a left element stays at p, and the k-th right element from position 0 goes to
//   n - 2 - lr[k-2] (k = 1: n - 1), where lr[j] = n - 1 - (position of the (j+1)-th left element
//   counted from n - 1); for p >= s a right element goes to p - 1 and the k-th left element counted
//   from n - 1 goes to rl[k-1], the position of the k-th right element counted from 0.
//
// Box arithmetic follows MINSS / MAXSS (math/dim_amd64.s): x < y ? x : y.  The boxes that reach the
// nodes (leaf boxes, unions of child boxes) are grown in the reference's order, so the sign of zero
// bounds matches as well.  The centroid bounds and bin boxes of a split decide only through subtractions,
// products and comparisons, which give the same split whichever zero a bound is, so those folds run in
// any order, as integer minima and maxima of order-preserving keys.
//
// Schedule.  Ranges above kSubtreeMax elements are split level by level with device-wide kernels
// over chunks (all nodes of a level in one batch of launches; the host reads the pivots
// back after each batch).  A range of at most kSubtreeMax elements becomes a subtree that one
// workgroup builds completely in LDS, its wavefronts taking nodes from a queue (k_subtree), into a
// scratch node area at its element offset.  The host then numbers the nodes in the reference's
// depth-first pre-order and one kernel moves every subtree into place.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <limits>
#include <mutex>
#include <thread>
#include <utility>
#include <vector>

#include "qbvh_build.h"

namespace vgpu {

namespace {

constexpr int kSegThreads = 256;                 // threads of a chunk kernel
// Elements per chunk: small chunks fill the chip (300,001 elements: 293 workgroups instead of 73; the kernels
// of a batch take 51 us instead of 85), large ones keep the per-task folds over chunks short.
constexpr int kChunkSmall = 1024, kChunkLarge = 4096, kChunkLargeFrom = 1 << 20;
constexpr int kSubtreeMax = 2048;                // largest range one workgroup builds in LDS
constexpr int kStackMax = 192;                   // subtree depth limit

// One element: a = (lo xyz, index bits), b = (hi xyz, 0), c = (centroid xyz, 0).
struct alignas(16) GElem {
    float4 a, b, c;
};

struct Box {
    float lo[3], hi[3];
};

__device__ __forceinline__ float mins(float x, float y) { return (x < y) ? x : y; }
__device__ __forceinline__ float maxs(float x, float y) { return (x > y) ? x : y; }

__device__ __forceinline__ Box box_empty() {
    const float inf = __builtin_inff();
    return Box{{inf, inf, inf}, {-inf, -inf, -inf}};
}
// BoundingBox.GrowBox (math/boundingbox.go:99-104): Min(acc, b), Max(acc, b); ties take b.
__device__ __forceinline__ void grow_box(Box& acc, const Box& b) {
    for (int k = 0; k < 3; k++) { acc.lo[k] = mins(acc.lo[k], b.lo[k]); acc.hi[k] = maxs(acc.hi[k], b.hi[k]); }
}
__device__ __forceinline__ float dim(const Box& b, int a) { return b.hi[a] - b.lo[a]; }
__device__ __forceinline__ float area(const Box& b) {
    return dim(b, 0) * dim(b, 1) * 2.0f + dim(b, 1) * dim(b, 2) * 2.0f + dim(b, 0) * dim(b, 2) * 2.0f;
}
__device__ __forceinline__ int longest(const Box& b) {
    if (dim(b, 0) < dim(b, 1)) return (dim(b, 1) < dim(b, 2)) ? 2 : 1;
    return (dim(b, 0) < dim(b, 2)) ? 2 : 0;
}
__device__ __forceinline__ Box elem_box(const GElem& e) {
    return Box{{e.a.x, e.a.y, e.a.z}, {e.b.x, e.b.y, e.b.z}};
}
__device__ __forceinline__ float cen(const float4& c, int axis) { return axis == 0 ? c.x : (axis == 1 ? c.y : c.z); }

// The binning of one split: bin(c) = int(k1 * (c[axis] - k0)); right side: bin >= best.
struct Cut {
    int axis, best;
    float k0, k1;
    __device__ __forceinline__ bool right(const float4& c) const { return !((int)(k1 * (cen(c, axis) - k0)) < best); }
};

// ---------------------------------------------------------------- folds

// Order-preserving integer keys of floats (no NaN): unsigned comparison of keys is comparison of values,
// with -0 below +0.
__device__ __forceinline__ uint32_t key_of(float f) {
    const uint32_t u = __float_as_uint(f);
    return u ^ ((uint32_t)((int32_t)u >> 31) | 0x80000000u);
}
__device__ __forceinline__ float of_key(uint32_t k) {
    return __uint_as_float(k ^ (((k >> 31) - 1u) | 0x80000000u));
}
constexpr uint32_t kKeyInf = 0xff800000u, kKeyNegInf = 0x007fffffu;   // key_of(+inf), key_of(-inf)

// DPP shifts: lanes without a source read `old`.
template <int CTRL, int ROWS = 0xf>
__device__ __forceinline__ uint32_t dpp(uint32_t old, uint32_t x) {
    return (uint32_t)__builtin_amdgcn_update_dpp((int)old, (int)x, CTRL, ROWS, 0xf, false);
}
__device__ __forceinline__ uint32_t wave_min(uint32_t x) {
    x = min(x, dpp<0x111>(~0u, x));
    x = min(x, dpp<0x112>(~0u, x));
    x = min(x, dpp<0x114>(~0u, x));
    x = min(x, dpp<0x118>(~0u, x));
    x = min(x, dpp<0x142, 0xa>(~0u, x));
    x = min(x, dpp<0x143, 0xc>(~0u, x));
    return (uint32_t)__builtin_amdgcn_readlane((int)x, 63);
}
__device__ __forceinline__ uint32_t wave_max(uint32_t x) { return ~wave_min(~x); }

// Keys of centroid bounds, folded over elements.
struct KeyBox {
    uint32_t lo[3], hi[3];
    __device__ __forceinline__ void reset() {
        for (int k = 0; k < 3; k++) { lo[k] = kKeyInf; hi[k] = kKeyNegInf; }
    }
    __device__ __forceinline__ void grow(float x, float y, float z) {
        const float q[3] = {x, y, z};
        for (int k = 0; k < 3; k++) {
            const uint32_t u = key_of(q[k]);
            lo[k] = min(lo[k], u);
            hi[k] = max(hi[k], u);
        }
    }
    __device__ __forceinline__ void join(const KeyBox& o) {
        for (int k = 0; k < 3; k++) { lo[k] = min(lo[k], o.lo[k]); hi[k] = max(hi[k], o.hi[k]); }
    }
    __device__ __forceinline__ void over_wave() {
        for (int k = 0; k < 3; k++) { lo[k] = wave_min(lo[k]); hi[k] = wave_max(hi[k]); }
    }
    __device__ __forceinline__ Box box() const {
        Box b;
        for (int k = 0; k < 3; k++) { b.lo[k] = of_key(lo[k]); b.hi[k] = of_key(hi[k]); }
        return b;
    }
};

// Orders one wavefront's LDS accesses for the compiler (the hardware keeps them in order).
__device__ __forceinline__ void wave_order() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); }

constexpr int kWaves = kSegThreads / 64;

// The split's axis and binning from the centroid bounds (build.go:40-58); false on a flat axis.
__device__ __forceinline__ bool cut_of(const Box& cb, Cut& cut) {
    cut.axis = longest(cb);
    cut.best = 0;
    const float lo = cut.axis == 0 ? cb.lo[0] : (cut.axis == 1 ? cb.lo[1] : cb.lo[2]);
    const float hi = cut.axis == 0 ? cb.hi[0] : (cut.axis == 1 ? cb.hi[1] : cb.hi[2]);
    cut.k1 = 7.99952f / (hi - lo);
    cut.k0 = lo;
    return !(hi == lo);
}

// Eight bins as kBinWords words: six keys (lo xyz, hi xyz) per bin, then the eight counts.
constexpr int kBinWords = 56;
__device__ __forceinline__ uint32_t bin_identity(int w) { return w >= 48 ? 0u : (w % 6 < 3 ? kKeyInf : kKeyNegInf); }
__device__ __forceinline__ uint32_t bin_join(int w, uint32_t x, uint32_t y) {
    return w >= 48 ? x + y : (w % 6 < 3 ? min(x, y) : max(x, y));
}
// A wavefront's bins in LDS: COPIES copies, lane l adding to copy l % COPIES, since atomics on one address are
// served one after another (about 8 cycles a lane).  Eight for the chunks of the device-wide splits (293 chunks
// of 1024 elements: 25 us with one copy, 18 with eight), one for the subtrees, whose ranges are too short to
// pay for more (k_subtree over 300,001 triangles: 220 us with one, 245 with eight, measured before its last permutation
// stayed in registers).  Eight boxes per lane in registers cost 130 instructions an element and 288 shuffles a fold.
constexpr int kBinStride = kBinWords + 1;   // the odd stride spreads the copies over the banks
template <int COPIES>
struct WaveBins {
    uint32_t w[COPIES * kBinStride];
    __device__ __forceinline__ uint32_t* mine() { return w + ((int)threadIdx.x % COPIES) * kBinStride; }
};
template <int COPIES>
__device__ __forceinline__ void bins_reset(WaveBins<COPIES>& B) {
    for (int i = threadIdx.x & 63; i < COPIES * kBinStride; i += 64) B.w[i] = bin_identity(i % kBinStride);
}
// Folds the copies into the first one.
template <int COPIES>
__device__ __forceinline__ void bins_fold(WaveBins<COPIES>& B) {
    const int w = threadIdx.x & 63;
    if (COPIES == 1 || w >= kBinWords) return;
    uint32_t x = B.w[w];
#pragma unroll
    for (int k = 1; k < COPIES; k++) x = bin_join(w, x, B.w[k * kBinStride + w]);
    B.w[w] = x;
}
// Adds a box whose centroid coordinate on the cut's axis is c to a lane's copy; sets err bit 1 for a bin
// outside [0, 7] (the reference's index panics there).
__device__ __forceinline__ void bins_add(uint32_t* bins, const Cut& cut, float c, const float* b, int* err) {
    const float f = cut.k1 * (c - cut.k0);
    const int bin = (int)f;
    if (f != f || bin < 0 || bin > 7) { atomicOr(err, 1); return; }
    uint32_t* w = bins + bin * 6;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        __hip_atomic_fetch_min(w + k, key_of(b[k]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        __hip_atomic_fetch_max(w + 3 + k, key_of(b[3 + k]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    __hip_atomic_fetch_add(bins + 48 + bin, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// calcMinCost's SAH choice (qbvh/build.go:60-107) over the folded bins, by one wavefront, lane b holding
// bin b: left boxes and counts grown from bin 0, right ones from bin 7 (DPP scans), the first strict
// minimum of area(L) * nL + area(R) * nR.
__device__ void sah_wave(const uint32_t* bins, int* best_out, int* nl_out) {
    const int lane = threadIdx.x & 63;
    const bool in = lane < 8;
    Box L, R;
#pragma unroll
    for (int j = 0; j < 6; j++) {
        const bool lo = j < 3;
        const uint32_t id = lo ? kKeyInf : kKeyNegInf;
        const uint32_t v = in ? bins[lane * 6 + j] : id;
        auto fold = [&](uint32_t x, uint32_t y) { return lo ? min(x, y) : max(x, y); };
        uint32_t p = v, q = v;
        p = fold(p, dpp<0x111>(id, p)); p = fold(p, dpp<0x112>(id, p)); p = fold(p, dpp<0x114>(id, p));
        q = fold(q, dpp<0x101>(id, q)); q = fold(q, dpp<0x102>(id, q)); q = fold(q, dpp<0x104>(id, q));
        p = dpp<0x111>(id, p);   // the bins before this one
        (lo ? L.lo : L.hi)[j % 3] = of_key(p);
        (lo ? R.lo : R.hi)[j % 3] = of_key(q);
    }
    const uint32_t n = in ? bins[48 + lane] : 0u;
    uint32_t m = n, rn = n;
    m += dpp<0x111>(0, m); m += dpp<0x112>(0, m); m += dpp<0x114>(0, m);
    rn += dpp<0x101>(0, rn); rn += dpp<0x102>(0, rn); rn += dpp<0x104>(0, rn);
    m = dpp<0x111>(0, m);
    const float cost = area(L) * (float)(int)m + area(R) * (float)(int)rn;
    int best = -1, nl = 0;
    float best_cost = __builtin_inff();
#pragma unroll
    for (int b = 1; b < 8; b++) {
        const float c = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(cost), b));
        if (c < best_cost) { best = b; best_cost = c; nl = __builtin_amdgcn_readlane((int)m, b); }
    }
    *best_out = best;
    *nl_out = nl;
}

// Destination of position p (rank r = right elements in [0, p], inclusive) under the closed form;
// -1 for an index outside [0, n), which only inconsistent bins (an error already flagged) produce.
template <class I>
__device__ __forceinline__ int dest_of(int p, bool right, int r, int n, int nl, int s, const I* rl, const I* lr) {
    int d;
    if (p < s) {
        if (!right) return p;
        if (r < 2) return n - 1;
        if (r - 2 >= n) return -1;
        d = n - 2 - lr[r - 2];
    } else {
        if (right) return p - 1;
        const int k = nl - (p - r) - 1;
        if (k < 0 || k >= n) return -1;
        d = rl[k];
    }
    return (d >= 0 && d < n) ? d : -1;
}
// Records position i in rl / lr (r: right elements in [0, i], inclusive); false if out of range.
template <class I>
__device__ __forceinline__ bool record_rank(int i, bool right, int r, int n, int nl, I* rl, I* lr) {
    if (right) {
        if (r - 1 >= n) return false;
        rl[r - 1] = (I)i;
        return true;
    }
    const int k = nl - (i - r) - 1;
    if (k < 0 || k >= n) return false;
    lr[k] = (I)(n - 1 - i);
    return true;
}

// ---------------------------------------------------------------- subtrees in LDS

struct SplitOut {
    int axis, pivot;
};

constexpr int kSubWaves = 8;
constexpr int kSubThreads = 64 * kSubWaves;
constexpr uint32_t kTaskReady = 0x80000000u;
constexpr int kNoParent = 0x7ff;   // of node 0 only, which no node has as a child

// A subtree's elements (boxes and centroids, in the order they came) and the split's index lists, and its
// nodes in the order they were found: node id's range, its place in the tree and what its completion needs.
struct SubLds {
    float box[6][kSubtreeMax];
    float cen[3][kSubtreeMax];
    uint16_t idx[2][kSubtreeMax];                // positions in split order; a split moves a range between the two
    uint16_t rl[kSubtreeMax], lr[kSubtreeMax];
    uint32_t task[kSubtreeMax];                  // kTaskReady | n << 16 | start, 0 until it is published
    uint32_t link[kSubtreeMax];                  // parent | child slot << 11 | depth << 13
    int pend[kSubtreeMax];                       // child nodes not yet complete
    uint16_t child[kSubtreeMax][4];              // node ids, 0xffff: none
    uint16_t size[kSubtreeMax], before[kSubtreeMax];   // nodes of the subtree; nodes of the siblings before it
    WaveBins<1> bins[kSubWaves];
    int head, tail, done;                        // next ticket; nodes found; 1: complete, 2: given up
};
static_assert(sizeof(SubLds) <= 160 * 1024, "one workgroup per CU");

// binarySplit (qbvh/build.go:151-178) of positions [start, start + n) of L.idx[from] into L.idx[1 - from] by one
// wavefront.
__device__ __forceinline__ SplitOut split_lds(SubLds& L, int from, int start, int n, int leafMax, int* err) {
    const int lane = threadIdx.x & 63;
    const uint16_t* src = &L.idx[from][start];
    uint16_t* dst = &L.idx[1 - from][start];
    uint16_t* rl = L.rl + start;
    uint16_t* lr = L.lr + start;
    WaveBins<1>& B = L.bins[threadIdx.x >> 6];
    Cut cut{0, 0, 0.0f, 0.0f};
    bool split = n > leafMax;
    if (split) {
        KeyBox kb;
        kb.reset();
        for (int i = lane; i < n; i += 64) {
            const int e = src[i];
            kb.grow(L.cen[0][e], L.cen[1][e], L.cen[2][e]);
        }
        kb.over_wave();
        split = cut_of(kb.box(), cut);
    }
    if (!split) {
        for (int i = lane; i < n; i += 64) dst[i] = src[i];
        wave_order();
        return SplitOut{cut.axis, n > leafMax ? n / 2 + 1 : n};
    }
    bins_reset(B);
    wave_order();
    uint32_t* bins = B.mine();
    const float* cen = L.cen[cut.axis];
    for (int i = lane; i < n; i += 64) {
        const int e = src[i];
        float b[6];
#pragma unroll
        for (int k = 0; k < 6; k++) b[k] = L.box[k][e];
        bins_add(bins, cut, cen[e], b, err);
    }
    wave_order();
    bins_fold(B);
    wave_order();
    int nl;
    sah_wave(B.w, &cut.best, &nl);
    auto right = [&](int e) { return !((int)(cut.k1 * (cen[e] - cut.k0)) < cut.best); };
    // rank: right elements at or before the position
    const uint64_t upto = ~0ull >> (63 - lane);
    int run = 0;
    for (int i0 = 0; i0 < n; i0 += 64) {
        const int i = i0 + lane;
        const bool rt = i < n && right(src[i]);
        const uint64_t m = __ballot(rt);
        if (i < n && !record_rank(i, rt, run + __popcll(m & upto), n, nl, rl, lr)) atomicOr(err, 1);
        run += __popcll(m);
    }
    wave_order();
    const int s = nl + ((nl < n && right(src[nl])) ? 1 : 0);
    run = 0;
    for (int i0 = 0; i0 < n; i0 += 64) {
        const int i = i0 + lane;
        const int e = i < n ? src[i] : 0;
        const bool rt = i < n && right(e);
        const uint64_t m = __ballot(rt);
        if (i < n) {
            const int d = dest_of(i, rt, run + __popcll(m & upto), n, nl, s, rl, lr);
            if (d >= 0) dst[d] = (uint16_t)e;
            else atomicOr(err, 1);
        }
        run += __popcll(m);
    }
    wave_order();
    return SplitOut{cut.axis, nl};
}

__device__ __forceinline__ int32_t leaf_code(uint32_t first, uint32_t count) {
    return (int32_t)((1u << 31) | ((first << 4) & 0xfffffff0u) | ((count - 1) & 0xfu));
}

// calcBox of a leaf (GrowBox in element order), by one thread.
__device__ Box leaf_box(const GElem* E, int n) {
    Box b = box_empty();
    for (int i = 0; i < n; i++) grow_box(b, elem_box(E[i]));
    return b;
}

// Node `me` is complete (its leaves' and child nodes' boxes are in its record): its box unions the
// non-empty child boxes in order (qbvh/build.go:277-284) and fills its slot in the parent; the wavefront
// that completes a node's last child completes the node too, up to the root.
__device__ void complete_node(SubLds& L, int me, vgpu_qbvh_node* nodes, float* root_box) {
    const int lane = threadIdx.x & 63;
    while (true) {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
        const vgpu_qbvh_node& nd = nodes[me];
        const bool lo = lane < 3;
        float v = lo ? __builtin_inff() : -__builtin_inff();
        if (lane < 6)
            for (int c = 0; c < 4; c++)
                if (nd.children[c] != -1) {
                    const float b = nd.boxes[c + 4 * lane];
                    v = lo ? mins(v, b) : maxs(v, b);
                }
        if (lane == 0) {
            int sum = 0;
            for (int c = 0; c < 4; c++) {
                const int id = L.child[me][c];
                if (id == 0xffff) continue;
                L.before[id] = (uint16_t)sum;
                sum += L.size[id];
            }
            L.size[me] = (uint16_t)(sum + 1);
        }
        const uint32_t link = L.link[me];
        const int parent = (int)(link & 0x7ffu), slot = (int)((link >> 11) & 3u);
        if (me == 0) {
            if (lane < 6) root_box[lane] = v;
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
            if (lane == 0) __hip_atomic_store(&L.done, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
            return;
        }
        if (lane < 6) nodes[parent].boxes[slot + 4 * lane] = v;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        int left = 0;
        if (lane == 0) left = __hip_atomic_fetch_add(&L.pend[parent], -1, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_WORKGROUP);
        if (__builtin_amdgcn_readfirstlane(left) != 1) return;
        me = parent;
    }
}

// buildAccelRec (qbvh/build.go:180-287) of one subtree per workgroup.  Elements of subtree s: E[roots[s].x,
// + roots[s].y), permuted in place; its nodes in the order they were found at nodes[roots[s].x ..] (at most
// max(n, 1)), their pre-order numbers at pre[roots[s].x ..]; counts[s]: the node count; root_boxes[s]: the
// root's box.  err bit 2: node area exceeded (only a range whose recursion never ends, as two coincident
// centroids with leafMax 1); bit 8: deeper than kStackMax levels.
//
// The elements stay in LDS for the whole build and splits move 16-bit positions.  Wavefronts take nodes from
// a queue in the order they were found: each takes a ticket and waits until that node is published or the
// root is complete (or the build is given up), which some wavefront always reaches, since a published node
// waits for no other.  Finding order puts parents before children; the numbers follow from the subtree sizes.
// One wavefront per subtree splitting in global memory, with eight bin boxes per lane folded through
// shuffles, took 2270 us for the 340 subtrees (882 elements and 39 nodes each on average) of 300,001 triangles of the
// icosphere field; this takes 208 us.  What bounds it: SubLds fills a CU (141,100 bytes of 160 K), so on 256 CUs the 340
// workgroups run in two rounds, and a subtree's nodes wait for one another near its root.
__global__ __launch_bounds__(kSubThreads) void k_subtree(GElem* E_all, const int2* roots, vgpu_qbvh_node* nodes_all,
                                                         int* pre_all, int* counts, float* root_boxes, int leafMax,
                                                         int* err) {
    __shared__ SubLds L;
    const int2 root = roots[blockIdx.x];
    GElem* E = E_all + root.x;
    vgpu_qbvh_node* nodes = nodes_all + root.x;
    const int cap = max(root.y, 1);
    const int t = threadIdx.x, lane = t & 63;
    for (int i = t; i < kSubtreeMax; i += kSubThreads) {
        L.task[i] = 0;
        // every index a valid one, whatever a broken split leaves
        L.idx[0][i] = (uint16_t)min(i, cap - 1);
        L.idx[1][i] = (uint16_t)min(i, cap - 1);
        if (i < root.y) {
            const GElem e = E[i];
            const float b[6] = {e.a.x, e.a.y, e.a.z, e.b.x, e.b.y, e.b.z};
            for (int k = 0; k < 6; k++) L.box[k][i] = b[k];
            L.cen[0][i] = e.c.x; L.cen[1][i] = e.c.y; L.cen[2][i] = e.c.z;
        }
    }
    if (t == 0) {
        L.head = 0;
        L.tail = 1;
        L.done = 0;
        L.link[0] = kNoParent;
    }
    __syncthreads();
    if (t == 0)
        __hip_atomic_store(&L.task[0], kTaskReady | ((uint32_t)root.y << 16), __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
    while (true) {
        int me = 0;
        if (lane == 0) me = __hip_atomic_fetch_add(&L.head, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        me = __builtin_amdgcn_readfirstlane(me);
        uint32_t task = 0;
        int done = 0;
        while (true) {
            done = __builtin_amdgcn_readfirstlane(__hip_atomic_load(&L.done, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP));
            if (done) break;
            if (me < kSubtreeMax)
                task = (uint32_t)__builtin_amdgcn_readfirstlane(
                    (int)__hip_atomic_load(&L.task[me], __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP));
            if (task) break;
            __builtin_amdgcn_s_sleep(1);
        }
        if (done) break;
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        const int start = (int)(task & 0xffffu), n = (int)((task >> 16) & 0x7fffu);
        // the node's three binary splits: idx[0] -> idx[1] over the range, then each half back
        SplitOut s0{}, s1{}, s2{};
#pragma unroll 1
        for (int k = 0; k < 3; k++) {
            const SplitOut o = split_lds(L, k == 0 ? 0 : 1, k == 2 ? start + s0.pivot : start,
                                         k == 0 ? n : (k == 1 ? s0.pivot : n - s0.pivot), leafMax, err);
            if (k == 0) s0 = o;
            else if (k == 1) s1 = o;
            else s2 = o;
        }
        const int p1 = s1.pivot, p0 = s0.pivot, p02 = s0.pivot + s2.pivot;
        auto lo_of = [&](int c) { return c == 0 ? 0 : (c == 1 ? p1 : (c == 2 ? p0 : (c == 3 ? p02 : n))); };
        int cn[4], id[4], found = 0;
#pragma unroll
        for (int c = 0; c < 4; c++) {
            cn[c] = lo_of(c + 1) - lo_of(c);
            id[c] = 0xffff;
            if (cn[c] > leafMax) found++;
        }
        const int depth = (int)(L.link[me] >> 13);
        int first = 0;
        if (found) {
            if (lane == 0) first = __hip_atomic_fetch_add(&L.tail, found, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            first = __builtin_amdgcn_readfirstlane(first);
            const int bad = first + found > cap ? 2 : (depth + 1 >= kStackMax ? 8 : 0);
            if (bad) {
                if (lane == 0) {
                    atomicOr(err, bad);
                    __hip_atomic_store(&L.done, 2, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
                }
                break;
            }
        }
        {
            int k = first;
#pragma unroll
            for (int c = 0; c < 4; c++)
                if (cn[c] > leafMax) id[c] = k++;
        }
        // the node's record, a word per lane: boxes (lane 4 j + c: bound j of child c), axes, children
        const float inf = __builtin_inff();
        uint32_t w = 0;
        if (lane < 24) {
            const int c = lane & 3, j = lane >> 2;
            const int lo = start + lo_of(c), m = c == 0 ? cn[0] : (c == 1 ? cn[1] : (c == 2 ? cn[2] : cn[3]));
            if (m == 0) {
                w = __float_as_uint(inf);   // an empty leaf's InfBox (qbvh/qbvh.go:67-79)
            } else if (m <= leafMax) {      // calcBox of a leaf: GrowBox in element order
                const bool low = j < 3;
                float v = low ? inf : -inf;
                for (int i = 0; i < m; i++) {
                    const float b = L.box[j][L.idx[0][lo + i]];
                    v = low ? mins(v, b) : maxs(v, b);
                }
                w = __float_as_uint(v);
            }
        } else if (lane < 27) {
            w = (uint32_t)(lane == 24 ? s0.axis : (lane == 25 ? s1.axis : s2.axis));
        } else if (lane < 31) {
            const int c = lane - 27;
            const int m = c == 0 ? cn[0] : (c == 1 ? cn[1] : (c == 2 ? cn[2] : cn[3]));
            const int k = c == 0 ? id[0] : (c == 1 ? id[1] : (c == 2 ? id[2] : id[3]));
            w = (uint32_t)(m == 0 ? -1 : (m <= leafMax ? leaf_code((uint32_t)(root.x + start + lo_of(c)), (uint32_t)m) : k));
            L.child[me][c] = (uint16_t)k;
        }
        if (lane < 32) reinterpret_cast<uint32_t*>(nodes + me)[lane] = w;
        if (lane == 0) L.pend[me] = found;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        if (found == 0) {
            complete_node(L, me, nodes, root_boxes + blockIdx.x * 6);
        } else if (lane < 4) {
            const int m = lane == 0 ? cn[0] : (lane == 1 ? cn[1] : (lane == 2 ? cn[2] : cn[3]));
            const int k = lane == 0 ? id[0] : (lane == 1 ? id[1] : (lane == 2 ? id[2] : id[3]));
            if (m > leafMax) {
                L.link[k] = (uint32_t)me | ((uint32_t)lane << 11) | ((uint32_t)(depth + 1) << 13);
                __hip_atomic_store(&L.task[k], kTaskReady | ((uint32_t)m << 16) | (uint32_t)(start + lo_of(lane)),
                                   __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
            }
        }
    }
    __syncthreads();
    if (L.done != 1) return;
    const int count = L.tail;
    for (int i = t; i < count; i += kSubThreads) {
        int p = 0;
        for (int x = i; x != 0; x = (int)(L.link[x] & 0x7ffu)) p += 1 + L.before[x];
        pre_all[root.x + i] = p;
    }
    if (t == 0) counts[blockIdx.x] = count;
    constexpr int kPer = kSubtreeMax / kSubThreads;
    if (root.y == 0) return;
    // Plain vectors, which stay in registers; as structures they took 256 bytes of scratch per lane.  With those the
    // guide's training kernel, which spills, took 46 us a step instead of 41 in a process that had built a scene.
    typedef float Row __attribute__((ext_vector_type(4)));
    static_assert(sizeof(GElem) == 3 * sizeof(Row), "three rows an element");
    Row er[kPer][3];
#pragma unroll
    for (int k = 0; k < kPer; k++) {
        const Row* p = reinterpret_cast<const Row*>(E + L.idx[0][min(t + k * kSubThreads, root.y - 1)]);
#pragma unroll
        for (int j = 0; j < 3; j++) er[k][j] = p[j];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kPer; k++) {
        const int i = t + k * kSubThreads;
        if (i >= root.y) continue;
        Row* p = reinterpret_cast<Row*>(E + i);
#pragma unroll
        for (int j = 0; j < 3; j++) p[j] = er[k][j];
    }
}

// ---------------------------------------------------------------- device-wide splits of large ranges

// A split of src[start, start + n) into dst, over chunks [chunk0, chunk0 + nchunk) of the batch, `chunk`
// elements each.
struct SegTask {
    int start, n, chunk0, nchunk, chunk;
};
// mode 0: partition; 1: n <= leafMax (no binning); 2: flat axis.  pivot: the split's result.
struct SegParam {
    int mode, axis, best, nl, s, pivot;
    float k0, k1;
};
struct BinPart {
    uint32_t w[kBinWords];
};

struct ChunkRange {
    int task, first, end;   // task index and the chunk's element range within the task
};
__device__ __forceinline__ ChunkRange chunk_range(const SegTask* tasks, const int* chunk_task) {
    ChunkRange c;
    c.task = chunk_task[blockIdx.x];
    const SegTask tk = tasks[c.task];
    c.first = ((int)blockIdx.x - tk.chunk0) * tk.chunk;
    c.end = min(tk.n, c.first + tk.chunk);
    return c;
}
// Right elements of the block's chunks before this one, then of its wavefronts before this one: the rank
// base of a wavefront's quarter of the chunk.  part: right elements per chunk.  sh: kWaves ints each.
__device__ int rank_base(const SegTask& tk, const int* part, int mine, int* sh_before, int* sh_mine) {
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int chunk = (int)blockIdx.x - tk.chunk0;
    int before = 0;
    for (int i = threadIdx.x; i < chunk; i += kSegThreads) before += part[tk.chunk0 + i];
    for (int d = 32; d >= 1; d >>= 1) before += __shfl_xor(before, d);
    if (lane == 0) { sh_before[wv] = before; sh_mine[wv] = mine; }
    __syncthreads();
    int base = 0;
    for (int k = 0; k < kWaves; k++) {
        base += sh_before[k];
        if (k < wv) base += sh_mine[k];
    }
    return base;
}
// A wavefront's quarter of the chunk, read 64 consecutive elements at a time.
__device__ __forceinline__ void wave_range(const ChunkRange& c, int chunk, int* a, int* b) {
    *a = min(c.end, c.first + (int)(threadIdx.x >> 6) * (chunk / kWaves));
    *b = min(c.end, *a + chunk / kWaves);
}
// Right elements in a wavefront's range.
__device__ __forceinline__ int wave_count(const GElem* E, const Cut& cut, int a, int b) {
    int cnt = 0;
    for (int i0 = a; i0 < b; i0 += 64) {
        const int i = i0 + (int)(threadIdx.x & 63);
        cnt += __popcll(__ballot(i < b && cut.right(E[i].c)));
    }
    return cnt;
}

__global__ __launch_bounds__(kSegThreads) void k_seg_cb(const GElem* src, const SegTask* tasks, const int* chunk_task,
                                                         int leafMax, KeyBox* part) {
    __shared__ KeyBox sh[kWaves];
    const ChunkRange c = chunk_range(tasks, chunk_task);
    if (tasks[c.task].n <= leafMax) return;
    const GElem* E = src + tasks[c.task].start;
    KeyBox v;
    v.reset();
    for (int i = c.first + (int)threadIdx.x; i < c.end; i += kSegThreads) v.grow(E[i].c.x, E[i].c.y, E[i].c.z);
    v.over_wave();
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int k = 1; k < kWaves; k++) v.join(sh[k]);
        part[blockIdx.x] = v;
    }
}

// The task's cut from its chunks' centroid bounds, by every block of the task (the bounds of a chunk are
// 24 bytes; a launch of its own cost 6 us), and the chunk's bins.  The task's first block keeps the cut.
__global__ __launch_bounds__(kSegThreads) void k_seg_bins(const GElem* src, const SegTask* tasks, const int* chunk_task,
                                                           const KeyBox* cb_part, int leafMax, SegParam* params,
                                                           BinPart* part, int* err) {
    __shared__ KeyBox sh[kWaves];
    __shared__ WaveBins<8> bins[kWaves];
    const ChunkRange c = chunk_range(tasks, chunk_task);
    const SegTask tk = tasks[c.task];
    const bool owner = (int)blockIdx.x == tk.chunk0 && threadIdx.x == 0;
    SegParam P{};
    if (tk.n <= leafMax) {
        P.mode = 1;
        P.pivot = tk.n;
        if (owner) params[c.task] = P;
        return;
    }
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    KeyBox v;
    v.reset();
    for (int i = threadIdx.x; i < tk.nchunk; i += kSegThreads) v.join(cb_part[tk.chunk0 + i]);
    v.over_wave();
    if (lane == 0) sh[wv] = v;
    bins_reset(bins[wv]);
    __syncthreads();
    v = sh[0];
    for (int k = 1; k < kWaves; k++) v.join(sh[k]);
    Cut cut;
    const bool flat = !cut_of(v.box(), cut);
    P.axis = cut.axis;
    if (flat) {
        P.mode = 2;
        P.pivot = tk.n / 2 + 1;
    } else {
        P.k1 = cut.k1;
        P.k0 = cut.k0;
    }
    if (owner) params[c.task] = P;
    if (flat) return;
    const GElem* E = src + tk.start;
    for (int i = c.first + (int)threadIdx.x; i < c.end; i += kSegThreads) {
        const GElem e = E[i];
        const float b[6] = {e.a.x, e.a.y, e.a.z, e.b.x, e.b.y, e.b.z};
        bins_add(bins[wv].mine(), cut, cen(e.c, cut.axis), b, err);
    }
    wave_order();
    bins_fold(bins[wv]);
    __syncthreads();
    if (threadIdx.x < kBinWords) {
        const int w = threadIdx.x;
        uint32_t x = bins[0].w[w];
        for (int k = 1; k < kWaves; k++) x = bin_join(w, x, bins[k].w[w]);
        part[blockIdx.x].w[w] = x;
    }
}

__global__ __launch_bounds__(kSegThreads) void k_seg_sah(const GElem* src, const SegTask* tasks, const BinPart* part,
                                                          SegParam* params) {
    __shared__ uint32_t sh[kWaves][kBinWords];
    const SegTask tk = tasks[blockIdx.x];
    SegParam P = params[blockIdx.x];
    if (P.mode != 0) return;
    const int wv = threadIdx.x >> 6, w = threadIdx.x & 63;
    if (w < kBinWords) {
        uint32_t x = bin_identity(w);
        for (int i = wv; i < tk.nchunk; i += kWaves) x = bin_join(w, x, part[tk.chunk0 + i].w[w]);
        sh[wv][w] = x;
    }
    __syncthreads();
    if (wv != 0) return;
    if (w < kBinWords) {
        uint32_t x = sh[0][w];
        for (int k = 1; k < kWaves; k++) x = bin_join(w, x, sh[k][w]);
        sh[0][w] = x;
    }
    wave_order();
    Cut cut{P.axis, 0, P.k0, P.k1};
    sah_wave(sh[0], &cut.best, &P.nl);
    P.best = cut.best;
    P.pivot = P.nl;
    P.s = P.nl + ((P.nl < tk.n && cut.right(src[tk.start + P.nl].c)) ? 1 : 0);
    if (threadIdx.x == 0) params[blockIdx.x] = P;
}

__global__ __launch_bounds__(kSegThreads) void k_seg_rcount(const GElem* src, const SegTask* tasks,
                                                             const int* chunk_task, const SegParam* params, int* part) {
    __shared__ int sh[kWaves];
    const ChunkRange c = chunk_range(tasks, chunk_task);
    const SegParam P = params[c.task];
    if (P.mode != 0) return;
    int a, b;
    wave_range(c, tasks[c.task].chunk, &a, &b);
    const int cnt = wave_count(src + tasks[c.task].start, Cut{P.axis, P.best, P.k0, P.k1}, a, b);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = cnt;
    __syncthreads();
    if (threadIdx.x == 0) {
        int tot = 0;
        for (int k = 0; k < kWaves; k++) tot += sh[k];
        part[blockIdx.x] = tot;
    }
}

// rl / lr of the closed form, at the task's element offset.
__global__ __launch_bounds__(kSegThreads) void k_seg_rank(const GElem* src, const SegTask* tasks, const int* chunk_task,
                                                           const SegParam* params, const int* part, int* rl_all,
                                                           int* lr_all, int* err) {
    __shared__ int sh_before[kWaves], sh_mine[kWaves];
    const ChunkRange c = chunk_range(tasks, chunk_task);
    const SegParam P = params[c.task];
    if (P.mode != 0) return;
    const SegTask tk = tasks[c.task];
    const GElem* E = src + tk.start;
    const Cut cut{P.axis, P.best, P.k0, P.k1};
    int a, b;
    wave_range(c, tk.chunk, &a, &b);
    int r = rank_base(tk, part, wave_count(E, cut, a, b), sh_before, sh_mine);
    const int lane = threadIdx.x & 63;
    const uint64_t upto = ~0ull >> (63 - lane);
    for (int i0 = a; i0 < b; i0 += 64) {
        const int i = i0 + lane;
        const bool right = i < b && cut.right(E[i].c);
        const uint64_t m = __ballot(right);
        if (i < b && !record_rank(i, right, r + __popcll(m & upto), tk.n, P.nl, rl_all + tk.start, lr_all + tk.start))
            atomicOr(err, 1);
        r += __popcll(m);
    }
}

__global__ __launch_bounds__(kSegThreads) void k_seg_scatter(const GElem* src, GElem* dst, const SegTask* tasks,
                                                              const int* chunk_task, const SegParam* params,
                                                              const int* part, const int* rl_all, const int* lr_all,
                                                              int* err) {
    __shared__ int sh_before[kWaves], sh_mine[kWaves];
    const ChunkRange c = chunk_range(tasks, chunk_task);
    const SegParam P = params[c.task];
    const SegTask tk = tasks[c.task];
    const GElem* S = src + tk.start;
    GElem* D = dst + tk.start;
    if (P.mode != 0) {
        for (int i = c.first + (int)threadIdx.x; i < c.end; i += kSegThreads) D[i] = S[i];
        return;
    }
    const Cut cut{P.axis, P.best, P.k0, P.k1};
    int a, b;
    wave_range(c, tk.chunk, &a, &b);
    int r = rank_base(tk, part, wave_count(S, cut, a, b), sh_before, sh_mine);
    const int lane = threadIdx.x & 63;
    const uint64_t upto = ~0ull >> (63 - lane);
    for (int i0 = a; i0 < b; i0 += 64) {
        const int i = i0 + lane;
        const GElem e = S[min(i, b - 1)];
        const bool right = i < b && cut.right(e.c);
        const uint64_t m = __ballot(right);
        if (i < b) {
            const int d = dest_of(i, right, r + __popcll(m & upto), tk.n, P.nl, P.s, rl_all + tk.start, lr_all + tk.start);
            if (d >= 0) D[d] = e;
            else atomicOr(err, 1);
        }
        r += __popcll(m);
    }
}

// ---------------------------------------------------------------- packing, leaves, placement

// Packs the caller's arrays; err bit 4 for a non-finite centroid coordinate (the reference's binning
// fails on it) or a NaN box coordinate (box folds in another grouping would differ on it).
__global__ void k_pack(const float* boxes, const float* cent, const int32_t* idx, int n, GElem* E, int* err) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    GElem e;
    e.a = make_float4(boxes[i * 6], boxes[i * 6 + 1], boxes[i * 6 + 2], __int_as_float(idx[i]));
    e.b = make_float4(boxes[i * 6 + 3], boxes[i * 6 + 4], boxes[i * 6 + 5], 0.0f);
    e.c = make_float4(cent[i * 3], cent[i * 3 + 1], cent[i * 3 + 2], 0.0f);
    bool ok = true;
    for (int k = 0; k < 6; k++) ok = ok && !isnan(boxes[i * 6 + k]);
    for (int k = 0; k < 3; k++) ok = ok && isfinite(cent[i * 3 + k]);
    if (!ok) atomicOr(err, 4);
    E[i] = e;
}

__global__ void k_unpack(const GElem* E, int n, float* boxes, float* cent, int32_t* idx) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const GElem e = E[i];
    boxes[i * 6] = e.a.x; boxes[i * 6 + 1] = e.a.y; boxes[i * 6 + 2] = e.a.z;
    boxes[i * 6 + 3] = e.b.x; boxes[i * 6 + 4] = e.b.y; boxes[i * 6 + 5] = e.b.z;
    cent[i * 3] = e.c.x; cent[i * 3 + 1] = e.c.y; cent[i * 3 + 2] = e.c.z;
    idx[i] = __float_as_int(e.a.w);
}

// Boxes of the leaves under large-range nodes ({start, count}), one thread each.
__global__ void k_leaf_boxes(const GElem* E, const int2* leaves, int n, float* out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const Box b = leaf_box(E + leaves[i].x, leaves[i].y);
    for (int k = 0; k < 3; k++) { out[i * 6 + k] = b.lo[k]; out[i * 6 + 3 + k] = b.hi[k]; }
}

// Moves subtree s's nodes from the scratch area (offset src[s], in the order they were found) to their
// pre-order place from dst[s] on, renumbering child nodes.  A block per subtree along x: the grid's other axes end at
// 65,535, which 38 million elements can pass (about 590 a subtree where the ranges above 2048 split evenly).
__global__ void k_place(const vgpu_qbvh_node* scratch, const int* pre_all, const int* src, const int* dst,
                        const int* counts, vgpu_qbvh_node* out) {
    const int s = blockIdx.x;
    const int* pre = pre_all + src[s];
    for (int i = threadIdx.x; i < counts[s]; i += blockDim.x) {
        vgpu_qbvh_node nd = scratch[src[s] + i];
        for (int c = 0; c < 4; c++)
            if (nd.children[c] >= 0) nd.children[c] = dst[s] + pre[nd.children[c]];
        out[dst[s] + pre[i]] = nd;
    }
}

// ---------------------------------------------------------------- host side

// ---------------------------------------------------------------- pinned staging of the host arrays
//
// A pageable hipMemcpy moves the builder's host arrays (40 bytes per element each way) at about
// 21 GB/s to the device and 14 GB/s back.  Here they go through kStageSlots pinned slots of
// kStageSlot bytes: the host side of each chunk is copied by kCopyThreads threads while the DMA of
// the neighbouring chunk runs.  The slots (128 MiB of pinned host memory per device) are allocated
// by the first build of at least kStageMin bytes on that device and kept until the process ends;
// builds that run at once take turns on them.  Smaller transfers use plain hipMemcpyAsync.
constexpr size_t kStageSlot = (size_t)32 << 20, kStageMin = (size_t)4 << 20;
constexpr int kStageSlots = 4, kCopyThreads = 8, kStageDevices = 64;

struct HostSeg {
    char* host;
    char* dev;
    size_t bytes;
};

struct PinnedStage {
    std::mutex mu;
    char* buf = nullptr;
    hipEvent_t ev[kStageSlots] = {};
    bool failed = false;   // the pinned allocation failed once: plain copies from then on

    bool ready() {   // under mu, with the stage's device current
        if (buf) return true;
        if (failed) return false;
        if (hipHostMalloc((void**)&buf, kStageSlot * kStageSlots, hipHostMallocDefault) != hipSuccess) {
            buf = nullptr;
            failed = true;
            return false;
        }
        for (int i = 0; i < kStageSlots; i++)
            if (hipEventCreateWithFlags(&ev[i], hipEventDisableTiming) != hipSuccess) {
                failed = true;
                return false;   // buf stays allocated and unused
            }
        return true;
    }
};

PinnedStage* stage_for_current_device() {
    static PinnedStage stages[kStageDevices];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kStageDevices) return nullptr;
    return &stages[dev];
}

// memcpy split over up to kCopyThreads threads (64-byte aligned pieces).
void par_copy(char* dst, const char* src, size_t bytes) {
    const int T = bytes >= ((size_t)1 << 22) ? kCopyThreads : 1;
    const size_t per = ((bytes + T - 1) / T + 63) & ~(size_t)63;
    std::thread th[kCopyThreads];
    for (int t = 1; t < T; t++) {
        const size_t a = std::min(bytes, per * t), b = std::min(bytes, a + per);
        if (b > a) th[t] = std::thread([=]() { std::memcpy(dst + a, src + a, b - a); });
    }
    std::memcpy(dst, src, std::min(bytes, per));
    for (int t = 1; t < T; t++)
        if (th[t].joinable()) th[t].join();
}

std::vector<HostSeg> chunks_of(const HostSeg* segs, int nseg, size_t& total) {
    std::vector<HostSeg> c;
    total = 0;
    for (int i = 0; i < nseg; i++) {
        total += segs[i].bytes;
        for (size_t off = 0; off < segs[i].bytes; off += kStageSlot)
            c.push_back(HostSeg{segs[i].host + off, segs[i].dev + off, std::min(kStageSlot, segs[i].bytes - off)});
    }
    return c;
}

// Host -> device; the copies are complete on the host side when it returns, and ordered before later
// work on st.
hipError_t stage_h2d(const HostSeg* segs, int nseg, hipStream_t st) {
    size_t total = 0;
    const std::vector<HostSeg> c = chunks_of(segs, nseg, total);
    PinnedStage* S = total >= kStageMin ? stage_for_current_device() : nullptr;
    std::unique_lock<std::mutex> lk;
    if (S) {
        lk = std::unique_lock<std::mutex>(S->mu);
        if (!S->ready()) S = nullptr;
    }
    if (!S) {
        for (int i = 0; i < nseg; i++) {
            if (segs[i].bytes == 0) continue;
            const hipError_t e = hipMemcpyAsync(segs[i].dev, segs[i].host, segs[i].bytes, hipMemcpyHostToDevice, st);
            if (e != hipSuccess) return e;
        }
        return hipSuccess;
    }
    for (size_t k = 0; k < c.size(); k++) {
        const int slot = (int)(k % kStageSlots);
        char* sb = S->buf + (size_t)slot * kStageSlot;
        // the slot's previous DMA (this call's, or an earlier call's that returned early) must be done
        // before it is refilled; an event never recorded completes at once
        const hipError_t w = hipEventSynchronize(S->ev[slot]);
        if (w != hipSuccess) return w;
        par_copy(sb, c[k].host, c[k].bytes);
        hipError_t e = hipMemcpyAsync(c[k].dev, sb, c[k].bytes, hipMemcpyHostToDevice, st);
        if (e == hipSuccess) e = hipEventRecord(S->ev[slot], st);
        if (e != hipSuccess) return e;
    }
    // the slots are free for the next user only once their DMAs are done
    for (size_t k = c.size() > (size_t)kStageSlots ? c.size() - kStageSlots : 0; k < c.size(); k++) {
        const hipError_t e = hipEventSynchronize(S->ev[k % kStageSlots]);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

// Device -> host after the work already on st; the host arrays are complete when it returns.
hipError_t stage_d2h(const HostSeg* segs, int nseg, hipStream_t st) {
    size_t total = 0;
    const std::vector<HostSeg> c = chunks_of(segs, nseg, total);
    PinnedStage* S = total >= kStageMin ? stage_for_current_device() : nullptr;
    std::unique_lock<std::mutex> lk;
    if (S) {
        lk = std::unique_lock<std::mutex>(S->mu);
        if (!S->ready()) S = nullptr;
    }
    if (!S) {
        for (int i = 0; i < nseg; i++) {
            if (segs[i].bytes == 0) continue;
            const hipError_t e = hipMemcpyAsync(segs[i].host, segs[i].dev, segs[i].bytes, hipMemcpyDeviceToHost, st);
            if (e != hipSuccess) return e;
        }
        return hipStreamSynchronize(st);
    }
    // chunk k's DMA is issued before chunk k - 1 is copied out on the host; a slot is refilled only
    // after its previous chunk was copied out (kStageSlots >= 2)
    auto drain = [&](size_t k) -> hipError_t {
        const int slot = (int)(k % kStageSlots);
        const hipError_t e = hipEventSynchronize(S->ev[slot]);
        if (e != hipSuccess) return e;
        par_copy(c[k].host, S->buf + (size_t)slot * kStageSlot, c[k].bytes);
        return hipSuccess;
    };
    for (size_t k = 0; k < c.size(); k++) {
        const int slot = (int)(k % kStageSlots);
        if (k < (size_t)kStageSlots) {   // a DMA into the slot left by an earlier call that returned early
            const hipError_t w = hipEventSynchronize(S->ev[slot]);
            if (w != hipSuccess) return w;
        }
        char* sb = S->buf + (size_t)slot * kStageSlot;
        hipError_t e = hipMemcpyAsync(sb, c[k].dev, c[k].bytes, hipMemcpyDeviceToHost, st);
        if (e == hipSuccess) e = hipEventRecord(S->ev[slot], st);
        if (e == hipSuccess && k >= 1) e = drain(k - 1);
        if (e != hipSuccess) return e;
    }
    if (!c.empty()) return drain(c.size() - 1);
    return hipSuccess;
}


// The device memory of one build: carved from one allocation sized for the element arrays and the usual
// small ones (a build made 28 allocations and as many frees, each a synchronisation: 0.6 ms of 3.8 at
// 300,001 elements), with further slabs where it does not suffice.  Freed together.
struct Arena {
    std::vector<void*> slabs;
    char* cur = nullptr;
    size_t left = 0;
    Arena() = default;
    Arena(const Arena&) = delete;
    Arena& operator=(const Arena&) = delete;
    ~Arena() { for (void* p : slabs) (void)hipFree(p); }
    static size_t padded(size_t bytes) { return (bytes + 255) & ~(size_t)255; }
    hipError_t slab(size_t bytes) {
        void* p = nullptr;
        const hipError_t e = hipMalloc(&p, bytes);
        if (e != hipSuccess) return e;
        slabs.push_back(p);
        cur = (char*)p;
        left = bytes;
        return hipSuccess;
    }
    hipError_t take(size_t bytes, void** out) {
        bytes = padded(bytes);
        if (bytes > left) {
            const hipError_t e = slab(std::max(bytes, (size_t)1 << 20));
            if (e != hipSuccess) return e;
        }
        *out = cur;
        cur += bytes;
        left -= bytes;
        return hipSuccess;
    }
};

template <class T>
struct DevBuf {
    Arena& arena;
    T* p = nullptr;
    size_t cap = 0;
    explicit DevBuf(Arena& a) : arena(a) {}
    DevBuf(const DevBuf&) = delete;
    DevBuf& operator=(const DevBuf&) = delete;
    hipError_t alloc(size_t n) {   // contents are not kept when it grows
        n = std::max<size_t>(n, 1);
        if (n <= cap) return hipSuccess;
        void* q = nullptr;
        const hipError_t e = arena.take(n * sizeof(T), &q);
        if (e == hipSuccess) { p = (T*)q; cap = n; }
        return e;
    }
};

// A node above the subtrees, assembled on the host from the splits of its range.
struct TopNode {
    int start, n;
    int axis[3];
    int lo[5];      // child c covers [lo[c], lo[c + 1]) within the node's range
    int kind[4];    // 0 leaf, 1 top node, 2 subtree
    int ref[4];     // leaf, top node or subtree index
    int index;      // pre-order index
};

#define BUILD_TRY(x)                         \
    do {                                     \
        if ((x) != hipSuccess) return -2;    \
    } while (0)

// One batch of device-wide splits, src -> dst over `ranges` ({start, n}); (axis, pivot) per range
// into `out`.
struct SegRunner {
    hipStream_t st;
    int leafMax, chunk;
    DevBuf<int> d_work, d_rpart;     // the tasks, then the task of every chunk
    DevBuf<SegParam> d_params;
    DevBuf<KeyBox> d_cbpart;
    DevBuf<BinPart> d_binpart;
    std::vector<SegTask> tasks;
    std::vector<int> chunk_task, work;
    std::vector<SegParam> params;

    SegRunner(Arena& a, hipStream_t s, int leaf_max, int chunk_elems)
        : st(s), leafMax(leaf_max), chunk(chunk_elems), d_work(a), d_rpart(a), d_params(a), d_cbpart(a), d_binpart(a) {}

    int run(const GElem* src, GElem* dst, const std::vector<int2>& ranges, int* rl, int* lr, int* err,
            std::vector<int2>& out) {
        tasks.clear();
        chunk_task.clear();
        for (size_t i = 0; i < ranges.size(); i++) {
            const int nch = std::max(1, (ranges[i].y + chunk - 1) / chunk);
            tasks.push_back(SegTask{ranges[i].x, ranges[i].y, (int)chunk_task.size(), nch, chunk});
            for (int k = 0; k < nch; k++) chunk_task.push_back((int)i);
        }
        const unsigned nt = (unsigned)tasks.size(), nc = (unsigned)chunk_task.size();
        constexpr size_t kTaskInts = sizeof(SegTask) / sizeof(int);
        work.resize(nt * kTaskInts + nc);
        std::memcpy(work.data(), tasks.data(), nt * sizeof(SegTask));
        std::memcpy(work.data() + nt * kTaskInts, chunk_task.data(), nc * sizeof(int));
        BUILD_TRY(d_work.alloc(work.size()));
        BUILD_TRY(d_params.alloc(nt));
        BUILD_TRY(d_rpart.alloc(nc));
        BUILD_TRY(d_cbpart.alloc(nc));
        BUILD_TRY(d_binpart.alloc(nc));
        BUILD_TRY(hipMemcpyAsync(d_work.p, work.data(), work.size() * sizeof(int), hipMemcpyHostToDevice, st));
        const SegTask* d_tasks = (const SegTask*)d_work.p;
        const int* d_chunk_task = d_work.p + nt * kTaskInts;
        const dim3 blk(kSegThreads);
        hipLaunchKernelGGL(k_seg_cb, dim3(nc), blk, 0, st, src, d_tasks, d_chunk_task, leafMax, d_cbpart.p);
        hipLaunchKernelGGL(k_seg_bins, dim3(nc), blk, 0, st, src, d_tasks, d_chunk_task, d_cbpart.p, leafMax,
                           d_params.p, d_binpart.p, err);
        hipLaunchKernelGGL(k_seg_sah, dim3(nt), blk, 0, st, src, d_tasks, d_binpart.p, d_params.p);
        hipLaunchKernelGGL(k_seg_rcount, dim3(nc), blk, 0, st, src, d_tasks, d_chunk_task, d_params.p, d_rpart.p);
        hipLaunchKernelGGL(k_seg_rank, dim3(nc), blk, 0, st, src, d_tasks, d_chunk_task, d_params.p, d_rpart.p, rl,
                           lr, err);
        hipLaunchKernelGGL(k_seg_scatter, dim3(nc), blk, 0, st, src, dst, d_tasks, d_chunk_task, d_params.p,
                           d_rpart.p, rl, lr, err);
        BUILD_TRY(hipGetLastError());
        params.resize(nt);
        BUILD_TRY(hipMemcpyAsync(params.data(), d_params.p, nt * sizeof(SegParam), hipMemcpyDeviceToHost, st));
        BUILD_TRY(hipStreamSynchronize(st));
        out.resize(nt);
        for (unsigned i = 0; i < nt; i++) out[i] = make_int2(params[i].axis, params[i].pivot);
        return 0;
    }
};

}  // namespace

hipError_t stage_upload(void* dev, const void* host, size_t bytes, hipStream_t st) {
    const HostSeg seg{(char*)host, (char*)dev, bytes};
    return stage_h2d(&seg, 1, st);
}

int build_qbvh_gpu(float* boxes, float* centroids, int32_t* idx, int32_t n, int32_t leafMax,
                   vgpu_qbvh_node* nodes_out, int32_t max_nodes, int32_t* nnodes_out, float* bounds_out,
                   hipStream_t st) {
    if (n < 0 || !nnodes_out || (n > 0 && (!boxes || !centroids || !idx))) return -1;
    if (n > (1 << 28)) return -1;   // leaf codes hold 28 bits of element offset
    if (leafMax > 16) leafMax = 16;
    if (leafMax < 1) leafMax = 1;
    const size_t N = (size_t)std::max(n, 1);
    // boxes, centroids, indices, elements (twice with ranges to split), ranks, pre-order numbers, scratch
    // nodes; and a 16th of those again for the final nodes (leafMax 16 makes one per 22 elements) and the small arrays
    Arena arena;
    const size_t per = 40 + sizeof(GElem) + 4 + sizeof(vgpu_qbvh_node) + (n > kSubtreeMax ? sizeof(GElem) + 8 : 0);
    BUILD_TRY(arena.slab(N * per + N * sizeof(vgpu_qbvh_node) / 16 + ((size_t)1 << 18)));
    DevBuf<float> d_boxes(arena), d_cent(arena), d_rootbox(arena), d_leafbox(arena);
    DevBuf<int32_t> d_idx(arena);
    DevBuf<GElem> d_E(arena), d_T(arena);
    DevBuf<int> d_rl(arena), d_lr(arena), d_err(arena), d_counts(arena), d_src(arena), d_dst(arena), d_pre(arena);
    DevBuf<int2> d_roots(arena), d_leaves(arena);
    DevBuf<vgpu_qbvh_node> d_scratch(arena), d_nodes(arena);
    BUILD_TRY(d_boxes.alloc(N * 6));
    BUILD_TRY(d_cent.alloc(N * 3));
    BUILD_TRY(d_idx.alloc(N));
    BUILD_TRY(d_E.alloc(N));
    BUILD_TRY(d_err.alloc(1));
    BUILD_TRY(d_pre.alloc(N));
    BUILD_TRY(d_scratch.alloc(N));
    BUILD_TRY(hipMemsetAsync(d_err.p, 0, sizeof(int), st));
    if (n > 0) {
        const HostSeg in[3] = {{(char*)boxes, (char*)d_boxes.p, sizeof(float) * 6 * n},
                               {(char*)centroids, (char*)d_cent.p, sizeof(float) * 3 * n},
                               {(char*)idx, (char*)d_idx.p, sizeof(int32_t) * n}};
        BUILD_TRY(stage_h2d(in, 3, st));
        hipLaunchKernelGGL(k_pack, dim3((n + 255) / 256), dim3(256), 0, st, d_boxes.p, d_cent.p, d_idx.p, n, d_E.p,
                           d_err.p);
        BUILD_TRY(hipGetLastError());
        int bad = 0;
        BUILD_TRY(hipMemcpyAsync(&bad, d_err.p, sizeof(int), hipMemcpyDeviceToHost, st));
        BUILD_TRY(hipStreamSynchronize(st));
        if (bad) return -3;
    }
    std::vector<TopNode> top;
    std::vector<int2> subtrees, leaves;   // {start, n}
    std::vector<int> level;
    auto add_child = [&](int start, int cn, int& kind, int& ref) {
        if (cn <= leafMax) {
            kind = 0;
            ref = (int)leaves.size();
            leaves.push_back(make_int2(start, cn));
        } else if (cn <= kSubtreeMax) {
            kind = 2;
            ref = (int)subtrees.size();
            subtrees.push_back(make_int2(start, cn));
        } else {
            kind = 1;
            ref = (int)top.size();
            TopNode tn{};
            tn.start = start;
            tn.n = cn;
            top.push_back(tn);
            level.push_back(ref);
        }
    };
    // the root is a top node when its range is large; otherwise one subtree builds the whole tree
    // (a root of at most leafMax elements included: the reference still makes a node for it)
    const int root_kind = n > kSubtreeMax ? 1 : 2;
    if (root_kind == 1) {
        TopNode r{};
        r.start = 0;
        r.n = n;
        top.push_back(r);
        level.push_back(0);
        BUILD_TRY(d_T.alloc(N));
        BUILD_TRY(d_rl.alloc(N));
        BUILD_TRY(d_lr.alloc(N));
    } else {
        subtrees.push_back(make_int2(0, n));
    }
    SegRunner seg(arena, st, leafMax, n < kChunkLargeFrom ? kChunkSmall : kChunkLarge);
    std::vector<int2> ranges, r0, r12;
    while (!level.empty()) {
        const std::vector<int> cur = level;
        level.clear();
        ranges.clear();
        for (int i : cur) ranges.push_back(make_int2(top[i].start, top[i].n));
        int rc = seg.run(d_E.p, d_T.p, ranges, d_rl.p, d_lr.p, d_err.p, r0);
        if (rc) return rc;
        ranges.clear();
        for (size_t k = 0; k < cur.size(); k++) {
            const TopNode& tn = top[cur[k]];
            ranges.push_back(make_int2(tn.start, r0[k].y));
            ranges.push_back(make_int2(tn.start + r0[k].y, tn.n - r0[k].y));
        }
        rc = seg.run(d_T.p, d_E.p, ranges, d_rl.p, d_lr.p, d_err.p, r12);
        if (rc) return rc;
        for (size_t k = 0; k < cur.size(); k++) {
            const int ti = cur[k];
            const int p0 = r0[k].y, p1 = r12[2 * k].y, p2 = r12[2 * k + 1].y;
            top[ti].axis[0] = r0[k].x;
            top[ti].axis[1] = r12[2 * k].x;
            top[ti].axis[2] = r12[2 * k + 1].x;
            const int lo[5] = {0, p1, p0, p0 + p2, top[ti].n};
            for (int c = 0; c < 5; c++) top[ti].lo[c] = lo[c];
            for (int c = 0; c < 4; c++) {
                // a valid split leaves both sides of the first split non-empty; a child as large as
                // its parent only comes from bins already flagged as broken
                if (lo[c + 1] - lo[c] >= top[ti].n || lo[c + 1] < lo[c]) return -3;
                int kind, ref;
                add_child(top[ti].start + lo[c], lo[c + 1] - lo[c], kind, ref);
                top[ti].kind[c] = kind;
                top[ti].ref[c] = ref;
            }
        }
    }
    const int nsub = (int)subtrees.size();
    std::vector<int> counts(std::max(nsub, 1), 0);
    std::vector<float> rootbox((size_t)std::max(nsub, 1) * 6, 0.0f);
    if (nsub > 0) {
        BUILD_TRY(d_roots.alloc(nsub));
        BUILD_TRY(d_counts.alloc(nsub));
        BUILD_TRY(d_rootbox.alloc((size_t)nsub * 6));
        BUILD_TRY(hipMemcpyAsync(d_roots.p, subtrees.data(), nsub * sizeof(int2), hipMemcpyHostToDevice, st));
        hipLaunchKernelGGL(k_subtree, dim3(nsub), dim3(kSubThreads), 0, st, d_E.p, d_roots.p, d_scratch.p, d_pre.p,
                           d_counts.p, d_rootbox.p, leafMax, d_err.p);
        BUILD_TRY(hipGetLastError());
        BUILD_TRY(hipMemcpyAsync(counts.data(), d_counts.p, nsub * sizeof(int), hipMemcpyDeviceToHost, st));
        BUILD_TRY(hipMemcpyAsync(rootbox.data(), d_rootbox.p, (size_t)nsub * 6 * sizeof(float), hipMemcpyDeviceToHost,
                                 st));
    }
    const int nleaf = (int)leaves.size();
    std::vector<float> leafbox((size_t)std::max(nleaf, 1) * 6, 0.0f);
    if (nleaf > 0) {
        BUILD_TRY(d_leaves.alloc(nleaf));
        BUILD_TRY(d_leafbox.alloc((size_t)nleaf * 6));
        BUILD_TRY(hipMemcpyAsync(d_leaves.p, leaves.data(), nleaf * sizeof(int2), hipMemcpyHostToDevice, st));
        hipLaunchKernelGGL(k_leaf_boxes, dim3((nleaf + 255) / 256), dim3(256), 0, st, d_E.p, d_leaves.p, nleaf,
                           d_leafbox.p);
        BUILD_TRY(hipGetLastError());
        BUILD_TRY(hipMemcpyAsync(leafbox.data(), d_leafbox.p, (size_t)nleaf * 6 * sizeof(float), hipMemcpyDeviceToHost,
                                 st));
    }
    int err = 0;
    BUILD_TRY(hipMemcpyAsync(&err, d_err.p, sizeof(int), hipMemcpyDeviceToHost, st));
    BUILD_TRY(hipStreamSynchronize(st));
    if (err & 7) return -3;
    if (err) return -4;
    // pre-order numbering: a top node takes the next index, then its children in order; a subtree
    // takes a block of its node count
    std::vector<int> sub_dst(std::max(nsub, 1), 0);
    int next = 0;
    std::vector<std::pair<int, int>> stack{{root_kind, 0}};
    while (!stack.empty()) {
        const std::pair<int, int> it = stack.back();
        stack.pop_back();
        if (it.first == 2) {
            sub_dst[it.second] = next;
            next += counts[it.second];
            continue;
        }
        top[it.second].index = next++;
        for (int c = 3; c >= 0; c--)
            if (top[it.second].kind[c] != 0) stack.push_back({top[it.second].kind[c], top[it.second].ref[c]});
    }
    const int total = next;
    *nnodes_out = total;
    if (total > max_nodes || !nodes_out) return -1;
    BUILD_TRY(d_nodes.alloc(total));
    if (nsub > 0) {
        std::vector<int> src(nsub);
        for (int s = 0; s < nsub; s++) src[s] = subtrees[s].x;
        BUILD_TRY(d_src.alloc(nsub));
        BUILD_TRY(d_dst.alloc(nsub));
        BUILD_TRY(hipMemcpyAsync(d_src.p, src.data(), nsub * sizeof(int), hipMemcpyHostToDevice, st));
        BUILD_TRY(hipMemcpyAsync(d_dst.p, sub_dst.data(), nsub * sizeof(int), hipMemcpyHostToDevice, st));
        hipLaunchKernelGGL(k_place, dim3(nsub), dim3(256), 0, st, d_scratch.p, d_pre.p, d_src.p, d_dst.p,
                           d_counts.p, d_nodes.p);
        BUILD_TRY(hipGetLastError());
    }
    if (n > 0) {
        hipLaunchKernelGGL(k_unpack, dim3((n + 255) / 256), dim3(256), 0, st, d_E.p, n, d_boxes.p, d_cent.p, d_idx.p);
        BUILD_TRY(hipGetLastError());
    }
    const HostSeg out[4] = {{(char*)nodes_out, (char*)d_nodes.p, (size_t)total * sizeof(vgpu_qbvh_node)},
                            {(char*)boxes, (char*)d_boxes.p, n > 0 ? sizeof(float) * 6 * n : 0},
                            {(char*)centroids, (char*)d_cent.p, n > 0 ? sizeof(float) * 3 * n : 0},
                            {(char*)idx, (char*)d_idx.p, n > 0 ? sizeof(int32_t) * n : 0}};
    BUILD_TRY(stage_d2h(out, 4, st));
    BUILD_TRY(hipStreamSynchronize(st));
    // the top nodes, children before parents (reverse creation order), with MINSS / MAXSS unions
    const float kInf = std::numeric_limits<float>::infinity();
    auto fmin_ss = [](float x, float y) { return (x < y) ? x : y; };
    auto fmax_ss = [](float x, float y) { return (x > y) ? x : y; };
    std::vector<float> topbox(top.size() * 6);
    for (int ti = (int)top.size() - 1; ti >= 0; ti--) {
        const TopNode& tn = top[ti];
        vgpu_qbvh_node nd;
        std::memset(&nd, 0, sizeof(nd));
        nd.axis0 = (uint32_t)tn.axis[0];
        nd.axis1 = (uint32_t)tn.axis[1];
        nd.axis2 = (uint32_t)tn.axis[2];
        float nb[6] = {kInf, kInf, kInf, -kInf, -kInf, -kInf};
        for (int c = 0; c < 4; c++) {
            const int cn = tn.lo[c + 1] - tn.lo[c];
            const float* b;
            if (tn.kind[c] == 0) {
                if (cn == 0) {
                    nd.children[c] = -1;
                    for (int k = 0; k < 3; k++) { nd.boxes[c + k * 4] = kInf; nd.boxes[c + 12 + k * 4] = kInf; }
                    continue;
                }
                b = &leafbox[(size_t)tn.ref[c] * 6];
                const uint32_t first = (uint32_t)(tn.start + tn.lo[c]);
                nd.children[c] = (int32_t)((1u << 31) | ((first << 4) & 0xfffffff0u) | ((uint32_t)(cn - 1) & 0xfu));
            } else if (tn.kind[c] == 1) {
                b = &topbox[(size_t)tn.ref[c] * 6];
                nd.children[c] = top[tn.ref[c]].index;
            } else {
                b = &rootbox[(size_t)tn.ref[c] * 6];
                nd.children[c] = sub_dst[tn.ref[c]];
            }
            for (int k = 0; k < 3; k++) { nd.boxes[c + k * 4] = b[k]; nd.boxes[c + 12 + k * 4] = b[3 + k]; }
            for (int k = 0; k < 3; k++) { nb[k] = fmin_ss(nb[k], b[k]); nb[3 + k] = fmax_ss(nb[3 + k], b[3 + k]); }
        }
        std::memcpy(&topbox[(size_t)ti * 6], nb, sizeof(nb));
        nodes_out[tn.index] = nd;
    }
    if (bounds_out) std::memcpy(bounds_out, root_kind == 1 ? &topbox[0] : &rootbox[0], 6 * sizeof(float));
    return 0;
}

}  // namespace vgpu
