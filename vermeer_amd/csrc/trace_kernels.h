// Internal interface between the scene object (scene.cpp) and the
// traversal kernels (trace.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>

#include "xform.h"

namespace vgpu {

// Idle lanes that trigger a refill of the wavefront in the traversal kernel; 48 of 64 measured
// fastest on incoherent bounce rays (64: refill only when the whole wavefront is idle).
constexpr int kRefillDefault = 48;

// Direction-sign bit of axis 0 in the traversal's packed ray word, and the bias of the split axes that
// nodes hold.
constexpr int kSignBit = 4;

// Device node, 128 bytes = one cache line: qbvh.Node (qbvh/qbvh.go:31-36) re-laid as eight 16-byte rows
// (lane c = child c).  The two bounds of axis k lie in rows whose byte offsets differ in one bit, 16, 32
// and 64 for x, y and z, so a ray's near and far planes are single loads at offsets made from its
// direction signs.  The bounds are in order (lo <= hi): the upload swaps the lanes that are not, the
// reference's empty box (+inf, -inf) above all, whose slab values are the same either way round.
constexpr int kRowLoX = 0, kRowHiX = 1, kRowLoY = 4, kRowHiY = 6, kRowLoZ = 3, kRowHiZ = 7, kRowChildren = 2, kRowAxes = 5;
struct alignas(16) DevNode {
    float rows[8][4];
    // rows[kRowChildren]: int32, the reference's encoding, node indices relative to the geom's node base
    // rows[kRowAxes]: int32 kSignBit + axis0, axis1, axis2; then bit 4 k + c set where the upload swapped
    // axis k of child c
};
static_assert(sizeof(DevNode) == 128, "DevNode is one 128-byte line");

// Motion node (qbvh.MotionNode + its per-key MotionNodeBoxes): a 32-byte topology record (children,
// then axes as kSignBit + axis) followed by nkeys box blocks of 96 bytes: lo x, hi x, lo y, hi y, lo z,
// hi z as float4 rows.  Stride in float4 units: 2 + 6*nkeys, so a row pair starts on 32 bytes.

// A static triangle: three vertices without padding, 36 bytes.  Leaf tests read runs of consecutive
// triangles, so the lines fetched shrink with the record (48 bytes as three float4 before: the 5.2M-triangle
// field falls from 250 to 190 MB and, nodes included, under the 256 MB of the last-level cache).
struct DevTri {
    float v[3][3];
};
static_assert(sizeof(DevTri) == 36, "DevTri is nine floats");

// Geom table entry.  Static geom: node_base indexes DevNode, tri_base indexes
// triangles (DevTri).  Motion geom:
// node_base/tri_base are float4 offsets into the motion arrays; a motion
// triangle is nkeys consecutive groups of 3 float4.
struct alignas(16) DevGeom {
    int32_t node_base;
    int32_t tri_base;
    int32_t nkeys;      // 1 = static
    float ray_bias;     // PolyMesh.RayBias (builtin/geom/polymesh/polymesh.go:19)
};

// Per geom slot: the transform a geom applies to rays before tracing what it holds.  kind:
//   kXfNone      a mesh or sphere without a transform
//   kXfMesh      a PolyMesh with its own Transform (builtin/geom/polymesh/trace.go:20-74)
//   kXfInstance  a GeomInstance of child 0 (builtin/geom/instance/instance.go:73-114)
//   kXfProc      a Proc over its children, in order (builtin/geom/proc/proc.go:88-139)
// One key: M and M^-1 precomputed at mat_base (32 floats; a mesh's single key is its raw matrix, an
// instance's or proc's the recomposed TransformDecomp).  More: nkeys TransformDecomp records
// (kXfKeyFloats each) at key_base, interpolated at the ray's time.
constexpr int kXfNone = 0, kXfMesh = 1, kXfInstance = 2, kXfProc = 3;
struct alignas(16) DevXform {
    int32_t kind;
    int32_t nkeys;
    int32_t key_base;      // float offset in SceneView::xkeys (more than one key)
    int32_t mat_base;      // float offset in SceneView::xkeys (one key)
    int32_t child_base;    // first entry in SceneView::xchildren (instances and procs: geom slots)
    int32_t nchild;
    int32_t pad0, pad1;
};

// The transform of a geom at a ray's time and its inverse (a singular matrix inverts to zero, as
// Matrix4Inverse leaves it).  Keys as polymesh/trace.go:27-44 and TransformSRTArray.TimeKey
// (instance.go:17-34) pick them; a time outside [0, 1] is held to the end keys.
__device__ inline void xform_at(const DevXform& x, const float* xkeys, float time, float* M, float* Minv) {
    if (x.nkeys == 1) {
        const float* m = xkeys + x.mat_base;
        for (int i = 0; i < 16; i++) { M[i] = m[i]; Minv[i] = m[16 + i]; }
        return;
    }
    const float k = time * (float)(x.nkeys - 1);
    const float fk = floorf(k);
    const float t = k - fk;
    const int k0 = min(max((int)fk, 0), x.nkeys - 1), k1 = min(max((int)ceilf(k), 0), x.nkeys - 1);
    xf_decomp_matrix(xkeys + x.key_base + k0 * kXfKeyFloats, xkeys + x.key_base + k1 * kXfKeyFloats, t, M);
    if (!xf_inverse(M, Minv))
        for (int i = 0; i < 16; i++) Minv[i] = 0.0f;
}

struct SceneView {
    const DevNode* nodes;     // static nodes: top level at [0, ntop) when the top is static
    const DevTri* tris;       // static triangles
    const float4* mnodes;     // motion nodes (topology + boxes)
    const float4* mtris;      // motion triangles
    const DevGeom* geoms;     // post-sort geom slots
    const float4* spheres;    // analytic sphere geoms (centre, radius), indexed by DevGeom::tri_base
    int32_t top_motion;       // 1: the top level is a motion QBVH at mnodes[top_mbase]
    int32_t top_keys;         // motion keys of the top level
    int32_t top_mbase;
    int32_t near_far;         // 1: box4_near's conditions hold for the nodes: no NaN bound, lo <= hi (motion
                              // boxes: finite too), and both node arrays lie within 32-bit byte offsets
    int32_t any_xform;        // 1: some geom applies a transform (k_trace_xform traces every ray)
    const DevXform* xforms;   // per geom slot (any_xform only)
    const float* xkeys;       // transform records
    const int32_t* xchildren; // geom slots held by instances and procs
};

struct TraceLaunch {
    int block;          // 64, 128, 256
    int lds_depth;      // 8, 12, 16, 24, 32
    int waves_per_cu;   // resident waves per CU used to size the grid
    int refill_min = kRefillDefault;   // idle lanes that make a wavefront take new rays together (1..64)
    int spread = 16;    // waves per CU that a short launch is spread over (trace_ray_shift)
};

// Launch shapes of static and motion scenes: of launch_trace_ext (the shading passes' closest-hit traversal; callers
// size the spill area for the larger grid) and of every other traversal where the caller chose none.
// The static kernel holds 86 to 88 VGPRs, five waves per SIMD: a grid of 20 waves per CU fills them and leaves no
// workgroup waiting (2.1M bounce rays, block 64: 706 us at 20 waves per CU, 743 at 16, 898 at 24; block 128: 703 at 20,
// 910 at 24).
// The motion kernel holds 112 VGPRs, four waves per SIMD.  Held to 96 (four spilled, and their reloads lie in the loop) it
// fitted five, and was slower.  Among moving spheres, this shape against five waves at 64 / 8 / 20, in us: 1M camera rays
// 591 against 687, 1M shadow rays from them 533 against 633, 1M uniform shadow rays 758 against 1010, 20,011 uniform
// rays 130 against 176, 1,024 rays 59 against 76; a pass over 512^2 pixels 843 against 864.
constexpr TraceLaunch kExtLaunch{64, 12, 20};
constexpr TraceLaunch kExtLaunchMotion{256, 16, 16};

// Launch shape of the traversals of a scene with transforms: block and LDS depth are its kernel's, waves per CU and
// refill threshold the scene's (these waves where the caller chose none, and in launch_trace_ext).
// Spread over 4 / 8 / 16 waves per CU: 5,003 rays take 328 / 268 / 261 us, 50,000 take 471 / 472 / 475, 120,001 take
// 533 / 533 / 573.
constexpr TraceLaunch kXformLaunch{64, 12, 16, kRefillDefault, 8};
static_assert(kXformLaunch.waves_per_cu <= kExtLaunch.waves_per_cu && kXformLaunch.waves_per_cu <= kExtLaunchMotion.waves_per_cu,
              "the shading passes' spill areas cover it");
inline TraceLaunch scene_launch(const SceneView& sv, const TraceLaunch& cfg) {
    if (!sv.any_xform) return cfg;
    TraceLaunch l = kXformLaunch;
    l.waves_per_cu = cfg.waves_per_cu;
    l.refill_min = cfg.refill_min;
    return l;
}

// Scratch of the ray sort (raysort.hip), sized for `capacity` rays.
struct RaySortBuffers {
    uint32_t* keys;      // capacity
    uint32_t* perm;      // capacity: sorted position -> original ray index
    float4* rays;        // 2 * capacity: sorted rays
    uint32_t* hist;      // ray_sort_buckets(bits) counters
    uint32_t* bsum;      // ray_sort_scan_blocks(bits)
    uint64_t capacity;
};
uint32_t ray_sort_buckets(int bits);
uint32_t ray_sort_scan_blocks(int bits);
// Sorts min(n, *n_dev) rays into sb.rays / sb.perm by (Morton cell of the origin in a 2^bits grid over
// box = lo xyz, hi xyz) x (direction octant); bits in [1,6].  list (nullable): ray i is the one at slot list[i], and
// sb.perm holds slots.
hipError_t launch_ray_sort(const float* box, int bits, const void* rays, uint64_t n, const uint32_t* n_dev,
                           const RaySortBuffers& sb, int num_cus, hipStream_t stream, const uint32_t* list = nullptr);

// Enqueues one traversal over n rays (device pointers).  spill_T / spill_N
// hold (VGPU_MAX_STACK - lds_depth) entries per spill column; the launch
// fails if it needs more than spill_columns.  n_dev (nullable): a device-resident
// ray count; the kernel traces min(n, *n_dev) rays (n sizes the grid).  perm (nullable):
// ray i's results go to slot perm[i] (rays reordered by launch_ray_sort); with gather, ray i is the one
// at slot perm[i] and its results go there (a list of the slots to trace).  cfg: a scene_launch shape.
// Returns hipSuccess or the launch error.
hipError_t launch_trace(const SceneView& sv, bool shadow, bool motion, const TraceLaunch& cfg,
                        const void* rays, uint64_t n, void* hits, int32_t* geoms, int32_t* counters,
                        float* spill_T, int32_t* spill_N, uint64_t spill_columns, int32_t* err_flag,
                        int num_cus, hipStream_t stream, const uint32_t* n_dev = nullptr,
                        const uint32_t* perm = nullptr, bool gather = false);

// Closest hit with 32-byte records {prim, geom, t, U, V, W, 0, 0} (U, V, W: barycentric weights of the
// triangle's three vertices), for the shading kernels.  Launch shape kExtLaunch, or kExtLaunchMotion
// with motion.
hipError_t launch_trace_ext(const SceneView& sv, bool motion, const void* rays, uint64_t n, void* hits32, float* spill_T,
                            int32_t* spill_N, uint64_t spill_columns, int32_t* err_flag, int num_cus, hipStream_t stream,
                            const uint32_t* n_dev = nullptr);

// Rays that a wavefront takes at a time, as a shift: 64, or fewer when that would leave wavefronts for fewer
// than cfg.spread per CU.  A short launch lasts as long as its slowest wavefront, and one with fewer rays
// diverges less, its idle lanes working in the leaf tests: 4096 pinhole rays over the sphere take 47 us
// instead of 72, 50,000 bounce rays in the field 86 instead of 101, 1024 rays among moving spheres 59 instead of 107.
int trace_ray_shift(const TraceLaunch& cfg, uint64_t n, int num_cus);
// Spill columns of a launch: a lane that can own a ray has one.  A column per launched thread made the spill area of
// a short launch four times as large as its rays need, and its allocation is part of a scene's first pass
// (65,536 pinhole rays: 460 us, now 91).  Rounded up to 256: min(n, resident lanes) rounded is then the same for
// every shape, so an area sized by one shape serves a launch of as many rays by a shape with no more waves.
uint64_t trace_spill_columns(const TraceLaunch& cfg, uint64_t n, int num_cus);

// Threads of a launch.
uint64_t trace_grid_threads(const TraceLaunch& cfg, uint64_t n, int num_cus);

// Allocation-free traversal (vgpu_trace_noalloc): the spill area and error flag live in a
// file-scope device array of kNoAllocScratchBytes in trace.hip, one copy per GPU.
constexpr uint64_t kNoAllocScratchBytes = 128ull << 20;
constexpr int kNoAllocMaxDevices = 64;
// Looks the array up on `device`, which must be current; once per device (later calls return at once).
hipError_t noalloc_init(int device);
// Spill columns that fit the array at LDS depth lds_depth.
uint64_t noalloc_max_columns(int lds_depth);
// Clears the error flag (status, or the array's own flag word when status is NULL) with a kernel,
// then enqueues launch_trace with the array as its spill area.  The grid of cfg must fit
// noalloc_max_columns.  hipErrorNotInitialized: noalloc_init has not run on `device`.
hipError_t launch_trace_noalloc(int device, const SceneView& sv, bool shadow, bool motion, const TraceLaunch& cfg,
                                const void* rays, uint64_t n, void* hits, int32_t* geoms, int32_t* counters,
                                int32_t* status, int num_cus, hipStream_t stream);

}  // namespace vgpu
