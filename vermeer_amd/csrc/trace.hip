// Ray traversal kernels for gfx950 (MI355X).
//
// One ray per lane.  Each lane runs the reference's two-level traversal —
// scene QBVH over geoms, then the hit geom's triangle QBVH — with the same
// box test lane semantics, the same child push order, the same pop-time
// culling and the same watertight triangle test, so hit IDs, t and
// barycentrics match the reference bit for bit:
//   core/ray.go:103-148                 Ray.Setup
//   qbvh/intersect_amd64.s:13-100       intersectBoxes
//   qbvh/intersect.go:91-246            Trace
//   qbvh/motionintersect.go:22-127      TraceMotion
//   builtin/scene/scene.go:30-97        Scene.Trace / TraceElems
//   builtin/geom/sphere/trace.go:13-103  Sphere.Trace (a SphereLight's analytic sphere)
//   builtin/geom/polymesh/trace.go:108-194, :520-669   TraceElems / TraceMotionElems
//
// The traversal stack (the reference's RenderTask.Traversal.Stack, shared by
// both levels, core/ray.go:153-162) lives in LDS for its first LDS entries,
// laid out lane-minor ([depth][lane]) so lanes never conflict on a bank;
// deeper entries spill to HBM, a column per lane that can own a ray
// (trace_spill_columns), also lane-minor so that lanes at equal depth coalesce.
//
// Compiled with -ffp-contract=off: every float operation rounds as the
// reference's unfused SSE code does.

#include <algorithm>
#include <mutex>

#include "trace_kernels.h"
#include "xform.h"
#include "../../include/vermeer_gpu.h"

namespace vgpu {

namespace {

struct RayS {
    float P[3];
    float Dinv[3];
    float S[3];
    int Kx, Ky, Kz;
    int neg;          // bit k set when D[k] < 0
    float time;
    float tclosest;
};

__device__ __forceinline__ float sel3(float a, float b, float c, int k) { return k == 0 ? a : (k == 1 ? b : c); }

__device__ __forceinline__ float absf(float x) { return __int_as_float(__float_as_int(x) & 0x7fffffff); }

// core/ray.go:103-148
__device__ __forceinline__ void ray_setup(RayS& r, const float D[3]) {
    int Kz = 0;
    if (absf(D[1]) > absf(D[2])) {
        if (absf(D[1]) > absf(D[0])) Kz = 1;
    } else {
        if (absf(D[2]) > absf(D[0])) Kz = 2;
    }
    int Kx = Kz + 1; if (Kx == 3) Kx = 0;
    int Ky = Kx + 1; if (Ky == 3) Ky = 0;
    const float dkz = sel3(D[0], D[1], D[2], Kz);
    if (dkz < 0.0f) { int t = Kx; Kx = Ky; Ky = t; }
    // The reference divides in float64 and rounds the quotient to float32.  For float32
    // operands that double rounding is innocuous (53 >= 2 * 24 + 2 bits: the float64 quotient
    // never lands on a float32 rounding midpoint unless the exact quotient does), so a
    // correctly rounded float32 division gives the same bits.
    r.S[2] = 1.0f / dkz;
    r.S[0] = sel3(D[0], D[1], D[2], Kx) / dkz;
    r.S[1] = sel3(D[0], D[1], D[2], Ky) / dkz;
    for (int k = 0; k < 3; k++) r.Dinv[k] = 1.0f / D[k];
    r.Kx = Kx; r.Ky = Ky; r.Kz = Kz;
    r.neg = (D[0] < 0.0f ? 1 : 0) | (D[1] < 0.0f ? 2 : 0) | (D[2] < 0.0f ? 4 : 0);
}

// One axis slab of intersectBoxes (qbvh/intersect_amd64.s:26-81), NaN rules of MINPS/MAXPS.
__device__ __forceinline__ void slab(float lo, float hi, float o, float di, float& tmin, float& tmax, bool first) {
    const float t1 = (lo - o) * di;
    const float t2 = (hi - o) * di;
    const float m = (t2 < t1) ? t2 : t1;
    const float M = (t2 > t1) ? t2 : t1;
    if (first) { tmin = m; tmax = M; }
    else { tmin = (tmin > m) ? tmin : m; tmax = (tmax < M) ? tmax : M; }
}

struct Box4 {
    float t[4];
    bool h[4];
};

__device__ __forceinline__ void box4(const RayS& r, const float4& lx, const float4& ly, const float4& lz,
                                     const float4& hx, const float4& hy, const float4& hz, Box4& b) {
    const float lxa[4] = {lx.x, lx.y, lx.z, lx.w}, lya[4] = {ly.x, ly.y, ly.z, ly.w}, lza[4] = {lz.x, lz.y, lz.z, lz.w};
    const float hxa[4] = {hx.x, hx.y, hx.z, hx.w}, hya[4] = {hy.x, hy.y, hy.z, hy.w}, hza[4] = {hz.x, hz.y, hz.z, hz.w};
#pragma unroll
    for (int c = 0; c < 4; c++) {
        float tmin, tmax;
        slab(lxa[c], hxa[c], r.P[0], r.Dinv[0], tmin, tmax, true);
        slab(lya[c], hya[c], r.P[1], r.Dinv[1], tmin, tmax, false);
        slab(lza[c], hza[c], r.P[2], r.Dinv[2], tmin, tmax, false);
        const float tn = (0.0f > tmin) ? 0.0f : tmin;   // MAXPS X6,X0 with X0 = 0
        b.t[c] = tn;
        b.h[c] = tn <= tmax;                             // CMPPS $2 (ordered <=)
    }
}

// The same four boxes given by their near and far planes: the lower or the upper bound of an axis,
// whichever the direction's sign meets first.  For boxes with lo <= hi, a finite origin and a finite
// non-zero 1/D no value is NaN, and rounding keeps the order of (lo - P) * Dinv and (hi - P) * Dinv, so
// the near plane's value is intersectBoxes' smaller one.  MINPS/MAXPS then agree with IEEE min/max
// except for which zero of +0/-0 they return, and the entry distances are only ever compared, where
// +0 == -0: the same hit flags and the same traversal for 24 instructions less than sorting each pair.
__device__ __forceinline__ void box4_near(const RayS& r, const float4& nx, const float4& ny, const float4& nz,
                                          const float4& fx, const float4& fy, const float4& fz, Box4& b) {
    const float nxa[4] = {nx.x, nx.y, nx.z, nx.w}, nya[4] = {ny.x, ny.y, ny.z, ny.w}, nza[4] = {nz.x, nz.y, nz.z, nz.w};
    const float fxa[4] = {fx.x, fx.y, fx.z, fx.w}, fya[4] = {fy.x, fy.y, fy.z, fy.w}, fza[4] = {fz.x, fz.y, fz.z, fz.w};
#pragma unroll
    for (int c = 0; c < 4; c++) {
        const float tn = fmaxf(fmaxf(fmaxf((nxa[c] - r.P[0]) * r.Dinv[0], (nya[c] - r.P[1]) * r.Dinv[1]),
                                     (nza[c] - r.P[2]) * r.Dinv[2]), 0.0f);
        const float tx = fminf(fminf((fxa[c] - r.P[0]) * r.Dinv[0], (fya[c] - r.P[1]) * r.Dinv[1]),
                               (fza[c] - r.P[2]) * r.Dinv[2]);
        b.t[c] = tn;
        b.h[c] = tn <= tx;
    }
}

__device__ __forceinline__ int leaf_base(int32_t l) { return (int)((l & 0x7ffffff) >> 4); }
__device__ __forceinline__ int leaf_count(int32_t l) { return (int)((l & 0xf) + 1); }

// Ray quantities the watertight test reads: the shear constants and the permuted origin.
// The axes are held as which of them is axis 0 and which is axis 1.
struct TriRay {
    float S0, S1, S2, Pkx, Pky, Pkz;
    bool x0, x1, y0, y1, z0, z1;
    __device__ __forceinline__ float x(const float4& v) const { return x0 ? v.x : (x1 ? v.y : v.z); }
    __device__ __forceinline__ float y(const float4& v) const { return y0 ? v.x : (y1 ? v.y : v.z); }
    __device__ __forceinline__ float z(const float4& v) const { return z0 ? v.x : (z1 ? v.y : v.z); }
    // from a pack_perm word; the three axes differ, so Kz's masks follow from the others without a compare
    __device__ __forceinline__ void axes(int kp) {
        const int Kx = (kp >> 7) & 3, Ky = (kp >> 9) & 3;
        x0 = Kx == 0; x1 = Kx == 1;
        y0 = Ky == 0; y1 = Ky == 1;
        z0 = !(x0 || y0); z1 = !(x1 || y1);
    }
};


struct TriPre {
    float T, det, fU, fV, fW;
};

// The direction-sign bits and the permutation packed in one register: bit kSignBit + k set when
// D[k] < 0, then Kx, Ky, Kz in two bits each.  Nodes hold their split axes as kSignBit + axis, so the
// sign bit of an axis is one bit-field extract; and the sign bits' values 16, 32 and 64 are the byte
// offsets between a node's near and far rows (box4_near).
__device__ __forceinline__ int pack_perm(const RayS& r) {
    return (r.neg << kSignBit) | (r.Kx << 7) | (r.Ky << 9) | (r.Kz << 11);
}
__device__ __forceinline__ TriRay tri_ray_packed(const RayS& r, int kp) {
    TriRay q;
    q.S0 = r.S[0]; q.S1 = r.S[1]; q.S2 = r.S[2];
    q.axes(kp);
    const float4 P = make_float4(r.P[0], r.P[1], r.P[2], 0.0f);
    q.Pkx = q.x(P);
    q.Pky = q.y(P);
    q.Pkz = q.z(P);
    return q;
}

// Watertight ray/triangle test (builtin/geom/polymesh/trace.go:123-194 static, :556-624 motion),
// the part that does not read the closest distance so far: edge functions (retried in double
// precision when one is zero), the sign test, det != 0 and the near bound.
template <bool MOTION_BOUND>
__device__ __forceinline__ bool tri_pre(const TriRay& q, const float4& v0, const float4& v1, const float4& v2, float bias,
                                        TriPre& p) {
    const float AKz = q.z(v0) - q.Pkz;
    const float BKz = q.z(v1) - q.Pkz;
    const float CKz = q.z(v2) - q.Pkz;
    const float Cx = (q.x(v2) - q.Pkx) - q.S0 * CKz;
    const float By = (q.y(v1) - q.Pky) - q.S1 * BKz;
    const float Cy = (q.y(v2) - q.Pky) - q.S1 * CKz;
    const float Bx = (q.x(v1) - q.Pkx) - q.S0 * BKz;
    const float Ax = (q.x(v0) - q.Pkx) - q.S0 * AKz;
    const float Ay = (q.y(v0) - q.Pky) - q.S1 * AKz;
    float fU = Cx * By - Cy * Bx;
    float fV = Ax * Cy - Ay * Cx;
    float fW = Bx * Ay - By * Ax;
    if (fminf(fminf(absf(fU), absf(fV)), absf(fW)) == 0.0f) {   // some edge function is zero (NaNs aside)
        fU = (float)((double)Cx * (double)By - (double)Cy * (double)Bx);
        fV = (float)((double)Ax * (double)Cy - (double)Ay * (double)Cx);
        fW = (float)((double)Bx * (double)Ay - (double)By * (double)Ax);
    }
    // some edge function negative and another positive; fmin and fmax pass over NaNs as the comparisons do
    if (fminf(fminf(fU, fV), fW) < 0.0f && fmaxf(fmaxf(fU, fV), fW) > 0.0f) return false;
    const float det = fU + fV + fW;
    if (det == 0.0f) return false;
    const float T = q.S2 * (fU * AKz + fV * BKz + fW * CKz);
    const int sgn = __float_as_int(det) & (int)0x80000000;
    const float Tx = __int_as_float(__float_as_int(T) ^ sgn);
    const float Dx = __int_as_float(__float_as_int(det) ^ sgn);
    if (MOTION_BOUND) {
        if (Tx <= bias * Dx) return false;
    } else {
        if (Tx < (1.19209290E-07f + bias) * Dx) return false;
    }
    p.T = T; p.det = det; p.fU = fU; p.fV = fV; p.fW = fW;
    return true;
}

// The rest of the test: far bound against the closest distance so far, then the hit update.
__device__ __forceinline__ bool tri_accept(RayS& r, const TriPre& p, float& U, float& V, float& W) {
    const int sgn = __float_as_int(p.det) & (int)0x80000000;
    const float Tx = __int_as_float(__float_as_int(p.T) ^ sgn);
    const float Dx = __int_as_float(__float_as_int(p.det) ^ sgn);
    if (Tx > r.tclosest * Dx) return false;
    const float rcp = 1.0f / p.det;
    U = p.fU * rcp;
    V = p.fV * rcp;
    W = p.fW * rcp;
    r.tclosest = p.T * rcp;
    return true;
}

__device__ __forceinline__ void load_tri(const DevTri* __restrict__ p, float4& v0, float4& v1, float4& v2) {
    v0 = make_float4(p->v[0][0], p->v[0][1], p->v[0][2], 0.0f);
    v1 = make_float4(p->v[1][0], p->v[1][1], p->v[1][2], 0.0f);
    v2 = make_float4(p->v[2][0], p->v[2][1], p->v[2][2], 0.0f);
}

__device__ __forceinline__ float4 lerp4(const float4& a, const float4& b, float t) {
    const float s = 1.0f - t;
    return make_float4(s * a.x + t * b.x, s * a.y + t * b.y, s * a.z + t * b.z, s * a.w + t * b.w);
}

// Vertices of a motion triangle (its nkeys groups of 3 float4 at q) at time t between keys k0 and k1
// (trace.go:547-554).
__device__ __forceinline__ void motion_tri(const float4* __restrict__ q, int k0, int k1, float t, float4& v0, float4& v1,
                                           float4& v2) {
    const float4* a = q + 3 * k0;
    const float4* b = q + 3 * k1;
    v0 = lerp4(a[0], b[0], t);
    v1 = lerp4(a[1], b[1], t);
    v2 = lerp4(a[2], b[2], t);
}

struct NodeData {
    float4 lx, ly, lz, hx, hy, hz;
    int ch[4];
    int ax[3];
};

__device__ __forceinline__ void swap_lane(float& a, float& b, bool sw) {
    const float t = a;
    a = sw ? b : a;
    b = sw ? t : b;
}

// A static node with its boxes as the reference holds them (the lanes that the upload put in order,
// DevNode::axes[3], swapped back), for box4.
__device__ __forceinline__ void fetch_static(const DevNode* __restrict__ nodes, int idx, NodeData& nd) {
    const float4* p = reinterpret_cast<const float4*>(nodes + idx);
    nd.lx = p[kRowLoX]; nd.ly = p[kRowLoY]; nd.lz = p[kRowLoZ];
    nd.hx = p[kRowHiX]; nd.hy = p[kRowHiY]; nd.hz = p[kRowHiZ];
    const int4 c = reinterpret_cast<const int4*>(p)[kRowChildren];
    const int4 a = reinterpret_cast<const int4*>(p)[kRowAxes];
    nd.ch[0] = c.x; nd.ch[1] = c.y; nd.ch[2] = c.z; nd.ch[3] = c.w;
    nd.ax[0] = a.x; nd.ax[1] = a.y; nd.ax[2] = a.z;
    if (a.w != 0) {
        const int m = a.w;
        swap_lane(nd.lx.x, nd.hx.x, m & 1); swap_lane(nd.lx.y, nd.hx.y, m & 2);
        swap_lane(nd.lx.z, nd.hx.z, m & 4); swap_lane(nd.lx.w, nd.hx.w, m & 8);
        swap_lane(nd.ly.x, nd.hy.x, m & 16); swap_lane(nd.ly.y, nd.hy.y, m & 32);
        swap_lane(nd.ly.z, nd.hy.z, m & 64); swap_lane(nd.ly.w, nd.hy.w, m & 128);
        swap_lane(nd.lz.x, nd.hz.x, m & 256); swap_lane(nd.lz.y, nd.hz.y, m & 512);
        swap_lane(nd.lz.z, nd.hz.z, m & 1024); swap_lane(nd.lz.w, nd.hz.w, m & 2048);
    }
}

// Motion node (qbvh/motionintersect.go:47-49): the boxes lerped per key and tested one axis at a
// time, in the slab order of box4, so only one axis of both keys is live at once.
__device__ __forceinline__ void box_motion(const RayS& r, const float4* __restrict__ mnodes, int base, int node,
                                           int nkeys, int key, int key2, float time, NodeData& nd, Box4& b) {
    const float4* p = mnodes + base + (size_t)node * (2 + 6 * nkeys);
    const int4 c = reinterpret_cast<const int4*>(p)[0];
    const int4 a = reinterpret_cast<const int4*>(p)[1];
    nd.ch[0] = c.x; nd.ch[1] = c.y; nd.ch[2] = c.z; nd.ch[3] = c.w;
    nd.ax[0] = a.x; nd.ax[1] = a.y; nd.ax[2] = a.z;
    const float4* b0 = p + 2 + 6 * key;
    const float4* b1 = p + 2 + 6 * key2;
    float tmin[4], tmax[4];
#pragma unroll
    for (int ax = 0; ax < 3; ax++) {
        const float4 lo = lerp4(b0[2 * ax], b1[2 * ax], time), hi = lerp4(b0[2 * ax + 1], b1[2 * ax + 1], time);
        const float la[4] = {lo.x, lo.y, lo.z, lo.w}, ha[4] = {hi.x, hi.y, hi.z, hi.w};
#pragma unroll
        for (int ch = 0; ch < 4; ch++) slab(la[ch], ha[ch], r.P[ax], r.Dinv[ax], tmin[ch], tmax[ch], ax == 0);
    }
#pragma unroll
    for (int ch = 0; ch < 4; ch++) {
        const float tn = (0.0f > tmin[ch]) ? 0.0f : tmin[ch];
        b.t[ch] = tn;
        b.h[ch] = tn <= tmax[ch];
    }
}

// The same for a node whose boxes are finite and ordered, as near and far planes (box4_near): the lerp
// keeps lo <= hi.  A row pair starts on 32 bytes, so the far plane's offset is the near one's with bit 4
// flipped; byte offsets fit 32 bits (SceneView::near_far).
__device__ __forceinline__ void box_motion_near(const RayS& r, int kp, const float4* __restrict__ mnodes, int base,
                                                int node, int nkeys, int key, int key2, float time, int (&ch)[4],
                                                int (&ax)[3], Box4& b) {
    const char* mp = reinterpret_cast<const char*>(mnodes);
    const uint32_t o = ((uint32_t)base + (uint32_t)node * (uint32_t)(2 + 6 * nkeys)) << 4;
    const int4 c = *reinterpret_cast<const int4*>(mp + o);
    const int4 a = *reinterpret_cast<const int4*>(mp + o + 16);
    ch[0] = c.x; ch[1] = c.y; ch[2] = c.z; ch[3] = c.w;
    ax[0] = a.x; ax[1] = a.y; ax[2] = a.z;
    const uint32_t o0 = o + 96u * (uint32_t)key, o1 = o + 96u * (uint32_t)key2;
    float tn[4], tx[4];
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const uint32_t s = ((uint32_t)kp >> k) & 16u;
        auto plane = [&](uint32_t flip) {
            return lerp4(*reinterpret_cast<const float4*>(mp + ((o0 | s) ^ flip) + 32 + 32 * k),
                         *reinterpret_cast<const float4*>(mp + ((o1 | s) ^ flip) + 32 + 32 * k), time);
        };
        const float4 nv = plane(0u), fv = plane(16u);
        const float na[4] = {nv.x, nv.y, nv.z, nv.w}, fa[4] = {fv.x, fv.y, fv.z, fv.w};
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const float x = (na[j] - r.P[k]) * r.Dinv[k], y = (fa[j] - r.P[k]) * r.Dinv[k];
            tn[j] = k == 0 ? x : fmaxf(tn[j], x);
            tx[j] = k == 0 ? y : fminf(tx[j], y);
        }
    }
#pragma unroll
    for (int j = 0; j < 4; j++) {
        b.t[j] = fmaxf(tn[j], 0.0f);
        b.h[j] = b.t[j] <= tx[j];
    }
}

// ray.Time -> (key, key2, t) (builtin/geom/polymesh/trace.go:79-84, scene.go:49-54)
// A time outside [0, 1] (the reference indexes out of range and panics) is held to the end keys,
// so no key index leaves the node or triangle.
__device__ __forceinline__ void motion_keys(float rtime, int nkeys, int& key, int& key2, float& t) {
    const float k = rtime * (float)(nkeys - 1);
    const float fk = floorf(k);
    t = k - fk;
    key = min(max((int)fk, 0), nkeys - 1);
    key2 = min(max((int)ceilf(k), 0), nkeys - 1);
}

// Sphere.Trace (builtin/geom/sphere/trace.go:13-52): the closed-form quadratic (solveQuadratic,
// raySphereIntersect :54-103), accepted when t < Tclosest, with no ray bias.
__device__ bool sphere_geom_hit(const float* P, const float4& d, const float4& sp, float tclosest, float& t) {
    const float Lx = P[0] - sp.x, Ly = P[1] - sp.y, Lz = P[2] - sp.z;
    const float a = d.x * d.x + d.y * d.y + d.z * d.z;
    const float b = 2 * (d.x * Lx + d.y * Ly + d.z * Lz);
    const float c = (Lx * Lx + Ly * Ly + Lz * Lz) - sp.w * sp.w;
    float x0, x1;
    const float discr = b * b - 4 * a * c;
    if (discr < 0) return false;
    if (discr == 0) {
        x1 = -0.5f * b / a;
        x0 = x1;
    } else {
        const float q = b > 0 ? -0.5f * (b + sqrtf(discr)) : -0.5f * (b - sqrtf(discr));
        x0 = q / a;
        x1 = c / q;
    }
    if (x0 > x1) { const float tt = x0; x0 = x1; x1 = tt; }
    if (x0 < 0) {
        x0 = x1;
        if (x0 < 0) return false;
    }
    if (!(x0 < tclosest)) return false;
    t = x0;
    return true;
}

// Scene.TraceElems over geoms [gcur, gend) of a top-level leaf (scene.go:61-78): analytic spheres
// (DevGeom nkeys 0) are tested here, in order, up to the first mesh.  Returns 1 with g = that mesh,
// 2 when a shadow ray hit a sphere (the traversal ends, qbvh/intersect.go:232-236), 0 at the leaf's end.
template <bool SHADOW>
__device__ __forceinline__ int next_geom(const SceneView& sv, const float4* __restrict__ rays, uint64_t ri, RayS& r,
                                         int& gcur, int gend, DevGeom& g, int& best_geom, int& best_prim, float& bu,
                                         float& bv, float& bw) {
    for (; gcur < gend; gcur++) {
        g = sv.geoms[gcur];
        if (g.nkeys != 0) return 1;
        float t;
        if (sphere_geom_hit(r.P, rays[2 * ri + 1], sv.spheres[g.tri_base], r.tclosest, t)) {
            r.tclosest = t;
            best_geom = gcur; best_prim = 0; bu = 0.0f; bv = 0.0f; bw = 0.0f;
            if (SHADOW) return 2;
        }
    }
    return 0;
}

// The ray in object space: P and D moved by Minv (D not renormalised).
__device__ __forceinline__ void ray_to_object(const float* Minv, float* P, float* D) {
    float p[3], d[3];
    xf_point(Minv, P, p);
    xf_vec(Minv, D, d);
    for (int k = 0; k < 3; k++) { P[k] = p[k]; D[k] = d[k]; }
}

// The ray at (px, py, pz) along (dx, dy, dz) moved by the inverse of x's transform at `time`.  A call and not inlined: the
// decomposed keys, the matrix and its inverse would be allocated beside the traversal's whole state, and the kernels
// spilled 38 to 116 registers, into the box and leaf steps too (trace_wide's XFORM form; figures at k_trace_xform).
struct RayPD {
    float p[3], d[3];
};
__device__ __noinline__ RayPD xform_ray(const DevXform* x, const float* xkeys, float time, float px, float py, float pz,
                                        float dx, float dy, float dz) {
    float M[16], Minv[16];
    xform_at(*x, xkeys, time, M, Minv);
    RayPD r{{px, py, pz}, {dx, dy, dz}};
    ray_to_object(Minv, r.p, r.d);
    return r;
}

// Whether the near/far box tests hold for the ray (box4_near).
template <bool MOTION>
__device__ __forceinline__ bool ray_plain(const RayS& r) {
    bool ok = !MOTION || absf(r.time) < 1e20f;   // time * keys stays finite
    for (int k = 0; k < 3; k++) ok = ok && absf(r.P[k]) < INFINITY && absf(r.Dinv[k]) < INFINITY && r.Dinv[k] != 0.0f;
    return ok;
}

// Where a lane stands among the geoms of a top-level leaf: child `child` of geom gcur (instances and
// procs), whose mesh or sphere is `slot`; hit: gcur reported a hit.
struct GeomWalk {
    int slot, child;
    bool hit;
};

// next_geom for scenes with transforms: the reference's recursion Scene.TraceElems -> Geom.Trace written
// out.  first: the leaf has just been popped, gcur is its first geom; otherwise mesh w.slot has been
// traced.  A geom with a transform moves the ray into its object space (P and D by the inverse transform
// at the ray's time, then Setup) and restores it, Tclosest excepted (instance.go:78-104, proc.go:93-131,
// polymesh/trace.go:20-74); a proc stops at the first geom reporting a hit unless the ray is a shadow ray
// (proc.go:112-120), which leaves the scene after the geom that was hit.  Returns as next_geom.
template <bool SHADOW>
__device__ __forceinline__ int next_geom_xf(const SceneView& sv, const float4* __restrict__ rays, uint64_t ri, RayS& r,
                                            int& kp, bool& ok, bool first, int& gcur, int gend, GeomWalk& w, DevGeom& g,
                                            int& best_geom, int& best_prim, int& best_leaf, float& bu, float& bv,
                                            float& bw) {
    const float4 ra = rays[2 * ri], rb = rays[2 * ri + 1];
    bool entered = !first;   // geom gcur has begun
    while (true) {
        if (entered) {
            const DevXform x = sv.xforms[gcur];
            if (x.kind >= kXfInstance && w.child + 1 < x.nchild && !(w.hit && (x.kind == kXfInstance || !SHADOW))) {
                w.child++;
            } else {
                if (SHADOW && w.hit) return 2;
                gcur++;
                entered = false;
            }
        }
        const bool end = !entered && gcur >= gend;
        DevXform x{};
        if (!end) {
            x = sv.xforms[gcur];
            if (!entered) {
                entered = true;
                w.child = 0;
                w.hit = false;
            }
            if (x.kind >= kXfInstance) {
                if (w.child >= x.nchild) continue;   // a proc without geoms
                w.slot = sv.xchildren[x.child_base + w.child];
            } else {
                w.slot = gcur;
            }
            g = sv.geoms[w.slot];
        }
        float P[3] = {ra.x, ra.y, ra.z}, D[3] = {rb.x, rb.y, rb.z};
        if (!end) {
            // the instance's or proc's transform, then the mesh's own
#pragma unroll 1
            for (int level = x.kind >= kXfInstance ? 0 : 1; level < 2; level++) {
                const DevXform* xl = sv.xforms + (level == 0 ? gcur : w.slot);
                if (xl->kind == kXfNone) continue;
                const RayPD o = xform_ray(xl, sv.xkeys, rb.w, P[0], P[1], P[2], D[0], D[1], D[2]);
                for (int k = 0; k < 3; k++) { P[k] = o.p[k]; D[k] = o.d[k]; }
            }
        }
        for (int k = 0; k < 3; k++) r.P[k] = P[k];
        ray_setup(r, D);
        kp = pack_perm(r);
        ok = ray_plain<true>(r);
        if (end) return 0;
        if (g.nkeys != 0) return 1;
        float t;
        if (sphere_geom_hit(P, make_float4(D[0], D[1], D[2], 0.0f), sv.spheres[g.tri_base], r.tclosest, t)) {
            r.tclosest = t;
            w.hit = true;
            best_geom = gcur; best_prim = 0; best_leaf = w.slot; bu = 0.0f; bv = 0.0f; bw = 0.0f;
        }
    }
}

// ---- cross-lane helpers of the wavefront-wide leaf tests

// Sums / maxima over lanes 0..lane on the DPP row shifts and broadcasts: six VALU operations with no
// LDS round trip.
template <int CTRL, int ROWS>
__device__ __forceinline__ int dpp0(int x) {   // lanes without a source read 0
    return __builtin_amdgcn_update_dpp(0, x, CTRL, ROWS, 0xf, false);
}
__device__ __forceinline__ int wave_scan_add(int x) {
    x += dpp0<0x111, 0xf>(x);
    x += dpp0<0x112, 0xf>(x);
    x += dpp0<0x114, 0xf>(x);
    x += dpp0<0x118, 0xf>(x);
    x += dpp0<0x142, 0xa>(x);
    x += dpp0<0x143, 0xc>(x);
    return x;
}
__device__ __forceinline__ int wave_scan_max(int x) {   // x >= 0
    x = max(x, dpp0<0x111, 0xf>(x));
    x = max(x, dpp0<0x112, 0xf>(x));
    x = max(x, dpp0<0x114, 0xf>(x));
    x = max(x, dpp0<0x118, 0xf>(x));
    x = max(x, dpp0<0x142, 0xa>(x));
    x = max(x, dpp0<0x143, 0xc>(x));
    return x;
}
// LDS words that other lanes of the wavefront read or write (a wavefront's LDS operations stay in order;
// relaxed atomics keep the compiler from assuming a lane's own stores).
__device__ __forceinline__ void lds_put(int* p, int x) { __hip_atomic_store(p, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT); }
__device__ __forceinline__ int lds_get(const int* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT); }
// x of lane (addr / 4); every lane of the wavefront takes part.
__device__ __forceinline__ float lane_f(int addr, float x) {
    return __int_as_float(__builtin_amdgcn_ds_bpermute(addr, __float_as_int(x)));
}
__device__ __forceinline__ int lane_i(int addr, int x) { return __builtin_amdgcn_ds_bpermute(addr, x); }

// In scenes with transforms, lanes at the end or the start of a geom wait until kTurnWait times as many
// wait as hold a node or a leaf: the transform of a moving instance is a thousand instructions.  262,144 rays
// in a room of 60 instances / 2^20 rays in one of 20, in us: 751 / 1064 when half as many suffice, 706 / 990 at 1,
// 682 / 917 at 2, 678 / 886 at 3, 671 / 880 at 4, 667 / 878 at 6, 675 / 884 at 8; shadow rays in the first: 568, 522,
// 496, 506, 510, 516, 527.
constexpr int kTurnWait = 4;

// What a lane does next, beside node indices (>= 0) and mesh leaves (< kIdle).
constexpr int kPop = -1;    // take the next stack entry (also the encoding of an empty child)
constexpr int kIdle = -2;   // no ray, or its traversal has ended

// The wavefront tests the leaves its lanes hold once kLeafRatio times as many lanes hold a leaf as hold a
// node: few waiting leaves cost less than a node step with idle lanes while most lanes hold nodes, more as
// the node lanes run out.  Measured on the icosphere field (2.1M bounce rays) / the 1M-triangle room (one
// plain 1024^2 pass) / the box of spheres (320 x 199, depth 5), in us: ratio 2: 709 / 7930 / 1606, 3: 705 / 8009 /
// 1615, 5: 714 / 8184 / 1634, 8: 708 / 8429 / 1659; a fixed count of 2 lanes: 732 / 9046 / 1667, 4: 730 / 8468 /
// 1638, 10: 743 / 8144 / 1705.  Moving spheres (1M camera rays): 586 at 2, 592 at 3, 599 at 5.
constexpr int kLeafRatio = 3;

// The traversal, one ray per lane.  A lane holds the node it visits next, a leaf of triangles it has
// popped, or nothing; every turn of the loop the wavefront either steps all lanes that hold nodes (box
// test, push) or tests all leaves held (kLeafRatio), so that neither runs for a few lanes while many wait;
// lanes without either pop up to their next entry that is not culled.  The order of steps within each ray
// is the reference's, whatever the other lanes do.
//
// What bounds it is VALU issue: 2.1M bounce rays in the icosphere field took 4.4e8 VALU instructions, 80%
// of the issue slots of 902 us, when every turn ran both phases; now 2.85e8 and 66% of 705 us (2.97
// Grays/s), the rest waiting for nodes and triangles beyond L2.  Hence the forms below: near and far planes
// by address instead of sorted pairs (box4_near), stack positions as byte offsets summed from hit flags,
// one 8-byte LDS entry per push, DPP scans, the workers' results handed to the owners instead of a second
// test, and the geom changes kept out of the pop loop.
//
// Leaf tests are dealt out over the wavefront: an inclusive prefix sum of the leaf sizes runs over the
// lanes, work item w belongs to the last lane whose items start at or before w (each owner marks its
// first slot in LDS, a running maximum spreads the mark), and the lane working on it reads the owner's
// ray with cross-lane shuffles.  Consecutive lanes take consecutive triangles of one leaf, so the loads
// coalesce.  That part of the watertight test does not read the closest distance; the owner then accepts
// the triangles that passed, in leaf order and with the values that the worker computed, which takes the
// same triangles in the same order as the reference's loop.
//
// A lane whose ray has ended idles (and works in the leaf tests) until refill_min lanes are idle; then
// the idle lanes write their results and take the next rays of the wavefront together.
// MOTION: the scene has motion keys (a motion top level and/or moving meshes); node boxes
// (qbvh/motionintersect.go:47-49) and triangles of moving meshes (trace.go:547-554) are
// interpolated at the ray's time.
// EXT: hits are 32-byte records {prim, geom, t, U, V, W, 0, 0} for the shading kernels.
// XFORM: the scene holds instances, procs or transformed meshes (MOTION is set too); a lane's ray is the
// one in the space of the geom it traverses, and EXT records hold the slot of the mesh or sphere hit in
// place of the first 0.
template <int BLOCK, int LDS, bool SHADOW, bool MOTION, bool COUNTERS, bool EXT, bool XFORM = false>
__device__ __forceinline__ void trace_wide(SceneView sv, const float4* __restrict__ rays, uint64_t n,
                                           int4* __restrict__ hits, int32_t* __restrict__ geoms_out,
                                           int4* __restrict__ counters, float* __restrict__ spT,
                                           int32_t* __restrict__ spN, int32_t* __restrict__ err,
                                           const uint32_t* __restrict__ n_dev, const uint32_t* __restrict__ perm,
                                           int gather, int ray_shift, int refill_min) {
    static_assert(BLOCK % 64 == 0, "whole wavefronts");
    static_assert(LDS >= 4, "a node step's pushes are checked against LDS - 3");
    constexpr int kEntry = BLOCK * 8;             // bytes from one stack entry of a lane to the next
    constexpr int kNoRay = -1;
    __shared__ uint2 stack_lds[LDS * BLOCK];      // {T bits, node}, entry-major: lanes never conflict on a bank
    __shared__ int owner[BLOCK];                  // written by one lane, read by another of its wavefront
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const uint64_t nwaves = (uint64_t)gridDim.x * (BLOCK / 64);
    const uint64_t wave = (uint64_t)blockIdx.x * (BLOCK / 64) + (uint32_t)__builtin_amdgcn_readfirstlane(tid >> 6);
    const int bottom = tid * 8;                   // the lane's empty stack: entry i at bottom + i * kEntry

    // A spill column per lane that can own a ray: with ray_shift below 6 the wavefront takes all its rays at once,
    // into its first 2^ray_shift lanes (trace_spill_columns).
    auto spill = [&](int sp) {
        return (uint64_t)((uint32_t)sp / kEntry - LDS) * (nwaves << ray_shift) + (wave << ray_shift) +
               (uint32_t)(lane & ((1 << ray_shift) - 1));
    };
    auto push = [&](int sp, float T, int32_t node) {
        if (sp < LDS * kEntry) *reinterpret_cast<uint2*>(reinterpret_cast<char*>(stack_lds) + sp) = make_uint2(__float_as_uint(T), (uint32_t)node);
        else { const uint64_t o = spill(sp); spT[o] = T; spN[o] = node; }
    };

    if (n_dev) n = min(n, (uint64_t)*n_dev);
    // Rays of this wavefront: v = 0, 1, 2, ... -> ray_of(v), increasing in v: 2^ray_shift consecutive rays, then
    // as many nwaves * 2^ray_shift further on (trace_ray_shift).
    auto ray_of = [&](uint32_t v) {
        return (((uint64_t)(v >> ray_shift) * nwaves + wave) << ray_shift) + (v & ((1u << ray_shift) - 1u));
    };
    uint32_t cursor = 0;
    bool ok = true, fast = false;
    int ri = kNoRay;                              // launches hold fewer than 2^32 rays; ~0 is never one
    int kp = 0;                                   // pack_perm of the current ray
    RayS r;
    r.P[0] = 0.0f; r.P[1] = 0.0f; r.P[2] = 0.0f; r.tclosest = 0.0f; r.time = 0.0f;
    {
        const float D1[3] = {1.0f, 1.0f, 1.0f};
        ray_setup(r, D1);
    }
    int nodesT = 0, leafsT = 0, trisT = 0, maxDepth = 0;
    int best_geom = -1, best_prim = -1;
    float bu = 0.0f, bv = 0.0f, bw = 0.0f;
    // The level traversed: the scene's (base == bottom, in_mesh false) or geom gcur's, whose stack starts
    // at base.  A motion top level starts it at the popped leaf's own slot, a static one above it
    // (qbvh/motionintersect.go:99-103 against intersect.go:219-226).
    const bool top_motion = MOTION && sv.top_motion;
    const bool reuse_slot = XFORM || top_motion;
    GeomWalk walk = {0, 0, false};
    int best_leaf = 0;
    bool in_mesh = false;
    int base = bottom, gcur = 0, gend = 0;
    DevGeom g = {0, 0, 1, 0.0f};
    int sp = bottom;
    int cur = kIdle;
    while (true) {
        const uint64_t dm = __ballot(cur == kIdle);
        const bool more = ray_of(cursor) < n;
        if (more ? __popcll(dm) >= refill_min : dm == ~0ull) {
            if (cur == kIdle) {
                if (ri != kNoRay) {
                    if (best_prim == -2) {   // the stack overflowed
                        atomicOr(err, 1);
                        best_geom = -1; best_prim = -1;
                        if (XFORM) best_leaf = -1;
                    }
                    const uint64_t oi = perm && !gather ? (uint64_t)perm[(uint32_t)ri] : (uint64_t)(uint32_t)ri;
                    if (EXT) {
                        hits[2 * oi] = make_int4(best_prim, best_geom, __float_as_int(r.tclosest), __float_as_int(bu));
                        hits[2 * oi + 1] = make_int4(__float_as_int(bv), __float_as_int(bw), best_leaf, 0);
                    } else {
                        hits[oi] = make_int4(best_prim, __float_as_int(r.tclosest), __float_as_int(bu), __float_as_int(bv));
                        if (geoms_out) geoms_out[oi] = best_geom;
                    }
                    if (COUNTERS) counters[oi] = make_int4(nodesT, leafsT, trisT, maxDepth);
                    ri = kNoRay;
                }
                if (more) {
                    const uint32_t v = cursor + (uint32_t)__popcll(dm & ((1ull << lane) - 1ull));
                    const uint64_t rnext = ray_of(v);
                    ok = true;
                    if (rnext < n) {
                        ri = (int)(gather ? perm[rnext] : (uint32_t)rnext);
                        const float4 ra = rays[2 * (uint64_t)(uint32_t)ri], rb4 = rays[2 * (uint64_t)(uint32_t)ri + 1];
                        r.P[0] = ra.x; r.P[1] = ra.y; r.P[2] = ra.z; r.tclosest = ra.w;
                        const float D[3] = {rb4.x, rb4.y, rb4.z};
                        r.time = rb4.w;
                        // A ray with tmax < 0 (the shading passes' unused shadow slots) culls every entry, since
                        // no entry distance is below 0: a miss that needs no set-up and no step.
                        const bool ends = !COUNTERS && ra.w < 0.0f;
                        if (!ends) {
                            ray_setup(r, D);
                            kp = pack_perm(r);
                            ok = ray_plain<MOTION>(r);
                        }
                        nodesT = 0; leafsT = 0; trisT = 0; maxDepth = 0;
                        best_geom = -1; best_prim = -1;
                        if (XFORM) best_leaf = -1;
                        bu = 0.0f; bv = 0.0f; bw = 0.0f;
                        in_mesh = false;
                        base = bottom;
                        sp = bottom;
                        cur = ends ? kIdle : 0;   // the root, whose entry distance is tclosest itself: never culled
                    }
                }
            }
            if (!more) break;
            cursor += (uint32_t)__popcll(dm);
            fast = sv.near_far && __all(ok ? 1 : 0) != 0;
        }

        // Pop: up to the next entry of the level that is not culled (a culled entry and an empty child both
        // leave kPop).
        while (cur == kPop && sp != base) {
            sp -= kEntry;
            float T; int32_t node;
            if (sp < LDS * kEntry) {
                const uint2 e = *reinterpret_cast<const uint2*>(reinterpret_cast<const char*>(stack_lds) + sp);
                T = __uint_as_float(e.x); node = (int32_t)e.y;
            } else {
                const uint64_t o = spill(sp);
                T = spT[o]; node = spN[o];
            }
            cur = r.tclosest < T ? kPop : node;
            if (COUNTERS && cur < kIdle) { leafsT++; if (in_mesh) trisT += leaf_count(cur); }
        }
        // Ends of levels, and the scene level's leaves: lanes that leave a mesh for the scene level pop there
        // in the next turn.
        const bool turn = cur == kPop || (cur < kIdle && !in_mesh);
        const uint64_t turns = __ballot(turn);
        if (XFORM ? turns != 0 && __popcll(turns) >= kTurnWait * __popcll(__ballot(!turn && cur != kIdle)) : turns != 0) {
            if (turn) {
                if (cur == kPop && !in_mesh) {
                    cur = kIdle;
                } else {
                    const bool first = cur != kPop;   // else PolyMesh.Trace returned: on to the leaf's next geom (scene.go:65-75)
                    int mb = base;
                    if (first) {   // Scene.TraceElems: the geoms of a top-level leaf (scene.go:61-78)
                        mb = reuse_slot ? sp : sp + kEntry;
                        gcur = leaf_base(cur); gend = gcur + leaf_count(cur);
                    } else if (!XFORM) {
                        gcur++;
                    }
                    if (mb >= VGPU_MAX_STACK * kEntry) {
                        best_prim = -2;
                        cur = kIdle;
                    } else {
                        int ng;
                        if constexpr (XFORM)
                            ng = next_geom_xf<SHADOW>(sv, rays, (uint32_t)ri, r, kp, ok, first, gcur, gend, walk, g, best_geom,
                                                      best_prim, best_leaf, bu, bv, bw);
                        else
                            ng = next_geom<SHADOW>(sv, rays, (uint32_t)ri, r, gcur, gend, g, best_geom, best_prim, bu, bv, bw);
                        in_mesh = ng == 1;
                        base = in_mesh ? mb : bottom;
                        sp = in_mesh || reuse_slot ? mb : mb - kEntry;
                        cur = ng == 2 ? kIdle : (ng == 1 ? 0 : kPop);
                    }
                }
            }
            if (XFORM) {
                if (cur == kIdle) ok = true;
                fast = sv.near_far && __all(ok ? 1 : 0) != 0;
                if (turns != 0) continue;
            }
        }

        const bool leaf = XFORM ? cur < kIdle && in_mesh : cur < kIdle;
        const uint64_t leaves = __ballot(leaf);
        const uint64_t nodes = __ballot(cur >= 0);
        if (__popcll(leaves) * kLeafRatio < __popcll(nodes)) {
            if (cur >= 0) {
                if (COUNTERS) nodesT++;
                Box4 b;
                int ch[4], ax[3];
                bool moving = false;
                if constexpr (MOTION) moving = in_mesh ? g.nkeys > 1 : top_motion;
                if (MOTION && moving) {
                    const int nk = in_mesh ? g.nkeys : sv.top_keys;
                    const int nb = in_mesh ? g.node_base : sv.top_mbase;
                    int k0, k1;
                    float t;
                    motion_keys(r.time, nk, k0, k1, t);
                    if (fast) {
                        box_motion_near(r, kp, sv.mnodes, nb, cur, nk, k0, k1, t, ch, ax, b);
                    } else {
                        NodeData nd;
                        box_motion(r, sv.mnodes, nb, cur, nk, k0, k1, t, nd, b);
                        for (int c = 0; c < 4; c++) ch[c] = nd.ch[c];
                        for (int k = 0; k < 3; k++) ax[k] = nd.ax[k];
                    }
                } else {
                    const int idx = in_mesh ? g.node_base + cur : cur;
                    if (fast) {
                        // 32-bit byte offsets from the uniform base; a near plane's row is its axis's lower or
                        // upper bound by the sign bit, the far plane's the other one (DevNode)
                        const char* nbp = reinterpret_cast<const char*>(sv.nodes);
                        const uint32_t o = (uint32_t)idx << 7;
                        const uint32_t ox = (kp & 16) | o, oy = (kp & 32) | o, oz = (kp & 64) | o;
                        auto row = [&](uint32_t ofs, int rr) { return *reinterpret_cast<const float4*>(nbp + ofs + 16 * rr); };
                        const float4 nx = row(ox, kRowLoX), fx = row(ox ^ 16, kRowLoX);
                        const float4 ny = row(oy, kRowLoY), fy = row(oy ^ 32, kRowLoY);
                        const float4 nz = row(oz, kRowLoZ), fz = row(oz ^ 64, kRowLoZ);
                        const int4 c = *reinterpret_cast<const int4*>(nbp + o + 16 * kRowChildren);
                        const int4 a = *reinterpret_cast<const int4*>(nbp + o + 16 * kRowAxes);
                        ch[0] = c.x; ch[1] = c.y; ch[2] = c.z; ch[3] = c.w;
                        ax[0] = a.x; ax[1] = a.y; ax[2] = a.z;
                        box4_near(r, nx, ny, nz, fx, fy, fz, b);
                    } else {
                        NodeData nd;
                        fetch_static(sv.nodes, idx, nd);
                        box4(r, nd.lx, nd.ly, nd.lz, nd.hx, nd.hy, nd.hz, b);
                        for (int c = 0; c < 4; c++) ch[c] = nd.ch[c];
                        for (int k = 0; k < 3; k++) ax[k] = nd.ax[k];
                    }
                }
                // Push order of qbvh/intersect.go:137-216 (same as motionintersect.go:53-97): the children
                // are pushed as two pairs.  m0, m1, m2 are all ones when the ray's direction is negative on
                // the node's axis: the first pair goes first when m0, child 0 before child 1 when m1, child 2
                // before child 3 when m2.  A hit child's slot is the sum of the hits pushed before it, so the
                // entries are exactly those the reference leaves below its stack top.
                const int m0 = __builtin_amdgcn_sbfe(kp, ax[0], 1);
                const int m1 = __builtin_amdgcn_sbfe(kp, ax[1], 1);
                const int m2 = __builtin_amdgcn_sbfe(kp, ax[2], 1);
                const int c0 = b.h[0] ? kEntry : 0, c1 = b.h[1] ? kEntry : 0;
                const int c2 = b.h[2] ? kEntry : 0, c3 = b.h[3] ? kEntry : 0;
                const int s01 = c0 + c1, s23 = c2 + c3;
                const int pa = sp + (s23 & ~m0), pb = sp + (s01 & m0);
                const int p0 = pa + (c1 & ~m1), p1 = pa + (c0 & m1);
                const int p2 = pb + (c3 & ~m2), p3 = pb + (c2 & m2);
                cur = kPop;
                if (sp < (LDS - 3) * kEntry) {   // every slot of this step lies in LDS
                    if (b.h[0]) *reinterpret_cast<uint2*>(reinterpret_cast<char*>(stack_lds) + p0) = make_uint2(__float_as_uint(b.t[0]), (uint32_t)ch[0]);
                    if (b.h[1]) *reinterpret_cast<uint2*>(reinterpret_cast<char*>(stack_lds) + p1) = make_uint2(__float_as_uint(b.t[1]), (uint32_t)ch[1]);
                    if (b.h[2]) *reinterpret_cast<uint2*>(reinterpret_cast<char*>(stack_lds) + p2) = make_uint2(__float_as_uint(b.t[2]), (uint32_t)ch[2]);
                    if (b.h[3]) *reinterpret_cast<uint2*>(reinterpret_cast<char*>(stack_lds) + p3) = make_uint2(__float_as_uint(b.t[3]), (uint32_t)ch[3]);
                    sp += s01 + s23;
                } else if (sp >= (VGPU_MAX_STACK - 3) * kEntry) {   // conservative: the reference writes up to 4 slots here
                    best_prim = -2;
                    cur = kIdle;
                } else {
                    if (b.h[0]) push(p0, b.t[0], ch[0]);
                    if (b.h[1]) push(p1, b.t[1], ch[1]);
                    if (b.h[2]) push(p2, b.t[2], ch[2]);
                    if (b.h[3]) push(p3, b.t[3], ch[3]);
                    sp += s01 + s23;
                }
                if (COUNTERS && cur == kPop) maxDepth = max(maxDepth, (int)((uint32_t)sp / kEntry));
            }
            continue;
        }
        if (leaves == 0) continue;   // every lane popped its last entry

        // ---- the leaves held, all of them
        const bool mine = leaf;
        const int cnt = mine ? leaf_count(cur) : 0;
        const int lbase = leaf_base(cur);
        const int pin = wave_scan_add(cnt);
        const int pex = pin - cnt;
        const int total = __builtin_amdgcn_readlane(pin, 63);
        const TriRay own = tri_ray_packed(r, kp);
        const bool mv = MOTION && g.nkeys > 1;
        // what item w adds to reach its triangle: an index (static) or, scaled by the worker, a float4 offset
        const int tb = mv ? g.tri_base + lbase * 3 * g.nkeys : g.tri_base + lbase - pex;
        bool any = false;
        for (int k0 = 0; k0 < total; k0 += 64) {
            const int s0 = max(pex - k0, 0), e0 = min(pin - k0, 64);   // this lane's items of the chunk
            const bool has = e0 > s0;
            lds_put(&owner[tid], 0);
            if (has) lds_put(&owner[(tid & ~63) + s0], lane);
            const int o = wave_scan_max(lds_get(&owner[tid])) << 2;
            const int w = k0 + lane;
            TriRay q;
            q.S0 = lane_f(o, own.S0); q.S1 = lane_f(o, own.S1); q.S2 = lane_f(o, own.S2);
            q.Pkx = lane_f(o, own.Pkx); q.Pky = lane_f(o, own.Pky); q.Pkz = lane_f(o, own.Pkz);
            q.axes(lane_i(o, kp));
            const float obias = lane_f(o, g.ray_bias);
            const int otb = lane_i(o, tb);
            int onk = 1, oex = 0;
            float otime = 0.0f;
            if constexpr (MOTION) {
                onk = lane_i(o, g.nkeys);
                oex = lane_i(o, pex);
                otime = lane_f(o, r.time);
            }
            bool pass = false;
            TriPre pr;
            if (w < total) {
                if (MOTION && onk > 1) {
                    int a0, a1;
                    float t;
                    motion_keys(otime, onk, a0, a1, t);
                    float4 v0, v1, v2;
                    motion_tri(sv.mtris + otb + (size_t)(w - oex) * 3 * onk, a0, a1, t, v0, v1, v2);
                    pass = tri_pre<true>(q, v0, v1, v2, obias, pr);
                } else {
                    float4 v0, v1, v2;
                    load_tri(sv.tris + (otb + w), v0, v1, v2);
                    pass = tri_pre<false>(q, v0, v1, v2, obias, pr);
                }
            }
            const uint64_t cm = __ballot(pass);
            if (cm == 0) continue;
            // the owners' passes over their candidates, in leaf order (trace.go:108-122)
            uint32_t cand = has ? (uint32_t)(cm >> s0) & ((1u << (e0 - s0)) - 1u) : 0;
            while (__ballot(cand != 0) != 0) {
                const int src = s0 + __builtin_ctz(cand | 0x10000u);
                const int sa = src << 2;
                TriPre ow;
                ow.T = lane_f(sa, pr.T); ow.det = lane_f(sa, pr.det);
                ow.fU = lane_f(sa, pr.fU); ow.fV = lane_f(sa, pr.fV); ow.fW = lane_f(sa, pr.fW);
                if (cand != 0) {
                    cand &= cand - 1;
                    if (tri_accept(r, ow, bu, bv, bw)) {
                        best_geom = gcur;
                        best_prim = lbase + k0 + src - pex;
                        if (XFORM) best_leaf = walk.slot;
                        any = true;
                    }
                }
            }
        }
        // a shadow ray's hit ends both levels (qbvh/intersect.go:232-236); under a transform, the mesh
        if (mine) cur = SHADOW && any && !XFORM ? kIdle : kPop;
        if (XFORM && any) {
            walk.hit = true;
            if (SHADOW) sp = base;
        }
    }
}

#define VGPU_TRACE_PARAMS                                                                                      \
    SceneView sv, const float4 *__restrict__ rays, uint64_t n, int4 *__restrict__ hits,                       \
        int32_t *__restrict__ geoms_out, int4 *__restrict__ counters, float *__restrict__ spT,                \
        int32_t *__restrict__ spN, int32_t *__restrict__ err, const uint32_t *__restrict__ n_dev,              \
        const uint32_t *__restrict__ perm, int gather, int ray_shift,           \
        int refill_min
#define VGPU_TRACE_ARGS \
    sv, rays, n, hits, geoms_out, counters, spT, spN, err, n_dev, perm, gather, ray_shift, refill_min

template <int BLOCK, int LDS, bool SHADOW, bool MOTION, bool COUNTERS, bool EXT>
__global__ __launch_bounds__(BLOCK) void k_trace_wide(VGPU_TRACE_PARAMS) {
    trace_wide<BLOCK, LDS, SHADOW, MOTION, COUNTERS, EXT>(VGPU_TRACE_ARGS);
}

// Scenes holding GeomInstances, Procs or meshes with their own Transform.  Four waves per SIMD: the walk
// over geoms takes registers, and its lanes wait for one another (kTurnWait).
// 262,144 rays in a room of 60 instances: 670 us of kernel, 12 registers spilled.  With the transform inlined
// (xform_ray) 73 were and the kernel took 1061 us, 875 without spills at three waves per SIMD; one ray per lane with
// the recursion inside it (the leaf triangles of a lane tested by that lane alone) took 1868.
template <int BLOCK, int LDS, bool SHADOW, bool EXT>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(4, 8))) void k_trace_xform(VGPU_TRACE_PARAMS) {
    trace_wide<BLOCK, LDS, SHADOW, true, false, EXT, true>(VGPU_TRACE_ARGS);
}

#undef VGPU_TRACE_PARAMS
#undef VGPU_TRACE_ARGS

template <bool SHADOW, bool EXT>
hipError_t launch_xform(const SceneView& sv, const TraceLaunch& cfg, const void* rays, uint64_t n, void* hits,
                        int32_t* geoms, float* spT, int32_t* spN, uint64_t spill_columns, int32_t* err, int num_cus,
                        const uint32_t* n_dev, const uint32_t* perm, bool gather, hipStream_t stream) {
    constexpr int kB = kXformLaunch.block, kL = kXformLaunch.lds_depth;
    const uint64_t threads = trace_grid_threads(cfg, n, num_cus);
    if (cfg.block != kB || cfg.lds_depth != kL || trace_spill_columns(cfg, n, num_cus) > spill_columns) return hipErrorInvalidValue;
    hipLaunchKernelGGL((k_trace_xform<kB, kL, SHADOW, EXT>), dim3((unsigned)(threads / kB)), dim3(kB), 0, stream, sv,
                       (const float4*)rays, n, (int4*)hits, geoms, (int4*)nullptr, spT, spN, err, n_dev, perm,
                       gather ? 1 : 0, trace_ray_shift(cfg, n, num_cus), cfg.refill_min);
    return hipGetLastError();
}

template <int BLOCK, int LDS, bool SHADOW, bool MOTION>
hipError_t launch_cfg(const SceneView& sv, const void* rays, uint64_t n, void* hits, int32_t* geoms, int32_t* counters,
                      float* spT, int32_t* spN, uint64_t grid, int32_t* err, const uint32_t* n_dev,
                      const uint32_t* perm, bool gather, hipStream_t stream, int ray_shift, int refill_min) {
    if (counters)
        hipLaunchKernelGGL((k_trace_wide<BLOCK, LDS, SHADOW, MOTION, true, false>), dim3((unsigned)grid), dim3(BLOCK), 0,
                           stream, sv, (const float4*)rays, n, (int4*)hits, geoms, (int4*)counters, spT, spN, err,
                           n_dev, perm, gather ? 1 : 0, ray_shift, refill_min);
    else
        hipLaunchKernelGGL((k_trace_wide<BLOCK, LDS, SHADOW, MOTION, false, false>), dim3((unsigned)grid), dim3(BLOCK), 0,
                           stream, sv, (const float4*)rays, n, (int4*)hits, geoms, (int4*)nullptr, spT, spN, err,
                           n_dev, perm, gather ? 1 : 0, ray_shift, refill_min);
    return hipGetLastError();
}

template <int BLOCK, int LDS>
hipError_t launch_mode(const SceneView& sv, bool shadow, bool motion, const void* rays, uint64_t n, void* hits,
                       int32_t* geoms, int32_t* counters, float* spT, int32_t* spN, uint64_t grid, int32_t* err,
                       const uint32_t* n_dev, const uint32_t* perm, bool gather, hipStream_t stream, int ray_shift, int refill_min) {
    if (shadow) {
        if (motion)
            return launch_cfg<BLOCK, LDS, true, true>(sv, rays, n, hits, geoms, counters, spT, spN, grid, err, n_dev, perm, gather, stream, ray_shift, refill_min);
        return launch_cfg<BLOCK, LDS, true, false>(sv, rays, n, hits, geoms, counters, spT, spN, grid, err, n_dev, perm, gather, stream, ray_shift, refill_min);
    }
    if (motion)
        return launch_cfg<BLOCK, LDS, false, true>(sv, rays, n, hits, geoms, counters, spT, spN, grid, err, n_dev, perm, gather, stream, ray_shift, refill_min);
    return launch_cfg<BLOCK, LDS, false, false>(sv, rays, n, hits, geoms, counters, spT, spN, grid, err, n_dev, perm, gather, stream, ray_shift, refill_min);
}

}  // namespace

hipError_t launch_trace_ext(const SceneView& sv, bool motion, const void* rays, uint64_t n, void* hits32, float* spT,
                            int32_t* spN, uint64_t spill_columns, int32_t* err, int num_cus, hipStream_t stream,
                            const uint32_t* n_dev) {
    if (n == 0) return hipSuccess;
    if (n > 0xffffffffull) return hipErrorInvalidValue;
    // the block size is the kernel's launch bound: each shape is a template constant
    constexpr int kB = kExtLaunch.block, kL = kExtLaunch.lds_depth;
    constexpr int kBM = kExtLaunchMotion.block, kLM = kExtLaunchMotion.lds_depth;
    if (sv.any_xform)
        return launch_xform<false, true>(sv, kXformLaunch, rays, n, hits32, nullptr, spT, spN, spill_columns, err, num_cus,
                                         n_dev, nullptr, false, stream);
    const TraceLaunch cfg = motion ? kExtLaunchMotion : kExtLaunch;
    const uint64_t threads = trace_grid_threads(cfg, n, num_cus);
    if (trace_spill_columns(cfg, n, num_cus) > spill_columns) return hipErrorInvalidValue;
    const unsigned grid = (unsigned)(threads / cfg.block);
    const int ray_shift = trace_ray_shift(cfg, n, num_cus);
    if (motion)
        hipLaunchKernelGGL((k_trace_wide<kBM, kLM, false, true, false, true>), dim3(grid), dim3(kBM), 0, stream, sv,
                           (const float4*)rays, n, (int4*)hits32, (int32_t*)nullptr, (int4*)nullptr, spT, spN, err, n_dev,
                           (const uint32_t*)nullptr, 0, ray_shift, kRefillDefault);
    else
        hipLaunchKernelGGL((k_trace_wide<kB, kL, false, false, false, true>), dim3(grid), dim3(kB), 0, stream, sv,
                           (const float4*)rays, n, (int4*)hits32, (int32_t*)nullptr, (int4*)nullptr, spT, spN, err, n_dev,
                           (const uint32_t*)nullptr, 0, ray_shift, kRefillDefault);
    return hipGetLastError();
}

int trace_ray_shift(const TraceLaunch& cfg, uint64_t n, int num_cus) {
    const uint64_t waves = (uint64_t)num_cus * (uint64_t)std::min(cfg.waves_per_cu, cfg.spread);
    int shift = 6;
    while (shift > 0 && (n >> (shift - 1)) < waves) shift--;
    return shift;
}

uint64_t trace_grid_threads(const TraceLaunch& cfg, uint64_t n, int num_cus) {
    const uint64_t resident = (uint64_t)num_cus * (uint64_t)cfg.waves_per_cu * 64ull;
    uint64_t blocks = (resident + cfg.block - 1) / cfg.block;
    const uint64_t per = (uint64_t)(cfg.block / 64) << trace_ray_shift(cfg, n, num_cus);   // rays per block and round
    const uint64_t need = (n + per - 1) / per;
    if (blocks > need) blocks = need;
    if (blocks < 1) blocks = 1;
    return blocks * (uint64_t)cfg.block;
}

uint64_t trace_spill_columns(const TraceLaunch& cfg, uint64_t n, int num_cus) {
    const uint64_t columns = (trace_grid_threads(cfg, n, num_cus) / 64) << trace_ray_shift(cfg, n, num_cus);
    return (columns + 255) / 256 * 256;
}

hipError_t launch_trace(const SceneView& sv, bool shadow, bool motion, const TraceLaunch& cfg, const void* rays, uint64_t n,
                        void* hits, int32_t* geoms, int32_t* counters, float* spT, int32_t* spN, uint64_t spill_columns,
                        int32_t* err, int num_cus, hipStream_t stream, const uint32_t* n_dev, const uint32_t* perm, bool gather) {
    if (n == 0) return hipSuccess;
    if (n > 0xffffffffull) return hipErrorInvalidValue;
    if (sv.any_xform) {   // no counters
        if (counters) return hipErrorInvalidValue;
        return shadow ? launch_xform<true, false>(sv, cfg, rays, n, hits, geoms, spT, spN, spill_columns, err, num_cus,
                                                  n_dev, perm, gather, stream)
                      : launch_xform<false, false>(sv, cfg, rays, n, hits, geoms, spT, spN, spill_columns, err, num_cus,
                                                   n_dev, perm, gather, stream);
    }
    const uint64_t threads = trace_grid_threads(cfg, n, num_cus);
    if (trace_spill_columns(cfg, n, num_cus) > spill_columns) return hipErrorInvalidValue;
    const uint64_t grid = threads / cfg.block;
    const int ray_shift = trace_ray_shift(cfg, n, num_cus);
#define VGPU_CASE(B, L)                                                                                         \
    if (cfg.block == B && cfg.lds_depth == L)                                                                   \
        return launch_mode<B, L>(sv, shadow, motion, rays, n, hits, geoms, counters, spT, spN, grid, err, n_dev, perm, \
                                 gather, stream, ray_shift, cfg.refill_min);
    VGPU_CASE(64, 8) VGPU_CASE(64, 12) VGPU_CASE(64, 16) VGPU_CASE(64, 24) VGPU_CASE(64, 32)
    VGPU_CASE(128, 8) VGPU_CASE(128, 12) VGPU_CASE(128, 16) VGPU_CASE(128, 24) VGPU_CASE(128, 32)
    VGPU_CASE(256, 8) VGPU_CASE(256, 12) VGPU_CASE(256, 16) VGPU_CASE(256, 24) VGPU_CASE(256, 32)
#undef VGPU_CASE
    return hipErrorInvalidValue;
}

// ------------------------------------------------------------- allocation-free traversal
//
// vgpu_trace_noalloc keeps its traversal spill area in this file-scope array instead of device
// memory the scene allocates.  Layout: the error flag in the first 256 bytes, then the spill
// depths T and nodes N, each (VGPU_MAX_STACK - lds) entries per spill column
// (trace_spill_columns), depth-major.  The array's host-side name is not a device address: host code
// uses only the pointer hipGetSymbolAddress returned for the current device.
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

namespace {

std::mutex g_scratch_mu;
void* g_scratch_ptr[kNoAllocMaxDevices] = {};

__global__ void k_clear_flag(int32_t* flag) {
    if (threadIdx.x == 0 && blockIdx.x == 0) *flag = 0;
}

}  // namespace

hipError_t noalloc_init(int device) {
    if (device < 0 || device >= kNoAllocMaxDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (g_scratch_ptr[device]) return hipSuccess;
    int cur = -1;
    hipError_t e = hipGetDevice(&cur);
    if (e != hipSuccess) return e;
    if (cur != device) return hipErrorInvalidDevice;   // the caller makes `device` current
    void* ptr = nullptr;
    e = hipGetSymbolAddress((void**)&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    g_scratch_ptr[device] = ptr;
    return hipSuccess;
}

uint64_t noalloc_max_columns(int lds_depth) {
    const uint64_t per = (uint64_t)(VGPU_MAX_STACK - lds_depth) * (sizeof(float) + sizeof(int32_t));
    return (kNoAllocScratchBytes - 256) / per;
}

hipError_t launch_trace_noalloc(int device, const SceneView& sv, bool shadow, bool motion, const TraceLaunch& cfg,
                                const void* rays, uint64_t n, void* hits, int32_t* geoms, int32_t* counters,
                                int32_t* status, int num_cus, hipStream_t stream) {
    if (device < 0 || device >= kNoAllocMaxDevices) return hipErrorInvalidDevice;
    unsigned char* base;
    {
        std::lock_guard<std::mutex> lk(g_scratch_mu);
        base = (unsigned char*)g_scratch_ptr[device];
    }
    if (!base) return hipErrorNotInitialized;
    const uint64_t columns = trace_spill_columns(cfg, n, num_cus);
    if (columns > noalloc_max_columns(cfg.lds_depth)) return hipErrorInvalidValue;
    int32_t* flag = status ? status : (int32_t*)base;
    hipLaunchKernelGGL(k_clear_flag, dim3(1), dim3(64), 0, stream, flag);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || n == 0) return e;
    const uint64_t per = (uint64_t)(VGPU_MAX_STACK - cfg.lds_depth);
    float* spT = (float*)(base + 256);
    int32_t* spN = (int32_t*)(base + 256 + per * columns * sizeof(float));
    return launch_trace(sv, shadow, motion, cfg, rays, n, hits, geoms, counters, spT, spN, columns, flag, num_cus,
                        stream, nullptr, nullptr, false);
}

}  // namespace vgpu
