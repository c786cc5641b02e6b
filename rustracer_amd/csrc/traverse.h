// traverse.h — device-side traceRayEXT: two-level 4-wide BVH traversal and the
// watertight ray/triangle test.
//
// Semantics follow what the reference pipeline asks of the driver
// (crates/examples/gltf_viewer/shaders/RayTracing.rgen:89-92,
//  RayTracing.rchit:51-55): closest accepted hit in [tmin, tmax], any-hit on
// non-opaque geometry unless the ray or instance forces opacity, optional
// termination on the first accepted hit, no face culling.  Ties in t are broken
// by the smaller (instance, primitive) so results do not depend on BVH shape.
//
// Stack: a per-lane ring of kDepth entries in LDS (one column per lane, so a
// wave's pushes hit 64 distinct banks).  When the ring overwrites an entry the
// traversal restarts from the top (flattened BVH, then TLAS root) with the current
// closest t once the ring drains: closest-hit and shadow results stay exact; only
// the number of any-hit invocations can change.  After kMaxRestarts restarts the ray gives up and raises
// kErrStackOverflow, so every traversal ends.
#pragma once

#include "common.h"

namespace rt {

constexpr int kStackDepth = 32;  // default ring depth (a power of two)
constexpr uint32_t kMaxRestarts = 64;

struct TraceStats {
    uint32_t nodes = 0, tris = 0, instances = 0, anyhits = 0, overflows = 0;
};

struct HitInfo {
    float t, u, v;
    uint32_t inst;  // index into TlasView::inst
    uint32_t prim;  // gl_PrimitiveID
    uint32_t rec;   // triangle record index in the BLAS pool
};

// Watertight ray/triangle test (Woop, Benthin & Wald, JCGT 2013).  The ray origin
// is passed separately (it is the traversal ray's origin).
struct WoopRay {
    uint32_t k;  // kx | ky << 2 | kz << 4
    float sx, sy, sz;
};

__device__ inline WoopRay woop_setup(float3 d) {
    float ax = fabsf(d.x), ay = fabsf(d.y), az = fabsf(d.z);
    int kz = (ax > ay) ? (ax > az ? 0 : 2) : (ay > az ? 1 : 2);
    int kx = kz == 2 ? 0 : kz + 1;
    int ky = kx == 2 ? 0 : kx + 1;
    float dz = comp(d, kz);
    if (dz < 0.f) { int t = kx; kx = ky; ky = t; }
    WoopRay w;
    w.k = uint32_t(kx) | uint32_t(ky) << 2 | uint32_t(kz) << 4;
    w.sx = comp(d, kx) / dz;
    w.sy = comp(d, ky) / dz;
    w.sz = 1.0f / dz;
    return w;
}

// Returns true and (t, u, v) for a hit with tmin <= t <= tmax.  The edge functions
// are evaluated without FMA contraction: the test is watertight only if a shared
// edge's function evaluates to exactly the negated value in the neighbouring
// triangle, which a fused a*b - c*d does not guarantee.  (The sheared vertex
// coordinates may be fused: a shared vertex gets the same value in both triangles.)
__device__ inline bool woop_hit(const WoopRay& w, float3 o, float3 v0, float3 v1, float3 v2, float tmin, float tmax,
                                float& t, float& bu, float& bv) {
    const int kx = int(w.k & 3u), ky = int((w.k >> 2) & 3u), kz = int(w.k >> 4);
    float3 A = v0 - o, B = v1 - o, C = v2 - o;
    float Akz = comp(A, kz), Bkz = comp(B, kz), Ckz = comp(C, kz);
    float Ax = comp(A, kx) - w.sx * Akz, Ay = comp(A, ky) - w.sy * Akz;
    float Bx = comp(B, kx) - w.sx * Bkz, By = comp(B, ky) - w.sy * Bkz;
    float Cx = comp(C, kx) - w.sx * Ckz, Cy = comp(C, ky) - w.sy * Ckz;
    float U, V, W;
    {
#pragma clang fp contract(off)
        U = Cx * By - Cy * Bx;
        V = Ax * Cy - Ay * Cx;
        W = Bx * Ay - By * Ax;
    }
    if (U == 0.f || V == 0.f || W == 0.f) {
        U = float(double(Cx) * double(By) - double(Cy) * double(Bx));
        V = float(double(Ax) * double(Cy) - double(Ay) * double(Cx));
        W = float(double(Bx) * double(Ay) - double(By) * double(Ax));
    }
    if ((U < 0.f || V < 0.f || W < 0.f) && (U > 0.f || V > 0.f || W > 0.f)) return false;
    float det = U + V + W;
    if (det == 0.f) return false;
    float T = U * (w.sz * Akz) + V * (w.sz * Bkz) + W * (w.sz * Ckz);
    float tt = T / det;
    if (!(tt >= tmin && tt <= tmax)) return false;
    t = tt;
    bu = V / det;
    bv = W / det;
    return true;
}

struct TravRay {
    float3 o, inv;
};

// 1/x of the components of a ray direction.  A component of magnitude under 1e-30 of the
// largest (of 1, for directions longer than that) counts as that magnitude: over the
// lengths rays have it moves the ray by less than any padding, and the box test's
// products stay finite, so an axis-parallel ray is still culled on the axes it does not
// move along.  Directions come in any length; those so short that the products overflow
// give NaN there, which the box test's minima and maxima pass over: they are not culled.
// (The limit is put on the reciprocals: a division then waits for no comparison.)
__device__ inline float3 safe_inv(float3 d) {
    const float3 r = mk3(1.0f / d.x, 1.0f / d.y, 1.0f / d.z);
    const float most = 1e30f * fmaxf(fminf(fabsf(r.x), fminf(fabsf(r.y), fabsf(r.z))), 1.0f);
    return mk3(copysignf(fminf(fabsf(r.x), most), r.x), copysignf(fminf(fabsf(r.y), most), r.y),
               copysignf(fminf(fabsf(r.z), most), r.z));
}

// What one traversal step reads: the 64 bytes of a node, the 48 of a triangle record
// (and 16 unused), or the first 64 of an instance record.
struct StepData {
    uint4 w0, w1, w2, w3;
};
__device__ inline StepData load_step(const void* at) {
    const uint4* p = reinterpret_cast<const uint4*>(at);
    return StepData{ldg_u4(p), ldg_u4(p + 1), ldg_u4(p + 2), ldg_u4(p + 3)};
}

__device__ inline float qbyte(uint32_t w, int k) { return float((w >> (8 * k)) & 255u); }

// Slab test of the four children of a quantised node: entry distance per child, or
// +inf for a child that is missed or empty, and the children's stack entries.
//
// The planes are not decoded: with plane = origin + q 2^e, the distance to it is
// q (2^e inv) + (origin - o) inv, one fused multiply-add per plane, and the sign of inv
// says which of an axis' two planes comes first.  With u = 2^-24 the rounded distance is
// off by at most 3u |b| + 3u |t|, b = (origin - o) inv.  Moving b outward by 5u |b| on
// both sides and the exit by 16u |t| covers both, so a box that the exact ray touches is
// never rejected (as the widened exit of Ize 2013 does for decoded planes).  The planes
// enclose the child unrounded (QNode).
__device__ inline void node_hits(const StepData& n, const TravRay& r, float tmin, float tmax, float key[4],
                                 uint32_t ent[4]) {
    constexpr float kB = 5.0f / 16777216.0f, kT = 16.0f / 16777216.0f;
    const float sx = pow2f(int(int8_t(n.w0.w & 255u))), sy = pow2f(int(int8_t((n.w0.w >> 8) & 255u)));
    const float sz = pow2f(int(int8_t((n.w0.w >> 16) & 255u)));
    const float ax = sx * r.inv.x, ay = sy * r.inv.y, az = sz * r.inv.z;
    const float bx = (__uint_as_float(n.w0.x) - r.o.x) * r.inv.x, by = (__uint_as_float(n.w0.y) - r.o.y) * r.inv.y;
    const float bz = (__uint_as_float(n.w0.z) - r.o.z) * r.inv.z;
    const float bxn = fmaf(-kB, fabsf(bx), bx), bxf = fmaf(kB, fabsf(bx), bx);
    const float byn = fmaf(-kB, fabsf(by), by), byf = fmaf(kB, fabsf(by), by);
    const float bzn = fmaf(-kB, fabsf(bz), bz), bzf = fmaf(kB, fabsf(bz), bz);
    const bool fx = r.inv.x < 0.f, fy = r.inv.y < 0.f, fz = r.inv.z < 0.f;
    const uint32_t xn = fx ? n.w1.y : n.w1.x, xf = fx ? n.w1.x : n.w1.y;
    const uint32_t yn = fy ? n.w1.w : n.w1.z, yf = fy ? n.w1.z : n.w1.w;
    const uint32_t zn = fz ? n.w2.y : n.w2.x, zf = fz ? n.w2.x : n.w2.y;
    const uint32_t child[4] = {n.w2.z, n.w2.w, n.w3.x, n.w3.y};
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const float t0 = fmaxf(fmaxf(fmaf(qbyte(xn, k), ax, bxn), fmaf(qbyte(yn, k), ay, byn)),
                               fmaxf(fmaf(qbyte(zn, k), az, bzn), tmin));
        float t1 = fminf(fminf(fmaf(qbyte(xf, k), ax, bxf), fmaf(qbyte(yf, k), ay, byf)),
                         fminf(fmaf(qbyte(zf, k), az, bzf), tmax));
        t1 = fmaf(kT, fabsf(t1), t1);
        key[k] = (t0 <= t1 && child[k] != kEmpty) ? t0 : INFINITY;
        // the leaf bit and count of the entry are bits 3..7 of byte k of the last word
        ent[k] = child[k] | ((n.w3.w << (24 - 8 * k)) & ~kLeafFirstMask);
    }
}

struct NoAnyHit {
    __device__ bool ignore(uint32_t, uint32_t, float, float) { return false; }
};

// Source of the ray in fp64, read when the traversal enters an instance: the ray is
// taken to object space in fp64 (InstanceRecord::w2o_d) and rounded to fp32 there,
// so the object-space ray carries the rounding of object-space coordinates rather
// than that of the (larger) world coordinates.
struct RayFromF32 {  // the caller's ray is fp32
    float3 o, d;
    __device__ void get(D3& O, D3& Dd) const {
        O = D3{double(o.x), double(o.y), double(o.z)};
        Dd = D3{double(d.x), double(d.y), double(d.z)};
    }
};
struct RayFromF64 {  // the caller holds the fp64 ray
    const D3& o;
    const D3& d;
    __device__ void get(D3& O, D3& Dd) const {
        O = o;
        Dd = d;
    }
};

enum : int { kLevelTlas = 0, kLevelBlas = 1, kLevelFlat = 2 };

// Closest-hit traversal of one ray as a resumable state machine: begin() sets it up,
// each step() processes one node or leaf and returns true once the traversal has
// ended (found / hit then hold the result).  `ah.ignore(inst_index, prim, u, v)` is
// the any-hit shader (true = ignoreIntersectionEXT).
//
// The nearest hit child of a node is kept in a register and only the others go to
// the stack.  The flattened BVH (identity instances) is traversed first, with the
// TLAS root beneath it on the stack, so its hits bound the TLAS traversal.
template <bool kAnyHit, bool kStats, int kDepth = kStackDepth>
struct Traversal {
    static_assert((kDepth & (kDepth - 1)) == 0, "the stack ring depth is a power of two");
    float3 o, d;
    float tmin, best_t;
    uint32_t ray_flags;
    TravRay cur;
    WoopRay wr;
    const QNode* nodes;
    const float4* tris;
    uint32_t inst_idx;
    bool inst_opaque, found, lost;
    int level;
    uint32_t blas_base, sp, base, restarts, e;
    HitInfo hit;

    __device__ void push(uint32_t* stack, uint32_t stride, uint32_t v) {
        stack[(sp & (kDepth - 1)) * stride] = v;
        sp++;
        if (sp - base > uint32_t(kDepth)) {
            base++;
            lost = true;
        }
    }
    __device__ void to_world() { cur = TravRay{o, safe_inv(d)}; }
    __device__ uint32_t enter(const TlasView& tl, uint32_t* stack, uint32_t stride) {
        to_world();
        if (tl.flat_nodes) {
            if (tl.num_tlas) push(stack, stride, tl.root);
            blas_base = sp;
            level = kLevelFlat;
            nodes = tl.flat_nodes;
            tris = tl.flat_tris;
            wr = woop_setup(d);
            return tl.flat_root;
        }
        level = kLevelTlas;
        nodes = tl.nodes;
        return tl.root;
    }
    __device__ void begin(const TlasView& tl, float3 ro, float3 rd, float t0, float t1, uint32_t flags,
                          uint32_t* stack, uint32_t stride) {
        o = ro;
        d = rd;
        tmin = t0;
        best_t = t1;
        ray_flags = flags;
        found = false;
        lost = false;
        hit.inst = kEmpty;
        hit.prim = kEmpty;
        tris = tl.flat_tris;
        inst_idx = 0;
        inst_opaque = true;
        blas_base = 0;
        sp = 0;
        base = 0;
        restarts = 0;
        e = enter(tl, stack, stride);
    }

    template <class AnyHit, class RaySrc>
    __device__ bool step(const TlasView& tl, const RaySrc& rs, AnyHit& ah, uint32_t* stack, uint32_t stride,
                         TraceStats& st) {
        // One load for whatever the entry is.  The lanes of a wave stand at nodes,
        // triangles and instances at once; loaded in each kind's own branch, a step
        // waited for memory once per kind.  A leaf's triangles are tested one per step, so
        // that no lane's second record is waited for by the others.  With the box test
        // above (about 160 vector operations a node instead of 260) the 1080p frame of
        // the 2M-triangle sphere went from 190 to 174 ms, a 720p frame of 1000
        // alpha-tested instances from 45.8 to 38.4 ms, 4096 ray queries from 140 to 117 us.
        const bool leaf = (e & kLeafBit) != 0u;
        const bool entry = leaf && level == kLevelTlas;
        const uint32_t first = e & kLeafFirstMask;
        const char* at;
        if (entry) at = reinterpret_cast<const char*>(tl.inst + first);
        else if (leaf) at = reinterpret_cast<const char*>(tris + 3 * size_t(first));
        else at = reinterpret_cast<const char*>(nodes + e);
        const StepData n = load_step(at);
        if (!leaf) {
            // internal node
            if (kStats) st.nodes++;
            float key[4];
            uint32_t ent[4];
            node_hits(n, cur, tmin, best_t, key, ent);
            // order the hit children near-to-far: continue with the nearest, push the
            // others far first
#define RT_CSWAP(i, j)                                                         \
    {                                                                          \
        const bool s_ = key[j] < key[i];                                       \
        const float tk = s_ ? key[j] : key[i], th = s_ ? key[i] : key[j];      \
        const uint32_t te = s_ ? ent[j] : ent[i], tf = s_ ? ent[i] : ent[j];   \
        key[i] = tk; key[j] = th; ent[i] = te; ent[j] = tf;                    \
    }
            RT_CSWAP(0, 1) RT_CSWAP(2, 3) RT_CSWAP(0, 2) RT_CSWAP(1, 3) RT_CSWAP(1, 2)
#undef RT_CSWAP
            if (key[0] < INFINITY) {
#pragma unroll
                for (int k = 3; k >= 1; k--)
                    if (key[k] < INFINITY) {
                        stack[(sp & (kDepth - 1)) * stride] = ent[k];
                        sp++;
                    }
                if (sp - base > uint32_t(kDepth)) {
                    base = sp - uint32_t(kDepth);
                    lost = true;
                }
                e = ent[0];
                return false;
            }
        } else if (entry) {
            // TLAS leaf: one instance
            const uint4* ip = reinterpret_cast<const uint4*>(at);
            const uint4 w4 = ldg_u4(ip + 4), w5 = ldg_u4(ip + 5), w6 = ldg_u4(ip + 6), w7 = ldg_u4(ip + 7);
            if (kStats) st.instances++;
            const uint32_t fl = w7.z;
            if ((w7.y & 0xFFu) != 0u && !(fl & kInstEmpty)) {
                D3 O, Dd;
                rs.get(O, Dd);
                const double m[12] = {pair_f64(n.w0.x, n.w0.y), pair_f64(n.w0.z, n.w0.w), pair_f64(n.w1.x, n.w1.y),
                                      pair_f64(n.w1.z, n.w1.w), pair_f64(n.w2.x, n.w2.y), pair_f64(n.w2.z, n.w2.w),
                                      pair_f64(n.w3.x, n.w3.y), pair_f64(n.w3.z, n.w3.w), pair_f64(w4.x, w4.y),
                                      pair_f64(w4.z, w4.w), pair_f64(w5.x, w5.y), pair_f64(w5.z, w5.w)};
                float3 oo = mk3(float(m[0] * O.x + m[1] * O.y + m[2] * O.z + m[3]),
                                float(m[4] * O.x + m[5] * O.y + m[6] * O.z + m[7]),
                                float(m[8] * O.x + m[9] * O.y + m[10] * O.z + m[11]));
                float3 od = mk3(float(m[0] * Dd.x + m[1] * Dd.y + m[2] * Dd.z),
                                float(m[4] * Dd.x + m[5] * Dd.y + m[6] * Dd.z),
                                float(m[8] * Dd.x + m[9] * Dd.y + m[10] * Dd.z));
                cur.o = oo;
                cur.inv = safe_inv(od);
                wr = woop_setup(od);
                nodes = reinterpret_cast<const QNode*>(pair_u64(w6.x, w6.y));
                tris = reinterpret_cast<const float4*>(pair_u64(w6.z, w6.w));
                inst_idx = first;
                bool opq = (fl & kInstOpaqueGeom) != 0;
                if (fl & kInstForceOpaque) opq = true;
                if (fl & kInstForceNoOpaque) opq = false;
                if (ray_flags & RT_RAY_FLAG_OPAQUE) opq = true;
                if (ray_flags & RT_RAY_FLAG_NO_OPAQUE) opq = false;
                inst_opaque = opq;
                level = kLevelBlas;
                blas_base = sp;
                e = w7.x;
                return false;
            }
        } else {
            // one triangle of a leaf of a BLAS or of the flattened BVH
            if (kStats) st.tris++;
            float t, bu, bv;
            if (woop_hit(wr, cur.o, as_f3(n.w0), as_f3(n.w1), as_f3(n.w2), tmin, best_t, t, bu, bv)) {
                const uint32_t prim = n.w0.w;
                uint32_t ii = inst_idx, rec = first;
                bool opq = inst_opaque;
                if (level == kLevelFlat) {
                    ii = n.w1.w & ~kFlatOpaque;
                    rec = n.w2.w;
                    opq = (n.w1.w & kFlatOpaque) != 0u;
                    if (ray_flags & RT_RAY_FLAG_OPAQUE) opq = true;
                    if (ray_flags & RT_RAY_FLAG_NO_OPAQUE) opq = false;
                }
                bool keep = true;
                if (found && t == best_t) {
                    const uint32_t hi = tl.inst[ii].instance_id, ho = tl.inst[hit.inst].instance_id;
                    keep = hi < ho || (hi == ho && prim <= hit.prim);
                }
                if (kAnyHit && keep && !opq) {
                    if (kStats) st.anyhits++;
                    keep = !ah.ignore(ii, prim, bu, bv);
                }
                if (keep) {
                    found = true;
                    best_t = t;
                    hit.t = t;
                    hit.u = bu;
                    hit.v = bv;
                    hit.inst = ii;
                    hit.prim = prim;
                    hit.rec = rec;
                    if (ray_flags & RT_RAY_FLAG_TERMINATE_ON_FIRST_HIT) return true;
                }
            }
            if (e & (15u << kLeafCountShift)) {  // more triangles in this leaf
                e = e - (1u << kLeafCountShift) + 1u;
                return false;
            }
        }
        // next entry from the stack
        if (sp == base) {
            if (!lost) return true;
            lost = false;
            if (kStats) st.overflows++;
            if (++restarts > kMaxRestarts) {
                if (tl.error_flags) atomicOr(tl.error_flags, kErrStackOverflow);
                return true;
            }
            e = enter(tl, stack, stride);
            return false;
        }
        sp--;
        e = stack[(sp & (kDepth - 1)) * stride];
        if (level != kLevelTlas && sp < blas_base) {
            level = kLevelTlas;
            to_world();
            nodes = tl.nodes;
        }
        return false;
    }
};

// Runs one traversal to completion.  Returns true on a hit.
template <bool kAnyHit, bool kStats, int kDepth = kStackDepth, class AnyHit, class RaySrc>
__device__ bool trace_ray(const TlasView& tl, float3 o, float3 d, const RaySrc& rs, float tmin, float tmax,
                          uint32_t ray_flags, AnyHit& ah, uint32_t* lds_stack, uint32_t stride, HitInfo& hit,
                          TraceStats& st) {
    Traversal<kAnyHit, kStats, kDepth> tr;
    tr.begin(tl, o, d, tmin, tmax, ray_flags, lds_stack, stride);
    while (!tr.step(tl, rs, ah, lds_stack, stride, st)) {
    }
    hit = tr.hit;
    return tr.found;
}

}  // namespace rt
