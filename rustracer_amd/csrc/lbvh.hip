// lbvh.hip — batched LBVH build for gfx950 (see lbvh.h).
//
// Pipeline per build (all on one stream):
//   1. primitive boxes + per-segment bounds (reduced per workgroup before the atomics)
//   2. 64-bit keys: segment id above an interleaved Morton code
//   3. LSD radix sort, 8 bits per pass: LDS histogram, three-kernel scan, and an
//      LDS-staged stable scatter that ranks keys with wave ballots; small builds sort
//      by rank in one launch
//   4. Karras (HPG 2012) radix-tree emission, one thread per internal node
//   5. bottom-up passes over tiles of the tree in LDS: treelet restructuring, boxes
//   6. top-down collapse into 4-wide quantised nodes, two launches per level.  With the
//      SAH collapse (default), the bottom-up pass also solves, bottom-up, for every
//      binary node n and every number of slots i = 1..4 it may take in its parent's
//      wide node, the least surface-area-heuristic cost of its subtree
//        C(n, 1) = min(leaf: c_tri |n| A(n) if |n| <= leaf size,
//                      wide node: c_node A(n) + min_{i=2..4} D(n, i))
//        D(n, i) = min_{k=1..i-1} C(left, k) + C(right, i - k)
//        C(n, i) = min(C(n, i - 1), D(n, i))
//      (the dynamic program of Ylitie, Karras & Laine, HPG 2017, for 4-wide nodes),
//      and the collapse follows the decisions; the greedy form opens the
//      largest-surface-area child that is too big for a leaf until four children
//      are gathered
#include <string>

#include "lbvh.h"

namespace rt {

namespace {

constexpr int kBlock = 256;
constexpr int kRsItems = 8;
constexpr int kRsTile = kBlock * kRsItems;
constexpr int kScanPerBlock = 1024;  // 256 threads x 4 elements

#define RT_CHECK_LAUNCH()                              \
    do {                                               \
        hipError_t e_ = hipGetLastError();             \
        if (e_ != hipSuccess) return int(e_);          \
    } while (0)
#define RT_CHECK(x)                                    \
    do {                                               \
        hipError_t e_ = (x);                           \
        if (e_ != hipSuccess) return int(e_);          \
    } while (0)

inline uint32_t blocks_for(uint64_t n, int per) { return uint32_t((n + per - 1) / per); }

__device__ inline uint32_t find_segment(const uint32_t* seg_start, uint32_t nseg, uint32_t p) {
    uint32_t lo = 0, hi = nseg;  // seg_start[lo] <= p < seg_start[hi]
    while (hi - lo > 1) {
        uint32_t mid = (lo + hi) >> 1;
        if (seg_start[mid] <= p) lo = mid; else hi = mid;
    }
    return lo;
}

// ------------------------------------------------------------ primitives
__global__ void k_prepare_triangles(const TriSegment* segs, uint32_t nseg, uint32_t n, float4* tri, float4* lo,
                                    float4* hi, uint32_t* bad) {
    uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    // segments: binary search over prim_start
    uint32_t a = 0, b = nseg;
    while (b - a > 1) {
        uint32_t m = (a + b) >> 1;
        if (segs[m].prim_start <= p) a = m; else b = m;
    }
    const TriSegment& s = segs[a];
    uint32_t local = p - s.prim_start;
    float3 v[3];
    bool ok = true;
    for (int k = 0; k < 3; k++) {
        uint32_t idx = s.index_data[3 * size_t(local) + k];
        if (idx > s.max_vertex) { ok = false; idx = 0; }
        const float* f = (const float*)(s.vertex_data + size_t(s.first_vertex + idx) * s.stride);
        v[k] = mk3(f[0], f[1], f[2]);
    }
    if (!ok) {
        atomicOr(bad, 1u);
        v[1] = v[0];
        v[2] = v[0];
    }
    tri[3 * size_t(p) + 0] = make_float4(v[0].x, v[0].y, v[0].z, __uint_as_float(local));
    tri[3 * size_t(p) + 1] = make_float4(v[1].x, v[1].y, v[1].z, 0.f);
    tri[3 * size_t(p) + 2] = make_float4(v[2].x, v[2].y, v[2].z, 0.f);
    float3 l = fmin3(fmin3(v[0], v[1]), v[2]);
    float3 h = fmax3(fmax3(v[0], v[1]), v[2]);
    lo[p] = make_float4(l.x, l.y, l.z, 0.f);
    hi[p] = make_float4(h.x, h.y, h.z, 0.f);
}

__global__ void k_reorder_tris(const float4* in, const uint32_t* perm, uint32_t n, float4* out) {
    uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    uint32_t s = perm[p];
    out[3 * size_t(p) + 0] = in[3 * size_t(s) + 0];
    out[3 * size_t(p) + 1] = in[3 * size_t(s) + 1];
    out[3 * size_t(p) + 2] = in[3 * size_t(s) + 2];
}

// One axis of a node: the grid (origin, exponent) and the 8-bit planes of the
// non-empty children, each rounded outward so that fmaf(q, 2^e, origin) lies on or
// outside the child's plane.  Traversal takes the plane unrounded, which is at most half
// an ulp further in: the padding of the child's plane covers it (QNode).
__device__ inline void quantize_axis(const float lo[4], const float hi[4], const uint32_t child[4], float& origin,
                                     int8_t& exp, uint8_t qlo[4], uint8_t qhi[4]) {
    float o = INFINITY, top = -INFINITY;
    for (int k = 0; k < 4; k++) {
        qlo[k] = 0;
        qhi[k] = 0;
        if (child[k] == kEmpty) continue;
        o = fminf(o, lo[k]);
        top = fmaxf(top, hi[k]);
    }
    if (!(o <= top)) {  // no child
        origin = 0.f;
        exp = 0;
        return;
    }
    // smallest e with 254 * 2^e >= the extent (one step of room for the outward fixes)
    const double ext = double(top) - double(o);
    int e = -126;
    if (ext > 0.0) {
        int k = 0;
        (void)frexp(ext / 254.0, &k);  // ext / 254 = m 2^k, m in [0.5, 1)
        e = k < -126 ? -126 : (k > 127 ? 127 : k);
    }
    for (; e <= 127; e++) {
        const float s = pow2f(e);
        bool fits = true;
        for (int k = 0; k < 4 && fits; k++) {
            if (child[k] == kEmpty) continue;
            float ql = floorf((lo[k] - o) / s);
            if (!(ql >= 0.f)) ql = 0.f;
            if (ql > 255.f) ql = 255.f;
            for (int it = 0; it < 4 && ql > 0.f && fmaf(ql, s, o) > lo[k]; it++) ql -= 1.f;
            if (fmaf(ql, s, o) > lo[k]) ql = 0.f;  // q = 0 decodes to the origin, the smallest lo
            float qh = ceilf((hi[k] - o) / s);
            if (!(qh >= ql)) qh = ql;
            if (qh > 256.f) qh = 256.f;
            for (int it = 0; it < 4 && fmaf(qh, s, o) < hi[k]; it++) qh += 1.f;
            if (qh > 255.f || fmaf(qh, s, o) < hi[k]) {
                fits = false;
                break;
            }
            qlo[k] = uint8_t(ql);
            qhi[k] = uint8_t(qh);
        }
        if (fits || e == 127) break;
    }
    if (e > 127) e = 127;
    origin = o;
    exp = int8_t(e);
}

__device__ inline QNode quantize_node(const WideNode& w) {
    QNode q;
    q._pad0 = 0;
    quantize_axis(w.lo_x, w.hi_x, w.child, q.origin[0], q.exp[0], q.q + 0, q.q + 4);
    quantize_axis(w.lo_y, w.hi_y, w.child, q.origin[1], q.exp[1], q.q + 8, q.q + 12);
    quantize_axis(w.lo_z, w.hi_z, w.child, q.origin[2], q.exp[2], q.q + 16, q.q + 20);
    for (int k = 0; k < 4; k++) {
        q.child[k] = w.child[k];
        q.count[k] = uint8_t(w.count[k]);
        // child | tag << 24 is the traversal's stack entry (a leaf's child is below 2^27)
        q.tag[k] = w.count[k] ? uint8_t(0x80u | (w.count[k] - 1u) << 3) : uint8_t(0);
    }
    return q;
}

__global__ void k_gather_flat(const FlatSource* src, uint32_t nsrc, uint32_t n, float4* tri, float4* lo, float4* hi) {
    uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    uint32_t a = 0, b = nsrc;
    while (b - a > 1) {
        uint32_t m = (a + b) >> 1;
        if (src[m].start <= p) a = m; else b = m;
    }
    const FlatSource& s = src[a];
    const uint32_t rec = s.first_rec + (p - s.start);
    const float4* t = s.tris + 3 * size_t(rec);
    float4 v0 = t[0], v1 = t[1], v2 = t[2];
    tri[3 * size_t(p) + 0] = v0;  // w: primitive index
    tri[3 * size_t(p) + 1] = make_float4(v1.x, v1.y, v1.z, __uint_as_float(s.inst_bits));
    tri[3 * size_t(p) + 2] = make_float4(v2.x, v2.y, v2.z, __uint_as_float(rec));
    float3 l = fmin3(fmin3(xyz(v0), xyz(v1)), xyz(v2));
    float3 h = fmax3(fmax3(xyz(v0), xyz(v1)), xyz(v2));
    lo[p] = make_float4(l.x, l.y, l.z, 0.f);
    hi[p] = make_float4(h.x, h.y, h.z, 0.f);
}

__global__ void k_prepare_instances(const InstanceRecord* inst, uint32_t n, float4* lo, float4* hi) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const InstanceRecord& r = inst[i];
    float3 l = mk3(INFINITY, INFINITY, INFINITY), h = mk3(-INFINITY, -INFINITY, -INFINITY);
    if (!(r.flags & kInstEmpty)) {
        const float* bb = r.blas->bounds;
        for (int c = 0; c < 8; c++) {
            float3 p = mk3((c & 1) ? bb[3] : bb[0], (c & 2) ? bb[4] : bb[1], (c & 4) ? bb[5] : bb[2]);
            float3 w = mk3(r.o2w[0].x * p.x + r.o2w[0].y * p.y + r.o2w[0].z * p.z + r.o2w[0].w,
                           r.o2w[1].x * p.x + r.o2w[1].y * p.y + r.o2w[1].z * p.z + r.o2w[1].w,
                           r.o2w[2].x * p.x + r.o2w[2].y * p.y + r.o2w[2].z * p.z + r.o2w[2].w);
            l = fmin3(l, w);
            h = fmax3(h, w);
        }
        // rounding of the transform: pad by a few ulp of the magnitude
        float3 m = fmax3(mk3(fabsf(l.x), fabsf(l.y), fabsf(l.z)), mk3(fabsf(h.x), fabsf(h.y), fabsf(h.z)));
        float pad = fmaxf(fmaxf(m.x, m.y), m.z) * 1.0e-6f + 1e-30f;
        l = l - mk3(pad, pad, pad);
        h = h + mk3(pad, pad, pad);
    } else {
        // empty BLAS: a degenerate box at the origin that no traversal needs to enter
        l = mk3(0.f, 0.f, 0.f);
        h = l;
    }
    lo[i] = make_float4(l.x, l.y, l.z, 0.f);
    hi[i] = make_float4(h.x, h.y, h.z, 0.f);
}

__global__ void k_reorder_instances(const InstanceRecord* in, const uint32_t* perm, uint32_t n, InstanceRecord* out) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    out[i] = in[perm[i]];
}

// ------------------------------------------------------- segment bounds
// bounds: per segment 12 uints: centroid lo/hi (ordered), box lo/hi (ordered)
__global__ void k_init_bounds(uint32_t* bounds, uint32_t nseg) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nseg * 12) return;
    uint32_t k = i % 12;
    bool is_lo = (k < 3) || (k >= 6 && k < 9);
    bounds[i] = is_lo ? f2ord(INFINITY) : f2ord(-INFINITY);
}

constexpr uint32_t kBoundsItems = 16;  // most primitives per thread of k_seg_bounds
// enough workgroups to fill the chip twice before a thread takes more than one
inline uint32_t bounds_span(uint32_t n) {
    return uint32_t(kBlock) * std::min(std::max(n / (uint32_t(kBlock) * 512u), 1u), kBoundsItems);
}

__device__ inline bool bound_is_lo(int k) { return k < 3 || (k >= 6 && k < 9); }
__device__ inline void bounds_none(float v[12]) {
#pragma unroll
    for (int k = 0; k < 12; k++) v[k] = bound_is_lo(k) ? INFINITY : -INFINITY;
}
__device__ inline void bounds_add(float v[12], float4 l, float4 h) {
    const float c[3] = {0.5f * (l.x + h.x), 0.5f * (l.y + h.y), 0.5f * (l.z + h.z)};
    const float b[6] = {l.x, l.y, l.z, h.x, h.y, h.z};
#pragma unroll
    for (int k = 0; k < 3; k++) {
        v[k] = fminf(v[k], c[k]);
        v[3 + k] = fmaxf(v[3 + k], c[k]);
        v[6 + k] = fminf(v[6 + k], b[k]);
        v[9 + k] = fmaxf(v[9 + k], b[3 + k]);
    }
}
__device__ inline void bounds_wave(float v[12]) {
#pragma unroll
    for (int k = 0; k < 12; k++)
        for (int o = 32; o > 0; o >>= 1) {
            const float y = __shfl_xor(v[k], o, 64);
            v[k] = bound_is_lo(k) ? fminf(v[k], y) : fmaxf(v[k], y);
        }
}
__device__ inline void bounds_atomic(uint32_t* b, int k, float v) {
    if (bound_is_lo(k)) atomicMin(&b[k], f2ord(v));
    else atomicMax(&b[k], f2ord(v));
}

// A workgroup reduces up to 4096 primitives before its 12 atomics: all of one segment's
// atomics go to the same 12 words, one after another (one set per wave took 4.2 ms for a
// segment of 2M primitives, this 87 us; 4096 for 5,120 primitives as well were 50 us).
__global__ __launch_bounds__(kBlock) void k_seg_bounds(const float4* lo, const float4* hi, uint32_t n,
                                                        const uint32_t* seg_start, uint32_t nseg, uint32_t span,
                                                        uint32_t* bounds) {
    __shared__ float s_v[kBlock / 64][12];
    const uint32_t base = blockIdx.x * span;
    const uint32_t end = base + min(span, n - base);
    const uint32_t s0 = find_segment(seg_start, nseg, base);
    float v[12];
    if (s0 == find_segment(seg_start, nseg, end - 1u)) {
        bounds_none(v);
        for (uint32_t p = base + threadIdx.x; p < end; p += kBlock) bounds_add(v, lo[p], hi[p]);
        bounds_wave(v);
        if ((threadIdx.x & 63u) == 0u)
            for (int k = 0; k < 12; k++) s_v[threadIdx.x >> 6][k] = v[k];
        __syncthreads();
        if (threadIdx.x < 12u) {
            const int k = int(threadIdx.x);
            float x = s_v[0][k];
            for (int w = 1; w < kBlock / 64; w++) x = bound_is_lo(k) ? fminf(x, s_v[w][k]) : fmaxf(x, s_v[w][k]);
            bounds_atomic(bounds + 12 * size_t(s0), k, x);
        }
        return;
    }
    // several segments: a wave at a time
    for (uint32_t row = base; row < end; row += kBlock) {
        const uint32_t p = row + threadIdx.x;
        const bool valid = p < end;
        const uint32_t seg = valid ? find_segment(seg_start, nseg, p) : 0u;
        bounds_none(v);
        if (valid) bounds_add(v, lo[p], hi[p]);
        const uint64_t live = __ballot(valid);
        if (!live) continue;  // the wave's row is past the end
        const uint32_t w0 = __shfl(seg, 0, 64);  // lane 0 is valid when any lane is
        if (__ballot(valid && seg != w0) == 0ull) {
            bounds_wave(v);
            if (__lane_id() == 0)
                for (int k = 0; k < 12; k++) bounds_atomic(bounds + 12 * size_t(w0), k, v[k]);
        } else if (valid) {
            for (int k = 0; k < 12; k++) bounds_atomic(bounds + 12 * size_t(seg), k, v[k]);
        }
    }
}

// ---------------------------------------------------------------- Morton
__device__ inline uint64_t split3(uint32_t a) {
    uint64_t x = a & 0x1fffffu;
    x = (x | x << 32) & 0x1f00000000ffffull;
    x = (x | x << 16) & 0x1f0000ff0000ffull;
    x = (x | x << 8) & 0x100f00f00f00f00full;
    x = (x | x << 4) & 0x10c30c30c30c30c3ull;
    x = (x | x << 2) & 0x1249249249249249ull;
    return x;
}

__global__ void k_morton(const float4* lo, const float4* hi, uint32_t n, const uint32_t* seg_start, uint32_t nseg,
                         const uint32_t* bounds, int bits, uint64_t* keys, uint32_t* vals) {
    uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    uint32_t seg = find_segment(seg_start, nseg, p);
    const uint32_t* b = bounds + 12 * seg;
    float4 l = lo[p], h = hi[p];
    float c[3] = {0.5f * (l.x + h.x), 0.5f * (l.y + h.y), 0.5f * (l.z + h.z)};
    float scale = float((1u << bits) - 1u);
    uint32_t q[3];
    for (int k = 0; k < 3; k++) {
        float cl = ord2f(b[k]), ch = ord2f(b[3 + k]);
        float ext = ch - cl;
        float t = ext > 0.f ? (c[k] - cl) / ext : 0.5f;
        t = fminf(fmaxf(t, 0.f), 1.f);
        q[k] = uint32_t(t * scale);
    }
    uint64_t code = (split3(q[0]) << 2) | (split3(q[1]) << 1) | split3(q[2]);
    keys[p] = (uint64_t(seg) << (3 * bits)) | code;
    vals[p] = p;
}

// ------------------------------------------------------------ radix sort
__global__ __launch_bounds__(kBlock) void k_rs_hist(const uint64_t* keys, uint32_t n, int shift, uint32_t* hist,
                                                     uint32_t nblocks) {
    __shared__ uint32_t h[256];
    h[threadIdx.x] = 0;
    __syncthreads();
    uint32_t base = blockIdx.x * kRsTile;
    for (int i = threadIdx.x; i < kRsTile; i += kBlock) {
        uint32_t idx = base + i;
        if (idx < n) atomicAdd(&h[uint32_t(keys[idx] >> shift) & 255u], 1u);
    }
    __syncthreads();
    hist[threadIdx.x * nblocks + blockIdx.x] = h[threadIdx.x];
}

__global__ __launch_bounds__(kBlock) void k_scan_local(uint32_t* data, uint32_t m, uint32_t* sums) {
    __shared__ uint32_t s[kBlock];
    uint32_t base = blockIdx.x * kScanPerBlock + threadIdx.x * 4;
    uint32_t v[4], t = 0;
    for (int k = 0; k < 4; k++) {
        v[k] = (base + k < m) ? data[base + k] : 0u;
        uint32_t x = v[k];
        v[k] = t;
        t += x;
    }
    s[threadIdx.x] = t;
    __syncthreads();
    for (int o = 1; o < kBlock; o <<= 1) {
        uint32_t y = threadIdx.x >= uint32_t(o) ? s[threadIdx.x - o] : 0u;
        __syncthreads();
        s[threadIdx.x] += y;
        __syncthreads();
    }
    uint32_t excl = s[threadIdx.x] - t;
    for (int k = 0; k < 4; k++)
        if (base + k < m) data[base + k] = v[k] + excl;
    if (threadIdx.x == kBlock - 1) sums[blockIdx.x] = s[kBlock - 1];
}

__global__ __launch_bounds__(kBlock) void k_scan_add(uint32_t* data, uint32_t m, const uint32_t* sums) {
    uint32_t base = blockIdx.x * kScanPerBlock + threadIdx.x * 4;
    uint32_t add = sums[blockIdx.x];
    for (int k = 0; k < 4; k++)
        if (base + k < m) data[base + k] += add;
}

__global__ __launch_bounds__(kBlock) void k_rs_scatter(const uint64_t* kin, const uint32_t* vin, uint64_t* kout,
                                                        uint32_t* vout, uint32_t n, int shift, const uint32_t* offs,
                                                        uint32_t nblocks) {
    __shared__ uint32_t s_base[256];
    __shared__ uint32_t s_cnt[kBlock / 64][256];
    const uint32_t tid = threadIdx.x, wave = tid >> 6;
    s_base[tid] = offs[tid * nblocks + blockIdx.x];
    const uint32_t base = blockIdx.x * kRsTile;
    for (int r = 0; r < kRsItems; r++) {
        for (int k = tid; k < (kBlock / 64) * 256; k += kBlock) (&s_cnt[0][0])[k] = 0u;
        __syncthreads();
        uint32_t idx = base + r * kBlock + tid;
        bool valid = idx < n;
        uint64_t key = valid ? kin[idx] : 0ull;
        uint32_t val = valid ? vin[idx] : 0u;
        uint32_t digit = uint32_t(key >> shift) & 255u;
        uint64_t peers = __ballot(valid);
        for (int b = 0; b < 8; b++) {
            bool bit = (digit >> b) & 1u;
            uint64_t bal = __ballot(bit);
            peers &= bit ? bal : ~bal;
        }
        uint32_t rank = __popcll(peers & lanemask_lt());
        if (valid && rank == 0) s_cnt[wave][digit] = __popcll(peers);
        __syncthreads();
        uint32_t total;
        {
            uint32_t c0 = s_cnt[0][tid], c1 = s_cnt[1][tid], c2 = s_cnt[2][tid], c3 = s_cnt[3][tid];
            s_cnt[0][tid] = 0;
            s_cnt[1][tid] = c0;
            s_cnt[2][tid] = c0 + c1;
            s_cnt[3][tid] = c0 + c1 + c2;
            total = c0 + c1 + c2 + c3;
        }
        __syncthreads();
        if (valid) {
            uint32_t pos = s_base[digit] + s_cnt[wave][digit] + rank;
            if (pos < n) {  // always true for a consistent histogram
                kout[pos] = key;
                vout[pos] = val;
            }
        }
        __syncthreads();
        s_base[tid] += total;
        __syncthreads();
    }
}

// Sort of at most kRankMax keys in one launch: the position of a key is the number of
// keys below it, counting equal keys of smaller index (the stable order of the radix
// passes).  kRankSlices lanes share a key's count.  Kernel time against that of the 24 to
// 40 radix launches: 22 us to 120 us at 5,120 keys, 66 to 167 at 16,384; at 32,768 the
// n^2 compares take 260 us, the radix passes 170.
constexpr uint32_t kRankMax = 16384;
constexpr int kRankKeys = 64, kRankSlices = 16;

__global__ __launch_bounds__(kRankKeys * kRankSlices) void k_rank_sort(const uint64_t* kin, const uint32_t* vin,
                                                                      uint32_t n, uint64_t* kout, uint32_t* vout) {
    __shared__ uint32_t s_rank[kRankKeys];
    const uint32_t e = threadIdx.x & (kRankKeys - 1), slice = threadIdx.x / kRankKeys;
    const uint32_t i = blockIdx.x * kRankKeys + e;
    if (threadIdx.x < kRankKeys) s_rank[threadIdx.x] = 0u;
    __syncthreads();
    const uint64_t key = i < n ? kin[i] : 0ull;
    const uint32_t per = (n + kRankSlices - 1) / kRankSlices;
    const uint32_t j0 = min(slice * per, n), j1 = min(j0 + per, n);
    uint32_t c = 0;
#pragma unroll 8
    for (uint32_t j = j0; j < j1; j++) {
        const uint64_t k = kin[j];  // the same address in every lane of a wave
        c += (k < key || (k == key && j < i)) ? 1u : 0u;
    }
    atomicAdd(&s_rank[e], c);
    __syncthreads();
    if (slice == 0 && i < n) {
        const uint32_t r = s_rank[e];  // below n: the counts of n keys are a permutation
        kout[r] = key;
        vout[r] = vin[i];
    }
}

int exclusive_scan(hipStream_t st, uint32_t* d, uint32_t m, uint32_t* tmp, uint32_t tmp_cap) {
    uint32_t nb = blocks_for(m, kScanPerBlock);
    if (nb > tmp_cap) return int(hipErrorInvalidValue);
    hipLaunchKernelGGL(k_scan_local, dim3(nb), dim3(kBlock), 0, st, d, m, tmp);
    RT_CHECK_LAUNCH();
    if (nb > 1) {
        int rc = exclusive_scan(st, tmp, nb, tmp + nb, tmp_cap - nb);
        if (rc) return rc;
        hipLaunchKernelGGL(k_scan_add, dim3(nb), dim3(kBlock), 0, st, d, m, tmp);
        RT_CHECK_LAUNCH();
    }
    return 0;
}

// ---------------------------------------------------------------- Karras
__device__ inline int delta(const uint64_t* k, int n, int i, int j) {
    if (j < 0 || j >= n) return -1;
    uint64_t a = k[i], b = k[j];
    if (a == b) return 64 + __clz(uint32_t(i ^ j));
    return __clzll(a ^ b);
}

__global__ void k_karras(const uint64_t* keys, int n, uint32_t* left, uint32_t* right, uint32_t* first,
                         uint32_t* last, uint32_t* parent_int, uint32_t* parent_leaf, const uint32_t* seg_start,
                         uint32_t nseg, int seg_shift, uint32_t* seg_root, uint32_t* is_root, uint32_t* split_node) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    // the root of the whole tree (node 0, or the only leaf) has no parent
    if (i == 0) {
        if (n == 1) parent_leaf[0] = kEmpty;
        else parent_int[0] = kEmpty;
    }
    if (i >= n - 1) return;
    int d = (delta(keys, n, i, i + 1) - delta(keys, n, i, i - 1)) >= 0 ? 1 : -1;
    int dmin = delta(keys, n, i, i - d);
    int lmax = 2;
    while (delta(keys, n, i, i + lmax * d) > dmin) lmax <<= 1;
    int l = 0;
    for (int t = lmax >> 1; t >= 1; t >>= 1)
        if (delta(keys, n, i, i + (l + t) * d) > dmin) l += t;
    int j = i + l * d;
    int dnode = delta(keys, n, i, j);
    int s = 0, t = l;
    do {
        t = (t + 1) >> 1;
        if (delta(keys, n, i, i + (s + t) * d) > dnode) s += t;
    } while (t > 1);
    int gamma = i + s * d + min(d, 0);
    int lo = min(i, j), hi = max(i, j);
    uint32_t lc = (lo == gamma) ? (kLeafBit | uint32_t(gamma)) : uint32_t(gamma);
    uint32_t rc = (hi == gamma + 1) ? (kLeafBit | uint32_t(gamma + 1)) : uint32_t(gamma + 1);
    left[i] = lc;
    right[i] = rc;
    split_node[gamma] = i;  // the node that parts leaf gamma from gamma + 1
    first[i] = lo;
    last[i] = hi;
    if (lc & kLeafBit) parent_leaf[gamma] = i; else parent_int[gamma] = i;
    if (rc & kLeafBit) parent_leaf[gamma + 1] = i; else parent_int[gamma + 1] = i;
    uint32_t seg = uint32_t(keys[lo] >> seg_shift);
    const bool root = seg < nseg && uint32_t(lo) == seg_start[seg] && uint32_t(hi) + 1 == seg_start[seg + 1];
    is_root[i] = root ? 1u : 0u;
    if (root) seg_root[seg] = i;
}

// --------------------------------------------------------------- box fit
__device__ inline void load_box(uint32_t ref, const float4* lo, const float4* hi, const uint32_t* perm,
                                const float4* nlo, const float4* nhi, float3& l, float3& h) {
    if (ref & kLeafBit) {
        uint32_t s = perm[ref & ~kLeafBit];
        l = xyz(lo[s]);
        h = xyz(hi[s]);
    } else {
        l = xyz(nlo[ref]);
        h = xyz(nhi[ref]);
    }
}

__device__ inline float half_area(float3 l, float3 h) {
    float3 e = h - l;
    return e.x * e.y + e.y * e.z + e.z * e.x;
}

// Surface-area-heuristic costs of the 4-wide collapse: a wide node's visit against
// a triangle test, per unit of (half) surface area.
constexpr float kSahNodeCost = 1.0f;
constexpr float kSahTriCost = 0.6f;

// Decision word of one binary node (SAH collapse):
//   bit 0       C(n, 1) is a wide node (else a leaf)
//   bits 2i..   for i = 2..4 (2 bits each, at 2, 4, 6): k of D(n, i), 0 = C(n, i - 1)
//   bits 8..9   i* - 2 of the node's own wide node, bits 10..11 its k*
__device__ inline uint32_t dec_slots(uint32_t d, int i) { return (d >> (2 * (i - 1))) & 3u; }

// Exclusive sum over the workgroup; `total` gets the sum of all.
template <int T> __device__ inline uint32_t block_exclusive(uint32_t v, uint32_t* s_wave, uint32_t& total) {
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    uint32_t x = v;
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = __shfl_up(x, o, 64);
        if (lane >= uint32_t(o)) x += y;
    }
    __syncthreads();
    if (lane == 63u) s_wave[wave] = x;
    __syncthreads();
    uint32_t before = 0;
    total = 0;
    for (uint32_t w = 0; w < uint32_t(T) / 64u; w++) {
        if (w < wave) before += s_wave[w];
        total += s_wave[w];
    }
    return before + x - v;
}

// ------------------------------------------------- bottom-up passes
// Boxes, treelet restructuring and SAH costs are computed bottom-up: of the two threads
// that reach a node from below, the second handles it.  Done over the whole tree in
// global memory, every node costs an agent-scope acquire-release, which writes back and
// invalidates caches (8.3 ms for the box fit alone of 2M primitives, 15.8 ms for a
// treelet pass).  So the tree is taken in tiles of consecutive leaves: the nodes whose
// leaves lie in one tile of kTile leaves are handled by one workgroup, in LDS, all passes
// in one launch; then those of a tile kFan times as large, over the subtrees that the
// smaller tiles left, and so on (k_tree_level).  A subtree of a smaller tile is not
// opened again, so a treelet does not reach across it: node visits per ray are the same
// to 0.1 %.  For 2M primitives both treelet passes, boxes and SAH costs take
// 2.0 ms, against 39.8 ms.
constexpr int kTile = 512;        // leaves of a first tile, and its threads
constexpr int kTileRefs = 768;    // subtrees a larger tile can hold
constexpr int kTileThreads = 256; // threads of a larger tile
// A tile leaves about 15 subtrees, so 16 tiles make a larger one; where a tile turns out to
// hold more than kTileRefs, the build starts over with 4, whose subtrees always fit.
constexpr uint32_t kFan = 16, kFanSafe = 4;
// Subtrees of unfinished segments that a tile leaves: they hang off the tree's paths to
// the tile's first and last leaf, one per node of a path, and a path is shorter than the
// key and index bits together.
constexpr uint32_t kTileRoots = 192;
static_assert(kFanSafe * kTileRoots <= uint32_t(kTileRefs), "four tiles' subtrees fit");
constexpr uint32_t kOverflowNodes = 1u, kOverflowRoots = 2u, kOverflowFan = 4u;  // bits of the overflow word

// SAH costs C(n, 1..4) of a node from its children's costs and boxes; the decision word
// is returned in d.
__device__ inline float4 sah_costs(float4 ca4, float4 cb4, float area, uint32_t count, uint32_t leaf_max, uint32_t& d) {
    const float ca[5] = {0.f, ca4.x, ca4.y, ca4.z, ca4.w}, cb[5] = {0.f, cb4.x, cb4.y, cb4.z, cb4.w};
    float dist[5];
    uint32_t kbest[5];
#pragma unroll
    for (int i = 2; i <= 4; i++) {
        dist[i] = INFINITY;
        kbest[i] = 1;
#pragma unroll
        for (int k = 1; k < i; k++) {
            const float c = ca[k] + cb[i - k];
            if (c < dist[i]) { dist[i] = c; kbest[i] = uint32_t(k); }
        }
    }
    uint32_t istar = 2, kstar = kbest[2];
    float dmin = dist[2];
#pragma unroll
    for (int i = 3; i <= 4; i++)
        if (dist[i] < dmin) { dmin = dist[i]; istar = uint32_t(i); kstar = kbest[i]; }
    const float c_int = kSahNodeCost * area + dmin;
    const float c_leaf = count <= leaf_max ? kSahTriCost * float(count) * area : INFINITY;
    float c[5];
    d = 0;
    if (c_int < c_leaf) { c[1] = c_int; d |= 1u; } else { c[1] = c_leaf; }
#pragma unroll
    for (int i = 2; i <= 4; i++) {
        if (dist[i] < c[i - 1]) { c[i] = dist[i]; d |= kbest[i] << (2 * (i - 1)); }
        else c[i] = c[i - 1];
    }
    d |= (istar - 2u) << 8;
    d |= kstar << 10;
    return make_float4(c[1], c[2], c[3], c[4]);
}
// a primitive costs one triangle test wherever it goes
__device__ inline float4 sah_leaf(float3 l, float3 h) {
    const float c = kSahTriCost * half_area(l, h);
    return make_float4(c, c, c, c);
}

// Treelet restructuring (Karras & Aila, "Fast Parallel Construction of High-Quality
// Bounding Volume Hierarchies", HPG 2013): bottom up, each node of the binary tree gathers
// a treelet of up to kTreeletLeaves leaves (it opens the largest-area internal leaf until
// that many are gathered), finds the binary tree over those leaves of least
// surface-area-heuristic cost by a dynamic program over the leaf subsets, and rebuilds
// the treelet that way when that is cheaper, reusing its internal nodes.  Cost of a
// subtree: kTreeletNodeCost * A(n) + C(left) + C(right), and kTreeletTriCost * A(p) for a
// primitive.  Subtrees stop covering contiguous runs of the sorted primitives; a
// renumbering in depth-first order restores that before the collapse.
// Five leaves: 90 splits of 26 subsets per node, all in registers (every index of the
// arrays below is a constant once unrolled).  Seven leaves gave 10.12 against 10.18 node
// visits per ray (10.71 without restructuring) for nine times the splits.
constexpr int kTreeletLeaves = 5;
constexpr float kTreeletNodeCost = 1.2f;
constexpr float kTreeletTriCost = 1.0f;
constexpr int kMaxWalk = 1 << 16;  // bound of the walks up the binary tree

struct TreeRef {  // what a pass needs of a node or leaf
    float3 l, h;
    float c;     // treelet cost
    uint32_t n;  // primitives
};

template <class T> __device__ inline T pick5(const T (&a)[5], uint32_t i) {
    T r = a[0];
#pragma unroll
    for (uint32_t k = 1; k < 5; k++) r = i == k ? a[k] : r;
    return r;
}

// box, cost and primitive count of `node` from its children, stored; the cost and count
// are returned
template <class Store> __device__ inline float tree_refresh(Store& st, uint32_t node, uint32_t& count) {
    const TreeRef a = st.get(st.left(node)), b = st.get(st.right(node));
    TreeRef r;
    r.l = fmin3(a.l, b.l);
    r.h = fmax3(a.h, b.h);
    r.c = kTreeletNodeCost * half_area(r.l, r.h) + a.c + b.c;
    r.n = a.n + b.n;
    st.put(node, r);
    count = r.n;
    return r.c;
}

template <class Store> __device__ inline void treelet_optimize(Store& st, uint32_t node, float cur) {
    constexpr int M = kTreeletLeaves;
    static_assert(M == 5, "the subset words below hold 5-bit subsets");
    uint32_t leaf[M], inner[M];
    TreeRef lf[M];
    leaf[0] = st.left(node);
    leaf[1] = st.right(node);
    lf[0] = st.get(leaf[0]);
    lf[1] = st.get(leaf[1]);
    inner[0] = node;
    uint32_t m = 2;
#pragma unroll
    for (int k = 2; k < M; k++) {
        leaf[k] = leaf[0];
        lf[k] = lf[0];
        inner[k - 1] = node;
    }
    inner[M - 1] = node;
#pragma unroll
    for (int k = 2; k < M; k++) {
        if (m != uint32_t(k)) break;
        int best = -1;
        float best_a = -1.f;
#pragma unroll
        for (int j = 0; j < k; j++) {
            const float ar = half_area(lf[j].l, lf[j].h);
            if (!st.is_leaf(leaf[j]) && ar > best_a) { best_a = ar; best = j; }
        }
        if (best < 0) break;
        const uint32_t x = pick5(leaf, uint32_t(best));
        inner[k - 1] = x;
        const uint32_t xl = st.left(x), xr = st.right(x);
        const TreeRef tl = st.get(xl), tr = st.get(xr);
#pragma unroll
        for (int j = 0; j < k; j++)
            if (j == best) {
                leaf[j] = xl;
                lf[j] = tl;
            }
        leaf[k] = xr;
        lf[k] = tr;
        m = uint32_t(k) + 1u;
    }
    if (m < 3u) return;
    // least cost of a binary tree over each subset S of the leaves; part(S), the subset of
    // S that goes to the left child, in 5 bits of pw
    const uint32_t full = (1u << m) - 1u;
    float cost[1 << M];
    uint64_t pw[3] = {0ull, 0ull, 0ull};
#pragma unroll
    for (int k = 0; k < M; k++) cost[1 << k] = lf[k].c;
    float all = INFINITY;
#pragma unroll
    for (uint32_t S = 3; S < (1u << M); S++) {
        if ((S & (S - 1u)) == 0u) continue;
        if (S > full) break;
        float3 l = mk3(INFINITY, INFINITY, INFINITY), h = mk3(-INFINITY, -INFINITY, -INFINITY);
#pragma unroll
        for (int i = 0; i < M; i++)
            if ((S >> i) & 1u) { l = fmin3(l, lf[i].l); h = fmax3(h, lf[i].h); }
        const uint32_t low = S & (0u - S);
        float best = INFINITY;
        uint32_t bp = low;
#pragma unroll
        for (uint32_t P = 1; P < S; P++) {  // the left part holds the lowest leaf
            if ((P & S) != P || !(P & low)) continue;
            const float c = cost[P] + cost[S ^ P];
            if (c < best) { best = c; bp = P; }
        }
        cost[S] = kTreeletNodeCost * half_area(l, h) + best;
        pw[S / 12] |= uint64_t(bp) << (5 * (S % 12));
        if (S == full) all = cost[S];
    }
    if (!(all < 0.9999f * cur)) return;
    // rebuild: internal node inner[k] takes subset k of the queue, top down
    uint32_t queue = full, next = 1;
#pragma unroll
    for (int k = 0; k < M - 1; k++) {
        if (uint32_t(k) >= next) break;
        const uint32_t S = (queue >> (5 * k)) & 31u;
        const uint32_t w = S / 12u;
        const uint32_t P = uint32_t((w == 0u ? pw[0] : (w == 1u ? pw[1] : pw[2])) >> (5u * (S - 12u * w))) & 31u;
        const uint32_t sub[2] = {P, S ^ P};
        uint32_t ref[2];
#pragma unroll
        for (int c = 0; c < 2; c++) {
            if ((sub[c] & (sub[c] - 1u)) == 0u) {
                ref[c] = pick5(leaf, uint32_t(__ffs(int(sub[c]))) - 1u);
            } else {
                ref[c] = pick5(inner, next);
                queue |= sub[c] << (5u * next);
                next++;
            }
            st.set_parent(ref[c], inner[k]);
        }
        st.set_children(inner[k], ref[0], ref[1]);
    }
    // children before parents (a child's place in the queue is behind its parent's)
    uint32_t count;
#pragma unroll
    for (int k = M - 2; k >= 0; k--)
        if (uint32_t(k) < next) (void)tree_refresh(st, inner[k], count);
}

struct TreeArgs {
    const float4* lo;   // primitive boxes
    const float4* hi;
    const uint32_t* perm;  // sorted position -> primitive
    const uint64_t* keys;  // sorted
    int seg_shift;
    const uint32_t* seg_start;
    const uint32_t* first;  // leaf range of each node as the radix tree was emitted
    const uint32_t* last;
    const uint32_t* split_node;
    uint32_t* left;
    uint32_t* right;
    uint32_t* parent_int;
    uint32_t* parent_leaf;
    float4* nlo;     // node boxes; nlo.w: treelet cost
    float4* nhi;
    uint32_t* cnt;   // primitives under each node
    float4* cost;    // C(n, 1..4) (SAH collapse)
    uint32_t* dec;   // decision words (SAH collapse)
    uint32_t* overflow;
    uint32_t n;
    uint32_t passes;   // treelet passes
    uint32_t leaf_max;
    uint32_t sah;
};

// The subtrees ("entities", 0..C-1, in leaf order) and nodes (C..2C-1) of one tile in LDS.
// Node k is the one whose split lies between entities k and k + 1.
template <int C> struct TileStore {
    static constexpr uint32_t kNone = 0xFFFFu;
    float lo[3][2 * C], hi[3][2 * C];
    float cost[2 * C];
    uint32_t cnt[2 * C];
    uint32_t ref[C];   // entity: kLeafBit | leaf position, or the subtree's root node
    uint32_t id[C];    // node id (kEmpty: the split's node is not of this tile)
    uint16_t child[2][C], parent[2 * C];
    uint32_t seen[C / 32];

    __device__ bool is_leaf(uint32_t e) const { return e < uint32_t(C); }
    __device__ uint32_t left(uint32_t e) const { return child[0][e - C]; }
    __device__ uint32_t right(uint32_t e) const { return child[1][e - C]; }
    __device__ TreeRef get(uint32_t e) const {
        TreeRef r;
        r.l = mk3(lo[0][e], lo[1][e], lo[2][e]);
        r.h = mk3(hi[0][e], hi[1][e], hi[2][e]);
        r.c = cost[e];
        r.n = cnt[e];
        return r;
    }
    __device__ void put(uint32_t e, const TreeRef& r) {
        lo[0][e] = r.l.x; lo[1][e] = r.l.y; lo[2][e] = r.l.z;
        hi[0][e] = r.h.x; hi[1][e] = r.h.y; hi[2][e] = r.h.z;
        cost[e] = r.c;
        cnt[e] = r.n;
    }
    __device__ void set_children(uint32_t e, uint32_t a, uint32_t b) {
        child[0][e - C] = uint16_t(a);
        child[1][e - C] = uint16_t(b);
    }
    __device__ void set_parent(uint32_t e, uint32_t p) { parent[e] = uint16_t(p); }
    // the second thread to arrive at a node handles it; workgroup scope: what the first one
    // wrote, to LDS or through this CU's cache, is visible
    __device__ bool second(uint32_t e) {
        const uint32_t k = e - C, bit = 1u << (k & 31u);
        return (__hip_atomic_fetch_or(&seen[k >> 5], bit, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_WORKGROUP) & bit) != 0u;
    }
};

// One level: tile blockIdx.x of `size` leaves, T threads.  kFirst: its entities are the
// leaves, else the subtrees that `fan` tiles of the level before left (roots_in,
// kTileRoots a tile).
template <int C, int T, bool kFirst>
__global__ __launch_bounds__(T, 4) void k_tree_level(TreeArgs a, uint32_t size, uint32_t fan, const uint32_t* roots_in,
                                                     const uint32_t* count_in, uint32_t tiles_in, uint32_t* roots_out,
                                                     uint32_t* count_out) {
    using Store = TileStore<C>;
    __shared__ Store ts;
    __shared__ uint32_t s_wave[T / 64];
    const uint32_t t = threadIdx.x, n = a.n;
    const uint32_t base = blockIdx.x * size, end = base + min(size, n - base);
    uint32_t* const lastpos = reinterpret_cast<uint32_t*>(ts.cost + C);  // until the node costs are written
    // entities
    uint32_t ne = 0;
    if (kFirst) {
        ne = end - base;
        for (uint32_t e = t; e < ne; e += T) ts.ref[e] = kLeafBit | (base + e);
    } else {
        // an earlier level that did not finish: its tiles' subtrees are missing (read once,
        // so that every thread decides alike)
        if (t == 0) s_wave[0] = *a.overflow;
        __syncthreads();
        if (s_wave[0]) return;
        __syncthreads();
        for (uint32_t k = 0; k < fan; k++) {
            const uint32_t tile = blockIdx.x * fan + k;
            const uint32_t c = tile < tiles_in ? count_in[tile] : 0u;
            if (ne + c > uint32_t(C)) {  // the same for every thread
                if (t == 0) {
                    atomicOr(a.overflow, kOverflowFan);
                    if (roots_out) count_out[blockIdx.x] = 0u;
                }
                return;
            }
            for (uint32_t i = t; i < c; i += T) ts.ref[ne + i] = roots_in[tile * kTileRoots + i];
            ne += c;
        }
    }
    __syncthreads();
    for (uint32_t e = t; e < ne; e += T) {
        const uint32_t r = ts.ref[e];
        TreeRef x;
        if (r & kLeafBit) {
            const uint32_t pos = r & ~kLeafBit, s = a.perm[pos];
            x.l = xyz(a.lo[s]);
            x.h = xyz(a.hi[s]);
            x.c = kTreeletTriCost * half_area(x.l, x.h);
            x.n = 1u;
            lastpos[e] = pos;
        } else {
            const float4 lw = a.nlo[r];
            x.l = xyz(lw);
            x.h = xyz(a.nhi[r]);
            x.c = lw.w;
            x.n = a.cnt[r];
            lastpos[e] = a.last[r];
        }
        ts.put(e, x);
        ts.parent[e] = Store::kNone;
    }
    // nodes: the one of each split between neighbouring entities, if its leaves are of this
    // tile and of one segment
    for (uint32_t k = t; k < uint32_t(C); k += T) {
        ts.id[k] = kEmpty;
        ts.parent[C + k] = Store::kNone;
    }
    __syncthreads();
    for (uint32_t k = t; k + 1u < ne; k += T) {
        const uint32_t q = a.split_node[lastpos[k]];
        const uint32_t f = a.first[q], l = a.last[q];
        if (f >= base && l < end && (a.keys[f] >> a.seg_shift) == (a.keys[l] >> a.seg_shift)) ts.id[k] = q;
    }
    __syncthreads();
    for (uint32_t k = t; k + 1u < ne; k += T) {
        const uint32_t q = ts.id[k];
        if (q == kEmpty) continue;
        // a child is the entity beside the split, or the node of a split found by its leaf
        // (the emitted tree's left child is numbered by the last leaf before the split)
        uint32_t c[2] = {a.left[q], a.right[q]};
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const uint32_t beside = k + uint32_t(j);
            if (ts.ref[beside] == c[j]) {
                c[j] = beside;
            } else {
                const uint32_t split = a.left[c[j]] & ~kLeafBit;
                uint32_t lo = 0, hi = ne - 1u;  // the entity that ends at leaf `split`
                while (lo < hi) {
                    const uint32_t mid = (lo + hi) >> 1;
                    if (lastpos[mid] < split) lo = mid + 1u;
                    else hi = mid;
                }
                c[j] = uint32_t(C) + lo;
            }
            ts.parent[c[j]] = uint16_t(C + k);
        }
        ts.child[0][k] = uint16_t(c[0]);
        ts.child[1][k] = uint16_t(c[1]);
    }
    __syncthreads();
    auto clear_seen = [&]() {
        if (t < uint32_t(C) / 32u) ts.seen[t] = 0u;
        __syncthreads();
    };
    // the treelet passes, or one pass that only fits the boxes
    for (uint32_t pass = 0; pass == 0u || pass < a.passes; pass++) {
        clear_seen();
        for (uint32_t e0 = t; e0 < ne; e0 += T) {
            for (uint32_t e = ts.parent[e0]; e != Store::kNone; e = ts.parent[e]) {
                if (!ts.second(e)) break;
                uint32_t count;
                const float cur = tree_refresh(ts, e, count);
                if (pass < a.passes && count >= 3u) treelet_optimize(ts, e, cur);
            }
        }
        __syncthreads();
    }
    if (a.sah) {
        clear_seen();
        for (uint32_t e0 = t; e0 < ne; e0 += T) {
            for (uint32_t e = ts.parent[e0]; e != Store::kNone; e = ts.parent[e]) {
                if (!ts.second(e)) break;
                const uint32_t k = e - C;
                float4 c[2];
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    const uint32_t r = ts.child[j][k];
                    const uint32_t g = ts.is_leaf(r) ? ts.ref[r] : ts.id[r - C];
                    if (g & kLeafBit) {
                        const TreeRef x = ts.get(r);
                        c[j] = sah_leaf(x.l, x.h);
                    } else {
                        c[j] = a.cost[g];
                    }
                }
                const TreeRef x = ts.get(e);
                uint32_t d;
                const uint32_t q = ts.id[k];
                a.cost[q] = sah_costs(c[0], c[1], half_area(x.l, x.h), x.n, a.leaf_max, d);
                a.dec[q] = d;
            }
        }
    }
    // back to global memory, and the subtrees without a parent here, in leaf order
    auto global_ref = [&](uint32_t e) { return e < uint32_t(C) ? ts.ref[e] : ts.id[e - C]; };
    for (uint32_t e = t; e < ne; e += T) {
        if (ts.parent[e] != Store::kNone) {
            const uint32_t r = ts.ref[e], q = ts.id[ts.parent[e] - C];
            if (r & kLeafBit) a.parent_leaf[r & ~kLeafBit] = q;
            else a.parent_int[r] = q;
        }
        const uint32_t q = ts.id[e];
        if (q == kEmpty) continue;
        const uint32_t x = C + e;
        a.left[q] = global_ref(ts.child[0][e]);
        a.right[q] = global_ref(ts.child[1][e]);
        if (ts.parent[x] != Store::kNone) a.parent_int[q] = ts.id[ts.parent[x] - C];
        a.nlo[q] = make_float4(ts.lo[0][x], ts.lo[1][x], ts.lo[2][x], ts.cost[x]);
        a.nhi[q] = make_float4(ts.hi[0][x], ts.hi[1][x], ts.hi[2][x], 0.f);
        a.cnt[q] = ts.cnt[x];
    }
    if (!roots_out) return;
    __syncthreads();
    // the root that starts at each entity: itself, or the topmost node it is the first
    // entity of (found from the node: its first leaf as emitted, which a root keeps); none
    // for a finished segment
    uint32_t* const start = reinterpret_cast<uint32_t*>(ts.lo);  // the boxes are stored
    auto first_leaf = [&](uint32_t r) { return (r & kLeafBit) ? (r & ~kLeafBit) : a.first[r]; };
    auto unfinished = [&](uint32_t r) {
        const uint32_t f = first_leaf(r), l = (r & kLeafBit) ? f : a.last[r];
        const uint32_t seg = uint32_t(a.keys[f] >> a.seg_shift);
        return a.seg_start[seg] != f || a.seg_start[seg + 1u] != l + 1u;
    };
    for (uint32_t e = t; e < ne; e += T)
        start[e] = ts.parent[e] == Store::kNone && unfinished(ts.ref[e]) ? ts.ref[e] : kEmpty;
    __syncthreads();
    for (uint32_t k = t; k + 1u < ne; k += T) {
        if (ts.id[k] == kEmpty || ts.parent[C + k] != Store::kNone || !unfinished(ts.id[k])) continue;
        const uint32_t f = a.first[ts.id[k]];
        uint32_t lo = 0, hi = ne - 1u;  // the entity that starts at leaf f
        while (lo < hi) {
            const uint32_t mid = (lo + hi) >> 1;
            if (first_leaf(ts.ref[mid]) < f) lo = mid + 1u;
            else hi = mid;
        }
        start[lo] = ts.id[k];
    }
    __syncthreads();
    uint32_t done = 0;
    for (uint32_t row = 0; row < ne; row += T) {
        const uint32_t r = row + t < ne ? start[row + t] : kEmpty;
        uint32_t total;
        const uint32_t at = done + block_exclusive<T>(r != kEmpty ? 1u : 0u, s_wave, total);
        if (r != kEmpty && at < kTileRoots) roots_out[blockIdx.x * kTileRoots + at] = r;
        done += total;
    }
    if (t == 0) {
        if (done > kTileRoots) atomicOr(a.overflow, kOverflowRoots);  // cannot happen (kTileRoots)
        count_out[blockIdx.x] = min(done, kTileRoots);
    }
}

// Depth-first renumbering after the treelet passes.  first/last of each internal
// node below a segment root: the root keeps its run, a right child starts after its
// left sibling's primitives.  Nodes above the roots are left as built.
__global__ void k_renumber_nodes(const uint32_t* left, const uint32_t* right, const uint32_t* parent_int,
                                 const uint32_t* is_root, const uint32_t* cnt, uint32_t* first, uint32_t* last, int ni,
                                 const uint32_t* overflow) {
    if (*overflow) return;  // the tree is not complete
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= ni) return;
    uint32_t off = 0, c = uint32_t(i);
    for (int up = 0; !is_root[c]; up++) {
        const uint32_t p = parent_int[c];
        if (p == kEmpty || up >= kMaxWalk) return;
        if (right[p] == c) {
            const uint32_t l = left[p];
            off += (l & kLeafBit) ? 1u : cnt[l];
        }
        c = p;
    }
    const uint32_t f = first[c] + off;  // c is the segment root, whose run stays
    first[i] = f;
    last[i] = f + cnt[i] - 1u;
}

// new sorted position of each primitive
__global__ void k_renumber_leaves(const uint32_t* left, const uint32_t* parent_leaf, const uint32_t* first,
                                  const uint32_t* cnt, const uint32_t* seg_start, uint32_t nseg, uint32_t* newpos,
                                  uint32_t n,
                                  const uint32_t* overflow) {
    if (*overflow) return;  // the tree is not complete
    const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    const uint32_t s = find_segment(seg_start, nseg, p);
    const uint32_t q = parent_leaf[p];
    if (q == kEmpty || seg_start[s + 1] - seg_start[s] < 2u) {
        newpos[p] = p;
        return;
    }
    const uint32_t l = left[q];
    newpos[p] = first[q] + (l == (kLeafBit | p) ? 0u : ((l & kLeafBit) ? 1u : cnt[l]));
}

__global__ void k_renumber_apply(const uint32_t* newpos, const uint32_t* perm_in, uint32_t* perm_out, uint32_t* left,
                                 uint32_t* right, uint32_t n,
                                 const uint32_t* overflow) {
    if (*overflow) return;  // the tree is not complete
    const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    perm_out[newpos[p]] = perm_in[p];
    if (p + 1u >= n) return;
    const uint32_t l = left[p], r = right[p];
    if (l & kLeafBit) left[p] = kLeafBit | newpos[l & ~kLeafBit];
    if (r & kLeafBit) right[p] = kLeafBit | newpos[r & ~kLeafBit];
}

// -------------------------------------------------------------- collapse
struct CollapseArgs {
    const float4* lo;
    const float4* hi;
    const uint32_t* perm;
    const float4* nlo;
    const float4* nhi;
    const uint32_t* left;
    const uint32_t* right;
    const uint32_t* first;
    const uint32_t* last;
    const uint32_t* seg_start;
    uint32_t nseg;
    const float* seg_pad;  // absolute padding per segment
    uint32_t leaf_max;
    QNode* nodes;
    uint32_t max_nodes;     // capacity of nodes and of each task array
    uint32_t* overflow;     // set when a capacity would be exceeded
    const uint32_t* dec;    // SAH decision words (NULL: the greedy largest-area collapse)
    uint2* levels;          // per tree level: tasks, first node of the next level
    uint32_t* block_sums;   // kCollapseBlocks: internal children of each workgroup's tasks
};

__device__ inline uint32_t ref_count(const CollapseArgs& a, uint32_t r) {
    return (r & kLeafBit) ? 1u : (a.last[r] - a.first[r] + 1u);
}
__device__ inline uint32_t ref_first(const CollapseArgs& a, uint32_t r) {
    return (r & kLeafBit) ? (r & ~kLeafBit) : a.first[r];
}
// Collapse of one level, in two launches so node numbering is deterministic: gather
// picks the (up to 4) children of every task and numbers the ones that become internal
// wide nodes within its workgroup; emit adds the counts of the workgroups before its own,
// writes the nodes, quantised, and numbers the new internal nodes level by level in task
// order.  Level sizes stay on the device, so the host enqueues the levels without
// waiting for each: a read-back leaves the device idle for 30 to 45 us, a level of 5,000
// primitives takes 12 us.
constexpr uint32_t kCollapseBlocks = 1024;
// task = (binary ref or kEmpty, wide node index, segment)
// SAH collapse: the children of the wide node made from binary node b, following
// the decisions (each (ref, slots) pair is expanded until it takes one slot).
__device__ inline int gather_children_sah(const CollapseArgs& a, uint32_t b, uint32_t c[4]) {
    const uint32_t d = a.dec[b];
    const uint32_t istar = ((d >> 8) & 3u) + 2u, kstar = (d >> 10) & 3u;
    uint32_t sr[4], ss[4];
    int sp = 0, nc = 0;
    sr[sp] = a.right[b]; ss[sp++] = istar - kstar;
    sr[sp] = a.left[b]; ss[sp++] = kstar;
    while (sp > 0 && nc < 4) {
        const uint32_t r = sr[--sp];
        uint32_t j = ss[sp];
        if (!(r & kLeafBit)) {
            while (j > 1u && dec_slots(a.dec[r], int(j)) == 0u) j--;  // C(r, j) = C(r, j - 1)
        }
        if ((r & kLeafBit) || j == 1u) {
            c[nc++] = r;
            continue;
        }
        const uint32_t k = dec_slots(a.dec[r], int(j));
        if (sp + 2 > 4) { c[nc++] = r; continue; }  // cannot happen: slots add up to at most 4
        sr[sp] = a.right[r]; ss[sp++] = j - k;
        sr[sp] = a.left[r]; ss[sp++] = k;
    }
    return nc;
}

__device__ inline int gather_children(const CollapseArgs& a, uint32_t b, uint32_t c[4], float3 cl[4], float3 ch[4]) {
    int nc;
    if (b == kEmpty) return 0;
    if (b & kLeafBit) { c[0] = b; nc = 1; }
    else if (a.dec) return gather_children_sah(a, b, c);
    else { c[0] = a.left[b]; c[1] = a.right[b]; nc = 2; }
    for (int k = 0; k < nc; k++) load_box(c[k], a.lo, a.hi, a.perm, a.nlo, a.nhi, cl[k], ch[k]);
    while (nc < 4) {
        int best = -1;
        float best_a = -1.f;
        for (int k = 0; k < nc; k++) {
            if ((c[k] & kLeafBit) || ref_count(a, c[k]) <= a.leaf_max) continue;
            float ar = half_area(cl[k], ch[k]);
            if (ar > best_a) { best_a = ar; best = k; }
        }
        if (best < 0) break;
        uint32_t node = c[best];
        c[best] = a.left[node];
        c[nc] = a.right[node];
        load_box(c[best], a.lo, a.hi, a.perm, a.nlo, a.nhi, cl[best], ch[best]);
        load_box(c[nc], a.lo, a.hi, a.perm, a.nlo, a.nhi, cl[nc], ch[nc]);
        nc++;
    }
    return nc;
}

__device__ inline bool becomes_internal(const CollapseArgs& a, uint32_t r) {
    if (r & kLeafBit) return false;
    if (a.dec) return (a.dec[r] & 1u) != 0u;
    return ref_count(a, r) > a.leaf_max;
}

// tasks of workgroup b of a level with n tasks: whole rows of kBlock
__device__ inline uint2 collapse_range(uint32_t n) {
    const uint32_t rows = (n + kBlock - 1) / kBlock, per = (rows + gridDim.x - 1) / gridDim.x;
    const uint32_t b = min(blockIdx.x * per * kBlock, n);
    return make_uint2(b, min(b + per * kBlock, n));
}

__global__ __launch_bounds__(kBlock) void k_collapse_gather(CollapseArgs a, uint32_t level, const uint4* tasks,
                                                             uint4* refs, uint32_t* offsets) {
    __shared__ uint32_t s_wave[kBlock / 64];
    // (a tree that is not complete has no levels)
    const uint2 r = collapse_range(*a.overflow ? 0u : a.levels[level].x);
    uint32_t sum = 0;
    for (uint32_t row = r.x; row < r.y; row += kBlock) {
        const uint32_t t = row + threadIdx.x;
        uint32_t internal = 0;
        if (t < r.y) {
            uint32_t c[4] = {kEmpty, kEmpty, kEmpty, kEmpty};
            float3 cl[4], ch[4];
            const int nc = gather_children(a, tasks[t].x, c, cl, ch);
            for (int k = 0; k < nc; k++) internal += becomes_internal(a, c[k]) ? 1u : 0u;
            refs[t] = make_uint4(c[0], c[1], c[2], c[3]);
        }
        uint32_t total;
        const uint32_t off = block_exclusive<kBlock>(internal, s_wave, total);
        if (t < r.y) offsets[t] = sum + off;
        sum += total;
    }
    if (threadIdx.x == 0) a.block_sums[blockIdx.x] = sum;
}

__global__ __launch_bounds__(kBlock) void k_collapse_emit(CollapseArgs a, uint32_t level, const uint4* tasks,
                                                           const uint4* refs, const uint32_t* offsets, uint4* tasks_out) {
    __shared__ uint32_t s_wave[kBlock / 64];
    const uint2 lv = a.levels[level];
    const uint2 r = collapse_range(*a.overflow ? 0u : lv.x);
    uint32_t mine = 0, before;
    for (uint32_t b = threadIdx.x; b < blockIdx.x; b += kBlock) mine += a.block_sums[b];
    (void)block_exclusive<kBlock>(mine, s_wave, before);
    if (blockIdx.x + 1u == gridDim.x && threadIdx.x == 0) {
        const uint32_t count = before + a.block_sums[blockIdx.x];
        a.levels[level + 1u] = make_uint2(count, lv.y + count);
    }
    for (uint32_t t = r.x + threadIdx.x; t < r.y; t += kBlock) {
        const uint4 task = tasks[t], r4 = refs[t];
        const uint32_t seg = task.z;
        const uint32_t c[4] = {r4.x, r4.y, r4.z, r4.w};
        const float pad = a.seg_pad[seg];
        uint32_t next = before + offsets[t];
        WideNode out;
        for (int k = 0; k < 4; k++) {
            if (c[k] == kEmpty) {
                out.lo_x[k] = out.lo_y[k] = out.lo_z[k] = 0.f;
                out.hi_x[k] = out.hi_y[k] = out.hi_z[k] = 0.f;
                out.child[k] = kEmpty;
                out.count[k] = 0;
                continue;
            }
            float3 cl, ch;
            load_box(c[k], a.lo, a.hi, a.perm, a.nlo, a.nhi, cl, ch);
            out.lo_x[k] = cl.x - pad; out.lo_y[k] = cl.y - pad; out.lo_z[k] = cl.z - pad;
            out.hi_x[k] = ch.x + pad; out.hi_y[k] = ch.y + pad; out.hi_z[k] = ch.z + pad;
            if (!becomes_internal(a, c[k])) {
                out.child[k] = ref_first(a, c[k]);
                out.count[k] = ref_count(a, c[k]);
            } else {
                const uint32_t idx = lv.y + next;
                if (idx >= a.max_nodes || next >= a.max_nodes) {
                    atomicOr(a.overflow, kOverflowNodes);
                    out.child[k] = kEmpty;
                    out.count[k] = 0;
                    continue;
                }
                tasks_out[next] = make_uint4(c[k], idx, seg, 0u);
                out.child[k] = idx;
                out.count[k] = 0;
                next++;
            }
        }
        if (task.y < a.max_nodes) a.nodes[task.y] = quantize_node(out);
    }
}

// level 0: one task per segment, its root is node s (kEmpty for an empty segment)
__global__ void k_init_tasks(const uint32_t* seg_root, uint32_t nseg, uint4* tasks, uint2* levels) {
    uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s == 0u) levels[0] = make_uint2(nseg, nseg);
    if (s >= nseg) return;
    tasks[s] = make_uint4(seg_root[s], s, s, 0u);
}

// padding and root bounds per segment, and the roots of segments without a binary node
__global__ void k_seg_pad(const uint32_t* bounds, const uint32_t* seg_start, uint32_t nseg, float* pad,
                          float* seg_bounds, uint32_t* seg_root, uint32_t* overflow) {
    uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s == 0u) *overflow = 0u;
    if (s >= nseg) return;
    const uint32_t prims = seg_start[s + 1] - seg_start[s];
    if (prims < 2u) seg_root[s] = prims ? (kLeafBit | seg_start[s]) : kEmpty;
    const uint32_t* b = bounds + 12 * s;
    float m = 0.f;
    float v[6];
    for (int k = 0; k < 6; k++) {
        v[k] = ord2f(b[6 + k]);
        if (isfinite(v[k])) m = fmaxf(m, fabsf(v[k]));
    }
    // about 8 ulp of the largest coordinate magnitude of the segment
    float p = m * 9.5367431640625e-07f + 1e-30f;  // 2^-20
    pad[s] = p;
    bool empty = !(v[0] <= v[3]);
    for (int k = 0; k < 3; k++) {
        seg_bounds[6 * s + k] = empty ? 0.f : v[k] - p;
        seg_bounds[6 * s + 3 + k] = empty ? 0.f : v[3 + k] + p;
    }
}

// ------------------------------------------------------------ refit
// Largest coordinate magnitudes (non-negative floats order as their bits).  The maxima of
// one segment go to one word, one after another: a wave brings one (when it is of one
// segment), a workgroup whose whole span is of one segment one.
__device__ inline uint32_t wave_max(uint32_t v) {
    for (int o = 32; o > 0; o >>= 1) v = max(v, uint32_t(__shfl_xor(int(v), o, 64)));
    return v;
}
__device__ inline void raise_block(uint32_t* word, uint32_t v) {  // every thread
    __shared__ uint32_t s_max[kBlock / 64];
    v = wave_max(v);
    if ((threadIdx.x & 63u) == 0u) s_max[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x != 0u) return;
    for (int w = 1; w < kBlock / 64; w++) v = max(v, s_max[w]);
    atomicMax(word, v);
}
__device__ inline void raise_wave(uint32_t* words, uint32_t seg, uint32_t v, bool valid) {  // every lane
    if (!__ballot(valid)) return;
    const uint32_t w0 = __shfl(seg, 0, 64);  // lane 0 is valid when any lane is
    if (__ballot(valid && seg != w0) == 0ull) {
        v = wave_max(valid ? v : 0u);
        if (__lane_id() == 0) atomicMax(words + w0, v);
    } else if (valid) {
        atomicMax(words + seg, v);
    }
}
__device__ inline uint32_t tri_mag(float3 a, float3 b, float3 c) {
    const float3 v[3] = {a, b, c};
    float mag = 0.f;
    for (int k = 0; k < 3; k++) mag = fmaxf(mag, fmaxf(fabsf(v[k].x), fmaxf(fabsf(v[k].y), fabsf(v[k].z))));
    return isfinite(mag) ? __float_as_uint(mag) : 0u;
}
__device__ inline uint32_t find_tri_segment(const TriSegment* segs, uint32_t nseg, uint32_t r) {
    uint32_t a = 0, b = nseg;
    while (b - a > 1) {
        uint32_t m = (a + b) >> 1;
        if (segs[m].prim_start <= r) a = m; else b = m;
    }
    return a;
}

// Record r of the pool gets new positions for its primitive (v0.w, kept) of the
// segment whose records contain r; the other words are kept.  Raises the segment's
// largest coordinate magnitude (200k triangles: 467 us with an atomic per triangle,
// 13 us with one per span).
__global__ __launch_bounds__(kBlock) void k_refit_records(const TriSegment* segs, uint32_t nseg, uint32_t n,
                                                          uint32_t span, float4* tri, uint32_t* seg_mag,
                                                          uint32_t* bad) {
    const uint32_t base = blockIdx.x * span, end = base + min(span, n - base);
    const uint32_t s0 = find_tri_segment(segs, nseg, base);
    const bool one = s0 == find_tri_segment(segs, nseg, end - 1u);
    uint32_t most = 0;
    for (uint32_t row = base; row < end; row += kBlock) {
        const uint32_t r = row + threadIdx.x;
        const bool valid = r < end;
        uint32_t a = s0, mag = 0;
        if (valid) {
            if (!one) a = find_tri_segment(segs, nseg, r);
            const TriSegment& s = segs[a];
            float4* t = tri + 3 * size_t(r);
            const float4 t0 = t[0], t1 = t[1], t2 = t[2];
            const uint32_t prim = __float_as_uint(t0.w);
            float3 v[3];
            bool ok = prim < s.prim_count;
            for (int k = 0; k < 3; k++) {
                uint32_t idx = ok ? s.index_data[3 * size_t(prim) + k] : 0u;
                if (idx > s.max_vertex) { ok = false; idx = 0; }
                const float* f = (const float*)(s.vertex_data + size_t(s.first_vertex + idx) * s.stride);
                v[k] = mk3(f[0], f[1], f[2]);
            }
            if (!ok) {
                atomicOr(bad, 1u);
                v[1] = v[0];
                v[2] = v[0];
            }
            t[0] = make_float4(v[0].x, v[0].y, v[0].z, t0.w);
            t[1] = make_float4(v[1].x, v[1].y, v[1].z, t1.w);
            t[2] = make_float4(v[2].x, v[2].y, v[2].z, t2.w);
            mag = tri_mag(v[0], v[1], v[2]);
        }
        most = max(most, mag);
        if (!one) raise_wave(seg_mag, a, mag, valid);
    }
    if (one) raise_block(seg_mag + s0, most);
}

// Bottom-up over the levels of a forest: child boxes from the triangle records or boxes
// (leaves) or from the refit boxes of the deeper level (internal children), padded by the
// segment's padding as the build pads them, quantised; the node's own (unpadded) box is
// kept for its parent, and so is its segment, which a leaf child finds by its record.
// Root bounds (padded, 0 for an empty segment) go to descs, as the build reports them.
struct RefitArgs {
    QNode* nodes;
    uint32_t nseg;           // roots: nodes 0..nseg-1, root s is of segment s
    const TriSegment* segs;  // NULL: one segment
    const float4* tri;
    const float4* leaf_lo;   // boxes in place of triangles (tri NULL)
    const float4* leaf_hi;
    const uint32_t* seg_mag;
    uint32_t* node_seg;
    float* node_box;
    BlasDesc* descs;
};

__device__ inline void refit_node(const RefitArgs& a, uint32_t i) {
    const QNode q = a.nodes[i];
    uint32_t seg = i < a.nseg ? i : 0u;
    if (a.segs && i >= a.nseg) {
        // (below a root a node has a child)
        if (q.count[0]) seg = find_tri_segment(a.segs, a.nseg, q.child[0]);
        else if (q.child[0] != kEmpty) seg = a.node_seg[q.child[0]];
        a.node_seg[i] = seg;
    }
    // about 8 ulp of the segment's largest coordinate magnitude (as the build pads)
    const float pad = __uint_as_float(a.seg_mag[seg]) * 9.5367431640625e-07f + 1e-30f;
    WideNode w;
    float3 nl = mk3(INFINITY, INFINITY, INFINITY), nh = mk3(-INFINITY, -INFINITY, -INFINITY);
    for (int k = 0; k < 4; k++) {
        const uint32_t c = q.child[k], cnt = q.count[k];
        w.child[k] = c;
        w.count[k] = cnt;
        if (c == kEmpty) {
            w.lo_x[k] = w.lo_y[k] = w.lo_z[k] = 0.f;
            w.hi_x[k] = w.hi_y[k] = w.hi_z[k] = 0.f;
            continue;
        }
        float3 l = mk3(INFINITY, INFINITY, INFINITY), h = mk3(-INFINITY, -INFINITY, -INFINITY);
        if (cnt) {
            for (uint32_t r = c; r < c + cnt; r++) {
                if (!a.tri) {
                    l = fmin3(l, xyz(a.leaf_lo[r]));
                    h = fmax3(h, xyz(a.leaf_hi[r]));
                    continue;
                }
                const float4* t = a.tri + 3 * size_t(r);
                for (int v = 0; v < 3; v++) {
                    const float3 p = xyz(t[v]);
                    l = fmin3(l, p);
                    h = fmax3(h, p);
                }
            }
        } else {
            const float* b = a.node_box + 6 * size_t(c);
            l = mk3(b[0], b[1], b[2]);
            h = mk3(b[3], b[4], b[5]);
        }
        nl = fmin3(nl, l);
        nh = fmax3(nh, h);
        w.lo_x[k] = l.x - pad; w.lo_y[k] = l.y - pad; w.lo_z[k] = l.z - pad;
        w.hi_x[k] = h.x + pad; w.hi_y[k] = h.y + pad; w.hi_z[k] = h.z + pad;
    }
    float* b = a.node_box + 6 * size_t(i);
    b[0] = nl.x; b[1] = nl.y; b[2] = nl.z;
    b[3] = nh.x; b[4] = nh.y; b[5] = nh.z;
    a.nodes[i] = quantize_node(w);
    if (i < a.nseg) {
        const bool empty = !(nl.x <= nh.x);
        const float v[6] = {nl.x - pad, nl.y - pad, nl.z - pad, nh.x + pad, nh.y + pad, nh.z + pad};
        for (int k = 0; k < 6; k++) a.descs[i].bounds[k] = empty ? 0.f : v[k];
    }
}

__global__ __launch_bounds__(kBlock) void k_refit_level(RefitArgs a, uint32_t begin, uint32_t end) {
    const uint32_t i = begin + blockIdx.x * blockDim.x + threadIdx.x;
    if (i < end) refit_node(a, i);
}

// Consecutive levels of at most kRefitSmall nodes in one workgroup, with a barrier between
// them.  A level takes about 8 us either way (a chain of loads, then the quantising); what
// goes is its launch: 627 to 593 us an animation step of 1,300 triangles, no change for
// 200k, where the large levels set the pace.
constexpr uint32_t kRefitSmall = 1024;
constexpr int kRefitLevels = 16, kRefitThreads = 1024;
struct RefitLevels {
    uint32_t count;
    uint32_t start[kRefitLevels + 1];  // ascending: levels are taken from the last to the first
};
__global__ __launch_bounds__(kRefitThreads) void k_refit_levels(RefitArgs a, RefitLevels lv) {
    for (uint32_t L = lv.count; L-- > 0;) {
        for (uint32_t i = lv.start[L] + threadIdx.x; i < lv.start[L + 1]; i += kRefitThreads) refit_node(a, i);
        __syncthreads();
    }
}

// Flattened-BVH refit: record p takes its positions again from its BLAS record (v1.w
// names the instance, v2.w the record in that instance's BLAS pool); the w words are
// kept.  Raises the largest coordinate magnitude (one segment).
__global__ __launch_bounds__(kBlock) void k_refit_flat_records(const InstanceRecord* inst, uint32_t n, uint32_t span,
                                                               float4* tri, uint32_t* seg_mag) {
    const uint32_t base = blockIdx.x * span, end = base + min(span, n - base);
    uint32_t most = 0;
    for (uint32_t p = base + threadIdx.x; p < end; p += kBlock) {
        float4* t = tri + 3 * size_t(p);
        const float4 t0 = t[0], t1 = t[1], t2 = t[2];
        const uint32_t ii = __float_as_uint(t1.w) & ~kFlatOpaque, rec = __float_as_uint(t2.w);
        const float4* src = inst[ii].tris + 3 * size_t(rec);
        const float4 a = src[0], b = src[1], c = src[2];
        t[0] = make_float4(a.x, a.y, a.z, t0.w);
        t[1] = make_float4(b.x, b.y, b.z, t1.w);
        t[2] = make_float4(c.x, c.y, c.z, t2.w);
        most = max(most, tri_mag(xyz(a), xyz(b), xyz(c)));
    }
    raise_block(seg_mag, most);
}

// Largest finite coordinate magnitude of a set of leaf boxes (one segment).
__global__ __launch_bounds__(kBlock) void k_box_mag(const float4* lo, const float4* hi, uint32_t n, uint32_t span,
                                                    uint32_t* seg_mag) {
    const uint32_t base = blockIdx.x * span, end = base + min(span, n - base);
    float m = 0.f;
    for (uint32_t i = base + threadIdx.x; i < end; i += kBlock) {
        const float v[6] = {lo[i].x, lo[i].y, lo[i].z, hi[i].x, hi[i].y, hi[i].z};
        for (int k = 0; k < 6; k++)
            if (isfinite(v[k])) m = fmaxf(m, fabsf(v[k]));
    }
    raise_block(seg_mag, __float_as_uint(m));
}

}  // namespace

// ------------------------------------------------------------------ host
int prepare_triangles(hipStream_t st, const TriSegment* d_segs, uint32_t nseg, uint32_t n, float4* d_tri, float4* d_lo,
                      float4* d_hi, uint32_t* d_bad) {
    if (n == 0) return 0;
    hipLaunchKernelGGL(k_prepare_triangles, dim3(blocks_for(n, kBlock)), dim3(kBlock), 0, st, d_segs, nseg, n, d_tri,
                       d_lo, d_hi, d_bad);
    RT_CHECK_LAUNCH();
    return 0;
}

int reorder_triangles(hipStream_t st, const float4* in, const uint32_t* perm, uint32_t n, float4* out) {
    if (n == 0) return 0;
    hipLaunchKernelGGL(k_reorder_tris, dim3(blocks_for(n, kBlock)), dim3(kBlock), 0, st, in, perm, n, out);
    RT_CHECK_LAUNCH();
    return 0;
}

int gather_flat(hipStream_t st, const FlatSource* src, uint32_t nsrc, uint32_t n, float4* tri, float4* lo, float4* hi) {
    if (n == 0) return 0;
    hipLaunchKernelGGL(k_gather_flat, dim3(blocks_for(n, kBlock)), dim3(kBlock), 0, st, src, nsrc, n, tri, lo, hi);
    RT_CHECK_LAUNCH();
    return 0;
}

int prepare_instances(hipStream_t st, const InstanceRecord* inst, uint32_t n, float4* lo, float4* hi) {
    if (n == 0) return 0;
    hipLaunchKernelGGL(k_prepare_instances, dim3(blocks_for(n, kBlock)), dim3(kBlock), 0, st, inst, n, lo, hi);
    RT_CHECK_LAUNCH();
    return 0;
}

int reorder_instances(hipStream_t st, const InstanceRecord* in, const uint32_t* perm, uint32_t n, InstanceRecord* out) {
    if (n == 0) return 0;
    hipLaunchKernelGGL(k_reorder_instances, dim3(blocks_for(n, kBlock)), dim3(kBlock), 0, st, in, perm, n, out);
    RT_CHECK_LAUNCH();
    return 0;
}

// ------------------------------------------------------------ scratch
ScratchPool::~ScratchPool() {
    for (void* p : extra) (void)hipFree(p);
    if (base) (void)hipFree(base);
}

void ScratchPool::begin(size_t bytes) {
    used = 0;
    if (bytes <= cap) return;
    if (base) (void)hipFree(base);
    base = nullptr;
    cap = 0;
    void* p = nullptr;
    if (hipMalloc(&p, bytes) == hipSuccess) {
        base = (char*)p;
        cap = bytes;
    } else {
        (void)hipGetLastError();  // every buffer is tried by itself then
    }
}

void* ScratchPool::alloc_bytes(size_t bytes) {
    bytes = (bytes + 16 + 255) & ~size_t(255);
    if (used + bytes <= cap) {
        void* p = base + used;
        used += bytes;
        return p;
    }
    void* p = nullptr;
    if (hipMalloc(&p, bytes) != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
    }
    extra.push_back(p);
    return p;
}

void ScratchPool::end() {
    used = 0;
    for (void* p : extra) (void)hipFree(p);
    extra.clear();
    if (cap > kScratchKeep) {
        (void)hipFree(base);
        base = nullptr;
        cap = 0;
    }
}

size_t lbvh_scratch_bytes(uint32_t n, uint32_t nseg) {
    const size_t hist = 256 * size_t(blocks_for(n, kRsTile));
    const size_t nodes = size_t(n) + nseg;
    const size_t roots = (size_t(blocks_for(n, kTile)) * 5 / 4 + 2) * (kTileRoots + 1) * 4;
    return size_t(n) * (16 + 8 + 24 + 4 + 4 + 32 + 4 + 16 + 4 + 4) + roots + nodes * (64 + 16 * 3 + 4) +
           hist * 4 + hist / 128 + size_t(nseg) * 96 + (1u << 16);
}

int lbvh_build(hipStream_t st, const float4* d_lo, const float4* d_hi, uint32_t n, const uint32_t* d_seg_start,
               const std::vector<uint32_t>& h_seg_start, uint32_t leaf_max, uint32_t collapse, uint32_t treelet_passes,
               ScratchPool& s, LbvhResult* out, std::string* err) {
    const uint32_t nseg = uint32_t(h_seg_start.size()) - 1;
    if (leaf_max < 1 || leaf_max > uint32_t(kMaxLeafPrims)) { *err = "leaf size out of range"; return int(hipErrorInvalidValue); }
    if (n >= (1u << kLeafCountShift)) { *err = "too many primitives in one build"; return int(hipErrorInvalidValue); }
    int segbits = 0;
    while ((1u << segbits) < nseg) segbits++;
    int bits = (64 - segbits) / 3;
    if (bits > 21) bits = 21;
    const int key_bits = 3 * bits + segbits;
    const uint32_t max_nodes = n + nseg;
    uint32_t* bounds = s.alloc<uint32_t>(12 * size_t(nseg));
    float* pad = s.alloc<float>(nseg);
    uint32_t* seg_root = s.alloc<uint32_t>(nseg);
    float* seg_bounds = s.alloc<float>(6 * size_t(nseg));
    QNode* nodes_tmp = s.alloc<QNode>(max_nodes);
    constexpr uint32_t kMaxLevels = 256;
    uint2* levels = s.alloc<uint2>(kMaxLevels + 1);
    uint32_t* words = s.alloc<uint32_t>(kCollapseBlocks + 1);  // workgroup sums, overflow flag
    uint4* ta = s.alloc<uint4>(max_nodes);
    uint4* tb = s.alloc<uint4>(max_nodes);
    uint4* refs = s.alloc<uint4>(max_nodes);
    uint32_t* offs = s.alloc<uint32_t>(max_nodes);
    uint64_t* k0 = s.alloc<uint64_t>(n);
    uint64_t* k1 = s.alloc<uint64_t>(n);
    uint32_t* v0 = s.alloc<uint32_t>(n);
    uint32_t* v1 = s.alloc<uint32_t>(n);
    uint32_t* left = s.alloc<uint32_t>(n);
    uint32_t* right = s.alloc<uint32_t>(n);
    uint32_t* first = s.alloc<uint32_t>(n);
    uint32_t* last = s.alloc<uint32_t>(n);
    uint32_t* parent_int = s.alloc<uint32_t>(n);
    uint32_t* parent_leaf = s.alloc<uint32_t>(n);
    uint32_t* is_root = s.alloc<uint32_t>(n);
    uint32_t* split = s.alloc<uint32_t>(n);
    float4* nlo = s.alloc<float4>(n);
    float4* nhi = s.alloc<float4>(n);
    uint32_t* cnt = s.alloc<uint32_t>(n);
    float4* cost = s.alloc<float4>(n);
    uint32_t* dec = s.alloc<uint32_t>(n);
    // the subtrees left by the tiles of a level, ping-pong; sized for the smaller fan, which
    // has more tiles in every level
    const size_t tiles0 = blocks_for(n, kTile), tiles1 = (tiles0 + kFanSafe - 1) / kFanSafe;
    uint32_t* roots0 = s.alloc<uint32_t>(tiles0 * kTileRoots);
    uint32_t* counts0 = s.alloc<uint32_t>(tiles0);
    uint32_t* roots1 = s.alloc<uint32_t>(tiles1 * kTileRoots);
    uint32_t* counts1 = s.alloc<uint32_t>(tiles1);
    for (const void* p : {(const void*)bounds, (const void*)pad, (const void*)seg_root, (const void*)seg_bounds,
                          (const void*)nodes_tmp, (const void*)levels, (const void*)words, (const void*)ta, (const void*)tb,
                          (const void*)refs, (const void*)offs, (const void*)k0, (const void*)k1, (const void*)v0,
                          (const void*)v1, (const void*)left, (const void*)right, (const void*)first, (const void*)last,
                          (const void*)parent_int, (const void*)parent_leaf, (const void*)is_root, (const void*)split,
                          (const void*)nlo, (const void*)nhi, (const void*)cnt, (const void*)cost,
                          (const void*)dec, (const void*)roots0, (const void*)counts0, (const void*)roots1,
                          (const void*)counts1})
        if (!p) { *err = "out of device memory"; return int(hipErrorOutOfMemory); }
    uint32_t* const overflow = words + kCollapseBlocks;
    auto fail = [&](int rc, const char* what) {
        *err = what;
        return rc;
    };
    // launch errors are sticky until read: one check after each group of launches
    auto launched = [&](const char* what) -> int {
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) *err = what;
        return int(e);
    };
    int rc;
    hipLaunchKernelGGL(k_init_bounds, dim3(blocks_for(12 * size_t(nseg), kBlock)), dim3(kBlock), 0, st, bounds, nseg);
    if (n > 0)
        hipLaunchKernelGGL(k_seg_bounds, dim3(blocks_for(n, bounds_span(n))), dim3(kBlock), 0, st, d_lo, d_hi,
                           n, d_seg_start, nseg, bounds_span(n), bounds);
    hipLaunchKernelGGL(k_seg_pad, dim3(blocks_for(nseg, kBlock)), dim3(kBlock), 0, st, bounds, d_seg_start, nseg, pad,
                       seg_bounds, seg_root, overflow);
    if ((rc = launched("launch of the segment bounds"))) return rc;

    const uint32_t* perm = v0;
    const bool sah = collapse == kCollapseSah;
    if (n > 0) {
        hipLaunchKernelGGL(k_morton, dim3(blocks_for(n, kBlock)), dim3(kBlock), 0, st, d_lo, d_hi, n, d_seg_start, nseg,
                           bounds, bits, k0, v0);
        if (n <= kRankMax) {
            hipLaunchKernelGGL(k_rank_sort, dim3(blocks_for(n, kRankKeys)), dim3(kRankKeys * kRankSlices), 0, st, k0, v0,
                               n, k1, v1);
            std::swap(k0, k1);
            std::swap(v0, v1);
            if ((rc = launched("launch k_rank_sort"))) return rc;
        } else {
            const uint32_t nblk = blocks_for(n, kRsTile);
            const uint32_t m = 256u * nblk;
            uint32_t* hist = s.alloc<uint32_t>(m);
            const uint32_t scan_cap = 2 * blocks_for(m, kScanPerBlock) + 64;
            uint32_t* scan_tmp = s.alloc<uint32_t>(scan_cap);
            if (!hist || !scan_tmp) return fail(int(hipErrorOutOfMemory), "out of device memory");
            for (int shift = 0; shift < key_bits; shift += 8) {
                hipLaunchKernelGGL(k_rs_hist, dim3(nblk), dim3(kBlock), 0, st, k0, n, shift, hist, nblk);
                rc = exclusive_scan(st, hist, m, scan_tmp, scan_cap);
                if (rc) return fail(rc, "scan");
                hipLaunchKernelGGL(k_rs_scatter, dim3(nblk), dim3(kBlock), 0, st, k0, v0, k1, v1, n, shift, hist, nblk);
                std::swap(k0, k1);
                std::swap(v0, v1);
            }
            if ((rc = launched("launch of the radix sort"))) return rc;
        }
        // v0: sorted position -> primitive, k0: sorted keys
    }
    const uint32_t* const sorted = v0;
    uint32_t fan = kFan, level = 0, num_nodes = 0, h_over = 0;
    std::vector<uint2> h_levels(kMaxLevels + 1);
    for (;; fan = kFanSafe) {
        if (n > 0) {
            hipLaunchKernelGGL(k_karras, dim3(blocks_for(n, kBlock)), dim3(kBlock), 0, st, k0, int(n), left, right, first,
                               last, parent_int, parent_leaf, d_seg_start, nseg, 3 * bits, seg_root, is_root, split);
            perm = sorted;
            const TreeArgs tr{d_lo,  d_hi,       sorted,      k0,  3 * bits, d_seg_start, first, last, split,    left, right,
                              parent_int, parent_leaf, nlo, nhi, cnt,      cost,        dec,   overflow, n, treelet_passes,
                              leaf_max, sah ? 1u : 0u};
            uint32_t tiles = blocks_for(n, kTile);
            uint32_t *ri = roots0, *ci = counts0, *ro = roots1, *co = counts1;
            hipLaunchKernelGGL((k_tree_level<kTile, kTile, true>), dim3(tiles), dim3(kTile), 0, st, tr, uint32_t(kTile), fan,
                               (const uint32_t*)nullptr, (const uint32_t*)nullptr, 0u, tiles > 1 ? ri : nullptr, ci);
            for (uint64_t size = uint64_t(kTile) * fan; tiles > 1; size *= fan) {
                const uint32_t tiles_in = tiles;
                tiles = (tiles + fan - 1) / fan;
                hipLaunchKernelGGL((k_tree_level<kTileRefs, kTileThreads, false>), dim3(tiles), dim3(kTileThreads), 0, st, tr,
                                   uint32_t(std::min<uint64_t>(size, 1ull << 31)), fan, ri, ci, tiles_in,
                                   tiles > 1 ? ro : nullptr, co);
                std::swap(ri, ro);
                std::swap(ci, co);
            }
            if ((rc = launched("launch of the tree passes"))) return rc;
            if (treelet_passes > 0 && n > 2) {
                // newpos in offs, which the collapse writes only afterwards
                hipLaunchKernelGGL(k_renumber_nodes, dim3(blocks_for(n - 1, kBlock)), dim3(kBlock), 0, st, left, right,
                                   parent_int, is_root, cnt, first, last, int(n) - 1, overflow);
                hipLaunchKernelGGL(k_renumber_leaves, dim3(blocks_for(n, kBlock)), dim3(kBlock), 0, st, left, parent_leaf,
                                   first, cnt, d_seg_start, nseg, offs, n, overflow);
                hipLaunchKernelGGL(k_renumber_apply, dim3(blocks_for(n, kBlock)), dim3(kBlock), 0, st, offs, sorted, v1, left,
                                   right, n, overflow);
                perm = v1;
                if ((rc = launched("launch of the renumbering"))) return rc;
            }
        }

        // collapse: level by level until a level has no tasks.  The number of levels is known
        // on the device only: about 1.25 log4 of the largest segment; more are enqueued when
        // the levels read back show that the tree goes deeper.
        CollapseArgs a{d_lo, d_hi, perm, nlo, nhi, left, right, first, last, d_seg_start, nseg, pad, leaf_max,
                       nodes_tmp, max_nodes, overflow, sah ? dec : nullptr, levels, words};
        hipLaunchKernelGGL(k_init_tasks, dim3(blocks_for(nseg, kBlock)), dim3(kBlock), 0, st, seg_root, nseg, ta, levels);
        uint32_t largest = 1;
        for (uint32_t k = 0; k < nseg; k++) largest = std::max(largest, h_seg_start[k + 1] - h_seg_start[k]);
        uint32_t want = 1;
        level = 0;
        for (uint64_t c = 1; c < largest; c *= 4) want++;
        want += want / 4;
        for (bool done = false; !done; want += 4) {
            for (; level < want && level < kMaxLevels; level++) {
                const uint64_t bound = std::min<uint64_t>(uint64_t(nseg) << std::min(2u * level, 32u), max_nodes);
                const dim3 grid(std::min(blocks_for(bound, kBlock), kCollapseBlocks));
                hipLaunchKernelGGL(k_collapse_gather, grid, dim3(kBlock), 0, st, a, level, ta, refs, offs);
                hipLaunchKernelGGL(k_collapse_emit, grid, dim3(kBlock), 0, st, a, level, ta, refs, offs, tb);
                std::swap(ta, tb);
            }
            if ((rc = launched("launch of the collapse"))) return rc;
            if (hipMemcpyAsync(h_levels.data(), levels, sizeof(uint2) * (level + 1), hipMemcpyDeviceToHost, st) != hipSuccess ||
                hipMemcpyAsync(&h_over, overflow, sizeof(h_over), hipMemcpyDeviceToHost, st) != hipSuccess ||
                hipStreamSynchronize(st) != hipSuccess)
                return fail(int(hipErrorUnknown), "read level sizes");
            if (h_over == kOverflowFan && fan != kFanSafe) break;
            if (h_over) return fail(int(hipErrorUnknown), "node capacity exceeded during collapse");
            done = h_levels[level].x == 0u;
            if (!done && level >= kMaxLevels) return fail(int(hipErrorUnknown), "collapse did not terminate");
        }
        if (!h_over) break;
        // a tile held too many subtrees: once more with tiles that cannot
        if (hipMemsetAsync(overflow, 0, sizeof(uint32_t), st) != hipSuccess) return fail(int(hipErrorUnknown), "memset");
    }
    out->level_start.assign({0u, nseg});
    num_nodes = nseg;
    for (uint32_t k = 1; k <= level && h_levels[k].x != 0u; k++) {
        num_nodes = h_levels[k].y;
        out->level_start.push_back(num_nodes);
    }
    if (num_nodes > max_nodes) return fail(int(hipErrorUnknown), "node capacity exceeded during collapse");
    QNode* nodes = nullptr;
    if (hipMalloc(&nodes, sizeof(QNode) * size_t(num_nodes)) != hipSuccess) return fail(int(hipErrorOutOfMemory), "out of device memory");
    if (hipMemcpyAsync(nodes, nodes_tmp, sizeof(QNode) * size_t(num_nodes), hipMemcpyDeviceToDevice, st) != hipSuccess) {
        (void)hipFree(nodes);
        return fail(int(hipErrorUnknown), "copy nodes");
    }
    out->nodes = nodes;
    out->num_nodes = num_nodes;
    out->perm = perm;
    out->seg_bounds = seg_bounds;
    return 0;
}

namespace {
bool levels_match(const std::vector<uint32_t>& level_start, uint32_t nseg, uint32_t num_nodes) {
    return level_start.size() >= 2 && level_start.front() == 0u && level_start[1] == nseg && level_start.back() == num_nodes;
}

// Refits every level, the deepest first; a.node_seg and a.node_box come from s.
int refit_levels(hipStream_t st, ScratchPool& s, RefitArgs a, uint32_t num_nodes, const std::vector<uint32_t>& level_start,
                 std::string* err) {
    a.node_seg = s.alloc<uint32_t>(num_nodes);
    a.node_box = s.alloc<float>(6 * size_t(num_nodes));
    if (!a.node_seg || !a.node_box) {
        *err = "out of device memory";
        return int(hipErrorOutOfMemory);
    }
    for (size_t L = level_start.size() - 1; L > 0;) {
        const uint32_t c = level_start[L];
        size_t top = L;  // levels top..L-1 are small
        while (top > 0 && L - top < size_t(kRefitLevels) && level_start[top] - level_start[top - 1] <= kRefitSmall) top--;
        if (top < L) {
            RefitLevels lv;
            lv.count = uint32_t(L - top);
            for (uint32_t k = 0; k <= lv.count; k++) lv.start[k] = level_start[top + k];
            hipLaunchKernelGGL(k_refit_levels, dim3(1), dim3(kRefitThreads), 0, st, a, lv);
            L = top;
        } else {
            const uint32_t b = level_start[--L];
            hipLaunchKernelGGL(k_refit_level, dim3(blocks_for(c - b, kBlock)), dim3(kBlock), 0, st, a, b, c);
        }
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) *err = "refit launch";
    return int(e);
}

// Refit of a one-segment tree (root node 0); seg_mag[0] is raised beforehand on the same
// stream.  Writes the padded root box to bounds.
int refit_tree(hipStream_t st, ScratchPool& s, RefitArgs a, uint32_t num_nodes, const std::vector<uint32_t>& level_start,
               float bounds[6], std::string* err) {
    a.nseg = 1u;
    a.descs = s.alloc<BlasDesc>(1);
    if (!a.descs) {
        *err = "out of device memory";
        return int(hipErrorOutOfMemory);
    }
    const int rc = refit_levels(st, s, a, num_nodes, level_start, err);
    if (rc) return rc;
    hipError_t e = hipMemcpyAsync(bounds, a.descs->bounds, sizeof(float) * 6, hipMemcpyDeviceToHost, st);
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    if (e != hipSuccess) *err = "refit launch";
    return int(e);
}
}  // namespace

size_t refit_scratch_bytes(uint32_t num_nodes, uint32_t nseg, uint32_t boxes) {
    return size_t(num_nodes) * 28 + size_t(nseg) * 4 + size_t(boxes) * 32 + 8192;
}

int lbvh_refit(hipStream_t st, const TriSegment* d_segs, uint32_t nseg, uint32_t n, float4* d_tri, QNode* d_nodes,
               uint32_t num_nodes, const std::vector<uint32_t>& level_start, BlasDesc* d_descs, uint32_t* d_bad,
               ScratchPool& s, std::string* err) {
    if (!levels_match(level_start, nseg, num_nodes)) {
        *err = "the pool's level table does not match its nodes";
        return int(hipErrorInvalidValue);
    }
    uint32_t* seg_mag = s.alloc<uint32_t>(nseg);
    if (!seg_mag) {
        *err = "out of device memory";
        return int(hipErrorOutOfMemory);
    }
    hipError_t e = hipMemsetAsync(seg_mag, 0, sizeof(uint32_t) * nseg, st);
    if (e != hipSuccess) {
        *err = "memset";
        return int(e);
    }
    if (n) hipLaunchKernelGGL(k_refit_records, dim3(blocks_for(n, bounds_span(n))), dim3(kBlock), 0, st, d_segs, nseg, n,
                              bounds_span(n), d_tri, seg_mag, d_bad);
    RefitArgs a = {};
    a.nodes = d_nodes;
    a.nseg = nseg;
    a.segs = d_segs;
    a.tri = d_tri;
    a.seg_mag = seg_mag;
    a.descs = d_descs;
    return refit_levels(st, s, a, num_nodes, level_start, err);
}

int lbvh_refit_flat(hipStream_t st, const InstanceRecord* d_inst, uint32_t n, float4* d_tri, QNode* d_nodes,
                    uint32_t num_nodes, const std::vector<uint32_t>& level_start, float bounds[6], ScratchPool& s,
                    std::string* err) {
    if (!levels_match(level_start, 1u, num_nodes)) {
        *err = "the tree's level table does not match its nodes";
        return int(hipErrorInvalidValue);
    }
    uint32_t* seg_mag = s.alloc<uint32_t>(1);
    if (!seg_mag) {
        *err = "out of device memory";
        return int(hipErrorOutOfMemory);
    }
    hipError_t e = hipMemsetAsync(seg_mag, 0, sizeof(uint32_t), st);
    if (e != hipSuccess) {
        *err = "memset";
        return int(e);
    }
    if (n) hipLaunchKernelGGL(k_refit_flat_records, dim3(blocks_for(n, bounds_span(n))), dim3(kBlock), 0, st, d_inst, n,
                              bounds_span(n), d_tri, seg_mag);
    RefitArgs a = {};
    a.nodes = d_nodes;
    a.tri = d_tri;
    a.seg_mag = seg_mag;
    return refit_tree(st, s, a, num_nodes, level_start, bounds, err);
}

int lbvh_refit_instances(hipStream_t st, const InstanceRecord* d_inst, uint32_t n, QNode* d_nodes, uint32_t num_nodes,
                         const std::vector<uint32_t>& level_start, float bounds[6], ScratchPool& s, std::string* err) {
    if (!levels_match(level_start, 1u, num_nodes)) {
        *err = "the tree's level table does not match its nodes";
        return int(hipErrorInvalidValue);
    }
    uint32_t* seg_mag = s.alloc<uint32_t>(1);
    float4* lo = s.alloc<float4>(n + 1);
    float4* hi = s.alloc<float4>(n + 1);
    if (!seg_mag || !lo || !hi) {
        *err = "out of device memory";
        return int(hipErrorOutOfMemory);
    }
    hipError_t e = hipMemsetAsync(seg_mag, 0, sizeof(uint32_t), st);
    if (e != hipSuccess) {
        *err = "memset";
        return int(e);
    }
    int rc = prepare_instances(st, d_inst, n, lo, hi);
    if (rc) {
        *err = "instance boxes";
        return rc;
    }
    if (n) hipLaunchKernelGGL(k_box_mag, dim3(blocks_for(n, bounds_span(n))), dim3(kBlock), 0, st, lo, hi, n, bounds_span(n),
                              seg_mag);
    RefitArgs a = {};
    a.nodes = d_nodes;
    a.leaf_lo = lo;
    a.leaf_hi = hi;
    a.seg_mag = seg_mag;
    return refit_tree(st, s, a, num_nodes, level_start, bounds, err);
}

}  // namespace rt
