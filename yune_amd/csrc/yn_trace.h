// yn_trace.h — traversal of one ray per lane, shared by the trace kernels
// (trace.hip) and the kernels that run whole paths (paths.hip).
//
// Template parameter ANY: 0 closest hit, 1 any hit, 2 either, by the lane's
// own RayState::any.
#pragma once

#include "yn_device.h"
#include "yn_exact.h"
#include "yn_internal.h"
#include "yn_slab.h"

namespace yune {

struct RayState {
    float ox, oy, oz, dx, dy, dz, ix, iy, iz;
    float lx, ly, lz;       // FMA slab form: o * dir_inv moved by 2^-21 |o * dir_inv|,
    float hx, hy, hz;       //   one way for the box's lo planes, the other for its hi planes
    float best;             // current tmax
    float cull;             // nodes entered beyond it are skipped: best * (1 + 1e-4) * kWiden
    int tri;                // best hit: triangle id (-1: none), u, v
    float u, v;
    bool any;               // ANY 2: this ray is done at its first hit
};

// Whether a ray that has found something (got) needs no more tests.
template <int ANY>
__device__ __forceinline__ bool ends(const RayState& r, bool got)
{
    return ANY == 0 ? false : ANY == 1 ? got : got && r.any;
}

// A child box of an interior node: the reference's slab arithmetic (EXACT)
// or the widened FMA form.
template <bool EXACT>
__device__ __forceinline__ bool child_hit(float lox, float loy, float loz, float hix, float hiy, float hiz,
                                          const RayState& r, float& enter)
{
    return EXACT ? box_hit(lox, loy, loz, hix, hiy, hiz, r.ox, r.oy, r.oz, r.ix, r.iy, r.iz, enter)
                 : box_hit_fma(lox, loy, loz, hix, hiy, hiz, r.ix, r.iy, r.iz, r.lx, r.ly, r.lz, r.hx, r.hy, r.hz,
                               enter);
}

// A ray's traversal state from its queue entry.  Returns whether the FMA
// slab form may be used (see box_hit_fma).
__device__ __forceinline__ bool start_ray(RayState& r, const float4& ot, const float4& dp, const DevScene& S)
{
    r.ox = ot.x; r.oy = ot.y; r.oz = ot.z;
    r.dx = dp.x; r.dy = dp.y; r.dz = dp.z;
    r.ix = x_rcp(r.dx); r.iy = x_rcp(r.dy); r.iz = x_rcp(r.dz);   // dir_inv (udpt.cl:395)
    fma_offsets(r.ox, r.ix, r.lx, r.hx);
    fma_offsets(r.oy, r.iy, r.ly, r.hy);
    fma_offsets(r.oz, r.iz, r.lz, r.hz);
    r.best = ot.w;
    r.cull = cull_of(ot.w);
    r.tri = -1; r.u = 0.0f; r.v = 0.0f;
    return S.fma_slab && fma_form_ok(r.ox, r.oy, r.oz, r.ix, r.iy, r.iz);
}

// A load from a scene array as a global-memory load.  Through a generic
// pointer (the scene table holds them) the compiler emits FLAT loads, which
// also count against the LDS wait counter: every access to the LDS stack
// would then wait for the node fetches still in flight.
// (Through a native vector type: a cast of float4* itself still copies
// through a generic reference.)
typedef float yn_v4f __attribute__((ext_vector_type(4)));
typedef int yn_v4i __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float4 gload(const float4* p)
{
    yn_v4f v = *(const __attribute__((address_space(1))) yn_v4f*)(const void*)p;
    return make_float4(v.x, v.y, v.z, v.w);
}

__device__ __forceinline__ int4 gload(const int4* p)
{
    yn_v4i v = *(const __attribute__((address_space(1))) yn_v4i*)(const void*)p;
    return make_int4(v.x, v.y, v.z, v.w);
}

// The same address in every lane, as one the scalar unit loads from.
typedef const __attribute__((address_space(4))) yn_v4f yn_cv4f;
__device__ __forceinline__ yn_cv4f* scalar_ptr(const float4* p)
{
    const uint64_t u = (uint64_t)p;
    const uint64_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)u);
    const uint64_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(u >> 32));
    return (yn_cv4f*)(hi << 32 | lo);
}

// rayTriangleIntersection (udpt.cl:326-390) on a stored slot {A, B, C}; xyz
// only (the w terms of the reference's dots are exact zeros).  Returns whether
// (u, v) lies in the triangle, with t.
template <typename V>
__device__ __forceinline__ bool tri_uvt(const V& A, const V& B, const V& C, const RayState& r, float& t, float& u,
                                        float& v)
{
    // pvec = cross(dir, v1v3)
    float px = r.dy * C.z - r.dz * C.y;
    float py = r.dz * C.x - r.dx * C.z;
    float pz = r.dx * C.y - r.dy * C.x;
    float det = B.x * px + B.y * py + B.z * pz;
    float inv_det = x_rcp(det);
    float sx = r.ox - A.x, sy = r.oy - A.y, sz = r.oz - A.z;
    u = (px * sx + py * sy + pz * sz) * inv_det;
    if (u < 0.0f || u > 1.0f) return false;
    // qvec = cross(dist, v1v2)
    float qx = sy * B.z - sz * B.y;
    float qy = sz * B.x - sx * B.z;
    float qz = sx * B.y - sy * B.x;
    v = (qx * r.dx + qy * r.dy + qz * r.dz) * inv_det;
    if (v < 0.0f || u + v > 1.0f) return false;
    t = (C.x * qx + C.y * qy + C.z * qz) * inv_det;
    return true;
}

template <int ANY, typename V>
__device__ __forceinline__ bool tri_test(const V& A, const V& B, const V& C, RayState& r)
{
    float t, u, v;
    if (tri_uvt(A, B, C, r, t, u, v) && t > 0.0f && t < r.best) {
        if (ANY != 1) {         // an any-hit ray ends here, and only whether it hit counts
            r.best = t;
            r.cull = cull_of(t);
            r.tri = __float_as_int(A.w);
            r.u = u;
            r.v = v;
        }
        return true;
    }
    return false;
}

template <int ANY>
__device__ __forceinline__ bool tri_test(const float4* __restrict__ tri, int s, RayState& r)
{
    return tri_test<ANY>(gload(tri + 3 * s), gload(tri + 3 * s + 1), gload(tri + 3 * s + 2), r);
}

// The result record {t, triangle id bits, u, v} of a finished closest-hit
// traversal.
__device__ __forceinline__ float4 hit_record(const RayState& r)
{
    return make_float4(r.best, __int_as_float(r.tri), r.u, r.v);
}

struct Counts { unsigned nodes, tris; };

template <int ANY, bool COUNT>
__device__ __forceinline__ bool leaf_test(const float4* __restrict__ tri, uint32_t ref, RayState& r, Counts& c)
{
    int s = (int)((ref >> 4) & 0x7FFFFFFu);
    int left = (int)(ref & 15u);
    bool got = false;
    do {                    // a leaf holds at least one triangle (kEmptyRef is never entered)
        if (COUNT) c.tris++;
        got |= tri_test<ANY>(tri, s, r);
        if (ends<ANY>(r, got)) return true;
        ++s;
    } while (--left > 0);
    return got;
}

// The stack's two parts in explicit address spaces: through plain (generic)
// pointers the compiler merges a pop's LDS and global branches into one
// FLAT load, which goes through the vector-memory pipeline the node fetches
// already saturate (and waits on both counters).
typedef __attribute__((address_space(3))) uint32_t lds_u32;
typedef __attribute__((address_space(3))) uint16_t lds_u16;
typedef __attribute__((address_space(1))) uint32_t gbl_u32;
typedef __attribute__((address_space(1))) uint16_t gbl_u16;

// Per-lane traversal stack: LDS for the top LST entries, global beyond.
template <int LST, int BLOCK>
struct Stack {
    lds_u32* lref;          // LDS, the block's arrays: entry e of column c at e * BLOCK + c
    lds_u16* lt;
    uint32_t col;           // this lane's column (one register for both arrays)
    gbl_u32* gref;          // global overflow area: entry k of grid thread g at
    gbl_u16* gt;            //   k * gstride + g, g = gbase + column()
    uint32_t gbase;         // the block's first grid thread
    uint32_t gstride;       // threads in the grid
    int gcap;               // overflow entries available
    uint32_t* full;         // set to 1 by a traversal that would overflow the stack (it ends there)
    int sp;

    // the column, opaque to the compiler at each use: otherwise it keeps
    // one precomputed address per array live through the whole loop, and
    // at the kernel's register bound one of them spills
    __device__ __forceinline__ uint32_t column() const
    {
        uint32_t c = col;
        __asm__ volatile("" : "+v"(c));
        return c;
    }

    __device__ __forceinline__ void put(uint32_t ref, float t)
    {
        const uint32_t i = sp * BLOCK + column();
        lref[i] = ref;
        lt[i] = (uint16_t)(__float_as_uint(t) >> 16);   // truncation: a lower bound of t >= 0
    }

    // An entry anywhere.  One that the overflow area has no room for is left
    // out and raises the flag: the caller's results are then refused.
    __device__ __forceinline__ void push(uint32_t ref, float t)
    {
        if (sp < LST) {
            put(ref, t);
        } else {
            int k = sp - LST;
            if (k >= gcap) { *full = 1u; return; }      // cannot happen: depth bound
            const size_t i = (size_t)k * gstride + gbase + column();
            gref[i] = ref;
            gt[i] = (uint16_t)(__float_as_uint(t) >> 16);
        }
        ++sp;
    }

    // The farther children of a node, k1 <= k2 <= k3 with +inf where there is
    // none, the nearest on top.  While every lane of the wave has room for
    // three in LDS, each is written whether there or not and the next goes
    // over it, without a branch for each.
    __device__ __forceinline__ void push3(float k1, uint32_t c1, float k2, uint32_t c2, float k3, uint32_t c3)
    {
        if (__builtin_expect(__ballot(sp > LST - 3) == 0, 1)) {
            put(c3, k3);
            sp += k3 != INFINITY ? 1 : 0;
            put(c2, k2);
            sp += k2 != INFINITY ? 1 : 0;
            put(c1, k1);
            sp += k1 != INFINITY ? 1 : 0;
        } else {
            if (k3 != INFINITY) push(c3, k3);
            if (k2 != INFINITY) push(c2, k2);
            if (k1 != INFINITY) push(c1, k1);
        }
    }

    __device__ __forceinline__ uint32_t pop(float& t)
    {
        --sp;
        uint32_t ref;
        uint16_t tb;
        if (__builtin_expect(__ballot(sp >= LST) == 0, 1) || sp < LST) {
            const uint32_t i = sp * BLOCK + column();
            ref = lref[i];
            tb = lt[i];
        } else {
            const size_t i = (size_t)(sp - LST) * gstride + gbase + column();
            ref = gref[i];
            tb = gt[i];
        }
        t = __uint_as_float((uint32_t)tb << 16);
        return ref;
    }
};

// Traverse one ray; returns true if a hit was found.
template <int W, int ANY, int LST, int BLOCK, bool COUNT, bool EXACT>
__device__ bool traverse(const DevScene& S, RayState& r, Stack<LST, BLOCK>& st, Counts& c)
{
    const float4* __restrict__ nodes = S.nodes;
    const float4* __restrict__ tri = S.tri_isect;
    bool got = false;
    if (S.brute) {
        for (int s = 0; s < S.n_slots; ++s) {
            if (COUNT) c.tris++;
            got |= tri_test<ANY>(tri, s, r);
            if (ends<ANY>(r, got)) return true;
        }
        return got;
    }
    // oversized triangles hoisted out of the tree, each behind its own box
    for (int s = 0; s < S.n_hoist; ++s) {
        float4 lo = gload(S.hoist_box + 2 * s), hi = gload(S.hoist_box + 2 * s + 1);
        float e;
        if (!box_hit(lo.x, lo.y, lo.z, hi.x, hi.y, hi.z, r.ox, r.oy, r.oz, r.ix, r.iy, r.iz, e) || e > r.cull)
            continue;
        if (COUNT) c.tris++;
        got |= tri_test<ANY>(tri, s, r);
        if (ends<ANY>(r, got)) return true;
    }
    uint32_t node = S.root_ref;
    if (node == kEmptyRef) return got;
    if (node & kLeafBit) {
        float e;
        if (!box_hit(S.root_box[0], S.root_box[1], S.root_box[2], S.root_box[3], S.root_box[4], S.root_box[5],
                     r.ox, r.oy, r.oz, r.ix, r.iy, r.iz, e))
            return got;
        return leaf_test<ANY, COUNT>(tri, node, r, c) || got;
    }
    for (;;) {
        if (!(node & kLeafBit)) {
            if (COUNT) c.nodes++;
            if (W == 2) {
                const float4* n = nodes + 4 * (size_t)node;
                float4 X = gload(n), Y = gload(n + 1), Z = gload(n + 2);
                int4 C = gload(reinterpret_cast<const int4*>(n + 3));
                float e0, e1;
                bool h0 = child_hit<EXACT>(X.x, Y.x, Z.x, X.z, Y.z, Z.z, r, e0);
                bool h1 = child_hit<EXACT>(X.y, Y.y, Z.y, X.w, Y.w, Z.w, r, e1);
                h0 = h0 && e0 <= r.cull && (uint32_t)C.x != kEmptyRef;
                h1 = h1 && e1 <= r.cull && (uint32_t)C.y != kEmptyRef;
                if (h0 && h1) {
                    uint32_t nearc = (uint32_t)C.x, farc = (uint32_t)C.y;
                    float fe = e1;
                    if (e1 < e0) { nearc = (uint32_t)C.y; farc = (uint32_t)C.x; fe = e0; }
                    st.push(farc, fe);
                    node = nearc;
                    continue;
                } else if (h0) { node = (uint32_t)C.x; continue; }
                else if (h1) { node = (uint32_t)C.y; continue; }
            } else {
                const float4* n = nodes + 8 * (size_t)node;
                float4 LX = gload(n), HX = gload(n + 1), LY = gload(n + 2), HY = gload(n + 3), LZ = gload(n + 4), HZ = gload(n + 5);
                int4 C = gload(reinterpret_cast<const int4*>(n + 6));
                float k0, k1, k2, k3;
                bool h0 = child_hit<EXACT>(LX.x, LY.x, LZ.x, HX.x, HY.x, HZ.x, r, k0);
                bool h1 = child_hit<EXACT>(LX.y, LY.y, LZ.y, HX.y, HY.y, HZ.y, r, k1);
                bool h2 = child_hit<EXACT>(LX.z, LY.z, LZ.z, HX.z, HY.z, HZ.z, r, k2);
                bool h3 = child_hit<EXACT>(LX.w, LY.w, LZ.w, HX.w, HY.w, HZ.w, r, k3);
                uint32_t c0 = (uint32_t)C.x, c1 = (uint32_t)C.y, c2 = (uint32_t)C.z, c3 = (uint32_t)C.w;
                // missed, culled or absent children sort last (key +inf); the
                // FMA form misses the NaN box of an absent child
                k0 = (h0 && k0 <= r.cull && (!EXACT || c0 != kEmptyRef)) ? k0 : INFINITY;
                k1 = (h1 && k1 <= r.cull && (!EXACT || c1 != kEmptyRef)) ? k1 : INFINITY;
                k2 = (h2 && k2 <= r.cull && (!EXACT || c2 != kEmptyRef)) ? k2 : INFINITY;
                k3 = (h3 && k3 <= r.cull && (!EXACT || c3 != kEmptyRef)) ? k3 : INFINITY;
                // 4-input sorting network, ascending entry distance
#define YN_CS(ka, ca, kb, cb)                                              \
    {                                                                      \
        bool sw = kb < ka;                                                 \
        float tk = sw ? kb : ka; kb = sw ? ka : kb; ka = tk;               \
        uint32_t tc = sw ? cb : ca; cb = sw ? ca : cb; ca = tc;            \
    }
                YN_CS(k0, c0, k1, c1);
                YN_CS(k2, c2, k3, c3);
                YN_CS(k0, c0, k2, c2);
                YN_CS(k1, c1, k3, c3);
                YN_CS(k1, c1, k2, c2);
#undef YN_CS
                if (k0 != INFINITY) {
                    st.push3(k1, c1, k2, c2, k3, c3);
                    node = c0;
                    continue;
                }
            }
        } else {
            got |= leaf_test<ANY, COUNT>(tri, node, r, c);
            if (ends<ANY>(r, got)) return true;
        }
        // pop; a deferred child whose entry now lies beyond the best hit is dropped
        for (;;) {
            if (st.sp == 0) return got;
            float et;
            uint32_t ref = st.pop(et);
            if (et > r.cull) continue;
            node = ref;
            break;
        }
    }
}


// The hoisted triangles of one scene: boxes and triangles come through the
// scalar unit, each box while the one before it is tested, instead of as
// loads of one address by every lane.  Those were a tenth of a walk's loads
// through the vector memory pipe, which bounds the walks of large trees, and
// a chain of a dozen trips to memory before each of them: 32 frames of
// 1920x1080 of a 1M-triangle room 171.0 -> 159.1 ms, 1280x720 of a
// 245k-triangle room 3,448 -> 3,235 us, 16.8M paths of the Cornell box (4
// hoisted) 12.5 -> 12.1 ms, 8 bidirectional frames of 1280x720 of it 12.5 ->
// 11.6 ms, twelve served jobs of three scenes 35.3 -> 33.5 ms.
// Returns whether the walk ends here.
template <int ANY, bool COUNT>
__device__ __forceinline__ bool hoisted(yn_cv4f* hb, yn_cv4f* ht, int n, RayState& r, bool& got, Counts& c)
{
    if (n <= 0) return false;
    yn_v4f lo = hb[0], hi = hb[1];
    for (int s = 0; s < n; ++s) {
        const int k = s + 1 < n ? s + 1 : s;
        const yn_v4f nlo = hb[2 * k], nhi = hb[2 * k + 1];
        float e;
        if (box_hit(lo.x, lo.y, lo.z, hi.x, hi.y, hi.z, r.ox, r.oy, r.oz, r.ix, r.iy, r.iz, e) && !(e > r.cull)) {
            if (COUNT) c.tris++;
            const yn_v4f A = ht[3 * s], B = ht[3 * s + 1], C = ht[3 * s + 2];
            got |= tri_test<ANY>(A, B, C, r);
            if (ends<ANY>(r, got)) return true;
        }
        lo = nlo;
        hi = nhi;
    }
    return false;
}

// The tests ahead of the tree, as in traverse(): every slot of a scene
// without a BVH; the hoisted slots; a root that is one leaf.  Returns whether
// the ray goes on to the tree, at `node`.  UNI: every lane of the wave is in
// the same scene.
template <int ANY, bool COUNT, bool UNI>
__device__ __forceinline__ bool trav_start(const DevScene& S, RayState& r, uint32_t& node, bool& got, Counts& c)
{
    const float4* __restrict__ tri = S.tri_isect;
    if (S.brute) {
        for (int s = 0; s < S.n_slots; ++s) {
            if (COUNT) c.tris++;
            got |= tri_test<ANY>(tri, s, r);
            if (ends<ANY>(r, got)) break;
        }
        return false;
    }
    if (UNI) {
        if (hoisted<ANY, COUNT>(scalar_ptr(S.hoist_box), scalar_ptr(tri), __builtin_amdgcn_readfirstlane(S.n_hoist), r,
                                got, c))
            return false;
    } else {
        for (;;) {      // the wave's scenes one after the other
            yn_cv4f* hb = scalar_ptr(S.hoist_box);
            yn_cv4f* ht = scalar_ptr(tri);
            const int n = __builtin_amdgcn_readfirstlane(S.n_hoist);
            if ((uint64_t)ht != (uint64_t)tri) continue;
            if (hoisted<ANY, COUNT>(hb, ht, n, r, got, c)) return false;
            break;
        }
    }
    node = S.root_ref;
    if (node == kEmptyRef) return false;
    if (node & kLeafBit) {
        float e;
        if (box_hit(S.root_box[0], S.root_box[1], S.root_box[2], S.root_box[3], S.root_box[4], S.root_box[5], r.ox,
                    r.oy, r.oz, r.ix, r.iy, r.iz, e))
            got |= leaf_test<ANY, COUNT>(tri, node, r, c);
        return false;
    }
    return true;
}

// The children of an interior node of width 4: the nearest one hit becomes
// `node`, the others go on the stack.  Returns whether any is hit.
template <bool EXACT, typename V, typename VI, typename ST>
__device__ __forceinline__ bool descend(const V& LX, const V& HX, const V& LY, const V& HY, const V& LZ, const V& HZ,
                                        const VI& C, uint32_t& node, RayState& r, ST& st)
{
    float k0, k1, k2, k3;
    bool h0 = child_hit<EXACT>(LX.x, LY.x, LZ.x, HX.x, HY.x, HZ.x, r, k0);
    bool h1 = child_hit<EXACT>(LX.y, LY.y, LZ.y, HX.y, HY.y, HZ.y, r, k1);
    bool h2 = child_hit<EXACT>(LX.z, LY.z, LZ.z, HX.z, HY.z, HZ.z, r, k2);
    bool h3 = child_hit<EXACT>(LX.w, LY.w, LZ.w, HX.w, HY.w, HZ.w, r, k3);
    uint32_t c0 = (uint32_t)C.x, c1 = (uint32_t)C.y, c2 = (uint32_t)C.z, c3 = (uint32_t)C.w;
    // missed, culled or absent children sort last (key +inf); the FMA form
    // misses the NaN box of an absent child
    k0 = (h0 && k0 <= r.cull && (!EXACT || c0 != kEmptyRef)) ? k0 : INFINITY;
    k1 = (h1 && k1 <= r.cull && (!EXACT || c1 != kEmptyRef)) ? k1 : INFINITY;
    k2 = (h2 && k2 <= r.cull && (!EXACT || c2 != kEmptyRef)) ? k2 : INFINITY;
    k3 = (h3 && k3 <= r.cull && (!EXACT || c3 != kEmptyRef)) ? k3 : INFINITY;
    // 4-input sorting network, ascending entry distance
    auto cs = [](float& ka, uint32_t& ca, float& kb, uint32_t& cb) {
        const bool sw = kb < ka;
        const float tk = sw ? kb : ka; kb = sw ? ka : kb; ka = tk;
        const uint32_t tc = sw ? cb : ca; cb = sw ? ca : cb; ca = tc;
    };
    cs(k0, c0, k1, c1);
    cs(k2, c2, k3, c3);
    cs(k0, c0, k2, c2);
    cs(k1, c1, k3, c3);
    cs(k1, c1, k2, c2);
    if (k0 == INFINITY) return false;
    st.push3(k1, c1, k2, c2, k3, c3);
    node = c0;
    return true;
}

// The first step of a walk over a tree of width 4 in a wave of one scene: the
// root through the scalar unit (every new ray of the wave is there), seven
// vector loads and one of their trips fewer.  8 bidirectional frames of
// 1280x720 of the Cornell box 11.63 -> 11.35 ms, a 160x90 frame 440 -> 431 us;
// rooms of 245k and 1M triangles within 0.4%.
template <bool COUNT, bool EXACT, typename ST>
__device__ __forceinline__ bool trav_root(const float4* __restrict__ nodes, uint32_t& node, RayState& r, ST& st,
                                          Counts& c)
{
    if (COUNT) c.nodes++;
    yn_cv4f* n = scalar_ptr(nodes) + 8 * (size_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)node);
    const yn_v4i C = *(const __attribute__((address_space(4))) yn_v4i*)(n + 6);
    return descend<EXACT>((yn_v4f)n[0], (yn_v4f)n[1], (yn_v4f)n[2], (yn_v4f)n[3], (yn_v4f)n[4], (yn_v4f)n[5], C, node,
                          r, st);
}

// One step of a ray's traversal: an interior node, descending to its
// nearest child; when that child is a leaf (or the step began at one), the
// leaf's triangles are tested in the same step and the next node is popped.
// The nodes and triangles are visited in traverse()'s order, so results and
// counts are the same; only the steps are fewer (a wave that runs interior
// and leaf lanes side by side no longer spends a step on each).  Returns true
// while the ray has nodes left; `node`, the stack and the best hit carry over
// between steps.
template <int W, int ANY, int LST, int BLOCK, bool COUNT, bool EXACT>
__device__ __forceinline__ bool trav_step(const float4* __restrict__ nodes, const float4* __restrict__ tri,
                                          uint32_t& node, RayState& r, Stack<LST, BLOCK>& st, bool& got, Counts& c)
{
    if (!(node & kLeafBit)) {
        if (COUNT) c.nodes++;
        if (W == 2) {
            const float4* n = nodes + 4 * (size_t)node;
            float4 X = gload(n), Y = gload(n + 1), Z = gload(n + 2);
            int4 C = gload(reinterpret_cast<const int4*>(n + 3));
            float e0, e1;
            bool h0 = child_hit<EXACT>(X.x, Y.x, Z.x, X.z, Y.z, Z.z, r, e0);
            bool h1 = child_hit<EXACT>(X.y, Y.y, Z.y, X.w, Y.w, Z.w, r, e1);
            h0 = h0 && e0 <= r.cull && (uint32_t)C.x != kEmptyRef;
            h1 = h1 && e1 <= r.cull && (uint32_t)C.y != kEmptyRef;
            if (h0 && h1) {
                uint32_t nearc = (uint32_t)C.x, farc = (uint32_t)C.y;
                float fe = e1;
                if (e1 < e0) { nearc = (uint32_t)C.y; farc = (uint32_t)C.x; fe = e0; }
                st.push(farc, fe);
                node = nearc;
                if (!(node & kLeafBit)) return true;
            } else if (h0) { node = (uint32_t)C.x; if (!(node & kLeafBit)) return true; }
            else if (h1) { node = (uint32_t)C.y; if (!(node & kLeafBit)) return true; }
            else goto pop;
        } else {
            const float4* n = nodes + 8 * (size_t)node;
            float4 LX = gload(n), HX = gload(n + 1), LY = gload(n + 2), HY = gload(n + 3), LZ = gload(n + 4), HZ = gload(n + 5);
            int4 C = gload(reinterpret_cast<const int4*>(n + 6));
            // loaded with the boxes: sunk below the tests (where it is used) it
            // would be one more trip to memory in every step's chain
            __asm__ volatile("" : "+v"(C.x), "+v"(C.y), "+v"(C.z), "+v"(C.w));
            if (!descend<EXACT>(LX, HX, LY, HY, LZ, HZ, C, node, r, st)) goto pop;
            if (!(node & kLeafBit)) return true;
        }
    }
    // a leaf: this iteration's node, or the nearest child just reached
    got |= leaf_test<ANY, COUNT>(tri, node, r, c);
    if (ends<ANY>(r, got)) return false;
pop:
    // pop; a deferred child whose entry now lies beyond the best hit is dropped
    for (;;) {
        if (st.sp == 0) return false;
        float et;
        uint32_t ref = st.pop(et);
        if (et > r.cull) continue;
        node = ref;
        return true;
    }
}

}  // namespace yune
