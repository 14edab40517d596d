// trace.hip — extend (closest hit) and shadow (any hit) kernels.
//
// Replaces traceRay/traverseBVH/rayAabbIntersection/rayTriangleIntersection
// of kernels/legacy/udpt.cl:240-431 for one queue of rays.  The light quad
// is tested by the shading kernel when it creates a ray (udpt.cl:244-276),
// which then passes the quad distance as the ray's tmax; so "no triangle
// nearer than tmax" reads back as the quad hit, exactly as in traceRay.
//
// Result semantics follow the reference:
//  * closest hit: the triangle with the smallest t in (0, tmax) over every
//    leaf whose box the ray meets.  The reference's breadth-first list never
//    shrinks and ignores t; this traversal visits children near-first and
//    skips a box whose entry distance is beyond the best hit so far (with a
//    1e-4 relative margin, so rounding in the box entry can never hide a
//    triangle the reference would find).  Moller-Trumbore uses the
//    reference's operands and order, so t, u, v and the accept/reject of
//    each triangle are bit-identical to the CPU restatement.  Boxes are
//    tested with the reference's slab arithmetic or with a widened FMA form
//    that enters every box the reference's arithmetic enters (yn_slab.h).
//    Only equal-t ties may resolve to a different triangle (test order).
//  * any hit (shadow rays, udpt.cl:307-308): true if some triangle has t in
//    (0, tmax).
//
// Each lane owns one ray.  Its traversal stack keeps the top LST entries in
// LDS, interleaved by lane so a wave's 64 lanes hit 64 banks, and spills
// deeper entries to a per-thread global area (rarely touched: stack depth
// stays far below the tree depth bound).  An entry is a child reference and
// a 16-bit lower bound of its entry distance, so a deferred child that now
// lies beyond the best hit is dropped on pop without fetching it.  Waves pull
// chunks of rays from the queue with one atomic per chunk.
#include "yn_internal_dev.h"
#include "yn_shade.h"
#include "yn_trace.h"

namespace yune {


// Occupancy the kernel is compiled for, per SIMD: the LDS stack (6 B per
// entry and lane, 160 KB per CU) allows 13 / 8 / 6 / 3 waves per SIMD for
// 8 / 12 / 16 / 32 entries, and registers are held to what 7 / 7 / 6 / 3
// waves leave (72 / 72 / 80 / 168).  More waves in flight hide more of the
// node-fetch latency; past 7 the register spills cost more than they hide.
template <int LST>
constexpr int trace_waves() { return LST <= 12 ? 7 : (LST == 16 ? 6 : 3); }

// Result of one ray into the path's slot.
template <bool ANY>
__device__ __forceinline__ void store_hit(const TraceArgs& a, int pidx, const RayState& r, bool got)
{
    if (ANY) a.occ_out[pidx] = got ? 1 : 0;
    else nt_store(a.hit_out + pidx, hit_record(r));
}

template <int W, bool ANY, int LST, int BLOCK, bool COUNT>
__global__ __launch_bounds__(BLOCK, trace_waves<LST>()) void k_trace(TraceArgs a)
{
    __shared__ uint32_t stk_all[LST * BLOCK];
    __shared__ uint16_t stkt_all[LST * BLOCK];
    Stack<LST, BLOCK> st;
    st.lref = (lds_u32*)stk_all;
    st.lt = (lds_u16*)stkt_all;
    st.col = threadIdx.x;
    st.gstride = gridDim.x * BLOCK;
    st.gref = (gbl_u32*)a.ovf_ref;
    st.gt = (gbl_u16*)a.ovf_t;
    st.gbase = blockIdx.x * BLOCK;
    st.gcap = a.ovf_depth;
    st.full = &a.ctr->q[7][0];
    const int lane = (int)__lane_id();
    if (blockIdx.x == 0 && threadIdx.x == 0 && a.zero0) { *a.zero0 = 0; if (a.zero1) *a.zero1 = 0; }
    const uint32_t n = *a.q.count;
    Counts c{0, 0};
    unsigned nrays = 0;
    // The queue is cut into one slice of chunks per XCD: workgroups go to
    // the XCDs round-robin, so block b runs on XCD b % n_slices and takes
    // its chunks from slice b % n_slices, where neighbouring rays (neighbouring
    // pixels) share that XCD's L2.  Each wave first takes its static chunk of
    // its slice without an atomic, then chunks past the slice's static ones
    // from the slice's counter; when the slice is used up it moves on to the
    // next slices in turn (never back), so every chunk is taken exactly once
    // and every wave ends after at most n_slices empty requests.  When the
    // static chunks cover the whole queue, a wave leaves without touching a
    // counter (same-address atomics from every wave would otherwise set a
    // floor on the launch time of short queues).
    const uint32_t ns = (uint32_t)a.n_slices;
    const uint32_t G = gridDim.x, wpb = BLOCK >> 6;
    const uint32_t xs = blockIdx.x % ns;
    const uint32_t wx = (blockIdx.x / ns) * wpb + (threadIdx.x >> 6);     // wave within its slice's XCD
    const uint32_t chunk = (uint32_t)a.chunk;
    const uint32_t n_chunks = (n + chunk - 1) / chunk;
    auto waves_of = [&](uint32_t y) { return ((G - y + ns - 1) / ns) * wpb; };
    auto slice_lo = [&](uint32_t y) { return (uint32_t)(((uint64_t)y * n_chunks) / ns); };
    const bool all_static = n_chunks <= ns * ((G / ns) * wpb);
    uint32_t y = xs, moved = 0;
    for (bool first = true;; first = false) {
        uint32_t ci;
        for (;;) {
            const uint32_t c0 = slice_lo(y), c1 = slice_lo(y + 1);
            if (first) {
                ci = c0 + wx;
            } else if (all_static) {
                ci = n_chunks;          // nothing past the static chunks
                break;
            } else {
                uint32_t k = 0;
                if (lane == 0) k = atomicAdd(a.work + y * kWorkStride, 1u);
                ci = c0 + waves_of(y) + __shfl(k, 0);
            }
            if (ci < c1) break;
            if (all_static) { ci = n_chunks; break; }
            first = false;
            if (++moved >= ns) { ci = n_chunks; break; }
            y = (y + 1) % ns;
        }
        if (ci >= n_chunks) break;
        const uint32_t base = ci * chunk;
        for (uint32_t off = (uint32_t)lane; off < (uint32_t)a.chunk; off += 64) {
            uint32_t i = base + off;
            if (i >= n) break;
            float4 ot = a.q.o_t[i];
            float4 dp = a.q.d_p[i];
            int pidx = __float_as_int(dp.w);
            int sc = a.single_scene >= 0 ? a.single_scene
                                         : a.jobs[a.by_queue ? pidx : a.path_job[pidx >> a.id_shift]].scene;
            if (a.by_queue) pidx = (int)i;      // the result goes beside the ray
            const DevScene& S = a.scenes[sc];
            RayState r;
            const bool fma_ok = start_ray(r, ot, dp, S);
            st.sp = 0;
            // A ray with a NaN in its origin, direction or length hits nothing:
            // u, v or t of every triangle test is NaN, and each acceptance
            // comparison is false.  Its traversal would still visit every
            // node (the NaN guard keeps each slab), one lane for the whole
            // tree, so it is answered without one.
            bool nan_ray = !(ot.x == ot.x && ot.y == ot.y && ot.z == ot.z && ot.w == ot.w && dp.x == dp.x &&
                             dp.y == dp.y && dp.z == dp.z);
            bool got = false;
            if (!nan_ray)
                got = __ballot(!fma_ok) ? traverse<W, ANY, LST, BLOCK, COUNT, true>(S, r, st, c)
                                        : traverse<W, ANY, LST, BLOCK, COUNT, false>(S, r, st, c);
            ++nrays;
            store_hit<ANY>(a, pidx, r, got);
        }
    }
    // one atomic per wave for the statistics
    unsigned long long tot = wave_sum_u64(nrays);
    if (lane == 0 && tot) atomicAdd(ANY ? &a.ctr->rays_shadow : &a.ctr->rays_ext, tot);
    if (COUNT) {
        unsigned long long tn = wave_sum_u64(c.nodes), tt = wave_sum_u64(c.tris);
        if (lane == 0) {
            atomicAdd(ANY ? &a.ctr->nodes_shadow : &a.ctr->nodes_ext, tn);
            atomicAdd(ANY ? &a.ctr->tris_shadow : &a.ctr->tris_ext, tt);
        }
    }
}

// Result of a caller's ray.
__device__ __forceinline__ void store_ray(const RaysArgs& a, uint32_t i, const RayState& r, bool quad)
{
    a.tri[i] = r.tri;
    a.light[i] = r.tri < 0 && quad ? 0 : -1;
    a.t[i] = r.best;
}

// Traversal with lanes refilled.  k_trace runs each lane's ray to its end
// while the wave waits for its slowest ray, so about a quarter of the vector
// lanes do work.  Here the loop takes one traversal step per lane per
// iteration (traverse()'s loop body), and once `a.refill` lanes of the wave
// have finished, those lanes take new rays from the queue, one atomic for
// all of them.  Each ray's own steps, tests and results are those of
// k_trace.  The first fetch of every wave is static (rays wave*64 ..),
// later ones come after the static range from the work counter.
// SS: every ray renders the one scene a.single_scene, whose node and
// triangle arrays are then wave-uniform (scalar registers; per-lane
// pointers would take four vector registers from a kernel held to 72).
template <int W, bool ANY, int LST, int BLOCK, bool COUNT, bool SS>
__global__ __launch_bounds__(BLOCK, trace_waves<LST>()) void k_trace_rf(TraceArgs a)
{
    __shared__ uint32_t stk_all[LST * BLOCK];
    __shared__ uint16_t stkt_all[LST * BLOCK];
    Stack<LST, BLOCK> st;
    st.lref = (lds_u32*)stk_all;
    st.lt = (lds_u16*)stkt_all;
    st.col = threadIdx.x;
    st.gstride = gridDim.x * BLOCK;
    st.gref = (gbl_u32*)a.ovf_ref;
    st.gt = (gbl_u16*)a.ovf_t;
    st.gbase = blockIdx.x * BLOCK;
    st.gcap = a.ovf_depth;
    st.full = &a.ctr->q[7][0];
    st.sp = 0;
    const int lane = (int)__lane_id();
    const unsigned long long below = (1ull << lane) - 1ull;
    if (blockIdx.x == 0 && threadIdx.x == 0 && a.zero0) { *a.zero0 = 0; if (a.zero1) *a.zero1 = 0; }
    const uint32_t n = *a.q.count;
    // a wave with every lane idle always fetches, so the queue drains
    const int refill = a.refill < 1 ? 1 : (a.refill > 64 ? 64 : a.refill);
    // Queue slices as in k_trace, in rays: the wave's first fetch is its
    // static 64 rays of its XCD's slice, later ones as many rays as idle
    // lanes from the slice's counter, past the slice's static rays; a used-up
    // slice sends the wave on to the next ones (never back).
    const uint32_t ns = (uint32_t)a.n_slices;
    const uint32_t G = gridDim.x, wpb = BLOCK >> 6;
    const uint32_t wx = (blockIdx.x / ns) * wpb + (threadIdx.x >> 6);
    auto waves_of = [&](uint32_t y) { return ((G - y + ns - 1) / ns) * wpb; };
    auto slice_lo = [&](uint32_t y) { return (uint32_t)(((uint64_t)y * n) / ns); };
    const bool all_static = (uint64_t)n <= (uint64_t)ns * ((G / ns) * wpb) * 64u;
    uint32_t y = blockIdx.x % ns, moved = 0;
    // the current slice's bounds and wave count, recomputed only when the
    // wave moves on (slice_lo divides 64-bit)
    auto sreg = [](uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); };   // wave-uniform
    uint32_t y_lo = sreg(slice_lo(y)), y_hi = sreg(slice_lo(y + 1)), y_waves = sreg(waves_of(y));
    Counts c{0, 0};
    unsigned nrays = 0;
    RayState r{};
    uint32_t node = 0;
    int pidx = 0;
    bool live = false, got = false, exact = false;
    const int ss = SS ? __builtin_amdgcn_readfirstlane(a.single_scene) : 0;
    const float4* nodes = SS ? a.scenes[ss].nodes : nullptr;
    const float4* tri = SS ? a.scenes[ss].tri_isect : nullptr;
    bool more = true, first = true;
    for (;;) {
        const unsigned long long idle = __ballot(!live);
        const int n_idle = __popcll(idle);
        if (more && n_idle >= refill) {
            uint32_t base = 0, lim = 0;
            for (;;) {
                if (first) {
                    base = y_lo + wx * 64u;          // every lane is idle on the first fetch
                    first = false;
                } else {
                    uint32_t b = 0;
                    if (lane == 0) b = atomicAdd(a.work + y * kWorkStride, (uint32_t)n_idle);
                    base = y_lo + y_waves * 64u + __shfl(b, 0);
                }
                if (base < y_hi) { lim = y_hi; break; }
                if (all_static || ++moved >= ns) { more = false; break; }
                y = (y + 1) % ns;
                y_lo = sreg(slice_lo(y));
                y_hi = sreg(slice_lo(y + 1));
                y_waves = sreg(waves_of(y));
            }
            if (all_static) more = false;            // nothing past the static rays
            const uint32_t i = base + (uint32_t)__popcll(idle & below);
            if (!live && i < lim) {
                float4 ot = nt_load(a.q.o_t + i);
                float4 dp = nt_load(a.q.d_p + i);
                pidx = __float_as_int(dp.w);
                int sc = SS ? ss
                            : a.single_scene >= 0 ? a.single_scene
                                                  : a.jobs[a.by_queue ? pidx : a.path_job[pidx >> a.id_shift]].scene;
                if (a.by_queue) pidx = (int)i;      // the result goes beside the ray
                const DevScene& S = a.scenes[sc];
                exact = !start_ray(r, ot, dp, S);
                st.sp = 0;
                got = false;
                ++nrays;
                // a ray with a NaN component hits nothing (see k_trace)
                live = ot.x == ot.x && ot.y == ot.y && ot.z == ot.z && ot.w == ot.w && dp.x == dp.x &&
                       dp.y == dp.y && dp.z == dp.z;
                if (!SS) {
                    nodes = S.nodes;
                    tri = S.tri_isect;
                }
                if (live) live = trav_start<ANY, COUNT, SS>(S, r, node, got, c);
                if (SS && W == 4 && live) {
                    if (__ballot(exact)) live = trav_root<COUNT, true>(nodes, node, r, st, c);
                    else live = trav_root<COUNT, false>(nodes, node, r, st, c);
                }
                if (!live) store_hit<ANY>(a, pidx, r, got);
            }
        }
        if (__ballot(live) == 0) {
            if (!more) break;
            continue;
        }
        const bool wexact = __ballot(live && exact) != 0;
        if (live) {
            live = wexact ? trav_step<W, ANY, LST, BLOCK, COUNT, true>(nodes, tri, node, r, st, got, c)
                          : trav_step<W, ANY, LST, BLOCK, COUNT, false>(nodes, tri, node, r, st, got, c);
            if (!live) store_hit<ANY>(a, pidx, r, got);
        }
    }
    unsigned long long tot = wave_sum_u64(nrays);
    if (lane == 0 && tot) atomicAdd(ANY ? &a.ctr->rays_shadow : &a.ctr->rays_ext, tot);
    if (COUNT) {
        unsigned long long tn = wave_sum_u64(c.nodes), tt = wave_sum_u64(c.tris);
        if (lane == 0) {
            atomicAdd(ANY ? &a.ctr->nodes_shadow : &a.ctr->nodes_ext, tn);
            atomicAdd(ANY ? &a.ctr->tris_shadow : &a.ctr->tris_ext, tt);
        }
    }
}

// Rays of a caller, in yn_trace's layout: the quad test of traceRay
// (udpt.cl:244-276) as the ray is taken, closest hit or any hit by the ray's
// own flag, and the results written as yn_trace reports them (a triangle
// nearer than the quad replaces the light hit, udpt.cl:386).  One launch for
// all of it, where a queue fill, a launch for each kind of ray and a result
// pass had their records in memory between them.  The loop is k_trace_rf's;
// with no more rays than the grid has lanes each wave takes an equal share
// of them and no counter is touched.
// What bounds it: at a million rays the vector memory pipe, as k_trace_rf
// (260 us for 1,000,003 rays over 123k triangles); at a few hundred the chain
// of one ray's dependent fetches (45 us).  yn_trace of 1,000,003 host rays
// 13.3 -> 2.15 ms (the rest is the bus: 32 MB in, 12 MB out), of 150,001
// shadow rays 1.27 -> 0.41 ms, of 200 rays 95 -> 50 us; yn_trace_noalloc of
// 200,003 rays 189 -> 105 us.
template <int W, int LST>
__global__ __launch_bounds__(kRaysBlock, trace_waves<LST>()) void k_rays(RaysArgs a)
{
    constexpr int BLOCK = kRaysBlock;
    __shared__ uint32_t stk_all[LST * BLOCK];
    __shared__ uint16_t stkt_all[LST * BLOCK];
    Stack<LST, BLOCK> st;
    st.lref = (lds_u32*)stk_all;
    st.lt = (lds_u16*)stkt_all;
    st.col = threadIdx.x;
    st.gstride = gridDim.x * BLOCK;
    st.gref = (gbl_u32*)a.ovf_ref;
    st.gt = (gbl_u16*)a.ovf_t;
    st.gbase = blockIdx.x * BLOCK;
    st.gcap = a.ovf_depth;
    st.full = a.full;
    st.sp = 0;
    const int lane = (int)__lane_id();
    const unsigned long long below = (1ull << lane) - 1ull;
    const uint32_t n = (uint32_t)a.n;
    const DevScene& S = *a.scene;
    const float4* nodes = S.nodes;
    const float4* tri = S.tri_isect;
    // slices of the rays, one per XCD, as in k_trace
    const uint32_t ns = (uint32_t)a.n_slices, G = gridDim.x, wpb = BLOCK >> 6;
    const uint32_t wx = (blockIdx.x / ns) * wpb + (threadIdx.x >> 6);
    auto waves_of = [&](uint32_t y) { return ((G - y + ns - 1) / ns) * wpb; };
    auto slice_lo = [&](uint32_t y) { return (uint32_t)(((uint64_t)y * n) / ns); };
    auto sreg = [](uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); };   // wave-uniform
    const uint32_t min_waves = (G / ns) * wpb;
    const bool all_static = (uint64_t)n <= (uint64_t)ns * min_waves * 64u;
    // rays of a wave's first fetch: its share of a slice (at most n / ns + 1 rays) when they all fit
    const uint32_t per = all_static ? min(64u, (n / ns + min_waves) / min_waves) : 64u;
    uint32_t y = blockIdx.x % ns, moved = 0;
    uint32_t y_lo = sreg(slice_lo(y)), y_hi = sreg(slice_lo(y + 1)), y_waves = sreg(waves_of(y));
    Counts c{0, 0};
    RayState r{};
    uint32_t node = 0, ray = 0;
    bool live = false, got = false, exact = false, quad = false;
    bool more = true, first = true;
    for (;;) {
        const unsigned long long idle = __ballot(!live);
        const int n_idle = __popcll(idle);
        if (more && (first || n_idle >= a.refill)) {
            uint32_t base = 0, lim = 0;
            for (;;) {
                if (first) {
                    base = y_lo + wx * per;          // every lane is idle on the first fetch
                    first = false;
                    if (base < y_hi) { lim = min(y_hi, base + per); break; }
                } else {
                    uint32_t b = 0;
                    if (lane == 0) b = atomicAdd(a.work + y * kWorkStride, (uint32_t)n_idle);
                    base = y_lo + y_waves * 64u + __shfl(b, 0);
                    if (base < y_hi) { lim = y_hi; break; }
                }
                if (all_static || ++moved >= ns) { more = false; break; }
                y = (y + 1) % ns;
                y_lo = sreg(slice_lo(y));
                y_hi = sreg(slice_lo(y + 1));
                y_waves = sreg(waves_of(y));
            }
            if (all_static) more = false;
            const uint32_t i = base + (uint32_t)__popcll(idle & below);
            if (!live && i < lim) {
                ray = i;
                float4 ot, dp;
                const float* q = a.rays + 8 * (size_t)i;
                if (a.aligned) {
                    ot = gload(reinterpret_cast<const float4*>(q));
                    dp = gload(reinterpret_cast<const float4*>(q) + 1);
                } else {
                    ot = make_float4(q[0], q[1], q[2], q[3]);
                    dp = make_float4(q[4], q[5], q[6], q[7]);
                }
                float t;
                quad = quad_hit(S.light, mk(ot.x, ot.y, ot.z, 1.0f), mk(dp.x, dp.y, dp.z, 0.0f), ot.w, t);
                if (quad) ot.w = t;
                exact = !start_ray(r, ot, dp, S);
                r.any = dp.w != 0.0f;
                st.sp = 0;
                got = false;
                // a ray with a NaN component hits nothing (see k_trace)
                live = ot.x == ot.x && ot.y == ot.y && ot.z == ot.z && ot.w == ot.w && dp.x == dp.x &&
                       dp.y == dp.y && dp.z == dp.z;
                if (live) live = trav_start<2, false, true>(S, r, node, got, c);
                if (W == 4 && live) {
                    if (__ballot(exact)) live = trav_root<false, true>(nodes, node, r, st, c);
                    else live = trav_root<false, false>(nodes, node, r, st, c);
                }
                if (!live) store_ray(a, ray, r, quad);
            }
        }
        if (__ballot(live) == 0) {
            if (!more) break;
            continue;
        }
        const bool wexact = __ballot(live && exact) != 0;
        if (live) {
            live = wexact ? trav_step<W, 2, LST, BLOCK, false, true>(nodes, tri, node, r, st, got, c)
                          : trav_step<W, 2, LST, BLOCK, false, false>(nodes, tri, node, r, st, got, c);
            if (!live) store_ray(a, ray, r, quad);
        }
    }
}

namespace {
template <int W, bool ANY, int LST, int BL>
void launch_b(const TraceArgs& a, int grid, bool count, hipStream_t s)
{
    if (a.refill > 0) {
        bool done = false;
        if constexpr (W == 4) {
            if (a.single_scene >= 0) {
                if (count) hipLaunchKernelGGL((k_trace_rf<W, ANY, LST, BL, true, true>), dim3(grid), dim3(BL), 0, s, a);
                else hipLaunchKernelGGL((k_trace_rf<W, ANY, LST, BL, false, true>), dim3(grid), dim3(BL), 0, s, a);
                done = true;
            }
        }
        if (!done) {
            if (count) hipLaunchKernelGGL((k_trace_rf<W, ANY, LST, BL, true, false>), dim3(grid), dim3(BL), 0, s, a);
            else hipLaunchKernelGGL((k_trace_rf<W, ANY, LST, BL, false, false>), dim3(grid), dim3(BL), 0, s, a);
        }
    } else {
        if (count) hipLaunchKernelGGL((k_trace<W, ANY, LST, BL, true>), dim3(grid), dim3(BL), 0, s, a);
        else hipLaunchKernelGGL((k_trace<W, ANY, LST, BL, false>), dim3(grid), dim3(BL), 0, s, a);
    }
}

template <bool ANY, int LST>
void launch_w(const TraceArgs& a, int width, int block, int grid, bool count, hipStream_t s)
{
    if (width == 2) {
        if (block == 64) launch_b<2, ANY, LST, 64>(a, grid, count, s);
        else if (block == 128) launch_b<2, ANY, LST, 128>(a, grid, count, s);
        else launch_b<2, ANY, LST, 256>(a, grid, count, s);
    } else {
        if (block == 64) launch_b<4, ANY, LST, 64>(a, grid, count, s);
        else if (block == 128) launch_b<4, ANY, LST, 128>(a, grid, count, s);
        else launch_b<4, ANY, LST, 256>(a, grid, count, s);
    }
}

template <bool ANY>
void launch_l(const TraceArgs& a, int width, int block, int grid, bool count, int lds, hipStream_t s)
{
    if (lds == 8) launch_w<ANY, 8>(a, width, block, grid, count, s);
    else if (lds == 12) launch_w<ANY, 12>(a, width, block, grid, count, s);
    else if (lds == 32) launch_w<ANY, 32>(a, width, block, grid, count, s);
    else launch_w<ANY, 16>(a, width, block, grid, count, s);
}
}  // namespace

// LDS part of the traversal stack: 8, 12, 16 or 32 entries per lane.
int trace_lds_stack(int lds) { return lds == 8 || lds == 12 || lds == 32 ? lds : 16; }

// Waves per SIMD a trace launch runs at for a configured LDS stack.
int trace_resident_waves(int lds)
{
    lds = trace_lds_stack(lds);
    return lds == 8 ? trace_waves<8>() : lds == 12 ? trace_waves<12>() : (lds == 32 ? trace_waves<32>() : trace_waves<16>());
}

// LDS part of a caller's rays' stack: 12 or 16 entries.
int rays_lds_stack(int lds) { return lds > 0 && lds <= 12 ? 12 : 16; }

void launch_rays(const RaysArgs& a, int width, int lds, int grid, hipStream_t s)
{
    const bool l12 = rays_lds_stack(lds) == 12;
    if (width == 2) {
        if (l12) hipLaunchKernelGGL((k_rays<2, 12>), dim3(grid), dim3(kRaysBlock), 0, s, a);
        else hipLaunchKernelGGL((k_rays<2, 16>), dim3(grid), dim3(kRaysBlock), 0, s, a);
    } else {
        if (l12) hipLaunchKernelGGL((k_rays<4, 12>), dim3(grid), dim3(kRaysBlock), 0, s, a);
        else hipLaunchKernelGGL((k_rays<4, 16>), dim3(grid), dim3(kRaysBlock), 0, s, a);
    }
}

// `stack`: traversal stack entries the scene can need; the launch is refused
// when LDS plus the overflow area cannot hold them.
int launch_trace(const TraceArgs& a, bool any_hit, int width, int stack, int block, int grid, bool count, int lds,
                 hipStream_t stream)
{
    lds = trace_lds_stack(lds);
    if (stack > lds + a.ovf_depth) return -1;
    if (any_hit) launch_l<true>(a, width, block, grid, count, lds, stream);
    else launch_l<false>(a, width, block, grid, count, lds, stream);
    return 0;
}

}  // namespace yune
