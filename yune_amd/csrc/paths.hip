// paths.hip — whole unidirectional paths in one launch.
//
// The wavefront (pt.hip, trace.hip) launches a trace and a shade for every
// ray of the deepest path and waits, in each, for the slowest ray of all.
// With few paths in flight that costs more than the work: 5,917 paths of a
// Cornell box need 82 launches, each as long as one ray's chain of dependent
// fetches.  Here each lane keeps its path: it traces the path's ray, runs the
// shade step (yn_path.h) with the result and the record in registers, and
// goes on with the ray the step made until the path ends, then takes the next
// path of the queues.  Paths never wait for each other beyond their wave, no
// ray, record or result goes through memory in between, and each path's
// arithmetic is that of the wavefront, so images are the same bit for bit.
//
// What bounds it: vector issue (91% busy on the Cornell box) with a quarter
// of the lanes at work, since a wave's lanes wait for its longest walk and
// run each other's shade steps; when a wave holds few paths, the chain of one
// path's fetches.  97x61 pixels of the Cornell box without a bounce limit:
// 2,100 -> 285 us; 1280x720 of a 245k-triangle room (NEE + MIS, depth 8):
// 7,590 -> 3,290 us.  Variants measured at 4.2M paths of that room: 3 waves
// per SIMD (no spills) 7.9 ms, 4 waves (8 registers spilled) 6.8, 5 waves
// (102) 6.5 but 7% slower at 262,144 paths; lanes that finish their walk
// shaded while the others walk on (30 spilled at 3 waves) 8.0; all closest-
// hit rays of a wave before its shadow rays 9.9; interior nodes and leaves as
// separate turns of the walk 8.6.
#include "yn_internal_dev.h"
#include "yn_path.h"
#include "yn_trace.h"

namespace yune {

namespace {

struct RegResult {
    float4 h;
    int o;
    __device__ __forceinline__ float4 hit() const { return h; }
    __device__ __forceinline__ int occ() const { return o; }
};

// (The arguments' address is opaque at each call: otherwise the compiler
// loads every field before the loop and spills what the registers cannot
// hold, instead of loading it again where it is used.)
template <bool ONE>
__device__ __forceinline__ auto tables_of(const PathsArgs& a)
{
    if constexpr (ONE) {
        auto* k = (const __attribute__((address_space(4))) PathsArgs*)__builtin_amdgcn_kernarg_segment_ptr();
        __asm__ volatile("" : "+s"(k));
        return OneJob{*(const DevJob*)&k->job, *(const DevScene*)&k->scene};
    } else {
        return JobTables{a.s.jobs, a.s.scenes};
    }
}

}  // namespace

// ONE: all paths of one job (LM 1).  PARK: see PathsArgs::parked.
template <int LM, bool ONE, bool PARK>
__global__ __launch_bounds__(kPathsBlock, paths_waves(LM)) void k_paths(PathsArgs a)
{
    constexpr int BL = kPathsBlock;
    __shared__ uint32_t stk_all[kPathsLds * BL];
    __shared__ uint16_t stkt_all[kPathsLds * BL];
    __shared__ float4 smat4[LM ? kLdsMats * 5 : 1];
    __shared__ float4 slight4[LM == 2 ? kLdsLights * 5 : LM == 1 ? 5 : 1];
    const ShadeArgs& s = a.s;
    if (LM) {
        for (int k = (int)threadIdx.x; k < s.n_lmats * 5; k += BL) smat4[k] = s.lmats[k];
        for (int k = (int)threadIdx.x; k < s.n_lights * 5; k += BL)
            slight4[k] = reinterpret_cast<const float4*>(&s.scenes[LM == 1 ? s.lscene : k / 5].light)[k % 5];
        __syncthreads();
    }
    const LdsScene lds{(lds_mat*)(void*)smat4, (lds_light*)(void*)slight4};
    Stack<kPathsLds, BL> st;
    st.lref = (lds_u32*)stk_all;
    st.lt = (lds_u16*)stkt_all;
    st.col = threadIdx.x;
    st.gstride = gridDim.x * BL;
    st.gref = (gbl_u32*)a.ovf_ref;
    st.gt = (gbl_u16*)a.ovf_t;
    st.gbase = blockIdx.x * BL;
    st.gcap = a.ovf_depth;
    st.full = &s.ctr->q[7][0];
    const int lane = (int)__lane_id();
    const unsigned long long below = (1ull << lane) - 1ull;
    const uint32_t n_ext = *s.ext_in.count, total = n_ext + *s.sh_in.count;
    // the paths spread over all the waves of the grid: with fewer paths than
    // lanes a wave holds only as many as it must, since its lanes wait for
    // each other in every ray and step
    const uint32_t n_waves = gridDim.x * (BL / 64);
    const uint32_t per = min(64u, (total + n_waves - 1) / n_waves);
    const uint32_t wave = blockIdx.x * (BL / 64) + (threadIdx.x >> 6);
    bool more = total > n_waves * per;              // paths beyond the static ones
    Rec R;
    R.m0 = make_int4(0, 0, 0, 0);
    float4 ot = make_float4(0, 0, 0, 0), dp = ot;
    bool any = false, live = false;
    // takes path i of the queues: first the extension queue's, then the shadow queue's
    auto take = [&](uint32_t i) {
        const bool ext = i < n_ext;
        const uint32_t qi = ext ? i : i - n_ext;
        live = true;
        any = !ext;
        ot = ext ? s.ext_in.o_t[qi] : s.sh_in.o_t[qi];
        dp = ext ? s.ext_in.d_p[qi] : s.sh_in.d_p[qi];
        load_rec<false>(s.in, ext ? qi : (uint32_t)(s.in.cap - 1 - (int64_t)qi), dp, R, ext && s.ext_primary);
    };
    if ((uint32_t)lane < per && wave * per + (uint32_t)lane < total) take(wave * per + (uint32_t)lane);
    unsigned long long n_rays[2] = {0, 0};          // closest-hit and any-hit, of the wave
    Counts c{0, 0};
    const DevCapture cap{};
    for (;;) {
        const unsigned long long lm = __ballot(live);
        if (!lm) break;
        const unsigned k = (unsigned)__popcll(__ballot(live && any));
        n_rays[0] += (unsigned)__popcll(lm) - k;
        n_rays[1] += k;
        if (live) {
            const auto tab = tables_of<ONE>(a);
            const DevScene& S = tab.scene(LM == 1 ? s.lscene : (R.m0.y >> SCENE_SHIFT) & 0xff);
            RayState r;
            const bool fma_ok = start_ray(r, ot, dp, S);
            r.any = any;
            st.sp = 0;
            // a ray with a NaN component hits nothing (see k_trace)
            const bool nan_ray = !(ot.x == ot.x && ot.y == ot.y && ot.z == ot.z && ot.w == ot.w && dp.x == dp.x &&
                                   dp.y == dp.y && dp.z == dp.z);
            bool got = false;
            uint32_t node = 0;
            bool go = !nan_ray && trav_start<2, false, LM == 1>(S, r, node, got, c);
            const float4 *nodes = S.nodes, *tri = S.tri_isect;
            if (__ballot(!fma_ok)) {
                if (LM == 1 && go) go = trav_root<false, true>(nodes, node, r, st, c);
                while (go) go = trav_step<4, 2, kPathsLds, BL, false, true>(nodes, tri, node, r, st, got, c);
            } else {
                if (LM == 1 && go) go = trav_root<false, false>(nodes, node, r, st, c);
                while (go) go = trav_step<4, 2, kPathsLds, BL, false, false>(nodes, tri, node, r, st, got, c);
            }
            R.dir = mk(dp.x, dp.y, dp.z, 0.0f);
            R.job = __float_as_int(dp.w);
            const Out o = advance<false, LM>(
                tab, cap, RegResult{hit_record(r), got ? 1 : 0}, R, lds);
            ot = o.o_t;
            dp = o.d_p;
            any = o.kind == 2;
            live = o.kind != 0;
            if constexpr (PARK) {   // once in every stretch: a bounce has one closest-hit ray
                if (o.kind == 1 && (R.m0.z & (kParkBounces - 1)) == kParkBounces - 1) {
                    const uint32_t at = atomicAdd(a.parked, 1u);
                    s.ext_out.o_t[at] = ot;
                    s.ext_out.d_p[at] = dp;
                    store_rec(s.out, at, R);
                    atomicAdd(a.left + (R.job - s.done_base), 1u);
                    live = false;
                }
            } else if (live && R.m0.z >= kMaxPathBounces) {
                *a.endless = 1;
                live = false;
            }
        }
        if (more) {         // lanes whose paths have ended take the next ones
            const unsigned long long idle = __ballot(!live);
            if (idle) {
                uint32_t b = 0;
                // after an endless path no more are taken
                if constexpr (PARK) {
                    if (lane == 0) b = n_waves * per + atomicAdd(a.next, (uint32_t)__popcll(idle));
                } else if (lane == 0) {
                    b = __hip_atomic_load(a.endless, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                            ? total
                            : n_waves * per + atomicAdd(a.next, (uint32_t)__popcll(idle));
                }
                b = __shfl(b, 0);
                if (b >= total) more = false;
                const uint32_t i = b + (uint32_t)__popcll(idle & below);
                if (!live && i < total) take(i);
            }
        }
    }
    if (lane == 0 && n_rays[0]) atomicAdd(&s.ctr->rays_ext, n_rays[0]);
    if (lane == 0 && n_rays[1]) atomicAdd(&s.ctr->rays_shadow, n_rays[1]);
}

void launch_paths(const PathsArgs& a, int grid, hipStream_t stream)
{
    const int lm = a.s.lmats != nullptr && a.s.n_lmats <= kLdsMats ? a.s.lmode : 0;
    const dim3 g(grid), b(kPathsBlock);
    if (a.parked) {
        if (lm == 1) hipLaunchKernelGGL((k_paths<1, false, true>), g, b, 0, stream, a);
        else if (lm == 2) hipLaunchKernelGGL((k_paths<2, false, true>), g, b, 0, stream, a);
        else hipLaunchKernelGGL((k_paths<0, false, true>), g, b, 0, stream, a);
    } else {
        if (lm == 1 && a.one) hipLaunchKernelGGL((k_paths<1, true, false>), g, b, 0, stream, a);
        else if (lm == 1) hipLaunchKernelGGL((k_paths<1, false, false>), g, b, 0, stream, a);
        else if (lm == 2) hipLaunchKernelGGL((k_paths<2, false, false>), g, b, 0, stream, a);
        else hipLaunchKernelGGL((k_paths<0, false, false>), g, b, 0, stream, a);
    }
}

}  // namespace yune
