// pt.hip — generate, shade and resolve kernels of the wavefront
// unidirectional path tracer (kernels/legacy/udpt.cl semantics).
//
// The reference runs one path per work-item from camera ray to the end
// (pathtracer -> shading -> evaluateDirectLighting, udpt.cl:158-609).  Here
// each path is a small state machine stored in HBM; a shade pass consumes
// the result of the path's one outstanding ray and runs until the path
// needs its next ray (or ends):
//
//   PRIMARY  --hit--> [NEE start] --shadow ray--> NEE_SH --> [lobe pick,
//   light sample, MIS direction] --MIS ray--> NEE_MIS --> [BOUNCE: sample
//   direction] --extension ray--> BOUNCE --hit--> [emission, throughput,
//   RR] --> NEE start at the new vertex ...
//
// The per-path xorshift state travels with the path and is consumed in the
// reference's order (including the lobe pick that only happens after an
// unoccluded shadow ray, udpt.cl:557-559), so primary and first shadow rays
// are bit-identical to the CPU restatement and later decisions agree up to
// libm-vs-device ulps in sin/cos/pow.
//
// Rays never recorded by the reference as separate entities:
//  * the quad light is tested here when a ray is made (udpt.cl:244-276);
//    a hit shortens the ray to the quad and marks it, so an extension ray
//    that finds no nearer triangle is a light hit;
//  * an NEE shadow ray the quad already blocks is occluded without a BVH
//    query (traceRay would return true either way);
//  * the MIS BRDF ray only matters if it reaches the light first
//    (udpt.cl:599), so it is an any-hit query up to the quad, skipped when
//    the quad is missed.
#include "yn_internal_dev.h"
#include "yn_path.h"
#include "yn_shade.h"

namespace yune {

// WAVES: the occupancy the register allocation is held to, per SIMD.
// Blocks of shade_block_pt(WAVES) threads walk the queues together, one atomic per
// block and output queue.  A path's record is read beside the ray whose
// result it consumes and written, once the block knows where the path's
// next ray goes, beside that ray.
// CAP: the variant that records the first frame's primary hits and shadow
// rays for the parity tests (without it, the kernel holds fewer values).
template <int WAVES, bool CAP, int LM>
__global__ __launch_bounds__(shade_block_pt(WAVES), WAVES) void k_shade_pt(ShadeArgs a, DevCapture cap)
{
    constexpr int BL = shade_block_pt(WAVES);
    __shared__ BlockReserveLds<2, BL> rsv;
    // LM: the materials of a.lmats (a.n_lmats <= kLdsMats) and the light quads
    __shared__ float4 smat4[LM ? kLdsMats * 5 : 1];
    __shared__ float4 slight4[LM ? kLdsLights * 5 : 1];
    if (LM) {
        for (int k = (int)threadIdx.x; k < a.n_lmats * 5; k += BL) smat4[k] = a.lmats[k];
        for (int k = (int)threadIdx.x; k < a.n_lights * 5; k += BL)
            slight4[k] = reinterpret_cast<const float4*>(&a.scenes[LM == 1 ? a.lscene : k / 5].light)[k % 5];
        __syncthreads();
    }
    const LdsScene lds{(lds_mat*)(void*)smat4, (lds_light*)(void*)slight4};
    // continuous serving: ended paths per job-table entry, gathered per block
    // in a small table and added to the device counters once at the end
    // (device-scope atomics on one cache line, one per wave, serialise)
    constexpr int kDoneSlots = 16;
    __shared__ int32_t dkey[kDoneSlots];
    __shared__ uint32_t dval[kDoneSlots];
    const uint32_t n_ext = *a.ext_in.count, n_sh = *a.sh_in.count;
    const uint32_t total = n_ext + n_sh;
    if (blockIdx.x == 0 && (int)threadIdx.x < a.n_zero) a.zero[threadIdx.x * kWorkStride] = 0;
    if (a.done_ctr) {
        if (threadIdx.x < (unsigned)kDoneSlots) { dkey[threadIdx.x] = -1; dval[threadIdx.x] = 0; }
        __syncthreads();
    }
    auto done_add = [&](int e, uint32_t n) {
        int h = e & (kDoneSlots - 1);
        for (int k = 0; k < kDoneSlots; ++k, h = (h + 1) & (kDoneSlots - 1)) {
            const int old = atomicCAS(&dkey[h], -1, e);
            if (old == -1 || old == e) { atomicAdd(&dval[h], n); return; }
        }
        atomicAdd(a.done_ctr + (e - a.done_base), n);     // table full: straight to the counter
    };
    uint32_t* const ctr[2] = {a.ext_out.count, a.sh_out.count};
    int par = 0;
    // the block walks the queues together: its appends are one atomic per queue
    constexpr uint32_t B = BL;
    for (uint32_t base = blockIdx.x * B; base < total; base += gridDim.x * B, par ^= 1) {
        uint32_t i = base + threadIdx.x;
        Out o;
        Rec R;
        if (i < total) {
            const bool ext = i < n_ext;
            const uint32_t qi = ext ? i : i - n_ext;
            const float4 dp = nt_load(ext ? &a.ext_in.d_p[qi] : &a.sh_in.d_p[qi]);
            load_rec<true>(a.in, ext ? qi : (uint32_t)(a.in.cap - 1 - (int64_t)qi), dp, R, ext && a.ext_primary);
            o = advance<CAP, LM>(JobTables{a.jobs, a.scenes}, cap, QueueResult{a.hit, a.occ, qi}, R, lds);
        }
        const uint32_t n[2] = {o.kind == 1 ? 1u : 0u, o.kind == 2 ? 1u : 0u};
        uint32_t at[2];
        block_reserve<2, BL>(rsv, par, ctr, n, at);
        if (o.kind == 1) {
            nt_store(&a.ext_out.o_t[at[0]], o.o_t);
            nt_store(&a.ext_out.d_p[at[0]], o.d_p);
            store_rec(a.out, at[0], R);
        }
        if (o.kind == 2) {
            nt_store(&a.sh_out.o_t[at[1]], o.o_t);
            nt_store(&a.sh_out.d_p[at[1]], o.d_p);
            store_rec(a.out, (uint32_t)(a.out.cap - 1 - (int64_t)at[1]), R);
        }
        if (a.done_ctr) {
            // ended paths per job-table entry, one table update per entry
            // present in the wave (mostly one: a queue's paths come in runs of one job)
            const bool dn = i < total && o.done;
            unsigned long long m = __ballot(dn);
            while (m) {
                const int leader = __ffsll((long long)m) - 1;
                const int e = __shfl(o.job, leader);
                const unsigned long long g = __ballot(dn && o.job == e);
                if ((int)__lane_id() == leader && e >= a.done_base) done_add(e, (uint32_t)__popcll(g));
                m &= ~g;
            }
        }
    }
    if (a.done_ctr) {       // the loop is block-uniform: every thread gets here
        __syncthreads();
        if (threadIdx.x < (unsigned)kDoneSlots && dkey[threadIdx.x] >= 0 && dval[threadIdx.x])
            atomicAdd(a.done_ctr + (dkey[threadIdx.x] - a.done_base), dval[threadIdx.x]);
    }
}

// Primary rays (pathtracer entry, udpt.cl:162-189) for a list of segments:
// work item -> (segment, pixel), a ray at the item's queue position and the
// new path's record beside it.
// ONE: every path belongs to the arguments' job.
template <bool ONE>
__global__ __launch_bounds__(256) void k_generate(GenArgs a, DevCapture cap)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.n_paths) return;
    const int item = a.item0 + i;
    // behind the rays already queued: k_queue_reserve took the count before
    // this launch and added n_paths to it
    const uint32_t qpos = a.queue_base ? *a.queue_base + (uint32_t)i : (uint32_t)i;
    const GenSeg g = seg_of<kOwnFrames>(a, item);
    int x, y;
    seg_pixel(item - g.path_base + g.first, g.w, g.h, x, y);
    x += g.x0;
    y += g.y0;
    const DevJob& J = ONE ? a.job : a.jobs[g.job];
    const yn_light_quad& light = ONE ? a.light : a.scenes[J.scene].light;
    uint32_t seed = pixel_seed(g.rand, x, y, J.W);
    float r1 = next_rand(seed);
    float r2 = next_rand(seed);
    f4 o, d;
    create_ray((float)x + r1, (float)y + r2, J.W, J.H, J.cam, o, d);
    float tq, tmax = INFINITY;
    int st = ST_PRIMARY | (J.scene << SCENE_SHIFT);
    if (quad_hit(light, o, d, INFINITY, tq)) { tmax = tq; st |= F_LCAND; }
    const uint32_t sample = (uint32_t)g.slot * (uint32_t)(J.W * J.H) + (uint32_t)(y * J.W + x);
    *reinterpret_cast<int4*>(a.rec.f(PathRecs::M0, qpos)) = make_int4((int)seed, st, (int)sample, 0);
    a.ext_out.o_t[qpos] = make_float4(o.x, o.y, o.z, tmax);
    a.ext_out.d_p[qpos] = make_float4(d.x, d.y, d.z, __int_as_float(g.job));
    if (!a.queue_base && i == 0) *a.ext_out.count = (uint32_t)a.n_paths;
    if (cap.prim_tri && g.slot == 0) {
        cap.shadow_occ[y * J.W + x] = -1;
        cap.shadow_d[y * J.W + x] = make_float4(0, 0, 0, 0);
    }
}

// Running average of the batch's frames, oldest first (udpt.cl:196-210).
__global__ __launch_bounds__(256) void k_resolve(ResolveArgs a)
{
    int q = blockIdx.x * blockDim.x + threadIdx.x;
    // paths that were given up, or not taken, have no sample to fold (the
    // flags stay up, since every block of the batch's folds reads them; they
    // are asked for here and looked at only before the store, behind the
    // samples' loads)
    const uint32_t failed = a.ctr->q[6][0] | a.ctr->q[7][0];
    if (a.host && blockIdx.x == 0 && threadIdx.x < 64) {    // the batch's last launch: its counters
        const int i = (int)threadIdx.x;
        unsigned long long *from = &a.ctr->rays_ext, *to = &a.host->rays_ext;
        if (i < 6) to[i] = from[i];
        if (i < 12) a.host->q[i][0] = a.ctr->q[i][0];
        clear_counters(a.ctr);
    }
    if (q >= a.w * a.h) return;
    int x = a.x0 + q % a.w, y = a.y0 + q / a.w;
    size_t pix = (size_t)y * a.W + x;
    size_t npix = (size_t)a.W * a.H;
    f4 acc = ld(a.prev[pix]);
    for (int k = 0; k < a.n_slots; ++k) {
        f4 c = ld(a.samples[(size_t)k * npix + pix]);
        if (k == 0 && a.reset_first) {
            c.w = 1;
        } else {
            int num_passes = (int)acc.w;
            c = c + acc * (float)num_passes;
            c = c / (float)(num_passes + 1);
            c.w = (float)(num_passes + 1);
        }
        acc = c;
    }
    if (failed == 0) a.accum[pix] = st4(acc);
}

// The kernels' sin / cos / pow evaluated on the device (diagnostics).
__global__ __launch_bounds__(256) void k_fmath(int op, const float* x, const float* y, int n, float* out)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    out[i] = op == 0 ? ynf_sinf(x[i]) : op == 1 ? ynf_cosf(x[i]) : ynf_powf(x[i], y[i]);
}

void launch_fmath(int op, const float* x, const float* y, int n, float* out, hipStream_t s)
{
    if (n > 0) hipLaunchKernelGGL(k_fmath, dim3((n + 255) / 256), dim3(256), 0, s, op, x, y, n, out);
}

// Reserves n entries at the end of a queue: base = count, count += n.
__global__ void k_queue_reserve(uint32_t* count, uint32_t n, uint32_t* base)
{
    if (threadIdx.x == 0) {
        const uint32_t c = *count;
        *base = c;
        *count = c + n;
    }
}

void launch_generate(const GenArgs& a, const DevCapture& cap, hipStream_t s)
{
    int grid = (a.n_paths + 255) / 256;
    if (grid <= 0) return;
    if (a.queue_base)
        hipLaunchKernelGGL(k_queue_reserve, dim3(1), dim3(64), 0, s, a.ext_out.count, (uint32_t)a.n_paths,
                           a.queue_base);
    if (a.one) hipLaunchKernelGGL((k_generate<true>), dim3(grid), dim3(256), 0, s, a, cap);
    else hipLaunchKernelGGL((k_generate<false>), dim3(grid), dim3(256), 0, s, a, cap);
}
void launch_shade_pt(const ShadeArgs& a, const DevCapture& cap, int grid, int waves, hipStream_t s)
{
    if (cap.prim_tri) {
        hipLaunchKernelGGL((k_shade_pt<4, true, 0>), dim3(grid), dim3(shade_block_pt(4)), 0, s, a, cap);
        return;
    }
    const int lm = a.lmats != nullptr && a.n_lmats <= kLdsMats ? a.lmode : 0;
    if (waves == 4) {
        if (lm == 1) hipLaunchKernelGGL((k_shade_pt<4, false, 1>), dim3(grid), dim3(shade_block_pt(4)), 0, s, a, cap);
        else if (lm == 2) hipLaunchKernelGGL((k_shade_pt<4, false, 2>), dim3(grid), dim3(shade_block_pt(4)), 0, s, a, cap);
        else hipLaunchKernelGGL((k_shade_pt<4, false, 0>), dim3(grid), dim3(shade_block_pt(4)), 0, s, a, cap);
    } else if (waves == 3) {
        hipLaunchKernelGGL((k_shade_pt<3, false, 0>), dim3(grid), dim3(shade_block_pt(3)), 0, s, a, cap);
    } else {
        hipLaunchKernelGGL((k_shade_pt<2, false, 0>), dim3(grid), dim3(shade_block_pt(2)), 0, s, a, cap);
    }
}
void launch_resolve(const ResolveArgs& a, hipStream_t s)
{
    int n = a.w * a.h;
    if (n > 0) hipLaunchKernelGGL(k_resolve, dim3((n + 255) / 256), dim3(256), 0, s, a);
}

}  // namespace yune
