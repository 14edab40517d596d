// yn_path.h — one shade step of a unidirectional path (kernels/legacy/udpt.cl
// semantics), shared by the wavefront's shade kernel (pt.hip) and the kernel
// that runs whole paths (paths.hip).
#pragma once

#include "yn_internal_dev.h"
#include "yn_shade.h"

namespace yune {

enum : int {
    ST_DONE = 0,
    ST_PRIMARY = 1,
    ST_BOUNCE = 2,
    ST_NEE_SH = 3,
    ST_NEE_MIS = 4,
    ST_MASK = 0xff,
    F_DIRECT = 1 << 8,      // NEE result is the first vertex's direct light
    F_LCAND = 1 << 9,       // pending extension ray ends on the quad
    F_NGLOSSY = 1 << 10,    // NEE lobe: glossy
    F_BGLOSSY = 1 << 11,    // bounce lobe: glossy
    F_CAPSH = 1 << 12,      // first shadow ray already captured
    SCENE_SHIFT = 16,       // bits 16..23: the path's scene (its job's), read without the job
};

constexpr float kPinkR = 0.988f, kPinkG = 0.0588f, kPinkB = 0.7529f;   // udpt.cl:110

struct Out {
    int kind = 0;           // 0 none, 1 extension, 2 shadow
    bool done = false;      // the path ended and wrote its sample
    int job = -1;           // the path's job-table entry
    float4 o_t;
    float4 d_p;
};

// A path's state between two shade steps (the fields of PathRecs, and of the
// pending ray, which holds the rest).
struct Rec {
    int4 m0;
    uint32_t sample;        // frame slot * W * H + pixel (below 4 * 2^30: what fits the card)
    int job;                // the ray's: job-table entry
    f4 dir;                 // the ray's: its direction, w = 0
    // of a bounce ray: pdf and lobe probability, or, off a specular surface,
    // the index-of-refraction factor and the direction's w; of a shadow ray:
    // light pdf and lobe probability; of a MIS ray also the BRDF's pdf
    float a, b, c;
    f4 hp, hn, rd, tp, direct, indirect, ls;
};

__device__ __forceinline__ void write_sample(const DevJob& J, uint32_t sample, f4 c)
{
    if (any_nan(c)) c = mk(kPinkR, kPinkG, kPinkB, 1.0f);     // udpt.cl:193-194
    J.samples[sample] = st4(c);
}

// The ray's w carries the path's job-table entry: the trace kernels look
// the scene up through it.
__device__ __forceinline__ Out make_ray(int kind, f4 o, f4 d, float tmax, int job)
{
    Out r;
    r.kind = kind;
    r.o_t = make_float4(o.x, o.y, o.z, tmax);
    r.d_p = make_float4(d.x, d.y, d.z, __int_as_float(job));
    return r;
}

template <bool NT>
__device__ __forceinline__ float4 rec_load(const float4* p)
{
    if constexpr (NT) return nt_load(p);
    else return *p;
}

// The record a step reads; dp: the pending ray's second half.  The shade pass
// is bound by memory traffic, so a record holds nothing that the ray or the
// state already says: the ray's direction and job are read from the queue, a
// new path has no fields but M0, and the first vertex's constants (half of
// all steps are there) are not stored.  What every later state uses is loaded
// without waiting for the state, the rest once it is known.
template <bool NT>
__device__ __forceinline__ void load_rec(const PathRecs& I, uint32_t ri, float4 dp, Rec& R, bool primary)
{
    using F = PathRecs;
    const float4 m0 = rec_load<NT>(I.f(F::M0, ri));
    R.m0 = make_int4(__float_as_int(m0.x), __float_as_int(m0.y), __float_as_int(m0.z), __float_as_int(m0.w));
    R.dir = mk(dp.x, dp.y, dp.z, 0.0f);
    R.job = __float_as_int(dp.w);
    R.hp = R.hn = R.rd = R.direct = R.indirect = R.ls = mk(0, 0, 0, 0);
    R.tp = mk(1, 1, 1, 1);
    R.a = R.b = R.c = 0;
    if (!primary) {
        const float4 m1 = rec_load<NT>(I.f(F::M1, ri));
        R.sample = __float_as_uint(m1.x);
        R.a = m1.y; R.b = m1.z; R.c = m1.w;
        R.hp = ld(rec_load<NT>(I.f(F::HP, ri)));
        R.hn = ld(rec_load<NT>(I.f(F::HN, ri)));
        R.rd = ld(rec_load<NT>(I.f(F::RD, ri)));
    }
    const int code = R.m0.y & ST_MASK;
    if (code == ST_PRIMARY) {
        R.sample = (uint32_t)R.m0.z;
        R.m0.z = 0;
    } else {
        if (R.m0.z > 0) {
            R.tp = ld(rec_load<NT>(I.f(F::TP, ri)));
            R.indirect = ld(rec_load<NT>(I.f(F::INDIRECT, ri)));
        }
        if (R.m0.z > 0 || code == ST_BOUNCE) R.direct = ld(rec_load<NT>(I.f(F::DIRECT, ri)));
        if (code == ST_NEE_MIS) R.ls = ld(rec_load<NT>(I.f(F::LS, ri)));
    }
}

// The record beside a ray just made: what the next step's state uses.
__device__ __forceinline__ void store_rec(const PathRecs& O, uint32_t ri, const Rec& R)
{
    using F = PathRecs;
    nt_store(O.f(F::M0, ri), make_float4(__int_as_float(R.m0.x), __int_as_float(R.m0.y), __int_as_float(R.m0.z),
                                         __int_as_float(R.m0.w)));
    nt_store(O.f(F::M1, ri), make_float4(__uint_as_float(R.sample), R.a, R.b, R.c));
    nt_store(O.f(F::HP, ri), st4(R.hp));
    nt_store(O.f(F::HN, ri), st4(R.hn));
    nt_store(O.f(F::RD, ri), st4(R.rd));
    const int code = R.m0.y & ST_MASK;
    if (R.m0.z > 0) {
        nt_store(O.f(F::TP, ri), st4(R.tp));
        nt_store(O.f(F::INDIRECT, ri), st4(R.indirect));
    }
    if (R.m0.z > 0 || code == ST_BOUNCE) nt_store(O.f(F::DIRECT, ri), st4(R.direct));
    if (code == ST_NEE_MIS) nt_store(O.f(F::LS, ri), st4(R.ls));
}

// The result of a path's ray in the results arrays, read when a step needs
// it.
struct QueueResult {
    const float4* hit_at;
    const int32_t* occ_at;
    uint32_t i;
    __device__ __forceinline__ float4 hit() const { return nt_load(hit_at + i); }
    __device__ __forceinline__ int occ() const { return occ_at[i]; }
};

// One shade step of the path whose record is R and whose ray's result is
// `res`; R is updated in place for the ray the step makes.  The ray whose
// result arrived is rebuilt, bit for bit as it was made, from its direction
// and the path state: a camera ray starts at the camera's eye (createRay,
// udpt.cl:236), a bounce ray at hp + nd * EPSILON along the bounce direction
// nd (udpt.cl:766, 906, 945).  (Sampled directions have w = 0, or are NaN in
// every component; a specular one's w is kept, see Rec.)
// `tab`: where the path's job and scene are found (JobTables or OneJob).
template <bool CAP, int LM, typename TAB, typename RES>
__device__ __forceinline__ Out advance(const TAB& tab, const DevCapture& cap, const RES& res, Rec& R,
                                       const LdsScene& lds)
{
    const int4 m0 = R.m0;
    const int jid = R.job;
    const DevJob& J = tab.job(jid);
    const yn_render_params& RP = J.p;
    const int sid = (m0.y >> SCENE_SHIFT) & 0xff;
    const DevScene& S = tab.scene(sid);                                // loaded beside J, not after it
    // LM: materials and light in LDS, the launch's one scene's (1) or every scene's (2)
    auto mat_of = [&](int id) {
        return LM == 1 ? load_mat(lds.mats, id) : LM == 2 ? load_mat(lds.mats, S.mat_base + id) : load_mat(S.mats, id);
    };
    auto& L = light_of<LM>(S.light, lds, sid);
    const bool on = RP.oren_nayar != 0;
    const bool fix = RP.fix_mis != 0;

    int st = m0.y;
    int code = st & ST_MASK;
    uint32_t seed = (uint32_t)m0.x;
    const uint32_t pix = R.sample;      // in frame slot 0, the only one captured
    const bool cap_on = CAP && cap.prim_tri != nullptr && pix < (uint32_t)(J.W * J.H);

    int vmat = m0.w;                    // material of the path's current vertex
    f4& hp = R.hp;
    f4& hn = R.hn;
    f4& rd = R.rd;
    f4& tp = R.tp;
    f4& direct = R.direct;
    f4& indirect = R.indirect;
    bool v_dirty = false;
    int bounce = m0.z;

    // NEE scratch
    f4 wi = mk(0, 0, 0, 0);
    float lpdf = 0.0f, nprob = 0.0f;
    f4 ls = mk(0, 0, 0, 0);
    f4 em = mk(0, 0, 0, 0);
    f4 nee_res = mk(0, 0, 0, 0);
    int occ = 0;

    enum Step { S_NEE_START, S_NEE_SHADOW, S_NEE_MIS, S_NEE_DONE, S_BOUNCE_SAMPLE, S_FINISH, S_FINISH_CONST };
    Step step;
    f4 const_color = mk(0, 0, 0, 0);

    if (code == ST_PRIMARY) {
        float4 h = res.hit();
        int htri = __float_as_int(h.y);
        if (cap_on) {
            cap.prim_tri[pix] = htri;
            cap.prim_light[pix] = (htri < 0 && (st & F_LCAND)) ? 0 : -1;
            cap.prim_t[pix] = h.x;
        }
        f4 d = R.dir;
        if (htri < 0) {
            if (st & F_LCAND) {     // udpt.cl:440-446
                const_color = dot(d, ld(L.normal)) < 0 ? mk(1, 1, 1, 1) : mk(0.1f, .1f, .1f, 1);
            } else {
                const_color = mk(RP.background[0], RP.background[1], RP.background[2], RP.background[3]);
            }
            step = S_FINISH_CONST;
        } else {
            f4 o = mk(J.cam.r1.w, J.cam.r2.w, J.cam.r3.w, 1.0f);
            vmat = tri_material(S.tri_shade, htri);
            hp = o + d * h.x;
            hn = shade_normal(S.tri_shade, htri, h.z, h.w);
            rd = d;
            tp = mk(1, 1, 1, 1);
            direct = mk(0, 0, 0, 0);
            indirect = mk(0, 0, 0, 0);
            v_dirty = true;
            bounce = 0;
            Mat m = mat_of(vmat);
            if (!m.spec) { st |= F_DIRECT; step = S_NEE_START; }
            else { step = S_BOUNCE_SAMPLE; }
        }
    } else {
        if (code == ST_NEE_SH) {
            occ = res.occ();
            step = S_NEE_SHADOW;
        } else if (code == ST_NEE_MIS) {
            occ = res.occ();
            step = S_NEE_MIS;
        } else {   // ST_BOUNCE: extension result (udpt.cl:488-529)
            float4 h = res.hit();
            int htri = __float_as_int(h.y);
            Mat m = mat_of(vmat);
            f4 nd = R.dir;
            if (m.spec) nd.w = R.b;
            if (htri < 0) {
                if ((st & F_LCAND) && m.spec) indirect = indirect + tp * ld(L.ke);
                step = S_FINISH;
            } else {
                f4 o = hp + nd * kEps;
                f4 nhp = o + nd * h.x;
                f4 nhn = shade_normal(S.tri_shade, htri, h.z, h.w);
                const int nmat = tri_material(S.tri_shade, htri);
                Mat nm = mat_of(nmat);
                indirect = indirect + tp * nm.ke;
                if (m.spec) tp = tp * R.a;
                else
                    tp = ((tp * eval_brdf(m, nd, -rd, hp, hn, (st & F_BGLOSSY) != 0, R.b, on, false)) *
                          fmaxf(dot(nd, hn), 0.0f)) / R.a;
                step = S_NEE_START;
                if (bounce > RP.rr_threshold) {    // udpt.cl:514-523
                    float pr = fminf(luminance(tp), 0.95f);
                    float r = next_rand(seed);
                    if (r >= pr) step = S_FINISH;
                    else tp = tp * (1 / pr);
                }
                if (step != S_FINISH) {
                    v_dirty = true;
                    vmat = nmat;
                    hp = nhp;
                    hn = nhn;
                    rd = nd;
                    bounce++;
                    st &= ~F_DIRECT;
                    if (nm.spec) step = S_BOUNCE_SAMPLE;
                }
            }
        }
    }

    Out out;
    bool ended = false;
    // The steps only ever move forward (NEE start, shadow, MIS, done, bounce
    // sample, finish), so they run as one forward sequence: a step that
    // hands over sets `step` to a later one and leaves its block, a step that
    // makes a ray jumps past the rest.  Without a loop back-edge, values of
    // one step are not kept live through the others.
    if (step == S_NEE_START) do {   // evaluateDirectLighting (udpt.cl:535-555)
        Mat m = mat_of(vmat);
        em = m.ke;
        f4 wraw;
        if (!sample_lights(L, hp, hn, seed, lpdf, wraw) || lpdf <= 0.0f) { nee_res = em; step = S_NEE_DONE; break; }
        float len = length(wraw);
        len -= kEps * 1.5f;
        wi = normalize(wraw);
        bool glossy = false;
        nprob = 0.0f;
        if (fix) {
            glossy = sample_glossy_pdf(m, seed, nprob, false);
            if (nprob == 0.0f) { nee_res = em; step = S_NEE_DONE; break; }
            st = glossy ? (st | F_NGLOSSY) : (st & ~F_NGLOSSY);
        }
        f4 so = hp + wi * kEps;
        float tq;
        if (cap_on && (st & F_DIRECT) && !(st & F_CAPSH)) {
            cap.shadow_o[pix] = make_float4(so.x, so.y, so.z, len);
            cap.shadow_d[pix] = make_float4(wi.x, wi.y, wi.z, 1.0f);
        }
        if (quad_hit(L, so, wi, len, tq)) { occ = 1; step = S_NEE_SHADOW; break; }
        R.a = lpdf;
        R.b = nprob;
        st = (st & ~ST_MASK) | ST_NEE_SH;
        out = make_ray(2, so, wi, len, jid);
        goto steps_done;
    } while (0);
    if (step == S_NEE_SHADOW) do {  // udpt.cl:557-565 and the MIS light weight
        if (code == ST_NEE_SH) {
            wi = R.dir;
            lpdf = R.a;
            nprob = R.b;
            code = ST_DONE;     // consumed
        }
        if (cap_on && (st & F_DIRECT) && !(st & F_CAPSH)) { cap.shadow_occ[pix] = occ; st |= F_CAPSH; }
        Mat m = mat_of(vmat);
        em = m.ke;
        f4 w_o = -rd;
        bool glossy = fix ? ((st & F_NGLOSSY) != 0) : false;
        ls = mk(0, 0, 0, 0);
        if (!occ) {
            if (!fix) {
                glossy = sample_glossy_pdf(m, seed, nprob, false);
                if (nprob == 0.0f) { nee_res = em; step = S_NEE_DONE; break; }
            }
            ls = (eval_brdf(m, wi, w_o, hp, hn, glossy, nprob, on, false) * ld(L.ke)) * fmaxf(dot(wi, hn), 0.0f);
            ls = ls * (1 / lpdf);
        }
        if (!RP.mis) { nee_res = ls + em; step = S_NEE_DONE; break; }
        float bpdf = glossy ? phong_pdf(m, wi, w_o, hn) : cos_pdf(wi, hn);
        float mw = power_heuristic(lpdf, lpdf, bpdf);
        ls = ls * mw;
        f4 bd = glossy ? phong_sample(m, bpdf, w_o, hp, hn, seed, false) : cosine_sample(bpdf, hp, hn, seed);
        if (bpdf <= 0.0f) { nee_res = ls + em; step = S_NEE_DONE; break; }
        f4 bo = hp + bd * kEps;
        float tq;
        if (!quad_hit(L, bo, bd, INFINITY, tq)) { nee_res = ls + em; step = S_NEE_DONE; break; }
        st = glossy ? (st | F_NGLOSSY) : (st & ~F_NGLOSSY);
        R.ls = ls;
        R.a = lpdf;
        R.b = nprob;
        R.c = bpdf;
        st = (st & ~ST_MASK) | ST_NEE_MIS;
        out = make_ray(2, bo, bd, tq, jid);
        goto steps_done;
    } while (0);
    if (step == S_NEE_MIS) do {     // udpt.cl:599-607
        Mat m = mat_of(vmat);
        em = m.ke;
        ls = R.ls;
        if (occ) { nee_res = ls + em; step = S_NEE_DONE; break; }
        f4 bd = R.dir;
        float bpdf = R.c;
        lpdf = R.a;
        nprob = R.b;
        bool glossy = (st & F_NGLOSSY) != 0;
        float mw = power_heuristic(bpdf, lpdf, bpdf);
        f4 bs = (eval_brdf(m, bd, -rd, hp, hn, glossy, nprob, on, false) * ld(L.ke)) * fmaxf(dot(bd, hn), 0.0f);
        bs = bs * (mw / bpdf);
        nee_res = (ls + bs) + em;
        step = S_NEE_DONE;
        break;
    } while (0);
    if (step == S_NEE_DONE) do {
        if (st & F_DIRECT) direct = nee_res;
        else indirect = indirect + tp * nee_res;
        step = S_BOUNCE_SAMPLE;
        break;
    } while (0);
    if (step == S_BOUNCE_SAMPLE) do {   // udpt.cl:458-487
        if (!RP.gi || bounce >= RP.max_bounces) { step = S_FINISH; break; }
        Mat m = mat_of(vmat);
        float pdf = 1.0f, bprob = 0.0f, ior = 1.0f;
        bool glossy = false;
        f4 nd;
        if (m.spec) nd = fresnel_sample(m, hn, -rd, ior, seed);
        else {
            glossy = sample_glossy_pdf(m, seed, bprob, false);
            if (bprob == 0.0f) { step = S_FINISH; break; }
            nd = glossy ? phong_sample(m, pdf, -rd, hp, hn, seed, false) : cosine_sample(pdf, hp, hn, seed);
        }
        if (pdf <= 0.0f) { step = S_FINISH; break; }
        f4 no = hp + nd * kEps;
        float tq, tmax = INFINITY;
        st &= ~F_LCAND;
        if (quad_hit(L, no, nd, INFINITY, tq)) { tmax = tq; st |= F_LCAND; }
        st = glossy ? (st | F_BGLOSSY) : (st & ~F_BGLOSSY);
        R.a = m.spec ? ior : pdf;
        R.b = m.spec ? nd.w : bprob;
        st = (st & ~ST_MASK) | ST_BOUNCE;
        out = make_ray(1, no, nd, tmax, jid);
        goto steps_done;
    } while (0);
    if (step == S_FINISH) do {
        write_sample(J, R.sample, direct + indirect);
        st = ST_DONE;
        ended = true;
        goto steps_done;
    } while (0);
    if (step == S_FINISH_CONST) { write_sample(J, R.sample, const_color); st = ST_DONE; ended = true; }
steps_done:
    if (out.kind == 0 && !ended) {   // unreachable by construction; never leave a path hanging
        write_sample(J, R.sample, mk(NAN, NAN, NAN, NAN));
        st = ST_DONE;
    }
    out.done = out.kind == 0;
    out.job = jid;
    R.m0 = make_int4((int)seed, st, v_dirty ? bounce : m0.z, v_dirty ? vmat : m0.w);
    return out;
}

}  // namespace yune
