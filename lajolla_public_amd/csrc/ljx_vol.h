// Volumetric path tracing on the wavefront loop (homogeneous and
// heterogeneous media).
//
// lajolla's vol_path_tracing is a homework stub returning zero
// (src/vol_path_tracing.h:59-64); this follows the handout's final
// algorithm (handouts/homework2.tex): homogenised free flight with one-sample
// spectral MIS over RGB (:713-758), next-event estimation with ratio tracking
// through index-matched surfaces (:770-812, :460-507), update_medium
// (:402-409), the MIS caches dir_pdf / nee_p_cache / multi_trans_pdf /
// never_scatter (:505-557), Russian roulette from rr_depth (:331-400), and the
// max_null_collisions cap (:760-764).
//
//   k_vol_flight  free flight (delta tracking) in scenes with grid media
//   k_vol_event   whether a path scatters before its hit, in scenes without
//   k_sort_*      orders the paths by what happens to them
//   k_vol_shade   by event: phase or BSDF sampling, NEE light-point sampling,
//                 RR, emission with MIS, index-matched pass-through
//   k_vol_shadow  the NEE shadow walk: closest hits through index-matched
//                 surfaces with ratio tracking in every medium on the way
//
// All NEE draws come from a sub-stream seeded by one draw of the path stream
// (stream id path_stream ^ 0x5bd1e9955bd1e995), so the shadow kernel can
// consume them after the shade kernel has moved on.
#pragma once

#include "ljx_kernels.h"

#include <vector>

namespace ljx {

constexpr bool kVolpathEnabled = true;
constexpr uint64_t kNeeStreamXor = 0x5bd1e9955bd1e995ULL;
constexpr int kMaxShadowSegments = 256;

// sigma_t = sigma_s + sigma_a at p; a grid medium's two are its density times
// the albedo and times the rest, so theirs is the density itself
__device__ __forceinline__ D3 sigma_t_at(const MediumRec &m, D3 p) {
    if (m.type == 0) return m.sigma_s + m.sigma_a;
    return vol_lookup(m.density, p);
}
__device__ __forceinline__ D3 sigma_s_at(const MediumRec &m, D3 p) {
    D3 s, a;
    medium_sigmas(m, p, s, a);
    return s;
}

// exp(-maj t) per channel.  A grey majorant (every channel equal: grid
// media, whose sigma_t is the density alone) gives three identical
// exponentials, computed once.
__device__ __forceinline__ D3 maj_exp(D3 maj, bool grey, double t) {
    if (grey) {
        const double e = exp(-1.0 * maj.x * t);
        return D3{e, e, e};
    }
    return vexp(-1.0 * maj * t);
}

// update_medium (homework2.tex:402-409)
__device__ __forceinline__ int update_medium(D3 dir, const Vertex &v, int medium) {
    if (v.interior_medium_id != v.exterior_medium_id)
        return dot(dir, v.g.ng) > 0 ? v.exterior_medium_id : v.interior_medium_id;
    return medium;
}

// Free-flight sampling of one path in a medium (homework2.tex:745-769, delta
// tracking; its first draw picks the channel).  It is the first use of the
// path's stream in a bounce, so in scenes with grid media (long loops of
// null collisions) k_vol_flight runs it for every path of the queue before
// k_vol_shade, which takes over the stream state; in homogeneous media (one
// collision) k_vol_event runs it to learn the outcome and k_vol_shade again,
// which is cheaper than 128 bytes of FP64 results written and read.
struct Flight {
    D3 T, trans_dir_pdf;
    double accum_t;
    bool scatter;
};
template <bool GREY>
__device__ __forceinline__ D3 grey_or(D3 v) {
    return GREY ? D3{v.x, v.x, v.x} : v;
}
// The loop of free_flight, resumable one collision at a time.
struct FlightRun {
    const MediumRec *m;
    D3 org, dir, maj;
    double t_hit, max_maj;
    int ch, it;
    bool grey;
    Flight fl;
};
__device__ __forceinline__ void flight_begin(FlightRun &r, const DeviceScene &S, int medium, D3 org, D3 dir,
                                             double t_hit, uint64_t &st, uint64_t inc) {
    r.fl = Flight{{1, 1, 1}, {1, 1, 1}, 0.0, false};
    r.m = &S.media[medium];
    r.org = org;
    r.dir = dir;
    r.t_hit = t_hit;
    r.maj = medium_majorant(*r.m, org, dir, __builtin_huge_val());
    r.max_maj = maxc(r.maj);
    r.grey = r.maj.x == r.maj.y && r.maj.y == r.maj.z;
    const double u = pcg_double(st, inc);
    r.ch = min(max(int(u * 3), 0), 2);
    r.it = 0;
}
// GREY, here and in the shadow walk: every medium of the scene is a grid
// medium of one density channel, so the majorant, transmittance and pdfs of
// the three channels stay equal and only the first is computed (x); majorant
// over largest majorant, one there, drops out.  A third of the FP64 lookups,
// divisions and state: the 128^3 smoke grid's flights and walks are bound by
// that arithmetic and by the waves per SIMD its registers allow (71 -> 37 and
// 87 -> 45 ms at 768x576, 64 samples, at four waves instead of three and three
// instead of two).
// One pass of the loop; true when the flight has ended.  decided: whether the
// path collides before its hit, where an earlier kernel has found that out (1
// or 0, else -1): two compilations of the comparison may round differently.
template <bool GREY = false>
__device__ __forceinline__ bool flight_step(FlightRun &r, const PathBufs &P, uint64_t &st, uint64_t inc,
                                            int decided = -1) {
    Flight &fl = r.fl;
    if constexpr (GREY) {
        const double maj = r.maj.x;
        if (maj <= 0) return true;
        if (r.it >= P.max_null) return true;
        const double t = -log(1 - pcg_double(st, inc)) / maj, dt = r.t_hit - fl.accum_t;
        fl.accum_t = fmin(fl.accum_t + t, r.t_hit);
        const bool collides = t < dt;
        const double e = exp(-1.0 * maj * (collides ? t : dt));
        fl.T.x *= e;
        fl.trans_dir_pdf.x *= e;
        if (!collides) return true;
        const double sig_t = vol_lookup_grey(r.m->density, r.org + fl.accum_t * r.dir);
        const double real_prob = sig_t / maj;
        if (pcg_double(st, inc) < real_prob) {
            fl.scatter = true;
            fl.T.x /= maj;
            fl.trans_dir_pdf.x *= real_prob;
            return true;
        }
        fl.T.x = fl.T.x * (maj - sig_t) / maj;
        fl.trans_dir_pdf.x *= 1.0 - real_prob;
        r.it++;
        return false;
    }
    const D3 maj = r.maj;
    const double max_maj = r.max_maj;
    const int ch = r.ch;
    const double mc = comp(maj, ch);
    if (mc <= 0) return true;
    if (r.it >= P.max_null) return true;
    const double t = -log(1 - pcg_double(st, inc)) / mc;
    const double dt = r.t_hit - fl.accum_t;
    fl.accum_t = fmin(fl.accum_t + t, r.t_hit);
    if (decided < 0 ? t < dt : decided > 0) {
        D3 sig_t = sigma_t_at(*r.m, r.org + fl.accum_t * r.dir);
        D3 real_prob = sig_t / maj;
        D3 e = maj_exp(maj, r.grey, t);
        if (pcg_double(st, inc) < comp(real_prob, ch)) {
            fl.scatter = true;
            fl.T = fl.T * e / max_maj;
            fl.trans_dir_pdf = fl.trans_dir_pdf * e * maj * real_prob / max_maj;
            return true;
        }
        D3 sig_n = maj - sig_t;
        fl.T = fl.T * e * sig_n / max_maj;
        fl.trans_dir_pdf = fl.trans_dir_pdf * e * maj * (1.0 - real_prob) / max_maj;
        r.it++;
        return false;
    }
    D3 e = maj_exp(maj, r.grey, dt);
    fl.T = fl.T * e;
    fl.trans_dir_pdf = fl.trans_dir_pdf * e;
    return true;
}
__device__ __forceinline__ Flight free_flight(const DeviceScene &S, const PathBufs &P, int medium, D3 org, D3 dir,
                                              double t_hit, uint64_t &st, uint64_t inc, int decided = -1) {
    FlightRun r;
    flight_begin(r, S, medium, org, dir, t_hit, st, inc);
    while (!flight_step<false>(r, P, st, inc, decided)) {
    }
    return r.fl;
}

// Distance to the surface a ray hit (infinite on a miss), from the vertex
// position the shading kernel computes.
template <bool SPH>
__device__ __forceinline__ double hit_distance(const DeviceScene &S, float4 h, D3 org, D3 dir) {
    const int slot = __float_as_int(h.w);
    if (slot < 0) return __builtin_huge_val();
    Vertex v = make_vertex<SPH>(S, slot, h.x, h.y, h.z, org, dir);
    return sqrt(dist2(org, v.pos));
}

// The bucket of a path: scattered in its medium, or the hit's (k_extend).
__device__ __forceinline__ uint8_t event_bucket(const DeviceScene &S, bool scatter, float4 hit) {
    const int slot = __float_as_int(hit.w);
    return uint8_t(scatter ? kBucketScatter : slot < 0 ? kBucketMiss : S.slot_bucket[slot]);
}
template <bool SPH>
__global__ __launch_bounds__(256) void k_vol_event(DeviceScene S, PathBufs P, int cur) {
    const uint32_t *q = cur ? P.extq1 : P.extq0;
    const int n = P.ctr[C_EXT + cur];
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const uint32_t pid = q[i];
        const float4 h = P.hit[pid];
        const int medium = P.medium[pid];
        bool scatter = false;
        if (medium >= 0) {
            const float4 ro = P.ray_o[pid], rd = P.ray_d[pid];
            const D3 org = f3d(ro), dir = f3d(rd);
            uint64_t st = P.rng[pid];
            const uint64_t inc = pcg_inc(slot_info(P, int(pid)).stream());
            scatter = free_flight(S, P, medium, org, dir, hit_distance<SPH>(S, h, org, dir), st, inc).scatter;
        }
        P.key[i] = event_bucket(S, scatter, h);
    }
}

// Free flight for the queue's paths that are in a medium, in a kernel small
// enough for three waves per SIMD (GREY: four).  The loops' lengths vary
// widely between paths, so a lane whose flight ended (or whose path is in no
// medium) takes its next path as soon as kFlightRefill lanes of its wave are
// idle rather than waiting for the wave's longest flight.
constexpr int kFlightRefill = 16;
template <bool SPH, bool GREY>
__global__ __launch_bounds__(256) void k_vol_flight(DeviceScene S, PathBufs P, int cur) {
    const uint32_t *q = cur ? P.extq1 : P.extq0;
    FlightRun r;
    uint64_t st = 0, inc = 0;
    uint32_t pid = 0;
    int i = 0;
    bool busy = false, fin = false;
    FeedRange range;
    range.start(P.ctr + C_FEED_FLIGHT, P.ctr[C_EXT + cur], kFeedTickets);
    while (true) {
        const uint64_t idle = __ballot(!busy);
        const int nidle = __popcll(idle);
        if ((nidle >= kFlightRefill && !range.done) || nidle == 64) {
            if (fin) {
                P.rng[pid] = st;
                const D3 T = grey_or<GREY>(r.fl.T), p = grey_or<GREY>(r.fl.trans_dir_pdf);
                P.vf_t[pid] = make_double4(T.x, T.y, T.z, r.fl.accum_t);
                P.vf_p[pid] = make_double4(p.x, p.y, p.z, r.fl.scatter ? 1.0 : 0.0);
                P.key[i] = event_bucket(S, r.fl.scatter, P.hit[pid]);
                fin = false;
            }
            const int k = range.take(!busy, [&](int j) {
                const uint32_t p = q[j];
                const bool in_medium = P.medium[p] >= 0;
                if (!in_medium) P.key[j] = event_bucket(S, false, P.hit[p]);
                return in_medium;
            });
            if (k >= 0) {
                i = k;
                pid = q[i];
                const float4 ro = P.ray_o[pid], rd = P.ray_d[pid];
                const D3 org = f3d(ro), dir = f3d(rd);
                st = P.rng[pid];
                inc = pcg_inc(slot_info(P, int(pid)).stream());
                flight_begin(r, S, P.medium[pid], org, dir, hit_distance<SPH>(S, P.hit[pid], org, dir), st, inc);
                busy = true;
            }
            if (__ballot(busy) == 0) break;
        }
        if (busy && flight_step<GREY>(r, P, st, inc)) {
            busy = false;
            fin = true;
        }
    }
}

// What happens to a path at the end of its flight, by bucket.  One kernel for
// all of them ran with 30 of 64 lanes active, one wave per SIMD and every
// field of the state read and written whatever the event; by event the kernels
// move only what theirs needs (scattering: no hit, vertex, radiance or MIS
// caches) and nothing for paths that left the scene: 126 -> 75 ms for the
// 1024x1024 128-sample nested media with k_vol_event and the sort.
constexpr int kEvScatter = 0, kEvSurface = 1, kEvPass = 2;
template <bool SPH, int DMT, int EV>
__device__ __forceinline__ void vol_shade(const DeviceScene &S, const PathBufs &P, uint32_t pid, bool &push_ext,
                                          bool &push_sh, float4 &sh_o, float4 &sh_d, float4 &sh_c, float4 &sh_x) {
    constexpr bool scatter = EV == kEvScatter, ENV = DMT == kMtEnv;
    push_ext = false;
    push_sh = false;
    float4 ro = P.ray_o[pid], rd = P.ray_d[pid];
    D3 org = f3d(ro), dir = f3d(rd);
    int bounces = P.depth[pid];
    // a path at the last depth may still reach a light
    const bool last = P.max_depth != -1 && bounces == P.max_depth - 1;
    if (scatter && last) return;
    uint64_t st = P.rng[pid];
    const uint64_t stream = slot_info(P, int(pid)).stream();
    uint64_t inc = pcg_inc(stream);
    float4 tp4 = P.tp[pid];
    D3 tp{tp4.x, tp4.y, tp4.z};
    double eta_scale = tp4.w;
    int medium = P.medium[pid];

    Vertex v;
    if constexpr (!scatter) {
        const float4 h = P.hit[pid];
        v = make_vertex<SPH>(S, __float_as_int(h.w), h.x, h.y, h.z, org, dir);
    }
    D3 p_scatter = org, trans_dir_pdf{1, 1, 1};
    if (medium >= 0) {
        D3 T;
        double accum_t;
        if (P.vol_flight) {
            // the free flight k_vol_flight sampled (it advanced the stream state)
            const double4 ft = P.vf_t[pid], fp = P.vf_p[pid];
            T = D3{ft.x, ft.y, ft.z};
            trans_dir_pdf = D3{fp.x, fp.y, fp.z};
            accum_t = ft.w;
        } else {
            const Flight fl = free_flight(S, P, medium, org, dir,
                                          scatter ? __builtin_huge_val() : sqrt(dist2(org, v.pos)), st, inc, scatter);
            T = fl.T;
            trans_dir_pdf = fl.trans_dir_pdf;
            accum_t = fl.accum_t;
        }
        if (scatter) p_scatter = org + accum_t * dir;
        tp = tp * T / avgc(trans_dir_pdf);
    }
    if constexpr (!scatter) {
        if (v.area_light_id >= 0) {
            const LightRec &l = S.lights[v.area_light_id];
            LightPoint lp{v.pos, v.g.ng};
            D3 add = tp * light_emission<ENV>(l, -dir, lp);
            const float4 mt = P.mtp[pid];
            if (mt.w == 0.f) {  // some vertex of the path scattered
                const float4 nc = P.nee_c[pid];
                const D3 nee_p_cache{nc.x, nc.y, nc.z};
                const D3 multi_trans_pdf = D3{mt.x, mt.y, mt.z} * trans_dir_pdf;
                double pdf_nee = S.light_pmf[v.area_light_id] * pdf_light_point<SPH, ENV>(S, l, lp, nee_p_cache);
                double G = fabs(dot(dir, v.g.ng)) / dist2(nee_p_cache, v.pos);
                double dp = double(nc.w) * avgc(multi_trans_pdf) * G;
                add = add * ((dp * dp) / (dp * dp + pdf_nee * pdf_nee));
            }
            const float4 r4 = P.rad[pid];
            P.rad[pid] = make_float4(float(r4.x + add.x), float(r4.y + add.y), float(r4.z + add.z), 0.f);
        }
        if (last) return;
    }
    if constexpr (EV == kEvPass) {
        // index-matched interface: continue straight through
        const float4 mt = P.mtp[pid];
        const D3 multi_trans_pdf = D3{mt.x, mt.y, mt.z} * trans_dir_pdf;
        P.ray_o[pid] = make_float4(float(v.pos.x), float(v.pos.y), float(v.pos.z), float(S.eps));
        P.ray_d[pid] = make_float4(float(dir.x), float(dir.y), float(dir.z), __builtin_huge_valf());
        P.depth[pid] = bounces + 1;
        if (!P.vol_flight) P.rng[pid] = st;
        P.medium[pid] = update_medium(dir, v, medium);
        P.tp[pid] = make_float4(float(tp.x), float(tp.y), float(tp.z), float(eta_scale));
        P.mtp[pid] = make_float4(float(multi_trans_pdf.x), float(multi_trans_pdf.y), float(multi_trans_pdf.z), mt.w);
        push_ext = true;
        return;
    } else {
        // constant materials are read in place; the runtime-dispatch kernel, which
        // also takes textured ones, works on a copy with the textures evaluated
        MatRec mat_tex;
        if constexpr (EV == kEvSurface && DMT < 0) {
            mat_tex = S.materials[v.material_id];
            if (mat_tex.textured) resolve_textures(S, mat_tex, v.tu, v.tv, 0.0);
        }
        const MatRec &mat = DMT < 0 ? mat_tex : S.materials[scatter ? 0 : v.material_id];
        D3 dir_view = -dir;
        // NEE sub-stream
        uint32_t k = pcg_next(st, inc);
        uint64_t nstream = stream ^ kNeeStreamXor;
        uint64_t ninc = pcg_inc(nstream);
        uint64_t nst = pcg_init_state(nstream, uint64_t(k));
        const D3 pos = scatter ? p_scatter : v.pos;
        double lu0 = pcg_double(nst, ninc), lu1 = pcg_double(nst, ninc);
        double lw = pcg_double(nst, ninc), sw = pcg_double(nst, ninc);
        D3 sigma_s{0, 0, 0};
        if (scatter) sigma_s = sigma_s_at(S.media[medium], p_scatter);
        if (S.num_lights > 0) {
            int lid = sample_cdf_guided(S.light_cdf, S.num_lights, lw, S.light_guide, S.light_guide_m);
            const LightRec &l = S.lights[lid];
            LightPoint lp = sample_light_point<SPH, ENV>(S, l, pos, lu0, lu1, sw);
            D3 dir_light = normalize(lp.pos - pos);
            double G = fmax(-dot(dir_light, lp.n), 0.0) / dist2(pos, lp.pos);
            double pdf_nee = S.light_pmf[lid] * pdf_light_point<SPH, ENV>(S, l, lp, pos);
            if (G > 0 && pdf_nee > 0) {
                D3 f;
                double pdf_f;
                D3 pre = tp;
                if constexpr (scatter) {
                    double pv = phase_value(S.media[medium], dir_view, dir_light);
                    f = D3{pv, pv, pv};
                    pdf_f = pv;
                    pre = pre * sigma_s;
                } else {
                    f = bsdf_eval<DMT>(mat, dir_view, dir_light, v.g);
                    pdf_f = bsdf_pdf<DMT>(mat, dir_view, dir_light, v.g);
                }
                D3 L = light_emission<ENV>(l, -dir_light, lp);
                D3 K = pre * G * f * L;
                if (K.x != 0 || K.y != 0 || K.z != 0) {
                    push_sh = true;
                    sh_o = make_float4(float(pos.x), float(pos.y), float(pos.z), __int_as_float(medium));
                    sh_d = make_float4(float(lp.pos.x), float(lp.pos.y), float(lp.pos.z), __int_as_float(bounces));
                    sh_c = make_float4(float(K.x), float(K.y), float(K.z), __int_as_float(int(pid)));
                    sh_x = make_float4(float(pdf_nee), float(pdf_f * G), __uint_as_float(uint32_t(nst)),
                                       __uint_as_float(uint32_t(nst >> 32)));
                }
            }
        }
        double dir_pdf;
        D3 next_dir;
        float tnear;
        if constexpr (scatter) {
            const MediumRec &m = S.media[medium];
            double u0 = pcg_double(st, inc), u1 = pcg_double(st, inc);
            next_dir = phase_sample(m, dir_view, u0, u1);
            dir_pdf = phase_value(m, dir_view, next_dir);
            if (dir_pdf <= 0) return;
            tp = tp * (D3{dir_pdf, dir_pdf, dir_pdf} / dir_pdf) * sigma_s;
            tnear = 0.f;
        } else {
            double u0 = pcg_double(st, inc), u1 = pcg_double(st, inc), w = pcg_double(st, inc);
            BsdfSample bs = bsdf_sample<DMT>(mat, dir_view, v.g, u0, u1, w);
            if (!bs.valid) return;
            if (bs.eta != 0) eta_scale /= (bs.eta * bs.eta);
            D3 f = bsdf_eval<DMT>(mat, dir_view, bs.dir, v.g);
            dir_pdf = bsdf_pdf<DMT>(mat, dir_view, bs.dir, v.g);
            if (dir_pdf <= 0) return;
            tp = tp * f / dir_pdf;
            medium = update_medium(bs.dir, v, medium);
            next_dir = bs.dir;
            tnear = float(S.eps);
        }
        if (bounces >= P.rr_depth) {
            double rr = fmin(maxc((1 / eta_scale) * tp), 0.95);
            if (pcg_double(st, inc) > rr) return;
            tp = tp / rr;
        }
        // a path that goes on; an ended one's state is not read again
        push_ext = true;
        P.ray_o[pid] = make_float4(float(pos.x), float(pos.y), float(pos.z), tnear);
        P.ray_d[pid] = make_float4(float(next_dir.x), float(next_dir.y), float(next_dir.z), __builtin_huge_valf());
        P.depth[pid] = bounces + 1;
        P.rng[pid] = st;
        if (!scatter) P.medium[pid] = medium;
        P.tp[pid] = make_float4(float(tp.x), float(tp.y), float(tp.z), float(eta_scale));
        P.nee_c[pid] = make_float4(float(pos.x), float(pos.y), float(pos.z), float(dir_pdf));
        P.mtp[pid] = make_float4(1.f, 1.f, 1.f, 0.f);
    }
}

// Surfaces: DMT is the material type of the kernel's bucket, -1 for the
// buckets from kVolTyped on, or kMtEnv for all of them.
constexpr int kVolTyped = 3;
template <bool SPH, int DMT, int EV>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(EV == kEvSurface && DMT >= 0 && !SPH ? 2 : 1))) void k_vol_shade(DeviceScene S, PathBufs P, int cur) {
    constexpr int first = EV == kEvScatter ? kBucketScatter : EV == kEvPass ? kBucketNoMat : DMT >= 0 ? DMT : DMT == kMtEnv ? 0 : kVolTyped;
    constexpr int end = EV == kEvSurface && DMT < 0 ? kBucketScatter : first + 1;
    const int j0 = bucket_start(P, first), j1 = bucket_start(P, end);
    for (int j = j0 + blockIdx.x * blockDim.x + threadIdx.x; j < j1; j += gridDim.x * blockDim.x) {
        const uint32_t pid = P.order[j];
        bool pe, ps;
        float4 so, sd, sc, sx;
        vol_shade<SPH, DMT, EV>(S, P, pid, pe, ps, so, sd, sc, sx);
        if (pe) P.alive[pid] = 1;
        if constexpr (EV != kEvPass) {
            // the shadow ray takes its path's place in the order (shade_queue)
            P.sh_occ[j] = ps ? uint8_t(0) : kShNone;
            if (ps) {
                P.sh_o[j] = so;
                P.sh_d[j] = sd;
                P.sh_c[j] = sc;
                P.sh_x[j] = sx;
            }
        }
    }
}

// NEE segments, first pass: one any-hit query per segment that passes
// through index-matched boundaries.  A surface with a material anywhere on
// the way to the light blocks the sample whatever the media, so this
// settles most segments before the FP64 walk: sh_occ = 1 when such a surface
// blocks the segment, 2 when it crosses index-matched boundaries only (the
// walk takes closest hits through them), 0 when nothing lies on it (the
// walk's first closest-hit query, over the same interval, would find
// nothing).  Traversal only, so it runs at the any-hit kernel's occupancy
// and with its lane refill; the walk's FP64 state would cut that to two
// waves per SIMD.  Triangle-only scenes cap it at eight waves per SIMD (64
// registers, a 16-byte spill).
template <bool STATS, bool SPH>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(SPH ? 1 : 8))) void k_vol_occlude(DeviceScene S, PathBufs P) {
    __shared__ int stack[kStackLds * 256];
    const TraceScene ts{S.qnodes, S.prims, S.spheres, S.slot_passthru};
    const int gtid = blockIdx.x * blockDim.x + threadIdx.x;
    const int stride = gridDim.x * blockDim.x;
    int *spill = P.spill + gtid;
    uint32_t nn = 0, np = 0;
    Tracer<true, STATS, SPH, true> tr;
    bool busy = false, fin = false;
    FeedRange range;
    range.start(P.ctr + C_FEED_SHADOW, bucket_start(P, kBucketMiss));
    int i = 0, rays = 0;
    while (true) {
        const uint64_t idle = __ballot(!busy);
        const int nidle = __popcll(idle);
        if ((nidle >= kShadowRefill && !range.done) || nidle == 64) {
            if (fin) P.sh_occ[i] = tr.found ? 1 : (tr.passed ? 2 : 0);
            fin = false;
            const int k = range.take(!busy, [&](int j) { return P.sh_occ[j] != kShNone; });
            if (k >= 0) {
                i = k;
                const float4 so = P.sh_o[i], sd = P.sh_d[i];
                const D3 p{so.x, so.y, so.z}, pp{sd.x, sd.y, sd.z};
                const D3 dir_light = normalize(pp - p);
                const double dl = sqrt(dist2(p, pp));
                tr.start(float(p.x), float(p.y), float(p.z), float(dir_light.x), float(dir_light.y),
                         float(dir_light.z), float(S.eps), float((1 - S.eps) * dl));
                busy = true;
            }
            const int now = __popcll(__ballot(busy));
            rays += now - (64 - nidle);
            if (now == 0) break;
        }
        if (busy) {
            if (S.num_nodes == 0 || tr.step(ts, stack + threadIdx.x, blockDim.x, spill, stride, nn, np)) {
                busy = false;
                fin = true;
            }
        }
    }
    if (S.num_nodes > 0 && __lane_id() == 0) P.wave_stat[gtid >> 6] += (unsigned long long)rays;
    if (STATS) {
        atomicAdd(&P.stat[S_SH_NODES], (unsigned long long)nn);
        atomicAdd(&P.stat[S_SH_PRIMS], (unsigned long long)np);
    }
}

// One NEE sample's walk towards the light: segments between index-matched
// boundaries, each with ratio tracking in its medium one collision at a time.
struct Walk {
    uint64_t nst, ninc;
    D3 p0, pp, dir;
    D3 T, p_nee, p_dir;
    D3 maj;
    double max_maj, next_t, accum_t;
    const MediumRec *m;
    int pid, bounces, medium, seg, shadow_bounces;
    int ch, it;
    int next_medium;   // medium beyond the boundary at the segment's end
    bool grey, crossings, hit, surface, blocked;
};
// Starts a segment: the boundary it ends at (only samples that cross
// boundaries have one) and its medium's majorant and channel.
template <bool STATS, bool SPH>
__device__ __forceinline__ void walk_segment(Walk &w, const DeviceScene &S, int *stack, int *spill, int stride,
                                             uint32_t &nn, uint32_t &np) {
    const double dl = sqrt(dist2(w.p0, w.pp));
    TraceHit h;
    w.hit = w.crossings && trace_ray<false, STATS, SPH>(TraceScene{S.qnodes, S.prims, S.spheres}, float(w.p0.x),
                                                        float(w.p0.y), float(w.p0.z), float(w.dir.x), float(w.dir.y),
                                                        float(w.dir.z), float(S.eps), float((1 - S.eps) * dl), stack,
                                                        blockDim.x, spill, stride, h, nn, np);
    w.next_t = dl;
    if (w.hit) {
        const Vertex v = make_vertex<SPH>(S, h.slot, h.t, h.u, h.v, w.p0, w.dir);
        w.next_t = sqrt(dist2(w.p0, v.pos));
        w.surface = v.material_id >= 0;
        w.next_medium = update_medium(w.dir, v, w.medium);
    }
    if (w.medium >= 0) {
        w.m = &S.media[w.medium];
        w.maj = medium_majorant(*w.m, w.p0, w.dir, (1 - S.eps) * dl);
        w.max_maj = maxc(w.maj);
        w.grey = w.maj.x == w.maj.y && w.maj.y == w.maj.z;
        const double u = pcg_double(w.nst, w.ninc);
        w.ch = min(max(int(u * 3), 0), 2);
        w.accum_t = 0;
        w.it = 0;
    }
}
// One collision of the segment's ratio tracking; true at the segment's end.
template <bool GREY>
__device__ __forceinline__ bool walk_collision(Walk &w, const PathBufs &P) {
    if (w.medium < 0) return true;
    if constexpr (GREY) {
        const double maj = w.maj.x;
        if (maj <= 0) return true;
        if (w.it >= P.max_null) return true;
        const double t = -log(1 - pcg_double(w.nst, w.ninc)) / maj, dt = w.next_t - w.accum_t;
        w.accum_t = fmin(w.accum_t + t, w.next_t);
        const bool collides = t < dt;
        const double e = exp(-1.0 * maj * (collides ? t : dt));
        w.T.x *= e;
        w.p_nee.x *= e;
        w.p_dir.x *= e;
        if (!collides) return true;
        const double sig_t = vol_lookup_grey(w.m->density, w.p0 + w.accum_t * w.dir);
        w.T.x = w.T.x * (maj - sig_t) / maj;
        w.p_dir.x *= 1.0 - sig_t / maj;
        w.it++;
        return w.T.x <= 0;
    }
    const D3 maj = w.maj;
    const double mc = comp(maj, w.ch);
    if (mc <= 0) return true;
    if (w.it >= P.max_null) return true;
    const double t = -log(1 - pcg_double(w.nst, w.ninc)) / mc;
    const double dt = w.next_t - w.accum_t;
    w.accum_t = fmin(w.accum_t + t, w.next_t);
    if (t < dt) {
        const D3 sig_t = sigma_t_at(*w.m, w.p0 + w.accum_t * w.dir);
        const D3 sig_n = maj - sig_t;
        const D3 e = maj_exp(maj, w.grey, t);
        w.T = w.T * e * sig_n / w.max_maj;
        w.p_nee = w.p_nee * e * maj / w.max_maj;
        const D3 real_prob = sig_t / maj;
        w.p_dir = w.p_dir * e * maj * (1.0 - real_prob) / w.max_maj;
        w.it++;
        return maxc(w.T) <= 0;
    }
    const D3 e = maj_exp(maj, w.grey, dt);
    w.T = w.T * e;
    w.p_nee = w.p_nee * e;
    w.p_dir = w.p_dir * e;
    return true;
}
// After a segment: true when the walk has ended.
__device__ __forceinline__ bool walk_advance(Walk &w, const PathBufs &P) {
    if (!w.hit) return true;
    if (w.surface) {
        w.blocked = true;
        return true;
    }
    w.shadow_bounces++;
    if (P.max_depth != -1 && w.bounces + w.shadow_bounces + 1 >= P.max_depth) {
        w.blocked = true;
        return true;
    }
    w.medium = w.next_medium;
    w.p0 = w.p0 + w.next_t * w.dir;
    if (++w.seg == kMaxShadowSegments) {
        w.blocked = true;
        return true;
    }
    return false;
}

// The NEE shadow walk with ratio tracking (homework2.tex:770-812), after
// k_vol_occlude: blocked segments are skipped, and only segments that cross
// boundaries take closest hits.  The walks' lengths vary widely (none to
// hundreds of collisions in a dense grid), so a wave advances all its walks
// by one collision at a time, and lanes whose walk ended take their next
// sample once kWalkRefill of them are idle; likewise a segment's start (its
// closest hit) waits for company.  One lane per sample from start to end
// left most of a wave idle behind its longest walk: 150 -> 100 ms for the
// 768x576 64-sample smoke render.
constexpr int kWalkRefill = 16;
template <bool STATS, bool SPH, bool GREY>
__global__ __launch_bounds__(256) void k_vol_shadow(DeviceScene S, PathBufs P) {
    __shared__ int stack[kStackLds * 256];
    const int gtid = blockIdx.x * blockDim.x + threadIdx.x;
    const int stride = gridDim.x * blockDim.x;
    int *spill = P.spill + gtid;
    uint32_t nn = 0, np = 0;
    int segs = 0;
    Walk w;
    int i = 0;
    // a busy lane is at a segment's start (wait) or inside one
    bool busy = false, fin = false, wait = false;
    FeedRange range;
    range.start(P.ctr + C_FEED_WALK, bucket_start(P, kBucketMiss), kFeedTickets);
    while (true) {
        const uint64_t idle = __ballot(!busy);
        const int nidle = __popcll(idle);
        if ((nidle >= kWalkRefill && !range.done) || nidle == 64) {
            const D3 T = grey_or<GREY>(w.T);
            if (fin && !w.blocked && maxc(T) > 0) {
                const float4 sc = P.sh_c[i], sx = P.sh_x[i];
                const double pdf_nee = double(sx.x) * avgc(grey_or<GREY>(w.p_nee));
                if (pdf_nee > 0) {
                    const double pdf_dir = double(sx.y) * avgc(grey_or<GREY>(w.p_dir));
                    const double wt = (pdf_nee * pdf_nee) / (pdf_nee * pdf_nee + pdf_dir * pdf_dir);
                    const D3 c = D3{sc.x, sc.y, sc.z} * T * (wt / pdf_nee);
                    const float4 r = P.rad[w.pid];
                    P.rad[w.pid] = make_float4(float(r.x + c.x), float(r.y + c.y), float(r.z + c.z), 0.f);
                }
            }
            fin = false;
            // k_vol_occlude's verdict picks the samples (the NEE stream is not
            // written back, so skipping a blocked one leaves every other draw
            // unchanged)
            const int k = range.take(!busy, [&](int j) {
                const uint8_t occ = P.sh_occ[j];
                return occ == 0 || occ == 2;
            });
            if (k >= 0) {
                i = k;
                const float4 so = P.sh_o[i], sd = P.sh_d[i], sx = P.sh_x[i];
                w.pid = __float_as_int(P.sh_c[i].w);
                w.medium = __float_as_int(so.w);
                w.bounces = __float_as_int(sd.w);
                w.p0 = D3{so.x, so.y, so.z};
                w.pp = D3{sd.x, sd.y, sd.z};
                w.dir = normalize(w.pp - w.p0);
                w.nst = uint64_t(__float_as_uint(sx.z)) | (uint64_t(__float_as_uint(sx.w)) << 32);
                w.ninc = pcg_inc(slot_info(P, w.pid).stream() ^ kNeeStreamXor);
                w.T = w.p_nee = w.p_dir = D3{1, 1, 1};
                w.crossings = P.sh_occ[i] == 2;
                w.seg = w.shadow_bounces = 0;
                w.blocked = false;
                busy = wait = true;
            }
            if (__ballot(busy) == 0) break;
        }
        const int nwait = __popcll(__ballot(wait));
        if (nwait >= kWalkRefill || (nwait > 0 && __ballot(busy && !wait) == 0)) {
            segs += __popcll(__ballot(wait && w.crossings));
            if (wait) walk_segment<STATS, SPH>(w, S, stack + threadIdx.x, spill, stride, nn, np);
            wait = false;
        }
        if (busy && !wait && walk_collision<GREY>(w, P)) {
            if (walk_advance(w, P)) {
                busy = false;
                fin = true;
            } else {
                wait = true;
            }
        }
    }
    if (__lane_id() == 0) P.wave_stat[gtid >> 6] += (unsigned long long)segs;
    if (STATS) {
        atomicAdd(&P.stat[S_SH_NODES], (unsigned long long)nn);
        atomicAdd(&P.stat[S_SH_PRIMS], (unsigned long long)np);
    }
}

// Volpath-specific path state initialisation after raygen.
__global__ void k_vol_init(DeviceScene S, PathBufs P) {
    int n = P.pass_ns * P.pass_nq;
    int stride = gridDim.x * blockDim.x;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        P.medium[i] = P.jobs ? P.jobs[slot_info(P, i).job].camera.medium_id : S.camera.medium_id;
        float4 o = P.ray_o[i];
        P.nee_c[i] = make_float4(o.x, o.y, o.z, 0.f);
        P.mtp[i] = make_float4(1.f, 1.f, 1.f, 1.f);
    }
}

template <class Alloc, class Bufs>
void vol_alloc(bool, size_t capacity, PathBufs &P, Bufs &bufs, Alloc alloc) {
    auto take = [&](size_t bytes) {
        void *p = alloc(bytes);
        bufs.push_back({p, bytes});
        return p;
    };
    P.medium = static_cast<int *>(take(capacity * sizeof(int)));
    P.nee_c = static_cast<float4 *>(take(capacity * sizeof(float4)));
    P.mtp = static_cast<float4 *>(take(capacity * sizeof(float4)));
    P.sh_x = static_cast<float4 *>(take(capacity * sizeof(float4)));
    P.vf_t = static_cast<double4 *>(take(capacity * sizeof(double4)));
    P.vf_p = static_cast<double4 *>(take(capacity * sizeof(double4)));
}

inline void vol_launch_check() {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) throw std::runtime_error(std::string("volpath kernel launch: ") + hipGetErrorString(e));
}

// What happens to each path of the extension queue: free flight and the sort's keys.
inline void vol_events(const DeviceScene &S, PathBufs &P, int cur, int grid, hipStream_t s, bool sph) {
    if (P.vol_flight) {
        auto kern = sph ? (P.vol_grey ? k_vol_flight<true, true> : k_vol_flight<true, false>)
                        : (P.vol_grey ? k_vol_flight<false, true> : k_vol_flight<false, false>);
        hipLaunchKernelGGL(kern, dim3(grid), dim3(256), 0, s, S, P, cur);
    } else {
        if (sph) hipLaunchKernelGGL(k_vol_event<true>, dim3(grid), dim3(256), 0, s, S, P, cur);
        else hipLaunchKernelGGL(k_vol_event<false>, dim3(grid), dim3(256), 0, s, S, P, cur);
    }
    vol_launch_check();
}
// The shading kernels, on the streams given (one may stand for all three).
// types: the material types present; textured: some material reads a texture;
// env: an envmap is among the lights (the kernels for spheres take scenes
// without them too).
template <bool SPH>
void vol_shade_t(const DeviceScene &S, PathBufs &P, int cur, int grid, const hipStream_t (&s)[3], unsigned types,
                 bool textured) {
    const dim3 g(grid), b(256);
    if (types & 4) hipLaunchKernelGGL((k_vol_shade<SPH, 2, kEvSurface>), g, b, 0, s[0], S, P, cur);
    hipLaunchKernelGGL((k_vol_shade<SPH, 0, kEvScatter>), g, b, 0, s[1], S, P, cur);
    if (types & 1) hipLaunchKernelGGL((k_vol_shade<SPH, 0, kEvSurface>), g, b, 0, s[2], S, P, cur);
    if (types & 2) hipLaunchKernelGGL((k_vol_shade<SPH, 1, kEvSurface>), g, b, 0, s[0], S, P, cur);
    if (textured || (types >> kVolTyped))
        hipLaunchKernelGGL((k_vol_shade<SPH, -1, kEvSurface>), g, b, 0, s[0], S, P, cur);
    hipLaunchKernelGGL((k_vol_shade<SPH, 0, kEvPass>), g, b, 0, s[2], S, P, cur);
    vol_launch_check();
}
inline void vol_shade_all(const DeviceScene &S, PathBufs &P, int cur, int grid, const hipStream_t (&s)[3], bool sph,
                          unsigned types, bool textured, bool env) {
    if (env) {
        const dim3 g(grid), b(256);
        hipLaunchKernelGGL((k_vol_shade<true, kMtEnv, kEvSurface>), g, b, 0, s[0], S, P, cur);
        hipLaunchKernelGGL((k_vol_shade<true, kMtEnv, kEvScatter>), g, b, 0, s[1], S, P, cur);
        hipLaunchKernelGGL((k_vol_shade<true, kMtEnv, kEvPass>), g, b, 0, s[2], S, P, cur);
        vol_launch_check();
    } else if (sph) vol_shade_t<true>(S, P, cur, grid, s, types, textured);
    else vol_shade_t<false>(S, P, cur, grid, s, types, textured);
}

inline void vol_shadow(const DeviceScene &S, PathBufs &P, int grid, hipStream_t s, bool stats, bool sph) {
    if (stats) {
        if (sph) hipLaunchKernelGGL((k_vol_occlude<true, true>), dim3(grid), dim3(256), 0, s, S, P);
        else hipLaunchKernelGGL((k_vol_occlude<true, false>), dim3(grid), dim3(256), 0, s, S, P);
    } else {
        if (sph) hipLaunchKernelGGL((k_vol_occlude<false, true>), dim3(grid), dim3(256), 0, s, S, P);
        else hipLaunchKernelGGL((k_vol_occlude<false, false>), dim3(grid), dim3(256), 0, s, S, P);
    }
    vol_launch_check();
    auto walk = P.vol_grey ? (stats ? (sph ? k_vol_shadow<true, true, true> : k_vol_shadow<true, false, true>)
                                    : (sph ? k_vol_shadow<false, true, true> : k_vol_shadow<false, false, true>))
                           : (stats ? (sph ? k_vol_shadow<true, true, false> : k_vol_shadow<true, false, false>)
                                    : (sph ? k_vol_shadow<false, true, false> : k_vol_shadow<false, false, false>));
    hipLaunchKernelGGL(walk, dim3(grid), dim3(256), 0, s, S, P);
    vol_launch_check();
}

}  // namespace ljx
