// bdpt.hip -- BidirectionalPathTracer (bidirPathTracer.cpp:10-313), VCMTracer
// and PhotonMap on gfx950.
//
// Several passes run side by side (a lane is a pixel of a pass: one pass of a
// 256^2 image alone does not fill the chip).  BidirectionalPathTracer:
//   1. the sub-paths, a path walk (walk_dev.h, SubpathWalk): per lane the eye
//      sub-path, the camera ray (camera.cpp:6-60) and MCRenderer::samplePath
//      (mcRenderer.cpp:16-57) from it, and the light sub-path,
//      Scene::genLightSample as AbstractObject::genSurfaceSample
//      (abstractObj.cpp:18-52) and samplePath from it, with the light-path
//      vertex counters, into one block of records per lane;
//   2. k_bdpt_prefix: what a connection needs of the records before its two
//      (BPrefix);
//   3. k_bdpt: every (light length, eye length) split of every joined length
//      (bidirPathTracer.cpp:53-140), the pairs of a wave's lanes dealt out to its
//      lanes: connectEdge (294-324), connectingColorProb (266-291) and
//      connectingMisWeight (142-221) with linkVertex (228-243).  Contributions
//      with an eye side of two or more vertices go to the lane's pixel,
//      light-tracing ones (the camera vertex alone on the eye side) are splatted
//      to the pixel Camera::convToRaster names (camera.cpp:148-170), scaled by
//      1 / pixel solid angle / pixel count;
//   4. the visibility tests (mcRenderer.cpp:59-65) of the connections, which
//      k_bdpt queues with their contribution and target pixel: the batch NoSelf
//      query (k_closest_hit: the same traversal, so the same answers), then
//      k_bdpt_accum; with a full queue a connection is traced in place;
//   5. k_bdpt_fold.  The pixel values of each pass are summed with float atomics
//      in a buffer of their own (the splats of other lanes land on any pixel);
//      it applies isLegalColor and fixVignetting and adds them to the Kahan film
//      in pass order.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <vector>

#include "grid_dev.h"
#include "merge_entry.h"
#include "pt_dev.h"
#include "walk_dev.h"
#include "wr_pt.h"

#pragma clang fp contract(off)

namespace wrd {

constexpr uint32_t kBdptLightVertex = 0x80000000u;  // as the light sub-paths of photon.hip
constexpr uint32_t kCameraObj = 0xFFFFFFFEu;        // the camera as a NoSelf contact: not an object, not NULL
constexpr uint32_t kVDelta = 1u, kVCamera = 2u;

// One Ray of a Path as the estimator reads it (ray.h:8-37).
struct BVert {
    f3 o, d, rad, n;  // n: the contact normal at o (the camera's: front)
    float op, dp;
    uint32_t inside, contact, flags, pad;
};

// terminateRay (mcRenderer.cpp:20-27) after a ray from o.
__device__ __forceinline__ BVert terminate_at(f3 o) {
    BVert t;
    t.o = o;
    t.d = mk(0.f, 0.f, 0.f);
    t.rad = t.d;
    t.n = t.d;
    t.op = 1.f;
    t.dp = 1.f;
    t.inside = WR_NONE;
    t.contact = WR_NONE;
    t.flags = kVDelta;
    t.pad = 0;
    return t;
}

// Camera::getPixelSolidAngle (camera.cpp:124-131).
__device__ __forceinline__ float pixel_solid_angle(const CamDev& c, uint32_t p) {
    const uint32_t x = p % c.W, y = p / c.W;
    const float xc = (float)((double)x + 0.5 - (c.W / 2.0)), yc = (float)((c.H / 2.0) - 0.5 - (double)y);
    const float pd = sqrtf(xc * xc + yc * yc + c.dist * c.dist);
    return c.dist / powf(pd, 3.f);
}

// Ray::cosineTerm (ray.cpp:52-58).
__device__ __forceinline__ float cos_term_v(const BVert& r) {
    float c = 1.f;
    if (((r.flags & kVCamera) || r.contact != WR_NONE) && (double)len(r.d) > 0.5) c = fabsf(dot(r.n, r.d));
    return (double)c > kEps ? c : (float)kEps;
}

// in.evalBSDF(out) (ray.cpp:15-22): the object of out's contact (else inside).
__device__ f3 eval_bsdf(const SceneDev& S, const BVert& in, const BVert& out) {
    if (out.flags & kVCamera) return mk(1.f, 1.f, 1.f);  // AbstractObject::evaluateBSDF
    const uint32_t obj = out.contact != WR_NONE ? out.contact : out.inside;
    if (obj == WR_NONE) return mk(0.f, 0.f, 0.f);
    const wr_object_gpu& ob = S.objs[obj];
    const f3 color = mk(ob.color[0], ob.color[1], ob.color[2]);
    if (ob.mat == WR_MAT_REFRACTIVE) return mk(0.f, 0.f, 0.f);  // refractiveObj.h:13-15
    if (ob.mat == WR_MAT_EMISSIVE) return color;                // emissiveObj.h:13
    if (out.contact == WR_NONE) return mk(0.f, 0.f, 0.f);       // diffuseObj.h:18, glossyObj.h:21
    const f3 n = out.n;
    if (!(dot(in.d, n) <= 0.f && dot(out.d, n) >= 0.f)) return mk(0.f, 0.f, 0.f);
    if (ob.mat == WR_MAT_DIFFUSE) return muls(color, (float)kInvPi);  // diffuseBsdf.h:29-34
    const f3 refl = normalize(add(muls(muls(n, -dot(n, in.d)), 2.f), in.d));  // isotropicPhong.h:41-48
    const f3 rho = muls(muls(muls(color, (float)((double)ob.power + 2.0)), 0.5f), (float)kInvPi);
    const float dRW = dot(refl, out.d);
    return muls(rho, powf(dRW > 0.f ? dRW : 0.f, ob.power));
}

// in.evalDirectionProbability(out) (ray.cpp:31-38); same: the emitted branch of
// AbstractObject::evalDirectionProbability (in and out one object).
__device__ float eval_dir_prob(const SceneDev& S, const CamDev& cam, uint32_t pixel, const BVert& in,
                               const BVert& out, bool same) {
    (void)in;
    if (out.flags & kVCamera) return (float)(1.0 / (double)pixel_solid_angle(cam, pixel));  // camera.cpp:144-146
    const uint32_t obj = out.contact != WR_NONE ? out.contact : out.inside;
    if (obj == WR_NONE) return 0.f;
    const wr_object_gpu& ob = S.objs[obj];
    if (ob.mat == WR_MAT_REFRACTIVE || ob.mat == WR_MAT_EMISSIVE)  // abstractObj.cpp:61-68
        return same ? (float)(kInvPi * 0.25f) * 2.f : 0.f;
    if (out.contact == WR_NONE) return 0.f;
    const float p = ob.pmax;
    const float c = dot(out.n, out.d);
    if (ob.mat == WR_MAT_DIFFUSE) return p * (c > 0.f ? (float)((double)c * kInvPi) : 0.f);  // diffuseBsdf.h:12-14
    const float cos_theta = (double)c > kEps ? c : (float)kEps;                                // isotropicPhong.h:13-18
    return p * (float)(((double)ob.power + 1.0) * (double)powf(cos_theta, ob.power) * (kInvPi * 0.5));
}

__device__ __forceinline__ bool is_delta(const BVert& v) { return (v.flags & kVDelta) != 0; }

// max(|a - b|, EPSILON)
__device__ __forceinline__ float vert_dist(const BVert& a, const BVert& b) {
    const float l = len(sub(a.o, b.o));
    return (double)l > kEps ? l : (float)kEps;
}

// PdfWtoA's factor cosine / distance^2.
__device__ __forceinline__ double area_factor(float cosine, float dist) {
    return (double)(1.0f * fabsf(cosine) / (dist * dist));
}

// linkVertex (bidirPathTracer.cpp:228-243): record v re-aimed at its neighbour.
__device__ __forceinline__ BVert link_to(const BVert& v, const BVert& to) {
    BVert l = v;
    l.d = normalize(sub(to.o, v.o));
    l.inside = to.inside;
    return l;
}

// What a connection or merge needs of all the records before one of its two
// records, i.e. the part of connectingColorProb (bidirPathTracer.cpp:266-291)
// and of the weight (142-221; vcmTracer.cpp:221-320) that does not depend on
// the other sub-path.
//
// Write the joined path light[0..c], eye[e..0]; direct[i] and reverse[i] are
// the weight's two recurrences, and the weight's sum is
//   sum over i of direct[i] * reverse[i + 1] * (vc_i + K * vm_i),
// vc_i = 1 for two non-delta neighbours, vm_i the merging strategy's factor at
// vertex i + 1 and K = pi r^2 * merging light paths.  On the light side,
// direct[i] does not depend on the connection up to i = c, and reverse[i] =
// reverse[c] * (factors f[i] .. f[c - 1] of single edges); on the eye side the
// same holds with the roles exchanged.  So
//   sum over i < c = reverse[c] * sum(direct[i] * (..) * f[i + 1] .. f[c - 1]),
// whose second factor obeys S[c + 1] = f[c] * S[c] + direct[c] * (..): one
// multiply-add per record.  The same holds for the products of the colour and
// of the probability.  These prefixes, kept per record by k_bdpt_prefix, leave
// each connection and each merge the two records and the edge between them,
// instead of a sweep over the joined path with its dozen arrays in scratch
// (3.5 KB a lane): Cornell 256^2 x 8 passes, maxPathLen 8, 14.7 ms in k_bdpt with
// the sweep, 7.5 with the prefixes (0.57 since connect_wave deals the pairs out)
// and 0.36 in k_bdpt_prefix; the merges of a 201 x 151 VCM render 0.83 and 0.29 ms.
struct BPrefix {
    double run;     // direct[i] of a light record, reverse of an eye record
    double vc, vm;  // S of the connections and of the merging factors (without K)
    double all;     // product of the edge factors: reverse[0] = reverse[c] * all
    f3 color;       // product over the records before this one (radiance * cosine)
    float prob;     // product of their probabilities
    uint32_t flags; // kPAny, kPEmissive, kPDelta
    uint32_t pad;
};
constexpr uint32_t kPAny = 1u;       // some neighbours among the records up to this one are both non-delta
constexpr uint32_t kPEmissive = 2u;  // the record's contact is an emitter
constexpr uint32_t kPDelta = 4u;     // the record is a delta scatter (or an end)

// One pass's grid (VCMTracer, PhotonMap): src and idx are of the pass's block of
// light points.
using VcmGrid = GridView;

struct VcmTerms {
    float r;     // the pass's merging radius
    double nvm;  // light sub-paths of the pass (one per pixel)
    bool vm;     // a merge (VM), else a connection (VC)
};

// The weight, colour and probability of the path light[0..c], eye[e..0] joined
// by its two records as connectEdge left them (evalOriginProbability compares
// two temporaries there, so it is 1; no participating media, so expTerm is 1
// and no record lies inside a medium).  The doubles are the reference's.
__device__ __forceinline__ float color_prob_weight(const SceneDev& S, const CamDev& cam, uint32_t pixel,
                                                   const BVert& lc, const BPrefix& pl, int c, const BVert& ec,
                                                   const BPrefix& pe, int e, f3& color, float& prob,
                                                   const VcmTerms* vt = nullptr) {
    const float d = vert_dist(ec, lc);
    const float cos_l = cos_term_v(lc), cos_e = cos_term_v(ec);
    color = mulv(pl.color, lc.rad);
    color = muls(color, cos_l * cos_e / (d * d));
    color = mulv(color, ec.rad);
    color = mulv(color, pe.color);
    prob = pl.prob * (lc.dp * lc.op);
    if (vt && vt->vm) {  // a merge: the merging disc and the area density at the eye-side vertex
        prob = (float)((double)prob * (kPi * (double)vt->r * (double)vt->r));
        prob *= 1.0f * fabsf(cos_e) / (d * d);
    }
    prob *= ec.dp * ec.op;
    prob *= pe.prob;
    if (prob == 0.f || len(color) == 0.f) return 0.f;  // the caller skips these
    const bool dl = is_delta(lc), de = is_delta(ec);
    const double pf = dl ? 1.0 : (double)eval_dir_prob(S, cam, pixel, lc, lc, c == 0);
    const double pb = de ? 1.0 : (double)eval_dir_prob(S, cam, pixel, ec, ec, e == 0);
    const double next = pl.run * area_factor(cos_e, d) * pf;  // direct[c + 1]
    const double back = pe.run * area_factor(cos_l, d) * pb;  // reverse[c]
    const double join = pl.run * pe.run;
    double all = back * pl.vc + next * pe.vc;
    const bool connects = !dl && !de;
    if (connects) all += join;
    if (!vt) {
        const double w = join / all;
        return (float)(w > 0.0 ? w : 0.0);
    }
    const double disc = kPi * (double)vt->r * (double)vt->r;
    // merging at the eye-side vertex, unless it is the camera
    const double merge = e > 0 && !de ? pe.run * next * disc : 0.0;
    all += (back * pl.vm + next * pe.vm) * disc * vt->nvm + merge * vt->nvm;
    if (!connects && !((pl.flags | pe.flags) & kPAny)) all += back * pl.all;  // pathCanNotConnect
    const double w = (vt->vm ? merge * vt->nvm : join) / all;
    if (!(w >= 0.0)) return 0.f;
    return (float)w;
}

// connectEdge (bidirPathTracer.cpp:294-324) on copies lc / ec of light[c] and
// eye[e]; the previous records are read after the edits (for c = 0, and for an
// eye side of one record, the previous record is the connection record itself).
__device__ __forceinline__ bool connect_edge(const SceneDev& S, const BVert* L, int c, const BVert* E, int e, BVert& lc,
                                             BVert& ec) {
    if (is_delta(lc) || is_delta(ec)) return false;
    lc.d = normalize(sub(ec.o, lc.o));
    ec.d = mk(-lc.d.x, -lc.d.y, -lc.d.z);
    lc.dp = 1.f;
    {
        BVert pre = lc;
        if (c > 0) {
            pre.d = L[c - 1].d;
            pre.inside = L[c - 1].inside;
        }
        lc.rad = eval_bsdf(S, pre, lc);
        if (lc.contact != WR_NONE && c > 0) lc.inside = dot(lc.n, lc.d) > 0.f ? pre.inside : lc.contact;
    }
    ec.dp = 1.f;
    {
        BVert pre = ec;
        if (e > 0) {
            pre.d = E[e - 1].d;
            pre.inside = E[e - 1].inside;
        }
        ec.rad = eval_bsdf(S, pre, ec);
        if (ec.contact != WR_NONE && e > 0) ec.inside = dot(ec.n, ec.d) > 0.f ? pre.inside : ec.contact;
    }
    return true;
}

// connectEdge for a merge (vcmTracer.cpp:366-398 with VM): both directions are
// re-aimed, only the eye-side record is edited (radiance, probability, delta,
// inside); its previous record is an eye record (the merged eye vertex is at
// least the second of its path).
__device__ __forceinline__ bool connect_edge_vm(const SceneDev& S, const BVert* E, int e, BVert& lc, BVert& ec) {
    if (is_delta(ec)) return false;
    lc.d = normalize(sub(ec.o, lc.o));
    ec.d = mk(-lc.d.x, -lc.d.y, -lc.d.z);
    ec.dp = 1.f;
    BVert pre = ec;
    pre.d = E[e - 1].d;
    pre.inside = E[e - 1].inside;
    ec.rad = eval_bsdf(S, pre, ec);
    if (ec.contact != WR_NONE) ec.inside = dot(ec.n, ec.d) > 0.f ? pre.inside : ec.contact;
    return true;
}

// A path that the eye side found alone: eye[e..0], eye[e] on an emitter (e >= 1);
// pe, pp: the prefixes of eye[e] and eye[e - 1].
// Only paths that pathCanNotConnect rejects for every connection are taken.
// Its sum has no connection terms; with vt, the merging ones.
__device__ __forceinline__ float eye_path_weight(const BVert* E, const BPrefix& pe, const BPrefix& pp, int e,
                                                 const BVert& last, f3& color, float& prob,
                                                 const VcmTerms* vt = nullptr) {
    color = mulv(last.rad, pe.color);
    prob = last.dp * last.op * pe.prob;
    if (prob == 0.f || len(color) == 0.f) return 0.f;
    double all = 0.0;
    if (vt) {
        // the emitter's record starts the path: its direction probability is that of an emission
        const double pf = is_delta(last) ? 1.0 : (double)((float)(kInvPi * 0.25f) * 2.f);
        const BVert prev = E[e - 1];
        const double next = last.op * area_factor(cos_term_v(prev), vert_dist(last, prev)) * pf;
        const double disc = kPi * (double)vt->r * (double)vt->r * vt->nvm;
        if (e > 1 && !is_delta(prev)) all += pp.run * next * disc;
        all += next * pp.vm * disc;
    }
    all += pe.run;
    const double w = pe.run / all;
    return (float)(w > 0.0 ? w : 0.0);
}

__device__ __forceinline__ bool emissive(const SceneDev& S, uint32_t obj) {
    return obj != WR_NONE && S.objs[obj].mat == WR_MAT_EMISSIVE;
}

// The visibility queue: rays in the batch NoSelf layout (o, d, inside,
// contact), per entry the contribution and the distance to the light-side
// record, and the target (pass buffer offset + pixel).
struct VisQueue {
    uint32_t* rays;   // 8 words per entry
    float* pay;       // 4 floats per entry: contribution, distance
    uint32_t* dst;    // pixel index into the pass buffers (k * npix + q)
    uint32_t* count;
    uint32_t cap;
};

__device__ __forceinline__ void atomic_add3(float* buf, uint32_t p, f3 v) {
    atomicAdd(buf + 3 * p + 0, v.x);
    atomicAdd(buf + 3 * p + 1, v.y);
    atomicAdd(buf + 3 * p + 2, v.z);
}

// The sub-paths of every lane (pixel and pass) as a path walk: paths [0, eyes)
// are the eye sub-paths of the lanes in order, the others their light
// sub-paths (eyes = 0: PhotonMap forms its own).  counts[2 * lane] = eye
// records, counts[2 * lane + 1] = light records.  Record k + 1 is written by
// step k; max_depth + 3 records hold the longest sub-path: its first ray,
// max_depth scatters, the end.
struct SubpathWalk {
    CamDev cam;
    uint32_t max_depth, pass0, npix, maxv, eyes;
    uint64_t seed;
    BVert* verts;
    uint32_t* counts;

    __device__ __forceinline__ void split(uint32_t path, bool& eye, uint32_t& lane, uint32_t& p, uint32_t& pass,
                                          BVert*& V) const {
        eye = path < eyes;
        lane = eye ? path : path - eyes;
        p = lane % npix;
        pass = pass0 + lane / npix;
        V = verts + ((size_t)lane * 2 + (eye ? 0 : 1)) * maxv;
    }

    __device__ __forceinline__ bool begin(const SceneCtx& sc, uint32_t path, LaneStack& st, f3& o, f3& d,
                                          uint32_t& inside, uint32_t& contact) const {
        bool eye;
        uint32_t lane, p, pass;
        BVert* V;
        split(path, eye, lane, p, pass, V);
        float rn[4];
        BVert r;
        r.op = 1.f;
        r.dp = 1.f;
        r.inside = WR_NONE;
        r.contact = WR_NONE;
        r.pad = 0;
        bool go = true;
        inside = contact = WR_NONE;
        if (eye) {  // the camera ray (camera.cpp:6-60), traced without a condition
            rng4(seed, p, pass, 0, rn);
            r.o = cam.pos;
            r.d = cam_dir(cam, p, rn[0], rn[1]);
            r.rad = mk(1.f, 1.f, 1.f);
            r.n = cam.front;
            r.flags = kVCamera;
            r.inside = find_inside(sc.S, r.o, r.d, WR_NONE, st);
        } else {  // the light ray (as LightWalk's first)
            rng4(seed, p, pass, kBdptLightVertex, rn);
            const LightSample ls = sample_light(sc, rn);
            r.o = mk(0.f, 0.f, 0.f);
            r.d = r.o;
            r.rad = r.o;
            r.n = r.o;
            r.flags = 0;
            go = ls.ok;
            if (ls.ok) {
                rng4(seed, p, pass, kBdptLightVertex + 1, rn);
                const float term1 = (float)(2.0 * kPi * (double)rn[0]);  // uniformSphereSampler.h:6-20
                const float term2 = 2.f * sqrtf(rn[1] - rn[1] * rn[1]);
                f3 dir = mk(cosf(term1) * term2, 1.f - 2.f * rn[1], sinf(term1) * term2);
                r.dp = (float)(kInvPi * 0.25f);
                if (dot(dir, ls.n) < 0.f) dir = mk(-dir.x, -dir.y, -dir.z);
                r.o = ls.o;
                r.n = ls.n;
                r.d = dir;
                r.rad = ls.rad;
                r.contact = ls.obj;
                r.inside = find_inside(sc.S, r.o, r.d, ls.obj, st);
                r.dp *= 2.f;
                r.op = ls.op;
                inside = r.inside;
                contact = r.contact;
            }
        }
        V[0] = r;
        if (!go) {  // an empty light sample: its ray hits nothing
            V[1] = terminate_at(r.o);
            counts[2 * lane + 1] = 2;
        }
        o = r.o;
        d = r.d;
        return go;
    }

    __device__ __forceinline__ bool step(const SceneCtx& sc, uint32_t path, uint32_t s, f3 o, f3 d, const PHit& hit,
                                         LaneStack& st, Out& out) const {
        bool eye;
        uint32_t lane, p, pass;
        BVert* V;
        split(path, eye, lane, p, pass, V);
        uint32_t* count = counts + 2 * lane + (eye ? 0 : 1);
        *count = s + 2;  // of a path that ends here; a later step overwrites it
        // an escaped ray ends the path at the origin before its own; a light
        // ray's hit counts only at dist > 0 (abstractObj.cpp:46)
        if (hit.rec == WR_NONE || (!eye && s == 0 && !(hit.t > 0.f))) {
            V[s + 1] = terminate_at(s == 0 ? o : V[s - 1].o);
            return false;
        }
        const uint32_t inside = V[s].inside;
        float rn[4];
        rng4(seed, p, pass, (eye ? 0u : kBdptLightVertex + 1) + s + 1, rn);
        out = scatter(sc, inside != WR_NONE ? inside : hit.obj, o, d, hit, inside, rn, st);
        const bool absorbed = (double)len(out.d) < 0.5;
        if (!absorbed && s + 1 > max_depth) {
            V[s + 1] = terminate_at(o);
            return false;
        }
        BVert nx;
        nx.o = out.o;
        nx.d = out.d;
        nx.rad = out.rad;
        nx.n = out.n;
        nx.op = out.op;
        nx.dp = out.dp;
        nx.inside = out.inside;
        nx.contact = out.contact;
        nx.flags = out.delta ? kVDelta : 0u;
        nx.pad = 0;
        V[s + 1] = nx;
        return !absorbed;
    }
};

// The prefix of a sub-path's first record.
__device__ __forceinline__ BPrefix prefix_first(const SceneDev& S, const BVert& v) {
    BPrefix p;
    p.run = v.op;
    p.vc = p.vm = 0.0;
    p.all = 1.0;
    p.color = mk(1.f, 1.f, 1.f);
    p.prob = 1.f;
    p.flags = (emissive(S, v.contact) ? kPEmissive : 0u) | (is_delta(v) ? kPDelta : 0u);
    p.pad = 0;
    return p;
}

// The prefix of record i > 0 (cur) from that of the record before it (prev).
__device__ __forceinline__ void prefix_next(const SceneDev& S, const CamDev& cam, uint32_t pixel, bool eye, uint32_t i,
                                            const BVert& prev, const BVert& cur, BPrefix& p) {
    const BVert link = link_to(cur, prev);
    const float d = vert_dist(cur, prev);
    const bool dp = is_delta(prev), dc = is_delta(cur);
    const float cos_prev = cos_term_v(prev);
    const double own = area_factor(cos_prev, d);         // of the edge, at prev
    const double at = area_factor(cos_term_v(link), d);  // of the edge, at cur
    const double own_p = dp ? 1.0 : (double)eval_dir_prob(S, cam, pixel, prev, prev, !eye && i == 1);
    const double link_p = dc ? 1.0 : (double)eval_dir_prob(S, cam, pixel, link, link, false);
    const double edge = own * link_p;  // the other recurrence's factor from cur to prev
    // merging at the far vertex of the pair: at cur on the light side, at prev on the eye side
    // (the camera merges with nothing)
    double merge = 0.0;
    if (!eye && !dc) merge = own_p * at;
    if (eye && i > 1 && !dp) merge = edge;
    const bool connects = !dp && !dc;
    p.vc = edge * p.vc + (connects ? p.run : 0.0);
    p.vm = edge * p.vm + merge * p.run;
    p.all *= edge;
    p.run = p.run * at * own_p;
    p.color = muls(mulv(p.color, prev.rad), cos_prev);
    p.prob *= prev.dp * prev.op;
    p.flags = (p.flags & kPAny) | (connects ? kPAny : 0u) | (emissive(S, cur.contact) ? kPEmissive : 0u) |
              (dc ? kPDelta : 0u);
}

// The prefixes of every sub-path of the lanes [first, end), one lane per
// sub-path: side 0 the light sub-path, side 1 the eye sub-path of each lane's
// SubpathWalk.  table: of the records of lane `first` on.
__global__ __launch_bounds__(256) void k_bdpt_prefix(SceneDev S, CamDev cam, uint32_t npix, uint32_t first,
                                                     uint32_t end, uint32_t maxv, const BVert* verts,
                                                     const uint32_t* counts, BPrefix* table) {
    const uint64_t id = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    const uint32_t lanes = end - first;
    if (id >= 2ull * lanes) return;
    const bool eye = id >= lanes;
    const uint32_t own = (uint32_t)(eye ? id - lanes : id), lane = first + own;
    const BVert* V = verts + ((size_t)lane * 2 + (eye ? 0 : 1)) * maxv;
    BPrefix* P = table + ((size_t)own * 2 + (eye ? 0 : 1)) * maxv;
    const uint32_t n = min(counts[2 * (size_t)lane + (eye ? 0 : 1)], maxv), pixel = lane % npix;
    if (n == 0) return;
    BVert prev = V[0];
    BPrefix p = prefix_first(S, prev);
    P[0] = p;
    for (uint32_t i = 1; i < n; i++) {
        const BVert cur = V[i];
        prefix_next(S, cam, pixel, eye, i, prev, cur, p);
        P[i] = p;
        prev = cur;
    }
}

// The prefixes as the connections and merges read them.  TABLE: from
// k_bdpt_prefix's table; else, where the device has no room for the table (56 B
// for each 72 B record), formed anew from the sub-path's records, which costs
// about what a sweep over them costs.
template <bool TABLE>
struct Prefixes {
    const BPrefix* table;  // indexed like verts
    const BVert* verts;
    uint32_t npix, maxv;
    // of record i of a lane's eye or light sub-path
    __device__ __forceinline__ BPrefix at(const SceneDev& S, const CamDev& cam, uint64_t lane, bool eye, int i) const {
        const size_t first = (lane * 2 + (eye ? 0 : 1)) * maxv;
        if (TABLE) return table[first + i];
        BVert prev = verts[first];
        BPrefix p = prefix_first(S, prev);
        for (int k = 1; k <= i; k++) {
            const BVert cur = verts[first + k];
            prefix_next(S, cam, (uint32_t)(lane % npix), eye, (uint32_t)k, prev, cur, p);
            prev = cur;
        }
        return p;
    }
    // the flags of record `rec`; before: those of the record before it, unless it is the first
    __device__ __forceinline__ uint32_t flags(const SceneDev& S, size_t rec, bool first, uint32_t before) const {
        if (TABLE) return table[rec].flags;
        const BVert& v = verts[rec];
        const bool d = is_delta(v);
        const bool any = (before & kPAny) || (!first && !d && !(before & kPDelta));
        return (any ? kPAny : 0u) | (emissive(S, v.contact) ? kPEmissive : 0u) | (d ? kPDelta : 0u);
    }
};

// Index of the n-th set bit.
__device__ __forceinline__ int nth_bit(uint64_t mask, uint32_t n) {
    for (; n > 0; n--) mask &= mask - 1;
    return __ffsll((unsigned long long)mask) - 1;
}

// Queue slots that a wave of connect_wave reserves ahead at most.  The one
// counter bounds the connections: with an atomic of each wave for every 64
// pairs k_bdpt took 1.6 ms for Cornell 256^2 x 8 passes (5.9M entries), of which
// its arithmetic is 0.6 ms.  With the expected number of entries reserved at
// once (slots that stay empty hold rays that leave the scene) the render takes
// 4.97 ms instead of 6.04; 192 ahead instead of 448: 5.00 ms.
constexpr uint32_t kReserve = 448;

// The pairs of records that a wave's lanes connect, for connect_wave.
struct PairTable {
    uint64_t eye[64], light[64];  // per lane: the records that connect to something, a bit each
    uint32_t upto[64];            // pairs of the lanes up to this one
};

// The connections of a wave's lanes (bidirPathTracer.cpp:53-140, and with grids
// vcmTracer.cpp:88-173): every eye record with no light record, and with every
// light record.  Sub-paths differ in length, and a lane that walked its own
// pairs would keep its wave for the longest of 64 products (k_bdpt: 7.5 ms for
// Cornell 256^2 x 8 passes); so each lane notes which of its records connect
// at all (neither delta nor an emitter), and the wave deals its lanes' pairs
// out one to each lane at a time.  Every lane of the wave makes the
// call; lane0: the lane (pixel and pass) of the wave's first; max_eye,
// max_light: 0 where a lane of the wave has none.  Adds what needs no visibility test to the lane's own pixel.
template <bool TABLE>
__device__ __forceinline__ f3 connect_wave(const SceneDev& S, const SceneCtx& sc, const CamDev& cam, uint32_t npix,
                                           uint32_t maxv, uint64_t lane0, const BVert* verts,
                                           const Prefixes<TABLE>& prefix, int max_eye, int max_light,
                                           float* pix_all, const VisQueue& Q, LaneStack& st, const VcmGrid* grids, PairTable& T) {
    static_assert(wr::kBdptMaxDepth + 3 <= 64, "a record per bit");
    const uint32_t wl = threadIdx.x & 63u;
    f3 own = mk(0.f, 0.f, 0.f);
    uint64_t eye = 0, light = 0;
    {
        const size_t ei = (lane0 + wl) * 2 * maxv, li = ei + maxv;
        uint32_t fl = 0;
        for (int e = 0; e < max_eye; e++) {
            fl = prefix.flags(S, ei + e, e == 0, fl);
            if (!(fl & kPEmissive)) {
                if (!(fl & kPDelta)) eye |= 1ull << e;
            } else if (e > 0 && !(fl & kPAny)) {
                // an emitter: the eye path alone, if no connection could have made it
                const VcmTerms vt{grids ? grids[(lane0 + wl) / npix].r : 0.f, (double)npix, false};
                f3 color;
                float prob;
                const float w = eye_path_weight(verts + ei, prefix.at(S, cam, lane0 + wl, true, e),
                                                prefix.at(S, cam, lane0 + wl, true, e - 1), e, verts[ei + e], color,
                                                prob, grids ? &vt : nullptr);
                if (prob != 0.f && len(color) != 0.f) own = add(own, muls(divs(color, prob), w));
            }
        }
        // light paths that start on no emitter (an empty light sample) connect to nothing
        if (max_light > 0 && eye != 0 && (prefix.flags(S, li, true, 0) & kPEmissive)) {
            fl = 0;
            for (int c = 0; c < max_light; c++) {
                fl = prefix.flags(S, li + c, c == 0, fl);
                if (!(fl & kPDelta) && (c == 0 || !(fl & kPEmissive))) light |= 1ull << c;
            }
        }
    }
    uint32_t upto = (uint32_t)(__popcll(eye) * __popcll(light));
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t t = __shfl_up(upto, off, 64);
        if (wl >= (uint32_t)off) upto += t;
    }
    T.eye[wl] = eye;
    T.light[wl] = light;
    T.upto[wl] = upto;
    __builtin_amdgcn_wave_barrier();  // the table is this wave's own: LDS operations of a wave stay in order
    const uint32_t total = __shfl(upto, 63, 64);
    uint32_t kept = 0, kept_end = 0, used = 0;  // the wave's reserved queue slots, and its entries so far
    // Once a reservation lies past the queue the wave makes no more, so a wave adds
    // at most one (512 slots) past it and the 32-bit counter does not come round
    // below 8M waves, more lanes than the device has memory for.
    bool full = false;
    for (uint32_t t0 = 0; t0 < total; t0 += 64) {
        BVert ec{};
        f3 contrib{};
        uint32_t target = 0, k = 0;
        float dist = 0.f;
        auto connect = [&](uint32_t t) {
            uint32_t o = 0;  // the first lane with upto > t
#pragma unroll
            for (uint32_t step = 32; step > 0; step >>= 1)
                if (T.upto[o + step - 1] <= t) o += step;
            const uint32_t r = o ? t - T.upto[o - 1] : t;
            const uint64_t lights = T.light[o];
            const uint32_t nl = (uint32_t)__popcll(lights);
            const int e = nth_bit(T.eye[o], r / nl), c = nth_bit(lights, r % nl);
            const uint64_t lane = lane0 + o;
            const uint32_t p = (uint32_t)(lane % npix);
            k = (uint32_t)(lane / npix);
            const size_t ei = lane * 2 * maxv, li = ei + maxv;
            BVert lc = verts[li + c];
            ec = verts[ei + e];
            if (!connect_edge(S, verts + li, c, verts + ei, e, lc, ec)) return false;
            const VcmTerms vt{grids ? grids[k].r : 0.f, (double)npix, false};
            f3 color;
            float prob;
            const float w = color_prob_weight(S, cam, p, lc, prefix.at(S, cam, lane, false, c), c, ec,
                                              prefix.at(S, cam, lane, true, e), e, color, prob, grids ? &vt : nullptr);
            if (prob == 0.f) return false;
            if (len(color) == 0.f) return false;
            contrib = muls(divs(color, prob), w);
            target = p;
            if (e == 0) {  // light tracing: splat to the pixel the camera sees the point in
                const f3 v = sub(lc.o, cam.pos);
                const float vfd = dot(v, cam.front);
                const float scale = cam.dist / vfd;
                const float rx = (float)(cam.W / 2.0 + (double)(dot(v, cam.right) * scale));
                const float ry = (float)(cam.H / 2.0 - (double)(dot(v, cam.top) * scale));
                const int x = (int)rx, y = (int)ry;  // checkPixelBound truncates (camera.cpp:164-170)
                if (!(x >= 0 && y >= 0 && x < (int)cam.W && y < (int)cam.H)) return false;
                target = (uint32_t)(y * (int)cam.W + x);
                const float factor = (float)(1.0 / (double)pixel_solid_angle(cam, target));
                contrib = muls(contrib, factor / (float)npix);
            }
            dist = len(sub(ec.o, lc.o));
            return true;
        };
        const bool want = t0 + wl < total && connect(t0 + wl);
        const uint64_t m = __ballot(want);
        if (m == 0) continue;
        // the slots: what is left of the wave's reservation, then of a new one
        // for as many more entries as its pairs so far let expect
        const uint32_t n = (uint32_t)__popcll(m), avail = kept_end - kept;
        used += n;
        uint32_t first = kept, fresh = 0;
        if (n > avail && full) {
            first = fresh = kept = kept_end = Q.cap;
        } else if (n > avail) {
            const uint32_t seen = min(t0 + 64, total);
            const uint32_t take = n - avail + min((uint32_t)((uint64_t)(total - seen) * used / seen), kReserve);
            if (wl == 0) fresh = atomicAdd(Q.count, take);
            fresh = __shfl(fresh, 0, 64);
            kept = fresh + (n - avail);
            kept_end = fresh + take;
            full = fresh >= Q.cap;
        } else {
            kept += n;
        }
        if (!want) continue;
        const uint32_t rank = (uint32_t)__popcll(m & ((1ull << wl) - 1ull));
        const uint32_t slot = rank < avail ? first + rank : fresh + (rank - avail);
        // MCRenderer::visibilityTest from the eye-side connection record
        const uint32_t contact = (ec.flags & kVCamera) ? kCameraObj : ec.contact;
        if (slot < Q.cap) {
            uint32_t* ray = Q.rays + 8 * (size_t)slot;
            ray[0] = __float_as_uint(ec.o.x); ray[1] = __float_as_uint(ec.o.y); ray[2] = __float_as_uint(ec.o.z);
            ray[3] = __float_as_uint(ec.d.x); ray[4] = __float_as_uint(ec.d.y); ray[5] = __float_as_uint(ec.d.z);
            ray[6] = ec.inside;
            ray[7] = contact;
            float* y = Q.pay + 4 * (size_t)slot;
            y[0] = contrib.x; y[1] = contrib.y; y[2] = contrib.z; y[3] = dist;
            Q.dst[slot] = k * npix + target;
        } else {  // queue full: trace here
            const PHit h = trace_scene<true>(sc, ec.o, ec.d, ec.inside, contact, st);
            if (nee_visible(h.rec, h.t, dist)) atomic_add3(pix_all + 3 * (size_t)k * npix, target, contrib);
        }
    }
    // slots reserved for more entries than came: rays that leave the scene, contributing nothing
    for (uint32_t slot = kept + wl; slot < min(kept_end, Q.cap); slot += 64) {
        uint32_t* ray = Q.rays + 8 * (size_t)slot;
        for (int a = 0; a < 6; a++) ray[a] = __float_as_uint(a < 3 ? 1e18f : 1.f);
        ray[6] = ray[7] = WR_NONE;
        float* y = Q.pay + 4 * (size_t)slot;
        y[0] = y[1] = y[2] = y[3] = 0.f;
        Q.dst[slot] = WR_NONE;
    }
    return own;
}

// The lanes [first, end); prefix: table indexed as if it held every lane's.
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void k_bdpt(
    SceneDev S, CamDev cam, uint32_t first, uint32_t end, uint32_t npix, uint32_t maxv, const BVert* verts,
    const BPrefix* prefix, const uint32_t* counts, float* pix_all, VisQueue Q, uint32_t width) {
    __shared__ PairTable tables[4];
    const uint32_t wl = threadIdx.x & 63u;
    const uint64_t lane0 = first + (uint64_t)(blockIdx.x * 4 + (threadIdx.x >> 6)) * width, lane = lane0 + wl;
    const bool valid = wl < width && lane < end;
    StackSpill spill;
    LaneStack st(&spill);
    const SceneCtx sc = make_scene_ctx(S);
    const uint32_t ne = valid ? counts[2 * lane] : 0u, nl = valid ? counts[2 * lane + 1] : 0u;
    const f3 own = connect_wave(S, sc, cam, npix, maxv, lane0, verts, Prefixes<true>{prefix, verts, npix, maxv},
                                (int)min(ne, maxv), (int)min(nl, maxv), pix_all, Q, st, nullptr,
                                tables[threadIdx.x >> 6]);
    if (valid) atomic_add3(pix_all + 3 * (size_t)(lane / npix) * npix, (uint32_t)(lane % npix), own);
}

// The queued visibility tests, answered by the batch NoSelf query (hits:
// prim WR_NONE on a miss, t): visible connections add their contribution.
// Connections of one pixel follow each other in the queue (connect_wave deals
// them out in that order), so a wave first sums every run of entries with one
// target and adds a run with one set of atomics (5.9M entries: 936 us with one
// set per entry, 96 us).
__global__ __launch_bounds__(256) void k_bdpt_accum(uint32_t n, const float* pay, const uint32_t* dst,
                                                    const uint4* hits, float* pix_all) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t to = WR_NONE;
    f3 v = mk(0.f, 0.f, 0.f);
    if (i < n) {
        const uint4 h = hits[i];
        const float* y = pay + 4 * (size_t)i;
        if (nee_visible(h.x == WR_NONE ? WR_NONE : 0u, __uint_as_float(h.y), y[3])) v = mk(y[0], y[1], y[2]);
        to = dst[i];
    }
    const uint32_t prev = __shfl_up(to, 1);
    const uint64_t heads = __ballot(lane == 0 || to != prev);
    // the lanes of this run that follow: up to the next head
    const uint64_t later = heads & ~((2ull << lane) - 1ull);
    const uint32_t end = later ? (uint32_t)__ffsll((unsigned long long)later) - 1 : 64u;
#pragma unroll
    for (uint32_t off = 1; off < 64; off <<= 1) {
        const f3 o = mk(__shfl_down(v.x, off), __shfl_down(v.y, off), __shfl_down(v.z, off));
        if (lane + off < end) v = add(v, o);
    }
    if (i < n && ((heads >> lane) & 1) && (v.x != 0.f || v.y != 0.f || v.z != 0.f)) atomic_add3(pix_all, to, v);
}

// Each pass's pixel values, in pass order: isLegalColor, fixVignetting, the Kahan film.
__global__ __launch_bounds__(256) void k_bdpt_fold(CamDev cam, uint32_t npass, uint32_t npix, const float* pix,
                                                   FilmDev film) {
    const uint32_t p = blockIdx.x * 256 + threadIdx.x;
    if (p >= npix) return;
    for (uint32_t k = 0; k < npass; k++) {
        const float* c = pix + 3 * ((size_t)k * npix + p);
        f3 v = mk(c[0], c[1], c[2]);
        if (!legal(v)) v = mk(0.f, 0.f, 0.f);
        film_add(film, p, fix_vignetting(cam, v, p));
    }
}

// ---- VCMTracer (vcmTracer.cpp:6-446) ---------------------------------------
// Several passes side by side (lane = pass x pixel, as k_bdpt), each with its
// own light points, radius and grid: the sub-paths of SubpathWalk (one
// light path per pixel); per pass the light points (vcmTracer.cpp:42-55: the
// pixel count of default-constructed ones, then every non-delta vertex past
// the first of each light path, up to an emitter, path-major) in a block of
// their own; HashGrid::Build over each block; then k_vcm, one lane per pixel
// and pass: the connections of k_bdpt with vcmMisWeight, and the merges.

// true: vertex i of a light path is a light point; stop: the path's points end there
__device__ __forceinline__ bool light_point(const SceneDev& S, const BVert& v, bool& stop) {
    stop = emissive(S, v.contact);
    return !stop && !(v.flags & kVDelta);
}

__global__ __launch_bounds__(256) void k_vcm_point_count(SceneDev S, const BVert* verts, const uint32_t* counts,
                                                         uint32_t lanes, uint32_t maxv, uint32_t* pc) {
    const uint32_t k = blockIdx.x * 256 + threadIdx.x;
    if (k >= lanes) return;
    const BVert* L = verts + (size_t)k * 2 * maxv + maxv;
    const uint32_t nl = min(counts[2 * k + 1], maxv);
    uint32_t m = 0;
    for (uint32_t i = 1; i < nl; i++) {
        bool stop;
        const bool keep = light_point(S, L[i], stop);
        if (stop) break;
        m += keep;
    }
    pc[k] = m;
}

// Pass b's block of points starts at b * npix + offs[b * npix] (offs: exclusive
// sums of the counts over all lanes): the npix default points (origin, no
// path), then the points of the pass's paths; src holds the lane in the batch
// and the vertex.
__global__ __launch_bounds__(256) void k_vcm_point_write(SceneDev S, const BVert* verts, const uint32_t* counts,
                                                         uint32_t npix, uint32_t lanes, uint32_t maxv,
                                                         const uint32_t* offs, float* pos, uint32_t* src) {
    const uint32_t k = blockIdx.x * 256 + threadIdx.x;
    if (k >= lanes) return;
    const uint32_t b = k / npix, p = k % npix;
    const size_t block = (size_t)b * npix + offs[(size_t)b * npix];
    pos[3 * (block + p)] = 0.f;
    pos[3 * (block + p) + 1] = 0.f;
    pos[3 * (block + p) + 2] = 0.f;
    src[2 * (block + p)] = WR_NONE;
    src[2 * (block + p) + 1] = WR_NONE;
    const BVert* L = verts + (size_t)k * 2 * maxv + maxv;
    const uint32_t nl = min(counts[2 * k + 1], maxv);
    size_t j = block + npix + (offs[k] - offs[(size_t)b * npix]);
    for (uint32_t i = 1; i < nl; i++) {
        bool stop;
        const bool keep = light_point(S, L[i], stop);
        if (stop) break;
        if (!keep) continue;
        pos[3 * j] = L[i].o.x;
        pos[3 * j + 1] = L[i].o.y;
        pos[3 * j + 2] = L[i].o.z;
        src[2 * j] = k;
        src[2 * j + 1] = i;
        j++;
    }
}

// The first offset of every pass: starts[b] = offs[b * npix], b = 0..npass.
__global__ void k_vcm_pass_starts(const uint32_t* offs, uint32_t npix, uint32_t npass, uint32_t* starts) {
    const uint32_t b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b <= npass) starts[b] = offs[(size_t)b * npix];
}

// The merges of the VCM lanes, one entry per light point in reach of an eye
// vertex: word 0 the eye vertex (merge_entry.h), word 1 the light point; count
// behind them, of all merges, queued or not: in 64 bits, since a pass of a
// megapixel with a radius of a tenth of the scene has more than 2^32.  A
// separate kernel takes one merge per lane, so the uneven number of merges per
// pixel does not leave most lanes of a wave idle.
struct MergeQueue {
    uint32_t* ent;
    uint32_t cap;
    __device__ __forceinline__ unsigned long long* count() const {
        return reinterpret_cast<unsigned long long*>(ent + 2 * (size_t)cap);
    }
};

// One merge (throughputByMerging, vcmTracer.cpp:196-213): the eye vertex i of
// lane `lane` with light point pi of the lane's pass.  Returns the contribution
// (before the division by the pixel count); zero when the merge gives nothing.
template <bool TABLE>
__device__ __forceinline__ f3 vcm_merge(const SceneDev& S, const CamDev& cam, uint32_t npix, uint32_t maxv,
                                        const BVert* verts, const Prefixes<TABLE>& prefix, const VcmGrid& G,
                                        uint64_t lane, int i, uint32_t pi) {
    const uint32_t p = (uint32_t)(lane % npix);
    const uint32_t k = G.src[2 * (size_t)pi], j = G.src[2 * (size_t)pi + 1];
    const size_t li = (size_t)k * 2 * maxv + maxv + (j - 1), ei = lane * 2 * maxv;
    BVert lc = verts[li], ec = verts[ei + i];
    if (!connect_edge_vm(S, verts + ei, i, lc, ec)) return mk(0.f, 0.f, 0.f);
    const VcmTerms vm{G.r, (double)npix, true};
    f3 color;
    float prob;
    const float w = color_prob_weight(S, cam, p, lc, prefix.at(S, cam, k, false, (int)j - 1), (int)j - 1, ec,
                                      prefix.at(S, cam, lane, true, i), i, color, prob, &vm);
    if (len(color) == 0.f || prob == 0.f) return mk(0.f, 0.f, 0.f);
    return divs(muls(color, w), prob);
}

template <bool TABLE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void k_vcm(
    SceneDev S, CamDev cam, uint32_t npix, uint32_t npass, uint32_t maxv, const BVert* verts, const BPrefix* table,
    const uint32_t* counts, float* pix_all, VisQueue Q, const VcmGrid* grids, MergeQueue M, uint32_t width) {
    const Prefixes<TABLE> prefix{table, verts, npix, maxv};
    // every lane of a wave stays to the end (the merge reservations below are
    // wave-wide scans); a lane past the last one stands in for lane 0 and does
    // nothing
    const uint32_t wl = threadIdx.x & 63u;
    const uint64_t lane0 = (uint64_t)(blockIdx.x * 4 + (threadIdx.x >> 6)) * width;
    const bool valid = wl < width && lane0 + wl < (uint64_t)npass * npix;
    const uint64_t lane = valid ? lane0 + wl : 0;
    const uint32_t kb = (uint32_t)(lane / npix), p = (uint32_t)(lane % npix);
    const VcmGrid G = grids[kb];
    float* pix = pix_all + 3 * (size_t)kb * npix;
    StackSpill spill;
    LaneStack st(&spill);
    const SceneCtx sc = make_scene_ctx(S);
    const BVert* E = verts + lane * 2 * maxv;
    const uint32_t ne = counts[2 * lane], nl = counts[2 * lane + 1];
    const int max_eye = (int)(ne < maxv ? ne : maxv), max_light = (int)(nl < maxv ? nl : maxv);
    // throughputByConnecting (vcmTracer.cpp:88-173): k_bdpt's connections with vcmMisWeight
    __shared__ PairTable tables[4];
    f3 own = connect_wave(S, sc, cam, npix, maxv, lane0, verts, prefix, valid ? max_eye : 0,
                          valid ? max_light : 0, pix_all, Q, st, grids, tables[threadIdx.x >> 6]);
    // throughputByMerging (vcmTracer.cpp:175-217): the light points within the
    // radius of every non-delta eye vertex before an emitter, in the grid's
    // order (HashGrid::Process); the default points have no path and give
    // nothing.  Each merge is queued for k_vcm_merge: per eye vertex the lane
    // counts its points in reach, the wave reserves their slots with one
    // atomic (an exclusive scan of the counts), and the lane writes them.
    bool alive = valid;
    for (int i = 1; i < (int)maxv; i++) {
        bool act = alive && i < max_eye;
        BVert ev;
        if (act) {
            ev = E[i];
            if (emissive(S, ev.contact)) {
                alive = false;
                act = false;
            } else if (ev.flags & kVDelta) {
                act = false;
            }
        }
        if (i + 1 >= max_eye) alive = false;
        int pc[6];
        const bool q = act && query_corner(G.g, ev.o, pc);
        uint32_t cnt = 0;
        for (int pass2 = 0; pass2 < 2; pass2++) {
            uint32_t k = 0;  // cap where the queue is full
            if (pass2) {     // the slots of this lane's merges: the wave's scan, one atomic
                unsigned long long v = cnt;
                for (int off = 1; off < 64; off <<= 1) {
                    const unsigned long long t = __shfl_up(v, off, 64);
                    if (wl >= (uint32_t)off) v += t;
                }
                const unsigned long long total = __shfl(v, 63, 64);
                unsigned long long base = 0;
                if (wl == 0 && total) base = atomicAdd(M.count(), total);
                k = (uint32_t)min(__shfl(base, 0, 64) + (v - cnt), (unsigned long long)M.cap);
                if (cnt == 0) break;
            }
            f3 contrib = mk(0.f, 0.f, 0.f);
            for (int c8 = 0; q && c8 < 8; c8++) {
                const uint32_t cell = query_cell(G.g, pc, c8);
                int a = cell == 0 ? 0 : G.ends[cell - 1];
                const int b = G.ends[cell];
                // the default points lead their cell's range (the sort keeps input order in a cell)
                int hi = b;
                while (a < hi) {
                    const int mid = (a + hi) >> 1;
                    if (G.idx[mid] < npix) a = mid + 1;
                    else hi = mid;
                }
                for (; a < b; a++) {
                    if (!grid_near(G.g, G.pos, ev.o, a)) continue;
                    const uint32_t pi = G.idx[a];
                    if (!pass2) {
                        cnt++;
                    } else if (k < M.cap) {
                        M.ent[2 * (size_t)k] = wr::merge_entry((uint32_t)lane, (uint32_t)i, maxv);
                        M.ent[2 * (size_t)k + 1] = pi;
                        k++;
                    } else {  // queue full: merge here
                        contrib = add(contrib, vcm_merge(S, cam, npix, maxv, verts, prefix, G, lane, i, pi));
                    }
                }
            }
            if (pass2) own = add(own, divs(contrib, (float)npix));
        }
        if (__ballot(alive) == 0) break;
    }
    if (valid) atomic_add3(pix, p, own);
}

// The queued merges of k_vcm, one per lane, each added to its pixel of its pass.
template <bool TABLE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void k_vcm_merge(
    SceneDev S, CamDev cam, uint32_t npix, uint32_t maxv, const BVert* verts, const BPrefix* table, float* pix_all,
    MergeQueue M, const VcmGrid* grids) {
    const Prefixes<TABLE> prefix{table, verts, npix, maxv};
    const uint32_t n = (uint32_t)min(*M.count(), (unsigned long long)M.cap);
    for (uint32_t e = blockIdx.x * 256 + threadIdx.x; e < n; e += gridDim.x * 256) {
        const uint32_t w0 = M.ent[2 * (size_t)e], pi = M.ent[2 * (size_t)e + 1];
        const uint32_t lane = wr::merge_lane(w0, maxv);
        const int i = (int)wr::merge_vertex(w0, maxv);
        const uint32_t kb = lane / npix, p = lane % npix;
        const f3 c = vcm_merge(S, cam, npix, maxv, verts, prefix, grids[kb], lane, i, pi);
        if (c.x != 0.f || c.y != 0.f || c.z != 0.f)
            atomic_add3(pix_all + 3 * (size_t)kb * npix, p, divs(c, (float)npix));
    }
}

// ---- PhotonMap (photonMap.cpp:21-680), progressive photon mapping ----------
// The light points and per-pass grids of VCMTracer (the same light paths);
// the eye "merge path" of every pixel and pass (PpmWalk: samplePath with
// maxPathLen MERGE_LEN = 10, photonMap.cpp:10,150-190) up to its first
// emitter (its emitted radiance) or first non-specular, i.e. diffuse, vertex
// (the kernel density estimate of the photons around it, photonMap.cpp:
// 198-248,656-668), times the camera vertex's factor only (photonMap.cpp:
// 670-674).  No object here is a volume or an anisotropic glossy object, so
// every photon is a surface photon and every estimate the plain range query.
constexpr uint32_t kMergeLen = 10;

// The throughput of every light path before each of its records (radiance /
// directionProb / originProb * cosine of the records before it), kept in the
// radiance of the eye-side record of the same index, which PhotonMap has no
// other use for: a photon in reach costs one record instead of its whole path
// (Cornell 256^2 x 8 passes: 0.6 ms less in the estimates, 0.11 here).
__global__ __launch_bounds__(256) void k_ppm_throughput(uint32_t lanes, uint32_t maxv, BVert* verts,
                                                        const uint32_t* counts) {
    const uint32_t lane = blockIdx.x * 256 + threadIdx.x;
    if (lane >= lanes) return;
    BVert* out = verts + (size_t)lane * 2 * maxv;
    const BVert* L = out + maxv;
    const uint32_t n = min(counts[2 * lane + 1], maxv);
    f3 thr = mk(1.f, 1.f, 1.f);
    for (uint32_t m = 0; m < n; m++) {
        out[m].rad = thr;
        const BVert lm = L[m];
        thr = mulv(thr, divs(divs(lm.rad, lm.dp), lm.op));
        thr = muls(thr, cos_term_v(lm));
    }
}

// Query::Process for the photons around outRay (the eye vertex, its direction
// towards the previous eye vertex).
__device__ f3 ppm_density(const SceneDev& S, const VcmGrid& G, const BVert* verts, uint32_t maxv, uint32_t npix,
                          const BVert& outRay) {
    f3 contrib = mk(0.f, 0.f, 0.f);
    int pc[6];
    if (!query_corner(G.g, outRay.o, pc)) return contrib;
    const float r = G.r;
    for (int c8 = 0; c8 < 8; c8++) {
        const uint32_t cell = query_cell(G.g, pc, c8);
        int a = cell == 0 ? 0 : G.ends[cell - 1];
        const int b = G.ends[cell];
        int hi = b;  // the default points lead their cell's range
        while (a < hi) {
            const int mid = (a + hi) >> 1;
            if (G.idx[mid] < npix) a = mid + 1;
            else hi = mid;
        }
        for (; a < b; a++) {
            if (!grid_near(G.g, G.pos, outRay.o, a)) continue;
            const uint32_t pi = G.idx[a];
            const uint32_t k = G.src[2 * (size_t)pi], j = G.src[2 * (size_t)pi + 1];
            const BVert* L = verts + (size_t)k * 2 * maxv + maxv;
            f3 thr = (L - maxv)[j].rad;  // k_ppm_throughput
            BVert ph = L[j];
            thr = divs(thr, ph.op);
            ph.d = L[j - 1].d;
            const f3 col = mulv(thr, eval_bsdf(S, ph, outRay));
            const float l = len(sub(outRay.o, ph.o));
            const float dist_sqr = l * l;  // powf(l, 2): the correctly rounded square
            if (!legal(col)) continue;
            const float q = 1.f - dist_sqr / (r * r);
            const float sk = 0.f > q ? 0.f : q;
            const float kernel = (float)((double)(3.f * sk * sk) / kPi);  // Kernel (photonMap.cpp:209-212)
            const float norm = kernel / ((float)npix * r * r);
            contrib = add(contrib, muls(col, norm));
        }
    }
    return contrib;
}

// The eye merge paths as a path walk, one per pixel and pass.  What the walk
// keeps of a path lies in its first two eye-side records, of which PhotonMap
// otherwise uses the radiance only (k_ppm_throughput): record 0 the path's
// inside object, then kPpmDensity or 0 in flags and the light it found in n;
// record 1 the vertex whose density k_ppm_density estimates.  (With the
// estimate inside the walk's steps, the lanes of a step waited for the
// longest list of photons in a kernel of 128 registers: 2.3 ms for 256^2 x 8
// passes; 0.36 and 0.47 ms apart.)
constexpr uint32_t kPpmDensity = 1u;
struct PpmWalk {
    CamDev cam;
    uint32_t pass0, npix, maxv;
    uint64_t seed;
    BVert* verts;

    __device__ __forceinline__ bool begin(const SceneCtx& sc, uint32_t lane, LaneStack& st, f3& o, f3& d,
                                          uint32_t& inside, uint32_t& contact) const {
        float rn[4];
        rng4(seed, lane % npix, pass0 + lane / npix, 0, rn);
        o = cam.pos;
        d = cam_dir(cam, lane % npix, rn[0], rn[1]);
        BVert* first = verts + (size_t)lane * 2 * maxv;
        first->inside = find_inside(sc.S, o, d, WR_NONE, st);
        first->n = mk(0.f, 0.f, 0.f);
        first->flags = 0;
        inside = contact = WR_NONE;  // traced without a condition
        return true;
    }

    __device__ __forceinline__ bool step(const SceneCtx& sc, uint32_t lane, uint32_t s, f3 o, f3 d, const PHit& hit,
                                         LaneStack& st, Out& out) const {
        if (hit.rec == WR_NONE) return false;
        BVert* first = verts + (size_t)lane * 2 * maxv;
        const uint32_t inside = first->inside;
        float rn[4];
        rng4(seed, lane % npix, pass0 + lane / npix, s + 1, rn);
        out = scatter(sc, inside != WR_NONE ? inside : hit.obj, o, d, hit, inside, rn, st);
        first->inside = out.inside;
        const bool absorbed = (double)len(out.d) < 0.5;
        if (!absorbed && s + 1 > kMergeLen) return false;  // the terminating record
        if (emissive(sc.S, out.contact)) {                 // the eye path hit a light
            first->n = out.rad;
            return false;
        }
        if (out.contact != WR_NONE && sc.S.objs[out.contact].mat == WR_MAT_DIFFUSE) {  // nonSpecular()
            first->flags = kPpmDensity;
            BVert* v = first + 1;
            v->o = out.o;
            v->d = mk(-d.x, -d.y, -d.z);
            v->n = out.n;
            v->inside = out.inside;
            v->contact = out.contact;
            return false;
        }
        return !absorbed;
    }
};

// Each pixel's value: the camera vertex's factor times what its path found.
__global__ __launch_bounds__(256) void k_ppm_density(SceneDev S, CamDev cam, uint32_t npix, uint32_t lanes,
                                                     uint32_t maxv, const BVert* verts, uint64_t seed, uint32_t pass0,
                                                     float* pix_all, const VcmGrid* grids) {
    const uint32_t lane = blockIdx.x * 256 + threadIdx.x;
    if (lane >= lanes) return;
    const uint32_t kb = lane / npix, p = lane % npix;
    const BVert* first = verts + (size_t)lane * 2 * maxv;
    f3 surface = first->n;
    if (first->flags & kPpmDensity) {
        BVert v = first[1];
        v.flags = 0;
        surface = ppm_density(S, grids[kb], verts, maxv, npix, v);
    }
    float rn[4];
    rng4(seed, p, pass0 + kb, 0, rn);
    BVert c;
    c.d = cam_dir(cam, p, rn[0], rn[1]);
    c.n = cam.front;
    c.flags = kVCamera;
    c.contact = WR_NONE;
    const f3 color = mulv(mulv(mk(1.f, 1.f, 1.f), surface),
                          divs(divs(muls(mk(1.f, 1.f, 1.f), cos_term_v(c)), 1.f), 1.f));
    float* px = pix_all + 3 * (size_t)lane;
    px[0] = color.x;
    px[1] = color.y;
    px[2] = color.z;
}

}  // namespace wrd

namespace wr {

size_t bdpt_vertex_bytes() { return sizeof(wrd::BVert); }

float vcm_radius(float base, uint32_t pass) {
    const float alpha = (float)(2.0 / 3);  // vcmTracer.h:39
    const float r = base * std::sqrt(std::pow((float)(pass + 1), alpha - 1.f));
    return (double)r > 1e-5 ? r : (float)1e-5;
}

static wrd::CamDev make_cam_dev(const CamHost& ch) {
    wrd::CamDev cam;
    cam.pos = wrd::f3{ch.pos[0], ch.pos[1], ch.pos[2]};
    cam.front = wrd::f3{ch.front[0], ch.front[1], ch.front[2]};
    cam.right = wrd::f3{ch.right[0], ch.right[1], ch.right[2]};
    cam.top = wrd::f3{ch.top[0], ch.top[1], ch.top[2]};
    cam.dist = ch.dist;
    cam.W = ch.W;
    cam.H = ch.H;
    return cam;
}

// The light sub-paths of `lanes` lanes, and their eye sub-paths when eye.
static hipError_t run_subpaths(wr_ctx* ctx, const SceneDev& S, const wr_tree_hdr& H, const wrd::CamDev& cam,
                               uint32_t max_depth, uint64_t seed, uint32_t pass0, uint32_t lanes, uint32_t npix,
                               uint32_t maxv, wrd::BVert* V, uint32_t* counts, bool eye) {
    const wrd::SubpathWalk P{cam, max_depth, pass0, npix, maxv, eye ? lanes : 0u, seed, V, counts};
    return run_walk(ctx, S, H, P, eye ? 2 * lanes : lanes, max_depth + 1);
}

// The light sub-paths of passes [pass0, pass0 + npass) (and their eye sub-paths
// when eye), their light points and one grid per pass, described in vb.grids;
// the grids' buffers come from mem.  vb.err is set on the device if a pass's
// points spread over too many cells.
static int light_point_grids(wr_ctx* ctx, Scratch& mem, const SceneDev& S, const wr_tree_hdr& H,
                             const wrd::CamDev& cam, uint32_t npix, uint32_t max_depth, uint64_t seed,
                             uint32_t pass0, uint32_t npass, float base_radius, uint32_t maxv, wrd::BVert* V, uint32_t* counts, const VcmBufs& vb, bool eye,
                             const char* who) {
    hipStream_t st = ctx->stream;
    const uint32_t lanes = npass * npix;  // the caller keeps npass * npix below 2^31
    const uint32_t blocks = (lanes + 255) / 256;
    hipError_t e = hipMemsetAsync(vb.pc + lanes, 0, sizeof(uint32_t), st);
    if (e == hipSuccess) e = hipMemsetAsync(vb.err, 0, sizeof(uint32_t), st);
    if (e != hipSuccess) return hip_fail(ctx, e, who);
    if ((e = run_subpaths(ctx, S, H, cam, max_depth, seed, pass0, lanes, npix, maxv, V, counts, eye)) != hipSuccess)
        return hip_fail(ctx, e, who);
    wrd::k_vcm_point_count<<<blocks, 256, 0, st>>>(S, V, counts, lanes, maxv, vb.pc);
    if ((e = hipGetLastError()) != hipSuccess) return hip_fail(ctx, e, who);
    size_t tb = vb.scan_bytes;
    if ((e = hipcub::DeviceScan::ExclusiveSum(vb.scan, tb, vb.pc, vb.offs, (int)lanes + 1, st)) != hipSuccess)
        return hip_fail(ctx, e, who);
    wrd::k_vcm_pass_starts<<<(npass + 1 + 63) / 64, 64, 0, st>>>(vb.offs, npix, npass, vb.starts);
    std::vector<uint32_t> starts(npass + 1);
    if ((e = hipGetLastError()) != hipSuccess ||
        (e = hipMemcpyAsync(starts.data(), vb.starts, sizeof(uint32_t) * (npass + 1), hipMemcpyDeviceToHost, st)) !=
            hipSuccess ||
        (e = hipStreamSynchronize(st)) != hipSuccess)
        return hip_fail(ctx, e, who);
    if ((uint64_t)lanes + starts[npass] > vb.cap)
        return fail(ctx, WR_EINVAL, std::string(who) + ": more light points than the buffer holds");
    wrd::k_vcm_point_write<<<blocks, 256, 0, st>>>(S, V, counts, npix, lanes, maxv, vb.offs, vb.pos, vb.src);
    if ((e = hipGetLastError()) != hipSuccess) return hip_fail(ctx, e, who);
    // per pass: HashGrid::Reserve(pixels) + Build(its light points, its radius)
    // (vcmTracer.cpp:30,33,57; photonMap.cpp:48,56,93), all passes together
    std::vector<wrd::GridParams> params(npass);
    for (uint32_t b = 0; b < npass; b++) {
        const float r = vcm_radius(base_radius, pass0 + b);
        params[b] = wrd::GridParams{1.f / (r * 2.f), r * r, r};
    }
    const uint64_t total = (uint64_t)lanes + starts[npass];
    e = build_grids(ctx, mem, vb.pos, vb.src, total, vb.starts, npix, npass, npix, params.data(),
                    (wrd::GridView*)vb.grids, vb.err, nullptr, vb.cap - total >= total ? vb.pos + 3 * total : nullptr);
    if (e != hipSuccess) return hip_fail(ctx, e, who);
    return WR_OK;
}

// Once the stream has been synchronised: the error of a pass's grid.
static int check_grids(wr_ctx* ctx, uint32_t err, const char* who) {
    if (!err) return WR_OK;
    return fail(ctx, WR_EINVAL, std::string(who) + ": too many cells across the light points' box for this radius");
}

// Lanes (pixel and pass) of each wave of the connection kernels: fewer than 64
// while that leaves fewer than `waves` waves, so that a small image fills the
// chip (the lanes without a pixel still take their share of the pairs).  Cornell
// 64x64, 1 pass: BidirectionalPathTracer 1,018 -> 916 us, VCMTracer 1,615 ->
// 1,278 us; 100x100, 2 passes, VCMTracer 2.01 -> 1.81 ms.  k_vcm's merges are a
// lane's own: with its line at 4,096 waves 256x256, 4 passes took 7.5 ms, 7.1 at 1,024.
constexpr uint64_t kBdptWaves = 2048, kVcmWaves = 1024;

static uint32_t connect_width(uint64_t lanes, uint64_t waves) {
    uint32_t width = 64;
    while (width > 4 && lanes < waves * width) width /= 2;
    return width;
}

int launch_vcm_passes(wr_ctx* ctx, const SceneDev& S, const wr_tree_hdr& H, const CamHost& ch, uint32_t max_depth,
                      uint64_t seed, uint32_t pass0, uint32_t npass, float base_radius, uint32_t maxv, void* verts,
                      float* pix, const BdptQueue& q, const VcmBufs& vb, const FilmBufs& film) {
    hipStream_t st = ctx->stream;
    const wrd::CamDev cam = make_cam_dev(ch);
    const uint32_t npix = ch.W * ch.H;
    const uint32_t lanes = npass * npix;
    wrd::BVert* V = (wrd::BVert*)verts;
    hipError_t e = hipMemsetAsync(pix, 0, sizeof(float) * 3 * (size_t)lanes, st);
    if (e == hipSuccess) e = hipMemsetAsync(q.count, 0, sizeof(uint32_t), st);
    if (e != hipSuccess) return hip_fail(ctx, e, "wr_render_vcm");
    Scratch mem(*ctx->pool);  // the grids'
    int rc = light_point_grids(ctx, mem, S, H, cam, npix, max_depth, seed, pass0, npass, base_radius, maxv, V, q.counts,
                               vb, true, "wr_render_vcm");
    if (rc != WR_OK) return rc;
    // a merge needs the prefixes of any light path of its pass: without room for
    // all of them they are formed where they are needed
    wrd::BPrefix* prefix = nullptr;
    e = mem.get(&prefix, sizeof(wrd::BPrefix) * 2 * maxv * (size_t)lanes);
    if (e != hipSuccess && e != hipErrorOutOfMemory) return hip_fail(ctx, e, "wr_render_vcm");
    if (prefix)
        wrd::k_bdpt_prefix<<<(uint32_t)((2ull * lanes + 255) / 256), 256, 0, st>>>(S, cam, npix, 0, lanes, maxv, V,
                                                                                  q.counts, prefix);
    const wrd::VisQueue Q{q.rays, q.pay, q.dst, q.count, q.cap};
    const wrd::MergeQueue M{vb.mq, vb.mq_cap};
    e = hipMemsetAsync(vb.mq + 2 * (size_t)vb.mq_cap, 0, sizeof(uint64_t), st);
    if (e != hipSuccess) return hip_fail(ctx, e, "wr_render_vcm");
    const uint32_t width = connect_width(lanes, kVcmWaves);
    (prefix ? wrd::k_vcm<true> : wrd::k_vcm<false>)<<<(lanes + 4 * width - 1) / (4 * width), 256, wrd::kStackLdsBytes,
                                                      st>>>(S, cam, npix, npass, maxv, V, prefix, q.counts, pix, Q,
                                                            (const wrd::VcmGrid*)vb.grids, M, width);
    e = hipGetLastError();
    if (e == hipSuccess) {
        (prefix ? wrd::k_vcm_merge<true> : wrd::k_vcm_merge<false>)<<<4096, 256, 0, st>>>(
            S, cam, npix, maxv, V, prefix, pix, M, (const wrd::VcmGrid*)vb.grids);
        e = hipGetLastError();
    }
    uint32_t nq = 0, grid_err = 0;
    if (e == hipSuccess) e = hipMemcpyAsync(&nq, q.count, sizeof(uint32_t), hipMemcpyDeviceToHost, st);
    if (e == hipSuccess) e = hipMemcpyAsync(&grid_err, vb.err, sizeof(uint32_t), hipMemcpyDeviceToHost, st);
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    if (e != hipSuccess) return hip_fail(ctx, e, "wr_render_vcm");
    if ((rc = check_grids(ctx, grid_err, "wr_render_vcm")) != WR_OK) return rc;
    if (nq > q.cap) nq = q.cap;
    if (nq) {
        if ((e = launch_closest_hit_path(S, H, q.rays, nq, q.hits, q.work, st)) != hipSuccess)
            return hip_fail(ctx, e, "wr_render_vcm: visibility");
        wrd::k_bdpt_accum<<<(nq + 255) / 256, 256, 0, st>>>(nq, q.pay, q.dst, (const uint4*)q.hits, pix);
    }
    wrd::k_bdpt_fold<<<(npix + 255) / 256, 256, 0, st>>>(cam, npass, npix, pix,
                                                         wrd::FilmDev{film.sum, film.comp, film.sumsq});
    if ((e = hipGetLastError()) != hipSuccess) return hip_fail(ctx, e, "wr_render_vcm");
    return WR_OK;
}

int launch_ppm_passes(wr_ctx* ctx, const SceneDev& S, const wr_tree_hdr& H, const CamHost& ch, uint32_t max_depth,
                      uint64_t seed, uint32_t pass0, uint32_t npass, float base_radius, uint32_t maxv, void* verts, uint32_t* counts,
                      float* pix, const VcmBufs& vb, const FilmBufs& film) {
    hipStream_t st = ctx->stream;
    const wrd::CamDev cam = make_cam_dev(ch);
    const uint32_t npix = ch.W * ch.H;
    const uint32_t lanes = npass * npix;
    const uint32_t blocks = (lanes + 255) / 256;
    wrd::BVert* V = (wrd::BVert*)verts;
    Scratch mem(*ctx->pool);  // the grids'
    int rc = light_point_grids(ctx, mem, S, H, cam, npix, max_depth, seed, pass0, npass, base_radius, maxv, V, counts,
                               vb, false, "wr_render_ppm");
    if (rc != WR_OK) return rc;
    wrd::k_ppm_throughput<<<blocks, 256, 0, st>>>(lanes, maxv, V, counts);
    const wrd::PpmWalk P{cam, pass0, npix, maxv, seed, V};
    hipError_t e = run_walk(ctx, S, H, P, lanes, wrd::kMergeLen + 1);
    if (e != hipSuccess) return hip_fail(ctx, e, "wr_render_ppm");
    wrd::k_ppm_density<<<blocks, 256, 0, st>>>(S, cam, npix, lanes, maxv, V, seed, pass0, pix,
                                               (const wrd::VcmGrid*)vb.grids);
    wrd::k_bdpt_fold<<<(npix + 255) / 256, 256, 0, st>>>(cam, npass, npix, pix,
                                                         wrd::FilmDev{film.sum, film.comp, film.sumsq});
    uint32_t grid_err = 0;
    e = hipGetLastError();
    if (e == hipSuccess) e = hipMemcpyAsync(&grid_err, vb.err, sizeof(uint32_t), hipMemcpyDeviceToHost, st);
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    if (e != hipSuccess) return hip_fail(ctx, e, "wr_render_ppm");
    return check_grids(ctx, grid_err, "wr_render_ppm");  // an error marks the film as part-written
}

size_t vcm_grid_bytes() { return sizeof(wrd::VcmGrid); }

size_t vcm_scan_bytes(uint32_t lanes) {
    size_t tb = 0;
    (void)hipcub::DeviceScan::ExclusiveSum(nullptr, tb, (uint32_t*)nullptr, (uint32_t*)nullptr, (int)lanes + 1);
    return tb;
}

hipError_t launch_bdpt_passes(wr_ctx* ctx, const SceneDev& S, const wr_tree_hdr& H, const CamHost& ch,
                              uint32_t max_depth, uint64_t seed, uint32_t pass0, uint32_t npass, uint32_t maxv, void* verts, float* pix,
                              const BdptQueue& q, const FilmBufs& film) {
    hipStream_t st = ctx->stream;
    const wrd::CamDev cam = make_cam_dev(ch);
    const uint32_t npix = ch.W * ch.H;
    const uint64_t lanes = (uint64_t)npass * npix;
    hipError_t e = hipMemsetAsync(pix, 0, sizeof(float) * 3 * (size_t)lanes, st);
    if (e == hipSuccess) e = hipMemsetAsync(q.count, 0, sizeof(uint32_t), st);
    if (e != hipSuccess) return e;
    const wrd::VisQueue Q{q.rays, q.pay, q.dst, q.count, q.cap};
    e = run_subpaths(ctx, S, H, cam, max_depth, seed, pass0, (uint32_t)lanes, npix, maxv, (wrd::BVert*)verts, q.counts,
                     true);
    if (e != hipSuccess) return e;
    // the prefixes of at most 4 GiB of lanes at a time (all of them up to a million
    // lanes at the longest paths), fewer where the device has no room for them
    Scratch mem(*ctx->pool);
    const size_t lane_bytes = sizeof(wrd::BPrefix) * 2 * maxv;
    uint64_t part = std::min<uint64_t>(lanes, (4ull << 30) / lane_bytes);
    wrd::BPrefix* prefix = nullptr;
    while ((e = mem.get(&prefix, lane_bytes * part)) == hipErrorOutOfMemory && part > 1024) part = (part + 3) / 4;
    if (e != hipSuccess) return e;
    for (uint64_t a = 0; a < lanes; a += part) {
        const uint32_t first = (uint32_t)a, end = (uint32_t)std::min<uint64_t>(lanes, a + part), n = end - first;
        wrd::k_bdpt_prefix<<<(uint32_t)((2ull * n + 255) / 256), 256, 0, st>>>(
            S, cam, npix, first, end, maxv, (const wrd::BVert*)verts, q.counts, prefix);
        const uint32_t width = connect_width(n, kBdptWaves);
        wrd::k_bdpt<<<(uint32_t)((n + 4ull * width - 1) / (4 * width)), 256, wrd::kStackLdsBytes, st>>>(
            S, cam, first, end, npix, maxv, (const wrd::BVert*)verts, prefix - (ptrdiff_t)first * 2 * maxv, q.counts,
            pix, Q, width);
    }
    uint32_t nq = 0;
    e = hipMemcpyAsync(&nq, q.count, sizeof(uint32_t), hipMemcpyDeviceToHost, st);
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    if (e != hipSuccess) return e;
    if (nq > q.cap) nq = q.cap;
    if (nq) {
        e = launch_closest_hit_path(S, H, q.rays, nq, q.hits, q.work, st);
        if (e != hipSuccess) return e;
        wrd::k_bdpt_accum<<<(nq + 255) / 256, 256, 0, st>>>(nq, q.pay, q.dst, (const uint4*)q.hits, pix);
    }
    wrd::k_bdpt_fold<<<(npix + 255) / 256, 256, 0, st>>>(cam, npass, npix, pix,
                                                         wrd::FilmDev{film.sum, film.comp, film.sumsq});
    return hipGetLastError();
}

}  // namespace wr
