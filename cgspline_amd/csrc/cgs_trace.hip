// SPDX-License-Identifier: MIT
//
// Ray-query and render kernels for gfx950.
//
// One ray per lane; 256-lane workgroups (4 waves).  A lane runs the reference's
// per-ray algorithm — top-level traversal, per-object local ray, per-object
// hashed traversal, Bézier clipping at each leaf — so every result equals the
// CPU restatement's bit for bit.  The objects a ray reaches are found through
// a cull tree where the scene has one, with the reference's top-level hashed
// traversal for the rays whose answer could depend on the visit order.
//
#include <hip/hip_runtime.h>

#include "cgs_internal.hpp"
#include "cgs_limits.hpp"
#include "cgs_scene_dev.hpp"
#include "cgs_clip_wave.hpp"
#include "cgs_sample.hpp"

namespace cgs
{

constexpr float kClipTol = 0x1p-12f;  // Spline.h:493
constexpr float kClipTol2 = 0x1p-24f; // tolSquare(kClipTol)

// Leaf method of the ray queries.  Clip: Bézier clipping (the reference's
// leaf call, Primitive.cu:234,260); ClipCapped: the same stopped after a
// number of loop passes; Subdiv: subdivision (the commented-out alternative
// at Primitive.cu:236,263, Spline_Subdivision.cu:168-288).  The last two,
// and the Newton polish, are opt-in modes; the default is Clip, unpolished.
enum LeafMethod : int
{
    Clip = 0,
    ClipCapped = 1,
    Subdiv = 2,
};

struct TraceParams
{
    float tol2;         // tolSquare of the clipping tolerance (Spline.h:493 default 2^-12)
    float threshold;    // subdivision threshold (Spline.h:500 default 2^-4)
    uint32_t maxIters;  // ClipCapped: loop passes per patch test
};

struct LocalRay
{
    V3 o, d;
    float max, dinv;
};

// RayTracer.cu:305-314,333: world ray -> object-local ray; t scales by |M d|.
CGS_DEV LocalRay toLocal(const DevObject& ob, V3 o, V3 d, float tmax)
{
    M4 M;
    M.c[0] = ob.w2l[0]; M.c[1] = ob.w2l[1]; M.c[2] = ob.w2l[2]; M.c[3] = ob.w2l[3];
    LocalRay l;
    l.o = project4(m4mul(M, make_float4(o.x, o.y, o.z, 1.0f)));
    V3 ld = m3mul(M, d);
    float len = len3(ld);
    l.max = tmax * len;
    float dinv = 1.0f / len;
    l.d = mul3(dinv, ld);
    l.dinv = dinv;
    return l;
}

// ---------------------------------------------------------------------------
// Subdivision intersection, host semantics (Spline_Subdivision.cu:168-288)
// ---------------------------------------------------------------------------

// Slab test over [0, +inf) (Ds Bounds3::intersect as restated).
CGS_DEV bool boxHit(V3 bmin, V3 bmax, V3 o, V3 d)
{
    float tmin = 0.0f, tmax = __builtin_inff();
    const float b0[3] = {bmin.x, bmin.y, bmin.z}, b1[3] = {bmax.x, bmax.y, bmax.z};
    const float oo[3] = {o.x, o.y, o.z}, dd[3] = {d.x, d.y, d.z};
#pragma unroll
    for (int i = 0; i < 3; i++)
    {
        float inv = 1.0f / dd[i];
        float t0 = (b0[i] - oo[i]) * inv;
        float t1 = (b1[i] - oo[i]) * inv;
        if (inv < 0.0f)
        {
            float s = t0;
            t0 = t1;
            t1 = s;
        }
        if (t0 > tmin) tmin = t0;
        if (t1 < tmax) tmax = t1;
        if (tmin > tmax) return false;
    }
    return true;
}

// Möller–Trumbore (Ds triangle::intersect as restated): t in (0, +inf).
CGS_DEV bool triHit(V3 o, V3 d, V3 p0, V3 p1, V3 p2, float& t)
{
    V3 e1 = sub3(p1, p0), e2 = sub3(p2, p0);
    V3 s1 = cross3(d, e2);
    float det = dot3(s1, e1);
    if (__builtin_fabsf(det) < 1.17549435e-38f) return false;
    float inv = 1.0f / det;
    V3 s = sub3(o, p0);
    float b1 = dot3(s, s1) * inv;
    if (b1 < 0.0f || b1 > 1.0f) return false;
    V3 s2 = cross3(s, e1);
    float b2 = dot3(d, s2) * inv;
    if (b2 < 0.0f || b1 + b2 > 1.0f) return false;
    float tt = dot3(e2, s2) * inv;
    if (!(tt > 0.0f)) return false;
    t = tt;
    return true;
}

CGS_DEV void subpatch4(float4 (&p)[16], bool vside, float a, float b)
{
    float iu = 1.0f - a;
    float vv = (b - a) / iu;
    float ivv = 1.0f - vv;
#pragma unroll
    for (int k = 0; k < 4; k++)
    {
        const int i0 = vside ? k : 4 * k;
        const int st = vside ? 4 : 1;
        slice1(p[i0].x, p[i0 + st].x, p[i0 + 2 * st].x, p[i0 + 3 * st].x, a, iu, vv, ivv);
        slice1(p[i0].y, p[i0 + st].y, p[i0 + 2 * st].y, p[i0 + 3 * st].y, a, iu, vv, ivv);
        slice1(p[i0].z, p[i0 + st].z, p[i0 + 2 * st].z, p[i0 + 3 * st].z, a, iu, vv, ivv);
        slice1(p[i0].w, p[i0 + st].w, p[i0 + 2 * st].w, p[i0 + 3 * st].w, a, iu, vv, ivv);
    }
}

CGS_DEV void projBox(const float4 (&p)[16], V3& mn, V3& mx)
{
    const float big = 3.40282347e+38f;
    mn = {big, big, big};
    mx = {-big, -big, -big};
#pragma unroll
    for (int i = 0; i < 16; i++)
    {
        V3 q = project4(p[i]);
        if (q.x < mn.x) mn.x = q.x;
        if (q.x > mx.x) mx.x = q.x;
        if (q.y < mn.y) mn.y = q.y;
        if (q.y > mx.y) mx.y = q.y;
        if (q.z < mn.z) mn.z = q.z;
        if (q.z > mx.z) mx.z = q.z;
    }
}

constexpr int kSubdivStack = 64;

// The subdivision test of one patch against a ray (o, d unit), host
// semantics: returns found; best/bu/bv updated by a nearer triangle hit;
// overflow when the region stack is exhausted.
template<bool ANY>
CGS_DEV bool subdividePatch(const float4* __restrict__ S, V3 o, V3 d, float threshold, float& best, float& bu,
                            float& bv, bool& overflow)
{
    bool found = false;
    float4 sub[16];
#pragma unroll
    for (int i = 0; i < 16; i++) sub[i] = S[i];
    V3 bmn, bmx;
    projBox(sub, bmn, bmx);
    if (!boxHit(bmn, bmx, o, d)) return false;
    float4 st[kSubdivStack]; // (umin, vmin, umax, vmax)
    uint8_t side[kSubdivStack];
    int sp = 0;
    st[sp] = {0.0f, 0.0f, 0.5f, 1.0f}; side[sp++] = 0;
    st[sp] = {0.5f, 0.0f, 1.0f, 1.0f}; side[sp++] = 0;
    while (sp > 0)
    {
        sp--;
        const float4 e = st[sp];
        const bool es = side[sp] != 0;
#pragma unroll
        for (int i = 0; i < 16; i++) sub[i] = S[i];
        subpatch4(sub, true, e.y, e.w);
        subpatch4(sub, false, e.x, e.z);
        projBox(sub, bmn, bmx);
        if (!boxHit(bmn, bmx, o, d)) continue;
        float x = 0.5f * (e.x + e.z);
        float y = 0.5f * (e.y + e.w);
        if ((e.z - e.x) < threshold && (e.w - e.y) < threshold)
        {
            V3 p00 = project4(sub[0]), p10 = project4(sub[3]), p01 = project4(sub[12]), p11 = project4(sub[15]);
            float t = 0.0f, t1 = 0.0f;
            bool b0 = triHit(o, d, p10, p01, p00, t);
            bool b1 = triHit(o, d, p01, p10, p11, t1);
            if (b0)
            {
                if (b1 && t1 < t) t = t1;
            }
            else if (b1)
            {
                t = t1;
                b0 = true;
            }
            if (b0 && t < best)
            {
                best = t;
                bu = x;
                bv = y;
                found = true;
                if (ANY) break;
            }
        }
        else
        {
            if (sp + 2 > kSubdivStack)
            {
                overflow = true;
                break;
            }
            if (es)
            {
                st[sp] = {e.x, e.y, x, e.w}; side[sp++] = !es;
                st[sp] = {x, e.y, e.z, e.w}; side[sp++] = !es;
            }
            else
            {
                st[sp] = {e.x, e.y, e.z, y}; side[sp++] = !es;
                st[sp] = {e.x, y, e.z, e.w}; side[sp++] = !es;
            }
        }
    }
    return found;
}

// ---------------------------------------------------------------------------
// Cull-tree enumeration (cgs_cull.cpp): the elements (objects or patches)
// whose reference leaf box a ray passes, in the tree's near-to-far order
// ---------------------------------------------------------------------------

CGS_DEV bool cullable(V3 o, V3 Dinv)
{
    auto ok = [](float oi, float di) { return __builtin_isfinite(oi) && __builtin_isfinite(di) && di != 0.0f; };
    return ok(o.x, Dinv.x) && ok(o.y, Dinv.y) && ok(o.z, Dinv.z);
}

// A lane's place in one traversal, kept between two patch tests.  In a cull
// tree: the next node (EMPTY: none) and the elements elem..elemEnd-1 of the
// leaf being read.  In a hashed BVH: its TravState, and the next slot of the
// leaf list being read (EMPTY: none).
struct Walk
{
    TravState st;        // cull tree: st.node is the next node
    uint32_t leaf;       // cull tree: elem
    CGS_DEV uint32_t& elem() { return leaf; }
    CGS_DEV uint32_t& elemEnd() { return st.key; }
};
CGS_DEV Walk cullWalk(uint32_t root) { return Walk {TravState {root, 0u, 0u, RingState {}}, 0u}; }
CGS_DEV Walk hashWalk(uint32_t root) { return Walk {TravState {root, 1u, 0u, RingState {}}, EMPTY}; }

// The next element whose reference leaf box the ray passes with entry
// below tmax and at most lim; its entry in L0.  EMPTY at the end.
CGS_DEV uint32_t cullNext(const SceneDev& sc, int oct, V3 o, V3 Dinv, float lim, float tmax, Walk& it, float& L0)
{
    uint32_t node = it.st.node, elem = it.elem(), elemEnd = it.elemEnd(), found = EMPTY;
    while (true)
    {
        if (elem < elemEnd)
        {
            CGS_COUNT(kWorkCullElem);
            const float4 a = sc.cullElems[2 * (size_t)elem], b = sc.cullElems[2 * (size_t)elem + 1];
            elem++;
            float l;
            if (nodeIntersect<-1>(l, {a.x, a.y, a.z}, {b.x, b.y, b.z}, o, Dinv) && l < tmax && l <= lim)
            {
                L0 = l;
                found = __float_as_uint(a.w);
                break;
            }
            continue;
        }
        if (node == EMPTY) break;
        CGS_COUNT(kWorkCullNode);
        const float4 a = sc.cullNodes[2 * (size_t)node], b = sc.cullNodes[2 * (size_t)node + 1];
        const uint2 l = sc.cullLinks[8 * (size_t)node + oct];
        float tn;
        const bool pass = nodeIntersect<-1>(tn, {a.x, a.y, a.z}, {b.x, b.y, b.z}, o, Dinv) && tn <= lim;
        const uint32_t count = __float_as_uint(b.w);
        if (pass && count)
        {
            elem = __float_as_uint(a.w);
            elemEnd = elem + count;
        }
        node = pass && !count ? l.x : l.y;
    }
    it.st.node = node;
    it.elem() = elem;
    it.elemEnd() = elemEnd;
    return found;
}

// The next element of a hashed BVH's stackless traversal (rt/BVH.h:178-350)
// against `limit`: the closest-hit traversal's is the caller's nearest hit so
// far, the any-hit one's the ray's end.  EMPTY at the end.  OCTANTS:
// specialise the node loop on the wave's direction octant (worth its code
// size where a wave's rays are coherent: in world space).  LOW: the BVH's
// nodes lie in the first 4 GiB of the node array (loadNodeLow).
template<bool OCTANTS, bool LOW, bool BIG>
CGS_DEV uint32_t hashNext(const BVHRef& b, V3 o, V3 Dinv, float limit, const NodeCache& nc, const SiblingRing& ring,
                          Walk& it)
{
    const int oct = OCTANTS ? waveOctant(o, Dinv, b.record->finiteBoxes) : -1;
    while (true)
    {
        if (it.leaf != EMPTY)
        {
            const uint32_t e = b.indices[it.leaf];
            if (e != EMPTY)
            {
                CGS_COUNT(kWorkLeaf);
                it.leaf++;
                return e;
            }
            it.leaf = EMPTY;
            if (!ascend<BIG>(b, nc, ring, it.st)) return EMPTY;
        }
        it.leaf = OCTANTS ? nextLeafOct<LOW, BIG>(oct, b, nc, ring, o, Dinv, limit, it.st)
                          : nextLeaf<-1, LOW, BIG>(b, nc, ring, o, Dinv, limit, it.st);
        if (it.leaf == EMPTY) return EMPTY;
    }
}

// How far beyond the nearest hit so far an object's box entry may lie and
// the object still be tested: 2^-10 of the distance plus the origin's
// magnitude, orders of magnitude above the FP32 rounding of a hit distance
// or a box entry.
CGS_DEV float cullLimit(float best, V3 o)
{
    const float mag = fmax_(__builtin_fabsf(o.x), fmax_(__builtin_fabsf(o.y), __builtin_fabsf(o.z)));
    return best + (best + mag) * 0x1p-10f;
}

CGS_DEV int dirOctant(V3 Dinv)
{
    return (__builtin_signbit(Dinv.x) ? 1 : 0) | (__builtin_signbit(Dinv.y) ? 2 : 0) | (__builtin_signbit(Dinv.z) ? 4 : 0);
}

// A shadow ray's own surface patch, clipped last.  An any-hit answer is the
// OR of the patch tests the traversal reaches, in whatever order, so a query
// may pass over one patch, note that the traversal reached it, and
// clip it only if no other patch is hit (sceneQuery).  A shadow ray that
// grazes its origin patch clips it for up to thousands of passes; one that
// another patch occludes then never does.
struct OriginSkip
{
    int32_t object;
    uint32_t patch;
};

// ---------------------------------------------------------------------------
// Scene queries (Context::intersect, RayTracer.cu:296-383)
// ---------------------------------------------------------------------------
//
// One ray per lane, all lanes of a wave together: each lane walks the objects
// its ray reaches and the patches of each (rt::intersect(BezierSurface),
// Primitive.cu:222-268, on the object-local ray of RayTracer.cu:305-333) until
// its next patch test, and then the wave clips all its lanes' patches in one
// shared clip (clipWave), to which the lanes whose rays are done lend a hand.
// With the test inside each lane's own traversal loops 11 of 64 lanes were
// active on the 1M-patch frame, and a lane whose ray grazes a patch for
// thousands of passes held its wave alone.
//
// Lanes on the reference's top-level traversal (rays with a zero direction
// component, as all of an orthographic view have that looks along an axis
// plane, and restarted ones) wait for each other before the next object.  That
// traversal reads about twice as many nodes as the cull tree's, and with lanes in
// different objects each round of a wave pays for it: 1M parallel rays through
// 2,048 grids took 5.5 ms (closest) and 4.9 (any hit) that way, 3.1 and 2.5 this.
//
// Objects through the cull tree.  The reference's top-level traversal reaches
// object X only if the ray passes X's leaf box with entry L0 below the hit
// distance at that moment (rt/BVH.h:147-266), and every ancestor box contains
// X's box, so it passes there whenever it passes X's (the slab test is
// monotone in the box).  Each object's own result does not depend on the visit
// order (its traversal starts from ray.max·|M d|, RayTracer.cu:311-314).  So:
//  - any hit: the reference's answer is whether some object whose leaf box
//    the ray passes with L0 < ray.max has a hit, in any order;
//  - closest: enumerating every such object whose L0 is not far beyond the
//    nearest hit found so far (a hit lies inside its object's box, up to
//    rounding, for which the slack below leaves a wide margin) finds the
//    nearest hit W.  The reference reaches W when L0_W < t_W (its limit is
//    never below t_W), and then reports W unless another object has a hit at
//    exactly t_W, where its visit order decides.
// A lane starts its ray over by the reference's traversal for a tie, for
// L0_W >= t_W, for a clip-stack overflow on the way (so that overflows are
// reported as in the reference order), and takes it from the first for rays on
// which the slab test could meet a NaN (a zero or non-finite direction
// component, a non-finite origin) and scenes without the tree.
//
// The patches of a large surface through its own cull tree: the same argument
// one level down.  A patch's clip accepts candidates by the running distance
// only (t < best), so a patch's own nearest hit does not depend on the
// distance its test starts from; every patch whose leaf box the local ray
// passes near or before the nearest hit so far is clipped from the local ray's
// max, and the nearest wins.  The object is started over by the reference's
// traversal under the same conditions.  Clipping only (the subdivision leaf
// keeps the reference's traversal).

struct ClosestHit
{
    float t, u, v;
    uint32_t patch;
    int32_t object;
};

// Sibling rings of a lane for the two traversal levels: the top-level BVH
// over objects (CGS_RING_TOP entries; 4096 objects make it 13 levels deep)
// and the patch BVH of one object (CGS_RING_BOT; 256 patches, 9 levels).
#ifndef CGS_RING_TOP
#define CGS_RING_TOP 8
#endif
#ifndef CGS_RING_BOT
#define CGS_RING_BOT 8
#endif
// Octant-specialised node loops in the patch BVHs too (object-local rays:
// lanes in different objects rarely share an octant).
#ifndef CGS_BOT_OCTANTS
#define CGS_BOT_OCTANTS false
#endif
struct Rings
{
    SiblingRing top, bot;
};
constexpr uint32_t kRingWords = CGS_RING_TOP + CGS_RING_BOT ? (CGS_RING_TOP + CGS_RING_BOT) * kRingStride : 1;

CGS_DEV Rings laneRings(uint32_t* lds)
{
    lds_u32* lane = (lds_u32*)lds + threadIdx.x;
    return Rings {{CGS_RING_TOP ? lane : nullptr, CGS_RING_TOP},
                  {CGS_RING_BOT ? lane + CGS_RING_TOP * kRingStride : nullptr, CGS_RING_BOT}};
}

// What a lane's queries work with: its rings, region stack and its wave's
// clip words.
struct LaneMem
{
    Rings rings;
    ClipStack stack;
    lds_u32* clip;
    lds_u32* shadow;     // the wave's shadow rays (ShadowList), else null
};

// One patch test of each lane that has one (`have`), by the chosen leaf
// method.  Every lane of the wave calls it together.
template<int METHOD, bool ANY>
CGS_DEV bool leafTest(bool have, const float4* __restrict__ S, V3 o, V3 d, const TraceParams& tp, float& best, float& bu,
                      float& bv, const LaneMem& lm, bool& overflow)
{
    if constexpr (METHOD == Subdiv)
        return have && subdividePatch<ANY>(S, o, d, tp.threshold, best, bu, bv, overflow);
    else if constexpr (METHOD == ClipCapped)
        return clipWave<ANY, true>(have, S, o, d, tp.tol2, best, bu, bv, lm.stack, lm.clip, overflow, tp.maxIters);
    else
        return clipWave<ANY>(have, S, o, d, kClipTol2, best, bu, bv, lm.stack, lm.clip, overflow);
}

// The closest hit of each lane's ray into h (ANY: whether it has a hit, the
// return value), for the lanes with `run`; every lane of the wave calls it
// together.  ANY with ORIGIN: the patch `origin` is passed over and clipped
// last.  BIG: the scene may have wide hashes and surface cull trees.
// With a List other than NoList the rays come from it (ANY and ORIGIN; the
// ray arguments are not read): a lane whose ray is done gives the answer to
// the list and takes the next one.
struct NoList
{
    static constexpr bool kList = false;
    CGS_DEV bool next(V3&, V3&, float&, OriginSkip&) { return false; }
    CGS_DEV void done(bool, bool) {}
};
template<int METHOD, bool ANY, bool BIG, bool ORIGIN = false, class List = NoList>
CGS_DEV bool sceneQuery(bool run, const SceneDev& sc, const NodeCache& nc, const LaneMem& lm, V3 o, V3 d, float tmax,
                        const TraceParams& tp, ClosestHit& h, bool& overflow, OriginSkip origin = {-1, EMPTY},
                        List list = List {})
{
    constexpr bool LIST = List::kList;
    static_assert(!LIST || (ANY && ORIGIN), "lists hold any-hit rays with an origin patch");
    bool open = LIST;                    // LIST: rays may be left
    bool over1 = false, last = false;    // LIST: this ray's overflow; its origin patch is the current test
    h = {tmax, 0.0f, 0.0f, EMPTY, -1};
    bool hit = false;                    // ANY: the answer
    bool seen = false;                   // ORIGIN: the traversal reached the origin patch
    // the objects
    bool culled = false, tie = false;
    float topL0 = 0.0f, hL0 = 0.0f;      // box entry of the current object, of the nearest hit's
    Walk top {};
    if (run)
    {
        const V3 Dinv {1.0f / d.x, 1.0f / d.y, 1.0f / d.z};
        culled = sc.top.cullRoot != EMPTY && cullable(o, Dinv);
        top = culled ? cullWalk(sc.top.cullRoot) : hashWalk(sc.top.root);
    }
    // the current object (EMPTY: none), its surface and its patches
    uint32_t obj = EMPTY, surface = EMPTY, patchBase = 0;
    LocalRay lr {};
    Walk bot {};
    bool botCulled = false, botTie = false;
    float botL0 = 0.0f, lL0 = 0.0f, lt = 0.0f, lu = 0.0f, lv = 0.0f;
    uint32_t lp = EMPTY;
    while (true)
    {
        uint32_t pid = EMPTY;
        // lanes on the reference's top-level traversal take their next objects together
        const bool inside = __ballot(run && !culled && obj != EMPTY) != 0;
        if (run ? culled || obj != EMPTY || !inside : LIST && open)
        {
            while (true)
            {
                if (LIST && !run)
                {
                    if (!open || !list.next(o, d, tmax, origin))
                    {
                        open = false;
                        break;
                    }
                    run = true;
                    over1 = seen = last = false;
                    obj = EMPTY;
                    culled = sc.top.cullRoot != EMPTY && cullable(o, {1.0f / d.x, 1.0f / d.y, 1.0f / d.z});
                    top = culled ? cullWalk(sc.top.cullRoot) : hashWalk(sc.top.root);
                }
                if (obj == EMPTY)
                {
                    const V3 Dinv {1.0f / d.x, 1.0f / d.y, 1.0f / d.z};
                    if (culled)
                    {
                        obj = cullNext(sc, dirOctant(Dinv), o, Dinv, ANY ? tmax : cullLimit(h.t, o), tmax, top, topL0);
                        if (!ANY && obj == EMPTY && (tie || (h.object >= 0 && !(hL0 < h.t))))
                        {
                            // the reference's visit order decides
                            culled = false;
                            h = {tmax, 0.0f, 0.0f, EMPTY, -1};
                            top = hashWalk(sc.top.root);
                            continue;
                        }
                    }
                    else
                        obj = hashNext<true, true, BIG>(bvhRef(sc, &sc.top), o, Dinv, ANY ? tmax : h.t, nc, lm.rings.top, top);
                    if (LIST && obj == EMPTY && seen)
                    {
                        // the origin patch that the traversal passed over: the same
                        // local ray and patch test as the traversal's leaf
                        const DevObject& ob = sc.objects[origin.object];
                        lr = toLocal(ob, o, d, tmax);
                        patchBase = sc.surfaces[ob.surface].patchBase;
                        pid = origin.patch;
                        last = true;
                        botCulled = false;
                        break;
                    }
                    if (obj == EMPTY)
                    {
                        run = false;
                        if (!LIST) break;
                        list.done(false, over1);
                        continue;
                    }
                    const DevObject& ob = sc.objects[obj];
                    if (ob.surface == EMPTY)   // no geometry (empty box: only a NaN ray gets here)
                    {
                        obj = EMPTY;
                        continue;
                    }
                    CGS_COUNT(kWorkObject);
                    lr = toLocal(ob, o, d, tmax);
                    surface = ob.surface;
                    const DevBVH& surf = sc.surfaces[surface];
                    patchBase = surf.patchBase;
                    botCulled = false;
                    if constexpr (BIG && METHOD != Subdiv)
                        botCulled = surf.cullRoot != EMPTY && cullable(lr.o, {1.0f / lr.d.x, 1.0f / lr.d.y, 1.0f / lr.d.z});
                    bot = botCulled ? cullWalk(surf.cullRoot) : hashWalk(surf.root);
                    lt = lr.max;
                    lp = EMPTY;
                    botTie = false;
                }
                const V3 Dinv {1.0f / lr.d.x, 1.0f / lr.d.y, 1.0f / lr.d.z};
                if (BIG && METHOD != Subdiv && botCulled)
                {
                    pid = cullNext(sc, dirOctant(Dinv), lr.o, Dinv, ANY ? lr.max : cullLimit(lt, lr.o), lr.max, bot, botL0);
                    if (!ANY && pid == EMPTY && (botTie || (lp != EMPTY && !(lL0 < lt))))
                    {
                        botCulled = false;
                        bot = hashWalk(sc.surfaces[surface].root);
                        lt = lr.max;
                        lp = EMPTY;
                        continue;
                    }
                }
                else
                    pid = hashNext<CGS_BOT_OCTANTS, false, BIG>(bvhRef(sc, sc.surfaces + surface), lr.o, Dinv, ANY ? lr.max : lt,
                                                                NodeCache {nullptr, 0}, lm.rings.bot, bot);
                if (pid != EMPTY)
                {
                    if (ORIGIN && (int32_t)obj == origin.object && pid == origin.patch)
                    {
                        seen = true;
                        pid = EMPTY;
                        continue;
                    }
                    break;
                }
                // the object is done: its hit at the world distance t / |M d|
                if (!ANY && lp != EMPTY)
                {
                    const float t = lt * lr.dinv;
                    if (t < h.t)
                    {
                        h = {t, lu, lv, lp, (int32_t)obj};
                        hL0 = topL0;
                        tie = false;
                    }
                    else if (t == h.t)
                        tie = true;
                }
                obj = EMPTY;
                if (!culled) break;
            }
        }
        // ends: a round moves every lane that does not wait, and while lanes wait others are inside objects
        const bool have = pid != EMPTY;
        if (__ballot(have) == 0)
        {
            if (__ballot(run)) continue;
            break;
        }
        // test the patches: a culled surface's from the local ray's max
        float t = ANY || botCulled ? lr.max : lt, u = 0.0f, v = 0.0f;
        bool over = false;
        const float4* S = sc.patches + 16 * (size_t)(have ? patchBase + pid : 0);
        const bool f = leafTest<METHOD, ANY>(have, S, lr.o, versor3(lr.d), tp, t, u, v, lm, over);
        if (have)
        {
            if (LIST && last)
            {
                list.done(f, over1 || over);
                run = false;
            }
            else if (over && botCulled)
            {
                // the object again, in the reference's order
                botCulled = false;
                bot = hashWalk(sc.surfaces[surface].root);
                lt = lr.max;
                lp = EMPTY;
            }
            else if (over && culled)
            {
                // the ray again, in the reference's order
                culled = false;
                h = {tmax, 0.0f, 0.0f, EMPTY, -1};
                top = hashWalk(sc.top.root);
                obj = EMPTY;
                seen = false;
            }
            else
            {
                if (over) (LIST ? over1 : overflow) = true;
                if (ANY)
                {
                    if (f)
                    {
                        hit = true;
                        run = false;
                        if (LIST) list.done(true, over1);
                    }
                }
                else if (f && (!botCulled || t < lt))
                {
                    lt = t;
                    lu = u;
                    lv = v;
                    lp = pid;
                    lL0 = botL0;
                    botTie = false;
                }
                else if (f && t == lt)
                    botTie = true;
            }
        }
    }
    if constexpr (ORIGIN && !LIST)
    {
        // the origin patch that the traversal passed over: the same local ray
        // and patch test as the traversal's leaf
        const bool have = seen && !hit;
        if (__ballot(have))
        {
            const float4* S = sc.patches;
            if (have)
            {
                const DevObject& ob = sc.objects[origin.object];
                lr = toLocal(ob, o, d, tmax);
                S += 16 * (size_t)(sc.surfaces[ob.surface].patchBase + origin.patch);
            }
            float best = lr.max, u, v;
            if (leafTest<METHOD, true>(have, S, lr.o, versor3(lr.d), tp, best, u, v, lm, overflow)) hit = true;
        }
    }
    return hit;
}

// Device totals of the work events (CGS_WORK_COUNTS builds), one set for the
// kernels of each translation unit; workCounts adds them up.
static __device__ unsigned long long g_workCounts[kWorkEvents];

// Clears the workgroup's event slots / adds them to g_workCounts at the end of
// a kernel.
CGS_DEV void workBegin()
{
#if CGS_WORK_COUNTS
    if (threadIdx.x < kWorkEvents) workSlots()[threadIdx.x] = 0;
    __syncthreads();
#endif
}
CGS_DEV void workEnd()
{
#if CGS_WORK_COUNTS
    __syncthreads();
    if (threadIdx.x < kWorkEvents) atomicAdd(g_workCounts + threadIdx.x, workSlots()[threadIdx.x]);
#endif
}

#ifndef CGS_TOP_LDS_KEYS
#define CGS_TOP_LDS_KEYS 256
#endif
static_assert(CGS_TOP_LDS_KEYS <= kTopKeyCap, "top-level LDS staging beyond the key map");

// Stages the top-level BVH's nodes with heap key < CGS_TOP_LDS_KEYS (its upper
// levels, visited by nearly every ray of a traversal without a cull tree) in
// LDS: 64 B per key.  256 keys (16 KiB per workgroup): with 512 the 1M-patch
// frame took 6.66 ms against 6.49, and three workgroups of the any-hit queries
// would not fit a CU.  In a scene with a cull tree only rays with a zero
// direction component and the few whose visit order decides read that BVH: ray
// and shading queries stage it there too (ALWAYS; parallel rays through 256
// grids take 837 and 729 us staged, 888 and 789 not), renders, whose camera rays
// have such a component in a column or two, do not (a 640x480 frame takes 2.23 ms
// staged, 2.12 not).
template<bool ALWAYS>
CGS_DEV NodeCache stageTopLevel(const SceneDev& sc, float4* lds)
{
    if (!ALWAYS && sc.top.cullRoot != EMPTY) return NodeCache {nullptr, 0};
    for (uint32_t k = threadIdx.x; k < 4 * CGS_TOP_LDS_KEYS; k += blockDim.x)
    {
        const uint32_t node = sc.topByKey[k >> 2];
        lds[k] = node != EMPTY ? sc.nodes[4 * (size_t)node + (k & 3)] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
    __syncthreads();
    return NodeCache {(lds_float*)(float*)lds, CGS_TOP_LDS_KEYS};
}

// A lane's query memory: its rings and its wave's clip words in LDS, its
// region stack in `stack`.
CGS_DEV LaneMem laneMem(uint32_t* ringLds, uint32_t* clipLds, float2* stack)
{
    return LaneMem {laneRings(ringLds), clipStackFor(stack, blockIdx.x * blockDim.x + threadIdx.x), waveClipWords(clipLds),
                    nullptr};
}

// Sum of a per-lane count over the wave, added with one atomic.
CGS_DEV void addWave(unsigned long long* ctr, unsigned long long v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    if ((threadIdx.x & 63) == 0 && v) atomicAdd(ctr, v);
}

// Persistent launches: the grid holds at most the resident waves; each wave takes
// chunks of work items (64, fewer in a small launch, the caller's number in a
// batch) from a counter.
struct Persist
{
    float2* stack;           // the waves' region stacks
    unsigned int* counter;
    uint32_t chunk;          // work items a wave takes at a time
};

// The first of the wave's next ps.chunk work items.
CGS_DEV uint32_t nextChunk(const Persist& ps)
{
    uint32_t base = 0;
    if ((threadIdx.x & 63) == 0) base = atomicAdd(ps.counter, ps.chunk);
    return __shfl(base, 0, 64);
}
// Whether this lane has one of the wave's items: lane k has item base + k.
CGS_DEV bool laneHas(const Persist& ps, uint32_t base, uint32_t n)
{
    const uint32_t k = threadIdx.x & 63;
    return k < ps.chunk && base + k < n;
}

#ifndef CGS_RENDER_WAVES
#define CGS_RENDER_WAVES 2
#endif
// Occupancy targets of the queries (waves per SIMD).  Three (168 registers)
// where a launch holds scattered rays, whose walks wait for memory: 200,000
// picks on 1,600 patches take 308 us (closest) and 287 (any) against 351 and 337
// at two, a batch of 64 scenes (17M rays, half of them scattered) 6.3 ms against
// 7.1 (smaller batches: batchAtTwoWaves), 777,777 scattered any-hit rays 820 us.  Closest hits stay at two: 700,000
// camera rays take 782 us against 844 at three, where 49 registers spill;
// 700,000 scattered ones take 964 against 912.
#ifndef CGS_ANY_WAVES
#define CGS_ANY_WAVES 3
#endif
#ifndef CGS_BATCH_WAVES
#define CGS_BATCH_WAVES 3
#endif
#ifndef CGS_PICK_WAVES
#define CGS_PICK_WAVES 3
#endif
#ifndef CGS_CLOSEST_WAVES
#define CGS_CLOSEST_WAVES 2
#endif

CGS_DEV cgs_hit hitRecord(const ClosestHit& h, bool overflow)
{
    return {h.t, h.object < 0 ? 0.0f : h.u, h.object < 0 ? 0.0f : h.v,
            overflow ? CGS_PATCH_OVERFLOW : (h.object < 0 ? EMPTY : h.patch)};
}

template<int METHOD, bool POLISH>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(CGS_CLOSEST_WAVES))) void kTraceClosest(SceneDev sc, Persist ps, const cgs_ray* __restrict__ rays, uint32_t n,
                                                     cgs_hit* __restrict__ hits, int32_t* __restrict__ objects,
                                                     unsigned long long* __restrict__ overflowCount, TraceParams tp)
{
    __shared__ float4 topLds[4 * CGS_TOP_LDS_KEYS];
    __shared__ uint32_t ringLds[kRingWords], clipLds[kClipGroupWords];
    const NodeCache nc = stageTopLevel<true>(sc, topLds);
    const LaneMem lm = laneMem(ringLds, clipLds, ps.stack);
    unsigned long long nOverflow = 0;
    for (uint32_t base = nextChunk(ps); base < n; base = nextChunk(ps))
    {
        const uint32_t r = base + (threadIdx.x & 63);
        const bool run = laneHas(ps, base, n);
        bool overflow = false;
        const cgs_ray ray = run ? rays[r] : cgs_ray {};
        ClosestHit h;
        sceneQuery<METHOD, false, true>(run, sc, nc, lm, {ray.ox, ray.oy, ray.oz}, {ray.dx, ray.dy, ray.dz}, ray.tmax, tp, h,
                                        overflow);
        if (!run) continue;
        if constexpr (POLISH)
            if (h.object >= 0 && !overflow)
            {
                // the reported hit only: the traversal's decisions are the reference's
                const DevObject& ob = sc.objects[h.object];
                const DevBVH surf = sc.surfaces[ob.surface];
                polishHit64(sc.patches + 16 * (size_t)(surf.patchBase + h.patch), ob.w2l, {ray.ox, ray.oy, ray.oz},
                            {ray.dx, ray.dy, ray.dz}, h.t, h.u, h.v);
            }
        hits[r] = hitRecord(h, overflow);
        if (objects) objects[r] = h.object;
        nOverflow += overflow;
    }
    addWave(overflowCount, nOverflow);
}

template<int METHOD>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(CGS_ANY_WAVES))) void kTraceAny(SceneDev sc, Persist ps, const cgs_ray* __restrict__ rays, uint32_t n,
                                                 uint32_t* __restrict__ occluded,
                                                 unsigned long long* __restrict__ overflowCount, TraceParams tp)
{
    __shared__ float4 topLds[4 * CGS_TOP_LDS_KEYS];
    __shared__ uint32_t ringLds[kRingWords], clipLds[kClipGroupWords];
    const NodeCache nc = stageTopLevel<true>(sc, topLds);
    const LaneMem lm = laneMem(ringLds, clipLds, ps.stack);
    unsigned long long nOverflow = 0;
    for (uint32_t base = nextChunk(ps); base < n; base = nextChunk(ps))
    {
        const uint32_t r = base + (threadIdx.x & 63);
        const bool run = laneHas(ps, base, n);
        bool overflow = false;
        const cgs_ray ray = run ? rays[r] : cgs_ray {};
        ClosestHit unused;
        const bool occ = sceneQuery<METHOD, true, true>(run, sc, nc, lm, {ray.ox, ray.oy, ray.oz}, {ray.dx, ray.dy, ray.dz},
                                                        ray.tmax, tp, unused, overflow);
        if (!run) continue;
        occluded[r] = overflow ? 2u : (occ ? 1u : 0u);
        nOverflow += overflow;
    }
    addWave(overflowCount, nOverflow);
}

// The job of ray r: the last with rayBase <= r.
template<class Job>
CGS_DEV uint32_t jobOf(const Job* __restrict__ jobs, uint32_t njobs, uint32_t r)
{
    uint32_t lo = 0, hi = njobs;
    while (hi - lo > 1)
    {
        const uint32_t mid = (lo + hi) / 2;
        if (jobs[mid].rayBase <= r) lo = mid;
        else hi = mid;
    }
    return lo;
}

// Batched ray queries over many resident scenes in one launch: rays of all
// jobs are numbered consecutively and waves take chunks of rays (a
// multiple of 64, ps.chunk) from one counter, so small and large jobs share the grid
// without a launch per scene.  Each lane finds its job by binary search over
// the jobs' first ray numbers and runs the same per-ray query as
// kTraceClosest / kTraceAny, with the same leaf methods and polish.
template<int METHOD, bool POLISH, bool BIG, int WAVES = CGS_BATCH_WAVES>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(WAVES))) void kTraceBatch(
    const BatchJob* __restrict__ jobs, uint32_t njobs, uint32_t total, Persist ps,
    unsigned long long* __restrict__ overflowCount, TraceParams tp)
{
    __shared__ uint32_t ringLds[kRingWords], clipLds[kClipGroupWords];
    const LaneMem lm = laneMem(ringLds, clipLds, ps.stack);
    const NodeCache none {nullptr, 0};
    unsigned long long nOverflow = 0;
    for (uint32_t base = nextChunk(ps); base < total; base = nextChunk(ps))
    {
        const uint32_t end = base + ps.chunk < total ? base + ps.chunk : total;
        for (uint32_t r0 = base; r0 < end; r0 += 64)
        {
            const uint32_t r = r0 + (threadIdx.x & 63);
            const bool run = r < end;
            const BatchJob& J = jobs[jobOf(jobs, njobs, run ? r : base)];
            const uint32_t k = r - J.rayBase;
            const cgs_ray ray = run ? J.rays[k] : cgs_ray {};
            const V3 o {ray.ox, ray.oy, ray.oz}, d {ray.dx, ray.dy, ray.dz};
            bool overflow = false;
            const bool any = run && J.any, closest = run && !J.any;
            ClosestHit h;
            if (__ballot(any))
            {
                const bool occ = sceneQuery<METHOD, true, BIG>(any, J.sc, none, lm, o, d, ray.tmax, tp, h, overflow);
                if (any) J.occluded[k] = overflow ? 2u : (occ ? 1u : 0u);
            }
            if (__ballot(closest))
            {
                sceneQuery<METHOD, false, BIG>(closest, J.sc, none, lm, o, d, ray.tmax, tp, h, overflow);
                if (closest)
                {
                    if constexpr (POLISH)
                        if (h.object >= 0 && !overflow)
                        {
                            const DevObject& ob = J.sc.objects[h.object];
                            const DevBVH surf = J.sc.surfaces[ob.surface];
                            polishHit64(J.sc.patches + 16 * (size_t)(surf.patchBase + h.patch), ob.w2l, o, d, h.t, h.u, h.v);
                        }
                    J.hits[k] = hitRecord(h, overflow);
                    if (J.objects) J.objects[k] = h.object;
                }
            }
            nOverflow += overflow;
        }
    }
    addWave(overflowCount, nOverflow);
}

#if !CGS_SAMPLED_TU && !CGS_LIGHTS_TU
// Batched doBezierClipping: ray r against patch r (Spline_BezierClipping.cu:46-114).
__global__ __launch_bounds__(256) void kClipBatch(Persist ps, const cgs_ray* __restrict__ rays,
                                                  const float4* __restrict__ patches, uint32_t n, float tol2,
                                                  cgs_hit* __restrict__ hits)
{
    __shared__ uint32_t clipLds[kClipGroupWords];
    const ClipStack stk = clipStackFor(ps.stack, blockIdx.x * blockDim.x + threadIdx.x);
    for (uint32_t base = nextChunk(ps); base < n; base = nextChunk(ps))
    {
        const uint32_t r = base + (threadIdx.x & 63);
        const bool run = laneHas(ps, base, n);
        const cgs_ray ray = run ? rays[r] : cgs_ray {};
        bool overflow = false;
        float t = ray.tmax, u = 0.0f, v = 0.0f;
        const bool f = clipWave<false>(run, patches + 16 * (size_t)(run ? r : 0), {ray.ox, ray.oy, ray.oz},
                                       versor3({ray.dx, ray.dy, ray.dz}), tol2, t, u, v, stk, waveClipWords(clipLds), overflow);
        if (run) hits[r] = {t, u, v, overflow ? CGS_PATCH_OVERFLOW : (f ? 1u : EMPTY)};
    }
}

// Batched subdivision (Spline_Subdivision.cu:168-288): ray r against patch r,
// `perWave` pairs to each (one-wave) workgroup.  A pair's regions depend on
// nothing but themselves: the nearest triangle hit wins whatever the order, so
// a wave's lanes share its pairs' regions as ClipLane's do (the oldest entry of
// a lane that has more than one, one for one by rank; entry indices are the
// reference's stack depths), and a pair whose order decides (two hits at
// exactly the winning distance, or an overflow where it was shared) is
// subdivided again unshared.  A region is small (its corners), and its net is
// cut from the patch's each time, so any lane can take it.  With one lane per
// pair, its stack in scratch memory and a workgroup of four waves, 30,001 pairs
// kept half the SIMDs idle and took 1,300 us; this way 147 us.
constexpr int kSubdivLds = 16;   // stack entries in LDS; deeper ones in scratch memory
enum SubdivField : uint32_t
{
    kSubOx, kSubOy, kSubOz, kSubDx, kSubDy, kSubDz, kSubPair, kSubKey, kSubTie, kSubU, kSubV, kSubFlags, kSubGiver,
    kSubFields
};

__global__ __launch_bounds__(64) void kSubdivBatch(const cgs_ray* __restrict__ rays, const float4* __restrict__ patches,
                                                   uint32_t n, uint32_t perWave, float threshold,
                                                   cgs_hit* __restrict__ hits)
{
    __shared__ float4 stackLds[kSubdivLds * 64];
    __shared__ uint32_t wordsLds[kSubFields * 64];
    lds_u32* w = (lds_u32*)wordsLds;
    const uint32_t lane = threadIdx.x, r = blockIdx.x * perWave + lane;
    const bool mine = lane < perWave && r < n;
    float4 deep[kSubdivStack - kSubdivLds];
    // an entry: (umin, vmin, umax, vmax), the side in umin's sign
    auto put = [&](int i, float4 e, bool side) {
        e.x = __uint_as_float(__float_as_uint(e.x) | (side ? 0x80000000u : 0u));
        if (i < kSubdivLds) stackLds[i * 64 + lane] = e;
        else deep[i - kSubdivLds] = e;
    };
    float tmax = 0.0f;
    bool todo = mine;
    if (mine)
    {
        const cgs_ray ray = rays[r];
        const V3 d = versor3({ray.dx, ray.dy, ray.dz});
        tmax = ray.tmax;
        w[kSubOx * 64 + lane] = __float_as_uint(ray.ox);
        w[kSubOy * 64 + lane] = __float_as_uint(ray.oy);
        w[kSubOz * 64 + lane] = __float_as_uint(ray.oz);
        w[kSubDx * 64 + lane] = __float_as_uint(d.x);
        w[kSubDy * 64 + lane] = __float_as_uint(d.y);
        w[kSubDz * 64 + lane] = __float_as_uint(d.z);
        w[kSubPair * 64 + lane] = r;
    }
    // hits lie at t > 0: none is nearer than a tmax of 0 or less or NaN
    const uint32_t first = tmax > 0.0f ? __float_as_uint(tmax) : 0u;
    uint32_t key = 0, flags = 0;
    for (bool alone = false;; alone = true)
    {
        if (todo)
        {
            w[kSubKey * 64 + lane] = first;
            w[kSubTie * 64 + lane] = 0xFFFFFFFFu;
            w[kSubFlags * 64 + lane] = 0u;
        }
        int sp = 0, lo = 0;          // entries lo..sp-1 of this lane's stack
        uint32_t own = lane;         // whose pair they belong to
        if (todo)
        {
            float4 net[16];
#pragma unroll
            for (int i = 0; i < 16; i++) net[i] = patches[16 * (size_t)r + i];
            V3 mn, mx;
            projBox(net, mn, mx);
            const V3 o {__uint_as_float(w[kSubOx * 64 + lane]), __uint_as_float(w[kSubOy * 64 + lane]),
                        __uint_as_float(w[kSubOz * 64 + lane])};
            const V3 d {__uint_as_float(w[kSubDx * 64 + lane]), __uint_as_float(w[kSubDy * 64 + lane]),
                        __uint_as_float(w[kSubDz * 64 + lane])};
            if (boxHit(mn, mx, o, d))
            {
                put(0, {0.0f, 0.0f, 0.5f, 1.0f}, false);
                put(1, {0.5f, 0.0f, 1.0f, 1.0f}, false);
                sp = 2;
            }
        }
        waveOrder();
        // ends: every lane with entries takes one region of its depth-first walk per turn
        while (const uint64_t busy = __ballot(sp > lo))
        {
            if (!alone && busy != ~0ull)
            {
                const bool spare = sp - lo > 1 && lo < kSubdivLds;
                if (const uint64_t give = __ballot(spare))
                {
                    const uint32_t rank = lanesBelow(give), idle = lanesBelow(~busy);
                    if (spare) w[kSubGiver * 64 + rank] = lane;
                    waveOrder();
                    const bool take = sp == lo && idle < (uint32_t)__popcll(give);
                    const uint32_t src = take ? w[kSubGiver * 64 + idle] : lane;
                    const int srcLo = __shfl(lo, (int)src, 64);
                    const uint32_t srcOwn = (uint32_t)__shfl((int)own, (int)src, 64);
                    float4 e {};
                    if (take) e = stackLds[srcLo * 64 + src];
                    waveOrder();
                    if (take)
                    {
                        own = srcOwn;
                        lo = srcLo;
                        sp = lo + 1;
                        stackLds[lo * 64 + lane] = e;
                        ldsOr(w + kSubFlags * 64 + own, kClipShared);
                    }
                    else if (spare && rank < 64u - (uint32_t)__popcll(busy))
                        lo++;
                    waveOrder();
                }
            }
            bool full = false;   // this lane's stack overflowed
            if (sp > lo)
            {
                sp--;
                float4 e = sp < kSubdivLds ? stackLds[sp * 64 + lane] : deep[sp - kSubdivLds];
                const bool side = __builtin_signbit(e.x);
                e.x = __builtin_fabsf(e.x);
                const float4* S = patches + 16 * (size_t)w[kSubPair * 64 + own];
                const V3 o {__uint_as_float(w[kSubOx * 64 + own]), __uint_as_float(w[kSubOy * 64 + own]),
                            __uint_as_float(w[kSubOz * 64 + own])};
                const V3 d {__uint_as_float(w[kSubDx * 64 + own]), __uint_as_float(w[kSubDy * 64 + own]),
                            __uint_as_float(w[kSubDz * 64 + own])};
                float4 sub[16];
#pragma unroll
                for (int i = 0; i < 16; i++) sub[i] = S[i];
                subpatch4(sub, true, e.y, e.w);
                subpatch4(sub, false, e.x, e.z);
                V3 mn, mx;
                projBox(sub, mn, mx);
                if (boxHit(mn, mx, o, d))
                {
                    const float x = 0.5f * (e.x + e.z);
                    const float y = 0.5f * (e.y + e.w);
                    if ((e.z - e.x) < threshold && (e.w - e.y) < threshold)
                    {
                        const V3 p00 = project4(sub[0]), p10 = project4(sub[3]), p01 = project4(sub[12]),
                                 p11 = project4(sub[15]);
                        float t = 0.0f, t1 = 0.0f;
                        const bool b0 = triHit(o, d, p10, p01, p00, t);
                        const bool b1 = triHit(o, d, p01, p10, p11, t1);
                        if (b1 && (!b0 || t1 < t)) t = t1;
                        if (b0 || b1)
                        {
                            const uint32_t tb = __float_as_uint(t), old = ldsMin(w + kSubKey * 64 + own, tb);
                            if (tb < old)
                            {
                                // unless another lane's hit of this turn is nearer still
                                if (ldsLoad(w + kSubKey * 64 + own) == tb)
                                {
                                    w[kSubU * 64 + own] = __float_as_uint(x);
                                    w[kSubV * 64 + own] = __float_as_uint(y);
                                }
                            }
                            else if (tb == old)
                                ldsMin(w + kSubTie * 64 + own, tb);
                        }
                    }
                    else if (sp + 2 > kSubdivStack)
                    {
                        ldsOr(w + kSubFlags * 64 + own, kClipOverflowed);
                        sp = lo;
                        full = true;
                    }
                    else
                    {
                        put(sp, side ? make_float4(e.x, e.y, x, e.w) : make_float4(e.x, e.y, e.z, y), !side);
                        put(sp + 1, side ? make_float4(x, e.y, e.z, e.w) : make_float4(e.x, y, e.z, e.w), !side);
                        sp += 2;
                    }
                }
            }
            waveOrder();
            // an overflowed pair ends for every lane at work on it
            if (__ballot(full) && (ldsLoad(w + kSubFlags * 64 + own) & kClipOverflowed)) sp = lo;
            waveOrder();
        }
        key = w[kSubKey * 64 + lane];
        flags = w[kSubFlags * 64 + lane];
        todo = todo && (flags & kClipShared) &&
               ((flags & kClipOverflowed) || (key < first && w[kSubTie * 64 + lane] == key));
        if (__ballot(todo) == 0) break;
    }
    if (!mine) return;
    const bool found = key < first;
    hits[r] = {found ? __uint_as_float(key) : tmax, found ? __uint_as_float(w[kSubU * 64 + lane]) : 0.0f,
               found ? __uint_as_float(w[kSubV * 64 + lane]) : 0.0f,
               (flags & kClipOverflowed) ? CGS_PATCH_OVERFLOW : (found ? 1u : EMPTY)};
}

// ---------------------------------------------------------------------------
// Patch evaluation (Spline.h:165-254 de Casteljau, Spline.cu:10-27 normal,
// SplineMat.h:125-187 matrix form) and subpatch (Spline.h:384-396)
// ---------------------------------------------------------------------------

// deCasteljau (Spline.h:168-178) over 4 float4 points
CGS_DEV float4 lerp4(float4 a, float4 b, float t, float u)
{
    return {t * a.x + u * b.x, t * a.y + u * b.y, t * a.z + u * b.z, t * a.w + u * b.w};
}
CGS_DEV float4 deCasteljau4(float4 (&p)[4], float u)
{
    const float t = 1.0f - u;
#pragma unroll
    for (int k = 1; k < 4; ++k)
#pragma unroll
        for (int i = 0; i < 4 - k; ++i) p[i] = lerp4(p[i], p[i + 1], t, u);
    return p[0];
}
// deCasteljauDx (Spline.h:183-195): the hodograph without its factor 3
CGS_DEV float4 deCasteljauDx4(float4 (&p)[4], float u)
{
    const float t = 1.0f - u;
#pragma unroll
    for (int i = 1; i < 4; ++i) p[i - 1] = {p[i].x - p[i - 1].x, p[i].y - p[i - 1].y, p[i].z - p[i - 1].z, p[i].w - p[i - 1].w};
#pragma unroll
    for (int k = 2; k < 4; ++k)
#pragma unroll
        for (int i = 0; i < 4 - k; ++i) p[i] = lerp4(p[i], p[i + 1], t, u);
    return p[0];
}
// interpolate (Spline.h:197-214), derivativeU (:216-234), derivativeV (:236-254)
CGS_DEV float4 interpolateDC(const float4* __restrict__ S, float u, float v)
{
    float4 q[4];
#pragma unroll
    for (int j = 0; j < 4; j++)
    {
        float4 p[4] = {S[4 * j], S[4 * j + 1], S[4 * j + 2], S[4 * j + 3]};
        q[j] = deCasteljau4(p, u);
    }
    return deCasteljau4(q, v);
}
CGS_DEV float4 derivativeU_DC(const float4* __restrict__ S, float u, float v)
{
    float4 q[4];
#pragma unroll
    for (int j = 0; j < 4; j++)
    {
        float4 p[4] = {S[4 * j], S[4 * j + 1], S[4 * j + 2], S[4 * j + 3]};
        q[j] = deCasteljauDx4(p, u);
    }
    return deCasteljau4(q, v);
}
CGS_DEV float4 derivativeV_DC(const float4* __restrict__ S, float u, float v)
{
    float4 p[4];
#pragma unroll
    for (int i = 0; i < 4; i++)
    {
        float4 q[4] = {S[i], S[4 + i], S[8 + i], S[12 + i]};
        p[i] = deCasteljauDx4(q, v);
    }
    return deCasteljau4(p, u);
}
// normal (Spline.cu:10-27): a vanishing derivative (a degenerate edge) is
// taken 1e-4 inside the patch instead
CGS_DEV V3 normalDC(const float4* __restrict__ S, float u, float v)
{
    const float e = 0.0001f;
    float4 dU = derivativeU_DC(S, u, v);
    float4 dV = derivativeV_DC(S, u, v);
    if (dU.x == 0.0f && dU.y == 0.0f && dU.z == 0.0f) dU = derivativeU_DC(S, u, __builtin_fabsf(v - e));
    if (dV.x == 0.0f && dV.y == 0.0f && dV.z == 0.0f) dV = derivativeV_DC(S, __builtin_fabsf(u - e), v);
    return cross3({dU.x, dU.y, dU.z}, {dV.x, dV.y, dV.z});
}
// mat::derivativeU (SplineMat.h:142-158) / mat::derivativeV (:160-176)
CGS_DEV float4 derivativeUMat(const float4* __restrict__ S, float u, float v)
{
    float4 x = dbasisMul(evalVecDt(u));
    float4 y = basisMul(evalVec(v));
    float4 a0 = comb4(S[0], S[1], S[2], S[3], x);
    float4 a1 = comb4(S[4], S[5], S[6], S[7], x);
    float4 a2 = comb4(S[8], S[9], S[10], S[11], x);
    float4 a3 = comb4(S[12], S[13], S[14], S[15], x);
    return comb4(a0, a1, a2, a3, y);
}
CGS_DEV float4 derivativeVMat(const float4* __restrict__ S, float u, float v)
{
    float4 xb = basisMul(evalVec(u));
    float4 yd = dbasisMul(evalVecDt(v));
    float4 b0 = comb4(S[0], S[4], S[8], S[12], yd);
    float4 b1 = comb4(S[1], S[5], S[9], S[13], yd);
    float4 b2 = comb4(S[2], S[6], S[10], S[14], yd);
    float4 b3 = comb4(S[3], S[7], S[11], S[15], yd);
    return comb4(b0, b1, b2, b3, xb);
}

// One evaluation per item: patch r at (u, v) = uv[r], by `kind` (CGS_EVAL_*).
__global__ __launch_bounds__(256) void kPatchEval(uint32_t kind, const float4* __restrict__ patches,
                                                  const float2* __restrict__ uv, uint32_t n, float4* __restrict__ out)
{
    const uint32_t r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= n) return;
    const float4* S = patches + 16 * (size_t)r;
    const float2 t = uv[r];
    float4 o;
    switch (kind)
    {
    case CGS_EVAL_INTERPOLATE: o = interpolateDC(S, t.x, t.y); break;
    case CGS_EVAL_INTERPOLATE_MAT: o = interpolateMat(S, t.x, t.y); break;
    case CGS_EVAL_DERIVATIVE_U: o = derivativeU_DC(S, t.x, t.y); break;
    case CGS_EVAL_DERIVATIVE_V: o = derivativeV_DC(S, t.x, t.y); break;
    case CGS_EVAL_DERIVATIVE_U_MAT: o = derivativeUMat(S, t.x, t.y); break;
    case CGS_EVAL_DERIVATIVE_V_MAT: o = derivativeVMat(S, t.x, t.y); break;
    case CGS_EVAL_NORMAL:
    {
        const V3 nv = normalDC(S, t.x, t.y);
        o = {nv.x, nv.y, nv.z, 0.0f};
        break;
    }
    default:
    {
        const V3 nv = normalMat(S, t.x, t.y);
        o = {nv.x, nv.y, nv.z, 0.0f};
        break;
    }
    }
    out[r] = o;
}

// subpatch (Spline.h:384-396): subpatchV to [vmin, vmax], then subpatchU to
// [umin, umax]; ranges[r] = (umin, umax, vmin, vmax).  One patch per lane, read
// and written through LDS so that a wave moves its 64 patches (16 KiB) in
// whole lines: with each lane reading its own 256 bytes, a line was fetched
// again for most of its sixteen points once a CU's waves held more than its
// 32-KiB L1.  A padded row of 17 points per patch spreads the lanes' 16-byte
// accesses over the banks.  Bound by memory: 300,001 patches (528 bytes each)
// took 46 us (3.4 TB/s) that way, 38 us (4.2 TB/s) this way.  Calls of few
// patches (subpatchPerLane) are latency: the way through LDS adds to it.
__global__ __launch_bounds__(64) void kSubpatch(const float4* __restrict__ patches, const float4* __restrict__ ranges,
                                                uint32_t n, float4* __restrict__ out)
{
    __shared__ float4 lds[64 * 17];
    const uint32_t lane = threadIdx.x, r0 = blockIdx.x * 64;
    const uint32_t points = (n - r0 < 64u ? n - r0 : 64u) * 16u;   // of this wave's patches
    const float4* in = patches + 16 * (size_t)r0;
    float4 p[16];
#pragma unroll
    for (uint32_t k = 0; k < 16; k++)
        if (k * 64 + lane < points) p[k] = in[k * 64 + lane];
    float4 g {0.0f, 1.0f, 0.0f, 1.0f};
    if (r0 + lane < n) g = ranges[r0 + lane];
    // point q of patch l at 17 l + q
#pragma unroll
    for (uint32_t k = 0; k < 16; k++)
        if (k * 64 + lane < points) lds[(k * 4 + (lane >> 4)) * 17 + (lane & 15)] = p[k];
    __syncthreads();
    if (r0 + lane < n)
    {
#pragma unroll
        for (int i = 0; i < 16; i++) p[i] = lds[lane * 17 + i];
        subpatch4(p, true, g.z, g.w);
        subpatch4(p, false, g.x, g.y);
#pragma unroll
        for (int i = 0; i < 16; i++) lds[lane * 17 + i] = p[i];
    }
    __syncthreads();
    float4* to = out + 16 * (size_t)r0;
#pragma unroll
    for (uint32_t k = 0; k < 16; k++)
        if (k * 64 + lane < points) to[k * 64 + lane] = lds[(k * 4 + (lane >> 4)) * 17 + (lane & 15)];
}

// The same with each lane moving its own patch.
__global__ __launch_bounds__(64) void kSubpatchFew(const float4* __restrict__ patches, const float4* __restrict__ ranges,
                                                   uint32_t n, float4* __restrict__ out)
{
    const uint32_t r = blockIdx.x * 64 + threadIdx.x;
    if (r >= n) return;
    const float4* S = patches + 16 * (size_t)r;
    float4 p[16];
#pragma unroll
    for (int i = 0; i < 16; i++) p[i] = S[i];
    const float4 g = ranges[r];
    subpatch4(p, true, g.z, g.w);
    subpatch4(p, false, g.x, g.y);
#pragma unroll
    for (int i = 0; i < 16; i++) out[16 * (size_t)r + i] = p[i];
}
#endif // !CGS_SAMPLED_TU && !CGS_LIGHTS_TU

// ---------------------------------------------------------------------------
// cg::PatchBVH (PatchBVH.h:13-28, PatchBVH.cpp:84-121): rays against the
// patches of one surface, in the surface's own frame
// ---------------------------------------------------------------------------
//
// The ray is a Ray3f: its direction normalized once.  Closest (intersect(ray,
// hit)): hit.distance starts at ray.tmax and each leaf clips its patch
// against it.  Any (intersect(ray)): a leaf clips with hit.distance = inf
// (PatchBVH.cpp:93-94), so a patch whose box the traversal reaches within
// ray.tmax counts with a hit at any distance in front.
template<bool ANY>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(CGS_PICK_WAVES))) void kPick(SceneDev sc, Persist ps, const cgs_ray* __restrict__ rays, uint32_t n,
                                                            cgs_hit* __restrict__ hits, uint32_t* __restrict__ occluded)
{
    __shared__ uint32_t ringLds[kRingWords], clipLds[kClipGroupWords];
    const LaneMem lm = laneMem(ringLds, clipLds, ps.stack);
    const DevBVH& surf = sc.surfaces[0];
    const BVHRef b = bvhRef(sc, &surf);
    for (uint32_t base = nextChunk(ps); base < n; base = nextChunk(ps))
    {
        const uint32_t r = base + (threadIdx.x & 63);
        const bool mine = laneHas(ps, base, n);
        bool run = mine;
        const cgs_ray ray = run ? rays[r] : cgs_ray {};
        const V3 o {ray.ox, ray.oy, ray.oz};
        const V3 d = versor3({ray.dx, ray.dy, ray.dz});
        const V3 Dinv {1.0f / d.x, 1.0f / d.y, 1.0f / d.z};
        bool overflow = false, hit = false;
        float t = ray.tmax, u = 0.0f, v = 0.0f;
        uint32_t patch = EMPTY;
        Walk walk = hashWalk(surf.root);
        while (true)
        {
            uint32_t pid = EMPTY;
            if (run)
            {
                pid = hashNext<true, false, true>(b, o, Dinv, ANY ? ray.tmax : t, NodeCache {nullptr, 0}, lm.rings.bot, walk);
                run = pid != EMPTY;
            }
            if (__ballot(run) == 0) break;
            const float4* S = sc.patches + 16 * (size_t)(run ? surf.patchBase + pid : 0);
            float inf = __builtin_inff();
            const bool f = clipWave<ANY>(run, S, o, d, kClipTol2, ANY ? inf : t, u, v, lm.stack, lm.clip, overflow);
            if (f)
            {
                patch = pid;
                hit = true;
                if (ANY) run = false;
            }
        }
        if (!mine) continue;
        if (ANY) occluded[r] = overflow ? 2u : (hit ? 1u : 0u);
        else hits[r] = {t, patch == EMPTY ? 0.0f : u, patch == EMPTY ? 0.0f : v, overflow ? CGS_PATCH_OVERFLOW : patch};
    }
}

// ---------------------------------------------------------------------------
// Renderer (RayTracer.cu:194-544, non-Monte-Carlo path)
// ---------------------------------------------------------------------------

struct CamDev
{
    float4 c[4];          // camera→world columns
    float px, py, pz;     // position
    float tlx, tly;       // top-left pixel centre
    float hdx, hdy;       // half pixel sizes
};

struct RenderDev
{
    float eps;
    int depth;
    uint32_t width, height;
    uint32_t stride;      // frame row pitch in pixels (>= width)
    uint32_t samples;     // camera rays per pixel of the sampled render (0: the plain render)
    uint32_t seed;        // the sampled render's random seed
};

// A render's camera, options and outputs, read by kRender from device memory
// where it needs them (once per tile, or per light for eps) rather than held
// in scalar registers for the whole launch: the traversal loops need those
// registers.
struct RenderArgs
{
    CamDev cam;
    RenderDev op;
    uint32_t* frame;
    float* color;
    unsigned long long* counts;
    const uint32_t* order;   // rank -> tile, or null for row order
    uint32_t* tileTicks;     // per tile: its wave's time in wall-clock ticks, or null
};

// PBR (rt/PBR.h, rt/PBR.cu)
CGS_DEV bool lightVector(float& d, V3& L, V3 P, const DevLight& lt)
{
    const float angle = lt.c.w;
    if (angle < 0.01f)
    {
        L = {-lt.c.x, -lt.c.y, -lt.c.z};
        d = __builtin_inff();
        return true;
    }
    L = sub3({lt.b.x, lt.b.y, lt.b.z}, P);
    d = len3(L);
    if (d < 1e-14f || (lt.b.w > 0.0f && d > lt.b.w)) return false;
    L = mul3(1.0f / d, L);
    if (angle > 1.57f) return true;
    float DL = dot3({lt.c.x, lt.c.y, lt.c.z}, L);
    return DL < 0.0f && angle > 2.0f * acosf(DL);
}
CGS_DEV V3 lightColor(float d, const DevLight& lt)
{
    const V3 col {lt.a.x, lt.a.y, lt.a.z};
    if (lt.c.w < 0.01f) return col;
    float range = lt.b.w, f;
    if (range == 0.0f)
    {
        f = 1.0f / d;
        f *= f;
    }
    else
    {
        f = d / range;
        f = 1.0f + f * (f - 2.0f);
    }
    return mul3(f, col);
}
CGS_DEV V3 schlick(V3 f0, float dotLH)
{
    float b = 1.0f - dotLH;
    float b2 = b * b;
    float s = b2 * b2 * b;
    return {f0.x + (1.0f - f0.x) * s, f0.y + (1.0f - f0.y) * s, f0.z + (1.0f - f0.z) * s};
}
CGS_DEV float G1(float dotNX, float k) { return dotNX / (dotNX * (1.0f - k) + k); }
CGS_DEV float Gsmith(float dotNL, float dotNV, float r)
{
    const float r1 = r + 1.0f;
    const float k = (r1 * r1) * 0.125f;
    return G1(dotNL, k) * G1(dotNV, k);
}
CGS_DEV float Dggx(float dotNH, float r)
{
    r = fmax_(r, 1e-3f);
    float a = r * r;
    float a2 = a * a;
    float d = dotNH * dotNH * (a2 - 1.0f) + 1.0f;
    return a2 / (0x1.921fb6p+1f * d * d);
}
CGS_DEV float microfacet(float dotNV, float dotNL, float dotNH, float r)
{
    return Gsmith(dotNL, dotNV, r) * Dggx(dotNH, r) / (4.0f * dotNL * dotNV);
}

// Ds-boundary pack_sRGB: sRGB encode, 8 bits per channel, 0xAABBGGRR.
CGS_DEV uint32_t packSRGB(float r, float g, float b)
{
    auto enc = [](float c) -> uint32_t {
        float e = c <= 0.0031308f ? 12.92f * c : 1.055f * powf(c, 1.0f / 2.4f) - 0.055f;
        int q = (int)(e * 255.0f + 0.5f);
        q = q < 0 ? 0 : (q > 255 ? 255 : q);
        return (uint32_t)q;
    };
    return enc(r) | (enc(g) << 8) | (enc(b) << 16) | 0xFF000000u;
}

CGS_DEV float saturate(float x) { return x > 0.0f ? (x < 1.0f ? x : 1.0f) : 0.0f; }

// One pixel's random stream in the sampled render: the seed, the pixel's cell
// of the 256×256 grid and the draws taken so far.
struct SampleState
{
    uint32_t seed, stream, draw;
};

// Per-wave LDS words of the shadow rays: 64 of each field (the surface points
// they start from), the list of rays and how many are taken.
enum ShadowField : uint32_t
{
    kShadowX, kShadowY, kShadowZ, kShadowObject, kShadowPatch, kShadowNext, kShadowFields
};
constexpr uint32_t kShadowList = 512;
constexpr uint32_t kShadowWaveWords = kShadowFields * 64 + kShadowList;
constexpr uint32_t kShadowGroupWords = 4 * kShadowWaveWords;

// The shadow rays of a wave's surface points towards a run of lights, any
// lane's ray taken by any lane.  With a lane's own rays in that lane only, one
// light after the other, the few lanes whose paths go on after a bounce were a
// wave's only busy ones for every light: half the time of a frame with 51
// lights went to 13% of its 87 million shadow rays.  From the list that frame
// takes 65 ms instead of 81 to 93.
struct ShadowList
{
    static constexpr bool kList = true;
    static constexpr uint32_t kHit = 1u << 30, kOver = 1u << 31;
    const SceneDev& sc;
    const float* eps;
    lds_u32* w;
    uint32_t l0 = 0, n = 0;
    uint32_t k = 0;              // this lane's ray: its entry

    // this lane's surface point and the patch it lies on
    CGS_DEV void from(V3 P, int32_t object, uint32_t patch) const
    {
        const uint32_t lane = threadIdx.x & 63;
        w[kShadowX * 64 + lane] = __float_as_uint(P.x);
        w[kShadowY * 64 + lane] = __float_as_uint(P.y);
        w[kShadowZ * 64 + lane] = __float_as_uint(P.z);
        w[kShadowObject * 64 + lane] = (uint32_t)object;
        w[kShadowPatch * 64 + lane] = patch;
    }
    CGS_DEV void add(uint32_t i, uint32_t light) const
    {
        w[kShadowFields * 64 + i] = (light << 6) | (threadIdx.x & 63);
    }
    // the list is complete: `count` rays towards lights from firstLight on
    CGS_DEV void open(uint32_t firstLight, uint32_t count)
    {
        l0 = firstLight;
        n = count;
        if ((threadIdx.x & 63) == 0) w[kShadowNext * 64] = 0u;
        waveOrder();
    }
    CGS_DEV uint32_t answer(uint32_t i) const { return w[kShadowFields * 64 + i]; }

    CGS_DEV bool next(V3& o, V3& d, float& tmax, OriginSkip& origin)
    {
        k = ldsAdd(w + kShadowNext * 64, 1u);
        if (k >= n) return false;
        const uint32_t e = w[kShadowFields * 64 + k], at = e & 63u;
        const V3 P {__uint_as_float(w[kShadowX * 64 + at]), __uint_as_float(w[kShadowY * 64 + at]),
                    __uint_as_float(w[kShadowZ * 64 + at])};
        lightVector(tmax, d, P, sc.lights[l0 + (e >> 6)]);
        o = add3(P, mul3(*eps, d));
        origin = {(int32_t)w[kShadowObject * 64 + at], w[kShadowPatch * 64 + at]};
        return true;
    }
    CGS_DEV void done(bool hit, bool over) const { w[kShadowFields * 64 + k] |= (hit ? kHit : 0u) | (over ? kOver : 0u); }
};

// The radiance carried back along one ray of each lane with `run`: the render
// kernel's iterative trace loop with Context::trace / miss / closestHit
// (RayTracer.cu:194-294, 385-544): closest hit, ambient + one shadow ray per
// light with the PBR terms, then the reflection bounce while depth remains and
// the attenuation exceeds 2^-8.  The first segment ends at rmax, bounces at
// infinity.  Every lane of the wave calls it together, and the wave goes
// through each stage together (sceneQuery); a lane whose path has ended helps
// with the others' clips.  eps is read from device memory per use (the
// traversal loops need the registers a kernel argument would hold for the
// whole launch).  With RECORD, the first segment's hit is returned in `first`.
// SAMPLED: the Monte Carlo branches (RayTracer.cu:403-407,473-522): no ambient
// term, and the bounce mirrors about a GGX microfacet normal drawn from `rs`
// (microfacet(roughness², x, y), PBR.h:159-176) with weight mix(diffuse BRDF,
// F(M·V) G(N·R, N·V) (M·V) / (N·V N·M), metalness); the result adds to `acc`,
// the colour carried over from the pixel's earlier samples.
// LIGHTS: the shadow rays go through a ShadowList (all lanes in one scene).
template<bool RECORD, bool BIG = true, bool SAMPLED = false, bool LIGHTS = false>
CGS_DEV V3 rayRadiance(bool run, const SceneDev& sc, const NodeCache& nc, const LaneMem& lm, V3 ro, V3 rd, float rmax,
                       int depth, const float* eps, bool& overflow, uint32_t& nShadow, uint32_t& nSecondary,
                       ClosestHit& first, V3 acc = {0.0f, 0.0f, 0.0f}, SampleState* rs = nullptr)
{
    const TraceParams tp {kClipTol2, 0x1p-4f, 0};
    V3 att {1.0f, 1.0f, 1.0f};
    bool primary = true;
    while (__ballot(run))
    {
        if (run && !primary) nSecondary++;
        ClosestHit h;
        sceneQuery<Clip, false, BIG>(run, sc, nc, lm, ro, rd, rmax, tp, h, overflow);
        if (RECORD && primary) first = h;
        primary = false;
        if (run && h.object < 0)
        {
            acc = add3(acc, mulv3({sc.background[0], sc.background[1], sc.background[2]}, att));
            run = false;
        }
        if (__ballot(run) == 0) break;
        float metal = 0.0f, rough = 0.0f, dotNV = 0.0f;
        V3 spec {}, diffuse {}, col {}, V {}, N {}, Pt {};
        const float invPi = 0x1.45f306p-2f; // std::numbers::inv_pi_v<float>
        if (run)
        {
            const DevObject& ob = sc.objects[h.object];
            const float4 m0 = ob.mat0, m1 = ob.mat1;
            metal = m0.w;
            rough = m1.w;
            spec = {m1.x, m1.y, m1.z};
            diffuse = mul3(1.0f - metal, mul3(invPi, {m0.x, m0.y, m0.z}));
            if (!SAMPLED) col = mulv3({sc.ambient[0], sc.ambient[1], sc.ambient[2]}, diffuse);
            V = neg3(rd);
            N = versor3(normalMat(sc.patches + 16 * (size_t)(sc.surfaces[ob.surface].patchBase + h.patch), h.u, h.v));
            M4 W;
            W.c[0] = ob.w2l[0]; W.c[1] = ob.w2l[1]; W.c[2] = ob.w2l[2]; W.c[3] = ob.w2l[3];
            N = versor3(m3tmul(W, N));
            dotNV = dot3(N, V);
            if (dotNV < 0.0f)
            {
                N = neg3(N);
                dotNV = -dotNV;
            }
            Pt = add3(ro, mul3(h.t, rd));
        }
        auto litBy = [&](uint32_t li, float& d, float& dotNL, V3& L) {
            if (!(run && li < sc.nlight) || !lightVector(d, L, Pt, sc.lights[li])) return false;
            dotNL = dot3(N, L);
            return !(dotNL < 1e-14f);
        };
        auto addLight = [&](uint32_t li, float d, float dotNL, V3 L) {
            V3 H = versor3(add3(L, V));
            float dotHN = dot3(H, N);
            float dotHL = dot3(H, L);
            V3 I = lightColor(d, sc.lights[li]);
            V3 bs = mul3(microfacet(dotNV, dotNL, dotHN, rough), schlick(spec, dotHL));
            col = add3(col, mulv3(mul3(dotNL, I), add3(diffuse, mul3(metal, bs))));
        };
        if constexpr (LIGHTS)
        {
            // light by light, all lanes' rays into one list (as many lights at a
            // time as fit it), then the lit ones' terms in light order
            waveOrder();
            ShadowList shadows {sc, eps, lm.shadow};
            if (run) shadows.from(Pt, h.object, h.patch);
            for (uint32_t l0 = 0, l1; __ballot(run && l0 < sc.nlight); l0 = l1)
            {
                float d, dotNL;
                V3 L;
                uint32_t n = 0;
                for (l1 = l0; n + 64 <= kShadowList && l1 - l0 < (1u << 20) && __ballot(run && l1 < sc.nlight); l1++)
                {
                    const bool lit = litBy(l1, d, dotNL, L);
                    const uint64_t on = __ballot(lit);
                    if (lit) shadows.add(n + lanesBelow(on), l1 - l0);
                    nShadow += lit;
                    n += (uint32_t)__popcll(on);
                }
                if (n == 0) continue;
                shadows.open(l0, n);
                ClosestHit unused;
                bool none = false;
                sceneQuery<Clip, true, BIG, true>(false, sc, nc, lm, V3 {}, V3 {}, 0.0f, tp, unused, none, {-1, EMPTY},
                                                  shadows);
                waveOrder();
                n = 0;
                for (uint32_t li = l0; li < l1; li++)
                {
                    const bool lit = litBy(li, d, dotNL, L);
                    const uint64_t on = __ballot(lit);
                    const uint32_t answer = lit ? shadows.answer(n + lanesBelow(on)) : 0u;
                    n += (uint32_t)__popcll(on);
                    if (answer & ShadowList::kOver) overflow = true;
                    if (lit && !(answer & ShadowList::kHit)) addLight(li, d, dotNL, L);
                }
                waveOrder();
            }
        }
        else
            for (uint32_t li = 0; __ballot(run && li < sc.nlight); li++)
            {
                float d = 0.0f, dotNL = 0.0f;
                V3 L {};
                const bool lit = litBy(li, d, dotNL, L);
                if (__ballot(lit) == 0) continue;
                nShadow += lit;
                // the hit's own patch last (OriginSkip): the answer is the same
                V3 so {};
                if (lit) so = add3(Pt, mul3(*eps, L));
                ClosestHit unused;
                const bool occluded = sceneQuery<Clip, true, BIG, true>(lit, sc, nc, lm, so, L, d, tp, unused, overflow,
                                                                        {h.object, h.patch});
                if (lit && !occluded) addLight(li, d, dotNL, L);
            }
        if (!run) continue;
        acc = add3(acc, mulv3(mul3(0x1.921fb6p+1f, col), att));
        run = false;   // until the bounce is known to go on
        if (depth <= 0) continue;
        V3 R, brdf;
        if constexpr (SAMPLED)
        {
            float x, y;
            drawPair(rs->seed, rs->stream, rs->draw, x, y);
            rs->draw += 2;
            const float alpha = rough * rough;
            const float thetaM = atan2Quadrant(alpha * sqrtf(x), sqrtf(1.0f - x));
            const float phiM = 0x1.921fb6p+2f * y;   // 2π y
            const V3 ts = versor3(cross3(N, V));
            const V3 tp2 = versor3(cross3(N, ts));
            float sinT, cosT, sinP, cosP;
            sinCosAngle(thetaM, sinT, cosT);
            sinCosAngle(phiM, sinP, cosP);
            const V3 M = versor3(add3(add3(mul3(sinT * cosP, ts), mul3(sinT * sinP, tp2)), mul3(cosT, N)));
            const float dotMV = dot3(M, V);
            const V3 refl = schlick(spec, dotMV);
            R = sub3(neg3(V), mul3(2.0f * -dotMV, M));
            const float dotMN = dot3(M, N);
            const float dotNR = dot3(N, R);
            if (dotNR < 1e-14f) continue;
            const float g = Gsmith(dotNR, dotNV, rough) * dotMV / (dotNV * dotMN);
            brdf = add3(diffuse, mul3(metal, mul3(g, refl)));
        }
        else
        {
            V3 refl = schlick(spec, dotNV);
            R = sub3(neg3(V), mul3(2.0f * -dotNV, N));
            float g = Gsmith(dotNV, dotNV, rough);
            float rr = 1.0f - rough;
            brdf = mul3(rr * rr, mul3(dotNV, add3(diffuse, mul3(metal, mul3(g, refl)))));
        }
        V3 a = mulv3(att, brdf);
        if (max3(a) <= 0x1p-8f) continue;
        ro = add3(Pt, mul3(*eps, R));
        rd = R;
        rmax = __builtin_inff();
        att = a;
        depth = depth - 1;
        run = true;
    }
    return acc;
}

// Occupancy target of the render megakernel (waves per SIMD): the compiler
// keeps VGPR + AGPR use within 512 / CGS_RENDER_WAVES.  Two (256 registers, none
// spilled in the plain renders): at three the frame of 4,096 displaced grids
// takes 5.4-5.6 ms against 6.1-6.3, but a 256x256 height field 324-335 us against
// 294, a 768x768 sampled frame 8.4-10.6 ms against 7.3-9.3, and the tea frame of
// 51 lights 112 ms against 64.
// BIG: the scene has a BVH hashed with the wide family or a surface with a
// cull tree (kernels for other scenes leave those paths out and keep their
// registers).
// LIGHTS: shadow rays through a ShadowList, for scenes of kListLights lights or
// more.
// SAMPLED: the Monte Carlo render (RayTracer.cu:212-246): op.samples camera
// rays per pixel through (i + s/n, j + vdc(s)), one running colour over them,
// scaled by 1/n; the pixel's stream is its cell of a 256×256 grid.
template<bool BIG, bool SAMPLED = false, bool LIGHTS = false>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(CGS_RENDER_WAVES))) void kRender(SceneDev sc, Persist ps, const RenderArgs* ra)
{
    __shared__ float4 topLds[4 * CGS_TOP_LDS_KEYS];
    __shared__ uint32_t ringLds[kRingWords], clipLds[kClipGroupWords];
    workBegin();
    const NodeCache nc = stageTopLevel<false>(sc, topLds);
    LaneMem lm = laneMem(ringLds, clipLds, ps.stack);
    if constexpr (LIGHTS)
    {
        __shared__ uint32_t shadowLds[kShadowGroupWords];
        lm.shadow = (lds_u32*)shadowLds + (threadIdx.x >> 6) * kShadowWaveWords;
    }
    const uint32_t lane = threadIdx.x & 63;
    uint32_t nItems;
    {
        const RenderDev op = ra->op;
        nItems = ((op.width + 7) / 8) * ((op.height + 7) / 8) * 64;
    }
    uint32_t nPrimary = 0, nShadow = 0, nSecondary = 0, nOverflow = 0;
    for (uint32_t base = nextChunk(ps); base < nItems; base = nextChunk(ps))
    {
        const RenderDev op = ra->op;
        const CamDev cam = ra->cam;
        const uint32_t tilesX = (op.width + 7) / 8;
        M4 C;
        C.c[0] = cam.c[0]; C.c[1] = cam.c[1]; C.c[2] = cam.c[2]; C.c[3] = cam.c[3];
        const V3 camPos {cam.px, cam.py, cam.pz};
        // one wave = one 8×8 pixel tile (some of its rows in a small frame), taken
        // in the order of ra->order
        const uint32_t rank = base / 64, pixel = base % 64 + lane;
        const uint32_t tile = ra->order ? ra->order[rank] : rank;
        const unsigned long long tileStart = wall_clock64();
        const uint32_t i = (tile % tilesX) * 8 + (pixel & 7), j = (tile / tilesX) * 8 + (pixel >> 3);
        const bool run = lane < ps.chunk && i < op.width && j < op.height;
        bool overflow = false;
        ClosestHit unused;
        V3 acc;
        if constexpr (SAMPLED)
        {
            SampleState rs {op.seed, (i & 255u) + 256u * (j & 255u), 0u};
            const uint32_t n = op.samples;
            const float nInv = 1.0f / (float)n;
            acc = {0.0f, 0.0f, 0.0f};
            for (uint32_t smp = 0; smp < n; smp++)
            {
                nPrimary += run;
                const CamDev cs = ra->cam;
                M4 Cs;
                Cs.c[0] = cs.c[0]; Cs.c[1] = cs.c[1]; Cs.c[2] = cs.c[2]; Cs.c[3] = cs.c[3];
                const V3 pos {cs.px, cs.py, cs.pz};
                const float x = (float)i + (float)smp * nInv, y = (float)j + vdc(smp);
                float4 P = make_float4(cs.tlx + cs.hdx * (2.0f * x), cs.tly - cs.hdy * (2.0f * y), -1.0f, 1.0f);
                const V3 rd = versor3(sub3(project4(m4mul(Cs, P)), pos));
                acc = rayRadiance<false, BIG, true, LIGHTS>(run, sc, nc, lm, pos, rd, __builtin_inff(), ra->op.depth, &ra->op.eps,
                                                    overflow, nShadow, nSecondary, unused, acc, &rs);
            }
            acc = mul3(nInv, acc);
        }
        else
        {
            nPrimary += run;
            // pixelRayDirection (RayTracer.cu:59-71)
            float4 P = make_float4(cam.tlx + cam.hdx * (2.0f * (float)i), cam.tly - cam.hdy * (2.0f * (float)j), -1.0f, 1.0f);
            const V3 rd = versor3(sub3(project4(m4mul(C, P)), camPos));
            acc = rayRadiance<false, BIG, false, LIGHTS>(run, sc, nc, lm, camPos, rd, __builtin_inff(), op.depth, &ra->op.eps, overflow,
                                          nShadow, nSecondary, unused);
        }
        if (!run) continue;
        const uint32_t q = j * ra->op.width + i;
        if (float* color = ra->color)
        {
            color[3 * (size_t)q] = acc.x;
            color[3 * (size_t)q + 1] = acc.y;
            color[3 * (size_t)q + 2] = acc.z;
        }
        ra->frame[(size_t)j * ra->op.stride + i] = packSRGB(saturate(acc.x), saturate(acc.y), saturate(acc.z));
        nOverflow += overflow;
        // The tile's time, for ordering the next render of this view.  Lane 0
        // holds the tile's first pixel, which always lies inside the frame.
        if (uint32_t* ticks = ra->tileTicks)
        {
            const unsigned long long dt = wall_clock64() - tileStart;
            if (pixel == 0) ticks[tile] = dt > 0xFFFFFFFFull ? 0xFFFFFFFFu : (uint32_t)dt;
        }
    }
    if (unsigned long long* counts = ra->counts)
    {
        addWave(counts + 0, nPrimary);
        addWave(counts + 1, nShadow);
        addWave(counts + 2, nSecondary);
        addWave(counts + 3, nOverflow);
    }
    workEnd();
}

// Shaded ray queries: each lane traces and shades one given world ray as the
// render does a camera ray (rayRadiance), over one or many jobs.  Rays of all
// jobs are numbered consecutively and waves take chunks of `chunk` rays from
// one counter; each lane finds its job by binary search over the jobs' first
// ray numbers.  With ONE_SCENE every job is on scene `sc0` (a kernel
// argument, like the render's) and the top-level BVH's upper levels are
// staged in LDS as in the render; otherwise each job's own scene is used.
template<bool ONE_SCENE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(CGS_RENDER_WAVES))) void kShade(
    SceneDev sc0, const ShadeJob* __restrict__ jobs, uint32_t njobs, uint32_t total, Persist ps,
    unsigned long long* __restrict__ counts)
{
    __shared__ uint32_t ringLds[kRingWords], clipLds[kClipGroupWords];
    NodeCache nc {nullptr, 0};
    if constexpr (ONE_SCENE)
    {
        __shared__ float4 topLds[4 * CGS_TOP_LDS_KEYS];
        nc = stageTopLevel<true>(sc0, topLds);
    }
    const LaneMem lm = laneMem(ringLds, clipLds, ps.stack);
    uint32_t nPrimary = 0, nShadow = 0, nSecondary = 0, nOverflow = 0;
    for (uint32_t base = nextChunk(ps); base < total; base = nextChunk(ps))
    {
        const uint32_t end = base + ps.chunk < total ? base + ps.chunk : total;
        for (uint32_t r0 = base; r0 < end; r0 += 64)
        {
            const uint32_t r = r0 + (threadIdx.x & 63);
            const bool run = r < end;
            const ShadeJob& J = jobs[jobOf(jobs, njobs, run ? r : base)];
            const uint32_t k = r - J.rayBase;
            const cgs_ray ray = run ? J.rays[k] : cgs_ray {};
            bool overflow = false;
            nPrimary += run;
            ClosestHit h;
            V3 acc;
            if constexpr (ONE_SCENE)
                acc = rayRadiance<true>(run, sc0, nc, lm, {ray.ox, ray.oy, ray.oz}, {ray.dx, ray.dy, ray.dz}, ray.tmax,
                                        J.depth, &J.eps, overflow, nShadow, nSecondary, h);
            else
                acc = rayRadiance<true>(run, J.sc, nc, lm, {ray.ox, ray.oy, ray.oz}, {ray.dx, ray.dy, ray.dz}, ray.tmax,
                                        J.depth, &J.eps, overflow, nShadow, nSecondary, h);
            if (!run) continue;
            J.color[3 * (size_t)k] = acc.x;
            J.color[3 * (size_t)k + 1] = acc.y;
            J.color[3 * (size_t)k + 2] = acc.z;
            if (uint32_t* px = J.pixels) px[k] = packSRGB(saturate(acc.x), saturate(acc.y), saturate(acc.z));
            if (cgs_hit* hits = J.hits) hits[k] = hitRecord(h, overflow);
            if (int32_t* objects = J.objects) objects[k] = h.object;
            nOverflow += overflow;
        }
    }
    if (counts)
    {
        addWave(counts + 0, nPrimary);
        addWave(counts + 1, nShadow);
        addWave(counts + 2, nSecondary);
        addWave(counts + 3, nOverflow);
    }
}

} // namespace cgs

namespace cgs
{
// Adds this translation unit's work-event totals to `out` and clears them when
// `reset`.
static hipError_t addWorkCounts(unsigned long long* out, bool reset)
{
    unsigned long long own[kWorkEvents];
    const hipError_t e = hipMemcpyFromSymbol(own, HIP_SYMBOL(g_workCounts), sizeof own);
    if (e != hipSuccess) return e;
    for (int k = 0; k < kWorkEvents; k++) out[k] += own[k];
    if (!reset) return hipSuccess;
    const unsigned long long zero[kWorkEvents] = {};
    return hipMemcpyToSymbol(HIP_SYMBOL(g_workCounts), zero, sizeof zero);
}
} // namespace cgs

#if CGS_LIGHTS_TU
namespace cgs
{
hipError_t workCountsLights(unsigned long long* out, bool reset) { return addWorkCounts(out, reset); }

hipError_t launchRenderLights(const SceneDev& sc, const PersistArgs& pa, const void* argsDev, hipStream_t s)
{
    Persist ps {pa.stack, pa.counter, pa.chunk};
    if (sc.big)
        hipLaunchKernelGGL((kRender<true, false, true>), dim3(pa.grid), dim3(256), 0, s, sc, ps, (const RenderArgs*)argsDev);
    else
        hipLaunchKernelGGL((kRender<false, false, true>), dim3(pa.grid), dim3(256), 0, s, sc, ps, (const RenderArgs*)argsDev);
    return hipGetLastError();
}
} // namespace cgs
#elif CGS_SAMPLED_TU
namespace cgs
{
hipError_t workCountsSampled(unsigned long long* out, bool reset) { return addWorkCounts(out, reset); }

hipError_t launchRenderSampled(const SceneDev& sc, const PersistArgs& pa, const void* argsDev, hipStream_t s)
{
    Persist ps {pa.stack, pa.counter, pa.chunk};
    hipLaunchKernelGGL((kRender<true, true>), dim3(pa.grid), dim3(256), 0, s, sc, ps, (const RenderArgs*)argsDev);
    return hipGetLastError();
}
} // namespace cgs
#else
// ---------------------------------------------------------------------------
// Launchers (called by the host library)
// ---------------------------------------------------------------------------
namespace cgs
{

static inline uint32_t blocks(uint32_t n, uint32_t b) { return (n + b - 1) / b; }

// Resident workgroups per CU of each persistent kernel (occupancy API).
hipError_t persistentGrid(PersistKernel k, uint32_t& blocksPerCU)
{
    int n = 0;
    hipError_t e = hipSuccess;
    switch (k)
    {
    case PersistKernel::TraceClosest: e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kTraceClosest<Clip, false>, 256, 0); break;
    case PersistKernel::TraceAny: e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kTraceAny<Clip>, 256, 0); break;
    case PersistKernel::ClipBatch: e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kClipBatch, 256, 0); break;
    case PersistKernel::Render: e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kRender<true>, 256, 0); break;
    case PersistKernel::Batch: e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kTraceBatch<Clip, false, true>, 256, 0); break;
    case PersistKernel::Pick: e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kPick<false>, 256, 0); break;
    case PersistKernel::Shade: e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kShade<true>, 256, 0); break;
    }
    blocksPerCU = n > 0 ? (uint32_t)n : 1u;
    return e;
}

// The least float x whose square root is at least tol, so that
// sqrt(x) < tol is x < tolSquare(tol) (the correctly rounded square root is
// monotone): two compares per clipping pass instead of two square roots.
// 0 where no square root is below tol (tol <= 0 or NaN).
static float tolSquare(float tol)
{
    if (!(tol > 0.0f)) return 0.0f;
    const uint32_t inf = 0x7F800000u;
    uint32_t lo = 0u, hi = inf;      // sqrt(lo) < tol; hi is inf or sqrt(hi) >= tol
    while (hi - lo > 1u)
    {
        const uint32_t m = lo + (hi - lo) / 2u;
        if (__builtin_sqrtf(std::bit_cast<float>(m)) < tol) lo = m;
        else hi = m;
    }
    return std::bit_cast<float>(hi);
}

// Trace launches with an explicit leaf method.  The opt-in modes use the
// default kernels' grid (the same VGPR budget and LDS; they spill to scratch
// where the default kernels do not).  The default kernels clip at the fixed
// 2^-12, so a clipping run with another tolerance takes the capped kernels
// with a cap no run reaches (2^32 - 1 passes).
static TraceParams traceParams(const TraceMode& m)
{
    return {tolSquare(m.tol), m.threshold, m.maxIters ? m.maxIters : 0xFFFFFFFFu};
}

hipError_t launchTraceClosest(const SceneDev& sc, const PersistArgs& pa, const cgs_ray* rays, uint32_t n, cgs_hit* hits,
                              int32_t* objects, unsigned long long* overflow, hipStream_t s, const TraceMode& m)
{
    if (n == 0) return hipSuccess;
    Persist ps {pa.stack, pa.counter, pa.chunk};
    const TraceParams tp = traceParams(m);
#define CGS_LAUNCH_CLOSEST(M, P) \
    hipLaunchKernelGGL((kTraceClosest<M, P>), dim3(pa.grid), dim3(256), 0, s, sc, ps, rays, n, hits, objects, overflow, tp)
    if (m.method == CGS_METHOD_SUBDIVISION)
    {
        if (m.polish) CGS_LAUNCH_CLOSEST(Subdiv, true);
        else CGS_LAUNCH_CLOSEST(Subdiv, false);
    }
    else if (m.maxIters || m.tol != kClipTol)
    {
        if (m.polish) CGS_LAUNCH_CLOSEST(ClipCapped, true);
        else CGS_LAUNCH_CLOSEST(ClipCapped, false);
    }
    else if (m.polish) CGS_LAUNCH_CLOSEST(Clip, true);
    else CGS_LAUNCH_CLOSEST(Clip, false);
#undef CGS_LAUNCH_CLOSEST
    return hipGetLastError();
}

hipError_t launchTraceAny(const SceneDev& sc, const PersistArgs& pa, const cgs_ray* rays, uint32_t n, uint32_t* occluded,
                          unsigned long long* overflow, hipStream_t s, const TraceMode& m)
{
    if (n == 0) return hipSuccess;
    Persist ps {pa.stack, pa.counter, pa.chunk};
    const TraceParams tp = traceParams(m);
    if (m.method == CGS_METHOD_SUBDIVISION)
        hipLaunchKernelGGL((kTraceAny<Subdiv>), dim3(pa.grid), dim3(256), 0, s, sc, ps, rays, n, occluded, overflow, tp);
    else if (m.maxIters || m.tol != kClipTol)
        hipLaunchKernelGGL((kTraceAny<ClipCapped>), dim3(pa.grid), dim3(256), 0, s, sc, ps, rays, n, occluded, overflow, tp);
    else
        hipLaunchKernelGGL((kTraceAny<Clip>), dim3(pa.grid), dim3(256), 0, s, sc, ps, rays, n, occluded, overflow, tp);
    return hipGetLastError();
}

hipError_t launchTraceBatch(const BatchJob* jobs, uint32_t njobs, uint32_t total, uint32_t chunk, float2* stack,
                            unsigned int* counter, uint32_t grid, unsigned long long* overflow, hipStream_t s,
                            const TraceMode& m, bool big)
{
    if (total == 0) return hipSuccess;
    Persist ps {stack, counter, chunk};
    const TraceParams tp = traceParams(m);
    if (m.method != CGS_METHOD_SUBDIVISION && !m.maxIters && m.tol == kClipTol && !m.polish)
    {
        // the default method has kernels without the wide-hash and surface-cull
        // paths, and both with a form for launches of few rays
        if (batchAtTwoWaves(total)) grid = std::min(grid, 2u * 256u);
        const auto kernel = batchAtTwoWaves(total) ? (big ? kTraceBatch<Clip, false, true, 2> : kTraceBatch<Clip, false, false, 2>)
                                                   : (big ? kTraceBatch<Clip, false, true> : kTraceBatch<Clip, false, false>);
        hipLaunchKernelGGL(kernel, dim3(grid), dim3(256), 0, s, jobs, njobs, total, ps, overflow, tp);
        return hipGetLastError();
    }
#define CGS_LAUNCH_BATCH(M, P) \
    hipLaunchKernelGGL((kTraceBatch<M, P, true>), dim3(grid), dim3(256), 0, s, jobs, njobs, total, ps, overflow, tp)
    if (m.method == CGS_METHOD_SUBDIVISION)
    {
        if (m.polish) CGS_LAUNCH_BATCH(Subdiv, true);
        else CGS_LAUNCH_BATCH(Subdiv, false);
    }
    else if (m.maxIters || m.tol != kClipTol)
    {
        if (m.polish) CGS_LAUNCH_BATCH(ClipCapped, true);
        else CGS_LAUNCH_BATCH(ClipCapped, false);
    }
    else CGS_LAUNCH_BATCH(Clip, true);
#undef CGS_LAUNCH_BATCH
    return hipGetLastError();
}

hipError_t launchClipBatch(const PersistArgs& pa, const cgs_ray* rays, const float* patches, uint32_t n, float tol,
                           cgs_hit* hits, hipStream_t s)
{
    if (n == 0) return hipSuccess;
    Persist ps {pa.stack, pa.counter, pa.chunk};
    hipLaunchKernelGGL(kClipBatch, dim3(pa.grid), dim3(256), 0, s, ps, rays, (const float4*)patches, n, tolSquare(tol), hits);
    return hipGetLastError();
}

hipError_t launchSubdivBatch(const cgs_ray* rays, const float* patches, uint32_t n, float threshold, cgs_hit* hits,
                             hipStream_t s)
{
    if (n == 0) return hipSuccess;
    // Pairs per wave: a full wave's where they fill the chip's 2,048 resident
    // waves, fewer below (down to 8: a pair's regions keep about 8 lanes at work)
    const uint32_t perWave = std::clamp<uint32_t>(n / 2048u / 8u * 8u, 8u, 64u);
    hipLaunchKernelGGL(kSubdivBatch, dim3(blocks(n, perWave)), dim3(64), 0, s, rays, (const float4*)patches, n, perWave,
                       threshold, hits);
    return hipGetLastError();
}

hipError_t launchPatchEval(uint32_t kind, const float* patches, const float* uv, uint32_t n, float* out, hipStream_t s)
{
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(kPatchEval, dim3(blocks(n, 256)), dim3(256), 0, s, kind, (const float4*)patches,
                       (const float2*)uv, n, (float4*)out);
    return hipGetLastError();
}

hipError_t launchSubpatch(const float* patches, const float* ranges, uint32_t n, float* out, hipStream_t s)
{
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(subpatchPerLane(n) ? kSubpatchFew : kSubpatch, dim3(blocks(n, 64)), dim3(64), 0, s,
                       (const float4*)patches, (const float4*)ranges, n, (float4*)out);
    return hipGetLastError();
}

hipError_t launchShade(const SceneDev* one, const ShadeJob* jobs, uint32_t njobs, uint32_t total, uint32_t chunk,
                       float2* stack, unsigned int* counter, uint32_t grid, unsigned long long* counts,
                       hipStream_t s)
{
    if (total == 0 || njobs == 0) return hipSuccess;
    Persist ps {stack, counter, chunk};
    if (one)
        hipLaunchKernelGGL(kShade<true>, dim3(grid), dim3(256), 0, s, *one, jobs, njobs, total, ps, counts);
    else
        hipLaunchKernelGGL(kShade<false>, dim3(grid), dim3(256), 0, s, SceneDev {}, jobs, njobs, total, ps,
                           counts);
    return hipGetLastError();
}

hipError_t launchPick(const SceneDev& sc, const PersistArgs& pa, const cgs_ray* rays, uint32_t n, cgs_hit* hits,
                      uint32_t* occluded, hipStream_t s)
{
    if (n == 0) return hipSuccess;
    Persist ps {pa.stack, pa.counter, pa.chunk};
    if (occluded)
        hipLaunchKernelGGL(kPick<true>, dim3(pa.grid), dim3(256), 0, s, sc, ps, rays, n, hits, occluded);
    else
        hipLaunchKernelGGL(kPick<false>, dim3(pa.grid), dim3(256), 0, s, sc, ps, rays, n, hits, occluded);
    return hipGetLastError();
}

hipError_t launchRender(const SceneDev& sc, const PersistArgs& pa, const float* toWorld16, const float* pos3, float tlx,
                        float tly, float hdx, float hdy, float eps, int depth, uint32_t w, uint32_t h, uint32_t* frame,
                        float* color, unsigned long long* counts, uint32_t stride, const uint32_t* order,
                        uint32_t* tileTicks, void* argsDev, hipStream_t s, uint32_t samples, uint32_t seed)
{
    CamDev cam;
    for (int c = 0; c < 4; c++)
        cam.c[c] = make_float4(toWorld16[4 * c], toWorld16[4 * c + 1], toWorld16[4 * c + 2], toWorld16[4 * c + 3]);
    cam.px = pos3[0];
    cam.py = pos3[1];
    cam.pz = pos3[2];
    cam.tlx = tlx;
    cam.tly = tly;
    cam.hdx = hdx;
    cam.hdy = hdy;
    if ((uint64_t)w * h == 0) return hipSuccess;
    const RenderArgs ra {cam, RenderDev {eps, depth, w, h, stride, samples, seed}, frame, color, counts, order, tileTicks};
    static_assert(sizeof(RenderArgs) <= kRenderArgsBytes, "render argument block");
    // `ra` is pageable (the stack): HIP performs such a copy synchronously,
    // so it has been read when the call returns.
    hipError_t e = hipMemcpyAsync(argsDev, &ra, sizeof ra, hipMemcpyHostToDevice, s);
    if (e != hipSuccess) return e;
    Persist ps {pa.stack, pa.counter, pa.chunk};
    if (samples > 0) return launchRenderSampled(sc, pa, argsDev, s);
    if (sc.nlight >= kListLights) return launchRenderLights(sc, pa, argsDev, s);
    if (sc.big)
        hipLaunchKernelGGL(kRender<true>, dim3(pa.grid), dim3(256), 0, s, sc, ps, (const RenderArgs*)argsDev);
    else
        hipLaunchKernelGGL(kRender<false>, dim3(pa.grid), dim3(256), 0, s, sc, ps, (const RenderArgs*)argsDev);
    return hipGetLastError();
}

// Tile order for the next render of a view: longest first, by a counting
// sort on the tile times (four buckets per octave; order within a bucket is
// arbitrary).  One workgroup; every tile gets exactly one rank.
constexpr int kOrderBuckets = 128;
CGS_DEV uint32_t timeBucket(uint32_t t)
{
    if (t < 2) return 0;
    const uint32_t l = 31 - __builtin_clz(t);
    return 4 * l + (l >= 2 ? (t >> (l - 2)) & 3 : (t << (2 - l)) & 3);
}

__global__ __launch_bounds__(1024) void kTileOrder(const uint32_t* __restrict__ ticks, uint32_t n,
                                                   uint32_t* __restrict__ order)
{
    __shared__ uint32_t count[kOrderBuckets];
    for (uint32_t b = threadIdx.x; b < kOrderBuckets; b += blockDim.x) count[b] = 0;
    __syncthreads();
    for (uint32_t t = threadIdx.x; t < n; t += blockDim.x) atomicAdd(&count[timeBucket(ticks[t])], 1u);
    __syncthreads();
    if (threadIdx.x == 0)
    {
        uint32_t first = 0;   // the longest bucket first
        for (int b = kOrderBuckets - 1; b >= 0; b--)
        {
            const uint32_t c = count[b];
            count[b] = first;
            first += c;
        }
    }
    __syncthreads();
    for (uint32_t t = threadIdx.x; t < n; t += blockDim.x) order[atomicAdd(&count[timeBucket(ticks[t])], 1u)] = t;
}

hipError_t launchTileOrder(const uint32_t* ticks, uint32_t n, uint32_t* order, hipStream_t s)
{
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(kTileOrder, dim3(1), dim3(1024), 0, s, ticks, n, order);
    return hipGetLastError();
}

// The work-event totals of the CGS_WORK_COUNTS build (zeros otherwise):
// copies kWorkEvents totals to `out` and clears them when `reset`.
hipError_t workCounts(unsigned long long* out, bool reset)
{
    std::fill(out, out + kWorkEvents, 0ull);
    hipError_t e = addWorkCounts(out, reset);
    if (e == hipSuccess) e = workCountsLights(out, reset);
    if (e == hipSuccess) e = workCountsSampled(out, reset);
    return e;
}

} // namespace cgs
#endif // CGS_SAMPLED_TU, CGS_LIGHTS_TU
