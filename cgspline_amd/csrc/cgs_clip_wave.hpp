// SPDX-License-Identifier: MIT
//
// The clipping test of a wave's lanes, shared between them: every lane of the
// wave calls clipWave with or without a (ray, patch) pair of its own, and a
// lane without work takes regions from the stack of one that has them.
//
#pragma once

#include "cgs_device.hpp"

namespace cgs
{

// Orders one lane's LDS and region-stack accesses against the other lanes' of
// its wave.  A wave's accesses to one memory are executed in program order,
// so this only stops the compiler from moving them.
CGS_DEV void waveOrder()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Per-wave LDS words of the shared clip, 64 of each field: a lane's own pair
// (ray, control points) and its result, read and updated by the lanes that
// work on its regions; and the list of lanes with regions to give.
enum ClipField : uint32_t
{
    kClipOx, kClipOy, kClipOz, kClipDx, kClipDy, kClipDz,
    kClipSLo, kClipSHi,
    kClipKey,      // nearest accepted distance (its bits: distances are >= 0)
    kClipTie,      // least distance accepted twice (its bits)
    kClipU, kClipV,
    kClipFlags,
    kClipGiver,
    kClipFields
};
constexpr uint32_t kClipWaveWords = kClipFields * 64;
constexpr uint32_t kClipGroupWords = 4 * kClipWaveWords;   // a 256-lane workgroup
enum ClipFlag : uint32_t { kClipFound = 1, kClipOverflowed = 2, kClipShared = 4 };

CGS_DEV lds_u32* waveClipWords(uint32_t* lds) { return (lds_u32*)lds + (threadIdx.x >> 6) * kClipWaveWords; }

CGS_DEV uint32_t lanesBelow(uint64_t mask)
{
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

// A lane's part in the clipping of its wave's (ray, patch) pairs:
// doBezierClipping with host semantics (Spline_BezierClipping.cu:46-114,
// 174-445), for every lane's pair at once.  start() makes a pair of the lane's
// own current, and share() and pass() are called by EVERY lane of the wave
// together until no lane has a region.  With ANY a pair stops at its first accepted candidate (the caller
// only needs "found").  tol2 is the clipping tolerance's tolSquare: a region's
// size is compared squared.  CAPPED (an opt-in mode with no counterpart in the
// reference): the test stops after maxIters passes of its loop and keeps what
// it found so far.
//
// Sharing.  Each lane works depth first through its pair's regions with a
// region stack of its own, as the reference does; entries lo..sp-1 of its
// column hold the postponed ones.  A lane without a region takes the oldest
// postponed region (the largest, and the last in the reference's order) of a
// lane that has some, one for one by rank, and works depth first from there;
// the entry's index is the region's depth, so stacks never grow beyond the
// reference's 32 entries and overflow where its does.  A region's passes
// depend on nothing but the region, and a candidate's acceptance on its own
// distance, so the results are the reference's except where its visit order
// decides; there the pair is clipped again unshared (`alone`):
//  - closest: the nearest candidate wins whatever the order; two candidates
//    at exactly the winning distance;
//  - any: what a lane finds among taken regions stops that lane only, since
//    an earlier region might still overflow; the lane that holds the first
//    regions stops the whole pair;
//  - an overflow anywhere in a pair that was shared, which ends at once for
//    all its lanes.
//
// What bounds it is the instruction count of a pass, on full waves and on the
// one lane that a wave's slowest pair would keep busy.  Convergence by squared
// sizes (no square roots), maxNum/minNum envelopes, straight-line hull edges,
// one de Casteljau step for a split's two halves and stack words at constant
// offsets took 200,000 (ray, patch) pairs from 752 to 571 us and a 64-ray pick
// from 111 to 97 us; sharing took the pairs to 157 us, the 1M-patch frame (views
// whose slowest pixel alone had taken 23 ms) to 6.5 ms and a 768² sampled frame
// from 45 to 8.6 ms.
template<bool ANY, bool CAPPED = false>
struct ClipLane
{
    lds_u32* w;                 // the wave's words
    ClipStack stk;              // this lane's column
    uint32_t lane;
    bool held = false;          // this lane has a current region
    bool taken = false;         // ... of regions taken from another lane
    bool alone = CAPPED;        // this lane's pair is not to be shared
    uint32_t own = 0;           // whose pair the current region belongs to
    int sp = 0, lo = 0;         // postponed regions: entries lo..sp-1 of this lane's column
    V2 p[16];
    V2 mn, mx, sz;
    bool vside = false, finite = true;
    uint32_t iters = 0;

    CGS_DEV ClipLane(lds_u32* words, const ClipStack& stack) : w(words), stk(stack), lane(threadIdx.x & 63) {}

    CGS_DEV float word(uint32_t field, uint32_t l) const { return __uint_as_float(w[field * 64 + l]); }
    // a distance is never below 0: no candidate beats a best of 0 or less or NaN
    CGS_DEV static uint32_t firstKey(float best) { return best > 0.0f ? __float_as_uint(best) : 0u; }

    // Takes ray (o, d), d the Ray3f direction, against the 16 control points S
    // (global) as this lane's pair; candidates below `best` count.
    CGS_DEV void start(const float4* S, V3 o, V3 d, float best, bool unshared)
    {
        w[kClipOx * 64 + lane] = __float_as_uint(o.x);
        w[kClipOy * 64 + lane] = __float_as_uint(o.y);
        w[kClipOz * 64 + lane] = __float_as_uint(o.z);
        w[kClipDx * 64 + lane] = __float_as_uint(d.x);
        w[kClipDy * 64 + lane] = __float_as_uint(d.y);
        w[kClipDz * 64 + lane] = __float_as_uint(d.z);
        w[kClipSLo * 64 + lane] = (uint32_t)(uint64_t)S;
        w[kClipSHi * 64 + lane] = (uint32_t)((uint64_t)S >> 32);
        w[kClipKey * 64 + lane] = firstKey(best);
        w[kClipTie * 64 + lane] = 0xFFFFFFFFu;
        w[kClipFlags * 64 + lane] = 0u;
        CGS_COUNT(kWorkPatch);
        const ClipRay R = makeClipRay(o, d);
        // 0 * x is NaN for the infinities and NaN
        float fin = 0.0f;
#pragma unroll
        for (int i = 0; i < 16; i++)
        {
            const float4 q = S[i];
            const V3 D {q.x - R.o.x, q.y - R.o.y, q.z - R.o.z};
            p[i] = {dot3(R.ax0, D), dot3(R.ax1, D)};
            fin += 0.0f * p[i].x + 0.0f * p[i].y;
        }
        finite = fin == 0.0f;
        mn = {0.0f, 0.0f};
        mx = sz = {1.0f, 1.0f};
        vside = taken = false;
        held = true;
        alone = CAPPED || unshared;
        own = lane;
        sp = lo = 0;
        iters = 0;
    }

    // The pair has to be clipped again, unshared: the order decides.
    CGS_DEV bool mustRepeat(float best) const
    {
        const uint32_t flags = w[kClipFlags * 64 + lane];
        if (!(flags & kClipShared)) return false;
        if (flags & kClipOverflowed) return true;
        const uint32_t key = w[kClipKey * 64 + lane];
        return !ANY && key < firstKey(best) && w[kClipTie * 64 + lane] == key;
    }
    CGS_DEV bool overflowed() const { return (w[kClipFlags * 64 + lane] & kClipOverflowed) != 0; }
    // The pair's answer; the nearest accepted candidate (closest)
    CGS_DEV bool found(float best) const
    {
        return ANY ? (w[kClipFlags * 64 + lane] & kClipFound) != 0 : w[kClipKey * 64 + lane] < firstKey(best);
    }
    CGS_DEV float t() const { return word(kClipKey, lane); }
    CGS_DEV float u() const { return word(kClipU, lane); }
    CGS_DEV float v() const { return word(kClipV, lane); }

    CGS_DEV void load(const float2* e)
    {
#pragma unroll
        for (int i = 0; i < 16; i++)
        {
            const float2 q = e[64 * i];
            p[i] = {q.x, q.y};
        }
        const float2 r0 = e[64 * 16], r1 = e[64 * 17], r2 = e[64 * 18], r3 = e[64 * 19];
        mn = {r0.x, r0.y};
        mx = {r1.x, r1.y};
        sz = {r2.x, r2.y};
        vside = r3.x != 0.0f;
    }

    // The current region's points are not needed any more.  Without these empty
    // definitions they count as live until the next region replaces them, also
    // through the evaluation of a candidate (16 points of the patch), as a second
    // copy beside the other lanes': a pick took 227 registers, 172 with them, and
    // at three waves per SIMD (168) spilled 182, now 5.
    CGS_DEV void forget()
    {
#ifdef __HIP_DEVICE_COMPILE__
#pragma unroll
        for (int i = 0; i < 16; i++)
        {
            asm("" : "=v"(p[i].x));
            asm("" : "=v"(p[i].y));
        }
#endif
    }

    CGS_DEV void release()
    {
        held = false;
        sp = lo;
    }

    // Lanes without a region take one from those that have some.
    CGS_DEV void share()
    {
        // An overflowed pair ends for every lane at work on it: its tree can be
        // far larger than the one path the reference follows to overflow.  (The
        // lane that overflowed is without a region now, so the wave gets here.)
        if (__ballot(held && taken))
            if (held && (ldsLoad(w + kClipFlags * 64 + own) & kClipOverflowed)) release();
        const bool spare = held && sp > lo && (taken || !alone);
        const uint64_t give = __ballot(spare), idle = __ballot(!held);
        if (give == 0 || idle == 0) return;
        const uint32_t rank = lanesBelow(give), idleRank = lanesBelow(idle);
        if (spare) w[kClipGiver * 64 + rank] = lane;
        waveOrder();
        const bool take = !held && idleRank < (uint32_t)__popcll(give);
        const uint32_t src = take ? w[kClipGiver * 64 + idleRank] : lane;
        const int srcLo = __shfl(lo, (int)src, 64);
        const uint32_t srcOwn = (uint32_t)__shfl((int)own, (int)src, 64);
        const int srcFinite = __shfl((int)finite, (int)src, 64);
        if (take)
        {
            load(stk.entry(srcLo) + ((int)src - (int)lane));
            held = taken = true;
            finite = srcFinite != 0;
            own = srcOwn;
            sp = lo = srcLo;
            ldsOr(w + kClipFlags * 64 + own, kClipShared);
        }
        else if (spare && rank < (uint32_t)__popcll(idle))
            lo++;
        waveOrder();
    }

    // One pass of every held lane's depth-first walk.
    CGS_DEV void pass(float tol2, uint32_t maxIters)
    {
        bool stop = false;   // ANY: this pair's test is decided
        if (held)
        {
            // The working patch is kept in the orientation of the current
            // cut side: natural (p[4j+i] = point(i,j)) while clipping in u,
            // transposed while clipping in v, so the curves being cut are
            // always the rows p[4r..4r+3] and one code path serves both
            // sides.  Transposing moves values only; every formula below
            // gives the natural-orientation result bit for bit: the
            // tolerance diagonals p3-p12 and p15-p0 change at most by an
            // exact negation, L = (p15-p0) + (p12-p3) in transposed storage
            // equals (p15-p0) - (p12-p3) in natural storage
            // (x + (-y) == x - y), and the envelope visits the same points
            // in the same order.
            bool pop = false, drop = false;
            const V2 t0 {p[3].x - p[12].x, p[3].y - p[12].y};
            const V2 t1 {p[15].x - p[0].x, p[15].y - p[0].y};
            if (CAPPED && iters++ >= maxIters)
                drop = true;
            else if (t0.x * t0.x + t0.y * t0.y < tol2 && t1.x * t1.x + t1.y * t1.y < tol2)
            {
                CGS_COUNT(kWorkConverged);
                // approximateIntersection (Spline.h:739-765) on the natural corners
                const V2 c30 = vside ? p[12] : p[3], c03 = vside ? p[3] : p[12];
                V2 c;
                bool cand[2];
                V2 at[2];
                cand[0] = triangleOrigin(c, p[0], c30, c03);
                at[0] = {mn.x + c.x * sz.x, mn.y + c.y * sz.y};
                cand[1] = triangleOrigin(c, p[15], c03, c30);
                at[1] = {mx.x - c.x * sz.x, mx.y - c.y * sz.y};
                forget();
#pragma unroll 1
                for (int k = 0; k < 2; k++)
                {
                    const float eu = k ? at[1].x : at[0].x, ev = k ? at[1].y : at[0].y;
                    if (!(k ? cand[1] : cand[0])) continue;
                    CGS_COUNT(kWorkOnHit);
                    const uint64_t sa =
                        (uint64_t)w[kClipSLo * 64 + own] | ((uint64_t)w[kClipSHi * 64 + own] << 32);
                    const V3 oo {__uint_as_float(w[kClipOx * 64 + own]), __uint_as_float(w[kClipOy * 64 + own]),
                                 __uint_as_float(w[kClipOz * 64 + own])};
                    const V3 od {__uint_as_float(w[kClipDx * 64 + own]), __uint_as_float(w[kClipDy * 64 + own]),
                                 __uint_as_float(w[kClipDz * 64 + own])};
                    const V3 V = sub3(project4(interpolateMat((const float4*)sa, eu, ev)), oo);
                    const float t = len3(V);
                    if (!(dot3(V, od) > 0.0f)) continue;
                    const uint32_t tb = __float_as_uint(t);
                    if (ANY)
                    {
                        if (t < __uint_as_float(w[kClipKey * 64 + own]))
                        {
                            ldsOr(w + kClipFlags * 64 + own, kClipFound);
                            drop = true;
                            stop = !taken;
                        }
                    }
                    else if (t == t)
                    {
                        const uint32_t old = ldsMin(w + kClipKey * 64 + own, tb);
                        if (tb < old)
                        {
                            // unless another lane's candidate of this turn is nearer still
                            if (ldsLoad(w + kClipKey * 64 + own) == tb)
                            {
                                w[kClipU * 64 + own] = __float_as_uint(eu);
                                w[kClipV * 64 + own] = __float_as_uint(ev);
                            }
                        }
                        else if (tb == old)
                            ldsMin(w + kClipTie * 64 + own, tb);
                    }
                }
                pop = true;
            }
            else
            {
                V2 L {p[15].x - p[0].x, p[15].y - p[0].y};
                const V2 Dv {p[12].x - p[3].x, p[12].y - p[3].y};
                L = {L.x + Dv.x, L.y + Dv.y};
                L = normalize2(L);
                const V2 N {-L.y, L.x};
                // signed distances N·p folded into the envelope as they are
                // computed.  maxNum / minNum: as the reference's fmax / fmin
                // but for the sign of a zero, which the hull below does not
                // depend on (it enters differences, compares, and quotients
                // times an abscissa that is added to a value never -0)
                float ytop[4], ybot[4];
#pragma unroll
                for (int i = 0; i < 4; i++)
                {
                    const float d0 = N.x * p[i].x + N.y * p[i].y;
                    ybot[i] = d0;
                    ytop[i] = d0;
#pragma unroll
                    for (int k = 1; k < 4; k++)
                    {
                        const float dk = N.x * p[4 * k + i].x + N.y * p[4 * k + i].y;
                        ytop[i] = __builtin_fmaxf(ytop[i], dk);
                        ybot[i] = __builtin_fminf(ybot[i], dk);
                    }
                }
                float lower = 1.0f, upper = 0.0f;
                const float o1 = 1.0f / 3.0f, o2 = 2.0f / 3.0f;
                const V2 hull[7] {{o2, ybot[2]}, {1.0f, ybot[3]}, {1.0f, ytop[3]}, {o2, ytop[2]},
                                  {o1, ytop[1]}, {0.0f, ytop[0]}, {0.0f, ybot[0]}};
                V2 P1 {0.0f, ybot[0]};
                V2 P2 {o1, ybot[1]};
#pragma unroll
                for (int h = 0; h < 7; h++)
                {
                    const V2 P3 = hull[h];
                    const bool ccw = isCCW({P2.x - P1.x, P2.y - P1.y}, {P3.x - P1.x, P3.y - P1.y}) >= 0.0f;
                    hullEdge(lower, upper, P1, P2, ccw);
                    P1.x = ccw ? P2.x : P1.x;
                    P1.y = ccw ? P2.y : P1.y;
                    P2 = P3;
                }
                hullEdge(lower, upper, P1, P2, true);
                lower = lower * 0x0FFp-8f;
                upper = upper + (1.0f - upper) * 0x001p-8f;
                const float delta = upper - lower;
                // delta > 0.8: split in half, keep the upper half and push
                // the lower half (Spline_BezierClipping.cu:373-409);
                // otherwise clip to [lower, upper] (:410-432).  Both keep a
                // slice of the rows.
                const bool split = delta > 0.8f;
                if (delta < 0.0f)
                {
                    CGS_COUNT(kWorkPrune);
                    pop = true;
                    forget();
                }
                else if (split && sp >= CGS_CLIP_STACK)
                {
                    ldsOr(w + kClipFlags * 64 + own, kClipOverflowed);
                    drop = true;
                    forget();
                }
                else
                {
                    CGS_COUNT(split ? kWorkSplit : kWorkClip);
                    // region along the cut side (u: x, v: y)
                    const float smn = vside ? mn.y : mn.x, smx = vside ? mx.y : mx.x, ssz = vside ? sz.y : sz.x;
                    float nmn, nmx, nsz;
                    if (split)
                    {
                        // the lower half, pushed for later: rows sliced to
                        // [0, 1/2], stored transposed (the popped entry cuts
                        // the other side: stored word 4c + r holds row r,
                        // point c); the upper half stays.  One de Casteljau
                        // step at 1/2 gives both: the reference slices the
                        // lower half first at 0 and the upper last at 1,
                        // which multiply by 0 and 1 and change nothing but
                        // the sign of a zero (no result depends on one)
                        // while the points are finite; a net with an
                        // infinity or NaN takes the two general slices.
                        float2* e = stk.entry(sp);
#pragma unroll
                        for (int r = 0; r < 4; r++)
                        {
                            V2 c0 = p[4 * r], c1 = p[4 * r + 1], c2 = p[4 * r + 2], c3 = p[4 * r + 3];
                            if (finite)
                            {
                                halve1(c0.x, c1.x, c2.x, c3.x, p[4 * r].x, p[4 * r + 1].x, p[4 * r + 2].x);
                                halve1(c0.y, c1.y, c2.y, c3.y, p[4 * r].y, p[4 * r + 1].y, p[4 * r + 2].y);
                            }
                            else
                            {
                                slice1(c0.x, c1.x, c2.x, c3.x, 0.0f, 1.0f, 0.5f, 0.5f);
                                slice1(c0.y, c1.y, c2.y, c3.y, 0.0f, 1.0f, 0.5f, 0.5f);
                                slice1(p[4 * r].x, p[4 * r + 1].x, p[4 * r + 2].x, p[4 * r + 3].x, 0.5f, 0.5f, 1.0f, 0.0f);
                                slice1(p[4 * r].y, p[4 * r + 1].y, p[4 * r + 2].y, p[4 * r + 3].y, 0.5f, 0.5f, 1.0f, 0.0f);
                            }
                            e[64 * r] = make_float2(c0.x, c0.y);
                            e[64 * (4 + r)] = make_float2(c1.x, c1.y);
                            e[64 * (8 + r)] = make_float2(c2.x, c2.y);
                            e[64 * (12 + r)] = make_float2(c3.x, c3.y);
                        }
                        const float hs = 0.5f * ssz;
                        const float hm = smn + hs;
                        const V2 emx = vside ? V2 {mx.x, hm} : V2 {hm, mx.y};
                        const V2 psz = vside ? V2 {sz.x, hs} : V2 {hs, sz.y};
                        e[64 * 16] = make_float2(mn.x, mn.y);
                        e[64 * 17] = make_float2(emx.x, emx.y);
                        e[64 * 18] = make_float2(psz.x, psz.y);
                        e[64 * 19] = make_float2(vside ? 0.0f : 1.0f, 0.0f);
                        sp++;
                        nmn = hm;
                        nmx = smx;
                        nsz = hs;
                    }
                    else
                    {
                        nmn = smn + ssz * lower;
                        nmx = smx - ssz * (1.0f - upper);
                        nsz = nmx - nmn;
                        subpatchU2(p, lower, upper);
                    }
                    if (vside)
                    {
                        mn.y = nmn;
                        mx.y = nmx;
                        sz.y = nsz;
                    }
                    else
                    {
                        mn.x = nmn;
                        mx.x = nmx;
                        sz.x = nsz;
                    }
                    // the other side is cut next: transpose
#pragma unroll
                    for (int r = 0; r < 4; r++)
#pragma unroll
                        for (int c = r + 1; c < 4; c++)
                        {
                            const V2 t = p[4 * r + c];
                            p[4 * r + c] = p[4 * c + r];
                            p[4 * c + r] = t;
                        }
                    vside = !vside;
                }
            }
            if (drop || (pop && sp == lo))
                release();
            else if (pop)
                load(stk.entry(--sp));
        }
        if (ANY)
        {
            // a lane that stopped its pair is that pair's own (`own` == its lane)
            const uint64_t stopped = __ballot(stop);
            if (held && ((stopped >> own) & 1u)) release();
        }
        waveOrder();
    }
};

// The clipping test of each lane's pair, shared between the wave's lanes;
// every lane calls it together, `have`: with a pair of its own.  best/bu/bv:
// its current hit, updated by accepted candidates (t < best && V·d > 0).
// Returns found; sets overflow when the region stack is exhausted.
template<bool ANY, bool CAPPED = false>
CGS_DEV bool clipWave(const bool have, const float4* __restrict__ S, const V3 o, const V3 d, const float tol2,
                      float& best, float& bu, float& bv, const ClipStack& stk, lds_u32* w, bool& overflow,
                      const uint32_t maxIters = 0)
{
    ClipLane<ANY, CAPPED> c(w, stk);
    bool todo = have;
    if (todo) c.start(S, o, d, best, false);
    waveOrder();
    while (true)
    {
        // ends: every held lane takes one pass of its depth-first walk per turn
        while (__ballot(c.held))
        {
            c.share();
            c.pass(tol2, maxIters);
        }
        todo = todo && c.mustRepeat(best);
        if (__ballot(todo) == 0) break;
        if (todo) c.start(S, o, d, best, true);
        waveOrder();
    }
    if (!have) return false;
    if (c.overflowed()) overflow = true;
    const bool f = c.found(best);
    if (f && !ANY)
    {
        best = c.t();
        bu = c.u();
        bv = c.v();
    }
    return f;
}

} // namespace cgs
