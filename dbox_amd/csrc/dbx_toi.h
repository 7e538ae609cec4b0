// dbx_toi.h -- continuous collision for the step kernels: b2Distance (GJK with a
// simplex cache, src/dbox/collision/b2distance.d:30-707) and b2TimeOfImpact
// (conservative advancement on separating axes, b2timeofimpact.d:67-530), one
// shape pair per lane pair (b2Distance for the overlap test: per lane).
//
// The simplex keeps its three vertices as named members and every access by a
// run-time index goes through a select, so the whole state stays in registers.
// Floating-point operations follow the reference's order; the library is built
// with -ffp-contract=off.
#pragma once

#include "dbx_geom.h"

namespace dbx {

constexpr int kToiUnknown = 0, kToiFailed = 1, kToiOverlapped = 2, kToiTouching = 3, kToiSeparated = 4;

// b2DistanceProxy (b2distance.d:30-140): the shape's vertices (circle centre,
// edge ends, polygon hull) and its radius.  No chain shapes.
struct DProxy {
    const float2 *__restrict__ v;
    int count;
    float radius;
};
__device__ __forceinline__ DProxy make_proxy(const Shape *s) {
    DProxy p;
    p.v = s->type == kCircle ? &s->c : s->v; // edge: v[0] = vertex1, v[1] = vertex2
    p.count = s->type == kCircle ? 1 : (s->type == kEdge ? 2 : s->count);
    p.radius = s->radius;
    return p;
}
// A proxy with its vertices in LDS (kMaxPolygonVertices entries), for the many support
// and evaluate calls of one TOI.
typedef float Float2Vec __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) Float2Vec LdsFloat2;
struct LdsProxy {
    const LdsFloat2 *v;
    int count;
    float radius;
    __device__ __forceinline__ float2 at(int i) const {
        const Float2Vec x = v[i];
        return v2(x.x, x.y);
    }
};
__device__ __forceinline__ LdsProxy make_proxy_in(const Shape *s, LdsFloat2 *buf) {
    const DProxy g = make_proxy(s);
#pragma unroll
    for (int i = 0; i < kMaxPolygonVertices; ++i)
        if (i < g.count) buf[i] = Float2Vec{g.v[i].x, g.v[i].y};
    LdsProxy p;
    p.v = buf;
    p.count = g.count;
    p.radius = g.radius;
    return p;
}
// GetSupport (b2distance.d:94-111): first vertex of largest dot product.
__device__ __forceinline__ int support(const DProxy &p, float2 d) {
    int best = 0;
    float bestValue = dot(p.v[0], d);
    for (int i = 1; i < p.count; ++i) {
        const float value = dot(p.v[i], d);
        if (value > bestValue) {
            best = i;
            bestValue = value;
        }
    }
    return best;
}
// From LDS all entries are read at once, those past the count to no effect: one
// latency for the whole search instead of one per vertex.
__device__ __forceinline__ int support(const LdsProxy &p, float2 d) {
    Float2Vec x[kMaxPolygonVertices];
#pragma unroll
    for (int i = 0; i < kMaxPolygonVertices; ++i) x[i] = p.v[i];
    int best = 0;
    float bestValue = dot(v2(x[0].x, x[0].y), d);
#pragma unroll
    for (int i = 1; i < kMaxPolygonVertices; ++i) {
        const float value = dot(v2(x[i].x, x[i].y), d);
        if (i < p.count && value > bestValue) {
            best = i;
            bestValue = value;
        }
    }
    return best;
}

// b2Sweep (b2math.d:552-593): c0 and a0 at alpha0, c and a at the step's end.
struct Sweep {
    float2 lc, c0, c;
    float a0, a, alpha0;
};
// GetTransform (b2math.d:556-564)
__device__ __forceinline__ Xf sweep_xf(const Sweep &s, float beta) {
    Xf xf;
    xf.p = add(scl(1.0f - beta, s.c0), scl(beta, s.c));
    const float angle = (1.0f - beta) * s.a0 + beta * s.a;
    xf.q = rot(angle);
    xf.p = sub(xf.p, mul(xf.q, s.lc));
    return xf;
}
// Advance (b2math.d:568-575)
__device__ __forceinline__ void sweep_advance(Sweep &s, float alpha) {
    const float beta = (alpha - s.alpha0) / (1.0f - s.alpha0);
    s.c0 = add(s.c0, scl(beta, sub(s.c, s.c0)));
    s.a0 += beta * (s.a - s.a0);
    s.alpha0 = alpha;
}
// Normalize (b2math.d:578-584)
__device__ __forceinline__ void sweep_normalize(Sweep &s) {
    const float twoPi = 2.0f * kPi;
    const float d = twoPi * floorf(s.a0 / twoPi);
    s.a0 -= d;
    s.a -= d;
}

struct SimplexCache {
    float metric;
    int count;
    int iA0, iA1, iA2, iB0, iB1, iB2;
};
struct SVert {
    float2 wA, wB, w;
    float a;
    int iA, iB;
};
struct Simplex {
    SVert v1, v2, v3;
    int count;
};

// Two proxies and their transforms on one lane.
struct LaneShapes {
    DProxy pA, pB;
    Xf xfA, xfB;
    __device__ __forceinline__ SVert vertex(int iA, int iB) const {
        SVert s;
        s.iA = iA;
        s.iB = iB;
        s.wA = mul(xfA, pA.v[iA]);
        s.wB = mul(xfB, pB.v[iB]);
        s.w = sub(s.wB, s.wA);
        s.a = 0.0f;
        return s;
    }
    __device__ __forceinline__ void supports(float2 d, int &iA, int &iB) const {
        iA = support(pA, mulT(xfA.q, neg(d)));
        iB = support(pB, mulT(xfB.q, d));
    }
};
// The same on a lane pair, which takes every branch together: the even lane holds and
// evaluates body A's side, the odd lane body B's, and the two exchange the results.  A
// TOI is one long chain of instructions whose transforms (a sine and a cosine in double
// precision for each body at each time looked at) are most of it; this way it does
// each body's half only.  64 rooms of 40 projectiles: 586 us a step with a TOI per lane,
// 560 so.
struct PairShapes {
    LdsProxy own;
    Xf xf;
    bool odd;
    __device__ __forceinline__ SVert vertex(int iA, int iB) const {
        SVert s;
        s.iA = iA;
        s.iB = iB;
        const float2 w = mul(xf, own.at(odd ? iB : iA)), o = pair_swap(w);
        s.wA = v2(odd ? o.x : w.x, odd ? o.y : w.y);
        s.wB = v2(odd ? w.x : o.x, odd ? w.y : o.y);
        s.w = sub(s.wB, s.wA);
        s.a = 0.0f;
        return s;
    }
    __device__ __forceinline__ void supports(float2 d, int &iA, int &iB) const {
        const int i = support(own, mulT(xf.q, odd ? d : neg(d))), o = pair_swap(i);
        iA = odd ? o : i;
        iB = odd ? i : o;
    }
};
// GetMetric (b2distance.d:710-728)
__device__ __forceinline__ float simplex_metric(const Simplex &s) {
    if (s.count == 1) return 0.0f;
    if (s.count == 2) {
        const float2 d = sub(s.v1.w, s.v2.w);
        return sqrtf(d.x * d.x + d.y * d.y);
    }
    return crs(sub(s.v2.w, s.v1.w), sub(s.v3.w, s.v1.w));
}
// ReadCache (b2distance.d:574-624)
template <class P>
__device__ __forceinline__ void read_cache(Simplex &s, const SimplexCache &c, const P &p) {
    s.count = c.count;
    if (c.count > 0) s.v1 = p.vertex(c.iA0, c.iB0);
    if (c.count > 1) s.v2 = p.vertex(c.iA1, c.iB1);
    if (c.count > 2) s.v3 = p.vertex(c.iA2, c.iB2);
    if (s.count > 1) {
        const float metric1 = c.metric;
        const float metric2 = simplex_metric(s);
        if (metric2 < 0.5f * metric1 || 2.0f * metric1 < metric2 || metric2 < kEps) s.count = 0;
    }
    if (s.count == 0) {
        s.v1 = p.vertex(0, 0);
        s.v1.a = 1.0f;
        s.count = 1;
    }
}
// WriteCache (b2distance.d:626-637)
__device__ __forceinline__ void write_cache(const Simplex &s, SimplexCache &c) {
    c.metric = simplex_metric(s);
    c.count = s.count;
    c.iA0 = s.v1.iA;
    c.iB0 = s.v1.iB;
    c.iA1 = s.v2.iA;
    c.iB1 = s.v2.iB;
    c.iA2 = s.v3.iA;
    c.iB2 = s.v3.iB;
}
// Solve2 (b2distance.d:373-406)
__device__ __forceinline__ void solve2(Simplex &s) {
    const float2 w1 = s.v1.w, w2 = s.v2.w;
    const float2 e12 = sub(w2, w1);
    const float d12_2 = -dot(w1, e12);
    if (d12_2 <= 0.0f) {
        s.v1.a = 1.0f;
        s.count = 1;
        return;
    }
    const float d12_1 = dot(w2, e12);
    if (d12_1 <= 0.0f) {
        s.v2.a = 1.0f;
        s.count = 1;
        s.v1 = s.v2;
        return;
    }
    const float inv_d12 = 1.0f / (d12_1 + d12_2);
    s.v1.a = d12_1 * inv_d12;
    s.v2.a = d12_2 * inv_d12;
    s.count = 2;
}
// Solve3 (b2distance.d:413-571)
__device__ __forceinline__ void solve3(Simplex &s) {
    const float2 w1 = s.v1.w, w2 = s.v2.w, w3 = s.v3.w;
    const float2 e12 = sub(w2, w1);
    const float w1e12 = dot(w1, e12), w2e12 = dot(w2, e12);
    const float d12_1 = w2e12, d12_2 = -w1e12;
    const float2 e13 = sub(w3, w1);
    const float w1e13 = dot(w1, e13), w3e13 = dot(w3, e13);
    const float d13_1 = w3e13, d13_2 = -w1e13;
    const float2 e23 = sub(w3, w2);
    const float w2e23 = dot(w2, e23), w3e23 = dot(w3, e23);
    const float d23_1 = w3e23, d23_2 = -w2e23;
    const float n123 = crs(e12, e13);
    const float d123_1 = n123 * crs(w2, w3);
    const float d123_2 = n123 * crs(w3, w1);
    const float d123_3 = n123 * crs(w1, w2);
    if (d12_2 <= 0.0f && d13_2 <= 0.0f) {
        s.v1.a = 1.0f;
        s.count = 1;
        return;
    }
    if (d12_1 > 0.0f && d12_2 > 0.0f && d123_3 <= 0.0f) {
        const float inv_d12 = 1.0f / (d12_1 + d12_2);
        s.v1.a = d12_1 * inv_d12;
        s.v2.a = d12_2 * inv_d12;
        s.count = 2;
        return;
    }
    if (d13_1 > 0.0f && d13_2 > 0.0f && d123_2 <= 0.0f) {
        const float inv_d13 = 1.0f / (d13_1 + d13_2);
        s.v1.a = d13_1 * inv_d13;
        s.v3.a = d13_2 * inv_d13;
        s.count = 2;
        s.v2 = s.v3;
        return;
    }
    if (d12_1 <= 0.0f && d23_2 <= 0.0f) {
        s.v2.a = 1.0f;
        s.count = 1;
        s.v1 = s.v2;
        return;
    }
    if (d13_1 <= 0.0f && d23_1 <= 0.0f) {
        s.v3.a = 1.0f;
        s.count = 1;
        s.v1 = s.v3;
        return;
    }
    if (d23_1 > 0.0f && d23_2 > 0.0f && d123_1 <= 0.0f) {
        const float inv_d23 = 1.0f / (d23_1 + d23_2);
        s.v2.a = d23_1 * inv_d23;
        s.v3.a = d23_2 * inv_d23;
        s.count = 2;
        s.v1 = s.v3;
        return;
    }
    const float inv_d123 = 1.0f / (d123_1 + d123_2 + d123_3);
    s.v1.a = d123_1 * inv_d123;
    s.v2.a = d123_2 * inv_d123;
    s.v3.a = d123_3 * inv_d123;
    s.count = 3;
}

// b2Distance (b2distance.d:185-345) without radii: the distance of the two
// shapes' cores and the simplex left in the cache.
template <class P>
__device__ __forceinline__ float gjk_distance(SimplexCache &cache, const P &p) {
    Simplex s;
    read_cache(s, cache, p);
    int sA0 = 0, sA1 = 0, sA2 = 0, sB0 = 0, sB1 = 0, sB2 = 0;
    for (int iter = 0; iter < 20;) {
        const int saveCount = s.count;
        sA0 = s.v1.iA;
        sB0 = s.v1.iB;
        sA1 = s.v2.iA;
        sB1 = s.v2.iB;
        sA2 = s.v3.iA;
        sB2 = s.v3.iB;
        if (s.count == 2) solve2(s);
        else if (s.count == 3) solve3(s);
        if (s.count == 3) break;
        // GetSearchDirection (b2distance.d:639-662)
        float2 d;
        if (s.count == 1) {
            d = neg(s.v1.w);
        } else {
            const float2 e12 = sub(s.v2.w, s.v1.w);
            const float sgn = crs(e12, neg(s.v1.w));
            d = sgn > 0.0f ? crs(1.0f, e12) : crs(e12, 1.0f);
        }
        if (lensq(d) < kEps * kEps) break;
        int iA, iB;
        p.supports(d, iA, iB);
        const SVert nv = p.vertex(iA, iB);
        ++iter;
        const bool dup = (saveCount > 0 && iA == sA0 && iB == sB0) || (saveCount > 1 && iA == sA1 && iB == sB1) ||
                         (saveCount > 2 && iA == sA2 && iB == sB2);
        if (dup) break;
        if (s.count == 1) s.v2 = nv;
        else s.v3 = nv;
        ++s.count;
    }
    // GetWitnessPoints (b2distance.d:686-708)
    float2 wa, wb;
    if (s.count == 1) {
        wa = s.v1.wA;
        wb = s.v1.wB;
    } else if (s.count == 2) {
        wa = add(scl(s.v1.a, s.v1.wA), scl(s.v2.a, s.v2.wA));
        wb = add(scl(s.v1.a, s.v1.wB), scl(s.v2.a, s.v2.wB));
    } else {
        wa = add(add(scl(s.v1.a, s.v1.wA), scl(s.v2.a, s.v2.wA)), scl(s.v3.a, s.v3.wA));
        wb = wa;
    }
    write_cache(s, cache);
    const float2 dd = sub(wa, wb);
    return sqrtf(dd.x * dd.x + dd.y * dd.y);
}

// b2TestOverlap of two shapes (b2collision.d:449-468): b2Distance with radii from
// an empty cache (b2distance.d:327-344); overlapping below 10 epsilon.
__device__ __noinline__ bool test_overlap(const Shape *a, const Xf &xfA, const Shape *b, const Xf &xfB) {
    SimplexCache cache;
    cache.count = 0;
    const LaneShapes p{make_proxy(a), make_proxy(b), xfA, xfB};
    const float d = gjk_distance(cache, p);
    const float r = p.pA.radius + p.pB.radius;
    const float dist = (d > r && d > kEps) ? d - r : 0.0f;
    return dist < 10.0f * kEps;
}

// b2SeparationFunction (b2timeofimpact.d:297-530) on a lane pair: the lane's own sweep
// and proxy.
struct SepFn {
    Sweep s;
    int type; // 0 points, 1 faceA, 2 faceB
    bool face; // the face (lp, axis) is on this lane's body
    float2 lp, axis;
};
// A lane's own value where `own`, else the other lane's.
__device__ __forceinline__ float2 pair_pick(bool own, float2 x) {
    const float2 o = pair_swap(x);
    return v2(own ? x.x : o.x, own ? x.y : o.y);
}
// dot(pB - pA, n) of the lanes' points (types 0 and 1), dot(pA - pB, n) for type 2.
__device__ __forceinline__ float pair_separation(bool minuend, float2 p, float2 n) {
    const float2 o = pair_swap(p);
    return dot(v2(minuend ? p.x - o.x : o.x - p.x, minuend ? p.y - o.y : o.y - p.y), n);
}
// Initialize (b2timeofimpact.d:331-410)
__device__ __forceinline__ void sep_init(SepFn &f, const SimplexCache &cache, const LdsProxy &own, bool odd,
                                         const Sweep &s, float t1) {
    f.s = s;
    const Xf xf = sweep_xf(s, t1);
    const float2 e0 = own.at(odd ? cache.iB0 : cache.iA0);
    if (cache.count == 1) {
        f.type = 0;
        f.face = false;
        const float2 w = mul(xf, e0), o = pair_swap(w);
        f.axis = odd ? sub(w, o) : sub(o, w);
        normalize(f.axis);
        f.lp = v2(0.0f, 0.0f);
        return;
    }
    const float2 e1 = own.at(odd ? cache.iB1 : cache.iA1);
    f.type = cache.iA0 == cache.iA1 ? 2 : 1;
    f.face = odd == (f.type == 2);
    const float2 f0 = pair_pick(f.face, e0), f1 = pair_pick(f.face, e1);
    f.axis = crs(sub(f1, f0), 1.0f);
    normalize(f.axis);
    const float2 normal = pair_pick(f.face, mul(xf.q, f.axis));
    f.lp = scl(0.5f, add(f0, f1));
    const float sep = pair_separation(!f.face, mul(xf, f.face ? f.lp : e0), normal);
    if (sep < 0.0f) f.axis = neg(f.axis);
}
// FindMinSeparation (b2timeofimpact.d:413-470); v: this lane's vertex.
__device__ __forceinline__ float sep_find_min(const SepFn &f, const LdsProxy &own, bool odd, float2 &v, float t) {
    const Xf xf = sweep_xf(f.s, t);
    if (f.type == 0) {
        v = own.at(support(own, mulT(xf.q, odd ? neg(f.axis) : f.axis)));
        return pair_separation(odd, mul(xf, v), f.axis);
    }
    const float2 normal = pair_pick(f.face, mul(xf.q, f.axis));
    v = own.at(support(own, mulT(xf.q, neg(normal))));
    return pair_separation(!f.face, mul(xf, f.face ? f.lp : v), normal);
}
// Evaluate (b2timeofimpact.d:473-518)
__device__ __forceinline__ float sep_eval(const SepFn &f, bool odd, float2 v, float t) {
    const Xf xf = sweep_xf(f.s, t);
    if (f.type == 0) return pair_separation(odd, mul(xf, v), f.axis);
    const float2 normal = pair_pick(f.face, mul(xf.q, f.axis));
    return pair_separation(!f.face, mul(xf, f.face ? f.lp : v), normal);
}

// b2TimeOfImpact (b2timeofimpact.d:67-295) over [0, tMax]; returns the output
// state and writes the time.  Every loop is bounded as in the reference (20
// outer iterations, b2_maxPolygonVertices push-backs, 50 root-finder steps).  On a lane
// pair: own and s are body A's on the even lane and body B's on the odd one; both
// lanes return the same.
__device__ __forceinline__ int time_of_impact(float &tOut, const LdsProxy &own, Sweep s, float tMax) {
    const bool odd = (threadIdx.x & 1) != 0;
    int state = kToiUnknown;
    tOut = tMax;
    sweep_normalize(s);
    const float totalRadius = own.radius + pair_swap(own.radius);
    const float target = fmaxr(kLinearSlop, totalRadius - 3.0f * kLinearSlop);
    const float tolerance = 0.25f * kLinearSlop;
    float t1 = 0.0f;
    SimplexCache cache;
    cache.count = 0;
    cache.metric = 0.0f;
    cache.iA0 = cache.iA1 = cache.iA2 = cache.iB0 = cache.iB1 = cache.iB2 = 0;
    for (int iter = 0;;) {
        const PairShapes p{own, sweep_xf(s, t1), odd};
        const float distance = gjk_distance(cache, p);
        if (distance <= 0.0f) {
            state = kToiOverlapped;
            tOut = 0.0f;
            break;
        }
        if (distance < target + tolerance) {
            state = kToiTouching;
            tOut = t1;
            break;
        }
        SepFn fcn;
        sep_init(fcn, cache, own, odd, s, t1);
        bool done = false;
        float t2 = tMax;
        for (int pushBackIter = 0;;) {
            float2 v;
            float s2 = sep_find_min(fcn, own, odd, v, t2);
            if (s2 > target + tolerance) {
                state = kToiSeparated;
                tOut = tMax;
                done = true;
                break;
            }
            if (s2 > target - tolerance) {
                t1 = t2;
                break;
            }
            float s1 = sep_eval(fcn, odd, v, t1);
            if (s1 < target - tolerance) {
                state = kToiFailed;
                tOut = t1;
                done = true;
                break;
            }
            if (s1 <= target + tolerance) {
                state = kToiTouching;
                tOut = t1;
                done = true;
                break;
            }
            float a1 = t1, a2 = t2;
            for (int rootIterCount = 0;;) {
                float t;
                if (rootIterCount & 1) t = a1 + (target - s1) * (a2 - a1) / (s2 - s1);
                else t = 0.5f * (a1 + a2);
                ++rootIterCount;
                const float sep = sep_eval(fcn, odd, v, t);
                if (fabsr(sep - target) < tolerance) {
                    t2 = t;
                    break;
                }
                if (sep > target) {
                    a1 = t;
                    s1 = sep;
                } else {
                    a2 = t;
                    s2 = sep;
                }
                if (rootIterCount == 50) break;
            }
            ++pushBackIter;
            if (pushBackIter == kMaxPolygonVertices) break;
        }
        ++iter;
        if (done) break;
        if (iter == 20) {
            state = kToiFailed;
            tOut = t1;
            break;
        }
    }
    return state;
}

} // namespace dbx
