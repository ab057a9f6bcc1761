// sphgeom.hpp -- FP64 spherical polygon geometry for the gfx950 kernels.
//
// Replaces the per-pair operator of the reference,
//   DefaultIntersectionOperator{Spherical}(p1, p2) =
//       GO.area(m, GO.intersection(ConvexConvexSutherlandHodgman(m), p1, p2))
//   (src/regridder/regridder.jl:96-103),
// and the cell areas of areas() (regridder.jl:165-178).
//
// Design for registers, not buffers: Sutherland-Hodgman is run as the
// re-entrant pipeline of its original paper -- one stage per clip edge, each
// stage holding only (first, previous) vertex and side value.  Subject vertices
// are streamed from memory one at a time and every vertex a stage emits is
// pushed straight into the next stage; the last stage feeds the area
// accumulator.  State is O(clip edges) doubles no matter how many vertices the
// subject polygon has (16 for a HEALPix step-4 cell), so the kernel needs no
// per-thread scratch arrays.
//
// Numerics (shared with the CPU oracle as published formulas, not as code):
//   edge a->b: great circle with normal n = a x (b - a); side(v) = n . (v - a),
//   inside iff side >= 0.  Crossing of edge p->q: the positive combination
//   |s_q| p + |s_p| q, renormalised (it lies on the plane for opposite signs).
//   Area: triangle solid angle tan(E/2) = a.((b-a)x(c-a)) / (1 + a.b + b.c + c.a)
//   (Van Oosterom & Strackee 1983), fan from the first vertex.  The fan's angles
//   are summed as the argument of a product of complex numbers, so each polygon
//   needs one atan2 instead of one per triangle.
#pragma once

#include "common.hpp"

namespace cr {

struct d3 {
    double x, y, z;
};

CR_HD d3 mk3(double x, double y, double z) { return d3{x, y, z}; }
CR_HD d3 operator-(const d3 &a, const d3 &b) { return d3{a.x - b.x, a.y - b.y, a.z - b.z}; }
CR_HD d3 operator+(const d3 &a, const d3 &b) { return d3{a.x + b.x, a.y + b.y, a.z + b.z}; }
CR_HD d3 operator*(double s, const d3 &a) { return d3{s * a.x, s * a.y, s * a.z}; }
CR_HD double dot(const d3 &a, const d3 &b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
CR_HD d3 cross(const d3 &a, const d3 &b) {
    return d3{a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}
CR_HD d3 load3(const double *p) { return d3{p[0], p[1], p[2]}; }
CR_HD d3 normalized(const d3 &a) { return (1.0 / sqrt(dot(a, a))) * a; }

// Squared length below which a clip edge is treated as degenerate (coincident
// vertices, e.g. the two pole corners of a lon-lat polar cell).
constexpr double kDegenerateEdge2 = 1e-26;

// Fan-area accumulator: angle sum as arg of a running complex product.
struct AreaAcc {
    d3 w0, prev;
    double re, im;
    int n;
    CR_HD void init() { re = 1.0; im = 0.0; n = 0; }
    CR_HD void push(const d3 &w) {
        if (n >= 2) {
            d3 e1 = prev - w0, e2 = w - w0;
            double num = dot(w0, cross(e1, e2));
            double den = 1.0 + dot(w0, prev) + dot(prev, w) + dot(w, w0);
            // scale by 1/4 (exact) to keep the product near unit magnitude
            num *= 0.25;
            den *= 0.25;
            double r = re * den - im * num;
            double i = re * num + im * den;
            re = r;
            im = i;
        } else if (n == 0) {
            w0 = w;
        }
        prev = w;
        ++n;
    }
    CR_HD double area() const { return n >= 3 ? 2.0 * atan2(im, re) : 0.0; }
};

// One clip stage per clip-polygon edge, unrolled at compile time (NC stages).
template <int NC>
struct ClipPipe {
    d3 anchor[NC];
    d3 nrm[NC];
    d3 first[NC];
    d3 prev[NC];
    double sfirst[NC];
    double sprev[NC];
    bool started[NC];
    AreaAcc acc;

    // Stage k clips against the great circle of edge (a -> b).  A degenerate
    // edge gets a zero normal: every vertex is then "inside" (side 0) and the
    // stage passes the polygon through unchanged.
    CR_HD void set_edge(int k, const d3 &a, const d3 &b) {
        d3 n = cross(a, b - a);
        if (dot(n, n) < kDegenerateEdge2) n = mk3(0.0, 0.0, 0.0);
        anchor[k] = a;
        nrm[k] = n;
        started[k] = false;
    }
    CR_HD void init() { acc.init(); }
};

// 1/sqrt(v): the device's rsqrt (one instruction sequence, no IEEE division);
// the host build divides.  Either is within an ulp or two, which only moves a
// renormalised point along its ray.
CR_HD double inv_norm(double v) {
#ifdef __HIP_DEVICE_COMPILE__
    return rsqrt(v);
#else
    return 1.0 / sqrt(v);
#endif
}

CR_HD d3 crossing(const d3 &p, double sp, const d3 &q, double sq) {
    d3 x = fabs(sq) * p + fabs(sp) * q;
    return inv_norm(dot(x, x)) * x;
}

template <int K, int NC>
CR_HD void pipe_push(ClipPipe<NC> &P, const d3 &v);

// Sutherland-Hodgman rule for edge p->q at stage K: a crossing when the side
// changes, then q when it is inside.  The (at most two) outputs are forwarded
// by a loop that is not unrolled, so each stage's downstream code exists once
// and the kernel grows linearly, not exponentially, with the number of stages.
template <int K, int NC>
CR_HD void pipe_edge(ClipPipe<NC> &P, const d3 &p, double sp, const d3 &q, double sq) {
    const bool qin = sq >= 0.0;
    const bool crosses = (sp >= 0.0) != qin;
    d3 x = q;
    if (crosses) x = crossing(p, sp, q, sq);
    const int m = (int)crosses + (int)qin;
#pragma unroll 1
    for (int e = 0; e < m; ++e) {
        d3 u = (e == 0) ? x : q;
        pipe_push<K + 1, NC>(P, u);
    }
}

template <int K, int NC>
CR_HD void pipe_push(ClipPipe<NC> &P, const d3 &v) {
    if constexpr (K == NC) {
        P.acc.push(v);
    } else {
        double s = dot(P.nrm[K], v - P.anchor[K]);
        if (!P.started[K]) {
            P.started[K] = true;
            P.first[K] = v;
            P.sfirst[K] = s;
        } else {
            pipe_edge<K, NC>(P, P.prev[K], P.sprev[K], v, s);
        }
        P.prev[K] = v;
        P.sprev[K] = s;
    }
}

// Close every stage in order: the closing edge (last -> first) of stage K may
// emit vertices into stage K+1 before that stage is closed.
template <int K, int NC>
CR_HD void pipe_close(ClipPipe<NC> &P) {
    if constexpr (K < NC) {
        if (P.started[K]) pipe_edge<K, NC>(P, P.prev[K], P.sprev[K], P.first[K], P.sfirst[K]);
        pipe_close<K + 1, NC>(P);
    }
}

// Area of (subject ∩ clip) for a clip polygon of at most NC vertices (padded by
// repeating its last vertex) and a subject of ns vertices read from memory.
template <int NC>
CR_HD double clip_area_stream(const double *clip, int nc, const double *subj, int ns) {
    ClipPipe<NC> P;
    P.init();
    d3 c[NC];
#pragma unroll
    for (int k = 0; k < NC; ++k) c[k] = load3(clip + 3 * (k < nc ? k : nc - 1));
#pragma unroll
    for (int k = 0; k < NC; ++k) P.set_edge(k, c[k], c[(k + 1) % NC]);
    // subject vertices are loaded two ahead of the one being clipped, so their
    // latency overlaps the pipeline's work
    d3 v0 = load3(subj), v1 = load3(subj + 3 * (ns > 1 ? 1 : 0));
    for (int i = 0; i < ns; ++i) {
        const d3 v2 = load3(subj + 3 * (i + 2 < ns ? i + 2 : ns - 1));
        pipe_push<0, NC>(P, v0);
        v0 = v1;
        v1 = v2;
    }
    pipe_close<0, NC>(P);
    return P.acc.area();
}

// The same with a pipeline of NS stages, one per clip edge whose bit is set in
// `mask` (exactly NS bits, in edge order).  An edge that has every subject
// vertex on its inside passes the clipped polygon through unchanged (the
// polygon stays inside the subject, which is inside that edge's hemisphere),
// so dropping its stage changes nothing but rounding.
template <int K, int NS, int NC>
CR_HD void pipe_set_masked(ClipPipe<NS> &P, const double *clip, int nc, unsigned mask) {
    if constexpr (K < NS) {
        const int e = __builtin_ctz(mask), e1 = (e + 1) % NC;
        P.set_edge(K, load3(clip + 3 * (e < nc ? e : nc - 1)), load3(clip + 3 * (e1 < nc ? e1 : nc - 1)));
        pipe_set_masked<K + 1, NS, NC>(P, clip, nc, mask & (mask - 1));
    }
}

template <int NS, int NC>
CR_HD double clip_area_stream_masked(const double *clip, int nc, unsigned mask, const double *subj, int ns) {
    ClipPipe<NS> P;
    P.init();
    pipe_set_masked<0, NS, NC>(P, clip, nc, mask);
    d3 v0 = load3(subj), v1 = load3(subj + 3 * (ns > 1 ? 1 : 0));
    for (int i = 0; i < ns; ++i) {
        const d3 v2 = load3(subj + 3 * (i + 2 < ns ? i + 2 : ns - 1));
        pipe_push<0, NS>(P, v0);
        v0 = v1;
        v1 = v2;
    }
    pipe_close<0, NS>(P);
    return P.acc.area();
}

// `mask` with its lowest clear bits set until it has n bits (n <= NC).
CR_HD unsigned pad_mask(unsigned mask, int n) {
    while (__builtin_popcount(mask) < n) mask |= ~mask & (mask + 1u);
    return mask;
}

// Where the subject lies against the clip polygon, by the pipeline's own side
// test n.(v - a) (a degenerate edge has n = 0: everything is on its inside):
// kSubjectOutside when every subject vertex is strictly outside one clip edge
// (the intersection is empty), kSubjectInside when every vertex is inside
// every edge (the pipeline would pass the subject through unchanged: the
// intersection is the subject), kSubjectCrosses otherwise.
enum { kSubjectOutside = 0, kSubjectInside = 1, kSubjectCrosses = 2 };

template <int NC>
CR_HD int classify_subject(const double *clip, int nc, const double *subj, int ns, unsigned *crossed = nullptr) {
    d3 a[NC], n[NC];
#pragma unroll
    for (int k = 0; k < NC; ++k) a[k] = load3(clip + 3 * (k < nc ? k : nc - 1));
    bool out[NC];
#pragma unroll
    for (int k = 0; k < NC; ++k) {
        d3 nk = cross(a[k], a[(k + 1) % NC] - a[k]);
        if (dot(nk, nk) < kDegenerateEdge2) nk = mk3(0.0, 0.0, 0.0);
        out[k] = true;
        n[k] = nk;
    }
    bool in = true;
    unsigned cut = 0;  // edges with a subject vertex outside
    for (int i = 0; i < ns; ++i) {
        const d3 v = load3(subj + 3 * i);
#pragma unroll
        for (int k = 0; k < NC; ++k) {
            const double s = dot(n[k], v - a[k]);
            out[k] = out[k] && s < 0.0;
            cut |= (s < 0.0 ? 1u : 0u) << k;
        }
    }
    in = cut == 0;
    if (crossed) *crossed = cut;
    bool any = false;
#pragma unroll
    for (int k = 0; k < NC; ++k) any = any || out[k];
    return any ? kSubjectOutside : (in ? kSubjectInside : kSubjectCrosses);
}

// Signed area of an open ring of n vertices.
CR_HD double ring_area(const double *xyz, int n) {
    AreaAcc a;
    a.init();
    for (int i = 0; i < n; ++i) a.push(load3(xyz + 3 * i));
    return a.area();
}


// ============================================================================
// Backward: d(area of subject ∩ clip) / d(vertices), by provenance.
//
// Every vertex of the clipped polygon is, in exact arithmetic, a subject
// vertex, a clip vertex, or the crossing of two great circles (a subject edge
// with a clip edge, or two clip edges).  The pipeline below is the forward one
// with a label carried next to each vertex; a crossing's label comes from the
// line the clipped segment lies on (the line its two endpoints share).  The
// area stage differentiates each fan triangle,
//   E = 2 atan2(T, D),  T = a.(b x c),  D = 1 + a.b + b.c + c.a,
//   dE/da = 2 (D (b x c) - T (b + c)) / (T^2 + D^2)   (and cyclic),
// and hands (label, position, gradient) to a sink, which chains through the
// crossing x = y/|y|, y = +-(n1 x n2), n = p x q, to the input vertices.
// ============================================================================

// label: bits 28-29 type, bits 8-27 and 0-7 indices (a subject vertex uses
// bits 0-27); -1 (sign bit) marks a vertex without provenance
constexpr int32_t kLabS = 0, kLabC = 1, kLabXF = 2, kLabXE = 3;
constexpr int32_t kLabIndexMask = 0x0fffffff;
CR_HD int32_t lab_make(int32_t type, int32_t a, int32_t b) { return (type << 28) | (a << 8) | b; }
CR_HD int32_t lab_type(int32_t l) { return (l >> 28) & 3; }
CR_HD int32_t lab_hi(int32_t l) { return (l >> 8) & 0xfffff; }
CR_HD int32_t lab_lo(int32_t l) { return l & 0xff; }

// line ids: subject edge e -> e, clip edge k -> kClipLine | k
constexpr int32_t kClipLine = 1 << 27;

template <int NC>
CR_HD void lab_lines(int32_t l, int ns, int32_t &l1, int32_t &l2) {
    int32_t t = lab_type(l), a = lab_hi(l), b = lab_lo(l);
    if (t == kLabS) {
        int32_t e = l & kLabIndexMask;
        l1 = e == 0 ? ns - 1 : e - 1;
        l2 = e;
    }
    else if (t == kLabC) { l1 = kClipLine | ((b + NC - 1) % NC); l2 = kClipLine | b; }
    else if (t == kLabXF) { l1 = a; l2 = kClipLine | b; }
    else { l1 = kClipLine | a; l2 = kClipLine | b; }
}

// Label of the crossing of segment p->q with clip edge K.
template <int NC>
CR_HD int32_t lab_crossing(int32_t lp, int32_t lq, int K, int ns) {
    int32_t p1, p2, q1, q2;
    lab_lines<NC>(lp, ns, p1, p2);
    lab_lines<NC>(lq, ns, q1, q2);
    int32_t line = (p1 == q1 || p1 == q2) ? p1 : ((p2 == q1 || p2 == q2) ? p2 : -1);
    if (line < 0) return -1;  // no shared line (degenerate input): no gradient
    if (!(line & kClipLine)) return lab_make(kLabXF, line, K);
    int a = line & 0xff;
    if (a == (K + NC - 1) % NC) return lab_make(kLabC, 0, K);
    if (a == (K + 1) % NC) return lab_make(kLabC, 0, (K + 1) % NC);
    return lab_make(kLabXE, a, K);
}

CR_HD d3 tangential(const d3 &g, const d3 &x) { return g - dot(g, x) * x; }

template <int NC, class Sink>
struct GradPipe {
    d3 anchor[NC];
    d3 *nrm;  // the NC edge normals, in caller memory (LDS) to spare registers
    d3 first[NC], prev[NC];
    double sfirst[NC], sprev[NC];
    int32_t lfirst[NC], lprev[NC];
    bool started[NC];
    int ns;
    double coef;
    Sink *sink;
    // area stage: fan triangles (w0, wp, w); the previous vertex's part from
    // the last triangle waits in pend until the next triangle completes it,
    // so each vertex reaches the sink once (the sink is linear in g)
    d3 w0, wp, g0, pend;
    int32_t l0, lp;
    int n;

    CR_HD void area_push(const d3 &w, int32_t l) {
        if (n == 0) {
            w0 = w;
            l0 = l;
            g0 = mk3(0, 0, 0);
            pend = mk3(0, 0, 0);
        } else if (n >= 2) {
            d3 a = w0, b = wp, c = w;
            double T = dot(a, cross(b, c));
            double D = 1.0 + dot(a, b) + dot(b, c) + dot(c, a);
            double f = 2.0 / (T * T + D * D);
            g0 = g0 + f * (D * cross(b, c) - T * (b + c));
            (*sink)(lp, b, pend + (coef * f) * (D * cross(c, a) - T * (a + c)));
            pend = (coef * f) * (D * cross(a, b) - T * (a + b));
        }
        wp = w;
        lp = l;
        ++n;
    }
    CR_HD void area_close() {
        if (n < 3) return;
        (*sink)(lp, wp, pend);
        (*sink)(l0, w0, coef * g0);
    }
};

template <int K, int NC, class Sink>
CR_HD void gpipe_push(GradPipe<NC, Sink> &P, const d3 &v, int32_t l);

template <int K, int NC, class Sink>
CR_HD void gpipe_edge(GradPipe<NC, Sink> &P, const d3 &p, double sp, int32_t lp, const d3 &q,
                      double sq, int32_t lq) {
    const bool qin = sq >= 0.0;
    const bool crosses = (sp >= 0.0) != qin;
    d3 x = q;
    int32_t lx = lq;
    if (crosses) {
        x = crossing(p, sp, q, sq);
        lx = lab_crossing<NC>(lp, lq, K, P.ns);
    }
    const int m = (int)crosses + (int)qin;
#pragma unroll 1
    for (int e = 0; e < m; ++e) {
        d3 u = (e == 0) ? x : q;
        int32_t lu = (e == 0) ? lx : lq;
        gpipe_push<K + 1, NC, Sink>(P, u, lu);
    }
}

template <int K, int NC, class Sink>
CR_HD void gpipe_push(GradPipe<NC, Sink> &P, const d3 &v, int32_t l) {
    if constexpr (K == NC) {
        P.area_push(v, l);
    } else {
        double s = dot(P.nrm[K], v - P.anchor[K]);
        if (!P.started[K]) {
            P.started[K] = true;
            P.first[K] = v;
            P.sfirst[K] = s;
            P.lfirst[K] = l;
        } else {
            gpipe_edge<K, NC, Sink>(P, P.prev[K], P.sprev[K], P.lprev[K], v, s, l);
        }
        P.prev[K] = v;
        P.sprev[K] = s;
        P.lprev[K] = l;
    }
}

template <int K, int NC, class Sink>
CR_HD void gpipe_close(GradPipe<NC, Sink> &P) {
    if constexpr (K < NC) {
        if (P.started[K])
            gpipe_edge<K, NC, Sink>(P, P.prev[K], P.sprev[K], P.lprev[K], P.first[K], P.sfirst[K],
                                    P.lfirst[K]);
        gpipe_close<K + 1, NC, Sink>(P);
    }
}

// Scatter coef * d(area)/d(vertex) of (subject ∩ clip) through `sink`;
// nrm_store holds NC normals (the caller's, e.g. a per-thread slice of LDS).
template <int NC, class Sink>
CR_HD void clip_area_backward(const double *clip, int nc, const double *subj, int ns, double coef,
                              Sink &sink, d3 *nrm_store) {
    GradPipe<NC, Sink> P;
    P.nrm = nrm_store;
    P.ns = ns;
    P.coef = coef;
    P.sink = &sink;
    P.n = 0;
    d3 c[NC];
#pragma unroll
    for (int k = 0; k < NC; ++k) c[k] = load3(clip + 3 * (k < nc ? k : nc - 1));
#pragma unroll
    for (int k = 0; k < NC; ++k) {
        d3 n = cross(c[k], c[(k + 1) % NC] - c[k]);
        if (dot(n, n) < kDegenerateEdge2) n = mk3(0.0, 0.0, 0.0);
        P.anchor[k] = c[k];
        P.nrm[k] = n;
        P.started[k] = false;
    }
    for (int i = 0; i < ns; ++i) gpipe_push<0, NC, Sink>(P, load3(subj + 3 * i), lab_make(kLabS, 0, 0) | i);
    gpipe_close<0, NC, Sink>(P);
    P.area_close();
}

// Gradient w.r.t. the great-circle crossing x = y/|y| (y = +-(n1 x n2),
// n1 = p1 x q1, n2 = p2 x q2) pushed back to p1, q1, p2, q2.
CR_HD bool crossing_backward(const d3 &x, const d3 &g, const d3 &p1, const d3 &q1, const d3 &p2,
                             const d3 &q2, d3 &gp1, d3 &gq1, d3 &gp2, d3 &gq2) {
    d3 n1 = cross(p1, q1), n2 = cross(p2, q2);
    d3 y = cross(n1, n2);
    double L = sqrt(dot(y, y));
    if (!(L > 1e-300)) return false;
    double sigma = dot(y, x) >= 0.0 ? 1.0 : -1.0;
    d3 yb = (sigma / L) * tangential(g, x);
    d3 n1b = cross(n2, yb), n2b = cross(yb, n1);
    gp1 = cross(q1, n1b);
    gq1 = cross(n1b, p1);
    gp2 = cross(q2, n2b);
    gq2 = cross(n2b, p2);
    return true;
}

// ============================================================================
// Backward by boundary arcs (no clip pipeline): pair_arcs, then line_grad.
//
// To first order the area of P = subject ∩ clip changes only by the motion of
// the great circles that carry its boundary (the motion of a corner along them
// is of second order), so no crossing point is differentiated.  When vertex p of
// the line p -> q (inside on its left, n = p x q) moves by d along n / |n|, a
// point x of the line moves inward by d sin(xq) / sin(pq) (angles to q), so an arc
// a -> b on it loses the area d / |n| (cos(bq) - cos(aq)), that is
//   dA/dp = -n / |n|^2 M_p,   M_p = (|a - q|^2 - |b - q|^2) / 2,
//   dA/dq = -n / |n|^2 M_q,   M_q = (|b - p|^2 - |a - p|^2) / 2
// (tangential by themselves).  M_p and M_q are sums over the line's arcs: all
// arcs of one line (of one pair, or of all pairs that share the cell) are summed
// first, and line_grad runs once per line.  An edge's squared lengths are taken
// from differences, so nothing of the order of the sphere is cancelled (the same
// sums kept as vectors b - a, with q x ((b - a) x n) / n.n at the end, lost three
// digits on quarter-degree cells).
//
// The arcs: (i) the part of each subject edge inside the convex clip polygon --
// one interval, from the edge's side values against every clip line: the latest
// entry and the earliest exit (Liang-Barsky on the chord parameter; the
// crossings are the forward's crossing() of the edge's own end points); (ii) the
// parts of the clip edges inside the subject: they begin where a subject edge
// leaves the clip polygon through that edge's line or at a clip vertex inside
// the subject, and end where a subject edge enters or at the next clip vertex,
// so their sums are signed sums over those points.
//
// pair_arcs returns false when the pair is near a configuration where the area is
// not differentiable or where the decisions above could differ from the forward
// clip's by rounding: a subject vertex within ~1e-10 of a clip edge's length from
// two clip lines, two neighbouring ones that near one line, a crossing that near
// a clip corner, an edge that enters and leaves at one point; or when a clip edge
// meets the subject's boundary more than twice; or when the boundaries meet only
// where the subject goes out and in again at one point (a reflex vertex on a clip
// edge), or nowhere while a subject vertex is that near a clip line (cells that only
// touch: n.(v - o) - h may round to another sign than the forward's n.(v - c)).  The
// caller then uses clip_area_backward.  (Any other single subject vertex on a clip
// line is fine, on whichever side it comes out: its side counts as one for both of
// its edges, and the two crossings it may make cancel.)
// A clip edge without a length (a polar cell's, a padded polygon's) is no line;
// its neighbours' crossing is the corner, as in the forward clip.
// ============================================================================
constexpr double kEdgeTol = 1e-10;

// M_p and M_q of a line's arcs.
struct LineSum {
    double p, q;
};
// ... of the arc a -> b of the line p -> q (as products of differences: a short
// arc keeps its relative accuracy), and of the whole line.
CR_HD LineSum arc_sum(const d3 &p, const d3 &q, const d3 &a, const d3 &b) {
    const d3 h = 0.5 * (b - a);
    return LineSum{-dot(h, (a - q) + (b - q)), dot(h, (a - p) + (b - p))};
}
CR_HD double whole_sum(const d3 &p, const d3 &q) {
    const d3 e = q - p;
    return 0.5 * dot(e, e);
}

// The derivative of the area w.r.t. the vertices p, q of a boundary line (zero
// for a line of no length).
CR_HD void line_grad(const d3 &p, const d3 &q, const LineSum &S, d3 &gp, d3 &gq) {
    const d3 n = cross(p, q - p);
    const double nn = dot(n, n), f = nn > 0.0 ? -1.0 / nn : 0.0;
    gp = (f * S.p) * n;
    gq = (f * S.q) * n;
}

// The vertices of clip line k of NC (padding: a cell of nc < NC vertices repeats
// its last one, and line NC - 1 closes the ring).
template <int NC>
CR_HD int clip_first(int k, int nc) {
    return k < nc ? k : nc - 1;
}
template <int NC>
CR_HD int clip_second(int k, int nc) {
    return k + 1 == NC ? 0 : clip_first<NC>(k + 1, nc);
}

// One interval of the subject edge p -> q: where it enters through a line and
// where it leaves, the side values' sizes at p and q against that line.
struct EdgeCut {
    double p_in, q_in, p_out, q_out;  // the chord parameter is p / (p + q)
    int k_in, k_out;
};

// The arcs of a pair: `full`, a bit per subject edge wholly inside the clip
// polygon; arc(i, j, sums) for the i-th subject edge inside it in part, edge j
// (returns false if it has no room: the pair is declined); S[k] for clip line k.
// M: an unsigned integer of at least ns bits.
template <int NC, class M, class Arc>
CR_HD bool pair_arcs(const double *clip, int nc, const double *subj, int ns, M &full, LineSum (&S)[NC], Arc &&arc) {
    // side values n.(v - c) of clip line k as n.(v - o) - h, o the first clip vertex
    // (v - o is exact, both terms are of the cells' size): 3 FMAs a line
    const d3 o = load3(clip);
    d3 n[NC];
    double h[NC], tol[NC];
    {
        d3 c = o;
#pragma unroll
        for (int k = 0; k < NC; ++k) {
            S[k] = LineSum{0.0, 0.0};
            const d3 c1 = load3(clip + 3 * clip_second<NC>(k, nc));
            n[k] = cross(c, c1 - c);
            const double nn = dot(n[k], n[k]);
            tol[k] = kEdgeTol * nn;  // |side| below this: within ~1e-10 edge lengths of the line
            if (nn < kDegenerateEdge2) {
                n[k] = mk3(0.0, 0.0, 0.0);  // every point is inside
                tol[k] = -1.0;              // and none is near
            }
            h[k] = dot(n[k], c - o);
            c = c1;
        }
    }
    auto side = [&](int k, const d3 &v) { return fma(n[k].x, v.x, fma(n[k].y, v.y, fma(n[k].z, v.z, -h[k]))); };
    M out[NC], near = 0;  // subject vertices outside each line, near one
#pragma unroll
    for (int k = 0; k < NC; ++k) out[k] = 0;
    for (int j = 0; j < ns; ++j) {
        const d3 v = load3(subj + 3 * j) - o;
        bool close = false;
#pragma unroll
        for (int k = 0; k < NC; ++k) {
            const double a = side(k, v);
            out[k] |= (M)(a < 0.0) << j;
            close = close || fabs(a) <= tol[k];
        }
        near |= (M)close << j;
    }
    const M all = (M)(~(M)0) >> (8 * sizeof(M) - ns);
    auto next = [&](M m) { return (M)((m >> 1 | m << (ns - 1)) & all); };  // bit j: vertex j + 1
    M any_out = 0, apart = 0;
#pragma unroll
    for (int k = 0; k < NC; ++k) {
        any_out |= out[k];
        apart |= out[k] & next(out[k]);
    }
    full = ~any_out & next(~any_out & all) & all;
    M part = all & ~apart & ~full;
    for (M left = near; left; left &= left - 1) {
        const int j = __builtin_ctzll((unsigned long long)left), j1 = j + 1 == ns ? 0 : j + 1;
        const d3 v = load3(subj + 3 * j) - o, w = load3(subj + 3 * j1) - o;
        int lines = 0;
#pragma unroll
        for (int k = 0; k < NC; ++k) {
            if (!(fabs(side(k, v)) <= tol[k])) continue;
            ++lines;
            if (!(fabs(side(k, w)) <= tol[k])) continue;
            // an edge along the line: declined unless another line keeps it away
            bool away = false;
#pragma unroll
            for (int m = 0; m < NC; ++m) away = away || (m != k && (out[m] & next(out[m])) >> j & 1);
            if (!away) return false;
        }
        if (lines > 1) return false;
    }
    // the crossings on each clip edge (at most two): the first's place along the
    // edge, and whether a clip-edge arc begins (the subject leaves) at the first
    // and at the last
    double u_lo[NC];
    unsigned one = 0, two = 0, lo_leaves = 0, hi_leaves = 0, none = 0;
#pragma unroll
    for (int k = 0; k < NC; ++k) u_lo[k] = 0.0;
    bool any_arc = full != 0;
    int count = 0;
    for (M left = part; left; left &= left - 1) {
        const int j = __builtin_ctzll((unsigned long long)left);
        const d3 p = load3(subj + 3 * j), q = load3(subj + 3 * (j + 1 == ns ? 0 : j + 1));
        EdgeCut cut{0.0, 1.0, 1.0, 0.0, -1, -1};
#pragma unroll
        for (int k = 0; k < NC; ++k) {
            const double ap = side(k, p - o), aq = side(k, q - o);
            const bool pin = ap >= 0.0;
            if (pin == (aq >= 0.0)) continue;
            const double fp = fabs(ap), fq = fabs(aq);
            // fp / (fp + fq) against the latest entry, the earliest exit
            if (!pin && fp * cut.q_in > cut.p_in * fq) {
                cut.p_in = fp;
                cut.q_in = fq;
                cut.k_in = k;
            }
            if (pin && fp * cut.q_out < cut.p_out * fq) {
                cut.p_out = fp;
                cut.q_out = fq;
                cut.k_out = k;
            }
        }
        if (cut.k_in >= 0 && cut.k_out >= 0) {
            const double in = cut.p_in * (cut.p_out + cut.q_out), out_ = cut.p_out * (cut.p_in + cut.q_in);
            if (fabs(in - out_) <= kEdgeTol * ((cut.p_in + cut.q_in) * (cut.p_out + cut.q_out))) return false;
            if (in > out_) continue;  // outside
        }
        any_arc = true;
        d3 end[2] = {p, q};
#pragma unroll
        for (int way = 0; way < 2; ++way) {
            const int k = way == 0 ? cut.k_in : cut.k_out;
            if (k < 0) continue;
            // crossing() of the edge's end points
            d3 x = (way == 0 ? cut.q_in : cut.q_out) * p + (way == 0 ? cut.p_in : cut.p_out) * q;
            x = inv_norm(dot(x, x)) * x;
            end[way] = x;
            const d3 c0 = load3(clip + 3 * clip_first<NC>(k, nc)), c1 = load3(clip + 3 * clip_second<NC>(k, nc));
            const d3 e = c1 - c0, d = x - c0, f = x - c1;
            const double ee = dot(e, e), u = dot(d, e);
            if (u <= kEdgeTol * ee || u >= (1.0 - kEdgeTol) * ee) return false;  // at a clip corner
            // a clip-edge arc ends where the subject enters, begins where it leaves
            const double half = way == 0 ? 0.5 : -0.5, sp = -half * dot(f, f), sq = half * dot(d, d);
            const unsigned bit = 1u << k, leaves = way == 1 ? bit : 0u;
            double first = 0.0;
#pragma unroll
            for (int m = 0; m < NC; ++m)
                if (m == k) {
                    S[m].p += sp;
                    S[m].q += sq;
                    first = u_lo[m];
                    if (!(one & bit) || u < first) u_lo[m] = u;
                }
            if (two & bit) return false;
            if (!(one & bit)) {
                one |= bit;
                lo_leaves |= leaves;
                hi_leaves |= leaves;
            } else {
                two |= bit;
                if (fabs(u - first) <= kEdgeTol * ee) none |= bit;  // out and in again at one point
                if (u > first) hi_leaves = (hi_leaves & ~bit) | leaves;
                else lo_leaves = (lo_leaves & ~bit) | leaves;
            }
        }
        if (!arc(count++, j, arc_sum(p, q, end[0], end[1]))) return false;
    }
    if (two & ~(lo_leaves ^ hi_leaves)) return false;  // not an arc's two ends
    // clip vertices inside the subject: a vertex's state is that after the last
    // crossing before it along the clip boundary; with no crossing P is the
    // subject, or the clip polygon if no subject edge lies in it
    unsigned corners = 0;
    one &= ~none;
    if (none && !one) return false;  // one cell inside the other but for a touch: which, the arcs there do not tell
    if (one) {
#pragma unroll
        for (int k = 0; k < NC; ++k) {
            bool found = false;
#pragma unroll
            for (int s = 1; s <= NC; ++s) {
                const int m = (k - s + NC) % NC;
                if (!found && (one >> m & 1u)) {
                    corners |= (hi_leaves >> m & 1u) << k;
                    found = true;
                }
            }
        }
    } else if (!any_arc) {
        if (near) return false;
        corners = (1u << NC) - 1u;
    }
#pragma unroll
    for (int k = 0; k < NC; ++k) {
        const double whole = whole_sum(load3(clip + 3 * clip_first<NC>(k, nc)), load3(clip + 3 * clip_second<NC>(k, nc)));
        if (corners >> k & 1u) S[k].p += whole;
        if (corners >> ((k + 1) % NC) & 1u) S[k].q += whole;
    }
    return true;
}

// coef * d(signed ring area)/d(vertices) through emit(slot, grad): one call per
// vertex (a vertex's parts from the two fan triangles that share it are summed
// before the call).
template <class Emit>
CR_HD void ring_area_backward(const double *xyz, int n, double coef, Emit &&emit) {
    if (n < 3) return;
    d3 a = load3(xyz);
    d3 ga = mk3(0, 0, 0), pend = mk3(0, 0, 0);
    d3 b = load3(xyz + 3);
    for (int i = 1; i + 1 < n; ++i) {
        const d3 c = load3(xyz + 3 * (i + 1));
        double T = dot(a, cross(b, c));
        double D = 1.0 + dot(a, b) + dot(b, c) + dot(c, a);
        double f = coef * 2.0 / (T * T + D * D);
        ga = ga + f * (D * cross(b, c) - T * (b + c));
        emit(i, tangential(pend + f * (D * cross(c, a) - T * (a + c)), b));
        pend = f * (D * cross(a, b) - T * (a + b));
        b = c;
    }
    emit(n - 1, tangential(pend, b));
    emit(0, tangential(ga, a));
}

// Part of ring_area_backward's fan, unrolled (the slots are compile-time
// indices): the triangles (v0, v_i, v_{i+1}) for I0 <= i < I1.  ga (not made
// tangential) gets their derivative w.r.t. v0, g[j] (made
// tangential) w.r.t. v_{I0+j}, 0 <= j <= I1 - I0.  Two parts that meet at a
// vertex each hold a share of its derivative; the projection is linear, so
// the shares add.
template <int I0, int I1>
CR_HD void ring_area_backward_part(const double *xyz, double coef, d3 &ga, d3 (&g)[I1 - I0 + 1]) {
    const d3 a = load3(xyz);
    d3 pend = mk3(0, 0, 0);
    d3 b = load3(xyz + 3 * I0);
#pragma unroll
    for (int i = I0; i < I1; ++i) {
        const d3 c = load3(xyz + 3 * (i + 1));
        const double T = dot(a, cross(b, c));
        const double D = 1.0 + dot(a, b) + dot(b, c) + dot(c, a);
        const double f = coef * 2.0 / (T * T + D * D);
        ga = ga + f * (D * cross(b, c) - T * (b + c));
        g[i - I0] = g[i - I0] + tangential(pend + f * (D * cross(c, a) - T * (a + c)), b);
        pend = f * (D * cross(a, b) - T * (a + b));
        b = c;
    }
    g[I1 - I0] = g[I1 - I0] + tangential(pend, b);
}


}  // namespace cr
