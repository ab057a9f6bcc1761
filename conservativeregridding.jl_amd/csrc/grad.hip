// grad.hip -- reverse mode of regrid!(y, R, x) w.r.t. the field and the grid
// vertices (no reference counterpart: the reference has no AD; this is what a
// ChainRulesCore rrule around regrid! calls).
//
// With y = (A x) ./ a_to (normalize) and upstream gradient gy:
//   dL/dx          = A^T (gy ./ a_to)                      (the transpose apply)
//   dL/dA_ij       = sum_f gy_if x_jf / a_to,i             (per intersection pair)
//   dL/da_to,i     = -sum_f gy_if y_if / a_to,i            (per destination cell)
// and every A_ij, a_to,i is an area of unit-sphere polygons, so the vertex
// gradient is the sum over pairs of dL/dA_ij * d(area of cell_i ∩ cell_j)/dV
// plus the sum over cells of dL/da_to,i * d(area of cell_i)/dV, scattered into
// per-vertex gradients with FP64 atomics (order-nondeterministic in the last
// bits).  Gradients are tangential: the areas depend on the vertices through
// v/|v|.  Areas here are on the unit sphere; `area_scale` converts.
#include <algorithm>
#include <mutex>
#include <string>
#include <type_traits>

#include "regridder.hpp"
#include "sphgeom.hpp"

namespace cr {

// Gradients of one line's two vertices into caller vertices.
__device__ __forceinline__ void add_line(double *g, const int32_t *vi, int j, int j1, const d3 &p, const d3 &q,
                                         double w, const LineSum &S) {
    if (!g) return;
    d3 gp, gq;
    line_grad(p, q, LineSum{w * S.p, w * S.q}, gp, gq);
    atomicAdd(g + 3 * (int64_t)vi[j], gp.x);
    atomicAdd(g + 3 * (int64_t)vi[j] + 1, gp.y);
    atomicAdd(g + 3 * (int64_t)vi[j] + 2, gp.z);
    atomicAdd(g + 3 * (int64_t)vi[j1], gq.x);
    atomicAdd(g + 3 * (int64_t)vi[j1] + 1, gq.y);
    atomicAdd(g + 3 * (int64_t)vi[j1] + 2, gq.z);
}

// The destination cells' area term: cell i's area has dL/da_i = -kappa / a_i
// sum_f gy_if y_if (y null: no term).
struct AreaTerm {
    const double *y, *gy, *a_to;
    const int64_t *rowptr;
    int64_t yc, yf, gc, gf, nf;
    double kappa;
};
__device__ __forceinline__ double area_coef(const AreaTerm &A, int64_t i) {
    if (A.a_to[i] == 0.0) return 0.0;  // zero-area (ghost) cells have no area term
    double s = 0.0;
    for (int64_t f = 0; f < A.nf; ++f) s += A.gy[i * A.gc + f * A.gf] * A.y[i * A.yc + f * A.yf];
    return -A.kappa * s / A.a_to[i];
}
// ... of a cell by itself, as lines that are boundary all along.
__device__ __forceinline__ void add_area(const double *cell, int nv, const int32_t *vi, double c, double *g) {
    for (int v = 0; v < nv; ++v) {
        const int v1 = v + 1 == nv ? 0 : v + 1;
        const d3 p = load3(cell + 3 * v), q = load3(cell + 3 * v1);
        const double h = whole_sum(p, q);
        add_line(g, vi, v, v1, p, q, c, LineSum{h, h});
    }
}

// Per non-zero of CSR(A) (rows = dst, cols = src), one thread each: the
// coefficient dL/dA_u,ij (unit-sphere areas).
__global__ void k_pair_coef(const int32_t *__restrict__ rowid, const int32_t *__restrict__ col, int64_t nnz,
                            int transpose, int normalize, double kappa,
                            const double *__restrict__ a_to, int64_t nf,
                            const double *__restrict__ x, int64_t xc, int64_t xf,
                            const double *__restrict__ gy, int64_t gc, int64_t gf,
                            double *__restrict__ coef) {
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= nnz) return;
    const int64_t i = rowid[k], j = col[k];
    // forward: y lives on dst rows i, x on src cols j; transpose: the reverse
    const int64_t to = transpose ? j : i, from = transpose ? i : j;
    double s = 0.0;
    for (int64_t f = 0; f < nf; ++f) s += gy[to * gc + f * gf] * x[from * xc + f * xf];
    coef[k] = normalize ? kappa * s / a_to[to] : kappa * s;
}

// Scatter target of the clip backward: caller-vertex gradients of both grids.
// The destination cell's slots may go to a block-local accumulator instead
// (lacc_subj or lacc_clip, 3 doubles per slot), flushed once per block.  NC:
// the clip slots of the kernel (clip index NC wraps to 0).
template <int NC>
struct VertexSink {
    const double *subj, *clip;
    int ns, nc;
    const int32_t *subj_vi, *clip_vi;  // caller vertex of each slot of the two cells
    double *g_subj, *g_clip;           // caller-vertex gradients (may be null)
    double *lacc_subj, *lacc_clip;     // LDS accumulators of one side's slots, or null
    double *own_clip;                  // the pair's own 4 x 3 clip-slot sums in LDS, or null
    double *own_subj;                  // the pair's own 4 x 3 subject-slot sums in LDS, or null

    // slot e of the subject, 0 <= e <= ns (an edge's end vertex e + 1 wraps)
    __device__ int wrap(int e) const { return e >= ns ? e - ns : e; }
    __device__ d3 sv(int e) const { return load3(subj + 3 * wrap(e)); }
    __device__ d3 cv(int k) const {
        const int kk = k >= NC ? k - NC : k;
        return load3(clip + 3 * (kk < nc ? kk : nc - 1));
    }
    __device__ static void add(double *g, int32_t v, const d3 &d) {
        if (!g) return;
        atomicAdd(g + 3 * (int64_t)v, d.x);
        atomicAdd(g + 3 * (int64_t)v + 1, d.y);
        atomicAdd(g + 3 * (int64_t)v + 2, d.z);
    }
    __device__ static void add_local(double *l, int slot, const d3 &d) {
        atomicAdd(l + 3 * slot, d.x);
        atomicAdd(l + 3 * slot + 1, d.y);
        atomicAdd(l + 3 * slot + 2, d.z);
    }
    __device__ void add_subj(int e, const d3 &g) const {
        e = wrap(e);
        if (lacc_subj) {
            add_local(lacc_subj, e, tangential(g, sv(e)));
        } else if (own_subj) {  // this pair's own sums
            const d3 t = tangential(g, sv(e));
            own_subj[3 * e] += t.x;
            own_subj[3 * e + 1] += t.y;
            own_subj[3 * e + 2] += t.z;
        } else {
            add(g_subj, subj_vi[e], tangential(g, sv(e)));
        }
    }
    __device__ void add_clip(int k, const d3 &g) const {
        int kk = k >= NC ? k - NC : k;
        kk = kk < nc ? kk : nc - 1;
        const d3 t = tangential(g, cv(kk));
        if (lacc_clip) {
            add_local(lacc_clip, kk, t);
        } else if (own_clip) {  // this pair's own sums
            own_clip[3 * kk] += t.x;
            own_clip[3 * kk + 1] += t.y;
            own_clip[3 * kk + 2] += t.z;
        } else {
            add(g_clip, clip_vi[kk], t);
        }
    }
    __device__ void operator()(int32_t l, const d3 &x, const d3 &g) const {
        if (l < 0) return;
        int32_t t = lab_type(l), a = lab_hi(l), b = lab_lo(l);
        if (t == kLabS) {
            add_subj(l & kLabIndexMask, g);  // the subject index is the low 30 bits
        } else if (t == kLabC) {
            add_clip(b, g);
        } else {
            d3 p1, q1, p2 = cv(b), q2 = cv(b + 1), gp1, gq1, gp2, gq2;
            if (t == kLabXF) { p1 = sv(a); q1 = sv(a + 1); }
            else { p1 = cv(a); q1 = cv(a + 1); }
            if (!crossing_backward(x, g, p1, q1, p2, q2, gp1, gq1, gp2, gq2)) return;
            if (t == kLabXF) { add_subj(a, gp1); add_subj(a + 1, gq1); }
            else { add_clip(a, gp1); add_clip(a + 1, gq1); }
            add_clip(b, gp2);
            add_clip(b + 1, gq2);
        }
    }
};

// One wave per 64 consecutive non-zeros.  CSR rows are destination cells, so a
// wave's pairs share few destination cells (about 12 on the benchmark): their
// slots' gradients are summed in LDS (rows r0 .. r0 + kGradRows - 1 of the
// wave) and reach memory once per wave.  A source cell of at most 4 vertices
// (clipping or clipped) has its slots summed per pair and written once per
// pair; other contributions use global FP64 atomics directly.
constexpr int kGradRows = 16;

// The sink of one pair: its two rings, its slots' accumulators (the wave's
// destination rows in LDS when `lacc` is given and the row is one of them,
// the pair's own source-cell sums in `own`) and the caller-vertex gradients;
// NC: the clip slots of the kernel.
template <int NC>
__device__ __forceinline__ VertexSink<NC> pair_sink(int64_t d, int64_t s, int64_t r0, double *lacc, double *own,
                                                const double *__restrict__ dst_cells, int dst_nv,
                                                const int32_t *__restrict__ dst_vi,
                                                const double *__restrict__ src_cells, int src_nv,
                                                const int32_t *__restrict__ src_vi, int clip_is_dst,
                                                double *__restrict__ g_dst, double *__restrict__ g_src) {
    const double *dp = dst_cells + 3 * (int64_t)dst_nv * d;
    const double *sp = src_cells + 3 * (int64_t)src_nv * s;
    double *mine = (lacc && g_dst && d - r0 < kGradRows) ? lacc + (d - r0) * dst_nv * 3 : nullptr;
    // a source cell of at most 4 vertices sums its slots per pair
    double *own4 = (g_src && src_nv <= 4) ? own : nullptr;
    return clip_is_dst
                       ? VertexSink<NC>{sp, dp, src_nv, dst_nv, src_vi + (int64_t)src_nv * s, dst_vi + (int64_t)dst_nv * d,
                                    g_src, g_dst, nullptr, mine, nullptr, own4}
                       : VertexSink<NC>{dp, sp, dst_nv, src_nv, dst_vi + (int64_t)dst_nv * d, src_vi + (int64_t)src_nv * s,
                                    g_dst, g_src, mine, nullptr, own4, nullptr};
}

// The per-pair sums of the source cell's 4 slots, one atomic per component.
template <int NC>
__device__ __forceinline__ void flush_own(const VertexSink<NC> &sink, int src_nv, double *own, double *g_src) {
    if (!sink.own_clip && !sink.own_subj) return;
    const int32_t *vi = sink.own_clip ? sink.clip_vi : sink.subj_vi;
    for (int kk = 0; kk < src_nv && kk < 4; ++kk) {
        const d3 v = mk3(own[3 * kk], own[3 * kk + 1], own[3 * kk + 2]);
        if (v.x != 0.0 || v.y != 0.0 || v.z != 0.0) VertexSink<NC>::add(g_src, vi[kk], v);
    }
}

// The wave's destination rows from LDS to memory.
__device__ __forceinline__ void flush_rows(const double *lacc, int64_t r0, int64_t nrows, int dst_nv,
                                           const int32_t *__restrict__ dst_vi, double *g_dst) {
    for (int i = threadIdx.x; i < nrows * dst_nv * 3; i += 64) {
        const double v = lacc[i];
        if (v == 0.0) continue;
        const int r = i / (dst_nv * 3), slot = (i / 3) % dst_nv, comp = i % 3;
        atomicAdd(g_dst + 3 * (int64_t)dst_vi[(r0 + r) * dst_nv + slot] + comp, v);
    }
}

// Destination rows of a wave summed in LDS: at most 256 lines of three doubles.
inline int arc_rows(int dst_nv) { return std::max(1, std::min(64, 256 / dst_nv)); }

// Subject edges a pair may have inside the clip polygon in part (more: declined),
// kept in LDS; a quad's are at most 4, a 16-gon's rarely more than 8.
template <class M>
constexpr int kArcs = sizeof(M) == 1 ? 6 : 8;
template <class M>
constexpr int kOwn = 2 * kArcs<M> + 1;  // a lane's doubles in LDS (odd: lanes on different banks)

// The vertex pass by boundary arcs (pair_arcs), one wave per 64 consecutive
// non-zeros, a lane each.  Nothing but two numbers per line is summed per pair: a
// destination cell's lines are summed in LDS over the wave's pairs (an edge
// wholly inside the other cell adds its coefficient alone, and so does the cell's
// own area term, in the wave that holds the row's first non-zero) and turned into
// vertex gradients once per wave and row; a source cell's lines once per pair, in
// registers.  A pair near a degenerate configuration is appended to `list` (wave
// by wave, in order) for k_clip_grad_list.  M: a bit per subject vertex.
//
// Bound: FP64 VALU of the arcs (side values of every subject vertex against the
// clip lines, then the few edges that cross) and the gradients' own traffic.
// Differentiating every crossing and fan triangle instead, with the crossings
// queued in LDS, took 15 600 VALU instructions a wave against 5 000 here: the whole
// vertex pass on quarter degree -> HEALPix 256 (16-gons, nnz 4.35 M), with the
// declined pairs and the area term, 4.39 -> 1.68 ms; C96 -> 1 degree 276 -> 100 us.
// The lane-to-double mapping of the atomics matters as much: with a lane per pair
// and vertex this kernel ran 2.55 ms.  Three waves a SIMD (168 registers, a few
// spilled) against two: 1.88 and 2.11 ms for the whole reverse mode.
template <int NC, class M>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(NC == 4 ? 3 : 2))) k_clip_grad_arcs(
    const int32_t *__restrict__ rowid, const int32_t *__restrict__ col, const double *__restrict__ coef,
    int64_t nnz, const double *__restrict__ dst_cells, int dst_nv, const int32_t *__restrict__ dst_vi,
    const double *__restrict__ src_cells, int src_nv, const int32_t *__restrict__ src_vi, int clip_is_dst, int window,
    AreaTerm area, double *__restrict__ g_dst, double *__restrict__ g_src, int32_t *__restrict__ list,
    uint32_t *__restrict__ count) {
    // a lane's arcs of subject edges (M_p, M_q), then its source vertices' gradients
    __shared__ double own[64 * kOwn<M>];
    __shared__ double acoef[64];  // the rows' area terms
    __shared__ uint8_t lead[64];  // a lane of each source cell
    extern __shared__ double rows[];  // window x dst_nv x (M_p, M_q, coefficient of whole edges)
    const int lane = threadIdx.x;
    const int nrow = window * dst_nv * 3;
    const bool use_own = src_nv <= 4;
    const int64_t k0 = (int64_t)blockIdx.x * 64, k = k0 + lane;
    const int64_t r0 = rowid[k0];
    for (int i = lane; i < nrow; i += 64) rows[i] = 0.0;
    __syncthreads();
    const double w = k < nnz ? coef[k] : 0.0;
    double *mine = own + kOwn<M> * lane;
    bool planned = true, zero = true;  // zero: no source vertex gradients in `mine`
    // the wave's rows; their area terms, a lane per row
    const int64_t last = rowid[min(nnz, k0 + 64) - 1] - r0 + 1;
    acoef[lane] = 0.0;
    if (area.y && g_dst) {
        for (int64_t r = lane; r < last; r += 64) {
            const double c = area.rowptr[r0 + r] >= k0 ? area_coef(area, r0 + r) : 0.0;
            if (r < window)
                acoef[r] = c;
            else if (c != 0.0)
                add_area(dst_cells + 3 * (int64_t)dst_nv * (r0 + r), dst_nv, dst_vi + (r0 + r) * dst_nv, c, g_dst);
        }
    }
    if (w != 0.0) {
        const int64_t d = rowid[k], s = col[k];
        const double *dp = dst_cells + 3 * (int64_t)dst_nv * d, *sp = src_cells + 3 * (int64_t)src_nv * s;
        const double *clip = clip_is_dst ? dp : sp, *subj = clip_is_dst ? sp : dp;
        const int nc = clip_is_dst ? dst_nv : src_nv, ns = clip_is_dst ? src_nv : dst_nv;
        const int32_t *dvi = dst_vi + (int64_t)dst_nv * d, *svi = src_vi + (int64_t)src_nv * s;
        double *row = d - r0 < window ? rows + (d - r0) * dst_nv * 3 : nullptr;
        M full;
        LineSum S[NC];
        int arcs = 0;
        uint64_t edge = 0;  // the arcs' subject edges, a byte each
        planned = pair_arcs<NC, M>(clip, nc, subj, ns, full, S, [&](int i, int j, const LineSum &a) {
            if (i >= kArcs<M>) return false;
            mine[2 * i] = a.p;
            mine[2 * i + 1] = a.q;
            edge |= (uint64_t)j << (8 * i);
            arcs = i + 1;
            return true;
        });
        if (planned) {
            auto after = [&](int j) { return j + 1 == ns ? 0 : j + 1; };
            auto clear = [&] {
                zero = false;
#pragma unroll
                for (int i = 0; i < 12; ++i) mine[i] = 0.0;
            };
            auto add_own = [&](int v, int v1, const d3 &p, const d3 &q, const LineSum &L) {
                d3 gp, gq;
                line_grad(p, q, L, gp, gq);
                mine[3 * v] += gp.x;
                mine[3 * v + 1] += gp.y;
                mine[3 * v + 2] += gp.z;
                mine[3 * v1] += gq.x;
                mine[3 * v1 + 1] += gq.y;
                mine[3 * v1 + 2] += gq.z;
            };
            if (!clip_is_dst && row) {
                for (M m = full; m; m &= m - 1) atomicAdd(row + 3 * __builtin_ctzll((unsigned long long)m) + 2, w);
                for (int i = 0; i < arcs; ++i, edge >>= 8) {
                    double *line = row + 3 * (int)(edge & 255);
                    atomicAdd(line, w * mine[2 * i]);
                    atomicAdd(line + 1, w * mine[2 * i + 1]);
                }
            } else if (clip_is_dst && use_own) {
                LineSum L[4];
#pragma unroll
                for (int m = 0; m < 4; ++m) {
                    L[m] = LineSum{0.0, 0.0};
                    if (m < ns && (full >> m & 1))
                        L[m].p = L[m].q = w * whole_sum(load3(subj + 3 * m), load3(subj + 3 * after(m)));
                }
                for (int i = 0; i < arcs; ++i, edge >>= 8) {
#pragma unroll
                    for (int m = 0; m < 4; ++m)
                        if (m == (int)(edge & 255)) L[m] = LineSum{w * mine[2 * i], w * mine[2 * i + 1]};
                }
                clear();
#pragma unroll
                for (int m = 0; m < 4; ++m) {
                    if (m >= ns) continue;
                    add_own(m, after(m), load3(subj + 3 * m), load3(subj + 3 * after(m)), L[m]);
                }
            } else {  // a subject of more vertices, or a row past the window
                double *g = clip_is_dst ? g_src : g_dst;
                const int32_t *vi = clip_is_dst ? svi : dvi;
                for (M m = full; m; m &= m - 1) {
                    const int j = __builtin_ctzll((unsigned long long)m);
                    const d3 p = load3(subj + 3 * j), q = load3(subj + 3 * after(j));
                    const double h = whole_sum(p, q);
                    add_line(g, vi, j, after(j), p, q, w, LineSum{h, h});
                }
                for (int i = 0; i < arcs; ++i, edge >>= 8) {
                    const int j = (int)(edge & 255);
                    add_line(g, vi, j, after(j), load3(subj + 3 * j), load3(subj + 3 * after(j)), w,
                             LineSum{mine[2 * i], mine[2 * i + 1]});
                }
            }
            if (NC == 4 && !clip_is_dst) clear();
            // the clip cell's lines (one without a length has no sums)
#pragma unroll
            for (int m = 0; m < NC; ++m) {
                const int i0 = clip_first<NC>(m, nc), i1 = clip_second<NC>(m, nc);
                if (i0 == i1) continue;
                if (clip_is_dst && row) {
                    atomicAdd(row + 3 * i0, w * S[m].p);
                    atomicAdd(row + 3 * i0 + 1, w * S[m].q);
                } else if (NC == 4 && !clip_is_dst) {  // nc <= 4: its vertices are the pair's own
                    add_own(i0, i1, load3(clip + 3 * i0), load3(clip + 3 * i1), LineSum{w * S[m].p, w * S[m].q});
                } else {
                    add_line(clip_is_dst ? g_dst : g_src, clip_is_dst ? dvi : svi, i0, i1, load3(clip + 3 * i0),
                             load3(clip + 3 * i1), w, S[m]);
                }
            }
        }
    }
    // declined pairs to the list: one atomic per wave, lanes in order
    const uint64_t m = __ballot(!planned);
    if (m) {
        uint32_t base = 0;
        if (lane == 0) base = atomicAdd(count, (uint32_t)__popcll(m));
        base = __shfl(base, 0);
        if (!planned) list[base + __popcll(m & ((1ull << lane) - 1ull))] = (int32_t)k;
    }
    // the pairs' source vertices: neighbouring lanes take neighbouring doubles (a
    // quad's 12 are two runs of 48 bytes: an atomic of 64 lanes then touches about
    // 11 lines; a lane per pair touched 64).  Subjects of few vertices, whose arcs
    // take little time, have the pairs of one source cell summed first (a wave
    // holds about half as many cells as pairs): C96 -> 1 degree 195 -> 177 us; for
    // 16-gons the search costs what it saves (1.88 -> 1.93 ms).
    if (use_own && g_src) {
        const int32_t s = k < nnz && !zero ? col[k] : -1;
        if constexpr (sizeof(M) == 1) {
            int leader = lane, place = 0, cells = 0;
            for (uint64_t todo = __ballot(s >= 0); todo; ++cells) {
                const int l = __builtin_ctzll(todo);
                const int32_t sl = __builtin_amdgcn_readlane(s, l);
                todo &= ~__ballot(s == sl);
                if (s == sl) leader = l;
                if (lane == l) place = cells;
            }
            __syncthreads();
            if (leader != lane) {
                double *to = own + kOwn<M> * leader;
#pragma unroll
                for (int i = 0; i < 12; ++i) atomicAdd(to + i, mine[i]);
            } else if (s >= 0) {
                lead[place] = (uint8_t)lane;
            }
            __syncthreads();
            for (int i = lane; i < (cells * 12 + 63) / 64 * 64; i += 64) {
                const int c = min(i / 12, cells - 1), e = i % 12, l = lead[c];
                const int64_t sp = __shfl(s, l, 64);
                const double v = i < cells * 12 ? own[kOwn<M> * l + e] : 0.0;
                if (v != 0.0) atomicAdd(g_src + 3 * (int64_t)src_vi[sp * src_nv + e / 3] + e % 3, v);
            }
        } else {
            if (s < 0) {
#pragma unroll
                for (int i = 0; i < 12; ++i) mine[i] = 0.0;
            }
            __syncthreads();
            for (int i = lane; i < 64 * 12; i += 64) {
                const int l = i / 12, e = i % 12;
                const int64_t sp = __shfl(s, l, 64);
                const double v = own[kOwn<M> * l + e];
                if (v != 0.0) atomicAdd(g_src + 3 * (int64_t)src_vi[sp * src_nv + e / 3] + e % 3, v);
            }
        }
    }
    if (!g_dst) return;
    // the destination rows: a lane per vertex, from the lines before and after it;
    // then a lane per double
    const int n = (int)min((int64_t)window, last) * dst_nv;
    __syncthreads();
    d3 g[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const int i = lane + 64 * t;
        g[t] = mk3(0.0, 0.0, 0.0);
        if (i >= n) continue;
        const int r = i / dst_nv, v = i - r * dst_nv, u = v == 0 ? dst_nv - 1 : v - 1, v1 = v + 1 == dst_nv ? 0 : v + 1;
        const double *cell = dst_cells + 3 * (int64_t)dst_nv * (r0 + r), *line = rows + 3 * dst_nv * r;
        const d3 pu = load3(cell + 3 * u), pv = load3(cell + 3 * v), pn = load3(cell + 3 * v1);
        const double cu = line[3 * u + 2] + acoef[r], cv = line[3 * v + 2] + acoef[r];
        d3 gp, gq, unused;
        line_grad(pu, pv, LineSum{0.0, line[3 * u + 1] + cu * whole_sum(pu, pv)}, unused, gq);
        line_grad(pv, pn, LineSum{line[3 * v] + cv * whole_sum(pv, pn), 0.0}, gp, unused);
        g[t] = gq + gp;
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const int i = lane + 64 * t;
        if (i >= n) continue;
        rows[3 * i] = g[t].x;
        rows[3 * i + 1] = g[t].y;
        rows[3 * i + 2] = g[t].z;
    }
    __syncthreads();
    // atomics for cells that own their vertices, too: the buffer may be g_src as
    // well, or another call's on another stream (plain adds to a wave's inner rows
    // took 1.81 ms instead of 1.87 for the whole reverse mode of quarter degree ->
    // HEALPix 256, and lost updates there)
    for (int i = lane; i < 3 * n; i += 64) {
        const double v = rows[i];
        if (v != 0.0) atomicAdd(g_dst + 3 * (int64_t)dst_vi[r0 * dst_nv + i / 3] + i % 3, v);
    }
}

// The vertex pass through the clip pipeline (clip_area_backward) for the
// pairs the boundary arcs decline: list[0 .. *count), 64 per wave,
// the waves striding over the list.  The list holds each wave's declined
// pairs in order, so a window of 64 entries mostly shares rows: rows r0 ..
// r0 + kGradRows - 1 of its first entry are summed in LDS, the rest go to
// memory directly.  Two waves per SIMD (256 registers): the second wave hides
// the atomics' and the FP64 chain's latency.  The clip pipeline's edge
// normals live in LDS (6 KB per workgroup), which cuts the register spills
// from 73 to about 30; moving its first vertices and clip vertices there too
// removes the rest but lowers the occupancy LDS allows and ran slower (as the
// whole vertex pass on C3: 8.4 ms with the normals in registers, 7.1 ms as
// here, 9.1 ms with none spilled), and so did one wave per SIMD with no
// spills (8.3 ms against 5.4).
template <int NC>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) k_clip_grad_list(
    const int32_t *__restrict__ rowid, const int32_t *__restrict__ col, const double *__restrict__ coef,
    const double *__restrict__ dst_cells, int dst_nv, const int32_t *__restrict__ dst_vi,
    const double *__restrict__ src_cells, int src_nv, const int32_t *__restrict__ src_vi, int clip_is_dst,
    double *__restrict__ g_dst, double *__restrict__ g_src, const int32_t *__restrict__ list,
    const uint32_t *__restrict__ count, int64_t n_rows) {
    extern __shared__ double lacc[];  // kGradRows * dst_nv * 3
    __shared__ double own[64 * 12];
    __shared__ d3 nrm_lds[64 * NC];  // each thread's NC clip-edge normals
    double *my_own = own + 12 * threadIdx.x;
    const int64_t total = *count;
    const int nacc = kGradRows * dst_nv * 3;
    // a short list is spread over all waves: fewer pairs a wave, fewer paths in it
    const int64_t per = min((int64_t)64, (total + gridDim.x - 1) / gridDim.x);
    for (int64_t base = (int64_t)blockIdx.x * per; base < total; base += (int64_t)gridDim.x * per) {
        const int64_t r0 = rowid[list[base]];
        for (int i = threadIdx.x; i < nacc; i += 64) lacc[i] = 0.0;
#pragma unroll
        for (int i = 0; i < 12; ++i) my_own[i] = 0.0;
        __syncthreads();
        const int64_t i = base + threadIdx.x;
        if (threadIdx.x < per && i < total) {
            const int64_t k = list[i];
            const double c = coef[k];
            const int64_t d = rowid[k];
            if (c != 0.0) {
                VertexSink<NC> sink = pair_sink<NC>(d, col[k], r0, d >= r0 ? lacc : nullptr, my_own, dst_cells, dst_nv,
                                            dst_vi, src_cells, src_nv, src_vi, clip_is_dst, g_dst, g_src);
                clip_area_backward<NC, VertexSink<NC>>(sink.clip, sink.nc, sink.subj, sink.ns, c, sink,
                                                   nrm_lds + NC * threadIdx.x);
                flush_own(sink, src_nv, my_own, g_src);
            }
        }
        __syncthreads();
        if (g_dst) flush_rows(lacc, r0, min((int64_t)kGradRows, n_rows - r0), dst_nv, dst_vi, g_dst);
        __syncthreads();
    }
}

// Before the vertex pass: its list's count, and the area term of the destination rows
// that no wave of the pass has -- rows without a non-zero that do not lie between two
// non-zeros of one wave.  (The term is 0 there, but for an upstream gradient that is
// not finite, or a y that is not the forward's.)
__global__ void k_vertex_start(uint32_t *__restrict__ count, AreaTerm area, int64_t n_rows, int64_t nnz,
                               const double *__restrict__ dst_cells, int dst_nv, const int32_t *__restrict__ dst_vi,
                               double *__restrict__ g_dst) {
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r == 0) *count = 0u;
    if (r >= n_rows || !area.y || !g_dst) return;
    const int64_t k = area.rowptr[r];
    if (k != area.rowptr[r + 1] || (k % 64 != 0 && k != nnz)) return;
    const double c = area_coef(area, r);
    if (c != 0.0) add_area(dst_cells + 3 * (int64_t)dst_nv * r, dst_nv, dst_vi + r * dst_nv, c, g_dst);
}

// Workgroups of the list pass (the waves stride over the declined pairs).
constexpr unsigned kListBlocks = 2048;

// d(area of each destination cell)/dV times dL/da_u.  (Like all of the reverse
// mode it adds to g by atomics, whoever owns a vertex: other calls may be adding
// to the same buffer.)
__global__ void k_area_grad(const double *__restrict__ cells, int nv, const int32_t *__restrict__ vi,
                            int64_t ncells, double kappa, const double *__restrict__ a_to, int64_t nf,
                            const double *__restrict__ y, int64_t yc, int64_t yf,
                            const double *__restrict__ gy, int64_t gc, int64_t gf,
                            double *__restrict__ g) {
    int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= ncells || a_to[t] == 0.0) return;  // zero-area (ghost) cells have no area term
    double s = 0.0;
    for (int64_t f = 0; f < nf; ++f) s += gy[t * gc + f * gf] * y[t * yc + f * yf];
    double c = -kappa * s / a_to[t];
    if (c == 0.0) return;
    const int32_t *v = vi + (int64_t)nv * t;
    ring_area_backward(cells + 3 * (int64_t)nv * t, nv, c, [&](int slot, const d3 &d) {
        double *gv = g + 3 * (int64_t)v[slot];
        atomicAdd(gv, d.x);
        atomicAdd(gv + 1, d.y);
        atomicAdd(gv + 2, d.z);
    });
}

// The same for grids whose cells own their vertices, with at most
// kStagedNv vertices per cell: a workgroup's 64 cells are one contiguous run of
// vertex data and of g (each cell's caller vertices are its own slots, in some
// order), so both are staged through LDS with coalesced loads and stores
// instead of a thread per cell reading and writing 24*nv bytes apart from its
// neighbours.
constexpr int kStagedNv = 16;
__global__ void __launch_bounds__(64) k_area_grad_private(const double *__restrict__ cells, int nv,
                                                          const int32_t *__restrict__ vi, int64_t ncells,
                                                          double kappa, const double *__restrict__ a_to, int64_t nf,
                                                          const double *__restrict__ y, int64_t yc, int64_t yf,
                                                          const double *__restrict__ gy, int64_t gc, int64_t gf,
                                                          double *__restrict__ g) {
    extern __shared__ double stage[];  // 2 * 64 * nv * 3 doubles: vertices, then g
    double *vin = stage, *gout = stage + 64 * 3 * nv;
    const int64_t c0 = (int64_t)blockIdx.x * 64;
    const int ncell = (int)min((int64_t)64, ncells - c0);
    const int n = ncell * nv * 3;
    const double *src = cells + 3 * (int64_t)nv * c0;
    double *gb = g + 3 * (int64_t)nv * c0;
    for (int i = threadIdx.x; i < n; i += 64) {
        vin[i] = src[i];
        gout[i] = 0.0;
    }
    __syncthreads();
    const int t = threadIdx.x;
    const int64_t c = c0 + t;
    if (t < ncell && a_to[c] != 0.0) {  // zero-area (ghost) cells have no area term
        double sum = 0.0;
        for (int64_t f = 0; f < nf; ++f) sum += gy[c * gc + f * gf] * y[c * yc + f * yf];
        const double coef = -kappa * sum / a_to[c];
        if (coef != 0.0) {
            const int32_t *v = vi + (int64_t)nv * c;
            const int64_t base = (int64_t)nv * c0;
            ring_area_backward(vin + 3 * nv * t, nv, coef, [&](int slot, const d3 &d) {
                double *o = gout + 3 * (v[slot] - base);
                o[0] += d.x;
                o[1] += d.y;
                o[2] += d.z;
            });
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += 64)
        if (gout[i] != 0.0) atomicAdd(gb + i, gout[i]);
}

// The same for tables of NV-vertex cells whose slot -> vertex map is the
// identity (cells own their vertices and none was re-oriented): two lanes per
// cell, each taking half of its fan (triangles (v0, v_i, v_{i+1}) below and
// from the middle vertex v_H on) with its slots' gradients in registers (the
// fan's slots are compile-time indices); the two shares of v0 and v_H meet by
// a lane shuffle.  One LDS buffer stages the block's 64 cells' vertices in
// and their gradients out, both with coalesced accesses (two lanes a cell:
// twice the waves one lane a cell had for the same LDS).
template <int NV>
__global__ void __launch_bounds__(128) k_area_grad_table(const double *__restrict__ cells, int64_t ncells,
                                                         double kappa, const double *__restrict__ a_to, int64_t nf,
                                                         const double *__restrict__ y, int64_t yc, int64_t yf,
                                                         const double *__restrict__ gy, int64_t gc, int64_t gf,
                                                         double *__restrict__ g) {
    constexpr int H = NV / 2;
    static_assert(NV >= 4 && NV % 2 == 0, "even rings of at least 4 vertices");
    __shared__ double stage[64 * NV * 3];
    const int64_t c0 = (int64_t)blockIdx.x * 64;
    const int ncell = (int)min((int64_t)64, ncells - c0);
    const int n = ncell * NV * 3;
    const double *src = cells + 3 * (int64_t)NV * c0;
    double *gb = g + 3 * (int64_t)NV * c0;
    for (int i = threadIdx.x; i < n; i += 128) stage[i] = src[i];
    __syncthreads();
    const int t = threadIdx.x >> 1;  // the cell; lanes 2t and 2t + 1 share it (one wave)
    const bool hi = (threadIdx.x & 1) != 0;
    const int64_t c = c0 + t;
    d3 ga = mk3(0.0, 0.0, 0.0);
    d3 gr[H];  // the lane's slots: 1 .. H (low lane) or H .. NV-1 (high lane)
#pragma unroll
    for (int k = 0; k < H; ++k) gr[k] = mk3(0.0, 0.0, 0.0);
    if (t < ncell && a_to[c] != 0.0) {  // zero-area (ghost) cells have no area term
        double sum = 0.0;
        for (int64_t f = 0; f < nf; ++f) sum += gy[c * gc + f * gf] * y[c * yc + f * yf];
        const double coef = -kappa * sum / a_to[c];
        if (coef != 0.0) {
            // the low lane: triangles 1 .. H-1 (slots 1 .. H), the high lane:
            // triangles H .. NV-2 (slots H .. NV-1)
            if (!hi) ring_area_backward_part<1, H>(stage + 3 * NV * t, coef, ga, gr);
            else ring_area_backward_part<H, NV - 1>(stage + 3 * NV * t, coef, ga, gr);
        }
    }
    // the shared slots: v0 from both lanes, v_H (the low lane's last, the high lane's first)
    const d3 ga_o = mk3(__shfl_xor(ga.x, 1), __shfl_xor(ga.y, 1), __shfl_xor(ga.z, 1));
    const d3 mid = hi ? gr[0] : gr[H - 1];
    const d3 mid_o = mk3(__shfl_xor(mid.x, 1), __shfl_xor(mid.y, 1), __shfl_xor(mid.z, 1));
    __syncthreads();
    if (t < ncell) {
        double *o = stage + 3 * NV * t;
        auto put = [&](int k, const d3 &v) {
            o[3 * k] = v.x;
            o[3 * k + 1] = v.y;
            o[3 * k + 2] = v.z;
        };
        if (!hi) {
            const double *a = o;  // v0, still staged: the low lane writes it only now
            put(0, tangential(ga + ga_o, load3(a)));
#pragma unroll
            for (int k = 1; k < H; ++k) put(k, gr[k - 1]);
            put(H, gr[H - 1] + mid_o);
        } else {
#pragma unroll
            for (int k = H + 1; k < NV; ++k) put(k, gr[k - H]);
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += 128)
        if (stage[i] != 0.0) atomicAdd(gb + i, stage[i]);
}

__global__ void k_div_rows(const double *__restrict__ gy, int64_t gc, int64_t gf, int64_t n, int64_t nf,
                           const double *__restrict__ a, double *__restrict__ w) {
    int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n * nf) return;
    int64_t f = t / n, i = t - f * n;
    w[t] = a ? gy[i * gc + f * gf] / a[i] : gy[i * gc + f * gf];
}

void apply(const cr_regridder *R, bool transpose, int dtype, int64_t nf, const void *src, int64_t sc,
           int64_t sf, void *dst, int64_t dc, int64_t df, bool normalize, hipStream_t s,
           int force_variant);
bool apply_ready(const cr_regridder *R, bool transpose, int dtype, int64_t nf, int64_t sf, int64_t df);

// Scratch of the reverse mode: w (n_to x nfields doubles, the field adjoint's
// input), coef (a double per non-zero), rowid (an int32 per non-zero), list
// (the non-zeros the boundary arcs decline, at most one int32 per
// non-zero) and its count.
struct BackwardScratch {
    double *w = nullptr, *coef = nullptr;
    int32_t *rowid = nullptr, *list = nullptr;
    uint32_t *count = nullptr;
};

// The reverse mode on the given stream.  ws == nullptr: the scratch is
// allocated for the call (stream-ordered) and the stream synchronised at the
// end; otherwise the caller's scratch is used, nothing is allocated, every
// per-direction plan must exist already, and the call returns without
// synchronising.
static void backward(const cr_regridder *R, const cr_grid *dst, const cr_grid *src, int32_t transpose,
                     int32_t normalize, int64_t nfields, const double *x, int64_t xc, int64_t xf, const double *y,
                     int64_t yc, int64_t yf, const double *gy, int64_t gc, int64_t gf, double *gx, int64_t gxc,
                     int64_t gxf, double *g_dst_verts, double *g_src_verts, hipStream_t s,
                     const BackwardScratch *ws) {
    CR_REQUIRE(R && nfields > 0 && x && gy, CR_INVALID_ARGUMENT, "cr_regrid_backward: bad arguments");
    CR_REQUIRE(xc > 0 && gc > 0 && (nfields == 1 || (xf > 0 && gf > 0)), CR_INVALID_ARGUMENT,
               "cr_regrid_backward: bad strides");
    const bool want_verts = g_dst_verts || g_src_verts;
    const Csr &F = R->fwd;
    const int64_t n_to = transpose ? F.ncols : F.nrows;
    const double *a_to = transpose ? R->a_src.p : R->a_dst.p;
    const int B = 256;
    // field gradient: gx = A_dir^T (gy ./ a_to)
    if (gx) {
        CR_REQUIRE(gxc > 0 && (nfields == 1 || gxf > 0), CR_INVALID_ARGUMENT, "bad gx strides");
        DevBuf<double> wb;
        double *w = ws ? ws->w : nullptr;
        if (!ws) {
            wb.alloc_async((size_t)n_to * nfields, s);
            w = wb.p;
        } else {
            CR_REQUIRE(apply_ready(R, !transpose, CR_F64, nfields, n_to, gxf), CR_UNSUPPORTED,
                       "the field adjoint's plan is not made: call cr_regrid_prepare(R, !transpose, CR_F64, "
                       "nfields, n_to, field stride of gx) first");
        }
        hipLaunchKernelGGL(k_div_rows, dim3(grid_for(n_to * nfields, B)), dim3(B), 0, s, gy, gc, gf, n_to,
                           nfields, normalize ? a_to : nullptr, w);
        CR_HIP(hipGetLastError());
        apply(R, !transpose, CR_F64, nfields, w, 1, n_to, gx, gxc, gxf, false, s, -1);
    }
    if (!want_verts) {
        if (!ws) synchronise(s);
        return;
    }
    CR_REQUIRE(R->area_scale > 0.0, CR_UNSUPPORTED,
               "vertex gradients need a regridder built from grids (cr_regridder_build)");
    CR_REQUIRE(dst && src && dst->ncells == F.nrows && src->ncells == F.ncols, CR_DIMENSION_MISMATCH,
               "cr_regrid_backward: grids do not match the regridder");
    CR_REQUIRE(!dst->planar && !src->planar, CR_UNSUPPORTED,
               "vertex gradients are of spherical intersection areas; these grids are planar");
    const int clip_nv = R->stats.clip_with_dst ? dst->nv : src->nv;
    CR_REQUIRE(clip_nv <= 8, CR_UNSUPPORTED, "vertex gradients need clip cells with at most 8 vertices");
    if (normalize) CR_REQUIRE(y, CR_INVALID_ARGUMENT, "cr_regrid_backward: the forward output y is needed");
    const double kappa = R->area_scale;
    DevBuf<double> coef_b;
    DevBuf<int32_t> rowid_b;
    double *coef = ws ? ws->coef : nullptr;
    int32_t *rowid = ws ? ws->rowid : nullptr;
    if (!ws) {
        coef_b.alloc_async(F.nnz, s);
        rowid_b.alloc_async(F.nnz, s);
        coef = coef_b.p;
        rowid = rowid_b.p;
    }
    row_ids(F, rowid, s);
    if (F.nnz)
        hipLaunchKernelGGL(k_pair_coef, dim3(grid_for(F.nnz, B)), dim3(B), 0, s, rowid, F.col.p, F.nnz,
                           (int)(transpose != 0), (int)(normalize != 0), kappa, a_to, nfields, x, xc, xf, gy, gc,
                           gf, coef);
    DevBuf<int32_t> list_b;
    DevBuf<uint32_t> count_b;
    int32_t *list = ws ? ws->list : nullptr;
    uint32_t *count = ws ? ws->count : nullptr;
    if (!ws) {
        list_b.alloc_async(F.nnz, s);
        count_b.alloc_async(1, s);
        list = list_b.p;
        count = count_b.p;
    }
    const AreaTerm area{normalize && !transpose ? y : nullptr, gy, a_to, F.rowptr.p, yc, yf, gc, gf, nfields, kappa};
    hipLaunchKernelGGL(k_vertex_start, dim3(grid_for(area.y ? F.nrows : 1, B)), dim3(B), 0, s, count, area, F.nrows,
                       F.nnz, dst->cells.p, dst->nv, dst->vidx.p, g_dst_verts);
    if (F.nnz) {
        // most pairs by boundary arcs; the pairs that declines through the clip pipeline
        const size_t lds = (size_t)kGradRows * dst->nv * 3 * sizeof(double);
        const bool cd = R->stats.clip_with_dst != 0;
        const int window = arc_rows(dst->nv);
        const size_t arcs_lds = (size_t)window * dst->nv * 3 * sizeof(double);
        auto vertex_pass = [&](auto nc, auto mask) {
            constexpr int NC = decltype(nc)::value;
            hipLaunchKernelGGL((k_clip_grad_arcs<NC, decltype(mask)>), dim3(grid_for(F.nnz, 64)), dim3(64), arcs_lds, s,
                               rowid, F.col.p, coef, F.nnz, dst->cells.p, dst->nv, dst->vidx.p, src->cells.p, src->nv,
                               src->vidx.p, (int)cd, window, area, g_dst_verts, g_src_verts,
                               list, count);
            hipLaunchKernelGGL(k_clip_grad_list<NC>, dim3(kListBlocks), dim3(64), lds, s, rowid, F.col.p, coef,
                               dst->cells.p, dst->nv, dst->vidx.p, src->cells.p, src->nv, src->vidx.p,
                               R->stats.clip_with_dst, g_dst_verts, g_src_verts, (const int32_t *)list,
                               (const uint32_t *)count, F.nrows);
        };
        using C4 = std::integral_constant<int, 4>;
        using C8 = std::integral_constant<int, 8>;
        const int ns = cd ? src->nv : dst->nv;  // the subject's vertices: a bit each
        auto with_clip = [&](auto nc) {
            if (ns <= 8) vertex_pass(nc, uint8_t());
            else if (ns <= 32) vertex_pass(nc, uint32_t());
            else vertex_pass(nc, uint64_t());
        };
        if (clip_nv <= 4) with_clip(C4());
        else with_clip(C8());
        CR_HIP(hipGetLastError());
    }
    double *g_to = g_src_verts;
    const cr_grid *gto = src;
    if (normalize && transpose && g_to) {  // forward: with the pairs above
        const bool table = gto->private_vertices && gto->flipped == 0;  // slot -> vertex is the identity
        if (table && gto->nv == 4)
            hipLaunchKernelGGL(k_area_grad_table<4>, dim3(grid_for(n_to, 64)), dim3(128), 0, s, gto->cells.p, n_to,
                               kappa, a_to, nfields, y, yc, yf, gy, gc, gf, g_to);
        else if (table && gto->nv == 8)
            hipLaunchKernelGGL(k_area_grad_table<8>, dim3(grid_for(n_to, 64)), dim3(128), 0, s, gto->cells.p, n_to,
                               kappa, a_to, nfields, y, yc, yf, gy, gc, gf, g_to);
        else if (table && gto->nv == 16)
            hipLaunchKernelGGL(k_area_grad_table<16>, dim3(grid_for(n_to, 64)), dim3(128), 0, s, gto->cells.p,
                               n_to, kappa, a_to, nfields, y, yc, yf, gy, gc, gf, g_to);
        else if (gto->private_vertices && gto->nv <= kStagedNv)
            hipLaunchKernelGGL(k_area_grad_private, dim3(grid_for(n_to, 64)), dim3(64),
                               2 * 64 * 3 * gto->nv * sizeof(double), s, gto->cells.p, gto->nv,
                               gto->vidx.p, n_to, kappa, a_to, nfields, y, yc, yf, gy, gc, gf, g_to);
        else
            hipLaunchKernelGGL(k_area_grad, dim3(grid_for(n_to, B)), dim3(B), 0, s, gto->cells.p, gto->nv,
                               gto->vidx.p, n_to, kappa, a_to, nfields, y, yc, yf, gy, gc, gf, g_to);
    }
    CR_HIP(hipGetLastError());
    release(coef_b, rowid_b, list_b, count_b);
    if (!ws) synchronise(s);
}

// The allocation-free reverse mode's scratch: one static array per device
// (every GPU the library runs on keeps its copy until the process ends).  Host
// code must use the per-device address from hipGetSymbolAddress, never the
// array's name (that is a host-side stand-in, not a device address).
constexpr size_t kNoAllocScratchBytes = (size_t)64 << 20;
__device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

static unsigned char *scratch_address() {
    static std::mutex mu;
    static unsigned char *ptr[256] = {};
    int dev = 0;
    CR_HIP(hipGetDevice(&dev));
    CR_REQUIRE(dev >= 0 && dev < 256, CR_UNSUPPORTED, "device index out of range");
    std::lock_guard<std::mutex> lock(mu);
    if (!ptr[dev]) {
        void *p = nullptr;
        CR_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        CR_REQUIRE(p, CR_INTERNAL, "hipGetSymbolAddress gave no address for the scratch array");
        ptr[dev] = (unsigned char *)p;
    }
    return ptr[dev];
}

}  // namespace cr

using namespace cr;

extern "C" {

cr_status cr_regrid_backward_noalloc(const cr_regridder *R, const cr_grid *dst, const cr_grid *src,
                                     int32_t transpose, int32_t normalize, int64_t nfields, const double *x,
                                     int64_t xc, int64_t xf, const double *y, int64_t yc, int64_t yf,
                                     const double *gy, int64_t gc, int64_t gf, double *gx, int64_t gxc,
                                     int64_t gxf, double *g_dst_verts, double *g_src_verts, void *stream) {
    return guard([&] {
        CR_REQUIRE(R && nfields > 0, CR_INVALID_ARGUMENT, "cr_regrid_backward_noalloc: bad arguments");
        const Csr &F = R->fwd;
        const int64_t n_to = transpose ? F.ncols : F.nrows;
        auto up = [](size_t b) { return (b + 255) / 256 * 256; };
        const size_t wbytes = gx ? up((size_t)n_to * (size_t)nfields * sizeof(double)) : 0;
        const bool verts = g_dst_verts || g_src_verts;
        const size_t cbytes = verts ? up((size_t)F.nnz * sizeof(double)) : 0;
        const size_t rbytes = verts ? up((size_t)F.nnz * sizeof(int32_t)) : 0;
        const size_t lbytes = verts ? up((size_t)F.nnz * sizeof(int32_t)) + 256 : 0;  // list + count
        const size_t need = wbytes + cbytes + rbytes + lbytes;
        CR_REQUIRE(need <= kNoAllocScratchBytes, CR_INVALID_ARGUMENT,
                   "cr_regrid_backward_noalloc: the call needs " + std::to_string(need) +
                       " bytes of scratch, over its maximum of " + std::to_string(kNoAllocScratchBytes) +
                       " (use cr_regrid_backward)");
        unsigned char *base = scratch_address();
        BackwardScratch ws;
        ws.w = wbytes ? (double *)base : nullptr;
        ws.coef = cbytes ? (double *)(base + wbytes) : nullptr;
        ws.rowid = rbytes ? (int32_t *)(base + wbytes + cbytes) : nullptr;
        ws.count = lbytes ? (uint32_t *)(base + wbytes + cbytes + rbytes) : nullptr;
        ws.list = lbytes ? (int32_t *)(base + wbytes + cbytes + rbytes + 256) : nullptr;
        R->uses.on(as_stream(stream));
        if (dst) dst->uses.on(as_stream(stream));
        if (src) src->uses.on(as_stream(stream));
        backward(R, dst, src, transpose, normalize, nfields, x, xc, xf, y, yc, yf, gy, gc, gf, gx, gxc, gxf,
                 g_dst_verts, g_src_verts, as_stream(stream), &ws);
    });
}

cr_status cr_regrid_backward(const cr_regridder *R, const cr_grid *dst, const cr_grid *src,
                             int32_t transpose, int32_t normalize, int64_t nfields, const double *x,
                             int64_t xc, int64_t xf, const double *y, int64_t yc, int64_t yf,
                             const double *gy, int64_t gc, int64_t gf, double *gx, int64_t gxc,
                             int64_t gxf, double *g_dst_verts, double *g_src_verts, void *stream) {
    return guard([&] {
        refuse_capture(as_stream(stream), "cr_regrid_backward (cr_regrid_backward_noalloc does neither)");
        backward(R, dst, src, transpose, normalize, nfields, x, xc, xf, y, yc, yf, gy, gc, gf, gx, gxc, gxf,
                 g_dst_verts, g_src_verts, as_stream(stream), nullptr);
    });
}

}  // extern "C"
