// Host build of the reverse mode's boundary arcs (sphgeom.hpp): the gradients one
// pair gets, and whether it is declined.
#include "../conservativeregridding.jl_amd/csrc/sphgeom.hpp"

using namespace cr;

static void add(double *g, int v, const d3 &d) {
    g[3 * v] += d.x;
    g[3 * v + 1] += d.y;
    g[3 * v + 2] += d.z;
}

template <int NC>
static int arcs(const double *clip, int nc, const double *subj, int ns, double *g_clip, double *g_subj) {
    uint64_t full = 0;
    LineSum S[NC], A[64];
    int edge[64], n = 0;
    if (!pair_arcs<NC, uint64_t>(clip, nc, subj, ns, full, S, [&](int, int j, const LineSum &a) {
            edge[n] = j;
            A[n++] = a;
            return true;
        }))
        return 0;
    auto line = [&](double *g, const double *ring, int j, int j1, const LineSum &L) {
        d3 gp, gq;
        line_grad(load3(ring + 3 * j), load3(ring + 3 * j1), L, gp, gq);
        add(g, j, gp);
        add(g, j1, gq);
    };
    for (int j = 0; j < ns; ++j)
        if (full >> j & 1) {
            const double h = whole_sum(load3(subj + 3 * j), load3(subj + 3 * ((j + 1) % ns)));
            line(g_subj, subj, j, (j + 1) % ns, LineSum{h, h});
        }
    for (int i = 0; i < n; ++i) line(g_subj, subj, edge[i], (edge[i] + 1) % ns, A[i]);
    for (int k = 0; k < NC; ++k) {
        const int i0 = clip_first<NC>(k, nc), i1 = clip_second<NC>(k, nc);
        if (i0 != i1) line(g_clip, clip, i0, i1, S[k]);
    }
    return 1;
}

extern "C" {

// 1: g_clip (nc x 3) and g_subj (ns x 3) hold d(area)/d(vertices); 0: declined
int arcs_grad(const double *clip, int nc, const double *subj, int ns, double *g_clip, double *g_subj) {
    return nc <= 4 ? arcs<4>(clip, nc, subj, ns, g_clip, g_subj) : arcs<8>(clip, nc, subj, ns, g_clip, g_subj);
}

double forward_area(const double *clip, int nc, const double *subj, int ns) {
    return nc <= 4 ? clip_area_stream<4>(clip, nc, subj, ns) : clip_area_stream<8>(clip, nc, subj, ns);
}
}
