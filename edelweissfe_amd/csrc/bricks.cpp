// Bricks of the hexa8 matrix-free operator (matfree.hip): the elements grouped into compact
// workgroup-sized sets, with every index table the product needs.
//
// A product stages each brick's distinct nodes once and writes one partial force per (brick,
// node), so its traffic beyond the tangents goes with the nodes per element of a brick: 2.5 for
// 256 consecutive elements of a box in lattice order (two thin slabs of nodes), 1.6 for the
// 8 x 8 x 4 sets found here.  The elements are split recursively across the longest side
// (measured in mean element sizes), at a gap between layers of elements where there is one, at
// the position that needs the fewest bricks, else nearest the middle; a set is a brick once it
// has at most EB elements and NB staged nodes, whatever the mesh.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <future>
#include <system_error>

#include "efe_internal.h"

namespace {

struct Splitter {
    const std::vector<float>& cen;  // [3][E] element centroids in mean element sizes
    std::vector<int32_t>& order;    // element indices, rearranged in place
    int E, EB, NB;

    // Splits [lo, hi) of the order and returns the position of the cut.
    int cut(int lo, int hi, std::vector<int32_t>& bins, std::vector<int32_t>& tmp) const {
        const int n = hi - lo;
        float mn[3] = {3e38f, 3e38f, 3e38f}, mx[3] = {-3e38f, -3e38f, -3e38f};
        for (int i = lo; i < hi; ++i)
            for (int k = 0; k < 3; ++k) {
                const float v = cen[(size_t)k * E + order[i]];
                mn[k] = std::min(mn[k], v);
                mx[k] = std::max(mx[k], v);
            }
        int ax = 0;
        for (int k = 1; k < 3; ++k)
            if (mx[k] - mn[k] > 1.001f * (mx[ax] - mn[ax])) ax = k;
        const float ext = mx[ax] - mn[ax];
        if (!(ext > 0.0f)) return lo + n / 2;  // coincident centroids: the order as it is
        const float* c = cen.data() + (size_t)ax * E;
        const int nb = std::min(4096, std::max(64, 4 * n));
        const float scale = (float)nb / ext;
        auto bin = [&](int e) {
            const float f = (c[e] - mn[ax]) * scale;
            return f >= (float)(nb - 1) ? nb - 1 : (f > 0.0f ? (int)f : 0);
        };
        bins.assign(nb + 1, 0);
        for (int i = lo; i < hi; ++i) ++bins[bin(order[i]) + 1];
        for (int b = 0; b < nb; ++b) bins[b + 1] += bins[b];  // bins[b]: elements before bin b
        int best = -1;
        int64_t bestCost = INT64_MAX;
        for (int b = 1; b < nb; ++b) {
            const int l = bins[b];
            if (4 * (int64_t)l < n || 4 * (int64_t)l > 3 * (int64_t)n) continue;
            const bool gap = bins[b + 1] == l;  // an empty bin: between two layers
            const int64_t bricks = (l + EB - 1) / EB + (n - l + EB - 1) / EB;
            const int64_t cost = ((gap ? 0 : 1) * (int64_t)(E + 1) + bricks) * (int64_t)(n + 1) + std::abs(2 * l - n);
            if (cost < bestCost) {
                bestCost = cost;
                best = b;
            }
        }
        if (best < 0) {  // most centroids in one bin: halve by position
            std::nth_element(order.begin() + lo, order.begin() + lo + n / 2, order.begin() + hi,
                             [&](int32_t a, int32_t b) { return c[a] != c[b] ? c[a] < c[b] : a < b; });
            return lo + n / 2;
        }
        tmp.clear();
        int w = lo;
        for (int i = lo; i < hi; ++i) {
            const int32_t e = order[i];
            if (bin(e) < best) order[w++] = e;
            else tmp.push_back(e);
        }
        std::copy(tmp.begin(), tmp.end(), order.begin() + w);
        return w;
    }
};

// the tables of one brick; entries are moved into the global tables afterwards
struct Brick {
    int lo = 0, hi = 0;
    std::vector<int32_t> nodes;   // staged nodes (a node with more than 8 incidences repeats)
    std::vector<uint16_t> linc;   // [nodes][8] incidences, 0xffff: none
    std::vector<uint16_t> lidx;   // [elements][8]
};

// Fills the tables of the elements order[lo, hi); false when more than NB nodes are staged.
bool fill(Brick& b, const Splitter& sp, const int32_t* conn, std::vector<int32_t>& scratch) {
    const std::vector<int32_t>& order = sp.order;
    const int ne = b.hi - b.lo;
    scratch.clear();
    for (int t = 0; t < ne; ++t)
        for (int a = 0; a < 8; ++a) scratch.push_back(conn[(size_t)order[b.lo + t] * 8 + a]);
    std::vector<int32_t> sorted(scratch);
    std::sort(sorted.begin(), sorted.end());
    b.nodes.clear();
    for (size_t i = 0; i < sorted.size();) {  // one entry per 8 incidences of a node
        size_t j = i;
        while (j < sorted.size() && sorted[j] == sorted[i]) ++j;
        for (size_t k = i; k < j; k += 8) b.nodes.push_back(sorted[i]);
        i = j;
    }
    if ((int)b.nodes.size() > sp.NB) return false;
    b.linc.assign(b.nodes.size() * 8, 0xffff);
    b.lidx.resize((size_t)ne * 8);
    std::vector<uint8_t> fillc(b.nodes.size(), 0);
    for (int t = 0; t < ne; ++t)  // element order inside every node's list
        for (int a = 0; a < 8; ++a) {
            const int32_t nd = scratch[(size_t)t * 8 + a];
            int l = (int)(std::lower_bound(b.nodes.begin(), b.nodes.end(), nd) - b.nodes.begin());
            while (fillc[l] == 8) ++l;
            b.lidx[(size_t)t * 8 + a] = (uint16_t)l;
            b.linc[(size_t)l * 8 + fillc[l]++] = (uint16_t)(sp.EB == kBrick ? a * kBrick + t : 8 * t + a);
        }
    return true;
}

// a task of its own thread, or run at get() when there is no thread to be had
template <typename Fn>
std::future<void> aside(Fn fn) {
    try {
        return std::async(std::launch::async, fn);
    } catch (const std::system_error&) {
        return std::async(std::launch::deferred, fn);
    }
}

void grow(const Splitter& sp, int lo, int hi, const int32_t* conn, std::vector<Brick>& out, int depth) {
    std::vector<int32_t> bins, tmp, scratch;
    if (hi - lo <= sp.EB) {
        Brick b;
        b.lo = lo;
        b.hi = hi;
        std::sort(sp.order.begin() + lo, sp.order.begin() + hi);
        if (fill(b, sp, conn, scratch)) {
            out.push_back(std::move(b));
            return;
        }
    }
    const int mid = sp.cut(lo, hi, bins, tmp);
    if (depth > 0 && hi - lo > 8192) {  // the two halves side by side
        std::vector<Brick> right;
        std::future<void> f = aside([&] { grow(sp, mid, hi, conn, right, depth - 1); });
        grow(sp, lo, mid, conn, out, depth - 1);
        f.get();
        out.insert(out.end(), std::make_move_iterator(right.begin()), std::make_move_iterator(right.end()));
        return;
    }
    grow(sp, lo, mid, conn, out, 0);
    grow(sp, mid, hi, conn, out, 0);
}

}  // namespace

void efe_build_bricks(BrickPattern& bp, int N, int E, const int32_t* conn, const double* coords,
                      const int32_t* specOfNode) {
    // centroids in the mean element sizes of their specimen, from its lowest coordinates: the bricks of a
    // specimen are the same whatever else is in the context
    // (numbers from 0 up; any other is taken as 0 here)
    auto spec = [&](int n) { return specOfNode && specOfNode[n] > 0 && specOfNode[n] < N ? specOfNode[n] : 0; };
    int nspec = 1;
    for (int n = 0; n < N; ++n) nspec = std::max(nspec, spec(n) + 1);
    std::vector<float> cen((size_t)3 * E);
    std::vector<double> lo3((size_t)3 * nspec, INFINITY), size((size_t)3 * nspec, 0.0);
    std::vector<int> count(nspec, 0);
    for (int n = 0; n < N; ++n)
        for (int k = 0; k < 3; ++k) {
            double& lo = lo3[3 * (size_t)spec(n) + k];
            lo = std::min(lo, coords[(size_t)3 * n + k]);
        }
    for (int e = 0; e < E; ++e) {
        const int s = spec(conn[(size_t)8 * e]);
        ++count[s];
        for (int k = 0; k < 3; ++k) {
            double mn = coords[(size_t)3 * conn[(size_t)8 * e] + k], mx = mn, sum = 0.0;
            for (int a = 0; a < 8; ++a) {
                const double v = coords[(size_t)3 * conn[(size_t)8 * e + a] + k];
                mn = std::min(mn, v);
                mx = std::max(mx, v);
                sum += v;
            }
            size[(size_t)3 * s + k] += mx - mn;
            cen[(size_t)k * E + e] = (float)(sum * 0.125 - lo3[(size_t)3 * s + k]);
        }
    }
    for (int e = 0; e < E; ++e) {
        const int s = spec(conn[(size_t)8 * e]);
        for (int k = 0; k < 3; ++k) {
            const double h = size[(size_t)3 * s + k] / count[s];
            if (h > 0.0 && std::isfinite(h)) cen[(size_t)k * E + e] = (float)(cen[(size_t)k * E + e] / h);
        }
    }
    std::vector<int32_t> order(E);
    for (int e = 0; e < E; ++e) order[e] = e;
    std::vector<int> seg;  // a brick holds elements of one specimen
    if (specOfNode) {
        auto of = [&](int e) { return specOfNode[conn[(size_t)8 * e]]; };
        std::stable_sort(order.begin(), order.end(), [&](int32_t a, int32_t b) { return of(a) < of(b); });
        for (int i = 0; i < E; ++i)
            if (i == 0 || of(order[i]) != of(order[i - 1])) seg.push_back(i);
    } else {
        seg.push_back(0);
    }
    seg.push_back(E);
    const int EB = bp.EB, NB = bp.NB = EB == kBrick ? kBrickNodes : 8 * EB;
    Splitter sp{cen, order, E, EB, NB};
    std::vector<Brick> bricks;
    if (seg.size() == 2) {
        grow(sp, 0, E, conn, bricks, 3);
    } else {  // specimens shared out over threads, collected in specimen order
        const int ns = (int)seg.size() - 1, nt = std::min(8, ns);
        std::vector<std::vector<Brick>> per(ns);
        std::vector<std::future<void>> th;
        for (int t = 0; t < nt; ++t)
            th.push_back(aside([&, t] {
                for (int s = t; s < ns; s += nt) grow(sp, seg[s], seg[s + 1], conn, per[s], 0);
            }));
        for (auto& x : th) x.get();
        for (auto& v : per)
            bricks.insert(bricks.end(), std::make_move_iterator(v.begin()), std::make_move_iterator(v.end()));
    }
    const int G = bp.G = (int)bricks.size();
    // tables at a fixed pitch per brick, so that a workgroup finds its own without reading offsets
    bp.pos.resize(E);
    bp.lidx.assign((size_t)G * EB * 8, 0xffff);
    bp.lnode.assign((size_t)G * NB, -1);
    bp.lpos.assign((size_t)G * NB, 0);
    bp.linc.assign((size_t)G * NB * 8, 0xffff);
    bp.pptr.assign(N + 1, 0);
    for (int g = 0; g < G; ++g) {
        const Brick& b = bricks[g];
        std::copy(b.nodes.begin(), b.nodes.end(), bp.lnode.begin() + (size_t)g * NB);
        std::copy(b.linc.begin(), b.linc.end(), bp.linc.begin() + (size_t)g * NB * 8);
        std::copy(b.lidx.begin(), b.lidx.end(), bp.lidx.begin() + (size_t)g * EB * 8);
        for (int i = b.lo; i < b.hi; ++i) bp.pos[order[i]] = g * EB + (i - b.lo);
        for (int32_t nd : b.nodes) ++bp.pptr[nd + 1];
        if (specOfNode) bp.spec.push_back(specOfNode[b.nodes[0]]);
    }
    // partial slots in node order, the bricks of a node in ascending order
    for (int n = 0; n < N; ++n) bp.pptr[n + 1] += bp.pptr[n];
    bp.L = bp.pptr[N];
    std::vector<int32_t> next(bp.pptr.begin(), bp.pptr.end() - 1);
    for (size_t i = 0; i < bp.lnode.size(); ++i)
        if (bp.lnode[i] >= 0) bp.lpos[i] = next[bp.lnode[i]]++;
}
