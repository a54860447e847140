// kgrad.hip -- launchers of the two-electron gradient kernels (kgrad.h):
// the list of surviving quartets (pairs ordered by bound inside each
// primitive count class, so the survivors of a bra are prefixes, enumerated as
// chunks) with the lanes each quartet gets, then one launch per class pair,
// whose kernels live in kgrad/kgrad_xX.hip (one translation unit per bra
// pair class, compiled in parallel).
#include "kgrad.h"

#include <algorithm>

namespace {

using RowLaunch = void (*)(const GradArgs&, int, int, int, unsigned, size_t, double*, hipStream_t);
using RowHost = void (*)(const GradArgs&, int, int, int, double*);
const RowLaunch kRowLaunch[6] = {polyeri_grad_row_launch_0, polyeri_grad_row_launch_1, polyeri_grad_row_launch_2,
                                 polyeri_grad_row_launch_3, polyeri_grad_row_launch_4, polyeri_grad_row_launch_5};
const RowHost kRowHost[6] = {polyeri_grad_row_host_0, polyeri_grad_row_host_1, polyeri_grad_row_host_2,
                             polyeri_grad_row_host_3, polyeri_grad_row_host_4, polyeri_grad_row_host_5};

// Primitive count class: the count rounded up to three significant bits, so
// that a class has few members more or less than its label and a row few
// groups of kets.
int count_class(int n) {
    int step = 1;
    while (n >= 8 * step) step *= 2;
    return (n + step - 1) / step * step;
}

int class_nint(int X) { return ncart(kGradPL[X][0]) * ncart(kGradPL[X][1]); }
int class_roots(int X, int Y) {
    return (kGradPL[X][0] + kGradPL[X][1] + kGradPL[Y][0] + kGradPL[Y][1] + 1) / 2 + 1;
}
// Operations of one unit, about: nodes and tables, then the components.
double unit_cost(int X, int Y) {
    const int nint = class_nint(X) * class_nint(Y);
    return (grad_root_units(nint) ? 1 : class_roots(X, Y)) * (60.0 + 22.0 * nint);
}

// Lanes are added until the launch has about kGradLanes (two wavefronts for
// each of the 1024 SIMDs), while a lane keeps at least kGradWork operations
// (its own set-up and twelve LDS atomics cost about a third of that).
constexpr double kGradLanes = 131072.0, kGradWork = 3000.0;
constexpr int kGradMaxLanes = 1024;

}  // namespace

bool polyeri_grad_sort_pairs(int* pa, int* pb, double* qp, int* pp0, int* pn, const int* seg) {
    for (int t = 0; t < seg[6]; ++t)
        if (!std::isfinite(qp[t])) return false;
    std::vector<int> idx, ti;
    std::vector<double> tq;
    for (int X = 0; X < 6; ++X) {
        const int s0 = seg[X], n = seg[X + 1] - seg[X];
        if (n <= 1) continue;
        idx.resize(n);
        for (int k = 0; k < n; ++k) idx[k] = s0 + k;
        std::stable_sort(idx.begin(), idx.end(), [&](int u, int v) {
            const int cu = count_class(pn[u]), cv = count_class(pn[v]);
            if (cu != cv) return cu > cv;
            return qp[u] > qp[v];
        });
        ti.resize(n);
        for (int* x : {pa, pb, pp0, pn}) {
            for (int k = 0; k < n; ++k) ti[k] = x[idx[k]];
            std::copy(ti.begin(), ti.end(), x + s0);
        }
        tq.resize(n);
        for (int k = 0; k < n; ++k) tq[k] = qp[idx[k]];
        std::copy(tq.begin(), tq.end(), qp + s0);
    }
    return true;
}

void polyeri_grad_chunks(const double* qp, const int* pn, const int* seg, double tol, bool sorted,
                         GradChunks& ch) {
    ch.off.clear();
    ch.ij.clear();
    std::vector<int> ni;                       // quartets of each chunk of one class pair
    for (int X = 0; X < 6; ++X)
        for (int Y = 0; Y < 6; ++Y) {
            const int k = 6 * X + Y;
            ch.off0[k] = ch.ij0[k] = 0;
            ch.n[k] = 0;
            ch.nlane[k] = 0;
            ch.units[k] = 0.0;
            if (Y > X) continue;
            const int x0 = seg[X], nx = seg[X + 1] - seg[X], y0 = seg[Y], ny = seg[Y + 1] - seg[Y];
            ch.off0[k] = ch.off.size();
            ch.ij0[k] = ch.ij.size();
            if (nx <= 0 || ny <= 0) continue;
            // groups of Y: runs of one primitive count class
            std::vector<int> gs{0};
            for (int j = 1; j < ny; ++j)
                if (count_class(pn[y0 + j]) != count_class(pn[y0 + j - 1])) gs.push_back(j);
            gs.push_back(ny);
            const int nr = grad_root_units(class_nint(X) * class_nint(Y)) ? class_roots(X, Y) : 1;
            ni.clear();
            double units = 0.0;
            for (int i = 0; i < nx; ++i) {
                const double qi = qp[x0 + i];
                if (pn[x0 + i] <= 0) continue;
                for (size_t gr = 0; gr + 1 < gs.size(); ++gr) {
                    const int lo = gs[gr], hi = X == Y ? std::min(gs[gr + 1], i + 1) : gs[gr + 1];
                    if (hi <= lo || pn[y0 + lo] <= 0) continue;
                    // first j of [lo, hi) with qi Q_j < tol (the products fall with j)
                    int a = lo, b = hi;
                    while (sorted && a < b) {
                        const int m = (a + b) >> 1;
                        if (qi * qp[y0 + m] >= tol) a = m + 1;
                        else b = m;
                    }
                    if (!sorted) a = hi;
                    if (a == lo) continue;
                    const int u = count_class(pn[x0 + i]) * count_class(pn[y0 + lo]) * nr;
                    ch.ij.push_back(i);
                    ch.ij.push_back(lo);
                    ch.ij.push_back(u);
                    ni.push_back(a - lo);
                    units += (double)u * (a - lo);
                    ++ch.n[k];
                }
            }
            const double grain = std::max(units / kGradLanes, kGradWork / unit_cost(X, Y));
            unsigned long long tot = 0;
            for (int c = 0; c < ch.n[k]; ++c) {
                int& u = ch.ij[ch.ij0[k] + 3 * c + 2];
                u = (int)std::min<double>(std::max(1.0, std::ceil(u / grain)), kGradMaxLanes);
                ch.off.push_back(tot);
                tot += (unsigned long long)ni[c] * u;
            }
            ch.off.push_back(tot);
            ch.nlane[k] = tot;
            ch.units[k] = units;
        }
}

int polyeri_grad_launch(const GradArgs& g, double* d_grad, const hipStream_t* streams, int ns, const GradChunks& ch,
                        const unsigned long long* d_off, const int* d_ij) {
    if (g.nsh <= 0 || g.npair <= 0 || g.natom <= 0 || ns <= 0 || 3 * g.natom * 8 > 48 * 1024) return -1;
    // costliest class pair first, each to the least loaded stream
    std::vector<std::pair<double, int>> order;
    for (int X = 0; X < 6; ++X)
        for (int Y = 0; Y <= X; ++Y)
            if (ch.nlane[6 * X + Y] > 0) order.push_back({ch.units[6 * X + Y] * unit_cost(X, Y), 6 * X + Y});
    std::stable_sort(order.begin(), order.end(), [](const auto& a, const auto& b) { return a.first > b.first; });
    std::vector<double> load(ns, 0.0);
    for (const auto& o : order) {
        const int k = o.second, X = k / 6, Y = k % 6;
        GradArgs gx = g;
        gx.coff = d_off + ch.off0[k];
        gx.cij = d_ij + ch.ij0[k];
        gx.nchunk = ch.n[k];
        const unsigned long long want = (ch.nlane[k] + 255) / 256;
        const unsigned grid = (unsigned)(want < 8192ULL ? want : 8192ULL);
        const int q = (int)(std::min_element(load.begin(), load.end()) - load.begin());
        load[q] += o.first;
        kRowLaunch[X](gx, Y, g.seg[X], g.seg[Y], grid, 3 * (size_t)g.natom * sizeof(double), d_grad, streams[q]);
        if (hipGetLastError() != hipSuccess) return -2;
    }
    return 0;
}

int polyeri_grad_host(const GradArgs& g, const GradShells& gs, double* grad) {
    const RysTabs rt = host_tabs();
    const int npair = g.npair;
    std::vector<double> Qp(npair);
    for (int t = 0; t < npair; ++t) Qp[t] = pair_bound(gs, rt, g.pa[t], g.pb[t]);
    // the survivors only, with the lanes of the device
    std::vector<int> pa(g.pa, g.pa + npair), pb(g.pb, g.pb + npair), pp0(g.pp0, g.pp0 + npair),
        pn(g.pn, g.pn + npair);
    const bool sorted = polyeri_grad_sort_pairs(pa.data(), pb.data(), Qp.data(), pp0.data(), pn.data(), g.seg);
    GradChunks ch;
    polyeri_grad_chunks(Qp.data(), pn.data(), g.seg, g.tol, sorted, ch);
    GradArgs gq = g;
    gq.Qp = Qp.data();
    gq.pa = pa.data();
    gq.pb = pb.data();
    gq.pp0 = pp0.data();
    gq.pn = pn.data();
    for (int i = 0; i < 3 * g.natom; ++i) grad[i] = 0.0;
    for (int X = 0; X < 6; ++X)
        for (int Y = 0; Y <= X; ++Y) {
            const int k = 6 * X + Y;
            if (ch.nlane[k] == 0) continue;
            GradArgs gx = gq;
            gx.coff = ch.off.data() + ch.off0[k];
            gx.cij = ch.ij.data() + ch.ij0[k];
            gx.nchunk = ch.n[k];
            kRowHost[X](gx, Y, g.seg[X], g.seg[Y], grad);
        }
    return 0;
}
