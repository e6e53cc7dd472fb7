// Host plan of the default field solve: see fdm_front.h.
#include "fdm_front.h"

#include <algorithm>

namespace sbf {

namespace {

// Column structures below the diagonal of the union pattern of L and U^T,
// closed under elimination (a column's structure past its first row is part of
// that row's structure), each ascending. For factors computed without
// off-diagonal pivots the union is closed already and nothing is added.
std::vector<std::vector<int>> closed_structure(const RowTerms& lower, const RowTerms& upper) {
    const int n = (int)lower.size();
    std::vector<std::vector<int>> st(n);
    std::vector<int> cnt(n, 0);
    for (int i = 0; i < n; i++)
        for (const auto& e : lower[i]) cnt[e.first]++;
    for (int j = 0; j < n; j++) st[j].reserve(cnt[j]);
    for (int i = 0; i < n; i++)   // ascending i: each column's rows come out ascending
        for (const auto& e : lower[i]) st[e.first].push_back(i);
    std::vector<int> mark(n, -1), kid(n, -1), next(n, -1);   // kid / next: lists of the columns whose first row is j
    for (int j = 0; j < n; j++) {
        std::vector<int>& s = st[j];
        bool sorted = true;
        for (int i : s) mark[i] = j;
        auto add = [&](int i) {
            if (mark[i] == j) return;
            mark[i] = j;
            s.push_back(i);
            sorted = false;
        };
        for (const auto& e : upper[j]) add(e.first);
        for (int c = kid[j]; c >= 0; c = next[c])
            for (size_t q = 1; q < st[c].size(); q++) add(st[c][q]);
        if (!sorted) std::sort(s.begin(), s.end());
        if (!s.empty()) {
            next[j] = kid[s[0]];
            kid[s[0]] = j;
        }
    }
    return st;
}

int tiles16(int x) { return (x + 15) / 16; }
int steps4(int x) { return (x + 3) / 4; }

}  // namespace

void plan_fronts(const RowTerms& lower, const RowTerms& upper, FrontPlan* out) {
    const int n = (int)lower.size();
    const std::vector<std::vector<int>> st = closed_structure(lower, upper);
    std::vector<int> par(n, -1), size(n, 1);
    for (int j = 0; j < n; j++) {
        if (!st[j].empty()) par[j] = st[j][0];
        if (par[j] >= 0) size[par[j]] += size[j];
    }
    // fr[j]: the root (last column) of j's front. First the leaves, every
    // other column a front of its own
    std::vector<int> fr(n);
    for (int j = n - 1; j >= 0; j--)
        fr[j] = size[j] <= kLeafCols && par[j] >= 0 && size[par[j]] <= kLeafCols ? fr[par[j]] : j;
    auto leaf = [&](int j) { return size[j] <= kLeafCols; };
    std::vector<int> w(n, 0);
    for (int j = 0; j < n; j++) w[fr[j]]++;
    // merge a front's upper children into it, longest boundary first, while the
    // operators grow by less than half (and a small front's by at most 2 tiles):
    // the fewer and wider the fronts, the fewer dependent steps a solve has
    std::vector<std::vector<int>> kids(n);
    std::vector<int> into(n);
    for (int j = 0; j < n; j++) into[j] = j;
    auto entries = [](double a, double r) { return a * a + 2.0 * a * r; };
    std::vector<int> cand;
    for (int j = 0; j < n; j++) {
        if (fr[j] != j) continue;
        const double r = (double)st[j].size();
        if (!leaf(j)) {
            cand.swap(kids[j]);
            kids[j].clear();
            std::stable_sort(cand.begin(), cand.end(), [&](int a, int b) { return st[a].size() > st[b].size(); });
            for (int c : cand) {
                const int W = w[j] + w[c];
                if (!leaf(c) && W <= kFrontCols
                    && entries(W, r) <= 1.5 * (entries(w[j], r) + entries(w[c], (double)st[c].size())) + 512.0) {
                    w[j] = W;
                    into[c] = j;
                    kids[j].insert(kids[j].end(), kids[c].begin(), kids[c].end());
                    kids[c].clear();
                } else {
                    kids[j].push_back(c);
                }
            }
            cand.clear();
        }
        if (par[j] >= 0) kids[fr[par[j]]].push_back(j);
    }
    // the root every column ends in (a merged root's target is a later column)
    for (int j = n - 1; j >= 0; j--) fr[j] = fr[j] == j ? (into[j] == j ? j : fr[into[j]]) : fr[fr[j]];
    std::vector<int> roots, height(n, 0);
    for (int j = 0; j < n; j++) {
        if (fr[j] != j) continue;
        roots.push_back(j);
        for (int c : kids[j]) height[j] = std::max(height[j], height[c] + 1);
    }
    std::stable_sort(roots.begin(), roots.end(), [&](int a, int b) { return height[a] < height[b]; });

    FrontPlan& o = *out;
    o = FrontPlan();
    const int nf = (int)roots.size();
    o.fronts.resize(nf);
    o.front_of.assign(n, 0);
    o.local.assign(n, 0);
    o.pos.assign(n, 0);
    std::vector<int> id(n, -1);
    int off = 0;
    for (int f = 0; f < nf; f++) {
        Front& F = o.fronts[f];
        id[roots[f]] = f;
        F.off = off;
        F.w = 0;
        F.r = (int)st[roots[f]].size();
        off += w[roots[f]];
        if (height[roots[f]] == 0) o.n_leaf = off;
    }
    for (int j = 0; j < n; j++) {   // ascending columns within a front
        const int f = id[fr[j]];
        o.front_of[j] = f;
        o.local[j] = o.fronts[f].w++;
        o.pos[j] = o.fronts[f].off + o.local[j];
    }
    int rows = 0;
    for (int f = 0; f < nf; f++) {
        Front& F = o.fronts[f];
        const std::vector<int>& B = st[roots[f]];
        F.brow = (int)o.bperm.size();
        for (int i : B) o.bperm.push_back(i);
        while (o.bperm.size() % 4) o.bperm.push_back(B.back());
        F.c = o.n_c;
        o.n_c += F.r;
        F.arow = height[roots[f]] ? rows : 0;
        if (height[roots[f]]) rows += F.w + F.r;
        const long long kw = steps4(F.w), kr = steps4(F.r);
        F.f = (long long)o.ops;
        o.ops += (size_t)(64 * tiles16(F.r) * kw);
        F.k = (long long)o.ops;
        o.ops += (size_t)(64 * tiles16(F.w) * (kw + kr));
    }
    for (int i : o.bperm) o.brow.push_back(o.pos[i]);
    // assembly: each child's contributions into its parent's rows
    o.arow.assign(std::max(rows, 1), AsmRow{});
    std::vector<std::vector<int>> src;
    std::vector<int> at(n, -1);
    for (int f = 0; f < nf; f++) {
        const Front& F = o.fronts[f];
        const int root = roots[f];
        if (!height[root]) continue;
        src.assign(F.w + F.r, {});
        for (int k = 0; k < F.r; k++) at[o.bperm[F.brow + k]] = F.w + k;
        for (int c : kids[root]) {
            const Front& K = o.fronts[id[c]];
            for (int k = 0; k < K.r; k++) {
                const int i = o.bperm[K.brow + k];
                src[o.front_of[i] == f ? o.local[i] : at[i]].push_back(K.c + k);
            }
        }
        for (int q = 0; q < F.w + F.r; q++) {
            AsmRow& a = o.arow[F.arow + q];
            for (int s = 0; s < 4; s++) a.s[s] = s < (int)src[q].size() ? src[q][s] : o.n_c;
            a.xb = (int)o.xsrc.size();
            for (size_t s = 4; s < src[q].size(); s++) o.xsrc.push_back(src[q][s]);
            a.xe = (int)o.xsrc.size();
        }
    }
    // tasks, a height at a time
    for (int f = 0; f < nf;) {
        const int h = height[roots[f]];
        int e = f;
        FrontLevel L{};
        while (e < nf && height[roots[e]] == h) L.wmax = std::max(L.wmax, o.fronts[e++].w);
        L.f0 = (int)o.tasks.size();
        for (int g = f; g < e; g++)
            for (int t = 0; t < std::max(tiles16(o.fronts[g].r), h ? 1 : 0); t++) o.tasks.push_back({g, t});
        L.nf = (int)o.tasks.size() - L.f0;
        L.k0 = (int)o.tasks.size();
        for (int g = f; g < e; g++)
            for (int t = 0; t < tiles16(o.fronts[g].w); t++) o.tasks.push_back({g, t});
        L.nk = (int)o.tasks.size() - L.k0;
        o.levels.push_back(L);
        f = e;
    }
    for (auto* v : {&o.bperm, &o.brow, &o.xsrc})
        if (v->empty()) v->push_back(0);
}

}  // namespace sbf
