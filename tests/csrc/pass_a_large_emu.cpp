// pass_a_large_emu.cpp — k_tp_pass_a on pairs whose endpoint pairs are past 32
// bits of a product or of a count (23171 segments, 32769 segments): the first,
// the middle and the last unit, against the serial tests of zdx_topo.h.  And the
// larger pairs of a step in workgroups of PA_BIG_THREADS: the rows and words of
// PA_THREADS, which pass_a_emu.cpp checks.
#define main pass_a_emu_main
#include "pass_a_emu.cpp"
#undef main

static bool check_large(int S) {
    const int R = 16;
    const double h = 1e-3;
    std::mt19937_64 g(S);
    std::vector<double> arena(6 * (size_t)S);
    auto point = [&](int k, double* p) { p[0] = 0.01 * (k % 211); p[1] = 0.01 * (k / 211 % 173); p[2] = 0.01 * (k / 211 / 173); };
    // a chain of points, one grid step apart; every third of the last segments
    // ends at earlier points of it
    for (int s = 0; s < S; ++s) {
        point(s, &arena[6 * (size_t)s]);
        point(s + 1, &arena[6 * (size_t)s + 3]);
        if (s >= S - 60 && s % 3 == 0) {
            const int k = (int)(g() % (uint64_t)S);
            point(k, &arena[6 * (size_t)s]);
            point(k + 1, &arena[6 * (size_t)s + 3]);
            arena[6 * (size_t)s] += 0.4 * h;
        }
    }
    const int nu = tp_pa_units(S);
    const int64_t npt = (int64_t)S * (2 * S - 1), nw = (npt + 63) / 64;
    int32_t pi = 0, mesh = 0, nseg = S, list = 0, nn = 1;
    int64_t seg_off = 0, adj_off = 0, snap_off = 0;
    double tol = h;
    const int units_of[] = {0, nu / 2, nu - 1};
    std::vector<int32_t> units;
    for (int b : units_of)
        if (b > 0) { units.push_back(0); units.push_back(b); }
    std::unique_ptr<int32_t[]> adj(new int32_t[(int64_t)S * (R + 1)]);
    std::unique_ptr<uint64_t[]> snap(new uint64_t[nw]);
    std::vector<int32_t> cell9(9 * (size_t)S);
    unsigned long long top[5] = {0, 0, 0, 0, units.size() / 2};
    TopoBufs T{cell9.data(), adj.get(), R, snap.get(), top, units.data(), (int64_t)units.size() / 2, &adj_off, &snap_off, 0.0};
    DPairs P{};
    P.pi = &pi; P.nseg = &nseg; P.seg_off = &seg_off; P.arena = arena.data(); P.topo_list = &list; P.topo_n = &nn;
    DMeshes M{};
    M.tol = &tol;
    DBodies B{};
    B.mesh = &mesh;
    const std::string err =
        simt::launch(1, PA_THREADS, (size_t)pass_a_lds_bytes(PA_THREADS, PA_WORDS, PA_SEGS),
                     [&] { k_tp_pass_a<PA_THREADS, PA_WORDS, 0>(P, M, B, T, PA_SEGS); });
    if (!err.empty()) {
        std::printf("FAIL %s\n", err.c_str());
        return false;
    }
    std::vector<int> c9(9 * (size_t)S), row(R);
    for (int s = 0; s < S; ++s) tp_cells(arena.data(), s, h, &c9[9 * (size_t)s]);
    int64_t nadj = 0, nsnap = 0;
    for (int b : units_of) {
        for (int i = (int)((int64_t)b * S / nu); i < (int)((int64_t)(b + 1) * S / nu); ++i) {
            const int m = tp_adj_row(arena.data(), c9.data(), h, S, i, row.data(), R);
            bool ok = adj[i] == m && m <= R;
            for (int e = 0; e < m && ok; ++e) ok = adj[S + (int64_t)i * R + e] == row[e];
            if (!ok) {
                std::printf("FAIL %d segments: row %d has %d, expected %d\n", S, i, adj[i], m);
                return false;
            }
            nadj += m;
        }
        for (int64_t w = b * nw / nu; w < (b + 1) * nw / nu; ++w) {
            uint64_t want = 0;
            for (int64_t t = 64 * w; t < 64 * w + 64 && t < npt; ++t) {
                int x, y;
                tp_pair_of(t, x, y);
                if (tp_snap_hit(arena.data(), c9.data(), h, x, y)) { want |= 1ull << (t & 63); ++nsnap; }
            }
            if (snap[w] != want) {
                std::printf("FAIL %d segments: unit %d, snap word %lld\n", S, b, (long long)w);
                return false;
            }
        }
    }
    std::printf("ok %d segments, %d units: %lld joined, %lld snap hits\n", S, nu, (long long)nadj, (long long)nsnap);
    return nsnap > 4;
}

// adjacency counts and rows (slots past a row's count as they were) and snap
// words of the larger pairs
template <int NT>
static std::vector<uint64_t> big_pairs(const Pairs& q, int groups) {
    const int n = (int)q.S.size(), R = 6;
    std::vector<int32_t> pi(n), nseg(q.S.begin(), q.S.end()), list(n), big, mesh(n), units;
    std::vector<int64_t> seg_off = q.off, adj_off(n), snap_off(n);
    std::vector<double> arena = q.arena, tol = q.tol;
    int64_t na = 0, nw = 0;
    for (int it = 0; it < n; ++it) {
        const int S = nseg[it];
        pi[it] = mesh[it] = list[it] = it;
        adj_off[it] = na; snap_off[it] = nw;
        na += (int64_t)S * (R + 1);
        nw += ((int64_t)S * (2 * S - 1) + 63) / 64;
        for (int b = 1; b < tp_pa_units(S); ++b) { units.push_back(it); units.push_back(b); }
        if (S >= TOPO_BIG_SEGS) big.push_back(it);
    }
    std::vector<int32_t> adj(na, -7), cell9(9 * arena.size() / 6);
    std::vector<uint64_t> snap(nw, 0x5555ull);
    unsigned long long top[5] = {0, 0, 0, 0, units.size() / 2};
    int32_t nn = n, nbig = (int)big.size(), none = 0;
    TopoBufs T{cell9.data(), adj.data(), R, snap.data(), top, units.data(), (int64_t)units.size() / 2, adj_off.data(),
               snap_off.data(), 0.02};
    DPairs P{};
    P.pi = pi.data(); P.nseg = nseg.data(); P.seg_off = seg_off.data(); P.arena = arena.data();
    P.topo_list = list.data(); P.topo_n = &nn; P.topo_big = big.data(); P.n_big = &nbig; P.n_small = &none;
    DMeshes M{};
    M.tol = tol.data();
    DBodies B{};
    B.mesh = mesh.data();
    const std::string err = simt::launch((unsigned)groups, NT, (size_t)pass_a_lds_bytes(NT, PA_WORDS, PA_SEGS),
                                         [&] { k_tp_pass_a<NT, PA_WORDS, 2>(P, M, B, T, PA_SEGS); });
    if (!err.empty()) {
        std::printf("FAIL %s\n", err.c_str());
        return {};
    }
    std::vector<uint64_t> out(snap);
    for (int32_t a : adj) out.push_back((uint64_t)(int64_t)a);
    out.push_back(top[3]);
    return out;
}
static bool check_big() {
    Pairs q = make_pairs();
    for (double& x : q.arena)
        if (!std::isfinite(x)) x = 0.25;   // the cells of others wrap
    const std::vector<uint64_t> a = big_pairs<PA_THREADS>(q, 2), b = big_pairs<PA_BIG_THREADS>(q, 3);
    const bool same = !a.empty() && a == b;
    std::printf("%s %d threads as %d: %zu words\n", same ? "ok" : "FAIL", PA_BIG_THREADS, PA_THREADS, a.size());
    return same;
}

int main() {
    const bool ok = check_big() && check_large(23300) && check_large(32900);
    std::printf(ok ? "pass_a_large ok\n" : "pass_a_large failed\n");
    return ok ? 0 : 1;
}
