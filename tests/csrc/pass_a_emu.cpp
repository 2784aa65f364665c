// pass_a_emu.cpp — k_tp_pass_a (zedm-x_amd/csrc/zdx_pass_a.h) run on the CPU
// under the SIMT emulation of simt_emu.h, against the serial tests of
// zdx_topo.h: adjacency counts and rows, the longest row, and the snap hit
// words of every pair.  Segment counts at the edges of a wave, of the staged
// LDS and of the units; loops whose endpoints coincide, lie within the
// tolerance, or miss it; clutter, degenerate and non-finite segments, and
// tolerances from none to larger than the pair.
#include "simt_emu.h"

#include <algorithm>
#include <cstdio>
#include <memory>
#include <random>

#define __builtin_amdgcn_readlane(v, l) __shfl((int)(v), (int)(l))
static unsigned long long atomicOr(unsigned long long* p, unsigned long long v) {
    const unsigned long long o = *p;
    *p = o | v;
    return o;
}
template <class T>
static T atomicMax(T* p, T v) {
    const T o = *p;
    if (v > o) *p = v;
    return o;
}

#include "../../zedm-x_amd/csrc/zdx_geom.h"
#include "../../zedm-x_amd/csrc/zdx_internal.h"
#include "../../zedm-x_amd/csrc/zdx_topo.h"

namespace zdx {
namespace {
constexpr int WAVE = 64;
struct TopoBufs {
    int32_t* cell9;
    int32_t* adj;
    int32_t adj_row;
    uint64_t* snapw;
    unsigned long long* top;
    int32_t* units;
    int64_t units_cap;
    int64_t *adj_off, *snap_off;
    double tol_override;
};
#include "../../zedm-x_amd/csrc/zdx_wave.h"
#include "../../zedm-x_amd/csrc/zdx_narrow.h"
#include "../../zedm-x_amd/csrc/zdx_cluster.h"
#include "../../zedm-x_amd/csrc/zdx_pass_a.h"
}  // namespace
}  // namespace zdx

using namespace zdx;

struct Pairs {
    std::vector<int> S;
    std::vector<double> tol;
    std::vector<int64_t> off;
    std::vector<double> arena;
};

static Pairs make_pairs() {
    std::mt19937_64 g(5);
    std::uniform_real_distribution<double> u(-1.0, 1.0);
    Pairs q;
    const int sizes[] = {1, 2, 3, 7, 21, 31, 32, 33, 39, 40, 63, 64, 65, 90, 127, 128, 129, 256, 257};
    const double tols[] = {1e-3, 0.0, 0.05, 1e-9, 3.0};
    int k = 0;
    for (int S : sizes)
        for (int rep = 0; rep < (S < 100 ? 3 : 1); ++rep, ++k) {
            const double h = tols[k % 5], far = k % 4 == 1 ? 1000.0 : 0.0;
            q.S.push_back(S);
            q.tol.push_back(h);
            q.off.push_back((int64_t)q.arena.size() / 6);
            std::vector<double> e(6 * (size_t)S);
            const int loops = 1 + k % 3;
            for (int s = 0; s < S; ++s) {
                const int l = s % loops, n = (S + loops - 1) / loops, m = s / loops;
                const double a = 6.283185307179586 * m / n, b = 6.283185307179586 * (m + 1) / n;
                const double p[6] = {far + 2.5 * l + std::cos(a), std::sin(a), 0.3 * l, far + 2.5 * l + std::cos(b), std::sin(b), 0.3 * l};
                for (int d = 0; d < 6; ++d) {
                    // endpoints apart by nothing, less than, about and more than the tolerance
                    const double gap[] = {0.0, 0.3 * h, h, 3.0 * h};
                    e[6 * s + d] = p[d] + gap[(s + k) % 4] * (d < 3 ? 0.0 : (s & 1 ? 1.0 : -1.0));
                    if (s % 11 == 5) e[6 * s + d] = far + u(g);          // clutter
                    if (s % 13 == 6 && d >= 3) e[6 * s + d] = e[6 * s + d - 3];   // a point
                }
                if (k % 6 == 5 && s == S / 2) e[6 * s + 1] = k % 12 == 5 ? NAN : INFINITY;
            }
            std::shuffle((double(*)[6])e.data(), (double(*)[6])e.data() + S, g);
            q.arena.insert(q.arena.end(), e.begin(), e.end());
        }
    return q;
}

template <int MODE>
static bool check(const Pairs& q, int R, int groups, int lds_segs, bool tol_given) {
    const int n = (int)q.S.size();
    std::vector<int32_t> pi(n), nseg(q.S.begin(), q.S.end()), list(n), big, small, mesh(n);
    std::vector<int64_t> seg_off = q.off, adj_off(n), snap_off(n);
    std::vector<double> arena = q.arena, tol = q.tol;
    std::vector<int32_t> units;
    int64_t na = 0, nw = 0;
    for (int p = 0; p < n; ++p) {
        const int it = n - 1 - p;   // items in another order than the pairs
        pi[p] = p; mesh[p] = p; list[it] = p;
    }
    for (int it = 0; it < n; ++it) {
        const int S = nseg[list[it]];
        adj_off[it] = na; snap_off[it] = nw;
        na += (int64_t)S * (R + 1);
        nw += ((int64_t)S * (2 * S - 1) + 63) / 64;
        for (int b = 1; b < tp_pa_units(S); ++b) { units.push_back(it); units.push_back(b); }
        (S < TOPO_BIG_SEGS ? small : big).push_back(it);
    }
    // exact sizes, so that a store past them is seen
    std::unique_ptr<int32_t[]> adj(new int32_t[na]);
    std::unique_ptr<uint64_t[]> snap(new uint64_t[nw]);
    std::fill(adj.get(), adj.get() + na, -7);
    std::fill(snap.get(), snap.get() + nw, 0x5555ull);
    std::vector<int32_t> cell9(9 * arena.size() / 6);
    unsigned long long top[5] = {0, 0, 0, 0, units.size() / 2};
    int32_t nn = n, nbig = (int)big.size(), nsmall = (int)small.size();
    units.push_back(-1);
    TopoBufs T{cell9.data(), adj.get(), R, snap.get(), top, units.data(), (int64_t)units.size() / 2, adj_off.data(),
               snap_off.data(), tol_given ? 0.02 : 0.0};
    DPairs P{};
    P.pi = pi.data(); P.nseg = nseg.data(); P.seg_off = seg_off.data(); P.arena = arena.data();
    P.topo_list = list.data(); P.topo_n = &nn; P.topo_big = big.data(); P.topo_small = small.data();
    P.n_big = &nbig; P.n_small = &nsmall;
    DMeshes M{};
    M.tol = tol.data();
    DBodies B{};
    B.mesh = mesh.data();
    std::string err;
    if (MODE == 2) {
        err = simt::launch((unsigned)groups, PA_SMALL_THREADS,
                           (size_t)pass_a_lds_bytes(PA_SMALL_THREADS, PA_SMALL_WORDS, TOPO_BIG_SEGS),
                           [&] { k_tp_pass_a<PA_SMALL_THREADS, PA_SMALL_WORDS, 1>(P, M, B, T, TOPO_BIG_SEGS); });
    }
    if (err.empty())
        err = simt::launch((unsigned)groups, PA_THREADS, (size_t)pass_a_lds_bytes(PA_THREADS, PA_WORDS, lds_segs),
                           [&] { k_tp_pass_a<PA_THREADS, PA_WORDS, MODE>(P, M, B, T, lds_segs); });
    if (!err.empty()) {
        std::printf("FAIL %s\n", err.c_str());
        return false;
    }
    int64_t nadj = 0, nsnap = 0;
    unsigned long long most = 0;
    for (int it = 0; it < n; ++it) {
        const int p = list[it], S = nseg[p];
        const double* seg = arena.data() + 6 * seg_off[p];
        const double h = tol_given ? 0.02 : tol[p];
        std::vector<int> c9(9 * (size_t)S), row(R);
        for (int s = 0; s < S; ++s) tp_cells(seg, s, h, &c9[9 * (size_t)s]);
        for (int i = 0; i < S; ++i) {
            const int m = tp_adj_row(seg, c9.data(), h, S, i, row.data(), R);
            const int32_t* got = adj.get() + adj_off[it];
            bool ok = got[i] == m;
            for (int e = 0; e < (m < R ? m : R); ++e) ok = ok && got[S + (int64_t)i * R + e] == row[e];
            if (!ok) {
                std::printf("FAIL mode %d pair %d of %d segments: row %d has %d, expected %d\n", MODE, p, S, i, got[i], m);
                return false;
            }
            nadj += m;
            if (m > R && (unsigned long long)m > most) most = m;
        }
        std::vector<uint64_t> w(((int64_t)S * (2 * S - 1) + 63) / 64, 0);
        for (int a = 0; a < 2 * S; ++a)
            for (int b = 0; b < a; ++b)
                if (tp_snap_hit(seg, c9.data(), h, a, b)) {
                    const int64_t t = (int64_t)a * (a - 1) / 2 + b;
                    w[t >> 6] |= 1ull << (t & 63);
                    ++nsnap;
                }
        for (size_t k = 0; k < w.size(); ++k)
            if (snap[snap_off[it] + k] != w[k]) {
                std::printf("FAIL mode %d pair %d of %d segments: snap word %zu\n", MODE, p, S, k);
                return false;
            }
    }
    if (top[3] != most) {
        std::printf("FAIL mode %d: longest row %llu, expected %llu\n", MODE, top[3], most);
        return false;
    }
    std::printf("ok mode %d, rows of %d, %d groups, %d staged: %lld joined, %lld snap hits, longest row %llu\n", MODE, R,
                groups, lds_segs, (long long)nadj, (long long)nsnap, most);
    return true;
}

int main() {
    const Pairs q = make_pairs();
    const bool ok = check<0>(q, 16, 3, PA_SEGS, false) && check<2>(q, 4, 2, PA_SEGS, false) &&
                    check<0>(q, 300, 1, 33, true);
    std::printf(ok ? "pass_a_emu ok\n" : "pass_a_emu failed\n");
    return ok ? 0 : 1;
}
