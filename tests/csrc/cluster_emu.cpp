// cluster_emu.cpp — the cluster kernels of zedm-x_amd/csrc/zdx_cluster.h run
// on the CPU under the SIMT emulation of simt_emu.h: k_cluster_spheres over the
// meshes, then k_pairs_wave followed by k_pairs_group over the pairs it
// leaves, or k_pairs_group alone over every pair, for every compiled workgroup
// size, then k_pairs_exact and k_pairs_sort, with shuffled work items from the
// queue and with items in pair order striding the grid, with and without
// provenance.
//
// Each run is checked against a plain restatement: the triangles of each body
// whose outward-rounded float box meets the other's float AABB, the pairs of
// them whose float boxes overlap (counted), and of those, in (ta, tb) order,
// the ones that pass the reference's exact test, with its segments -- which
// must be the arena's, bit for bit.  Small segment capacities and arenas must
// raise their status bits and store nothing.
//
//   cluster_emu INPUT     (binary written by tests/test_cluster_emu.py)
#include "simt_emu.h"

#include <algorithm>
#include <cfenv>
#include <numeric>
#include <random>
#include <set>

#define __builtin_amdgcn_readlane(v, l) __shfl((int)(v), (int)(l))

#include "../../zedm-x_amd/csrc/zdx_geom.h"
#include "../../zedm-x_amd/csrc/zdx_internal.h"

namespace zdx {
namespace {
constexpr int WAVE = 64;
#include "../../zedm-x_amd/csrc/zdx_wave.h"
#include "../../zedm-x_amd/csrc/zdx_narrow.h"
#include "../../zedm-x_amd/csrc/zdx_cluster.h"
}  // namespace
}  // namespace zdx

using namespace zdx;

struct Scene {
    std::vector<HostMesh> hm;
    std::vector<int32_t> nverts, ntris, tri_off, vert_off, clus_off, sph_off, nclus;
    std::vector<double> verts;
    std::vector<Cluster> clus;
    std::vector<float> sph;
    std::vector<int32_t> mesh, nondeg, pi, pj;
    std::vector<int64_t> wv_off;
    std::vector<double> state, wv, aabb;
    int32_t tmax = 1;
    DMeshes M{};
};

static bool read_scene(const char* path, Scene& s) {
    FILE* f = std::fopen(path, "rb");
    if (!f) return false;
    auto rd = [&](void* p, size_t n) { return std::fread(p, 1, n, f) == n; };
    int32_t nm = 0, np = 0;
    if (!rd(&nm, 4)) return false;
    int32_t nc = 0;
    for (int m = 0; m < nm; ++m) {
        int32_t T;
        if (!rd(&T, 4)) return false;
        std::vector<double> t(9 * (size_t)T);
        if (!rd(t.data(), 72 * (size_t)T)) return false;
        s.hm.push_back(build_mesh(t, true));
        const HostMesh& h = s.hm.back();
        s.nverts.push_back((int32_t)(h.verts.size() / 3));
        s.ntris.push_back(T);
        s.tri_off.push_back(0);
        s.vert_off.push_back((int32_t)(s.verts.size() / 3));
        s.verts.insert(s.verts.end(), h.verts.begin(), h.verts.end());
        // every triangle once, with its own corners
        const std::vector<Cluster> cl = cluster_mesh(h);
        std::vector<int> seen(T, 0);
        int n = 0;
        for (const Cluster& q : cl)
            for (uint32_t w : q.t) {
                if (w >> 16 == CLUS_NONE) continue;
                const int t = (int)(w >> 16);
                bool ok = t < T && !seen[t]++;
                for (int k = 0; ok && k < 3; ++k) ok = q.v[(w >> (4 * k)) & 15u] == h.tri_idx[3 * t + k];
                if (!ok) { std::printf("FAIL: cluster triangle\n"); return false; }
                ++n;
            }
        if (n != T) { std::printf("FAIL: clusters hold %d of %d triangles\n", n, T); return false; }
        s.clus_off.push_back((int32_t)s.clus.size());
        s.sph_off.push_back(nc + 3 * m);   // gaps between the meshes' spheres
        s.nclus.push_back((int32_t)cl.size());
        s.clus.insert(s.clus.end(), cl.begin(), cl.end());
        nc += (int32_t)cl.size();
        s.tmax = std::max(s.tmax, T);
    }
    if (!rd(&np, 4)) return false;
    for (int p = 0; p < np; ++p)
        for (int side = 0; side < 2; ++side) {
            int32_t m;
            double pose[7];
            if (!rd(&m, 4) || !rd(pose, sizeof pose)) return false;
            (side ? s.pj : s.pi).push_back((int32_t)s.mesh.size());
            s.mesh.push_back(m);
            s.nondeg.push_back(s.ntris[m]);
            s.wv_off.push_back((int64_t)(s.wv.size() / 3));
            for (int k = 0; k < 16; ++k) s.state.push_back(k < 7 ? pose[k] : 0.0);
            Qt q;
            q.w = pose[3]; q.x = pose[4]; q.y = pose[5]; q.z = pose[6];
            double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
            for (int v = 0; v < s.nverts[m]; ++v) {
                const double* b = &s.verts[3 * ((size_t)s.vert_off[m] + v)];
                const V3 w = add(qrotate(q, v3(b[0], b[1], b[2])), v3(pose[0], pose[1], pose[2]));
                const double x[3] = {w.x, w.y, w.z};
                for (int k = 0; k < 3; ++k) {
                    s.wv.push_back(x[k]);
                    lo[k] = std::min(lo[k], x[k]);
                    hi[k] = std::max(hi[k], x[k]);
                }
            }
            s.aabb.insert(s.aabb.end(), lo, lo + 3);
            s.aabb.insert(s.aabb.end(), hi, hi + 3);
        }
    std::fclose(f);
    s.sph.assign(4 * (size_t)(nc + 3 * nm), NAN);
    DMeshes& M = s.M;
    M.verts = s.verts.data(); M.nverts = s.nverts.data(); M.vert_off = s.vert_off.data();
    M.tri_off = s.tri_off.data(); M.ntris = s.ntris.data();
    M.clusters = s.clus.data(); M.clus_off = s.clus_off.data(); M.nclus = s.nclus.data();
    M.clus_sph = s.sph.data(); M.sph_off = s.sph_off.data();
    const std::string e = simt::launch((unsigned)nm, 256, 0, [&] { k_cluster_spheres(M, s.sph.data()); });
    if (!e.empty()) { std::printf("FAIL k_cluster_spheres: %s\n", e.c_str()); return false; }
    return true;
}

// ---- the plain restatement
static float round_dir(double x, int mode) {
    const int old = std::fegetround();
    std::fesetround(mode);
    volatile double xv = x;
    volatile float f = (float)xv;
    std::fesetround(old);
    return f;
}
struct FBox { float v[6]; };
static FBox fbox(const double* lo, const double* hi) {
    FBox b;
    for (int k = 0; k < 3; ++k) { b.v[k] = round_dir(lo[k], FE_DOWNWARD); b.v[3 + k] = round_dir(hi[k], FE_UPWARD); }
    return b;
}
static bool meets(const FBox& a, const FBox& b) {
    for (int k = 0; k < 3; ++k)
        if (a.v[3 + k] < b.v[k] || a.v[k] > b.v[3 + k]) return false;
    return true;
}
struct Expect {
    int64_t tests = 0;
    int kept = 0, hits = 0;
    std::vector<double> seg;       // 6 each
    std::vector<int32_t> prov;     // 4 each
};
static Expect expect(const Scene& s, int i, int j) {
    Expect e;
    std::vector<int> kept[2];
    std::vector<FBox> fb[2];
    const int body[2] = {i, j};
    auto corners = [&](int b, int t, V3* o) {
        for (int c = 0; c < 3; ++c) {
            const double* w = &s.wv[3 * (size_t)(s.wv_off[b] + s.hm[s.mesh[b]].tri_idx[3 * (size_t)t + c])];
            o[c] = v3(w[0], w[1], w[2]);
        }
    };
    for (int a = 0; a < 2; ++a) {
        const FBox other = fbox(&s.aabb[6 * body[1 - a]], &s.aabb[6 * body[1 - a] + 3]);
        for (int t = 0; t < s.ntris[s.mesh[body[a]]]; ++t) {
            V3 c[3];
            corners(body[a], t, c);
            double lo[3], hi[3];
            tri_box(c, lo, hi);
            const FBox f = fbox(lo, hi);
            if (meets(f, other)) { kept[a].push_back(t); fb[a].push_back(f); }
        }
    }
    e.tests = (int64_t)kept[0].size() * (int64_t)kept[1].size();
    e.kept = (int)(kept[0].size() + kept[1].size());
    for (size_t a = 0; a < kept[0].size(); ++a)
        for (size_t b = 0; b < kept[1].size(); ++b) {
            if (!meets(fb[0][a], fb[1][b])) continue;
            ++e.hits;
            V3 A[3], Bt[3];
            corners(i, kept[0][a], A);
            corners(j, kept[1][b], Bt);
            double alo[3], ahi[3], blo[3], bhi[3];
            tri_box(A, alo, ahi);
            tri_box(Bt, blo, bhi);
            bool rej = false;
            for (int k = 0; k < 3; ++k) rej = rej || ahi[k] < blo[k] || alo[k] > bhi[k];
            if (rej) continue;
            V3 nA, nB, p0, p1;
            double dA, dB;
            int c0 = 0, c1 = 0;
            plane_of(A[0], A[1], A[2], nA, dA);
            plane_of(Bt[0], Bt[1], Bt[2], nB, dB);
            if (!tri_tri_prov(A, nA, dA, Bt, nB, dB, p0, p1, c0, c1)) continue;
            e.seg.insert(e.seg.end(), {p0.x, p0.y, p0.z, p1.x, p1.y, p1.z});
            e.prov.insert(e.prov.end(), {kept[0][a], kept[1][b], c0, c1});
        }
    return e;
}

struct Run {
    int bs;
    bool batched, prov, wave;
    int groups, shards, seg_cap;   // seg_cap 0: as many as the largest pair has
    bool full;                     // an arena one slot too small
    int heavy_tests;
    bool lists;                    // with the lists of big and small pairs
};

template <int BS>
static std::string launch_group(const Scene& s, const DBodies& B, const DPairs& P, const Run& r, unsigned* q, int back) {
    return simt::launch((unsigned)r.groups, BS, (size_t)pairs_group_lds_bytes(BS), [&] {
        k_pairs_group<BS>(B, s.M, P, r.batched, q + (back > 0 ? NQ_WG : NQ_WG_FRONT), back < 0 ? nullptr : P.heavy,
                          back < 0 ? P.n : (const int32_t*)(q + (back ? NQ_HEAVY_BACK : NQ_HEAVY)), back, nullptr);
    });
}

static int check_run(const Scene& s, const std::vector<Expect>& ex, const Run& r) {
    const int np = (int)s.pi.size();
    std::vector<double> wv = s.wv, aabb = s.aabb;
    std::vector<int32_t> nondeg = s.nondeg;
    DBodies B{};
    B.n = (int)s.mesh.size(); B.mesh = s.mesh.data(); B.state = s.state.data(); B.wv_off = s.wv_off.data();
    B.wv = wv.data(); B.nondeg = nondeg.data(); B.aabb = aabb.data();
    std::vector<int32_t> perm(np);
    std::iota(perm.begin(), perm.end(), 0);
    if (r.batched) std::shuffle(perm.begin(), perm.end(), std::mt19937(54321));
    int smax = 0, hmax = 0;
    std::vector<int64_t> load(r.shards, 0);
    for (int q = 0; q < np; ++q) {
        smax = std::max(smax, (int)ex[perm[q]].seg.size() / 6);
        hmax = std::max(hmax, ex[perm[q]].hits);
        load[q % r.shards] += ex[perm[q]].hits;
    }
    const int seg_cap = r.seg_cap ? r.seg_cap : std::max(1, smax);
    int64_t cap = (int64_t)r.shards * std::max<int64_t>(1, *std::max_element(load.begin(), load.end()));
    if (r.full) cap -= r.shards;
    std::unique_ptr<PairItem[]> items(new PairItem[np]);
    std::vector<int32_t> list(np), lists[3];
    for (auto& l : lists) l.assign(np, -7);
    int32_t counts[3] = {0, 0, 0};
    std::vector<int64_t> seg_off(np, -7), checks(np, -7), tests(np, -7);
    std::vector<int32_t> nseg(np, -7), hits(np, -7), scanned(np, -7), heavy(np, -7);
    std::unique_ptr<double[]> arena(new double[6 * (size_t)std::max<int64_t>(cap, 1)]);
    std::unique_ptr<double[]> tmp(new double[6 * (size_t)std::max<int64_t>(cap, 1)]);
    std::unique_ptr<int32_t[]> prov(new int32_t[4 * (size_t)std::max<int64_t>(cap, 1)]);
    std::unique_ptr<PairHit[]> rec(new PairHit[(size_t)std::max<int64_t>(cap, 1)]);
    std::unique_ptr<int32_t[]> flag(new int32_t[(size_t)std::max<int64_t>(cap, 1)]),
        tri(new int32_t[2 * (size_t)std::max<int64_t>(cap, 1)]);
    std::vector<int64_t> hit_off(np, -7);
    int32_t n = np, status = 0;
    unsigned long long top[HIT_SHARDS * HIT_TOP_STRIDE] = {};
    unsigned queue[NQ_COUNTERS] = {};
    DPairs P{};
    P.cap = np; P.n = &n; P.pi = s.pi.data(); P.pj = s.pj.data();
    P.pitems = items.get();
    P.hits = (int32_t*)rec.get(); P.hit_off = hit_off.data(); P.hit_flag = flag.get(); P.hit_tri = tri.get();
    P.seg_tmp = tmp.get(); P.topo_list = lists[0].data(); P.topo_n = counts;
    if (r.lists) { P.topo_big = lists[1].data(); P.topo_small = lists[2].data(); P.n_big = counts + 1; P.n_small = counts + 2; }
    for (int q = 0; q < np; ++q) make_pair_item(P, s.M, B, perm[q], items[q]);
    P.seg_off = seg_off.data(); P.nseg = nseg.data(); P.tri_checks = checks.data(); P.tri_tests = tests.data();
    P.tri_hits = hits.data(); P.tri_scanned = scanned.data(); P.status = &status; P.arena = arena.get();
    P.arena_cap = P.hit_cap = cap; P.hit_top = top; P.hit_shards = r.shards; P.heavy = heavy.data();
    P.prov = r.prov ? prov.get() : nullptr;
    char tag[128];
    std::snprintf(tag, sizeof tag, "%s %d threads %s%s groups %d seg_cap %d%s", r.wave ? "wave+group" : "group", r.bs,
                  r.batched ? "queue" : "strided", r.prov ? " prov" : "", r.groups, seg_cap, r.full ? " full arena" : "");
    std::string err;
    if (r.wave)
        err = simt::launch((unsigned)r.groups, NWV * WAVE, (size_t)pairs_wave_lds_bytes(), [&] {
            k_pairs_wave(B, s.M, P, P.heavy, queue, r.batched, r.heavy_tests, nullptr);
        });
    const unsigned left = queue[NQ_HEAVY] + queue[NQ_HEAVY_BACK];
    if (err.empty() && r.wave) err = launch_group<GROUP_BIG>(s, B, P, r, queue, 0);
    const int back = r.wave ? 1 : -1;
    if (err.empty()) switch (r.bs) {
        case 64: err = launch_group<64>(s, B, P, r, queue, back); break;
        case 128: err = launch_group<128>(s, B, P, r, queue, back); break;
        case 256: err = launch_group<256>(s, B, P, r, queue, back); break;
        default: err = launch_group<512>(s, B, P, r, queue, back); break;
    }
    if (err.empty())
        err = simt::launch((unsigned)r.groups, 256, 0, [&] {
            if (r.prov) k_pairs_exact<true>(B, P);
            else k_pairs_exact<false>(B, P);
        });
    if (err.empty())
        err = simt::launch((unsigned)r.groups, 256, 0, [&] {
            if (r.prov) k_pairs_sort<true>(P, seg_cap);
            else k_pairs_sort<false>(P, seg_cap);
        });
    if (!err.empty()) {
        std::printf("FAIL %s: emulation: %s\n", tag, err.c_str());
        return 1;
    }
    int bad = 0;
    auto fail = [&](int p, const char* what, long a, long b) {
        if (bad++ < 12) std::printf("FAIL %s: pair %d: %s: got %ld want %ld\n", tag, p, what, a, b);
    };
    const bool small = smax > seg_cap;
    if (((status & ST_STAGE) != 0) != small) fail(-1, "ST_STAGE", status, small);
    if (((status & ST_HITS) != 0) != r.full) fail(-1, "ST_HITS", status, r.full);
    long stored = 0;
    std::set<int> want_list[3];
    std::vector<std::pair<int64_t, int64_t>> ranges;
    for (int p = 0; p < np; ++p) {
        const Expect& e = ex[p];
        const int i = s.pi[p], j = s.pj[p], S = (int)e.seg.size() / 6;
        const int TA = s.ntris[s.mesh[i]], TB = s.ntris[s.mesh[j]];
        if (hits[p] != e.hits && !(r.full && hits[p] == 0)) fail(p, "tri_hits", hits[p], e.hits);
        if (tests[p] != e.tests) fail(p, "tri_tests", (long)tests[p], (long)e.tests);
        if (scanned[p] != TA + TB) fail(p, "tri_scanned", scanned[p], TA + TB);
        if (checks[p] != (int64_t)s.nondeg[i] * TB) fail(p, "tri_checks", (long)checks[p], (long)s.nondeg[i] * TB);
        const int want = r.full || S > seg_cap ? 0 : S;   // a full arena: nothing is tested
        if (nseg[p] != want) { fail(p, "nseg", nseg[p], want); continue; }
        if (nseg[p] == 0) continue;
        want_list[0].insert(p);
        want_list[S >= TOPO_BIG_SEGS ? 1 : 2].insert(p);
        stored += S;
        ranges.emplace_back(seg_off[p], seg_off[p] + S);
        if (seg_off[p] < 0 || seg_off[p] + S > cap) { fail(p, "range", (long)seg_off[p], S); continue; }
        if (std::memcmp(arena.get() + 6 * seg_off[p], e.seg.data(), 48 * (size_t)S)) fail(p, "segments", 0, 0);
        if (r.prov && std::memcmp(prov.get() + 4 * seg_off[p], e.prov.data(), 16 * (size_t)S)) fail(p, "provenance", 0, 0);
    }
    std::sort(ranges.begin(), ranges.end());
    for (size_t k = 1; k < ranges.size(); ++k)
        if (ranges[k].first < ranges[k - 1].second) fail(-1, "overlapping ranges", (long)ranges[k].first, 0);
    for (int l = 0; l < (r.lists ? 3 : 1); ++l) {
        std::set<int> got;
        for (int k = 0; k < counts[l]; ++k) got.insert(l == 0 ? lists[0][k] : lists[0][lists[l][k]]);
        if (got != want_list[l] || counts[l] != (int)got.size()) fail(-1, "work list", l, counts[l]);
    }
    if (bad == 0) std::printf("ok %s: %d pairs (%u to the workgroup kernel), %ld segments\n", tag, np, left, stored);
    return bad ? 1 : 0;
}

int main(int argc, char** argv) {
    Scene s;
    if (argc < 2 || !read_scene(argv[1], s)) {
        std::fprintf(stderr, "cluster_emu: no input\n");
        return 2;
    }
    const int np = (int)s.pi.size();
    std::vector<Expect> ex(np);
    int smax = 0, hmax = 0, kmax = 0, none = 0;
    for (int p = 0; p < np; ++p) {
        ex[p] = expect(s, s.pi[p], s.pj[p]);
        smax = std::max(smax, (int)ex[p].seg.size() / 6);
        kmax = std::max(kmax, ex[p].kept);
        hmax = std::max(hmax, ex[p].hits);
        none += ex[p].tests == 0;
    }
    std::printf("most segments %d, most hits %d, most kept triangles %d, pairs without tests %d\n", smax, hmax, kmax, none);
    const Run runs[] = {
        {256, true, false, true, 2, 64, 0, false, 16384, true}, {64, true, true, true, 4, 1, 0, false, 100, true},
        {128, false, false, true, 1, 5, 40, false, 16384, false}, {512, true, false, false, 2, 64, 0, false, 0, false},
        {256, false, true, false, 2, 1, 0, false, 0, true},     {256, true, false, true, 2, 1, 0, true, 16384, true},
    };
    int fails = 0;
    for (const Run& r : runs) fails += check_run(s, ex, r);
    if (fails) {
        std::printf("cluster_emu: %d runs failed\n", fails);
        return 1;
    }
    std::printf("cluster_emu ok: %d runs\n", (int)(sizeof(runs) / sizeof(runs[0])));
    return 0;
}
