// cluster_extremes_emu.cpp — the cluster kernels on bodies at the ends of their
// range (tests/test_cluster_extremes.py): quaternions that qnormalize takes for
// the identity, for zero, and beside those; world vertices that are no numbers or
// infinite.  The kept triangles are restated by their vertices' outcodes, as the
// hit-arena kernels take them (a vertex that is no number lies beyond no side),
// the rest as in cluster_emu.cpp, whose runs are used.
//
//   cluster_extremes_emu INPUT FIRST     (from pair FIRST on, vertices are spoilt)
#define main cluster_emu_main
#define expect expect_by_boxes
#include "cluster_emu.cpp"
#undef expect
#undef main

static Expect expect(const Scene& s, int i, int j) {
    Expect e;
    std::vector<int> kept[2];
    std::vector<FBox> fb[2];
    const int body[2] = {i, j};
    for (int a = 0; a < 2; ++a) {
        const FBox other = fbox(&s.aabb[6 * body[1 - a]], &s.aabb[6 * body[1 - a] + 3]);
        const OcThr thr = oc_thresholds(other.v);
        for (int t = 0; t < s.ntris[s.mesh[body[a]]]; ++t) {
            V3 c[3];
            unsigned all = ~0u;
            for (int k = 0; k < 3; ++k) {
                const double* w = &s.wv[3 * (size_t)(s.wv_off[body[a]] + s.hm[s.mesh[body[a]]].tri_idx[3 * (size_t)t + k])];
                all &= vertex_outcode(w, thr);
                c[k] = v3(w[0], w[1], w[2]);
            }
            if (all) continue;
            double lo[3], hi[3];
            tri_box(c, lo, hi);
            kept[a].push_back(t);
            fb[a].push_back(fbox(lo, hi));
        }
    }
    e.tests = (int64_t)kept[0].size() * (int64_t)kept[1].size();
    e.kept = (int)(kept[0].size() + kept[1].size());
    auto corners = [&](int b, int t, V3* o) {
        for (int c = 0; c < 3; ++c) {
            const double* w = &s.wv[3 * (size_t)(s.wv_off[b] + s.hm[s.mesh[b]].tri_idx[3 * (size_t)t + c])];
            o[c] = v3(w[0], w[1], w[2]);
        }
    };
    for (size_t a = 0; a < kept[0].size(); ++a)
        for (size_t b = 0; b < kept[1].size(); ++b) {
            if (!meets(fb[0][a], fb[1][b])) continue;
            ++e.hits;
            PairHit h{};
            V3 p0, p1;
            int c0 = 0, c1 = 0;
            double w[18];
            V3 A[3], Bt[3];
            corners(i, kept[0][a], A);
            corners(j, kept[1][b], Bt);
            for (int k = 0; k < 3; ++k) {
                const V3 q[2] = {A[k], Bt[k]};
                for (int d = 0; d < 2; ++d) {
                    w[9 * d + 3 * k] = q[d].x; w[9 * d + 3 * k + 1] = q[d].y; w[9 * d + 3 * k + 2] = q[d].z;
                }
            }
            for (int k = 0; k < 6; ++k) h.v[k] = k;
            if (!exact_hit<true>(w, h, p0, p1, c0, c1)) continue;
            e.seg.insert(e.seg.end(), {p0.x, p0.y, p0.z, p1.x, p1.y, p1.z});
            e.prov.insert(e.prov.end(), {kept[0][a], kept[1][b], c0, c1});
        }
    return e;
}

int main(int argc, char** argv) {
    Scene s;
    if (argc < 3 || !read_scene(argv[1], s)) return 2;
    const int np = (int)s.pi.size(), first = std::atoi(argv[2]);
    const double bad[] = {NAN, INFINITY, -INFINITY};
    for (int p = first; p < np; ++p)
        for (int b : {s.pi[p], s.pj[p]}) {
            const int nv = s.nverts[s.mesh[b]];
            double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
            for (int v = 0; v < nv; ++v) {
                double* w = &s.wv[3 * (size_t)(s.wv_off[b] + v)];
                if (v % 7 == p % 7 && (b & 1) == (p & 1)) w[(v + p) % 3] = bad[(p - first) % 3];
                for (int k = 0; k < 3; ++k) { lo[k] = std::fmin(lo[k], w[k]); hi[k] = std::fmax(hi[k], w[k]); }
            }
            for (int k = 0; k < 3; ++k) { s.aabb[6 * b + k] = lo[k]; s.aabb[6 * b + 3 + k] = hi[k]; }
        }
    // the spoilt bodies' clusters are never skipped: their spheres know nothing of it
    for (float& x : s.sph)
        if (first < np) x = INFINITY;
    std::vector<Expect> ex(np);
    int hits = 0, segs = 0;
    for (int p = 0; p < np; ++p) {
        ex[p] = expect(s, s.pi[p], s.pj[p]);
        hits += ex[p].hits;
        segs += (int)ex[p].seg.size() / 6;
    }
    const Run runs[] = {{256, true, false, true, 2, 64, 0, false, 65536, true}, {512, true, false, false, 2, 64, 0, false, 0, false}};
    int fails = 0;
    for (const Run& r : runs) fails += check_run(s, ex, r);
    std::printf("%d pairs, %d hits, %d segments: cluster_extremes %s\n", np, hits, segs, fails ? "failed" : "ok");
    return fails ? 1 : 0;
}
