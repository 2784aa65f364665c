// zdx_cluster.h — narrow phase by triangle clusters: k_pairs_wave (one wave
// per pair) and k_pairs_group (one workgroup per pair, for the pairs a wave
// leaves) find the hits, k_pairs_exact tests them, k_pairs_sort puts the
// segments in order.
//
// Textually included inside namespace zdx::{anonymous} after zdx_narrow.h: by
// zdx_kernels.hip for gfx950 and by the host SIMT emulation of the kernels
// (tests/csrc/cluster_emu.cpp).  No includes or namespaces of its own.
//
//   1. Each side's clusters (patches of at most CT triangles and vertices, a
//      bounding sphere each) against the other body's float box, then the
//      triangles of those that may meet it, by the vertex outcodes of
//      zdx_narrow.h: the kept triangles are those whose outward-rounded box
//      meets the other's, whichever clusters they came from.
//   2. The kept triangles' boxes in groups of GT: boxes of groups against boxes
//      of groups, then the GT x GT triangle boxes of two groups that meet, one
//      lane each.  The pairs that pass are the hits, in no fixed order; the
//      product of the kept counts is what the counter of box tests reports.
//   3. The exact tests (src/main.cpp:2130-2145), one thread per hit of all
//      pairs; segments go to their pair's range of seg_tmp as they come.
//   4. One wave per pair ranks its segments by (ta, tb), the reference's order
//      (2123-2145), and moves them to the arena.
//
// Why: both of the kernels in zdx_narrow.h read every vertex and triangle of
// both bodies and test the whole product of the kept triangles.  In the
// 60k concave packing 5 % of the triangles are kept and 0.4 % of the product
// hits, so most of that work is left out.  What bounds these: in the packing
// instruction issue as far as its waves go (the vector units 51 % busy in the
// wave kernel, 56 in the groups, 65 in the exact tests), in the 100k bed the
// latency of a pair's chain (40, 22 and 51 %, 0.95 TB/s of memory traffic over
// all four).  Narrow phase, those kernels / these, on an MI355X: 60k
// packing 4241 / 1540 us, 4096 pairs of mixed meshes 1112 / 426, 257 pairs
// with sensitivities 706 / 193, 100k bed 381 / 264.  (The exact test inside
// the wave kernel, for its own hits, took 2760 us in the packing: partial
// waves and 160 registers.)

constexpr int GT = 8;    // triangles per group (GT x GT box tests fill a wave)
static_assert(WAVE == GT * GT && WAVE % CT == 0, "a wave holds a pair of groups and whole clusters");

// LDS of one wave of k_pairs_wave: the cluster list (later the hits), then the
// kept triangles' boxes and corners (A's from the front, B's from the back)
// and the groups' boxes.  CW_WPS workgroups of four waves share a CU's 160 KB.
constexpr int CW_WPS = 4;
constexpr int CW_SLICE = ((160 * 1024 / CW_WPS - 64) / NWV) & ~31;
constexpr int CW_CLUS = 512;    // clusters of one side that may meet the other's box
constexpr int CW_HITS = 512;    // hits of one pair
constexpr int CW_TESTS = 65536; // box tests of one pair (unless tuned)
constexpr int CW_HEAD = 4 * CW_HITS;
constexpr int CW_KEPT = (CW_SLICE - CW_HEAD - 48) / 35;   // kept triangles of both sides
static_assert(CW_HEAD + 32 * CW_KEPT + 24 * (CW_KEPT / GT + 2) <= CW_SLICE, "a wave's LDS");
static_assert(2 * CW_CLUS <= CW_HEAD, "the cluster list and the hits share their place");
static_assert(CW_WPS * (NWV * CW_SLICE + 64) <= 160 * 1024, "workgroups per CU");
__host__ __device__ constexpr int pairs_wave_lds_bytes() { return NWV * CW_SLICE; }

// LDS of k_pairs_group: a range's cluster list, each wave's hits, then the
// kept triangles; 16 waves per CU.
__host__ __device__ constexpr int group_hits(int bs) { return bs >= 512 ? 512 : 320; }
__host__ __device__ constexpr int pairs_group_lds_bytes(int bs) { return 155 * bs; }
__host__ __device__ constexpr int group_kept(int bs) {
    return (pairs_group_lds_bytes(bs) - 4 * bs - 4 * group_hits(bs) * (bs / WAVE) - 48) / 35;
}
// The pairs a wave leaves: those of more than CW_FRONT kept triangles (or of
// too many clusters to count them) at the front of the list, for workgroups of
// GROUP_BIG threads; the others at its back, for the launch's workgroups
// (256 threads unless tuned).  On the 100k bed, where one pair in eight that a
// wave leaves keeps 700 to 1300 triangles (a small body inside the box of a
// large one), workgroups of 256 alone took 332 us for the narrow phase, of 512
// alone 251; in the 60k packing, where none keeps more than 600, 1465 and
// 1676.
constexpr int GROUP_BIG = 512;
constexpr int CW_FRONT = 640;
static_assert(4 * (pairs_group_lds_bytes(256) + 256) <= 160 * 1024, "16 waves per CU");
static_assert(group_kept(64) >= 3 * WAVE, "a round of both sides fits");

// Bounding sphere of every cluster of a mesh, one thread each: the centre of
// the corners' box, rounded to float, and the largest distance from that float
// centre with the margin of cluster_meets, rounded up.  A cluster with a
// non-finite corner gets an infinite radius (it is never skipped).
__global__ void __launch_bounds__(256) k_cluster_spheres(DMeshes M, float* sph) {
    const int m = blockIdx.x;
    const double* v = M.verts + 3 * (int64_t)M.vert_off[m];
    const Cluster* cl = M.clusters + M.clus_off[m];
    float* out = sph + 4 * (int64_t)M.sph_off[m];
    for (int c = threadIdx.x; c < M.nclus[m]; c += blockDim.x) {
        double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
        for (int l = 0; l < CT; ++l) {
            const double* p = v + 3 * (int)cl[c].v[l];
            for (int k = 0; k < 3; ++k) { lo[k] = fmin(lo[k], p[k]); hi[k] = fmax(hi[k], p[k]); }
        }
        float o[3];
        for (int k = 0; k < 3; ++k) o[k] = (float)(0.5 * (lo[k] + hi[k]));
        double r2 = 0.0;
        for (int l = 0; l < CT; ++l) {
            const double* p = v + 3 * (int)cl[c].v[l];
            const double x = p[0] - o[0], y = p[1] - o[1], z = p[2] - o[2];
            const double d2 = x * x + y * y + z * z;
            r2 = d2 < INFINITY ? fmax(r2, d2) : INFINITY;
        }
        for (int k = 0; k < 3; ++k) out[4 * c + k] = o[k];
        out[4 * c + 3] = __double2float_ru(sqrt(r2) * (1.0 + 1e-5) +
                                           1e-5 * (fabs((double)o[0]) + fabs((double)o[1]) + fabs((double)o[2])));
    }
}

// Whether a cluster (body-frame centre c[0..3), radius c[3] with its margin)
// may hold a triangle whose outward-rounded box meets the other body's: R the
// rotation, t the body's position relative to the other's box centre, H the
// box's half edges with their margin (make_pair_item).  False only when every
// vertex in the sphere lies beyond one side by more than a float step of it.
// The margins (1e-5 of the centre and radius here, 1e-5 of t and H there) are
// far above the roundings of this test to float, which are 1e-7 of them.
__device__ inline bool cluster_meets(const float* R, const float* t, const float* H, const float* c) {
    bool out = false;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const float w = R[3 * k] * c[0] + R[3 * k + 1] * c[1] + R[3 * k + 2] * c[2] + t[k];
        out = out | (fabsf(w) > H[k] + c[3]);
    }
    return !out;
}
// The work item of pair p: counts, offsets and the geometry of the cluster
// test (R, t, H) and of the triangles' (th: the outcode thresholds of the
// OTHER body's float box, lower then upper).
__device__ inline void make_pair_item(const DPairs& P, const DMeshes& M, const DBodies& B, int p, PairItem& o) {
    const int b[2] = {P.pi[p], P.pj[p]};
    o.p = p;
    for (int s = 0; s < 2; ++s) {
        const int m = B.mesh[b[s]];
        const double* st = B.state + 16 * (int64_t)b[s];
        const double* ob = B.aabb + 6 * (int64_t)b[1 - s];
        o.T[s] = M.ntris[m]; o.wo[s] = (int32_t)B.wv_off[b[s]];
        o.nc[s] = M.nclus[m]; o.co[s] = M.clus_off[m]; o.so[s] = M.sph_off[m];
        double w = st[3], x = st[4], y = st[5], z = st[6];
        const double n = w * w + x * x + y * y + z * z;
        if (n < 1e-28) { w = 1.0; x = y = z = 0.0; }   // as qnormalize
        const double f = n < 1e-28 ? 2.0 : 2.0 / n;
        float* R = o.R[s];
        R[0] = (float)(1.0 - f * (y * y + z * z)); R[1] = (float)(f * (x * y - z * w)); R[2] = (float)(f * (x * z + y * w));
        R[3] = (float)(f * (x * y + z * w)); R[4] = (float)(1.0 - f * (x * x + z * z)); R[5] = (float)(f * (y * z - x * w));
        R[6] = (float)(f * (x * z - y * w)); R[7] = (float)(f * (y * z + x * w)); R[8] = (float)(1.0 - f * (x * x + y * y));
        float bx[6];
        box_f(ob, ob + 3, bx);
        for (int k = 0; k < 3; ++k) {
            const double lo = bx[k], hi = bx[3 + k], c = 0.5 * (lo + hi), t = st[k] - c;
            o.t[s][k] = (float)t;
            // 1e-5 for the roundings to float, a float step of the box (1.2e-7
            // of the coordinate) and the vertices' own rounding (some 1e-16 of
            // the position)
            o.H[s][k] = __double2float_ru(0.5 * (hi - lo) * (1.0 + 1e-5) + 1e-5 * fabs(t) +
                                          2.4e-7 * fmax(fabs(lo), fabs(hi)) + 1e-12 * fabs(st[k]) + 1e-38);
            o.th[s][k] = nextafterf(bx[k], -INFINITY);
            o.th[s][3 + k] = nextafterf(bx[3 + k], INFINITY);
        }
    }
    o.nondegA = B.nondeg[b[0]];
    for (int k = 0; k < 10; ++k) o.pad[k] = 0;
}
// An item's words, word l in lane l: one load per wave; fields are read
// uniformly over the wave.
static_assert(sizeof(PairItem) == WAVE * 4, "a work item is 64 words");
struct PairView {
    int word;
    __device__ int i(int k) const { return __builtin_amdgcn_readlane(word, k); }
    __device__ float f(int k) const { return __int_as_float(i(k)); }
    static constexpr int P_ = 0, ND = 1, T = 2, WO = 4, NC = 6, CO = 8, SO = 10, R = 12, TT = 30, H = 36, TH = 42;
    // the pair's results, by one lane
    __device__ void put(const DPairs& P, int64_t base, int hits, int64_t tests) const {
        const int p = i(P_), ta = i(T), tb = i(T + 1), nd = i(ND);
        if (lane_id() == 0) {
            P.hit_off[p] = base;
            P.tri_hits[p] = hits;
            P.tri_checks[p] = (int64_t)nd * tb;
            P.tri_tests[p] = tests;
            P.tri_scanned[p] = ta + tb;
            P.nseg[p] = 0;      // counted by the exact tests
        }
    }
};
__device__ inline int pair_word(const DPairs& P, int item) { return ((const int*)(P.pitems + item))[lane_id()]; }

// Geometry of one side, in uniform registers.
struct SideView {
    const Cluster* cl;
    const float* sph;
    const double* wv;
    float R[9], t[3], H[3];
    double lo[3], hi[3];
    __device__ SideView(const PairView& c, const DMeshes& M, const DBodies& B, int s) {
        cl = M.clusters + c.i(PairView::CO + s);
        sph = M.clus_sph + 4 * (int64_t)c.i(PairView::SO + s);
        wv = B.wv + 3 * (int64_t)c.i(PairView::WO + s);
#pragma unroll
        for (int k = 0; k < 9; ++k) R[k] = c.f(PairView::R + 9 * s + k);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            t[k] = c.f(PairView::TT + 3 * s + k);
            H[k] = c.f(PairView::H + 3 * s + k);
            lo[k] = (double)c.f(PairView::TH + 6 * s + k);
            hi[k] = (double)c.f(PairView::TH + 6 * s + 3 + k);
        }
    }
    __device__ bool meets(int k) const { return cluster_meets(R, t, H, sph + 4 * (int64_t)k); }
};
// One cluster per CT lanes: lane l holds vertex and triangle l % CT of its
// cluster.  A wave so reads about 15 vertices, nearly consecutive in memory,
// per 16 triangles, and takes a triangle's corners' outcodes from the lanes
// that hold them.
struct CLoad { double x[3]; uint32_t t; int v; };
__device__ inline CLoad load_cluster(const SideView& s, int k, bool on) {
    CLoad c;
    c.t = CLUS_NONE << 16;
    c.v = 0;
    c.x[0] = c.x[1] = c.x[2] = 0.0;
    if (on) {
        const int l = lane_id() % CT;
        c.v = s.cl[k].v[l];
        c.t = s.cl[k].t[l];
        const double* p = s.wv + 3 * c.v;
        c.x[0] = p[0]; c.x[1] = p[1]; c.x[2] = p[2];
    }
    return c;
}
// whether the lane's triangle is kept, and its corners
__device__ inline bool cluster_tri(const SideView& s, const CLoad& c, TriQ& q) {
    unsigned oc = 0;
#pragma unroll
    for (int k = 0; k < 3; ++k) oc |= ((unsigned)(c.x[k] <= s.lo[k]) << (2 * k)) | ((unsigned)(c.x[k] >= s.hi[k]) << (2 * k + 1));
    // outcode and vertex in one word: one fetch per corner
    const int w = (int)((oc << 16) | (unsigned)c.v);
    const int base = lane_id() & ~(CT - 1);
    const int w0 = __shfl(w, base + (int)(c.t & 15u), WAVE), w1 = __shfl(w, base + (int)((c.t >> 4) & 15u), WAVE),
              w2 = __shfl(w, base + (int)((c.t >> 8) & 15u), WAVE);
    q.a = (uint16_t)w0; q.b = (uint16_t)w1; q.c = (uint16_t)w2;
    q.id = (uint16_t)(c.t >> 16);
    return (((unsigned)(w0 & w1 & w2) >> 16) == 0u) & ((c.t >> 16) != CLUS_NONE);
}
// outward-rounded float box of a kept triangle; a bound that is no number is
// past every other, as the box test takes it, so that the boxes of groups hold it
__device__ inline void kept_box(const double* wv, TriQ q, float* box) {
    V3 t[3] = {ld3(wv + 3 * (int)q.a), ld3(wv + 3 * (int)q.b), ld3(wv + 3 * (int)q.c)};
    double lo[3], hi[3];
    tri_box(t, lo, hi);
    box_f(lo, hi, box);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        box[k] = fmaxf(box[k], -INFINITY);
        box[3 + k] = fminf(box[3 + k], INFINITY);
    }
}

// boxes in LDS are read two floats at a time
struct F2 { float x, y; };
__device__ inline void ld_box(const float* p, float* b) {
    const F2* q = (const F2*)p;
    const F2 u = q[0], v = q[1], w = q[2];
    b[0] = u.x; b[1] = u.y; b[2] = v.x; b[3] = v.y; b[4] = w.x; b[5] = w.y;
}
// The boxes of the groups: A's kept triangles at bx + 6 k, B's at bx + 6 (cap
// - 1 - k); thread `first` of `stride`.
__device__ inline void group_boxes(const float* bx, float* gx, int cap, int nA, int nB, int first, int stride) {
    const int gA = (nA + GT - 1) / GT, gB = (nB + GT - 1) / GT;
    for (int g = first; g < gA + gB; g += stride) {
        const bool a = g < gA;
        const int k0 = GT * (a ? g : g - gA), n = (a ? nA : nB) - k0;
        const float* p = bx + 6 * (a ? k0 : cap - 1 - k0);
        float o[6];
        ld_box(p, o);
        for (int k = 1; k < (n < GT ? n : GT); ++k) {
            float b[6];
            ld_box(p + (a ? 6 * k : -6 * k), b);
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                if (b[c] < o[c]) o[c] = b[c];
                if (o[3 + c] < b[3 + c]) o[3 + c] = b[3 + c];
            }
        }
#pragma unroll
        for (int c = 0; c < 6; ++c) gx[6 * g + c] = o[c];
    }
}
// The box tests of wave w of nw: its share of the group pairs (every nw-th, so
// that the waves' shares are alike), 64 at a time, and the GT x GT triangles of
// each that meets, two at a time: f(hit, a, b, mask) for each, by the whole
// wave.
template <class F>
__device__ inline void sweep_groups(const float* bx, const float* gx, int cap, int nA, int nB, int w, int nw, F&& f) {
    const int lane = lane_id();
    const int gA = (nA + GT - 1) / GT, gB = (nB + GT - 1) / GT, total = gA * gB;
    auto test = [&](int a, int b) {
        bool hit = false;
        if (a < nA && b < nB) {
            float fa[6], fb[6];
            ld_box(bx + 6 * a, fa);
            ld_box(bx + 6 * (cap - 1 - b), fb);
            hit = ovl_f(fa, fb);
        }
        return hit;
    };
    for (int t0 = 0; t0 < total; t0 += WAVE * nw) {
        const int t = t0 + lane * nw + w;
        const int ga = (int)((unsigned)t / (unsigned)gB), gb = t - ga * gB;
        bool meet = false;
        if (t < total) {
            float fa[6], fb[6];
            ld_box(gx + 6 * ga, fa);
            ld_box(gx + 6 * (gA + gb), fb);
            meet = ovl_f(fa, fb);
        }
        const int gab = ga | (gb << 16);
        for (uint64_t m = __ballot(meet); m;) {
            const int l0 = __builtin_ctzll(m);
            m &= m - 1;
            const int l1 = m ? __builtin_ctzll(m) : l0;
            const bool two = m != 0ull;
            m &= m - 1;
            const int g0 = __builtin_amdgcn_readlane(gab, l0), g1 = __builtin_amdgcn_readlane(gab, l1);
            const int a0 = GT * (g0 & 0xffff) + lane / GT, b0 = GT * (g0 >> 16) + lane % GT;
            const int a1 = GT * (g1 & 0xffff) + lane / GT, b1 = GT * (g1 >> 16) + lane % GT;
            const bool h0 = test(a0, b0), h1 = test(a1, b1) & two;
            f(h0, a0, b0, __ballot(h0));
            f(h1, a1, b1, __ballot(h1));
        }
    }
}
// the hit record of two kept triangles
__device__ inline void put_hit(const DPairs& P, int64_t at, const TriQ& a, const TriQ& b, int woA, int woB, int p) {
    int4* o = (int4*)((PairHit*)P.hits + at);
    o[0] = make_int4(woA + a.a, woA + a.b, woA + a.c, woB + b.a);
    o[1] = make_int4(woB + b.b, woB + b.c, (int)(((unsigned)a.id << 16) | (unsigned)b.id), p);
}

// One wave per pair.  Work items as k_narrow_wave takes them, each loaded
// while the one before it is worked on; a pair beyond the wave's limits
// (clusters, kept triangles, heavy_tests box tests, hits) goes to hlist for
// k_pairs_group, which writes all of that pair's results.
__global__ void __launch_bounds__(NWV * WAVE, CW_WPS) k_pairs_wave(DBodies B, DMeshes M, DPairs P, int32_t* hlist,
                                                             unsigned int* queue, int32_t use_queue,
                                                             int32_t heavy_tests, unsigned long long* stamp) {
    stamp_here(stamp);
    ZDX_DYN_LDS(s_nb);
    const int lane = lane_id();
    const int w = threadIdx.x / WAVE;
    char* sl = s_nb + w * CW_SLICE;
    uint16_t* cl = (uint16_t*)sl;
    uint32_t* hb = (uint32_t*)sl;
    float* bx = (float*)(sl + CW_HEAD);
    TriQ* ix = (TriQ*)(bx + 6 * CW_KEPT);
    float* gx = (float*)(ix + CW_KEPT);
    const uint64_t below = (1ull << lane) - 1ull;
    const int npairs = *P.n;
    const int nw = (int)gridDim.x * NWV;
    const int gw = (int)blockIdx.x * NWV + w;
    const int nq = nw < WQ ? nw : WQ;
    const int wq = gw % nq;
    auto take = [&](int round) {
        int it = 0;
        if (use_queue) {
            if (lane == 0) it = wq + nq * (int)atomicAdd(queue + wq * QSTRIDE, 1u);
        } else {
            it = round * nw + ((round & 1) ? nw - 1 - gw : gw);
        }
        return it;
    };
    int round = 0;
    int item = uni(__shfl(take(0), 0, WAVE));
    PairView c{item < npairs ? pair_word(P, item) : 0};
    while (item < npairs) {
        ++round;
        const int next = take(round);
        // ---- 1. each side's clusters, then their triangles, four rounds of
        // four clusters in flight
        bool heavy = false, front = false;
        int n[2] = {0, 0};
#pragma unroll 1
        for (int s = 0; s < 2; ++s) {
            const SideView v(c, M, B, s);
            const int nc = c.i(PairView::NC + s);
            int ncl = 0;
            for (int k0 = 0; k0 < nc; k0 += WAVE) {
                const int k = k0 + lane;
                const bool in = v.meets(k < nc ? k : nc - 1) & (k < nc);
                const uint64_t m = __ballot(in);
                const int r = ncl + __popcll(m & below);
                if (in && r < CW_CLUS) cl[r] = (uint16_t)k;
                ncl += __popcll(m);
            }
            heavy = front = front || ncl > CW_CLUS;
            ncl = ncl < CW_CLUS ? ncl : CW_CLUS;
            wave_sync();
            constexpr int PER = WAVE / CT, U = 4;
            int nk = 0;
            for (int k0 = 0; k0 < ncl; k0 += U * PER) {
                CLoad cu[U];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int e = k0 + u * PER + lane / CT;
                    cu[u] = load_cluster(v, e < ncl ? (int)cl[e] : 0, e < ncl);
                }
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    TriQ q;
                    const bool keep = cluster_tri(v, cu[u], q);
                    const uint64_t m = __ballot(keep);
                    const int r = nk + __popcll(m & below);
                    if (keep && r < CW_KEPT) ix[s ? CW_KEPT - 1 - r : r] = q;
                    nk += __popcll(m);
                }
            }
            if (s) n[1] = nk; else n[0] = nk;
            wave_sync();   // the cluster list is rewritten
        }
        // the next item, in flight from here on
        const int nitem = uni(__shfl(next, 0, WAVE));
        const int nword = nitem < npairs ? pair_word(P, nitem) : 0;
        const int nA = n[0], nB = n[1];
        const int64_t tests = (int64_t)nA * nB;
        heavy = heavy || nA + nB > CW_KEPT || tests > heavy_tests;
        const int woA = c.i(PairView::WO), woB = c.i(PairView::WO + 1), pair = c.i(PairView::P_);
        int hits = 0;
        if (!heavy && tests > 0) {
            // ---- 2. boxes, groups, hits
            for (int k = lane; k < nA + nB; k += WAVE) {
                const bool a = k < nA;
                const int at = a ? k : CW_KEPT - 1 - (k - nA);
                kept_box(B.wv + 3 * (int64_t)(a ? woA : woB), ix[at], bx + 6 * at);
            }
            wave_sync();
            group_boxes(bx, gx, CW_KEPT, nA, nB, lane, WAVE);
            wave_sync();
            sweep_groups(bx, gx, CW_KEPT, nA, nB, 0, 1, [&](bool hit, int a, int b, uint64_t m) {
                const int r = hits + __popcll(m & below);
                if (hit && r < CW_HITS) hb[r] = (uint32_t)a | ((uint32_t)b << 16);
                hits += __popcll(m);
            });
            heavy = hits > CW_HITS;
        }
        if (heavy) {
            if (lane == 0) {
                if (front || nA + nB > CW_FRONT) hlist[atomicAdd(queue + NQ_HEAVY, 1u)] = item;
                else hlist[npairs - 1 - (int)atomicAdd(queue + NQ_HEAVY_BACK, 1u)] = item;
            }
        } else {
            unsigned long long base = 0;
            if (hits > 0) {
                if (lane == 0) base = reserve_hits(P, item, hits);
                base = __shfl(base, 0, WAVE);
                wave_sync();
                if (base != ~0ull) {
                    for (int k = lane; k < hits; k += WAVE) {
                        const uint32_t ab = hb[k];
                        put_hit(P, (int64_t)base + k, ix[ab & 0xffffu], ix[CW_KEPT - 1 - (int)(ab >> 16)], woA, woB,
                                pair);
                    }
                } else {
                    hits = 0;
                    base = 0;
                }
            }
            c.put(P, (int64_t)base, hits, tests);
        }
        wave_sync();   // the wave's LDS is rewritten by the next item
        item = nitem;
        c.word = nword;
    }
}

// One workgroup per pair, of the list's front (*count entries from its start),
// of its back (from its end) or, without a list, of all *count work items; the
// same work spread over its waves.  The kept triangles are taken a batch at a
// time, as many of A's and then of B's as the LDS holds.  Each wave
// keeps its hits in LDS; when they fit and there is one batch (nearly always),
// they are written from there, else the box tests run again with the hits'
// slots reserved.
template <int BS>
__global__ void __launch_bounds__(BS, 4) k_pairs_group(DBodies B, DMeshes M, DPairs P, int32_t use_queue,
                                                      unsigned int* queue, const int32_t* hlist,
                                                      const int32_t* count, int32_t back,
                                                      unsigned long long* stamp) {
    stamp_here(stamp);
    constexpr int NW = BS / WAVE, KC = group_kept(BS), PER = WAVE / CT, HB = group_hits(BS);
    ZDX_DYN_LDS(s_nb);
    uint32_t* s_cl = (uint32_t*)s_nb;      // clusters of a range that meet, ascending
    uint32_t* s_hb = s_cl + BS;            // per wave its hits
    float* s_bx = (float*)(s_hb + NW * HB);
    TriQ* s_ix = (TriQ*)(s_bx + 6 * KC);
    float* s_gx = (float*)(s_ix + KC);
    __shared__ int s_wc[NW];
    __shared__ int s_next, s_n, s_hits;
    __shared__ unsigned long long s_base;
    const int tid = threadIdx.x, lane = lane_id(), wid = tid / WAVE;
    const uint64_t below = (1ull << lane) - 1ull;
    uint32_t* hb = s_hb + HB * wid;
    const int nq = *count, hend = *P.n - 1;
    // exclusive prefix of a count per wave (the same in all its lanes), and the
    // total; ends with a barrier pending on s_wc
    auto wave_prefix = [&](int n, int& total) {
        if (lane == 0) s_wc[wid] = n;
        __syncthreads();
        int o = 0, t = 0;
#pragma unroll
        for (int q = 0; q < NW; ++q) {
            const int x = s_wc[q];
            o += q < wid ? x : 0;
            t += x;
        }
        total = uni(t);
        return o;
    };
    if (tid == 0) s_next = use_queue ? (int)atomicAdd(queue, 1u) : (int)blockIdx.x;
    __syncthreads();
    int qi = uni(s_next);
    while (qi < nq) {
        int next = 0;
        if (tid == 0) next = use_queue ? (int)atomicAdd(queue, 1u) : qi + (int)gridDim.x;
        const int item = uni(!hlist ? qi : hlist[back ? hend - qi : qi]);
        const PairView c{pair_word(P, item)};
        const int nc[2] = {c.i(PairView::NC), c.i(PairView::NC + 1)};
        const int woA = c.i(PairView::WO), woB = c.i(PairView::WO + 1), pair = c.i(PairView::P_);
        if (tid == 0) s_hits = 0;
        int k2[2] = {0, 0};                    // the next cluster of A and of B
        int nA = 0, nB = 0, boxed = 0, batches = 0, hits = 0;
        int64_t totA = 0, totB = 0;
        unsigned long long base = 0;
        int s = 0;
        bool firstB = true, write = false;
        for (;;) {
            // ---- 1. a batch of side s: its clusters from k on, BS of them at a
            // time, until they end or the room does
            {
                const SideView v(c, M, B, s);
                const int end = s ? nc[1] : nc[0], room = s ? KC - nA : KC - NW * WAVE;
                int k = s ? k2[1] : k2[0], n = 0;
                bool full = false;
                if (tid == 0) s_n = 0;
                while (k < end && !full) {
                    const int r1 = k + BS < end ? k + BS : end;
                    const bool in = v.meets(k + tid < r1 ? k + tid : k) & (k + tid < r1);
                    const uint64_t m = __ballot(in);
                    int ncl;
                    const int o = wave_prefix(__popcll(m), ncl) + __popcll(m & below);
                    if (in) s_cl[o] = (uint32_t)(k + tid);
                    __syncthreads();
                    // up to U rounds of PER clusters per wave in flight while
                    // they are sure to fit, else one
                    constexpr int U = 4;
                    for (int done = 0, step; done < ncl; done += step) {
                        step = NW * PER * U;
                        if (n + (ncl - done < step ? ncl - done : step) * CT > room) step = NW * PER;
                        if (n + (ncl - done < step ? ncl - done : step) * CT > room) {
                            full = true;
                            k = uni((int)s_cl[done]);
                            break;
                        }
                        CLoad cu[U];
#pragma unroll
                        for (int u = 0; u < U; ++u) {
                            const int e = done + (u * NW + wid) * PER + lane / CT;
                            const bool on = e < ncl && u * NW * PER < step;
                            cu[u] = load_cluster(v, on ? (int)s_cl[e] : 0, on);
                        }
#pragma unroll
                        for (int u = 0; u < U; ++u) {
                            TriQ q;
                            const bool keep = cluster_tri(v, cu[u], q);
                            const uint64_t mk = __ballot(keep);
                            int r = 0;
                            if (lane == 0 && mk) r = atomicAdd(&s_n, __popcll(mk));
                            r = __shfl(r, 0, WAVE) + __popcll(mk & below);
                            if (keep) s_ix[s ? KC - 1 - r : r] = q;
                        }
                        __syncthreads();
                        n = uni(s_n);
                        __syncthreads();
                    }
                    if (!full) k = r1;
                }
                if (s == 0) {
                    nA = n;
                    boxed = 0;
                    k2[0] = k;
                    if (!write) totA += n;
                    s = 1;
                    // without A's there is nothing to do unless B is still to be counted
                    k2[1] = n > 0 || firstB ? 0 : nc[1];
                    __syncthreads();
                    if (k2[1] < nc[1]) continue;
                    nB = 0;
                } else {
                    nB = n;
                    k2[1] = k;
                    if (!write && firstB) totB += n;
                    __syncthreads();
                }
            }
            // the boxes of this batch (A's once)
            if (nA > 0 && nB > 0) {
                for (int q = boxed + tid; q < nA + nB; q += BS) {
                    const bool a = q < nA;
                    const int at = a ? q : KC - 1 - (q - nA);
                    kept_box(B.wv + 3 * (int64_t)(a ? woA : woB), s_ix[at], s_bx + 6 * at);
                }
                boxed = nA;
                __syncthreads();
                group_boxes(s_bx, s_gx, KC, nA, nB, tid, BS);
            }
            __syncthreads();
            ++batches;
            // ---- 2. the box tests: count and keep the hits, or write them
            int at = 0;
            if (nA > 0 && nB > 0)
                sweep_groups(s_bx, s_gx, KC, nA, nB, wid, NW, [&](bool hit, int a, int b, uint64_t m) {
                    if (!write) {
                        const int r = at + __popcll(m & below);
                        if (hit && r < HB) hb[r] = (uint32_t)a | ((uint32_t)b << 16);
                        at += __popcll(m);
                    } else if (m) {
                        int r = 0;
                        if (lane == 0) r = atomicAdd(&s_hits, __popcll(m));
                        r = __shfl(r, 0, WAVE) + __popcll(m & below);
                        if (hit) put_hit(P, (int64_t)base + r, s_ix[a], s_ix[KC - 1 - b], woA, woB, pair);
                    }
                });
            const bool last = k2[1] >= nc[1] && k2[0] >= nc[0];
            if (!write) {
                int total;
                const int mine = wave_prefix(at, total);
                hits += total;
                __syncthreads();
                int spill;
                (void)wave_prefix(at > HB ? 1 : 0, spill);
                if (last && batches == 1 && spill == 0) {
                    if (tid == 0) s_base = reserve_hits(P, item, hits);
                    __syncthreads();
                    base = s_base;
                    if (base != ~0ull)
                        for (int q = lane; q < at; q += WAVE) {
                            const uint32_t ab = hb[q];
                            put_hit(P, (int64_t)base + mine + q, s_ix[ab & 0xffffu], s_ix[KC - 1 - (int)(ab >> 16)], woA,
                                    woB, pair);
                        }
                    break;
                }
            }
            __syncthreads();   // the kept triangles are rewritten
            if (k2[1] < nc[1]) continue;   // more of B against this batch of A
            firstB = false;
            s = 0;
            if (!last) continue;
            if (write) break;
            // several batches, or more hits than a wave keeps: again, with
            // their slots
            if (tid == 0) s_base = reserve_hits(P, item, hits);
            __syncthreads();
            base = s_base;
            if (base == ~0ull || hits == 0) break;
            write = true;
            k2[0] = k2[1] = 0;
        }
        if (base == ~0ull) { base = 0; hits = 0; }
        if (wid == 0) c.put(P, (int64_t)base, hits, totA * totB);
        if (tid == 0) s_next = next;
        __syncthreads();
        qi = uni(s_next);
    }
}

// The reference's exact test of one hit (src/main.cpp:2130-2145): the AABB
// reject, both planes, the triangle-triangle intersection.
template <bool PROV>
__device__ inline bool exact_hit(const double* wv, const PairHit& h, V3& p0, V3& p1, int& c0, int& c1) {
    V3 A[3] = {ld3(wv + 3 * (int64_t)h.v[0]), ld3(wv + 3 * (int64_t)h.v[1]), ld3(wv + 3 * (int64_t)h.v[2])};
    V3 Bt[3] = {ld3(wv + 3 * (int64_t)h.v[3]), ld3(wv + 3 * (int64_t)h.v[4]), ld3(wv + 3 * (int64_t)h.v[5])};
    double alo[3], ahi[3], blo[3], bhi[3];
    tri_box(A, alo, ahi);
    tri_box(Bt, blo, bhi);
    if (ahi[0] < blo[0] || alo[0] > bhi[0] || ahi[1] < blo[1] || alo[1] > bhi[1] || ahi[2] < blo[2] || alo[2] > bhi[2])
        return false;
    V3 nA, nB;
    double dA, dB;
    plane_of(A[0], A[1], A[2], nA, dA);
    plane_of(Bt[0], Bt[1], Bt[2], nB, dB);
    if (PROV) return tri_tri_prov(A, nA, dA, Bt, nB, dB, p0, p1, c0, c1);
    return tri_tri(A, nA, dA, Bt, nB, dB, p0, p1);
}
// The exact tests, one thread per hit of the arena.  A pair's segments go to
// its range of seg_tmp in the order they come (nseg counts them), with their
// keys (hit_flag) and, in sensitivity runs, the endpoints' codes (hit_tri).
template <bool PROV>
__global__ void __launch_bounds__(256) k_pairs_exact(DBodies B, DPairs P) {
    // the used prefix of every shard: the slot of linear index i is found in
    // the prefix sums of the shards' counts (after an overflow part of the
    // arena was never written: nothing is tested, the step is run again)
    static_assert(HIT_SHARDS == WAVE, "one lane per shard");
    __shared__ long long s_pre[HIT_SHARDS + 1];
    const int64_t size = P.hit_cap / P.hit_shards;
    if (threadIdx.x < WAVE) {
        const int l = threadIdx.x;
        long long x = 0;
        if (l < P.hit_shards) {
            const long long t = (long long)P.hit_top[l * HIT_TOP_STRIDE];
            x = t < size ? t : size;
        }
#pragma unroll
        for (int d = 1; d < WAVE; d <<= 1) {
            const long long y = __shfl_up(x, d, WAVE);
            if (l >= d) x += y;
        }
        s_pre[l + 1] = x;
        if (l == 0) s_pre[0] = 0;
    }
    __syncthreads();
    const int64_t lim = (*P.status & (int)ST_HITS) ? 0 : s_pre[HIT_SHARDS];
    for (int64_t i0 = blockIdx.x * (int64_t)blockDim.x + (threadIdx.x & ~(WAVE - 1)); i0 < lim;
         i0 += (int64_t)gridDim.x * blockDim.x) {
        // the whole wave takes part; lanes past the end repeat the last hit
        const bool on = i0 + lane_id() < lim;
        const int64_t i = on ? i0 + lane_id() : lim - 1;
        int lo = 0, hi = HIT_SHARDS;   // s_pre[lo] <= i < s_pre[hi]
        while (hi - lo > 1) {
            const int mid = (lo + hi) / 2;
            if (s_pre[mid] <= i) lo = mid; else hi = mid;
        }
        const int4* r = (const int4*)((const PairHit*)P.hits + ((int64_t)lo * size + (i - s_pre[lo])));
        const int4 r0 = r[0], r1 = r[1];
        const PairHit h{{r0.x, r0.y, r0.z, r0.w, r1.x, r1.y}, (uint32_t)r1.z, r1.w};
        V3 p0, p1;
        int c0 = 0, c1 = 0;
        // the wave's segments of one pair at a time: one count per pair and wave
        const bool is = exact_hit<PROV>(B.wv, h, p0, p1, c0, c1) & on;
        int64_t at = 0;
        for (uint64_t m = __ballot(is); m;) {
            const int pair = __builtin_amdgcn_readlane(h.pair, __builtin_ctzll(m));
            const uint64_t same = __ballot(is & (h.pair == pair)) & m;
            int first = 0;
            if (lane_id() == __builtin_ctzll(same)) first = atomicAdd(&P.nseg[pair], __popcll(same));
            first = __builtin_amdgcn_readlane(first, __builtin_ctzll(same));
            if (is & (h.pair == pair)) at = P.hit_off[pair] + first + __popcll(same & ((1ull << lane_id()) - 1ull));
            m &= ~same;
        }
        if (is) {
            double* o = P.seg_tmp + 6 * at;
            o[0] = p0.x; o[1] = p0.y; o[2] = p0.z; o[3] = p1.x; o[4] = p1.y; o[5] = p1.z;
            P.hit_flag[at] = (int32_t)h.key;
            if (PROV) ((int2*)P.hit_tri)[at] = make_int2(c0, c1);
        }
    }
}

// pairs with at least this many segments are walked first (their walks are
// the longest, so they should not wait for a free workgroup)
constexpr int TOPO_BIG_SEGS = 40;

// The segments of every pair from seg_tmp to the arena in the order of their
// keys, and the topology's work lists: the pairs with stored segments in
// topo_list, and (with P.topo_big) their indices there in topo_big
// (TOPO_BIG_SEGS or more) or topo_small.  4 to 256 pairs per workgroup, as the
// grid needs: the lists take one atomic each per workgroup, then each wave
// takes the next pair that has segments.  A pair with more than seg_cap stores
// none (ST_STAGE).  S^2/64 steps of one wave a pair: 26 us for the bed's 1900
// pairs of up to 160 segments; a pair of 641 takes 0.29 ms of a call of 9.9.
template <bool PROV>
__global__ void __launch_bounds__(256) k_pairs_sort(DPairs P, int32_t seg_cap) {
    constexpr int NW = 256 / WAVE;
    __shared__ int s_cnt[3][NW], s_base[3], s_p[256], s_s[256];
    const int lane = lane_id(), wid = threadIdx.x / WAVE;
    const uint64_t below = (1ull << lane) - 1ull;
    const int npairs = (*P.status & (int)ST_HITS) ? 0 : *P.n;
    int per = (npairs + (int)gridDim.x - 1) / (int)gridDim.x;
    per = per < NW ? NW : (per > 256 ? 256 : per);
    for (int64_t p0 = blockIdx.x * (int64_t)per; p0 < npairs; p0 += gridDim.x * (int64_t)per) {
        const int p = (int)p0 + (int)threadIdx.x;
        const bool on = (int)threadIdx.x < per && p < npairs;
        int S = on ? P.nseg[p] : 0;
        if (on) P.seg_off[p] = P.hit_off[p];
        if (S > seg_cap) {
            atomicOr(P.status, (int)ST_STAGE);
            P.nseg[p] = 0;
            S = 0;
        }
        const uint64_t m0 = __ballot(S > 0), m1 = __ballot(S >= TOPO_BIG_SEGS), m2 = m0 & ~m1;
        if (lane == 0) { s_cnt[0][wid] = __popcll(m0); s_cnt[1][wid] = __popcll(m1); s_cnt[2][wid] = __popcll(m2); }
        __syncthreads();
        int before[3] = {0, 0, 0}, total = 0;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            total += s_cnt[0][w];
#pragma unroll
            for (int l = 0; l < 3; ++l) before[l] += w < wid ? s_cnt[l][w] : 0;
        }
        if (threadIdx.x < 3) {
            int t = 0;
#pragma unroll
            for (int w = 0; w < NW; ++w) t += s_cnt[threadIdx.x][w];
            int* counter = threadIdx.x == 0 ? P.topo_n : (threadIdx.x == 1 ? P.n_big : P.n_small);
            s_base[threadIdx.x] = t > 0 && counter ? atomicAdd(counter, t) : 0;
        }
        const int r = before[0] + __popcll(m0 & below);
        if (S > 0) { s_p[r] = p; s_s[r] = S; }
        __syncthreads();
        if (S > 0) {
            const int idx = s_base[0] + r;
            P.topo_list[idx] = p;
            if (P.topo_big) {
                if (S >= TOPO_BIG_SEGS) P.topo_big[s_base[1] + before[1] + __popcll(m1 & below)] = idx;
                else P.topo_small[s_base[2] + before[2] + __popcll(m2 & below)] = idx;
            }
        }
        for (int q = wid; q < total; q += NW) {
            const int n = uni(s_s[q]);
            const int64_t h0 = P.hit_off[uni(s_p[q])];
            const unsigned* keys = (const unsigned*)P.hit_flag + h0;
            for (int e0 = 0; e0 < n; e0 += WAVE) {
                const int e = e0 + lane;
                const unsigned key = e < n ? keys[e] : ~0u;
                double v[6];
                int2 cc = make_int2(0, 0);
                if (e < n) {
#pragma unroll
                    for (int d = 0; d < 6; ++d) v[d] = P.seg_tmp[6 * (h0 + e) + d];
                    if (PROV) cc = ((const int2*)P.hit_tri)[h0 + e];
                }
                int rank = 0;
                for (int f0 = 0; f0 < n; f0 += WAVE) {
                    const int fn = n - f0 < WAVE ? n - f0 : WAVE;
                    const int kf = f0 == e0 ? (int)key : (lane < fn ? (int)keys[f0 + lane] : -1);
                    for (int l = 0; l < fn; ++l) rank += (unsigned)__builtin_amdgcn_readlane(kf, l) < key ? 1 : 0;
                }
                if (e < n) {
                    double* o = P.arena + 6 * (h0 + rank);
#pragma unroll
                    for (int d = 0; d < 6; ++d) o[d] = v[d];
                    if (PROV) ((int4*)P.prov)[h0 + rank] = make_int4((int)(key >> 16), (int)(key & 0xffffu), cc.x, cc.y);
                }
            }
        }
        __syncthreads();   // the lists are rewritten
    }
}
