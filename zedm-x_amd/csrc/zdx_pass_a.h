// zdx_pass_a.h — pass A of the phased topology on the device: the adjacency
// rows and the snap hit words of every pair (zdx_topo.h has the tests).
//
// Textually included inside namespace zdx::{anonymous} after zdx_narrow.h and
// zdx_cluster.h: by zdx_kernels.hip for gfx950 and by the host SIMT emulation
// (tests/csrc/pass_a_emu.cpp).  No includes or namespaces of its own.
//
// Of the S x S segment pairs only a few per row pass.  A pair can pass the
// adjacency test only if the segments' boxes grown by the tolerance overlap
// (the test has that reject on the same boxes), and two endpoints within the
// tolerance of each other lie in both boxes; so each wave first runs through
// its rows' pairs on float copies of those boxes, rounded outward, and collects
// the pairs that overlap in LDS, and the cell and distance tests run on 64
// collected pairs at a time, every lane busy.
// What is left is the latency of a pair's few batches: 128 threads for a small
// pair and units of 8192 tests for a large one.  On an MI355X, 4096 pairs of
// about 80 segments: 660 us with every pair taking the full tests (into an LDS
// matrix of keys that one thread per row compacted, in 1024-thread workgroups),
// 190 us so.  The pairs of the 100k bed (1900 small ones, 200 of 40 to 160
// segments beside them, whose walks wait for it): 39 and 50 us before, 30 and
// 32 so, the larger pairs in workgroups of 1024 threads (of 256 they take 64 us,
// of 512 36: their 300 units leave the chip idle otherwise); one wave per small
// pair 47.

// Snap / adjacency tolerance of a pair: mesh A's (main.cpp:2118-2121) unless
// the caller of the per-pair API gave one.
__device__ inline double topo_tol(const TopoBufs& T, const DMeshes& M, int mesh_a) {
    return T.tol_override > 0.0 ? T.tol_override : M.tol[mesh_a];
}

constexpr int PA_THREADS = 256;       // threads per unit of the larger pairs
constexpr int PA_SEGS = 256;          // segments staged in LDS; a larger pair is read from memory
constexpr int PA_WORDS = 512;         // snap words a unit builds in LDS at a time
constexpr int PA_TESTS = 8192;        // segment-pair tests per unit (sets the units of a big pair)
constexpr int PA_BIG_THREADS = 1024;  // where those are the few larger pairs of a step
constexpr int PA_SMALL_THREADS = 128; // threads per pair of fewer than TOPO_BIG_SEGS segments
constexpr int PA_SMALL_WORDS = 64;    // snap words of a pair of fewer than TOPO_BIG_SEGS segments
static_assert((TOPO_BIG_SEGS - 1) * (2 * TOPO_BIG_SEGS - 3) <= 64 * PA_SMALL_WORDS, "a small pair's words");
__host__ __device__ constexpr int pass_a_lds_bytes(int threads, int words, int segs) {
    return 8 * words + 16 * threads + 108 * segs + 4 * (segs & 1);
}

// Units of pass A for a pair of S segments: enough that each unit has at most
// PA_TESTS candidate tests (rows x S) and PA_WORDS snap words, and at least one
// row.
__device__ inline int tp_pa_units(int S) {
    const int64_t npt = (int64_t)S * (2 * S - 1);
    const int64_t nw = (npt + 63) >> 6;
    int64_t m = ((int64_t)S * S + PA_TESTS - 1) / PA_TESTS;
    const int64_t mw = (nw + PA_WORDS - 1) / PA_WORDS;
    if (mw > m) m = mw;
    if (m > S) m = S;
    return m < 1 ? 1 : (int)m;
}

// Unit b of nu of one pair, by a workgroup: a band of rows and a range of snap
// words.  STAGED: segments, cells and boxes in LDS (seg, c9, fb), else seg and
// c9 in memory and the boxes from the segments.
template <int NT, int WORDS, bool STAGED>
__device__ inline void pass_a_unit(const double* seg, const int* c9, const float* fb, int2* list,
                                            unsigned long long* sw, int S, double h, int R, int b, int nu, int* cntp,
                                            uint64_t* w, unsigned long long* most) {
    constexpr int NW = NT / WAVE;
    const int tid = threadIdx.x, lane = lane_id(), wid = uni(tid / WAVE);
    const uint64_t below = (1ull << lane) - 1ull;
    int* rows = cntp + S;
    const int64_t npt = (int64_t)S * (2 * S - 1);   // endpoint pairs of 2S points: past 31 bits at 32769 segments
    const int nw = (int)((npt + 63) >> 6);
    auto meet = [&](int i, int j) {
        bool r = true;
        if (STAGED) {
            float fi[6], fj[6];
            ld_box(fb + 6 * i, fi);
            ld_box(fb + 6 * j, fj);
            r = ovl_f(fi, fj);
        } else {
            const double *a = seg + 6 * (int64_t)i, *c = seg + 6 * (int64_t)j;
#pragma unroll
            for (int k = 0; k < 3; ++k)
                r = r & !(dmax(a[k], a[3 + k]) + h < dmin(c[k], c[3 + k]) - h ||
                          dmin(a[k], a[3 + k]) - h > dmax(c[k], c[3 + k]) + h);
        }
        return r | (i == j);
    };
    // rows [ra, rb) by the workgroup's waves: their adjacency (adj), or only
    // j <= i; and the snap hits in words [c0, c1)
    auto sweep = [&](int ra, int rb, bool adj, int c0, int c1) {
        const int64_t tb = 64 * (int64_t)c0, te = 64 * (int64_t)c1 < npt ? 64 * (int64_t)c1 : npt;
        const int r0 = ra + (int)((int64_t)(rb - ra) * wid / NW), r1 = ra + (int)((int64_t)(rb - ra) * (wid + 1) / NW);
        int crow = -1, ccnt = 0;   // the row that the last tested pair belonged to, and its count so far
        auto test = [&](int n) {   // the first n <= WAVE pairs of the list
            const bool on = lane < n;
            const int2 e = list[on ? lane : 0];
            if (adj) {
                int key = TP_NOADJ;
                if (on) key = tp_adj_key(seg, c9, h, e.x, e.y);
                const bool hit = key != TP_NOADJ;
                const int prev = __shfl_up(e.x, 1, WAVE);
                const uint64_t acc = __ballot(hit);
                const uint64_t starts = __ballot(on & ((lane == 0) | (prev != e.x)));   // first lane of each row
                const uint64_t mine = ~0ull << (63 - __builtin_clzll(starts & (below | (1ull << lane))));
                const int at = (e.x == crow ? ccnt : 0) + __popcll(acc & below & mine);
                if (hit && at < R) rows[(int64_t)e.x * R + at] = e.y | (key << 24);
                const int cnt = at + (hit ? 1 : 0);
                // the row's last lane here: a later batch of the same row, by
                // this wave, stores over it
                if (on && (lane == n - 1 || ((starts >> lane) >> 1 & 1ull))) {
                    cntp[e.x] = cnt;
                    if (cnt > R) atomicMax(most, (unsigned long long)cnt);
                }
                crow = __builtin_amdgcn_readlane(e.x, n - 1);
                ccnt = __builtin_amdgcn_readlane(cnt, n - 1);
            }
            if (on && e.y <= e.x && c1 > c0) {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int a = 2 * e.x + (q >> 1), c = 2 * e.y + (q & 1);
                    const int64_t t = (int64_t)a * (a - 1) / 2 + c;   // a (a - 1): past 31 bits at 23171 segments
                    if (c < a && t >= tb && t < te && tp_snap_hit(seg, c9, h, a, c))
                        atomicOr(&sw[(t >> 6) - c0], 1ull << (t & 63));
                }
            }
        };
        // pairs (i, j) in row order, 64 at a time
        const int di = WAVE / S, dj = WAVE - di * S;
        int i = r0 + lane / S, j = lane - lane / S * S, n = 0;
        for (int k = 0, total = (r1 - r0) * S; k < total; k += WAVE) {
            bool on = (i < r1) & (adj | (j <= i));
            if (on) on = meet(i, j);
            const uint64_t m = __ballot(on);
            if (on) list[n + __popcll(m & below)] = make_int2(i, j);
            n += __popcll(m);
            wave_sync();
            if (n >= WAVE) {
                test(WAVE);
                n -= WAVE;
                wave_sync();
                const int2 rest = list[WAVE + (lane < n ? lane : 0)];
                wave_sync();
                if (lane < n) list[lane] = rest;
                wave_sync();
            }
            i += di;
            j += dj;
            if (j >= S) {
                j -= S;
                ++i;
            }
        }
        if (n > 0) test(n);
        wave_sync();   // the list is rewritten
    };
    const int r0 = (int)((int64_t)b * S / nu), r1 = (int)((int64_t)(b + 1) * S / nu);
    const int w0 = (int)((int64_t)b * nw / nu), w1 = (int)((int64_t)(b + 1) * nw / nu);
    if (nu > 1) sweep(r0, r1, true, 0, 0);
    for (int c0 = w0; c0 < w1; c0 += WORDS) {
        const int c1 = c0 + WORDS < w1 ? c0 + WORDS : w1;
        for (int k = tid; k < c1 - c0; k += NT) sw[k] = 0ull;
        // the segments i of the points a of the words' endpoint pairs
        int ra = 0, rb = S;
        if (nu > 1) {
            int a0, a1, x;
            tp_pair_of(64 * (int64_t)c0, a0, x);
            tp_pair_of((64 * (int64_t)c1 < npt ? 64 * (int64_t)c1 : npt) - 1, a1, x);
            ra = a0 >> 1;
            rb = (a1 >> 1) + 1;
        }
        __syncthreads();
        sweep(ra, rb, nu == 1, c0, c1);
        __syncthreads();
        for (int k = tid; k < c1 - c0; k += NT) w[c0 + k] = sw[k];
        __syncthreads();
    }
}

// One workgroup per unit: unit 0 of every item, then the extra units of the big
// pairs.  MODE 0: every item and every extra unit; MODE 1: the items of
// P.topo_small only (fewer than TOPO_BIG_SEGS segments, so one unit each); MODE 2: the items of P.topo_big and every extra unit.  lds_segs:
// segments that the launch's LDS holds.
template <int NT, int WORDS, int MODE>
__global__ void __launch_bounds__(NT, 4) k_tp_pass_a(DPairs P, DMeshes M, DBodies B, TopoBufs T, int32_t lds_segs) {
    ZDX_DYN_LDS(s_nb);
    unsigned long long* sw = (unsigned long long*)s_nb;
    int2* list = (int2*)(sw + WORDS) + 2 * WAVE * (threadIdx.x / WAVE);
    double* s_seg = (double*)((int2*)(sw + WORDS) + 2 * NT);
    int* s_c9 = (int*)(s_seg + 6 * (int64_t)lds_segs);
    float* s_fb = (float*)(s_c9 + 9 * (int64_t)lds_segs + (lds_segs & 1));
    const int n = MODE == 0 ? *P.topo_n : (MODE == 1 ? *P.n_small : *P.n_big);
    const int nunits = n + (MODE == 1 ? 0 : (int)*(T.top + 4));
    const int tid = threadIdx.x;
    for (int u = blockIdx.x; u < nunits; u += gridDim.x) {
        int it = MODE == 0 ? u : (u < n ? (MODE == 1 ? P.topo_small[u] : P.topo_big[u]) : 0), b = 0;
        if (u >= n) {
            if (u - n >= T.units_cap) continue;
            const int2 e = ((const int2*)T.units)[u - n];
            it = e.x;
            b = e.y;
            // k_tp_alloc wrote every slot below units_cap this step; this only
            // guards against a slot it did not write
            if (it < 0 || it >= *P.topo_n || b < 1) continue;
        }
        const long long ao = T.adj_off[it], so = T.snap_off[it];
        if (ao < 0) continue;
        const int p = P.topo_list[it];
        const int S = uni(P.nseg[p]);
        const int nu = tp_pa_units(S);
        if (b >= nu) continue;
        const int64_t sb = P.seg_off[p];
        const double h = topo_tol(T, M, B.mesh[P.pi[p]]);
        const double* gseg = P.arena + 6 * sb;
        int* cntp = T.adj + ao;
        uint64_t* w = T.snapw + so;
#ifdef ZDX_WALK_PROFILE
        const unsigned long long t0 = wall_clock64();
#endif
        __syncthreads();   // the last unit's LDS is rewritten
        if (MODE == 1 || S <= lds_segs) {
            for (int k = tid; k < 6 * S; k += NT) s_seg[k] = gseg[k];
            __syncthreads();
            for (int k = tid; k < S; k += NT) {
                tp_cells(s_seg, k, h, s_c9 + 9 * k);
                const double* q = s_seg + 6 * k;
                double lo[3], hi[3];
#pragma unroll
                for (int d = 0; d < 3; ++d) {
                    lo[d] = dmin(q[d], q[3 + d]) - h;
                    hi[d] = dmax(q[d], q[3 + d]) + h;
                }
                box_f(lo, hi, s_fb + 6 * k);
            }
            __syncthreads();
            pass_a_unit<NT, WORDS, true>(s_seg, s_c9, s_fb, list, sw, S, h, T.adj_row, b, nu, cntp, w, T.top + 3);
        } else {
            // every unit of the pair writes the same cells
            int* gc9 = T.cell9 + 9 * sb;
            for (int k = tid; k < S; k += NT) tp_cells(gseg, k, h, gc9 + 9 * (int64_t)k);
            __syncthreads();
            pass_a_unit<NT, WORDS, false>(gseg, gc9, nullptr, list, sw, S, h, T.adj_row, b, nu, cntp, w, T.top + 3);
        }
#ifdef ZDX_WALK_PROFILE
        if (tid == 0 && it < 8192 && b == 0) {
            g_topo_pairs[4 * it] = S;
            g_topo_pairs[4 * it + 1] = (long long)(wall_clock64() - t0);
        }
#endif
    }
}
