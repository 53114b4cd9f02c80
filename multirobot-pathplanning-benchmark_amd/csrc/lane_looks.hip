// lane_looks.hip — batches of plane edges (scenes with a cell table) without a queue (gfx950).
//
// A cell look-up costs a few dozen instructions, so most of a batch's time went into feeding the
// pass-ordered queue: five launches, the rows read and the steps written and read again, and four
// dependent round trips per slot.  Here a wave owns 1..16 edges from rows to verdict:
//   rows   : its edges' rows in one coalesced round into LDS; N, window and steps from there
//   look   : 64 / edges evenly spread states per edge by the cell table alone; most colliding edges
//            end here
//   rounds : the edges left, in groups of 16, 32 or 64 lanes by their state count, every state by
//            the full evaluator; long edges 64 spread states a round, in the binary order of rounds
// Edges of more than LOOK_MAX_R rounds are cut into items for k_lane_items, which runs after on the
// whole chip and normally finds nothing.
// 10,000 disk edges of ~290 states 128 -> 21 us, 262,144 planar edges of ~40 states 220 -> 42 us
// against the queue on the same evaluators; free edges of 2,500 states (20,000) 730 -> 621, 10 edges of
// 200,000 states 4,044 -> 33.
#include "lanes.hpp"

#define LOOK_NW 4       // waves per workgroup
#define LOOK_MAX_E 16   // edges per wave at most
#define LOOK_MAX_R 16   // rounds of 64 states that a wave takes on its own
#define LOOK_ITEM_R 4   // rounds per item of a long edge
#define LOOK_ITEM_SHARE 16  // an edge takes at most this fraction of the item list

// Counters of a run (PlanWork.meta): a run uses the pair (items, errors) of its parity; the parity
// goes from run to run through two words, each written by the kernel that does not read it, and
// k_lane_items clears the other pair.  So a workspace needs clearing once, not once per run.
enum { LOOK_EPOCH = 0, LOOK_EPOCH2 = 1, LOOK_PAIR = 3 };
__device__ inline long long* look_pair(const PlanWork& W, long long epoch) { return W.meta + LOOK_PAIR + 2 * (epoch & 1); }

// items (waves) of an edge of R rounds
__device__ inline int look_parts(int R, long long cap) {
    const long long m = (R + LOOK_ITEM_R - 1) / LOOK_ITEM_R, most = cap / LOOK_ITEM_SHARE;
    return (int)(m < most ? m : (most > 1 ? most : 1));
}

template <int T1, int T2, bool LOOK, class Q>
__device__ inline bool lane_state(const DiskGridView& S, const Q& q, unsigned mask, unsigned& rc) {
    return disk2_state<T2, LOOK>(S, q, mask, rc);
}
template <int T1, int T2, bool LOOK, class Q>
__device__ inline bool lane_state(const PlanarGridView& S, const Q& q, unsigned mask, unsigned& rc) {
    return planar_state<T1, LOOK>(S, q, mask, rc);
}

template <class View, int T1, int T2>
__global__ void __launch_bounds__(64 * LOOK_NW) k_lane_looks(View S, EdgeBatchView B, PlanWork W, int lgE) {
    extern __shared__ double look_lds[];
    __shared__ int4 s_rec[LOOK_NW][LOOK_MAX_E];  // N, M, window start, full
    const int lane = wave_lane(), wid = threadIdx.x >> 6, D = S.D;
    const int E = 1 << lgE, lgg = 6 - lgE, g = 1 << lgg;
    const long long epoch = W.meta[LOOK_EPOCH];
    if (blockIdx.x == 0 && threadIdx.x == 0) W.meta[LOOK_EPOCH2] = epoch;
    const long long e0 = ((long long)blockIdx.x * LOOK_NW + wid) << lgE;
    if (e0 >= B.n) return;  // no workgroup barrier below
    const int nE = (int)(B.n - e0 < E ? B.n - e0 : E);
    double* sa = look_lds + (size_t)wid * 2 * E * D;
    double* sd = sa + E * D;
    int4* rec = s_rec[wid];
    for (int t = lane; t < nE * D; t += 64) {
        const int j = t / D, k = t - j * D;
        sa[t] = row1(B, e0 + j)[k * B.ds];
        sd[t] = row2(B, e0 + j)[k * B.ds];
    }
    wave_sync();
    const int jg = lane >> lgg, sub = lane & (g - 1);  // the look's edge and place
    int N = 2;
    if (B.N || B.N0 > 0) {
        if (jg < nE) N = B.N ? B.N[e0 + jg] : B.N0;
    } else {
        // edge_N_dev's rule: a NaN in coordinate 0 sticks (lane 0 of the group starts from it), a
        // NaN elsewhere is skipped
        double m = 0.0;
        if (jg < nE) {
            const double* a = sa + jg * D;
            const double* b = sd + jg * D;
            if (sub == 0) m = __builtin_fabs(a[0] - b[0]);
            for (int k = sub ? sub : g; k < D; k += g) {
                const double v = __builtin_fabs(a[k] - b[k]);
                m = v > m ? v : m;
            }
        }
        for (int o = 1; o < g; o <<= 1) {
            const double v = __shfl_xor(m, o, g);
            m = v > m ? v : m;
        }
        m = __shfl(m, 0, g);
        N = edge_N_from_max(m, B.res);
    }
    EdgeWin w;
    w.err = 0;
    w.M = 0;
    if (jg < nE) {
        w = edge_window(N, batch_N_start(B, e0 + jg), batch_N_max(B, e0 + jg), B.incl);
        if (sub == 0) rec[jg] = make_int4(N, w.M, w.w0, w.full);
    }
    // bits of the wave's edges (lane j < E stands for edge j below)
    auto edge_bits = [&](bool b) -> unsigned {  // b of any lane of the edge's group
        const unsigned long long v = __ballot(b);
        const unsigned long long gm = g == 64 ? ~0ull : (1ull << g) - 1ull;
        return (unsigned)__ballot(lane < E && ((v >> ((lane & (E - 1)) << lgg)) & gm) != 0ull);
    };
    const unsigned err = edge_bits(w.err != 0);
    if (err && lane == 0) atomicAdd((unsigned long long*)look_pair(W, epoch) + 1, (unsigned long long)__builtin_popcount(err));
    wave_sync();
    for (int t = lane; t < nE * D; t += 64) sd[t] = interp_step_f64(sa[t], sd[t], rec[t / D].x);
    wave_sync();
    unsigned rechecks = 0;
    unsigned alive = edge_bits(w.M > 0);
    unsigned dead = err;
    auto win_at = [&](const int4 r) {
        EdgeWin v;
        v.N = r.x;
        v.M = r.y;
        v.w0 = r.z;
        v.full = r.w;
        v.first = B.incl ? 0 : 1;
        v.err = 0;
        return v;
    };
    {
        bool hit = false;
        const int local = w.M <= g ? sub : (int)(((unsigned)(2 * sub + 1) * (unsigned)w.M) >> (lgg + 1));
        if (local < w.M) {
            w.N = N;
            const int i = edge_state_index(w, local, B.incl);
            const double* a = sa + jg * D;
            const double* d = sd + jg * D;
            if (i >= 0)
                hit = lane_state<T1, T2, true>(S, [&](int k) { return interp_dir_f64(a[k], d[k], i); }, B.mask, rechecks);
        }
        const unsigned h = edge_bits(hit);
        dead |= h;
        alive &= ~h;
    }
    if (alive) {
        const int Ml = lane < nE ? rec[lane].y : 0;
        unsigned c16 = alive & (unsigned)__ballot(Ml <= 16), c32 = alive & (unsigned)__ballot(Ml > 16 && Ml <= 32),
                 c64 = alive & (unsigned)__ballot(Ml > 32);
        for (unsigned c = c64 & (unsigned)__ballot(Ml > 64 * LOOK_MAX_R); c; c &= c - 1u) {  // long edges: items
            const int j = __builtin_ctz(c);
            const int parts = look_parts((rec[j].y + 63) >> 6, W.items_cap);
            unsigned long long at = 0;
            if (lane == 0) at = atomicAdd((unsigned long long*)look_pair(W, epoch), (unsigned long long)parts);
            at = (unsigned long long)__builtin_amdgcn_readfirstlane((unsigned)at) |
                 ((unsigned long long)__builtin_amdgcn_readfirstlane((unsigned)(at >> 32)) << 32);
            const bool fits = (long long)at + parts <= W.items_cap;
            for (int k = lane; k < parts && (long long)at + k < W.items_cap; k += 64)
                W.items[at + k] = make_int2(fits ? (int)(e0 + j) : -1, k);
            if (fits) c64 &= ~(1u << j);  // no room: the wave keeps the edge
        }
        while (c16 | c32 | c64) {
            unsigned& c = c16 ? c16 : (c32 ? c32 : c64);
            const int lgw = c16 ? 4 : (c32 ? 5 : 6), wd = 1 << lgw;
            const int slot = lane >> lgw, s = lane & (wd - 1);
            unsigned t = c;
            for (int k = 0; k < slot; ++k) t &= t - 1u;
            const int j = t ? __builtin_ctz(t) : -1;
            for (int k = 0; k < 64 >> lgw; ++k) c &= c - 1u;
            const EdgeWin v = win_at(rec[j < 0 ? 0 : j]);
            const int R = lgw == 6 ? (v.M + 63) >> 6 : 1;
            const double* a = sa + j * D;
            const double* d = sd + j * D;
            for (int r = 0; r < R; ++r) {
                const int local = s * R + (R > 1 ? bfs_index(R, r) : 0);
                bool hit = false;
                if (j >= 0 && local < v.M) {
                    const int i = edge_state_index(v, local, B.incl);
                    if (i >= 0)
                        hit = lane_state<T1, T2, false>(S, [&](int k) { return interp_dir_f64(a[k], d[k], i); }, B.mask,
                                                        rechecks);
                }
                unsigned long long b = __ballot(hit);
                if (lgw == 6 && b) {
                    dead |= 1u << j;
                    break;
                }
                while (b) {  // groups with a hit
                    const int l = __builtin_ctzll(b);
                    dead |= 1u << __builtin_amdgcn_readlane(j, l);
                    b &= ~(((1ull << wd) - 1ull) << (l & ~(wd - 1)));
                }
            }
        }
    }
    if (lane < nE) B.out[e0 + lane] = (dead >> lane) & 1u ? 0 : 1;
}

// The items of long edges, one wave each: rounds part, part + parts, ... of the edge's 64-state
// rounds in the binary order, until the edge is found in collision.
template <class View, int T1, int T2>
__global__ void __launch_bounds__(64 * LOOK_NW) k_lane_items(View S, EdgeBatchView B, PlanWork W) {
    __shared__ double s_row[LOOK_NW][2 * MRCC_MAX_D];
    const int lane = wave_lane(), wid = threadIdx.x >> 6, D = S.D;
    const long long epoch = W.meta[LOOK_EPOCH2];
    const long long* pair = look_pair(W, epoch);
    const long long n = pair[0] < W.items_cap ? pair[0] : W.items_cap;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        long long* other = look_pair(W, epoch + 1);
        W.meta[META_ERRORS] = pair[1];
        other[0] = 0;
        other[1] = 0;
        W.meta[LOOK_EPOCH] = epoch + 1;
    }
    double* sa = s_row[wid];
    double* sd = sa + MRCC_MAX_D;
    unsigned rechecks = 0;
    for (long long it = (long long)blockIdx.x * LOOK_NW + wid; it < n; it += (long long)gridDim.x * LOOK_NW) {
        const int2 item = W.items[it];
        const int e = item.x;
        if (e < 0 || edge_dead(B.out, e)) continue;
        const double av = lane < D ? row1(B, e)[lane * B.ds] : 0.0;
        const double bv = lane < D ? row2(B, e)[lane * B.ds] : 0.0;
        int N;
        if (B.N || B.N0 > 0) {
            N = B.N ? B.N[e] : B.N0;
        } else {
            const double m = lane < D ? __builtin_fabs(av - bv) : 0.0;
            const double m0 = readlane_f64(m, 0), mx = wave_max_f64(__builtin_isnan(m) ? 0.0 : m);
            N = edge_N_from_max(__builtin_isnan(m0) ? m0 : mx, B.res);
        }
        const EdgeWin v = edge_window(N, batch_N_start(B, e), batch_N_max(B, e), B.incl);
        wave_sync();
        if (lane < D) {
            sa[lane] = av;
            sd[lane] = interp_step_f64(av, bv, N);
        }
        wave_sync();
        const int R = (v.M + 63) >> 6, parts = look_parts(R, W.items_cap);
        for (int r = item.y; r < R; r += parts) {
            const int local = lane * R + bfs_index(R, r);
            bool hit = false;
            if (local < v.M) {
                const int i = edge_state_index(v, local, B.incl);
                if (i >= 0)
                    hit = lane_state<T1, T2, false>(S, [&](int k) { return interp_dir_f64(sa[k], sd[k], i); }, B.mask, rechecks);
            }
            if (__any(hit)) {
                if (lane == 0) edge_kill(B.out, e);
                break;
            }
            if (edge_dead(B.out, e)) break;
        }
    }
}

__global__ void k_look_reset(PlanWork W) {
    if (threadIdx.x < 8) W.meta[threadIdx.x] = 0;
}

bool lane_looks_apply(const SceneRec& sc) {
    return (sc.kind == KIND_DISKS && sc.disk.grid.n > 0 && sc.disk.nr <= 4) || (sc.kind == KIND_PLANAR && sc.planar.grid.n > 0);
}

void launch_lane_looks(const SceneRec& sc, const EdgeBatchView& B, const PlanWork& W, bool reset, hipStream_t st) {
    if (reset) k_look_reset<<<1, 64, 0, st>>>(W);
    // Edges per wave: as many as leave 4,000 waves, about four per SIMD.  More edges share one chain
    // of round trips (rows, look, rounds), but a wave takes the rounds of its edges one after another.
    // 4 boxes, 100 obstacles, 200,000 edges: 218 / 121 / 69 / 49 / 37 / 36 us at 1 / 2 / 4 / 8 / 16 / 32
    // edges; 2 disks, 20 rectangles, half of 4,000 edges colliding: 20 / 20 / 22 / 22 / 23 / 31 us.
    int lgE = 0;
    while ((2 << lgE) <= LOOK_MAX_E && (B.n >> (lgE + 1)) >= 4000) ++lgE;
    const long long waves = (B.n + (1 << lgE) - 1) >> lgE;
    const int blocks = (int)((waves + LOOK_NW - 1) / LOOK_NW);
    const size_t lds = (size_t)LOOK_NW * 2 * (sizeof(double) << lgE) * sc.D;
    lane_dispatch(sc, [&](const auto& view, auto t1, auto t2) {
        using V = typename std::decay<decltype(view)>::type;
        if constexpr (!LaneKind<V>::all) {  // scenes with a table
            k_lane_looks<V, t1, t2><<<blocks, 64 * LOOK_NW, lds, st>>>(view, B, W, lgE);
            k_lane_items<V, t1, t2><<<4 * mrcc_internal::device_cus(), 64 * LOOK_NW, 0, st>>>(view, B, W);
        }
    });
}
