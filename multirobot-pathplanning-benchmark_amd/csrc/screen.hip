// screen.hip — self-collision screen of arm states ahead of the full evaluators (gfx950).
//
// Most random states of arm scenes collide within one arm.  The full evaluator spends one wavefront
// per state and places every arm; this kernel takes 16 (state, arm) items per wavefront, 4 lanes
// each, tests the deepest link pair of the arm and passes a state on to its next arm only when no
// contact is certain.  It only ever reports certain collisions: the frames, sphere centres and the
// margin M are those of the full evaluator (binary64 kinematics in the same order, centres rounded
// to binary32, d^2 - (r_i + r_j)^2 < -M), so a state it reports collides by the binary64 predicate
// too.  States it does not report go on to the full evaluator, which decides alone; the booleans are
// the same with and without the screen.
#include "lanes.hpp"

#define SCREEN_ITEMS 16       // (state, arm) items per wave and step
#define SCREEN_QUEUE 80       // pending items: 15 left over + one chunk of 64
#define SCREEN_BINS 1024      // pass counts histogrammed in LDS
#define SCREEN_MAX_NW 8       // waves per workgroup
#define SCREEN_MAX_N (1 << 28)  // queue entries hold the index in 28 bits, the arm count above

// LDS of a wave: per item the two frames of its deepest link pair ([row][R0 R1 R2 t] doubles, 16
// bytes of padding against bank conflicts), the link spheres, the queue of pending items.
#define SCREEN_X_STRIDE (2 * 96 + 16)
__host__ __device__ inline int screen_wave_bytes(int dof) {
    return SCREEN_ITEMS * (SCREEN_X_STRIDE + 16 * dof) + 8 * SCREEN_QUEUE;
}

struct ScreenArgs {
    const double* q1;   // rows of the configurations, or of the edges' first ends
    const int* idx1;
    const double* q2;   // EDGES: rows of the second ends
    const int* idx2;
    int4* erec;         // EDGES: per-edge records
    int* hist;          // EDGES: pass histogram
    unsigned long long* stats;
    const int* modes;
    unsigned char* out;
    long long rs, ds;
    int n, md0, incl, lgG;
    unsigned mask;
};

template <int J>
__device__ inline float sq_bcast(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), J * 0x55, 0xf, 0xf, false));
}
__device__ inline unsigned quad_min(unsigned v) {
    v = min(v, (unsigned)__builtin_amdgcn_mov_dpp((int)v, 0xb1, 0xf, 0xf, false));  // lanes [1, 0, 3, 2]
    return min(v, (unsigned)__builtin_amdgcn_mov_dpp((int)v, 0x4e, 0xf, 0xf, false));  // [2, 3, 0, 1]
}

// centre of sphere `s` in the frame X ([row][R0 R1 R2 t]): xform_point_f64's operations
__device__ inline float4 screen_place(const ArmLds& W, const double* X, int s, bool act) {
#pragma clang fp contract(off)
    const double l0 = W.sphL[3 * s], l1 = W.sphL[3 * s + 1], l2 = W.sphL[3 * s + 2];
    float c[3];
#pragma unroll
    for (int r = 0; r < 3; ++r) c[r] = (float)(((X[4 * r] * l0 + X[4 * r + 1] * l1) + X[4 * r + 2] * l2) + X[4 * r + 3]);
    return make_float4(act ? c[0] : __builtin_nanf(""), c[1], c[2], W.sphR[s]);  // NaN: no test holds
}

// One step: lane group s = lane / 4 takes the arm `a` (of the group) of the state `ent` (index and
// arm count, state number of an edge); act: the group has an item.  Returns the lanes (all four of
// a group) whose state certainly collides.
template <bool CHAIN, bool EDGES>
__device__ inline unsigned long long screen_step(const ArmK& V, const ArmLds& W, const ScreenArgs& A, int a, int2 ent,
                                                 bool act, unsigned char* wave_lds) {
    const int lane = wave_lane();
    const int s = lane >> 2, r = lane & 3, rr = r < 3 ? r : 2;
    const int dof = V.dof;
    const long long id = ent.x & (SCREEN_MAX_N - 1);
    // 1. joint values: lane r of the group holds joints r and r + 4 of the arm
    const double* row = A.q1 + (A.idx1 ? (long long)A.idx1[id] : id) * A.rs;
    double qv[2];
    if constexpr (EDGES) {
        const double* end = A.q2 + (A.idx2 ? (long long)A.idx2[id] : id) * A.rs;
        const int N = A.erec[id].x;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int k = r + 4 * h, c = a * dof + (k < dof ? k : 0);
            qv[h] = interp_f64(row[c * A.ds], end[c * A.ds], N, ent.y & 0xffffff);
        }
    } else {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int k = r + 4 * h, c = a * dof + (k < dof ? k : 0);
            qv[h] = row[c * A.ds];
        }
    }
    const SinCos t0 = sincos_f64(qv[0]), t1 = sincos_f64(qv[1]);
    // 2. kinematics: lane r < 3 carries row r of the arm's frame through the joints (rows are
    //    independent: dh_row_f64); the group's lanes hand out each joint's sine and cosine
    //    The rows of every link stay in registers until the state's link pair is known.
    double* X = (double*)(wave_lds + s * SCREEN_X_STRIDE);
    float* LC = (float*)(wave_lds + SCREEN_ITEMS * SCREEN_X_STRIDE) + 4 * dof * s;
    double Xr[MRCC_MAX_DOF][4];
    double R0 = W.base[12 * a + 3 * rr], R1 = W.base[12 * a + 3 * rr + 1], R2 = W.base[12 * a + 3 * rr + 2],
           t = W.base[12 * a + 9 + rr];
#pragma unroll
    for (int k = 0; k < MRCC_MAX_DOF; ++k) {
        if (k >= dof) break;  // wave-uniform
        const int l = a * dof + k;
        double cs = quad_bcast_f64(k < 4 ? t0.c : t1.c, k & 3);
        double sn = quad_bcast_f64(k < 4 ? t0.s : t1.s, k & 3);
        if constexpr (CHAIN) {
#pragma clang fp contract(off)
            const double* C = W.dh + 12 * l;
            const bool pr = (V.prism >> l) & 1ull;
            const double q = quad_bcast_f64(k < 4 ? qv[0] : qv[1], k & 3);
            cs = pr ? 1.0 : cs;
            sn = pr ? 0.0 : sn;
            double y[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const ChainCoef kc = chain_coef_f64(cs, sn, C[c], C[4 + c]);
                const double a2 = c == 3 ? chain_a23_f64(C, pr, q) : C[8 + c];
                y[c] = (R0 * kc.a0 + R1 * kc.a1) + R2 * a2;
            }
            R0 = y[0];
            R1 = y[1];
            R2 = y[2];
            t = y[3] + t;
        } else {
            dh_row_f64(R0, R1, R2, t, W.dh + 4 * l, cs, sn);
        }
        __builtin_amdgcn_sched_barrier(0);  // one joint's coefficients in flight, not all
        Xr[k][0] = R0;
        Xr[k][1] = R1;
        Xr[k][2] = R2;
        Xr[k][3] = t;
        // the link's bounding sphere: coordinate r of its centre, the radius from lane 3
        float v;
        {
#pragma clang fp contract(off)
            const double* b = W.linkBC + 3 * l;
            v = (float)(((R0 * b[0] + R1 * b[1]) + R2 * b[2]) + t);
        }
        LC[4 * k + r] = r < 3 ? v : W.linkR[l];
    }
    wave_sync();
    // 3. the deepest of the arm's link pairs with close bounding spheres (least squared distance over
    //    squared sum of radii; the pair's number in the low bits of the key)
    const int p_lo = W.sets[a], np = W.sets[a + 1] - p_lo;  // np <= (dof - 1)(dof - 2) / 2 <= 21
    const int np_max = (dof - 1) * (dof - 2) / 2;
    const float4* L4 = (const float4*)LC;
    unsigned best = ~0u;
#pragma unroll
    for (int j = 0; j < 6; ++j) {
        if (4 * j >= np_max) break;  // wave-uniform
        const int p = r + 4 * j;
        const bool in = act && p < np;
        const int2 pr = arm_pair(V, W, in ? p_lo + p : 0);
        const float4 Ca = L4[in ? ((pr.x >> 8) & 255) - a * dof : 0], Cb = L4[in ? (pr.x & 255) - a * dof : 0];
        const float dx = Ca.x - Cb.x, dy = Ca.y - Cb.y, dz = Ca.z - Cb.z;
        const float d2 = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
        const float Rs = Ca.w + Cb.w, T = Rs * Rs;
        const unsigned key = (__float_as_uint(d2 * __builtin_amdgcn_rcpf(T)) & ~31u) | (unsigned)p;
        best = in && d2 <= T + V.Mcull && key < best ? key : best;
    }
    best = quad_min(best);
    const bool test = best != ~0u;
    if (__ballot(test) == 0ull) {
        wave_sync();
        return 0ull;
    }
    // 4. every sphere pair of that link pair (lane r places spheres r and r + 4 of both links; the
    //    second link's are handed round the group)
    const float M = V.Msph;
    const int2 pr = arm_pair(V, W, test ? p_lo + (int)(best & 31u) : 0);  // !test: masked by NaN below
    const int fl = pr.y & 511, nl = (pr.y >> 9) & 15, fm = (pr.y >> 13) & 511, nm = (pr.y >> 22) & 15;
    const int ll = ((pr.x >> 8) & 255) - a * dof, lm = (pr.x & 255) - a * dof;
#pragma unroll
    for (int k = 0; k < MRCC_MAX_DOF; ++k) {
        if (k >= dof) break;  // wave-uniform
        if (r < 3 && (ll == k || lm == k)) {  // ll != lm
            double2* x = (double2*)(X + (ll == k ? 0 : 12) + 4 * r);
            x[0] = make_double2(Xr[k][0], Xr[k][1]);
            x[1] = make_double2(Xr[k][2], Xr[k][3]);
        }
    }
    wave_sync();
    const double *Xl = X, *Xm = X + 12;
    float4 ca[2], cb[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int k = r + 4 * h;
        ca[h] = screen_place(W, Xl, fl + (k < nl ? k : 0), test && k < nl);
        cb[h] = screen_place(W, Xm, fm + (k < nm ? k : 0), k < nm);
    }
    float dist = 0.0f;  // least d^2 - (r_i + r_j)^2 (fminf skips the NaN of lanes without a sphere)
    auto against = [&](float4 c) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const float dx = ca[h].x - c.x, dy = ca[h].y - c.y, dz = ca[h].z - c.z;
            const float d2 = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
            const float Rs = ca[h].w + c.w;
            dist = fminf(dist, fmaf(-Rs, Rs, d2));
        }
    };
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        against(make_float4(sq_bcast<0>(cb[h].x), sq_bcast<0>(cb[h].y), sq_bcast<0>(cb[h].z), sq_bcast<0>(cb[h].w)));
        against(make_float4(sq_bcast<1>(cb[h].x), sq_bcast<1>(cb[h].y), sq_bcast<1>(cb[h].z), sq_bcast<1>(cb[h].w)));
        against(make_float4(sq_bcast<2>(cb[h].x), sq_bcast<2>(cb[h].y), sq_bcast<2>(cb[h].z), sq_bcast<2>(cb[h].w)));
        against(make_float4(sq_bcast<3>(cb[h].x), sq_bcast<3>(cb[h].y), sq_bcast<3>(cb[h].z), sq_bcast<3>(cb[h].w)));
    }
    const unsigned long long m = __ballot(dist < -M);
    const unsigned long long hits = __ballot(((m >> (lane & ~3)) & 15ull) != 0ull);
    wave_sync();  // the wave's LDS is rewritten by the next step
    return hits;
}

// EDGES: edges e with passes (erec[e].z > 0); a certain collision of its middle state writes
// out[e] = 0, takes the edge out of the queue (erec[e].z = 0) and out of the histogram.
// Otherwise configurations r: out[r] = 0 for a certain collision, 1 for one that the full evaluator
// has to decide.  A wave stops screening when fewer than 1 in 8 of its states were caught: there the
// full evaluator alone is faster.
template <bool CHAIN, bool EDGES>
__global__ void __launch_bounds__(64 * SCREEN_MAX_NW, 4) k_arm_screen(ArmK V, ScreenArgs A, int chunk) {
    extern __shared__ double lds_scr[];
    unsigned char* lds = (unsigned char*)lds_scr;
    int* h = (int*)(lds + V.img_bytes);
    if constexpr (EDGES)
        for (int i = threadIdx.x; i < SCREEN_BINS; i += blockDim.x) h[i] = 0;
    arm_stage_scene(lds, V);  // ends with a barrier
    ArmLds W;
    {
        const ArmStaticLayout o = arm_static_layout(V.L, V.na, V.nb, V.S, V.NP, V.nm, V.nclu, V.chain);
        W.dh = (const double*)(lds + o.o_dh);
        W.base = (const double*)(lds + o.o_base);
        W.sphL = (const double*)(lds + o.o_sphL);
        W.linkBC = (const double*)(lds + o.o_linkBC);
        W.sphR = (const float*)(lds + o.o_sphR);
        W.linkR = (const float*)(lds + o.o_linkR);
        W.pairs = (const int2*)(lds + o.o_pairs);
        W.mact = (const int*)(lds + o.o_mact);
        W.sets = (const int*)(lds + o.o_sets);
    }
    const int lane = wave_lane(), nw = blockDim.x >> 6, wv = threadIdx.x >> 6;
    unsigned char* wl = lds + V.img_bytes + (EDGES ? 4 * SCREEN_BINS : 0) + wv * screen_wave_bytes(V.dof);
    int2* queue = (int2*)(wl + SCREEN_ITEMS * (SCREEN_X_STRIDE + 16 * V.dof));
    const unsigned amask = A.mask & ((1u << V.na) - 1u);
    const int first = amask ? __builtin_ctz(amask) : MRCC_MAX_ARMS;
    int pend = 0;  // items in the queue
    int tested = 0, caught = 0;
    bool stop = amask == 0;
    const long long nchunks = ((long long)A.n + chunk - 1) / chunk;
    long long c = (long long)blockIdx.x * nw + wv;
    const long long cstep = (long long)gridDim.x * nw;
    for (;;) {
        if (pend < SCREEN_ITEMS && c < nchunks) {  // a chunk of states, each at its first arm
            const long long id = c * chunk + lane;
            c += cstep;
            const bool in = lane < chunk && id < A.n;
            int na = 0, i = 0;
            if (in) {
                if constexpr (EDGES) {
                    const int4 rec = A.erec[id];
                    if (rec.z > 0) {
                        EdgeWin w;
                        w.N = rec.x;
                        w.M = rec.y;
                        w.w0 = erec_w0(rec);
                        w.full = erec_full(rec);
                        w.first = A.incl ? 0 : 1;
                        w.err = 0;
                        // the middle slot: the state least like the ends, which a planner has
                        // usually checked
                        i = edge_state_index(w, w.M >> 1, A.incl);
                        if (i >= 0) na = arm_mact(V, W, A.modes ? A.modes[id] : A.md0);
                    }
                } else {
                    const int md = A.modes ? A.modes[id] : A.md0;
                    if (md >= 0 && md < V.nm) na = arm_mact(V, W, md);
                }
            }
            const bool push = !stop && in && na > first;
            const unsigned long long m = __ballot(push);
            if (push) queue[pend + (int)lanes_below(m)] = make_int2((int)id | ((na - 1) << 28), i | (first << 24));
            if (!EDGES && in && !push) A.out[id] = 1;
            pend += __popcll(m);
            wave_sync();
            if (EDGES && stop) break;  // nothing to write for the states left
            continue;
        }
        if (pend == 0) break;
        const int ns = pend < SCREEN_ITEMS ? pend : SCREEN_ITEMS;
        pend -= ns;
        // group g takes item g % ns; the groups beyond the last item take the next arms of the same
        // states (a single state left over goes to the full evaluator)
        const int g = lane >> 2, gi = g % ns, ahead = g / ns;
        const int2 ent = queue[pend + gi];
        unsigned arms = amask & ((2u << ((ent.x >> 28) & 7)) - 1u) & ~((1u << (ent.y >> 24)) - 1u);
        for (int k = 0; k < ahead; ++k) arms &= arms - 1u;
        const bool act = arms != 0u;
        const int a = act ? __builtin_ctz(arms) : 0;
        const bool run = !stop && ns > 1;
        unsigned long long hits = run ? screen_step<CHAIN, EDGES>(V, W, A, a, ent, act, wl) : 0ull;
        const bool lead = g < ns && (lane & 3) == 0;
        bool hit = false;
        unsigned rest = arms;  // of a lead lane: the state's arms not tested yet
        for (int k = 0; k < SCREEN_ITEMS; k += ns) {  // the state's groups g, g + ns, ...
            if (g + k < SCREEN_ITEMS) {
                hit |= (hits >> ((lane + 4 * k) & 63)) & 1ull;
                rest &= rest - 1u;
            }
        }
        const long long id = ent.x & (SCREEN_MAX_N - 1);
        if (run) {
            tested += ns;
            caught += __popcll(__ballot(lead && hit));
            stop = caught * 8 < tested;
        }
        const bool next = lead && !hit && run && rest != 0u;
        if (lead && hit) {
            A.out[id] = 0;
            if constexpr (EDGES) {
                const int4 rec = A.erec[id];
                ((int*)(A.erec + id))[2] = 0;
                if (rec.z < SCREEN_BINS) atomicAdd(&h[rec.z], 1);
                else atomicSub(&A.hist[rec.z], 1);
                if (A.stats) {  // a caught edge: one state evaluated, its other slots skipped
                    atomicAdd(A.stats, 1ull);
                    atomicAdd(A.stats + 2, (unsigned long long)(rec.y - 1));
                    atomicAdd(A.stats + 3, (unsigned long long)rec.z << A.lgG);
                }
            }
        } else if (!EDGES && lead && !next) {
            A.out[id] = 1;
        }
        const unsigned long long m = __ballot(next);
        wave_sync();  // the queue's entries are read before they are rewritten
        if (next) queue[pend + (int)lanes_below(m)] = make_int2(ent.x, (ent.y & 0xffffff) | (__builtin_ctz(rest) << 24));
        pend += __popcll(m);
        wave_sync();
    }
    if constexpr (EDGES) {
        __syncthreads();
        for (int i = threadIdx.x; i < SCREEN_BINS; i += blockDim.x)
            if (h[i]) atomicSub(&A.hist[i], h[i]);
    }
}

// host side --------------------------------------------------------------------------------------
struct ScreenShape {
    int nw, wgs;
    size_t lds;
};

// waves per workgroup: the most resident waves per CU in 160 KiB of LDS
static ScreenShape screen_shape(const SceneRec& sc, bool edges) {
    const ArmK& V = sc.armk;
    const size_t fixed = (size_t)V.img_bytes + (edges ? 4 * SCREEN_BINS : 0);
    ScreenShape b = {0, 0, 0};
    for (int nw = 1; nw <= SCREEN_MAX_NW; ++nw) {
        const size_t lds = fixed + (size_t)nw * screen_wave_bytes(V.dof);
        if (lds > 163840) break;
        const int wgs = (int)(163840 / lds) < 16 / nw ? (int)(163840 / lds) : 16 / nw;
        if (wgs * nw > b.nw * b.wgs) b = {nw, wgs, lds};
    }
    return b;
}

// chunk of states per wave and turn: every resident wave gets some, at most a wave's lanes
static int screen_chunk(long long n, long long waves) {
    int chunk = SCREEN_ITEMS;
    while (chunk < 64 && n > waves * chunk) chunk *= 2;
    return chunk;
}

template <bool EDGES>
static void launch_screen(const SceneRec& sc, const ScreenArgs& A, hipStream_t st) {
    const ScreenShape b = screen_shape(sc, EDGES);
    const long long waves = (long long)b.nw * b.wgs * mrcc_internal::device_cus();
    const int chunk = screen_chunk(A.n, waves);
    const long long nchunks = ((long long)A.n + chunk - 1) / chunk;
    const int blocks = (int)(((nchunks < waves ? nchunks : waves) + b.nw - 1) / b.nw);
    if (sc.arm.chain) k_arm_screen<true, EDGES><<<blocks, 64 * b.nw, b.lds, st>>>(sc.armk, A, chunk);
    else k_arm_screen<false, EDGES><<<blocks, 64 * b.nw, b.lds, st>>>(sc.armk, A, chunk);
}

bool arm_screen_applies(const SceneRec& sc, long long n, long long n_min) {
    return sc.kind == KIND_ARMS && sc.armk.broadphase && n >= n_min && n < SCREEN_MAX_N &&
           screen_shape(sc, true).nw > 0;
}

void launch_screen_edges(const SceneRec& sc, const EdgeBatchView& B, const PlanWork& W, int lgG, hipStream_t st) {
    ScreenArgs A;
    A.q1 = B.q1;
    A.idx1 = B.idx1;
    A.q2 = B.q2;
    A.idx2 = B.idx2;
    A.erec = W.erec;
    A.hist = W.hist;
    A.stats = W.stats;
    A.modes = B.modes;
    A.out = B.out;
    A.rs = B.rs;
    A.ds = B.ds;
    A.n = (int)B.n;
    A.md0 = B.md0;
    A.incl = B.incl;
    A.lgG = lgG;
    A.mask = B.mask;
    launch_screen<true>(sc, A, st);
}

void launch_screen_configs(const SceneRec& sc, const double* q, long long n, long long rs, long long ds,
                           const int* modes, unsigned mask, unsigned char* out, hipStream_t st) {
    ScreenArgs A;
    A.q1 = q;
    A.idx1 = nullptr;
    A.q2 = nullptr;
    A.idx2 = nullptr;
    A.erec = nullptr;
    A.hist = nullptr;
    A.stats = nullptr;
    A.modes = modes;
    A.out = out;
    A.rs = rs;
    A.ds = ds;
    A.n = (int)n;
    A.md0 = 0;
    A.incl = 0;
    A.lgG = 0;
    A.mask = mask;
    launch_screen<false>(sc, A, st);
}
