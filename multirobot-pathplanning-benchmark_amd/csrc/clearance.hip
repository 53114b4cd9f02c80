// clearance.hip — differentiable clearance cost of arm scenes (binary32).
//
//   cost(q) = sum over the checked pair set of max(0, m + r_i + r_j - |c_i - c_j|)^2
//           + sum over spheres x boxes of max(0, m + r_i - dist(c_i, box))^2
// with the pair set of the boolean check (links >= 2 apart in one arm, all links of different
// arms), culled exactly with the links' bounding spheres.  The backward recomputes the forward
// kinematics, sums the force of every term and its moment (d cost / d c and c x that) per link in
// LDS, and maps them to the joints with d c / d q_k = z_{k-1} x (c - o_{k-1}) (revolute joints) or
// z_{k-1} (prismatic chain joints) for spheres on links >= k of the same arm.
//
// Bound by instruction issue and LDS latency (the inputs are 4 D bytes a waypoint).  One waypoint per
// wave at a time, its kinematics in pairs of waypoints; a workgroup of several waves stages the
// scene's binary32 tables in LDS once and walks the batch.
#include "engine.hpp"

namespace {

#define CLR_MAX_NW 8  // waves per workgroup

struct ClrLds {
    // per wave
    float4* X;     // [2][L*3] rows (R0 R1 R2 t) of every link frame, two waypoints
    float2* cs;    // [2*D] cosine, sine of every joint (kinematics; shares memory with sph)
    float4* sph;   // [S] sphere centres, radii
    float4* lk;    // [L] link bounding spheres (x, y, z, R)
    float* tf;     // [L*6] per link: sum of c x f and sum of f over its spheres (backward)
    int* cand;     // [64] candidates of one culling round
    int* cand2;    // [64] second-level candidates (link, box) of the clustered box test
    // per workgroup (the scene)
    const float4* joint;  // [L] d a cos(alpha) sin(alpha), or [L*3] rows of C (chain joints)
    const float4* base;   // [na*3] rows
    const float4* sphL;   // [S] centre in the link frame, radius
    const float4* lbc;    // [L] bounding-sphere centre in the link frame, radius
    const int* fc;        // [L] first sphere | count << 16
    const int* slink;     // [S] link of the sphere
    const float4* box;    // [nb*2] lo, hi (LDS; scenes with box clusters only)
    const float4* clu;    // [nclu*2] lo xyz | first box, hi xyz | box count
    const int2* pairs;    // [NP] (NP <= ARM_PAIRS_LDS_MAX)
};

inline __host__ __device__ int clr_sph_bytes(int D, int S) { return 16 * (S > D ? S : D); }
inline __host__ __device__ int clr_wave_bytes(int D, int L, int S) {
    return 96 * L + clr_sph_bytes(D, S) + 16 * L + ((24 * L + 15) & ~15) + 512;
}

__device__ inline ClrLds clr_lds(unsigned char* b, const ClrK& V) {
    const ClrLayout o = clr_layout(V.L, V.na, V.nb, V.S, V.NP, V.nclu, V.chain);
    ClrLds W;
    W.joint = (const float4*)(b + o.o_joint);
    W.base = (const float4*)(b + o.o_base);
    W.sphL = (const float4*)(b + o.o_sph);
    W.lbc = (const float4*)(b + o.o_lbc);
    W.fc = (const int*)(b + o.o_fc);
    W.slink = (const int*)(b + o.o_slink);
    W.box = (const float4*)(b + o.o_box);
    W.clu = (const float4*)(b + o.o_clu);
    W.pairs = (const int2*)(b + o.o_pairs);
    unsigned char* w = b + o.bytes + (threadIdx.x >> 6) * clr_wave_bytes(V.D, V.L, V.S);
    W.X = (float4*)w;
    w += 96 * V.L;
    W.sph = (float4*)w;
    W.cs = (float2*)w;
    w += clr_sph_bytes(V.D, V.S);
    W.lk = (float4*)w;
    w += 16 * V.L;
    W.tf = (float*)w;
    w += (24 * V.L + 15) & ~15;
    W.cand = (int*)w;
    W.cand2 = W.cand + 64;
    return W;
}

// Forward kinematics of `nw` (1 or 2) waypoints: the rows of every link frame into W.X.  Lane
// (waypoint, arm, row) carries a row through its arm's joints (rows are independent of each other).
template <bool CHAIN>
__device__ inline void clr_fk(const ClrK& V, const ClrLds& W, const float* q, int nw) {
#pragma clang fp contract(off)
    const int lane = wave_lane();
    for (int t = lane; t < nw * V.D; t += 64) {
        float s, c;
        sincosf(q[t], &s, &c);
        const int k = t < V.D ? t : t - V.D;
        const bool pr = CHAIN && ((V.prism >> k) & 1ull);  // prismatic: Tz(q) C = Rz(0) C + q e_z
        W.cs[t] = pr ? make_float2(1.f, 0.f) : make_float2(c, s);
    }
    wave_sync();
    const int rows = 3 * V.na;  // <= 24
    if (lane < nw * rows) {
        const int w = lane >= rows ? 1 : 0, ar = lane - w * rows, a = ar / 3, r = ar - 3 * a;
        const float4 b = W.base[ar];
        float R0 = b.x, R1 = b.y, R2 = b.z, t = b.w;
        const int l0 = a * V.dof;
        for (int k = 0; k < V.dof; ++k) {
            const int l = l0 + k;
            const float2 cs = W.cs[w * V.D + l];
            float y0, y1, y2, y3;
            if constexpr (CHAIN) {  // A = Rz(q) C (revolute), Tz(q) C (prismatic)
                const float4 c0 = W.joint[3 * l], c1 = W.joint[3 * l + 1], c2 = W.joint[3 * l + 2];
                const float u = fmaf(R1, cs.y, R0 * cs.x), v = fmaf(-R0, cs.y, R1 * cs.x);
                const float q3 = ((V.prism >> l) & 1ull) ? q[w * V.D + l] : 0.f;
                y0 = fmaf(R2, c2.x, fmaf(v, c1.x, u * c0.x));
                y1 = fmaf(R2, c2.y, fmaf(v, c1.y, u * c0.y));
                y2 = fmaf(R2, c2.z, fmaf(v, c1.z, u * c0.z));
                y3 = fmaf(R2, c2.w + q3, fmaf(v, c1.w, fmaf(u, c0.w, t)));
            } else {  // A = Rz(q) Tz(d) Tx(a) Rx(alpha)
                const float4 p = W.joint[l];
                const float u = fmaf(R1, cs.y, R0 * cs.x), v = fmaf(-R0, cs.y, R1 * cs.x);
                y0 = u;
                y1 = fmaf(R2, p.w, v * p.z);
                y2 = fmaf(-v, p.w, R2 * p.z);
                y3 = fmaf(R2, p.x, fmaf(u, p.y, t));
            }
            W.X[(w * V.L + l) * 3 + r] = make_float4(y0, y1, y2, y3);
            R0 = y0;
            R1 = y1;
            R2 = y2;
            t = y3;
        }
    }
    wave_sync();
}

// Fused operations are written out here and in the terms: the kernels with and without the gradient
// then round the same, and a cost does not depend on whether its gradient is wanted.
__device__ inline float clr_row(float4 a, float4 l) { return fmaf(a.z, l.z, fmaf(a.y, l.y, fmaf(a.x, l.x, a.w))); }
__device__ inline float4 clr_point(const float4* X, float4 l) {
    return make_float4(clr_row(X[0], l), clr_row(X[1], l), clr_row(X[2], l), l.w);
}
__device__ inline float clr_sq(float ex, float ey, float ez) { return fmaf(ez, ez, fmaf(ey, ey, ex * ex)); }

// Slack of the link-level cull (metres): covers the binary32 rounding of the link and sphere
// centres (micrometres) with a wide margin.
#define CLR_CULL_EPS 1e-4f

// within reach (up to rounding)
__device__ inline bool clr_near(float e2, float R) { return e2 <= R * R * 1.0001f; }

// One penetration term: cost += pen^2 for pen = R - d > 0, and with GRAD the force g e on the first
// sphere (g = -2 pen / d).  The square root only for pairs within reach: d < R implies
// e2 < R^2 (1 + 2^-21), so the bound passes every pair with pen > 0.
template <bool GRAD>
__device__ inline bool clr_term(float ex, float ey, float ez, float R, float& cost, float& gx, float& gy, float& gz) {
    const float e2 = clr_sq(ex, ey, ez);
    if (!clr_near(e2, R)) return false;
    const float d = sqrtf(e2);
    const float pen = R - d;
    if (!(pen > 0.f)) return false;
    cost = fmaf(pen, pen, cost);
    if (!GRAD || !(d > 0.f)) return false;
    const float g = -2.f * pen / d;
    gx = g * ex;
    gy = g * ey;
    gz = g * ez;
    return true;
}

// Force and moment sums of the links, lane (arm a, joint k) = 8 a + k holding link (a, k).  Summed in
// registers by lane shifts: LDS atomics of the lanes of one candidate all go to the same two links,
// one after the other (262,144 waypoints: 694 us with them).
struct ClrSums {
    float T0, T1, T2, F0, F1, F2;
};

// adds the force g at the point c to the link's sums in LDS (the walk over the full pair set)
__device__ inline void clr_add(float* tf, float4 c, float gx, float gy, float gz) {
    atomicAdd(tf, c.y * gz - c.z * gy);
    atomicAdd(tf + 1, c.z * gx - c.x * gz);
    atomicAdd(tf + 2, c.x * gy - c.y * gx);
    atomicAdd(tf + 3, gx);
    atomicAdd(tf + 4, gy);
    atomicAdd(tf + 5, gz);
}

// v + the value of the lane a row shift away (0 beyond the row of 16: one add with a DPP operand)
template <int CTRL>
__device__ inline float dpp_add(float v) {
    return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
// sum over the lane's group of 8, in the group's last lane (row_shr 1, 2, 4; lanes whose source lies
// in the group before take it too: their value is not used)
__device__ inline float group8_sum(float v) { return dpp_add<0x114>(dpp_add<0x112>(dpp_add<0x111>(v))); }
// sum over the lane's row of 16, in the row's last lane
__device__ inline float row16_sum(float v) { return dpp_add<0x118>(group8_sum(v)); }
// sum over the wave, wave-uniform
__device__ inline float wave_sum_f32(float v) {
    v = row16_sum(v);
    return readlane_f(v, 15) + readlane_f(v, 31) + (readlane_f(v, 47) + readlane_f(v, 63));
}

// squared distance from c to the box [lo, hi], and its vector
__device__ inline float3 clr_box_e(float4 c, float4 lo, float4 hi) {
    return make_float3(c.x - fminf(fmaxf(c.x, lo.x), hi.x), c.y - fminf(fmaxf(c.y, lo.y), hi.y),
                       c.z - fminf(fmaxf(c.z, lo.z), hi.z));
}
__device__ inline float clr_box_e2(float4 c, float4 lo, float4 hi) {
    const float3 e = clr_box_e(c, lo, hi);
    return clr_sq(e.x, e.y, e.z);
}

// sum of the lane's value and those of the lanes after it in its group of 8 (DPP row_shl; the last
// lanes of a group take nothing from the next group)
__device__ inline float clr_suffix8(float v) {
    const int k = threadIdx.x & 7;
    const float a = dpp_add<0x101>(v), b = k < 7 ? a : v;
    const float c = dpp_add<0x102>(b), d = k < 6 ? c : b;
    const float e = dpp_add<0x104>(d);
    return k < 4 ? e : d;
}

// The full pair set without culling (the scene's broad phase off): lane = sphere i, every partner
// j >= sph_lo[i] and every box in turn.  With the gradient a partner that no lane has in reach ends
// at its distance (262,144 waypoints 5.16 ms when every lane branched for itself, 4.12 now; the cost alone is
// faster by lanes, 3.43 against 3.80).  Returns the lane's share of the cost.
template <bool GRAD>
__device__ inline float clr_pairs_all(const ClrK& V, const ClrLds& W, float m) {
    const int lane = wave_lane();
    const int S = V.S;
    float cost = 0.f;
    for (int base = 0; base < S; base += 64) {
        const int i = base + lane;
        const bool act = i < S;
        const float4 ci = W.sph[act ? i : 0];
        float fx = 0.f, fy = 0.f, fz = 0.f;
        for (int b = 0; b < V.nb; ++b) {
            const float3 e = clr_box_e(ci, V.box32[2 * b], V.box32[2 * b + 1]);
            const float R = m + ci.w;
            const bool near = act && clr_near(clr_sq(e.x, e.y, e.z), R);
            if (GRAD && __ballot(near) == 0ull) continue;
            float gx, gy, gz;
            if (near && clr_term<GRAD>(e.x, e.y, e.z, R, cost, gx, gy, gz)) {
                fx += gx;
                fy += gy;
                fz += gz;
            }
        }
        const int lo = act ? V.sph_lo[i] : 0x7fffffff;
        for (int j = V.sph_lo[base]; j < S; ++j) {
            const float4 cj = W.sph[j];
            const float ex = ci.x - cj.x, ey = ci.y - cj.y, ez = ci.z - cj.z, R = m + ci.w + cj.w;
            const bool near = j >= lo && clr_near(clr_sq(ex, ey, ez), R);
            if (GRAD && __ballot(near) == 0ull) continue;
            float gx, gy, gz;
            if (near && clr_term<GRAD>(ex, ey, ez, R, cost, gx, gy, gz)) {
                fx += gx;
                fy += gy;
                fz += gz;
                clr_add(W.tf + 6 * W.slink[j], cj, -gx, -gy, -gz);
            }
        }
        if (GRAD && act) clr_add(W.tf + 6 * W.slink[i], ci, fx, fy, fz);
    }
    return cost;
}

// The lane's share of the cost of the pair set; with GRAD also the links' forces and moments in W.tf.
// Terms are nonzero only for pairs within reach, so both parts are culled with the links'
// bounding spheres first (the triangle inequality: a sphere of link A lies within R_A - r of A's
// centre, so no pair of two links farther apart than m + R_A + R_B, and no sphere of a link
// farther than m + R_A from a box, penetrates); the surviving (link, box) and (link, link)
// candidates are expanded to their spheres, 8 x 8 lanes at a time.  With the scene's broad phase
// off (V.broadphase = 0) the full pair set is walked instead (clr_pairs_all).
template <bool GRAD>
__device__ inline float clr_pairs(const ClrK& V, const ClrLds& W, float m, int my_link, ClrSums& S) {
    const int lane = wave_lane();
    const int L = V.L;
    float cost = 0.f;
    // the spheres of (link, box) candidate `cd` (lane k of its group of 8 takes the link's sphere k)
    auto sphere_box = [&](bool act, int cd, int k, const float4* box) {
        const int l = cd & 255, b = cd >> 8;
        const int fc = W.fc[l];
        act = act && k < (fc >> 16);
        const float4 ci = W.sph[(fc & 0xffff) + (act ? k : 0)];
        const float3 e = clr_box_e(ci, box[2 * b], box[2 * b + 1]);
        float gx = 0.f, gy = 0.f, gz = 0.f;
        const bool f = act && clr_term<GRAD>(e.x, e.y, e.z, m + ci.w, cost, gx, gy, gz);
        if constexpr (GRAD) {
            unsigned long long mk = __ballot(f);
            if (mk == 0ull) return;  // wave-uniform
            if (!f) gx = gy = gz = 0.f;
            const float t0 = group8_sum(ci.y * gz - ci.z * gy), t1 = group8_sum(ci.z * gx - ci.x * gz),
                        t2 = group8_sum(ci.x * gy - ci.y * gx), f0 = group8_sum(gx), f1 = group8_sum(gy),
                        f2 = group8_sum(gz);
            while (mk) {  // the groups with a force
                const int g = __builtin_ctzll(mk) >> 3, last = 8 * g + 7;
                mk &= ~(255ull << (8 * g));
                const float w = __builtin_amdgcn_readlane(l, last) == my_link ? 1.f : 0.f;
                S.T0 += w * readlane_f(t0, last);
                S.T1 += w * readlane_f(t1, last);
                S.T2 += w * readlane_f(t2, last);
                S.F0 += w * readlane_f(f0, last);
                S.F1 += w * readlane_f(f1, last);
                S.F2 += w * readlane_f(f2, last);
            }
        }
    };
    // 1. spheres vs boxes: links against the box around all obstacles, then, in scenes with box
    //    clusters (at most 16, of at most 8 boxes), (link, cluster) pairs lane-parallel, the boxes of
    //    the candidate clusters 8 lanes per pair, the spheres of the candidate (link, box) pairs 8
    //    lanes per pair; otherwise each link against 64 boxes at a time
    bool lsurv = false;
    if (lane < L && (W.fc[lane] >> 16) > 0) {
        const float4 c = W.lk[lane];
        const float R = m + c.w + CLR_CULL_EPS;
        lsurv = clr_box_e2(c, make_float4(V.bb_lo[0], V.bb_lo[1], V.bb_lo[2], 0.f),
                           make_float4(V.bb_hi[0], V.bb_hi[1], V.bb_hi[2], 0.f)) <= R * R && V.nb > 0;
    }
    const unsigned long long smask = __ballot(lsurv);
    if (V.nclu > 0 && smask) {
        if (lsurv) W.cand2[lanes_below(smask)] = lane;
        wave_sync();
        const int nsv = __popcll(smask);
        const int lgKG = V.nclu <= 8 ? 3 : 4;  // lanes per link: 8 or 16
        const int per = 64 >> lgKG;
        for (int k0 = 0; k0 < nsv; k0 += per) {
            const int k = k0 + (lane >> lgKG), cc = lane & ((1 << lgKG) - 1);
            const bool in = k < nsv && cc < V.nclu;
            const int l = W.cand2[in ? k : k0];
            const float4 lk = W.lk[l];
            const float R = m + lk.w + CLR_CULL_EPS;
            const int ci = in ? cc : 0;
            const bool cand = in && clr_box_e2(lk, W.clu[2 * ci], W.clu[2 * ci + 1]) <= R * R;
            const unsigned long long mk = __ballot(cand);
            if (mk == 0ull) continue;  // wave-uniform
            if (cand) W.cand[lanes_below(mk)] = l | (cc << 8);
            wave_sync();
            const int nA = __popcll(mk);
            for (int a0 = 0; a0 < nA; a0 += 8) {  // 8 (link, cluster) candidates x 8 boxes
                const int g = lane >> 3, j = lane & 7;
                const bool ga = a0 + g < nA;
                const int c2 = W.cand[ga ? a0 + g : a0];
                const int l2 = c2 & 255, cl = c2 >> 8;
                const int first = __float_as_int(W.clu[2 * cl].w), count = __float_as_int(W.clu[2 * cl + 1].w);
                const bool act = ga && j < count;
                const int b = act ? first + j : 0;
                const float4 lk2 = W.lk[l2];
                const float R2 = m + lk2.w + CLR_CULL_EPS;
                const bool bc = act && clr_box_e2(lk2, W.box[2 * b], W.box[2 * b + 1]) <= R2 * R2;
                unsigned long long bm = __ballot(bc);
                const int code = l2 | (b << 8);
                while (bm) {  // 8 (link, box) candidates x 8 spheres: lane group g takes the g-th set lane
                    int src = -1;
#pragma unroll
                    for (int t = 0; t < 8; ++t) {
                        const int z = bm ? __builtin_ctzll(bm) : -1;
                        bm &= bm - 1ull;
                        src = g == t ? z : src;
                    }
                    const int cd = __shfl(code, src < 0 ? 0 : src, 64);
                    sphere_box(src >= 0, src >= 0 ? cd : 0, j, W.box);
                }
            }
            wave_sync();  // W.cand is rewritten by the next round
        }
    }
    for (unsigned long long lm = V.nclu > 0 ? 0ull : smask; lm; lm &= lm - 1ull) {
        const int l = __builtin_ctzll(lm);
        const float4 lk = W.lk[l];
        const float R = m + lk.w + CLR_CULL_EPS;
        for (int b0 = 0; b0 < V.nb; b0 += 64) {
            const int b = b0 + lane;
            const int bi = b < V.nb ? b : 0;
            const bool cand = b < V.nb && clr_box_e2(lk, V.box32[2 * bi], V.box32[2 * bi + 1]) <= R * R;
            const unsigned long long mk = __ballot(cand);
            if (mk == 0ull) continue;  // wave-uniform
            if (cand) W.cand[lanes_below(mk)] = l | (b << 8);
            wave_sync();
            const int n = __popcll(mk);
            for (int c0 = 0; c0 < n; c0 += 8) {  // 8 candidates x 8 spheres per round
                const int k = c0 + (lane >> 3);
                sphere_box(k < n, W.cand[k < n ? k : c0], lane & 7, V.box32);
            }
            wave_sync();  // W.cand is rewritten by the next round
        }
    }
    // 2. sphere pairs of the link pairs in the pair set
    for (int p0 = 0; p0 < V.NP; p0 += 64) {
        const int pi = p0 + lane;
        const bool in = pi < V.NP;
        int2 pr;
        if (V.NP <= ARM_PAIRS_LDS_MAX) {
            const unsigned long long v = ((lds_cu64*)W.pairs)[in ? pi : p0];
            pr = make_int2((int)(unsigned)v, (int)(unsigned)(v >> 32));
        } else {
            pr = V.lpairs2[in ? pi : p0];
        }
        const float4 A = W.lk[(pr.x >> 8) & 255], B = W.lk[pr.x & 255];
        const float dx = A.x - B.x, dy = A.y - B.y, dz = A.z - B.z;
        const float R = m + A.w + B.w + CLR_CULL_EPS;
        const bool cand = in && clr_sq(dx, dy, dz) <= R * R;
        unsigned long long mk = __ballot(cand);
        while (mk) {  // one link pair per round: lane (i, j) of its 8 x 8 spheres
            const int src = __builtin_ctzll(mk);
            mk &= mk - 1ull;
            const int xc = __builtin_amdgcn_readlane(pr.x, src), yc = __builtin_amdgcn_readlane(pr.y, src);
            const int fl = yc & 511, nl = (yc >> 9) & 15, fm = (yc >> 13) & 511, nm = (yc >> 22) & 15;
            const int i = lane >> 3, j = lane & 7;
            const bool act = i < nl && j < nm;
            const float4 ci = W.sph[fl + (act ? i : 0)], cj = W.sph[fm + (act ? j : 0)];
            float gx = 0.f, gy = 0.f, gz = 0.f;
            const bool f = act && clr_term<GRAD>(ci.x - cj.x, ci.y - cj.y, ci.z - cj.z, m + ci.w + cj.w, cost, gx, gy, gz);
            if constexpr (GRAD) {
                unsigned long long hm = __ballot(f);
                if (hm) {
                    if (!f) gx = gy = gz = 0.f;
                    // the opposite force on the second link; c_i x g = c_j x g, since the force acts
                    // along the line of the centres
                    const float w = ((xc >> 8) & 255) == my_link ? 1.f : ((xc & 255) == my_link ? -1.f : 0.f);
                    const float t0 = row16_sum(ci.y * gz - ci.z * gy), t1 = row16_sum(ci.z * gx - ci.x * gz),
                                t2 = row16_sum(ci.x * gy - ci.y * gx), f0 = row16_sum(gx), f1 = row16_sum(gy),
                                f2 = row16_sum(gz);
                    do {  // the rows of 16 lanes with a force
                        const int row = __builtin_ctzll(hm) >> 4, last = 16 * row + 15;
                        hm &= ~(65535ull << (16 * row));
                        S.T0 += w * readlane_f(t0, last);
                        S.T1 += w * readlane_f(t1, last);
                        S.T2 += w * readlane_f(t2, last);
                        S.F0 += w * readlane_f(f0, last);
                        S.F1 += w * readlane_f(f1, last);
                        S.F2 += w * readlane_f(f2, last);
                    } while (hm);
                }
            }
        }
    }
    return cost;
}

template <bool GRAD, bool CHAIN>
__global__ void __launch_bounds__(64 * CLR_MAX_NW, 4) k_clearance(ClrK V, const float* q, long long n, float m,
                                                                  const float* grad_cost, float* cost, float* grad_q) {
    extern __shared__ float4 lds_clr[];
    {
        const int n16 = V.img_bytes >> 4;
        for (int i = threadIdx.x; i < n16; i += blockDim.x) lds_clr[i] = V.img[i];
    }
    __syncthreads();
    const ClrLds W = clr_lds((unsigned char*)lds_clr, V);
    const int lane = wave_lane(), nw = blockDim.x >> 6;
    const long long waves = (long long)gridDim.x * nw, w0 = (long long)blockIdx.x * nw + (threadIdx.x >> 6);
    const int per = n > waves ? 2 : 1;  // waypoints per turn: small batches one per wave
    for (long long r0 = w0 * per; r0 < n; r0 += waves * per) {
        const int k_end = r0 + per <= n ? per : (int)(n - r0);
        clr_fk<CHAIN>(V, W, q + r0 * V.D, k_end);
        for (int k = 0; k < k_end; ++k) {
            const long long r = r0 + k;
            const float4* X = W.X + 3 * V.L * k;
            const float gw = GRAD && grad_cost ? grad_cost[r] : 1.f;  // in flight during the pairs
            for (int s = lane; s < V.S; s += 64) W.sph[s] = clr_point(X + 3 * W.slink[s], W.sphL[s]);
            if (lane < V.L) W.lk[lane] = clr_point(X + 3 * lane, W.lbc[lane]);
            // lane (arm a, joint kj), 8 lanes per arm
            const int a = lane >> 3, kj = lane & 7;
            const bool in = a < V.na && kj < V.dof;
            const int l = in ? a * V.dof + kj : 0;
            ClrSums S = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            float c;
            if (V.broadphase) {
                wave_sync();
                c = clr_pairs<GRAD>(V, W, m, in ? l : -1, S);
            } else {
                if (GRAD)
                    for (int t = lane; t < 6 * V.L; t += 64) W.tf[t] = 0.f;
                wave_sync();
                c = clr_pairs_all<GRAD>(V, W, m);
                wave_sync();
                const float* tf = W.tf + 6 * l;
                if (GRAD && in) S = {tf[0], tf[1], tf[2], tf[3], tf[4], tf[5]};
            }
            if (cost) {
                const float total = wave_sum_f32(c);
                if (lane == 0) cost[r] = total;
            }
            if (GRAD) {
                // g of joint k = z_{k-1} . sum over spheres on links >= k
                // of (c_s - o_{k-1}) x f_s = z_{k-1} . (T_k - o_{k-1} x F_k), T_k and F_k the sums of
                // c_s x f_s and of f_s over the arm's links >= k (suffix sums by lane shifts)
                const float T0 = clr_suffix8(S.T0), T1 = clr_suffix8(S.T1), T2 = clr_suffix8(S.T2),
                            F0 = clr_suffix8(S.F0), F1 = clr_suffix8(S.F1), F2 = clr_suffix8(S.F2);
                if (in) {
                    const float4* P = kj == 0 ? W.base + 3 * a : X + 3 * (l - 1);
                    const float2* P2 = (const float2*)P;  // (R0 R1) (R2 t) per row
                    const float2 p0 = P2[1], p1 = P2[3], p2 = P2[5];
                    const float z0 = p0.x, z1 = p1.x, z2 = p2.x, o0 = p0.y, o1 = p1.y, o2 = p2.y;
                    const bool pr = CHAIN && ((V.prism >> l) & 1ull);  // prismatic: g = z . F
                    const float g = pr ? z0 * F0 + z1 * F1 + z2 * F2
                                       : z0 * (T0 - (o1 * F2 - o2 * F1)) + z1 * (T1 - (o2 * F0 - o0 * F2)) +
                                             z2 * (T2 - (o0 * F1 - o1 * F0));
                    grad_q[r * V.D + l] = gw * g;
                }
            }
            wave_sync();  // the wave's LDS is rewritten for the next waypoint
        }
    }
}

// waves per workgroup and workgroups per CU: the most resident waves in 160 KiB of LDS, 16 at most
// (4 per SIMD, the kernels' register budget)
struct ClrShape {
    int nw, wgs;
    size_t lds;
};
ClrShape clr_shape(const ClrK& K) {
    ClrShape b = {0, 0, 0};
    for (int nw = 1; nw <= CLR_MAX_NW; ++nw) {
        const size_t lds = (size_t)K.img_bytes + (size_t)nw * clr_wave_bytes(K.D, K.L, K.S);
        if (lds > 163840) break;
        const int fit = (int)(163840 / lds), wgs = fit < 16 / nw ? fit : 16 / nw;
        if (wgs * nw > b.nw * b.wgs) b = {nw, wgs, lds};
    }
    return b;
}

// out[r][k] = w[r] x[r][k]: the chain rule of a cost whose gradient is already there.  Bound by
// memory: 16-byte accesses where the rows are a multiple of 4 wide and the tensors aligned.
template <bool VEC>
__global__ void __launch_bounds__(256) k_scale_rows(const float* x, const float* w, long long n, int D, float* out) {
    const long long total = n * D / (VEC ? 4 : 1), step = (long long)gridDim.x * blockDim.x;
    for (long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x; t < total; t += step) {
        if constexpr (VEC) {
            const float c = w[4 * t / D];
            const float4 v = ((const float4*)x)[t];
            ((float4*)out)[t] = make_float4(c * v.x, c * v.y, c * v.z, c * v.w);
        } else {
            out[t] = w[t / D] * x[t];
        }
    }
}

}  // namespace

void launch_scale_rows(const float* x, const float* w, long long n, int D, float* out, hipStream_t st) {
    const bool vec = (D & 3) == 0 && (((uintptr_t)x | (uintptr_t)out) & 15) == 0;
    const long long total = n * D / (vec ? 4 : 1), cap = 16ll * mrcc_internal::device_cus();
    const long long blocks = (total + 255) / 256;
    const int g = (int)(blocks < cap ? blocks : cap);
    if (vec) k_scale_rows<true><<<g, 256, 0, st>>>(x, w, n, D, out);
    else k_scale_rows<false><<<g, 256, 0, st>>>(x, w, n, D, out);
}

void launch_clearance(const SceneRec& sc, const float* q, long long n, float margin,
                      const float* grad_cost, float* cost, float* grad_q, hipStream_t st) {
    ClrK K = sc.clr;
    K.broadphase = sc.arm.broadphase;
    const ClrShape b = clr_shape(K);
    const long long waves = (long long)b.nw * b.wgs * mrcc_internal::device_cus();
    const int blocks = (int)(((n < waves ? n : waves) + b.nw - 1) / b.nw);
#define MRCC_CLR(G, C) k_clearance<G, C><<<blocks, 64 * b.nw, b.lds, st>>>(K, q, n, margin, grad_cost, cost, grad_q)
    if (grad_q) {
        if (K.chain) MRCC_CLR(true, true);
        else MRCC_CLR(true, false);
    } else {
        if (K.chain) MRCC_CLR(false, true);
        else MRCC_CLR(false, false);
    }
#undef MRCC_CLR
}
