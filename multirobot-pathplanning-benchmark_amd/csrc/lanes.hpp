// lanes.hpp — what the edge kernels share: rows, interpolation, verdict bytes, and the choice of
// the lane-per-state evaluator.
#pragma once

#include "engine.hpp"

using namespace mrcc;

__device__ inline void stat_add(unsigned long long* stats, int idx, unsigned long long v) {
    if (stats && v) atomicAdd(stats + idx, v);
}

// row pointers of edge e
__device__ inline const double* row1(const EdgeBatchView& B, long long e) {
    long long r = B.idx1 ? (long long)B.idx1[e] : e;
    return B.q1 + r * B.rs;
}
__device__ inline const double* row1(const ArmQueue& B, long long e) {
    long long r = B.idx1 ? (long long)B.idx1[e] : e;
    return B.q1 + r * B.rs;
}
__device__ inline const double* row2(const EdgeBatchView& B, long long e) {
    long long r = B.idx2 ? (long long)B.idx2[e] : e;
    return B.q2 + r * B.rs;
}

__device__ inline const double* row2(const ArmQueue& B, long long e) {
    long long r = B.idx2 ? (long long)B.idx2[e] : e;
    return B.q2 + r * B.rs;
}

// What the kernel that forms a queue's records clears for the kernels after it.
__device__ inline void plan_prep_clear(const PlanWork& W) {
    for (int b = blockIdx.x * blockDim.x + threadIdx.x; b <= MRCC_MAX_PASSES; b += gridDim.x * blockDim.x) W.cursor[b] = 0;
    if (blockIdx.x == 0 && threadIdx.x < 8) W.ticket[32 * threadIdx.x] = 0;
}

// interpolated state (abstract_env.py:341, :348): q1 + ((q2 - q1) / (N - 1)) * i, unfused
__device__ inline double interp_f64(double a, double b, int N, int i) {
#pragma clang fp contract(off)
    double dir = (b - a) / (double)(N - 1);
    return a + dir * (double)i;
}
__device__ inline double interp_dir_f64(double a, double dir, int i) {
#pragma clang fp contract(off)
    return a + dir * (double)i;
}

// binary64 interpolation step of one coordinate, (b - a) / (N - 1), as interp_f64 forms it
__device__ inline double interp_step_f64(double a, double b, int N) {
#pragma clang fp contract(off)
    return (b - a) / (double)(N - 1);
}

// The verdict byte of an edge in the persistent kernels, as every XCD sees it: another wave
// writes an edge's 0 when one of its states collides, and the later slots of the edge are skipped
// when they read it.  Each XCD has its own L2 and plain accesses may stay in it (a plain read can
// return an XCD's stale copy until the kernel ends); agent-scope accesses reach the level that all
// XCDs share.  (The direct kernels keep plain accesses: there the agent-scope ones measured slower,
// 47 -> 248 us for a list of 30 arm edges with 64 waves per edge.)
__device__ inline bool edge_dead(const unsigned char* out, int e) {
    return __hip_atomic_load(out + e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0;
}
__device__ inline void edge_kill(unsigned char* out, int e) {
    __hip_atomic_store(out + e, (unsigned char)0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Disks in the plane: <DiskGridView, 2, NRB>, at most NRB robots; planar boxes: <PlanarGridView, NRB, 0>,
// likewise.  Views without the table (LaneKind::all): every obstacle is tested, by the evaluators that are
// the faster ones then: <DiskView, 2, 2> two disks in the plane, <DiskView, 0, 0> any disks,
// <PlanarView, 4, 0> four boxes, <PlanarView, 0, 0> any number.
template <class View>
struct LaneKind {
    static constexpr bool planar = std::is_base_of<PlanarView, View>::value;
    static constexpr bool all = std::is_same<View, DiskView>::value || std::is_same<View, PlanarView>::value;
};
// register length of the per-lane state
template <class View, int T1, int T2>
struct LaneDim {
    static constexpr int value = LaneKind<View>::planar ? 3 * (T1 ? T1 : MRCC_PLANAR_MAX_ROBOTS)
                                                        : (T1 ? T1 * T2 : MRCC_DISK_MAX_RD * 4);
};

// Calls F(view, T1, T2) with the smallest bounds that hold the scene.
// Without a table, us of 200,000 configurations by planar_collides / disk_collides and by
// planar_state / disk2_state with every obstacle: 4 boxes 85 / 120, 2 disks 34 / 38; 1 and 2 boxes 87 / 46, 55 /
// 36, 1, 3 and 4 disks 162 / 37, 568 / 134, 787 / 177; 8 boxes 264 / 249, but queues of 200,000 edges 1,271 /
// 1,430.
template <class F>
static void lane_dispatch(const SceneRec& sc, F f) {
    using std::integral_constant;
    const integral_constant<int, 0> c0{};
    const integral_constant<int, 2> c2{};
    const integral_constant<int, 4> c4{};
    if (sc.kind == KIND_DISKS) {
        const DiskGridView& V = sc.disk;
        const DiskView& all = V;
        if (V.rd != 2 || V.nr > 4) f(all, c0, c0);
        else if (V.nr == 2 && V.grid.n == 0) f(all, c2, c2);
        else if (V.nr <= 2) f(V, c2, c2);
        else f(V, c2, c4);
    } else {
        const PlanarGridView& V = sc.planar;
        const PlanarView& all = V;
        const bool none = V.grid.n == 0;
        if (V.nr == 4 && none) f(all, c4, c0);
        else if (V.nr <= 4) f(V, c4, c0);
        else if (none) f(all, c0, c0);
        else if (V.nr <= 8) f(V, integral_constant<int, 8>(), c0);
        else f(V, integral_constant<int, MRCC_PLANAR_MAX_ROBOTS>(), c0);
    }
}
