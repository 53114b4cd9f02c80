// engine.hpp — host-side records of the collision engine and the kernel launchers.
#pragma once

#include "../../include/mrcc.h"
#include "evaluators.hpp"

#include <algorithm>

// An arm scene as the clearance kernels see it: scalars and the binary32 tables as one image that a
// workgroup stages in LDS (clr_layout); tables too large for it are read from global memory.
struct ClrK {
    int na, dof, D, L, S, nb, NP, nclu, chain, broadphase;
    unsigned long long prism;
    float bb_lo[3], bb_hi[3];
    const float4* img;
    int img_bytes;
    const float4* box32;  // [nb*2] lo, hi
    const int2* lpairs2;  // [NP]
    const int* sph_lo;    // [S]
};
struct ClrLayout {
    int o_joint, o_base, o_sph, o_lbc, o_fc, o_slink, o_box, o_clu, o_pairs, bytes;
};
__host__ __device__ inline ClrLayout clr_layout(int L, int na, int nb, int S, int NP, int nclu, int chain) {
    ClrLayout o;
    int b = 0;
    o.o_joint = b;  b += 16 * (chain ? 3 : 1) * L;  // d a cos(alpha) sin(alpha), or the rows of C
    o.o_base = b;   b += 48 * na;                   // rows R0 R1 R2 t
    o.o_sph = b;    b += 16 * S;                    // centre in the link frame, radius
    o.o_lbc = b;    b += 16 * L;                    // bounding-sphere centre in the link frame, radius
    o.o_fc = b;     b += align16(4 * L);            // first sphere | count << 16
    o.o_slink = b;  b += align16(4 * S);            // link of each sphere
    o.o_box = b;    b += (nclu > 0 ? 32 * nb : 0);
    o.o_clu = b;    b += 32 * nclu;
    o.o_pairs = b;  b += (NP <= ARM_PAIRS_LDS_MAX ? align16(8 * NP) : 0);
    o.bytes = b;
    return o;
}

// A scene as held by the library: the kind, its device view and the device allocation behind it.
struct SceneRec {
    int kind;
    int D;
    int n_robots;
    int device;
    DiskGridView disk;
    PlanarGridView planar;
    ArmView arm;          // every array of an arm scene (clearance and kinematics kernels)
    ArmK armk;            // the edge and configuration kernels' view of the same scene
    ClrK clr;             // the clearance kernels' view
    size_t arm_lds;       // dynamic LDS bytes of the arm kernels (arm_nw waves per workgroup)
    size_t arm_lds1;      // dynamic LDS bytes of an arm kernel with one wave per workgroup
    int arm_nw;           // waves per workgroup of the arm kernels
    int arm_nw_pers;      // waves per workgroup of the persistent kernel
    int arm_wg_pers;      // its resident workgroups per CU (registers and LDS)
    int arm_blocks_pers;  // its largest useful grid: resident workgroups on every CU
    size_t arm_lds_pers;  // its dynamic LDS bytes
    int arm_nw_edge;      // waves of the per-call kernel's one workgroup
    size_t arm_lds_edge;  // its dynamic LDS bytes
    void* dev_mem;        // one allocation holding every array the views point to
    size_t dev_bytes;
    // host copies needed by host code
    int arm_na, arm_dof, arm_S, arm_nm;
    int arm_has_grasp;    // some mode holds a box: the evaluator with the held-box phase
    // staging block of the host-pointer per-call entry points (lazily allocated): pinned coherent
    // host memory, read and written by the kernels in place; stage_dev is its device address
    double* stage_dev;
    double* stage_host;
    unsigned char* stage_out_dev;
    unsigned char* stage_out_host;
    // staging of the host-memory batch entry point (grown on demand)
    unsigned char* batch_dev;
    unsigned char* batch_host;
    size_t batch_cap;
    // block of the short host lists (at most MRCC_HOST_LIST_ZC edges): pinned coherent host memory
    // that the kernels read and write in place; list_dev is its device address; a flag byte after
    // the verdicts is set by a one-thread kernel after the check
    unsigned char* list_host;
    unsigned char* list_dev;
};

// `clear`: the workspace is not as a finished run (or launch_plan_clear) left it
void launch_plan_build(const SceneRec& sc, const EdgeBatchView& B, const PlanWork& W, int lgG, bool clear,
                       hipStream_t st);
void launch_plan_clear(const PlanWork& W, hipStream_t st);
void launch_plan_run(const SceneRec& sc, const EdgeBatchView& B, const PlanWork& W, int lgG,
                     int spt, int grid, hipStream_t st);
void launch_direct(const SceneRec& sc, const EdgeBatchView& B, int wpe, int init_out, int max_grid,
                   unsigned long long* stats, hipStream_t st);
// lane_looks.hip: edge batches of plane scenes with a cell table, two launches, no queue; W.meta is
// zero before the workspace's first run (`reset`: cleared here, for workspaces used otherwise too)
bool lane_looks_apply(const SceneRec& sc);
void launch_lane_looks(const SceneRec& sc, const EdgeBatchView& B, const PlanWork& W, bool reset, hipStream_t st);
#define MRCC_NO_QUEUE (-1)  // lgG of such a run
// cells.hip: fills the cell table of a plane scene; tally: two zeroed device words or null
void launch_cells(const SceneRec& sc, int* tally, hipStream_t st);
void cell_size(const CellGrid& C, double* hd, double* slack);
void launch_fill_u8(unsigned char* p, long long n, unsigned char v, hipStream_t st);
// plain per-call form: edge 0 of B in one workgroup (k_arm_edge / k_lane_edge)
void launch_edge1(const SceneRec& sc, const EdgeBatchView& B, hipStream_t st);
// one thread writes 1 to *flag (after the work queued before it on the stream)
void launch_flag(unsigned char* flag, hipStream_t st);
// one configuration (row q1 of B) of a disk or planar scene: the per-call lane kernel, obstacles
// split over lanes
void launch_config1(const SceneRec& sc, const EdgeBatchView& B, hipStream_t st);
// k_arm_edge on `blocks` workgroups (blocks > 1: the verdict must be preset to 1)
void launch_arm_edge_spread(const SceneRec& sc, const EdgeBatchView& B, int blocks, hipStream_t st);
void launch_configs(const SceneRec& sc, const double* q, long long n, long long rs, long long ds,
                    const int* modes, unsigned mask, unsigned char* out, int max_grid,
                    hipStream_t st);
// self-collision screen of arm states (screen.hip), ahead of the full evaluators
bool arm_screen_applies(const SceneRec& sc, long long n, long long n_min);
// From these sizes on.  us with the screen / without, 2, 4 and 6 arms of 7 joints, 50 boxes: 512 uniform edges 50 /
// 46, 47 / 43, 54 / 43, 1,536: 51 / 56, 50 / 46, 53 / 47, 4,096: 53 / 66, 52 / 60, 55 / 63 (0.4 rad around home: 49 /
// 58, 54 / 61, 65 / 65; 56 / 87, 58 / 79, 68 / 82; 67 / 92, 74 / 83, 85 / 106).  Configurations 0.4 rad around home,
// where it catches least: 16,384: 55 / 47, 65 / 52, 99 / 105, 49,152: 97 / 107, 115 / 121, 158 / 270; uniform ones
// 47 / 43, 43 / 45, 46 / 78 and 68 / 93, 49 / 98, 52 / 196.
#define MRCC_SCREEN_MIN_EDGES 1536
#define MRCC_SCREEN_MIN_CONFIGS 49152
void launch_screen_edges(const SceneRec& sc, const EdgeBatchView& B, const PlanWork& W, int lgG, hipStream_t st);
void launch_screen_configs(const SceneRec& sc, const double* q, long long n, long long rs, long long ds,
                           const int* modes, unsigned mask, unsigned char* out, hipStream_t st);
void launch_arm_fk(const SceneRec& sc, const double* q, long long n, long long rs, long long ds,
                   double* out, hipStream_t st);
void launch_sincos(const double* x, long long n, double* s, double* c, hipStream_t st);
void launch_clearance(const SceneRec& sc, const float* q, long long n, float margin,
                      const float* grad_cost, float* cost, float* grad_q, hipStream_t st);
void launch_scale_rows(const float* x, const float* w, long long n, int D, float* out, hipStream_t st);

// configuration-pair costs (cost.hip): row r of the result reduces d = P[r*ps + k] - Q[r*qs + k]
// (k < D) over the slices [sl[2i], sl[2i+1])
#define MRCC_COST_MAX_SLICES 64
#define MRCC_COST_MAX_D 1024
#define MRCC_COST_TILE_BYTES 8192  // LDS of one workgroup's tile of rows (narrow rows)
struct CostArgs {
    const double* P;
    long long ps;
    const double* Q;
    long long qs;
    long long n;
    int D, ns, metric, red;
    double w;
    double* out;
    int sl[2 * MRCC_COST_MAX_SLICES];
};
void launch_config_cost(const CostArgs& A, int max_grid, hipStream_t st);

// api.hip internals shared with the no-allocation entry point (noalloc.hip)
namespace mrcc_internal {
int fail(int code, const char* fmt, ...);  // sets the thread's last-error message, returns code
int injected();                            // an injected failure (mrcc_debug_inject_failure), or 0
int device_cus();
const SceneRec* scene_rec(const mrcc_scene* s);
int check_batch(const SceneRec* sc, const mrcc_edge_batch* b);
EdgeBatchView batch_view(const mrcc_edge_batch* b);
// execution shape: defaults filled in and checked (mrcc_edge_plan_create's rules)
int tune_defaults(const SceneRec* sc, const mrcc_tune* tune, mrcc_tune* t);
int plan_grid(const SceneRec* sc, const mrcc_tune& t);
// Bytes of a plan's workspace for n_edges edges; with W, lays it out from base.  D: coordinates of the
// stored steps, 0 without them (plan_step_dim).
size_t plan_layout(long long n_edges, int D, unsigned char* base, PlanWork* W);
int plan_step_dim(const SceneRec* sc, const mrcc_tune& t);
// queue build and persistent kernel on stream st (lgG = MRCC_NO_QUEUE: the two launches of
// lane_looks.hip); `clear` as for launch_plan_build
void launch_plan_sequence(const SceneRec& sc, const EdgeBatchView& B, const PlanWork& W, int lgG, int spt,
                          int grid, hipStream_t st, bool clear);
int plan_lgG(const mrcc_tune& t);
}  // namespace mrcc_internal

// noalloc.hip: looks up the current device's scratch array (called by mrcc_init)
int mrcc_noalloc_setup();
