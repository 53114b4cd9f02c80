// cells.hip — the cell table of plane scenes (CellGrid), built on the device when a scene is made.
#include "engine.hpp"

namespace {

// One thread per (robot, cell): every obstacle's distance to the cell's centre against the robot's
// circumscribed and inscribed radii, widened by the cell's half diagonal and the slack.
// Triangle inequality: a centre within `hd` of the cell's centre is at d - hd .. d + hd from the
// obstacle; beyond the circumscribed radius nothing overlaps (and a separating axis of the two boxes
// exceeds the gap over sqrt 2), within the inscribed radius the overlap is certain.
// 128 x 128 cells: 10 us (2 disks, 20 rectangles), 30 us (4 boxes, 100 obstacles), once per scene.
__device__ inline void cell_fill(CellGrid C, double hd, double slack, int i, double r_in, double r_out, int n_obs,
                                 int t, const DiskView* D, const PlanarView* P, int* tally) {
    const int cy = t / C.n, cx = t - cy * C.n;
    const double x = (double)C.x0 + (cx + 0.5) / (double)C.ix, y = (double)C.y0 + (cy + 0.5) / (double)C.iy;
    unsigned short h[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    const double wx = 0.5 / (double)C.ix, wy = 0.5 / (double)C.iy;
    unsigned n = 0;
    int own = 0;  // obstacles centred in the cell
    // obstacles through LDS, 64 at a time: read one by one they were a chain of dependent round trips
    // (100 boxes: 40 us)
    __shared__ double s_ob[64][8];
    for (int o = 0; o < n_obs; ++o) {
        if ((o & 63) == 0) {
            __syncthreads();
            const int k = threadIdx.x >> 2, c = (threadIdx.x & 3) * 2, u = o + k;  // 256 threads: 2 words each
            if (u < n_obs) {
                double v[2] = {0.0, 0.0};
                if (P) {
                    v[0] = P->ob64[8 * u + c];
                    v[1] = P->ob64[8 * u + c + 1];
                } else if (u < D->ns) {
                    if (c == 0) v[0] = D->sc64[2 * u], v[1] = D->sc64[2 * u + 1];
                    if (c == 2) v[0] = D->srT64[i * D->ns + u];
                } else if (c < 4) {
                    const double* e = (c == 0 ? D->lo64 : D->hi64) + 2 * (u - D->ns);
                    v[0] = e[0];
                    v[1] = e[1];
                }
                s_ob[k][c] = v[0];
                s_ob[k][c + 1] = v[1];
            }
            __syncthreads();
        }
        const double* b = s_ob[o & 63];
        if (tally) {
            const bool rect = !P && o >= D->ns;
            own += fabs(x - (rect ? 0.5 * (b[0] + b[2]) : b[0])) <= wx && fabs(y - (rect ? 0.5 * (b[1] + b[3]) : b[1])) <= wy;
        }
        if (n == CELL_HIT) continue;
        double d2, lo = r_in, hi = r_out;  // squared distance
        if (P) {
            const double tx = x - b[0], ty = y - b[1];
            const double ex = fmax(fabs(tx * b[2] + ty * b[3]) - b[6], 0.0);
            const double ey = fmax(fabs(tx * b[4] + ty * b[5]) - b[7], 0.0);
            d2 = ex * ex + ey * ey;
        } else if (o < D->ns) {
            const double tx = x - b[0], ty = y - b[1];
            d2 = tx * tx + ty * ty;
            lo = hi = sqrt(b[2]);  // the sum of the radii, to rounding
        } else {
            const double ex = fmax(fmax(b[0] - x, x - b[2]), 0.0);
            const double ey = fmax(fmax(b[1] - y, y - b[3]), 0.0);
            d2 = ex * ex + ey * ey;
        }
        const double far = hi + slack + hd, near = lo - slack - hd;
        if (d2 > far * far) continue;
        if (near > 0.0 && d2 < near * near) {
            n = CELL_HIT;
            continue;
        }
        if (n <= CELL_LIST) ++n;  // no further: 65,535 of them would read as CELL_HIT
#pragma unroll
        for (int k = 1; k <= CELL_LIST; ++k)
            if ((int)n == k) h[k] = (unsigned short)o;
    }
    if (n != CELL_HIT && n > CELL_LIST) n = CELL_MANY;
    if (t >= C.n * C.n) return;
    uint4 r;
    r.x = n | ((unsigned)h[1] << 16);
    r.y = h[2] | ((unsigned)h[3] << 16);
    r.z = h[4] | ((unsigned)h[5] << 16);
    r.w = h[6] | ((unsigned)h[7] << 16);
    ((uint4*)C.rec)[(size_t)i * C.n * C.n + t] = r;
    if (own) {
        atomicAdd(tally, own);
        atomicAdd(tally + 1, own * (n == CELL_HIT ? 0 : min((int)n, CELL_LIST + 1)));
    }
}

__global__ void __launch_bounds__(256) k_cells_disk(DiskGridView S, double hd, double slack, int* tally) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x, i = blockIdx.y;
    const double r = sqrt(S.rp2_64[i]);
    cell_fill(S.grid, hd, slack, i, r, r, S.ns + S.nrect, t, &S, nullptr, tally);
}

__global__ void __launch_bounds__(256) k_cells_planar(PlanarGridView S, double hd, double slack, int* tally) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x, i = blockIdx.y;
    const double a = S.rh64[2 * i], b = S.rh64[2 * i + 1];
    cell_fill(S.grid, hd, slack, i, fmin(a, b), sqrt(a * a + b * b), S.no, t, nullptr, &S, tally);
}

}  // namespace

// Fills the table that sc's view points to (grid.rec, corner and scale set).  tally[0] counts the
// obstacles by the cells that hold their centres, over all robots, tally[1] the tests that those cells
// leave open (none where contact is certain, 8 for CELL_MANY); null: not counted.
void launch_cells(const SceneRec& sc, int* tally, hipStream_t st) {
    const CellGrid& C = sc.kind == KIND_DISKS ? sc.disk.grid : sc.planar.grid;
    double hd, slack;
    cell_size(C, &hd, &slack);
    const dim3 grid((C.n * C.n + 255) / 256, sc.n_robots);
    if (sc.kind == KIND_DISKS) k_cells_disk<<<grid, 256, 0, st>>>(sc.disk, hd, slack, tally);
    else k_cells_planar<<<grid, 256, 0, st>>>(sc.planar, hd, slack, tally);
}

// half diagonal of a cell, slack of the table
void cell_size(const CellGrid& C, double* hd, double* slack) {
    const double wx = 1.0 / (double)C.ix, wy = 1.0 / (double)C.iy;
    const double ext = std::max(std::max(fabs((double)C.x0), fabs((double)C.y0)), C.n * std::max(wx, wy));
    *hd = 0.5 * sqrt(wx * wx + wy * wy);
    *slack = cell_slack(ext, std::max(wx, wy));
}
