// raytrace.hip -- the causal column-density ray trace of the star-on thermo
// operator (Thermodynamics::rayTrace + updateColDen,
// src/Integrators/Thermodynamics.cpp:339-417) and the star geometry kernel.
//
// The reference walks the cells in a causal order (Grid::buildCausal) so
// that a cell's four upstream neighbours (Grid::calculateNearestNeighbours)
// are done before it.  Those neighbours always lie exactly one Chebyshev
// shell (max_d |i_d - star_d|) closer to the star: one step along the ray
// plane and at most one along the other axes, whose offsets are no larger.
// So the GPU sweeps the shells outwards, SWEEP_SHELLS of them per launch.
// Neighbours of zero weight may be in the same shell (ties between axes); they
// are not read (their term is 0 x a finite value, as the reference adds it).
//
// One launch per shell was bound by the launch, not by its few thousand cells
// (26 B each): 71 launches of 6.7 us on a 128^3 grid with the star near its
// centre.  Here a workgroup follows a patch of one face of the shells (a
// face's cells depend only on that face of the shell before, edges and
// corners included) and computes, beside its own cells, those between them
// and the star that a later shell of the launch reads: one step towards the
// star per shell, 1.3 times the cells.  Each shell is now bound by the chain
// of its divisions behind a barrier.  Hydro, cooling and radiation around that
// star, 2 steps (5 traces): 8.32 ms before, 7.46 with 4 shells of 12 x 12
// patches, 7.6 with 8 of 16 x 16 (twice the chain's waves per SIMD), 7.8 with
// 12.

#include <algorithm>

#include <hip/hip_runtime.h>

#include "star_device.hpp"
#include "torchgpu_internal.hpp"

namespace tg {

constexpr int SWEEP_SHELLS = 4, SWEEP_TILE = 12;
constexpr int SWEEP_W = SWEEP_TILE + SWEEP_SHELLS;  // region of the shell before the launch's first
constexpr int SWEEP_THREADS = SWEEP_W * SWEEP_W;

// Offsets from the star, along one axis of a face, of the cells that a tile
// [t, t + SWEEP_TILE) of shell k + j needs at shell k.
__device__ __forceinline__ void sweep_range(int t, int j, int k, int& lo, int& hi) {
    lo = t > 0 ? max(t - j, 0) : t;
    hi = t + SWEEP_TILE - 1 < 0 ? min(t + SWEEP_TILE - 1 + j, 0) : t + SWEEP_TILE - 1;
    lo = max(lo, -k);
    hi = min(hi, k);
}

// updateColDen (Thermodynamics.cpp:339-363) for shells k0 .. k1: tile
// blockIdx.x of the faces f of shell k1 (not clipped: tiles of offsets, w0 of
// them along the first axis from lo0/lo1).  Each thread has one cell per
// shell; COL_DEN + DCOL_DEN, all that the next shell reads, goes through LDS.
// An edge's or a corner's cells are written by the first of their faces.
__global__ __launch_bounds__(SWEEP_THREADS) void coldens_sweep_kernel(StarGeom s, ShellFaces f, int k0, int k1,
                                                                      const double* __restrict__ den,
                                                                      double den_floor, double* col, double* dcol) {
    __shared__ double sum[2][SWEEP_THREADS];
    int q = 0;
    while (q + 1 < f.nf && (long long)blockIdx.x >= f.start[q + 1]) ++q;
    const int l = (int)(blockIdx.x - f.start[q]);
    const int axis = f.axis[q], sg = f.fixed[q];
    const int t0 = f.lo0[q] + l % f.w0[q] * SWEEP_TILE, t1 = f.lo1[q] + l / f.w0[q] * SWEEP_TILE;
    const int px = threadIdx.x % SWEEP_W, py = threadIdx.x / SWEEP_W;
    // the thread's cell of shell k (false: none, or off the grid)
    const auto cell = [&](int k, int ijk[3], int& lo0, int& lo1) {
        int hi0, hi1;
        sweep_range(t0, k1 - k, k, lo0, hi0);
        sweep_range(t1, k1 - k, k, lo1, hi1);
        const int o0 = lo0 + px, o1 = lo1 + py;
        ijk[0] = s.s[0] + (axis == 0 ? sg * k : o0);
        ijk[1] = s.s[1] + (axis == 1 ? sg * k : axis == 0 ? o0 : o1);
        ijk[2] = s.s[2] + (axis == 2 ? sg * k : o1);
        return o0 <= hi0 && o1 <= hi1 && ijk[0] >= 0 && ijk[0] < s.n[0] && ijk[1] >= 0 && ijk[1] < s.n[1] &&
               ijk[2] >= 0 && ijk[2] < s.n[2];
    };
    int ijk[3], lo0 = 0, lo1 = 0;
    if (k0 > 0 && cell(k0 - 1, ijk, lo0, lo1)) {
        const long long c = star_flat(s, ijk[0], ijk[1], ijk[2]);
        sum[(k0 - 1) & 1][threadIdx.x] = col[c] + dcol[c];
    }
    int pl0 = lo0, pl1 = lo1;  // where the region of the shell before starts
    bool mine = cell(k0, ijk, lo0, lo1);
    double den_next = mine ? den[star_flat(s, ijk[0], ijk[1], ijk[2])] : 0.0;
    for (int k = k0; k <= k1; ++k) {
        __syncthreads();
        const double den_raw = den_next;
        const int c0 = lo0, c1 = lo1, me[3] = {ijk[0], ijk[1], ijk[2]};
        const bool on = mine;
        if (k < k1) {  // the next shell's density is on its way meanwhile
            mine = cell(k + 1, ijk, lo0, lo1);
            if (mine) den_next = den[star_flat(s, ijk[0], ijk[1], ijk[2])];
        }
        if (on) {
            // floored as fixPrimitives floors it (den_floor -HUGE_VAL: as given)
            const double den_c = den_raw < den_floor ? den_floor : den_raw;
            // distance to the star in cell units
            double dist2 = 0;
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                const double e = star_offset(s, me, a);
                dist2 += e * e;
            }
            double v = 0;
            if (dist2 > 0.95 * 0.95) {
                int nbc[4][3];
                bool valid[4];
                double w[4], cd[4], wr[4];
                star_neighbour_cells(s, me, nbc, valid, w);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    cd[j] = 0.0;
                    // its place in the region before: in range by construction
                    const int n0 = (axis == 0 ? nbc[j][1] - s.s[1] : nbc[j][0] - s.s[0]) - pl0;
                    const int n1 = (axis == 2 ? nbc[j][1] - s.s[1] : nbc[j][2] - s.s[2]) - pl1;
                    if (valid[j] && w[j] != 0.0 && (unsigned)n0 < SWEEP_W && (unsigned)n1 < SWEEP_W)
                        cd[j] = sum[(k - 1) & 1][n1 * SWEEP_W + n0];
                    wr[j] = cd[j] == 0 ? 0.0 : w[j] / cd[j];
                }
                const double sum_w = wr[0] + wr[1] + wr[2] + wr[3];
                if (sum_w != 0) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) v += (wr[j] / sum_w) * cd[j];
                }
            }
            const double dc = (den_c / s.hydrogen_mass) * star_path_length(s, me);
            sum[k & 1][threadIdx.x] = v + dc;
            const int ox = me[0] - s.s[0], oy = me[1] - s.s[1], oz = me[2] - s.s[2];
            const int o0 = axis == 0 ? oy : ox, o1 = axis == 2 ? oy : oz;
            const bool first = axis == 0 ? (k > 0 || sg > 0) : (ox > -k && ox < k && (axis == 1 || (oy > -k && oy < k)));
            if (first && o0 >= t0 && o0 < t0 + SWEEP_TILE && o1 >= t1 && o1 < t1 + SWEEP_TILE) {
                const long long c = star_flat(s, me[0], me[1], me[2]);
                col[c] = v;
                dcol[c] = dc;
            }
        }
        pl0 = c0;
        pl1 = c1;
    }
}

__global__ void star_geometry_kernel(StarGeom s, long long* __restrict__ nb, double* __restrict__ w,
                                     double* __restrict__ ds, double* __restrict__ shell_vol) {
    const long long n = (long long)s.n[0] * s.n[1] * s.n[2];
    for (long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x; c < n; c += (long long)gridDim.x * blockDim.x) {
        const int ijk[3] = {(int)(c % s.n[0]), (int)((c / s.n[0]) % s.n[1]), (int)(c / ((long long)s.n[0] * s.n[1]))};
        long long b[4];
        double wq[4];
        star_neighbours(s, ijk, b, wq);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            nb[4 * c + q] = b[q];
            w[4 * c + q] = wq[q];
        }
        const double d = star_path_length(s, ijk);
        ds[c] = d;
        shell_vol[c] = star_shell_volume(s, ijk, d);
    }
}

// Faces of shell k clipped to the grid (see ShellFaces).
void shell_faces(const StarGeom& s, int k, ShellFaces& f) {
    f.nf = 0;
    f.start[0] = 0;
    auto add = [&](int axis, int fixed, int lo0, int hi0, int lo1, int hi1) {
        const int b0 = axis == 0 ? 1 : 0, b1 = axis == 2 ? 1 : 2;
        if (fixed < 0 || fixed >= s.n[axis]) return;
        lo0 = lo0 < 0 ? 0 : lo0;
        lo1 = lo1 < 0 ? 0 : lo1;
        hi0 = hi0 > s.n[b0] - 1 ? s.n[b0] - 1 : hi0;
        hi1 = hi1 > s.n[b1] - 1 ? s.n[b1] - 1 : hi1;
        if (hi0 < lo0 || hi1 < lo1) return;
        const int q = f.nf++;
        f.axis[q] = axis;
        f.fixed[q] = fixed;
        f.lo0[q] = lo0;
        f.lo1[q] = lo1;
        f.w0[q] = hi0 - lo0 + 1;
        f.start[q + 1] = f.start[q] + (long long)f.w0[q] * (hi1 - lo1 + 1);
    };
    const int x = s.s[0], y = s.s[1], z = s.s[2];
    if (k == 0) {
        add(0, x, y, y, z, z);
        return;
    }
    for (int sgn = -1; sgn <= 1; sgn += 2) add(0, x + sgn * k, y - k, y + k, z - k, z + k);
    for (int sgn = -1; sgn <= 1; sgn += 2) add(1, y + sgn * k, x - k + 1, x + k - 1, z - k, z + k);
    for (int sgn = -1; sgn <= 1; sgn += 2) add(2, z + sgn * k, x - k + 1, x + k - 1, y - k + 1, y + k - 1);
}

int shell_max(const StarGeom& s) {
    int kmax = 0;
    for (int a = 0; a < 3; ++a) {
        const int m = s.s[a] > s.n[a] - 1 - s.s[a] ? s.s[a] : s.n[a] - 1 - s.s[a];
        kmax = m > kmax ? m : kmax;
    }
    return kmax;
}

// The tiles of the faces of shell k1 that lie on the grid at shell k0: fixed
// is the face's side (-1, 1), lo0/lo1 the first tiles' offsets.
static void sweep_tiles(const StarGeom& s, int k0, int k1, ShellFaces& f) {
    f.nf = 0;
    f.start[0] = 0;
    const auto tiles = [&](int a, int& lo) {  // along axis a
        const int o_lo = std::max(-k1, -s.s[a]), o_hi = std::min(k1, s.n[a] - 1 - s.s[a]);
        lo = -((-o_lo + SWEEP_TILE - 1) / SWEEP_TILE) * SWEEP_TILE;
        return (o_hi - lo) / SWEEP_TILE + 1;
    };
    for (int axis = 0; axis < 3; ++axis)
        for (int sg = -1; sg <= 1; sg += 2) {
            const int at = s.s[axis] + sg * k0;
            if (at < 0 || at >= s.n[axis]) continue;
            const int q = f.nf++;
            f.axis[q] = axis;
            f.fixed[q] = sg;
            f.w0[q] = tiles(axis == 0 ? 1 : 0, f.lo0[q]);
            f.start[q + 1] = f.start[q] + (long long)f.w0[q] * tiles(axis == 2 ? 1 : 2, f.lo1[q]);
        }
}

hipError_t launch_thermo_ray_trace(const StarGeom& s, const double* den, double den_floor, double* col, double* dcol,
                                   hipStream_t stream) {
    const int kmax = shell_max(s);
    ShellFaces f;
    for (int k0 = 0; k0 <= kmax; k0 += SWEEP_SHELLS) {
        const int k1 = std::min(k0 + SWEEP_SHELLS - 1, kmax);
        sweep_tiles(s, k0, k1, f);
        hipLaunchKernelGGL(coldens_sweep_kernel, dim3((unsigned)f.start[f.nf]), dim3(SWEEP_THREADS), 0, stream, s, f,
                           k0, k1, den, den_floor, col, dcol);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t launch_star_geometry(const StarGeom& s, long long* nb, double* w, double* ds, double* shell_vol,
                                hipStream_t stream) {
    const long long n = (long long)s.n[0] * s.n[1] * s.n[2];
    long long b = (n + 255) / 256;
    if (b > 65536) b = 65536;
    hipLaunchKernelGGL(star_geometry_kernel, dim3((unsigned)b), dim3(256), 0, stream, s, nb, w, ds, shell_vol);
    return hipGetLastError();
}

}  // namespace tg
