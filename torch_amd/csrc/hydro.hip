// hydro.hip -- fused hydro stage kernels for CDNA4 (gfx950).
//
// One launch = one stage of the reference's midpoint predictor-corrector
// (Torch::hydroStep, src/Torch/Torch.cpp:366-387) over the whole grid:
//
//   Q   = QfromU(Usrc)                       (+ fixPrimitives in stage 1)
//   ghost cells by boundary condition        Grid::applyBCs, Grid.cpp:649-802
//   QL/QR = linear reconstruction            Hydrodynamics::reconstruct, Hydro.cpp:44-67
//   F    = Riemann solve per face            Hydrodynamics::calcFluxes, Hydro.cpp:91-115
//   UDOT = sum_dim (A/V)(F_left - F_right)   Hydrodynamics::updateSourceTerms, Hydro.cpp:117-137
//   Udst = fixSolution(Ubase + dtf * UDOT)   Fluid::advSolution/fixSolution, Fluid.cpp:80-136
//   stage 2 only: max_cells inv_t of fixPrimitives(QfromU(Udst)), the CFL
//   reduction of the next step (Hydro.cpp:77-89), via wave shuffles + one
//   atomicMax per block on the bit pattern of a non-negative double.
//
// Data layout: conserved state U is structure-of-arrays in HBM,
// U[v * ncell + x + nx * (y + ny * z)], v in UID order, x fastest.
//
// These are the FP64 parity kernels: compiled with -ffp-contract=off they
// keep the reference's operand order and are bitwise equal to its x86-64
// build.  Two layouts of one stage, chosen by the grid's size
// (launch_hydro_stage):
//
//  hydro_march_kernel  a workgroup of 256 threads owns a 16 x 16 column of
//      cells and marches it along z.  Each thread keeps the primitives of its
//      column at planes k .. k+2, the limited z slope of plane k and the last
//      z flux in registers; plane k with its 2-deep x and y halos, and each
//      cell's x and y slope (limited once for both its faces), go through
//      LDS.  Per cell 3.125 face solves (and 1/planes), 21 limited slopes and
//      1.5 cell loads, where the 8^3 tiles this replaces took 3.375, 47 and
//      2.5; 72 KB of LDS and 256 registers leave two workgroups per CU (eight
//      waves on four SIMDs), where those tiles' 140 KB left one of nine waves.
//  hydro_tile_kernel   an 8 x 4 x 4 tile per workgroup of 512 threads, all
//      faces of the three directions solved at once, one per thread: a grid
//      too small to fill the chip is bound by the length of one workgroup's
//      serial chain, here one load, one solve and one update, where the
//      tiles took three sweeps and a march takes a solve per plane.
//
// Workgroups are handed out XCD-contiguously (consecutive workgroups
// round-robin over the 8 XCDs, so workgroup b is given tile (b % 8) *
// (ntiles / 8) + b / 8) so that each XCD's L2 sees neighbouring halos.  The
// mixed-precision kernel is in hydro_mixed.hip.

#include <type_traits>

#include "hydro_device.hpp"

namespace tg {

// Limited slope of cell b between its neighbours a and c (0 at first order).
// ALB: van Albada, the default, without the other limiters' code.
// FAST: the three cells keep the divisions in range (Recip, hydro_math.hpp).
template <bool ALB, bool FAST>
__device__ __forceinline__ void cell_slope(const HydroGeom& g, const double a[7], const double b[7], const double c[7],
                                           double s[7]) {
    if (g.spatial_order == 1) {
#pragma unroll
        for (int v = 0; v < 7; ++v) {
            if constexpr (ALB) s[v] = albada<FAST>(b[v] - a[v], c[v] - b[v]);
            else s[v] = limiter<double>(g.limiter, b[v] - a[v], c[v] - b[v]);
        }
    } else {
#pragma unroll
        for (int v = 0; v < 7; ++v) s[v] = 0.0;
    }
}

// Flux along DIM through the face between cells b and c with limited slopes
// sb and sc: QR of b and QL of c (Hydrodynamics::reconstruct) and the Riemann
// solve.  yswap (DIM 0): a y face, solved as an x face with the x and y
// velocity components exchanged (see hydro_math.hpp).  Returns true if the
// HII flux is NaN or, FAST, the flux not to be trusted.
template <int SOLVER, int DIM, bool FAST>
__device__ __forceinline__ bool slope_flux(const HydroGeom& g, const double b[7], const double sb[7], const double c[7],
                                           const double sc[7], const GasConsts<double>& gc, double F[7],
                                           bool yswap = false) {
    double ql[7], qr[7];
#pragma unroll
    for (int v = 0; v < 7; ++v) {
        ql[v] = b[v] + 0.5 * sb[v];
        qr[v] = c[v] - 0.5 * sc[v];
    }
    if (DIM == 0 && yswap) {
        const double lx = ql[VEL], rx = qr[VEL];
        ql[VEL] = ql[VEL + 1];
        qr[VEL] = qr[VEL + 1];
        ql[VEL + 1] = lx;
        qr[VEL + 1] = rx;
    }
    const double a_l2 = div_r<FAST>(gc.g * ql[PRE], ql[DEN]);
    const double a_r2 = div_r<FAST>(gc.g * qr[PRE], qr[DEN]);
    const bool bad = riemann<SOLVER, FAST, DIM>(F, ql, qr, a_l2, a_r2, gc, yswap);
    if (DIM == 0 && yswap) {
        const double fx = F[VEL];
        F[VEL] = F[VEL + 1];
        F[VEL + 1] = fx;
    }
    return bad;
}

// Fluid::advSolution + fixSolution of one cell from its base state u and
// flux divergence (the gravity source is zero, GRAV = 0), in place; inv_t: the
// CFL term of the new state (stage 2).  Returns false (FAST) where the result
// is not to be trusted.
template <int STAGE, bool FAST>
__device__ __forceinline__ bool update_cell(const HydroGeom& g, double u[7], const double udot[7], double dtf,
                                            StepState* st, double& inv_t) {
#pragma unroll
    for (int v = 0; v < 7; ++v) u[v] += dtf * udot[v];
    const bool ok = !FAST || (conserved_in_range(u) & (dtf * g.kflux < 0x1p200));
    if (fix_solution<FAST>(g, u) && ok) set_error(st, STAGE == 1 ? ERR_FIX_SOLUTION_1 : ERR_FIX_SOLUTION_2);
    if (STAGE == 2) {
        double q[7];
        QfromU<FAST>(q, u, g.gm1);
        fix_primitives<FAST>(g, q, u[DEN]);
        inv_t = cfl_inv_t<FAST>(g, q);
    }
    return ok;
}

// ---------------------------------------------------------------------------
// Small grids: 8 x 4 x 4 tiles, every face of the tile at once
// ---------------------------------------------------------------------------
constexpr int QX = 8, QY = 4, QZ = 4, QCELLS = QX * QY * QZ;
constexpr int QHX = 4 * QY * QZ, QHY = 4 * QX * QZ, QHZ = 4 * QX * QY;  // 2-deep halos at both ends
constexpr int QNX = (QX + 1) * QY * QZ, QNY = QX * (QY + 1) * QZ, QNZ = QX * QY * (QZ + 1);
constexpr int QTHREADS = 512;
constexpr int QZ0 = 320;  // first thread of the z faces: whole waves per solver
static_assert(QNX + QNY <= QZ0 && QZ0 % 64 == 0 && QZ0 + QNZ <= QTHREADS, "one face per thread");
static_assert(QCELLS + QHX + QHY + QHZ <= QTHREADS, "one cell per thread");

struct SmallLDS {
    double q[7][QCELLS + QHX + QHY + QHZ];
    double fx[7][QNX], fy[7][QNY], fz[7][QNZ];
    double red[QTHREADS / 64];
    int slow;  // a cell, face or result is out of the quick divisions' range
};

// LDS slot of tile position (x, y, z), of which one may lie in a 2-deep halo.
__device__ __forceinline__ int qslot(int x, int y, int z) {
    if ((unsigned)x >= (unsigned)QX) return QCELLS + (x < 0 ? x + 2 : x - QX + 2) * (QY * QZ) + y + QY * z;
    if ((unsigned)y >= (unsigned)QY) return QCELLS + QHX + (y < 0 ? y + 2 : y - QY + 2) * (QX * QZ) + x + QX * z;
    if ((unsigned)z >= (unsigned)QZ)
        return QCELLS + QHX + QHY + (z < 0 ? z + 2 : z - QZ + 2) * (QX * QY) + x + QX * y;
    return x + QX * (y + QY * z);
}

// Face f of tile row (ox, oy, oz) + f along DIM: the four stencil cells, both
// slopes and the solve.
template <int SOLVER, bool ALB, int DIM, bool FAST>
__device__ __forceinline__ bool small_face(const HydroGeom& g, const SmallLDS& s, int x, int y, int z, bool yface,
                                           const GasConsts<double>& gc, double F[7]) {
    const int dx = DIM == 0 && !yface, dy = DIM == 0 && yface, dz = DIM == 2;
    double q[4][7], sb[7], sc[7];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int c = qslot(x + dx * (i - 2), y + dy * (i - 2), z + dz * (i - 2));
#pragma unroll
        for (int v = 0; v < 7; ++v) q[i][v] = s.q[v][c];
    }
    cell_slope<ALB, FAST>(g, q[0], q[1], q[2], sb);
    cell_slope<ALB, FAST>(g, q[1], q[2], q[3], sc);
    return slope_flux<SOLVER, DIM, FAST>(g, q[1], sb, q[2], sc, gc, F, yface);
}

template <int SOLVER, bool ALB, int STAGE>
__global__ __launch_bounds__(QTHREADS) void hydro_tile_kernel(HydroGeom g, int ntx, int nty, int ntz,
                                                              const double* __restrict__ Usrc, const double* Ubase,
                                                              double* Udst, StepState* st, double dtf_host) {
    __shared__ SmallLDS s;
    if (st->halted) return;  // a halted sub-step's pass-through is launch_halted_copy's
    const int tile = tile_of_block(blockIdx.x, ntx * nty * ntz);
    const int ox = (tile % ntx) * QX, oy = (tile / ntx % nty) * QY, oz = tile / (ntx * nty) * QZ;
    const int tid = threadIdx.x;
    const GasConsts<double> gc = {g.g, g.gm1, g.g2};
    const int lx = tid % QX, ly = tid / QX % QY, lz = tid / (QX * QY);
    const bool active = tid < QCELLS && ox + lx < g.nx && oy + ly < g.ny && oz + lz < g.nz;
    if (tid == 0) s.slow = 0;
    __syncthreads();
    if (tid < QCELLS + QHX + QHY + QHZ) {
        int x = lx, y = ly, z = lz;
        if (tid >= QCELLS + QHX + QHY) {
            const int h = tid - (QCELLS + QHX + QHY), l = h / (QX * QY);
            x = h % QX, y = h / QX % QY, z = l < 2 ? l - 2 : QZ + l - 2;
        } else if (tid >= QCELLS + QHX) {
            const int h = tid - (QCELLS + QHX), l = h / (QX * QZ);
            x = h % QX, z = h / QX % QZ, y = l < 2 ? l - 2 : QY + l - 2;
        } else if (tid >= QCELLS) {
            const int h = tid - QCELLS, l = h / (QY * QZ);
            y = h % QY, z = h / QY % QZ, x = l < 2 ? l - 2 : QX + l - 2;
        }
        double q[7];
        if (!load_q<STAGE, Q_BOTH>(g, Usrc, ox + x, oy + y, oz + z, q, st, active)) s.slow = 1;
#pragma unroll
        for (int v = 0; v < 7; ++v) s.q[v][tid] = q[v];
    }
    double ub[7];  // the cell's base state, on its way while the faces are solved
    const long long c = (long long)(ox + lx) + (long long)g.nx * ((long long)(oy + ly) + (long long)g.ny * (oz + lz));
    if (active) {
#pragma unroll
        for (int v = 0; v < 7; ++v) ub[v] = Ubase[v * g.ncell + c];
    }
    __syncthreads();
    const double dtf = stage_dtf(dtf_host, st, STAGE);
    double inv_t = 0.0, u[7];
    const auto solve = [&](auto fast_c) {
        constexpr bool FAST = decltype(fast_c)::value;
        bool bad = false;
        double F[7] = {0, 0, 0, 0, 0, 0, 0};
        if (tid < QZ0) {
            const bool yface = tid >= QNX;
            const int j = yface ? tid - QNX : tid;
            const int x = yface ? j % QX : j % (QX + 1), y = yface ? j / (QX * QZ) : j / (QX + 1) % QY;
            const int z = yface ? j / QX % QZ : j / ((QX + 1) * QY);
            if (tid < QNX + QNY) {
                if (ox + x < g.nx + !yface && oy + y < g.ny + yface && oz + z < g.nz)
                    bad = small_face<SOLVER, ALB, 0, FAST>(g, s, x, y, z, yface, gc, F);
                double* dst = yface ? &s.fy[0][j] : &s.fx[0][j];
                const int n = yface ? QNY : QNX;
#pragma unroll
                for (int v = 0; v < 7; ++v) dst[v * n] = F[v];
            }
        } else if (tid < QZ0 + QNZ) {
            const int j = tid - QZ0, x = j % QX, y = j / QX % QY, z = j / (QX * QY);
            if (ox + x < g.nx && oy + y < g.ny && oz + z <= g.nz)
                bad = small_face<SOLVER, ALB, 2, FAST>(g, s, x, y, z, false, gc, F);
#pragma unroll
            for (int v = 0; v < 7; ++v) s.fz[v][j] = F[v];
        }
        if (bad && !FAST) set_error(st, STAGE == 1 ? ERR_RIEMANN_NAN_1 : ERR_RIEMANN_NAN_2);
        __syncthreads();
        bool ok = true;
        if (active) {
            // += (A/V) F_L, -= (A/V) F_R per dimension (Hydro.cpp:117-137)
            double udot[7];
            const int jx = lx + (QX + 1) * (ly + QY * lz), jy = lx + QX * (lz + QZ * ly), jz = lx + QX * (ly + QY * lz);
#pragma unroll
            for (int v = 0; v < 7; ++v) {
                double d = 0.0;
                d += g.kflux * s.fx[v][jx];
                d -= g.kflux * s.fx[v][jx + 1];
                d += g.kflux * s.fy[v][jy];
                d -= g.kflux * s.fy[v][jy + QX * QZ];
                d += g.kflux * s.fz[v][jz];
                d -= g.kflux * s.fz[v][jz + QX * QY];
                udot[v] = d;
                u[v] = ub[v];
            }
            ok = update_cell<STAGE, FAST>(g, u, udot, dtf, st, inv_t);
        }
        return ok && !bad;
    };
    if (s.slow == 0) {
        const bool ok = solve(std::true_type{});
        if (!ok) s.slow = 1;
        __syncthreads();
    }
    if (s.slow != 0) solve(std::false_type{});
    if (active) {
#pragma unroll
        for (int v = 0; v < 7; ++v) Udst[v * g.ncell + c] = u[v];
    }
    if (STAGE == 2) block_max_to<QTHREADS>(inv_t, &st->maxinv, s.red);
}

// ---------------------------------------------------------------------------
// The z march
// ---------------------------------------------------------------------------
constexpr int DT = 16;                      // columns are DT x DT cells
constexpr int DTHREADS = DT * DT;
constexpr int DPW = DT + 4;                 // plane row with its halos
constexpr int DHALO = 8 * DT;               // x and y halo cells per plane
constexpr int DNF = (DT + 1) * DT;          // x (and y) faces per plane
constexpr int DNS = (DT + 2) * DT;          // cells with an x (and y) slope per plane
constexpr int DN3 = 2 * DNF - 2 * DTHREADS; // faces past two per thread

struct ColumnLDS {
    double p[7][DPW * DPW];   // plane k: cell (x, y) at (y + 2) DPW + x + 2
    // the limited slopes of plane k, then (after a barrier) its face fluxes
    union {
        struct {
            double x[7][DNS];  // x slope of cell (x, y): y (DT + 2) + x + 1
            double y[7][DNS];  // y slope of cell (x, y): (y + 1) DT + x
        } s;
        struct {
            double x[7][DNF];  // x faces of plane k: y (DT + 1) + f
            double y[7][DNF];  // y faces of plane k: f DT + x
        } f;
    } sf;
    // fluxes that wait for the slopes' LDS: a thread's first face and the
    // faces past two per thread
    double park0[7][DTHREADS];
    double park2[7][DN3];
    double red[DTHREADS / 64];
    int stop[2];  // plane k & 1: a cell or face is out of the quick divisions' range
};

__device__ __forceinline__ int dslot(int x, int y) { return (y + 2) * DPW + x + 2; }

// Element at byte offset `off` (within one plane) of variable v at plane
// base U + plane: scalar base plus 32-bit offset.
template <typename T>
__device__ __forceinline__ T* plane_at(T* U, long long ncell, int v, long long plane, unsigned int off) {
    return (T*)((char*)(U + (v * ncell + plane)) + off);
}

// Halo cell h (0 .. DHALO - 1) of a plane: x halos first, then y halos.
__device__ __forceinline__ void dhalo_pos(int h, int& x, int& y) {
    const int l = (h & (4 * DT - 1)) / DT, r = h & (DT - 1), e = l < 2 ? l - 2 : DT + l - 2;
    x = h < 4 * DT ? e : r;
    y = h < 4 * DT ? r : e;
}

// x and y slopes of plane k: each thread its own cell's, 4 DT threads those of
// the 1-deep halo cells, which the column's boundary faces read.
template <bool ALB, bool FAST>
__device__ __forceinline__ void dmarch_slopes(const HydroGeom& g, ColumnLDS& s, int tid, int ht, int tx, int ty,
                                              const double w[7]) {
    double a[7], c[7], sl[7];
    const int o = dslot(tx, ty);
#pragma unroll
    for (int v = 0; v < 7; ++v) {
        a[v] = s.p[v][o - 1];
        c[v] = s.p[v][o + 1];
    }
    cell_slope<ALB, FAST>(g, a, w, c, sl);
#pragma unroll
    for (int v = 0; v < 7; ++v) s.sf.s.x[v][ty * (DT + 2) + tx + 1] = sl[v];
#pragma unroll
    for (int v = 0; v < 7; ++v) {
        a[v] = s.p[v][o - DPW];
        c[v] = s.p[v][o + DPW];
    }
    cell_slope<ALB, FAST>(g, a, w, c, sl);
#pragma unroll
    for (int v = 0; v < 7; ++v) s.sf.s.y[v][(ty + 1) * DT + tx] = sl[v];
    if (ht < 4 * DT) {
        const bool yh = ht >= 2 * DT;
        const int side = (ht / DT) & 1, r = ht & (DT - 1);
        const int hx = yh ? r : (side ? DT : -1), hy = yh ? (side ? DT : -1) : r;
        const int ho = dslot(hx, hy), st = yh ? DPW : 1;
        double b[7];
#pragma unroll
        for (int v = 0; v < 7; ++v) {
            a[v] = s.p[v][ho - st];
            b[v] = s.p[v][ho];
            c[v] = s.p[v][ho + st];
        }
        cell_slope<ALB, FAST>(g, a, b, c, sl);
        double* dst = yh ? &s.sf.s.y[0][(hy + 1) * DT + hx] : &s.sf.s.x[0][hy * (DT + 2) + hx + 1];
#pragma unroll
        for (int v = 0; v < 7; ++v) dst[v * DNS] = sl[v];
    }
}

// One x face (item < DNF: row y = item / (DT + 1), face f) or y face (face f
// = j / DT of column x) of plane k: flux in F (zero outside the grid).  Returns
// as slope_flux does.
template <int SOLVER, bool FAST>
__device__ __forceinline__ bool dmarch_face(const HydroGeom& g, const ColumnLDS& s, int item, int ox, int oy,
                                            const GasConsts<double>& gc, double F[7]) {
    const bool yface = item >= DNF;
    int qb, qs, sb, ss;
    bool valid;
    if (!yface) {
        const int y = item / (DT + 1), f = item - y * (DT + 1);
        valid = (ox + f <= g.nx) && (oy + y < g.ny);
        qb = dslot(f - 1, y);
        qs = 1;
        sb = y * (DT + 2) + f;
        ss = 1;
    } else {
        const int j = item - DNF, f = j / DT, x = j - f * DT;
        valid = (oy + f <= g.ny) && (ox + x < g.nx);
        qb = dslot(x, f - 1);
        qs = DPW;
        sb = DNS * 7 + f * DT + x;  // into the y slopes, which follow the x slopes
        ss = DT;
    }
#pragma unroll
    for (int v = 0; v < 7; ++v) F[v] = 0.0;
    if (valid) {
        double b[7], c[7], sbv[7], scv[7];
        const double* sl = &s.sf.s.x[0][0];
#pragma unroll
        for (int v = 0; v < 7; ++v) {
            b[v] = s.p[v][qb];
            c[v] = s.p[v][qb + qs];
            sbv[v] = sl[v * DNS + sb];
            scv[v] = sl[v * DNS + sb + ss];
        }
        return slope_flux<SOLVER, 0, FAST>(g, b, sbv, c, scv, gc, F, yface);
    }
    return false;
}

__device__ __forceinline__ void dstore_flux(ColumnLDS& s, int item, const double F[7]) {
    double* dst = item >= DNF ? &s.sf.f.y[0][item - DNF] : &s.sf.f.x[0][item];
#pragma unroll
    for (int v = 0; v < 7; ++v) dst[v * DNF] = F[v];
}

// FAST: the quick divisions and square roots (Recip, hydro_math.hpp) alone.  A
// workgroup that meets a cell or face out of their range ends before that
// plane's update, having noted the plane in `resume`, and the instance with the full ones, launched
// next, goes on from there (resume null: from the start), leaving at once
// where nothing is left (4 us; 7 at 256^3, 27 at 512^3).  Us per step: 256^3 6,609 with full divisions
// only, 5,715 so; 205x173x190 2,943 and 2,527; 128^3 864 and 750.  Both in one
// kernel, chosen per plane, held 105 spilled registers and were slower than
// full divisions alone (256^3 7,170).  What bounds the march is the latency of
// its instruction stream: two waves per SIMD issue vector instructions 0.55 to
// 0.63 of the time (3,800 per cell and stage).
template <int SOLVER, bool ALB, int STAGE, bool FAST>
__global__ __launch_bounds__(DTHREADS) __attribute__((amdgpu_waves_per_eu(2))) void hydro_march_kernel(
    HydroGeom g, int ntx, int nty, int ntz, int mz, const double* __restrict__ Usrc, const double* Ubase, double* Udst,
    StepState* st, double dtf_host, int* __restrict__ resume) {
    __shared__ ColumnLDS s;
    if (st->halted) return;  // a halted sub-step's pass-through is launch_halted_copy's
    const int tile = tile_of_block(blockIdx.x, ntx * nty * ntz);
    const int ox = (tile % ntx) * DT, oy = (tile / ntx % nty) * DT;
    int z0 = tile / (ntx * nty) * mz;
    const int z1 = min(z0 + mz, g.nz);
    if (!FAST && resume) z0 = resume[blockIdx.x];
    if (z0 >= z1) return;
    const int tid = threadIdx.x, tx = tid % DT, ty = tid / DT;
    const int gx = ox + tx, gy = oy + ty;
    const bool col = gx < g.nx && gy < g.ny;
    const GasConsts<double> gc = {g.g, g.gm1, g.g2};
    const double dtf = stage_dtf(dtf_host, st, STAGE);
    const long long pl = (long long)g.nx * g.ny;
    // the own column's source in a plane and, past the x or y end of the grid
    // (a ghost column that the last faces read), its velocity rule
    const CellSrc own = cell_source(g, gx, gy, z0);
    const unsigned int off = 8u * (unsigned int)(own.idx - pl * z0);
    // Q of the own column's plane z (ghost planes by the z boundary
    // condition; own cells are checked once, by the workgroup that owns them)
    const auto load_u = [&](int z, double u[7]) {
        const int zs = ghost_map(z, g.nz, g.bc_l[2], g.bc_r[2]).src;
#pragma unroll
        for (int v = 0; v < 7; ++v) u[v] = *plane_at(Usrc, g.ncell, v, pl * zs, off);
    };
    const auto to_q = [&](int z, const double u[7], double q[7]) {
        const bool zg = (unsigned)z >= (unsigned)g.nz;
        const int zmode = ghost_map(z, g.nz, g.bc_l[2], g.bc_r[2]).mode;
        return q_of_cell<STAGE, FAST ? Q_FAST : Q_FULL>(g, u, own.mdim ? own.mode : zmode,
                                                        own.mdim ? own.mdim : (zg ? 3 : 0), q, st,
                                                        col && z >= z0 && z < z1);
    };
    unsigned int ok;  // FAST, bit j: plane k + 2 - j of the own column is in range

    double sk[7], w1[7], w2[7], w3[7], fz[7];
    {
        double a[7], w0[7], s0[7], u[7];
        load_u(z0 - 2, u);
        ok = to_q(z0 - 2, u, a);
        load_u(z0 - 1, u);
        ok = 2 * ok + to_q(z0 - 1, u, w0);
        load_u(z0, u);
        ok = 2 * ok + to_q(z0, u, w1);
        load_u(z0 + 1, u);
        ok = 2 * ok + to_q(z0 + 1, u, w2);
        cell_slope<ALB, FAST>(g, a, w0, w1, s0);
        cell_slope<ALB, FAST>(g, w0, w1, w2, sk);
        bool bad = false;
        if (col) bad = slope_flux<SOLVER, 2, FAST>(g, w0, s0, w1, sk, gc, fz);  // face z0 - 1/2
        if (FAST) ok = bad ? 0 : ok;
        else if (bad) set_error(st, STAGE == 1 ? ERR_RIEMANN_NAN_1 : ERR_RIEMANN_NAN_2);
        load_u(z0 + 2, u);
        ok = 2 * ok + to_q(z0 + 2, u, w3);
    }
    if (FAST) {
        if (tid < 2) s.stop[tid] = 0;
        __syncthreads();
    }
    int done = z1;
    double inv_t = 0.0;
    for (int k = z0; k < z1; ++k) {
        // The extra work of a plane (halo cells, halo slopes, third faces)
        // goes to another wave each plane.
        const int turn = (tid + 64 * (k & 3)) & (DTHREADS - 1);
        double un[7];
        if (k + 1 < z1) load_u(k + 3, un);  // used at the plane's end
#pragma unroll
        for (int v = 0; v < 7; ++v) s.p[v][dslot(tx, ty)] = w1[v];
        if (FAST) {
            // planes k - 1 .. k + 2 of the own column, and k - 2 behind its first face
            const unsigned int need = k == z0 ? 31u : 15u;
            if ((ok & need) != need) s.stop[k & 1] = 1;
        }
        if (turn < DHALO) {
            int hx, hy;
            dhalo_pos(turn, hx, hy);
            double hq[7];
            const bool in = load_q<STAGE, FAST ? Q_FAST : Q_FULL>(g, Usrc, ox + hx, oy + hy, k, hq, st, false);
            if (FAST && !in) s.stop[k & 1] = 1;
            const int hs = dslot(hx, hy);
#pragma unroll
            for (int v = 0; v < 7; ++v) s.p[v][hs] = hq[v];
        }
        __syncthreads();
        // x and y slopes, then the faces; each flux waits (in LDS or, the
        // last one solved, in registers) until every face has read the
        // slopes, whose LDS the fluxes then take over
        dmarch_slopes<ALB, FAST>(g, s, tid, turn, tx, ty, w1);
        __syncthreads();
        {
            double F[7];
#pragma unroll 1
            for (int j = turn < DN3 ? -1 : 0; j < 2; ++j) {
                const int item = j < 0 ? 2 * DTHREADS + turn : tid + j * DTHREADS;
                if (dmarch_face<SOLVER, FAST>(g, s, item, ox, oy, gc, F)) {
                    if (FAST) s.stop[k & 1] = 1;
                    else set_error(st, STAGE == 1 ? ERR_RIEMANN_NAN_1 : ERR_RIEMANN_NAN_2);
                }
                if (j < 0) {
#pragma unroll
                    for (int v = 0; v < 7; ++v) s.park2[v][turn] = F[v];
                } else if (j == 0) {
#pragma unroll
                    for (int v = 0; v < 7; ++v) s.park0[v][tid] = F[v];
                }
            }
            __syncthreads();
            dstore_flux(s, tid + DTHREADS, F);
#pragma unroll
            for (int v = 0; v < 7; ++v) F[v] = s.park0[v][tid];
            dstore_flux(s, tid, F);
            if (turn < DN3) {
#pragma unroll
                for (int v = 0; v < 7; ++v) F[v] = s.park2[v][turn];
                dstore_flux(s, turn + 2 * DTHREADS, F);
            }
        }
        // z face k + 1/2 from registers
        double fzn[7] = {0, 0, 0, 0, 0, 0, 0}, u[7];
        {
            double sn[7];
            cell_slope<ALB, FAST>(g, w1, w2, w3, sn);
            if (col && slope_flux<SOLVER, 2, FAST>(g, w1, sk, w2, sn, gc, fzn)) {
                if (FAST) s.stop[k & 1] = 1;
                else set_error(st, STAGE == 1 ? ERR_RIEMANN_NAN_1 : ERR_RIEMANN_NAN_2);
            }
#pragma unroll
            for (int v = 0; v < 7; ++v) sk[v] = sn[v];
        }
        if (col) {
#pragma unroll
            for (int v = 0; v < 7; ++v) u[v] = *plane_at(Ubase, g.ncell, v, pl * k, off);
        }
        __syncthreads();
        double t = 0.0;
        if (col) {
            // += (A/V) F_L, -= (A/V) F_R per dimension (Hydro.cpp:117-137)
            double udot[7];
            const int fxl = ty * (DT + 1) + tx, fyl = ty * DT + tx;
#pragma unroll
            for (int v = 0; v < 7; ++v) {
                double d = 0.0;
                d += g.kflux * s.sf.f.x[v][fxl];
                d -= g.kflux * s.sf.f.x[v][fxl + 1];
                d += g.kflux * s.sf.f.y[v][fyl];
                d -= g.kflux * s.sf.f.y[v][fyl + DT];
                d += g.kflux * fz[v];
                d -= g.kflux * fzn[v];
                udot[v] = d;
            }
            if (!update_cell<STAGE, FAST>(g, u, udot, dtf, st, t)) s.stop[k & 1] = 1;
        }
        if (FAST) {
            __syncthreads();
            if (s.stop[k & 1]) {  // nothing of this plane has left the workgroup
                done = k;
                break;
            }
        }
        if (col) {
            if (STAGE == 2 && t > inv_t) inv_t = t;
#pragma unroll
            for (int v = 0; v < 7; ++v) *plane_at(Udst, g.ncell, v, pl * k, off) = u[v];
        }
#pragma unroll
        for (int v = 0; v < 7; ++v) {
            fz[v] = fzn[v];
            w1[v] = w2[v];
            w2[v] = w3[v];
        }
        if (k + 1 < z1) ok = 2 * ok + to_q(k + 3, un, w3);
    }
    if (FAST && tid == 0) resume[blockIdx.x] = done;
    if (STAGE == 2) block_max_to<DTHREADS>(inv_t, &st->maxinv, s.red);
}

// Standalone CFL reduction over U (Hydrodynamics::calculateTimeStep on
// fixPrimitives(QfromU(U))).
__global__ __launch_bounds__(256) void cfl_kernel(HydroGeom g, const double* __restrict__ U, StepState* st) {
    __shared__ double red[4];
    double m = 0.0;
    for (long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x; c < g.ncell; c += (long long)gridDim.x * blockDim.x) {
        double u[7], q[7];
#pragma unroll
        for (int v = 0; v < 7; ++v) u[v] = U[v * g.ncell + c];
        QfromU(q, u, g.gm1);
        fix_primitives(g, q, u[DEN]);
        double it = cfl_inv_t(g, q);
        if (it >= 0.0) m = fmax(m, it);
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) m = fmax(m, __shfl_xor(m, off, 64));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        double b = fmax(fmax(red[0], red[1]), fmax(red[2], red[3]));
        atomicMax(&st->maxinv, (unsigned long long)__double_as_longlong(b));
    }
}

// Checkpointer::update's count for time t (Checkpointer.cpp:14-26): the
// number of the checkpoint percentages 100 / ncheckpoints passed.
__device__ __forceinline__ int checkpoint_count(const StepState* st, double t) {
    const double delta = 100.0 / st->ncheckpoints;
    const double pct = smin(100.0, 100.0 * t / st->tmax);
    int count = st->ckpt_count;
    while (pct - count * delta > delta - 1.0e-8) count += 1;
    return count;
}

__global__ void set_time_kernel(StepState* st, double t) {
    st->time = t;
    st->ckpt_count = 0;
    st->ckpt_count = checkpoint_count(st, t);
    st->paused = 0;
    st->halted = 0;
}

__global__ void resume_kernel(StepState* st) {
    if (st->paused) {
        st->paused = 0;
        st->halted = 0;
    }
}

// Start of a step: dt = min(dt_nextCheckpoint, dt_cfl) as Torch::run +
// Torch::fullStep + Torch::calculateTimeStep (Torch.cpp:266-270,304-339,397),
// with the checkpoint arithmetic of Checkpointer::update (Checkpointer.cpp:14-26).
// use_cfl = 0 takes dt_override instead of the CFL/first-step value.
__global__ void step_begin_kernel(StepState* st, int use_cfl, double dt_override,
                                  const unsigned long long* thermo_dt_bits,
                                  const unsigned long long* rad_dt_bits) {
    if (!use_cfl) {  // an explicit Torch::hydroStep(dt): no clock rules apply
        st->halted = 0;
        st->dt = dt_override;
        st->keep_ustar = 1;
        return;
    }
    if (st->halted) return;
    // a step that raised an error ends the run as the reference's exception
    // does; the error is reported by the next synchronising call; the loop
    // condition of Torch::run (Torch.cpp:266) also ends it once quitting
    if (!(st->time < st->tmax) || st->err || st->quitting) {
        st->halted = 1;
        return;
    }
    const int count = checkpoint_count(st, st->time);
    if (st->pause_ckpt && count > st->ckpt_count) {
        // a new checkpoint is due before this step: Torch::run prints here
        st->ckpt_count = count;
        st->paused = 1;
        st->halted = 1;
        return;
    }
    st->ckpt_count = count;
    const double delta = 100.0 / st->ncheckpoints;
    double pct = smin(100.0, 100.0 * st->time / st->tmax);
    const double dt_next = ((count + 1) * delta - pct) * st->tmax / 100.0;
    double dt;
    if (st->first) {
        dt = st->dt_max * 1.0e-20;
        st->first = 0;
    } else {
        const double maxinv = __longlong_as_double((long long)st->maxinv);
        double tmin = st->dt_max;
        if (maxinv > 0.0) tmin = smin(tmin, 0.5 / maxinv);
        dt = smin(tmin, st->dt_max);
        // Torch::calculateTimeStep's debug test (Torch.cpp:321-332): its
        // condition reads the hydro percentage only; the step still runs and
        // Torch::run's loop ends after it
        if (st->debug && 100.0 * dt / st->tmax <= 1.0e-6) st->quitting = 1;
        if (thermo_dt_bits) {
            // Thermodynamics::calculateTimeStep: dt_max lowered by every
            // smaller |f E/RATE| (Thermodynamics.cpp:465-474)
            const double m = __longlong_as_double((long long)*thermo_dt_bits);
            dt = smin(dt, smin(m, st->dt_max));
        }
        if (rad_dt_bits) {
            // Radiation::calculateTimeStep's minimum, at most dt_max
            const double m = __longlong_as_double((long long)*rad_dt_bits);
            dt = smin(dt, smin(m, st->dt_max));
        }
    }
    st->dt = smin(dt_next, dt);
    st->maxinv = 0ull;
    // the next step_begin's tests on this step's end time (step_end adds dt
    // to time the same way): a pause for a new checkpoint, tmax, quitting
    const double t_end = st->time + st->dt;
    st->keep_ustar = checkpoint_count(st, t_end) > count || !(t_end < st->tmax) || st->quitting;
}

__global__ void step_end_kernel(StepState* st) {
    if (st->halted) return;
    st->time += st->dt;
    st->step += 1;
}

__global__ void q_from_u_kernel(HydroGeom g, const double* __restrict__ U, double* __restrict__ Q, int fix) {
    for (long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x; c < g.ncell; c += (long long)gridDim.x * blockDim.x) {
        double u[7], q[7];
#pragma unroll
        for (int v = 0; v < 7; ++v) u[v] = U[v * g.ncell + c];
        QfromU(q, u, g.gm1);
        if (fix) fix_primitives(g, q, u[DEN]);
#pragma unroll
        for (int v = 0; v < 7; ++v) Q[v * g.ncell + c] = q[v];
    }
}

// Torch::initialise tail (Torch.cpp:117-119): fixPrimitives on the uploaded
// Q (U is still zero there, so the temperature floor reads U[DEN] = 0), then
// globalUfromQ.  Q is fixed in place.
__global__ void u_from_q_kernel(HydroGeom g, double* __restrict__ Q, double* __restrict__ U) {
    const GasConsts<double> gc = {g.g, g.gm1, g.g2};
    for (long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x; c < g.ncell; c += (long long)gridDim.x * blockDim.x) {
        double u[7], q[7];
#pragma unroll
        for (int v = 0; v < 7; ++v) q[v] = Q[v * g.ncell + c];
        fix_primitives(g, q, 0.0);
        UfromQ<double>(u, q, gc);
#pragma unroll
        for (int v = 0; v < 7; ++v) {
            Q[v * g.ncell + c] = q[v];
            U[v * g.ncell + c] = u[v];
        }
    }
}

// Thermodynamics::updateSourceTerms + Fluid::advSolution + fixSolution on
// the grid: UDOT[PRE] = rate (other UDOT zero), U += dtf * UDOT, then
// fixSolution (Thermodynamics.cpp:478-485, Fluid.cpp:80-136).
// cerr: the cooling operator's error word; a subcycle count beyond the int
// range raised by the integrate that produced `rate` is moved into the step
// state here (reported at this step, like the fixSolution errors) and the
// word cleared.
__global__ void apply_rate_fix_kernel(HydroGeom g, double* __restrict__ U, const double* __restrict__ rate, double dtf,
                                      StepState* st, unsigned int* cerr) {
    if (dtf < 0.0 && st->halted) return;
    if (cerr && blockIdx.x == 0 && threadIdx.x == 0) {
        const unsigned int e = *cerr;
        if (e & ERR_THERMO_NSTEPS) {
            set_error(st, ERR_THERMO_NSTEPS);
            *cerr = 0u;
        }
    }
    dtf = stage_dtf(dtf, st, 0);
    for (long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x; c < g.ncell; c += (long long)gridDim.x * blockDim.x) {
        double u[7];
#pragma unroll
        for (int v = 0; v < 7; ++v) u[v] = U[v * g.ncell + c];
        double udot[7] = {0, 0, 0, 0, 0, 0, 0};
        udot[PRE] += rate ? rate[c] : 0.0;
#pragma unroll
        for (int v = 0; v < 7; ++v) u[v] += dtf * udot[v];
        if (fix_solution(g, u)) set_error(st, ERR_THERMO_FIX);
#pragma unroll
        for (int v = 0; v < 7; ++v) U[v * g.ncell + c] = u[v];
    }
}

// The cooling sub-step's update of U (as apply_rate_fix_kernel:
// Thermodynamics::updateSourceTerms + advSolution + fixSolution) fused with
// the float Q the next mixed stage reads (as q_float_kernel in fix mode), so
// the updated state is not read back.  A halted run leaves U as it is but
// still refreshes the float Q from it.  Compiled without FMA contraction,
// as the FP64 grids' update: the same arithmetic whichever kernel applies
// a cooling sub-step.
__global__ void apply_rate_fix_qf_kernel(HydroGeom g, double* __restrict__ U, const double* __restrict__ rate,
                                         double dtf, StepState* st, unsigned int* cerr, float* __restrict__ qout) {
    const bool halted = dtf < 0.0 && st->halted;
    if (!halted && cerr && blockIdx.x == 0 && threadIdx.x == 0) {
        const unsigned int e = *cerr;
        if (e & ERR_THERMO_NSTEPS) {
            set_error(st, ERR_THERMO_NSTEPS);
            *cerr = 0u;
        }
    }
    if (!halted) dtf = stage_dtf(dtf, st, 0);
    for (long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x; c < g.ncell; c += (long long)gridDim.x * blockDim.x) {
        double u[7];
#pragma unroll
        for (int v = 0; v < 7; ++v) u[v] = U[v * g.ncell + c];
        if (!halted) {
            double udot[7] = {0, 0, 0, 0, 0, 0, 0};
            udot[PRE] += rate ? rate[c] : 0.0;
#pragma unroll
            for (int v = 0; v < 7; ++v) u[v] += dtf * udot[v];
            if (fix_solution(g, u)) set_error(st, ERR_THERMO_FIX);
#pragma unroll
            for (int v = 0; v < 7; ++v) U[v * g.ncell + c] = u[v];
        }
        double q[7];
        q_from_u_mixed(q, u, g.gm1);
        store_qf(g, q, u, qout, c, 1, false);
    }
}

hipError_t launch_fix_solution_qf(const HydroGeom& g, double* U, const double* rate, double dtf, StepState* st,
                                  hipStream_t stream, unsigned int* cerr, float* qout) {
    long long nb = (g.ncell + 255) / 256;
    if (nb > 65536) nb = 65536;
    hipLaunchKernelGGL(apply_rate_fix_qf_kernel, dim3((unsigned)nb), dim3(256), 0, stream, g, U, rate, dtf, st, cerr,
                       qout);
    return hipGetLastError();
}

// A halted run's single-stage sub-step (dt code DT_HALF / DT_FULL) still
// passes its input through to its output, float primitives included: the
// host swaps the two state buffers after every such sub-step without knowing
// whether the run halted.  Launched after each such sub-step; returns at
// once while the run is going.
__global__ void halted_copy_kernel(HydroGeom g, const StepState* st, const double* __restrict__ Usrc,
                                   double* __restrict__ Udst, const float* __restrict__ qin,
                                   float* __restrict__ qout) {
    if (!st->halted) return;
    for (long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x; c < g.ncell; c += (long long)gridDim.x * blockDim.x) {
#pragma unroll
        for (int v = 0; v < 7; ++v) Udst[v * g.ncell + c] = Usrc[v * g.ncell + c];
        if (qin) {
#pragma unroll
            for (int v = 0; v < 7; ++v) qout[v * g.ncell + c] = qin[v * g.ncell + c];
        }
    }
}

__global__ void zero_kernel(double* __restrict__ p, long long n) {
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
        p[i] = 0.0;
}

hipError_t launch_zero(double* p, long long n, hipStream_t stream) {
    long long nb = (n + 255) / 256;
    if (nb > 8192) nb = 8192;
    if (nb < 1) nb = 1;
    hipLaunchKernelGGL(zero_kernel, dim3((unsigned)nb), dim3(256), 0, stream, p, n);
    return hipGetLastError();
}

hipError_t launch_halted_copy(const HydroGeom& g, const StepState* st, const double* Usrc, double* Udst,
                              const float* qin, float* qout, hipStream_t stream) {
    long long nb = (g.ncell + 255) / 256;
    if (nb > 8192) nb = 8192;
    hipLaunchKernelGGL(halted_copy_kernel, dim3((unsigned)nb), dim3(256), 0, stream, g, st, Usrc, Udst, qin, qout);
    return hipGetLastError();
}

hipError_t launch_fix_solution(const HydroGeom& g, double* U, const double* rate, double dtf, StepState* st,
                               hipStream_t stream, unsigned int* cerr) {
    long long nb = (g.ncell + 255) / 256;
    if (nb > 65536) nb = 65536;
    hipLaunchKernelGGL(apply_rate_fix_kernel, dim3((unsigned)nb), dim3(256), 0, stream, g, U, rate, dtf, st, cerr);
    return hipGetLastError();
}

// Which layout, and how many planes per march workgroup: the smallest of
// estimates from times measured on this part (one stage, rotated solver, van
// Albada).  A march workgroup takes about 13.5 us per plane alone on a CU and
// 20.5 us beside a second one, with 1.2 planes' worth of work before its
// first; up to 512 run at once, and of more the last leave half a workgroup's
// time unfilled; the second launch takes 4 us.  The tiles take 12 us and 0.29
// ns per cell.  Measured us per step (two stages), tiles / march / the single
// 8^3-tile kernel before: 16^3 25 / 169 (pieces of 4 planes) / 97; 48^3 86 /
// 118; 64^3 162 / 154 / 200; 72^3 236 / 209; 80^3 312 / 215 / 383; 128^3 1,203
// / 750 / 1,487; 205x173x190 4,227 / 2,527 / 5,093; 256^3 10,044 / 5,715 /
// 12,251 (1,369 -> 2,936 Mcell-updates/s).
struct StagePlan {
    bool march;
    int mz;
};

static StagePlan stage_plan(const HydroGeom& g) {
    const long long cols = (long long)((g.nx + DT - 1) / DT) * ((g.ny + DT - 1) / DT);
    StagePlan p{false, g.nz};
    double best = 12.0 + 0.29e-3 * (double)g.ncell;
    // the march's 32-bit offsets cover planes of fewer than 2^29 cells
    if ((long long)g.nx * g.ny >= (1LL << 29)) return p;
    // pieces of 2 .. 32 planes (longer ones lose the halo's reuse in L2)
    for (int pieces = (g.nz + 31) / 32; pieces <= 4 * ((g.nz + 31) / 32) + 12; ++pieces) {
        const int mz = (g.nz + pieces - 1) / pieces;
        if (mz < 2 && g.nz > 1) break;
        const long long blocks = cols * ((g.nz + mz - 1) / mz);
        const double rounds = blocks <= 256 ? 13.5 / 20.5 : blocks <= 512 ? 1.0 : 0.5 + (double)blocks / 512.0;
        const double t = 4.0 + 20.5 * rounds * (mz + 1.2);
        if (t < best) {
            best = t;
            p = StagePlan{true, mz};
        }
    }
    return p;
}

long long march_blocks(const HydroGeom& g) {
    const StagePlan p = stage_plan(g);
    return p.march ? (long long)((g.nx + DT - 1) / DT) * ((g.ny + DT - 1) / DT) * ((g.nz + p.mz - 1) / p.mz) : 0;
}

template <int SOLVER, bool ALB>
static hipError_t launch_stage_t(const HydroGeom& g, int stage, const double* Usrc, const double* Ubase, double* Udst,
                                 StepState* st, double dtf, hipStream_t stream) {
    const StagePlan plan = stage_plan(g);
    if (plan.march) {
        const int mtx = (g.nx + DT - 1) / DT, mty = (g.ny + DT - 1) / DT, mtz = (g.nz + plan.mz - 1) / plan.mz;
        dim3 grid(mtx * mty * mtz), block(DTHREADS);
        const auto launch = [&](auto fast, int* resume) {
            if (stage == 1)
                hipLaunchKernelGGL((hydro_march_kernel<SOLVER, ALB, 1, decltype(fast)::value>), grid, block, 0, stream,
                                   g, mtx, mty, mtz, plan.mz, Usrc, Ubase, Udst, st, dtf, resume);
            else
                hipLaunchKernelGGL((hydro_march_kernel<SOLVER, ALB, 2, decltype(fast)::value>), grid, block, 0, stream,
                                   g, mtx, mty, mtz, plan.mz, Usrc, Ubase, Udst, st, dtf, resume);
        };
        if (g.fast) launch(std::true_type{}, g.resume);
        launch(std::false_type{}, g.fast ? g.resume : nullptr);
        return hipGetLastError();
    }
    const int ntx = (g.nx + QX - 1) / QX, nty = (g.ny + QY - 1) / QY, ntz = (g.nz + QZ - 1) / QZ;
    dim3 grid(ntx * nty * ntz), block(QTHREADS);
    if (stage == 1)
        hipLaunchKernelGGL((hydro_tile_kernel<SOLVER, ALB, 1>), grid, block, 0, stream, g, ntx, nty, ntz, Usrc, Ubase,
                           Udst, st, dtf);
    else
        hipLaunchKernelGGL((hydro_tile_kernel<SOLVER, ALB, 2>), grid, block, 0, stream, g, ntx, nty, ntz, Usrc, Ubase,
                           Udst, st, dtf);
    return hipGetLastError();
}

template <int SOLVER>
static hipError_t launch_stage_l(const HydroGeom& g, int stage, const double* Usrc, const double* Ubase, double* Udst,
                                 StepState* st, double dtf, hipStream_t stream) {
    if (g.limiter == LIM_ALBADA) return launch_stage_t<SOLVER, true>(g, stage, Usrc, Ubase, Udst, st, dtf, stream);
    return launch_stage_t<SOLVER, false>(g, stage, Usrc, Ubase, Udst, st, dtf, stream);
}

hipError_t launch_hydro_stage(const HydroGeom& g, int solver, int stage, const double* Usrc, const double* Ubase,
                              double* Udst, StepState* st, hipStream_t stream, double dtf) {
    switch (solver) {
    case SOLVER_HLL:  return launch_stage_l<SOLVER_HLL>(g, stage, Usrc, Ubase, Udst, st, dtf, stream);
    case SOLVER_HLLC: return launch_stage_l<SOLVER_HLLC>(g, stage, Usrc, Ubase, Udst, st, dtf, stream);
    default:          return launch_stage_l<SOLVER_ROTATED>(g, stage, Usrc, Ubase, Udst, st, dtf, stream);
    }
}

hipError_t launch_cfl(const HydroGeom& g, const double* U, StepState* st, hipStream_t stream) {
    long long nb = (g.ncell + 255) / 256;
    if (nb > 8192) nb = 8192;
    hipLaunchKernelGGL(cfl_kernel, dim3((unsigned)nb), dim3(256), 0, stream, g, U, st);
    return hipGetLastError();
}

hipError_t launch_step_begin(StepState* st, int use_cfl, double dt_override, hipStream_t stream,
                             const unsigned long long* thermo_dt_bits, const unsigned long long* rad_dt_bits) {
    hipLaunchKernelGGL(step_begin_kernel, dim3(1), dim3(1), 0, stream, st, use_cfl, dt_override, thermo_dt_bits,
                       rad_dt_bits);
    return hipGetLastError();
}

// dst = src (n doubles) unless the run has halted.
__global__ void copy_if_running_kernel(const StepState* st, const double* __restrict__ src, double* __restrict__ dst,
                                       long long n) {
    if (st->halted) return;
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
        dst[i] = src[i];
}

hipError_t launch_copy_if_running(const StepState* st, const double* src, double* dst, long long n,
                                  hipStream_t stream) {
    long long nb = (n + 255) / 256;
    if (nb > 65536) nb = 65536;
    hipLaunchKernelGGL(copy_if_running_kernel, dim3((unsigned)nb), dim3(256), 0, stream, st, src, dst, n);
    return hipGetLastError();
}

hipError_t launch_set_time(StepState* st, double t, hipStream_t stream) {
    hipLaunchKernelGGL(set_time_kernel, dim3(1), dim3(1), 0, stream, st, t);
    return hipGetLastError();
}

hipError_t launch_resume(StepState* st, hipStream_t stream) {
    hipLaunchKernelGGL(resume_kernel, dim3(1), dim3(1), 0, stream, st);
    return hipGetLastError();
}

hipError_t launch_step_end(StepState* st, hipStream_t stream) {
    hipLaunchKernelGGL(step_end_kernel, dim3(1), dim3(1), 0, stream, st);
    return hipGetLastError();
}

hipError_t launch_q_from_u(const HydroGeom& g, const double* U, double* Q, int fix, hipStream_t stream) {
    long long nb = (g.ncell + 255) / 256;
    if (nb > 65536) nb = 65536;
    hipLaunchKernelGGL(q_from_u_kernel, dim3((unsigned)nb), dim3(256), 0, stream, g, U, Q, fix);
    return hipGetLastError();
}

__global__ void q_from_u_if_running_kernel(HydroGeom g, const StepState* st, const double* __restrict__ U,
                                           double* __restrict__ Q) {
    if (st->halted) return;
    for (long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x; c < g.ncell; c += (long long)gridDim.x * blockDim.x) {
        double u[7], q[7];
#pragma unroll
        for (int v = 0; v < 7; ++v) u[v] = U[v * g.ncell + c];
        QfromU(q, u, g.gm1);
        fix_primitives(g, q, u[DEN]);
#pragma unroll
        for (int v = 0; v < 7; ++v) Q[v * g.ncell + c] = q[v];
    }
}

hipError_t launch_q_from_u_if_running(const HydroGeom& g, const StepState* st, const double* U, double* Q,
                                      hipStream_t stream) {
    long long nb = (g.ncell + 255) / 256;
    if (nb > 65536) nb = 65536;
    hipLaunchKernelGGL(q_from_u_if_running_kernel, dim3((unsigned)nb), dim3(256), 0, stream, g, st, U, Q);
    return hipGetLastError();
}

hipError_t launch_u_from_q(const HydroGeom& g, double* Q, double* U, hipStream_t stream) {
    long long nb = (g.ncell + 255) / 256;
    if (nb > 65536) nb = 65536;
    hipLaunchKernelGGL(u_from_q_kernel, dim3((unsigned)nb), dim3(256), 0, stream, g, Q, U);
    return hipGetLastError();
}

}  // namespace tg
