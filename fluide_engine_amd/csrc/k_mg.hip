// k_mg.hip -- geometric multigrid V-cycle used as the preconditioner of the
// pressure CG (no reference counterpart: the reference's CG has an identity
// preconditioner, src/linear_system/conjugate_gradient_solver.cpp:57-63).
//
// Levels: level 0 is the pressure grid; each coarser level halves every axis
// (rounding up).  A coarse cell is AIR if any child is AIR, else FLUID if any
// child is FLUID, else BOUNDRY (the free surface keeps its Dirichlet cells on
// every level, as in McAdams, Sifakis and Teran, "A parallel multigrid Poisson
// solver for fluids simulation on large grids", SCA 2010), and its operator is
// BuildSystem's 7-point rule on those markers with twice the spacing.
//
// The V-cycle is symmetric, so the preconditioner is SPD and CG stays CG:
//   * smoothing: two steps of Chebyshev iteration on D^-1 A over [0.15, 2]
//     on the finest level and [0.07, 2] below it, before and the same two after (mg_cheb2; levels inside the
//     one-workgroup tail on small grids: two damped Jacobi sweeps with the
//     first step's weight before and after);
//   * prolongation: trilinear interpolation of the cell-centred coarse
//     correction (weights 3/4, 1/4 per axis; out-of-range coarse neighbours
//     clamp onto the boundary cell, which is the Neumann wall);
//   * restriction: the transpose of that prolongation divided by 8;
//   * coarsest level (<= 512 cells): 8 steps of Chebyshev iteration on D^-1 A over [0.05, 2]
//     from zero, a fixed polynomial in the operator.
// Non-FLUID cells carry no residual into the coarse levels and take no
// correction; on level 0 they are smoothed like the identity rows they are.
//
// Kernels per V-cycle (FE_MG_FUSED): a descent and an ascent per level over LDS
// tiles (k_mg_down, k_mg_up), the last two levels in one workgroup
// (k_mg_bottom), or, where they do not fit it, the coarsest alone (k_mg_tail).
// FE_MG_SPLIT takes one kernel per sweep, residual, restriction and
// prolongation, the first sweep from zero fused into the kernel that produces
// the level's right-hand side.
#include <algorithm>

#include "fe_stencil.hpp"

namespace fe {

// Coarsest level: kCoarseSweeps steps of Chebyshev iteration from zero on
// D^-1 A over [kChebLo, kChebHi].  Gershgorin bounds every eigenvalue of D^-1 A
// (diagonal >= the sum of the off-diagonal magnitudes on every row) by 2, so
// with kChebHi = 2 the residual polynomial's Chebyshev form lies in (0, 1] at
// every eigenvalue, below kChebLo included: the step is a fixed symmetric
// positive-definite polynomial of D^-1 A, as PCG needs.
constexpr int kCoarseSweeps = 8;
constexpr float kChebLo = 0.05f, kChebHi = 2.0f;
constexpr int kCoarseMax = 512;       // cells of the coarsest level
constexpr int kTailMax = kCoarseMax;  // levels of at most this many cells run in k_mg_tail
constexpr int kTailLds = kCoarseMax;  // cells of all tail levels together (5 floats + a row code each in LDS)
constexpr int kTailThreads = kTailMax;  // one cell per thread
constexpr int kMaxTail = 8;
constexpr int kTailPer = (kTailMax + kTailThreads - 1) / kTailThreads;  // cells per thread on a tail level

// ---------------------------------------------------------------------------
// Level construction
// ---------------------------------------------------------------------------
__device__ inline void cell_ijk(int64_t c, int nx, int ny, int& i, int& j, int& k) {
    const uint32_t cu = (uint32_t)c;
    i = (int)(cu % (uint32_t)nx);
    j = (int)((cu / (uint32_t)nx) % (uint32_t)ny);
    k = (int)(cu / ((uint32_t)nx * (uint32_t)ny));
}

__global__ __launch_bounds__(kBlock) void k_mg_coarsen(const uint8_t* __restrict__ ff, int fx, int fy, int fz,
                                                       uint8_t* __restrict__ cf, int cx, int cy, int cz) {
    const int64_t c = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    const int64_t nc = (int64_t)cx * cy * cz;
    if (c >= nc) return;
    int I, J, K;
    cell_ijk(c, cx, cy, I, J, K);
    bool fluid = false, air = false;
    for (int dk = 0; dk < 2; ++dk) {
        const int k = 2 * K + dk;
        if (k >= fz) continue;
        for (int dj = 0; dj < 2; ++dj) {
            const int j = 2 * J + dj;
            if (j >= fy) continue;
            for (int di = 0; di < 2; ++di) {
                const int i = 2 * I + di;
                if (i >= fx) continue;
                const uint8_t f = ff[(int64_t)i + (int64_t)fx * ((int64_t)j + (int64_t)fy * k)];
                fluid |= f == FE_FLUID;
                air |= f == FE_AIR;
            }
        }
    }
    cf[c] = air ? (uint8_t)FE_AIR : (fluid ? (uint8_t)FE_FLUID : (uint8_t)FE_BOUNDRY);
}

// The coarse markers of levels 1 .. m (m <= kPyr) in one launch: a
// workgroup takes a block of 8 x 8 x 8 level-1 cells and the pyramid above
// it (4^3, 2^3 and 1 cells of levels 2, 3, 4; a level-q cell's children are
// level-(q-1) cells of the same block), each level from the one below in LDS
// by k_mg_coarsen's rule -- AIR if a child is AIR, else FLUID if a child is
// FLUID, else BOUNDRY, over the children that exist.  It also leaves the
// fine-tile flags of the fused V-cycle's finest level (a block's level-0
// region is two 16 x 16 x 8 tiles or eight 8 x 8 x 8 ones): whether the tile
// holds a FLUID cell.
constexpr int kPyr = 4;
constexpr int kPyrThreads = 512;
constexpr uint8_t kNoCell = 255;  // a cell beyond its level's dims

struct PyrArgs {
    int levels;           // m, levels 1 .. m computed here
    int n[kPyr + 1][3];   // dims of levels 0 .. m
    uint8_t* flags[kPyr + 1];
    uint8_t* tfl;         // tile flags of level 0 (null: not wanted)
    int tiles[3];         // tile counts of level 0's fused tiles
    int rx, ry, rz;       // and their level-1 cells per axis (8 or 4)
};

__global__ __launch_bounds__(kPyrThreads) void k_mg_pyramid(PyrArgs a) {
    __shared__ uint8_t L[2][512];
    const int t = (int)threadIdx.x;
    const int bx = (a.n[1][0] + 7) / 8, by = (a.n[1][1] + 7) / 8;
    const int b = (int)blockIdx.x;
    const int B[3] = {b % bx, (b / bx) % by, b / (bx * by)};
    // level 1 from level 0, plus the tile flags
    int fluid0 = 0;
    {
        const int I = 8 * B[0] + t % 8, J = 8 * B[1] + (t / 8) % 8, K = 8 * B[2] + t / 64;
        uint8_t out = kNoCell;
        if (I < a.n[1][0] && J < a.n[1][1] && K < a.n[1][2]) {
            const int fx = a.n[0][0], fy = a.n[0][1], fz = a.n[0][2];
            bool fluid = false, air = false;
            for (int dk = 0; dk < 2; ++dk) {
                const int k = 2 * K + dk;
                if (k >= fz) continue;
                for (int dj = 0; dj < 2; ++dj) {
                    const int j = 2 * J + dj;
                    if (j >= fy) continue;
                    for (int di = 0; di < 2; ++di) {
                        const int i = 2 * I + di;
                        if (i >= fx) continue;
                        const uint8_t f = a.flags[0][(int64_t)i + (int64_t)fx * ((int64_t)j + (int64_t)fy * k)];
                        fluid |= f == FE_FLUID;
                        air |= f == FE_AIR;
                    }
                }
            }
            out = air ? (uint8_t)FE_AIR : (fluid ? (uint8_t)FE_FLUID : (uint8_t)FE_BOUNDRY);
            a.flags[1][(int64_t)I + (int64_t)a.n[1][0] * ((int64_t)J + (int64_t)a.n[1][1] * K)] = out;
            fluid0 = fluid ? 1 : 0;
        }
        L[0][t] = out;
    }
    if (a.tfl) {
        // the tiles of this block: 8 / rx by 8 / ry by 8 / rz
        __shared__ int has[8];
        if (t < 8) has[t] = 0;
        __syncthreads();
        const int mx = 8 / a.rx, my = 8 / a.ry, mz = 8 / a.rz;
        if (fluid0) has[(t % 8) / a.rx + mx * ((t / 8) % 8 / a.ry + my * (t / 64 / a.rz))] = 1;
        __syncthreads();
        if (t < mx * my * mz) {
            const int tx = mx * B[0] + t % mx, ty = my * B[1] + (t / mx) % my, tz = mz * B[2] + t / (mx * my);
            if (tx < a.tiles[0] && ty < a.tiles[1] && tz < a.tiles[2])
                a.tfl[(int64_t)tx + (int64_t)a.tiles[0] * ((int64_t)ty + (int64_t)a.tiles[1] * tz)] = (uint8_t)has[t];
        }
    } else {
        __syncthreads();
    }
    // levels 2 .. m from the level below, in LDS
    int side = 8;
    for (int q = 2; q <= a.levels; ++q) {
        const uint8_t* below = L[q & 1];
        uint8_t* here = L[(q + 1) & 1];
        const int cs = side / 2;  // this level's block side
        if (t < cs * cs * cs) {
            const int tx = t % cs, ty = (t / cs) % cs, tz = t / (cs * cs);
            const int I = cs * B[0] + tx, J = cs * B[1] + ty, K = cs * B[2] + tz;
            uint8_t out = kNoCell;
            if (I < a.n[q][0] && J < a.n[q][1] && K < a.n[q][2]) {
                bool fluid = false, air = false;
                for (int d = 0; d < 8; ++d) {
                    const uint8_t f = below[(2 * tx + (d & 1)) + side * ((2 * ty + ((d >> 1) & 1)) + side * (2 * tz + (d >> 2)))];
                    fluid |= f == FE_FLUID;
                    air |= f == FE_AIR;
                }
                out = air ? (uint8_t)FE_AIR : (fluid ? (uint8_t)FE_FLUID : (uint8_t)FE_BOUNDRY);
                a.flags[q][(int64_t)I + (int64_t)a.n[q][0] * ((int64_t)J + (int64_t)a.n[q][1] * K)] = out;
            }
            here[t] = out;
        }
        __syncthreads();
        side = cs;
    }
}

// The row codes of levels 1 .. L-1 in one launch: thread c of the flattened
// cell range, level by level (offsets in off[]).
constexpr int kMaxLevels = 16;
struct CodesArgs {
    int levels;                  // coarse levels (1 .. levels)
    int64_t off[kMaxLevels + 1]; // first flattened cell of each coarse level
    int n[kMaxLevels][3];
    const uint8_t* flags[kMaxLevels];
    uint16_t* code[kMaxLevels];
};

__global__ __launch_bounds__(kBlock) void k_mg_codes_all(CodesArgs a) {
    const int64_t g = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (g >= a.off[a.levels]) return;
    int q = 0;
    while (q + 1 < a.levels && g >= a.off[q + 1]) ++q;
    const int64_t c = g - a.off[q];
    const int nx = a.n[q][0], ny = a.n[q][1], nz = a.n[q][2];
    int i, j, k;
    cell_ijk(c, nx, ny, i, j, k);
    a.code[q][c] = row_code(a.flags[q], c, (uint32_t)i, (uint32_t)j, (uint32_t)k, (uint32_t)nx, (uint32_t)ny,
                            (uint32_t)nz);
}

__global__ __launch_bounds__(kBlock) void k_mg_codes(const uint8_t* __restrict__ flags, int nx, int ny, int nz,
                                                     uint16_t* __restrict__ code) {
    const int64_t c = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    const int64_t nc = (int64_t)nx * ny * nz;
    if (c >= nc) return;
    int i, j, k;
    cell_ijk(c, nx, ny, i, j, k);
    code[c] = row_code(flags, c, (uint32_t)i, (uint32_t)j, (uint32_t)k, (uint32_t)nx, (uint32_t)ny, (uint32_t)nz);
}

// ---------------------------------------------------------------------------
// Transfer weights
// ---------------------------------------------------------------------------
// Prolongation of fine index fi on one axis: two coarse neighbours a, b.
__device__ inline void prolong_axis(int fi, int nc, int& a, float& wa, int& b, float& wb) {
    const int m = fi >> 1;
    if (fi & 1) {
        a = m;
        wa = 0.75f;
        b = min(m + 1, nc - 1);
        wb = 0.25f;
    } else {
        a = max(m - 1, 0);
        wa = 0.25f;
        b = m;
        wb = 0.75f;
    }
}

// Weight with which fine index fi feeds coarse index I (the transpose).
__device__ inline float restrict_w(int fi, int I, int nc) {
    int a, b;
    float wa, wb;
    prolong_axis(fi, nc, a, wa, b, wb);
    return (a == I ? wa : 0.0f) + (b == I ? wb : 0.0f);
}

// The fine indices 2I-1 .. 2I+2 whose prolongation reaches coarse index I,
// clamped into range, with their weights (0 outside the grid).
__device__ inline void restrict_taps(int I, int nf, int nc, int (&idx)[4], float (&w)[4]) {
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const int fi = 2 * I - 1 + t;
        const bool in = fi >= 0 && fi < nf;
        idx[t] = min(max(fi, 0), nf - 1);
        w[t] = in ? restrict_w(fi, I, nc) : 0.0f;
    }
}

// One x row of a coarse cell's window; R(t) is the residual at tap t.
template <typename F>
__device__ inline float restrict_row(const float (&w)[4], F R) {
    float s = 0.0f;
#pragma unroll
    for (int t = 0; t < 4; ++t) s += w[t] * R(t);
    return s;
}

// (1/8) sum of the 4x4x4 fine window, 64 independent loads.
template <typename F>
__device__ inline float restrict_sum(int I, int J, int K, int fx, int fy, int fz, int cx, int cy, int cz, F R) {
    int ix[4], iy[4], iz[4];
    float wx[4], wy[4], wz[4];
    restrict_taps(I, fx, cx, ix, wx);
    restrict_taps(J, fy, cy, iy, wy);
    restrict_taps(K, fz, cz, iz, wz);
    float acc = 0.0f;
#pragma unroll
    for (int tk = 0; tk < 4; ++tk) {
#pragma unroll
        for (int tj = 0; tj < 4; ++tj) {
            const int64_t row = (int64_t)fx * ((int64_t)iy[tj] + (int64_t)fy * iz[tk]);
            acc += (wy[tj] * wz[tk]) * restrict_row(wx, [&](int ti) { return R(row + ix[ti]); });
        }
    }
    return acc * 0.125f;
}

// Trilinear prolongation of the coarse correction at fine cell (i, j, k);
// V(a, b, c) is the coarse value at coarse index (a, b, c).
template <typename F>
__device__ inline float prolong_at3(int i, int j, int k, int cx, int cy, int cz, F V) {
    int ia, ib, ja, jb, ka, kb;
    float wia, wib, wja, wjb, wka, wkb;
    prolong_axis(i, cx, ia, wia, ib, wib);
    prolong_axis(j, cy, ja, wja, jb, wjb);
    prolong_axis(k, cz, ka, wka, kb, wkb);
    return wka * (wja * (wia * V(ia, ja, ka) + wib * V(ib, ja, ka)) + wjb * (wia * V(ia, jb, ka) + wib * V(ib, jb, ka))) +
           wkb * (wja * (wia * V(ia, ja, kb) + wib * V(ib, ja, kb)) + wjb * (wia * V(ia, jb, kb) + wib * V(ib, jb, kb)));
}

// The same with X(n) the coarse value at linear index n.
template <typename F>
__device__ inline float prolong_at(int i, int j, int k, int cx, int cy, int cz, F X) {
    return prolong_at3(i, j, k, cx, cy, cz,
                       [&](int a, int b, int c) { return X((int64_t)a + (int64_t)cx * ((int64_t)b + (int64_t)cy * c)); });
}

// One damped-Jacobi update of a cell, x + w (b - A x): the smoother of every
// level and kernel variant (the same expression, so the same rounding).
__device__ inline float mg_sweep_cell(uint16_t cd, float xc, float bc, const float (&nb)[6], const float ih2[3],
                                     float omega) {
    const float dgn = code_center(cd, ih2);
    const float w = mg_weight(cd, ih2, omega);
    return xc + w * (bc - code_apply_nb(cd, dgn, ih2, xc, nb));
}
// The second smoothing step at cell c (mg_cheb2 with the cell's weights).
__device__ inline float mg_cheb2_cell(uint16_t cd, float xc, float x0, float bc, const float (&nb)[6],
                                      const float ih2[3], const MgSmooth& sm) {
    const float dgn = code_center(cd, ih2);
    const float w = mg_weight(cd, ih2, sm.omega);
    return mg_cheb2(xc, x0, sm.w21 * w, bc - code_apply_nb(cd, dgn, ih2, xc, nb), sm.beta);
}

// The residual b - A x of a FLUID cell, 0 elsewhere.
__device__ inline float mg_residual_cell(uint16_t cd, float xc, float bc, const float (&nb)[6], const float ih2[3]) {
    return (cd & kFluidBit) ? bc - code_apply_nb(cd, code_center(cd, ih2), ih2, xc, nb) : 0.0f;
}

// A level's diagonal and smoother weight for FLUID rows, one entry per lane:
// lane n + 3 m + 9 p of every wavefront holds code_center and mg_weight of a
// FLUID row with n, m and p non-BOUNDRY neighbours along x, y and z (the only
// bits of a FLUID row's code that the two functions read), so the values are
// theirs.  Each wavefront builds its own copy (no LDS, no barrier) and reads it
// with a cross-lane permute.
struct CodeLanes {
    float cen, wgt;
};

__device__ inline CodeLanes code_lanes(const float ih2[3], float omega) {
    const int L = (int)(threadIdx.x & 63) % 27;  // lanes 27..63 repeat entries, never read
    const uint16_t cd = (uint16_t)(kFluidBit | ((L % 3) << 6) | (((L / 3) % 3) << 8) | ((L / 9) << 10));
    return CodeLanes{code_center(cd, ih2), mg_weight(cd, ih2, omega)};
}

// Lane of a FLUID row's entry.  Every lane of the wavefront must execute the
// permutes that read it (call outside divergent code).
__device__ inline int code_lane(uint32_t cd) {
    return (int)(((cd >> 6) & 3) + 3 * ((cd >> 8) & 3) + 9 * ((cd >> 10) & 3));
}

__device__ inline float lane_read(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_ds_bpermute(lane << 2, __float_as_int(v)));
}

// A x at a FLUID row whose neighbours outside FLUID hold 0: a FLUID row
// couples to exactly its FLUID neighbours, and every vector of the V-cycle is
// 0 outside FLUID cells (the CG start puts the solution's non-FLUID entries at
// 0, the residual is 0 there from then on, restriction and prolongation skip
// those cells), so each coupling term is taken without consulting the code:
// an uncoupled neighbour adds -ih2 * 0.  The terms and their order are
// code_apply_nb's, so the value is too.  cen = code_center of the row; nih2 =
// -1/h^2 per axis.
__device__ inline float mg_apply_fluid_row(float cen, float xc, const float (&nb)[6], const float nih2[3]) {
    float acc = cen * xc;
    acc = fmaf(nih2[0], nb[0], acc);
    acc = fmaf(nih2[0], nb[1], acc);
    acc = fmaf(nih2[1], nb[2], acc);
    acc = fmaf(nih2[1], nb[3], acc);
    acc = fmaf(nih2[2], nb[4], acc);
    acc = fmaf(nih2[2], nb[5], acc);
    return acc;
}

// mg_sweep_cell at a FLUID row under the same condition (w = mg_weight).  At a
// non-FLUID cell (x and b 0) mg_sweep_cell gives 0, which the callers write
// without reading the neighbours.
__device__ inline float mg_sweep_fluid_row(float cen, float w, float xc, float bc, const float (&nb)[6],
                                           const float nih2[3]) {
    return xc + w * (bc - mg_apply_fluid_row(cen, xc, nb, nih2));
}

// ---------------------------------------------------------------------------
// Large levels: one kernel per step
// ---------------------------------------------------------------------------
struct LevelArgs {
    int64_t nc;
    Stride st;
    float ih2[3];
    int64_t chunk, padded;
};

// What a smoothing sweep or a residual reads for cell c.
struct StencilIn {
    uint16_t cd;
    float xc, bc, nb[6];
};

template <typename F>
__device__ inline StencilIn stencil_in(int64_t c, const uint16_t* __restrict__ code, const float* __restrict__ x,
                                       const float* __restrict__ b, const Stride& st, F X) {
    StencilIn t;
    t.cd = code[c];
    t.xc = x[c];
    t.bc = b[c];
    code_neighbours(c, st, X, t.nb);
    return t;
}

// x_out = x_in + w (b - A x_in).  With prz != nullptr (the last level-0 sweep)
// also leaves partials of b . x_out, which is r . z of the CG.  With pconf !=
// nullptr (the V-cycle's first kernel) and a pending confirmation, the
// residual the CG update just recomputed as b - A x is tested first: when it
// meets the relative stop the solve ends here (iteration count of that
// update), without this V-cycle and the next spmv.  cfl (level 0 only): the
// solver chunks holding a FLUID cell; the others hold zeros and are skipped.
__global__ __launch_bounds__(kBlock) void k_mg_smooth(LevelArgs L, const uint16_t* __restrict__ code,
                                                      const float* __restrict__ b, const float* __restrict__ xin,
                                                      float* xout, const SolverScalars* st,
                                                      double* __restrict__ prz, const double* __restrict__ pconf,
                                                      int nparts, const uint8_t* __restrict__ cfl, int second,
                                                      const float* x0, int fine) {
    // The stop flag is read with the data and tested before the first write,
    // so its load adds no latency of its own (the loads before it are in bounds).
    const int done = st->done;
    if (pconf && done) return;
    if (pconf && st->confirm) {
        double t[2];
        sum_partials<2>(pconf, nparts, t);
        if (stop_rule(st, st->bnorm2, t[0], t[1])) {
            if (blockIdx.x == 0 && threadIdx.x == 0) {
                SolverScalars* w = const_cast<SolverScalars*>(st);
                w->rr = t[1];
                w->it = st->it + 1;
                w->converged = 1;
                w->done = 1;
            }
            return;
        }
    }
    const Span sp = block_span(L.nc, L.chunk, L.padded);
    if (cfl && !cfl[sp.lb]) {  // level 0 chunk without FLUID cells: x stays 0
        if (prz && threadIdx.x == 0) prz[blockIdx.x] = 0.0;
        return;
    }
    const Stride stv = L.st;
    double v[1] = {0.0};
    auto X = [&](int64_t n) { return xin[n]; };
    span_groups<8, StencilIn>(
        sp.c0, sp.c1, [&](int64_t c) { return stencil_in(c, code, xin, b, stv, X); },
        [&](int64_t c, const StencilIn& t) {
            if (done) return;  // uniform: the solve has stopped
            // second: the second smoothing step, from x0 (null: 0); x0 may be
            // xout (each cell reads its own x0 before writing it)
            const MgSmooth& sm = fine ? kMgFine : kMgCoarse;
            const float xo = second ? mg_cheb2_cell(t.cd, t.xc, x0 ? x0[c] : 0.0f, t.bc, t.nb, L.ih2, sm)
                                    : mg_sweep_cell(t.cd, t.xc, t.bc, t.nb, L.ih2, sm.omega);
            xout[c] = xo;
            v[0] += (double)t.bc * (double)xo;
        });
    if (done) return;
    if (prz) write_partials<1>(v, prz);
}

__global__ __launch_bounds__(kBlock) void k_mg_residual(LevelArgs L, const uint16_t* __restrict__ code,
                                                        const float* __restrict__ b, const float* __restrict__ x,
                                                        float* __restrict__ r, const SolverScalars* __restrict__ st,
                                                        const uint8_t* __restrict__ cfl) {
    const int done = st->done;  // tested before the first write (see k_mg_smooth)
    const Span sp = block_span(L.nc, L.chunk, L.padded);
    if (cfl && !cfl[sp.lb]) return;  // level 0 chunk without FLUID cells: r stays 0
    const Stride stv = L.st;
    auto X = [&](int64_t n) { return x[n]; };
    span_groups<8, StencilIn>(
        sp.c0, sp.c1, [&](int64_t c) { return stencil_in(c, code, x, b, stv, X); },
        [&](int64_t c, const StencilIn& t) {
            if (done) return;
            r[c] = mg_residual_cell(t.cd, t.xc, t.bc, t.nb, L.ih2);
        });
}

// b_c = R r_f on coarse FLUID cells (0 elsewhere); with x1 != nullptr also the
// coarse level's first sweep from zero, x1 = w b_c.  A workgroup covers an
// 8x8x4 coarse tile and first stages the 18x18x10 fine window it reads in LDS.
constexpr int kRtx = 8, kRty = 8, kRtz = 4;
constexpr int kRwx = 2 * kRtx + 2, kRwy = 2 * kRty + 2, kRwz = 2 * kRtz + 2;
static_assert(kRtx * kRty * kRtz == kBlock, "one coarse cell per thread");

__global__ __launch_bounds__(kBlock) void k_mg_restrict(const float* __restrict__ rf, int fx, int fy, int fz,
                                                        const uint16_t* __restrict__ ccode, float* __restrict__ bc,
                                                        float* __restrict__ x1, int cx, int cy, int cz, float cihx2,
                                                        float cihy2, float cihz2,
                                                        const SolverScalars* __restrict__ st) {
    const int done = st->done;  // tested before the first write (see k_mg_smooth)
    __shared__ float win[kRwz][kRwy][kRwx];
    const int I0 = blockIdx.x * kRtx, J0 = blockIdx.y * kRty, K0 = blockIdx.z * kRtz;
    const int fi0 = 2 * I0 - 1, fj0 = 2 * J0 - 1, fk0 = 2 * K0 - 1;
    const int tx = threadIdx.x % kRtx, ty = (threadIdx.x / kRtx) % kRty, tz = threadIdx.x / (kRtx * kRty);
    const int I = I0 + tx, J = J0 + ty, K = K0 + tz;
    const bool inside = I < cx && J < cy && K < cz;
    const int64_t c = (int64_t)I + (int64_t)cx * ((int64_t)J + (int64_t)cy * K);
    const uint16_t cd = inside ? ccode[c] : (uint16_t)0;  // issued with the window loads
    // All of a thread's window loads are issued before the first LDS store, so
    // the window costs one memory latency rather than one per element.
    constexpr int kWin = kRwx * kRwy * kRwz;
    constexpr int kPer = (kWin + kBlock - 1) / kBlock;
    float wv[kPer];
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
        const int e = threadIdx.x + u * kBlock;
        wv[u] = 0.0f;
        if (e < kWin) {
            const int wi = e % kRwx, wj = (e / kRwx) % kRwy, wk = e / (kRwx * kRwy);
            const int fi = min(max(fi0 + wi, 0), fx - 1);
            const int fj = min(max(fj0 + wj, 0), fy - 1);
            const int fk = min(max(fk0 + wk, 0), fz - 1);
            wv[u] = rf[(int64_t)fi + (int64_t)fx * ((int64_t)fj + (int64_t)fy * fk)];
        }
    }
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
        const int e = threadIdx.x + u * kBlock;
        if (e < kWin) (&win[0][0][0])[e] = wv[u];
    }
    __syncthreads();
    if (done || !inside) return;
    float v = 0.0f;
    if (cd & kFluidBit) {
        // window coordinates of fine index 2I-1+t are 2*tx+t (clamped taps carry weight 0)
        int ix[4], iy[4], iz[4];
        float wx[4], wy[4], wz[4];
        restrict_taps(I, fx, cx, ix, wx);
        restrict_taps(J, fy, cy, iy, wy);
        restrict_taps(K, fz, cz, iz, wz);
        float acc = 0.0f;
#pragma unroll
        for (int tk = 0; tk < 4; ++tk) {
#pragma unroll
            for (int tj = 0; tj < 4; ++tj) {
                acc += (wy[tj] * wz[tk]) *
                       restrict_row(wx, [&](int ti) { return win[2 * tz + tk][2 * ty + tj][2 * tx + ti]; });
            }
        }
        v = acc * 0.125f;
    }
    bc[c] = v;
    if (x1) {
        const float ih2[3] = {cihx2, cihy2, cihz2};
        x1[c] = mg_weight(cd, ih2, kMgCoarse.omega) * v;
    }
}

// x_f += P x_c on FLUID fine cells.
__global__ __launch_bounds__(kBlock) void k_mg_prolong(const float* __restrict__ xc, int cx, int cy, int cz,
                                                       const uint16_t* __restrict__ fcode, float* __restrict__ xf,
                                                       int fx, int fy, int fz, const SolverScalars* __restrict__ st) {
    const int done = st->done;  // tested before the write (see k_mg_smooth)
    const int64_t f = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    const int64_t nf = (int64_t)fx * fy * fz;
    if (f >= nf) return;
    // the marker, the fine value and the coarse values are loaded together
    const uint16_t cd = fcode[f];
    const float x0 = xf[f];
    int i, j, k;
    cell_ijk(f, fx, fy, i, j, k);
    const float add = prolong_at(i, j, k, cx, cy, cz, [&](int64_t n) { return xc[n]; });
    if (done || !(cd & kFluidBit)) return;
    xf[f] = x0 + add;
}

// ---------------------------------------------------------------------------
// Large levels, fused (FE_MG_FUSED): one descent and one ascent kernel per
// level.  A workgroup owns a coarse tile of T::rx x T::ry x T::rz cells and the
// fine tile of twice that size below it.  It stages what the tile's sweeps
// read, with halos, in LDS and recomputes the halo cells of each sweep itself
// instead of waiting for a neighbour tile, so a level takes two launches
// instead of six.  The terms of every value are the split kernels' (a neighbour
// outside the grid, which enters with weight 0, reads 0 here), and so is their
// order but for the restriction, whose four planes are added as a tree: the
// variants agree to FP32 rounding.  The sweeps and residuals take the FLUID-row forms (mg_sweep_fluid_row: diagonal and weight
// from a per-wavefront lane table, coupling terms without the code's selects),
// half the instructions of the general ones: the finest level's phases are
// VALU-bound (16 waves of a tile share one CU's four SIMDs).
// For the same reason a thread keeps one column of the window through all
// phases, P consecutive planes of it (FCols): its cells' place is decoded
// once instead of in every phase, their own values, diagonals and weights and
// the neighbours along z within its planes stay in registers, and every other
// neighbour is at a constant distance in LDS.  With the window's cells dealt
// to the threads anew in each phase the finest level's descent and ascent of a
// 128^3 dam break took 14.0 and 16.1 us, now 11.4 and 12.7; the small tiles
// below 5.6 us each, now 4.3 and 3.8.
//   descent:  x1 = w b (first sweep from zero), x2 = x1 + w (b - A x1) (kept
//             for the ascent), r = b - A x2, coarse b = R r;
//   ascent:   y = x2 + P xc, x' = y + w (b - A y), out = x' + w (b - A x'),
//             with level 0's out = z and the partials of r.z.
// Window of halo H around the fine tile: coordinates 0 .. T::fx + 2H - 1
// stand for fine indices f0 - H ...
// Two tile shapes (small_tiles): a level of many tiles is throughput-bound and
// takes large ones (little halo per cell); the others are latency-bound (a 32^3
// level has 16 large tiles for 256 CUs, and each workgroup's chain of LDS
// phases sets the kernel's time), so they take small tiles: 2.5x fewer cells
// per thread in every phase for more halo work in all.  A cell's value does
// not depend on the tile it is computed in.
// ---------------------------------------------------------------------------
template <int RX, int RY, int RZ>
struct FusedTile {
    static constexpr int rx = RX, ry = RY, rz = RZ;              // coarse tile
    static constexpr int fx = 2 * RX, fy = 2 * RY, fz = 2 * RZ;  // fine tile
    static constexpr int coarse = RX * RY * RZ;
};
using TileLarge = FusedTile<8, 8, 4>;
using TileSmall = FusedTile<4, 4, 4>;
template <class T, int H>
struct FWin {
    static constexpr int x = T::fx + 2 * H, y = T::fy + 2 * H, z = T::fz + 2 * H;
    static constexpr int sy = x, sz = x * y, n = x * y * z;
};
// coarse window of the ascent: coarse indices I0 - 2 .. I0 + T::rx + 1 per axis
template <class T>
struct CWin {
    static constexpr int x = T::rx + 4, y = T::ry + 4, z = T::rz + 4;
    static constexpr int sy = x, sz = x * y, n = x * y * z;
};

// Columns of the window of halo H, lane-contiguous in LDS: thread g * cols + c
// has planes [g P, (g + 1) P) of column c, P the least that kFusedThreads
// threads cover the window with.  Arrays hold G * P planes.
constexpr int kFusedThreads = 1024;  // 16 waves per tile
template <class T, int H>
struct FCols {
    using W = FWin<T, H>;
    static constexpr int cols = W::sz;
    static constexpr int planes() {
        int p = 1;
        while (cols * ((W::z + p - 1) / p) > kFusedThreads) ++p;
        return p;
    }
    static constexpr int P = planes(), G = (W::z + P - 1) / P;
    static constexpr int threads = (cols * G + 63) / 64 * 64;
    static constexpr int n = cols * G * P;
};

struct FusedArgs {
    int n[3];        // the fine level
    int c[3];        // the coarse level
    float ih2[3];    // the fine level's 1/h^2
    int tiles[3];    // coarse tiles per axis
    int64_t padded;  // launched workgroups (XCD remap), >= the tile count
};

__device__ inline int64_t fused_tile(const FusedArgs& a) { return xcd_remap(blockIdx.x, a.padded); }

__device__ inline bool fine_in(const FusedArgs& a, int i, int j, int k) {
    return i >= 0 && j >= 0 && k >= 0 && i < a.n[0] && j < a.n[1] && k < a.n[2];
}

// Linear index of an in-grid cell of a level with dims n: 32-bit arithmetic
// (a scene holds at most 2^30 cells).
__device__ inline uint32_t fused_index(int i, int j, int k, const int n[3]) {
    return (uint32_t)i + (uint32_t)n[0] * ((uint32_t)j + (uint32_t)n[1] * (uint32_t)k);
}

// tfl (level 0 only): per tile, whether its fine tile holds a FLUID cell.  A
// tile without one has every output 0 (its right-hand side and its coarse
// cells' are 0), and those stay as the solve's start left them.

// sum_partials for a kFusedThreads workgroup: every workgroup adds the NV-wide
// partials in the same fixed order (threads strided over the partials, lanes
// by wave_sum, waves in order), so all derive identical totals.
template <int NV>
__device__ inline void sum_partials_fused(const double* __restrict__ part, int nparts, double (&tot)[NV]) {
    __shared__ double sm[NV][kFusedThreads / 64];
#pragma unroll
    for (int q = 0; q < NV; ++q) tot[q] = 0.0;
    add_partials<NV, 1>(part, NV, 0, (int)threadIdx.x, kFusedThreads, nparts, tot);
    wave_sums(tot, sm);
    __syncthreads();
#pragma unroll
    for (int q = 0; q < NV; ++q) tot[q] = waves_total(sm[q]);
    __syncthreads();
}

template <bool L0, class T>
__global__ __launch_bounds__(kFusedThreads) void k_mg_down(FusedArgs a, const float* __restrict__ b,
                                                    const uint16_t* __restrict__ code, float* __restrict__ x2out,
                                                    const uint16_t* __restrict__ ccode, float* __restrict__ cb,
                                                    const SolverScalars* st, const double* __restrict__ pconf,
                                                    int nconf, const uint8_t* __restrict__ tfl) {
    using C = FCols<T, 3>;
    using W = typename C::W;
    constexpr int P = C::P;
    __shared__ float sX1[C::n];  // x1; later the residual
    __shared__ float sX2[C::n];
    const int done = st->done;  // read with the data, tested before the first write
    if (L0 && pconf) {
        // the V-cycle's first kernel: after a stop it returns; a relative stop
        // pending confirmation is tested on the residual the CG update just
        // recomputed (as k_mg_smooth), by every workgroup (workgroup 0 records
        // a stop).  Tested before the tile's loads: with the loads' registers
        // live across the test the kernel needs more than 64 VGPRs, and two
        // tiles no longer share a CU.
        if (done) return;
        if (st->confirm) {
            double tt[2];
            sum_partials_fused<2>(pconf, nconf, tt);
            if (stop_rule(st, st->bnorm2, tt[0], tt[1])) {
                if (blockIdx.x == 0 && threadIdx.x == 0) {
                    SolverScalars* w = const_cast<SolverScalars*>(st);
                    w->rr = tt[1];
                    w->it = st->it + 1;
                    w->converged = 1;
                    w->done = 1;
                }
                return;
            }
        }
    }
    const uint32_t t = (uint32_t)fused_tile(a);
    const bool real = t < (uint32_t)(a.tiles[0] * a.tiles[1] * a.tiles[2]) && !(L0 && tfl && !tfl[t]);
    if (!real) return;
    const uint32_t tx0 = (uint32_t)a.tiles[0], txy = tx0 * (uint32_t)a.tiles[1];
    const int TX = (int)(t % tx0), TY = (int)((t % txy) / tx0), TZ = (int)(t / txy);
    const int I0 = TX * T::rx, J0 = TY * T::ry, K0 = TZ * T::rz;
    const int fx0 = 2 * I0, fy0 = 2 * J0, fz0 = 2 * K0;
    // this thread's coarse cell (the restriction: four lanes per cell, one per
    // fine plane of its taps)
    const int tq = threadIdx.x & 3, tc = threadIdx.x >> 2;
    const int tx = tc % T::rx, ty = (tc / T::rx) % T::ry, tz = tc / (T::rx * T::ry);
    const int I = I0 + tx, J = J0 + ty, K = K0 + tz;
    const bool cin = tc < T::coarse && I < a.c[0] && J < a.c[1] && K < a.c[2];
    const uint32_t ci = fused_index(I, J, K, a.c);
    // this thread's column of the tile + 3
    const int g = threadIdx.x / C::cols, col = threadIdx.x - g * C::cols, z0 = g * P;
    const int wx = col % W::x, wy = col / W::x;
    const int i = fx0 - 3 + wx, j = fy0 - 3 + wy, k0 = fz0 - 3 + z0;
    const bool mine = g < C::G;
    const bool col_in = mine && i >= 0 && j >= 0 && i < a.n[0] && j < a.n[1];
    const uint32_t slab = (uint32_t)a.n[0] * (uint32_t)a.n[1];
    const uint32_t f0 = fused_index(i, j, k0, a.n);
    const int e = col + W::sz * z0;
    const int em = z0 > 0 ? e - W::sz : e;                                         // the plane below its planes
    const int ep = e + W::sz * (g < C::G - 1 ? P : P - 1);                         // and the one above
    const auto inner = [&](int h) { return mine && wx >= h && wx < W::x - h && wy >= h && wy < W::y - h; };
    // b and the row codes: every load issued before any LDS store (the codes
    // in whole registers, so no load waits for another)
    float vb[P];
    uint32_t vc[P];
#pragma unroll
    for (int u = 0; u < P; ++u) {
        vb[u] = 0.0f;
        vc[u] = 0;
        if (col_in && (unsigned)(k0 + u) < (unsigned)a.n[2]) {
            vb[u] = b[f0 + u * slab];
            vc[u] = code[f0 + u * slab];
        }
    }
    const uint32_t ccd = cin ? (uint32_t)ccode[ci] : 0u;
    constexpr MgSmooth SM = L0 ? kMgFine : kMgCoarse;
    const CodeLanes lanes = code_lanes(a.ih2, SM.omega);
    const float nih2[3] = {-a.ih2[0], -a.ih2[1], -a.ih2[2]};
    float cen[P], wgt[P], x[P];
    uint32_t fluid = 0;
#pragma unroll
    for (int u = 0; u < P; ++u) {
        const int li = code_lane(vc[u]);  // every lane: cross-lane reads
        cen[u] = lane_read(lanes.cen, li);
        wgt[u] = lane_read(lanes.wgt, li);
        const bool fl = vc[u] & kFluidBit;
        fluid |= fl ? 1u << u : 0u;
        x[u] = (fl ? wgt[u] : SM.omega) * vb[u];  // the first sweep from zero
        if (mine) sX1[e + W::sz * u] = x[u];
    }
    __syncthreads();
    if (done) return;  // uniform: the solve has stopped
    // x2 on the tile + 2; the tile's own cells also go to global memory.  The
    // planes past the window's halo take values that nothing reads.
    if (inner(1)) {
        const bool tile_col = inner(3) && col_in;
        float lo = sX1[em];
        const float hi = sX1[ep];
#pragma unroll
        for (int u = 0; u < P; ++u) {
            const float* q = sX1 + e + W::sz * u;
            const float nb[6] = {q[-1], q[1], q[-W::x], q[W::x], lo, u < P - 1 ? x[u < P - 1 ? u + 1 : u] : hi};
            lo = x[u];
            const float x2 = mg_cheb2(x[u], 0.0f, SM.w21 * wgt[u], vb[u] - mg_apply_fluid_row(cen[u], x[u], nb, nih2),
                                      SM.beta);
            x[u] = (fluid >> u) & 1u ? x2 : 0.0f;
            sX2[e + W::sz * u] = x[u];
            if (tile_col && z0 + u >= 3 && z0 + u < 3 + T::fz && k0 + u < a.n[2]) x2out[f0 + u * slab] = x[u];
        }
    }
    __syncthreads();
    // r on the tile + 1 (into sX1, whose x1 is no longer read)
    float* sR = sX1;
    if (inner(2)) {
        float lo = sX2[em];
        const float hi = sX2[ep];
#pragma unroll
        for (int u = 0; u < P; ++u) {
            const float* q = sX2 + e + W::sz * u;
            const float nb[6] = {q[-1], q[1], q[-W::x], q[W::x], lo, u < P - 1 ? x[u < P - 1 ? u + 1 : u] : hi};
            lo = x[u];
            const float r = vb[u] - mg_apply_fluid_row(cen[u], x[u], nb, nih2);
            sR[e + W::sz * u] = (fluid >> u) & 1u ? r : 0.0f;
        }
    }
    __syncthreads();
    // coarse b = R r: fine index 2I-1+t sits at window coordinate 2*(I - I0) + 2 + t
    if (tc >= T::coarse) return;  // whole wavefronts
    float acc = 0.0f;
    if (cin && (ccd & kFluidBit)) {
        int ix[4], iy[4], iz[4];
        float cx[4], cy[4], cz[4];
        restrict_taps(I, a.n[0], a.c[0], ix, cx);
        restrict_taps(J, a.n[1], a.c[1], iy, cy);
        restrict_taps(K, a.n[2], a.c[2], iz, cz);
        const float wk = tq < 2 ? (tq == 0 ? cz[0] : cz[1]) : (tq == 2 ? cz[2] : cz[3]);
        const float* q = sR + (2 * tx + 2) + W::sy * (2 * ty + 2) + W::sz * (2 * tz + 2 + tq);
#pragma unroll
        for (int tj = 0; tj < 4; ++tj) {
            acc += (cy[tj] * wk) * restrict_row(cx, [&](int ti) { return q[ti + W::sy * tj]; });
        }
    }
    acc += __shfl_xor(acc, 1, 4);
    acc += __shfl_xor(acc, 2, 4);
    if (cin && tq == 0) cb[ci] = acc * 0.125f;
}

// out = the level's corrected and post-smoothed solution.  With prz (level 0)
// every launched workgroup leaves one partial of b . out (r.z).
template <bool L0, class T>
__global__ __launch_bounds__((FCols<T, 2>::threads)) void k_mg_up(FusedArgs a, const float* __restrict__ x2,
                                                  const float* __restrict__ xc, const float* __restrict__ b,
                                                  const uint16_t* __restrict__ code, float* __restrict__ out,
                                                  double* __restrict__ prz, const SolverScalars* __restrict__ st,
                                                  const uint8_t* __restrict__ tfl) {
    using C = FCols<T, 2>;
    using W = typename C::W;
    using Wc = CWin<T>;
    constexpr int P = C::P;
    static_assert(P % 2 == 0, "a thread's planes start at an even fine index");
    __shared__ float sY[C::n];
    __shared__ float sXp[C::n];
    __shared__ float sXc[Wc::n];
    const int done = st->done;  // read with the data, tested before the first write
    const uint32_t t = (uint32_t)fused_tile(a);
    const bool real = t < (uint32_t)(a.tiles[0] * a.tiles[1] * a.tiles[2]) && !(L0 && tfl && !tfl[t]);
    const uint32_t tx0 = (uint32_t)a.tiles[0], txy = tx0 * (uint32_t)a.tiles[1];
    const int TX = (int)(t % tx0), TY = (int)((t % txy) / tx0), TZ = (int)(t / txy);
    const int fx0 = 2 * TX * T::rx, fy0 = 2 * TY * T::ry, fz0 = 2 * TZ * T::rz;
    // this thread's column of the tile + 2
    const int g = threadIdx.x / C::cols, col = threadIdx.x - g * C::cols, z0 = g * P;
    const int wx = col % W::x, wy = col / W::x;
    const int i = fx0 - 2 + wx, j = fy0 - 2 + wy, k0 = fz0 - 2 + z0;
    const bool mine = g < C::G;
    const bool col_in = mine && i >= 0 && j >= 0 && i < a.n[0] && j < a.n[1];
    const uint32_t slab = (uint32_t)a.n[0] * (uint32_t)a.n[1];
    const uint32_t f0 = fused_index(i, j, k0, a.n);
    const int e = col + W::sz * z0;
    const int em = z0 > 0 ? e - W::sz : e;                  // the plane below its planes
    const int ep = e + W::sz * (g < C::G - 1 ? P : P - 1);  // and the one above
    const auto inner = [&](int h) { return mine && wx >= h && wx < W::x - h && wy >= h && wy < W::y - h; };
    float y[P], vb[P];
    uint32_t vc[P];
    if (real) {
        // x2, b and the row codes of the column and the coarse correction on
        // its window (clamped into the grid, as the prolongation clamps): every
        // load issued before any LDS store (the codes in whole registers, so no
        // load waits for another)
#pragma unroll
        for (int u = 0; u < P; ++u) {
            y[u] = vb[u] = 0.0f;
            vc[u] = 0;
            if (col_in && (unsigned)(k0 + u) < (unsigned)a.n[2]) {
                y[u] = x2[f0 + u * slab];
                vb[u] = b[f0 + u * slab];
                vc[u] = code[f0 + u * slab];
            }
        }
        constexpr int kPc = (Wc::n + C::threads - 1) / C::threads;
        float vxc[kPc];
#pragma unroll
        for (int u = 0; u < kPc; ++u) {
            const int q = threadIdx.x + u * C::threads;
            vxc[u] = 0.0f;
            if (q < Wc::n) {
                const int qx = q % Wc::x, qy = (q / Wc::x) % Wc::y, qz = q / Wc::sz;
                const int I = min(max(fx0 / 2 - 2 + qx, 0), a.c[0] - 1), J = min(max(fy0 / 2 - 2 + qy, 0), a.c[1] - 1),
                          K = min(max(fz0 / 2 - 2 + qz, 0), a.c[2] - 1);
                vxc[u] = xc[fused_index(I, J, K, a.c)];
            }
        }
#pragma unroll
        for (int u = 0; u < kPc; ++u) {
            const int q = threadIdx.x + u * C::threads;
            if (q < Wc::n) sXc[q] = vxc[u];
        }
    }
    constexpr MgSmooth SM = L0 ? kMgFine : kMgCoarse;
    const CodeLanes lanes = code_lanes(a.ih2, SM.omega);
    const float nih2[3] = {-a.ih2[0], -a.ih2[1], -a.ih2[2]};
    float cen[P], wgt[P];
    uint32_t fluid = 0;
    if (real) {  // the whole workgroup: cross-lane reads
#pragma unroll
        for (int u = 0; u < P; ++u) {
            const int li = code_lane(vc[u]);
            cen[u] = lane_read(lanes.cen, li);
            wgt[u] = lane_read(lanes.wgt, li);
            fluid |= vc[u] & kFluidBit ? 1u << u : 0u;
        }
    }
    __syncthreads();
    if (done) return;  // uniform: the solve has stopped
    double v[1] = {0.0};
    if (real && mine) {
        // y = x2 + P xc on FLUID cells: prolong_at3's terms, the window's
        // coarse index (fine index >> 1) - (tile's first - 2); the bilinear
        // part of a coarse plane serves the two to four fine planes it feeds
        const int ia = (wx >> 1) + (wx & 1), ja = (wy >> 1) + (wy & 1);  // the lower neighbour of each axis
        const float wia = wx & 1 ? 0.75f : 0.25f, wja = wy & 1 ? 0.75f : 0.25f;
        const float wib = 1.0f - wia, wjb = 1.0f - wja;
        const float* q = sXc + ia + Wc::sy * ja + Wc::sz * (z0 >> 1);
        float S[P / 2 + 2];
#pragma unroll
        for (int m = 0; m < P / 2 + 2; ++m) {
            const float* r = q + Wc::sz * m;
            S[m] = wja * (wia * r[0] + wib * r[1]) + wjb * (wia * r[Wc::sy] + wib * r[Wc::sy + 1]);
        }
#pragma unroll
        for (int u = 0; u < P; ++u) {
            const float add = u & 1 ? 0.75f * S[u / 2 + 1] + 0.25f * S[u / 2 + 2] : 0.25f * S[u / 2] + 0.75f * S[u / 2 + 1];
            y[u] = (fluid >> u) & 1u ? y[u] + add : y[u];
            sY[e + W::sz * u] = y[u];
        }
    }
    __syncthreads();
    float xp[P];
    if (real && inner(1)) {
        // x' on the tile + 1 (the planes past it take values that nothing reads)
        float lo = sY[em];
        const float hi = sY[ep];
#pragma unroll
        for (int u = 0; u < P; ++u) {
            const float* q = sY + e + W::sz * u;
            const float nb[6] = {q[-1], q[1], q[-W::x], q[W::x], lo, u < P - 1 ? y[u < P - 1 ? u + 1 : u] : hi};
            lo = y[u];
            const float x1 = mg_sweep_fluid_row(cen[u], wgt[u], y[u], vb[u], nb, nih2);
            xp[u] = (fluid >> u) & 1u ? x1 : 0.0f;
            sXp[e + W::sz * u] = xp[u];
        }
    }
    __syncthreads();
    if (real && inner(2) && col_in) {
        // out on the tile
        float lo = sXp[em];
        const float hi = sXp[ep];
#pragma unroll
        for (int u = 0; u < P; ++u) {
            const float* q = sXp + e + W::sz * u;
            const float nb[6] = {q[-1], q[1], q[-W::x], q[W::x], lo, u < P - 1 ? xp[u < P - 1 ? u + 1 : u] : hi};
            lo = xp[u];
            if (z0 + u < 2 || z0 + u >= 2 + T::fz || k0 + u >= a.n[2]) continue;
            float o = 0.0f;
            if ((fluid >> u) & 1u) {
                o = mg_cheb2(xp[u], y[u], SM.w21 * wgt[u], vb[u] - mg_apply_fluid_row(cen[u], xp[u], nb, nih2), SM.beta);
                if (L0) v[0] += (double)vb[u] * (double)o;
            }
            out[f0 + u * slab] = o;
        }
    }
    if (L0 && prz) {  // one partial per workgroup
        __shared__ double sm[1][C::threads / 64];
        wave_sums(v, sm);
        __syncthreads();
        if (threadIdx.x == 0) prz[blockIdx.x] = waves_total(sm[0]);
    }
}


// ---------------------------------------------------------------------------
// Small levels: the rest of the V-cycle in one workgroup
// ---------------------------------------------------------------------------
struct TailArgs {
    int levels;  // tail levels; the last is the coarsest
    int n[kMaxTail][3];
    float ih2[kMaxTail][3];
    const uint16_t* code[kMaxTail];
    int off[kMaxTail];  // offset of each level in the LDS arrays
};

// Tail level t in LDS: values at V + o, row codes at Cd + o.
struct TailLevel {
    int nx, ny, nz, nc, o;
    Stride32 st;
    float ih2[3];
};

__device__ inline TailLevel tail_level(const TailArgs& a, int t) {
    TailLevel l;
    l.nx = a.n[t][0];
    l.ny = a.n[t][1];
    l.nz = a.n[t][2];
    l.nc = l.nx * l.ny * l.nz;
    l.o = a.off[t];
    l.st = Stride32{l.nx, l.nx * l.ny, l.nc - 1};
    for (int q = 0; q < 3; ++q) l.ih2[q] = a.ih2[t][q];
    return l;
}

// One Jacobi sweep: out = in + w (b - A in), or out = w b when `in` is null.
// dg, wt: the level's diagonal and smoother weight per cell (precomputed).
// One Chebyshev step on the coarsest level (wt = 1/diagonal): d = c1 d +
// c2 D^-1 (b - A in), out = in + d; from zero (in == nullptr) d = c2 D^-1 b.
// d is per cell, so it is updated in place.
__device__ inline void tail_cheb(const TailLevel& l, const uint16_t* code, const float* dg, const float* wt,
                                 const float* in, float* out, const float* b, float* d, float c1, float c2) {
#pragma unroll
    for (int u = 0; u < kTailPer; ++u) {
        const int c = threadIdx.x + u * kTailThreads;
        if (c >= l.nc) break;
        const uint16_t cd = code[c];
        const float w = wt[c];
        float xo, dn;
        if (in) {
            const float xc = in[c];
            const float r = w * (b[c] - code_apply(cd, dg[c], c, l.st, l.ih2, xc, [&](int n) { return in[n]; }));
            dn = c1 * d[c] + c2 * r;
            xo = xc + dn;
        } else {
            dn = c2 * (w * b[c]);
            xo = dn;
        }
        d[c] = dn;
        out[c] = xo;
    }
    __syncthreads();
}

__device__ inline void tail_sweep(const TailLevel& l, const uint16_t* code, const float* dg, const float* wt,
                                  const float* in, float* out, const float* b) {
    // a tail level holds at most kTailMax cells: a fixed trip count lets the
    // LDS reads of a thread's cells overlap
#pragma unroll
    for (int u = 0; u < kTailPer; ++u) {
        const int c = threadIdx.x + u * kTailThreads;
        if (c >= l.nc) break;
        const uint16_t cd = code[c];
        const float w = wt[c];
        float xo;
        if (in) {
            const float xc = in[c];
            xo = xc + w * (b[c] - code_apply(cd, dg[c], c, l.st, l.ih2, xc, [&](int n) { return in[n]; }));
        } else {
            xo = w * b[c];
        }
        out[c] = xo;
    }
    __syncthreads();
}

// Solves level T's right-hand side bT approximately with the V-cycle of the
// tail levels; the result goes to xT.  Everything lives in LDS: five values
// (two iterates, right-hand side, diagonal, smoother weight) and the row code
// per cell of every tail level (at most kTailLds cells).
__global__ __launch_bounds__(kTailThreads) void k_mg_tail(TailArgs a, const float* __restrict__ bT,
                                                          float* __restrict__ xT,
                                                          const SolverScalars* __restrict__ st) {
    const int done = st->done;  // tested after the loads below (see k_mg_smooth)
    __shared__ float X[kTailLds], Tm[kTailLds], B[kTailLds], Dg[kTailLds], Wt[kTailLds];
    __shared__ float Dd[kCoarseMax];  // the coarsest level's Chebyshev direction
    __shared__ uint16_t Cd[kTailLds];
    // Row codes and the right-hand side: every load is issued before the
    // first LDS store (one memory latency in all).
    constexpr int kPer = kTailPer;
    const int n0 = a.n[0][0] * a.n[0][1] * a.n[0][2];
    {
        float bv[kPer];
        uint16_t cv[kMaxTail][kPer];
#pragma unroll
        for (int u = 0; u < kPer; ++u) {
            const int c = threadIdx.x + u * kTailThreads;
            bv[u] = c < n0 ? bT[c] : 0.0f;
        }
#pragma unroll
        for (int t = 0; t < kMaxTail; ++t) {
            const int nc = t < a.levels ? a.n[t][0] * a.n[t][1] * a.n[t][2] : 0;
#pragma unroll
            for (int u = 0; u < kPer; ++u) {
                const int c = threadIdx.x + u * kTailThreads;
                cv[t][u] = c < nc ? a.code[t][c] : (uint16_t)0;
            }
        }
#pragma unroll
        for (int u = 0; u < kPer; ++u) {
            const int c = threadIdx.x + u * kTailThreads;
            if (c < n0) B[c] = bv[u];
        }
#pragma unroll
        for (int t = 0; t < kMaxTail; ++t) {
            const int nc = t < a.levels ? a.n[t][0] * a.n[t][1] * a.n[t][2] : 0;
#pragma unroll
            for (int u = 0; u < kPer; ++u) {
                const int c = threadIdx.x + u * kTailThreads;
                if (c < nc) Cd[a.off[t] + c] = cv[t][u];
            }
        }
    }
    __syncthreads();
    if (done) return;
    // per cell: the diagonal and the damped-Jacobi weight (the coarsest level
    // with its own damping)
    for (int t = 0; t < a.levels; ++t) {
        const TailLevel l = tail_level(a, t);
        const float omega = t == a.levels - 1 ? 1.0f : kMgCoarse.omega;  // the coarsest: 1/diagonal for Chebyshev
#pragma unroll
        for (int u = 0; u < kTailPer; ++u) {
            const int c = threadIdx.x + u * kTailThreads;
            if (c >= l.nc) break;
            const uint16_t cd = Cd[l.o + c];
            Dg[l.o + c] = code_center(cd, l.ih2);
            Wt[l.o + c] = mg_weight(cd, l.ih2, omega);
        }
    }
    __syncthreads();
    // down: the solution of every level ends in Tm after its pre-smoothing
    for (int t = 0; t < a.levels - 1; ++t) {
        const TailLevel l = tail_level(a, t), lc = tail_level(a, t + 1);
        const int o = l.o;
        const uint16_t* code = Cd + o;
        tail_sweep(l, code, Dg + o, Wt + o, nullptr, X + o, B + o);
        tail_sweep(l, code, Dg + o, Wt + o, X + o, Tm + o, B + o);
        // residual into X (free now)
        {
            const float* xs = Tm + o;
#pragma unroll
            for (int u = 0; u < kTailPer; ++u) {
                const int c = threadIdx.x + u * kTailThreads;
                if (c >= l.nc) break;
                const uint16_t cd = code[c];
                float rc = 0.0f;
                if (cd & kFluidBit)
                    rc = B[o + c] - code_apply(cd, Dg[o + c], c, l.st, l.ih2, xs[c],
                                               [&](int n) { return xs[n]; });
                X[o + c] = rc;
            }
            __syncthreads();
        }
        // restriction into the next level's B
        {
            const float* rs = X + o;
#pragma unroll
            for (int u = 0; u < kTailPer; ++u) {
                const int c = threadIdx.x + u * kTailThreads;
                if (c >= lc.nc) break;
                float v = 0.0f;
                if (Cd[lc.o + c] & kFluidBit) {
                    int I, J, K;
                    cell_ijk(c, lc.nx, lc.ny, I, J, K);
                    v = restrict_sum(I, J, K, l.nx, l.ny, l.nz, lc.nx, lc.ny, lc.nz,
                                     [&](int64_t n) { return rs[n]; });
                }
                B[lc.o + c] = v;
            }
            __syncthreads();
        }
    }
    // coarsest level: Chebyshev iteration from zero, ending in Tm (the
    // three-term recurrence with rho_k = 1 / (2 sigma - rho_(k-1)), rho_0 = 1 / sigma)
    {
        const TailLevel l = tail_level(a, a.levels - 1);
        const int o = l.o;
        const uint16_t* code = Cd + o;
        static_assert(kCoarseSweeps % 2 == 0, "the steps ping-pong X -> Tm");
        const float theta = 0.5f * (kChebHi + kChebLo), delta = 0.5f * (kChebHi - kChebLo);
        const float sigma = theta / delta;
        float rho = 1.0f / sigma;
        tail_cheb(l, code, Dg + o, Wt + o, nullptr, X + o, B + o, Dd, 0.0f, 1.0f / theta);
        for (int k = 1; k < kCoarseSweeps; ++k) {
            const float rn = 1.0f / (2.0f * sigma - rho);
            const float c1 = rn * rho, c2 = 2.0f * rn / delta;
            if (k & 1)
                tail_cheb(l, code, Dg + o, Wt + o, X + o, Tm + o, B + o, Dd, c1, c2);
            else
                tail_cheb(l, code, Dg + o, Wt + o, Tm + o, X + o, B + o, Dd, c1, c2);
            rho = rn;
        }
    }
    // up: prolongation, two sweeps Tm -> X -> Tm
    for (int t = a.levels - 2; t >= 0; --t) {
        const TailLevel l = tail_level(a, t), lc = tail_level(a, t + 1);
        const int o = l.o;
        const uint16_t* code = Cd + o;
        const float* xc = Tm + lc.o;
#pragma unroll
        for (int u = 0; u < kTailPer; ++u) {
            const int f = threadIdx.x + u * kTailThreads;
            if (f >= l.nc) break;
            if (!(code[f] & kFluidBit)) continue;
            int i, j, k;
            cell_ijk(f, l.nx, l.ny, i, j, k);
            Tm[o + f] += prolong_at(i, j, k, lc.nx, lc.ny, lc.nz, [&](int64_t n) { return xc[n]; });
        }
        __syncthreads();
        tail_sweep(l, code, Dg + o, Wt + o, Tm + o, X + o, B + o);
        tail_sweep(l, code, Dg + o, Wt + o, X + o, Tm + o, B + o);
    }
#pragma unroll
    for (int u = 0; u < kTailPer; ++u) {
        const int c = threadIdx.x + u * kTailThreads;
        if (c < n0) xT[c] = Tm[c];
    }
}

// ---------------------------------------------------------------------------
// The last two levels of the fused V-cycle in one workgroup: the descent into
// the coarsest level, its Chebyshev iteration, and the ascent.  Bound by the
// chain of phases between barriers (a level of 16^3 over one of 8^3: 16
// barriers); it replaces three launches (4.7 + 4.2 + 5.1 us and the gaps
// between them) with one of 10 us.
//
// A thread keeps up to four fine cells (right-hand side, diagonal, weight and
// place, in registers) and at most one coarse cell.  The iterates lie in LDS
// with a border of zeros, so the FLUID-row forms need neither codes nor
// clamps there: a cell's neighbours are at fixed offsets, and every cell that
// is not FLUID holds 0, as does the border.  The terms are the tiles' and the
// tail's, in their order but for the restriction's rows, which are added one
// after another as in the split kernels: the values agree to FP32 rounding.
// ---------------------------------------------------------------------------
constexpr int kBotThreads = 1024;
constexpr int kBotPer = 4;  // fine cells per thread: a coarsest level of 512 cells halves one of at most 4096
constexpr int kBotLds = 20000;  // floats of LDS at most (80 KB)
static_assert(kBotThreads * kBotPer >= 8 * kCoarseMax && kBotThreads >= kCoarseMax, "a place for every cell");

struct BottomArgs {
    int n[3], c[3];          // the fine and the coarsest level
    float ih2[3], cih2[3];
    int pf, pc;              // padded cells of each
};

// cell_ijk of a cell below 4096 without integer divisions: (c + 1/2) / n lies
// at least 1 / (2 n) from an integer, and its rounding error is below
// 4096 * 2^-22 / n.
__device__ inline void small_cell_ijk(int c, int nx, int ny, float rx, float ry, int& i, int& j, int& k) {
    const int q = (int)(((float)c + 0.5f) * rx);
    i = c - __mul24(q, nx);
    k = (int)(((float)q + 0.5f) * ry);
    j = q - __mul24(k, ny);
}

// Offset of cell (i, j, k) in an array of dims n with a border of one (24-bit
// products: a 32-bit one takes four times the issue time).
__device__ inline int bordered(int i, int j, int k, const int n[3]) {
    return (i + 1) + __mul24(n[0] + 2, (j + 1) + __mul24(n[1] + 2, k + 1));
}

__device__ inline void bordered_neighbours(const float* x, int p, int sy, int sz, float (&nb)[6]) {
    nb[0] = x[p - 1];
    nb[1] = x[p + 1];
    nb[2] = x[p - sy];
    nb[3] = x[p + sy];
    nb[4] = x[p - sz];
    nb[5] = x[p + sz];
}

__global__ __launch_bounds__(kBotThreads) void k_mg_bottom(BottomArgs a, const float* __restrict__ b,
                                                           const uint16_t* __restrict__ code,
                                                           const uint16_t* __restrict__ ccode,
                                                           float* __restrict__ out,
                                                           const SolverScalars* __restrict__ st) {
    extern __shared__ float lds[];
    float* X = lds;           // fine iterates
    float* Y = X + a.pf;
    float* U = Y + a.pf;      // coarse iterates
    float* V = U + a.pc;
    const int done = st->done;  // read with the data, tested before the first write
    const int nf = a.n[0] * a.n[1] * a.n[2], nc = a.c[0] * a.c[1] * a.c[2];
    float bf[kBotPer];
    uint32_t cd[kBotPer];
#pragma unroll
    for (int u = 0; u < kBotPer; ++u) {
        const int f = threadIdx.x + u * kBotThreads;
        bf[u] = f < nf ? b[f] : 0.0f;
        cd[u] = f < nf ? (uint32_t)code[f] : 0u;
    }
    const bool con = (int)threadIdx.x < nc;
    const uint32_t ccd = con ? (uint32_t)ccode[threadIdx.x] : 0u;
    for (int e = threadIdx.x; e < (2 * (a.pf + a.pc) + 3) / 4; e += kBotThreads)
        reinterpret_cast<float4*>(lds)[e] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    constexpr MgSmooth SM = kMgCoarse;
    const CodeLanes fl = code_lanes(a.ih2, SM.omega), cl = code_lanes(a.cih2, 1.0f);
    const float nih2[3] = {-a.ih2[0], -a.ih2[1], -a.ih2[2]}, cnih2[3] = {-a.cih2[0], -a.cih2[1], -a.cih2[2]};
    const int sy = a.n[0] + 2, sz = sy * (a.n[1] + 2), csy = a.c[0] + 2, csz = csy * (a.c[1] + 2);
    float cen[kBotPer], wgt[kBotPer];
    int p[kBotPer];
    const float rx = __builtin_amdgcn_rcpf((float)a.n[0]), ry = __builtin_amdgcn_rcpf((float)a.n[1]);
#pragma unroll
    for (int u = 0; u < kBotPer; ++u) {
        const int li = code_lane(cd[u]);
        cen[u] = lane_read(fl.cen, li);
        wgt[u] = lane_read(fl.wgt, li);
        int i, j, k;
        small_cell_ijk(threadIdx.x + u * kBotThreads, a.n[0], a.n[1], rx, ry, i, j, k);
        p[u] = bordered(i, j, k, a.n);
    }
    const int cli = code_lane(ccd);
    const float ccen = lane_read(cl.cen, cli), cw = lane_read(cl.wgt, cli);
    int I, J, K;
    small_cell_ijk(threadIdx.x, a.c[0], a.c[1], __builtin_amdgcn_rcpf((float)a.c[0]),
                   __builtin_amdgcn_rcpf((float)a.c[1]), I, J, K);
    const int cp = bordered(I, J, K, a.c);
    const bool cfl = (ccd & kFluidBit) != 0;  // false where there is no cell
    __syncthreads();
    if (done) return;  // uniform: the solve has stopped
    // x1, the first sweep from zero
#pragma unroll
    for (int u = 0; u < kBotPer; ++u)
        if (cd[u] & kFluidBit) X[p[u]] = wgt[u] * bf[u];
    __syncthreads();
    // x2, kept for the ascent
    float x2[kBotPer];
#pragma unroll
    for (int u = 0; u < kBotPer; ++u) {
        x2[u] = 0.0f;
        if (!(cd[u] & kFluidBit)) continue;
        float nb[6];
        bordered_neighbours(X, p[u], sy, sz, nb);
        const float x1 = X[p[u]];
        x2[u] = mg_cheb2(x1, 0.0f, SM.w21 * wgt[u], bf[u] - mg_apply_fluid_row(cen[u], x1, nb, nih2), SM.beta);
        Y[p[u]] = x2[u];
    }
    __syncthreads();
    // r = b - A x2 (over x1, which nothing reads any more)
#pragma unroll
    for (int u = 0; u < kBotPer; ++u) {
        if (!(cd[u] & kFluidBit)) continue;
        float nb[6];
        bordered_neighbours(Y, p[u], sy, sz, nb);
        X[p[u]] = bf[u] - mg_apply_fluid_row(cen[u], x2[u], nb, nih2);
    }
    __syncthreads();
    // the coarsest level: b = R r and kCoarseSweeps steps of Chebyshev
    // iteration from zero (the three-term recurrence of k_mg_tail)
    const float theta = 0.5f * (kChebHi + kChebLo), delta = 0.5f * (kChebHi - kChebLo);
    const float sigma = theta / delta;
    float rho = 1.0f / sigma;
    float bc = 0.0f, d = 0.0f, xc = 0.0f;
    if (cfl) {
        // the taps 2I-1 .. 2I+2 per axis at constant distances; where the last
        // lies beyond the border (odd dims) it has weight 0 and takes the one before
        int ix[4], iy[4], iz[4];
        float wx[4], wy[4], wz[4];
        restrict_taps(I, a.n[0], a.c[0], ix, wx);
        restrict_taps(J, a.n[1], a.c[1], iy, wy);
        restrict_taps(K, a.n[2], a.c[2], iz, wz);
        const float* row = X + bordered(2 * I - 1, 2 * J - 1, 2 * K - 1, a.n);
        const int lx = 2 * I + 2 > a.n[0] ? 2 : 3, ly = sy * (2 * J + 2 > a.n[1] ? 2 : 3),
                  lz = sz * (2 * K + 2 > a.n[2] ? 2 : 3);
        float acc = 0.0f;
#pragma unroll
        for (int tk = 0; tk < 4; ++tk) {
#pragma unroll
            for (int tj = 0; tj < 4; ++tj) {
                const float* q = row + (tk < 3 ? tk * sz : lz) + (tj < 3 ? tj * sy : ly);
                acc += (wy[tj] * wz[tk]) * restrict_row(wx, [&](int ti) { return q[ti < 3 ? ti : lx]; });
            }
        }
        bc = acc * 0.125f;
        d = (1.0f / theta) * (cw * bc);
        xc = d;
        U[cp] = xc;
    }
    __syncthreads();
    static_assert(kCoarseSweeps % 2 == 0, "the last step writes V");
    for (int q = 1; q < kCoarseSweeps; ++q) {
        const float rn = 1.0f / (2.0f * sigma - rho);
        const float c1 = rn * rho, c2 = 2.0f * rn / delta;
        const float* in = q & 1 ? U : V;
        float* to = q & 1 ? V : U;
        if (cfl) {
            float nb[6];
            bordered_neighbours(in, cp, csy, csz, nb);
            d = c1 * d + c2 * (cw * (bc - mg_apply_fluid_row(ccen, xc, nb, cnih2)));
            xc = xc + d;
            to[cp] = xc;
        }
        rho = rn;
        __syncthreads();
    }
    // the ascent: y = x2 + P xc, two steps
#pragma unroll
    for (int u = 0; u < kBotPer; ++u) {
        if (!(cd[u] & kFluidBit)) continue;
        // prolong_at3's terms from its lowest neighbour, the others one step on
        // (none where the axis clamps both to one cell)
        int i, j, k;
        small_cell_ijk(threadIdx.x + u * kBotThreads, a.n[0], a.n[1], rx, ry, i, j, k);
        const int A = (i - 1) >> 1, B = (j - 1) >> 1, C = (k - 1) >> 1;
        const float wa = i & 1 ? 0.75f : 0.25f, wb = j & 1 ? 0.75f : 0.25f, wc = k & 1 ? 0.75f : 0.25f;
        const float wa1 = 1.0f - wa, wb1 = 1.0f - wb, wc1 = 1.0f - wc;
        const float* q = V + bordered(max(A, 0), max(B, 0), max(C, 0), a.c);
        const int dx = A >= 0 && A + 1 < a.c[0] ? 1 : 0, dy = B >= 0 && B + 1 < a.c[1] ? csy : 0,
                  dz = C >= 0 && C + 1 < a.c[2] ? csz : 0;
        x2[u] = x2[u] + (wc * (wb * (wa * q[0] + wa1 * q[dx]) + wb1 * (wa * q[dy] + wa1 * q[dy + dx])) +
                         wc1 * (wb * (wa * q[dz] + wa1 * q[dz + dx]) + wb1 * (wa * q[dz + dy] + wa1 * q[dz + dy + dx])));
        Y[p[u]] = x2[u];
    }
    __syncthreads();
    float xp[kBotPer];
#pragma unroll
    for (int u = 0; u < kBotPer; ++u) {
        xp[u] = 0.0f;
        if (!(cd[u] & kFluidBit)) continue;
        float nb[6];
        bordered_neighbours(Y, p[u], sy, sz, nb);
        xp[u] = mg_sweep_fluid_row(cen[u], wgt[u], x2[u], bf[u], nb, nih2);
        X[p[u]] = xp[u];
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kBotPer; ++u) {
        const int f = threadIdx.x + u * kBotThreads;
        if (f >= nf) break;
        float o = 0.0f;
        if (cd[u] & kFluidBit) {
            float nb[6];
            bordered_neighbours(X, p[u], sy, sz, nb);
            o = mg_cheb2(xp[u], x2[u], SM.w21 * wgt[u], bf[u] - mg_apply_fluid_row(cen[u], xp[u], nb, nih2), SM.beta);
        }
        out[f] = o;
    }
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------
static inline dim3 grid1(int64_t n) { return dim3((unsigned)((n + kBlock - 1) / kBlock)); }

static LevelArgs level_args(const MGLevel& l) {
    const SolverShape sh = solver_shape_n(l.cells);
    LevelArgs a;
    a.nc = l.cells;
    a.st = stride_of(l.n[0], l.n[1], l.n[2]);
    for (int q = 0; q < 3; ++q) a.ih2[q] = l.ih2[q];
    a.chunk = sh.chunk;
    a.padded = sh.blocks;
    return a;
}

template <class T>
static FusedArgs fused_args(const MGLevel& l, const MGLevel& c) {
    FusedArgs a;
    for (int q = 0; q < 3; ++q) {
        a.n[q] = l.n[q];
        a.c[q] = c.n[q];
        a.ih2[q] = l.ih2[q];
    }
    a.tiles[0] = (c.n[0] + T::rx - 1) / T::rx;
    a.tiles[1] = (c.n[1] + T::ry - 1) / T::ry;
    a.tiles[2] = (c.n[2] + T::rz - 1) / T::rz;
    a.padded = pad_blocks((int64_t)a.tiles[0] * a.tiles[1] * a.tiles[2]);
    return a;
}

// Whether a level takes the small tiles: up to 1.5 of them per CU.  There the
// level's kernels are bound by the latency of a workgroup's chain of phases,
// and a small tile has 2.5x fewer cells per thread in each; above, by
// throughput, and the small tiles' halos cost more than they save.  Measured
// on whole solves to 1e-10, finest level on large tiles / small: 32^3 0.473 /
// 0.423 ms, 48^3 (216 small tiles) 0.549 / 0.500, 56^3 (343) 0.573 / 0.571,
// 64^3 (512) 0.680 / 0.695, 96^3 0.99 / 1.18, 128^3 1.51 / 1.90.
static bool small_tiles(const MGLevel& l) {
    constexpr int64_t kCus = 256;
    return 2 * l.cells <= 3 * kCus * TileSmall::coarse * 8;
}

static FusedArgs tile_args(const MGLevel& l, const MGLevel& c) {
    return small_tiles(l) ? fused_args<TileSmall>(l, c) : fused_args<TileLarge>(l, c);
}

void mg_free(fe_scene* s);

// First level of the tail: the first level below the finest with at most
// kTailMax cells whose tail fits the LDS arrays and the level table.
static int tail_start(const std::vector<MGLevel>& lv) {
    const int L = (int)lv.size();
    for (int q = 1; q < L; ++q) {
        int64_t sum = 0;
        for (int t = q; t < L; ++t) sum += lv[t].cells;
        if (lv[q].cells <= kTailMax && sum <= kTailLds && L - q <= kMaxTail) return q;
    }
    return L - 1;
}

static hipError_t mg_alloc(fe_scene* s) {
    const Geom& g = s->g;
    std::vector<MGLevel> lv;
    MGLevel l0;
    for (int a = 0; a < 3; ++a) {
        l0.n[a] = g.n[a];
        l0.ih2[a] = (float)(g.ihd[a] * g.ihd[a]);
    }
    l0.cells = cell_count(g);
    lv.push_back(l0);
    // every axis has at least 2 cells, so the first coarsening always shrinks
    while (lv.back().cells > kCoarseMax || lv.size() < 2) {
        const MGLevel& f = lv.back();
        MGLevel c;
        for (int a = 0; a < 3; ++a) {
            c.n[a] = (f.n[a] + 1) / 2;
            c.ih2[a] = f.ih2[a] * 0.25f;  // twice the spacing
        }
        c.cells = (int64_t)c.n[0] * c.n[1] * c.n[2];
        if (c.cells == f.cells) break;
        c.owns = true;
        lv.push_back(c);
    }
    if (lv.size() < 2 || lv.back().cells > kCoarseMax) return hipErrorInvalidValue;
    hipError_t e = hipSuccess;
    for (size_t q = 0; q < lv.size(); ++q) {
        MGLevel& l = lv[q];
        const size_t n = (size_t)l.cells;
        if (l.owns) {
            if ((e = hipMalloc((void**)&l.flags, n)) != hipSuccess) break;
            if ((e = hipMalloc((void**)&l.code, n * sizeof(uint16_t))) != hipSuccess) break;
            if ((e = hipMalloc((void**)&l.b, n * sizeof(float))) != hipSuccess) break;
        }
        if ((e = hipMalloc((void**)&l.x, n * sizeof(float))) != hipSuccess) break;
        if ((e = hipMalloc((void**)&l.x2, n * sizeof(float))) != hipSuccess) break;
        if ((e = hipMalloc((void**)&l.r, n * sizeof(float))) != hipSuccess) break;
    }
    // the fused V-cycle's level-0 tile flags and r.z partials
    const FusedArgs fa = tile_args(lv[0], lv[1]);
    s->mg_npz = fa.padded;
    if (e == hipSuccess) e = hipMalloc((void**)&s->mg_tfl, (size_t)fa.padded);
    if (e == hipSuccess) e = hipMalloc((void**)&s->mg_pz, sizeof(double) * (size_t)fa.padded);
    s->mg = lv;
    s->mg_tail = tail_start(lv);
    if (e != hipSuccess) mg_free(s);  // leaves the hierarchy empty: the next solve retries
    return e;
}

void mg_free(fe_scene* s) {
    for (MGLevel& l : s->mg) {
        if (l.owns) {
            (void)hipFree(l.flags);
            (void)hipFree(l.code);
            (void)hipFree(l.b);
        }
        (void)hipFree(l.x);
        (void)hipFree(l.x2);
        (void)hipFree(l.r);
    }
    s->mg.clear();
    (void)hipFree(s->mg_tfl);
    (void)hipFree(s->mg_pz);
    s->mg_tfl = nullptr;
    s->mg_pz = nullptr;
    s->mg_npz = 0;
}

// Per solve: coarse markers and row codes from the current level-0 markers
// (the level-0 codes come from k_build_system).
hipError_t mg_setup(fe_scene* s) {
    hipError_t e;
    if (s->mg.empty() && (e = mg_alloc(s)) != hipSuccess) return e;
    std::vector<MGLevel>& lv = s->mg;
    lv[0].flags = s->flags;
    lv[0].code = s->code;
    const int L = (int)lv.size();
    // markers of levels 1 .. m and the finest tiles' flags in one launch,
    // deeper levels (grids above 128^3) one launch each
    const int m = std::min(L - 1, kPyr);
    PyrArgs pa{};
    pa.levels = m;
    for (int q = 0; q <= m; ++q) {
        for (int a = 0; a < 3; ++a) pa.n[q][a] = lv[q].n[a];
        pa.flags[q] = lv[q].flags;
    }
    if (s->tune.mg == FE_MG_FUSED) {
        const FusedArgs fa = tile_args(lv[0], lv[1]);
        pa.tfl = s->mg_tfl;
        for (int a = 0; a < 3; ++a) pa.tiles[a] = fa.tiles[a];
        const bool small = small_tiles(lv[0]);
        pa.rx = small ? TileSmall::rx : TileLarge::rx;
        pa.ry = small ? TileSmall::ry : TileLarge::ry;
        pa.rz = small ? TileSmall::rz : TileLarge::rz;
    }
    const unsigned nb = (unsigned)(((lv[1].n[0] + 7) / 8) * ((lv[1].n[1] + 7) / 8) * ((lv[1].n[2] + 7) / 8));
    hipLaunchKernelGGL(k_mg_pyramid, dim3(nb), dim3(kPyrThreads), 0, s->stream, pa);
    for (int q = m + 1; q < L; ++q) {
        const MGLevel& f = lv[q - 1];
        MGLevel& c = lv[q];
        hipLaunchKernelGGL(k_mg_coarsen, grid1(c.cells), dim3(kBlock), 0, s->stream, (const uint8_t*)f.flags, f.n[0],
                           f.n[1], f.n[2], c.flags, c.n[0], c.n[1], c.n[2]);
    }
    // row codes of every coarse level in one launch
    if (L - 1 <= kMaxLevels) {
        CodesArgs ca{};
        ca.levels = L - 1;
        ca.off[0] = 0;
        for (int q = 1; q < L; ++q) {
            for (int a = 0; a < 3; ++a) ca.n[q - 1][a] = lv[q].n[a];
            ca.flags[q - 1] = lv[q].flags;
            ca.code[q - 1] = lv[q].code;
            ca.off[q] = ca.off[q - 1] + lv[q].cells;
        }
        hipLaunchKernelGGL(k_mg_codes_all, grid1(ca.off[L - 1]), dim3(kBlock), 0, s->stream, ca);
    } else {
        for (int q = 1; q < L; ++q)
            hipLaunchKernelGGL(k_mg_codes, grid1(lv[q].cells), dim3(kBlock), 0, s->stream, (const uint8_t*)lv[q].flags,
                               lv[q].n[0], lv[q].n[1], lv[q].n[2], lv[q].code);
    }
    return hipGetLastError();
}

float* mg_first_sweep_target(fe_scene* s) { return s->mg.empty() ? nullptr : s->mg[0].x; }

// The one-workgroup tail of a V-cycle (z = M^-1 r, mg_apply below).  Once `st`
// says the solve has stopped, every multigrid kernel still issues its first
// loads (the stop flag is read together with them) and then returns before its
// first write, except the finest-level descent, which tests the flag before
// its loads; the CG spmv and update issue their first group of cells' loads
// and the partial-sum loads before testing it.
static void launch_tail(fe_scene* s, SolverScalars* st) {
    std::vector<MGLevel>& lv = s->mg;
    const int L = (int)lv.size();
    const int T = s->mg_tail;
    TailArgs ta{};
    ta.levels = L - T;
    int off = 0;
    for (int t = 0; t < ta.levels; ++t) {
        const MGLevel& l = lv[T + t];
        for (int q = 0; q < 3; ++q) {
            ta.n[t][q] = l.n[q];
            ta.ih2[t][q] = l.ih2[q];
        }
        ta.code[t] = l.code;
        ta.off[t] = off;
        off += (int)l.cells;
    }
    hipLaunchKernelGGL(k_mg_tail, dim3(1), dim3(kTailThreads), 0, s->stream, ta, (const float*)lv[T].b, lv[T].x2, st);
}

// Level q and the coarsest one below it, for k_mg_bottom.
static BottomArgs bottom_args(const MGLevel& l, const MGLevel& c) {
    BottomArgs a;
    a.pf = a.pc = 1;
    for (int q = 0; q < 3; ++q) {
        a.n[q] = l.n[q];
        a.c[q] = c.n[q];
        a.ih2[q] = l.ih2[q];
        a.cih2[q] = c.ih2[q];
        a.pf *= l.n[q] + 2;
        a.pc *= c.n[q] + 2;
    }
    return a;
}

// The fused V-cycle: level q's descent writes its pre-smoothed x2 and level
// q+1's right-hand side; the tail leaves level T's result in lv[T].x2; level
// q's ascent reads x2 and the coarse result and writes its own result to x
// (level 0: z).  x is never read before the ascent writes it, so no level
// holds a first sweep in memory.
static hipError_t mg_apply_fused(fe_scene* s, const float* r, float* z, SolverScalars* st, double* prz, int tag,
                                 const double* pconf, int nparts) {
    std::vector<MGLevel>& lv = s->mg;
    const int T = s->mg_tail;
    lv[0].b = const_cast<float*>(r);
    auto down = [&](int q) {
        const MGLevel& l = lv[q];
        const MGLevel& c = lv[q + 1];
        const FusedArgs a = tile_args(l, c);
        const bool sm = small_tiles(l);
        const dim3 grid((unsigned)a.padded);
        if (q == 0)
            launch_timed(s, FE_KERNEL_MG_DOWN, tag, sm ? k_mg_down<true, TileSmall> : k_mg_down<true, TileLarge>, grid,
                         dim3(kFusedThreads), a, (const float*)l.b, (const uint16_t*)l.code, l.x2,
                         (const uint16_t*)c.code, c.b, (const SolverScalars*)st, pconf, nparts,
                         (const uint8_t*)s->mg_tfl);
        else
            hipLaunchKernelGGL((sm ? k_mg_down<false, TileSmall> : k_mg_down<false, TileLarge>), grid,
                               dim3(kFusedThreads), 0, s->stream, a, (const float*)l.b, (const uint16_t*)l.code, l.x2,
                               (const uint16_t*)c.code, c.b, (const SolverScalars*)st, (const double*)nullptr, 0,
                               (const uint8_t*)nullptr);
    };
    auto up = [&](int q) {
        const MGLevel& l = lv[q];
        const MGLevel& c = lv[q + 1];
        const FusedArgs a = tile_args(l, c);
        const bool sm = small_tiles(l);
        const dim3 grid((unsigned)a.padded);
        const dim3 threads((unsigned)(sm ? FCols<TileSmall, 2>::threads : FCols<TileLarge, 2>::threads));
        const float* xc = q + 1 == T ? c.x2 : c.x;
        if (q == 0)
            launch_timed(s, FE_KERNEL_MG_UP, tag, sm ? k_mg_up<true, TileSmall> : k_mg_up<true, TileLarge>, grid,
                         threads, a, (const float*)l.x2, xc, (const float*)l.b, (const uint16_t*)l.code, z, prz,
                         (const SolverScalars*)st, (const uint8_t*)s->mg_tfl);
        else
            hipLaunchKernelGGL((sm ? k_mg_up<false, TileSmall> : k_mg_up<false, TileLarge>), grid, threads, 0,
                               s->stream, a, (const float*)l.x2, xc, (const float*)l.b, (const uint16_t*)l.code, l.x,
                               (double*)nullptr, (const SolverScalars*)st, (const uint8_t*)nullptr);
    };
    down(0);
    // the last level above the coarsest goes with it into one workgroup, where
    // their iterates fit its LDS (all but very long grids)
    BottomArgs ba{};
    const bool bottom = T >= 2 && T + 1 == (int)lv.size() &&
                        2 * ((ba = bottom_args(lv[T - 1], lv[T])).pf + ba.pc) <= kBotLds;
    const int B = bottom ? T - 1 : T;
    for (int q = 1; q < B; ++q) down(q);
    if (bottom)
        hipLaunchKernelGGL(k_mg_bottom, dim3(1), dim3(kBotThreads), sizeof(float) * (2 * (ba.pf + ba.pc) + 3), s->stream, ba,
                           (const float*)lv[B].b, (const uint16_t*)lv[B].code, (const uint16_t*)lv[T].code, lv[B].x,
                           (const SolverScalars*)st);
    else
        launch_tail(s, st);
    for (int q = B - 1; q >= 0; --q) up(q);
    return hipGetLastError();
}

// z = M^-1 r with one V-cycle, leaving partials of r.z in prz.  With the split
// kernels the caller has already written level 0's first sweep (x1 = w r)
// into mg[0].x; the fused descent sweeps from r itself.
hipError_t mg_apply(fe_scene* s, const float* r, float* z, SolverScalars* st, double* prz, int tag,
                    const double* pconf, int nparts) {
    if (s->tune.mg == FE_MG_FUSED) return mg_apply_fused(s, r, z, st, prz, tag, pconf, nparts);
    std::vector<MGLevel>& lv = s->mg;
    const int T = s->mg_tail;
    lv[0].b = const_cast<float*>(r);
    const uint8_t* cfl0 = s->chunk_fluid;
    for (int q = 0; q < T; ++q) {
        MGLevel& l = lv[q];
        MGLevel& c = lv[q + 1];
        const LevelArgs a = level_args(l);
        const dim3 grid((unsigned)a.padded);
        if (q == 0)
            launch_timed(s, FE_KERNEL_MG_SMOOTH, tag, k_mg_smooth, grid, dim3(kBlock), a, (const uint16_t*)l.code,
                         (const float*)l.b, (const float*)l.x, l.x2, st, (double*)nullptr, pconf, nparts, cfl0, 1,
                         (const float*)nullptr, 1);
        else
            hipLaunchKernelGGL(k_mg_smooth, grid, dim3(kBlock), 0, s->stream, a, (const uint16_t*)l.code,
                               (const float*)l.b, (const float*)l.x, l.x2, (const SolverScalars*)st, (double*)nullptr,
                               (const double*)nullptr, 0, (const uint8_t*)nullptr, 1, (const float*)nullptr, 0);
        hipLaunchKernelGGL(k_mg_residual, grid, dim3(kBlock), 0, s->stream, a, (const uint16_t*)l.code,
                           (const float*)l.b, (const float*)l.x2, l.r, st, q == 0 ? cfl0 : (const uint8_t*)nullptr);
        const dim3 rgrid((unsigned)((c.n[0] + kRtx - 1) / kRtx), (unsigned)((c.n[1] + kRty - 1) / kRty),
                         (unsigned)((c.n[2] + kRtz - 1) / kRtz));
        hipLaunchKernelGGL(k_mg_restrict, rgrid, dim3(kBlock), 0, s->stream, (const float*)l.r, l.n[0],
                           l.n[1], l.n[2], (const uint16_t*)c.code, c.b, q + 1 < T ? c.x : (float*)nullptr, c.n[0],
                           c.n[1], c.n[2], c.ih2[0], c.ih2[1], c.ih2[2], st);
    }
    launch_tail(s, st);
    for (int q = T - 1; q >= 0; --q) {
        MGLevel& l = lv[q];
        const MGLevel& c = lv[q + 1];
        const LevelArgs a = level_args(l);
        const dim3 grid((unsigned)a.padded);
        hipLaunchKernelGGL(k_mg_prolong, grid1(l.cells), dim3(kBlock), 0, s->stream, (const float*)c.x2, c.n[0],
                           c.n[1], c.n[2], (const uint16_t*)l.code, l.x2, l.n[0], l.n[1], l.n[2], st);
        if (q == 0) {
            launch_timed(s, FE_KERNEL_MG_SMOOTH, tag, k_mg_smooth, grid, dim3(kBlock), a, (const uint16_t*)l.code,
                         (const float*)l.b, (const float*)l.x2, l.x, st, (double*)nullptr, (const double*)nullptr, 0,
                         cfl0, 0, (const float*)nullptr, 1);
            launch_timed(s, FE_KERNEL_MG_SMOOTH, tag, k_mg_smooth, grid, dim3(kBlock), a, (const uint16_t*)l.code,
                         (const float*)l.b, (const float*)l.x, z, st, prz, (const double*)nullptr, 0, cfl0, 1,
                         (const float*)l.x2, 1);
        } else {
            hipLaunchKernelGGL(k_mg_smooth, grid, dim3(kBlock), 0, s->stream, a, (const uint16_t*)l.code,
                               (const float*)l.b, (const float*)l.x2, l.x, st, (double*)nullptr, (const double*)nullptr, 0,
                               (const uint8_t*)nullptr, 0, (const float*)nullptr, 0);
            hipLaunchKernelGGL(k_mg_smooth, grid, dim3(kBlock), 0, s->stream, a, (const uint16_t*)l.code,
                               (const float*)l.b, (const float*)l.x, l.x2, st, (double*)nullptr, (const double*)nullptr, 0,
                               (const uint8_t*)nullptr, 1, (const float*)l.x2, 0);
        }
    }
    return hipGetLastError();
}

}  // namespace fe
