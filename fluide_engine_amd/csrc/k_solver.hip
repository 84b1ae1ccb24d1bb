// k_solver.hip -- pressure projection of SinglePhasePressureSolver
// (src/fluid_solvers/single_phase_pressure_solver.cpp) on gfx950.
//
// The reference stores A as {center,right,up,front} doubles per cell
// (src/linear_system/linear_system.hpp:9-15, 32 B/cell).  Here BuildSystem's
// rules (:99-164) -- center = sum of 1/h^2 over in-range, non-BOUNDRY
// neighbours; off-diagonal -1/h^2 between two FLUID cells; non-FLUID rows are
// the identity -- are packed once per solve into a 16-bit code per cell
// (which neighbours are coupled, how many neighbours count per axis), so the
// iteration kernels read 2 B/cell of matrix and never divide an index.
// r, z, d, q are FP32, the solution is FP64, and every dot product and norm
// accumulates in FP64.
//
// Reductions: each kernel runs at most 1024 blocks over contiguous cell chunks
// and leaves one FP64 partial per block and value.  The next kernel's blocks
// each sum those partials in the same fixed order, so all blocks derive
// bit-identical scalars with no atomics and no inter-block fences (the kernel
// boundary orders the writes); block 0 records the solver state.
#include <algorithm>
#include <type_traits>
#include <utility>

#include "fe_stencil.hpp"

namespace fe {



// ---------------------------------------------------------------------------
// BuildSystem (single_phase_pressure_solver.cpp:99-164): the row codes and the
// right-hand side b = DivergenceAtCallCenter (face_centered_grid3d.cpp:157-166)
// on FLUID cells, 0 elsewhere; partials of b.b.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void k_build_system(Geom g, FaceSet u, const uint8_t* __restrict__ flags,
                                                         uint16_t* __restrict__ code, float* __restrict__ b,
                                                         double* __restrict__ pout, uint8_t* __restrict__ cfl,
                                                         int64_t chunk, int64_t padded, SolverScalars* __restrict__ sc,
                                                         SolverScalars init) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *sc = init;  // the solver's start state (read by the later kernels)
    const int64_t nc = cell_count(g);
    const Span sp = block_span(nc, chunk, padded);
    const uint32_t nx = (uint32_t)g.n[0], ny = (uint32_t)g.n[1], nz = (uint32_t)g.n[2];
    const int64_t sy = nx, sz = (int64_t)nx * ny;
    double v[1] = {0.0};
    int fluid = 0;
    // Groups of G cells: their flags loaded together, then every FLUID cell's
    // neighbour flags and faces together (two dependent load rounds per group
    // instead of per cell); the cells are then written in order.
    const FaceSet fs = u;
    constexpr int G = 4;
    for (int64_t c0 = sp.c0 + threadIdx.x; c0 < sp.c1; c0 += (int64_t)G * kBlock) {
        uint8_t fc[G];
#pragma unroll
        for (int u = 0; u < G; ++u) {
            const int64_t c = c0 + (int64_t)u * kBlock;
            fc[u] = c < sp.c1 ? flags[c] : (uint8_t)FE_AIR;
        }
        uint8_t fn[G][6];
        float fv[G][6];
#pragma unroll
        for (int u = 0; u < G; ++u) {
            const int64_t c = c0 + (int64_t)u * kBlock;
#pragma unroll
            for (int q = 0; q < 6; ++q) {
                fn[u][q] = (uint8_t)FE_BOUNDRY;
                fv[u][q] = 0.0f;
            }
            if (fc[u] != FE_FLUID) continue;
            const uint32_t cu = (uint32_t)c;  // grids hold fewer than 2^30 cells
            const uint32_t i = cu % nx, j = (cu / nx) % ny, k = cu / (nx * ny);
            const bool in[6] = {i > 0, i + 1 < nx, j > 0, j + 1 < ny, k > 0, k + 1 < nz};
            const int64_t nb[6] = {c - 1, c + 1, c - sy, c + sy, c - sz, c + sz};
#pragma unroll
            for (int q = 0; q < 6; ++q)
                if (in[q]) fn[u][q] = flags[nb[q]];
            const int64_t iu = (int64_t)i + (int64_t)(nx + 1) * ((int64_t)j + (int64_t)ny * k);
            const int64_t iv = (int64_t)i + (int64_t)nx * ((int64_t)j + (int64_t)(ny + 1) * k);
            fv[u][0] = fs.a[0][iu];
            fv[u][1] = fs.a[0][iu + 1];
            fv[u][2] = fs.a[1][iv];
            fv[u][3] = fs.a[1][iv + nx];
            fv[u][4] = fs.a[2][c];
            fv[u][5] = fs.a[2][c + sz];
        }
#pragma unroll
        for (int u = 0; u < G; ++u) {
            const int64_t c = c0 + (int64_t)u * kBlock;
            if (c >= sp.c1) break;
            float bb = 0.0f;
            uint16_t cd = 0;
            if (fc[u] == FE_FLUID) {
                cd = kFluidBit;
                fluid = 1;
#pragma unroll
                for (int q = 0; q < 6; ++q) {
                    const uint8_t f = fn[u][q];  // FE_BOUNDRY outside the grid
                    if (f == FE_BOUNDRY) continue;
                    cd = (uint16_t)(cd + (1u << (6 + 2 * (q >> 1))));
                    if (f == FE_FLUID) cd |= (uint16_t)(1u << q);
                }
                bb = (fv[u][1] - fv[u][0]) / g.h[0] + (fv[u][3] - fv[u][2]) / g.h[1] + (fv[u][5] - fv[u][4]) / g.h[2];
            }
            code[c] = cd;
            b[c] = bb;
            v[0] += (double)bb * (double)bb;
        }
    }
    // chunks without FLUID cells hold zeros in every CG and level-0 multigrid
    // vector throughout the solve, so those kernels skip them
    fluid = __syncthreads_or(fluid);
    if (threadIdx.x == 0) cfl[sp.lb] = (uint8_t)(fluid != 0);
    write_partials<1>(v, pout);
}

// ---------------------------------------------------------------------------
// Jacobi sweep (JacobiIterationSolver::Relax, src/linear_system/jacobi_iteration_solver.cpp:39-76):
// x' = (b - sum_offdiag A x) / center, on FP32 working copies of the FP64
// pressure.  When a residual check ran before this sweep its partials are
// summed first (CalculateTolerance, :78-82: ||b - A x||_2 < tol stops the
// solve); after the stop every sweep only copies, so the buffer rotation stays
// consistent.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void k_jacobi(Geom g, const uint16_t* __restrict__ code,
                                                   const float* __restrict__ b, const float* __restrict__ xo,
                                                   float* __restrict__ xn, SolverScalars* sc,
                                                   const double* __restrict__ pcheck, int nparts, int check_it,
                                                   float ihx2, float ihy2, float ihz2, int64_t chunk,
                                                   int64_t padded) {
    // block 0 may set sc->done during this kernel: read it once per block so
    // every thread takes the same path through the barriers below
    __shared__ int sdone;
    if (threadIdx.x == 0) sdone = sc->done;
    __syncthreads();
    bool done = sdone != 0;
    if (pcheck && !done) {
        double t[1];
        sum_partials<1>(pcheck, nparts, t);
        if (sqrt(t[0]) < sc->tol) {
            done = true;
            if (blockIdx.x == 0 && threadIdx.x == 0) {
                sc->done = 1;
                sc->converged = 1;
                sc->it = check_it + 1;
            }
        }
    }
    const int64_t nc = cell_count(g);
    const Span sp = block_span(nc, chunk, padded);
    const float ih2[3] = {ihx2, ihy2, ihz2};
    const Stride st = stride_of(g.n[0], g.n[1], g.n[2]);
    auto X = [&](int64_t n) { return xo[n]; };
    for (int64_t c = sp.c0 + threadIdx.x; c < sp.c1; c += kBlock) {
        if (done) {
            xn[c] = xo[c];
            continue;
        }
        const uint16_t cd = code[c];
        const float center = code_center(cd, ih2);
        // off-diagonal sum in the reference order (i-1, i+1, j-1, j+1, k-1, k+1)
        const float off = code_apply(cd, 0.0f, c, st, ih2, 0.0f, X);
        xn[c] = (b[c] - off) / center;
    }
}

// Partials of ||b - A x||^2 for the Jacobi convergence check (FP64 sums).
__global__ __launch_bounds__(kBlock) void k_jacobi_residual(Geom g, const uint16_t* __restrict__ code,
                                                            const float* __restrict__ b,
                                                            const float* __restrict__ x, const SolverScalars* sc,
                                                            double* __restrict__ pout, float ihx2, float ihy2,
                                                            float ihz2, int64_t chunk, int64_t padded) {
    const int64_t nc = cell_count(g);
    const Span sp = block_span(nc, chunk, padded);
    const double ih2d[3] = {ihx2, ihy2, ihz2};
    const Stride st = stride_of(g.n[0], g.n[1], g.n[2]);
    double v[1] = {0.0};
    if (!sc->done) {
        for (int64_t c = sp.c0 + threadIdx.x; c < sp.c1; c += kBlock) {
            const double ax = code_apply64(code[c], c, st, ih2d, (double)x[c], [&](int64_t n) { return (double)x[n]; });
            const double res = (double)b[c] - ax;
            v[0] += res * res;
        }
    }
    write_partials<1>(v, pout);
}

__global__ __launch_bounds__(kBlock) void k_f64_to_f32(const double* __restrict__ a, float* __restrict__ o,
                                                       int64_t n) {
    const int64_t c = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (c < n) o[c] = (float)a[c];
}

__global__ __launch_bounds__(kBlock) void k_f32_to_f64(const float* __restrict__ a, double* __restrict__ o,
                                                       int64_t n) {
    const int64_t c = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (c < n) o[c] = (double)a[c];
}

__global__ __launch_bounds__(kBlock) void k_zero_f64(double* __restrict__ x, int64_t n) {
    const int64_t c = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (c < n) x[c] = 0.0;
}

// What a residual b - A x on the FP64 solution reads for cell c.
struct Stencil64In {
    uint16_t cd;
    float bc;
    double xc, nb[6];
};

__device__ inline Stencil64In stencil64_in(int64_t c, const uint16_t* __restrict__ code,
                                           const double* __restrict__ x, const float* __restrict__ b,
                                           const Stride& st) {
    Stencil64In t;
    t.cd = code[c];
    t.bc = b[c];
    t.xc = x[c];
    code_neighbours(c, st, [&](int64_t n) { return x[n]; }, t.nb);
    return t;
}

// ---------------------------------------------------------------------------
// Conjugate gradient (ConjugateGradientSolver::Solve, src/linear_system/conjugate_gradient_solver.cpp:14-55).
// With the multigrid preconditioner, two kernels and a V-cycle per iteration:
//   spmv:   [prologue: sigma' = r.z, r.r of the last update -> beta, trigger,
//           stopping rule, next replacement flag]  d = z + beta*d_old (also at
//           the 6 neighbours, on the fly), q = A d, partials of d.q
//   update: [prologue: alpha = sigma / d.q]  x' = alpha*d + x (FP64);
//           r = -alpha*q + r, or r = b - A x' in FP64 on residual replacement
//           (every 50 iterations or after sigma grew, :32-49; x' at the
//           neighbours is formed on the fly from x and d); partials of r.r
// Without it one kernel per iteration, k_cg_step below.
// With the relative rule a stop is only accepted on a freshly replaced
// residual, so the decision is taken on b - A x, not on the recurrence (with
// the multigrid preconditioner the next V-cycle's first kernel tests the
// replaced residual, so a confirmed stop costs no V-cycle and no spmv).
// The FP32 recurrence drifts from b - A x by about eps32 * ||A|| * sum|alpha d|,
// which grows with the residual at the last recomputation: the residual is
// also recomputed whenever ||r|| has fallen 100x below that value ("reliable
// updates", Sleijpen and van der Vorst 1996), so the drift stays well below
// ||r|| and beta stays meaningful across recomputations.
// ---------------------------------------------------------------------------
constexpr double kReliableDrop2 = 1e-4;  // (100x in ||r||)^2
// Sums per block without multigrid: r.r, d.q, q.M^-1 q, q.z and, where z is not
// r itself, r.z.
constexpr int cg_sums(bool diag) { return diag ? 5 : 4; }
__global__ __launch_bounds__(kBlock) void k_cg_init(Geom g, const uint16_t* __restrict__ code,
                                                    const float* __restrict__ b, double* __restrict__ x,
                                                    float* __restrict__ r, float* __restrict__ d0, float* __restrict__ mgx, SolverScalars* sc,
                                                    const double* __restrict__ pbb, double* __restrict__ pout,
                                                    int stride, int nparts, float ihx2, float ihy2, float ihz2,
                                                    int64_t chunk, int64_t padded) {
    const int64_t nc = cell_count(g);
    const Span sp = block_span(nc, chunk, padded);
    const Stride st = stride_of(g.n[0], g.n[1], g.n[2]);
    // the thread's first group of cells loaded before the partial sum is
    // waited for (it does not depend on it)
    constexpr int G = 4;
    const int64_t g0 = sp.c0 + threadIdx.x;
    const bool early = g0 + (int64_t)(G - 1) * kBlock < sp.c1;
    Stencil64In raw[G];
    if (early) {
#pragma unroll
        for (int u = 0; u < G; ++u) raw[u] = stencil64_in(g0 + (int64_t)u * kBlock, code, x, b, st);
    }
    double bb[1];
    sum_partials<1>(pbb, nparts, bb);
    if (blockIdx.x == 0 && threadIdx.x == 0) sc->bnorm2 = bb[0];
    const float ih2[3] = {ihx2, ihy2, ihz2};
    const double ih2d[3] = {ihx2, ihy2, ihz2};
    const int pre = sc->precond;  // 0 none, 1 diagonal, 2 multigrid (z and r.z come later)
    double v[2] = {0.0, 0.0};
    auto use = [&](int64_t c, const Stencil64In& t) {
        // the identity rows of non-FLUID cells have the solution 0: the
        // start takes it there (FLUID rows couple only to FLUID cells), so
        // r is 0 outside FLUID from the start and stays so
        const bool fl = (t.cd & kFluidBit) != 0;
        if (!fl && t.xc != 0.0) x[c] = 0.0;  // written only where it is not 0 already
        const float rc = fl ? (float)((double)t.bc - code_apply64_nb(t.cd, ih2d, t.xc, t.nb)) : 0.0f;
        r[c] = rc;
        const float zc = pre == 1 ? rc / code_center(t.cd, ih2) : rc;
        if (mgx) mgx[c] = mg_weight(t.cd, ih2) * rc;  // the V-cycle's first sweep from zero
        d0[c] = 0.0f;
        if (pre != 2) v[0] += (double)rc * (double)zc;
        v[1] += (double)rc * (double)rc;
    };
    if (early) {
#pragma unroll
        for (int u = 0; u < G; ++u) use(g0 + (int64_t)u * kBlock, raw[u]);
    }
    span_groups_from<G, Stencil64In>(
        early ? g0 + (int64_t)G * kBlock : g0, sp.c1, [&](int64_t c) { return stencil64_in(c, code, x, b, st); },
        use);
    if (stride == 2) {
        write_partials<2>(v, pout);
    } else if (stride == cg_sums(false)) {
        const double w[1] = {v[1]};
        write_partials<1, cg_sums(false)>(w, pout);
    } else {
        const double w[cg_sums(true)] = {v[1], 0.0, 0.0, 0.0, v[0]};
        write_partials<cg_sums(true)>(w, pout);
    }
}

// The CG kernels' prologue: every block derives the iteration's scalars from the
// last kernels' partials, alike.  The loads of the partials, of the state and
// of the thread's first group of cells go out together; the first wavefront
// alone adds up and decides (some hundred FP64 instructions with the quotients
// and roots, which all waves of a SIMD would otherwise issue in turn), and
// hands the plan to the others through LDS.
//
// G: cells per thread of a group, kBlock apart.  A chunk of 256 cells (grids up
// to 2^18) is one group of 1, larger chunks take groups of 4; a thread with
// fewer cells reads its chunk's last one again.
template <typename F>
inline void with_group(const SolverShape& sh, F f) {
    if (sh.chunk <= kBlock)
        f(std::integral_constant<int, 1>{});
    else
        f(std::integral_constant<int, 4>{});
}

// State slots alternate with the iteration (spmv k reads slot k&1 and writes
// slot (k+1)&1), so no block can see a half-updated state.
template <int G>
__global__ __launch_bounds__(kBlock) void k_cg_spmv(Geom g, const uint16_t* __restrict__ code,
                                                    const float* __restrict__ z, const float* __restrict__ dold,
                                                    float* __restrict__ dnew, float* __restrict__ q,
                                                    const SolverScalars* __restrict__ in,
                                                    SolverScalars* __restrict__ out, const double* __restrict__ pin,
                                                    const double* __restrict__ pz, int nz, double* __restrict__ pout,
                                                    int nparts, float ihx2, float ihy2, float ihz2,
                                                    const uint8_t* __restrict__ cfl, int64_t chunk, int64_t padded) {
    const int64_t nc = cell_count(g);
    const Span sp = block_span(nc, chunk, padded);
    const Stride st = stride_of(g.n[0], g.n[1], g.n[2]);
    const bool body = sp.c0 < sp.c1 && cfl[sp.lb] != 0;
    struct Raw {
        uint16_t cd;
        float zc, dc, zn[6], dn[6];
    };
    auto fetch = [&](int64_t c) {
        Raw w;
        w.cd = code[c];
        w.zc = z[c];
        w.dc = dold[c];
        code_neighbours(c, st, [&](int64_t n) { return z[n]; }, w.zn);
        code_neighbours(c, st, [&](int64_t n) { return dold[n]; }, w.dn);
        return w;
    };
    const int64_t g0 = sp.c0 + threadIdx.x;
    Raw raw[G];
    if (body) {
#pragma unroll
        for (int u = 0; u < G; ++u) raw[u] = fetch(min(g0 + (int64_t)u * kBlock, sp.c1 - 1));
    }
    // r.z of the V-cycle's last sweep and r.r of the last update
    __shared__ double sm[2][kBlock / 64];
    __shared__ double plan_beta;
    __shared__ int plan_done;
    {
        double tz[1] = {0.0}, tr[1] = {0.0};
        add_partials<1>(pz, 1, 0, (int)threadIdx.x, kBlock, nz, tz);
        add_partials<1>(pin, 2, 1, (int)threadIdx.x, kBlock, nparts, tr);
        const double t[2] = {tz[0], tr[0]};
        wave_sums(t, sm);
    }
    __syncthreads();
    if (threadIdx.x < 64) {
        SolverScalars o = *in;
        if (!o.done) {  // else: an earlier spmv stopped the solve
            const double sigma = waves_total(sm[0]), rr = waves_total(sm[1]), sold = o.sigma;
            const bool replaced = o.replace != 0;
            o.sigma_old = sold;
            o.sigma = sigma;
            o.rr = rr;
            o.confirm = 0;
            if (o.it < 0) {  // first iteration: partials come from k_cg_init
                o.it = 0;
                o.beta = 0.0;
                o.trigger = 0;
                o.rr_ref = rr;
                o.converged = stop_rule(in, o.bnorm2, sigma, rr) ? 1 : 0;
                o.done = (o.converged || o.max_it <= 0) ? 1 : 0;
            } else {
                if (replaced) o.rr_ref = rr;
                ++o.it;
                o.trigger = sigma > sold ? 1 : 0;
                o.beta = sigma / sold;
                bool stop = stop_rule(in, o.bnorm2, sigma, rr);
                if (stop && o.relative && !replaced) {  // confirm on the true residual
                    stop = false;
                    o.trigger = 1;
                    o.confirm = 1;
                }
                o.converged = stop ? 1 : 0;
                o.done = (stop || o.it >= o.max_it) ? 1 : 0;
            }
            o.replace = (o.trigger || (o.it % 50 == 0 && o.it > 0) || rr < kReliableDrop2 * o.rr_ref) ? 1 : 0;
        }
        if (threadIdx.x == 0) {
            plan_beta = o.beta;
            plan_done = o.done;
            if (blockIdx.x == 0) *out = o;
        }
    }
    __syncthreads();
    if (plan_done) return;
    if (!body) {  // no FLUID cell: d, q stay 0
        if (threadIdx.x == 0) pout[blockIdx.x] = 0.0;
        return;
    }
    const float ih2[3] = {ihx2, ihy2, ihz2};
    const float fb = (float)plan_beta;
    double v[1] = {0.0};
    auto use = [&](int64_t c, const Raw& w) {  // AXpY(beta, d, s, &d), here and at the neighbours
        const float dc = fb * w.dc + w.zc;
        float nb[6];
#pragma unroll
        for (int k = 0; k < 6; ++k) nb[k] = fb * w.dn[k] + w.zn[k];
        const float qc = code_apply_nb(w.cd, code_center(w.cd, ih2), ih2, dc, nb);
        dnew[c] = dc;
        q[c] = qc;
        v[0] += (double)dc * (double)qc;
    };
#pragma unroll
    for (int u = 0; u < G; ++u)
        if (g0 + (int64_t)u * kBlock < sp.c1) use(g0 + (int64_t)u * kBlock, raw[u]);
    span_groups_from<G, Raw>(g0 + (int64_t)G * kBlock, sp.c1, fetch, use);
    write_partials<1>(v, pout);
}

template <int G>
__global__ __launch_bounds__(kBlock) void k_cg_update(Geom g, const uint16_t* __restrict__ code,
                                                      const float* __restrict__ b, const double* __restrict__ xo,
                                                      double* __restrict__ xn, const float* __restrict__ d,
                                                      const float* __restrict__ q, float* __restrict__ r,
                                                      float* __restrict__ mgx, SolverScalars* sc,
                                                      const double* __restrict__ pin, double* __restrict__ pout,
                                                      int nparts, float ihx2, float ihy2, float ihz2,
                                                      const uint8_t* __restrict__ cfl, int64_t chunk, int64_t padded) {
    const int64_t nc = cell_count(g);
    const Span sp = block_span(nc, chunk, padded);
    const bool body = sp.c0 < sp.c1 && cfl[sp.lb] != 0;
    struct In {
        double x;
        float d, q, r;
        uint16_t cd;
    };
    auto fetch = [&](int64_t c) {
        In t;
        t.x = xo[c];
        t.d = d[c];
        t.q = q[c];
        t.r = r[c];
        t.cd = mgx ? code[c] : (uint16_t)0;  // for the first sweep
        return t;
    };
    const int64_t g0 = sp.c0 + threadIdx.x;
    In raw[G];
    if (body) {
#pragma unroll
        for (int u = 0; u < G; ++u) raw[u] = fetch(min(g0 + (int64_t)u * kBlock, sp.c1 - 1));
    }
    __shared__ double sm[1][kBlock / 64];
    __shared__ double plan_alpha;
    __shared__ int plan_done, plan_replace;
    {
        double t[1] = {0.0};
        add_partials<1>(pin, 1, 0, (int)threadIdx.x, kBlock, nparts, t);
        wave_sums(t, sm);
    }
    __syncthreads();
    if (threadIdx.x < 64) {
        const int done = sc->done, replaces = sc->replace;
        const double sigma = sc->sigma, dq = waves_total(sm[0]);
        if (threadIdx.x == 0) {
            plan_done = done;
            plan_replace = replaces;
            plan_alpha = sigma / dq;
            if (blockIdx.x == 0 && !done) {
                sc->dq = dq;
                sc->alpha = plan_alpha;
            }
        }
    }
    __syncthreads();
    if (plan_done) {  // keep the x rotation consistent
        for (int64_t c = sp.c0 + threadIdx.x; c < sp.c1; c += kBlock) xn[c] = xo[c];
        return;
    }
    if (!body) {  // no FLUID cell: x, r and the first sweep stay 0
        if (threadIdx.x == 0) pout[2 * blockIdx.x] = pout[2 * blockIdx.x + 1] = 0.0;
        return;
    }
    const double alpha = plan_alpha;
    const bool replace = plan_replace != 0;
    const float ih2[3] = {ihx2, ihy2, ihz2};
    const double ih2d[3] = {ihx2, ihy2, ihz2};
    const Stride st = stride_of(g.n[0], g.n[1], g.n[2]);
    const float fa = (float)alpha;
    auto X = [&](int64_t n) { return alpha * (double)d[n] + xo[n]; };
    double v[2] = {0.0, 0.0};  // r.z comes from the V-cycle
    auto finish = [&](int64_t c, uint16_t cd, float rc) {
        r[c] = rc;
        if (mgx) mgx[c] = mg_weight(cd, ih2) * rc;  // the V-cycle's first sweep from zero
        v[1] += (double)rc * (double)rc;
    };
    if (replace) {  // r = b - A x recomputed in FP64
        for (int64_t c = sp.c0 + threadIdx.x; c < sp.c1; c += kBlock) {
            const double xc = X(c);
            xn[c] = xc;
            const uint16_t cd = code[c];
            finish(c, cd, (float)((double)b[c] - code_apply64(cd, c, st, ih2d, xc, X)));
        }
    } else {
        auto use = [&](int64_t c, const In& t) {
            xn[c] = alpha * (double)t.d + t.x;
            finish(c, t.cd, -fa * t.q + t.r);
        };
#pragma unroll
        for (int u = 0; u < G; ++u)
            if (g0 + (int64_t)u * kBlock < sp.c1) use(g0 + (int64_t)u * kBlock, raw[u]);
        span_groups_from<G, In>(g0 + (int64_t)G * kBlock, sp.c1, fetch, use);
    }
    write_partials<2>(v, pout);
}

// ---------------------------------------------------------------------------
// One CG iteration without multigrid in one launch: (r, d, q = A d, x) of the
// read buffers to those of the written ones,
//   alpha = sigma / d.q,  r' = r - alpha q,  x' = x + alpha d (FP64),
//   d' = z' + beta d,  q' = A d',
// with r', z' and d' formed at the six neighbours too.  beta = sigma' / sigma
// needs sigma' = r'.z' before d' exists: r' being r - alpha q, it is sigma -
// 2 alpha q.z + alpha^2 q.M^-1 q, of sums that the launch before has left.
// That is r'.z' but for the FP32 roundings of r' and z', 1e-9 of it, which the
// rounding of beta to FP32 for d' (6e-8) covers; with q.d in the place of q.z,
// equal to it by conjugacy, beta would be off by 1e-6, as the vectors in FP32
// are.  Only beta takes that value: alpha and every test use the r.z and r.r
// summed from r itself.  Where it is not positive (all rounding), and where the
// residual is recomputed, the iteration takes two launches: r' = b - A x' with
// x', then d' and q' with the sums of that r'.
//
// Bound by latency on all but large grids: the launch, one round of loads, the
// partial sums, the state, the block's sums.  An iteration of 190 k cells in
// two launches took 12.7 us, in one 6.6 us.
// After a stop at x of buffer xbuf every launch returns.
// ---------------------------------------------------------------------------
enum CGPhase { kHaveR = 0, kHaveAll = 1, kHaveAllSummed = 2 };  // r; r, d, q; the same with sigma and r.r in the state

struct CGBuffers {
    const float *r, *d, *q;
    const double* x;
    float *ro, *dn, *qo;
    double* xo;
};

// G: cells per thread of a group, kBlock apart.
template <int G, bool DIAG>
__global__ __launch_bounds__(kBlock) void k_cg_step(Geom g, const uint16_t* __restrict__ code,
                                                    const float* __restrict__ b, CGBuffers B, int parity,
                                                    const SolverScalars* __restrict__ in,
                                                    SolverScalars* __restrict__ out, const double* __restrict__ pin,
                                                    double* __restrict__ pout, int nparts, float ihx2, float ihy2,
                                                    float ihz2, const uint8_t* __restrict__ cfl, int64_t chunk,
                                                    int64_t padded) {
    constexpr int NS = cg_sums(DIAG);
    const int64_t nc = cell_count(g);
    const Span sp = block_span(nc, chunk, padded);
    const Stride st = stride_of(g.n[0], g.n[1], g.n[2]);
    const bool body = sp.c0 < sp.c1 && cfl[sp.lb] != 0;
    struct Raw {
        uint16_t cd, cn[DIAG ? 6 : 1];
        float r, d, q, rn[6], dn[6], qn[6];
        double x;
    };
    auto fetch = [&](int64_t c) {
        Raw w;
        w.cd = code[c];
        w.r = B.r[c];
        w.d = B.d[c];
        w.q = B.q[c];
        w.x = B.x[c];
        code_neighbours(c, st, [&](int64_t n) { return B.r[n]; }, w.rn);
        code_neighbours(c, st, [&](int64_t n) { return B.d[n]; }, w.dn);
        code_neighbours(c, st, [&](int64_t n) { return B.q[n]; }, w.qn);
        if constexpr (DIAG) code_neighbours(c, st, [&](int64_t n) { return code[n]; }, w.cn);
        return w;
    };
    // the thread's first group, at its last cell where it has fewer
    Raw raw[G];
    const int64_t g0 = sp.c0 + threadIdx.x;
    if (body) {
#pragma unroll
        for (int u = 0; u < G; ++u) raw[u] = fetch(min(g0 + (int64_t)u * kBlock, sp.c1 - 1));
    }
    __shared__ double sm[NS][kBlock / 64];
    __shared__ double plan_alpha, plan_beta;
    __shared__ int plan_done, plan_only_d, plan_only_r;
    {
        double t[NS] = {};
        add_partials<NS, 4>(pin, NS, 0, (int)threadIdx.x, kBlock, nparts, t);
        wave_sums(t, sm);
    }
    __syncthreads();
    if (threadIdx.x < 64) {
        SolverScalars o = *in;
        const int phase = o.phase;
        if (!o.done) {
            const double sold = o.sigma;
            const bool first = o.it < 0, replaced = phase == kHaveR;
            if (phase != kHaveAllSummed) {
                o.sigma_old = sold;
                o.rr = waves_total(sm[0]);
                o.sigma = DIAG ? waves_total(sm[NS - 1]) : o.rr;
                o.confirm = 0;
                bool stop = stop_rule(in, o.bnorm2, o.sigma, o.rr);
                if (first) {  // the sums are k_cg_init's
                    o.it = 0;
                    o.trigger = 0;
                    o.rr_ref = o.rr;
                } else {
                    if (replaced) o.rr_ref = o.rr;
                    ++o.it;
                    o.trigger = o.sigma > sold ? 1 : 0;
                    if (stop && o.relative && !replaced) {  // confirm on the true residual
                        stop = false;
                        o.trigger = 1;
                        o.confirm = 1;
                    }
                }
                o.converged = stop ? 1 : 0;
                o.done = (stop || o.it >= o.max_it) ? 1 : 0;
                o.replace = (o.trigger || (o.it % 50 == 0 && o.it > 0) || o.rr < kReliableDrop2 * o.rr_ref) ? 1 : 0;
            }
            if (phase == kHaveR) {
                o.beta = first ? 0.0 : o.sigma / sold;
            } else {
                o.dq = waves_total(sm[1]);
                o.alpha = o.sigma / o.dq;
                const double fa = (double)(float)o.alpha;  // as r' takes it
                o.beta = (o.sigma - 2.0 * fa * waves_total(sm[3]) + fa * fa * waves_total(sm[2])) / o.sigma;
                if (!(o.beta > 0.0)) o.replace = 1;
            }
            o.phase = phase == kHaveR ? kHaveAllSummed : (o.replace ? kHaveR : kHaveAll);
            ++o.launches;
            o.xbuf = parity;
        }
        if (threadIdx.x == 0) {
            plan_alpha = o.alpha;
            plan_beta = o.beta;
            plan_done = o.done;
            plan_only_d = phase == kHaveR;
            plan_only_r = phase != kHaveR && o.replace;
            if (blockIdx.x == 0) *out = o;
        }
    }
    __syncthreads();
    if (plan_done) return;
    const double alpha = plan_alpha, beta = plan_beta;
    const bool only_d = plan_only_d != 0, only_r = plan_only_r != 0;
    if (!body) {  // no FLUID cell: every vector stays 0
        if (threadIdx.x < NS) pout[NS * (int64_t)blockIdx.x + threadIdx.x] = 0.0;
        return;
    }
    const float ih2[3] = {ihx2, ihy2, ihz2};
    const double ih2d[3] = {ihx2, ihy2, ihz2};
    const float fa = (float)alpha, fb = (float)beta;
    double v[NS] = {};
    auto precond = [&](float r, uint16_t cd) { return DIAG ? r / code_center(cd, ih2) : r; };
    auto direction = [&](int64_t c, uint16_t cd, float zc, float dc, const float (&nb)[6]) {
        const float center = code_center(cd, ih2);
        const float qc = code_apply_nb(cd, center, ih2, dc, nb);
        B.dn[c] = dc;
        B.qo[c] = qc;
        v[1] += (double)dc * (double)qc;
        v[2] += (double)qc * (double)(DIAG ? qc / center : qc);
        v[3] += (double)qc * (double)zc;
    };
    auto residual = [&](int64_t c, float rc, float zc) {
        B.ro[c] = rc;
        v[0] += (double)rc * (double)rc;
        if constexpr (DIAG) v[NS - 1] += (double)rc * (double)zc;
    };
    auto use = [&](int64_t c, const Raw& w) {
        float nb[6];
        if (only_r) {
            auto X = [&](int64_t n) { return alpha * (double)B.d[n] + B.x[n]; };
            const double xc = alpha * (double)w.d + w.x;
            B.xo[c] = xc;
            B.dn[c] = w.d;
            const float rc = (float)((double)b[c] - code_apply64(w.cd, c, st, ih2d, xc, X));
            residual(c, rc, precond(rc, w.cd));
        } else if (only_d) {
            B.xo[c] = w.x;
            B.ro[c] = w.r;
#pragma unroll
            for (int k = 0; k < 6; ++k) nb[k] = fmaf(fb, w.dn[k], precond(w.rn[k], w.cn[DIAG ? k : 0]));
            const float zc = precond(w.r, w.cd);
            direction(c, w.cd, zc, fmaf(fb, w.d, zc), nb);
        } else {
            B.xo[c] = alpha * (double)w.d + w.x;
            const float rc = fmaf(-fa, w.q, w.r), zc = precond(rc, w.cd);
            residual(c, rc, zc);
#pragma unroll
            for (int k = 0; k < 6; ++k)
                nb[k] = fmaf(fb, w.dn[k], precond(fmaf(-fa, w.qn[k], w.rn[k]), w.cn[DIAG ? k : 0]));
            direction(c, w.cd, zc, fmaf(fb, w.d, zc), nb);
        }
    };
#pragma unroll
    for (int u = 0; u < G; ++u)
        if (g0 + (int64_t)u * kBlock < sp.c1) use(g0 + (int64_t)u * kBlock, raw[u]);
    for (int64_t c = g0 + (int64_t)G * kBlock; c < sp.c1; c += kBlock) use(c, fetch(c));
    write_partials<NS>(v, pout);
}

// Final ||b - A p||^2 and ||b||^2 in FP64 on the FP64 solution, with FP64
// coefficients 1/h^2.
__global__ __launch_bounds__(kBlock) void k_final_residual(Geom g, const uint16_t* __restrict__ code,
                                                           const float* __restrict__ b, const double* __restrict__ x,
                                                           double* __restrict__ pout, double ihx2, double ihy2,
                                                           double ihz2, int64_t chunk, int64_t padded) {
    const int64_t nc = cell_count(g);
    const Span sp = block_span(nc, chunk, padded);
    const double ih2[3] = {ihx2, ihy2, ihz2};
    const Stride st = stride_of(g.n[0], g.n[1], g.n[2]);
    double v[2] = {0.0, 0.0};
    span_groups<4, Stencil64In>(
        sp.c0, sp.c1, [&](int64_t c) { return stencil64_in(c, code, x, b, st); },
        [&](int64_t c, const Stencil64In& t) {
            const double res = (double)t.bc - code_apply64_nb(t.cd, ih2, t.xc, t.nb);
            v[0] += res * res;
            v[1] += (double)t.bc * (double)t.bc;
        });
    write_partials<2>(v, pout);
}

// One block: totals of NV-wide partials into out[0..NV).
template <int NV>
__global__ __launch_bounds__(kBlock) void k_finish(const double* __restrict__ part, int nparts, double* out) {
    double t[NV];
    sum_partials<NV>(part, nparts, t);
    if (threadIdx.x == 0)
        for (int q = 0; q < NV; ++q) out[q] = t[q];
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------
static inline dim3 grid1(int64_t n) { return dim3((unsigned)((n + kBlock - 1) / kBlock)); }

static SolverShape solver_shape(const Geom& g) { return solver_shape_n(cell_count(g)); }

hipError_t launch_final_residual(fe_scene* s) {
    const Geom& g = s->g;
    const SolverShape sh = solver_shape(g);
    double* part = s->partials;
    hipLaunchKernelGGL(k_final_residual, dim3((unsigned)sh.blocks), dim3(kBlock), 0, s->stream, g, s->code, s->b,
                       s->p, part, g.ihd[0] * g.ihd[0], g.ihd[1] * g.ihd[1], g.ihd[2] * g.ihd[2], sh.chunk, sh.blocks);
    // totals (||r||^2, ||b||^2) land after the partials; read_final_residual fetches them
    hipLaunchKernelGGL(k_finish<2>, dim3(1), dim3(kBlock), 0, s->stream, part, (int)sh.blocks,
                       part + 2 * sh.blocks);
    return hipGetLastError();
}

static hipError_t read_scalars(fe_scene* s, int slot) {
    hipError_t e = hipMemcpyAsync(s->sc_host, s->sc + slot, sizeof(SolverScalars), hipMemcpyDeviceToHost, s->stream);
    if (e != hipSuccess) return e;
    return hipStreamSynchronize(s->stream);
}

hipError_t read_final_residual(fe_scene* s, double* rr, double* bb) {
    const SolverShape sh = solver_shape(s->g);
    double tot[2] = {0.0, 0.0};
    hipError_t e = hipMemcpyAsync(tot, s->partials + 2 * sh.blocks, sizeof(tot), hipMemcpyDeviceToHost, s->stream);
    if (e != hipSuccess) return e;
    if ((e = hipStreamSynchronize(s->stream)) != hipSuccess) return e;
    *rr = tot[0];
    *bb = tot[1];
    return hipSuccess;
}

// Zeros for up to 8 buffers in one launch: buffer q takes blocks
// [first[q], first[q + 1]), four 32-bit words per thread (one 16-byte store;
// every buffer starts 256-byte aligned).
struct ZeroList {
    int n = 0;
    uint32_t* p[8] = {};
    int64_t words[8] = {};
    int64_t first[9] = {};
};

__global__ __launch_bounds__(kBlock) void k_zero_many(ZeroList L) {
    const int64_t blk = blockIdx.x;
    int q = 0;
    while (q + 1 < L.n && blk >= L.first[q + 1]) ++q;
    const int64_t w0 = ((blk - L.first[q]) * kBlock + threadIdx.x) * 4;
    uint32_t* __restrict__ p = L.p[q];
    if (w0 + 4 <= L.words[q]) {
        *reinterpret_cast<uint4*>(p + w0) = make_uint4(0u, 0u, 0u, 0u);
    } else {
        for (int64_t w = w0; w < L.words[q]; ++w) p[w] = 0u;
    }
}

static void zero_add(ZeroList& L, void* p, int64_t bytes) {
    if (!p || bytes <= 0) return;
    L.p[L.n] = static_cast<uint32_t*>(p);
    L.words[L.n] = bytes / 4;
    L.first[L.n + 1] = L.first[L.n] + (L.words[L.n] + 4 * kBlock - 1) / (4 * kBlock);
    ++L.n;
}

// The solver's start: its scalars, BuildSystem and the initial guess.
static hipError_t solve_begin(fe_scene* s, const fe_solver_desc* d, SolverScalars& init) {
    const Geom& g = s->g;
    const int64_t nc = cell_count(g);
    const SolverShape sh = solver_shape(g);
    init = SolverScalars{};
    init.tol = d->tolerance;
    init.relative = d->relative;
    init.precond = d->kind == FE_SOLVER_PCG_JACOBI ? 1 : (d->kind == FE_SOLVER_MGPCG ? 2 : 0);
    init.max_it = d->max_iterations;
    init.it = -1;
    // the scalars' start goes with BuildSystem's launch (a kernel argument
    // rather than a host copy, so a captured substep carries the values)
    FaceSet u{{s->u[0], s->u[1], s->u[2]}};
    hipLaunchKernelGGL(k_build_system, dim3((unsigned)sh.blocks), dim3(kBlock), 0, s->stream, g, u, s->flags, s->code,
                       s->b, s->partials, s->chunk_fluid, sh.chunk, sh.blocks, s->sc, init);
    if (d->warm_start == FE_WARM_START_LEARNED) {
        if (!s->net) return hipErrorInvalidValue;
        hipError_t e = net_warm_start(s->net, s);
        if (e != hipSuccess) return e;
    } else if (!d->warm_start) {
        hipLaunchKernelGGL(k_zero_f64, grid1(nc), dim3(kBlock), 0, s->stream, s->p, nc);
    }
    return hipGetLastError();
}

// Jacobi sweeps (JacobiIterationSolver::Solve), host-driven.
static hipError_t jacobi_solve(fe_scene* s, const fe_solver_desc* d) {
    const Geom& g = s->g;
    const int64_t nc = cell_count(g);
    const SolverShape sh = solver_shape(g);
    const int nparts = (int)sh.blocks;
    double* PA = s->partials;
    double* PB = s->partials + 2 * sh.blocks;
    const float ih2[3] = {(float)(g.ihd[0] * g.ihd[0]), (float)(g.ihd[1] * g.ihd[1]), (float)(g.ihd[2] * g.ihd[2])};
    hipError_t e;
    // The reference's CudaJacobiIterationSolver uploads the previous x (warm start).
    float* xa = s->r;
    float* xb = s->z;
    hipLaunchKernelGGL(k_f64_to_f32, grid1(nc), dim3(kBlock), 0, s->stream, s->p, xa, nc);
    bool pending = false;
    int pending_it = 0;
    for (int it = 0; it < d->max_iterations; ++it) {
        launch_timed(s, FE_KERNEL_JACOBI, 0, k_jacobi, dim3((unsigned)sh.blocks), dim3(kBlock), g,
                     (const uint16_t*)s->code, (const float*)s->b, (const float*)xa, xb, s->sc,
                     (const double*)(pending ? PB : nullptr), nparts, pending_it, ih2[0], ih2[1], ih2[2], sh.chunk,
                     sh.blocks);
        std::swap(xa, xb);
        pending = false;
        if (it != 0 && d->check_interval > 0 && it % d->check_interval == 0) {
            hipLaunchKernelGGL(k_jacobi_residual, dim3((unsigned)sh.blocks), dim3(kBlock), 0, s->stream, g,
                               s->code, s->b, xa, s->sc, PB, ih2[0], ih2[1], ih2[2], sh.chunk, sh.blocks);
            pending = true;
            pending_it = it;
        }
    }
    if (pending)  // a check after the last sweep: the loop ends anyway, only record convergence
        hipLaunchKernelGGL(k_finish<1>, dim3(1), dim3(kBlock), 0, s->stream, PB, nparts, PA);
    hipLaunchKernelGGL(k_f32_to_f64, grid1(nc), dim3(kBlock), 0, s->stream, xa, s->p, nc);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if ((e = read_scalars(s, 0)) != hipSuccess) return e;
    if (pending && !s->sc_host->done) {
        double tot = 0.0;
        if ((e = hipMemcpy(&tot, PA, sizeof(double), hipMemcpyDeviceToHost)) != hipSuccess) return e;
        if (std::sqrt(tot) < d->tolerance) {
            s->sc_host->done = 1;
            s->sc_host->converged = 1;
            s->sc_host->it = pending_it + 1;
        }
    }
    kt_flush(s);
    return hipSuccess;
}

// ---------------------------------------------------------------------------
// CG / PCG, host side.  spmv k decides the stop of update k-1, so every batch
// of launches ends with an spmv whose state slot the host reads; launches
// after the stop leave before their first write (after at most one group of
// loads) and are left out of the kernel timer (tags >= the stopping iteration).
// ---------------------------------------------------------------------------
struct CGSetup {
    Geom g;
    SolverShape sh;
    int nparts = 0;
    double *PA = nullptr, *PB = nullptr, *PZ = nullptr;
    float ih2[3] = {0, 0, 0};
    int precond = 0;
    bool mg = false, fused = false;
    float* mgx = nullptr;
    int nz = 0;
};

// The per-solve constants (after mg_setup: the fused V-cycle's partials are
// allocated with its levels).
static CGSetup cg_setup(fe_scene* s, int precond) {
    CGSetup c;
    c.g = s->g;
    c.sh = solver_shape(s->g);
    c.nparts = (int)c.sh.blocks;
    c.PA = s->partials;                    // 2 per block, without multigrid cg_sums
    c.PB = s->partials + (precond == 2 ? 2 : cg_sums(precond == 1)) * c.sh.blocks;  // as many
    c.PZ = s->partials + 4 * c.sh.blocks;  // r.z of the V-cycle, 1 per block
    // BuildSystem's invH * invH (single_phase_pressure_solver.cpp:102-103); exact
    // in FP32 for power-of-two spacings
    for (int a = 0; a < 3; ++a) c.ih2[a] = (float)(s->g.ihd[a] * s->g.ihd[a]);
    c.precond = precond;
    c.mg = precond == 2;
    c.fused = c.mg && s->tune.mg == FE_MG_FUSED;
    if (c.fused) c.PZ = s->mg_pz;  // one r.z partial per workgroup of the level-0 ascent
    c.mgx = c.mg && !c.fused ? mg_first_sweep_target(s) : nullptr;  // the fused descent sweeps from b itself
    c.nz = c.fused ? (int)s->mg_npz : c.nparts;
    return c;
}

static void cg_update(fe_scene* s, const CGSetup& c, CGRun& R, int kk) {
    R.dcur = 1 - R.dcur;
    with_group(c.sh, [&](auto G) {
        launch_timed(s, FE_KERNEL_CG_UPDATE, kk, k_cg_update<G.value>, dim3((unsigned)c.sh.blocks), dim3(kBlock), c.g,
                     (const uint16_t*)s->code, (const float*)s->b, (const double*)R.xa, R.xb,
                     (const float*)s->d[R.dcur], (const float*)s->q, s->r, c.mgx, s->sc + ((kk + 1) & 1),
                     (const double*)c.PA, c.PB, c.nparts, c.ih2[0], c.ih2[1], c.ih2[2],
                     (const uint8_t*)s->chunk_fluid, c.sh.chunk, c.sh.blocks);
    });
    std::swap(R.xa, R.xb);
    (void)mg_apply(s, s->r, s->z, s->sc + ((kk + 1) & 1), c.PZ, kk, c.PB, c.nparts);
}

// nb spmv launches with an update (and V-cycle) between each two; R.k is the
// last spmv's iteration afterwards.
static void cg_batch(fe_scene* s, const CGSetup& c, CGRun& R, int nb) {
    for (int t = 0; t < nb; ++t) {
        with_group(c.sh, [&](auto G) {
            launch_timed(s, FE_KERNEL_CG_SPMV, R.k, k_cg_spmv<G.value>, dim3((unsigned)c.sh.blocks), dim3(kBlock), c.g,
                         (const uint16_t*)s->code, (const float*)s->z, (const float*)s->d[R.dcur], s->d[1 - R.dcur],
                         s->q, (const SolverScalars*)(s->sc + (R.k & 1)), s->sc + ((R.k + 1) & 1),
                         (const double*)c.PB, (const double*)c.PZ, c.nz, c.PA, c.nparts, c.ih2[0], c.ih2[1], c.ih2[2],
                         (const uint8_t*)s->chunk_fluid, c.sh.chunk, c.sh.blocks);
        });
        if (t == nb - 1) break;
        cg_update(s, c, R, R.k);
        ++R.k;
    }
}

// n launches of k_cg_step.
static void cg_steps(fe_scene* s, const CGSetup& c, CGRun& R, int n) {
    double* const X[2] = {s->p, s->p2};
    float* const r[2] = {s->r, s->z};
    float* const q[2] = {s->q, s->q2};
    double* const part[2] = {c.PB, c.PA};
    auto step = [&](auto kernel) {
        const int i = R.k & 1, o = 1 - i;
        const CGBuffers B{r[i], s->d[i], q[i], X[i], r[o], s->d[o], q[o], X[o]};
        launch_timed(s, FE_KERNEL_CG_SPMV, R.k, kernel, dim3((unsigned)c.sh.blocks), dim3(kBlock), c.g,
                     (const uint16_t*)s->code, (const float*)s->b, B, i, (const SolverScalars*)(s->sc + i), s->sc + o,
                     (const double*)part[i], part[o], c.nparts, c.ih2[0], c.ih2[1], c.ih2[2],
                     (const uint8_t*)s->chunk_fluid, c.sh.chunk, c.sh.blocks);
    };
    // One cell per thread up to 2^18 cells; above, two at a time: an iteration of
    // half full tanks, CG / diagonal preconditioner, 80x56x68 7.0 / 9.4 us (one
    // at a time 7.5 / 9.7, four 7.9 / 12.3), 128^3 20.9 / 33.0 (20.9 / 32.7,
    // 26.7 / 42.8).
    const bool one = c.sh.chunk <= kBlock;
    for (; n > 0; --n, ++R.k) {
        if (c.precond)
            one ? step(k_cg_step<1, true>) : step(k_cg_step<2, true>);
        else
            one ? step(k_cg_step<1, false>) : step(k_cg_step<2, false>);
    }
}

// The iterations' start: the solver vectors' zeros, the initial residual and
// the first V-cycle.  The CG and level-0 multigrid kernels skip the chunks
// without FLUID cells (s->chunk_fluid): every vector they would write there
// starts at 0 and, FLUID rows coupling only to FLUID cells, stays 0
// (k_cg_init writes r, d, the first sweep and the solution's zeros outside
// FLUID itself).
static hipError_t cg_start(fe_scene* s, const CGSetup& c, CGRun& R) {
    const int64_t nc = cell_count(c.g);
    hipError_t e;
    ZeroList L;
    zero_add(L, s->z, 4 * nc);
    zero_add(L, s->q, 4 * nc);
    if (!c.mg) zero_add(L, s->q2, 4 * nc);
    zero_add(L, s->d[1], 4 * nc);
    if (c.mg) zero_add(L, s->mg[0].x2, 4 * nc);
    // the fused V-cycle skips level-0 tiles without FLUID cells: the coarse
    // right-hand side below them stays 0
    if (c.fused) zero_add(L, s->mg[1].b, 4 * s->mg[1].cells);
    if (c.mg) zero_add(L, s->mg[0].r, 4 * nc);
    zero_add(L, s->p2, 8 * nc);
    hipLaunchKernelGGL(k_zero_many, dim3((unsigned)L.first[L.n]), dim3(kBlock), 0, s->stream, L);
    hipLaunchKernelGGL(k_cg_init, dim3((unsigned)c.sh.blocks), dim3(kBlock), 0, s->stream, c.g, s->code, s->b, s->p,
                       s->r, s->d[0], c.mgx, s->sc, c.PA, c.PB, c.mg ? 2 : cg_sums(c.precond == 1), c.nparts, c.ih2[0],
                       c.ih2[1], c.ih2[2], c.sh.chunk, c.sh.blocks);
    if (c.mg && (e = mg_apply(s, s->r, s->z, s->sc, c.PZ, -1, nullptr, 0)) != hipSuccess) return e;
    R = CGRun{};
    R.xa = s->p;
    R.xb = s->p2;
    return hipGetLastError();
}

// Launches of k_cg_step that end any solve: the start's, then at most two an
// iteration.
static int cg_step_bound(const fe_solver_desc* d) {
    return (int)std::min<int64_t>(2 * (int64_t)std::max(d->max_iterations, 0) + 1, 1 << 30);
}

// Host-driven iterations without multigrid: batches of steps, the host reading
// the last one's state slot.  expect: launches that the solve may take, from
// the last one (0: there was none); alike: that had the same settings.
// Waiting for the device between two batches costs about 30 us, an iteration
// 6.5 (190 k cells) and a launch after the stop 3.  So a solve like the last
// takes 512 at a time up to its length, any other at most as many as have run
// (64 at first) up to there; beyond, or where nothing is known, a batch is a
// quarter of what has run since.  No batch passes the bound.
static hipError_t cg_step_loop(fe_scene* s, const fe_solver_desc* d, const CGSetup& c, CGRun& R, int expect,
                               bool alike) {
    hipError_t e;
    const int bound = cg_step_bound(d);
    for (;;) {
        int n;
        if (R.k < expect)
            n = std::min(alike ? 512 : std::max(R.k, 64), expect - R.k);
        else
            n = std::max((R.k - expect) / 4, R.k > 0 ? 8 : 16);
        cg_steps(s, c, R, std::max(1, std::min(n, bound - R.k)));
        if ((e = hipGetLastError()) != hipSuccess) return e;
        if ((e = read_scalars(s, R.k & 1)) != hipSuccess) return e;
        kt_flush(s, s->sc_host->done ? s->sc_host->launches - 1 : (1 << 30));
        if (s->sc_host->done) break;  // the iteration cap ends every solve
    }
    s->last_cg_launches[c.precond] = s->sc_host->launches;
    s->last_cg_desc[c.precond] = *d;
    return hipSuccess;
}

// Host-driven iterations with multigrid: batches of spmv launches, the host
// reading the last one's state slot.  resume: the state slot read last said
// "not done" after a batch launched elsewhere (a captured substep), so the
// next update comes first.  first: spmv launches in the first batch.
static hipError_t cg_host_loop(fe_scene* s, const fe_solver_desc* d, const CGSetup& c, CGRun& R, int first,
                               bool resume) {
    hipError_t e;
    if (resume) {
        cg_update(s, c, R, R.k);
        ++R.k;
    }
    for (;;) {
        const int nb = std::min(first, d->max_iterations + 1 - R.k);
        first = 2;
        cg_batch(s, c, R, nb);
        if ((e = hipGetLastError()) != hipSuccess) return e;
        if ((e = read_scalars(s, (R.k + 1) & 1)) != hipSuccess) return e;
        kt_flush(s, s->sc_host->done ? s->sc_host->it : (1 << 30));
        if (s->sc_host->done || nb <= 0) break;
        cg_update(s, c, R, R.k);
        ++R.k;
    }
    return hipSuccess;
}

hipError_t pressure_alloc(fe_scene* s, const fe_solver_desc* d) {
    if (s->q2 || (d->kind != FE_SOLVER_CG && d->kind != FE_SOLVER_PCG_JACOBI)) return hipSuccess;
    return hipMalloc((void**)&s->q2, sizeof(float) * cell_count(s->g) + 64);
}

hipError_t launch_pressure_solve(fe_scene* s, const fe_solver_desc* d) {
    SolverScalars init;
    hipError_t e = pressure_alloc(s, d);
    if (e != hipSuccess) return e;
    if ((e = solve_begin(s, d, init)) != hipSuccess) return e;
    if (d->kind == FE_SOLVER_JACOBI) return jacobi_solve(s, d);
    if (init.precond == 2 && (e = mg_setup(s)) != hipSuccess) return e;
    const CGSetup c = cg_setup(s, init.precond);
    CGRun R;
    if ((e = cg_start(s, c, R)) != hipSuccess) return e;
    // the first host check comes where the previous solve of this kind stopped
    // (warm-started solves of consecutive substeps take similar counts), so a
    // typical solve waits for the device once; a launch after the stop costs
    // about 2 us
    if (c.mg) {
        const int prev = s->last_cg_iters[2];
        if ((e = cg_host_loop(s, d, c, R, prev > 0 ? std::min(prev + 1, 64) : 4, false)) != hipSuccess) return e;
    } else {
        const int prev = s->last_cg_launches[c.precond];
        if ((e = cg_step_loop(s, d, c, R, prev > 0 ? prev + 1 : 0, same_solver(s->last_cg_desc[c.precond], *d))) !=
            hipSuccess)
            return e;
        if (s->sc_host->xbuf) R.xa = s->p2;
    }
    if (R.xa != s->p) {
        s->p2 = s->p;
        s->p = R.xa;
    }
    s->last_cg_iters[init.precond] = s->sc_host->done ? s->sc_host->it : d->max_iterations;
    return hipSuccess;
}

// A captured substep's part of the solve: the start and the first `iters`
// spmv launches, then the state slot of the last one copied into the pinned
// host mirror.  Returns the run's state after them.
hipError_t capture_pressure_head(fe_scene* s, const fe_solver_desc* d, int iters, CGRun* out) {
    SolverScalars init;
    hipError_t e = solve_begin(s, d, init);
    if (e != hipSuccess) return e;
    if (init.precond == 2 && (e = mg_setup(s)) != hipSuccess) return e;
    const CGSetup c = cg_setup(s, init.precond);
    CGRun R;
    if ((e = cg_start(s, c, R)) != hipSuccess) return e;
    int slot;
    if (c.mg) {
        cg_batch(s, c, R, std::max(1, std::min(iters, d->max_iterations + 1)));
        slot = (R.k + 1) & 1;
    } else {  // recomputed residuals take a second launch
        const int prev = s->last_cg_launches[c.precond];
        cg_steps(s, c, R, std::min(prev > 0 ? prev + 2 : iters, cg_step_bound(d)));
        slot = R.k & 1;
    }
    if ((e = hipMemcpyAsync(s->sc_host, s->sc + slot, sizeof(SolverScalars), hipMemcpyDeviceToHost, s->stream)) !=
        hipSuccess)
        return e;
    *out = R;
    return hipGetLastError();
}

// After a captured head has run (s->sc_host holds its last state slot): the
// host-driven iterations it left, if any, then the solution copied into s->p
// when the iteration count left it in the partner buffer (a captured tail
// reads s->p).  *resumed: whether iterations were added.
hipError_t finish_pressure_after_head(fe_scene* s, const fe_solver_desc* d, const CGRun& head, bool* resumed) {
    const int precond = d->kind == FE_SOLVER_PCG_JACOBI ? 1 : (d->kind == FE_SOLVER_MGPCG ? 2 : 0);
    const CGSetup c = cg_setup(s, precond);
    CGRun R = head;
    hipError_t e;
    *resumed = false;
    if (!c.mg) {
        if (!s->sc_host->done) {
            *resumed = true;
            if ((e = cg_step_loop(s, d, c, R, R.k, false)) != hipSuccess) return e;
        }
        s->last_cg_launches[c.precond] = s->sc_host->launches;
        s->last_cg_desc[c.precond] = *d;
        if (s->sc_host->xbuf) R.xa = s->p2;
    } else if (!s->sc_host->done && R.k + 1 <= d->max_iterations) {
        *resumed = true;
        if ((e = cg_host_loop(s, d, c, R, 2, true)) != hipSuccess) return e;
    }
    if (R.xa != s->p &&
        (e = hipMemcpyAsync(s->p, R.xa, sizeof(double) * cell_count(s->g), hipMemcpyDeviceToDevice, s->stream)) !=
            hipSuccess)
        return e;
    s->last_cg_iters[precond] = s->sc_host->done ? s->sc_host->it : d->max_iterations;
    return hipSuccess;
}

}  // namespace fe
