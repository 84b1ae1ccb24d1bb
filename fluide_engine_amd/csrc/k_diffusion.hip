// k_diffusion.hip -- BackwardEulerDiffusionSolver (viscosity) on the device.
//
// src/fluid_solvers/backward_euler_diffusion_solver.cpp:20-242, called by
// PICSimulator::ComputeDiffusion (src/pic_simulator.cpp:214-222) when the
// viscosity is positive.  Per face component:
//   * face markers: FLUID iff the fluid SDF sampled at the face position is
//     negative, else BOUNDRY iff the collider SDF is, else AIR (BuildX/Y/ZMarkers,
//     :71-128);
//   * system (BuildMatrix :136-198, BuildVectors :200-242): a FLUID row has
//     centre 1 + c_a per in-range non-AIR neighbour and -c_a to every FLUID
//     neighbour, b = u + c_a * u(neighbour) per BOUNDRY neighbour; other rows
//     are the identity with b = u; x0 = u.  c_a = dt * viscosity / h_a^2.
//   * solver: the reference's CudaJacobiIterationSolver(1000, 5, 1e-14) (:10)
//     semantics: sweep, and after sweep it (it > 0, it % interval == 0) stop
//     when ||b - A x||_2 < tolerance.
// The three components' solves are independent; on all but large grids they
// run side by side in the same launches, each with its own stop (DiffState).
// Everything is FP64 (x, b, the row arithmetic in the reference's operation
// order with contraction off, the residual); the face velocities stay FP32
// and are exact in FP64.  The 16-bit row code has the pressure
// solver's layout: bits 0-5 coupled (FLUID) neighbours in the order i-1, i+1,
// j-1, j+1, k-1, k+1; bits 6-11 in-range non-AIR neighbours per axis; bit 12
// the row is FLUID.
#include <algorithm>
#include <cmath>

#include "fe_kernels.hpp"
#include "fe_stencil.hpp"

namespace fe {

namespace {

// The solved components' faces back to back: component c's start at off[c] in
// every array, its workgroups are blk[c] .. blk[c + 1] (multiples of 8 each,
// so the XCD remap holds within a component; none where it is not solved).
struct DiffGrid {
    int nx[3], ny[3];
    int64_t nf[3], off[3];
    int64_t blk[4];
};

constexpr int kDiffPer = 2;  // faces per thread of a sweep, kBlock apart
constexpr int kDiffOpen = INT32_MAX;  // DiffState::end of a solve that goes on

__device__ inline int diff_component(const DiffGrid& D, int64_t b) { return (b >= D.blk[1]) + (b >= D.blk[2]); }

// The workgroup's component and its first face there.
__device__ inline int64_t diff_first(const DiffGrid& D, int c) {
    const int64_t lb = xcd_remap((int64_t)blockIdx.x - D.blk[c], D.blk[c + 1] - D.blk[c]);
    return lb * (kBlock * kDiffPer);
}

// Face markers of the three components and the solves' start.
__global__ __launch_bounds__(kBlock) void k_diff_markers(Geom g, DiffGrid D, const double* __restrict__ sdf,
                                                         const double* __restrict__ csdf, uint8_t* __restrict__ m0,
                                                         uint8_t* __restrict__ m1, uint8_t* __restrict__ m2,
                                                         DiffState* __restrict__ st, DiffState init) {
#pragma clang fp contract(off)
    if (blockIdx.x == 0 && threadIdx.x < 3) st[threadIdx.x] = init;
    const int C = diff_component(D, blockIdx.x);
    uint8_t* mark = C == 0 ? m0 : (C == 1 ? m1 : m2);
    const int64_t f0 = diff_first(D, C) + threadIdx.x;
#pragma unroll
    for (int t = 0; t < kDiffPer; ++t) {
        const int64_t f = f0 + t * kBlock;
        if (f >= D.nf[C]) return;
        int idx[3];
        split_index(f, D.nx[C], D.ny[C], idx[0], idx[1], idx[2]);
        double p[3];
#pragma unroll
        for (int a = 0; a < 3; ++a) p[a] = g.cod[C][a] + g.hd[a] * (double)idx[a];  // GetX/Y/ZPos
        uint8_t m = FE_AIR;
        if (sample_sdf64(g, sdf, p) < 0)
            m = FE_FLUID;
        else if (csdf && sample_collider64(g, csdf, p) < 0)
            m = FE_BOUNDRY;
        mark[f] = m;
    }
}

// Row codes, right-hand sides and x0 = u, into both iterates: an identity row
// has the solution b = u, so no sweep needs to visit it, and the residual 0, or
// none that any tolerance meets where u is not finite.
__global__ __launch_bounds__(kBlock) void k_diff_build(DiffGrid D, FaceSet uu, const uint8_t* __restrict__ m0,
                                                       const uint8_t* __restrict__ m1, const uint8_t* __restrict__ m2,
                                                       uint16_t* __restrict__ code, double* __restrict__ x0,
                                                       double* __restrict__ x1, double* __restrict__ b, double cx,
                                                       double cy, double cz, DiffState* __restrict__ st) {
#pragma clang fp contract(off)
    const int C = diff_component(D, blockIdx.x);
    const uint8_t* __restrict__ mark = C == 0 ? m0 : (C == 1 ? m1 : m2);
    const float* __restrict__ u = uu.a[C];
    const int64_t f0 = diff_first(D, C) + threadIdx.x;
    const int nx = D.nx[C], ny = D.ny[C];
    const int64_t sy = nx, sz = (int64_t)nx * ny, nf = D.nf[C];
#pragma unroll
    for (int e = 0; e < kDiffPer; ++e) {
        const int64_t f = f0 + e * kBlock;
        if (f >= nf) return;
        uint16_t cd = 0;
        double bb = (double)u[f];
        const int64_t o = D.off[C] + f;
        x0[o] = bb;
        x1[o] = bb;
        if (mark[f] == FE_FLUID) {
            int i, j, k;
            split_index(f, nx, ny, i, j, k);
            const int nz = (int)(nf / sz);
            const bool in[6] = {i > 0, i + 1 < nx, j > 0, j + 1 < ny, k > 0, k + 1 < nz};
            const int64_t nb[6] = {f - 1, f + 1, f - sy, f + sy, f - sz, f + sz};
            cd = kFluidBit;
#pragma unroll
            for (int q = 0; q < 6; ++q) {
                if (!in[q]) continue;
                const uint8_t m = mark[nb[q]];
                if (m == FE_AIR) continue;
                cd = (uint16_t)(cd + (1u << (6 + 2 * (q >> 1))));
                if (m == FE_FLUID) cd |= (uint16_t)(1u << q);
            }
            // BuildVectors' BOUNDRY terms in its order: i+1, i-1, j+1, j-1, k+1, k-1
            const double c[3] = {cx, cy, cz};
            const int order[6] = {1, 0, 3, 2, 5, 4};
#pragma unroll
            for (int t = 0; t < 6; ++t) {
                const int q = order[t];
                if (in[q] && mark[nb[q]] == FE_BOUNDRY) bb += c[q >> 1] * (double)u[nb[q]];
            }
        } else if (!(bb - bb == 0.0)) {
            st[C].nonfinite = 1;  // every writer writes the same
        }
        code[o] = cd;
        b[o] = bb;
    }
}

// Centre 1 + c_a per non-AIR neighbour, summed in BuildMatrix's order (x, y, z).
__device__ inline double diff_center(uint16_t cd, const double (&c)[3]) {
#pragma clang fp contract(off)
    double center = 1.0;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const int cnt = (cd >> (6 + 2 * a)) & 3;
        if (cnt > 0) center += c[a];
        if (cnt > 1) center += c[a];
    }
    return center;
}

// Sum of the off-diagonal terms A_ij x_j of a FLUID row in the reference
// Jacobi order (i-1, i+1, j-1, j+1, k-1, k+1).  An uncoupled term adds 0,
// which changes no sum that started at +0.
__device__ inline double diff_offdiag(uint16_t cd, const double (&c)[3], const double (&nb)[6]) {
#pragma clang fp contract(off)
    double r = 0.0;
#pragma unroll
    for (int q = 0; q < 6; ++q) r += (cd & (1u << q)) ? (-c[q >> 1]) * nb[q] : 0.0;
    return r;
}

// Jacobi sweep number `it` of the three components, x_{it+1} from x_it = xo
// into xn.  CHECK: also the partials of ||b - A x_it||^2 (BLAS::Residual,
// src/linear_system/blas.cpp:21-37; the off-diagonal sums are the sweep's),
// and whether any value differs from the snapshot of an earlier state, which
// `snap` 1 renews.  !WRITE: the partials only (a check after the last sweep).
//
// Bound by the latency of its loads (1.5 M faces at 96x80x64 in 7.4 us, where
// a launch per component took 3 x 5.2 us and every fifth sweep 3 x 7.9 us more; of
// which about 20 MB are read for the fluid rows, from cache): the row code
// decides only whether a thread reads at all, and the six neighbours and b of
// all its rows are then loaded together instead of one after another under the
// code's bits.
template <bool CHECK, bool WRITE>
__global__ __launch_bounds__(kBlock) void k_diff_sweep(DiffGrid D, const uint16_t* __restrict__ code,
                                                       const double* __restrict__ b, const double* __restrict__ xo,
                                                       double* __restrict__ xn, double cx, double cy, double cz,
                                                       int it, int snap, double* __restrict__ xs,
                                                       DiffState* __restrict__ st, double* __restrict__ part) {
#pragma clang fp contract(off)
    const int C = diff_component(D, blockIdx.x);
    const int64_t f0 = diff_first(D, C) + threadIdx.x;
    const int64_t nf = D.nf[C], sy = D.nx[C], sz = sy * D.ny[C], last = nf - 1;
    code += D.off[C];
    b += D.off[C];
    xo += D.off[C];
    xn += D.off[C];
    xs += D.off[C];
    uint16_t cd[kDiffPer];
#pragma unroll
    for (int t = 0; t < kDiffPer; ++t) {
        const int64_t f = f0 + t * kBlock;
        cd[t] = f < nf ? code[f] : (uint16_t)0;
    }
    if (it >= st[C].end) return;  // uniform: x_end stays in its buffer
    const double c[3] = {cx, cy, cz};
    double bb[kDiffPer], xc[kDiffPer], xp[kDiffPer], nb[kDiffPer][6];
#pragma unroll
    for (int t = 0; t < kDiffPer; ++t) {
        if (!(cd[t] & kFluidBit)) continue;
        const int64_t f = f0 + t * kBlock;
        bb[t] = b[f];
        nb[t][0] = xo[f > 0 ? f - 1 : 0];
        nb[t][1] = xo[f < last ? f + 1 : last];
        nb[t][2] = xo[f >= sy ? f - sy : 0];
        nb[t][3] = xo[f + sy <= last ? f + sy : last];
        nb[t][4] = xo[f >= sz ? f - sz : 0];
        nb[t][5] = xo[f + sz <= last ? f + sz : last];
        if (CHECK) xc[t] = xo[f];
        if (CHECK && WRITE) xp[t] = xs[f];
    }
    double v[1] = {0.0};
    int changed = 0;
#pragma unroll
    for (int t = 0; t < kDiffPer; ++t) {
        if (!(cd[t] & kFluidBit)) continue;  // b - x is 0 on an identity row
        const double off = diff_offdiag(cd[t], c, nb[t]);
        const double center = diff_center(cd[t], c);
        if (WRITE) xn[f0 + t * kBlock] = (bb[t] - off) / center;
        if (CHECK) {
            const double r = (bb[t] - center * xc[t]) - off;
            v[0] += r * r;
            if (WRITE) {
                changed |= __double_as_longlong(xc[t]) != __double_as_longlong(xp[t]);
                if (snap) xs[f0 + t * kBlock] = xc[t];
            }
        }
    }
    if (CHECK) {
        if (WRITE) {
            changed = __syncthreads_or(changed);
            if (changed && threadIdx.x == 0) st[C].changed = 1;  // every writer writes the same
        }
        write_partials<1>(v, part);
    }
}

// One workgroup per component: check number q (q >= 1, after sweep
// j = q * interval, on the state x_{j+1}), from the partials that sweep j + 1
// left.
//
// A state that equals the snapshot L <= kDiffRing checks before it, bit for
// bit, starts the same L * interval sweeps again: all later states and checks
// are ones already seen, none of which met the tolerance, so the solve's last
// state is at most L * interval sweeps away and its last residual is known.
// Rounding brings every solve there (the sweep is a contraction; cycles of 2
// and 4 sweeps seen), and the reference's tolerance of 1e-14 on an absolute
// norm is below what rounding leaves on all but tiny grids: at 96x80x64 the
// states repeat from sweep 155 of the 1000.
__global__ __launch_bounds__(kBlock) void k_diff_check(DiffGrid D, const double* __restrict__ part, int q,
                                                       int interval, int compared, DiffState* __restrict__ st) {
    const int C = blockIdx.x;
    DiffState* S = st + C;
    if (D.blk[C + 1] == D.blk[C] || S->end != kDiffOpen) return;
    double t[1];
    sum_partials<1>(part + D.blk[C], (int)(D.blk[C + 1] - D.blk[C]), t);
    if (threadIdx.x != 0) return;
    const int k = q * interval + 1;  // the state checked
    if (S->nonfinite) t[0] = __builtin_nan("");
    S->rr = t[0];
    S->ring[q % kDiffRing] = t[0];
    if (sqrt(t[0]) < S->tol) {
        S->converged = 1;
        S->it = k;
        S->end = k;
        return;
    }
    if (compared && !S->changed) {
        const int L = (q - 1) % kDiffRing + 1;  // checks since the snapshot
        const int last = (S->max_it - 1) / interval;
        S->rr = S->ring[(q - ((q - last) % L + L) % L) % kDiffRing];
        S->end = k + (S->max_it - k) % (L * interval);
    }
    S->changed = 0;
}

__global__ __launch_bounds__(kBlock) void k_diff_store(DiffGrid D, const double* __restrict__ x0,
                                                       const double* __restrict__ x1, int odd, FaceSet u) {
    const int C = diff_component(D, blockIdx.x);
    const double* __restrict__ x = ((odd >> C) & 1 ? x1 : x0) + D.off[C];
    const int64_t f0 = diff_first(D, C) + threadIdx.x;
#pragma unroll
    for (int t = 0; t < kDiffPer; ++t) {
        const int64_t f = f0 + t * kBlock;
        if (f < D.nf[C]) u.a[C][f] = (float)x[f];  // output->x/y/z(i, j, k) = _system.x(i, j, k)
    }
}

// Up to here the three components are solved side by side, which saves two
// launches' latency a sweep; above, a sweep of one component fills the chip and
// its iterates stay in the last cache better, so they are solved one after
// another, in buffers of the largest only (34 bytes a face of one component,
// not of three).  100 sweeps of half full tanks, side by side / one after
// another: 96x80x64 1.01 / 2.02 ms, 128^3 2.44 / 3.48, 160^3 4.11 / 5.04, 192^3
// 9.03 / 7.61, 256^3 20.9 / 20.8.
constexpr int64_t kDiffTogether = 1 << 22;  // faces of the largest component

int64_t diff_faces(const Geom& g) {
    return std::max(face_count(g, 0), std::max(face_count(g, 1), face_count(g, 2)));
}

// Components from c0 up to c1.
DiffGrid diff_grid(const Geom& g, int c0, int c1) {
    DiffGrid D{};
    int64_t off = 0;
    for (int c = 0; c < 3; ++c) {
        D.blk[c + 1] = D.blk[c];
        if (c < c0 || c >= c1) continue;
        D.nx[c] = face_dim(g, c, 0);
        D.ny[c] = face_dim(g, c, 1);
        D.nf[c] = face_count(g, c);
        D.off[c] = off;
        off += (D.nf[c] + 15) / 16 * 16;
        D.blk[c + 1] += pad_blocks((D.nf[c] + kBlock * kDiffPer - 1) / (kBlock * kDiffPer));
    }
    return D;
}

}  // namespace

hipError_t diffusion_alloc(fe_scene* s) {
    if (s->dstate_host) return hipSuccess;
    const bool together = diff_faces(s->g) <= kDiffTogether;
    const DiffGrid D = diff_grid(s->g, 0, 3);
    const int64_t n = together ? D.off[2] + D.nf[2] : diff_faces(s->g);
    hipError_t e;
    for (int b = 0; b < 2; ++b)
        if ((e = hipMalloc((void**)&s->dx[b], sizeof(double) * n)) != hipSuccess) return e;
    if ((e = hipMalloc((void**)&s->dcode, sizeof(uint16_t) * n)) != hipSuccess) return e;
    if ((e = hipMalloc((void**)&s->db, sizeof(double) * n)) != hipSuccess) return e;
    if (hipMalloc((void**)&s->dsnap, sizeof(double) * n) != hipSuccess) {
        (void)hipGetLastError();  // without it repeated states go unseen, and every sweep is made
        s->dsnap = nullptr;
    }
    if ((e = hipMalloc((void**)&s->dpart, sizeof(double) * D.blk[3])) != hipSuccess) return e;
    if ((e = hipMalloc((void**)&s->dstate, sizeof(DiffState) * 3)) != hipSuccess) return e;
    for (int c = 0; c < 3; ++c)
        if ((e = hipMalloc((void**)&s->dmark[c], face_count(s->g, c))) != hipSuccess) return e;
    return hipHostMalloc((void**)&s->dstate_host, sizeof(DiffState) * 3, hipHostMallocDefault);
}

void diffusion_free(fe_scene* s) {
    auto release = [](auto*& p) {
        if (p) (void)hipFree(p);
        p = nullptr;
    };
    for (int b = 0; b < 2; ++b) release(s->dx[b]);
    release(s->dcode);
    release(s->db);
    release(s->dsnap);
    release(s->dpart);
    release(s->dstate);
    for (int c = 0; c < 3; ++c) release(s->dmark[c]);
    if (s->dstate_host) (void)hipHostFree(s->dstate_host);
    s->dstate_host = nullptr;
}

// The solves of components c0 up to c1, side by side on the scene's stream, in
// batches of sweeps with one host read of the stopping flags per batch.  The
// check after sweep j is taken from sweep j + 1, which reads the same rows: it
// leaves x_{j+1} in its input buffer, so a stop found there loses nothing.
static hipError_t solve_components(fe_scene* s, const double (&c)[3], const fe_solver_desc* d, int c0, int c1) {
    const Geom& g = s->g;
    hipError_t e;
    const DiffGrid D = diff_grid(g, c0, c1);
    const dim3 grid((unsigned)D.blk[3]), block(kBlock);
    const FaceSet u{{s->u[0], s->u[1], s->u[2]}};
    DiffState init{};
    init.tol = d->tolerance;
    init.max_it = d->max_iterations;
    init.it = d->max_iterations;
    init.end = kDiffOpen;
    hipLaunchKernelGGL(k_diff_markers, grid, block, 0, s->stream, g, D, (const double*)s->sdf,
                       (const double*)(s->has_collider ? s->csdf : nullptr), s->dmark[0], s->dmark[1], s->dmark[2],
                       s->dstate, init);
    hipLaunchKernelGGL(k_diff_build, grid, block, 0, s->stream, D, u, (const uint8_t*)s->dmark[0],
                       (const uint8_t*)s->dmark[1], (const uint8_t*)s->dmark[2], s->dcode, s->dx[0], s->dx[1], s->db,
                       c[0], c[1], c[2], s->dstate);
    constexpr int kBatch = 50;  // sweeps between host reads of the stopping flags
    const int interval = d->check_interval;
    auto checked = [&](int j) { return interval > 0 && j > 0 && j % interval == 0; };  // after sweep j
    double* const snapshot = s->dsnap ? s->dsnap : s->db;  // without one: read, for nothing, and never written
    auto sweep = [&](auto kernel, int it, int snap) {
        hipLaunchKernelGGL(kernel, grid, block, 0, s->stream, D, (const uint16_t*)s->dcode, (const double*)s->db,
                           (const double*)s->dx[it & 1], s->dx[(it + 1) & 1], c[0], c[1], c[2], it, snap, snapshot,
                           s->dstate, s->dpart);
    };
    auto check = [&](int q, int compared) {
        hipLaunchKernelGGL(k_diff_check, dim3(3), block, 0, s->stream, D, (const double*)s->dpart, q, interval,
                           compared, s->dstate);
    };
    for (int comp = c0; comp < c1; ++comp) s->dstate_host[comp] = init;
    int it = 0;
    bool done = false;
    while (it < d->max_iterations && !done) {
        const int end = std::min(d->max_iterations, it + kBatch);
        for (; it < end; ++it) {
            if (checked(it - 1)) {
                const int q = (it - 1) / interval;
                sweep(k_diff_sweep<true, true>, it, s->dsnap && q % kDiffRing == 0);
                check(q, s->dsnap && q > kDiffRing);
            } else {
                sweep(k_diff_sweep<false, true>, it, 0);
            }
        }
        if (it == d->max_iterations && checked(it - 1)) {
            sweep(k_diff_sweep<true, false>, it, 0);
            check((it - 1) / interval, 0);
        }
        if ((e = hipGetLastError()) != hipSuccess) return e;
        if ((e = hipMemcpyAsync(s->dstate_host, s->dstate, sizeof(DiffState) * 3, hipMemcpyDeviceToHost,
                                s->stream)) != hipSuccess)
            return e;
        if ((e = hipStreamSynchronize(s->stream)) != hipSuccess) return e;
        done = true;
        for (int comp = c0; comp < c1; ++comp) done = done && s->dstate_host[comp].end <= it;
    }
    int odd = 0;
    for (int comp = c0; comp < c1; ++comp) {
        const DiffState& h = s->dstate_host[comp];
        odd |= (std::min(h.end, d->max_iterations) & 1) << comp;
        fe_solve_stats& st = s->diff_stats[comp];
        st = fe_solve_stats{};
        st.iterations = h.it;
        st.converged = h.converged;
        st.abs_residual = interval > 0 && h.it > interval ? std::sqrt(h.rr) : -1.0;
        st.rel_residual = -1.0;
        st.ms = 0.0;
    }
    hipLaunchKernelGGL(k_diff_store, grid, block, 0, s->stream, D, (const double*)s->dx[0], (const double*)s->dx[1],
                       odd, u);
    return hipGetLastError();
}

// ComputeDiffusion without its trailing ApplyBoundryCondition: the three
// component solves (each reads and writes its own component only).
hipError_t launch_diffusion(fe_scene* s, double dt, const fe_solver_desc* d) {
    const Geom& g = s->g;
    const double nu = s->desc.viscosity;
    const double c[3] = {(dt * nu) / (g.hd[0] * g.hd[0]), (dt * nu) / (g.hd[1] * g.hd[1]),
                         (dt * nu) / (g.hd[2] * g.hd[2])};
    hipError_t e;
    if ((e = diffusion_alloc(s)) != hipSuccess) {
        diffusion_free(s);
        return e;
    }
    if (diff_faces(g) <= kDiffTogether) return solve_components(s, c, d, 0, 3);
    for (int comp = 0; comp < 3; ++comp)
        if ((e = solve_components(s, c, d, comp, comp + 1)) != hipSuccess) return e;
    return hipSuccess;
}

}  // namespace fe
