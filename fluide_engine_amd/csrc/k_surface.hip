// k_surface.hip -- fluid surface: MarchingCubesSolver::BuildSurface
// (src/3d/marching_cubes_solver.cpp:25-51) on the fluid SDF.
//
// Nodes are the SDF samples (cell centres, origin o + h/2); a node is inside
// when its value is <= 0.  The reference builds the mesh in four parts: the
// cubes between nodes (CalculateXYZMeshPart) and caps on the six boundary
// node planes (CalculateXY/YZ/XZMeshPart).  Here:
//   * cubes, on the device: every crossed node edge carries one vertex (the
//     reference's edge-keyed vertex map); vertices are numbered by a scan over
//     the crossed-edge flags (x edges, then y, then z), triangles by a scan
//     over per-cube counts, so the output is deterministic and needs no map;
//   * caps, on the device too: every square of the six boundary node planes
//     knows from its case and its place which of its corners and crossings no
//     earlier square of the plane has met, so a scan over the squares numbers
//     the vertices in the order of the reference's loops (one vertex set per
//     plane, its separate vertex maps).  On the host, from a copy of the planes,
//     that took 0.7 ms of the 0.95 ms of a 128x96x112 build; with the SDF's
//     upload and the mesh's download the whole went from 1.26 to 0.70 ms.
// Vertex position: linear zero of the SDF along the edge, alpha =
// |phi0| / (|phi0| + |phi1|) clamped to [1e-6, 0.999999]; normal: the same
// interpolation of the central-difference gradients at the two nodes,
// normalised (MarchingCubesSolver::Gradient and SafeNormalize).  The case
// tables come from fe_mc_rule.hpp (one face rule for cubes and caps, so the
// surface is closed); the reference's own table can leave holes on faces with
// diagonally opposite inside nodes.
#include <algorithm>
#include <cmath>
#include <vector>

#include "fe_kernels.hpp"
#include "fe_mc_rule.hpp"

namespace fe {

namespace {

struct NodeGrid {
    int n[3];
    double o[3], h[3], ih[3];  // node origin o + h/2, spacing, 1/h
    int64_t ne[3];             // edges per axis
};

__device__ __host__ inline int64_t node_index(const NodeGrid& G, int i, int j, int k) {
    return (int64_t)i + (int64_t)G.n[0] * ((int64_t)j + (int64_t)G.n[1] * k);
}

// Edge e of the concatenated x, y, z edge lists -> axis and low node.
__device__ inline void edge_node(const NodeGrid& G, int64_t e, int& axis, int& i, int& j, int& k) {
    axis = e < G.ne[0] ? 0 : (e < G.ne[0] + G.ne[1] ? 1 : 2);
    const int64_t l = e - (axis == 0 ? 0 : (axis == 1 ? G.ne[0] : G.ne[0] + G.ne[1]));
    const int dx = G.n[0] - (axis == 0), dy = G.n[1] - (axis == 1);
    split_index(l, dx, dy, i, j, k);
}

__device__ inline int64_t edge_id(const NodeGrid& G, int axis, int i, int j, int k) {
    if (axis == 0) return (int64_t)i + (int64_t)(G.n[0] - 1) * ((int64_t)j + (int64_t)G.n[1] * k);
    if (axis == 1) return G.ne[0] + (int64_t)i + (int64_t)G.n[0] * ((int64_t)j + (int64_t)(G.n[1] - 1) * k);
    return G.ne[0] + G.ne[1] + (int64_t)i + (int64_t)G.n[0] * ((int64_t)j + (int64_t)G.n[1] * k);
}

// MarchingCubesSolver::Gradient (src/3d/marching_cubes_solver.cpp:116-160).
__device__ inline void node_gradient(const NodeGrid& G, const double* __restrict__ sdf, int i, int j, int k,
                                     double g[3]) {
#pragma clang fp contract(off)
    const int idx[3] = {i, j, k};
    for (int a = 0; a < 3; ++a) {
        int p[3] = {i, j, k}, m[3] = {i, j, k};
        if (idx[a] > G.n[a] - 2) {
            p[a] = idx[a];
            m[a] = idx[a] - 1;
        } else if (idx[a] == 0) {
            p[a] = 1;
            m[a] = 0;
        } else {
            p[a] = idx[a] + 1;
            m[a] = idx[a] - 1;
        }
        g[a] = 0.5 * G.ih[a] * (sdf[node_index(G, p[0], p[1], p[2])] - sdf[node_index(G, m[0], m[1], m[2])]);
    }
}

__global__ __launch_bounds__(kBlock) void k_mc_edges(NodeGrid G, const double* __restrict__ sdf,
                                                     int32_t* __restrict__ flag, int64_t nedges) {
    const int64_t e = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (e >= nedges) return;
    int axis, i, j, k;
    edge_node(G, e, axis, i, j, k);
    const double a = sdf[node_index(G, i, j, k)];
    const double b = sdf[node_index(G, i + (axis == 0), j + (axis == 1), k + (axis == 2))];
    flag[e] = (a <= 0.0) != (b <= 0.0) ? 1 : 0;
}

__device__ inline int cube_case(const NodeGrid& G, const double* __restrict__ sdf, int i, int j, int k) {
    int cs = 0;
#pragma unroll
    for (int c = 0; c < 8; ++c)
        if (sdf[node_index(G, i + (c & 1), j + ((c >> 1) & 1), k + ((c >> 2) & 1))] <= 0.0) cs |= 1 << c;
    return cs;
}

__global__ __launch_bounds__(kBlock) void k_mc_count(NodeGrid G, const double* __restrict__ sdf,
                                                     const McTables* __restrict__ T, int32_t* __restrict__ cnt,
                                                     int64_t ncubes) {
    const int64_t c = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (c >= ncubes) return;
    int i, j, k;
    split_index(c, G.n[0] - 1, G.n[1] - 1, i, j, k);
    cnt[c] = T->ntri[cube_case(G, sdf, i, j, k)];
}

__global__ __launch_bounds__(kBlock) void k_mc_vertices(NodeGrid G, const double* __restrict__ sdf,
                                                        const int32_t* __restrict__ vid, double* __restrict__ pos,
                                                        double* __restrict__ nrm, int64_t nedges) {
#pragma clang fp contract(off)
    const int64_t e = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (e >= nedges) return;
    const int32_t v = vid[e];
    if (vid[e + 1] == v) return;  // not crossed
    int axis, i, j, k;
    edge_node(G, e, axis, i, j, k);
    const int i1 = i + (axis == 0), j1 = j + (axis == 1), k1 = k + (axis == 2);
    const double phi0 = sdf[node_index(G, i, j, k)], phi1 = sdf[node_index(G, i1, j1, k1)];
    // DistanceToZeroLevelSet (:591-601) and the clamps of SolveSingleCube (:263-268)
    double alpha = fabs(phi0) + fabs(phi1) > 0.000000001 ? fabs(phi0) / (fabs(phi0) + fabs(phi1)) : 0.5;
    alpha = alpha < 0.000001 ? 0.000001 : (alpha > 0.999999 ? 0.999999 : alpha);
    // The reference's edges run from the lower to the higher node
    // (_edgeConnection with its corner order) and its end points are
    // BoundingBox3D::Corner of the first cube in its i, j, k loop order that
    // holds the edge (the vertex map keeps that cube's vertex): the cube at
    // node - 1 on the two other axes, clamped at 0.
    const int a0[3] = {i, j, k};
    double g0[3], g1[3], nv[3];
    node_gradient(G, sdf, i, j, k, g0);
    node_gradient(G, sdf, i1, j1, k1, g1);
    for (int a = 0; a < 3; ++a) {
        const int cube = a == axis ? a0[a] : (a0[a] > 0 ? a0[a] - 1 : 0);
        const int off0 = a0[a] - cube, off1 = off0 + (a == axis);
        const double oc = G.o[a] + cube * G.h[a];  // GridIndexToPosition of the cube
        const double p0 = (G.h[a] * (off0 ? 0.5 : -0.5) + oc) + 0.5 * G.h[a];
        const double p1 = (G.h[a] * (off1 ? 0.5 : -0.5) + oc) + 0.5 * G.h[a];
        pos[3 * (int64_t)v + a] = (1.0 - alpha) * p0 + alpha * p1;
        nv[a] = (1.0 - alpha) * g0[a] + alpha * g1[a];
    }
    const double l2 = nv[0] * nv[0] + nv[1] * nv[1] + nv[2] * nv[2];
    if (l2 > 0.0) {  // SafeNormalize: Vector3::Normalize divides by the length
        const double l = sqrt(l2);
        for (int a = 0; a < 3; ++a) nv[a] = nv[a] / l;
    }
    for (int a = 0; a < 3; ++a) nrm[3 * (int64_t)v + a] = nv[a];
}

__global__ __launch_bounds__(kBlock) void k_mc_emit(NodeGrid G, const double* __restrict__ sdf,
                                                    const McTables* __restrict__ T, const int32_t* __restrict__ toff,
                                                    const int32_t* __restrict__ vid, int32_t* __restrict__ tri,
                                                    int64_t ncubes) {
    const int64_t c = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (c >= ncubes) return;
    const int32_t t0 = toff[c], nt = toff[c + 1] - t0;
    if (nt == 0) return;
    int i, j, k;
    split_index(c, G.n[0] - 1, G.n[1] - 1, i, j, k);
    const int cs = cube_case(G, sdf, i, j, k);
    for (int t = 0; t < nt; ++t)
        for (int q = 0; q < 3; ++q) {
            const int e = T->tri[cs][3 * t + q];
            const int axis = e >> 2, u = e & 1, w = (e >> 1) & 1;
            int64_t ge;
            if (axis == 0) ge = edge_id(G, 0, i, j + u, k + w);
            else if (axis == 1) ge = edge_id(G, 1, i + u, j, k + w);
            else ge = edge_id(G, 2, i + u, j + w, k);
            tri[3 * (int64_t)(t0 + t) + q] = vid[ge];
        }
}

inline dim3 grid_of(int64_t n) { return dim3((unsigned)((n + kBlock - 1) / kBlock)); }

NodeGrid node_grid(const Geom& g) {
    NodeGrid G;
    for (int a = 0; a < 3; ++a) {
        G.n[a] = g.n[a];
        G.h[a] = g.hd[a];
        G.ih[a] = 1.0 / g.hd[a];
        G.o[a] = g.od[a] + g.hd[a] / 2.0;  // the fluid SDF grid origin (src/hybrid_simulator.cpp:13-15)
    }
    G.ne[0] = (int64_t)(G.n[0] - 1) * G.n[1] * G.n[2];
    G.ne[1] = (int64_t)G.n[0] * (G.n[1] - 1) * G.n[2];
    G.ne[2] = (int64_t)G.n[0] * G.n[1] * (G.n[2] - 1);
    return G;
}

template <typename T>
hipError_t grow(T** p, int64_t* cap, int64_t need) {
    if (*cap >= need) return hipSuccess;
    if (*p) (void)hipFree(*p);
    *p = nullptr;
    *cap = 0;
    const int64_t n = std::max<int64_t>(need + need / 4, 1024);
    hipError_t e = hipMalloc((void**)p, sizeof(T) * n);
    if (e == hipSuccess) *cap = n;
    return e;
}

// ---------------------------------------------------------------------------
// Caps of the boundary planes (SolveXY / SolveYZ / SolveXZ with
// SolveSingleSquare, :272-589): squares of the plane's nodes, inside nodes and
// crossing points as vertices, the plane's outward axis normal for every
// vertex.  Plane p = 2 * axis + side; u, v the other axes, lower first.  The
// loops run v outer, u inner on every plane (z planes j, i; x planes k, j; y
// planes k, i).
// ---------------------------------------------------------------------------
constexpr int kCapOrder[6] = {4, 5, 0, 1, 2, 3};  // XY (z planes), YZ (x planes), XZ (y planes), as the reference

// A square's case: its slots in the order in which its triangles first name
// them (0-3 a corner, 4-7 the crossing on the edge from corner slot-4 to the
// next), and the triangles.
struct CapCase {
    int8_t nslot = 0, slot[8] = {};
    int8_t ntri = 0, tri[12] = {};
};
struct CapTables {
    int8_t corner[6][4][2];  // (du, dv) of the corners
    CapCase c[6][16];        // by plane and inside corners
};

// FE_SURFACE_CLOSED: the face rule of fe_mc_rule.hpp, corners in the (u, v)
// cyclic order, which turns counter-clockwise about u x v: +x for x planes, -y
// for y planes, +z for z planes.
CapTables make_cap_tables() {
    CapTables T;
    static const int8_t cyc[4][2] = {{0, 0}, {1, 0}, {1, 1}, {0, 1}};
    for (int p = 0; p < 6; ++p) {
        const double outward = p & 1 ? 1.0 : -1.0, natural = (p >> 1) == 1 ? -1.0 : 1.0;
        for (int t = 0; t < 4; ++t)
            for (int a = 0; a < 2; ++a) T.corner[p][t][a] = cyc[t][a];
        for (int cs = 0; cs < 16; ++cs) {
            CapCase c;
            bool in[4];
            for (int t = 0; t < 4; ++t) in[t] = (cs >> t) & 1;
            int poly[2][5], len[2];
            const int np = mc_square_caps(in, poly, len);
            for (int q = 0; q < np; ++q) {
                for (int s = 0; s < len[q]; ++s) c.slot[c.nslot++] = (int8_t)poly[q][s];
                for (int s = 1; s + 1 < len[q]; ++s) {
                    const bool flip = natural != outward;
                    const int f[3] = {poly[q][0], poly[q][flip ? s + 1 : s], poly[q][flip ? s : s + 1]};
                    for (int r = 0; r < 3; ++r) c.tri[3 * c.ntri + r] = (int8_t)f[r];
                    ++c.ntri;
                }
            }
            T.c[p][cs] = c;
        }
    }
    return T;
}

// FE_SURFACE_REFERENCE: the reference's corner order per plane and its square
// table (kMcRefSquare).
CapTables make_cap_tables_reference() {
    static const int8_t kRefSq[6][4][2] = {
        {{0, 0}, {0, 1}, {1, 1}, {1, 0}},  // left  (u = y, v = z): (j,k) (j,k+1) (j+1,k+1) (j+1,k)
        {{0, 1}, {0, 0}, {1, 0}, {1, 1}},  // right: (j,k+1) (j,k) (j+1,k) (j+1,k+1)
        {{0, 0}, {1, 0}, {1, 1}, {0, 1}},  // down  (u = x, v = z): (i,k) (i+1,k) (i+1,k+1) (i,k+1)
        {{1, 0}, {0, 0}, {0, 1}, {1, 1}},  // up:    (i+1,k) (i,k) (i,k+1) (i+1,k+1)
        {{1, 0}, {0, 0}, {0, 1}, {1, 1}},  // back  (u = x, v = y): (i+1,j) (i,j) (i,j+1) (i+1,j+1)
        {{0, 0}, {1, 0}, {1, 1}, {0, 1}},  // front: (i,j) (i+1,j) (i+1,j+1) (i,j+1)
    };
    CapTables T;
    for (int p = 0; p < 6; ++p) {
        for (int t = 0; t < 4; ++t)
            for (int a = 0; a < 2; ++a) T.corner[p][t][a] = kRefSq[p][t][a];
        for (int cs = 0; cs < 16; ++cs) {
            CapCase c;
            bool met[8] = {};
            for (const char* q = kMcRefSquare[cs]; *q; ++q) {
                const int8_t slot = (int8_t)mc_hex(*q);
                if (!met[slot]) c.slot[c.nslot++] = slot;
                met[slot] = true;
                c.tri[c.ntri++] = slot;
            }
            c.ntri /= 3;
            T.c[p][cs] = c;
        }
    }
    return T;
}

struct CapGrid {
    int64_t first[7];  // the planes' first squares, in the loops' plane order
    int64_t key[6];    // and their first vertex keys: nodes, then u edges, then v edges
};

// What a square knows of itself.
struct CapSquare {
    int p, axis, u, v, iu, jv, cs;
    double phi[4];
};

__device__ inline bool cap_square(const NodeGrid& G, const CapGrid& Q, const CapTables* __restrict__ T,
                                  const double* __restrict__ sdf, int64_t s, CapSquare& S) {
    if (s >= Q.first[6]) return false;
    int q = 0;
    while (s >= Q.first[q + 1]) ++q;
    S.p = (q + 4) % 6;  // kCapOrder
    S.axis = S.p >> 1;
    S.u = S.axis == 0 ? 1 : 0;
    S.v = S.axis == 2 ? 1 : 2;
    const int64_t r = s - Q.first[q], w = G.n[S.u] - 1;
    S.jv = (int)(r / w);
    S.iu = (int)(r - S.jv * w);
    S.cs = 0;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const int cu = S.iu + T->corner[S.p][t][0], cv = S.jv + T->corner[S.p][t][1];
        const int fixed = S.p & 1 ? G.n[S.axis] - 1 : 0;
        const int i = S.axis == 0 ? fixed : cu, j = S.axis == 1 ? fixed : (S.axis == 0 ? cu : cv),
                  k = S.axis == 2 ? fixed : cv;
        S.phi[t] = sdf[node_index(G, i, j, k)];
        if (S.phi[t] <= 0.0) S.cs |= 1 << t;
    }
    return true;
}

// The vertex of a slot: its key in the plane, and whether this square is the
// first to meet it.  Every square with an inside corner or a crossing names
// it, so the first is the lowest in the loops' order: the one before it in v
// (and, for what does not lie along u, before it in u) where there is one.
__device__ inline int64_t cap_key(const NodeGrid& G, const CapTables* __restrict__ T, const CapSquare& S, int slot,
                                  bool& first) {
    const int64_t nu = G.n[S.u], nv = G.n[S.v];
    const int t = slot & 3;
    int cu = S.iu + T->corner[S.p][t][0], cv = S.jv + T->corner[S.p][t][1];
    if (slot < 4) {
        first = S.iu == max(cu - 1, 0) && S.jv == max(cv - 1, 0);
        return cu + nu * cv;
    }
    const int t1 = (t + 1) & 3, eu = S.iu + T->corner[S.p][t1][0], ev = S.jv + T->corner[S.p][t1][1];
    const bool along_u = cv == ev;
    cu = min(cu, eu);
    cv = min(cv, ev);
    if (along_u) {
        first = S.jv == max(cv - 1, 0);
        return nu * nv + cu + (nu - 1) * cv;
    }
    first = S.iu == max(cu - 1, 0);
    return nu * nv + (nu - 1) * nv + cu + nu * cv;
}

__global__ __launch_bounds__(kBlock) void k_cap_count(NodeGrid G, CapGrid Q, const CapTables* __restrict__ T,
                                                      const double* __restrict__ sdf, int32_t* __restrict__ nvert,
                                                      int32_t* __restrict__ ntri) {
    const int64_t s = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    CapSquare S;
    if (!cap_square(G, Q, T, sdf, s, S)) return;
    const CapCase& c = T->c[S.p][S.cs];
    int own = 0;
    for (int q = 0; q < c.nslot; ++q) {
        bool first;
        (void)cap_key(G, T, S, c.slot[q], first);
        own += first;
    }
    nvert[s] = own;
    ntri[s] = c.ntri;
}

// The vertices a square meets first, from vbase + voff[s] on; their indices by
// key for the triangles.  CLOSED places a crossing from its lower node, the
// reference from the corner its square's edge starts at, with SolveSingleSquare's
// alpha and clamps (:536-549) either way.
__global__ __launch_bounds__(kBlock) void k_cap_vertices(NodeGrid G, CapGrid Q, const CapTables* __restrict__ T,
                                                         const double* __restrict__ sdf,
                                                         const int32_t* __restrict__ voff, int64_t vbase, int closed,
                                                         int32_t* __restrict__ id, double* __restrict__ pos,
                                                         double* __restrict__ nrm) {
#pragma clang fp contract(off)
    const int64_t s = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    CapSquare S;
    if (!cap_square(G, Q, T, sdf, s, S)) return;
    const CapCase& c = T->c[S.p][S.cs];
    int64_t vi = vbase + voff[s];
    for (int q = 0; q < c.nslot; ++q) {
        const int slot = c.slot[q];
        bool first;
        const int64_t key = cap_key(G, T, S, slot, first);
        if (!first) continue;
        auto node = [&](int t, double out[3]) {
            const int cu = S.iu + T->corner[S.p][t][0], cv = S.jv + T->corner[S.p][t][1];
            const int fixed = S.p & 1 ? G.n[S.axis] - 1 : 0;
            const int idx[3] = {S.axis == 0 ? fixed : cu, S.axis == 1 ? fixed : (S.axis == 0 ? cu : cv),
                                S.axis == 2 ? fixed : cv};
            for (int a = 0; a < 3; ++a) out[a] = G.o[a] + idx[a] * G.h[a];
        };
        double w[3];
        if (slot < 4) {
            node(slot, w);
        } else {
            int t = slot - 4, t1 = (t + 1) & 3;
            const int sum = T->corner[S.p][t][0] + T->corner[S.p][t][1],
                      sum1 = T->corner[S.p][t1][0] + T->corner[S.p][t1][1];
            if (closed && sum > sum1) {
                const int h = t;
                t = t1;
                t1 = h;
            }
            const double f0 = fabs(S.phi[t]), f1 = fabs(S.phi[t1]);
            double alpha = f0 + f1 > 1e-12 ? f0 / (f0 + f1) : 0.5;
            if (alpha < 0.000001f) alpha = 0.000001f;
            if (alpha > 0.999999f) alpha = 0.999999f;
            double p0[3], p1[3];
            node(t, p0);
            node(t1, p1);
            for (int a = 0; a < 3; ++a) w[a] = (1.0 - alpha) * p0[a] + alpha * p1[a];
        }
        id[Q.key[S.p] + key] = (int32_t)vi;
        for (int a = 0; a < 3; ++a) {
            pos[3 * vi + a] = w[a];
            nrm[3 * vi + a] = a == S.axis ? (S.p & 1 ? 1.0 : -1.0) : 0.0;
        }
        ++vi;
    }
}

__global__ __launch_bounds__(kBlock) void k_cap_triangles(NodeGrid G, CapGrid Q, const CapTables* __restrict__ T,
                                                          const double* __restrict__ sdf,
                                                          const int32_t* __restrict__ toff, int64_t tbase,
                                                          const int32_t* __restrict__ id, int32_t* __restrict__ tri) {
    const int64_t s = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    CapSquare S;
    if (!cap_square(G, Q, T, sdf, s, S)) return;
    const CapCase& c = T->c[S.p][S.cs];
    const int64_t t0 = 3 * (tbase + toff[s]);
    for (int q = 0; q < 3 * c.ntri; ++q) {
        bool first;
        tri[t0 + q] = id[Q.key[S.p] + cap_key(G, T, S, c.tri[q], first)];
    }
}

CapGrid cap_grid(const NodeGrid& G, int64_t* keys) {
    CapGrid Q{};
    int64_t n = 0;
    for (int q = 0; q < 6; ++q) {
        const int p = kCapOrder[q], axis = p >> 1, u = axis == 0 ? 1 : 0, v = axis == 2 ? 1 : 2;
        const int64_t nu = G.n[u], nv = G.n[v];
        Q.first[q + 1] = Q.first[q] + (nu - 1) * (nv - 1);
        Q.key[p] = n;
        n += nu * nv + (nu - 1) * nv + nu * (nv - 1);
    }
    *keys = n;
    return Q;
}

// The surface SDF with a collider: the fluid SDF, replaced by minus the
// collider SDF where both are negative (GetSurface, src/hybrid_simulator.cpp:29-37).
__global__ __launch_bounds__(kBlock) void k_mc_combine(const double* __restrict__ sdf,
                                                       const double* __restrict__ csdf, double* __restrict__ out,
                                                       int64_t n) {
    const int64_t c = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (c >= n) return;
    const double a = sdf[c], b = csdf[c];
    out[c] = (a < 0 && b < 0) ? -b : a;
}

}  // namespace

void surface_free(fe_scene* s) {
    McState& m = s->mc;
    auto F = [](auto*& p) {
        if (p) (void)hipFree(p);
        p = nullptr;
    };
    F(m.flag);
    F(m.vid);
    F(m.cnt);
    F(m.toff);
    F(m.sums);
    F(m.tables);
    F(m.tables_ref);
    F(m.caps);
    F(m.caps_ref);
    F(m.capv);
    F(m.capt);
    F(m.capvo);
    F(m.capto);
    F(m.capid);
    F(m.pos);
    F(m.nrm);
    F(m.tri);
    F(m.comb);
    m = McState{};
}

hipError_t surface_build(fe_scene* s) {
    McState& m = s->mc;
    const NodeGrid G = node_grid(s->g);
    const int64_t nedges = G.ne[0] + G.ne[1] + G.ne[2];
    const int64_t ncubes = (int64_t)(G.n[0] - 1) * (G.n[1] - 1) * (G.n[2] - 1);
    int64_t keys = 0;
    const CapGrid Q = cap_grid(G, &keys);
    const int64_t squares = Q.first[6];
    hipError_t e;
    const bool ref = s->surface_mode == FE_SURFACE_REFERENCE;
    if (!m.capid) {  // the last to be allocated
        surface_free(s);
        const McTables host = make_mc_tables();
        if ((e = hipMalloc((void**)&m.tables, sizeof(McTables))) != hipSuccess) return e;
        if ((e = hipMemcpy(m.tables, &host, sizeof(McTables), hipMemcpyHostToDevice)) != hipSuccess) return e;
        const McTables href = make_mc_tables_reference();
        if ((e = hipMalloc((void**)&m.tables_ref, sizeof(McTables))) != hipSuccess) return e;
        if ((e = hipMemcpy(m.tables_ref, &href, sizeof(McTables), hipMemcpyHostToDevice)) != hipSuccess) return e;
        const CapTables hc = make_cap_tables(), hcr = make_cap_tables_reference();
        if ((e = hipMalloc((void**)&m.caps, sizeof(CapTables))) != hipSuccess) return e;
        if ((e = hipMemcpy(m.caps, &hc, sizeof(CapTables), hipMemcpyHostToDevice)) != hipSuccess) return e;
        if ((e = hipMalloc((void**)&m.caps_ref, sizeof(CapTables))) != hipSuccess) return e;
        if ((e = hipMemcpy(m.caps_ref, &hcr, sizeof(CapTables), hipMemcpyHostToDevice)) != hipSuccess) return e;
        const int64_t tiles = scan_tiles(std::max(std::max(nedges, ncubes), squares));
        if ((e = hipMalloc((void**)&m.flag, sizeof(int32_t) * (nedges + 1))) != hipSuccess) return e;
        if ((e = hipMalloc((void**)&m.vid, sizeof(int32_t) * (nedges + 1))) != hipSuccess) return e;
        if ((e = hipMalloc((void**)&m.cnt, sizeof(int32_t) * (ncubes + 1))) != hipSuccess) return e;
        if ((e = hipMalloc((void**)&m.toff, sizeof(int32_t) * (ncubes + 1))) != hipSuccess) return e;
        if ((e = hipMalloc((void**)&m.sums, sizeof(int32_t) * (tiles + 1))) != hipSuccess) return e;
        for (int32_t** q : {&m.capv, &m.capt, &m.capvo, &m.capto})
            if ((e = hipMalloc((void**)q, sizeof(int32_t) * (squares + 1))) != hipSuccess) return e;
        if ((e = hipMalloc((void**)&m.capid, sizeof(int32_t) * keys)) != hipSuccess) return e;
    }
    hipStream_t st = s->stream;
    // the reference's SDF values: the 8-bucket search over the same particles
    // where the last SDF came from the cell scan (the negative values, and so
    // the markers, are the same either way)
    if (s->sdf_from_cells && (e = launch_sdf(s, true)) != hipSuccess) return e;
    const McTables* tables = (const McTables*)(ref ? m.tables_ref : m.tables);
    const double* sdf = s->sdf;
    if (s->has_collider) {
        const int64_t nc = cell_count(s->g);
        if (!m.comb && (e = hipMalloc((void**)&m.comb, sizeof(double) * nc)) != hipSuccess) return e;
        hipLaunchKernelGGL(k_mc_combine, grid_of(nc), dim3(kBlock), 0, st, sdf,
                           (const double*)s->csdf, m.comb, nc);
        sdf = m.comb;
    }
    // cubes: crossed edges -> vertex ids; per-cube triangle counts -> offsets
    hipLaunchKernelGGL(k_mc_edges, grid_of(nedges), dim3(kBlock), 0, st, G, sdf, m.flag, nedges);
    if ((e = launch_scan_with(st, m.flag, m.vid, nedges, m.sums)) != hipSuccess) return e;
    hipLaunchKernelGGL(k_mc_count, grid_of(ncubes), dim3(kBlock), 0, st, G, sdf, tables, m.cnt, ncubes);
    if ((e = launch_scan_with(st, m.cnt, m.toff, ncubes, m.sums)) != hipSuccess) return e;
    // caps: the vertices each square meets first and its triangles -> offsets
    const CapTables* caps = (const CapTables*)(ref ? m.caps_ref : m.caps);
    hipLaunchKernelGGL(k_cap_count, grid_of(squares), dim3(kBlock), 0, st, G, Q, caps, sdf, m.capv, m.capt);
    if ((e = launch_scan_with(st, m.capv, m.capvo, squares, m.sums)) != hipSuccess) return e;
    if ((e = launch_scan_with(st, m.capt, m.capto, squares, m.sums)) != hipSuccess) return e;
    if ((e = hipGetLastError()) != hipSuccess) return e;
    int32_t nv = 0, nt = 0, ncv = 0, nct = 0;
    if ((e = hipMemcpyAsync(&nv, m.vid + nedges, sizeof(int32_t), hipMemcpyDeviceToHost, st)) != hipSuccess) return e;
    if ((e = hipMemcpyAsync(&nt, m.toff + ncubes, sizeof(int32_t), hipMemcpyDeviceToHost, st)) != hipSuccess) return e;
    if ((e = hipMemcpyAsync(&ncv, m.capvo + squares, sizeof(int32_t), hipMemcpyDeviceToHost, st)) != hipSuccess) return e;
    if ((e = hipMemcpyAsync(&nct, m.capto + squares, sizeof(int32_t), hipMemcpyDeviceToHost, st)) != hipSuccess) return e;
    if ((e = hipStreamSynchronize(st)) != hipSuccess) return e;
    const int64_t vertices = (int64_t)nv + ncv, triangles = (int64_t)nt + nct;
    if ((e = grow(&m.pos, &m.vcap, 3 * vertices)) != hipSuccess) return e;
    if ((e = grow(&m.nrm, &m.ncap, 3 * vertices)) != hipSuccess) return e;
    if ((e = grow(&m.tri, &m.tcap, 3 * triangles)) != hipSuccess) return e;
    if (nv > 0)
        hipLaunchKernelGGL(k_mc_vertices, grid_of(nedges), dim3(kBlock), 0, st, G, sdf,
                           (const int32_t*)m.vid, m.pos, m.nrm, nedges);
    if (nt > 0)
        hipLaunchKernelGGL(k_mc_emit, grid_of(ncubes), dim3(kBlock), 0, st, G, sdf, tables,
                           (const int32_t*)m.toff, (const int32_t*)m.vid, m.tri, ncubes);
    if (nct > 0) {
        hipLaunchKernelGGL(k_cap_vertices, grid_of(squares), dim3(kBlock), 0, st, G, Q, caps, sdf,
                           (const int32_t*)m.capvo, (int64_t)nv, ref ? 0 : 1, m.capid, m.pos, m.nrm);
        hipLaunchKernelGGL(k_cap_triangles, grid_of(squares), dim3(kBlock), 0, st, G, Q, caps, sdf,
                           (const int32_t*)m.capto, (int64_t)nt, (const int32_t*)m.capid, m.tri);
    }
    if ((e = hipGetLastError()) != hipSuccess) return e;
    m.vertices = vertices;
    m.triangles = triangles;
    m.built = true;
    return hipStreamSynchronize(st);
}

hipError_t surface_download(fe_scene* s, double* pos, double* nrm, int32_t* tri) {
    McState& m = s->mc;
    hipError_t e;
    const size_t v3 = 3 * (size_t)m.vertices, t3 = 3 * (size_t)m.triangles;
    if (pos && v3 && (e = hipMemcpy(pos, m.pos, sizeof(double) * v3, hipMemcpyDeviceToHost)) != hipSuccess) return e;
    if (nrm && v3 && (e = hipMemcpy(nrm, m.nrm, sizeof(double) * v3, hipMemcpyDeviceToHost)) != hipSuccess) return e;
    if (tri && t3 && (e = hipMemcpy(tri, m.tri, sizeof(int32_t) * t3, hipMemcpyDeviceToHost)) != hipSuccess) return e;
    return hipSuccess;
}

}  // namespace fe
