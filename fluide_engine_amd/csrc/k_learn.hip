// k_learn.hip -- the pressure warm-start network on the device: forward,
// backward and Adam, BF16 operands on MFMA with
// FP32 accumulation.  No counterpart in the reference.
//
// Convolutions are implicit GEMMs over channel-last BF16 activations, K = 27
// taps x input channels, 16 at a time (v_mfma_f32_16x16x16_bf16; a lane holds
// A[l % 16][4 (l / 16) + j], B[4 (l / 16) + j][l % 16] and returns
// C[4 (l / 16) + i][l % 16], checked on the device).
// The backward data pass is the same kernel on the flipped, transposed weights;
// the weight gradient is a GEMM over voxels (M = input channel, N = output
// channel, K = voxel) on channel planes, one partial per workgroup summed in a
// fixed order, so every gradient is reproducible run to run.
#include <algorithm>
#include <cmath>
#include <vector>

#include "fe_learn.hpp"
#include "fe_stencil.hpp"

namespace fe {

namespace {

typedef float f4 __attribute__((ext_vector_type(4)));

struct Lv {
    int nx, ny, nz;
    int64_t V;
};

inline Lv lv_of(const NetLevel& l) { return Lv{l.n[0], l.n[1], l.n[2], l.V}; }

__device__ inline uint16_t to_bf16(float f) {  // round to nearest, ties to even
    uint32_t u = __float_as_uint(f);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}
__device__ inline float from_bf16(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

__device__ inline void decode(const Lv& d, int64_t v, int& x, int& y, int& z) {
    const int64_t nxy = (int64_t)d.nx * d.ny;
    z = (int)(v / nxy);
    const int64_t r = v - (int64_t)z * nxy;
    y = (int)(r / d.nx);
    x = (int)(r - (int64_t)y * d.nx);
}

inline dim3 g1(int64_t n) { return dim3((unsigned)((n + 255) / 256)); }

// ---------------------------------------------------------------------------
// Convolution (forward, and backward data on the flipped weights)
// ---------------------------------------------------------------------------
// A wavefront computes 16 MT consecutive voxels x 16 NT output channels.  K
// runs over blocks of one tap and 16 channels, taps outermost, two blocks per
// step.  An output is one chain of products in that order whatever the tile,
// so no launch shape moves the BF16 roundings of the layers behind; an
// instruction of twice the depth, or shares of K added up, do (26 % of its sums
// change by a bit at the same error of 3.9e-8, and a gradient by 6.5e-4).
// A lane loads 16 bytes, half a block's channels of a voxel; two swaps of 16
// lanes turn the step's four halves into its blocks' operands, where lane group
// q holds channels 4 q .. 4 q + 3 (8-byte loads straight into that place touch
// twice the cache lines: 130 us for the 92 below).  A voxel outside the grid
// reads at an offset past the buffer's end, which the load gives as zeros.
// Bound by the first-level cache: per step it reads MT KB of activations and
// NT KB of packed weights for 2 MT NT matrix instructions.  A step's loads are
// issued AHEAD steps before its products; a small level, bound by the latency
// of a wavefront's chain of steps, keeps more of them in flight.  At 64x96x80
// (us per launch): 16 and 48 -> 16 channels on the finest level 32 and 92, 16
// -> 48 there 64, all launches of the three levels below together 157; with a
// 16-voxel tile, 8-byte loads and a step of one block they took 200 for the
// first two, 73 and 245.
typedef __bf16 b8 __attribute__((ext_vector_type(8)));
typedef short s4 __attribute__((ext_vector_type(4)));
typedef uint32_t u2 __attribute__((ext_vector_type(2)));
typedef uint32_t u4 __attribute__((ext_vector_type(4)));
__device__ inline b8 as_b8(const u4& w) { return __builtin_bit_cast(b8, w); }
__device__ inline s4 as_s4(const u2& w) { return __builtin_bit_cast(s4, w); }

__host__ __device__ inline int conv_chunks(int cin) { return (27 * cin + 31) / 32; }
constexpr int kMaxCh = 112;
constexpr int kMaxChunks = (27 * kMaxCh + 31) / 32;
// Bytes a load may reach from its wave's base, below the offset that stands for
// outside.  A wave's taps lie within 2 (nx ny + nx + 1) + 16 MT voxels of 96
// bytes at most on the finest level, 2.42e9 bytes on the largest grid
// (kNetMaxVoxels on the least 8 planes of 8 rows), a quarter of that below.
constexpr uint32_t kConvReach = 0xFFFFFFE0u;

template <int MT, int NT, int AHEAD>
__global__ __launch_bounds__(256) void k_conv(Lv d, const uint16_t* __restrict__ X, int cin, int cout,
                                              const u4* __restrict__ Wp, const float* __restrict__ bias, int relu,
                                              uint16_t* __restrict__ Ybf, float* __restrict__ Yf) {
    __shared__ int2 table[4 * kMaxChunks];  // per half block: byte offset, tap (27: none)
    const int chunks = conv_chunks(cin);
    for (int e = threadIdx.x; e < 4 * chunks; e += 256) {
        const int t = 8 * e / cin, ch = 8 * e - t * cin;
        const int dx = t % 3 - 1, dy = (t / 3) % 3 - 1, dz = t / 9 - 1;
        table[e] = t < 27 ? make_int2(2 * ((dx + d.nx * (dy + d.ny * dz)) * cin + ch), t) : make_int2(0, 27);
    }
    __syncthreads();
    const int wave = threadIdx.x >> 6, l = threadIdx.x & 63, row = l & 15, kq = l >> 4;
    const int64_t v0 = ((int64_t)blockIdx.x * 4 + wave) * (16 * MT);
    if (v0 >= d.V) return;  // uniform per wavefront
    const int nt0 = blockIdx.y * NT, nts = cout / 16;
    // the buffer starts a z slice and a row before the wave's first voxel
    const int64_t reach = (int64_t)d.nx * d.ny + d.nx + 1;
    const int64_t vb = v0 > reach ? v0 - reach : 0;
    const int64_t bytes = (d.V - vb) * cin * 2;
    const __amdgpu_buffer_rsrc_t buf =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(X + vb * cin), 0,
                                          (int)(uint32_t)min(bytes, (int64_t)kConvReach), 0x00020000);
    // per tile: which of the 27 taps lie inside the grid, and the voxel's offset
    uint32_t mask[MT], at[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        const int64_t v = v0 + 16 * m + row;
        mask[m] = 0;
        at[m] = (uint32_t)((v - vb) * cin * 2);
        if (v < d.V) {
            int x, y, z;
            decode(d, v, x, y, z);
            const uint32_t xm = (x > 0) | 2 | ((x + 1 < d.nx) << 2);
            const bool ym[3] = {y > 0, true, y + 1 < d.ny}, zm[3] = {z > 0, true, z + 1 < d.nz};
#pragma unroll
            for (int q = 0; q < 9; ++q) mask[m] |= ym[q % 3] && zm[q / 3] ? xm << (3 * q) : 0u;
        }
    }
    f4 acc[MT][NT];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[m][nt] = f4{0.f, 0.f, 0.f, 0.f};
    const u4* wb = Wp + (int64_t)nt0 * 64 + l;
    const int half = (kq >> 1) | ((kq & 1) << 1);  // of the step's four half blocks
    u4 a[AHEAD][MT], b[AHEAD][NT];
    auto load = [&](int c, u4 (&a)[MT], u4 (&b)[NT]) {
        const int2 e = table[4 * c + half];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) b[nt] = wb[((int64_t)c * nts + nt) * 64];
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const uint32_t o = (mask[m] >> e.y) & 1u ? at[m] + (uint32_t)e.x : 0xFFFFFFF0u;
            a[m] = __builtin_bit_cast(u4, __builtin_amdgcn_raw_buffer_load_b128(buf, (int)o, 0, 0));
        }
    };
#pragma unroll
    for (int s = 0; s < AHEAD; ++s) load(s, a[s], b[s]);  // 14 steps at least
    auto products = [&](const u4 (&a)[MT], const u4 (&b)[NT]) {
        u2 block[2][MT];
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int w = 0; w < 2; ++w) {  // lane groups 1, 3 of the lower half for 0, 2 of the upper
                const auto r = __builtin_amdgcn_permlane16_swap(a[m][w], a[m][w + 2], false, false);
                block[0][m][w] = r[0];
                block[1][m][w] = r[1];
            }
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int nt = 0; nt < NT; ++nt)
                    acc[m][nt] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(
                        as_s4(block[h][m]), as_s4(u2{b[nt][2 * h], b[nt][2 * h + 1]}), acc[m][nt], 0, 0, 0);
    };
    int c = 0;
    for (; c + AHEAD <= chunks; c += AHEAD) {
#pragma unroll
        for (int s = 0; s < AHEAD; ++s) {
            products(a[s], b[s]);
            load(min(c + s + AHEAD, chunks - 1), a[s], b[s]);
        }
    }
#pragma unroll
    for (int s = 0; s < AHEAD - 1; ++s)
        if (c + s < chunks) products(a[s], b[s]);
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int64_t v = v0 + 16 * m + 4 * kq + i;
            if (v >= d.V) continue;
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                const int co = (nt0 + nt) * 16 + row;
                float val = acc[m][nt][i] + (bias ? bias[co] : 0.0f);
                if (relu) val = fmaxf(val, 0.0f);
                if (Ybf) Ybf[v * cout + co] = to_bf16(val);
                if (Yf) Yf[v * cout + co] = val;
            }
        }
}

// Packed BF16 weights: forward [chunk][nt][lane][j] = W[t][ci][16 nt + lane % 16],
// t = q / (cin / 16), ci = 16 (q % (cin / 16)) + 4 (lane / 16) + j % 4 for block
// q = 2 chunk + j / 4 of the 27 cin / 16, zero past the end;
// backward data (cin' = cout, cout' = cin): W'[t][a][b] = W[26 - t][b][a], packed the same way.
__device__ inline void packed_place(int64_t i, int cin, int cout, int& t, int& ci, int& co) {
    const int j = (int)(i & 7), l = (int)(i >> 3) & 63, NT = cout / 16;
    const int64_t r = i >> 9;
    const int c = (int)(r / NT), nt = (int)(r - (int64_t)c * NT);
    const int q = 2 * c + (j >> 2), kcs = cin / 16;
    t = q / kcs;
    ci = 16 * (q - t * kcs) + 4 * (l >> 4) + (j & 3);
    co = 16 * nt + (l & 15);
}

__host__ __device__ inline int64_t packed_size(int cin, int cout) { return 32LL * conv_chunks(cin) * cout; }

__global__ __launch_bounds__(256) void k_pack(int cin, int cout, const float* __restrict__ w,
                                              uint16_t* __restrict__ wp, uint16_t* __restrict__ wpt) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    int t, a, b;
    if (i < packed_size(cin, cout)) {
        packed_place(i, cin, cout, t, a, b);
        wp[i] = t < 27 ? to_bf16(w[((int64_t)t * cin + a) * cout + b]) : (uint16_t)0;
    }
    if (i < packed_size(cout, cin)) {
        packed_place(i, cout, cin, t, a, b);  // a: an output channel of W, b: an input channel
        wpt[i] = t < 27 ? to_bf16(w[((int64_t)(26 - t) * cin + b) * cout + a]) : (uint16_t)0;
    }
}

// ---------------------------------------------------------------------------
// Weight gradient: dW[t][ci][co] = sum_v X[v + off(t)][ci] * G[v][co], and the
// bias gradient db[co] = sum_v G[v][co].
//
// The contraction runs over voxels, so both operands are taken from channel
// planes, where a lane's 8 voxels are one 16-byte load.  Rows are filled up to
// segments of 8 voxels: G as [co][segment], zero in the fill, X as
// [ci][nz + 2][ny + 2][row] with a border of zeros (8 wide in x, which keeps
// rows aligned), so no tap tests bounds.  A wavefront holds the 9 taps of one z offset
// for 16 input channels and all output channels: per y offset one 16-byte and
// two 4-byte loads give all three x offsets by shifting, so 9 NT matrix
// instructions (v_mfma_f32_16x16x32_bf16) take 3 + NT wide loads.  Bound by
// the first-level cache's loads.  The bias is one more product, with ones.
// At 64x96x80, the layers of the finest level (48 -> 16 and 16 -> 16
// channels): 450 and 417 us with one tap per wavefront and 2-byte loads.
// ---------------------------------------------------------------------------
constexpr int kEdge = 8;  // the zero border of X's rows

struct Planes {
    int nx8;         // segments of a row
    int px, py;      // X: row length and rows of a z slice
    int64_t xn, gn;  // elements of a channel's plane of X and G
    int64_t steps;   // 4 segments each, the last one's rest zero in G
};
__host__ __device__ inline Planes planes_of(const Lv& d) {
    Planes P;
    P.nx8 = (d.nx + 7) / 8;
    P.px = 8 * P.nx8 + 2 * kEdge;
    P.py = d.ny + 2;
    P.xn = (int64_t)P.px * P.py * (d.nz + 2);
    P.steps = ((int64_t)P.nx8 * d.ny * d.nz + 3) / 4;
    P.gn = 32 * P.steps;
    return P;
}

// A workgroup's 8 segments of a channel-last array, as pairs of channels:
// f(voxel, channel pair) gives a pair's bits; they go to channel planes (X's
// or G's place for each segment) by way of LDS (rows of C + 2: the transposed
// reads spread over the banks).  The fill of a segment is zero.
template <bool IS_X, typename F>
__device__ inline void segments_to_planes(const Lv& d, int C, uint16_t* __restrict__ out, F f) {
    __shared__ uint16_t lds[64 * (kMaxCh + 2)];
    __shared__ int64_t voxel[8], place[8];
    __shared__ int count[8];
    const Planes P = planes_of(d);
    if (threadIdx.x < 8) {
        const int64_t seg = (int64_t)blockIdx.x * 8 + threadIdx.x, r = seg / P.nx8;
        const int x = 8 * (int)(seg - r * P.nx8);
        const int64_t z = r / d.ny;
        const int y = (int)(r - z * d.ny);
        voxel[threadIdx.x] = r * d.nx + x;
        place[threadIdx.x] = IS_X ? ((z + 1) * P.py + (y + 1)) * P.px + kEdge + x : 8 * seg;
        count[threadIdx.x] = z < d.nz ? min(8, d.nx - x) : 0;
    }
    __syncthreads();
    const int half = C / 2;
    for (int e = threadIdx.x; e < 64 * half; e += 256) {
        const int slot = e / half, pair = e - slot * half;
        uint32_t w = 0;
        if ((slot & 7) < count[slot >> 3]) w = f(voxel[slot >> 3] + (slot & 7), pair);
        *reinterpret_cast<uint32_t*>(lds + slot * (C + 2) + 2 * pair) = w;
    }
    __syncthreads();
    for (int e = threadIdx.x; e < C * 8; e += 256) {
        const int c = e >> 3, q = e & 7;
        if (count[q] == 0) continue;
        u4 w;
#pragma unroll
        for (int h = 0; h < 4; ++h)
            w[h] = (uint32_t)lds[(8 * q + 2 * h) * (C + 2) + c] |
                   ((uint32_t)lds[(8 * q + 2 * h + 1) * (C + 2) + c] << 16);
        *reinterpret_cast<u4*>(out + c * (IS_X ? P.xn : P.gn) + place[q]) = w;
    }
}

// Channel-last X to planes (their border is zero from the allocation on).
__global__ __launch_bounds__(256) void k_planes(Lv d, int C, const uint16_t* __restrict__ X,
                                                uint16_t* __restrict__ Xt) {
    const uint32_t* in = reinterpret_cast<const uint32_t*>(X);
    segments_to_planes<true>(d, C, Xt, [&](int64_t v, int pair) { return in[v * (C / 2) + pair]; });
}

// dpre = bf16(y > 0 ? g : 0), channel-last and as planes
__global__ __launch_bounds__(256) void k_mask(Lv d, int C, const float* __restrict__ g,
                                              const uint16_t* __restrict__ y, uint16_t* __restrict__ dpre,
                                              uint16_t* __restrict__ Gt) {
    const float2* gi = reinterpret_cast<const float2*>(g);
    const uint32_t* yi = reinterpret_cast<const uint32_t*>(y);
    uint32_t* o = reinterpret_cast<uint32_t*>(dpre);
    auto mask = [](uint32_t h, float v) { return h != 0 && !(h & 0x8000u) ? (uint32_t)to_bf16(v) : 0u; };
    segments_to_planes<false>(d, C, Gt, [&](int64_t v, int pair) {
        const int64_t e = v * (C / 2) + pair;
        const float2 a = gi[e];
        const uint32_t h = yi[e];
        const uint32_t w = mask(h & 0xFFFFu, a.x) | (mask(h >> 16, a.y) << 16);
        o[e] = w;
        return w;
    });
}

// 16 input channels and the finest level's 491 520 voxels: 44 us, 48 channels
// 116 us, where voxel-major operands gathered a value at a time took 1.1 ms for
// the seven layers and their partials' sum 0.6 ms (now 0.26, 0.15 for the
// planes, and 0.04 ms).
// blockIdx.y = 3 kc + dz (16 input channels, z offset dz - 1).  Wave w of block
// b takes the 32-voxel steps [ (4 b + w) spw, ... + spw ).
template <int NT>
__global__ __launch_bounds__(256) void k_wgrad(Lv d, int cin, const uint16_t* __restrict__ Xt,
                                               const uint16_t* __restrict__ Gt, float* __restrict__ part,
                                               float* __restrict__ bpart, int64_t spw) {
    __shared__ float sm[4][NT * 256];
    const int wave = threadIdx.x >> 6, l = threadIdx.x & 63, row = l & 15, kq = l >> 4;
    const int kc = blockIdx.y / 3, dz = blockIdx.y % 3;
    constexpr int cout = NT * 16;
    const Planes P = planes_of(d);
    const int64_t s0 = min((4 * (int64_t)blockIdx.x + wave) * spw, P.steps), s1 = min(s0 + spw, P.steps);
    // this lane's 8 voxels: segment 4 s + kq (past the last one G is zero, and
    // X is read at the last z)
    const int nx8 = P.nx8;
    int x8 = 0, y = 0, z = 0;
    {
        const int64_t seg = 4 * s0 + kq, r = seg / nx8;
        x8 = (int)(seg - r * nx8);
        z = (int)(r / d.ny);
        y = (int)(r - (int64_t)z * d.ny);
    }
    const uint16_t* xp = Xt + (int64_t)(kc * 16 + row) * P.xn + kEdge;
    const uint16_t* gp = Gt + (int64_t)row * P.gn + 8 * kq;
    const bool bias = kc == 0 && dz == 1;  // uniform
    f4 acc[9][NT], accb[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        accb[nt] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < 9; ++t) acc[t][nt] = f4{0.f, 0.f, 0.f, 0.f};
    }
    const b8 ones = as_b8(u4{0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u});
    for (int64_t s = s0; s < s1; ++s) {
        b8 b[NT];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
            b[nt] = as_b8(*reinterpret_cast<const u4*>(gp + (int64_t)nt * 16 * P.gn + 32 * s));
        u4 m[3];
        uint32_t lo[3], hi[3];
#pragma unroll
        for (int dy = 0; dy < 3; ++dy) {
            const uint16_t* p = xp + ((int64_t)(min(z, d.nz - 1) + dz) * P.py + (y + dy)) * P.px + 8 * x8;
            m[dy] = *reinterpret_cast<const u4*>(p);
            lo[dy] = *reinterpret_cast<const uint32_t*>(p - 2);
            hi[dy] = *reinterpret_cast<const uint32_t*>(p + 8);
        }
#pragma unroll
        for (int dy = 0; dy < 3; ++dy) {
            const uint32_t a01 = __builtin_amdgcn_alignbit(m[dy][1], m[dy][0], 16),
                           a12 = __builtin_amdgcn_alignbit(m[dy][2], m[dy][1], 16),
                           a23 = __builtin_amdgcn_alignbit(m[dy][3], m[dy][2], 16);
            const b8 left = as_b8(u4{__builtin_amdgcn_alignbit(m[dy][0], lo[dy], 16), a01, a12, a23}),
                     mid = as_b8(m[dy]),
                     right = as_b8(u4{a01, a12, a23, __builtin_amdgcn_alignbit(hi[dy], m[dy][3], 16)});
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                acc[3 * dy][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(left, b[nt], acc[3 * dy][nt], 0, 0, 0);
                acc[3 * dy + 1][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(mid, b[nt], acc[3 * dy + 1][nt], 0, 0, 0);
                acc[3 * dy + 2][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(right, b[nt], acc[3 * dy + 2][nt], 0, 0, 0);
            }
        }
        if (bias) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
                accb[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, b[nt], accb[nt], 0, 0, 0);
        }
        x8 += 4;
        while (x8 >= nx8) {
            x8 -= nx8;
            if (++y == d.ny) {
                y = 0;
                ++z;
            }
        }
    }
    // the block's sum, waves in order, tap by tap
#pragma unroll
    for (int t = 0; t < 9; ++t) {
        __syncthreads();
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int i = 0; i < 4; ++i) sm[wave][(4 * kq + i) * cout + nt * 16 + row] = acc[t][nt][i];
        __syncthreads();
        float* o = part + (((int64_t)blockIdx.x * 27 + 9 * dz + t) * cin + kc * 16) * cout;
#pragma unroll
        for (int e = 0; e < NT; ++e) {
            const int i = threadIdx.x + 256 * e;
            o[i] = ((sm[0][i] + sm[1][i]) + sm[2][i]) + sm[3][i];
        }
    }
    if (bias) {  // every row of ones . G is the column sum
        __syncthreads();
        if (kq == 0) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) sm[wave][nt * 16 + row] = accb[nt][0];
        }
        __syncthreads();
        if (threadIdx.x < cout) {
            const int i = threadIdx.x;
            bpart[(int64_t)blockIdx.x * cout + i] = ((sm[0][i] + sm[1][i]) + sm[2][i]) + sm[3][i];
        }
    }
}

// out[i] = sum_p part[p * size + i] for the weights and, behind them, the
// biases: 16 outputs per block, the partials dealt to 16 threads each and
// their sums added in order.
__global__ __launch_bounds__(256) void k_reduce_parts(int nparts, int64_t wsize, const float* __restrict__ wpart,
                                                      float* __restrict__ w, int bsize,
                                                      const float* __restrict__ bpart, float* __restrict__ b) {
    __shared__ float sm[16][17];
    const int col = threadIdx.x & 15, sl = threadIdx.x >> 4;
    int64_t i = (int64_t)blockIdx.x * 16 + col;  // both sizes are multiples of 16
    const bool isw = i < wsize;
    if (!isw) i -= wsize;
    const float* part = isw ? wpart : bpart;
    const int64_t size = isw ? wsize : bsize;
    float s = 0.0f;
    for (int p = sl; p < nparts; p += 16) s += part[p * size + i];
    sm[sl][col] = s;
    __syncthreads();
    if (sl != 0) return;
    for (int q = 1; q < 16; ++q) s += sm[q][col];
    (isw ? w : b)[i] = s;
}

// ---------------------------------------------------------------------------
// Elementwise and resampling passes
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_features(int64_t V, const float* __restrict__ b,
                                                  const uint8_t* __restrict__ flags, double rms,
                                                  uint16_t* __restrict__ X0) {
    const int64_t v = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (v >= V) return;
    uint16_t* o = X0 + v * kNetIn;
    o[0] = to_bf16((float)((double)b[v] / rms));
    o[1] = flags[v] == FE_FLUID ? (uint16_t)0x3F80 : (uint16_t)0;  // 1.0 in BF16
    o[2] = flags[v] == FE_AIR ? (uint16_t)0x3F80 : (uint16_t)0;
    for (int c = 3; c < kNetIn; ++c) o[c] = 0;
}

// The passes between levels move data and are bound by it once a thread takes
// 16 bytes (8 BF16 or 4 FP32 channels) and finds its voxel with 32-bit
// divisions by constants: the concatenation at 64x96x80 takes 12 us (63 MB, the
// rate of a copy) where one channel per thread behind 64-bit divisions took 68,
// the seven passes of a gradient 65 us for 175.  A level's groups, 6 per finest
// voxel at most, stay below 2^32 (kNetMaxVoxels).
template <int GROUPS>
__device__ inline bool group_of(int64_t V, uint32_t& v, uint32_t& g) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    v = i / GROUPS;
    g = i - v * GROUPS;
    return v < (uint32_t)V;
}

__device__ inline void decode32(const Lv& d, uint32_t v, uint32_t& x, uint32_t& y, uint32_t& z) {
    const uint32_t r = v / (uint32_t)d.nx;
    x = v - r * (uint32_t)d.nx;
    z = r / (uint32_t)d.ny;
    y = r - z * (uint32_t)d.ny;
}

// The voxel of the coarser level that v lies in.
__device__ inline int64_t parent(const Lv& f, const Lv& c, uint32_t v) {
    uint32_t x, y, z;
    decode32(f, v, x, y, z);
    return (x / 2) + (int64_t)c.nx * ((y / 2) + (int64_t)c.ny * (z / 2));
}

// F(voxel) for the eight voxels of the finer level in v, x fastest.
template <typename F>
__device__ inline void children(const Lv& f, const Lv& c, uint32_t v, F fn) {
    uint32_t X, Y, Z;
    decode32(c, v, X, Y, Z);
#pragma unroll
    for (int q = 0; q < 8; ++q)
        fn((2 * X + (q & 1)) + (int64_t)f.nx * ((2 * Y + ((q >> 1) & 1)) + (int64_t)f.ny * (2 * Z + (q >> 2))));
}

template <int C>
__global__ __launch_bounds__(256) void k_pool(Lv f, Lv c, const uint16_t* __restrict__ in,
                                              uint16_t* __restrict__ out) {
    uint32_t vc, g;
    if (!group_of<C / 8>(c.V, vc, g)) return;
    float s[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    children(f, c, vc, [&](int64_t v) {
        const u4 w = *reinterpret_cast<const u4*>(in + v * C + 8 * g);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            s[2 * q] += from_bf16((uint16_t)w[q]);
            s[2 * q + 1] += from_bf16((uint16_t)(w[q] >> 16));
        }
    });
    u4 o;
#pragma unroll
    for (int q = 0; q < 4; ++q)
        o[q] = (uint32_t)to_bf16(s[2 * q] / 8.0f) | ((uint32_t)to_bf16(s[2 * q + 1] / 8.0f) << 16);
    *reinterpret_cast<u4*>(out + (int64_t)vc * C + 8 * g) = o;
}

// out[v] = [coarse[parent(v)] (CC channels), skip[v] (CS channels)]
template <int CC, int CS>
__global__ __launch_bounds__(256) void k_upcat(Lv f, Lv c, const uint16_t* __restrict__ coarse,
                                               const uint16_t* __restrict__ skip, uint16_t* __restrict__ out) {
    uint32_t v, g;
    if (!group_of<(CC + CS) / 8>(f.V, v, g)) return;
    const uint16_t* in = g < CC / 8 ? coarse + parent(f, c, v) * CC + 8 * g : skip + (int64_t)v * CS + (8 * g - CC);
    *reinterpret_cast<u4*>(out + (int64_t)v * (CC + CS) + 8 * g) = *reinterpret_cast<const u4*>(in);
}

__global__ __launch_bounds__(256) void k_head(int64_t V, const float* __restrict__ D0, const float* __restrict__ hw,
                                              const float* __restrict__ hb, float* __restrict__ out) {
    const int64_t v = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (v >= V) return;
    float s = 0.0f;
    for (int c = 0; c < 16; ++c) s += D0[v * 16 + c] * hw[c];
    out[v] = s + hb[0];
}

// dout = 2 (out - target) / nf on FLUID cells; per-block FP64 sums of the squares
__global__ __launch_bounds__(256) void k_loss(int64_t V, const float* __restrict__ out,
                                              const float* __restrict__ target, const uint8_t* __restrict__ flags,
                                              float nf, float* __restrict__ dout, double* __restrict__ part) {
    const int64_t v = (int64_t)blockIdx.x * 256 + threadIdx.x;
    double s = 0.0;
    if (v < V) {
        const float diff = flags[v] == FE_FLUID ? out[v] - target[v] : 0.0f;
        dout[v] = 2.0f * diff / nf;
        s = (double)diff * diff;
    }
    double sv[1] = {s};
    write_partials<1>(sv, part);
}

// gD0 = dout * hw; per-block FP64 sums of D0 * dout (16) and dout (1)
__global__ __launch_bounds__(256) void k_head_bwd(int64_t V, const float* __restrict__ D0,
                                                  const float* __restrict__ dout, const float* __restrict__ hw,
                                                  float* __restrict__ gD0, double* __restrict__ part) {
    const int64_t v = (int64_t)blockIdx.x * 256 + threadIdx.x;
    double s[17];
    for (int q = 0; q < 17; ++q) s[q] = 0.0;
    if (v < V) {
        const float g = dout[v];
        for (int c = 0; c < 16; ++c) {
            gD0[v * 16 + c] = g * hw[c];
            s[c] = (double)D0[v * 16 + c] * g;
        }
        s[16] = g;
    }
    write_partials<17>(s, part);
}

template <int NV>
__global__ __launch_bounds__(256) void k_sum_to(const double* __restrict__ part, int nparts, float* __restrict__ out,
                                                double* __restrict__ out64, double scale) {
    double tot[NV];
    sum_partials<NV>(part, nparts, tot);
    if (threadIdx.x == 0)
        for (int q = 0; q < NV; ++q) {
            if (out) out[q] = (float)(tot[q] * scale);
            if (out64) out64[q] = tot[q] * scale;
        }
}

// Energy loss: with q = A p (p zero outside FLUID), per-block FP64 sums of
// b.p and p.q over FLUID cells; q kept for the gradient.
__global__ __launch_bounds__(256) void k_energy_stats(Lv d, const uint16_t* __restrict__ code, double ihx, double ihy,
                                                      double ihz, const float* __restrict__ p,
                                                      const float* __restrict__ b, float* __restrict__ aq,
                                                      double* __restrict__ part) {
#pragma clang fp contract(off)
    const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
    double s[2] = {0.0, 0.0};
    if (c < d.V) {
        const uint16_t cd = code[c];
        double q = 0.0;
        if (cd & kFluidBit) {
            const double ih2[3] = {ihx, ihy, ihz};
            const Stride st = stride_of(d.nx, d.ny, d.nz);
            auto val = [&](int64_t k) { return (code[k] & kFluidBit) ? (double)p[k] : 0.0; };
            const double pc = (double)p[c];
            q = code_apply64(cd, c, st, ih2, pc, val);
            s[0] = (double)b[c] * pc;
            s[1] = pc * q;
        }
        aq[c] = (float)q;
    }
    write_partials<2>(s, part);
}

// loss = 1 - s^2 / (qq E); scal[0] = loss, scal[1] = 2 s / (qq E), scal[2] = s / qq
__global__ __launch_bounds__(256) void k_energy_finish(const double* __restrict__ part, int nparts, double energy,
                                                       float* __restrict__ loss_slot, double* __restrict__ scal) {
    double tot[2];
    sum_partials<2>(part, nparts, tot);
    if (threadIdx.x == 0) {
        const double sv = tot[0], qq = tot[1];
        const bool ok = qq > 0 && energy > 0;
        const double loss = ok ? 1.0 - sv * sv / (qq * energy) : 1.0;
        scal[0] = loss;
        scal[1] = ok ? 2.0 * sv / (qq * energy) : 0.0;
        scal[2] = ok ? sv / qq : 0.0;
        if (loss_slot) *loss_slot = (float)loss;
    }
}

// dout = 2 s / (qq E) (s / qq A p - b) on FLUID cells (FP64, stored FP32)
__global__ __launch_bounds__(256) void k_energy_grad(int64_t V, const uint16_t* __restrict__ code,
                                                     const float* __restrict__ aq, const float* __restrict__ b,
                                                     const double* __restrict__ scal, float* __restrict__ dout) {
#pragma clang fp contract(off)
    const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (c >= V) return;
    dout[c] = (code[c] & kFluidBit) ? (float)(scal[1] * (scal[2] * (double)aq[c] - (double)b[c])) : 0.0f;
}

__global__ __launch_bounds__(256) void k_codes(Lv d, const uint8_t* __restrict__ flags, uint16_t* __restrict__ code) {
    const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (c >= d.V) return;
    int x, y, z;
    decode(d, c, x, y, z);
    code[c] = row_code(flags, c, (uint32_t)x, (uint32_t)y, (uint32_t)z, (uint32_t)d.nx, (uint32_t)d.ny,
                       (uint32_t)d.nz);
}

// The coarse voxel's gradient: the sum over its children of the first CC of
// the concatenation's channels.
template <int CC, int CS>
__global__ __launch_bounds__(256) void k_up_bwd(Lv f, Lv c, const float* __restrict__ gC,
                                                float* __restrict__ gCoarse) {
    uint32_t p, g;
    if (!group_of<CC / 4>(c.V, p, g)) return;
    float4 s = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    children(f, c, p, [&](int64_t v) {
        const float4 a = *reinterpret_cast<const float4*>(gC + v * (CC + CS) + 4 * g);
        s.x += a.x;
        s.y += a.y;
        s.z += a.z;
        s.w += a.w;
    });
    *reinterpret_cast<float4*>(gCoarse + (int64_t)p * CC + 4 * g) = s;
}

// An encoder level's gradient: the concatenation's last CS channels plus an
// eighth of the pooled level's.
template <int CC, int CS>
__global__ __launch_bounds__(256) void k_enc_bwd(Lv f, Lv c, const float* __restrict__ gC,
                                                 const float* __restrict__ gPool, float* __restrict__ gE) {
    uint32_t v, g;
    if (!group_of<CS / 4>(f.V, v, g)) return;
    const float4 a = *reinterpret_cast<const float4*>(gC + (int64_t)v * (CC + CS) + CC + 4 * g);
    const float4 b = *reinterpret_cast<const float4*>(gPool + parent(f, c, v) * CS + 4 * g);
    *reinterpret_cast<float4*>(gE + (int64_t)v * CS + 4 * g) =
        make_float4(a.x + b.x / 8.0f, a.y + b.y / 8.0f, a.z + b.z / 8.0f, a.w + b.w / 8.0f);
}

__global__ __launch_bounds__(256) void k_adam(int64_t n, float* __restrict__ w, const float* __restrict__ g,
                                              float* __restrict__ m, float* __restrict__ v, float lr, float bc1,
                                              float bc2) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.0f - b1) * gi;
    const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    w[i] -= lr * (mi / bc1) / (sqrtf(vi / bc2) + eps);
}

// FP64 sums of b^2 over all cells, and of p^2, the count and b.p over FLUID cells
template <typename P>
__global__ __launch_bounds__(256) void k_sample_stats(int64_t V, const float* __restrict__ b,
                                                      const P* __restrict__ p, const uint8_t* __restrict__ flags,
                                                      double* __restrict__ part) {
    const int64_t v = (int64_t)blockIdx.x * 256 + threadIdx.x;
    double s[4] = {0.0, 0.0, 0.0, 0.0};
    if (v < V) {
        s[0] = (double)b[v] * b[v];
        if (flags[v] == FE_FLUID) {
            const double pv = p ? (double)p[v] : 0.0;
            s[1] = pv * pv;
            s[2] = 1.0;
            s[3] = p ? (double)b[v] * pv : 0.0;
        }
    }
    write_partials<4>(s, part);
}

__global__ __launch_bounds__(256) void k_target(int64_t V, const double* __restrict__ p,
                                                const uint8_t* __restrict__ flags, double rms,
                                                float* __restrict__ t) {
    const int64_t v = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (v >= V) return;
    t[v] = flags[v] == FE_FLUID ? (float)(p[v] / rms) : 0.0f;
}

// Scale of the warm start: with q = A phat (phat zero outside FLUID), per-block
// FP64 sums of b.q, q.q (residual-optimal alpha = b.q / q.q) and b.phat,
// phat.q (energy-optimal alpha = b.phat / phat.A.phat, the A-norm error's
// minimiser, which is what CG reduces).
__global__ __launch_bounds__(256) void k_ls(Lv d, const uint16_t* __restrict__ code, double ihx, double ihy,
                                            double ihz, const float* __restrict__ phat, const float* __restrict__ b,
                                            double* __restrict__ part) {
#pragma clang fp contract(off)
    const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
    double s[4] = {0.0, 0.0, 0.0, 0.0};
    if (c < d.V) {
        const uint16_t cd = code[c];
        if (cd & kFluidBit) {
            const double ih2[3] = {ihx, ihy, ihz};
            const Stride st = stride_of(d.nx, d.ny, d.nz);
            auto val = [&](int64_t q) { return (code[q] & kFluidBit) ? (double)phat[q] : 0.0; };
            const double ph = (double)phat[c];
            const double q = code_apply64(cd, c, st, ih2, ph, val);
            s[0] = (double)b[c] * q;
            s[1] = q * q;
            s[2] = (double)b[c] * ph;
            s[3] = ph * q;
        }
    }
    write_partials<4>(s, part);
}

__global__ __launch_bounds__(256) void k_set_guess(int64_t V, const uint16_t* __restrict__ code,
                                                   const float* __restrict__ phat, double alpha,
                                                   double* __restrict__ p) {
    const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (c >= V) return;
    p[c] = (code[c] & kFluidBit) ? alpha * (double)phat[c] : 0.0;
}

__global__ __launch_bounds__(256) void k_zero_f(int64_t n, float* __restrict__ a) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) a[i] = 0.0f;
}

// ---------------------------------------------------------------------------
// Host drivers
// ---------------------------------------------------------------------------
template <int MT, int NT, int AHEAD>
hipError_t launch_conv_tile(hipStream_t st, const Lv& d, const uint16_t* X, int cin, int cout, const uint16_t* wp,
                            const float* bias, int relu, uint16_t* ybf, float* yf) {
    const dim3 grid((unsigned)((d.V + 64 * MT - 1) / (64 * MT)), (unsigned)(cout / 16 / NT));
    hipLaunchKernelGGL((k_conv<MT, NT, AHEAD>), grid, dim3(256), 0, st, d, X, cin, cout,
                       reinterpret_cast<const u4*>(wp), bias, relu, ybf, yf);
    return hipGetLastError();
}

// Two tiles a wavefront as long as they leave every SIMD one (1024 SIMDs); the
// smallest levels take the most wavefronts, single tiles of an output group
// each.  At 64x96x80, us per launch on the finest level (48 -> 16, 16 -> 48):
// two tiles 92, 64, four 95, 83 (their registers leave fewer waves); 61 440
// voxels (32 -> 32): two 34, one 39.  Steps ahead: two 92, 64, 34; one 101, 62,
// 37; four with two tiles the same as two; single tiles of 7680 voxels (112 ->
// 48 channels) six 18.8, four 19.2.
hipError_t launch_conv(hipStream_t st, const Lv& d, const uint16_t* X, int cin, int cout, const uint16_t* wp,
                       const float* bias, int relu, uint16_t* ybf, float* yf) {
    if (d.V < 32 * 1024) return launch_conv_tile<1, 1, 6>(st, d, X, cin, cout, wp, bias, relu, ybf, yf);
    switch (cout / 16) {
        case 1: return launch_conv_tile<2, 1, 2>(st, d, X, cin, cout, wp, bias, relu, ybf, yf);
        case 2: return launch_conv_tile<2, 2, 2>(st, d, X, cin, cout, wp, bias, relu, ybf, yf);
        case 3: return launch_conv_tile<2, 3, 2>(st, d, X, cin, cout, wp, bias, relu, ybf, yf);
        case 4: return launch_conv_tile<2, 4, 2>(st, d, X, cin, cout, wp, bias, relu, ybf, yf);
        case 5: return launch_conv_tile<2, 5, 2>(st, d, X, cin, cout, wp, bias, relu, ybf, yf);
        case 7: return launch_conv_tile<2, 7, 2>(st, d, X, cin, cout, wp, bias, relu, ybf, yf);
        default: return hipErrorInvalidValue;
    }
}

// Workgroups along the voxels: about 16 waves per CU in all, and a few steps
// (32 voxels each) per wave at least.
struct WgradShape {
    int64_t spw;  // steps per wave
    int blocks;   // partials
};
WgradShape wgrad_shape(const Lv& d, int cin) {
    const int64_t steps = planes_of(d).steps;
    const int64_t want = 4096 / (4 * 3 * (cin / 16)), most = std::max<int64_t>(1, steps / 16);
    const int64_t blocks = std::max<int64_t>(1, std::min(want, most));
    WgradShape w;
    w.spw = (steps + 4 * blocks - 1) / (4 * blocks);
    w.blocks = (int)((steps + 4 * w.spw - 1) / (4 * w.spw));
    return w;
}

hipError_t launch_wgrad(hipStream_t st, const Lv& d, const uint16_t* Xt, int cin, const uint16_t* Gt, int cout,
                        float* part, float* bpart, const WgradShape& w) {
    const dim3 grid((unsigned)w.blocks, (unsigned)(3 * (cin / 16)));
    switch (cout / 16) {
        case 1: hipLaunchKernelGGL(k_wgrad<1>, grid, dim3(256), 0, st, d, cin, Xt, Gt, part, bpart, w.spw); break;
        case 2: hipLaunchKernelGGL(k_wgrad<2>, grid, dim3(256), 0, st, d, cin, Xt, Gt, part, bpart, w.spw); break;
        case 3: hipLaunchKernelGGL(k_wgrad<3>, grid, dim3(256), 0, st, d, cin, Xt, Gt, part, bpart, w.spw); break;
        case 4: hipLaunchKernelGGL(k_wgrad<4>, grid, dim3(256), 0, st, d, cin, Xt, Gt, part, bpart, w.spw); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

int red_blocks(int64_t V) { return (int)std::min<int64_t>((V + 255) / 256, 1 << 30); }

template <typename T>
hipError_t alloc(T** p, int64_t count) {
    *p = nullptr;
    return hipMalloc((void**)p, sizeof(T) * (size_t)std::max<int64_t>(count, 1));
}

template <typename T>
void release(T*& p) {
    if (p) (void)hipFree(p);
    p = nullptr;
}

void free_buffers(fe_net* n) {
    release(n->X0); release(n->E0); release(n->P1); release(n->E1); release(n->P2); release(n->E2);
    release(n->P3); release(n->E3); release(n->C2); release(n->D2); release(n->C1); release(n->D1);
    release(n->C0); release(n->D0); release(n->dpre); release(n->out); release(n->dout); release(n->aq);
    release(n->D0f);
    release(n->gD0); release(n->gC0); release(n->gE0); release(n->gD1); release(n->gC1); release(n->gE1);
    release(n->gP1); release(n->gD2); release(n->gC2); release(n->gE2); release(n->gP2); release(n->gE3);
    release(n->gP3); release(n->wpart); release(n->bpart); release(n->red);
    release(n->in_b); release(n->in_target); release(n->in_loss); release(n->in_flags); release(n->in_code);
    for (int l = 0; l < 4; ++l) {
        release(n->Xt[l]);
        release(n->Gt[l]);
    }
    n->red_cap = 0;
    for (auto& l : n->lv) l = NetLevel{};
}

// layer_back: dpre = mask(gY, Y); dW, db; gX = conv_bwd_data(dpre) when asked
hipError_t layer_back(fe_net* n, int li, const Lv& d, const uint16_t* X, const uint16_t* Y, const float* gY,
                      float* gX) {
    NetLayer& L = n->L[li];
    hipStream_t st = n->stream;
    hipError_t e;
    const dim3 segments((unsigned)((planes_of(d).steps + 1) / 2));  // 8 per workgroup
    uint16_t *Xt = n->Xt[kNetLayerLevel[li]], *Gt = n->Gt[kNetLayerLevel[li]];
    hipLaunchKernelGGL(k_mask, segments, dim3(256), 0, st, d, L.cout, gY, Y, n->dpre, Gt);
    hipLaunchKernelGGL(k_planes, segments, dim3(256), 0, st, d, L.cin, X, Xt);
    const WgradShape w = wgrad_shape(d, L.cin);
    if ((e = launch_wgrad(st, d, Xt, L.cin, Gt, L.cout, n->wpart, n->bpart, w)) != hipSuccess) return e;
    const int64_t wsz = 27LL * L.cin * L.cout;
    hipLaunchKernelGGL(k_reduce_parts, dim3((unsigned)((wsz + L.cout) / 16)), dim3(256), 0, st, w.blocks, wsz,
                       (const float*)n->wpart, L.gw, L.cout, (const float*)n->bpart, L.gb);
    if (gX) return launch_conv(st, d, n->dpre, L.cout, L.cin, L.wpt, nullptr, 0, nullptr, gX);
    return hipGetLastError();
}

hipError_t pack_all(fe_net* n) {
    for (auto& L : n->L) {
        const int64_t sz = std::max(packed_size(L.cin, L.cout), packed_size(L.cout, L.cin));
        hipLaunchKernelGGL(k_pack, g1(sz), dim3(256), 0, n->stream, L.cin, L.cout, (const float*)L.w, L.wp, L.wpt);
    }
    return hipGetLastError();
}

uint64_t splitmix(uint64_t z) {
    z += 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

}  // namespace

int64_t net_param_count() {
    int64_t c = 0;
    for (int i = 0; i < kNetLayers; ++i) c += 27LL * kNetLayerIn[i] * kNetLayerOut[i] + kNetLayerOut[i];
    return c + 17;
}

hipError_t net_alloc(fe_net* n, uint64_t seed) {
    hipError_t e;
    if ((e = hipStreamCreate(&n->stream)) != hipSuccess) return e;
    uint64_t state = seed;
    auto normal = [&]() {  // Box-Muller on SplitMix64 uniforms
        const double u1 = ((splitmix(state++) >> 11) + 1.0) * 0x1.0p-53, u2 = (splitmix(state++) >> 11) * 0x1.0p-53;
        return std::sqrt(-2.0 * std::log(u1)) * std::cos(6.283185307179586 * u2);
    };
    if ((e = alloc(&n->grads, net_param_count())) != hipSuccess) return e;
    float* g = n->grads;
    for (int i = 0; i < kNetLayers; ++i) {
        NetLayer& L = n->L[i];
        L.cin = kNetLayerIn[i];
        L.cout = kNetLayerOut[i];
        const int64_t wsz = 27LL * L.cin * L.cout;
        for (float** p : {&L.w, &L.mw, &L.vw})
            if ((e = alloc(p, wsz)) != hipSuccess) return e;
        for (float** p : {&L.b, &L.mb, &L.vb})
            if ((e = alloc(p, L.cout)) != hipSuccess) return e;
        L.gw = g;
        L.gb = g + wsz;
        g += wsz + L.cout;
        if ((e = alloc(&L.wp, packed_size(L.cin, L.cout))) != hipSuccess ||
            (e = alloc(&L.wpt, packed_size(L.cout, L.cin))) != hipSuccess)
            return e;
        std::vector<float> w((size_t)wsz), z((size_t)wsz, 0.0f), zb((size_t)L.cout, 0.0f);
        const double sd = std::sqrt(2.0 / (27.0 * L.cin));  // He initialisation
        for (auto& x : w) x = (float)(normal() * sd);
        if ((e = hipMemcpy(L.w, w.data(), sizeof(float) * wsz, hipMemcpyHostToDevice)) != hipSuccess) return e;
        for (float* p : {L.mw, L.vw})
            if ((e = hipMemcpy(p, z.data(), sizeof(float) * wsz, hipMemcpyHostToDevice)) != hipSuccess) return e;
        for (float* p : {L.b, L.mb, L.vb})
            if ((e = hipMemcpy(p, zb.data(), sizeof(float) * L.cout, hipMemcpyHostToDevice)) != hipSuccess) return e;
    }
    n->ghead = g;
    for (float** p : {&n->head, &n->mhead, &n->vhead})
        if ((e = alloc(p, 17)) != hipSuccess) return e;
    if ((e = alloc(&n->scal, 8)) != hipSuccess) return e;
    std::vector<float> hd(17, 0.0f), z17(17, 0.0f);
    for (int c = 0; c < 16; ++c) hd[c] = (float)(normal() * 0.25);
    if ((e = hipMemcpy(n->head, hd.data(), sizeof(float) * 17, hipMemcpyHostToDevice)) != hipSuccess) return e;
    for (float* p : {n->mhead, n->vhead})
        if ((e = hipMemcpy(p, z17.data(), sizeof(float) * 17, hipMemcpyHostToDevice)) != hipSuccess) return e;
    if ((e = pack_all(n)) != hipSuccess) return e;
    return hipStreamSynchronize(n->stream);
}

void net_free(fe_net* n) {
    if (n->stream) (void)hipStreamSynchronize(n->stream);
    free_buffers(n);
    for (auto& L : n->L) {
        release(L.w); release(L.b); release(L.mw); release(L.vw);
        release(L.mb); release(L.vb); release(L.wp); release(L.wpt);
    }
    release(n->head); release(n->mhead); release(n->vhead);
    release(n->grads); release(n->scal); release(n->losses);
    for (auto& s : n->samples) {
        release(s.b); release(s.flags); release(s.target); release(s.code);
    }
    n->samples.clear();
    if (n->stream) (void)hipStreamDestroy(n->stream);
    n->stream = nullptr;
}

hipError_t net_get_params(fe_net* n, float* host) {
    hipError_t e;
    for (auto& L : n->L) {
        const int64_t wsz = 27LL * L.cin * L.cout;
        if ((e = hipMemcpy(host, L.w, sizeof(float) * wsz, hipMemcpyDeviceToHost)) != hipSuccess) return e;
        host += wsz;
        if ((e = hipMemcpy(host, L.b, sizeof(float) * L.cout, hipMemcpyDeviceToHost)) != hipSuccess) return e;
        host += L.cout;
    }
    return hipMemcpy(host, n->head, sizeof(float) * 17, hipMemcpyDeviceToHost);
}

hipError_t net_set_params(fe_net* n, const float* host) {
    hipError_t e;
    for (auto& L : n->L) {
        const int64_t wsz = 27LL * L.cin * L.cout;
        if ((e = hipMemcpy(L.w, host, sizeof(float) * wsz, hipMemcpyHostToDevice)) != hipSuccess) return e;
        host += wsz;
        if ((e = hipMemcpy(L.b, host, sizeof(float) * L.cout, hipMemcpyHostToDevice)) != hipSuccess) return e;
        host += L.cout;
    }
    if ((e = hipMemcpy(n->head, host, sizeof(float) * 17, hipMemcpyHostToDevice)) != hipSuccess) return e;
    if ((e = pack_all(n)) != hipSuccess) return e;
    return hipStreamSynchronize(n->stream);
}

hipError_t net_ensure(fe_net* n, const int nn[3]) {
    if (n->lv[0].n[0] == nn[0] && n->lv[0].n[1] == nn[1] && n->lv[0].n[2] == nn[2] && n->X0) return hipSuccess;
    if ((int64_t)nn[0] * nn[1] * nn[2] > kNetMaxVoxels) return hipErrorInvalidConfiguration;
    (void)hipStreamSynchronize(n->stream);
    free_buffers(n);
    for (int l = 0; l < 4; ++l) {
        for (int a = 0; a < 3; ++a) n->lv[l].n[a] = nn[a] >> l;
        n->lv[l].V = (int64_t)n->lv[l].n[0] * n->lv[l].n[1] * n->lv[l].n[2];
    }
    const int64_t V0 = n->lv[0].V, V1 = n->lv[1].V, V2 = n->lv[2].V, V3 = n->lv[3].V;
    hipError_t e;
#define NA(p, cnt)                                     \
    if ((e = alloc(&n->p, (cnt))) != hipSuccess) {     \
        free_buffers(n); /* the next call starts over */ \
        return e;                                      \
    }
    NA(X0, V0 * 16); NA(E0, V0 * 16); NA(P1, V1 * 16); NA(E1, V1 * 32); NA(P2, V2 * 32); NA(E2, V2 * 48);
    NA(P3, V3 * 48); NA(E3, V3 * 64); NA(C2, V2 * 112); NA(D2, V2 * 48); NA(C1, V1 * 80); NA(D1, V1 * 32);
    NA(C0, V0 * 48); NA(D0, V0 * 16);
    NA(dpre, std::max({V0 * 16, V1 * 32, V2 * 48, V3 * 64}));
    NA(out, V0); NA(dout, V0); NA(aq, V0); NA(D0f, V0 * 16);
    NA(gD0, V0 * 16); NA(gC0, V0 * 48); NA(gE0, V0 * 16); NA(gD1, V1 * 32); NA(gC1, V1 * 80); NA(gE1, V1 * 32);
    NA(gP1, V1 * 16); NA(gD2, V2 * 48); NA(gC2, V2 * 112); NA(gE2, V2 * 48); NA(gP2, V2 * 32); NA(gE3, V3 * 64);
    NA(gP3, V3 * 48);
    int64_t wp = 0, bp = 0;
    for (int i = 0; i < kNetLayers; ++i) {
        const int64_t blocks = wgrad_shape(lv_of(n->lv[kNetLayerLevel[i]]), kNetLayerIn[i]).blocks;
        wp = std::max<int64_t>(wp, blocks * 27LL * kNetLayerIn[i] * kNetLayerOut[i]);
        bp = std::max<int64_t>(bp, blocks * kNetLayerOut[i]);
    }
    NA(wpart, wp);
    NA(bpart, bp);
    // the layers of a level share its planes, whose fill and border stay zero
    for (int l = 0; l < 4; ++l) {
        int ci = 0, co = 0;
        for (int i = 0; i < kNetLayers; ++i)
            if (kNetLayerLevel[i] == l) {
                ci = std::max(ci, kNetLayerIn[i]);
                co = std::max(co, kNetLayerOut[i]);
            }
        const Planes P = planes_of(lv_of(n->lv[l]));
        const int64_t xw = ci * P.xn / 2, gw = co * P.gn / 2;  // in 32-bit words
        NA(Xt[l], 2 * xw);
        NA(Gt[l], 2 * gw);
        hipLaunchKernelGGL(k_zero_f, g1(xw), dim3(256), 0, n->stream, xw, reinterpret_cast<float*>(n->Xt[l]));
        hipLaunchKernelGGL(k_zero_f, g1(gw), dim3(256), 0, n->stream, gw, reinterpret_cast<float*>(n->Gt[l]));
    }
    NA(red, (int64_t)red_blocks(V0) * 17);  // at most 17 sums per block
    n->red_cap = (int64_t)red_blocks(V0) * 17;
#undef NA
    return hipSuccess;
}

hipError_t net_forward(fe_net* n, const float* b, const uint8_t* flags, double rms_b) {
    hipStream_t st = n->stream;
    const Lv l0 = lv_of(n->lv[0]), l1 = lv_of(n->lv[1]), l2 = lv_of(n->lv[2]), l3 = lv_of(n->lv[3]);
    hipError_t e;
    hipLaunchKernelGGL(k_features, g1(l0.V), dim3(256), 0, st, l0.V, b, flags, rms_b, n->X0);
    auto conv = [&](int li, const Lv& d, const uint16_t* X, uint16_t* Y) {
        const NetLayer& L = n->L[li];
        return launch_conv(st, d, X, L.cin, L.cout, L.wp, L.b, 1, Y, nullptr);
    };
    if ((e = conv(0, l0, n->X0, n->E0)) != hipSuccess) return e;
    hipLaunchKernelGGL(k_pool<16>, g1(l1.V * (16 / 8)), dim3(256), 0, st, l0, l1, (const uint16_t*)n->E0, n->P1);
    if ((e = conv(1, l1, n->P1, n->E1)) != hipSuccess) return e;
    hipLaunchKernelGGL(k_pool<32>, g1(l2.V * (32 / 8)), dim3(256), 0, st, l1, l2, (const uint16_t*)n->E1, n->P2);
    if ((e = conv(2, l2, n->P2, n->E2)) != hipSuccess) return e;
    hipLaunchKernelGGL(k_pool<48>, g1(l3.V * (48 / 8)), dim3(256), 0, st, l2, l3, (const uint16_t*)n->E2, n->P3);
    if ((e = conv(3, l3, n->P3, n->E3)) != hipSuccess) return e;
    hipLaunchKernelGGL((k_upcat<64, 48>), g1(l2.V * ((64 + 48) / 8)), dim3(256), 0, st, l2, l3, (const uint16_t*)n->E3,
                       (const uint16_t*)n->E2, n->C2);
    if ((e = conv(4, l2, n->C2, n->D2)) != hipSuccess) return e;
    hipLaunchKernelGGL((k_upcat<48, 32>), g1(l1.V * ((48 + 32) / 8)), dim3(256), 0, st, l1, l2, (const uint16_t*)n->D2,
                       (const uint16_t*)n->E1, n->C1);
    if ((e = conv(5, l1, n->C1, n->D1)) != hipSuccess) return e;
    hipLaunchKernelGGL((k_upcat<32, 16>), g1(l0.V * ((32 + 16) / 8)), dim3(256), 0, st, l0, l1, (const uint16_t*)n->D1,
                       (const uint16_t*)n->E0, n->C0);
    {
        const NetLayer& L = n->L[6];
        if ((e = launch_conv(st, l0, n->C0, L.cin, L.cout, L.wp, L.b, 1, n->D0, n->D0f)) != hipSuccess) return e;
    }
    hipLaunchKernelGGL(k_head, g1(l0.V), dim3(256), 0, st, l0.V, (const float*)n->D0f, (const float*)n->head,
                       (const float*)(n->head + 16), n->out);
    return hipGetLastError();
}

hipError_t net_backward(fe_net* n, const LossIn& in, float* loss_slot) {
    hipStream_t st = n->stream;
    const Lv l0 = lv_of(n->lv[0]), l1 = lv_of(n->lv[1]), l2 = lv_of(n->lv[2]), l3 = lv_of(n->lv[3]);
    hipError_t e;
    const int nb = red_blocks(l0.V);
    if (n->loss_mode == 0) {
        const double nf = (double)std::max<int64_t>(in.nfluid, 1);
        hipLaunchKernelGGL(k_loss, dim3(nb), dim3(256), 0, st, l0.V, (const float*)n->out, in.target, in.flags,
                           (float)nf, n->dout, n->red);
        hipLaunchKernelGGL(k_sum_to<1>, dim3(1), dim3(256), 0, st, (const double*)n->red, nb, loss_slot, n->scal,
                           1.0 / nf);
    } else {
        hipLaunchKernelGGL(k_energy_stats, dim3(nb), dim3(256), 0, st, l0, in.code, in.ih2[0], in.ih2[1], in.ih2[2],
                           (const float*)n->out, in.b, n->aq, n->red);
        hipLaunchKernelGGL(k_energy_finish, dim3(1), dim3(256), 0, st, (const double*)n->red, nb, in.energy, loss_slot,
                           n->scal);
        hipLaunchKernelGGL(k_energy_grad, g1(l0.V), dim3(256), 0, st, l0.V, in.code, (const float*)n->aq, in.b,
                           (const double*)n->scal, n->dout);
    }
    hipLaunchKernelGGL(k_head_bwd, dim3(nb), dim3(256), 0, st, l0.V, (const float*)n->D0f, (const float*)n->dout,
                       (const float*)n->head, n->gD0, n->red);
    hipLaunchKernelGGL(k_sum_to<17>, dim3(1), dim3(256), 0, st, (const double*)n->red, nb, n->ghead, (double*)nullptr,
                       1.0);
    // decoder
    if ((e = layer_back(n, 6, l0, n->C0, n->D0, n->gD0, n->gC0)) != hipSuccess) return e;
    hipLaunchKernelGGL((k_up_bwd<32, 16>), g1(l1.V * (32 / 4)), dim3(256), 0, st, l0, l1, (const float*)n->gC0, n->gD1);
    if ((e = layer_back(n, 5, l1, n->C1, n->D1, n->gD1, n->gC1)) != hipSuccess) return e;
    hipLaunchKernelGGL((k_up_bwd<48, 32>), g1(l2.V * (48 / 4)), dim3(256), 0, st, l1, l2, (const float*)n->gC1, n->gD2);
    if ((e = layer_back(n, 4, l2, n->C2, n->D2, n->gD2, n->gC2)) != hipSuccess) return e;
    hipLaunchKernelGGL((k_up_bwd<64, 48>), g1(l3.V * (64 / 4)), dim3(256), 0, st, l2, l3, (const float*)n->gC2, n->gE3);
    // encoder
    if ((e = layer_back(n, 3, l3, n->P3, n->E3, n->gE3, n->gP3)) != hipSuccess) return e;
    hipLaunchKernelGGL((k_enc_bwd<64, 48>), g1(l2.V * (48 / 4)), dim3(256), 0, st, l2, l3, (const float*)n->gC2,
                       (const float*)n->gP3, n->gE2);
    if ((e = layer_back(n, 2, l2, n->P2, n->E2, n->gE2, n->gP2)) != hipSuccess) return e;
    hipLaunchKernelGGL((k_enc_bwd<48, 32>), g1(l1.V * (32 / 4)), dim3(256), 0, st, l1, l2, (const float*)n->gC1,
                       (const float*)n->gP2, n->gE1);
    if ((e = layer_back(n, 1, l1, n->P1, n->E1, n->gE1, n->gP1)) != hipSuccess) return e;
    hipLaunchKernelGGL((k_enc_bwd<32, 16>), g1(l0.V * (16 / 4)), dim3(256), 0, st, l0, l1, (const float*)n->gC0,
                       (const float*)n->gP1, n->gE0);
    if ((e = layer_back(n, 0, l0, n->X0, n->E0, n->gE0, nullptr)) != hipSuccess) return e;
    return hipGetLastError();
}

hipError_t net_adam(fe_net* n, float lr) {
    ++n->adam_t;
    const float bc1 = (float)(1.0 - std::pow(0.9, (double)n->adam_t));
    const float bc2 = (float)(1.0 - std::pow(0.999, (double)n->adam_t));
    hipStream_t st = n->stream;
    for (auto& L : n->L) {
        const int64_t wsz = 27LL * L.cin * L.cout;
        hipLaunchKernelGGL(k_adam, g1(wsz), dim3(256), 0, st, wsz, L.w, (const float*)L.gw, L.mw, L.vw, lr, bc1, bc2);
        hipLaunchKernelGGL(k_adam, g1(L.cout), dim3(256), 0, st, (int64_t)L.cout, L.b, (const float*)L.gb, L.mb, L.vb,
                           lr, bc1, bc2);
    }
    hipLaunchKernelGGL(k_adam, dim3(1), dim3(256), 0, st, (int64_t)17, n->head, (const float*)n->ghead, n->mhead,
                       n->vhead, lr, bc1, bc2);
    return pack_all(n);
}

hipError_t net_add_sample(fe_net* n, fe_scene* s) {
    const int64_t V = cell_count(s->g);
    NetSample smp;
    for (int a = 0; a < 3; ++a) smp.n[a] = s->g.n[a];
    hipError_t e;
    if ((e = alloc(&smp.b, V)) != hipSuccess) return e;
    if ((e = alloc(&smp.flags, V)) != hipSuccess) {
        release(smp.b);
        return e;
    }
    if ((e = alloc(&smp.target, V)) != hipSuccess || (e = alloc(&smp.code, V)) != hipSuccess) {
        release(smp.b);
        release(smp.flags);
        release(smp.target);
        return e;
    }
    for (int a = 0; a < 3; ++a) smp.ih2[a] = s->g.ihd[a] * s->g.ihd[a];
    (void)hipStreamSynchronize(s->stream);
    const int nb = red_blocks(V);
    double* part = nullptr;
    if ((e = alloc(&part, (int64_t)nb * 4 + 4)) != hipSuccess) return e;
    double sums[4] = {0, 0, 0, 0};
    if ((e = hipMemcpyAsync(smp.b, s->b, sizeof(float) * V, hipMemcpyDeviceToDevice, n->stream)) == hipSuccess &&
        (e = hipMemcpyAsync(smp.flags, s->flags, V, hipMemcpyDeviceToDevice, n->stream)) == hipSuccess &&
        (e = hipMemcpyAsync(smp.code, s->code, sizeof(uint16_t) * V, hipMemcpyDeviceToDevice, n->stream)) ==
            hipSuccess) {
        hipLaunchKernelGGL(k_sample_stats<double>, dim3(nb), dim3(256), 0, n->stream, V, (const float*)s->b,
                           (const double*)s->p, (const uint8_t*)s->flags, part);
        hipLaunchKernelGGL(k_sum_to<4>, dim3(1), dim3(256), 0, n->stream, (const double*)part, nb, (float*)nullptr,
                           part + (int64_t)nb * 4, 1.0);
        e = hipMemcpyAsync(sums, part + (int64_t)nb * 4, sizeof(sums), hipMemcpyDeviceToHost, n->stream);
        if (e == hipSuccess) e = hipStreamSynchronize(n->stream);
    }
    if (e == hipSuccess) {
        smp.nfluid = (int64_t)sums[2];
        smp.energy = sums[3];
        smp.rms_b = std::sqrt(sums[0] / (double)V);
        const double rms_p = smp.nfluid > 0 ? std::sqrt(sums[1] / (double)smp.nfluid) : 0.0;
        hipLaunchKernelGGL(k_target, g1(V), dim3(256), 0, n->stream, V, (const double*)s->p,
                           (const uint8_t*)s->flags, rms_p > 0 ? rms_p : 1.0, smp.target);
        e = hipGetLastError();
        if (e == hipSuccess) e = hipStreamSynchronize(n->stream);
    }
    release(part);
    if (e != hipSuccess || !(smp.rms_b > 0) || smp.nfluid == 0 || !(smp.energy > 0)) {
        release(smp.b);
        release(smp.flags);
        release(smp.target);
        release(smp.code);
        return e != hipSuccess ? e : hipErrorInvalidValue;
    }
    n->samples.push_back(smp);
    return hipSuccess;
}

hipError_t net_train(fe_net* n, int steps, float lr, uint64_t seed) {
    if (n->samples.empty() || steps <= 0) return hipErrorInvalidValue;
    hipError_t e;
    if (n->losses_cap < steps) {
        release(n->losses);
        if ((e = alloc(&n->losses, steps)) != hipSuccess) return e;
        n->losses_cap = steps;
    }
    for (int it = 0; it < steps; ++it) {
        const NetSample& smp = n->samples[splitmix(seed + (uint64_t)it) % n->samples.size()];
        if ((e = net_ensure(n, smp.n)) != hipSuccess) return e;
        if ((e = net_forward(n, smp.b, smp.flags, smp.rms_b)) != hipSuccess) return e;
        LossIn in;
        in.target = smp.target;
        in.flags = smp.flags;
        in.nfluid = smp.nfluid;
        in.code = smp.code;
        for (int a = 0; a < 3; ++a) in.ih2[a] = smp.ih2[a];
        in.b = smp.b;
        in.energy = smp.energy;
        if ((e = net_backward(n, in, n->losses + it)) != hipSuccess) return e;
        if ((e = net_adam(n, lr)) != hipSuccess) return e;
    }
    return hipStreamSynchronize(n->stream);
}

hipError_t net_codes(fe_net* n, const int nn[3], const uint8_t* flags, uint16_t* code) {
    const Lv d{nn[0], nn[1], nn[2], (int64_t)nn[0] * nn[1] * nn[2]};
    hipLaunchKernelGGL(k_codes, g1(d.V), dim3(256), 0, n->stream, d, flags, code);
    return hipGetLastError();
}

hipError_t net_fluid_count(fe_net* n, const uint8_t* flags, int64_t V, int64_t* count) {
    const int nb = red_blocks(V);
    double* part = nullptr;
    hipError_t e;
    if ((e = alloc(&part, (int64_t)nb * 4 + 4)) != hipSuccess) return e;
    float* bz = nullptr;
    if ((e = alloc(&bz, V)) != hipSuccess) {
        release(part);
        return e;
    }
    hipLaunchKernelGGL(k_zero_f, g1(V), dim3(256), 0, n->stream, V, bz);
    hipLaunchKernelGGL(k_sample_stats<double>, dim3(nb), dim3(256), 0, n->stream, V, (const float*)bz, (const double*)nullptr,
                       flags, part);
    hipLaunchKernelGGL(k_sum_to<4>, dim3(1), dim3(256), 0, n->stream, (const double*)part, nb, (float*)nullptr,
                       part + (int64_t)nb * 4, 1.0);
    double sums[4] = {0, 0, 0, 0};
    e = hipMemcpyAsync(sums, part + (int64_t)nb * 4, sizeof(sums), hipMemcpyDeviceToHost, n->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(n->stream);
    release(part);
    release(bz);
    *count = (int64_t)sums[2];
    return e;
}

// On the host the sums over b, the target and the flags took 0.6 ms at
// 64x96x80 (491 520 cells), more than half of the device's forward and backward
// pass; one pass here with a 32-byte copy back takes 0.03 ms.
hipError_t net_host_inputs(fe_net* n, const int dims[3], const float* b, const uint8_t* flags, const float* target,
                           LossIn& in, double* rms_b) {
    hipError_t e;
    if ((e = net_ensure(n, dims)) != hipSuccess) return e;
    const int64_t V = n->lv[0].V;
    if (!n->in_loss) {  // the last to be allocated
        release(n->in_b); release(n->in_target); release(n->in_flags); release(n->in_code);
        if ((e = alloc(&n->in_b, V)) != hipSuccess || (e = alloc(&n->in_target, V)) != hipSuccess ||
            (e = alloc(&n->in_flags, V)) != hipSuccess || (e = alloc(&n->in_code, V)) != hipSuccess ||
            (e = alloc(&n->in_loss, 1)) != hipSuccess)
            return e;
    }
    // an earlier call that failed after its launches may have left kernels reading the buffers
    if ((e = hipStreamSynchronize(n->stream)) != hipSuccess ||
        (e = hipMemcpy(n->in_b, b, sizeof(float) * V, hipMemcpyHostToDevice)) != hipSuccess ||
        (e = hipMemcpy(n->in_target, target, sizeof(float) * V, hipMemcpyHostToDevice)) != hipSuccess ||
        (e = hipMemcpy(n->in_flags, flags, V, hipMemcpyHostToDevice)) != hipSuccess)
        return e;
    const int nb = red_blocks(V);
    hipLaunchKernelGGL(k_sample_stats<float>, dim3(nb), dim3(256), 0, n->stream, V, (const float*)n->in_b,
                       (const float*)n->in_target, (const uint8_t*)n->in_flags, n->red);
    hipLaunchKernelGGL(k_sum_to<4>, dim3(1), dim3(256), 0, n->stream, (const double*)n->red, nb, (float*)nullptr,
                       n->scal, 1.0);
    if ((e = net_codes(n, dims, n->in_flags, n->in_code)) != hipSuccess) return e;
    double sums[4] = {0, 0, 0, 0};
    if ((e = hipMemcpyAsync(sums, n->scal, sizeof(sums), hipMemcpyDeviceToHost, n->stream)) != hipSuccess) return e;
    if ((e = hipStreamSynchronize(n->stream)) != hipSuccess) return e;
    *rms_b = std::sqrt(sums[0] / (double)V);
    in.b = n->in_b;
    in.target = n->in_target;
    in.flags = n->in_flags;
    in.code = n->in_code;
    in.nfluid = (int64_t)sums[2];
    in.energy = sums[3];
    return hipSuccess;
}

hipError_t net_warm_start(fe_net* n, fe_scene* s) {
    std::lock_guard<std::mutex> lock(n->mu);
    const Geom& g = s->g;
    const int64_t V = cell_count(g);
    hipError_t e;
    if ((e = net_ensure(n, g.n)) != hipSuccess) return e;
    // the scene's stream has built b and the row codes; the network runs on its own stream after that
    if ((e = hipStreamSynchronize(s->stream)) != hipSuccess) return e;
    const int nb = red_blocks(V);
    hipLaunchKernelGGL(k_sample_stats<double>, dim3(nb), dim3(256), 0, n->stream, V, (const float*)s->b,
                       (const double*)nullptr, (const uint8_t*)s->flags, n->red);
    hipLaunchKernelGGL(k_sum_to<4>, dim3(1), dim3(256), 0, n->stream, (const double*)n->red, nb, (float*)nullptr,
                       n->scal, 1.0);
    double sums[4] = {0, 0, 0, 0};
    if ((e = hipMemcpyAsync(sums, n->scal, sizeof(sums), hipMemcpyDeviceToHost, n->stream)) != hipSuccess) return e;
    if ((e = hipStreamSynchronize(n->stream)) != hipSuccess) return e;
    const double rms_b = std::sqrt(sums[0] / (double)V);
    double alpha = 0.0;
    if (rms_b > 0) {
        if ((e = net_forward(n, s->b, s->flags, rms_b)) != hipSuccess) return e;
        const Lv d{g.n[0], g.n[1], g.n[2], V};
        hipLaunchKernelGGL(k_ls, dim3(nb), dim3(256), 0, n->stream, d, (const uint16_t*)s->code,
                           g.ihd[0] * g.ihd[0], g.ihd[1] * g.ihd[1], g.ihd[2] * g.ihd[2], (const float*)n->out,
                           (const float*)s->b, n->red);
        hipLaunchKernelGGL(k_sum_to<4>, dim3(1), dim3(256), 0, n->stream, (const double*)n->red, nb, (float*)nullptr,
                           n->scal, 1.0);
        double sm[4] = {0, 0, 0, 0};
        if ((e = hipMemcpyAsync(sm, n->scal, sizeof(sm), hipMemcpyDeviceToHost, n->stream)) != hipSuccess) return e;
        if ((e = hipStreamSynchronize(n->stream)) != hipSuccess) return e;
        const double num = n->scale_mode == 0 ? sm[0] : sm[2], den = n->scale_mode == 0 ? sm[1] : sm[3];
        if (den > 0 && std::isfinite(num / den)) alpha = num / den;
    }
    s->net_alpha = alpha;
    hipLaunchKernelGGL(k_set_guess, g1(V), dim3(256), 0, n->stream, V, (const uint16_t*)s->code,
                       (const float*)n->out, alpha, s->p);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    return hipStreamSynchronize(n->stream);
}

}  // namespace fe
