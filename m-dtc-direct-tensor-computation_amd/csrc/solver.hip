// solver.hip -- batched matrix-free Jacobi-PCG for the 24 load cases of HEX08
// voxel domains on gfx950.
//
// Replaces the PETSc path of f-src/mod_dtc_main_subroutines.f90:426-1238:
// MatSetValues assembly of K_e = Hexe08(bone) per element, Dirichlet lifting
// f = -A x_bc with f[bc] = 0, MatZeroRowsColumns(diag 0.0), KSPSolve with
// CG + Jacobi and x0 = 0 for each load case, and the reactions r = A_org u.
//
// Design
//  * Operator: never assembled.  Every element is a voxel with modulus E_v,
//    so K_e = E_v * Khat.  In the signed Walsh basis of the 8 element nodes
//    Khat is block diagonal (3x3, 2x2, 1x1 blocks, 45 coefficients), so one
//    element product costs two 8-point Hadamard butterflies per direction
//    plus 45 multiplies instead of a dense 24x24 product.
//  * Tiling: the lattice of kept nodes is cut into bricks of 8x4x4 nodes, taken
//    along a Z-curve, and runs of them into clusters of at most 128 nodes.  A
//    workgroup computes every element that touches a node of its cluster,
//    adds their outputs up in LDS in a fixed order and writes its nodes once
//    (ebe.hpp).  No atomics, deterministic.
//  * Vectors: node-major [node][3][24], nodes numbered brick by brick so a
//    cluster's nodes are contiguous.  All 24 load cases advance in
//    lockstep with their own alpha/beta; a converged load case freezes.
//  * Reductions: per-brick partial sums in FP64, then one workgroup per
//    domain sums them in brick order (deterministic).
//  * Precision: DTC_FP64 runs PCG in FP64; DTC_FP32_REFINE runs the inner
//    PCG in FP32 on the residual equation and keeps x, the true residual
//    r = -(K u)_free and the reactions in FP64.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <thread>
#include <type_traits>

#include "bc.hpp"
#include "solver.hpp"

namespace dtc {

namespace {

constexpr int R = R24;
constexpr int NT_UPD = 192;    // multiple of 24: a thread keeps one load case

// IN_U: x with the Dirichlet values; IN_JS (FP32 Chebyshev step only): x = cin D^-1 v, the
// first smoothing step from x = 0 formed while reading v, so that it is never stored
enum InMode { IN_V = 0, IN_U = 1, IN_JS = 2 };
enum OutMode { OUT_MASKED_DOT = 0, OUT_RESID = 1, OUT_PLAIN = 2, OUT_MASKED = 3, OUT_CHEB = 4, OUT_BRES = 5 };

template <typename T> struct WK { T g[45]; };

template <typename T> WK<T> cast_wk(const WalshK& w) {
    WK<T> o;
    for (int i = 0; i < 45; ++i) o.g[i] = (T)w.g[i];
    return o;
}

__device__ inline bool is_bc(const DomInfo& D, int gx, int gy, int gz) {
    return gx == 0 || gy == 0 || gz == 0 || gx == D.nx || gy == D.ny || gz == D.nz;
}

__device__ inline void node_coord(const DomInfo& D, int gx, int gy, int gz, double c[3]) {
    c[0] = ((double)gx + D.xa1[0]) * D.delta[0];
    c[1] = ((double)gy + D.xa1[1]) * D.delta[1];
    c[2] = ((double)gz + D.xa1[2]) * D.delta[2];
}

// ---------------------------------------------------------------- element operator
// modes after the forward butterflies: index bit0 <-> x, bit1 <-> y, bit2 <-> z
template <typename T>
__device__ inline void fht_fwd(T v[8]) {
#pragma unroll
    for (int s = 1; s < 8; s <<= 1)
#pragma unroll
        for (int b = 0; b < 8; ++b)
            if (!(b & s)) {
                T a = v[b], c = v[b + s];
                v[b] = a + c;
                v[b + s] = c - a;
            }
}
template <typename T>
__device__ inline void fht_inv(T v[8]) {
#pragma unroll
    for (int s = 1; s < 8; s <<= 1)
#pragma unroll
        for (int b = 0; b < 8; ++b)
            if (!(b & s)) {
                T a = v[b], c = v[b + s];
                v[b] = a - c;
                v[b + s] = a + c;
            }
}
// fht_inv after its first butterfly stage (s = 1)
template <typename T>
__device__ inline void fht_inv_tail(T v[8]) {
#pragma unroll
    for (int s = 2; s < 8; s <<= 1)
#pragma unroll
        for (int b = 0; b < 8; ++b)
            if (!(b & s)) {
                T a = v[b], c = v[b + s];
                v[b] = a - c;
                v[b + s] = a + c;
            }
}

// y = Kw w on the (mode, direction) groups; w, y indexed [mode][dir]
template <typename K, typename T>
__device__ inline void walsh_apply(const WK<K>& k, const T w[8][3], T y[8][3]) {
#define M3(o, i0, d0, i1, d1, i2, d2)                                                         \
    {                                                                                         \
        T a0 = w[i0][d0], a1 = w[i1][d1], a2 = w[i2][d2];                                     \
        y[i0][d0] = k.g[o + 0] * a0 + k.g[o + 1] * a1 + k.g[o + 2] * a2;                      \
        y[i1][d1] = k.g[o + 3] * a0 + k.g[o + 4] * a1 + k.g[o + 5] * a2;                      \
        y[i2][d2] = k.g[o + 6] * a0 + k.g[o + 7] * a1 + k.g[o + 8] * a2;                      \
    }
#define M2(o, i0, d0, i1, d1)                                                                 \
    {                                                                                         \
        T a0 = w[i0][d0], a1 = w[i1][d1];                                                     \
        y[i0][d0] = k.g[o + 0] * a0 + k.g[o + 1] * a1;                                        \
        y[i1][d1] = k.g[o + 2] * a0 + k.g[o + 3] * a1;                                        \
    }
    y[0][0] = y[0][1] = y[0][2] = T(0);
    M3(0, 1, 0, 2, 1, 4, 2)          // x.ux, y.uy, z.uz
    M2(9, 1, 1, 2, 0)                // x.uy, y.ux
    M2(13, 1, 2, 4, 0)               // x.uz, z.ux
    M2(17, 2, 2, 4, 1)               // y.uz, z.uy
    M2(21, 3, 0, 6, 2)               // xy.ux, yz.uz
    M2(25, 3, 1, 5, 2)               // xy.uy, xz.uz
    M3(29, 3, 2, 5, 1, 6, 0)         // xy.uz, xz.uy, yz.ux
    M2(38, 5, 0, 6, 1)               // xz.ux, yz.uy
    y[7][0] = k.g[42] * w[7][0];     // xyz
    y[7][1] = k.g[43] * w[7][1];
    y[7][2] = k.g[44] * w[7][2];
#undef M3
#undef M2
}

// ---------------------------------------------------------------- matvec
// RC load cases of one (node, direction) are one 16-byte vector V (float4 / double2)
template <typename T> struct MvCfg;
template <> struct MvCfg<float> { static constexpr int RC = 4; using V = float4; };
template <> struct MvCfg<double> { static constexpr int RC = 2; using V = double2; };
constexpr int NET = EX * EY * EZ, NO = BX * BY * BZ;   // elements that touch a brick, its nodes

__device__ inline float vcomp(const float4& v, int w) { return w == 0 ? v.x : w == 1 ? v.y : w == 2 ? v.z : v.w; }
__device__ inline double vcomp(const double2& v, int w) { return w == 0 ? v.x : v.y; }
__device__ inline void vzero(float4& v) { v = make_float4(0.f, 0.f, 0.f, 0.f); }
__device__ inline void vzero(double2& v) { v = make_double2(0.0, 0.0); }
__device__ inline float4 vneg(const float4& v) { return make_float4(-v.x, -v.y, -v.z, -v.w); }
__device__ inline double2 vneg(const double2& v) { return make_double2(-v.x, -v.y); }
__device__ inline void vadd(float4& a, const float4& b) { a.x += b.x; a.y += b.y; a.z += b.z; a.w += b.w; }
__device__ inline void vadd(double2& a, const double2& b) { a.x += b.x; a.y += b.y; }

// OUT_CHEB direction handling: the previous direction d is read from dvec
// (CH_READ_D), or equals the current iterate (CH_D_FROM_X: the step after a
// zero-start step, where x_1 = d_0), or is absent (c1 = 0); the new direction
// is stored only when a later step reads it (CH_WRITE_D).
constexpr int CH_READ_D = 1, CH_D_FROM_X = 2, CH_WRITE_D = 4;

// the zero-start smoothing step fused into the next step (DTC_CHEB_FUSE=0: stored by k_cheb)
inline bool cheb_fuse() {
    const char* e = std::getenv("DTC_CHEB_FUSE");
    return !(e && e[0] == '0');
}

#include "ebe.hpp"

// ---------------------------------------------------------------- vector kernels
// One workgroup per brick; a vector row is one (node, direction) pair holding the 24 load
// cases.  Each thread takes 16 bytes of a row (VecN load cases) and keeps its load cases,
// ROW_U rows at a time with their loads issued together: bounded by HBM, or by the
// Infinity Cache for small batches.
template <typename T> constexpr int VecN = 16 / (int)sizeof(T);
template <typename T, int N> struct alignas(16) Vec {
    T v[N];
};
template <typename T, int N> __device__ inline Vec<T, N> vload(const T* p) { return *reinterpret_cast<const Vec<T, N>*>(p); }
template <typename T, int N> __device__ inline void vstore(T* p, const Vec<T, N>& a) { *reinterpret_cast<Vec<T, N>*>(p) = a; }
constexpr int ROW_U = 4;

// rows of the brick taken by this thread: row0, row0 + RPP, ... below row1; load cases lc0 ..
template <int N> struct BrickRows {
    static constexpr int LPR = R / N;          // threads per row
    static constexpr int RPP = NT_UPD / LPR;   // rows per pass
    int64_t row0, row1;
    int lc0;
    __device__ explicit BrickRows(const BrickInfo& B)
        : row0((int64_t)B.node_begin * 3 + (int)threadIdx.x / LPR), row1((int64_t)B.node_end * 3),
          lc0((int)threadIdx.x % LPR * N) {}
    // f(row, u) for the rows of one group; groups of ROW_U rows
    template <typename L, typename F> __device__ void each(L load, F use) const {
        for (int64_t row = row0; row < row1; row += ROW_U * RPP) {
#pragma unroll
            for (int u = 0; u < ROW_U; ++u) load(min(row + u * RPP, row1 - 1), u);   // (the last row again past the end)
#pragma unroll
            for (int u = 0; u < ROW_U; ++u)
                if (row + u * RPP < row1) use(row + u * RPP, u);
        }
    }
    // out[lc] = sum over the brick's threads of acc, in a fixed order
    __device__ void sum(const double (&acc)[N], double* s /* [RPP][R] */, double* __restrict__ out) const {
        const int tid = threadIdx.x;
        __syncthreads();
#pragma unroll
        for (int k = 0; k < N; ++k) s[tid / LPR * R + lc0 + k] = acc[k];
        __syncthreads();
        if (tid < R) {
            double t = 0.0;
#pragma unroll
            for (int g = 0; g < RPP; ++g) t += s[g * R + tid];
            out[tid] = t;
        }
    }
};

template <typename T>
__global__ __launch_bounds__(NT_UPD) void k_cg_init(const BrickInfo* __restrict__ bricks, const int* __restrict__ done,
                                                    const int* __restrict__ active, T* __restrict__ x,
                                                    const T* __restrict__ r, T* __restrict__ p,
                                                    const T* __restrict__ dinv, double* __restrict__ prz,
                                                    double* __restrict__ prr, int zero_x, int set_p,
                                                    const int* __restrict__ keep_p, const T* __restrict__ zin) {
    constexpr int N = VecN<T>;
    using V = Vec<T, N>;
    using Rows = BrickRows<N>;
    __shared__ double s_sum[Rows::RPP * R];
    const BrickInfo B = bricks[blockIdx.x];
    const Rows rows(B);
    double a1[N] = {}, a2[N] = {};
    if (!(done && done[B.dom])) {
        // keep the search direction of a load case still iterating when its
        // residual was replaced; restart it otherwise
        bool act[N], sp[N];
#pragma unroll
        for (int k = 0; k < N; ++k) {
            const int lc = B.dom * R + rows.lc0 + k;
            act[k] = active[lc] != 0;
            sp[k] = act[k] && (set_p || !(keep_p && keep_p[lc]));
        }
        V rv[ROW_U], zv[ROW_U], pv[ROW_U];
        T di[ROW_U];
        rows.each([&](int64_t row, int u) {
            const int64_t o = row * R + rows.lc0;
            rv[u] = vload<T, N>(r + o);
            pv[u] = vload<T, N>(p + o);
            if (zin) zv[u] = vload<T, N>(zin + o);
            else di[u] = dinv[row];
        }, [&](int64_t row, int u) {
            const int64_t o = row * R + rows.lc0;
            V xz;
#pragma unroll
            for (int k = 0; k < N; ++k) {
                const T z = act[k] ? (zin ? zv[u].v[k] : rv[u].v[k] * di[u]) : T(0);
                if (sp[k]) pv[u].v[k] = z;
                xz.v[k] = T(0);
                a1[k] += (double)rv[u].v[k] * (double)z;
                a2[k] += (double)rv[u].v[k] * (double)rv[u].v[k];
            }
            vstore(p + o, pv[u]);
            if (zero_x) vstore(x + o, xz);
        });
    }
    rows.sum(a1, s_sum, prz + (int64_t)blockIdx.x * R);
    rows.sum(a2, s_sum, prr + (int64_t)blockIdx.x * R);
}

// Three 33^3 domains in FP64 (40,000 nodes, 23 MB a vector, six of them moved): 36 -> 23.5 us
// (5.9 TB/s) against one load case per thread; k_cg_dir, three vectors, 36 -> 12.5
template <typename T>
__global__ __launch_bounds__(NT_UPD) void k_cg_update(const BrickInfo* __restrict__ bricks, const int* __restrict__ done,
                                                      const double* __restrict__ alpha, T* __restrict__ x,
                                                      T* __restrict__ r, const T* __restrict__ p,
                                                      const T* __restrict__ q, const T* __restrict__ dinv,
                                                      double* __restrict__ prz, double* __restrict__ prr) {
    constexpr int N = VecN<T>;
    using V = Vec<T, N>;
    using Rows = BrickRows<N>;
    __shared__ double s_sum[Rows::RPP * R];
    const BrickInfo B = bricks[blockIdx.x];
    if (done && done[B.dom]) return;
    const Rows rows(B);
    T a[N];
#pragma unroll
    for (int k = 0; k < N; ++k) a[k] = (T)alpha[B.dom * R + rows.lc0 + k];
    double a1[N] = {}, a2[N] = {};
    V xv[ROW_U], rv[ROW_U], pv[ROW_U], qv[ROW_U];
    T di[ROW_U];
    rows.each([&](int64_t row, int u) {
        const int64_t o = row * R + rows.lc0;
        rv[u] = vload<T, N>(r + o);
        qv[u] = vload<T, N>(q + o);
        xv[u] = vload<T, N>(x + o);
        pv[u] = vload<T, N>(p + o);
        di[u] = dinv[row];
    }, [&](int64_t row, int u) {
        const int64_t o = row * R + rows.lc0;
#pragma unroll
        for (int k = 0; k < N; ++k) {
            T t = rv[u].v[k];
            if (a[k] != T(0)) {      // frozen load cases keep x and r
                t -= a[k] * qv[u].v[k];
                xv[u].v[k] += a[k] * pv[u].v[k];
                rv[u].v[k] = t;
            }
            a1[k] += (double)t * (double)(t * di[u]);
            a2[k] += (double)t * (double)t;
        }
        vstore(x + o, xv[u]);
        vstore(r + o, rv[u]);
    });
    if (prz) rows.sum(a1, s_sum, prz + (int64_t)blockIdx.x * R);
    rows.sum(a2, s_sum, prr + (int64_t)blockIdx.x * R);
}

template <typename T>
__global__ __launch_bounds__(NT_UPD) void k_cg_dir(const BrickInfo* __restrict__ bricks, const int* __restrict__ done,
                                                   const double* __restrict__ beta, const T* __restrict__ r,
                                                   T* __restrict__ p, const T* __restrict__ dinv,
                                                   const T* __restrict__ zin) {
    constexpr int N = VecN<T>;
    using V = Vec<T, N>;
    const BrickInfo B = bricks[blockIdx.x];
    if (done && done[B.dom]) return;
    const BrickRows<N> rows(B);
    T b[N];
#pragma unroll
    for (int k = 0; k < N; ++k) b[k] = (T)beta[B.dom * R + rows.lc0 + k];
    V zv[ROW_U], pv[ROW_U];
    T di[ROW_U];
    rows.each([&](int64_t row, int u) {
        const int64_t o = row * R + rows.lc0;
        zv[u] = vload<T, N>((zin ? zin : r) + o);
        pv[u] = vload<T, N>(p + o);
        di[u] = zin ? T(1) : dinv[row];
    }, [&](int64_t row, int u) {
#pragma unroll
        for (int k = 0; k < N; ++k) pv[u].v[k] = zv[u].v[k] * di[u] + b[k] * pv[u].v[k];
        vstore(p + row * R + rows.lc0, pv[u]);
    });
}

// ---------------------------------------------------------------- per-domain reductions (one block per domain)
// sum over the bricks (clusters, slices) b0..b1-1 of a domain of part[b][lc] for the 24 load
// cases, in a fixed order: thread row g takes b0 + g, b0 + g + 32, ..., eight loads at a
// time (the sum takes as long as its chain of loads), and the rows are added in a tree of
// fixed shape; thread lc < 24 receives the sum of load case lc
constexpr int RED_G = 32, RED_NT = RED_G * R;
__device__ inline double dom_sum24(const double* __restrict__ part, int b0, int b1, double* s_w /* [RED_G][R] */) {
    const int tid = threadIdx.x, g = tid / R, lc = tid % R;
    constexpr int U = 8;
    double t = 0.0;
    for (int b = b0 + g; b < b1; b += U * RED_G) {
        double a[U];
#pragma unroll
        for (int u = 0; u < U; ++u) a[u] = b + u * RED_G < b1 ? part[(int64_t)(b + u * RED_G) * R + lc] : 0.0;
#pragma unroll
        for (int u = 0; u < U; ++u) t += a[u];
    }
    s_w[tid] = t;
    __syncthreads();
    for (int w = RED_G / 2; w > 0; w >>= 1) {
        if (g < w) s_w[tid] += s_w[tid + w * R];
        __syncthreads();
    }
    t = tid < R ? s_w[tid] : 0.0;
    __syncthreads();
    return t;
}

__global__ __launch_bounds__(RED_NT) void k_red_init(const DomInfo* __restrict__ doms, const int* __restrict__ skip,
                                                     const double* __restrict__ prz, const double* __restrict__ prr,
                                                     const double* __restrict__ thr2, int* __restrict__ active,
                                                     double* __restrict__ rz, int* __restrict__ done) {
    __shared__ double s_out[RED_NT];
    const int d = blockIdx.x, tid = threadIdx.x, i = d * R + tid;
    const DomInfo D = doms[d];
    const double z = dom_sum24(prz, D.brick_begin, D.brick_end, s_out);
    const double rr = dom_sum24(prr, D.brick_begin, D.brick_end, s_out);
    if (tid >= 64) return;
    int a = 0;
    if (tid < R) {
        a = (skip && skip[d]) ? 0 : active[i];
        if (a && !(rr > thr2[i])) a = 0;
        active[i] = a;
        rz[i] = z;
    }
    const bool any = __ballot(a != 0) != 0;
    if (tid == 0) done[d] = any ? 0 : 1;
}

__global__ __launch_bounds__(RED_NT) void k_red_alpha(const DomInfo* __restrict__ doms, const int* __restrict__ done,
                                                      const double* __restrict__ ppq, int clus,
                                                      int* __restrict__ active, const double* __restrict__ rz,
                                                      double* __restrict__ alpha) {
    __shared__ double s_out[RED_NT];
    const int d = blockIdx.x, tid = threadIdx.x;
    if (done[d]) return;
    const DomInfo D = doms[d];
    const double pq = dom_sum24(ppq, clus ? D.cl_begin : D.brick_begin, clus ? D.cl_end : D.brick_end, s_out);
    if (tid < R) {
        const int i = d * R + tid;
        double al = 0.0;
        if (active[i]) {
            if (pq > 0.0) al = rz[i] / pq;
            else active[i] = 0;      // breakdown: freeze this load case
        }
        alpha[i] = al;
    }
}

__global__ __launch_bounds__(RED_NT) void k_red_beta(const DomInfo* __restrict__ doms, int* __restrict__ done,
                                                     const double* __restrict__ prz, const double* __restrict__ prr,
                                                     const double* __restrict__ thr2, int* __restrict__ active,
                                                     double* __restrict__ rz, double* __restrict__ beta,
                                                     int64_t* __restrict__ iters, int64_t max_iters) {
    __shared__ double s_out[RED_NT];
    const int d = blockIdx.x, tid = threadIdx.x;
    if (done[d]) return;
    const DomInfo D = doms[d];
    const double z = dom_sum24(prz, D.brick_begin, D.brick_end, s_out);
    const double rr = dom_sum24(prr, D.brick_begin, D.brick_end, s_out);
    if (tid >= 64) return;
    const int i = d * R + tid;
    int a = 0;
    if (tid < R) {
        a = active[i];
        double bt = 0.0;
        if (a) {
            if (!(rr > thr2[i])) a = 0;
            else {
                const double old = rz[i];
                bt = old != 0.0 ? z / old : 0.0;
            }
        }
        active[i] = a;
        rz[i] = z;
        beta[i] = bt;
    }
    const bool any = __ballot(a != 0) != 0;
    if (tid == 0) {
        const int64_t it = iters[d] + 1;
        iters[d] = it;
        if (!any || it >= max_iters) done[d] = 1;
    }
}

// outer (FP64) residual bookkeeping after a RESID pass: rr = ||f - K u||^2 per load case;
// load cases above tol^2 ||f||^2 stay active.  The recursive PCG residual target
// is the larger of (tol/2)^2 ||f||^2 (so the true residual check passes after
// drift) and itol2 * rr (an inner solve reduces the residual it started from by
// at most sqrt(itol2), itol2 per domain; null: no relative target)
__global__ __launch_bounds__(RED_NT) void k_red_outer(const DomInfo* __restrict__ doms, const double* __restrict__ prr,
                                                      int first, double tol2, const double* __restrict__ itol2v,
                                                      double* __restrict__ rr0,
                                                      double* __restrict__ rrcur, int* __restrict__ active64,
                                                      int* __restrict__ active, double* __restrict__ thr2,
                                                      int* __restrict__ done64, int* __restrict__ done) {
    __shared__ double s_out[RED_NT];
    const int d = blockIdx.x, tid = threadIdx.x;
    const DomInfo D = doms[d];
    const double rr = dom_sum24(prr, D.brick_begin, D.brick_end, s_out);
    if (tid >= 64) return;
    const int i = d * R + tid;
    int a = 0;
    if (tid < R) {
        const double itol2 = itol2v ? itol2v[d] : 0.0;
        if (first) rr0[i] = rr;
        const double r0 = rr0[i];
        rrcur[i] = rr;
        a = (r0 > 0.0) && (rr > tol2 * r0);
        active64[i] = a;
        active[i] = a;
        thr2[i] = fmax(0.25 * tol2 * r0, itol2 * rr);
    }
    const bool any = __ballot(a != 0) != 0;
    if (tid == 0) {
        done64[d] = any ? 0 : 1;
        done[d] = any ? 0 : 1;
    }
}

// column scale of the FP32 correction problem: 1 / ||r64|| of the load case
// (rr = ||r64||^2 per load case), 1 without scaling or for a zero residual
__device__ inline double col_scale(const double* __restrict__ rr, int dom, int lc) {
    if (!rr) return 1.0;
    const double v = rr[dom * R + lc];
    return v > 0.0 ? 1.0 / sqrt(v) : 1.0;
}

// r32 = r64 (times its column scale when rr is given), x32 = 0 when given (residual replacement)
__global__ __launch_bounds__(NT_UPD) void k_to32(const BrickInfo* __restrict__ bricks, const int* __restrict__ done,
                                                 const double* __restrict__ r64, float* __restrict__ r32,
                                                 float* __restrict__ x32, const double* __restrict__ rr) {
    const BrickInfo B = bricks[blockIdx.x];
    if (done[B.dom]) return;
    const BrickRows<4> rows(B);
    double sc[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) sc[k] = col_scale(rr, B.dom, rows.lc0 + k);
    Vec<double, 4> v[ROW_U];
    rows.each([&](int64_t row, int u) { v[u] = vload<double, 4>(r64 + row * R + rows.lc0); }, [&](int64_t row, int u) {
        Vec<float, 4> f;
#pragma unroll
        for (int k = 0; k < 4; ++k) f.v[k] = (float)(v[u].v[k] * sc[k]);
        vstore(r32 + row * R + rows.lc0, f);
        if (x32) vstore(x32 + row * R + rows.lc0, Vec<float, 4>{});
    });
}

// x64 += x32 (divided by its column scale when rr is given), x32 = 0 (group
// update of the FP32 correction)
__global__ __launch_bounds__(NT_UPD) void k_acc64(const BrickInfo* __restrict__ bricks, const int* __restrict__ skip,
                                                  float* __restrict__ x32, double* __restrict__ x64,
                                                  const double* __restrict__ rr) {
    const BrickInfo B = bricks[blockIdx.x];
    if (skip[B.dom]) return;
    const BrickRows<4> rows(B);
    double sc[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) sc[k] = 1.0 / col_scale(rr, B.dom, rows.lc0 + k);
    Vec<double, 4> v[ROW_U];
    Vec<float, 4> f[ROW_U];
    rows.each([&](int64_t row, int u) {
        v[u] = vload<double, 4>(x64 + row * R + rows.lc0);
        f[u] = vload<float, 4>(x32 + row * R + rows.lc0);
    }, [&](int64_t row, int u) {
#pragma unroll
        for (int k = 0; k < 4; ++k) v[u].v[k] += (double)f[u].v[k] * sc[k];
        vstore(x64 + row * R + rows.lc0, v[u]);
        vstore(x32 + row * R + rows.lc0, Vec<float, 4>{});
    });
}

// ---------------------------------------------------------------- block PCG
// The 24 load cases of a domain share one Krylov block: block PCG in the
// A-orthogonal form
//   Q = A P,  W = P^T Q,  alpha = W^+ (P^T R),  X += P alpha,  R -= Q alpha,
//   Z = M R,  beta = -W^+ (Q^T Z),  P = Z + P beta.
// A vector row is one (node, direction) pair holding the 24 load cases.
constexpr int GR_NT = 256;          // 4 waves
// Slices of a domain's nodes, one workgroup each in the block's vector kernels: a slice is a
// serial walk over its rows, so a domain is cut into as many as pay (domains alone, 22 / 56 /
// 146 iterations: 512 nodes a slice 12.0 ms at 12^3, 39 at 33^3, 131 at 64^3; 32 nodes, at most
// 512 slices 6.5, 26 and 104; 1024 slices 106).  In a batch that fills the chip the
// longer partial-sum lists cost what the shorter walks give (16 x 64^3: 512 against 508 ms).
// The cut follows from the domain alone, so its sums do not depend on the batch.
constexpr int SLICE_NODES = 32;     // nodes per slice (at least)
constexpr int MAX_SLICES = 512;     // slices per domain (at most)
constexpr int RR = R * R;           // entries of a 24 x 24 coefficient matrix

// Gram partial sums over the rows of one slice of a domain's nodes:
//   g[0] = A^T B, g[1] = A^T C (NGR = 2; not written for NGR = 1), FP64 sums of the
// products of FP32 (or FP64) operands.  Lane (i, j) of a wave keeps rows 3i..3i+2 x
// columns 3j..3j+2.  The workgroup loads blocks of GB_ROWS vector rows of A, B (and C)
// with coalesced 16-byte loads (the next block's loads issued before the current
// block's products) into LDS, where the 8 lanes sharing an address are served by one
// broadcast; wave w takes rows w, w + 4, ... of each block in order, and the waves' sums
// are added in wave order.
constexpr int GB_ROWS = 32;
template <int NGR, typename TA = float, typename TB = float>
__global__ __launch_bounds__(GR_NT) void k_gram(const int4* __restrict__ slices, const int* __restrict__ done,
                                                   const TA* __restrict__ A, const TB* __restrict__ B,
                                                   const TB* __restrict__ C, double* __restrict__ gpart) {
    constexpr int EA = 16 / sizeof(TA), EB = 16 / sizeof(TB);      // elements per 16-byte vector
    constexpr int VA = GB_ROWS * R / EA, VB = GB_ROWS * R / EB;     // 16-byte vectors per block and array
    constexpr int VT = VA + NGR * VB;
    constexpr int NPF = (VT + GR_NT - 1) / GR_NT;                   // prefetch vectors per thread
    __shared__ uint4 sAv[VA];
    __shared__ uint4 sBv[NGR][VB];
    __shared__ double s_g[NGR * RR];
    const int4 sl = slices[blockIdx.x];   // domain, first node, end node
    if (done[sl.x]) return;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int ci = 3 * (lane >> 3), cj = 3 * (lane & 7);
    const int64_t r0 = (int64_t)sl.y * 3, r1 = (int64_t)sl.z * 3;
    double g[NGR][9];
#pragma unroll
    for (int t = 0; t < NGR; ++t)
#pragma unroll
        for (int k = 0; k < 9; ++k) g[t][k] = 0.0;
    uint4 pf[NPF];
    // vector v of block row0: array (0 = A, 1 = B, 2 = C), rows beyond r1 read as zero
    auto load = [&](int64_t row0) {
#pragma unroll
        for (int k = 0; k < NPF; ++k) {
            const int v = tid + k * GR_NT;
            uint4 val = make_uint4(0u, 0u, 0u, 0u);
            if (v < VA) {
                const int64_t e = row0 * R + (int64_t)v * EA;
                if (e < r1 * R) val = reinterpret_cast<const uint4*>(A + e)[0];
            } else if (v < VT) {
                const int w = v - VA, t = w / VB, u = w % VB;
                const int64_t e = row0 * R + (int64_t)u * EB;
                const TB* src = t == 0 ? B : C;
                if (e < r1 * R) val = reinterpret_cast<const uint4*>(src + e)[0];
            }
            pf[k] = val;
        }
    };
    auto store = [&]() {
#pragma unroll
        for (int k = 0; k < NPF; ++k) {
            const int v = tid + k * GR_NT;
            if (v < VA) sAv[v] = pf[k];
            else if (v < VT) sBv[(v - VA) / VB][(v - VA) % VB] = pf[k];
        }
    };
    const TA* sA = reinterpret_cast<const TA*>(sAv);
    if (r0 < r1) load(r0);
    for (int64_t row0 = r0; row0 < r1; row0 += GB_ROWS) {
        __syncthreads();                              // the previous block's products are done
        store();
        __syncthreads();
        if (row0 + GB_ROWS < r1) load(row0 + GB_ROWS);
#pragma unroll 2
        for (int k = 0; k < GB_ROWS / 4; ++k) {
            const int rr = wave + 4 * k;
            if (row0 + rr >= r1) break;
            double ad[3], bd[NGR][3];
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                ad[i] = (double)sA[rr * R + ci + i];
#pragma unroll
                for (int t = 0; t < NGR; ++t) bd[t][i] = (double)reinterpret_cast<const TB*>(sBv[t])[rr * R + cj + i];
            }
#pragma unroll
            for (int t = 0; t < NGR; ++t)
#pragma unroll
                for (int i = 0; i < 3; ++i)
#pragma unroll
                    for (int j = 0; j < 3; ++j) g[t][3 * i + j] = fma(ad[i], bd[t][j], g[t][3 * i + j]);
        }
    }
    __syncthreads();
    for (int w = 0; w < 4; ++w) {
        if (wave == w)
#pragma unroll
            for (int t = 0; t < NGR; ++t)
#pragma unroll
                for (int i = 0; i < 3; ++i)
#pragma unroll
                    for (int j = 0; j < 3; ++j) {
                        const int e = t * RR + (ci + i) * R + cj + j;
                        s_g[e] = w == 0 ? g[t][3 * i + j] : s_g[e] + g[t][3 * i + j];
                    }
        __syncthreads();
    }
    double* out = gpart + (int64_t)blockIdx.x * 2 * RR;
    for (int e = tid; e < NGR * RR; e += GR_NT) out[e] = s_g[e];
}

// gsum[d] = sum over the domain's slices of the Gram partials, in a fixed order: workgroup
// (d, c) sums entries 16c..16c+15; thread row g takes the slices g, g + 64, ..., eight loads
// at a time, and the rows are added in a tree of fixed shape.  (A chain of loads: it takes
// as long as its longest row; 512 slices of a 64^3 domain 12 us with 64 entries a
// workgroup, 4.6 us so.)
constexpr int GS_E = 16, GS_G = 64;
__global__ __launch_bounds__(GS_E * GS_G) void k_gram_sum(const int* __restrict__ dslice, const int* __restrict__ done,
                                                         const double* __restrict__ gpart, double* __restrict__ gsum) {
    __shared__ double s_w[GS_G][GS_E];
    const int d = blockIdx.x;
    if (done[d]) return;
    const int tid = threadIdx.x, g = tid / GS_E, e = (int)blockIdx.y * GS_E + tid % GS_E;
    const int s0 = dslice[d], s1 = dslice[d + 1];
    constexpr int U = 8;
    double t = 0.0;
    for (int s = s0 + g; s < s1; s += U * GS_G) {
        double a[U];
#pragma unroll
        for (int u = 0; u < U; ++u)
            a[u] = s + u * GS_G < s1 ? gpart[(int64_t)(s + u * GS_G) * 2 * RR + e] : 0.0;
#pragma unroll
        for (int u = 0; u < U; ++u) t += a[u];
    }
    s_w[g][tid % GS_E] = t;
    __syncthreads();
    for (int w = GS_G / 2; w > 0; w >>= 1) {
        if (g < w) s_w[g][tid % GS_E] += s_w[g + w][tid % GS_E];
        __syncthreads();
    }
    if (g == 0) gsum[(int64_t)d * 2 * RR + e] = s_w[0][tid];
}

// value of another lane (uniform over the wave)
__device__ inline double lane_f64(double v, int lane) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffll), lane);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
    return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}

#include "bsolve.hpp"

// X += P alpha, R -= Q alpha on the rows of each node slice of a domain (the Gram
// slices; alpha: k_bsolve mode 0), and per-slice sums of r.r per load case.  Of the 6 threads of a row, thread q
// keeps load cases 4q..4q+3.
__global__ __launch_bounds__(NT_UPD) void k_bupdate(const int4* __restrict__ slices, const int* __restrict__ done,
                                                   const float* __restrict__ coef, float* __restrict__ x,
                                                   float* __restrict__ r, const float* __restrict__ p,
                                                   const float* __restrict__ q, double* __restrict__ prr) {
    __shared__ float4 s_c[R * 6];
    __shared__ double s_a[NT_UPD][4];
    __shared__ float4 s_pq[2][NT_UPD / 6][6];   // P and Q rows of the current block
    const int4 sl = slices[blockIdx.x];   // domain, first node, end node
    if (done[sl.x]) return;
    const int tid = threadIdx.x, qd = tid % 6, rw = tid / 6;
    const float4* c4 = reinterpret_cast<const float4*>(coef + (int64_t)sl.x * RR);
    for (int e = tid; e < R * 6; e += NT_UPD) s_c[e] = c4[e];
    double acc[4] = {0.0, 0.0, 0.0, 0.0};
    const int64_t r0 = (int64_t)sl.y * 3, r1 = (int64_t)sl.z * 3;
    // the block's P and Q rows are loaded once (thread t: 16-byte vector t of P and
    // of Q, coalesced) and read from LDS by the 6 threads of a row (a broadcast),
    // instead of every thread loading both whole rows; the next block's vectors are
    // in flight during the current block's products
    constexpr int RB = NT_UPD / 6;   // rows per block (one per row lane)
    float4 pf_p, pf_q;
    auto load = [&](int64_t b0) {
        const int64_t row = b0 + tid / 6;
        pf_p = pf_q = make_float4(0.f, 0.f, 0.f, 0.f);
        if (row < r1) {
            pf_p = reinterpret_cast<const float4*>(p + row * R)[qd];
            pf_q = reinterpret_cast<const float4*>(q + row * R)[qd];
        }
    };
    if (r0 < r1) load(r0);
    for (int64_t b0 = r0; b0 < r1; b0 += RB) {
        __syncthreads();                 // the previous block's reads of s_pq are done (and s_c is set)
        s_pq[0][tid / 6][qd] = pf_p;
        s_pq[1][tid / 6][qd] = pf_q;
        __syncthreads();
        if (b0 + RB < r1) load(b0 + RB);
        const int64_t row = b0 + rw;
        if (row >= r1) continue;
        float4* xr = reinterpret_cast<float4*>(x + row * R) + qd;
        float4* rr = reinterpret_cast<float4*>(r + row * R) + qd;
        float4 xv = *xr, rv = *rr;
#pragma unroll
        for (int c = 0; c < 6; ++c) {
            const float4 pv = s_pq[0][rw][c], qv = s_pq[1][rw][c];
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                const float4 a = s_c[(4 * c + w) * 6 + qd];
                const float pk = vcomp(pv, w), qk = vcomp(qv, w);
                xv.x += pk * a.x; xv.y += pk * a.y; xv.z += pk * a.z; xv.w += pk * a.w;
                rv.x -= qk * a.x; rv.y -= qk * a.y; rv.z -= qk * a.z; rv.w -= qk * a.w;
            }
        }
        *xr = xv;
        *rr = rv;
        acc[0] += (double)rv.x * (double)rv.x;
        acc[1] += (double)rv.y * (double)rv.y;
        acc[2] += (double)rv.z * (double)rv.z;
        acc[3] += (double)rv.w * (double)rv.w;
    }
#pragma unroll
    for (int w = 0; w < 4; ++w) s_a[tid][w] = acc[w];
    __syncthreads();
    if (tid < R) {
        const int qq = tid / 4, w = tid % 4;
        double s = 0.0;
        for (int k = 0; k < NT_UPD / 6; ++k) s += s_a[k * 6 + qq][w];
        prr[(int64_t)blockIdx.x * R + tid] = s;
    }
}

// The FP64 form of k_bupdate (block PCG on FP64 vectors): x += P alpha,
// r -= Q alpha with x, r, Q in FP64 and the directions P in FP32, per-slice r.r.
// Of the 6 threads of a row, thread q keeps load cases 4q..4q+3 (as k_bupdate).
__global__ __launch_bounds__(NT_UPD) void k_bupdate64(const int4* __restrict__ slices, const int* __restrict__ done,
                                                     const float* __restrict__ coef, double* __restrict__ x,
                                                     double* __restrict__ r, const float* __restrict__ p,
                                                     const double* __restrict__ q, double* __restrict__ prr) {
    __shared__ float4 s_c[R * 6];
    __shared__ double s_a[NT_UPD][4];
    __shared__ float4 s_p[NT_UPD / 6][6];      // the block's P rows and
    __shared__ double2 s_q[NT_UPD / 6][12];    // Q rows (staged as in k_bupdate)
    const int4 sl = slices[blockIdx.x];   // domain, first node, end node
    if (done[sl.x]) return;
    const int tid = threadIdx.x, qd = tid % 6, rw = tid / 6;
    const float4* c4 = reinterpret_cast<const float4*>(coef + (int64_t)sl.x * RR);
    for (int e = tid; e < R * 6; e += NT_UPD) s_c[e] = c4[e];
    double acc[4] = {0.0, 0.0, 0.0, 0.0};
    constexpr int RB = NT_UPD / 6;
    const int64_t r0b = (int64_t)sl.y * 3, r1 = (int64_t)sl.z * 3;
    float4 pf_p;
    double2 pf_q[2];
    auto load = [&](int64_t b0) {
        const int64_t row = b0 + tid / 6;
        pf_p = make_float4(0.f, 0.f, 0.f, 0.f);
        pf_q[0] = pf_q[1] = make_double2(0.0, 0.0);
        if (row < r1) {
            pf_p = reinterpret_cast<const float4*>(p + row * R)[qd];
            pf_q[0] = reinterpret_cast<const double2*>(q + row * R)[2 * qd];
            pf_q[1] = reinterpret_cast<const double2*>(q + row * R)[2 * qd + 1];
        }
    };
    if (r0b < r1) load(r0b);
    for (int64_t b0 = r0b; b0 < r1; b0 += RB) {
        __syncthreads();
        s_p[tid / 6][qd] = pf_p;
        s_q[tid / 6][2 * qd] = pf_q[0];
        s_q[tid / 6][2 * qd + 1] = pf_q[1];
        __syncthreads();
        if (b0 + RB < r1) load(b0 + RB);
        const int64_t row = b0 + rw;
        if (row >= r1) continue;
        const float4* pr = s_p[rw];
        const double2* qr = s_q[rw];
        double2* xr = reinterpret_cast<double2*>(x + row * R) + 2 * qd;
        double2* rr = reinterpret_cast<double2*>(r + row * R) + 2 * qd;
        double xv[4], rv[4];
        {
            const double2 x0 = xr[0], x1 = xr[1], r0 = rr[0], r1v = rr[1];
            xv[0] = x0.x; xv[1] = x0.y; xv[2] = x1.x; xv[3] = x1.y;
            rv[0] = r0.x; rv[1] = r0.y; rv[2] = r1v.x; rv[3] = r1v.y;
        }
#pragma unroll
        for (int c = 0; c < 6; ++c) {
            const float4 pv = pr[c];
            const double2 qa = qr[2 * c], qb = qr[2 * c + 1];
            const double qk[4] = {qa.x, qa.y, qb.x, qb.y};
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                const float4 a = s_c[(4 * c + w) * 6 + qd];
                const double pk = (double)vcomp(pv, w);
                xv[0] += pk * (double)a.x; xv[1] += pk * (double)a.y; xv[2] += pk * (double)a.z; xv[3] += pk * (double)a.w;
                rv[0] -= qk[w] * (double)a.x; rv[1] -= qk[w] * (double)a.y;
                rv[2] -= qk[w] * (double)a.z; rv[3] -= qk[w] * (double)a.w;
            }
        }
        xr[0] = make_double2(xv[0], xv[1]);
        xr[1] = make_double2(xv[2], xv[3]);
        rr[0] = make_double2(rv[0], rv[1]);
        rr[1] = make_double2(rv[2], rv[3]);
#pragma unroll
        for (int w = 0; w < 4; ++w) acc[w] += rv[w] * rv[w];
    }
#pragma unroll
    for (int w = 0; w < 4; ++w) s_a[tid][w] = acc[w];
    __syncthreads();
    if (tid < R) {
        const int qq = tid / 4, w = tid % 4;
        double s = 0.0;
        for (int k = 0; k < NT_UPD / 6; ++k) s += s_a[k * 6 + qq][w];
        prr[(int64_t)blockIdx.x * R + tid] = s;
    }
}

// pn = Z + P coef (z null: pn = P coef); pn aliases neither p nor z.  With beta
// (k_bsolve mode 1) the new direction block, with L^-T (mode 2) its orthonormal
// columns
// GRAM: also the per-slice Gram partials pnᵀpn of the rows written (for the
// orthonormalisation that follows): the block's new rows are staged in LDS and wave w
// sums rows w, w + 3, ... of each block, lane (i, j) its 3 x 3 entries, in FP64 (the
// layout of k_gram's partials, another summation order)
template <bool GRAM>
__global__ __launch_bounds__(NT_UPD) void k_bdir(const int4* __restrict__ slices, const int* __restrict__ done,
                                                const float* __restrict__ coef, const float* __restrict__ p,
                                                const float* __restrict__ z, float* __restrict__ pn,
                                                double* __restrict__ gpart) {
    __shared__ float4 s_c[R * 6];
    __shared__ float4 s_p[NT_UPD / 6][6];   // P rows of the current block (staged as in k_bupdate)
    __shared__ float4 s_n[GRAM ? NT_UPD / 6 : 1][6];   // GRAM: the block's new rows
    __shared__ double s_g[GRAM ? RR : 1];
    const int4 sl = slices[blockIdx.x];   // domain, first node, end node
    if (done[sl.x]) return;
    const int tid = threadIdx.x, qd = tid % 6, rw = tid / 6;
    const int wave = tid >> 6, lane = tid & 63, ci = 3 * (lane >> 3), cj = 3 * (lane & 7);
    const float4* c4 = reinterpret_cast<const float4*>(coef + (int64_t)sl.x * RR);
    for (int e = tid; e < R * 6; e += NT_UPD) s_c[e] = c4[e];
    constexpr int RB = NT_UPD / 6, NWV = NT_UPD / 64;
    double g[GRAM ? 9 : 1];
#pragma unroll
    for (int k = 0; k < (GRAM ? 9 : 1); ++k) g[k] = 0.0;
    const int64_t r0 = (int64_t)sl.y * 3, r1 = (int64_t)sl.z * 3;
    float4 pf = make_float4(0.f, 0.f, 0.f, 0.f);
    auto load = [&](int64_t b0) {
        const int64_t row = b0 + tid / 6;
        pf = row < r1 ? reinterpret_cast<const float4*>(p + row * R)[qd] : make_float4(0.f, 0.f, 0.f, 0.f);
    };
    if (r0 < r1) load(r0);
    for (int64_t b0 = r0; b0 < r1; b0 += RB) {
        __syncthreads();
        s_p[tid / 6][qd] = pf;
        __syncthreads();
        if (b0 + RB < r1) load(b0 + RB);
        const int64_t row = b0 + rw;
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (row < r1) {
            if (z) v = reinterpret_cast<const float4*>(z + row * R)[qd];
#pragma unroll
            for (int c = 0; c < 6; ++c) {
                const float4 pv = s_p[rw][c];
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    const float4 a = s_c[(4 * c + w) * 6 + qd];
                    const float pk = vcomp(pv, w);
                    v.x += pk * a.x; v.y += pk * a.y; v.z += pk * a.z; v.w += pk * a.w;
                }
            }
            reinterpret_cast<float4*>(pn + row * R)[qd] = v;
        }
        if constexpr (GRAM) {
            s_n[rw][qd] = v;   // rows past the slice hold zeros
            __syncthreads();
            const float* sn = reinterpret_cast<const float*>(s_n);
            for (int rr = wave; rr < RB; rr += NWV) {
                double ad[3], bd[3];
#pragma unroll
                for (int i = 0; i < 3; ++i) {
                    ad[i] = (double)sn[rr * R + ci + i];
                    bd[i] = (double)sn[rr * R + cj + i];
                }
#pragma unroll
                for (int i = 0; i < 3; ++i)
#pragma unroll
                    for (int j = 0; j < 3; ++j) g[3 * i + j] = fma(ad[i], bd[j], g[3 * i + j]);
            }
        }
    }
    if constexpr (GRAM) {
        __syncthreads();
        for (int w = 0; w < NWV; ++w) {
            if (wave == w)
#pragma unroll
                for (int i = 0; i < 3; ++i)
#pragma unroll
                    for (int j = 0; j < 3; ++j) {
                        const int e = (ci + i) * R + cj + j;
                        s_g[e] = w == 0 ? g[3 * i + j] : s_g[e] + g[3 * i + j];
                    }
            __syncthreads();
        }
        double* out = gpart + (int64_t)blockIdx.x * 2 * RR;
        for (int e = tid; e < RR; e += NT_UPD) out[e] = s_g[e];
    }
}

// Where a domain's next phase between residual replacements ends at the latest: the first
// (and with FP64 vectors every) phase runs to its target or to the cap of all domains; a
// later one that has not got there after one and a half times the first one's iterations
// has lost its Krylov space to FP32 rounding (seen with clusters that hang on single
// voxels) and gains from the restart: a 64^3 domain, 73 iterations in the first phase, took 1004
// in all with phases of up to 400, 215 with the second one ended after 100.  Ends before the
// first phase's length cost far more: its directions are not resolved by then (1680 with 60).
__global__ void k_phase(const int64_t* __restrict__ iters, int n, int phase, int64_t* __restrict__ len0,
                        int64_t* __restrict__ phase_end) {
    const int d = blockIdx.x * blockDim.x + threadIdx.x;
    if (d >= n) return;
    if (phase == 1) len0[d] = iters[d];
    phase_end[d] = phase <= 0 ? INT64_MAX : iters[d] + len0[d] + len0[d] / 2 + 16;
}

// per domain: the inner block iteration has finished when every load case's
// recursive residual (scaled back by its column scale, see k_to32) is at or
// below its target (a non-finite one is not), at the end of its phase (k_phase), or at the
// iteration cap
__global__ __launch_bounds__(RED_NT) void k_bcheck(const int* __restrict__ dslice, int* __restrict__ done,
                                                  const double* __restrict__ prr, const double* __restrict__ thr2,
                                                  const double* __restrict__ rrcur, int64_t* __restrict__ iters,
                                                  const int64_t* __restrict__ phase_end, int64_t max_iters) {
    __shared__ double s_out[RED_NT];
    const int d = blockIdx.x, tid = threadIdx.x;
    if (done[d]) return;
    const double rr = dom_sum24(prr, dslice[d], dslice[d + 1], s_out);   // per-slice partials of k_bupdate
    if (tid >= 64) return;
    bool left = false;
    if (tid < R) {
        const double sc = col_scale(rrcur, d, tid);
        left = !(rr <= thr2[d * R + tid] * sc * sc);
    }
    const bool any = __ballot(left) != 0;
    if (tid == 0) {
        const int64_t it = iters[d] + 1;
        iters[d] = it;
        if (!any || it >= max_iters || it >= phase_end[d]) done[d] = 1;
    }
}

// algorithmic bytes of one timed launch: over the domains not done, vpass
// vectors (FP32, or FP64 with fp64), the element moduli (4 or 8 bytes each) and,
// with jac, the FP32 Jacobi scaling; and its dense element-product flops
// 2 (3 nen)^2 R N_e; dom_bytes[d] = {V32, E32, J32, V64, F}.  out = {bytes, flops},
// each summed by one workgroup in a fixed order.
__global__ __launch_bounds__(256) void k_launch_bytes(const int* __restrict__ done, const double* __restrict__ dom_bytes,
                                                      int n_dom, int vpass, int fp64, int jac, double* __restrict__ out) {
    __shared__ double sh[2][256];
    double acc = 0.0, fl = 0.0;
    for (int d = threadIdx.x; d < n_dom; d += 256) {
        if (done && done[d]) continue;
        const double* q = dom_bytes + 5 * d;
        acc += vpass * (fp64 ? q[3] : q[0]) + (fp64 ? 2.0 : 1.0) * q[1] + (jac ? q[2] : 0.0);
        fl += q[4];
    }
    sh[0][threadIdx.x] = acc;
    sh[1][threadIdx.x] = fl;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (threadIdx.x < w) {
            sh[0][threadIdx.x] += sh[0][threadIdx.x + w];
            sh[1][threadIdx.x] += sh[1][threadIdx.x + w];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        out[0] = sh[0][0];
        out[1] = sh[1][0];
    }
}

__global__ void k_fill_f64(double* __restrict__ a, int64_t n, double v) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) a[i] = v;
}
__global__ void k_fill_f32(float* __restrict__ a, int64_t n, float v) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) a[i] = v;
}
__global__ void k_fill_i32b(int* __restrict__ a, int64_t n, int v) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) a[i] = v;
}
__global__ void k_fill_i64(int64_t* __restrict__ a, int64_t n, int64_t v) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) a[i] = v;
}

// ---------------------------------------------------------------- topology
// nodes of every brick of the lattice, and those on the box faces (page-locked host memory)
__global__ void k_brick_count(const int* __restrict__ numLat, const int* __restrict__ keepN, int Lx, int Ly,
                              int Lz, int bnx, int bny, int2* __restrict__ cnt) {
    __shared__ int s[2];
    const int b = blockIdx.x, t = threadIdx.x;     // blockDim = BX*BY*BZ
    if (t < 2) s[t] = 0;
    __syncthreads();
    const int bx = b % bnx, by = (b / bnx) % bny, bz = b / (bnx * bny);
    const int gx = bx * BX + t % BX, gy = by * BY + (t / BX) % BY, gz = bz * BZ + t / (BX * BY);
    if (gx < Lx && gy < Ly && gz < Lz) {
        int num = numLat[gx + Lx * (gy + Ly * gz)];
        if (num > 0 && keepN[num - 1]) {
            atomicAdd(&s[0], 1);
            if (gx == 0 || gy == 0 || gz == 0 || gx == Lx - 1 || gy == Ly - 1 || gz == Lz - 1) atomicAdd(&s[1], 1);
        }
    }
    __syncthreads();
    if (t == 0) cnt[b] = make_int2(s[0], s[1]);
}

__global__ void k_brick_assign(const BrickInfo* __restrict__ bl, int brick0, const int* __restrict__ numLat,
                               const int* __restrict__ keepN, const int* __restrict__ cref, int Lx, int Ly, int Lz,
                               int64_t lat_off, int* __restrict__ lat2node, int* __restrict__ sol2ref) {
    constexpr int NO = BX * BY * BZ;
    __shared__ int flag[NO];
    const BrickInfo B = bl[brick0 + blockIdx.x];
    const int t = threadIdx.x;
    const int gx = B.x0 + t % BX, gy = B.y0 + (t / BX) % BY, gz = B.z0 + t / (BX * BY);
    int kept = 0, num = 0;
    if (gx < Lx && gy < Ly && gz < Lz) {
        num = numLat[gx + Lx * (gy + Ly * gz)];
        kept = (num > 0 && keepN[num - 1]) ? 1 : 0;
    }
    flag[t] = kept;
    __syncthreads();
    if (kept) {
        int rank = 0;
        for (int k = 0; k < t; ++k) rank += flag[k];   // lexicographic order inside the brick
        int s = B.node_begin + rank;
        lat2node[lat_off + gx + (int64_t)Lx * (gy + (int64_t)Ly * gz)] = s;
        sol2ref[s] = cref[num - 1] + 1;
    }
}

// element modulus of every voxel; escale folds a domain's edge length a into
// the modulus (K_e is linear in a), so one Walsh table serves the batch
__global__ void k_emod(const int* __restrict__ keepE, const double* __restrict__ modulus, double E, double escale,
                       int64_t nvox, double* __restrict__ emod) {
    int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nvox) return;
    emod[v] = keepE[v] ? (modulus ? modulus[v] : E) * escale : 0.0;
}

// Jacobi: diag(K)_node,d = kdiag * sum of the moduli of the adjacent elements
__global__ void k_dinv(const BrickInfo* __restrict__ bricks, const DomInfo* __restrict__ doms,
                       const int* __restrict__ lat2node, const double* __restrict__ emod, double kdiag,
                       double* __restrict__ d64, float* __restrict__ d32) {
    const BrickInfo B = bricks[blockIdx.x];
    const DomInfo D = doms[B.dom];
    const int t = threadIdx.x;
    const int gx = B.x0 + t % BX, gy = B.y0 + (t / BX) % BY, gz = B.z0 + t / (BX * BY);
    const int Lx = D.nx + 1, Ly = D.ny + 1, Lz = D.nz + 1;
    if (gx >= Lx || gy >= Ly || gz >= Lz) return;
    int q = lat2node[D.lat_off + gx + (int64_t)Lx * (gy + (int64_t)Ly * gz)];
    if (q < 0) return;
    double s = 0.0;
    for (int dz = -1; dz <= 0; ++dz)
        for (int dy = -1; dy <= 0; ++dy)
            for (int dx = -1; dx <= 0; ++dx) {
                int vx = gx + dx, vy = gy + dy, vz = gz + dz;
                if (vx < 0 || vy < 0 || vz < 0 || vx >= D.nx || vy >= D.ny || vz >= D.nz) continue;
                s += emod[D.vox_off + vx + (int64_t)D.nx * (vy + (int64_t)D.ny * vz)];
            }
    double dg = kdiag * s;
    double inv = dg != 0.0 ? 1.0 / dg : 1.0;   // PCJACOBI uses 1 for a zero diagonal
    if (is_bc(D, gx, gy, gz)) inv = 0.0;        // constrained DOFs stay zero
    for (int d = 0; d < 3; ++d) {              // one value per DOF (isotropic for the HEX08 voxel)
        if (d64) d64[3 * q + d] = inv;   // (the finest level only)
        d32[3 * q + d] = (float)inv;
    }
}

// ---------------------------------------------------------------- force projection
// ff(d*NEN + l, lc) = sum over owned nodes r_d(node, lc) N_l(xi(node))
// (f-src/mod_struct_calcmat.f90:254-280) with the NEN macro shape functions;
// partial per brick [brick][24 lc][FFD]; bricks of the other macro order are skipped
constexpr int FFD = 60;   // macro DOF slots of the force partials (3 x 20)

template <int NEN>
__global__ __launch_bounds__(NT_UPD) void k_project(const BrickInfo* __restrict__ bricks, const DomInfo* __restrict__ doms,
                                                    const int* __restrict__ lat2node, const double* __restrict__ rf,
                                                    double* __restrict__ pff) {
    constexpr int G = NT_UPD / R;    // 8 node groups
    constexpr int FD = 3 * NEN, PASS = 12;
    __shared__ double s[G][R][PASS];
    const BrickInfo B = bricks[blockIdx.x];
    const DomInfo D = doms[B.dom];
    if (macro_nodes(D.macro_order) != NEN) return;
    const int tid = threadIdx.x, lc = tid % R, g = tid / R;
    const int Lx = D.nx + 1, Ly = D.ny + 1;
    double acc[FD];
#pragma unroll
    for (int k = 0; k < FD; ++k) acc[k] = 0.0;
    for (int o = g; o < BX * BY * BZ; o += G) {
        int gx = B.x0 + o % BX, gy = B.y0 + (o / BX) % BY, gz = B.z0 + o / (BX * BY);
        if (gx > D.nx || gy > D.ny || gz > D.nz) continue;
        int q = lat2node[D.lat_off + gx + (int64_t)Lx * (gy + (int64_t)Ly * gz)];
        if (q < 0) continue;
        double c[3], N[20];
        node_coord(D, gx, gy, gz, c);
        macro_shape(D.macro_order, c, D.min_c, D.max_c, N);
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            double rv = rf[((int64_t)q * 3 + d) * R + lc];
#pragma unroll
            for (int l = 0; l < NEN; ++l) acc[d * NEN + l] += rv * N[l];
        }
    }
#pragma unroll
    for (int k0 = 0; k0 < FD; k0 += PASS) {
#pragma unroll
        for (int k = 0; k < PASS; ++k) s[g][lc][k] = k0 + k < FD ? acc[k0 + k] : 0.0;
        __syncthreads();
        for (int i = tid; i < R * PASS; i += NT_UPD) {
            const int l2 = i / PASS, k = i % PASS;
            if (k0 + k >= FD) continue;
            double v = 0.0;
            for (int gg = 0; gg < G; ++gg) v += s[gg][l2][k];
            pff[((int64_t)blockIdx.x * R + l2) * FFD + k0 + k] = v;
        }
        __syncthreads();
    }
}

// ff[d] = sum over the domain's bricks of the force partials: workgroup (d, g) takes
// entries 32 g .. 32 g + 31 of the R x FFD block; its 8 thread rows sum every 8th
// brick, and the 8 row sums are added in row order (fixed order)
constexpr int RFF_E = 32, RFF_P = 8;   // entries per workgroup, brick partitions
__global__ __launch_bounds__(RFF_E * RFF_P) void k_red_ff(const DomInfo* __restrict__ doms,
                                                         const double* __restrict__ pff, double* __restrict__ ff) {
    __shared__ double s_p[RFF_P][RFF_E];
    const int d = blockIdx.x;
    const DomInfo D = doms[d];
    const int FD = 3 * macro_nodes(D.macro_order);
    const int e = threadIdx.x % RFF_E, part = threadIdx.x / RFF_E;
    const int i = (int)blockIdx.y * RFF_E + e;
    double v = 0.0;
    if (i < R * FFD && i % FFD < FD)
        for (int b = D.brick_begin + part; b < D.brick_end; b += RFF_P) v += pff[(int64_t)b * R * FFD + i];
    s_p[part][e] = v;
    __syncthreads();
    if (part == 0 && i < R * FFD) {
        double t = 0.0;
        for (int k = 0; k < RFF_P; ++k) t += s_p[k][e];
        ff[(int64_t)d * R * FFD + i] = t;
    }
}

// u (mesh numbering) = x + x_bc, column-major (3N, ncol): load cases lc_base ..
// lc_base + ncol - 1 of the domain's group
__global__ __launch_bounds__(NT_UPD) void k_fields(const BrickInfo* __restrict__ bricks, const DomInfo* __restrict__ doms,
                                                   const int* __restrict__ lat2node, const int* __restrict__ sol2ref,
                                                   const double* __restrict__ x, const double* __restrict__ rf,
                                                   int dom, int64_t nn, int ncol, double* __restrict__ uo,
                                                   double* __restrict__ ro) {
    const BrickInfo B = bricks[blockIdx.x];
    if (B.dom != dom) return;
    const DomInfo D = doms[B.dom];
    const int Lx = D.nx + 1, Ly = D.ny + 1;
    for (int i = threadIdx.x; i < BX * BY * BZ * 3 * R; i += NT_UPD) {
        int o = i / (3 * R), rem = i % (3 * R), d = rem / R, lc = rem % R;
        if (lc >= ncol) continue;
        int gx = B.x0 + o % BX, gy = B.y0 + (o / BX) % BY, gz = B.z0 + o / (BX * BY);
        if (gx > D.nx || gy > D.ny || gz > D.nz) continue;
        int q = lat2node[D.lat_off + gx + (int64_t)Lx * (gy + (int64_t)Ly * gz)];
        if (q < 0) continue;
        int64_t ref = sol2ref[q] - 1;
        int64_t out = (3 * ref + d) + 3 * nn * lc;
        double v = x[((int64_t)q * 3 + d) * R + lc];
        if (is_bc(D, gx, gy, gz)) {
            double c[3], N[20];
            node_coord(D, gx, gy, gz, c);
            macro_shape(D.macro_order, c, D.min_c, D.max_c, N);
            v = bc_value_m(D.macro_order, N, d, D.lc_base + lc);
        }
        if (uo) uo[out] = v;
        if (ro) ro[out] = rf[((int64_t)q * 3 + d) * R + lc];
    }
}

// ---------------------------------------------------------------- sensitivity
// h[node][j][d] (+)= sum_lc M[lc][j] u_lc(node, d), u = x + x_bc, over the load cases
// of domain group dom (M: its 24 rows); h is indexed by the node numbers of group
// h_begin's range (the groups of one domain share one mesh and its numbering),
// add = 0 for the first group
__global__ __launch_bounds__(NT_UPD) void k_grad_h(const BrickInfo* __restrict__ bricks, const DomInfo* __restrict__ doms,
                                                   const int* __restrict__ lat2node, const double* __restrict__ x,
                                                   const double* __restrict__ Mj, int dom, int64_t h_begin, int add,
                                                   double* __restrict__ h) {
    const BrickInfo B = bricks[blockIdx.x];
    if (B.dom != dom) return;
    const DomInfo D = doms[B.dom];
    const int Lx = D.nx + 1, Ly = D.ny + 1;
    for (int i = threadIdx.x; i < BX * BY * BZ * 18; i += NT_UPD) {
        int o = i / 18, j = (i % 18) / 3, d = i % 3;
        int gx = B.x0 + o % BX, gy = B.y0 + (o / BX) % BY, gz = B.z0 + o / (BX * BY);
        if (gx > D.nx || gy > D.ny || gz > D.nz) continue;
        int q = lat2node[D.lat_off + gx + (int64_t)Lx * (gy + (int64_t)Ly * gz)];
        if (q < 0) continue;
        bool bc = is_bc(D, gx, gy, gz);
        double N[20];
        if (bc) {
            double c[3];
            node_coord(D, gx, gy, gz, c);
            macro_shape(D.macro_order, c, D.min_c, D.max_c, N);
        }
        double s = 0.0;
        for (int lc = 0; lc < R; ++lc) {
            double u = bc ? bc_value_m(D.macro_order, N, d, D.lc_base + lc) : x[((int64_t)q * 3 + d) * R + lc];
            s += Mj[lc * 6 + j] * u;
        }
        double* hp = h + ((q - D.node_begin + h_begin) * 6 + j) * 3 + d;
        *hp = add ? *hp + s : s;
    }
}

__device__ inline double u_at(const DomInfo& D, const int* lat2node, const double* x, int gx, int gy, int gz, int d,
                              int lc) {
    const int Lx = D.nx + 1, Ly = D.ny + 1;
    int q = lat2node[D.lat_off + gx + (int64_t)Lx * (gy + (int64_t)Ly * gz)];
    if (q < 0) return 0.0;
    if (is_bc(D, gx, gy, gz)) {
        double c[3], N[20];
        node_coord(D, gx, gy, gz, c);
        macro_shape(D.macro_order, c, D.min_c, D.max_c, N);
        return bc_value_m(D.macro_order, N, d, D.lc_base + lc);
    }
    return x[((int64_t)q * 3 + d) * R + lc];
}

// dL/dE_v = sum_j h_j,e^T Khat u_j,e for every voxel of domain dom
__global__ void k_grad_elem(const DomInfo* __restrict__ doms, const int* __restrict__ lat2node,
                            const double* __restrict__ emod, const double* __restrict__ x,
                            const double* __restrict__ h, WK<double> wk, int dom, double* __restrict__ g) {
    const DomInfo D = doms[dom];
    const int64_t nvox = (int64_t)D.nx * D.ny * D.nz;
    int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nvox) return;
    double out = 0.0;
    if (emod[D.vox_off + v] != 0.0) {
        const int vx = v % D.nx, vy = (v / D.nx) % D.ny, vz = v / ((int64_t)D.nx * D.ny);
        const int Lx = D.nx + 1, Ly = D.ny + 1;
        int qb[8];
#pragma unroll
        for (int b = 0; b < 8; ++b)
            qb[b] = lat2node[D.lat_off + (vx + (b & 1)) + (int64_t)Lx * ((vy + ((b >> 1) & 1)) + (int64_t)Ly * (vz + (b >> 2)))];
        for (int j = 0; j < 6; ++j) {
            double w[8][3], y[8][3];
            for (int d = 0; d < 3; ++d) {
                double t[8];
                for (int b = 0; b < 8; ++b)
                    t[b] = u_at(D, lat2node, x, vx + (b & 1), vy + ((b >> 1) & 1), vz + (b >> 2), d, j);
                fht_fwd(t);
                for (int b = 0; b < 8; ++b) w[b][d] = t[b];
            }
            walsh_apply(wk, w, y);
            for (int d = 0; d < 3; ++d) {
                double t[8];
                for (int b = 0; b < 8; ++b) t[b] = y[b][d];
                fht_inv(t);
                for (int b = 0; b < 8; ++b)
                    if (qb[b] >= 0) out += t[b] * h[((int64_t)qb[b] * 6 + j) * 3 + d];
            }
        }
    }
    g[v] = out;
}

// ---------------------------------------------------------------- multigrid (FP32 preconditioner)
// Level l+1 has voxels of 2x2x2 voxels of level l.  Its voxel modulus is the sum
// of the 8 children / 4: their mean times 2, because the element stiffness is
// linear in the edge length and the Walsh table is the one of the fine edge.
__global__ void k_coarsen(const double* __restrict__ ef, int fx, int fy, int fz, double* __restrict__ ec, int cx,
                          int cy, int cz) {
    const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= (int64_t)cx * cy * cz) return;
    const int x = (int)(v % cx), y = (int)((v / cx) % cy), z = (int)(v / ((int64_t)cx * cy));
    double s = 0.0;
    for (int k = 0; k < 2; ++k)
        for (int j = 0; j < 2; ++j)
            for (int i = 0; i < 2; ++i) {
                const int X = 2 * x + i, Y = 2 * y + j, Z = 2 * z + k;
                if (X < fx && Y < fy && Z < fz) s += ef[X + (int64_t)fx * (Y + (int64_t)fy * Z)];
            }
    ec[v] = 0.25 * s;
}

// lattice node flag: 1 if a voxel touching the node carries a modulus
__global__ void k_exist(const double* __restrict__ e, int nx, int ny, int nz, int* __restrict__ ex) {
    const int Lx = nx + 1, Ly = ny + 1, Lz = nz + 1;
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= (int64_t)Lx * Ly * Lz) return;
    const int x = (int)(p % Lx), y = (int)((p / Lx) % Ly), z = (int)(p / ((int64_t)Lx * Ly));
    int f = 0;
    for (int dz = -1; dz <= 0; ++dz)
        for (int dy = -1; dy <= 0; ++dy)
            for (int dx = -1; dx <= 0; ++dx) {
                const int vx = x + dx, vy = y + dy, vz = z + dz;
                if (vx < 0 || vy < 0 || vz < 0 || vx >= nx || vy >= ny || vz >= nz) continue;
                if (e[vx + (int64_t)nx * (vy + (int64_t)ny * vz)] != 0.0) f = 1;
            }
    ex[p] = f;
}

// nodes per brick from a node flag array (blockDim = BX*BY*BZ)
__global__ void k_brick_count_ex(const int* __restrict__ ex, int Lx, int Ly, int Lz, int bnx, int bny,
                                 int* __restrict__ cnt) {
    __shared__ int s;
    const int b = blockIdx.x, t = threadIdx.x;
    if (t == 0) s = 0;
    __syncthreads();
    const int bx = b % bnx, by = (b / bnx) % bny, bz = b / (bnx * bny);
    const int gx = bx * BX + t % BX, gy = by * BY + (t / BX) % BY, gz = bz * BZ + t / (BX * BY);
    if (gx < Lx && gy < Ly && gz < Lz && ex[gx + Lx * (gy + Ly * gz)]) atomicAdd(&s, 1);
    __syncthreads();
    if (t == 0) cnt[b] = s;
}

// solver node numbers of the flagged nodes, lexicographic inside each brick
__global__ void k_brick_assign_ex(const BrickInfo* __restrict__ bl, const int* __restrict__ ex, int Lx, int Ly, int Lz,
                                  int64_t lat_off, int* __restrict__ lat2node) {
    __shared__ int flag[NO];
    const BrickInfo B = bl[blockIdx.x];
    const int t = threadIdx.x;
    const int gx = B.x0 + t % BX, gy = B.y0 + (t / BX) % BY, gz = B.z0 + t / (BX * BY);
    int f = 0;
    if (gx < Lx && gy < Ly && gz < Lz) f = ex[gx + Lx * (gy + Ly * gz)];
    flag[t] = f;
    __syncthreads();
    if (f) {
        int rank = 0;
        for (int k = 0; k < t; ++k) rank += flag[k];
        lat2node[lat_off + gx + (int64_t)Lx * (gy + (int64_t)Ly * gz)] = B.node_begin + rank;
    }
}

// ---- transfers between levels
// Every transfer is, per node of its output, a weighted sum over a few nodes of its
// input; which ones is written once per set-up into a table row per node (T_ROW ints).
// 18 lanes per node, each lane one float4 = 4 load cases of one direction.
//   T_RESTRICT   b_c = P^T r_f, trilinear weights over the 3^3 fine nodes around (free ones)
//   T_PROLONG    x_f += P x_c, the mean of 1, 2, 4 or 8 coarse nodes
//   T_PRESTRICT  HEX20 -> HEX08: the corner node and half of its (up to 6) mid-edge ones
//   T_PPROLONG   HEX08 -> HEX20: the corner node, or the mean of an edge's two ends
// Rows: input nodes; -1: none, -2 (prolongations): counted in the mean, but without a
// node.  A Dirichlet node's row is all -1.
enum TransferKind { T_RESTRICT = 0, T_PROLONG = 1, T_PRESTRICT = 2, T_PPROLONG = 3 };
__host__ __device__ constexpr int t_row(int kind) { return kind == T_RESTRICT ? 28 : kind == T_PPROLONG ? 2 : 8; }
__host__ __device__ constexpr int t_terms(int kind) {
    return kind == T_RESTRICT ? 27 : kind == T_PROLONG ? 8 : kind == T_PRESTRICT ? 7 : 2;
}
constexpr int T_LPN = 3 * R / 4;           // float4 per node
constexpr int T_NPP = 256 / T_LPN;         // nodes per pass of a 256-thread workgroup

__device__ inline void f4_axpy(float4& s, float w, const float4& a) {
    s.x += w * a.x; s.y += w * a.y; s.z += w * a.z; s.w += w * a.w;
}

// One workgroup per (brick of the output, blockIdx.y-th share of its nodes).  All loads of a
// node are issued together: a missing node's lane loads node 0 and selects zero (it takes
// no part in any product).  Memory latency bounds the small levels, HBM the large ones.
// Sixteen 64^3 trabecular domains (1.05 M fine nodes), us per launch against lattice look-ups
// staged in LDS per brick: restriction 221 -> 152 and 64 -> 37 (second level), prolongation
// 240 -> 219 and 60 -> 57 (600 MB of the 700 MB it moves are x_f, read and written: 3 TB/s);
// a 48^3 greyscale domain 22.6 -> 11 and 13.5 -> 11.6; HEX20 prolongation (27^3) 43 -> 5.
template <int KIND>
__global__ __launch_bounds__(256) void k_transfer(const BrickInfo* __restrict__ bricks, const int* __restrict__ tab,
                                                  const int* __restrict__ done, const float* __restrict__ x,
                                                  float* __restrict__ y) {
    constexpr int K = t_terms(KIND), ROW = t_row(KIND);
    constexpr bool ADD = KIND == T_PROLONG || KIND == T_PPROLONG;
    const BrickInfo B = bricks[blockIdx.x];
    if (done && done[B.dom]) return;
    const int tid = threadIdx.x;
    if (tid >= T_NPP * T_LPN) return;
    const int slot = tid / T_LPN, j = tid % T_LPN;
    const float4* x4 = reinterpret_cast<const float4*>(x);
    float4* y4 = reinterpret_cast<float4*>(y);
    for (int q = B.node_begin + slot + (int)blockIdx.y * T_NPP; q < B.node_end; q += T_NPP * (int)gridDim.y) {
        int id[ROW];
        if constexpr (ROW % 4 == 0) {
#pragma unroll
            for (int k = 0; k < ROW; k += 4) {
                const int4 v = reinterpret_cast<const int4*>(tab)[(int64_t)q * (ROW / 4) + k / 4];
                id[k] = v.x; id[k + 1] = v.y; id[k + 2] = v.z; id[k + 3] = v.w;
            }
        } else {
            const int2 v = reinterpret_cast<const int2*>(tab)[q];
            id[0] = v.x;
            id[1] = v.y;
        }
        float4 old;
        if (ADD) old = y4[(int64_t)q * T_LPN + j];
        float4 v[K];
#pragma unroll
        for (int k = 0; k < K; ++k) v[k] = x4[(int64_t)max(id[k], 0) * T_LPN + j];
        float4 sum = make_float4(0.f, 0.f, 0.f, 0.f);
        int cnt = 0;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const bool on = id[k] >= 0;
            const float4 a = make_float4(on ? v[k].x : 0.f, on ? v[k].y : 0.f, on ? v[k].z : 0.f, on ? v[k].w : 0.f);
            if constexpr (KIND == T_RESTRICT) {
                constexpr float W[3] = {0.5f, 1.f, 0.5f};
                f4_axpy(sum, W[k % 3] * W[(k / 3) % 3] * W[k / 9], a);
            } else {
                f4_axpy(sum, KIND == T_PRESTRICT && k > 0 ? 0.5f : 1.f, a);
                cnt += id[k] != -1;
            }
        }
        if constexpr (ADD) {
            if (cnt == 0) continue;   // Dirichlet
            f4_axpy(old, cnt == 1 ? 1.f : cnt == 2 ? 0.5f : cnt == 4 ? 0.25f : 0.125f, sum);
            sum = old;
        }
        y4[(int64_t)q * T_LPN + j] = sum;
    }
}

// lattice position of a brick's thread t (t < NO) and its node, -1 outside
__device__ inline int brick_node(const BrickInfo& B, const DomInfo& D, const int* __restrict__ l2n, int t, int g[3]) {
    g[0] = B.x0 + t % BX;
    g[1] = B.y0 + (t / BX) % BY;
    g[2] = B.z0 + t / (BX * BY);
    if (g[0] > D.nx || g[1] > D.ny || g[2] > D.nz) return -1;
    return l2n[D.lat_off + g[0] + (int64_t)(D.nx + 1) * (g[1] + (int64_t)(D.ny + 1) * g[2])];
}

// T_RESTRICT rows of the coarse nodes (one workgroup of NO threads per coarse brick)
__global__ void k_rtab(const BrickInfo* __restrict__ cbr, const DomInfo* __restrict__ cdom, const int* __restrict__ cl2n,
                       const DomInfo* __restrict__ fdom, const int* __restrict__ fl2n, int* __restrict__ tab) {
    const BrickInfo B = cbr[blockIdx.x];
    const DomInfo C = cdom[B.dom], F = fdom[B.dom];
    int g[3];
    const int q = brick_node(B, C, cl2n, threadIdx.x, g);
    if (q < 0) return;
    int* row = tab + (int64_t)q * t_row(T_RESTRICT);
    const bool bc = is_bc(C, g[0], g[1], g[2]);
    for (int k = 0; k < t_row(T_RESTRICT); ++k) {
        const int X = 2 * g[0] + k % 3 - 1, Y = 2 * g[1] + (k / 3) % 3 - 1, Z = 2 * g[2] + k / 9 - 1;
        int f = -1;
        if (!bc && k < 27 && X > 0 && Y > 0 && Z > 0 && X < F.nx && Y < F.ny && Z < F.nz)   // free fine node
            f = fl2n[F.lat_off + X + (int64_t)(F.nx + 1) * (Y + (int64_t)(F.ny + 1) * Z)];
        row[k] = f;
    }
}

// T_PROLONG rows of the fine nodes (one workgroup of NO threads per fine brick)
__global__ void k_ptab(const BrickInfo* __restrict__ fbr, const DomInfo* __restrict__ fdom, const int* __restrict__ fl2n,
                       const DomInfo* __restrict__ cdom, const int* __restrict__ cl2n, int* __restrict__ tab) {
    const BrickInfo B = fbr[blockIdx.x];
    const DomInfo F = fdom[B.dom], C = cdom[B.dom];
    int g[3];
    const int q = brick_node(B, F, fl2n, threadIdx.x, g);
    if (q < 0) return;
    int* row = tab + (int64_t)q * t_row(T_PROLONG);
    const bool bc = is_bc(F, g[0], g[1], g[2]);
    for (int k = 0; k < 8; ++k) {
        const int i = k & 1, j = (k >> 1) & 1, l = k >> 2;
        int c = -1;
        if (!bc && !(i && !(g[0] & 1)) && !(j && !(g[1] & 1)) && !(l && !(g[2] & 1))) {
            const int X = (g[0] >> 1) + i, Y = (g[1] >> 1) + j, Z = (g[2] >> 1) + l;
            if (X <= C.nx && Y <= C.ny && Z <= C.nz)
                c = cl2n[C.lat_off + X + (int64_t)(C.nx + 1) * (Y + (int64_t)(C.ny + 1) * Z)];
            if (c < 0) c = -2;
        }
        row[k] = c;
    }
}

// one Chebyshev-Jacobi step on the owned nodes of each brick:
//   zero:      d = c2 D^-1 b,              x = d        (first step from x = 0; t unused)
//   otherwise: d = c1 d + c2 D^-1 (b - t), x = x + d    (t = A x)
// d == null: the new direction is not stored (zero start: it equals x).
// prz (optional): per-brick sums of b . x per load case
__global__ __launch_bounds__(NT_UPD) void k_cheb(const BrickInfo* __restrict__ bricks, const int* __restrict__ done,
                                                 const float* __restrict__ b, const float* __restrict__ t,
                                                 const float* __restrict__ dinv, float* __restrict__ d,
                                                 float* __restrict__ x, float c1, float c2, int zero,
                                                 double* __restrict__ prz) {
    using V = Vec<float, 4>;
    using Rows = BrickRows<4>;
    __shared__ double s_sum[Rows::RPP * R];
    const BrickInfo B = bricks[blockIdx.x];
    if (done && done[B.dom]) return;
    const Rows rows(B);
    double a1[4] = {};
    V bv[ROW_U], dv[ROW_U], tv[ROW_U], xv[ROW_U];
    float di[ROW_U];
    rows.each([&](int64_t row, int u) {
        const int64_t o = row * R + rows.lc0;
        bv[u] = vload<float, 4>(b + o);
        di[u] = dinv[row];
        if (!zero) {
            dv[u] = vload<float, 4>(d + o);
            tv[u] = vload<float, 4>(t + o);
            xv[u] = vload<float, 4>(x + o);
        }
    }, [&](int64_t row, int u) {
        const int64_t o = row * R + rows.lc0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const float bk = bv[u].v[k];
            if (zero) {
                dv[u].v[k] = c2 * di[u] * bk;
                xv[u].v[k] = dv[u].v[k];
            } else {
                dv[u].v[k] = cheb_dir(c1, dv[u].v[k], c2, di[u], bk, tv[u].v[k]);
                xv[u].v[k] += dv[u].v[k];
            }
            a1[k] += (double)bk * (double)xv[u].v[k];
        }
        if (d) vstore(d + o, dv[u]);
        vstore(x + o, xv[u]);
    });
    if (prz) rows.sum(a1, s_sum, prz + (int64_t)blockIdx.x * R);
}

// ---------------------------------------------------------------- p-multigrid transfers (HEX20 -> HEX08)
// The HEX20 nodes of a voxel mesh sit on the half-voxel lattice: corners at even
// coordinates (the HEX08 nodes of the same voxels), mid-edge nodes with one odd
// coordinate.  P (HEX08 -> HEX20) is the trilinear interpolation of the HEX08
// element: identity at corners, the mean of the edge's two ends at a mid-edge
// node.  Restriction is P^T in gather form, in a fixed order per coarse node.

// T_PRESTRICT rows of the HEX08 twin's nodes of one domain group (one thread per lattice
// point): its corner node and the mid-edge nodes around it on the half-voxel lattice
__global__ void k_pmg_rtab(Dom20Dev G, DomInfo D08, const int* __restrict__ lat2node08, int* __restrict__ tab) {
    const int Lx = D08.nx + 1, Ly = D08.ny + 1, Lz = D08.nz + 1;
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= (int64_t)Lx * Ly * Lz) return;
    const int c = lat2node08[D08.lat_off + p];
    if (c < 0) return;
    const int f[3] = {2 * (int)(p % Lx), 2 * (int)((p / Lx) % Ly), 2 * (int)(p / ((int64_t)Lx * Ly))};
    auto fine = [&](int x, int y, int z) -> int {
        if (x < 0 || y < 0 || z < 0 || x >= G.Lx || y >= G.Ly || z >= G.Lz) return -1;
        const int q = G.lat20[x + (int64_t)G.Lx * (y + (int64_t)G.Ly * z)];
        return q < 0 ? -1 : (int)(G.node_begin + q);
    };
    int* row = tab + (int64_t)c * t_row(T_PRESTRICT);
    const int q0 = fine(f[0], f[1], f[2]);
    const bool bc = q0 >= 0 && G.bcf[q0 - G.node_begin];
    row[0] = bc ? -1 : q0;
    for (int k = 0; k < 6; ++k) {
        const int dx = k == 0 ? -1 : k == 1 ? 1 : 0, dy = k == 2 ? -1 : k == 3 ? 1 : 0, dz = k == 4 ? -1 : k == 5 ? 1 : 0;
        row[1 + k] = bc ? -1 : fine(f[0] + dx, f[1] + dy, f[2] + dz);
    }
    row[7] = -1;
}

// T_PPROLONG rows of the HEX20 nodes: the HEX08 node at a corner, an edge's two ends
__global__ void k_pmg_ptab(const BrickInfo* __restrict__ bricks, const DomInfo* __restrict__ doms,
                           const Dom20Dev* __restrict__ d20, const DomInfo* __restrict__ doms08,
                           const int* __restrict__ lat2node08, int* __restrict__ tab) {
    const BrickInfo B = bricks[blockIdx.x];
    const DomInfo D = doms[B.dom], C = doms08[B.dom];
    const Dom20Dev G = d20[B.dom];
    const int Lx = C.nx + 1, Ly = C.ny + 1;
    for (int q = B.node_begin + (int)threadIdx.x; q < B.node_end; q += blockDim.x) {
        const int ql = (int)(q - G.node_begin);
        int c[2] = {-1, -1};
        if (!G.bcf[ql]) {
            int lo[3], odd = -1;
            for (int k = 0; k < 3; ++k) {
                const int l = (int)lrint(2.0 * (G.coords[3 * ql + k] / D.delta[k] - D.xa1[k]));
                if (l & 1) odd = k;
                lo[k] = l >> 1;
            }
            for (int k = 0; k < (odd >= 0 ? 2 : 1); ++k) {
                if (k) lo[odd] += 1;
                c[k] = lat2node08[C.lat_off + lo[0] + (int64_t)Lx * (lo[1] + (int64_t)Ly * lo[2])];
                if (c[k] < 0) c[k] = -2;
            }
        }
        tab[2 * (int64_t)q] = c[0];
        tab[2 * (int64_t)q + 1] = c[1];
    }
}

// per-brick sums of a . b per load case
template <typename T>
__global__ __launch_bounds__(NT_UPD) void k_dot(const BrickInfo* __restrict__ bricks, const int* __restrict__ done,
                                                const T* __restrict__ a, const T* __restrict__ b,
                                                double* __restrict__ part) {
    constexpr int N = VecN<T>;
    using Rows = BrickRows<N>;
    __shared__ double s_sum[Rows::RPP * R];
    const BrickInfo B = bricks[blockIdx.x];
    if (done && done[B.dom]) return;
    const Rows rows(B);
    double acc[N] = {};
    Vec<T, N> av[ROW_U], bv[ROW_U];
    rows.each([&](int64_t row, int u) {
        av[u] = vload<T, N>(a + row * R + rows.lc0);
        bv[u] = vload<T, N>(b + row * R + rows.lc0);
    }, [&](int64_t, int u) {
#pragma unroll
        for (int k = 0; k < N; ++k) acc[k] += (double)av[u].v[k] * (double)bv[u].v[k];
    });
    rows.sum(acc, s_sum, part + (int64_t)blockIdx.x * R);
}

// x = Dirichlet values on the box-face nodes of each brick, unchanged elsewhere;
// blockIdx.y takes a share of the brick's positions
__global__ __launch_bounds__(NT_UPD) void k_set_bc(const BrickInfo* __restrict__ bricks, const DomInfo* __restrict__ doms,
                                                   const int* __restrict__ lat2node, double* __restrict__ x) {
    const BrickInfo B = bricks[blockIdx.x];
    const DomInfo D = doms[B.dom];
    if (B.x0 != 0 && B.y0 != 0 && B.z0 != 0 && B.x0 + BX <= D.nx && B.y0 + BY <= D.ny && B.z0 + BZ <= D.nz) return;
    const int Lx = D.nx + 1, Ly = D.ny + 1;
    const int lc = threadIdx.x % R;
    for (int o = threadIdx.x / R + NT_UPD / R * (int)blockIdx.y; o < BX * BY * BZ; o += NT_UPD / R * (int)gridDim.y) {
        const int gx = B.x0 + o % BX, gy = B.y0 + (o / BX) % BY, gz = B.z0 + o / (BX * BY);
        if (gx > D.nx || gy > D.ny || gz > D.nz || !is_bc(D, gx, gy, gz)) continue;
        const int q = lat2node[D.lat_off + gx + (int64_t)Lx * (gy + (int64_t)Ly * gz)];
        if (q < 0) continue;
        double c[3], N[20];
        node_coord(D, gx, gy, gz, c);
        macro_shape(D.macro_order, c, D.min_c, D.max_c, N);
        for (int d = 0; d < 3; ++d)
            x[((int64_t)q * 3 + d) * R + lc] = bc_value_m(D.macro_order, N, d, D.lc_base + lc);
    }
}

inline unsigned nb(int64_t n, int t) { return (unsigned)((n + t - 1) / t); }

// Grids of fewer than FILL_BLOCKS workgroups leave CUs idle: the transfer kernels then
// split each brick's nodes over blockIdx.y
constexpr int FILL_BLOCKS = 2048;
inline int node_split(int n_bricks) {
    const int want = n_bricks > 0 ? (FILL_BLOCKS + n_bricks - 1) / n_bricks : 1;
    return want < 1 ? 1 : want > 8 ? 8 : want;
}

}  // namespace

// ---------------------------------------------------------------- host side
int element_stiffness(int nen, double E, double nu, double a, double* K) {
    if (nen != 8) return set_error(DTC_ERR_UNSUPPORTED, "element stiffness: only HEX08 is implemented here");
    if (!(a > 0.0) || !(nu > -1.0 && nu < 0.5)) return set_error(DTC_ERR_BAD_ARGUMENT, "element stiffness: a=%g nu=%g", a, nu);
    const int nd = 24;
    double D[6][6] = {};
    const double lam = E * nu / ((1.0 + nu) * (1.0 - 2.0 * nu)), mu = E / (2.0 * (1.0 + nu));
    for (int i = 0; i < 3; ++i) for (int j = 0; j < 3; ++j) D[i][j] = lam;
    for (int i = 0; i < 3; ++i) D[i][i] += 2.0 * mu;
    D[3][3] = D[4][4] = D[5][5] = mu;
    std::memset(K, 0, sizeof(double) * nd * nd);
    const double g = 1.0 / std::sqrt(3.0), jac = 2.0 / a, detJ = (a / 2.0) * (a / 2.0) * (a / 2.0);
    for (int qi = 0; qi < 8; ++qi) {
        const double q[3] = {(qi & 1) ? g : -g, (qi & 2) ? g : -g, (qi & 4) ? g : -g};
        double B[6][24] = {};
        for (int l = 0; l < 8; ++l) {
            const double sx = 2.0 * h08_off(l, 0) - 1, sy = 2.0 * h08_off(l, 1) - 1, sz = 2.0 * h08_off(l, 2) - 1;
            const double dx = sx * (1 + sy * q[1]) * (1 + sz * q[2]) / 8.0 * jac;
            const double dy = (1 + sx * q[0]) * sy * (1 + sz * q[2]) / 8.0 * jac;
            const double dz = (1 + sx * q[0]) * (1 + sy * q[1]) * sz / 8.0 * jac;
            B[0][3 * l] = dx; B[1][3 * l + 1] = dy; B[2][3 * l + 2] = dz;
            B[3][3 * l] = dy; B[3][3 * l + 1] = dx;
            B[4][3 * l] = dz; B[4][3 * l + 2] = dx;
            B[5][3 * l + 1] = dz; B[5][3 * l + 2] = dy;
        }
        for (int r = 0; r < nd; ++r)
            for (int c = 0; c < nd; ++c) {
                double s = 0.0;
                for (int m = 0; m < 6; ++m)
                    for (int p = 0; p < 6; ++p) s += B[m][r] * D[m][p] * B[p][c];
                K[r + nd * c] += detJ * s;
            }
    }
    return DTC_OK;
}

int walsh_blocks(const double* Khat, WalshK* out) {
    // node l <-> bit index b = ox + 2 oy + 4 oz; H[m][b] = prod over set bits i of m of (2 bit_i(b) - 1)
    int l_of_b[8];
    for (int l = 0; l < 8; ++l) l_of_b[h08_off(l, 0) + 2 * h08_off(l, 1) + 4 * h08_off(l, 2)] = l;
    auto H = [](int m, int b) {
        double s = 1.0;
        for (int i = 0; i < 3; ++i)
            if (m & (1 << i)) s *= ((b >> i) & 1) ? 1.0 : -1.0;
        return s;
    };
    // Kw[(m,d),(m',d')] = sum H[m][b] Khat[(l(b),d),(l(b'),d')] H[m'][b'] / 64
    double Kw[24][24];
    double kmax = 0.0;
    for (int m = 0; m < 8; ++m)
        for (int d = 0; d < 3; ++d)
            for (int m2 = 0; m2 < 8; ++m2)
                for (int d2 = 0; d2 < 3; ++d2) {
                    double s = 0.0;
                    for (int b = 0; b < 8; ++b)
                        for (int b2 = 0; b2 < 8; ++b2)
                            s += H(m, b) * Khat[(3 * l_of_b[b] + d) + 24 * (3 * l_of_b[b2] + d2)] * H(m2, b2);
                    Kw[3 * m + d][3 * m2 + d2] = s / 64.0;
                    kmax = std::fmax(kmax, std::fabs(s / 64.0));
                }
    // groups in the order walsh_apply reads them
    const int groups[11][3][2] = {
        {{1, 0}, {2, 1}, {4, 2}}, {{1, 1}, {2, 0}, {-1, 0}}, {{1, 2}, {4, 0}, {-1, 0}}, {{2, 2}, {4, 1}, {-1, 0}},
        {{3, 0}, {6, 2}, {-1, 0}}, {{3, 1}, {5, 2}, {-1, 0}}, {{3, 2}, {5, 1}, {6, 0}}, {{5, 0}, {6, 1}, {-1, 0}},
        {{7, 0}, {-1, 0}, {-1, 0}}, {{7, 1}, {-1, 0}, {-1, 0}}, {{7, 2}, {-1, 0}, {-1, 0}}};
    int grp_of[24];
    for (int i = 0; i < 24; ++i) grp_of[i] = -1;
    int o = 0;
    for (int g = 0; g < 11; ++g) {
        int n = 0;
        while (n < 3 && groups[g][n][0] >= 0) ++n;
        for (int i = 0; i < n; ++i) grp_of[3 * groups[g][i][0] + groups[g][i][1]] = g;
        for (int i = 0; i < n; ++i)
            for (int j = 0; j < n; ++j)
                out->g[o++] = Kw[3 * groups[g][i][0] + groups[g][i][1]][3 * groups[g][j][0] + groups[g][j][1]];
    }
    if (o != 45) return set_error(DTC_ERR_DEVICE, "walsh_blocks: %d coefficients", o);
    for (int i = 0; i < 24; ++i)
        for (int j = 0; j < 24; ++j)
            if ((grp_of[i] < 0 || grp_of[i] != grp_of[j]) && std::fabs(Kw[i][j]) > 1e-12 * kmax)
                return set_error(DTC_ERR_UNSUPPORTED, "element stiffness is not block diagonal in the Walsh basis");
    return DTC_OK;
}

int batch_begin(SolverBatch& b, const dtc_domain_desc* d, int64_t n_dom) {
    int64_t nlat = 0, nvox = 0;
    for (int64_t i = 0; i < n_dom; ++i) {
        nlat += (d[i].n[0] + 1) * (d[i].n[1] + 1) * (d[i].n[2] + 1);
        nvox += d[i].n[0] * d[i].n[1] * d[i].n[2];
    }
    DTC_TRY(b.lat2node.ensure((size_t)nlat * 4));
    DTC_TRY(b.sol2ref.ensure((size_t)nlat * 4));
    DTC_TRY(b.emod.ensure((size_t)nvox * 8));
    k_fill_i32b<<<nb(nlat, 256), 256, 0, b.stream>>>(b.lat2node.as<int>(), nlat, -1);
    k_fill_f64<<<nb(nvox, 256), 256, 0, b.stream>>>(b.emod.as<double>(), nvox, 0.0);
    DTC_HIP(hipGetLastError());
    b.n_dom = 0; b.n_nodes = 0; b.n_lat = 0; b.n_vox = 0;
    b.h_dom.clear(); b.h_brick.clear(); b.h_elems.clear(); b.h_nodes.clear(); b.h_bnodes.clear(); b.h_status.clear();
    b.h_contrast.clear();
    b.n_slices = 0;   // the block PCG slices follow the batch's domains (block_setup)
    // captured with the previous composition's buffers, and filled by them
    if (b.block_graph.e || !b.d20.empty()) {
        DTC_HIP(stream_wait(b.stream));
        b.block_graph.reset();
        Recycle idle(true);
        b.d20.clear();
    }
    return DTC_OK;
}

// Empty or failed domains keep a DomInfo with no bricks so indices stay aligned.
int batch_add_empty(SolverBatch& b, const dtc_domain_desc& d, int status, int lc_base) {
    DomInfo D{};
    D.nx = (int)d.n[0]; D.ny = (int)d.n[1]; D.nz = (int)d.n[2];
    D.macro_order = d.macro_order;
    D.lc_base = lc_base;
    D.brick_begin = D.brick_end = (int)b.h_brick.size();
    D.node_begin = D.node_end = b.n_nodes;
    D.lat_off = b.n_lat; D.vox_off = b.n_vox;
    b.h_dom.push_back(D);
    b.n_lat += (d.n[0] + 1) * (d.n[1] + 1) * (d.n[2] + 1);
    b.n_vox += d.n[0] * d.n[1] * d.n[2];
    b.n_dom += 1;
    b.h_elems.push_back(0);
    b.h_nodes.push_back(0);
    b.h_bnodes.push_back(0);
    b.h_status.push_back(status);
    if (b.micro20) b.d20.emplace_back();
    return DTC_OK;
}

// Order of a domain's bricks: a Z-curve over the brick grid (y, z, x from the lowest bit
// up, which makes runs of the 8x4x4 bricks compact), so that consecutive nodes, and with
// them the clusters, are close together.
static std::vector<int> brick_order(int bnx, int bny, int bnz) {
    auto spread = [](int v) {   // bit i -> bit 3 i
        int64_t r = 0;
        for (int i = 0; (v >> i) != 0; ++i) r |= (int64_t)((v >> i) & 1) << (3 * i);
        return r;
    };
    std::vector<std::pair<int64_t, int>> key;
    key.reserve((size_t)bnx * bny * bnz);
    for (int z = 0; z < bnz; ++z)
        for (int y = 0; y < bny; ++y)
            for (int x = 0; x < bnx; ++x)
                key.emplace_back(spread(y) | spread(z) << 1 | spread(x) << 2, x + bnx * (y + bny * z));
    std::sort(key.begin(), key.end());
    std::vector<int> o;
    o.reserve(key.size());
    for (const auto& k : key) o.push_back(k.second);
    return o;
}

int batch_add_domain(SolverBatch& b, const MeshDev& m, const dtc_domain_desc& d, const double* modulus_dev,
                     double escale, int lc_base, hipStream_t s) {
    if (m.nen != 8) return set_error(DTC_ERR_UNSUPPORTED, "the solver implements HEX08 micro elements");
    DomInfo D{};
    D.nx = m.nx; D.ny = m.ny; D.nz = m.nz;
    D.macro_order = d.macro_order;
    D.lc_base = lc_base;
    const int Lx = m.Lx, Ly = m.Ly, Lz = m.Lz;
    D.bnx = (Lx + BX - 1) / BX; D.bny = (Ly + BY - 1) / BY; D.bnz = (Lz + BZ - 1) / BZ;
    const int nbr = D.bnx * D.bny * D.bnz;
    for (int k = 0; k < 3; ++k) {
        D.delta[k] = d.delta[k];
        D.xa1[k] = (double)(d.xa_n[k] - 1);
        D.min_c[k] = (double)(d.xa_n[k] - 1) * d.delta[k];
        D.max_c[k] = (double)(d.xa_n[k] + d.n[k] - 1) * d.delta[k];
    }
    HostWords cnt;
    DTC_TRY(cnt.alloc((size_t)nbr * sizeof(int2)));
    k_brick_count<<<nbr, BX * BY * BZ, 0, s>>>(m.numLat.as<int>(), m.keepN.as<int>(), Lx, Ly, Lz, D.bnx, D.bny, (int2*)cnt.p);
    DTC_HIP(hipGetLastError());
    DTC_HIP(stream_wait(s));
    std::vector<int> hc(nbr);
    int64_t hb = 0;
    for (int i = 0; i < nbr; ++i) {
        hc[i] = ((const int2*)cnt.p)[i].x;
        hb += ((const int2*)cnt.p)[i].y;
    }
    cnt.recycle();
    // boundary nodes: fewer than 6 constrained DOFs fails the domain (f-src/mod_struct_preprocess.f90:471-473)
    if (3 * hb < 6) {
        DTC_TRY(batch_add_empty(b, d, DTC_ERR_FEW_CONSTRAINTS, lc_base));
        b.h_elems.back() = m.n_elems;
        b.h_nodes.back() = m.n_nodes;
        b.h_bnodes.back() = hb;
        return DTC_OK;
    }
    b.h_bnodes.push_back(hb);
    D.brick_begin = (int)b.h_brick.size();
    D.node_begin = b.n_nodes;
    int64_t node = b.n_nodes;
    std::vector<BrickInfo> mine;
    for (int i : brick_order(D.bnx, D.bny, D.bnz)) {
        if (!hc[i]) continue;
        BrickInfo B{};
        B.dom = b.n_dom;
        B.x0 = (i % D.bnx) * BX; B.y0 = ((i / D.bnx) % D.bny) * BY; B.z0 = (i / (D.bnx * D.bny)) * BZ;
        B.node_begin = (int)node;
        node += hc[i];
        B.node_end = (int)node;
        mine.push_back(B);
    }
    if (node >= INT32_MAX / 72) return set_error(DTC_ERR_BAD_ARGUMENT, "batch exceeds %d solver nodes", INT32_MAX / 72);
    D.brick_end = D.brick_begin + (int)mine.size();
    D.node_end = node;
    D.lat_off = b.n_lat;
    D.vox_off = b.n_vox;
    const int64_t nvox = (int64_t)m.nx * m.ny * m.nz;
    DevMem bl;
    if (!mine.empty()) {
        DTC_TRY(bl.alloc(mine.size() * sizeof(BrickInfo)));
        DTC_HIP(hipMemcpyAsync(bl.p, mine.data(), mine.size() * sizeof(BrickInfo), hipMemcpyHostToDevice, s));
        k_brick_assign<<<(unsigned)mine.size(), BX * BY * BZ, 0, s>>>(bl.as<BrickInfo>(), 0, m.numLat.as<int>(), m.keepN.as<int>(),
                                                                   m.cref.as<int>(), Lx, Ly, Lz, D.lat_off, b.lat2node.as<int>(),
                                                                   b.sol2ref.as<int>());
        DTC_HIP(hipGetLastError());
    }
    k_emod<<<nb(nvox, 256), 256, 0, s>>>(m.keepE.as<int>(), modulus_dev, d.E, escale, nvox, b.emod.as<double>() + D.vox_off);
    DTC_HIP(hipGetLastError());
    DTC_HIP(stream_wait(s));
    bl.recycle();
    b.h_brick.insert(b.h_brick.end(), mine.begin(), mine.end());
    b.h_dom.push_back(D);
    b.n_nodes = node;
    b.n_lat += (int64_t)Lx * Ly * Lz;
    b.n_vox += nvox;
    b.n_dom += 1;
    b.h_elems.push_back(m.n_elems);
    b.h_nodes.push_back(m.n_nodes);
    b.h_status.push_back(DTC_OK);
    return DTC_OK;
}

namespace {

// largest eigenvalue of a symmetric positive semidefinite n x n matrix (power iteration)
double sym_lmax(const double* A, int n) {
    std::vector<double> v(n, 1.0), w(n);
    for (int i = 0; i < n; ++i) v[i] += 0.01 * i;
    double lam = 0.0;
    for (int it = 0; it < 2000; ++it) {
        double nrm = 0.0;
        for (int i = 0; i < n; ++i) {
            double t = 0.0;
            for (int j = 0; j < n; ++j) t += A[i + n * j] * v[j];
            w[i] = t;
            nrm += t * t;
        }
        nrm = std::sqrt(nrm);
        double num = 0.0, den = 0.0;
        for (int i = 0; i < n; ++i) { num += v[i] * w[i]; den += v[i] * v[i]; }
        lam = num / den;
        for (int i = 0; i < n; ++i) v[i] = w[i] / nrm;
    }
    return lam;
}

// Most nodes of a level's clusters.  The matvec sums a node in the same order whatever
// its cluster is, so with the block PCG, which takes no other sums from it, the cap
// follows the grid: nodes / CL_GRID, so that small levels still make enough workgroups,
// each with a short walk over its elements (single 64^3 domain, 146 iterations: 148 ms with
// 128 everywhere, 132 ms so; 16 of them 517 and 509 ms).  The one-column PCGs also sum p.q per cluster;
// theirs is fixed, so that a domain's sums do not depend on the batch it is in.
constexpr int CL_GRID = 1024, CL_MIN = 8;
int cluster_cap(int64_t nodes, bool block, int precision) {
    if (!block) return precision == DTC_FP64 ? CL_CAP64 : CL_CAP;
    return (int)std::min<int64_t>(CL_CAP, std::max<int64_t>(CL_MIN, nodes / CL_GRID));
}

// Clusters of a level: consecutive nodes of each domain in brick order, whole bricks
// while they fit the cap, a brick of more nodes alone in equal pieces.
void make_clusters(std::vector<DomInfo>& hd, const std::vector<BrickInfo>& hb, int cap, Clusters& c) {
    c.h.clear();
    c.cap = cap;
    for (size_t d = 0; d < hd.size(); ++d) {
        DomInfo& D = hd[d];
        D.cl_begin = (int)c.h.size();
        ClusterInfo cur{};
        auto close = [&]() {
            if (cur.node_end > cur.node_begin) c.h.push_back(cur);
            cur = ClusterInfo{};
        };
        for (int i = D.brick_begin; i < D.brick_end; ++i) {
            const BrickInfo& B = hb[i];
            const int n = B.node_end - B.node_begin;
            if (cur.node_end - cur.node_begin + n > cap) close();
            if (n > cap) {
                const int pieces = (n + cap - 1) / cap;
                for (int k = 0; k < pieces; ++k)
                    c.h.push_back(ClusterInfo{(int)d, B.node_begin + n * k / pieces, B.node_begin + n * (k + 1) / pieces,
                                              i, i + 1, 0, 0});
                continue;
            }
            if (cur.node_end == cur.node_begin) {
                cur.dom = (int)d;
                cur.node_begin = B.node_begin;
                cur.brick_begin = i;
            }
            cur.node_end = B.node_end;
            cur.brick_end = i + 1;
        }
        close();
        D.cl_end = (int)c.h.size();
    }
    c.n = (int)c.h.size();
}

// element tables of a level's clusters (fine: FP64 moduli too)
int build_clusters(hipStream_t s, Clusters& c, const DevMem& brick, const DevMem& dom, const DevMem& lat2node,
                   const DevMem& emod, bool fine) {
    if (c.n == 0) return DTC_OK;
    HostWords cnt;
    DTC_TRY(cnt.alloc((size_t)c.n * 4));
    DTC_TRY(c.info.ensure(c.h.size() * sizeof(ClusterInfo)));
    DTC_HIP(hipMemcpyAsync(c.info.p, c.h.data(), c.h.size() * sizeof(ClusterInfo), hipMemcpyHostToDevice, s));
    k_cluster_elems<false><<<c.n, 256, 0, s>>>(c.info.as<ClusterInfo>(), brick.as<BrickInfo>(), dom.as<DomInfo>(),
                                               lat2node.as<int>(), emod.as<double>(), (int*)cnt.p, nullptr, nullptr,
                                               nullptr, nullptr, c.cap);
    DTC_HIP(hipGetLastError());
    DTC_HIP(stream_wait(s));
    const int* hc = (const int*)cnt.p;
    int64_t off = 0;
    for (int i = 0; i < c.n; ++i) {
        c.h[i].e_off = (int)off;
        c.h[i].e_cnt = hc[i];
        off += hc[i];
    }
    if (off >= INT32_MAX) return set_error(DTC_ERR_BAD_ARGUMENT, "batch exceeds %d cluster elements", INT32_MAX);
    DTC_HIP(hipMemcpyAsync(c.info.p, c.h.data(), c.h.size() * sizeof(ClusterInfo), hipMemcpyHostToDevice, s));
    const size_t ne = (size_t)off + 1;   // and the spare record
    DTC_TRY(c.enode.ensure(ne * 32));
    DTC_TRY(c.eown.ensure(ne * 8));
    if (fine) DTC_TRY(c.eE64.ensure(ne * 8));
    DTC_TRY(c.eE32.ensure(ne * 4));
    k_cluster_elems<true><<<c.n, 256, 0, s>>>(c.info.as<ClusterInfo>(), brick.as<BrickInfo>(), dom.as<DomInfo>(),
                                              lat2node.as<int>(), emod.as<double>(), nullptr, c.enode.as<int4>(),
                                              c.eown.as<uint2>(), fine ? c.eE64.as<double>() : nullptr,
                                              c.eE32.as<float>(), c.cap);
    DTC_HIP(hipGetLastError());
    cnt.recycle();
    return DTC_OK;
}

}  // namespace

// the mixed multigrid solve iterates the load cases as one block (DTC_BLOCK_PCG=0: one
// PCG per load case)
static bool block_pcg(const SolverBatch& b) {
    const char* e = std::getenv("DTC_BLOCK_PCG");
    return b.precond == DTC_PC_MG && !(e && e[0] == '0');
}

int batch_finalize(SolverBatch& b, int precision) {
    b.n_bricks = (int)b.h_brick.size();
    hipStream_t s = b.stream;
    b.cl.n = 0;
    const bool block = precision == DTC_FP32_REFINE && block_pcg(b);
    if (!b.micro20) make_clusters(b.h_dom, b.h_brick, cluster_cap(b.n_nodes, block, precision), b.cl);
    DTC_TRY(b.dom.ensure(b.h_dom.size() * sizeof(DomInfo)));
    DTC_HIP(hipMemcpyAsync(b.dom.p, b.h_dom.data(), b.h_dom.size() * sizeof(DomInfo), hipMemcpyHostToDevice, s));
    DTC_TRY(b.brick.ensure((b.h_brick.size() + 1) * sizeof(BrickInfo)));
    if (!b.h_brick.empty())
        DTC_HIP(hipMemcpyAsync(b.brick.p, b.h_brick.data(), b.h_brick.size() * sizeof(BrickInfo), hipMemcpyHostToDevice, s));
    const int64_t nn = b.n_nodes > 0 ? b.n_nodes : 1;
    const size_t v64 = (size_t)nn * 3 * R * 8, v32 = (size_t)nn * 3 * R * 4;
    DTC_TRY(b.dinv64.ensure((size_t)nn * 3 * 8));
    DTC_TRY(b.dinv32.ensure((size_t)nn * 3 * 4));
    DTC_TRY(b.x64.ensure(v64));
    DTC_TRY(b.r64.ensure(v64));
    if (precision == DTC_FP64) {
        DTC_TRY(b.p64.ensure(v64));
        DTC_TRY(b.q64.ensure(v64));
    } else {
        DTC_TRY(b.x32.ensure(v32));
        DTC_TRY(b.r32.ensure(v32));
        DTC_TRY(b.p32.ensure(v32));
        DTC_TRY(b.q32.ensure(v32));
    }
    // partial sums per brick, or per cluster (matvec)
    const size_t nbk = (size_t)std::max({b.n_bricks, b.cl.n, 1});
    DTC_TRY(b.part_a.ensure(nbk * R * 8));
    DTC_TRY(b.part_b.ensure(nbk * R * 8));
    DTC_TRY(b.part_c.ensure(nbk * R * 8));
    if (!b.micro20) DTC_TRY(b.part_ff.ensure((size_t)std::max(b.n_bricks, 1) * R * FFD * 8));
    const size_t nd = (size_t)(b.n_dom > 0 ? b.n_dom : 1);
    for (DevMem* m : {&b.alpha, &b.beta, &b.rz, &b.rr, &b.rr0, &b.thr2}) DTC_TRY(m->ensure(nd * R * 8));
    DTC_TRY(b.active.ensure(nd * R * 4));
    DTC_TRY(b.active64.ensure(nd * R * 4));
    DTC_TRY(b.active_prev.ensure(nd * R * 4));
    DTC_TRY(b.done.ensure(nd * 4));
    DTC_TRY(b.done64.ensure(nd * 4));
    DTC_TRY(b.iters.ensure(nd * 8));
    DTC_TRY(b.len0.ensure(nd * 8));
    DTC_TRY(b.phase_end.ensure(nd * 8));
    DTC_TRY(b.ff.ensure(nd * R * FFD * 8));
    // element stiffness (E = 1) and its Walsh blocks
    double Khat[576];
    DTC_TRY(element_stiffness(8, 1.0, b.nu, b.a, Khat));
    DTC_TRY(walsh_blocks(Khat, &b.wk64));
    b.kdiag = Khat[0];
    // element-by-element bound lambda_max(D^-1 K) <= lambda_max(diag(Khat)^-1/2 Khat diag(Khat)^-1/2);
    // the diagonal of the cube element is constant
    b.cheb_lmax = sym_lmax(Khat, 24) / b.kdiag;
    if (b.micro20) {
        DTC_TRY(finalize20(b));
    } else if (b.n_bricks > 0) {
        k_dinv<<<b.n_bricks, BX * BY * BZ, 0, s>>>(b.brick.as<BrickInfo>(), b.dom.as<DomInfo>(), b.lat2node.as<int>(),
                                                   b.emod.as<double>(), b.kdiag, b.dinv64.as<double>(), b.dinv32.as<float>());
        DTC_HIP(hipGetLastError());
        DTC_TRY(build_clusters(s, b.cl, b.brick, b.dom, b.lat2node, b.emod, true));
    }
    DTC_HIP(stream_wait(s));
    b.precision = precision;
    return DTC_OK;
}

int batch_build_mg(SolverBatch& b, int max_levels) {
    if (b.micro20) return set_error(DTC_ERR_UNSUPPORTED, "the multigrid preconditioner implements HEX08 micro elements");
    b.block_graph.reset();   // the levels' buffers are rebuilt
    hipStream_t s = b.stream;
    int maxn = 0;
    for (const DomInfo& D : b.h_dom) maxn = std::max(maxn, std::max(D.nx, std::max(D.ny, D.nz)));
    int L = 0;
    for (int n = maxn; n > 8 && L < max_levels; n = (n + 1) / 2) ++L;
    b.mg.resize(L);
    const size_t v0 = (size_t)(b.n_nodes > 0 ? b.n_nodes : 1) * 3 * R * 4;
    DTC_TRY(b.z32.ensure(v0));
    DTC_TRY(b.t32.ensure(v0));
    DTC_TRY(b.d32.ensure(v0));
    std::vector<DevMem> exist((size_t)L);   // of each level: lattice nodes of its voxels
    for (int l = 0; l < L; ++l) {
        Level& C = b.mg[l];
        const std::vector<DomInfo>& FD = l == 0 ? b.h_dom : b.mg[l - 1].h_dom;
        const double* fe = l == 0 ? b.emod.as<double>() : b.mg[l - 1].emod.as<double>();
        C.h_dom.assign(FD.begin(), FD.end());
        int64_t nlat = 0, nvox = 0, nbt = 0;
        std::vector<int64_t> boff(C.h_dom.size());
        for (size_t d = 0; d < C.h_dom.size(); ++d) {
            DomInfo& D = C.h_dom[d];
            D.nx = (D.nx + 1) / 2; D.ny = (D.ny + 1) / 2; D.nz = (D.nz + 1) / 2;
            for (int k = 0; k < 3; ++k) D.delta[k] *= 2.0;
            D.bnx = (D.nx + BX) / BX; D.bny = (D.ny + BY) / BY; D.bnz = (D.nz + BZ) / BZ;
            D.lat_off = nlat;
            D.vox_off = nvox;
            boff[d] = nbt;
            nlat += (int64_t)(D.nx + 1) * (D.ny + 1) * (D.nz + 1);
            nvox += (int64_t)D.nx * D.ny * D.nz;
            nbt += (int64_t)D.bnx * D.bny * D.bnz;
        }
        C.n_lat = nlat;
        C.n_vox = nvox;
        DTC_TRY(C.emod.ensure((size_t)std::max<int64_t>(nvox, 1) * 8));
        DTC_TRY(C.lat2node.ensure((size_t)std::max<int64_t>(nlat, 1) * 4));
        DevMem& ex = exist[l];
        HostWords cnt;
        DTC_TRY(ex.alloc((size_t)std::max<int64_t>(nlat, 1) * 4));
        DTC_TRY(cnt.alloc((size_t)std::max<int64_t>(nbt, 1) * 4));
        k_fill_i32b<<<nb(nlat, 256), 256, 0, s>>>(C.lat2node.as<int>(), nlat, -1);
        for (size_t d = 0; d < C.h_dom.size(); ++d) {
            const DomInfo &F = FD[d], &D = C.h_dom[d];
            const int64_t cv = (int64_t)D.nx * D.ny * D.nz, cl = (int64_t)(D.nx + 1) * (D.ny + 1) * (D.nz + 1);
            k_coarsen<<<nb(cv, 256), 256, 0, s>>>(fe + F.vox_off, F.nx, F.ny, F.nz, C.emod.as<double>() + D.vox_off,
                                                 D.nx, D.ny, D.nz);
            k_exist<<<nb(cl, 256), 256, 0, s>>>(C.emod.as<double>() + D.vox_off, D.nx, D.ny, D.nz,
                                               ex.as<int>() + D.lat_off);
            k_brick_count_ex<<<D.bnx * D.bny * D.bnz, NO, 0, s>>>(ex.as<int>() + D.lat_off, D.nx + 1, D.ny + 1,
                                                                   D.nz + 1, D.bnx, D.bny, (int*)cnt.p + boff[d]);
        }
        DTC_HIP(hipGetLastError());
        DTC_HIP(stream_wait(s));
        const int* hc = (const int*)cnt.p;
        C.h_brick.clear();
        int64_t node = 0;
        for (size_t d = 0; d < C.h_dom.size(); ++d) {
            DomInfo& D = C.h_dom[d];
            D.brick_begin = (int)C.h_brick.size();
            D.node_begin = node;
            for (int i : brick_order(D.bnx, D.bny, D.bnz)) {
                const int c = hc[boff[d] + i];
                if (!c) continue;
                BrickInfo B{};
                B.dom = (int)d;
                B.x0 = (i % D.bnx) * BX; B.y0 = ((i / D.bnx) % D.bny) * BY; B.z0 = (i / (D.bnx * D.bny)) * BZ;
                B.node_begin = (int)node;
                node += c;
                B.node_end = (int)node;
                C.h_brick.push_back(B);
            }
            D.brick_end = (int)C.h_brick.size();
            D.node_end = node;
        }
        cnt.recycle();
        C.n_bricks = (int)C.h_brick.size();
        C.n_nodes = node;
        make_clusters(C.h_dom, C.h_brick, cluster_cap(node, true, DTC_FP32_REFINE), C.cl);
        DTC_TRY(C.dom.ensure(C.h_dom.size() * sizeof(DomInfo)));
        DTC_HIP(hipMemcpyAsync(C.dom.p, C.h_dom.data(), C.h_dom.size() * sizeof(DomInfo), hipMemcpyHostToDevice, s));
        DTC_TRY(C.brick.ensure((C.h_brick.size() + 1) * sizeof(BrickInfo)));
        if (C.n_bricks > 0)
            DTC_HIP(hipMemcpyAsync(C.brick.p, C.h_brick.data(), C.h_brick.size() * sizeof(BrickInfo),
                                   hipMemcpyHostToDevice, s));
        for (size_t d = 0; d < C.h_dom.size(); ++d) {
            const DomInfo& D = C.h_dom[d];
            if (D.brick_end > D.brick_begin)
                k_brick_assign_ex<<<D.brick_end - D.brick_begin, NO, 0, s>>>(
                    C.brick.as<BrickInfo>() + D.brick_begin, ex.as<int>() + D.lat_off, D.nx + 1, D.ny + 1, D.nz + 1,
                    D.lat_off, C.lat2node.as<int>());
        }
        DTC_HIP(hipGetLastError());
        const size_t nn = (size_t)(C.n_nodes > 0 ? C.n_nodes : 1);
        DTC_TRY(C.dinv32.ensure(nn * 3 * 4));
        for (DevMem* m : {&C.b, &C.x, &C.t, &C.d}) DTC_TRY(m->ensure(nn * 3 * R * 4));
        if (C.n_bricks > 0) {
            k_dinv<<<C.n_bricks, NO, 0, s>>>(C.brick.as<BrickInfo>(), C.dom.as<DomInfo>(), C.lat2node.as<int>(),
                                            C.emod.as<double>(), b.kdiag, nullptr, C.dinv32.as<float>());
            DTC_HIP(hipGetLastError());
            DTC_TRY(build_clusters(s, C.cl, C.brick, C.dom, C.lat2node, C.emod, false));
            // transfer tables between this level and the finer one
            const int fbn = l == 0 ? b.n_bricks : b.mg[l - 1].n_bricks;
            const int64_t fnn = l == 0 ? b.n_nodes : b.mg[l - 1].n_nodes;
            const DevMem &fbr = l == 0 ? b.brick : b.mg[l - 1].brick, &fdm = l == 0 ? b.dom : b.mg[l - 1].dom,
                         &fln = l == 0 ? b.lat2node : b.mg[l - 1].lat2node;
            DTC_TRY(C.rtab.ensure(nn * t_row(T_RESTRICT) * 4));
            DTC_TRY(C.ptab.ensure((size_t)std::max<int64_t>(fnn, 1) * t_row(T_PROLONG) * 4));
            k_rtab<<<C.n_bricks, NO, 0, s>>>(C.brick.as<BrickInfo>(), C.dom.as<DomInfo>(), C.lat2node.as<int>(),
                                             fdm.as<DomInfo>(), fln.as<int>(), C.rtab.as<int>());
            if (fbn > 0)
                k_ptab<<<fbn, NO, 0, s>>>(fbr.as<BrickInfo>(), fdm.as<DomInfo>(), fln.as<int>(), C.dom.as<DomInfo>(),
                                          C.lat2node.as<int>(), C.ptab.as<int>());
            DTC_HIP(hipGetLastError());
        }
    }
    if (L > 0) {
        DTC_HIP(stream_wait(s));
        for (DevMem& ex : exist) ex.recycle();
    }
    return DTC_OK;
}

namespace {

constexpr int MAX_SLOTS = 4096;   // timed launches between two stream synchronisations

// Start of a timed launch of kernel kind `kind`: records the first event on the
// batch stream.  *slot = -1 when timing is off (or the slot table is full).
int timed_begin(SolverBatch& b, int kind, int* slot) {
    *slot = -1;
    if (!b.timing || b.n_slots >= MAX_SLOTS) return DTC_OK;
    if (b.ev_free.size() < 2) {
        for (int k = 0; k < 2; ++k) {
            hipEvent_t e;
            DTC_HIP(hipEventCreate(&e));
            b.ev.push_back(e);
            b.ev_free.push_back(e);
        }
    }
    SolverBatch::Timed t;
    t.e1 = b.ev_free.back(); b.ev_free.pop_back();
    t.e0 = b.ev_free.back(); b.ev_free.pop_back();
    t.kind = kind;
    t.slot = b.n_slots++;
    DTC_HIP(hipEventRecord(t.e0, b.stream));
    b.ev_used.push_back(t);
    *slot = t.slot;
    return DTC_OK;
}

// End of a timed launch: second event, then the launch's algorithmic bytes over
// the domains still iterating: vpass vectors of the working precision, the
// element moduli and (jac) the Jacobi scaling
int timed_end(SolverBatch& b, int slot, int vpass, bool fp64, bool jac, const int* done) {
    if (slot < 0) return DTC_OK;
    DTC_HIP(hipEventRecord(b.ev_used.back().e1, b.stream));
    k_launch_bytes<<<1, 256, 0, b.stream>>>(done, b.dom_bytes.as<double>(), b.n_dom, vpass, fp64 ? 1 : 0, jac ? 1 : 0,
                                           b.launch_bytes.as<double>() + 2 * slot);
    DTC_HIP(hipGetLastError());
    return DTC_OK;
}

// after a stream synchronisation: accumulate the timed launches
int harvest_events(SolverBatch& b) {
    if (b.ev_used.empty()) return DTC_OK;
    std::vector<double> by((size_t)b.n_slots * 2);
    DTC_HIP(hipMemcpy(by.data(), b.launch_bytes.p, by.size() * 8, hipMemcpyDeviceToHost));
    for (const SolverBatch::Timed& t : b.ev_used) {
        float ms = 0.f;
        DTC_HIP(hipEventElapsedTime(&ms, t.e0, t.e1));
        KernelStat& k = b.kstat[t.kind];
        k.ms_sum += ms;
        k.bytes_sum += by[2 * t.slot];
        k.flops_sum += by[2 * t.slot + 1];
        k.count += 1;
        b.ev_free.push_back(t.e0);
        b.ev_free.push_back(t.e1);
    }
    b.ev_used.clear();
    b.n_slots = 0;
    return DTC_OK;
}

// Load cases per wave of k_ebe (LCW): eight from EBE_FILL clusters on, where the vector
// cache's lookups bound the kernel (one per 32-byte run of x); on smaller grids (coarse
// levels, single domains) four, which halves the elements that each wave walks through.
// The sums do not depend on it.
constexpr int EBE_FILL = 1024;
template <int LCW, int CAP, typename T, typename TI, typename TO, int IN, int OUT>
void ebe_grid(int n, hipStream_t s, const EbeArgs& a, const WK<T>& wk, const TI* x, TO* y) {
    k_ebe<T, TI, TO, IN, OUT, LCW, CAP><<<n, 64 * R / LCW, 0, s>>>(a, wk, x, y);
}
template <typename T, typename TI, typename TO, int IN, int OUT>
int ebe_launch(const Clusters& c, hipStream_t s, EbeArgs a, const WK<T>& wk, const TI* x, TO* y) {
    if (c.n == 0) return DTC_OK;
    a.cl = c.info.as<ClusterInfo>();
    a.enode = c.enode.as<int4>();
    a.eown = c.eown.as<uint2>();
    a.eE = sizeof(T) == 4 ? c.eE32.p : c.eE64.p;
    const bool wide = c.n >= EBE_FILL;
    if (c.cap != CL_CAP64 || sizeof(T) == 4) {
        if (wide) ebe_grid<8, CL_CAP, T, TI, TO, IN, OUT>(c.n, s, a, wk, x, y);
        else ebe_grid<4, CL_CAP, T, TI, TO, IN, OUT>(c.n, s, a, wk, x, y);
    } else if constexpr (sizeof(T) == 8) {
        if (wide) ebe_grid<8, CL_CAP64, T, TI, TO, IN, OUT>(c.n, s, a, wk, x, y);
        else ebe_grid<4, CL_CAP64, T, TI, TO, IN, OUT>(c.n, s, a, wk, x, y);
    }
    DTC_HIP(hipGetLastError());
    return DTC_OK;
}

// x of the IN_U modes holds the Dirichlet values itself (set_bc in batch_solve)
template <typename T, int IN, int OUT>
int launch_mv(SolverBatch& b, const WK<T>& wk, const T* xin, T* yout, double* part, const int* done) {
    if (b.n_bricks == 0) return DTC_OK;
    // timed: the CG matvec (OUT_MASKED: of the block PCG) and the FP64 true residual
    constexpr int kind = (IN == IN_V && (OUT == OUT_MASKED_DOT || OUT == OUT_MASKED)) ? DTC_KSTAT_MV
                       : (IN == IN_U && OUT == OUT_RESID)                              ? DTC_KSTAT_RESID
                                                                                       : -1;
    int slot = -1;
    if (kind >= 0) DTC_TRY(timed_begin(b, kind, &slot));
    if (b.micro20) {
        DTC_TRY(mv20(b, sizeof(T) == 8, OUT, xin, yout, part, done));
    } else {
        EbeArgs a{};
        a.done = done;
        a.dinv = sizeof(T) == 4 ? b.dinv32.p : b.dinv64.p;
        a.partial = part;
        DTC_TRY((ebe_launch<T, T, T, IN_V, OUT>(b.cl, b.stream, a, wk, xin, yout)));
    }
    DTC_TRY(timed_end(b, slot, 2, sizeof(T) == 8, false, done));
    return DTC_OK;
}

// topology of one level for the FP32 matvec
struct MvTopo {
    const Clusters* cl;
    int n_bricks;
    const BrickInfo* bricks;
};

// tb: the batch whose fine level this is (its launches are timed), else null
// cin != 0 (OUT_CHEB only): x is cin D^-1 x
// (the zero-start step formed on the fly, IN_JS)
template <int OUT>
int launch_mv32(const MvTopo& T, hipStream_t s, const WK<float>& wk, const float* x, float* y, const int* done,
                const float* bv, const float* dinv, float* dv, float c1, float c2, int cflags, SolverBatch* tb,
                float cin) {
    static_assert(OUT == OUT_CHEB || OUT == OUT_BRES, "smoothing step or restriction residual");
    if (T.n_bricks == 0) return DTC_OK;
    if (cin != 0.f && OUT != OUT_CHEB) return set_error(DTC_ERR_BAD_ARGUMENT, "zero-start input needs the Chebyshev step");
    constexpr int kind = OUT == OUT_CHEB ? DTC_KSTAT_CHEB : DTC_KSTAT_BRES;
    int slot = -1;
    if (tb) DTC_TRY(timed_begin(*tb, kind, &slot));
    EbeArgs a{};
    a.done = done;
    a.dinv = dinv;
    a.bvec = bv;
    a.dvec = dv;
    a.c1 = c1;
    a.c2 = c2;
    a.cflags = cflags;
    a.cin = cin;
    bool js = false;
    if constexpr (OUT == OUT_CHEB) {
        js = cin != 0.f;
        if (js) DTC_TRY((ebe_launch<float, float, float, IN_JS, OUT>(*T.cl, s, a, wk, x, y)));
    }
    if (!js) DTC_TRY((ebe_launch<float, float, float, IN_V, OUT>(*T.cl, s, a, wk, x, y)));
    if (tb) {
        // x, y, b (with the zero-start input x is b itself: 2 vectors); Chebyshev: the
        // direction read and written as the flags say
        const int vp = (cin != 0.f ? 2 : 3) + (OUT == OUT_CHEB && (cflags & CH_READ_D) ? 1 : 0) +
                       (OUT == OUT_CHEB && (cflags & CH_WRITE_D) ? 1 : 0);
        DTC_TRY(timed_end(*tb, slot, vp, false, OUT == OUT_CHEB, done));
    }
    return DTC_OK;
}

// vectors and topology of multigrid level l (0 = the fine level, whose right-hand
// side is the PCG residual); the iterate alternates between buf[0] and buf[1]
struct LvView {
    MvTopo T;
    const float* dinv;
    float* b;
    float* buf[2];
    float* d;
};

// Chebyshev smoothing parameters: interval [lmax / ratio, lmax] of D^-1 K.  lmax is the
// element-by-element bound, about twice the largest eigenvalue of a porous mesh, and what the
// coarse space misses on thin struts reaches far down, so the intervals are wide.  The levels
// below the finest are an eighth of its work and less: they smooth with degree 4.  Iterations
// to 1e-11 and time against degree 2 and ratio 7 on every level: 64^3 trabecular 187 and 146
// -> 147 and 114, 191 -> 179 ms; 33^3 56 -> 44, 72 -> 67 ms for four; 27^3 HEX20 42 -> 30, 75 -> 65 ms
// for three; 48^3 greyscale 109 -> 80.  Degree 3 there: 184, 66 and 67 ms; degree 5: 180, 70 and 67;
// ratio 20: 183, 68 and 66.  (Measured with one launch per step on the coarsest level, degree 4.)
// The coarsest level takes degree 6: with 4 a domain whose batch has fewer levels (its own
// coarsest level carries the smooth modes) needed three iterations more than in a deeper one.
struct MgParams {
    double ratio = 0.0;        // finest level; 0: by its degree (fine_ratio)
    int level_degree = 4;      // intermediate levels (at least the finest level's degree)
    double level_ratio = 30.0;
    int coarse_degree = 6;     // coarsest level
    double coarse_ratio = 50.0;
    double lscale = 1.0;       // multiplies the element-by-element bound of lambda_max
    double fine_ratio(int deg) const { return ratio > 0.0 ? ratio : deg <= 1 ? 7.0 : deg == 2 ? 12.0 : deg == 3 ? 20.0 : 30.0; }
};

MgParams mg_params() {
    MgParams p;
    if (const char* e = std::getenv("DTC_MG_RATIO")) p.ratio = std::atof(e);
    if (const char* e = std::getenv("DTC_MG_LDEG")) p.level_degree = std::max(1, std::atoi(e));
    if (const char* e = std::getenv("DTC_MG_LRATIO")) p.level_ratio = std::atof(e);
    if (const char* e = std::getenv("DTC_MG_CDEG")) p.coarse_degree = std::max(1, std::atoi(e));
    if (const char* e = std::getenv("DTC_MG_CRATIO")) p.coarse_ratio = std::atof(e);
    if (const char* e = std::getenv("DTC_MG_LSCALE")) p.lscale = std::atof(e);
    return p;
}

// z = V(r): one V-cycle over the levels with Chebyshev-Jacobi pre- and
// post-smoothing by the same polynomial (a symmetric preconditioner), trilinear
// prolongation and its transpose as restriction.  Every smoothing step after the
// first is one fused matvec (OUT_CHEB); the residual before restriction is one
// OUT_BRES matvec.  prz (optional) receives per-brick sums of r . z.
int pmg_vcycle(SolverBatch& b, const float* r, float* z, double* prz);

int mg_vcycle(SolverBatch& b, const WK<float>& wk, const float* r, float* z, double* prz) {
    if (b.micro20) return pmg_vcycle(b, r, z, prz);
    hipStream_t s = b.stream;
    const int L = (int)b.mg.size();
    const int* done = b.done_ext ? b.done_ext : b.done.as<int>();
    static const MgParams P = mg_params();
    // (the twin's finest level is an intermediate level of the p-multigrid)
    const bool given = b.mg_degree > 0;   // by the caller: the intermediate levels take it too
    const int deg0 = given ? b.mg_degree : 2, ldeg = given ? deg0 : std::max(P.level_degree, deg0);
    const double lratio = given ? P.fine_ratio(deg0) : P.level_ratio;
    const int deg = b.done_ext ? ldeg : deg0;
    const double ratio0 = b.done_ext ? lratio : P.fine_ratio(deg0);
    auto view = [&](int l) {
        LvView v;
        if (l == 0) {
            v.T = {&b.cl, b.n_bricks, b.brick.as<BrickInfo>()};
            v.dinv = b.dinv32.as<float>();
            v.b = const_cast<float*>(r);
            v.buf[0] = z;
            v.buf[1] = b.t32.as<float>();
            v.d = b.d32.as<float>();
        } else {
            Level& C = b.mg[l - 1];
            v.T = {&C.cl, C.n_bricks, C.brick.as<BrickInfo>()};
            v.dinv = C.dinv32.as<float>();
            v.b = C.b.as<float>();
            v.buf[0] = C.x.as<float>();
            v.buf[1] = C.t.as<float>();
            v.d = C.d.as<float>();
        }
        return v;
    };
    std::vector<int> cur(L + 1, 0);
    auto smooth = [&](int l, int m, bool zero, double ratio) -> int {
        const LvView v = view(l);
        if (v.T.n_bricks == 0) return DTC_OK;
        const double hi = b.cheb_lmax * P.lscale, lo = hi / ratio;
        const double theta = 0.5 * (hi + lo), delta = 0.5 * (hi - lo), sigma = theta / delta;
        double rho = 1.0 / sigma;
        float c0 = 0.f;   // the zero-start step's coefficient, when that step is fused into the next
        for (int k = 0; k < m; ++k) {
            float c1 = 0.f, c2 = (float)(1.0 / theta);
            if (k > 0) {
                const double rn = 1.0 / (2.0 * sigma - rho);
                c1 = (float)(rn * rho);
                c2 = (float)(2.0 * rn / delta);
                rho = rn;
            }
            // the zero-start step x_1 = c2 D^-1 b is formed inside the next step's
            // staging (IN_JS) instead of being stored, where that kernel form runs
            const bool fuse = zero && m >= 2 && cheb_fuse();
            if (zero && k == 0 && fuse) {
                c0 = c2;
            } else if (zero && k == 0) {
                // x_1 = d_0: the next step takes its previous direction from x
                k_cheb<<<v.T.n_bricks, NT_UPD, 0, s>>>(v.T.bricks, done, v.b, nullptr, v.dinv, nullptr, v.buf[cur[l]],
                                                       c1, c2, 1, nullptr);
                DTC_HIP(hipGetLastError());
            } else {
                const int fl = (k == 0 ? 0 : (zero && k == 1) ? CH_D_FROM_X : CH_READ_D) | (k < m - 1 ? CH_WRITE_D : 0);
                const bool js = fuse && k == 1;
                DTC_TRY(launch_mv32<OUT_CHEB>(v.T, s, wk, js ? v.b : v.buf[cur[l]], v.buf[1 - cur[l]], done, v.b,
                                              v.dinv, v.d, c1, c2, fl, l == 0 ? &b : nullptr, js ? c0 : 0.f));
                cur[l] = 1 - cur[l];
            }
        }
        return DTC_OK;
    };
    // the coarsest level in one launch where it fits k_coarse: always, but for domains of more
    // than 2048 voxels an edge
    const std::vector<DomInfo>& cdom = L > 0 ? b.mg[L - 1].h_dom : b.h_dom;
    int edge = 0, nodes = 0;
    for (const DomInfo& D : cdom) {
        edge = std::max({edge, D.nx, D.ny, D.nz});
        nodes = std::max<int64_t>(nodes, (int64_t)(D.nx + 1) * (D.ny + 1) * (D.nz + 1));
    }
    const bool one_launch = edge <= COARSE_EDGE && P.coarse_degree <= COARSE_STEPS;
    auto coarsest = [&]() -> int {
        const LvView v = view(L);
        if (!one_launch) return smooth(L, P.coarse_degree, true, P.coarse_ratio);
        if (v.T.n_bricks == 0) return DTC_OK;
        const double hi = b.cheb_lmax * P.lscale, lo = hi / P.coarse_ratio;
        const double theta = 0.5 * (hi + lo), delta = 0.5 * (hi - lo), sigma = theta / delta;
        double rho = 1.0 / sigma;
        CoarseCheb cc{};
        cc.m = P.coarse_degree;
        cc.c2[0] = (float)(1.0 / theta);
        for (int k = 1; k < cc.m; ++k) {
            const double rn = 1.0 / (2.0 * sigma - rho);
            cc.c1[k] = (float)(rn * rho);
            cc.c2[k] = (float)(2.0 * rn / delta);
            rho = rn;
        }
        const DevMem& dom = L > 0 ? b.mg[L - 1].dom : b.dom;
        const DevMem& l2n = L > 0 ? b.mg[L - 1].lat2node : b.lat2node;
        const DevMem& emod = L > 0 ? b.mg[L - 1].emod : b.emod;
        const dim3 grid((unsigned)cdom.size(), R);
        auto run = [&](auto kernel, int nt) {
            kernel<<<grid, nt, 0, s>>>(dom.as<DomInfo>(), l2n.as<int>(), emod.as<double>(), v.dinv, done, wk, v.b, v.buf[0],
                                       cc);
        };
        if (nodes <= 256) run(k_coarse<256>, 256);
        else if (nodes <= 384) run(k_coarse<384>, 384);
        else if (nodes <= 512) run(k_coarse<512>, 512);
        else run(k_coarse<768>, 768);
        DTC_HIP(hipGetLastError());
        return DTC_OK;
    };
    // the fine iterate makes (deg - 1) + deg swaps (without coarse levels none, or
    // coarse_degree - 1): start in the buffer that makes it end in z
    cur[0] = (L > 0 ? 2 * deg - 1 : one_launch ? 0 : P.coarse_degree - 1) % 2;
    for (int l = 0; l < L; ++l) {
        DTC_TRY(smooth(l, l == 0 ? deg : ldeg, true, l == 0 ? ratio0 : lratio));
        const LvView f = view(l), c = view(l + 1);
        cur[l + 1] = 0;
        if (c.T.n_bricks == 0 || f.T.n_bricks == 0) continue;
        float* res = f.buf[1 - cur[l]];
        DTC_TRY(launch_mv32<OUT_BRES>(f.T, s, wk, f.buf[cur[l]], res, done, f.b, f.dinv, nullptr, 0.f, 0.f, 0,
                                      l == 0 ? &b : nullptr, 0.f));
        k_transfer<T_RESTRICT><<<dim3(c.T.n_bricks, node_split(c.T.n_bricks)), 256, 0, s>>>(
            c.T.bricks, b.mg[l].rtab.as<int>(), done, res, c.b);
        DTC_HIP(hipGetLastError());
    }
    DTC_TRY(coarsest());
    for (int l = L - 1; l >= 0; --l) {
        const LvView f = view(l), c = view(l + 1);
        if (f.T.n_bricks > 0 && c.T.n_bricks > 0) {
            k_transfer<T_PROLONG><<<dim3(f.T.n_bricks, node_split(f.T.n_bricks)), 256, 0, s>>>(
                f.T.bricks, b.mg[l].ptab.as<int>(), done, c.buf[cur[l + 1]], f.buf[cur[l]]);
            DTC_HIP(hipGetLastError());
        }
        DTC_TRY(smooth(l, l == 0 ? deg : ldeg, false, l == 0 ? ratio0 : lratio));
    }
    if (prz && b.n_bricks > 0) {
        k_dot<<<b.n_bricks, NT_UPD, 0, s>>>(b.brick.as<BrickInfo>(), done, r, z, prz);
        DTC_HIP(hipGetLastError());
    }
    return DTC_OK;
}

// p-multigrid V-cycle of HEX20 micro domains (FP32): Chebyshev-Jacobi smoothing
// on the HEX20 operator (degree mg_degree, zero start), the residual restricted
// to the HEX08 discretisation of the same voxels (P^T), that batch's geometric
// V-cycle, the correction prolongated (P), and the same Chebyshev polynomial
// after it (a symmetric preconditioner).
int pmg_vcycle(SolverBatch& b, const float* r, float* z, double* prz) {
    if (!b.p08) return set_error(DTC_ERR_DEVICE, "p-multigrid without its HEX08 level");
    SolverBatch& c = *b.p08;
    hipStream_t s = b.stream;
    const int* done = b.done.as<int>();
    static const MgParams P = mg_params();
    const int deg = b.mg_degree > 0 ? b.mg_degree : 2;
    const BrickInfo* bl = b.brick.as<BrickInfo>();
    float* t = b.t32.as<float>();
    float* d = b.d32.as<float>();
    const double hi = b.cheb_lmax * P.lscale, lo = hi / P.fine_ratio(deg);
    const double theta = 0.5 * (hi + lo), delta = 0.5 * (hi - lo), sigma = theta / delta;
    auto smooth = [&](bool zero, double* dot) -> int {
        double rho = 1.0 / sigma;
        for (int k = 0; k < deg; ++k) {
            float c1 = 0.f, c2 = (float)(1.0 / theta);
            if (k > 0) {
                const double rn = 1.0 / (2.0 * sigma - rho);
                c1 = (float)(rn * rho);
                c2 = (float)(2.0 * rn / delta);
                rho = rn;
            }
            double* dk = k == deg - 1 ? dot : nullptr;
            if (zero && k == 0) {
                k_cheb<<<b.n_bricks, NT_UPD, 0, s>>>(bl, done, r, nullptr, b.dinv32.as<float>(), d, z, c1, c2, 1, dk);
            } else if (!dk && cheb_fuse()) {
                // the step in the epilogue of the operator's node gather (no t vector)
                DTC_TRY(mv20_cheb(b, z, done, r, b.dinv32.as<float>(), d, c1, c2));
            } else {
                DTC_TRY(mv20(b, false, OUT_MASKED, z, t, nullptr, done));
                k_cheb<<<b.n_bricks, NT_UPD, 0, s>>>(bl, done, r, t, b.dinv32.as<float>(), d, z, c1, c2, 0, dk);
            }
            DTC_HIP(hipGetLastError());
        }
        return DTC_OK;
    };
    DTC_TRY(smooth(true, nullptr));
    // residual, restricted to the HEX08 nodes
    DTC_TRY(mv20_bres(b, z, t, done, r));
    float* r08 = c.r32.as<float>();
    float* z08 = c.z32.as<float>();
    if (c.n_bricks > 0)
        k_transfer<T_PRESTRICT><<<dim3(c.n_bricks, node_split(c.n_bricks)), 256, 0, s>>>(
            c.brick.as<BrickInfo>(), b.pmg_rtab.as<int>(), done, t, r08);
    DTC_HIP(hipGetLastError());
    c.done_ext = done;
    DTC_TRY(mg_vcycle(c, cast_wk<float>(c.wk64), r08, z08, nullptr));
    k_transfer<T_PPROLONG><<<dim3(b.n_bricks, node_split(b.n_bricks)), 256, 0, s>>>(bl, b.pmg_ptab.as<int>(), done,
                                                                                    z08, z);
    DTC_HIP(hipGetLastError());
    return smooth(false, prz);
}

// p-multigrid set-up of a HEX20 batch over its HEX08 twin c (same domain groups,
// finalised): the twin's geometric levels, the fine Chebyshev bound and vectors
int build_pmg(SolverBatch& b, SolverBatch& c) {
    if (!b.micro20 || c.micro20) return set_error(DTC_ERR_BAD_ARGUMENT, "p-multigrid needs a HEX20 batch and its HEX08 twin");
    if (c.n_dom != b.n_dom) return set_error(DTC_ERR_DEVICE, "p-multigrid: %d HEX08 groups for %d HEX20 groups", c.n_dom,
                                             b.n_dom);
    b.block_graph.reset();
    c.stream = b.stream;
    c.mg_degree = b.mg_degree;
    DTC_TRY(batch_build_mg(c, 8));
    // element-by-element bound of lambda_max(D^-1 K) for HEX20:
    // lambda_max(diag(Khat)^-1/2 Khat diag(Khat)^-1/2)
    std::vector<double> S(3600);
    for (int i = 0; i < 60; ++i)
        for (int j = 0; j < 60; ++j)
            S[i + 60 * j] = b.khat20[i + 60 * j] / std::sqrt(b.khat20[i + 60 * i] * b.khat20[j + 60 * j]);
    b.cheb_lmax = sym_lmax(S.data(), 60);
    const size_t v0 = (size_t)(b.n_nodes > 0 ? b.n_nodes : 1) * 3 * R * 4;
    DTC_TRY(b.z32.ensure(v0));
    DTC_TRY(b.t32.ensure(v0));
    DTC_TRY(b.d32.ensure(v0));
    DTC_TRY(b.pmg_rtab.ensure((size_t)std::max<int64_t>(c.n_nodes, 1) * t_row(T_PRESTRICT) * 4));
    DTC_TRY(b.pmg_ptab.ensure((size_t)std::max<int64_t>(b.n_nodes, 1) * t_row(T_PPROLONG) * 4));
    // rows without a HEX20 domain of their own stay empty
    if (c.n_nodes > 0)
        k_fill_i32b<<<nb(c.n_nodes * t_row(T_PRESTRICT), 256), 256, 0, b.stream>>>(b.pmg_rtab.as<int>(), c.n_nodes * t_row(T_PRESTRICT), -1);
    for (int g = 0; g < b.n_dom && g < c.n_dom; ++g) {
        const DomInfo& D08 = c.h_dom[g];
        if (b.h_status[g] != DTC_OK || c.h_status[g] != DTC_OK) continue;
        const int64_t n = (int64_t)(D08.nx + 1) * (D08.ny + 1) * (D08.nz + 1);
        k_pmg_rtab<<<nb(n, 256), 256, 0, b.stream>>>(b.h_d20dev[g], D08, c.lat2node.as<int>(), b.pmg_rtab.as<int>());
    }
    if (b.n_bricks > 0)
        k_pmg_ptab<<<b.n_bricks, 64, 0, b.stream>>>(b.brick.as<BrickInfo>(), b.dom.as<DomInfo>(), b.d20dev.as<Dom20Dev>(),
                                                    c.dom.as<DomInfo>(), c.lat2node.as<int>(), b.pmg_ptab.as<int>());
    DTC_HIP(hipGetLastError());
    b.p08 = &c;
    return DTC_OK;
}

// one PCG iteration on (x, r, p, q) in precision T; zmg != null: multigrid
// preconditioner (FP32 only), z = V(r) stored in zmg
template <typename T>
int pcg_iteration(SolverBatch& b, const WK<T>& wk, T* x, T* r, T* p, T* q, const T* dinv, int64_t max_iters, T* zmg) {
    const int D = b.n_dom, NBk = b.n_bricks;
    int* done = b.done.as<int>();
    DTC_TRY((launch_mv<T, IN_V, OUT_MASKED_DOT>(b, wk, p, q, b.part_a.as<double>(), done)));
    k_red_alpha<<<D, RED_NT, 0, b.stream>>>(b.dom.as<DomInfo>(), done, b.part_a.as<double>(),
                                            !b.micro20, b.active.as<int>(),
                                        b.rz.as<double>(), b.alpha.as<double>());
    k_cg_update<T><<<NBk, NT_UPD, 0, b.stream>>>(b.brick.as<BrickInfo>(), done, b.alpha.as<double>(), x, r, p, q, dinv,
                                                 zmg ? nullptr : b.part_a.as<double>(), b.part_b.as<double>());
    if constexpr (std::is_same<T, float>::value) {
        if (zmg) DTC_TRY(mg_vcycle(b, wk, r, zmg, b.part_a.as<double>()));
    }
    k_red_beta<<<D, RED_NT, 0, b.stream>>>(b.dom.as<DomInfo>(), done, b.part_a.as<double>(), b.part_b.as<double>(),
                                       b.thr2.as<double>(), b.active.as<int>(), b.rz.as<double>(), b.beta.as<double>(),
                                       b.iters.as<int64_t>(), max_iters);
    k_cg_dir<T><<<NBk, NT_UPD, 0, b.stream>>>(b.brick.as<BrickInfo>(), done, b.beta.as<double>(), r, p, dinv, zmg);
    DTC_HIP(hipGetLastError());
    return DTC_OK;
}

int all_done(SolverBatch& b, const DevMem& flags, bool* out) {
    std::vector<int> h(b.n_dom);
    DTC_HIP(hipMemcpyAsync(h.data(), flags.p, (size_t)b.n_dom * 4, hipMemcpyDeviceToHost, b.stream));
    DTC_HIP(stream_wait(b.stream));
    DTC_TRY(harvest_events(b));
    bool all = true;
    for (int v : h) all = all && (v != 0);
    *out = all;
    return DTC_OK;
}

// ---- convergence words
// After a run of iterations k_all_set counts the run in a device word and writes
// 2 * runs + (every domain's done flag is set) to a page-locked host word, one 8-byte
// store.  The host reads that word while the next run already executes (a copy of the
// flags between the runs left the GPU idle for 20 us each time).
__global__ __launch_bounds__(256) void k_all_set(const int* __restrict__ flags, int n, unsigned long long* __restrict__ runs,
                                                 unsigned long long* __restrict__ host) {
    __shared__ int s_any[256];
    int miss = 0;
    for (int d = threadIdx.x; d < n; d += 256) miss |= flags[d] == 0;
    s_any[threadIdx.x] = miss;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (threadIdx.x < w) s_any[threadIdx.x] |= s_any[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const unsigned long long k = *runs + 1;
        *runs = k;
        __hip_atomic_store(host, 2 * k + (s_any[0] ? 0 : 1), __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

__global__ void k_fill_u64(unsigned long long* __restrict__ p, int n, unsigned long long v) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// per domain [done64, iterations, rr (24), rr0 (24)] to page-locked host memory
constexpr int STAT_N = 2 + 2 * R;
__global__ __launch_bounds__(64) void k_status(const int* __restrict__ done64, const int64_t* __restrict__ iters,
                                               const double* __restrict__ rr, const double* __restrict__ rr0,
                                               double* __restrict__ host) {
    const int d = blockIdx.x, t = threadIdx.x;
    if (t >= STAT_N) return;
    host[(int64_t)d * STAT_N + t] = t == 0   ? (double)done64[d]
                                    : t == 1 ? (double)iters[d]
                                    : t < 2 + R ? rr[d * R + t - 2]
                                                : rr0[d * R + t - 2 - R];
}

int words_setup(SolverBatch& b) {
    const size_t need = 64 + (size_t)b.n_dom * STAT_N * 8;
    if (b.host_words.n < need) {
        if (b.host_words.p) DTC_HIP(stream_wait(b.stream));
        b.host_words.reset();
        DTC_TRY(b.host_words.alloc(need));
        *b.host_words.word() = 0;
        b.runs = 0;
        DTC_TRY(b.runs_dev.ensure(8));
        k_fill_u64<<<1, 1, 0, b.stream>>>(b.runs_dev.as<unsigned long long>(), 1, 0);
        DTC_HIP(hipGetLastError());
    }
    return DTC_OK;
}

int post_done(SolverBatch& b) {
    k_all_set<<<1, 256, 0, b.stream>>>(b.done.as<int>(), b.n_dom, b.runs_dev.as<unsigned long long>(),
                                       b.host_words.word());
    DTC_HIP(hipGetLastError());
    return DTC_OK;
}

// waits for the summary of run number `run`
int wait_done(SolverBatch& b, uint64_t run, bool* fin) {
    const unsigned long long* w = b.host_words.word();
    DTC_TRY(wait_word(b.stream, w, 2 * run));
    *fin = (__atomic_load_n(w, __ATOMIC_ACQUIRE) & 1) != 0;
    return DTC_OK;
}

// status of every domain on the host (the stream is idle afterwards)
int read_status(SolverBatch& b, const double** out) {
    DTC_TRY(words_setup(b));
    k_status<<<b.n_dom, 64, 0, b.stream>>>(b.done64.as<int>(), b.iters.as<int64_t>(), b.rr.as<double>(),
                                           b.rr0.as<double>(), b.host_words.status());
    DTC_HIP(hipGetLastError());
    DTC_HIP(stream_wait(b.stream));
    *out = b.host_words.status();
    return DTC_OK;
}

// iterations until every domain is done or max_steps (rounded up to CHECK) ran.  The host
// is one run of CHECK iterations ahead of the summary that it decides by: iterations after
// the last domain finished are early exits, every kernel skips done domains
template <typename T>
int pcg_run(SolverBatch& b, const WK<T>& wk, T* x, T* r, T* p, T* q, const T* dinv, int64_t max_iters,
            int64_t max_steps, T* zmg) {
    const int CHECK = zmg ? 4 : 8;
    if (!b.timing) DTC_TRY(words_setup(b));
    const uint64_t first = b.runs;
    for (int64_t steps = 0; steps < max_steps; steps += CHECK) {
        bool fin = false;
        if (b.timing) DTC_TRY(all_done(b, b.done, &fin));
        else if (b.runs > first + 1) DTC_TRY(wait_done(b, b.runs - 1, &fin));
        if (fin) break;
        for (int k = 0; k < CHECK; ++k) DTC_TRY(pcg_iteration<T>(b, wk, x, r, p, q, dinv, max_iters, zmg));
        if (!b.timing) {
            DTC_TRY(post_done(b));
            ++b.runs;
        }
    }
    return DTC_OK;
}

// Q = A P of the block PCG: FP32 vectors, FP64 arithmetic.  The Gram matrix
// W = P^T Q resolves the directions of the block only as far as Q is accurate:
// for smooth directions FP32 sums lose most digits of A P to cancellation, and
// W's small eigenvalues (the ones that steer the block) drown in that error.
// q64 set: Q is written as an FP64 vector (the block PCG on FP64 vectors)
int launch_mv_q64(SolverBatch& b, const float* p, float* q, const int* done, double* q64 = nullptr) {
    EbeArgs a{};
    a.done = done;
    a.dinv = b.dinv64.p;
    int slot = -1;
    DTC_TRY(timed_begin(b, DTC_KSTAT_MV, &slot));
    const WK<double> wk = cast_wk<double>(b.wk64);
    if (q64) DTC_TRY((ebe_launch<double, float, double, IN_V, OUT_MASKED>(b.cl, b.stream, a, wk, p, q64)));
    else DTC_TRY((ebe_launch<double, float, float, IN_V, OUT_MASKED>(b.cl, b.stream, a, wk, p, q)));
    DTC_TRY(timed_end(b, slot, 2, false, false, done));
    return DTC_OK;
}

// block PCG set-up: slices of SLICE_NODES nodes (more for domains of over
// MAX_SLICES * SLICE_NODES nodes) within each domain for the block's vector kernels, and
// the per-domain factor and coefficient storage
int block_setup(SolverBatch& b) {
    if (b.n_slices > 0) return DTC_OK;
    std::vector<int4>& sl = b.h_slices;
    std::vector<int>& ds = b.h_dslice;
    sl.clear();
    ds.assign((size_t)b.n_dom + 1, 0);
    for (int d = 0; d < b.n_dom; ++d) {
        ds[d] = (int)sl.size();
        const DomInfo& D = b.h_dom[d];
        const int64_t nn = D.node_end - D.node_begin;
        const int64_t step = std::max<int64_t>(SLICE_NODES, (nn + MAX_SLICES - 1) / MAX_SLICES);
        for (int64_t n0 = D.node_begin; n0 < D.node_end; n0 += step)
            sl.push_back(make_int4(d, (int)n0, (int)std::min<int64_t>(n0 + step, D.node_end), 0));
    }
    ds[b.n_dom] = (int)sl.size();
    DTC_TRY(b.slices.ensure(std::max<size_t>(sl.size(), 1) * sizeof(int4)));
    DTC_TRY(b.dslice.ensure(ds.size() * 4));
    DTC_TRY(b.gpart.ensure(std::max<size_t>(sl.size(), 1) * 2 * RR * 8));
    DTC_TRY(b.gsum.ensure((size_t)std::max(b.n_dom, 1) * 2 * RR * 8));
    DTC_TRY(b.lfac.ensure((size_t)std::max(b.n_dom, 1) * RR * 8));
    DTC_TRY(b.bcoef.ensure((size_t)std::max(b.n_dom, 1) * RR * 4));
    // per-slice r.r partials of the block update (slices of at least 32 nodes, bricks of up to 128)
    DTC_TRY(b.part_b.ensure(std::max<size_t>({sl.size(), (size_t)b.n_bricks, 1}) * R * 8));
    if (!sl.empty())
        DTC_HIP(hipMemcpyAsync(b.slices.p, sl.data(), sl.size() * sizeof(int4), hipMemcpyHostToDevice, b.stream));
    DTC_HIP(hipMemcpyAsync(b.dslice.p, ds.data(), ds.size() * 4, hipMemcpyHostToDevice, b.stream));
    b.n_slices = (int)sl.size();
    return DTC_OK;
}

// per-domain Grams a^T b and a^T c (c may be null) into gsum
template <typename T> struct NoDeduce { using type = T; };
template <typename TA = float, typename TB = float>
int block_gram(SolverBatch& b, const TA* a, const TB* bb, const typename NoDeduce<TB>::type* c) {
    hipStream_t s = b.stream;
    int* done = b.done.as<int>();
    if (b.n_slices > 0) {
        const int4* sl = b.slices.as<int4>();
        double* gp = b.gpart.as<double>();
        if (c) k_gram<2, TA, TB><<<b.n_slices, GR_NT, 0, s>>>(sl, done, a, bb, c, gp);
        else k_gram<1, TA, TB><<<b.n_slices, GR_NT, 0, s>>>(sl, done, a, bb, nullptr, gp);
    }
    k_gram_sum<<<dim3(b.n_dom, (c ? 2 : 1) * RR / GS_E), GS_E * GS_G, 0, s>>>(b.dslice.as<int>(), done,
                                                                            b.gpart.as<double>(), b.gsum.as<double>());
    DTC_HIP(hipGetLastError());
    return DTC_OK;
}

// dst = src with orthonormal columns per domain (dropped directions zero).  In
// FP32, combinations of nearly dependent columns with large coefficients that
// cancel lose the directions they should keep: the residual columns of a
// domain line up with its slowest modes after the first residual replacement.
int block_orth(SolverBatch& b, const float* src, float* dst, bool partials_done = false) {
    hipStream_t s = b.stream;
    int* done = b.done.as<int>();
    if (partials_done) {   // the direction kernel wrote src's Gram partials
        k_gram_sum<<<dim3(b.n_dom, RR / GS_E), GS_E * GS_G, 0, s>>>(b.dslice.as<int>(), done, b.gpart.as<double>(),
                                                                   b.gsum.as<double>());
    } else {
        DTC_TRY(block_gram(b, src, src, nullptr));
    }
    k_bsolve<2><<<b.n_dom, 64, 0, s>>>(done, b.gsum.as<double>(), b.lfac.as<double>(), b.bcoef.as<float>());
    k_bdir<false><<<b.n_slices, NT_UPD, 0, s>>>(b.slices.as<int4>(), done, b.bcoef.as<float>(), src, nullptr, dst,
                                                nullptr);
    DTC_HIP(hipGetLastError());
    return DTC_OK;
}

// the new direction block Z + P beta and its Gram partials in one kernel, then the
// orthonormalisation into p
int block_dir_orth(SolverBatch& b, float* p, const float* z, float* q) {
    hipStream_t s = b.stream;
    int* done = b.done.as<int>();
    k_bdir<true><<<b.n_slices, NT_UPD, 0, s>>>(b.slices.as<int4>(), done, b.bcoef.as<float>(), p, z, q,
                                               b.gpart.as<double>());
    DTC_HIP(hipGetLastError());
    return block_orth(b, q, p, true);
}

// one block PCG iteration on FP64 vectors (x64, r64) with the FP32 multigrid as
// preconditioner: Q = K P in FP64 (FP32 directions P, FP64 arithmetic), the
// Grams in FP64, x += P alpha and r -= Q alpha in FP64; r is rounded to FP32
// only as the V-cycle's input.  Used for high-contrast (greyscale) batches, whose
// FP32 recursive residual loses the soft regions' part to the rounding of the
// stiff regions' terms.
int block_iteration64(SolverBatch& b, const WK<float>& wk, float* p, float* q, float* z, int64_t max_iters) {
    hipStream_t s = b.stream;
    const int D = b.n_dom, NBk = b.n_bricks, NSl = b.n_slices;
    const int4* sl = b.slices.as<int4>();
    int* done = b.done.as<int>();
    const BrickInfo* bl = b.brick.as<BrickInfo>();
    double* x = b.x64.as<double>();
    double* r = b.r64.as<double>();
    double* q64 = b.q64.as<double>();
    if (b.micro20) DTC_TRY(mv20_q64(b, p, nullptr, done, q64));
    else DTC_TRY(launch_mv_q64(b, p, nullptr, done, q64));
    DTC_TRY((block_gram<float, double>(b, p, q64, r)));
    k_bsolve<0><<<D, 64, 0, s>>>(done, b.gsum.as<double>(), b.lfac.as<double>(), b.bcoef.as<float>());
    k_bupdate64<<<NSl, NT_UPD, 0, s>>>(sl, done, b.bcoef.as<float>(), x, r, p, q64, b.part_b.as<double>());
    k_bcheck<<<D, RED_NT, 0, s>>>(b.dslice.as<int>(), done, b.part_b.as<double>(), b.thr2.as<double>(), nullptr,
                                  b.iters.as<int64_t>(), b.phase_end.as<int64_t>(), max_iters);
    k_to32<<<NBk, NT_UPD, 0, s>>>(bl, done, r, b.r32.as<float>(), nullptr, nullptr);
    DTC_HIP(hipGetLastError());
    DTC_TRY(mg_vcycle(b, wk, b.r32.as<float>(), z, nullptr));
    DTC_TRY((block_gram<double, float>(b, q64, z, nullptr)));
    k_bsolve<1><<<D, 64, 0, s>>>(done, b.gsum.as<double>(), b.lfac.as<double>(), b.bcoef.as<float>());
    return block_dir_orth(b, p, z, q);
}

// one block PCG iteration on (x, r); p is the direction block (orthonormal
// columns), q and z are work vectors
int block_iteration(SolverBatch& b, const WK<float>& wk, float* x, float* r, float* p, float* q, float* z,
                    int64_t max_iters) {
    if (b.block64) return block_iteration64(b, wk, p, q, z, max_iters);
    hipStream_t s = b.stream;
    const int D = b.n_dom, NSl = b.n_slices;
    const int4* sl = b.slices.as<int4>();
    int* done = b.done.as<int>();
    if (b.block_q64 && b.micro20) DTC_TRY(mv20_q64(b, p, q, done));
    else if (b.block_q64) DTC_TRY(launch_mv_q64(b, p, q, done));
    else DTC_TRY((launch_mv<float, IN_V, OUT_MASKED>(b, wk, p, q, nullptr, done)));
    DTC_TRY(block_gram(b, p, q, r));
    k_bsolve<0><<<D, 64, 0, s>>>(done, b.gsum.as<double>(), b.lfac.as<double>(), b.bcoef.as<float>());
    k_bupdate<<<NSl, NT_UPD, 0, s>>>(sl, done, b.bcoef.as<float>(), x, r, p, q, b.part_b.as<double>());
    k_bcheck<<<D, RED_NT, 0, s>>>(b.dslice.as<int>(), done, b.part_b.as<double>(), b.thr2.as<double>(),
                                  b.rr.as<double>(), b.iters.as<int64_t>(), b.phase_end.as<int64_t>(), max_iters);
    DTC_HIP(hipGetLastError());
    DTC_TRY(mg_vcycle(b, wk, r, z, nullptr));
    DTC_TRY(block_gram(b, q, z, nullptr));
    k_bsolve<1><<<D, 64, 0, s>>>(done, b.gsum.as<double>(), b.lfac.as<double>(), b.bcoef.as<float>());
    return block_dir_orth(b, p, z, q);
}

// block PCG iterations until every domain is done or max_steps iterations ran.
//
// Without kernel timing (the default), RUN iterations and their summary (k_all_set) are
// captured once per solve into a HIP graph and replayed; the host stays one replay ahead of
// the summary that it decides by, so the GPU never waits for it, and at most 2 RUN - 1
// iterations of early exits follow the last one that counts.  An empty iteration costs its
// launches, 2-4 us each: a 12^3 domain (22 iterations in two phases) took 5.07 ms with runs of
// 4 and the flags copied between them, 4.55 with runs of 4, 4.36 with 2, 4.40 with 1.
// DTC_GRAPH=0 (or kernel timing) launches the iterations one by one with a synchronous
// check every GROUP iterations.
inline bool trace_on() {
    static const bool on = std::getenv("DTC_TRACE") && std::getenv("DTC_TRACE")[0] == '1';
    return on;
}

int block_run(SolverBatch& b, const WK<float>& wk, float* x, float* r, float* p, float* q, float* z,
              int64_t max_iters, int64_t max_steps) {
    constexpr int GROUP = 4, RUN = 2;   // max_steps is rounded up to GROUP iterations
    static_assert(GROUP % RUN == 0, "");
    const char* ge = std::getenv("DTC_GRAPH");
    const bool use_graph = !(ge && ge[0] == '0') && !b.timing;
    bool fin = false;
    if (!use_graph) {
        DTC_TRY(all_done(b, b.done, &fin));
        if (fin) return DTC_OK;
        for (int64_t steps = 0; steps < max_steps; steps += GROUP) {
            if (steps > 0) {
                DTC_TRY(all_done(b, b.done, &fin));
                if (fin) return DTC_OK;
            }
            for (int k = 0; k < GROUP; ++k) DTC_TRY(block_iteration(b, wk, x, r, p, q, z, max_iters));
        }
        return DTC_OK;
    }
    hipStream_t s = b.stream;
    const void* key[6] = {x, r, p, q, z, b.done.p};
    bool same = b.block_graph.e && b.graph_iters == max_iters && b.graph_bricks == b.n_bricks &&
                b.graph_mode == (int)b.block64;
    for (int k = 0; k < 6; ++k) same = same && b.graph_key[k] == key[k];
    if (!same) {
        if (b.block_graph.e) DTC_HIP(stream_wait(s));   // no replay of the old one is in flight
        b.block_graph.reset();
        DTC_TRY(words_setup(b));
        hipGraph_t g = nullptr;
        DTC_HIP(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
        int rc = DTC_OK;
        for (int k = 0; k < RUN && rc == DTC_OK; ++k) rc = block_iteration(b, wk, x, r, p, q, z, max_iters);
        if (rc == DTC_OK) rc = post_done(b);
        const hipError_t ec = hipStreamEndCapture(s, &g);
        if (rc != DTC_OK && g) (void)hipGraphDestroy(g);
        DTC_TRY(rc);
        if (ec != hipSuccess) return set_error(DTC_ERR_DEVICE, "hipStreamEndCapture: %s", hipGetErrorString(ec));
        const hipError_t ei = hipGraphInstantiate(&b.block_graph.e, g, nullptr, nullptr, 0);
        b.block_graph.g = g;
        if (ei != hipSuccess) {
            b.block_graph.e = nullptr;
            b.block_graph.reset();
            return set_error(DTC_ERR_DEVICE, "hipGraphInstantiate: %s", hipGetErrorString(ei));
        }
        for (int k = 0; k < 6; ++k) b.graph_key[k] = key[k];
        b.graph_iters = max_iters;
        b.graph_bricks = b.n_bricks;
        b.graph_mode = (int)b.block64;
    }
    const int64_t total = (std::min<int64_t>(max_steps, INT64_MAX - GROUP) + GROUP - 1) / GROUP * GROUP;
    auto run = [&](int64_t steps) -> int {
        DTC_HIP(hipGraphLaunch(b.block_graph.e, s));
        ++b.runs;
        if (steps > 0) DTC_TRY(wait_done(b, b.runs - 1, &fin));   // the replay before this one
        return DTC_OK;
    };
    for (int64_t steps = 0; steps < total && !fin; steps += RUN) {
        const int rc = run(steps);
        if (rc != DTC_OK) {
            (void)stream_wait(s);   // nothing is in flight when the caller gives up
            return rc;
        }
        // DTC_TRACE=1: a progress line every 1,000 block iterations of a long phase
        if (trace_on() && (steps + RUN) % 1000 < RUN)
            std::fprintf(stderr, "[dtc] block phase: %lld iterations\n", (long long)(steps + RUN));
    }
    return DTC_OK;
}

// FP64 true residual r64 = -(K u)_free, u = x64, which holds the Dirichlet values,
// then per load case activity and targets (k_red_outer)
int residual64(SolverBatch& b, const WK<double>& wk, const double* x64, int first, const dtc_solve_opts& o) {
    double* r64 = b.r64.as<double>();
    DTC_TRY((launch_mv<double, IN_U, OUT_RESID>(b, wk, x64, r64, b.part_c.as<double>(), nullptr)));
    if (!b.micro20)   // (the HEX20 operator forms the sums itself)
        k_dot<double><<<b.n_bricks, NT_UPD, 0, b.stream>>>(b.brick.as<BrickInfo>(), nullptr, r64, r64, b.part_c.as<double>());
    const double* itol2 = b.precision == DTC_FP32_REFINE && !b.block64 ? b.itol2.as<double>() : nullptr;
    k_red_outer<<<b.n_dom, RED_NT, 0, b.stream>>>(b.dom.as<DomInfo>(), b.part_c.as<double>(), first,
                                                  o.rel_tol * o.rel_tol, itol2, b.rr0.as<double>(), b.rr.as<double>(),
                                                  b.active64.as<int>(), b.active.as<int>(), b.thr2.as<double>(),
                                                  b.done64.as<int>(), b.done.as<int>());
    DTC_HIP(hipGetLastError());
    return DTC_OK;
}

// Progress of the FP64 true residual over the residual replacements of the mixed
// solve: a domain whose worst load case has not halved its relative residual in
// STALL replacements, or whose residual is not finite, is given up (the caller
// repeats it in FP64).
struct Progress {
    static constexpr int STALL = 10;
    std::vector<double> best;
    std::vector<int64_t> at;
};

// inner iteration cap reached (or no progress, see Progress) for some domains:
// mark them finished
int apply_cap(SolverBatch& b, int64_t cap, std::vector<int64_t>& nouter, bool* any_left, Progress* pg = nullptr) {
    const int D = b.n_dom;
    const double* st = nullptr;
    DTC_TRY(read_status(b, &st));
    std::vector<int> h(D);
    std::vector<int64_t> hi(D);
    for (int d = 0; d < D; ++d) {
        h[d] = st[(size_t)d * STAT_N] != 0.0;
        hi[d] = (int64_t)st[(size_t)d * STAT_N + 1];
    }
    auto rr_of = [&](int d, int lc) { return st[(size_t)d * STAT_N + 2 + lc]; };
    auto rr0_of = [&](int d, int lc) { return st[(size_t)d * STAT_N + 2 + R + lc]; };
    if (pg && (int)pg->best.size() != D) {
        pg->best.assign(D, -1.0);
        pg->at.assign(D, 0);
    }
    // DTC_TRACE=1: one stderr line per residual replacement of the mixed solve
    // (domain: PCG iterations so far / worst relative FP64 residual)
    static const bool trace = std::getenv("DTC_TRACE") && std::getenv("DTC_TRACE")[0] == '1';
    if (trace && pg) {
        std::fprintf(stderr, "[dtc] replacement:");
        for (int d = 0; d < D; ++d) {
            double worst = 0.0;
            for (int lc = 0; lc < R; ++lc) {
                const double r0 = rr0_of(d, lc);
                if (r0 > 0.0) worst = std::fmax(worst, std::sqrt(rr_of(d, lc) / r0));
            }
            std::fprintf(stderr, " %d:%lld/%.1e", d, (long long)hi[d], worst);
        }
        std::fprintf(stderr, "\n");
    }
    bool any = false, changed = false;
    for (int d = 0; d < D; ++d) {
        bool stop = !h[d] && hi[d] >= cap;
        if (pg && !h[d] && !stop) {
            double worst = 0.0;
            for (int lc = 0; lc < R; ++lc) {
                const double r0 = rr0_of(d, lc), rr = rr_of(d, lc);
                const double v = r0 > 0.0 ? std::sqrt(rr / r0) : 0.0;
                worst = std::isfinite(v) && std::isfinite(r0) ? std::fmax(worst, v) : INFINITY;
            }
            if (!std::isfinite(worst)) stop = true;
            else if (pg->best[d] < 0.0 || worst < 0.5 * pg->best[d]) {
                pg->best[d] = worst;
                pg->at[d] = nouter[d];
            } else if (nouter[d] - pg->at[d] >= Progress::STALL) {
                stop = true;
            }
        }
        if (stop) { h[d] = 1; changed = true; }
        if (!h[d]) { nouter[d] += 1; any = true; }
    }
    if (changed) {
        DTC_HIP(hipMemcpyAsync(b.done64.p, h.data(), (size_t)D * 4, hipMemcpyHostToDevice, b.stream));
        DTC_HIP(hipMemcpyAsync(b.done.p, h.data(), (size_t)D * 4, hipMemcpyHostToDevice, b.stream));
        DTC_HIP(stream_wait(b.stream));   // h goes
    }
    *any_left = any;
    return DTC_OK;
}

}  // namespace

int batch_build_pmg(SolverBatch& b, SolverBatch& c) { return build_pmg(b, c); }

int batch_solve(SolverBatch& b, const dtc_solve_opts& opts, std::vector<int64_t>& iters,
                std::vector<int64_t>& outer, std::vector<double>& relres) {
    const int D = b.n_dom;
    // with the multigrid, the 24 load cases of a domain iterate as one block
    // (DTC_BLOCK_PCG=0: one PCG per load case)
    const bool block = b.precision == DTC_FP32_REFINE && block_pcg(b) && (!b.micro20 || b.p08);
    // inner_tol outside (0, 1): automatic, per domain.  The block restarts at every
    // FP64 residual replacement, so it takes its FP32 phases as deep as FP32
    // allows: 1e-6 (two phases to 1e-8 instead of three) where the moduli of the
    // domain's solid voxels differ by at most 100x; high-contrast (greyscale)
    // domains stall in FP32 before that and use 1e-4, as does one PCG per load
    // case (it keeps its direction over a replacement)
    const dtc_solve_opts& o = opts;
    if (D > 0) {
        std::vector<double>& it2 = b.h_itol2;
        it2.resize(D);
        for (int d = 0; d < D; ++d) {
            double t = o.inner_tol;
            if (!(t > 0.0 && t < 1.0)) {
                const double c = d < (int)b.h_contrast.size() ? b.h_contrast[d] : 1.0;
                t = block && c <= 100.0 ? 1e-6 : 1e-4;
            }
            it2[d] = t * t;
        }
        DTC_TRY(b.itol2.ensure((size_t)D * 8));
        DTC_HIP(hipMemcpyAsync(b.itol2.p, it2.data(), (size_t)D * 8, hipMemcpyHostToDevice, b.stream));
    }
    iters.assign(D, 0);
    outer.assign(D, 0);
    relres.assign(D, 0.0);
    if (D == 0 || b.n_bricks == 0) return DTC_OK;
    hipStream_t s = b.stream;
    const int64_t nv = b.n_nodes * 3 * R;
    const WK<double> wk64 = cast_wk<double>(b.wk64);
    const WK<float> wk32 = cast_wk<float>(b.wk64);
    const int64_t cap = o.max_iter > 0 ? o.max_iter : 100000;
    const BrickInfo* bl = b.brick.as<BrickInfo>();
    const DomInfo* dl = b.dom.as<DomInfo>();
    k_fill_i64<<<nb(D, 64), 64, 0, s>>>(b.iters.as<int64_t>(), D, 0);
    k_fill_f64<<<nb(nv, 256), 256, 0, s>>>(b.x64.as<double>(), nv, 0.0);
    if (b.precision == DTC_FP64) {
        k_fill_f64<<<nb(nv, 256), 256, 0, s>>>(b.p64.as<double>(), nv, 0.0);
        k_fill_f64<<<nb(nv, 256), 256, 0, s>>>(b.q64.as<double>(), nv, 0.0);
    } else {
        k_fill_f32<<<nb(nv, 256), 256, 0, s>>>(b.p32.as<float>(), nv, 0.f);
        k_fill_f32<<<nb(nv, 256), 256, 0, s>>>(b.q32.as<float>(), nv, 0.f);
    }
    DTC_HIP(hipGetLastError());
    for (KernelStat& k : b.kstat) k = KernelStat{};
    b.reactions_valid = false;
    if (b.timing) {
        // per domain group: vector bytes (FP32), moduli (FP32), Jacobi scaling (FP32), vector
        // bytes (FP64), dense element-product flops 2 (3 nen)^2 R N_e
        std::vector<double> db((size_t)D * 5, 0.0);
        const double nd = 3.0 * (b.micro20 ? 20 : 8);
        for (int d = 0; d < D; ++d) {
            const double nn = (double)(b.h_dom[d].node_end - b.h_dom[d].node_begin);
            const double ne = b.h_status[d] == DTC_OK ? (double)b.h_elems[d] : 0.0;
            db[5 * d] = 3.0 * nn * R * 4.0;
            db[5 * d + 1] = 4.0 * ne;
            db[5 * d + 2] = 3.0 * nn * 4.0;
            db[5 * d + 3] = 3.0 * nn * R * 8.0;
            db[5 * d + 4] = 2.0 * nd * nd * R * ne;
        }
        DTC_TRY(b.dom_bytes.ensure(db.size() * 8));
        DTC_TRY(b.launch_bytes.ensure((size_t)MAX_SLOTS * 2 * 8));
        DTC_HIP(hipMemcpyAsync(b.dom_bytes.p, db.data(), db.size() * 8, hipMemcpyHostToDevice, s));
        DTC_HIP(stream_wait(s));
        b.n_slots = 0;
    }
    std::vector<int64_t> nouter(D, 0);
    // high-contrast batches (solid moduli differing by more than 100x): the block
    // iterates on FP64 vectors with the FP32 V-cycle (DTC_BLOCK64=1 / 0 overrides)
    {
        double cmax = 1.0;
        for (double c : b.h_contrast) cmax = std::fmax(cmax, c);
        const char* e64 = std::getenv("DTC_BLOCK64");
        b.block64 = block && (e64 ? e64[0] == '1' : cmax > 100.0);
        if (b.block64) DTC_TRY(b.q64.ensure((size_t)nv * 8));
    }
    // r64 = f (lifted right-hand side).  The Dirichlet values are written into x64 once;
    // every update of x64 adds zero there, and its other readers form them again
    if (b.micro20) DTC_TRY(set_bc20(b, b.x64.as<double>()));
    else k_set_bc<<<dim3(b.n_bricks, 8), NT_UPD, 0, s>>>(bl, dl, b.lat2node.as<int>(), b.x64.as<double>());
    DTC_HIP(hipGetLastError());
    DTC_TRY(residual64(b, wk64, b.x64.as<double>(), 1, o));

    if (b.precision == DTC_FP64) {
        // PCG in FP64 on (x64, r64); a true-residual check restarts it if the
        // recursive residual drifted
        for (int it = 0; it < 16; ++it) {
            bool left = false;
            DTC_TRY(apply_cap(b, cap, nouter, &left));
            if (!left) break;
            double* x = b.x64.as<double>();
            double* r = b.r64.as<double>();
            k_cg_init<double><<<b.n_bricks, NT_UPD, 0, s>>>(bl, b.done64.as<int>(), b.active.as<int>(), x, r,
                                                            b.p64.as<double>(), b.dinv64.as<double>(),
                                                            b.part_a.as<double>(), b.part_b.as<double>(), 0, 1, nullptr,
                                                            nullptr);
            k_red_init<<<D, RED_NT, 0, s>>>(dl, b.done64.as<int>(), b.part_a.as<double>(), b.part_b.as<double>(),
                                            b.thr2.as<double>(), b.active.as<int>(), b.rz.as<double>(), b.done.as<int>());
            DTC_HIP(hipGetLastError());
            DTC_TRY(pcg_run<double>(b, wk64, x, r, b.p64.as<double>(), b.q64.as<double>(), b.dinv64.as<double>(), cap,
                                    INT64_MAX, nullptr));
            DTC_TRY(residual64(b, wk64, b.x64.as<double>(), 0, o));
        }
    } else {
        // FP32 PCG with FP64 residual replacement: the FP32 correction x32 is
        // folded into x64 when the recursive residual has dropped by inner_tol
        // (or meets the final target, or after REPLACE iterations), r32 is
        // replaced by the true FP64 residual and the search direction p32 is
        // kept.
        const bool mg = b.precond == DTC_PC_MG && (!b.micro20 || b.p08);
        Progress progress;   // domains that stop converging are given up (the caller repeats them in FP64)
        const int64_t REPLACE = mg ? 100 : 1000;
        float* x32 = b.x32.as<float>();
        float* r32 = b.r32.as<float>();
        float* p32 = b.p32.as<float>();
        float* z32 = mg ? b.z32.as<float>() : nullptr;
        // the block's A P in FP64 arithmetic (FP32 vectors) for HEX20 micro meshes,
        // in FP32 for HEX08 (DTC_BLOCK_Q64=1 / 0 overrides).  HEX20 rows sum up to
        // 480 products of mixed sign; in FP32 that sum loses the small eigenvalues
        // of W = P^T A P, and on meshes with corner- or edge-hinged voxel clusters
        // (near-mechanisms) the block then drifts along them and diverges.
        const char* bq64 = std::getenv("DTC_BLOCK_Q64");
        b.block_q64 = bq64 ? bq64[0] == '1' : b.micro20;
        const char* brs = std::getenv("DTC_BLOCK_RESTART");
        const bool block_restart = !(brs && brs[0] == '0');
        // a block phase ends at its targets; the cap only bounds FP32 drift
        const char* brp = std::getenv("DTC_BLOCK_REPLACE");
        const int64_t block_replace = brp ? std::max(1, std::atoi(brp)) : 400;
        // FP64 vectors: the recursion drifts far less, and a restart discards the
        // block's Krylov space, so a phase runs to its target (the true residual
        // is checked then).  A cap of 500 took the worst of sixteen 48^3 greyscale domains
        // from 4,846 to 1,501 iterations, but a 128^3 one from 708 to 1,316 (3.6 -> 6.7 s) and
        // a 96^3 HEX20/HEX20 one, which needs over a thousand in one phase, past 5,500
        const int64_t block_replace64 = brp ? block_replace : 20000;
        float* bp = p32;
        float* bq = b.q32.as<float>();
        float* bz = z32;
        if (block) DTC_TRY(block_setup(b));
        bool first = true;
        for (int it = 0; it < 100000; ++it) {
            bool left = false;
            DTC_TRY(apply_cap(b, cap, nouter, &left, &progress));
            if (!left) break;
            if (block)
                k_phase<<<nb(D, 64), 64, 0, s>>>(b.iters.as<int64_t>(), D, b.block64 ? 0 : it, b.len0.as<int64_t>(),
                                                 b.phase_end.as<int64_t>());
            // the block solves the correction problem with unit-norm columns: FP32
            // directions mix all 24 load cases, whose residuals drift apart in size
            k_to32<<<b.n_bricks, NT_UPD, 0, s>>>(bl, b.done64.as<int>(), b.r64.as<double>(), r32, x32,
                                                 block ? b.rr.as<double>() : nullptr);
            if (block && b.block64) {
                // FP64 vectors: the block restarts from M r at every true-residual check
                k_to32<<<b.n_bricks, NT_UPD, 0, s>>>(bl, b.done64.as<int>(), b.r64.as<double>(), r32, nullptr, nullptr);
                DTC_HIP(hipGetLastError());
                DTC_TRY(mg_vcycle(b, wk32, r32, bz, nullptr));
                DTC_TRY(block_orth(b, bz, bp));
                first = false;
                DTC_TRY(block_run(b, wk32, x32, r32, bp, bq, bz, cap, block_replace64));
                DTC_TRY(residual64(b, wk64, b.x64.as<double>(), 0, o));
                continue;
            }
            if (block) {
                // the direction block restarts from M r at every residual replacement
                // (DTC_BLOCK_RESTART=0: it is kept, spanning the same space after the
                // column scaling)
                if (first || block_restart) {
                    DTC_TRY(mg_vcycle(b, wk32, r32, bz, nullptr));
                    DTC_TRY(block_orth(b, bz, bp));
                }
                first = false;
                DTC_TRY(block_run(b, wk32, x32, r32, bp, bq, bz, cap, block_replace));
                k_acc64<<<b.n_bricks, NT_UPD, 0, s>>>(bl, b.done64.as<int>(), x32, b.x64.as<double>(), b.rr.as<double>());
                DTC_HIP(hipGetLastError());
                DTC_TRY(residual64(b, wk64, b.x64.as<double>(), 0, o));
                continue;
            }
            if (mg) DTC_TRY(mg_vcycle(b, wk32, r32, z32, nullptr));
            k_cg_init<float><<<b.n_bricks, NT_UPD, 0, s>>>(bl, b.done64.as<int>(), b.active.as<int>(), x32, r32, p32,
                                                           b.dinv32.as<float>(), b.part_a.as<double>(),
                                                           b.part_b.as<double>(), 0, first ? 1 : 0,
                                                           b.active_prev.as<int>(), z32);
            k_red_init<<<D, RED_NT, 0, s>>>(dl, b.done64.as<int>(), b.part_a.as<double>(), b.part_b.as<double>(),
                                            b.thr2.as<double>(), b.active.as<int>(), b.rz.as<double>(), b.done.as<int>());
            DTC_HIP(hipGetLastError());
            first = false;
            DTC_TRY(pcg_run<float>(b, wk32, x32, r32, p32, b.q32.as<float>(), b.dinv32.as<float>(), cap, REPLACE,
                                   z32));
            DTC_HIP(hipMemcpyAsync(b.active_prev.p, b.active.p, (size_t)D * R * 4, hipMemcpyDeviceToDevice, s));
            k_acc64<<<b.n_bricks, NT_UPD, 0, s>>>(bl, b.done64.as<int>(), x32, b.x64.as<double>(), nullptr);
            DTC_HIP(hipGetLastError());
            DTC_TRY(residual64(b, wk64, b.x64.as<double>(), 0, o));
        }
    }
    // results: iterations, true relative residual, convergence status
    const double* st = nullptr;
    DTC_TRY(read_status(b, &st));
    DTC_TRY(harvest_events(b));
    for (int d = 0; d < D; ++d) {
        const double* sd = st + (size_t)d * STAT_N;
        iters[d] = (int64_t)sd[1];
        outer[d] = nouter[d];
        double mx = 0.0;
        bool finite = true;
        for (int lc = 0; lc < R; ++lc) {
            const double r0 = sd[2 + R + lc], rr = sd[2 + lc];
            if (!std::isfinite(r0) || !std::isfinite(rr)) finite = false;
            else if (r0 > 0.0) mx = std::fmax(mx, std::sqrt(rr / r0));
        }
        relres[d] = finite ? mx : NAN;
        if (b.h_status[d] == DTC_OK && !(finite && mx <= o.rel_tol)) b.h_status[d] = DTC_ERR_NO_CONVERGENCE;
    }
    return DTC_OK;
}

int batch_forces(SolverBatch& b, std::vector<double>& ff) {
    const int D = b.n_dom;
    ff.assign((size_t)D * R * FFD, 0.0);
    if (D == 0 || b.n_bricks == 0) {
        DTC_HIP(stream_wait(b.stream));
        return DTC_OK;
    }
    const WK<double> wk64 = cast_wk<double>(b.wk64);
    // reactions on the unmodified operator: rf = K (x + x_bc), stored in r64
    DTC_TRY((launch_mv<double, IN_U, OUT_PLAIN>(b, wk64, b.x64.as<double>(), b.r64.as<double>(), nullptr, nullptr)));
    if (b.micro20) {
        DTC_TRY(project20(b));
    } else {
        k_project<8><<<b.n_bricks, NT_UPD, 0, b.stream>>>(b.brick.as<BrickInfo>(), b.dom.as<DomInfo>(),
                                                          b.lat2node.as<int>(), b.r64.as<double>(),
                                                          b.force_partials());
        k_project<20><<<b.n_bricks, NT_UPD, 0, b.stream>>>(b.brick.as<BrickInfo>(), b.dom.as<DomInfo>(),
                                                           b.lat2node.as<int>(), b.r64.as<double>(),
                                                           b.force_partials());
    }
    k_red_ff<<<dim3(D, (R * FFD + RFF_E - 1) / RFF_E), RFF_E * RFF_P, 0, b.stream>>>(b.dom.as<DomInfo>(),
                                                                                b.force_partials(), b.ff.as<double>());
    DTC_HIP(hipGetLastError());
    DTC_HIP(hipMemcpyAsync(ff.data(), b.ff.p, ff.size() * 8, hipMemcpyDeviceToHost, b.stream));
    DTC_HIP(stream_wait(b.stream));
    b.reactions_valid = true;
    return DTC_OK;
}

int batch_fields(SolverBatch& b, int i, int ncol, double* u_out, double* r_out) {
    if (i < 0 || i >= b.n_dom) return set_error(DTC_ERR_BAD_ARGUMENT, "domain index %d", i);
    const int64_t nn = b.h_nodes[i];
    if (nn == 0) return DTC_OK;
    if (r_out && !b.reactions_valid) return set_error(DTC_ERR_BAD_ARGUMENT, "reactions requested before the force pass");
    DevMem du, dr;
    if (ncol < 1 || ncol > R) return set_error(DTC_ERR_BAD_ARGUMENT, "field columns %d", ncol);
    const size_t bytes = (size_t)nn * 3 * ncol * 8;
    if (u_out) DTC_TRY(du.alloc(bytes));
    if (r_out) DTC_TRY(dr.alloc(bytes));
    if (b.micro20) {
        DTC_TRY(fields20(b, i, ncol, u_out ? du.as<double>() : nullptr, r_out ? dr.as<double>() : nullptr));
    } else {
        k_fields<<<b.n_bricks, NT_UPD, 0, b.stream>>>(b.brick.as<BrickInfo>(), b.dom.as<DomInfo>(),
                                                      b.lat2node.as<int>(), b.sol2ref.as<int>(), b.x64.as<double>(),
                                                      b.r64.as<double>(), i, nn, ncol, u_out ? du.as<double>() : nullptr,
                                                      r_out ? dr.as<double>() : nullptr);
        DTC_HIP(hipGetLastError());
    }
    if (u_out) DTC_HIP(hipMemcpyAsync(u_out, du.p, bytes, hipMemcpyDeviceToHost, b.stream));
    if (r_out) DTC_HIP(hipMemcpyAsync(r_out, dr.p, bytes, hipMemcpyDeviceToHost, b.stream));
    DTC_HIP(stream_wait(b.stream));
    du.recycle();
    dr.recycle();
    return DTC_OK;
}

int batch_grad(SolverBatch& b, int i, int ng, const double* M, double* dL_dE_host) {
    if (i < 0 || ng < 1 || i + ng > b.n_dom) return set_error(DTC_ERR_BAD_ARGUMENT, "domain groups %d..%d", i, i + ng - 1);
    if (b.micro20) return grad20(b, i, ng, M, dL_dE_host);
    const DomInfo& D = b.h_dom[i];
    const int64_t nvox = (int64_t)D.nx * D.ny * D.nz;
    const int64_t nn = b.n_nodes > 0 ? b.n_nodes : 1;
    DevMem h, Md, g;
    DTC_TRY(h.alloc((size_t)nn * 18 * 8));
    DTC_TRY(Md.alloc((size_t)ng * R * 6 * 8));
    DTC_TRY(g.alloc((size_t)nvox * 8));
    DTC_HIP(hipMemcpyAsync(Md.p, M, (size_t)ng * R * 6 * 8, hipMemcpyHostToDevice, b.stream));
    for (int k = 0; k < ng; ++k)
        if (b.h_dom[i + k].brick_end > b.h_dom[i + k].brick_begin)
            k_grad_h<<<b.n_bricks, NT_UPD, 0, b.stream>>>(b.brick.as<BrickInfo>(), b.dom.as<DomInfo>(),
                                                          b.lat2node.as<int>(), b.x64.as<double>(),
                                                          Md.as<double>() + (size_t)k * R * 6, i + k, D.node_begin,
                                                          k > 0, h.as<double>());
    k_grad_elem<<<nb(nvox, 128), 128, 0, b.stream>>>(b.dom.as<DomInfo>(), b.lat2node.as<int>(), b.emod.as<double>(),
                                                     b.x64.as<double>(), h.as<double>(), cast_wk<double>(b.wk64), i,
                                                     g.as<double>());
    DTC_HIP(hipGetLastError());
    DTC_HIP(hipMemcpyAsync(dL_dE_host, g.p, (size_t)nvox * 8, hipMemcpyDeviceToHost, b.stream));
    DTC_HIP(stream_wait(b.stream));
    for (DevMem* m : {&h, &Md, &g}) m->recycle();
    return DTC_OK;
}

}  // namespace dtc
