// ebe.hpp -- the element-by-element matvec of HEX08 voxel levels and its tables.
// Included by solver.hip inside its anonymous namespace.

// ---------------------------------------------------------------- cluster element tables
// Elements of a cluster: every element with a corner among the cluster's nodes, found
// by scanning the 9x5x5 element tiles of the cluster's bricks; an element that touches
// several of those bricks is taken in the brick that holds its lowest node of the
// cluster.  FILL = false counts them; FILL = true writes them in descending
// lexicographic order of their voxels (rank by counting, in LDS), so that the matvec
// adds a node's contributions in corner order 0..7 whatever the clusters are.  Behind the
// last cluster's elements FILL writes a spare record (nodes 0, modulus 0): a last cluster
// without an element reads it.
template <bool FILL>
__global__ __launch_bounds__(256) void k_cluster_elems(const ClusterInfo* __restrict__ cl, const BrickInfo* __restrict__ bricks,
                                                       const DomInfo* __restrict__ doms, const int* __restrict__ lat2node,
                                                       const double* __restrict__ emod, int* __restrict__ cnt,
                                                       int4* __restrict__ enode, uint2* __restrict__ eown,
                                                       double* __restrict__ eE64, float* __restrict__ eE32, int cap) {
    __shared__ int64_t s_key[FILL ? 8 * CL_CAP : 1];
    __shared__ int s_n;
    const ClusterInfo C = cl[blockIdx.x];
    const DomInfo D = doms[C.dom];
    const int tid = threadIdx.x;
    const int64_t Lx = D.nx + 1, Ly = D.ny + 1;
    auto corner = [&](int vx, int vy, int vz, int b) {
        return lat2node[D.lat_off + (vx + (b & 1)) + Lx * ((vy + ((b >> 1) & 1)) + Ly * (vz + (b >> 2)))];
    };
    if (tid == 0) s_n = 0;
    __syncthreads();
    for (int br = C.brick_begin; br < C.brick_end; ++br) {
        const BrickInfo B = bricks[br];
        if (tid < NET) {
            const int vx = B.x0 - 1 + tid % EX, vy = B.y0 - 1 + (tid / EX) % EY, vz = B.z0 - 1 + tid / (EX * EY);
            if (vx >= 0 && vy >= 0 && vz >= 0 && vx < D.nx && vy < D.ny && vz < D.nz) {
                const int64_t v = vx + (int64_t)D.nx * (vy + (int64_t)D.ny * vz);
                if (emod[D.vox_off + v] != 0.0) {
                    int low = INT32_MAX;
                    for (int b = 0; b < 8; ++b) {
                        const int q = corner(vx, vy, vz, b);
                        if (q >= C.node_begin && q < C.node_end) low = min(low, q);
                    }
                    if (low >= B.node_begin && low < B.node_end) {
                        const int k = atomicAdd(&s_n, 1);
                        if constexpr (FILL) s_key[k] = v;
                    }
                }
            }
        }
    }
    __syncthreads();
    const int n = s_n;
    if constexpr (!FILL) {
        if (tid == 0) cnt[blockIdx.x] = n;
    } else {
        for (int k = tid; k < n; k += 256) {
            const int64_t v = s_key[k];
            int rank = 0;
            for (int j = 0; j < n; ++j) rank += s_key[j] > v;
            const int vx = (int)(v % D.nx), vy = (int)((v / D.nx) % D.ny), vz = (int)(v / ((int64_t)D.nx * D.ny));
            int q[8];
            unsigned w[8];
            for (int b = 0; b < 8; ++b) {
                q[b] = corner(vx, vy, vz, b);
                w[b] = q[b] >= C.node_begin && q[b] < C.node_end ? (unsigned)(q[b] - C.node_begin) : (unsigned)cap;
            }
            const int64_t o = (int64_t)C.e_off + rank;
            enode[2 * o] = make_int4(q[0], q[1], q[2], q[3]);
            enode[2 * o + 1] = make_int4(q[4], q[5], q[6], q[7]);
            eown[o] = make_uint2(w[0] | w[1] << 8 | w[2] << 16 | w[3] << 24, w[4] | w[5] << 8 | w[6] << 16 | w[7] << 24);
            const double e = emod[D.vox_off + v];
            if (eE64) eE64[o] = e;
            eE32[o] = (float)e;
        }
        if (blockIdx.x == gridDim.x - 1 && tid == 0) {
            const int64_t o = (int64_t)C.e_off + n;
            enode[2 * o] = enode[2 * o + 1] = make_int4(0, 0, 0, 0);
            eown[o] = make_uint2(cap * 0x01010101u, cap * 0x01010101u);
            if (eE64) eE64[o] = 0.0;
            eE32[o] = 0.f;
        }
    }
}

// ---------------------------------------------------------------- matvec
// a * b rounded, never part of a fused multiply-add: the zero-start step's x must be the
// value that the stored form keeps
template <typename T> __device__ __forceinline__ T mul_rounded(T a, T b) {
#pragma clang fp contract(off)
    return a * b;
}

struct EbeArgs {
    const ClusterInfo* cl;
    const int* done;            // finished domains are skipped; may be null
    const int4* enode;
    const uint2* eown;
    const void* eE;             // element moduli (T)
    const void* dinv;           // Jacobi scaling per DOF (T), 0 exactly on Dirichlet rows
    double* partial;            // OUT_MASKED_DOT: [cluster][24]
    // OUT_CHEB / OUT_BRES only
    const void* bvec;           // right-hand side b
    void* dvec;                 // Chebyshev direction
    float c1, c2;               // Chebyshev coefficients of this step
    int cflags;                 // CH_*
    float cin;                  // IN_JS: the zero-start step's coefficient
};

// y = K x over the clusters of a level; one workgroup per cluster, one wave per LCW of
// the 24 load cases.
//   product  a wave takes 64 / LCW elements at a time, a lane one (element, load case):
//            it gathers the 24 values of x straight from memory (neighbouring elements
//            share nodes: most of these loads hit the vector cache), forms the
//            Walsh-basis product, and adds corner b to the accumulator of the node it
//            belongs to in LDS, b = 0..7.  For one b the lanes of a wave write different
//            nodes, a wave's LDS operations complete in order, and no other wave has
//            these load cases, so plain read-add-write needs no atomics and no
//            barriers and the order of a node's sum is fixed;
//   write    after one barrier the nodes' values leave as one contiguous run.
// What bounds it (16 trabecular 64^3 domains, 1.25 M nodes, one launch over all of them):
// the vector cache's lookups (65-80 % busy: a load of x takes one per 32-byte run) and the
// VALU (55 %) together, with 12 waves a CU, as many as the LDS accumulators allow; the
// Chebyshev step also moves 1.66 GB (4.2 TB/s, a copy reaches 5.1).  Against bricks staged in LDS
// in six load-case chunks with corner buffers and two barriers a chunk (16 waves, most
// lanes idle on sparse bricks): Q = K P 678 -> 340 us, Chebyshev step 762 -> 411, residual
// before restriction 693 -> 354, FP64 residual 4114 -> 960.  Measured beside it: clusters of
// 64 nodes 370 / 455 us (2.0 against 1.7 elements computed per element of the mesh), of 160
// and 192 361 / 428 and 418 / 481 (fewer waves); two load cases a lane 355 / 431; twelve
// load cases a wave 378 / 445, four 406 / 489 (more lookups); LDS float atomics 3269;
// consecutive clusters on one XCD unchanged.
// OUT_MASKED writes y with zero Dirichlet rows; OUT_MASKED_DOT also sums x.y per
// cluster; OUT_RESID writes -y on free rows and 0 on Dirichlet rows;
// OUT_PLAIN writes y; OUT_BRES writes b - y on free rows and 0 on Dirichlet rows;
// OUT_CHEB applies one Chebyshev-Jacobi step, d = c1 d + c2 D^-1 (b - y), yout = x + d
// (yout must not alias x).  TI / TO: types of the vectors x and y, T of the arithmetic.
template <typename T, typename TI, typename TO, int IN, int OUT, int LCW, int CAP>
__global__ __launch_bounds__(64 * R / LCW) void k_ebe(EbeArgs A, WK<T> wk, const TI* __restrict__ xin,
                                                    TO* __restrict__ yout) {
    constexpr int NT = 64 * R / LCW, EPW = 64 / LCW, RC = MvCfg<T>::RC, NV = 3 * R / RC;
    constexpr bool SUMS = OUT == OUT_MASKED_DOT;
    using V = typename MvCfg<T>::V;
    static_assert(IN != IN_U && (IN == IN_V || OUT == OUT_CHEB), "zero-start input: Chebyshev step");
    static_assert(R % LCW == 0 && 64 % LCW == 0 && CAP < 256, "whole waves, byte-sized node indices");
    __shared__ V s_yv[(CAP + 1) * NV];        // the last row takes the corners outside the cluster
    constexpr int SEG = 8;
    __shared__ double s_red[SUMS ? SEG * R : 1];
    T* s_y = reinterpret_cast<T*>(s_yv);
    const ClusterInfo C = A.cl[blockIdx.x];
    const int tid = threadIdx.x, lane = tid & 63;
    const int lc = (tid >> 6) * LCW + lane % LCW, le = lane / LCW;
    const int ne = C.e_cnt, nv = (C.node_end - C.node_begin) * NV;
    const int4* __restrict__ en = A.enode + 2 * (int64_t)C.e_off;
    const uint2* __restrict__ eo = A.eown + C.e_off;
    const T* __restrict__ eE = static_cast<const T*>(A.eE) + C.e_off;
    const T* __restrict__ dinv = static_cast<const T*>(A.dinv);
    // (A cluster has no element where every voxel around its nodes is solid with modulus 0: it
    // reads the record at its offset, the next cluster's or the spare one at the end.)
    // Software pipeline: the records of the group after next and x of the next group are
    // loaded while the current group is computed.  Lanes past the last element repeat it
    // into the row that is not read; nothing is selected from a loaded record before it
    // is used (a select would wait for the record and, loads completing in order, for
    // the x loads before it)
    int4 n0, n1;
    uint2 ow;
    T E;
    const int last = max(ne - 1, 0);
    auto fetch = [&](int e) {
        const int i = min(e, last);
        n0 = en[2 * i];
        n1 = en[2 * i + 1];
        ow = eo[i];
        E = eE[i];
    };
    T w[8][3];
    T sc[IN == IN_JS ? 8 : 1];
    auto gather = [&]() {
        const int nd[8] = {n0.x, n0.y, n0.z, n0.w, n1.x, n1.y, n1.z, n1.w};
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const TI* xp = xin + (int64_t)nd[b] * (3 * R) + lc;
#pragma unroll
            for (int d = 0; d < 3; ++d) w[b][d] = (T)xp[d * R];
            if constexpr (IN == IN_JS) sc[b] = dinv[(int64_t)nd[b] * 3];
        }
    };
    fetch(le);
    if (A.done && A.done[C.dom]) return;
    for (int i = tid; i < nv; i += NT) vzero(s_yv[i]);
    gather();
    uint2 oc = ow;
    T Ec = E;
    fetch(EPW + le);
    __syncthreads();
    for (int e0 = 0; e0 < ne; e0 += EPW) {
        T y[8][3];
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            T v[8];
#pragma unroll
            for (int b = 0; b < 8; ++b) {
                v[b] = w[b][d];
                // the product order of k_cheb's zero start: (c2 dinv) v
                if constexpr (IN == IN_JS) v[b] = mul_rounded(mul_rounded((T)A.cin, sc[b]), v[b]);
            }
            fht_fwd(v);
#pragma unroll
            for (int b = 0; b < 8; ++b) w[b][d] = v[b];
        }
        walsh_apply(wk, w, y);
        const uint2 oy = e0 + le < ne ? oc : make_uint2(CAP * 0x01010101u, CAP * 0x01010101u);
        const T Ey = Ec;
        if (e0 + EPW < ne) {
            gather();
            oc = ow;
            Ec = E;
            if (e0 + 2 * EPW < ne) fetch(e0 + 2 * EPW + le);
        }
        T o[3][8];
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            // mode 0 (rigid translation) carries no force: the first inverse
            // butterfly of the pair (0, 1) reduces to (-y1, y1)
            const T y1 = y[1][d] * Ey;
            o[d][0] = -y1;
            o[d][1] = y1;
#pragma unroll
            for (int b = 2; b < 8; b += 2) {
                const T a = y[b][d] * Ey, c = y[b + 1][d] * Ey;
                o[d][b] = a - c;
                o[d][b + 1] = a + c;
            }
            fht_inv_tail(o[d]);
        }
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const unsigned k = ((b < 4 ? oy.x : oy.y) >> (8 * (b & 3))) & 255u;
            T* yp = s_y + k * (3 * R) + lc;
            T a[3];
#pragma unroll
            for (int d = 0; d < 3; ++d) a[d] = yp[d * R];
#pragma unroll
            for (int d = 0; d < 3; ++d) yp[d * R] = a[d] + o[d][b];
            // other lanes of the wave read these rows at the next corner
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        }
    }
    __syncthreads();
    const int64_t v0 = (int64_t)C.node_begin * NV;
    for (int i = tid; i < nv; i += NT) {
        V y = s_yv[i];
        const int64_t vi = v0 + i;
        const T di = OUT == OUT_PLAIN ? T(1) : dinv[vi / (R / RC)];
        const bool bc = di == T(0);
        if constexpr (OUT == OUT_MASKED || OUT == OUT_MASKED_DOT) {
            if (bc) vzero(y);
        } else if constexpr (OUT == OUT_RESID) {
            if (bc) vzero(y); else y = vneg(y);
        } else if constexpr (OUT == OUT_BRES) {
            V t = reinterpret_cast<const V*>(A.bvec)[vi];
            vadd(t, vneg(y));
            if (bc) vzero(t);
            y = t;
        } else if constexpr (OUT == OUT_CHEB) {
            const V bv = reinterpret_cast<const V*>(A.bvec)[vi];
            V* dp = reinterpret_cast<V*>(A.dvec) + vi;
            V xo, dv, dn, xn;
            if constexpr (IN == IN_JS) {
                const T s0 = mul_rounded((T)A.cin, di);
                T* xq = reinterpret_cast<T*>(&xo);
#pragma unroll
                for (int k = 0; k < RC; ++k) xq[k] = mul_rounded(s0, vcomp(bv, k));
            } else {
                xo = reinterpret_cast<const V*>(xin)[vi];
            }
            vzero(dv);
            if (A.cflags & CH_READ_D) dv = *dp;
            if (A.cflags & CH_D_FROM_X) dv = xo;
            vzero(dn);
            vzero(xn);
            if (!bc) {
                T* dq = reinterpret_cast<T*>(&dn);
                T* xq = reinterpret_cast<T*>(&xn);
#pragma unroll
                for (int k = 0; k < RC; ++k) {
                    const T r = vcomp(bv, k) - vcomp(y, k);
                    dq[k] = (T)A.c1 * vcomp(dv, k) + (T)A.c2 * di * r;
                    xq[k] = vcomp(xo, k) + dq[k];
                }
            }
            if (A.cflags & CH_WRITE_D) *dp = dn;
            y = xn;
        }
        if constexpr (SUMS) s_yv[i] = y;
        if constexpr (sizeof(TO) < sizeof(T)) {
            reinterpret_cast<float2*>(yout)[vi] = make_float2((float)vcomp(y, 0), (float)vcomp(y, 1));
        } else {
            reinterpret_cast<V*>(yout)[vi] = y;
        }
    }
    if constexpr (SUMS) {
        // fixed order whatever LCW is: 8 interleaved row sums per load case, added in order
        __syncthreads();
        const int rows = (C.node_end - C.node_begin) * 3;
        for (int t = tid; t < SEG * R; t += NT) {
            const int l = t % R;
            double s = 0.0;
            for (int j = t / R; j < rows; j += SEG) {
                s += (double)xin[(int64_t)C.node_begin * (3 * R) + j * R + l] * (double)s_y[j * R + l];
            }
            s_red[t] = s;
        }
        __syncthreads();
        if (tid < R) {
            double s = 0.0;
#pragma unroll
            for (int k = 0; k < SEG; ++k) s += s_red[k * R + tid];
            A.partial[(int64_t)blockIdx.x * R + tid] = s;
        }
    }
}

// ---------------------------------------------------------------- coarsest level
// All m steps of the coarsest level's Chebyshev-Jacobi pass from x = 0 in one launch: one
// workgroup per (domain, load case), everything in LDS and registers.  A step is two
// passes: thread v forms the forces of voxel v into s_y, then thread t (a lattice node)
// sums its up to 8 corners in ascending order of voxel offset and updates its d and x.  At
// most 8 voxels an edge: 512 voxels, 729 nodes.  One launch per step took 5-7 us each whatever
// the size, 28 us for degree 6 under a 12^3 domain (343 nodes) and 33 under a 64^3 one (729);
// this takes 7.8 and 12.3.
constexpr int COARSE_EDGE = 8, COARSE_STEPS = 16;
struct CoarseCheb {
    int m;
    float c1[COARSE_STEPS], c2[COARSE_STEPS];
};
template <int NT>
__global__ __launch_bounds__(NT) void k_coarse(const DomInfo* __restrict__ doms, const int* __restrict__ lat2node,
                                               const double* __restrict__ emod, const float* __restrict__ dinv,
                                               const int* __restrict__ done, WK<float> wk, const float* __restrict__ bvec,
                                               float* __restrict__ xout, CoarseCheb C) {
    constexpr int NVX = NT < COARSE_EDGE * COARSE_EDGE * COARSE_EDGE ? NT : COARSE_EDGE * COARSE_EDGE * COARSE_EDGE;
    __shared__ float s_x[3][NT];
    __shared__ float s_y[24][NVX];
    const int dom = blockIdx.x, lc = blockIdx.y, t = threadIdx.x;
    if (done && done[dom]) return;
    const DomInfo D = doms[dom];
    const int Lx = D.nx + 1, Ly = D.ny + 1, NL = Lx * Ly * (D.nz + 1), NV = D.nx * D.ny * D.nz;
    const int q = t < NL ? lat2node[D.lat_off + t] : -1;
    const int g[3] = {t % Lx, (t / Lx) % Ly, t / (Lx * Ly)};
    const float E = t < NV ? (float)emod[D.vox_off + t] : 0.f;
    const int n0 = t % D.nx + Lx * ((t / D.nx) % D.ny + Ly * (t / (D.nx * D.ny)));   // corner 0 of voxel t
    float b[3] = {0.f, 0.f, 0.f}, di[3] = {0.f, 0.f, 0.f}, d[3], x[3];
    if (q >= 0) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            b[k] = bvec[((int64_t)q * 3 + k) * R + lc];
            di[k] = dinv[(int64_t)q * 3 + k];
        }
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) x[k] = d[k] = C.c2[0] * di[k] * b[k];
    for (int st = 1; st < C.m; ++st) {
#pragma unroll
        for (int k = 0; k < 3; ++k) s_x[k][t] = x[k];
        __syncthreads();
        if (t < NV) {
            float w[8][3], y[8][3];
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                float v[8];
#pragma unroll
                for (int c = 0; c < 8; ++c) v[c] = s_x[k][n0 + (c & 1) + Lx * (((c >> 1) & 1) + Ly * (c >> 2))];
                fht_fwd(v);
#pragma unroll
                for (int c = 0; c < 8; ++c) w[c][k] = v[c];
            }
            walsh_apply(wk, w, y);
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                float o[8];
                const float y1 = y[1][k] * E;
                o[0] = -y1;
                o[1] = y1;
#pragma unroll
                for (int c = 2; c < 8; c += 2) {
                    const float p = y[c][k] * E, r = y[c + 1][k] * E;
                    o[c] = p - r;
                    o[c + 1] = p + r;
                }
                fht_inv_tail(o);
#pragma unroll
                for (int c = 0; c < 8; ++c) s_y[3 * c + k][t] = o[c];
            }
        }
        __syncthreads();
        if (t < NL) {
            float y[3] = {0.f, 0.f, 0.f};
#pragma unroll
            for (int c = 7; c >= 0; --c) {   // this node is corner c of the voxel
                const int vx = g[0] - (c & 1), vy = g[1] - ((c >> 1) & 1), vz = g[2] - (c >> 2);
                const bool in = vx >= 0 && vy >= 0 && vz >= 0 && vx < D.nx && vy < D.ny && vz < D.nz;
                const int v = in ? vx + D.nx * (vy + D.ny * vz) : 0;
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    const float f = s_y[3 * c + k][v];
                    y[k] += in ? f : 0.f;
                }
            }
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                d[k] = C.c1[st] * d[k] + C.c2[st] * di[k] * (b[k] - y[k]);
                x[k] += d[k];
            }
        }
    }
    if (q >= 0) {
#pragma unroll
        for (int k = 0; k < 3; ++k) xout[((int64_t)q * 3 + k) * R + lc] = x[k];
    }
}

