// mesh.hip -- voxel -> hex meshing on gfx950, bit-exact to gen_quadmesh_from_phi
// (f-src/mod_gen_quadmesh.f90:22-679).
//
// The reference works sequentially: elements in voxel scan order (x fastest),
// first-touch node numbering, max-label colouring until no change, a keep
// rule per colour and a stable compaction.  Here every step is a data-parallel
// integer pass over voxels, lattice nodes or node numbers:
//   * element index     = exclusive scan of the solid flags;
//   * node numbering    = the first toucher of a lattice node is its touching
//                         solid voxel with the smallest voxel index (element
//                         order follows voxel order), so each voxel counts the
//                         local nodes it touches first, a scan gives the base
//                         number and the local order gives the rest;
//   * colouring         = lock-free union-find over 26-neighbouring solid
//                         voxels (the colour partition is the connected-
//                         component partition; the label values are not output);
//   * keep rule         = component of the first element, or any voxel of the
//                         component on the node bounding box (the reference's
//                         0.1*delta coordinate tests are exact lattice equalities);
//   * compaction        = scans over the keep flags, with the last element and
//                         the last node always kept (:597-651).

#include <algorithm>

#include "dtc_internal.hpp"

namespace dtc {

namespace {

constexpr int NT = 256;

__host__ __device__ constexpr int h20_off(int l, int d) {
    // HEX20 local node offsets on the doubled lattice (f-src/mod_gen_quadmesh.f90:244-265)
    constexpr signed char T[20][3] = {
        {0, 0, 0}, {1, 0, 0}, {2, 0, 0}, {2, 1, 0}, {2, 2, 0}, {1, 2, 0}, {0, 2, 0}, {0, 1, 0},
        {0, 0, 1}, {2, 0, 1}, {2, 2, 1}, {0, 2, 1},
        {0, 0, 2}, {1, 0, 2}, {2, 0, 2}, {2, 1, 2}, {2, 2, 2}, {1, 2, 2}, {0, 2, 2}, {0, 1, 2}};
    return T[l][d];
}

__device__ inline int local_of_offset(int nen, int ox, int oy, int oz) {
    if (nen == 8) {
        constexpr signed char L8[8] = {0, 1, 3, 2, 4, 5, 7, 6};   // index ox + 2oy + 4oz
        return L8[ox + 2 * oy + 4 * oz];
    }
    for (int l = 0; l < 20; ++l)
        if (h20_off(l, 0) == ox && h20_off(l, 1) == oy && h20_off(l, 2) == oz) return l;
    return -1;
}

__host__ __device__ constexpr int node_off(int nen, int l, int d) { return nen == 8 ? h08_off(l, d) : h20_off(l, d); }

// Candidate voxels touching lattice coordinate a along one axis, in increasing
// voxel order, with the node's offset inside that voxel.
__device__ inline int axis_candidates(int a, int mul, int n, int vox[2], int off[2]) {
    int c = 0;
    if (mul == 1) {
        if (a - 1 >= 0 && a - 1 < n) { vox[c] = a - 1; off[c] = 1; ++c; }
        if (a >= 0 && a < n) { vox[c] = a; off[c] = 0; ++c; }
    } else if ((a & 1) == 0) {
        int x = a >> 1;
        if (x - 1 >= 0 && x - 1 < n) { vox[c] = x - 1; off[c] = 2; ++c; }
        if (x >= 0 && x < n) { vox[c] = x; off[c] = 0; ++c; }
    } else {
        int x = a >> 1;
        if (x >= 0 && x < n) { vox[c] = x; off[c] = 1; ++c; }
    }
    return c;
}

// First toucher of lattice node (a,b,c): the solid voxel with the smallest
// voxel index among the voxels containing it; -1 if none.
__device__ inline int first_toucher(const uint8_t* __restrict__ solid, int nx, int ny, int nz, int mul,
                                    int a, int b, int c, int* ox, int* oy, int* oz) {
    int vx[2], fx[2], vy[2], fy[2], vz[2], fz[2];
    int cx = axis_candidates(a, mul, nx, vx, fx);
    int cy = axis_candidates(b, mul, ny, vy, fy);
    int cz = axis_candidates(c, mul, nz, vz, fz);
    for (int k = 0; k < cz; ++k)
        for (int j = 0; j < cy; ++j)
            for (int i = 0; i < cx; ++i) {
                int v = vx[i] + nx * (vy[j] + ny * vz[k]);
                if (solid[v]) { *ox = fx[i]; *oy = fy[j]; *oz = fz[k]; return v; }
            }
    return -1;
}

// solid voxels and the start values of what the following passes collect
template <typename P>
__global__ void k_solid(const P* __restrict__ phi, int nvox, int64_t llimit, uint8_t* __restrict__ solid,
                        int* __restrict__ flag, int* __restrict__ parent, uint8_t* __restrict__ touch,
                        int* __restrict__ bbox) {
    int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v < 6) bbox[v] = v & 1 ? -1 : INT32_MAX;
    if (v >= nvox) return;
    int s = (int64_t)phi[v] >= llimit;   // f-src/mod_gen_quadmesh.f90:242,296
    solid[v] = (uint8_t)s;
    flag[v] = s;
    parent[v] = v;
    touch[v] = 0;
}

__global__ void k_fill_i32(int* __restrict__ a, int64_t n, int v) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) a[i] = v;
}

__device__ inline int uf_find(int* parent, int x) {
    volatile int* pv = parent;
    for (;;) {
        int p = pv[x];
        if (p == x) return x;
        int gp = pv[p];
        if (gp != p) pv[x] = gp;   // path halving; any stale value is still an ancestor
        x = p;
    }
}

// the same without writes
__device__ inline int uf_root(const int* parent, int x) {
    const volatile int* pv = parent;
    for (;;) {
        const int p = pv[x];
        if (p == x) return x;
        x = p;
    }
}

// node numbers, and a first pass of shortcuts through the components: it leaves short
// paths, not roots (a halving write can land on a parent that another thread has just set)
__global__ void k_number(const uint8_t* __restrict__ solid, const uint32_t* __restrict__ ftmask,
                         const int* __restrict__ nbase, int nx, int ny, int nz, int nen, int mul, int Lx, int Ly,
                         int* __restrict__ numLat, int* __restrict__ latOfNum, int* parent) {
    int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nx * ny * nz || !solid[v]) return;
    parent[v] = uf_find(parent, v);
    uint32_t mask = ftmask[v];
    int x = v % nx, y = (v / nx) % ny, z = v / (nx * ny);
    for (int l = 0; l < nen; ++l) {
        if (!(mask & (1u << l))) continue;
        int num = nbase[v] + __popc(mask & ((1u << l) - 1u)) + 1;
        int p = (x * mul + node_off(nen, l, 0)) + Lx * ((y * mul + node_off(nen, l, 1)) + Ly * (z * mul + node_off(nen, l, 2)));
        numLat[p] = num;
        latOfNum[num - 1] = p;
    }
}

__device__ inline void uf_unite(int* parent, int a, int b) {
    for (;;) {
        a = uf_find(parent, a);
        b = uf_find(parent, b);
        if (a == b) return;
        if (a < b) { int t = a; a = b; b = t; }
        // hook the larger root under the smaller one: the final root of a
        // component is its smallest voxel index
        if (atomicCAS(&parent[a], a, b) == a) return;
    }
}

// The 13 neighbours of a voxel with a smaller index among the 26 that share a node with it:
// bit 0..8 the plane z - 1, 9..11 the row y - 1, 12 the voxel x - 1.
__host__ __device__ constexpr int prev_off(int k, int d) {
    return k < 9 ? (d == 0 ? k % 3 - 1 : d == 1 ? k / 3 - 1 : -1) : k < 12 ? (d == 0 ? k - 10 : d == 1 ? -1 : 0)
                                                                          : (d == 0 ? -1 : 0);
}
// those that contain local node l
constexpr uint32_t prev_sharing(int nen, int l) {
    uint32_t m = 0;
    for (int k = 0; k < 13; ++k) {
        bool in = true;
        for (int d = 0; d < 3; ++d) {
            const int o = node_off(nen, l, d), p = prev_off(k, d);
            in = in && (p == 0 || (p < 0 ? o == 0 : o == (nen == 8 ? 1 : 2)));
        }
        if (in) m |= 1u << k;
    }
    return m;
}
// those that share a node with neighbour k (itself included)
constexpr uint32_t prev_adjacent(int k) {
    uint32_t m = 0;
    for (int j = 0; j < 13; ++j) {
        bool in = true;
        for (int d = 0; d < 3; ++d) {
            const int t = prev_off(j, d) - prev_off(k, d);
            in = in && t >= -1 && t <= 1;
        }
        if (in) m |= 1u << j;
    }
    return m;
}
template <int NEN> struct PrevTables {
    uint32_t share[NEN] = {}, adj[13] = {};
    constexpr PrevTables() {
        for (int l = 0; l < NEN; ++l) share[l] = prev_sharing(NEN, l);
        for (int k = 0; k < 13; ++k) adj[k] = prev_adjacent(k);
    }
};

// One look at a voxel's earlier neighbours gives
//  * the nodes it touches first (none of the earlier voxels that share them is solid);
//  * its unions.  Two solid voxels are connected when they share a node; a neighbour that
//    shares a node with one already united is connected to that one by the unions of the
//    later of the two, so faces come first and most voxels need one union instead of up
//    to 13 (trabecular 64^3: 13 unions and 8 first-touch searches a voxel 197 + 30 us, with the
//    bounding box, whose 6,144 atomics took 71; 51 us now);
//  * the bounding box of the solid voxels.
template <int NEN>
__global__ __launch_bounds__(NT) void k_voxel(const uint8_t* __restrict__ solid, int nx, int ny, int nz,
                                              uint32_t* __restrict__ ftmask, int* __restrict__ cnt, int* parent,
                                              int* bbox) {
    constexpr PrevTables<NEN> T;
    constexpr int ORD[13] = {4, 10, 12, 1, 3, 5, 7, 9, 11, 0, 2, 6, 8};   // faces, edges, corners
    __shared__ int s_box[6][NT / 64];
    const int v = blockIdx.x * NT + threadIdx.x, nvox = nx * ny * nz;
    int lo[3] = {INT32_MAX, INT32_MAX, INT32_MAX}, hi[3] = {-1, -1, -1};
    uint32_t mask = 0;
    if (v < nvox && solid[v]) {
        const int c[3] = {v % nx, (v / nx) % ny, v / (nx * ny)};
        uint32_t nb = 0;
#pragma unroll
        for (int k = 0; k < 13; ++k) {
            const int x = c[0] + prev_off(k, 0), y = c[1] + prev_off(k, 1), z = c[2] + prev_off(k, 2);
            if (x >= 0 && y >= 0 && z >= 0 && x < nx && y < ny && solid[x + nx * (y + ny * z)]) nb |= 1u << k;
        }
#pragma unroll
        for (int l = 0; l < NEN; ++l)
            if (!(nb & T.share[l])) mask |= 1u << l;
#pragma unroll
        for (int i = 0; i < 13; ++i) {
            const int k = ORD[i];
            if (!(nb >> k & 1u)) continue;
            uf_unite(parent, v, v + prev_off(k, 0) + nx * (prev_off(k, 1) + ny * prev_off(k, 2)));
            nb &= ~T.adj[k];
        }
        for (int d = 0; d < 3; ++d) lo[d] = hi[d] = c[d];
    }
    if (v < nvox) {
        ftmask[v] = mask;
        cnt[v] = __popc(mask);
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        for (int w = 32; w > 0; w >>= 1) {
            lo[d] = min(lo[d], __shfl_xor(lo[d], w));
            hi[d] = max(hi[d], __shfl_xor(hi[d], w));
        }
        if (lane == 0) {
            s_box[2 * d][wave] = lo[d];
            s_box[2 * d + 1][wave] = hi[d];
        }
    }
    __syncthreads();
    if (threadIdx.x < 6) {
        const int q = threadIdx.x;
        int b = s_box[q][0];
        for (int w = 1; w < NT / 64; ++w) b = q & 1 ? max(b, s_box[q][w]) : min(b, s_box[q][w]);
        // the bound only tightens: no atomic where the value read is already as tight
        const int now = *(volatile int*)&bbox[q];
        if (q & 1) {
            if (b > now) atomicMax(&bbox[q], b);
        } else {
            if (b < now) atomicMin(&bbox[q], b);
        }
    }
}

// keep rule, f-src/mod_gen_quadmesh.f90:482-553: the first colour (component
// of node 1 = component of the first element) always; any other component
// with a node on the bounding box of all nodes
__global__ void k_touch(const uint8_t* __restrict__ solid, const int* __restrict__ eidx, int* parent,
                        const int* __restrict__ bbox, int nx, int ny, int nz, uint8_t* __restrict__ touch) {
    int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nx * ny * nz || !solid[v]) return;
    const int root = uf_root(parent, v);   // every write of this pass is a root: parent[] ends as roots
    parent[v] = root;
    int x = v % nx, y = (v / nx) % ny, z = v / (nx * ny);
    bool hit = (eidx[v] == 0) || x == bbox[0] || x == bbox[1] || y == bbox[2] || y == bbox[3] ||
               z == bbox[4] || z == bbox[5];
    if (hit) touch[root] = 1;
}

__global__ void k_keepE(const uint8_t* __restrict__ solid, const int* __restrict__ eidx,
                        const int* __restrict__ parent, const uint8_t* __restrict__ touch, int nvox,
                        const int* __restrict__ tot, int* __restrict__ keepE) {
    int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nvox) return;
    int k = 0;
    if (solid[v]) k = (touch[parent[v]] || eidx[v] == tot[0] - 1) ? 1 : 0;   // last element kept (:597-614)
    keepE[v] = k;
}

__global__ void k_keepN(const uint8_t* __restrict__ solid, const int* __restrict__ latOfNum,
                        const int* __restrict__ parent, const uint8_t* __restrict__ touch, int nx, int ny, int nz,
                        int mul, int Lx, int Ly, int nmax, const int* __restrict__ tot, int* __restrict__ keepN) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= nmax) return;
    const int nn0 = tot[1];
    if (k >= nn0) {
        keepN[k] = 0;
        return;
    }
    int p = latOfNum[k];
    int a = p % Lx, b = (p / Lx) % Ly, c = p / (Lx * Ly);
    int ox, oy, oz;
    int ft = first_toucher(solid, nx, ny, nz, mul, a, b, c, &ox, &oy, &oz);
    keepN[k] = (touch[parent[ft]] || k == nn0 - 1) ? 1 : 0;   // last node kept (:619-651)
}

__global__ void k_out_elems(const int* __restrict__ keepE, const int* __restrict__ newE,
                            const int* __restrict__ numLat, const int* __restrict__ keepN,
                            const int* __restrict__ cref, int nx, int ny, int nz, int nen, int mul, int Lx,
                            int Ly, int64_t* __restrict__ elems) {
    int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nx * ny * nz || !keepE[v]) return;
    int x = v % nx, y = (v / nx) % ny, z = v / (nx * ny);
    int64_t e = newE[v];
    for (int l = 0; l < nen; ++l) {
        int p = (x * mul + node_off(nen, l, 0)) + Lx * ((y * mul + node_off(nen, l, 1)) + Ly * (z * mul + node_off(nen, l, 2)));
        int num = numLat[p];
        elems[e * nen + l] = keepN[num - 1] ? (int64_t)cref[num - 1] + 1 : 0;   // :656-660
    }
}

// coordinates, f-src/mod_gen_quadmesh.f90:346-384 (same IEEE operations)
__global__ void k_out_nodes(const int* __restrict__ keepN, const int* __restrict__ cref,
                            const int* __restrict__ latOfNum, int nn0, int mul, int Lx, int Ly, double dx,
                            double dy, double dz, int64_t xa0, int64_t xa1, int64_t xa2, double* __restrict__ nodes) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= nn0 || !keepN[k]) return;
    int p = latOfNum[k];
    int64_t ii = p % Lx, jj = (p / Lx) % Ly, kk = p / (Lx * Ly);
    int64_t o = 3 * (int64_t)cref[k];
    if (mul == 2) {
        nodes[o + 2] = ((double)kk / 2.0 + (double)(xa2 - 1)) * dz;
        nodes[o + 1] = ((double)jj / 2.0 + (double)(xa1 - 1)) * dy;
        nodes[o + 0] = ((double)ii / 2.0 + (double)(xa0 - 1)) * dx;
    } else {
        nodes[o + 2] = (double)(kk + xa2 - 1) * dz;
        nodes[o + 1] = (double)(jj + xa1 - 1) * dy;
        nodes[o + 0] = (double)(ii + xa0 - 1) * dx;
    }
}

inline unsigned grid_of(int64_t n) { return (unsigned)((n + NT - 1) / NT); }

}  // namespace

namespace {

// Exclusive prefix sums of int32 values: tiles of SCAN_TILE values (256 threads x
// 4), then every tile's values rescanned with the sum of the tiles before it.  Up to
// SCAN_LOOK tiles each workgroup adds those sums itself, which saves a launch; more
// are scanned by one workgroup in between.  Integer sums: exact and independent of the
// order.  The total goes to device and page-locked host memory.
constexpr int SCAN_NT = 256, SCAN_ITEMS = 4, SCAN_TILE = SCAN_NT * SCAN_ITEMS;
constexpr int64_t SCAN_LOOK = 4096;

// inclusive scan of one value per thread over the workgroup; returns the
// workgroup total in *total
__device__ inline int block_incl_scan(int v, int* s_w, int* total) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int u = __shfl_up(v, o);
        if (lane >= o) v += u;
    }
    if (lane == 63) s_w[wave] = v;
    __syncthreads();
    int base = 0, tot = 0;
#pragma unroll
    for (int w = 0; w < SCAN_NT / 64; ++w) {
        const int c = s_w[w];
        if (w < wave) base += c;
        tot += c;
    }
    __syncthreads();
    *total = tot;
    return v + base;
}

__global__ __launch_bounds__(SCAN_NT) void k_scan_tiles(const int* __restrict__ in, int64_t n, int* __restrict__ tile_sum) {
    __shared__ int s_w[SCAN_NT / 64];
    const int64_t t0 = (int64_t)blockIdx.x * SCAN_TILE + (int64_t)threadIdx.x * SCAN_ITEMS;
    int v = 0;
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; ++k)
        if (t0 + k < n) v += in[t0 + k];
    int tot;
    (void)block_incl_scan(v, s_w, &tot);
    if (threadIdx.x == 0) tile_sum[blockIdx.x] = tot;
}

// exclusive scan of the tile totals in place (one workgroup, SCAN_NT per step)
__global__ __launch_bounds__(SCAN_NT) void k_scan_totals(int* __restrict__ tile_sum, int64_t n_tiles) {
    __shared__ int s_w[SCAN_NT / 64];
    int carry = 0;
    for (int64_t b0 = 0; b0 < n_tiles; b0 += SCAN_NT) {
        const int64_t i = b0 + threadIdx.x;
        const int v = i < n_tiles ? tile_sum[i] : 0;
        int tot;
        const int inc = block_incl_scan(v, s_w, &tot);
        if (i < n_tiles) tile_sum[i] = carry + inc - v;
        carry += tot;
    }
}

// LOOK: tile_off holds the tiles' own sums, otherwise the sums before them
template <bool LOOK>
__global__ __launch_bounds__(SCAN_NT) void k_scan_apply(const int* __restrict__ in, int64_t n,
                                                       const int* __restrict__ tile_off, int* __restrict__ out,
                                                       int* __restrict__ tot_dev, int* __restrict__ tot_host) {
    __shared__ int s_w[SCAN_NT / 64];
    const int64_t t0 = (int64_t)blockIdx.x * SCAN_TILE + (int64_t)threadIdx.x * SCAN_ITEMS;
    int v[SCAN_ITEMS], sum = 0, base = 0, tot;
    if (LOOK) {
        int mine = 0;
        for (int b = threadIdx.x; b < (int)blockIdx.x; b += SCAN_NT) mine += tile_off[b];
        (void)block_incl_scan(mine, s_w, &base);
    } else {
        base = tile_off[blockIdx.x];
    }
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; ++k) {
        v[k] = t0 + k < n ? in[t0 + k] : 0;
        sum += v[k];
    }
    int run = block_incl_scan(sum, s_w, &tot) - sum + base;
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; ++k) {
        if (t0 + k < n) out[t0 + k] = run;
        run += v[k];
    }
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) {
        if (tot_dev) *tot_dev = base + tot;
        *tot_host = base + tot;
    }
}

size_t scan_bytes(int64_t n) { return (size_t)((n + SCAN_TILE - 1) / SCAN_TILE) * sizeof(int); }

// tmp: scan_bytes(n) at least, allocated before anything that uses it is in flight
int scan_launch(const int* in, int* out, int64_t n, int* tot_dev, int* tot_host, DevMem& tmp, hipStream_t s) {
    const int64_t tiles = (n + SCAN_TILE - 1) / SCAN_TILE;
    k_scan_tiles<<<(unsigned)tiles, SCAN_NT, 0, s>>>(in, n, tmp.as<int>());
    if (tiles <= SCAN_LOOK) {
        k_scan_apply<true><<<(unsigned)tiles, SCAN_NT, 0, s>>>(in, n, tmp.as<int>(), out, tot_dev, tot_host);
    } else {
        k_scan_totals<<<1, SCAN_NT, 0, s>>>(tmp.as<int>(), tiles);
        k_scan_apply<false><<<(unsigned)tiles, SCAN_NT, 0, s>>>(in, n, tmp.as<int>(), out, tot_dev, tot_host);
    }
    DTC_HIP(hipGetLastError());
    return DTC_OK;
}

}  // namespace

int scan_exclusive_i32(const int* in, int* out, int64_t n, int64_t* total, DevMem& tmp, hipStream_t s) {
    if (n <= 0) { *total = 0; return DTC_OK; }
    HostWords w;
    DTC_TRY(w.alloc(sizeof(int)));
    DTC_TRY(tmp.ensure(scan_bytes(n)));
    DTC_TRY(scan_launch(in, out, n, nullptr, (int*)w.p, tmp, s));
    DTC_HIP(stream_wait(s));
    *total = *(const volatile int*)w.p;
    w.recycle();
    return DTC_OK;
}

int mesh_build_device(const void* phi_dev, int kind, const int64_t n[3], int64_t llimit, int nen,
                      MeshDev& m, hipStream_t s) {
    if (nen != 8 && nen != 20) return set_error(DTC_ERR_BAD_ARGUMENT, "micro element nodes must be 8 or 20, got %d", nen);
    if (kind != DTC_IK1 && kind != DTC_IK2 && kind != DTC_IK4)
        return set_error(DTC_ERR_BAD_ARGUMENT, "voxel kind must be 1, 2 or 4, got %d", kind);
    for (int d = 0; d < 3; ++d)
        if (n[d] <= 0) return set_error(DTC_ERR_BAD_ARGUMENT, "domain extent n[%d] = %lld", d, (long long)n[d]);
    m.nx = (int)n[0]; m.ny = (int)n[1]; m.nz = (int)n[2];
    m.nen = nen; m.mul = nen == 8 ? 1 : 2;
    const int64_t Lx = n[0] * m.mul + 1, Ly = n[1] * m.mul + 1, Lz = n[2] * m.mul + 1;
    const int64_t nvox = n[0] * n[1] * n[2];
    if (Lx * Ly * Lz >= (int64_t)INT32_MAX / 2)
        return set_error(DTC_ERR_BAD_ARGUMENT, "domain of %lld^3 voxels exceeds the 32-bit lattice index", (long long)n[0]);
    m.Lx = (int)Lx; m.Ly = (int)Ly; m.Lz = (int)Lz;
    const int64_t nlat = Lx * Ly * Lz;
    const int nv = (int)nvox;

    // nodes: at most the lattice's, and nen per voxel (the counts stay on the device until
    // the end: one wait for the host instead of one per scan, 20-25 us each)
    const int64_t nmax = std::min<int64_t>(nlat, nvox * nen);
    DTC_TRY(m.solid.ensure(nvox));
    DTC_TRY(m.eidx.ensure(nvox * 4));
    DTC_TRY(m.ftmask.ensure(nvox * 4));
    DTC_TRY(m.nbase.ensure(nvox * 4));
    DTC_TRY(m.parent.ensure(nvox * 4));
    DTC_TRY(m.touch.ensure(nvox));
    DTC_TRY(m.keepE.ensure(nvox * 4));
    DTC_TRY(m.newE.ensure(nvox * 4));
    DTC_TRY(m.numLat.ensure(nlat * 4));
    DTC_TRY(m.latOfNum.ensure(nmax * 4));
    DTC_TRY(m.keepN.ensure(nmax * 4));
    DTC_TRY(m.cref.ensure(nmax * 4));
    DTC_TRY(m.bbox.ensure(6 * 4));
    DTC_TRY(m.tot.ensure(4 * 4));
    DTC_TRY(m.flag.ensure(nvox * 4));
    DTC_TRY(m.scratch.ensure(scan_bytes(std::max(nvox, nmax))));
    if (!m.words.p) DTC_TRY(m.words.alloc(4 * 4));
    int* flag = m.flag.as<int>();
    int* tot = m.tot.as<int>();          // elements, nodes before filtering; elements, nodes kept
    int* hw = (int*)m.words.p;

    auto solid = [&](auto* phi) {
        k_solid<<<grid_of(nvox), NT, 0, s>>>(phi, nv, llimit, m.solid.as<uint8_t>(), flag, m.parent.as<int>(),
                                             m.touch.as<uint8_t>(), m.bbox.as<int>());
    };
    switch (kind) {
    case DTC_IK1: solid((const int8_t*)phi_dev); break;
    case DTC_IK2: solid((const int16_t*)phi_dev); break;
    default: solid((const int32_t*)phi_dev); break;
    }
    DTC_HIP(hipGetLastError());
    DTC_TRY(scan_launch(flag, m.eidx.as<int>(), nvox, tot, hw, m.scratch, s));
    // first-touch numbering, connected components, bounding box of all nodes (in voxel terms)
    if (nen == 8)
        k_voxel<8><<<grid_of(nvox), NT, 0, s>>>(m.solid.as<uint8_t>(), m.nx, m.ny, m.nz, m.ftmask.as<uint32_t>(), flag,
                                                m.parent.as<int>(), m.bbox.as<int>());
    else
        k_voxel<20><<<grid_of(nvox), NT, 0, s>>>(m.solid.as<uint8_t>(), m.nx, m.ny, m.nz, m.ftmask.as<uint32_t>(), flag,
                                                 m.parent.as<int>(), m.bbox.as<int>());
    DTC_HIP(hipGetLastError());
    DTC_TRY(scan_launch(flag, m.nbase.as<int>(), nvox, tot + 1, hw + 1, m.scratch, s));
    k_fill_i32<<<grid_of(nlat), NT, 0, s>>>(m.numLat.as<int>(), nlat, 0);
    k_number<<<grid_of(nvox), NT, 0, s>>>(m.solid.as<uint8_t>(), m.ftmask.as<uint32_t>(), m.nbase.as<int>(), m.nx, m.ny, m.nz,
                                          nen, m.mul, m.Lx, m.Ly, m.numLat.as<int>(), m.latOfNum.as<int>(), m.parent.as<int>());
    // keep rule
    k_touch<<<grid_of(nvox), NT, 0, s>>>(m.solid.as<uint8_t>(), m.eidx.as<int>(), m.parent.as<int>(), m.bbox.as<int>(),
                                         m.nx, m.ny, m.nz, m.touch.as<uint8_t>());
    k_keepE<<<grid_of(nvox), NT, 0, s>>>(m.solid.as<uint8_t>(), m.eidx.as<int>(), m.parent.as<int>(), m.touch.as<uint8_t>(),
                                         nv, tot, m.keepE.as<int>());
    DTC_HIP(hipGetLastError());
    DTC_TRY(scan_launch(m.keepE.as<int>(), m.newE.as<int>(), nvox, tot + 2, hw + 2, m.scratch, s));
    k_keepN<<<grid_of(nmax), NT, 0, s>>>(m.solid.as<uint8_t>(), m.latOfNum.as<int>(), m.parent.as<int>(),
                                         m.touch.as<uint8_t>(), m.nx, m.ny, m.nz, m.mul, m.Lx, m.Ly, (int)nmax, tot,
                                         m.keepN.as<int>());
    DTC_HIP(hipGetLastError());
    DTC_TRY(scan_launch(m.keepN.as<int>(), m.cref.as<int>(), nmax, tot + 3, hw + 3, m.scratch, s));
    DTC_HIP(stream_wait(s));
    const volatile int* h = hw;
    m.n_elems0 = h[0];
    m.n_nodes0 = h[1];
    m.n_elems = h[2];
    m.n_nodes = h[3];
    if (m.n_elems0 == 0) {
        m.n_elems = m.n_nodes = m.n_nodes0 = 0;
        return set_error(DTC_ERR_EMPTY_MESH, "no voxel reaches the iso value limit %lld", (long long)llimit);
    }
    return DTC_OK;
}

int mesh_write_outputs(const MeshDev& m, const double delta[3], const int64_t xa_n[3], double* nodes_dev,
                       int64_t* elems_dev, hipStream_t s) {
    const int64_t nvox = (int64_t)m.nx * m.ny * m.nz;
    if (elems_dev) {
        k_out_elems<<<grid_of(nvox), NT, 0, s>>>(m.keepE.as<int>(), m.newE.as<int>(), m.numLat.as<int>(), m.keepN.as<int>(),
                                                 m.cref.as<int>(), m.nx, m.ny, m.nz, m.nen, m.mul, m.Lx, m.Ly, elems_dev);
        DTC_HIP(hipGetLastError());
    }
    if (nodes_dev) {
        k_out_nodes<<<grid_of(m.n_nodes0), NT, 0, s>>>(m.keepN.as<int>(), m.cref.as<int>(), m.latOfNum.as<int>(),
                                                       (int)m.n_nodes0, m.mul, m.Lx, m.Ly, delta[0], delta[1], delta[2],
                                                       xa_n[0], xa_n[1], xa_n[2], nodes_dev);
        DTC_HIP(hipGetLastError());
    }
    return DTC_OK;
}

}  // namespace dtc
