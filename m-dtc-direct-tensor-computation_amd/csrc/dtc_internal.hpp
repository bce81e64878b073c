// dtc_internal.hpp -- shared declarations of the gfx950 library (not part of the C ABI).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>
#include <string>
#include <vector>

#include "../../include/dtc_capi.h"

namespace dtc {

// ---------------------------------------------------------------- errors
int set_error(int code, const char* fmt, ...);

#define DTC_HIP(call)                                                                    \
    do {                                                                                 \
        hipError_t e_ = (call);                                                          \
        if (e_ != hipSuccess) {                                                          \
            if (e_ == hipErrorOutOfMemory)                                               \
                return ::dtc::set_error(DTC_ERR_OOM, "%s: %s", #call, hipGetErrorString(e_)); \
            return ::dtc::set_error(DTC_ERR_DEVICE, "%s: %s (%s:%d)", #call,              \
                                    hipGetErrorString(e_), __FILE__, __LINE__);          \
        }                                                                                \
    } while (0)

#define DTC_TRY(expr)              \
    do {                           \
        int rc_ = (expr);          \
        if (rc_ != DTC_OK) return rc_; \
    } while (0)

// Host waits.  Nothing relies on hipStreamSynchronize or hipStreamQuery: where several threads
// launch on streams of their own, both have returned success at once with 0.2 to 0.9 ms of
// work in flight, about once in ten million waits; an event recorded at that moment was
// waited for every time.
// Waits for everything enqueued on s so far: an event's wait decides.  The call before it does
// most of the waiting and clears what the runtime keeps of finished work, which otherwise
// waits for the next such call or the stream's destruction (the mesher, 64^3: 1.08 ms with the
// event alone, 1.02 so, 1.00 with that call alone).
inline hipError_t stream_wait(hipStream_t s) {
    hipEvent_t e;
    hipError_t rc = hipEventCreateWithFlags(&e, hipEventDisableTiming);
    if (rc != hipSuccess) return rc;
    rc = hipEventRecord(e, s);
    if (rc == hipSuccess) {
        (void)hipStreamSynchronize(s);
        rc = hipEventSynchronize(e);
    }
    (void)hipEventDestroy(e);
    return rc;
}
// Waits until *w, a page-locked word that work on s stores, is at least v: where more work is
// enqueued behind it, or a copy of the results is saved.
int wait_word(hipStream_t s, const unsigned long long* w, unsigned long long v);

// ---------------------------------------------------------------- device buffers
// Idle device memory and page-locked host words, kept from one call or object for the next.
// hipFree waits for the device and unmaps: 40 us each, 5 ms after one 64^3 solve, 19 ms
// after 40 domains of 21^3 (one-shot solves 93 -> 85 and 88 -> 62 ms; 27^3 HEX20 32.4 -> 25).
// Only what no stream uses any more goes in (its owner has synchronised them: recycle()
// and Recycle below; anything else is freed), so that any thread may take it out for any
// stream.  What is kept is bounded (POOL_BYTES, POOL_PINNED), the oldest goes first, what
// was not used for POOL_SECONDS is freed at the next call that uses the pool, and all of it
// when an allocation fails or the program asks (dtc_release_memory).  Streams are not kept:
// kept ones end up on one hardware queue, and the parts of a batch no longer overlap (40
// domains of 21^3 61 -> 70 ms).
constexpr size_t POOL_BYTES = (size_t)4 << 30;
// (page-locked: blocks kept, and the largest; a multigrid solve takes up to a dozen sizes)
constexpr size_t POOL_PINNED = 32, POOL_PINNED_BYTES = (size_t)1 << 20;
constexpr double POOL_SECONDS = 20.0;
// allocation size of an n-byte request: up to 1/8 more, so that requests of nearby sizes
// meet; 2 MiB steps from 16 MiB on
inline size_t pool_size(size_t n) {
    size_t step = 4096;
    while (step < ((size_t)2 << 20) && step * 16 <= n) step *= 2;
    return (n + step - 1) / step * step;
}
void* pool_take(size_t n, int dev);               // an idle allocation of n = pool_size(n) bytes, or null
void pool_put(void* p, size_t n, int dev);        // takes ownership
void pool_trim();                                 // frees all idle memory, device and page-locked
void* pool_take_pinned(size_t n);
void pool_put_pinned(void* p, size_t n);

// While one with idle = true lives, what this thread destroys is recycled: no stream may
// use it any more.
extern thread_local bool t_recycle;
struct Recycle {
    bool prev;
    explicit Recycle(bool idle) : prev(t_recycle) { t_recycle = idle; }
    ~Recycle() { t_recycle = prev; }
    Recycle(const Recycle&) = delete;
    Recycle& operator=(const Recycle&) = delete;
};
// The device objects of one call on one stream: a CallEnd declared before them, an
// IdleOnExit after them (it runs first, waits for the stream, and they are recycled).
struct CallEnd {
    bool prev = t_recycle;
    ~CallEnd() { t_recycle = prev; }
};
struct IdleOnExit {
    const hipStream_t& s;
    bool waited = false;   // set by the function: nothing was enqueued after its last wait
    ~IdleOnExit() { t_recycle = s && (waited || stream_wait(s) == hipSuccess); }
};

// Owning device allocation; allocation failure is reported as DTC_ERR_OOM.
struct DevMem {
    void* p = nullptr;
    size_t bytes = 0;
    int dev = 0;
    DevMem() = default;
    DevMem(const DevMem&) = delete;
    DevMem& operator=(const DevMem&) = delete;
    DevMem(DevMem&& o) noexcept : p(o.p), bytes(o.bytes), dev(o.dev) { o.p = nullptr; o.bytes = 0; }
    DevMem& operator=(DevMem&& o) noexcept {
        if (this != &o) {
            release();
            p = o.p; bytes = o.bytes; dev = o.dev;
            o.p = nullptr; o.bytes = 0;
        }
        return *this;
    }
    ~DevMem() { release(); }
    void release() {
        if (p && t_recycle) pool_put(p, bytes, dev);
        else if (p) (void)hipFree(p);
        p = nullptr;
        bytes = 0;
    }
    // gives the memory up; the caller has waited for every stream that uses it
    void recycle() {
        Recycle r(true);
        release();
    }
    int alloc(size_t n) {
        release();
        n = pool_size(n == 0 ? 16 : n);
        DTC_HIP(hipGetDevice(&dev));
        p = pool_take(n, dev);
        if (!p) {
            hipError_t e = hipMalloc(&p, n);
            if (e == hipErrorOutOfMemory) {
                (void)hipGetLastError();
                pool_trim();
                e = hipMalloc(&p, n);
            }
            if (e != hipSuccess) {
                p = nullptr;
                (void)hipGetLastError();
                return set_error(DTC_ERR_OOM, "hipMalloc(%zu bytes) failed: %s", n, hipGetErrorString(e));
            }
        }
        bytes = n;
        return DTC_OK;
    }
    // keep the allocation when it is large enough (repeated runs reuse buffers)
    int ensure(size_t n) {
        if (p && bytes >= n) return DTC_OK;
        return alloc(n);
    }
    template <typename T> T* as() const { return static_cast<T*>(p); }
};

// Page-locked host memory that the device writes, given up with the owner.  The solver keeps
// a summary word and then each domain's status in it.
struct HostWords {
    void* p = nullptr;
    size_t n = 0;
    HostWords() = default;
    HostWords(const HostWords&) = delete;
    HostWords& operator=(const HostWords&) = delete;
    ~HostWords() { reset(); }
    int alloc(size_t bytes) {
        bytes = pool_size(bytes);
        p = pool_take_pinned(bytes);
        if (!p) DTC_HIP(hipHostMalloc(&p, bytes, hipHostMallocDefault));
        n = bytes;
        return DTC_OK;
    }
    void reset() {
        if (p && t_recycle) pool_put_pinned(p, n);
        else if (p) (void)hipHostFree(p);
        p = nullptr;
        n = 0;
    }
    // as DevMem::recycle
    void recycle() {
        Recycle r(true);
        reset();
    }
    unsigned long long* word() const { return (unsigned long long*)p; }
    double* status() const { return (double*)p + 8; }
};

// ---------------------------------------------------------------- constants
constexpr int R24 = 24;          // load cases of the HEX08 macro element
constexpr int BX = 8, BY = 4, BZ = 4;   // owned nodes of one solver brick
constexpr int EX = BX + 1, EY = BY + 1, EZ = BZ + 1;   // elements that touch a brick's nodes

// HEX08 local node offsets in gen_quadmesh order (f-src/mod_gen_quadmesh.f90:298-306)
__host__ __device__ constexpr int h08_off(int l, int d) {
    // l: 0..7, d: 0..2
    return (d == 0) ? ((l == 1 || l == 2 || l == 5 || l == 6) ? 1 : 0)
         : (d == 1) ? ((l == 2 || l == 3 || l == 6 || l == 7) ? 1 : 0)
                    : (l >= 4 ? 1 : 0);
}

// ---------------------------------------------------------------- mesher
struct MeshDev {
    int nx = 0, ny = 0, nz = 0, nen = 8, mul = 1;
    int Lx = 0, Ly = 0, Lz = 0;       // lattice extents
    int64_t n_elems0 = 0, n_nodes0 = 0;   // before connectivity filtering
    int64_t n_elems = 0, n_nodes = 0;     // kept
    DevMem flag;      // int32 per voxel: counts of the running scan
    DevMem solid;     // uint8 per voxel
    DevMem eidx;      // int32 per voxel: element index before filtering
    DevMem ftmask;    // uint32 per voxel: first-touched local nodes
    DevMem nbase;     // int32 per voxel: first node number - 1 of the voxel's first touches
    DevMem numLat;    // int32 per lattice node: node number (1-based), 0 = unused
    DevMem latOfNum;  // int32 per node number: lattice index
    DevMem parent;    // int32 per voxel: union-find
    DevMem touch;     // uint8 per voxel (component roots)
    DevMem keepE;     // int32 per voxel
    DevMem newE;      // int32 per voxel: kept element index
    DevMem keepN;     // int32 per node number
    DevMem cref;      // int32 per node number: kept node number - 1
    DevMem bbox;      // int32[6]
    DevMem tot;       // int32[4]: counts of the four scans
    HostWords words;  // the same on the host
    DevMem scratch;   // scan temp storage
};

// Builds the mesh of one voxel block already resident on the device.
// Returns DTC_ERR_EMPTY_MESH when no voxel reaches llimit.
int mesh_build_device(const void* phi_dev, int kind, const int64_t n[3], int64_t llimit, int nen,
                      MeshDev& m, hipStream_t s);
// Writes nodes (3 x N, column-major) and elems (nen x N_e, 1-based) to device buffers.
int mesh_write_outputs(const MeshDev& m, const double delta[3], const int64_t xa_n[3],
                       double* nodes_dev, int64_t* elems_dev, hipStream_t s);

// exclusive prefix sum of int32 (n items), total returned through *total (host)
int scan_exclusive_i32(const int* in, int* out, int64_t n, int64_t* total, DevMem& tmp, hipStream_t s);

// ---------------------------------------------------------------- solver topology
struct DomInfo {
    int nx, ny, nz;           // voxels per edge
    int macro_order;          // 1: HEX08 macro element (24 load cases), 2: HEX20 (60)
    int lc_base;              // first macro load case of this group of 24
    int bnx, bny, bnz;        // brick grid
    int brick_begin, brick_end;
    int cl_begin, cl_end;     // HEX08: matvec clusters (ClusterInfo)
    int64_t lat_off;          // offset into the lattice map
    int64_t vox_off;          // offset into the voxel modulus array
    int64_t node_begin, node_end;
    double min_c[3], max_c[3];   // domain box (f-src/mod_struct_preprocess.f90:516-517)
    double xa1[3];               // (xa_n - 1)
    double delta[3];
};

struct BrickInfo {
    int dom;
    int x0, y0, z0;           // first owned lattice node
    int node_begin, node_end; // owned solver nodes (contiguous)
};

// A HEX08 matvec work unit: a run of consecutive solver nodes (of one or more bricks)
// with every element that touches one of them.  At most CL_CAP nodes, CL_CAP64 in the
// batches solved in FP64: the cap bounds the accumulators that a workgroup of k_ebe
// keeps in LDS (288 or 576 bytes a node).
constexpr int CL_CAP = 128, CL_CAP64 = 64;
struct ClusterInfo {
    int dom;
    int node_begin, node_end;
    int brick_begin, brick_end;   // bricks that hold the nodes
    int e_off, e_cnt;             // elements in the cluster element tables
};

// New Chebyshev-Jacobi direction of one unknown, c1 d + c2 D^-1 (b - t) with t = (K x)
// of the unknown: one expression for every kernel that forms it, so that a step fused
// into an operator's epilogue rounds like the separate vector kernel (the fused
// multiply-add is written out: left to contraction it may take either product)
__device__ __forceinline__ float cheb_dir(float c1, float d, float c2, float di, float b, float t) {
    return __builtin_fmaf(c1, d, c2 * di * (b - t));
}

// 45 coefficients of the HEX08 element stiffness in the signed Walsh basis
// (E = 1); see walsh_blocks() in solver.hip.
struct WalshK {
    double g[45];
};

}  // namespace dtc
