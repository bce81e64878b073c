// bsolve.hpp -- the 24 x 24 solves of the block PCG.  Included by solver.hip inside its
// anonymous namespace, after lane_f64 (v of lane `lane`, the same for the whole wave).

constexpr double PIVOT_DROP = 1e-9;   // of P^T A P
constexpr double ORTH_DROP = 1e-10;   // of P^T P

// Per domain: takes the Gram sums of k_gram_sum, then
//   mode 0: W = sym(g[0]) = P^T A P is factored as L L^T and L kept; a pivot at
//           or below 1e-9 of its diagonal entry before elimination (or not
//           finite) marks a direction that depends on the previous ones: its
//           column of L is zero and the solves give it a zero coefficient.
//           coef = W^+ g[1];
//   mode 1: coef = -W^+ g[0] with the kept factor;
//   mode 2: G = sym(g[0]) = P^T P is factored the same way (pivots at or below
//           1e-10 dropped, L not kept) and coef = L^-T, so that P coef has
//           orthonormal columns (zero columns for the dropped directions).
// coef[k * 24 + j] multiplies vector column k in the update of column j.
//
// A chain of 24 pivots: latency is all there is.  One wave per domain, no LDS and no barrier
// inside the chain: lane i holds row i of the matrix in registers, and the entries that
// all lanes need are read from the row's lane into scalar registers (v_readlane); for the
// solves lane j holds column j of the right-hand sides.  The three modes take 13, 9 and
// 10 us; 256 threads with the matrix in LDS and three barriers a pivot took 25 each.
template <int MODE>
__global__ __launch_bounds__(64) void k_bsolve(const int* __restrict__ done, const double* __restrict__ gsum,
                                              double* __restrict__ lfac, float* __restrict__ coef) {
    const int d = blockIdx.x, lane = threadIdx.x;
    if (done[d]) return;
    const int row = lane < R ? lane : R - 1;      // (the lanes past 23 repeat the last row)
    double* L = lfac + (int64_t)d * RR;
    const double* G = gsum + (int64_t)d * 2 * RR;
    double a[R], b[R];                            // row `row` of the matrix, column `row` of the right-hand sides
    if (MODE == 1) {
#pragma unroll
        for (int k = 0; k < R; ++k) a[k] = L[row * R + k];
    } else {
#pragma unroll
        for (int k = 0; k < R; ++k) a[k] = 0.5 * (G[row * R + k] + G[k * R + row]);
    }
#pragma unroll
    for (int k = 0; k < R; ++k)
        b[k] = MODE == 2 ? (k == row ? 1.0 : 0.0) : G[(MODE == 0 ? RR : 0) + k * R + row];
    // Entries that are not finite become 0 before the chain: a direction that brings them in
    // has such a diagonal entry too and is dropped, and the products with its 0 stay 0
    double sum = 0.0;
#pragma unroll
    for (int k = 0; k < R; ++k) sum += a[k] + b[k];
    if (!(fabs(sum) < INFINITY))
#pragma unroll
        for (int k = 0; k < R; ++k) {
            if (!(fabs(a[k]) < INFINITY)) a[k] = 0.0;
            if (!(fabs(b[k]) < INFINITY)) b[k] = 0.0;
        }
    double rd = 0.0;                              // 1 / L_kk of this row, 0 for a dropped direction
    if (MODE != 1) {
        constexpr double DROP = MODE == 0 ? PIVOT_DROP : ORTH_DROP;
        double diag = 0.0;                        // this row's diagonal entry before elimination
#pragma unroll
        for (int k = 0; k < R; ++k)
            if (k == row) diag = a[k];
#pragma unroll
        for (int k = 0; k < R; ++k) {
            const double dk = lane_f64(a[k], k);
            const bool keep = dk > DROP * lane_f64(diag, k) && dk < INFINITY;
            const double lk = keep ? sqrt(dk) : 0.0, rk = keep ? 1.0 / lk : 0.0;
            if (row == k) rd = rk;
            a[k] = row == k ? lk : row > k ? a[k] * rk : 0.0;
#pragma unroll
            for (int m = k + 1; m < R; ++m) a[m] -= a[k] * lane_f64(a[k], m);
        }
        if (MODE == 0 && lane < R)
#pragma unroll
            for (int k = 0; k < R; ++k) L[row * R + k] = k <= row ? a[k] : 0.0;
    }
    if (MODE == 1)
#pragma unroll
        for (int k = 0; k < R; ++k)
            if (k == row) rd = a[k] > 0.0 ? 1.0 / a[k] : 0.0;
    // L L^T y = b (modes 0, 1) or L^T y = I (mode 2), each lane its column.  The empty
    // statements hold each entry's lane reads at their step: moved to the front, as the
    // compiler would have them, the 276 values overflow the scalar registers
    if (MODE != 2)
#pragma unroll
        for (int k = 0; k < R; ++k) {
            b[k] *= lane_f64(rd, k);
            asm volatile("" : "+v"(a[k]), "+v"(b[k]));
#pragma unroll
            for (int m = k + 1; m < R; ++m) b[m] -= lane_f64(a[k], m) * b[k];
        }
#pragma unroll
    for (int k = R - 1; k >= 0; --k) {
        b[k] *= lane_f64(rd, k);
#pragma unroll
        for (int m = 0; m < k; ++m) {
            asm volatile("" : "+v"(a[m]), "+v"(b[m]));
            b[m] -= lane_f64(a[m], k) * b[k];
        }
    }
    if (lane < R)
#pragma unroll
        for (int k = 0; k < R; ++k) coef[(int64_t)d * RR + k * R + row] = (float)(MODE == 1 ? -b[k] : b[k]);
}
